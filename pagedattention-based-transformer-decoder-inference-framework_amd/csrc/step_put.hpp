// What a decode step's launch takes along for the device: words (the rows' tokens) and the place of
// the step's logits.
#pragma once

#include <algorithm>
#include <cstdint>

namespace llm {

// Up to kPut words and the place of a step's logits, out of the launch's own arguments: one launch in
// place of copies from pageable memory before a step and of the logits' copy behind it (which a
// captured step needs, since its own arguments are fixed).  A prompt of 113 tokens and 16 steps
// of one row, 2 layers of hidden 256: 1,191 us, now 1,137.
constexpr int kPut = 128;
struct StepPut {
  int32_t* to;
  int32_t* to2;  // (optional) takes v2
  float** place; // (optional) takes logits
  float* logits;
  int n;
  int32_t v2, v[kPut];
};

// tokens (null: those on the device) of `rows` rows to `to`, `logits` (null: nowhere) to *place, by
// launches, which return a status (0: done).  `placed`: *place is not null; nothing is launched where
// nothing changes.  The place goes with the last launch, so that after one that failed *place and
// `placed` are as they were: a place that is no longer the caller's is never left behind.
template <typename Launch>
int put_step(const int32_t* tokens, int rows, int32_t* to, float** place, float* logits, bool& placed,
             const Launch& launch) {
  if (!tokens && !logits && !placed) return 0;
  const int words = tokens ? rows : 0;
  int at = 0;
  do {
    StepPut a{};
    a.to = to + at;
    a.n = std::min(kPut, words - at);
    std::copy_n(tokens + at, a.n, a.v);
    at += a.n;
    if (at == words) {
      a.place = place;
      a.logits = logits;
    }
    if (const int rc = launch(a)) return rc;
  } while (at < words);
  placed = logits != nullptr;
  return 0;
}

}  // namespace llm
