// The executables of a decode step.
#pragma once

#include <algorithm>

namespace llm {

// One for each of the ways that a step can go (llm_decoder::rows_alone): a step that takes the other way as
// its rows grow finds that one's where it was left, and makes none anew in the middle of a sequence.
template <typename Exec, int WAYS>
struct StepGraphs {
  Exec exec[WAYS] = {};
  int rows[WAYS];  // that it steps (-1: to be made anew)

  StepGraphs() { stale(); }
  void stale() { std::fill_n(rows, WAYS, -1); }  // what a step does has changed

  // The executable of `n` rows by `way`.  wait() returns once no launch of the one that is replaced runs any
  // more; make(Exec*) builds; both return a status (0: done).  What fails leaves nothing that a later call
  // would take for whole.
  template <typename Wait, typename Drop, typename Make>
  int get(int way, int n, const Wait& wait, const Drop& drop, const Make& make, Exec* out) {
    if (rows[way] != n) {
      if (const int rc = wait()) return rc;
      rows[way] = -1;
      if (exec[way]) drop(exec[way]);
      exec[way] = Exec{};
      Exec made{};
      if (const int rc = make(&made)) return rc;
      exec[way] = made;
      rows[way] = n;
    }
    *out = exec[way];
    return 0;
  }

  template <typename Drop>
  void clear(const Drop& drop) {
    stale();
    for (Exec& e : exec) {
      if (e) drop(e);
      e = Exec{};
    }
  }
};

}  // namespace llm
