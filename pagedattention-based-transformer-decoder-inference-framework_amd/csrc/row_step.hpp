// A decode step's layers of a small INT8 decoder as one launch (csrc/row_step.hip).
#pragma once

#include <hip/hip_runtime.h>

#include <cstddef>
#include <cstdint>

#include "llm_decoder.h"

namespace llm {

// One projection of all layers: packed weights (`stride` bytes a layer), [L][N] column scales, [L][N]
// biases (NULL: none).
struct RowProduct {
  const uint8_t* w = nullptr;
  size_t stride = 0;
  const float* scale = nullptr;
  const float* bias = nullptr;
};

// Row m is page-table row m, its new token at pos[m] and its embedding E[tok[m]].  Pages of fp16.
struct RowStep {
  int L = 0, D = 0, V = 0, rows = 0;
  const _Float16* emb = nullptr;
  const int32_t* tok = nullptr;
  const int32_t* pos = nullptr;
  const float *ln1_g = nullptr, *ln1_b = nullptr, *ln2_g = nullptr, *ln2_b = nullptr;  // [L][hidden]
  float eps = 1e-5f;
  RowProduct qkv, o, fc1, fc2;
  const int32_t* page_table = nullptr;  // [L][beams][H][max_tiles]
  int beams = 0, max_tiles = 0, num_pages = 0;
  int page_shift = 0;  // log2 of a page's tokens
  _Float16* k_pool = nullptr;
  _Float16* v_pool = nullptr;
  size_t page_stride = 0;  // elements
  float attn_scale = 1.f;
  float* x = nullptr;  // [rows][hidden] after the last layer
  float* q = nullptr;  // [rows][hidden] the last layer's queries (llm_decoder_run_attention)
  // Taps (llm_decoder_set_taps; NULL: none): slot 4 layer + stage has int8 rows in packed-A order from
  // tap_q + slot tap_stride and their scales from tap_s + slot tap_rows.
  int8_t* tap_q = nullptr;
  float* tap_s = nullptr;
  size_t tap_stride = 0;
  int tap_rows = 0;
};

constexpr int kRowStepHidden = 256;
// Sizes that it is made for, and whether it is faster than the layers' own launches for so many rows of at
// most `longest` tokens.
bool row_step_ok(int hidden, int inter, int D, int page_size, int rows, int longest);
hipError_t row_step(const RowStep& a, hipStream_t st);

}  // namespace llm
