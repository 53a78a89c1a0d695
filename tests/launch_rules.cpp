// The launch rules (csrc/launch_rules.hpp) behind a C interface, for the CPU tests.
#include "launch_rules.hpp"

using namespace iehip;

extern "C" int prefill_kernel(int T, int n_heads, int n_kv_heads, int split, int cus) {
  return int(choose_prefill(T, n_heads, n_kv_heads, split != 0, cus));
}
extern "C" int prefill_f32_kernel(int T, int n_heads, int cus) {
  return int(choose_prefill_f32(T, n_heads, cus));
}
extern "C" int tile(int gate, int rows, int cols, int T, int cus) {
  return choose_tile(gate != 0, rows, cols, T, cus);
}
extern "C" int short_k(int64_t tiles, int cols, int norm, int cus) {
  return short_k_staged(tiles, cols, norm != 0, cus);
}
extern "C" int decode_waves(int chunk_tokens) { return decode_f32_waves(chunk_tokens); }
extern "C" int offsets_fit(int rows, int tokens, int64_t cols, int weight_bytes) {
  return tile_offsets_fit(rows, tokens, cols, weight_bytes);
}
extern "C" int wide_kernel(int gate, int cols, int T) { return int(choose_wide(gate != 0, cols, T)); }
