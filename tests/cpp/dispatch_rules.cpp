// The library's rules on sizes (csrc/dispatch.hpp) for a test to ask.
#include "dispatch.hpp"

extern "C" {
int gemm_tall_shape(int rows, int K, int N, int vs_lds) {
  return nnhip::gemm_tall_shape(rows, K, N, vs_lds != 0);
}
int attention_prompt_shape(int B, int S, int H, int D, int q8, int max_keys) {
  return nnhip::attention_prompt_shape(B, S, H, D, q8 != 0, max_keys);
}
int gemm_f32_shape(int rows, int N) { return nnhip::gemm_f32_shape(rows, N); }
int gemm_f32_waves(int rows, int K, int N) { return nnhip::gemm_f32_waves(rows, K, N); }
int sum_short_shape(long long n_out, long long n_red, int along_r) {
  return nnhip::sum_short_shape(n_out, n_red, along_r != 0);
}
int matmul_short_shape(long long M, long long N, long long K) {
  return nnhip::matmul_short_shape(M, N, K);
}
}
