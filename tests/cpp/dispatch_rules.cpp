// The library's rules on sizes (csrc/dispatch.hpp) for a test to ask.
#include "dispatch.hpp"

extern "C" {
int gemm_tall_shape(int rows, int K, int N, int vs_lds) {
  return nnhip::gemm_tall_shape(rows, K, N, vs_lds != 0);
}
}
