// C entry points of csrc/gemm_split.hpp for tests/test_gemm_split_host.py.
#include "../../tensornetworks.jl_amd/csrc/gemm_split.hpp"

extern "C" {
int ksplit_wanted(int cu, int prec, int M, int N, int K) { return tnh::gs::ksplit_wanted(cu, prec, M, N, K); }
int wide_slices(int cu, int prec, int M, int N, int K, int may_split) {
  return tnh::gs::wide_slices(cu, prec, M, N, K, may_split != 0);
}
int slice_width(int K, int slices) { return tnh::gs::slice_width(K, slices); }
}
