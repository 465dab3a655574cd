// Launch of one block_gemm_kernel configuration, shared by the files that instantiate them.
#pragma once

#include "gemm_kernel.h"

namespace hn {

// WPE: waves per SIMD the kernel is compiled for; above WN * WM / 4, several workgroups share a CU and the
// persistent grid grows to match.
template <int KIND, int EPI, bool G128, int WN, int WM, int TN, int TM, int OUT_DT, int BK, int NS, bool WBLK = false,
          int WPE = WN * WM / 4>
static int launch_cfg(GemmArgs& a, hipStream_t st) {
  constexpr int BN = WN * TN * 32, BM = WM * TM * 32;
  const int64_t tm = (a.M + BM - 1) / BM, tn = (a.N + BN - 1) / BN;
  if (tm * tn > 0x7fffffff) {
    set_error("hn_block_gemm: problem too large (%lld tiles)", (long long)(tm * tn));
    return HN_ERR_UNSUPPORTED;
  }
  a.tiles_m = (int)tm;
  a.tiles_n = (int)tn;
  const int64_t slots = (int64_t)cu_count() * (WPE * 4 / (WN * WM));
  const int64_t grid = NS > 2 || tm * tn < slots ? tm * tn : slots;  // a ring (NS > 2) takes one tile per workgroup
  hipLaunchKernelGGL((block_gemm_kernel<KIND, EPI, G128, WN, WM, TN, TM, OUT_DT, BK, NS, WBLK, WPE>),
                     dim3((unsigned)grid), dim3(WN * WM * 64), 0, st, a);
  return HN_LAUNCH_CHECK("block_gemm_kernel");
}

// The ring tiles (gemm_ring.h), by code kind: small problems of the plain and GELU epilogues with 2-byte outputs.
// Sets `taken` if a ring tile serves the problem.
int launch_ring_int8(GemmArgs& a, bool g128, int epilogue, int out_dtype, hipStream_t st, bool* taken);
int launch_ring_fp8(GemmArgs& a, int epilogue, int out_dtype, hipStream_t st, bool* taken);

}  // namespace hn
