// Ring tiles: block_gemm_kernel with one small tile per workgroup and three or more stage buffers, for problems
// whose 256 x 256 or 128 x 128 tiles would leave compute units idle.
//
// Such a problem is bound by latency: a workgroup has a compute unit nearly to itself, and its chain of stages
// (wait, barrier, fragment reads, products, fold) sets the time, K / 128 times over.  So the tile is the smallest
// that still gives every compute unit work once, each wave gets one or two 32 x 32 blocks (a short chain and a
// short fold), and two or more stages are always in flight.  Time per 128-channel stage with one workgroup on a
// compute unit, int8 g128 / int8 per token / fp8 blocks (us): 64 channels x 32 tokens 0.42 / 0.25 / 0.31, 64 x 64
// 0.45 / 0.28 / 0.36, 128 x 64 0.63 / 0.41 / 0.47, 128 x 128 in eight waves 0.90 / 0.47 / 0.60, against 0.90 / 0.79 /
// 0.83 for the two-stage 128 x 128 tile of four waves and 1.97 / 1.2 / 1.35 for the 256 x 256 tile.  (The g128 fold leaves
// the 128 x 128 ring nothing to gain, and it is not built.)
#pragma once

#include "gemm_launch.h"

namespace hn {

enum class RingTile { kNone, k64x32, k64x64, k128x64, k128x128 };  // channels x tokens

// The smallest tile that covers the problem in one round of workgroups; 128 x 64 also serves two per compute unit,
// where it fills the chip better than 128 x 128 tiles that no longer fit one round (300 x 2048 -> 12288: 25.8 -> 22.1
// us g128, 20.1 -> 17.4 per token).  Larger problems keep the persistent tiles: from two full rounds of 128 x 128 on
// those move fewer bytes per product (1024 x 3072 -> 12288: 72 us against 85).  So do, over random sizes of the class:
//   int8 g128 where only 128 x 128 tiles fit one round: that ring took 0.89 to 1.14 of the two-stage tile's time, 1.04 at
//     the median (844 x 2816 -> 3584 19.8 against 22.2 us, 605 x 3840 -> 6400 32.6 against 36.7); 128 x 64 two to a
//     compute unit up to 1.23 of it;
//   fp8 blocks of K > 8192 with two 128 x 64 to a compute unit: 0.84 to 1.07 of it (555 x 15488 -> 7100 118 against 126);
//     0.69 to 1.00 of it up to 8192.
// GEMM alone, old and new (us):
//   tokens x K -> N        int8 g128        int8 per token   fp8 blocks
//   32 x 12288 -> 3072     92.8 -> 44.4     85.1 -> 28.3     90.7 -> 32.3
//   100 x 3072 -> 3072     27.1 -> 11.1     24.8 -> 9.4      26.5 -> 10.2
//   200 x 12288 -> 3072    94.5 -> 36.1     84.0 -> 29.3     91.0 -> 32.1
//   500 x 3072 -> 3072     26.9 -> 19.8     24.1 -> 15.0     25.6 -> 16.8
//   1024 x 3072 -> 3072    23.4             20.3 -> 16.1     21.6 -> 18.6
template <int KIND, bool G128>
inline RingTile choose_ring(int64_t M, int64_t N, int64_t K) {
  const int64_t cus = cu_count();
  auto tiles = [&](int64_t bn, int64_t bm) { return ((N + bn - 1) / bn) * ((M + bm - 1) / bm); };
  if (tiles(64, 32) <= cus) return RingTile::k64x32;
  if (tiles(64, 64) <= cus) return RingTile::k64x64;
  if (tiles(128, 64) <= cus) return RingTile::k128x64;
  if (tiles(128, 128) <= cus) return KIND == HN_KIND_INT8 && G128 ? RingTile::kNone : RingTile::k128x128;
  if (tiles(128, 64) <= 2 * cus && (KIND != HN_KIND_FP8 || K <= 8192)) return RingTile::k128x64;
  return RingTile::kNone;
}

template <int KIND, int EPI, bool G128, int OUT_DT, bool WBLK>
static int launch_ring_tile(RingTile tile, GemmArgs& a, hipStream_t st) {
  switch (tile) {
    case RingTile::k64x32: return launch_cfg<KIND, EPI, G128, 2, 1, 1, 1, OUT_DT, 128, 4, WBLK, 2>(a, st);
    case RingTile::k64x64: return launch_cfg<KIND, EPI, G128, 2, 2, 1, 1, OUT_DT, 128, 4, WBLK, 2>(a, st);
    case RingTile::k128x64: return launch_cfg<KIND, EPI, G128, 2, 2, 2, 1, OUT_DT, 128, 3, WBLK, 2>(a, st);
    default:
      if constexpr (KIND == HN_KIND_INT8 && G128) return HN_ERR_UNSUPPORTED;  // (choose_ring names no such tile)
      else return launch_cfg<KIND, EPI, G128, 2, 4, 2, 1, OUT_DT, 128, 4, WBLK, 2>(a, st);
  }
}

template <int KIND, bool G128, bool WBLK>
static int launch_ring(GemmArgs& a, int epilogue, int out_dtype, hipStream_t st, bool* taken) {
  const RingTile tile = choose_ring<KIND, G128>(a.M, a.N, a.K);
  *taken = tile != RingTile::kNone && (epilogue == HN_EPI_NONE || epilogue == HN_EPI_GELU) &&
           (out_dtype == HN_DTYPE_BF16 || out_dtype == HN_DTYPE_F16);
  if (!*taken) return HN_OK;
  if (epilogue == HN_EPI_NONE)
    return out_dtype == HN_DTYPE_BF16 ? launch_ring_tile<KIND, HN_EPI_NONE, G128, HN_DTYPE_BF16, WBLK>(tile, a, st)
                                      : launch_ring_tile<KIND, HN_EPI_NONE, G128, HN_DTYPE_F16, WBLK>(tile, a, st);
  return out_dtype == HN_DTYPE_BF16 ? launch_ring_tile<KIND, HN_EPI_GELU, G128, HN_DTYPE_BF16, WBLK>(tile, a, st)
                                    : launch_ring_tile<KIND, HN_EPI_GELU, G128, HN_DTYPE_F16, WBLK>(tile, a, st);
}

}  // namespace hn
