// Dispatch and C ABI of the block-scaled 8-bit GEMM (hy_nomas/kernels.py:152-170, block_gemm).
// The kernel template and its design notes are in gemm_kernel.h.
#include "gemm_launch.h"
#include "skinny_kernel.h"

namespace hn {

// int8 codes lie in [-128, 127], so a whole-K int32 dot product is exact for K < 2^17.
constexpr int64_t kWholeKInt32Limit = 131072;

// ---------------------------------------------------------------------------------------------
// configurations

// The rows of a problem, as two launches: a.M rows from row 0 with the big tile, then the rest with a 128 x 128
// tile.  Tile rows are independent and every output keeps its fold order, so the results do not depend on
// where the split falls.
enum class TileSplit { kBig, kMid, kSmall, kBoth };

// Which tiles serve an M x N problem whose big tile is bm x bn with `slots` workgroups resident (one round of
// tiles), and for kBoth the rows the big tile takes.  A persistent grid runs ceil(tiles / slots) rounds of
// tiles; when the last round would leave more than half of the compute units idle, its rows go to 128 x 128
// tiles (four per big tile, on every compute unit).  A problem with fewer big tiles than half a round runs on
// small tiles alone, and one whose bn x 192 tiles still fit one round takes those: the round is shorter (256 x 192
// against 256 x 256 tiles, us, g128 / per token / fp8 blocks: 3520 x 12288 -> 3072 227 / 129 / 138 -> 190 / 120 / 131,
// 3520 x 3072 -> 3072 55.5 / 38.4 / 41.1 -> 50.2 / 35.2 / 37.1, 5000 x 8192 -> 2048 130 / 84 / 96 -> 118 / 79 / 89).  With
// more rounds than one they lose what they gain: a round of them takes 0.9 of the big tile's for 0.75 of its work.
static TileSplit choose_tiles(int64_t M, int64_t N, int bm, int bn, int64_t slots, int64_t* big_rows) {
  const int64_t tm = (M + bm - 1) / bm, tn = (N + bn - 1) / bn, tiles = tm * tn;
  const int64_t full = tiles / slots, rem = tiles % slots;
  if (full == 0 && rem > slots / 2 && (M + 191) / 192 * tn <= slots) return TileSplit::kMid;
  if (rem == 0 || rem > slots / 2) return TileSplit::kBig;
  if (full == 0) return TileSplit::kSmall;
  const int64_t rows = (full * slots / tn) * bm;  // whole tile rows of the full rounds
  if (rows <= 0 || rows >= M) return TileSplit::kBig;
  *big_rows = rows;
  return TileSplit::kBoth;
}

// Launch the tile configurations BIG, MID and SMALL (each a launch_cfg instantiation) over the rows choose_tiles
// assigns them.
template <int BM, int BN, int WN, int WM, int WPE, typename Big, typename Mid, typename Small>
static int launch_split(GemmArgs& a, int out_esz, hipStream_t st, Big big, Mid mid, Small small) {
  const int64_t slots = (int64_t)cu_count() * (WPE * 4 / (WN * WM));
  int64_t rows = 0;
  const TileSplit how = choose_tiles(a.M, a.N, BM, BN, slots, &rows);
  if (how == TileSplit::kBig) return big(a);
  if (how == TileSplit::kMid) return mid(a);
  if (how == TileSplit::kSmall) return small(a);
  GemmArgs head = a, tail = a;
  head.M = rows;
  tail.M = a.M - rows;
  tail.qa = a.qa + rows * a.lda;
  tail.sa = a.sa + rows * a.ldsa;
  tail.out = static_cast<char*>(a.out) + rows * a.ldo * out_esz;
  const int rc = big(head);
  return rc != HN_OK ? rc : small(tail);
}

// per-token / per-channel: 256 x 256 tile, 8 waves of 128 x 64.  fp8 with block weight scales: the same
// tile (the running sum is rescaled in place, so there is no second accumulator set).  Other g128 layouts:
// 256 x 128, 8 waves of 128 x 32 (the int32 group partial and the fp32 running sum both fit in 256
// VGPRs).  128-byte K stages in two LDS buffers.  The plain and GELU epilogues also have tiles for problems, or
// tails of problems, that would leave many compute units idle with the big tile (choose_tiles): 256 channels x 192
// tokens in eight waves of 64 x 96, and 128 x 128 in four waves (64 x 64 each, or 128 x 32 with block weight scales), of
// which two workgroups share a compute unit (about 70 KB of LDS each).
template <int KIND, int EPI, int OUT_DT>
static int launch_group(GemmArgs& a, bool g128, hipStream_t st) {
  constexpr bool SWIGLU = EPI == HN_EPI_SWIGLU_QUANT;
  constexpr bool SMALL_OK = EPI == HN_EPI_NONE || EPI == HN_EPI_GELU;
  // epilogues that need a token's 128 channels in one wave: four waves of 128 x 32 where the problem would fill at
  // most half of the compute units with the big tile (200 x 3072 -> 9216 q/k/v heads 64 -> 32 us g128, 49 -> 28 per
  // token; -> 12288 GELU + requantization 68 -> 32 and 54 -> 30)
  constexpr bool WAVE_ROWS = KIND == HN_KIND_INT8 && (EPI == HN_EPI_GELU_QUANT || EPI == kEpiQkvHeads);
  constexpr int ESZ = OUT_DT == HN_DTYPE_F32 ? 4 : 2;
  if (!g128) {
    auto big = [&](GemmArgs& x) { return launch_cfg<KIND, EPI, false, 2, 4, 4, 2, OUT_DT, 128, 2>(x, st); };
    if constexpr (SMALL_OK) {
      auto mid = [&](GemmArgs& x) { return launch_cfg<KIND, EPI, false, 4, 2, 2, 3, OUT_DT, 128, 2>(x, st); };
      auto small = [&](GemmArgs& x) { return launch_cfg<KIND, EPI, false, 2, 2, 2, 2, OUT_DT, 128, 2, false, 2>(x, st); };
      return launch_split<256, 256, 2, 4, 2>(a, ESZ, st, big, mid, small);
    }
    if constexpr (WAVE_ROWS)
      if (int64_t rows = 0; choose_tiles(a.M, a.N, 256, 256, cu_count(), &rows) == TileSplit::kSmall)
        return launch_cfg<KIND, EPI, false, 1, 4, 4, 1, OUT_DT, 128, 2, false, 2>(a, st);
    return big(a);
  }
  if constexpr (KIND == HN_KIND_FP8) {
    if (a.sw_rows == 128) {
      auto big = [&](GemmArgs& x) { return launch_cfg<KIND, EPI, true, 2, 4, 4, 2, OUT_DT, 128, 2, true>(x, st); };
      if constexpr (SMALL_OK) {
        auto mid = [&](GemmArgs& x) { return launch_cfg<KIND, EPI, true, 4, 2, 2, 3, OUT_DT, 128, 2, true>(x, st); };
        auto small = [&](GemmArgs& x) {
          return launch_cfg<KIND, EPI, true, 1, 4, 4, 1, OUT_DT, 128, 2, true, 2>(x, st);
        };
        return launch_split<256, 256, 2, 4, 2>(a, ESZ, st, big, mid, small);
      }
      return big(a);
    }
  }
  if constexpr (!SWIGLU) {
    if constexpr (KIND == HN_KIND_INT8) {  // (fp8 block scales took the branch above)
      if (a.sw_rows == 128) return launch_cfg<KIND, EPI, true, 2, 4, 4, 1, OUT_DT, 128, 2, true>(a, st);
    }
    auto big = [&](GemmArgs& x) { return launch_cfg<KIND, EPI, true, 2, 4, 4, 2, OUT_DT, 128, 2>(x, st); };
    if constexpr (SMALL_OK) {
      auto mid = [&](GemmArgs& x) { return launch_cfg<KIND, EPI, true, 4, 2, 2, 3, OUT_DT, 128, 2>(x, st); };
      auto small = [&](GemmArgs& x) { return launch_cfg<KIND, EPI, true, 2, 2, 2, 2, OUT_DT, 128, 2, false, 2>(x, st); };
      return launch_split<256, 256, 2, 4, 2>(a, ESZ, st, big, mid, small);
    }
    if constexpr (WAVE_ROWS)
      if (int64_t rows = 0; choose_tiles(a.M, a.N, 256, 256, cu_count(), &rows) == TileSplit::kSmall)
        return launch_cfg<KIND, EPI, true, 1, 4, 4, 1, OUT_DT, 128, 2, false, 2>(a, st);
    return big(a);
  }
  set_error("hn_block_gemm: swiglu_quant needs per-token scales or fp8 with 128 x 128 block weight scales");
  return HN_ERR_UNSUPPORTED;
}

template <int KIND, int EPI>
static int launch_out(GemmArgs& a, bool g128, int out_dtype, hipStream_t st) {
  if constexpr (EPI == HN_EPI_GELU_QUANT || EPI == HN_EPI_ACC32 || EPI == HN_EPI_SWIGLU_QUANT) {
    return launch_group<KIND, EPI, HN_DTYPE_BF16>(a, g128, st);
  } else {
    if (out_dtype == HN_DTYPE_BF16) return launch_group<KIND, EPI, HN_DTYPE_BF16>(a, g128, st);
    if (out_dtype == HN_DTYPE_F16) return launch_group<KIND, EPI, HN_DTYPE_F16>(a, g128, st);
    return launch_group<KIND, EPI, HN_DTYPE_F32>(a, g128, st);
  }
}

template <int KIND>
static int launch_kind(GemmArgs& a, bool g128, int epilogue, int out_dtype, hipStream_t st) {
  switch (epilogue) {
    case HN_EPI_NONE: return launch_out<KIND, HN_EPI_NONE>(a, g128, out_dtype, st);
    case HN_EPI_GELU: return launch_out<KIND, HN_EPI_GELU>(a, g128, out_dtype, st);
    case HN_EPI_GELU_QUANT: return launch_out<KIND, HN_EPI_GELU_QUANT>(a, g128, out_dtype, st);
    case HN_EPI_SWIGLU_QUANT: return launch_out<KIND, HN_EPI_SWIGLU_QUANT>(a, g128, out_dtype, st);
    default: break;
  }
  set_error("hn_block_gemm: bad epilogue %d", epilogue);
  return HN_ERR_ARG;
}

// M <= 4 int8 (the per-sample linears): one wave per 4 weight rows, v_dot4 on the streamed weights.
template <int MT, int MODE, int EPI>
static int launch_skinny_out(GemmArgs& a, int out_dtype, hipStream_t st) {
  constexpr int64_t ROWS = kSkinnyRows * kSkinnyWaves;
  const int64_t grid = (a.N + ROWS - 1) / ROWS;
  if (grid > 0x7fffffff) {
    set_error("hn_block_gemm: problem too large (N=%lld)", (long long)a.N);
    return HN_ERR_UNSUPPORTED;
  }
  const dim3 g((unsigned)grid), b(kSkinnyWaves * 64);
  if (out_dtype == HN_DTYPE_BF16) hipLaunchKernelGGL((skinny_gemm_kernel<MT, MODE, EPI, HN_DTYPE_BF16>), g, b, 0, st, a);
  else if (out_dtype == HN_DTYPE_F16) hipLaunchKernelGGL((skinny_gemm_kernel<MT, MODE, EPI, HN_DTYPE_F16>), g, b, 0, st, a);
  else hipLaunchKernelGGL((skinny_gemm_kernel<MT, MODE, EPI, HN_DTYPE_F32>), g, b, 0, st, a);
  return HN_LAUNCH_CHECK("skinny_gemm_kernel");
}

template <int MT, int MODE>
static int launch_skinny_epi(GemmArgs& a, int epilogue, int out_dtype, hipStream_t st) {
  if (epilogue == HN_EPI_GELU) return launch_skinny_out<MT, MODE, HN_EPI_GELU>(a, out_dtype, st);
  return launch_skinny_out<MT, MODE, HN_EPI_NONE>(a, out_dtype, st);
}

template <int MODE>
static int launch_skinny_mode(GemmArgs& a, int epilogue, int out_dtype, hipStream_t st) {
  if (a.M == 1) return launch_skinny_epi<1, MODE>(a, epilogue, out_dtype, st);
  if (a.M == 2) return launch_skinny_epi<2, MODE>(a, epilogue, out_dtype, st);
  return launch_skinny_epi<4, MODE>(a, epilogue, out_dtype, st);
}

// The same from a 16-bit source (skinny_takes_source): codes and scales in LDS, outputs in the source's dtype.
template <int MT, int MODE, int DT>
static int launch_skinny_x(GemmArgs& a, int rounding, hipStream_t st) {
  constexpr int64_t ROWS = kSkinnyRows * kSkinnyWaves;
  const int64_t grid = (a.N + ROWS - 1) / ROWS;
  if (grid > 0x7fffffff) {
    set_error("hn_block_gemm: problem too large (N=%lld)", (long long)a.N);
    return HN_ERR_UNSUPPORTED;
  }
  const dim3 g((unsigned)grid), b(kSkinnyWaves * 64);
  const unsigned lds = (unsigned)(a.M * a.K + a.M * (MODE == 0 ? 1 : a.K / 128) * 4);
  if (rounding == HN_ROUND_HALF_EVEN)
    hipLaunchKernelGGL((skinny_gemm_kernel<MT, MODE, HN_EPI_NONE, DT, DT, HN_ROUND_HALF_EVEN>), g, b, lds, st, a);
  else
    hipLaunchKernelGGL((skinny_gemm_kernel<MT, MODE, HN_EPI_NONE, DT, DT, HN_ROUND_HALF_AWAY>), g, b, lds, st, a);
  return HN_LAUNCH_CHECK("skinny_gemm_kernel");
}

template <int MODE, int DT>
static int launch_skinny_x_mode(GemmArgs& a, int rounding, hipStream_t st) {
  if (a.M == 1) return launch_skinny_x<1, MODE, DT>(a, rounding, st);
  if constexpr (MODE != 0)  // (skinny_takes_source: at most two rows there)
    if (a.M > 2) return launch_skinny_x<4, MODE, DT>(a, rounding, st);
  return launch_skinny_x<2, MODE, DT>(a, rounding, st);
}

template <int DT>
static int launch_skinny_x_dt(GemmArgs& a, bool g128, int rounding, hipStream_t st) {
  if (!g128) return launch_skinny_x_mode<0, DT>(a, rounding, st);
  if (a.sw_rows == 128) return launch_skinny_x_mode<2, DT>(a, rounding, st);
  return launch_skinny_x_mode<1, DT>(a, rounding, st);
}

// Whether the kernel that quantizes x itself takes a linear: 16-byte aligned 16-bit rows in a quantization that the quantizer
// takes, where it was measured no slower than quantizer and GEMM.  Every workgroup (16 outputs wide) repeats the
// quantization of all rows, so its cost grows with the rows, K and the workgroups that a compute unit runs, and past a point
// exceeds the launch that it saves.  Times of the two launches over the one kernel's (graphs of calls over rotating
// weights; worst of bf16 and fp16, 256 compute units), by K -> N:
//   1 row    g128, blocks     1024 -> 512 1.44   3072 -> 18432 1.09   12288 -> 18432 1.02   3072 -> 36864 1.01   16384 -> 18432 0.97
//            per token        1024 -> 512 1.37   3072 -> 18432 1.09   16384 -> 18432 1.07   3072 -> 36864 1.03
//   2 rows   all              1024 -> 256 1.15   4096 -> 12288 1.04   6144 -> 12288 0.89    3072 -> 18432 0.90
//            per token        8192 -> 4096 1.09  16384 -> 3072 1.08   8192 -> 18432 0.95
//   3 rows   g128, blocks     1024 -> 4096 1.18  2048 -> 4096 1.11    4096 -> 5120 0.95     3072 -> 18432 0.87
//   4 rows   g128, blocks     1024 -> 3072 1.18  3072 -> 3072 1.00    8192 -> 3072 0.87     12288 -> 18432 0.70
//   3, 4 rows per token       1024 -> 512 1.03, 0.96                  3072 -> 18432 0.85, 0.78
bool skinny_takes_source(const void* x, int x_dtype, int64_t ldx, int64_t M, int64_t N, int64_t K, int64_t group, int kind,
                         int rounding, int out_dtype) {
  if (M <= 0 || M > kSkinnyMaxM || N <= 0 || kind != HN_KIND_INT8 || (x_dtype != HN_DTYPE_BF16 && x_dtype != HN_DTYPE_F16) ||
      out_dtype != x_dtype || ldx < K || ldx % 8 || ((uintptr_t)x & 15) ||
      (rounding != HN_ROUND_HALF_AWAY && rounding != HN_ROUND_HALF_EVEN))
    return false;
  const int64_t per_round = (int64_t)cu_count() * kSkinnyRows * kSkinnyWaves;  // outputs of one workgroup on each unit
  if (M == 1) return K <= (group == 128 ? 12288 : 16384) && N <= 5 * per_round;
  if (M == 2) return (K <= 4096 && N <= 3 * per_round) || (group != 128 && K <= 16384 && N <= per_round);
  return group == 128 && K > 128 && M * K <= 8192 && N <= per_round;
}

// hn_block_gemm, or (x given, skinny_takes_source) the linear of x itself; qa [M, K] and sa [M, K / group] are then written.
static int block_gemm_impl(const void* x, int64_t ldx, int rounding, const void* qa, int64_t lda, const float* sa,
                           int64_t ldsa, const void* qw, int64_t ldw, const float* sw, int64_t ldsw, int64_t sw_rows,
                           const void* bias, int bias_dtype, int64_t M, int64_t N, int64_t K, int64_t group, int kind,
                           int epilogue, void* out, int out_dtype, int64_t ldo, float* qs, int64_t ldqs, void* stream) {
  HN_REQUIRE(M >= 0 && N > 0 && K > 0, "hn_block_gemm: bad shape M=%lld N=%lld K=%lld", (long long)M, (long long)N,
             (long long)K);
  HN_REQUIRE(K % 128 == 0, "hn_block_gemm: K=%lld is not a multiple of 128", (long long)K);
  HN_REQUIRE(group == 128 || group == K, "hn_block_gemm: group must be 128 or K (got %lld)", (long long)group);
  HN_REQUIRE(kind == HN_KIND_INT8 || kind == HN_KIND_FP8, "hn_block_gemm: bad kind %d", kind);
  HN_REQUIRE(epilogue >= HN_EPI_NONE && epilogue <= HN_EPI_SWIGLU_QUANT, "hn_block_gemm: bad epilogue %d", epilogue);
  HN_REQUIRE(epilogue != HN_EPI_ACC32 || kind == HN_KIND_INT8, "hn_block_gemm: ACC32 is int8 only");
  // whole-K int8 accumulation holds the exact dot product in int32: |sum| <= 128 * 128 * K < 2^31
  HN_REQUIRE(kind != HN_KIND_INT8 || (group != K && epilogue != HN_EPI_ACC32) || K < kWholeKInt32Limit,
             "hn_block_gemm: int8 with one scale group over K=%lld would overflow the int32 accumulator "
             "(K < %lld; use group 128)", (long long)K, (long long)kWholeKInt32Limit);
  HN_REQUIRE(epilogue != HN_EPI_GELU_QUANT || (N % 128 == 0 && qs != nullptr && ldqs >= N / 128),
             "hn_block_gemm: gelu_quant needs N %% 128 == 0 and qs [M, N/128]");
  HN_REQUIRE(out_dtype >= HN_DTYPE_BF16 && out_dtype <= HN_DTYPE_F32, "hn_block_gemm: bad out dtype %d", out_dtype);
  HN_REQUIRE(bias == nullptr || (bias_dtype >= HN_DTYPE_BF16 && bias_dtype <= HN_DTYPE_F32),
             "hn_block_gemm: bad bias dtype %d", bias_dtype);
  HN_REQUIRE(epilogue != HN_EPI_SWIGLU_QUANT || (N % 256 == 0 && qs != nullptr && ldqs >= N / 256),
             "hn_block_gemm: swiglu_quant needs N %% 256 == 0 (gate and up interleaved in 128-row blocks) and "
             "qs [M, N/256]");
  HN_REQUIRE((epilogue != HN_EPI_GELU_QUANT && epilogue != HN_EPI_SWIGLU_QUANT) ||
                 (ldo % 4 == 0 && ((uintptr_t)out & 3) == 0),
             "hn_block_gemm: quantized outputs are stored 4 codes at a time: ldo %% 4 == 0, 4-byte aligned out");
  HN_REQUIRE(lda >= K && ldw >= K && ldo >= (epilogue == HN_EPI_SWIGLU_QUANT ? N / 2 : N),
             "hn_block_gemm: row strides smaller than the rows");
  HN_REQUIRE(lda % 16 == 0 && ldw % 16 == 0, "hn_block_gemm: code row strides must be multiples of 16 bytes");
  HN_REQUIRE(lda < (1 << 22) && ldw < (1 << 22) && ldsa < (1 << 22) && ldsw < (1 << 22) && ldo < (1 << 22),
             "hn_block_gemm: row strides must be below 2^22 elements");
  HN_REQUIRE(sw_rows == 1 || (sw_rows == 128 && group == 128 && epilogue != HN_EPI_ACC32),
             "hn_block_gemm: sw_rows must be 1, or 128 with group 128 (got %lld)", (long long)sw_rows);
  HN_REQUIRE(qa && qw && out, "hn_block_gemm: null pointer");
  HN_REQUIRE(((uintptr_t)qa & 15) == 0 && ((uintptr_t)qw & 15) == 0, "hn_block_gemm: codes must be 16-byte aligned");
  if (epilogue != HN_EPI_ACC32) {
    HN_REQUIRE(sa && sw, "hn_block_gemm: null scales");
    HN_REQUIRE(ldsa >= K / group && ldsw >= K / group, "hn_block_gemm: scale row strides too small");
  }
  if (M == 0) return HN_OK;
  GemmArgs a{};
  a.qa = (const uint8_t*)qa; a.lda = lda; a.sa = sa; a.ldsa = ldsa;
  a.qw = (const uint8_t*)qw; a.ldw = ldw; a.sw = sw; a.ldsw = ldsw; a.sw_rows = (int)sw_rows;
  a.bias = bias; a.bias_dtype = bias_dtype;
  a.M = M; a.N = N; a.K = K;
  a.out = out; a.ldo = ldo; a.qs = qs; a.ldqs = ldqs;
  const int esz = out_dtype == HN_DTYPE_F32 ? 4 : 2;
  a.vec_store = (N % 4 == 0) && (ldo % 4 == 0) && ((((uintptr_t)out) & (4 * esz - 1)) == 0);
  a.stage_store = esz == 2 && (N % 8 == 0) && (ldo % 8 == 0) && ((((uintptr_t)out) & 15) == 0);
  hipStream_t st = (hipStream_t)stream;
  // per-token mode also serves a single-group K == 128 problem with one scale row per channel
  const bool g128 = group == 128 && (K != 128 || sw_rows == 128);
  if (epilogue == HN_EPI_ACC32) return launch_group<HN_KIND_INT8, HN_EPI_ACC32, HN_DTYPE_BF16>(a, false, st);
  if (x != nullptr) {
    a.x = (const uint16_t*)x;
    a.ldx = ldx;
    return out_dtype == HN_DTYPE_BF16 ? launch_skinny_x_dt<HN_DTYPE_BF16>(a, g128, rounding, st)
                                      : launch_skinny_x_dt<HN_DTYPE_F16>(a, g128, rounding, st);
  }
  if (kind == HN_KIND_INT8 && M <= kSkinnyMaxM && (epilogue == HN_EPI_NONE || epilogue == HN_EPI_GELU)) {
    if (!g128) return launch_skinny_mode<0>(a, epilogue, out_dtype, st);
    if (sw_rows == 128) return launch_skinny_mode<2>(a, epilogue, out_dtype, st);
    return launch_skinny_mode<1>(a, epilogue, out_dtype, st);
  }
  bool taken = false;
  if (kind == HN_KIND_INT8 && (!g128 || sw_rows == 1)) {
    const int rc = launch_ring_int8(a, g128, epilogue, out_dtype, st, &taken);
    if (taken) return rc;
  } else if (kind == HN_KIND_FP8 && g128 && sw_rows == 128) {
    const int rc = launch_ring_fp8(a, epilogue, out_dtype, st, &taken);
    if (taken) return rc;
  }
  if (kind == HN_KIND_INT8) return launch_kind<HN_KIND_INT8>(a, g128, epilogue, out_dtype, st);
  return launch_kind<HN_KIND_FP8>(a, g128, epilogue, out_dtype, st);
}


int skinny_linear(const void* x, int64_t ldx, int rounding, const void* qa, const float* sa, const void* qw, int64_t ldw,
                  const float* sw, int64_t ldsw, int64_t sw_rows, const void* bias, int bias_dtype, int64_t M, int64_t N,
                  int64_t K, int64_t group, void* out, int out_dtype, int64_t ldo, void* stream) {
  return block_gemm_impl(x, ldx, rounding, qa, K, sa, K / group, qw, ldw, sw, ldsw, sw_rows, bias, bias_dtype, M, N, K, group,
                         HN_KIND_INT8, HN_EPI_NONE, out, out_dtype, ldo, nullptr, 0, stream);
}

}  // namespace hn

extern "C" int hn_block_gemm(const void* qa, int64_t lda, const float* sa, int64_t ldsa, const void* qw, int64_t ldw,
                             const float* sw, int64_t ldsw, int64_t sw_rows, const void* bias, int bias_dtype, int64_t M, int64_t N,
                             int64_t K, int64_t group, int kind, int epilogue, void* out, int out_dtype, int64_t ldo,
                             float* qs, int64_t ldqs, void* stream) {
  using namespace hn;
  return block_gemm_impl(nullptr, 0, 0, qa, lda, sa, ldsa, qw, ldw, sw, ldsw, sw_rows, bias, bias_dtype, M, N, K, group, kind,
                         epilogue, out, out_dtype, ldo, qs, ldqs, stream);
}

static int qkv_heads_impl(const void* qa, int64_t lda, const float* sa, int64_t ldsa, const void* qw, int64_t ldw,
                          const float* sw, int64_t ldsw, int64_t sw_rows, const void* bias, int bias_dtype, int64_t B,
                          int64_t L, int64_t hidden, int64_t K, int64_t group, int kind, const float* q_norm_w,
                          const float* k_norm_w, const float* cos_t, const float* sin_t, float eps, void* out,
                          int64_t L_total, int64_t l_offset, void* vt, int64_t svb, int64_t svh, int64_t svd,
                          void* stream) {
  using namespace hn;
  HN_REQUIRE(B >= 0 && L >= 0 && hidden > 0 && K > 0, "hn_qkv_heads: bad shape");
  HN_REQUIRE(hidden % 128 == 0, "hn_qkv_heads: hidden=%lld is not a multiple of the head dim 128", (long long)hidden);
  HN_REQUIRE(K % 128 == 0, "hn_qkv_heads: K=%lld is not a multiple of 128", (long long)K);
  HN_REQUIRE(group == 128 || group == K, "hn_qkv_heads: group must be 128 or K (got %lld)", (long long)group);
  HN_REQUIRE(kind == HN_KIND_INT8 || kind == HN_KIND_FP8, "hn_qkv_heads: bad kind %d", kind);
  HN_REQUIRE(sw_rows == 1 || (sw_rows == 128 && group == 128), "hn_qkv_heads: sw_rows must be 1, or 128 with group 128");
  HN_REQUIRE(kind != HN_KIND_INT8 || group != K || K < kWholeKInt32Limit,
             "hn_qkv_heads: int8 with one scale group over K=%lld would overflow the int32 accumulator (K < %lld)",
             (long long)K, (long long)kWholeKInt32Limit);
  HN_REQUIRE(l_offset >= 0 && L_total >= l_offset + L, "hn_qkv_heads: tokens [%lld, %lld) exceed L_total=%lld",
             (long long)l_offset, (long long)(l_offset + L), (long long)L_total);
  HN_REQUIRE(B * L < ((int64_t)1 << 31), "hn_qkv_heads: B * L must be below 2^31");
  HN_REQUIRE(lda >= K && ldw >= K && lda % 16 == 0 && ldw % 16 == 0, "hn_qkv_heads: bad code row strides");
  HN_REQUIRE(lda < (1 << 22) && ldw < (1 << 22) && ldsa < (1 << 22) && ldsw < (1 << 22),
             "hn_qkv_heads: row strides must be below 2^22 elements");
  HN_REQUIRE(ldsa >= K / group && ldsw >= K / group, "hn_qkv_heads: scale row strides too small");
  HN_REQUIRE(bias == nullptr || (bias_dtype >= HN_DTYPE_BF16 && bias_dtype <= HN_DTYPE_F32), "hn_qkv_heads: bad bias dtype");
  HN_REQUIRE(qa && sa && qw && sw && q_norm_w && k_norm_w && out, "hn_qkv_heads: null pointer");
  HN_REQUIRE((cos_t == nullptr) == (sin_t == nullptr), "hn_qkv_heads: cos and sin must both be given or both NULL");
  HN_REQUIRE(((uintptr_t)qa & 15) == 0 && ((uintptr_t)qw & 15) == 0 && ((uintptr_t)out & 15) == 0 &&
                 ((uintptr_t)q_norm_w & 15) == 0 && ((uintptr_t)k_norm_w & 15) == 0 &&
                 ((uintptr_t)cos_t & 15) == 0 && ((uintptr_t)sin_t & 15) == 0,
             "hn_qkv_heads: codes, output, norm weights and rope tables must be 16-byte aligned");
  if (B * L == 0) return HN_OK;
  GemmArgs a{};
  a.qa = (const uint8_t*)qa; a.lda = lda; a.sa = sa; a.ldsa = ldsa;
  a.qw = (const uint8_t*)qw; a.ldw = ldw; a.sw = sw; a.ldsw = ldsw; a.sw_rows = (int)sw_rows;
  a.bias = bias; a.bias_dtype = bias_dtype;
  a.M = B * L; a.N = 3 * hidden; a.K = K;
  a.out = out; a.ldo = 3 * hidden;
  a.stage_store = 1;
  a.hm_L = L; a.hm_Ltot = L_total; a.hm_loff = l_offset; a.hm_hidden = hidden; a.hm_B = B;
  a.hm_wq = q_norm_w; a.hm_wk = k_norm_w; a.hm_cos = cos_t; a.hm_sin = sin_t; a.hm_eps = eps;
  a.hm_vt = (uint16_t*)vt; a.hm_svb = svb; a.hm_svh = svh; a.hm_svd = svd;
  hipStream_t st = (hipStream_t)stream;
  const bool g128 = group == 128 && (K != 128 || sw_rows == 128);
  if (kind == HN_KIND_INT8) return launch_group<HN_KIND_INT8, kEpiQkvHeads, HN_DTYPE_BF16>(a, g128, st);
  return launch_group<HN_KIND_FP8, kEpiQkvHeads, HN_DTYPE_BF16>(a, g128, st);
}

extern "C" int hn_qkv_heads(const void* qa, int64_t lda, const float* sa, int64_t ldsa, const void* qw, int64_t ldw,
                            const float* sw, int64_t ldsw, int64_t sw_rows, const void* bias, int bias_dtype, int64_t B,
                            int64_t L, int64_t hidden, int64_t K, int64_t group, int kind, const float* q_norm_w,
                            const float* k_norm_w, const float* cos_t, const float* sin_t, float eps, void* out,
                            int64_t L_total, int64_t l_offset, void* stream) {
  return qkv_heads_impl(qa, lda, sa, ldsa, qw, ldw, sw, ldsw, sw_rows, bias, bias_dtype, B, L, hidden, K, group, kind,
                        q_norm_w, k_norm_w, cos_t, sin_t, eps, out, L_total, l_offset, nullptr, 0, 0, 0, stream);
}

extern "C" int hn_qkv_heads_vt(const void* qa, int64_t lda, const float* sa, int64_t ldsa, const void* qw, int64_t ldw,
                               const float* sw, int64_t ldsw, int64_t sw_rows, const void* bias, int bias_dtype,
                               int64_t B, int64_t L, int64_t hidden, int64_t K, int64_t group, int kind,
                               const float* q_norm_w, const float* k_norm_w, const float* cos_t, const float* sin_t,
                               float eps, void* out, int64_t L_total, int64_t l_offset, void* vt, int64_t svb,
                               int64_t svh, int64_t svd, void* stream) {
  HN_REQUIRE(vt != nullptr && ((uintptr_t)vt & 15) == 0, "hn_qkv_heads_vt: V^T must be a 16-byte aligned pointer");
  HN_REQUIRE(L % 32 == 0 && l_offset % 16 == 0,
             "hn_qkv_heads_vt: L=%lld must be a multiple of 32 and l_offset=%lld of 16", (long long)L,
             (long long)l_offset);
  HN_REQUIRE(svd % 8 == 0 && svh % 8 == 0 && svb % 8 == 0 && svd >= l_offset + L && svh >= 128 * svd &&
                 svb >= (hidden / 128) * svh,
             "hn_qkv_heads_vt: V^T strides (%lld, %lld, %lld) must be multiples of 8 holding [B, H, 128, >= %lld]",
             (long long)svb, (long long)svh, (long long)svd, (long long)(l_offset + L));
  return qkv_heads_impl(qa, lda, sa, ldsa, qw, ldw, sw, ldsw, sw_rows, bias, bias_dtype, B, L, hidden, K, group, kind,
                        q_norm_w, k_norm_w, cos_t, sin_t, eps, out, L_total, l_offset, vt, svb, svh, svd, stream);
}
