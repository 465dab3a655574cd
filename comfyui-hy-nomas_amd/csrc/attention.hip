// Softmax attention on the gfx950 bf16 matrix cores: the attention backend of the double-stream block
// (hy_nomas/model.py:145-150 `attention`, the scaled-dot-product attention the reference hands to ComfyUI's
// backend), in one pass over the keys with an online softmax.
//
//   out[b, i, h, :] = sum_j softmax_j(q[b, i, h, :] . k[b, j, h, :] * scale) v[b, j, h, :]
//
// Head dim 128, bf16 q / k / v / out, fp32 scores, running max and sums, bf16 probabilities for the
// second product (as flash attention does), no mask.
//
// Work split.  A workgroup of 4 waves owns 128 queries of one (batch, head); each wave 32.  Keys are walked
// in tiles of 64, staged in LDS by gfx950's direct-to-LDS loads one tile ahead (two buffers, one barrier per
// tile).
//
// Layouts.  The scores are computed transposed, S^T = K Q^T (keys as the MFMA A rows, queries as the B
// columns), so each lane's accumulators hold one query and 16 keys of each 32-key block: the row statistics
// of a query are in-lane reductions plus one exchange with lane l ^ 32, which holds the other 16 keys.  Each
// lane keeps its own partial row sum and the two are added once at the end.  The output is accumulated
// transposed too, O^T = V^T P^T, with the probabilities as the B operand straight from the score registers:
// an MFMA's operands run along the reduced dimension (here the keys), so the 8 keys of a lane's B fragment
// are the ones its score registers hold, keys 16 g + 8 (e / 4) + 4 h + e % 4 (e = 0..7) of 16-key group g in
// lane half h.  V^T therefore comes with the keys of each 16-key group stored in the order 0-3, 8-11, 4-7,
// 12-15 (`hn_attention`'s V^T layout): lane half h's 8 keys are then one 16-byte chunk, read with one
// ds_read_b128.
//
// LDS.  K tile: 64 rows of 256 bytes, 16-byte chunk c of row r at c ^ (r & 15); V^T tile: 128 rows of 128
// bytes, chunk c of row r at c ^ ((r >> 1) & 7).  Both are read conflict-free (16 lanes per 256-byte pass hit
// 16 different bank quads).  The direct loads write 1 KB per wave instruction in lane order, so the swizzle
// is applied on the global side (the lane fetches the logical chunk of its physical slot).
//
// Key segments.  The keys of a query are the concatenation of up to three segments, read where they lie: up to two
// shared ones (the history cache and the current tokens, each with its own strides) and the text keys of the
// query's group.  Every segment starts a new 64-key tile, and its last tile is masked, so nothing is joined in
// memory first; V^T holds the segments one after another, each padded to whole tiles (attention_pack_kernel).  All
// groups share one launch, which fills the chip where one group would not.  Joining, gathering and transposing per
// group took two thirds of such a call.  With the split keys below, 24 heads, 3520 + 200 tokens over 15840 history keys in
// three groups went from 2608 to 905 us; 16 heads x 26656 tokens, where the V^T pass and the split are new, from 5649 to
// 4995 us.
//
// Lazy rescale.  The running reference max m moves only when a tile's max exceeds it by more than 8 (base-2
// units), so the probabilities exp2(s - m) stay below 2^8 and the accumulators are rescaled only a few times
// per query instead of whenever the max grows.  The result is the same quotient: numerator and denominator
// share the reference.
// A query whose scores so far are all -inf has no reference yet: m = -inf, and its products start from 0.
#include "hn_common.h"

namespace hn {
namespace {

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef int v4i_a __attribute__((ext_vector_type(4)));
typedef float v16f_a __attribute__((ext_vector_type(16)));

constexpr int kHeadDim = 128;
constexpr int kBQ = 128;                        // queries per workgroup
constexpr int kBK = 64;                         // keys per tile
constexpr int kAttnWaves = 4;
constexpr int kKTile = kBK * kHeadDim * 2;      // 16 KB
constexpr int kVTile = kHeadDim * kBK * 2;      // 16 KB
constexpr int kAttnStage = kKTile + kVTile;
constexpr float kSlack = 8.0f;                  // headroom of the lazy max (base-2 units)

constexpr int kMaxGroups = 64;                  // query groups of one launch (the table rides in the kernel arguments)

// One shared key segment: key j of batch b, head h at k + b skb + h skh + j skj, V^T position vpos + j.
struct AttnSeg {
  const uint16_t* k;
  int64_t skb, skh, skj;
  int64_t len;
  int64_t vpos;
};

// One query group: queries rows[q_off .. q_off + q_n), workgroups from query block qb0 on, text keys t_n at row
// t_pos (a multiple of 64) of the packed text keys.
struct AttnGroup {
  int qb0, q_off, q_n, t_n, t_pos;
};

struct AttnArgs {
  const uint16_t* q;
  int64_t sqb, sqh, sqi;  // element strides of batch, head, token (dims contiguous)
  AttnSeg seg[2];
  int nseg;
  const uint16_t* tk;     // packed text keys [B, H, t_rows, 128], V^T positions from tvpos on
  int64_t t_rows, tvpos;
  const uint16_t* vt;     // V^T: element (b, h, d, key position p) at vt + b svb + h svh + d svd + p
  int64_t svb, svh, svd;
  uint16_t* o;
  int64_t sob, soh, soi;
  const int64_t* rows;    // query rows of the groups, or null: query i is row i
  const int* owner;       // with rows: the last group that names each row, whose result it takes
  int H;
  float scale_log2;       // softmax scale times log2(e): the scores are exponentiated base 2
  int qblocks;            // query blocks of one (batch, head)
  // Query blocks of all heads, in order: the first `whole` walk all their keys, one workgroup each; the `tail` after
  // them have `splits` workgroups each, which take a contiguous range of the tiles.
  int whole, tail, splits;
  float4* po;             // the tail's unnormalized partial outputs [split][tail block][32 chunks of 4 dims][128 queries]
  float2* pml;            // and their reference max and sum [split][tail block][128 queries]
  int ngroups;
  AttnGroup group[kMaxGroups];
};

__device__ __forceinline__ void wait_vm0() { __builtin_amdgcn_s_waitcnt((7 << 4) | (15 << 8)); }

// max of x over lanes l and l ^ 32 (one v_permlane32_swap instead of an LDS permute)
__device__ __forceinline__ float max_xor32(float x) {
  const auto r = __builtin_amdgcn_permlane32_swap(__builtin_bit_cast(uint32_t, x), __builtin_bit_cast(uint32_t, x),
                                                  false, false);
  return __builtin_fmaxf(__builtin_bit_cast(float, (uint32_t)r[0]), __builtin_bit_cast(float, (uint32_t)r[1]));
}

template <bool SPLIT>
__global__ __launch_bounds__(kAttnWaves * 64) __attribute__((amdgpu_waves_per_eu(2, 2)))
void attention_kernel(const AttnArgs a) {
  __shared__ __align__(16) char smem[2 * kAttnStage];
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int h2 = lane >> 5, l32 = lane & 31;
  // (query blocks of one head run side by side, so that their tiles are read once from HBM)
  const bool part = SPLIT && (int)blockIdx.x >= a.whole;
  const int slot = part ? blockIdx.x - a.whole : 0;  // of the partials
  const int split = part ? slot / a.tail : 0;
  const int unit = part ? a.whole + slot % a.tail : blockIdx.x;
  const int bh = unit / a.qblocks, qb = unit % a.qblocks;
  const int64_t b = bh / a.H, hh = bh % a.H;
  int gi = 0;
  while (gi + 1 < a.ngroups && qb >= a.group[gi + 1].qb0) gi++;
  const int q_n = a.group[gi].q_n, t_n = a.group[gi].t_n;
  const uint16_t* qbase = a.q + b * a.sqb + hh * a.sqh;
  const char* vbase = reinterpret_cast<const char*>(a.vt + b * a.svb + hh * a.svh);
  const uint32_t vstride = (uint32_t)(a.svd * 2);  // bytes per dim row
  const int q0 = (qb - a.group[gi].qb0) * kBQ + wave * 32;
  const int qi = q0 + l32 < q_n ? q0 + l32 : q_n - 1;
  const int64_t qrow = a.rows ? a.rows[a.group[gi].q_off + qi] : qi;

  // the wave's 32 queries: B fragments of S^T = K Q^T for the 8 steps of 16 dims (query l32, dims 16 ks + 8 h2 ..)
  bf16x8 qf[8];
#pragma unroll
  for (int ks = 0; ks < 8; ks++) qf[ks] = *reinterpret_cast<const bf16x8*>(qbase + qrow * a.sqi + 16 * ks + 8 * h2);

  // direct loads of one tile: wave w fills the 1 KB blocks w, w + 4, w + 8, w + 12 of the K tile (4 rows of
  // 256 bytes each) and of the V^T tile (8 rows of 128 bytes), each lane 16 bytes at a fixed 32-bit offset
  // from the tile's buffer descriptor (wave-uniform base: no per-lane 64-bit address arithmetic)
  uint32_t koff[4], voff[4], kstride = 0;
#pragma unroll
  for (int u = 0; u < 4; u++) {
    const int vrow = (wave + 4 * u) * 8 + lane / 8, vphys = lane % 8;
    voff[u] = (uint32_t)vrow * vstride + (uint32_t)((vphys ^ ((vrow >> 1) & 7)) << 4);
  }
  // the next tile to load: its first key's address, its V^T column, and the keys from it to its segment's end
  const char *kcur = nullptr, *vcur = nullptr;
  int64_t left = 0;
  int seg = -1;
  auto next_segment = [&]() {
    do {
      seg++;
      if (seg < a.nseg) {
        const AttnSeg& sg = a.seg[seg];
        kcur = reinterpret_cast<const char*>(sg.k + b * sg.skb + hh * sg.skh);
        vcur = vbase + sg.vpos * 2;
        kstride = (uint32_t)(sg.skj * 2);  // bytes per key
        left = sg.len;
      } else {  // the group's text keys
        kcur = reinterpret_cast<const char*>(a.tk + ((b * a.H + hh) * a.t_rows + a.group[gi].t_pos) * kHeadDim);
        vcur = vbase + (a.tvpos + a.group[gi].t_pos) * 2;
        kstride = kHeadDim * 2;
        left = t_n;
      }
    } while (left == 0 && seg < a.nseg);
#pragma unroll
    for (int u = 0; u < 4; u++) {
      const int krow = (wave + 4 * u) * 4 + lane / 16, kphys = lane % 16;
      koff[u] = (uint32_t)krow * kstride + (uint32_t)((kphys ^ (krow & 15)) << 4);
    }
  };
  // loads the tile at the cursor into a buffer and moves the cursor; returns the tile's keys (64, or fewer at a
  // segment's end)
  auto issue_tile = [&](int buf) __attribute__((always_inline)) {
    char* kt = smem + buf * kAttnStage;
    char* vt = kt + kKTile;
    const __amdgpu_buffer_rsrc_t kr = buffer_rsrc(kcur);
    const __amdgpu_buffer_rsrc_t vr = buffer_rsrc(vcur);
    const int here = left < kBK ? (int)left : kBK;
    if (here == kBK) {
#pragma unroll
      for (int u = 0; u < 4; u++) b2lds16(kr, koff[u], 0, kt + (wave + 4 * u) * 1024);
    } else {
      // a segment's last tile: rows past the last key re-read it (their scores are masked)
#pragma unroll
      for (int u = 0; u < 4; u++) {
        const int krow = (wave + 4 * u) * 4 + lane / 16, kphys = lane % 16;
        const int r = krow < here - 1 ? krow : here - 1;
        b2lds16(kr, (uint32_t)r * kstride + (uint32_t)((kphys ^ (krow & 15)) << 4), 0, kt + (wave + 4 * u) * 1024);
      }
    }
#pragma unroll
    for (int u = 0; u < 4; u++) b2lds16(vr, voff[u], 0, vt + (wave + 4 * u) * 1024);
    left -= here;
    kcur += (int64_t)kBK * kstride;
    vcur += kBK * 2;
    if (left == 0 && seg < a.nseg) next_segment();
    return here;
  };

  v16f_a oacc[4];
#pragma unroll
  for (int db = 0; db < 4; db++)
#pragma unroll
    for (int r = 0; r < 16; r++) oacc[db][r] = 0.0f;
  float m = -__builtin_inff();  // reference max of the scaled scores (base-2 units), shared by lanes l, l ^ 32
  // -m / (scale log2(e)) in every register: the score products start from it, so the scores come out already
  // relative to the reference and a probability is exp2(s scale log2(e)).  0 until the first tile sets m.
  v16f_a mref;
#pragma unroll
  for (int r = 0; r < 16; r++) mref[r] = 0.0f;
  const float inv_scale = 1.0f / a.scale_log2;
  float mref_m = 0.0f;  // the reference mref holds (m', base-2 units)
  float lsum = 0.0f;            // this lane's partial sum of the probabilities
  float pv[32];                 // the last tile's probabilities, not yet in lsum
#pragma unroll
  for (int i = 0; i < 32; i++) pv[i] = 0.0f;
  const int kswz = l32 & 15, vswz = (l32 >> 1) & 7;   // the lane's rows' swizzles (rows 32 i + l32)

  int nt = (t_n + kBK - 1) / kBK;  // tiles of all segments
  for (int i = 0; i < a.nseg; i++) nt += (int)((a.seg[i].len + kBK - 1) / kBK);
  next_segment();
  if (part) {  // this workgroup's tiles [skip, skip + nt)
    int skip = (int)((int64_t)nt * split / a.splits);
    nt = (int)((int64_t)nt * (split + 1) / a.splits) - skip;
    for (int64_t here; (here = (left + kBK - 1) / kBK) <= skip;) {
      skip -= (int)here;
      next_segment();
    }
    kcur += (int64_t)skip * kBK * kstride;
    vcur += (int64_t)skip * kBK * 2;
    left -= (int64_t)skip * kBK;
  }
  int keys = 0, keys_next = 0;     // keys of the current and of the loading tile
  // tile t in stage buffer BUF (a constant, so the buffer offset rides in the LDS reads' immediate field
  // and the lane's fragment offsets stay fixed across the loop)
  auto tile = [&](int t, auto buf_c) __attribute__((always_inline)) {
    constexpr int BUF = decltype(buf_c)::value;
    // tile t has landed for every wave, and every wave is done with the buffer tile t + 1 refills
    wait_vm0();
    __builtin_amdgcn_s_waitcnt(0xc07f);  // lgkmcnt(0)
    __builtin_amdgcn_s_barrier();
    keys = keys_next;
    if (t + 1 < nt) keys_next = issue_tile(BUF ^ 1);
    const char* kt = smem + BUF * kAttnStage;
    const char* vt = kt + kKTile;

    // S^T for the tile's two 32-key blocks (interleaved): lane holds query l32, keys 32 kb + 8 (r / 4) + 4 h2 + r % 4
    v16f_a s[2];
    // the K fragments two steps ahead of their products (a ring of three), so each read has two steps of
    // products to land in
    bf16x8 kf[3][2];
    auto read_k = [&](int ks, bf16x8* f) __attribute__((always_inline)) {
#pragma unroll
      for (int kb = 0; kb < 2; kb++)
        f[kb] = *reinterpret_cast<const bf16x8*>(kt + (32 * kb + l32) * 256 + (((2 * ks + h2) ^ kswz) << 4));
    };
    read_k(0, kf[0]);
    read_k(1, kf[1]);
    __builtin_amdgcn_sched_group_barrier(0x100, 4, 0);
#pragma unroll
    for (int ks = 0; ks < 8; ks++) {
#pragma unroll
      for (int kb = 0; kb < 2; kb++)
        s[kb] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(kf[ks % 3][kb], qf[ks], ks == 0 ? mref : s[kb], 0, 0, 0);
      __builtin_amdgcn_sched_group_barrier(0x008, 2, 0);
      if (ks + 2 < 8) {
        read_k(ks + 2, kf[(ks + 2) % 3]);
        __builtin_amdgcn_sched_group_barrier(0x100, 2, 0);
      }
      // the previous tile's probabilities join the running sum while the matrix core works (the
      // reference m' has not moved since they were formed: a move below rescales lsum after this)
#pragma unroll
      for (int i = 0; i < 4; i++) lsum += pv[4 * ks + i];
      __builtin_amdgcn_sched_group_barrier(0x002, 4, 0);
    }
    if (keys < kBK) {  // a segment's last tile: keys past its end take no weight
      // register r of block kb holds the tile's key 32 kb + 8 (r / 4) + (r % 4) + 4 h2: a constant per register
      // against one per-lane limit
      const int lim = keys - 4 * h2;
#pragma unroll
      for (int kb = 0; kb < 2; kb++)
#pragma unroll
        for (int r = 0; r < 16; r++)
          if (32 * kb + 8 * (r / 4) + (r % 4) >= lim) s[kb][r] = -__builtin_inff();
    }
    // online softmax: the tile's max for this query (both lanes), then the lazy move of the reference max.
    // The scores hold s - m' / (scale log2(e)), m' the reference their products started from (m after the
    // first tile), so the tile's max in base-2 units is mx scale log2(e) + m'.
    float mx = s[0][0];
#pragma unroll
    for (int kb = 0; kb < 2; kb++)
#pragma unroll
      for (int r = 0; r < 16; r++) mx = __builtin_fmaxf(mx, s[kb][r]);
    const float mrel = max_xor32(mx) * a.scale_log2;  // the tile's max relative to m'
    // m' = m outside the move below; the first tile (m = -inf) always moves it
    if (__builtin_amdgcn_ballot_w64(!(mrel + mref_m <= m + kSlack)) != 0) {
      const float mt = mrel + mref_m;
      const bool grow = mt > m + kSlack;
      // where the reference stays nothing changes (m and m' differ only while every score so far was -inf: m = -inf and
      // m' = 0, whose difference is no factor)
      const float mnew = grow ? mt : mref_m;
      const float alpha = grow ? __builtin_amdgcn_exp2f(m - mt) : 1.0f;  // 0 for the first tile
      m = grow ? mt : m;
      lsum *= alpha;
#pragma unroll
      for (int db = 0; db < 4; db++)
#pragma unroll
        for (int r = 0; r < 16; r++) oacc[db][r] *= alpha;
      // this tile's scores moved to the new reference, and the next tiles' products start from it
      const float delta = (mref_m - mnew) * inv_scale;
#pragma unroll
      for (int kb = 0; kb < 2; kb++)
#pragma unroll
        for (int r = 0; r < 16; r++) s[kb][r] += delta;
      mref_m = mnew;
      const float mr = -mnew * inv_scale;
#pragma unroll
      for (int r = 0; r < 16; r++) mref[r] = mr;
    }
    // probabilities exp2(s scale log2(e)) against the reference, this lane's sum, bf16 pairs
    uint32_t pk[2][8];
#pragma unroll
    for (int kb = 0; kb < 2; kb++)
#pragma unroll
      for (int p = 0; p < 8; p++) {
        const float e0 = __builtin_amdgcn_exp2f(s[kb][2 * p] * a.scale_log2);
        const float e1 = __builtin_amdgcn_exp2f(s[kb][2 * p + 1] * a.scale_log2);
        pv[16 * kb + 2 * p] = e0;
        pv[16 * kb + 2 * p + 1] = e1;
        pk[kb][p] = bf16x2_finite(e0, e1);
      }
    // O^T += V^T P^T over the four 16-key groups g = 2 kb + ks2: the B fragment is score registers
    // 8 ks2 .. 8 ks2 + 7 of block kb, the A fragment chunk 2 g + h2 of each V^T row (the keys in the same order)
#pragma unroll
    for (int kb = 0; kb < 2; kb++)
#pragma unroll
      for (int ks2 = 0; ks2 < 2; ks2++) {
        const v4i_a bi = {(int)pk[kb][4 * ks2], (int)pk[kb][4 * ks2 + 1], (int)pk[kb][4 * ks2 + 2],
                          (int)pk[kb][4 * ks2 + 3]};
        const int chunk = (4 * kb + 2 * ks2 + h2) ^ vswz;
#pragma unroll
        for (int db = 0; db < 4; db++) {
          const bf16x8 af = *reinterpret_cast<const bf16x8*>(vt + (32 * db + l32) * 128 + (chunk << 4));
          oacc[db] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(af, __builtin_bit_cast(bf16x8, bi), oacc[db], 0, 0, 0);
        }
      }
  };
  keys_next = issue_tile(0);
  for (int t = 0; t < nt; t += 2) {
    tile(t, std::integral_constant<int, 0>());
    if (t + 1 < nt) tile(t + 1, std::integral_constant<int, 1>());
  }
#pragma unroll
  for (int i = 0; i < 32; i++) lsum += pv[i];
  // normalize and store: lane holds query l32, dims 32 db + 8 rr + 4 h2 + 0..3 in registers 4 rr .. 4 rr + 3
  const float ltot = lsum + __shfl_xor(lsum, 32);
  if (part) {  // fp32 partials, 16 bytes per lane with the 32 queries side by side
    float4* po = a.po + (int64_t)slot * 32 * kBQ + wave * 32 + l32;
#pragma unroll
    for (int db = 0; db < 4; db++)
#pragma unroll
      for (int rr = 0; rr < 4; rr++)
        po[(8 * db + 2 * rr + h2) * kBQ] =
            make_float4(oacc[db][4 * rr], oacc[db][4 * rr + 1], oacc[db][4 * rr + 2], oacc[db][4 * rr + 3]);
    if (h2 == 0) a.pml[(int64_t)slot * kBQ + wave * 32 + l32] = make_float2(m, ltot);
    return;
  }
  const float inv = 1.0f / ltot;
  if (q0 + l32 < q_n && (a.owner == nullptr || a.owner[qrow] == gi)) {
    uint16_t* orow = a.o + b * a.sob + hh * a.soh + qrow * a.soi;
#pragma unroll
    for (int db = 0; db < 4; db++)
#pragma unroll
      for (int rr = 0; rr < 4; rr++) {
        const int d = 32 * db + 8 * rr + 4 * h2;
        const uint2 w = make_uint2(bf16x2_finite(oacc[db][4 * rr] * inv, oacc[db][4 * rr + 1] * inv),
                                   bf16x2_finite(oacc[db][4 * rr + 2] * inv, oacc[db][4 * rr + 3] * inv));
        *reinterpret_cast<uint2*>(orow + d) = w;
      }
  }
}

// The result of queries whose keys were split: out = sum_s w_s O_s / sum_s w_s l_s with w_s = exp2(m_s - max m).
// A workgroup takes 32 queries of one query block, a thread 16 dims of one query; bound by reading the partials
// (64 KB per 128 queries and split).
constexpr int kCombineThreads = 256;

__global__ __launch_bounds__(kCombineThreads) void attention_combine_kernel(const AttnArgs a) {
  const int ql = (blockIdx.x % 4) * 32 + (threadIdx.x & 31), part = threadIdx.x >> 5;
  const int unit = a.whole + blockIdx.x / 4;
  const int bh = unit / a.qblocks, qb = unit % a.qblocks;
  int gi = 0;
  while (gi + 1 < a.ngroups && qb >= a.group[gi + 1].qb0) gi++;
  const int qi = (qb - a.group[gi].qb0) * kBQ + ql;
  if (qi >= a.group[gi].q_n) return;
  const int64_t qrow = a.rows ? a.rows[a.group[gi].q_off + qi] : qi;
  if (a.owner != nullptr && a.owner[qrow] != gi) return;
  const int64_t first = blockIdx.x / 4;  // the block's partial of split s: first + s tail
  float mmax = -__builtin_inff();
  for (int s = 0; s < a.splits; s++) mmax = __builtin_fmaxf(mmax, a.pml[(first + (int64_t)s * a.tail) * kBQ + ql].x);
  float o[16], l = 0.0f;
#pragma unroll
  for (int i = 0; i < 16; i++) o[i] = 0.0f;
  for (int s = 0; s < a.splits; s++) {
    const int64_t wg = first + (int64_t)s * a.tail;
    const float2 ml = a.pml[wg * kBQ + ql];
    const float w = __builtin_amdgcn_exp2f(ml.x - mmax);
    l = __builtin_fmaf(w, ml.y, l);
    const float4* po = a.po + (wg * 32 + part * 4) * kBQ + ql;
#pragma unroll
    for (int c = 0; c < 4; c++) {
      const float4 v = po[c * kBQ];
      o[4 * c] = __builtin_fmaf(w, v.x, o[4 * c]);
      o[4 * c + 1] = __builtin_fmaf(w, v.y, o[4 * c + 1]);
      o[4 * c + 2] = __builtin_fmaf(w, v.z, o[4 * c + 2]);
      o[4 * c + 3] = __builtin_fmaf(w, v.w, o[4 * c + 3]);
    }
  }
  const float inv = 1.0f / l;
  uint16_t* orow = a.o + (bh / a.H) * a.sob + (bh % a.H) * a.soh + qrow * a.soi + part * 16;
#pragma unroll
  for (int c = 0; c < 4; c++)
    *reinterpret_cast<uint2*>(orow + 4 * c) = make_uint2(bf16x2_finite(o[4 * c] * inv, o[4 * c + 1] * inv),
                                                         bf16x2_finite(o[4 * c + 2] * inv, o[4 * c + 3] * inv));
}

// V^T of every key segment, and the packed text keys, for attention_kernel.
//
// One workgroup takes 64 keys (one tile of one segment) of one (batch, head): it reads the 64 rows of 256 bytes
// whole, turns them in LDS (rows of 65 dwords, so the column reads spread over the banks) and writes 128 bytes of
// each of the 128 V^T rows, keys past the segment's end as zeros.  HBM bound: 2 bytes read and 2 written per
// element.  Text keys are gathered by row on the way (a few hundred rows at most), and their K rows copied to the
// packed buffer, where the attention kernel's tile loads can take them as a segment.  46 us for 24 heads x 19600
// keys, 5.3 TB/s; torch's permuting copy of one such V took about 400 us.
struct PackPart {
  const uint16_t* v;
  int64_t svb, svh, svj;
  int64_t len, tile0;
};

struct PackArgs {
  PackPart part[2];       // shared segments, then the text source below
  int nparts;
  int64_t text_tile0, tiles;
  const uint16_t *tk_src, *tv_src;
  int64_t tkb, tkh, tkj, tvb, tvh, tvj;
  const int64_t* rows;
  int64_t text_off;       // the text rows start here in rows
  uint16_t* vt;
  int64_t svb, svh, svd;
  uint16_t* tk;
  int64_t t_rows;
  int* owner;
  int64_t Lq;
  int H;
  int ngroups;
  AttnGroup group[kMaxGroups];
  int t_off[kMaxGroups];  // each group's first text row, from text_off
};

constexpr int kPackThreads = 256;

__global__ __launch_bounds__(kPackThreads) void attention_pack_kernel(const PackArgs a) {
  __shared__ uint32_t rows32[kBK * 65];  // row = key, 64 dwords of dim pairs, one dword of padding
  const int tid = threadIdx.x;
  const int64_t tile = blockIdx.x;
  const int64_t b = blockIdx.y / a.H, h = blockIdx.y % a.H;
  if (tile == a.tiles) {  // one more workgroup: the group whose result each query row takes (the last naming it)
    if (blockIdx.y != 0) return;
    for (int64_t i = tid; i < a.Lq; i += kPackThreads) a.owner[i] = -1;
    __threadfence();
    __syncthreads();
    for (int g = 0; g < a.ngroups; g++)
      for (int i = tid; i < a.group[g].q_n; i += kPackThreads) atomicMax(&a.owner[a.rows[a.group[g].q_off + i]], g);
    return;
  }
  // the tile's rows
  const uint16_t *vsrc, *ksrc = nullptr;
  int64_t vj, first = 0, len;
  const int64_t* idx = nullptr;
  int64_t kpos = 0;
  if (tile < a.text_tile0) {
    const PackPart& p = a.part[a.nparts > 1 && tile >= a.part[1].tile0 ? 1 : 0];
    first = (tile - p.tile0) * kBK;
    len = p.len - first;
    vsrc = p.v + b * p.svb + h * p.svh + first * p.svj;
    vj = p.svj;
  } else {
    kpos = (tile - a.text_tile0) * kBK;
    int g = 0;
    while (g + 1 < a.ngroups && kpos >= a.group[g + 1].t_pos) g++;
    first = kpos - a.group[g].t_pos;
    len = a.group[g].t_n - first;
    idx = a.rows + a.text_off + a.t_off[g] + first;
    vsrc = a.tv_src + b * a.tvb + h * a.tvh;
    ksrc = a.tk_src + b * a.tkb + h * a.tkh;
    vj = a.tvj;
  }
  const int n = len < kBK ? (int)len : kBK;
  const int c = tid & 15;
#pragma unroll
  for (int u = 0; u < 4; u++) {
    const int r = (tid >> 4) + 16 * u;
    uint4 v = make_uint4(0, 0, 0, 0);
    if (r < n) {
      const int64_t row = idx ? idx[r] : r;
      v = ld_nt16(vsrc + row * vj + c * 8);
      if (ksrc)
        *reinterpret_cast<uint4*>(a.tk + ((b * a.H + h) * a.t_rows + kpos + r) * kHeadDim + c * 8) =
            *reinterpret_cast<const uint4*>(ksrc + row * a.tkj + c * 8);
    }
    uint32_t* d = rows32 + r * 65 + c * 4;
    d[0] = v.x; d[1] = v.y; d[2] = v.z; d[3] = v.w;
  }
  __syncthreads();
  // chunk ch = 2 g + s of dim rows 2 p and 2 p + 1: the keys 16 g + 4 s + 0..3 and 16 g + 8 + 4 s + 0..3
  uint16_t* out = a.vt + b * a.svb + h * a.svh + tile * kBK;
#pragma unroll
  for (int u = 0; u < 2; u++) {
    const int ch = tid & 7, p = (tid >> 3) + 32 * u;
    uint32_t x[8];
#pragma unroll
    for (int e = 0; e < 8; e++) x[e] = rows32[((ch >> 1) * 16 + (e >> 2) * 8 + (ch & 1) * 4 + (e & 3)) * 65 + p];
    uint4 lo, hi;
    lo.x = __builtin_amdgcn_perm(x[1], x[0], 0x05040100u); hi.x = __builtin_amdgcn_perm(x[1], x[0], 0x07060302u);
    lo.y = __builtin_amdgcn_perm(x[3], x[2], 0x05040100u); hi.y = __builtin_amdgcn_perm(x[3], x[2], 0x07060302u);
    lo.z = __builtin_amdgcn_perm(x[5], x[4], 0x05040100u); hi.z = __builtin_amdgcn_perm(x[5], x[4], 0x07060302u);
    lo.w = __builtin_amdgcn_perm(x[7], x[6], 0x05040100u); hi.w = __builtin_amdgcn_perm(x[7], x[6], 0x07060302u);
    *reinterpret_cast<uint4*>(out + (2 * p) * a.svd + ch * 8) = lo;
    *reinterpret_cast<uint4*>(out + (2 * p + 1) * a.svd + ch * 8) = hi;
  }
}

int64_t tiles_of(int64_t n) { return (n + kBK - 1) / kBK; }

// How the query blocks (units) of a call share their key tiles: the first `whole` take one workgroup each, the others
// `splits`.  Times are in tiles of a compute unit that holds two workgroups: a round of workgroups takes its tiles plus
// about four for its start and end, a last round of at most one workgroup per unit 0.7 of that (its waves have the SIMD
// to themselves), a combine pass its launch and 128 KB of traffic per workgroup.  Whole rounds stay whole (their partials
// would be traffic for nothing), or nothing does; ranges stay at four tiles or more, split workgroups at four rounds (the
// partials' memory), and a split has to promise a thirtieth, of a
// last round alone a sixtieth.
// Measured whole calls, no split against the chosen one (us): 16 units x 290 tiles 316 -> 61, 40 x 73 89 -> 40, 144 x 49
// 69 -> 58, 216 x 129 191 -> 148, 336 x 182 330 -> 281, 592 x 213 618 -> 506; with a split last round only, 1024 x 157
// 760 -> 665, 1560 x 129 853 -> 790, 3168 x 264 3165 -> 3038, 3344 x 416 5330 -> 5090.
struct Split {
  int64_t whole;
  int splits;
};
Split choose_splits(int64_t units, int64_t tiles) {
  const int64_t cus = cu_count(), slots = 2 * cus;
  auto cost = [&](int64_t whole, int64_t s) {
    const int64_t wgs = (units - whole) * s, full = wgs / slots, rem = wgs % slots;
    const double rounds = full + (rem == 0 ? 0.0 : rem <= cus ? 0.7 : 1.0);
    return (double)(whole / slots) * (tiles + 4) + rounds * ((tiles + s - 1) / s + 4) + (s > 1 ? 2.0 + 0.016 * wgs : 0.0);
  };
  Split best{0, 1};
  const double one = cost(0, 1);
  double least = one;
  const int64_t rounds = units / slots * slots;
  for (int64_t whole : {(int64_t)0, rounds})
    for (int64_t s = 2; s <= 64 && s * 4 <= tiles && (units - whole) * s <= 4 * slots && units > whole; s++)
      if (cost(whole, s) < least && cost(whole, s) < one * (whole ? 59.0 / 60 : 29.0 / 30)) {
        best = Split{whole, (int)s};
        least = cost(whole, s);
      }
  return best;
}

// Bytes of the partials of `units` query blocks: outputs, then maxima and sums.
int64_t partial_bytes(int64_t units, Split sp) {
  return sp.splits > 1 ? (units - sp.whole) * sp.splits * kBQ * (kHeadDim * 4 + 8) : 0;
}

// Launches the attention kernel over args whose pointers, strides, segments and groups are set; `partials` is
// where the partials of split blocks go.
int launch_attention(AttnArgs& a, int64_t B, float scale, Split sp, char* partials, hipStream_t st) {
  int64_t qblocks = 0;
  for (int g = 0; g < a.ngroups; g++) {
    a.group[g].qb0 = (int)qblocks;
    qblocks += ((int64_t)a.group[g].q_n + kBQ - 1) / kBQ;
  }
  const int64_t units = B * a.H * qblocks;
  HN_REQUIRE(units * sp.splits <= 0x7fffffff, "hn_attention: problem too large");
  if (units == 0) return HN_OK;
  a.scale_log2 = scale * 1.4426950408889634f;
  a.qblocks = (int)qblocks;
  a.splits = sp.splits;
  a.whole = (int)sp.whole;
  a.tail = (int)(units - sp.whole);
  const dim3 grid((unsigned)(sp.splits > 1 ? sp.whole + a.tail * (int64_t)sp.splits : units)), block(kAttnWaves * 64);
  if (sp.splits == 1) {
    hipLaunchKernelGGL(attention_kernel<false>, grid, block, 0, st, a);
    return HN_LAUNCH_CHECK("attention_kernel");
  }
  a.po = (float4*)partials;
  a.pml = (float2*)(partials + (int64_t)a.tail * sp.splits * kBQ * kHeadDim * 4);
  hipLaunchKernelGGL(attention_kernel<true>, grid, block, 0, st, a);
  const int rc = HN_LAUNCH_CHECK("attention_kernel");
  if (rc != HN_OK) return rc;
  hipLaunchKernelGGL(attention_combine_kernel, dim3((unsigned)a.tail * 4), dim3(kCombineThreads), 0, st, a);
  return HN_LAUNCH_CHECK("attention_combine_kernel");
}

// The workspace of hn_segment_attention: V^T [B, H, 128, positions], packed text keys [B, H, t_rows, 128], the
// owner of each query row, the partials of split keys; each from a 256-byte boundary.
struct SegmentLayout {
  int64_t positions, t_rows, tk, owner, partials, bytes;
  Split split;
};
SegmentLayout segment_layout(const int64_t* parts, int n_parts, const int64_t* groups, int n_groups, int64_t B,
                             int64_t H, int64_t Lq) {
  SegmentLayout l{};
  int64_t qblocks = 0, tiles = 0, fewest = -1;  // of all groups; of the shared parts; text tiles of the shortest group
  for (int g = 0; g < n_groups; g++) {
    const int64_t q_n = groups[4 * g + 1], t = tiles_of(groups[4 * g + 3]);
    l.t_rows += t * kBK;
    qblocks += (q_n + kBQ - 1) / kBQ;
    if (q_n > 0 && (fewest < 0 || t < fewest)) fewest = t;
  }
  if (n_groups == 0) qblocks = (Lq + kBQ - 1) / kBQ;
  for (int p = 0; p < n_parts; p++) tiles += tiles_of(parts[9 * p + 8]);
  l.positions = l.t_rows + tiles * kBK;
  const int64_t units = B * H * qblocks;
  l.split = choose_splits(units, tiles + (fewest > 0 ? fewest : 0));  // every group has a tile for every range
  auto align = [](int64_t x) { return (x + 255) / 256 * 256; };
  l.tk = align(B * H * kHeadDim * l.positions * 2);
  l.owner = l.tk + align(B * H * kHeadDim * l.t_rows * 2);
  l.partials = l.owner + (n_groups ? align(Lq * 4) : 0);
  l.bytes = l.partials + partial_bytes(units, l.split);
  return l;
}

}  // namespace
}  // namespace hn

static int attention_impl(const void* q, int64_t sqb, int64_t sqh, int64_t sqi, const void* k, int64_t skb,
                            int64_t skh, int64_t skj, const void* vt, int64_t svb, int64_t svh, int64_t svd,
                            void* out, int64_t sob, int64_t soh, int64_t soi, int64_t B, int64_t H, int64_t Lq,
                            int64_t Lk, int64_t D, float scale, void* workspace, int64_t workspace_bytes, void* stream) {
  using namespace hn;
  HN_REQUIRE(B >= 0 && H > 0 && Lq >= 0 && Lk > 0, "hn_attention: bad shape B=%lld H=%lld Lq=%lld Lk=%lld",
             (long long)B, (long long)H, (long long)Lq, (long long)Lk);
  HN_REQUIRE(D == kHeadDim, "hn_attention: head dim %lld (128 only)", (long long)D);
  HN_REQUIRE(q && k && vt && out, "hn_attention: null pointer");
  HN_REQUIRE(svd >= (Lk + kBK - 1) / kBK * kBK,
             "hn_attention: V^T rows must hold ceil(Lk / 64) * 64 keys (svd=%lld for Lk=%lld)", (long long)svd,
             (long long)Lk);
  HN_REQUIRE(((uintptr_t)q & 15) == 0 && ((uintptr_t)k & 15) == 0 && ((uintptr_t)vt & 15) == 0 &&
                 ((uintptr_t)out & 7) == 0,
             "hn_attention: q, k, v^T must be 16-byte and out 8-byte aligned");
  HN_REQUIRE(sqi % 8 == 0 && skj % 8 == 0 && svd % 8 == 0 && sqh % 8 == 0 && skh % 8 == 0 && svh % 8 == 0 &&
                 sqb % 8 == 0 && skb % 8 == 0 && svb % 8 == 0 && soi % 4 == 0 && soh % 4 == 0 && sob % 4 == 0,
             "hn_attention: strides must keep rows 16-byte aligned (out 8-byte)");
  HN_REQUIRE(skj > 0 && skj <= (1 << 23) && svd > 0 && svd <= (1 << 22),
             "hn_attention: key stride %lld / V^T row stride %lld out of range (tile offsets are 32-bit)",
             (long long)skj, (long long)svd);
  HN_REQUIRE(scale > 0.0f && scale < 1e30f, "hn_attention: bad scale");
  HN_REQUIRE(Lq <= 0x7fffffff - kBQ && Lk <= ((int64_t)1 << 36) && H <= 0x7fffffff, "hn_attention: problem too large");
  if (B == 0 || Lq == 0) return HN_OK;
  AttnArgs a{};
  a.q = (const uint16_t*)q; a.sqb = sqb; a.sqh = sqh; a.sqi = sqi;
  a.seg[0] = AttnSeg{(const uint16_t*)k, skb, skh, skj, Lk, 0};
  a.nseg = 1;
  a.vt = (const uint16_t*)vt; a.svb = svb; a.svh = svh; a.svd = svd;
  a.o = (uint16_t*)out; a.sob = sob; a.soh = soh; a.soi = soi;
  a.H = (int)H;
  a.ngroups = 1;
  a.group[0] = AttnGroup{0, 0, (int)Lq, 0, 0};
  const int64_t units = B * H * ((Lq + kBQ - 1) / kBQ);
  const Split split = workspace ? choose_splits(units, tiles_of(Lk)) : Split{0, 1};
  HN_REQUIRE(workspace_bytes >= partial_bytes(units, split) && ((uintptr_t)workspace & 15) == 0,
             "hn_attention_ws: workspace of %lld bytes (16-byte aligned), %lld needed", (long long)workspace_bytes,
             (long long)partial_bytes(units, split));
  return launch_attention(a, B, scale, split, (char*)workspace, (hipStream_t)stream);
}

extern "C" int hn_attention(const void* q, int64_t sqb, int64_t sqh, int64_t sqi, const void* k, int64_t skb,
                            int64_t skh, int64_t skj, const void* vt, int64_t svb, int64_t svh, int64_t svd,
                            void* out, int64_t sob, int64_t soh, int64_t soi, int64_t B, int64_t H, int64_t Lq,
                            int64_t Lk, int64_t D, float scale, void* stream) {
  return attention_impl(q, sqb, sqh, sqi, k, skb, skh, skj, vt, svb, svh, svd, out, sob, soh, soi, B, H, Lq, Lk, D, scale,
                        nullptr, 0, stream);
}

extern "C" int64_t hn_attention_workspace_bytes(int64_t B, int64_t H, int64_t Lq, int64_t Lk) {
  using namespace hn;
  if (B < 0 || H <= 0 || Lq < 0 || Lk <= 0) return -1;
  const int64_t units = B * H * ((Lq + kBQ - 1) / kBQ);
  return partial_bytes(units, choose_splits(units, tiles_of(Lk)));
}

extern "C" int hn_attention_ws(const void* q, int64_t sqb, int64_t sqh, int64_t sqi, const void* k, int64_t skb,
                               int64_t skh, int64_t skj, const void* vt, int64_t svb, int64_t svh, int64_t svd,
                               void* out, int64_t sob, int64_t soh, int64_t soi, int64_t B, int64_t H, int64_t Lq,
                               int64_t Lk, int64_t D, float scale, void* workspace, int64_t workspace_bytes,
                               void* stream) {
  return attention_impl(q, sqb, sqh, sqi, k, skb, skh, skj, vt, svb, svh, svd, out, sob, soh, soi, B, H, Lq, Lk, D, scale,
                        workspace, workspace_bytes, stream);
}

extern "C" int64_t hn_segment_attention_workspace_bytes(const int64_t* parts, int n_parts, const int64_t* groups,
                                                        int n_groups, int64_t B, int64_t H, int64_t Lq) {
  using namespace hn;
  if (!parts || n_parts < 1 || n_parts > 2 || n_groups < 0 || n_groups > kMaxGroups || (n_groups && !groups) || B < 0 ||
      H <= 0 || Lq < 0)
    return -1;
  return segment_layout(parts, n_parts, groups, n_groups, B, H, Lq).bytes;
}

extern "C" int hn_segment_attention(const void* q, int64_t sqb, int64_t sqh, int64_t sqi, const int64_t* parts,
                                    int n_parts, const int64_t* text, const int64_t* groups, int n_groups,
                                    const int64_t* rows, int64_t text_off, void* out, int64_t sob, int64_t soh,
                                    int64_t soi, int64_t B, int64_t H, int64_t Lq, int64_t D, float scale,
                                    void* workspace, int64_t workspace_bytes, void* stream) {
  using namespace hn;
  HN_REQUIRE(B >= 0 && H > 0 && H <= 65535 && B * H <= 65535 && Lq >= 0 && Lq <= 0x7fffffff - kBQ,
             "hn_segment_attention: bad shape B=%lld H=%lld Lq=%lld", (long long)B, (long long)H, (long long)Lq);
  HN_REQUIRE(D == kHeadDim, "hn_segment_attention: head dim %lld (128 only)", (long long)D);
  HN_REQUIRE(n_parts >= 1 && n_parts <= 2 && parts, "hn_segment_attention: one or two shared key parts, got %d", n_parts);
  HN_REQUIRE(n_groups >= 0 && n_groups <= kMaxGroups, "hn_segment_attention: at most %d query groups, got %d", kMaxGroups,
             n_groups);
  HN_REQUIRE(n_groups == 0 || (groups && rows && text), "hn_segment_attention: groups without rows or text source");
  HN_REQUIRE(q && out && workspace, "hn_segment_attention: null pointer");
  HN_REQUIRE(scale > 0.0f && scale < 1e30f, "hn_segment_attention: bad scale");
  auto rows16 = [](const int64_t* t) {  // pointer, then batch / head / token strides: 16-byte aligned rows
    return t[0] != 0 && (t[0] & 15) == 0 && t[1] % 8 == 0 && t[2] % 8 == 0 && t[3] % 8 == 0 && t[3] > 0 && t[3] <= (1 << 23);
  };
  int64_t shared = 0;
  for (int p = 0; p < n_parts; p++) {
    HN_REQUIRE(rows16(parts + 9 * p) && rows16(parts + 9 * p + 4) && parts[9 * p + 8] >= 0,
               "hn_segment_attention: key part %d must have 16-byte aligned rows, token strides in (0, 2^23]", p);
    shared += parts[9 * p + 8];
  }
  HN_REQUIRE(((uintptr_t)q & 15) == 0 && sqb % 8 == 0 && sqh % 8 == 0 && sqi % 8 == 0 && ((uintptr_t)out & 7) == 0 &&
                 sob % 4 == 0 && soh % 4 == 0 && soi % 4 == 0,
             "hn_segment_attention: q rows must be 16-byte and out rows 8-byte aligned");
  HN_REQUIRE(n_groups == 0 || (rows16(text) && rows16(text + 4)), "hn_segment_attention: text rows must be 16-byte aligned");
  const SegmentLayout l = segment_layout(parts, n_parts, groups, n_groups, B, H, Lq);
  HN_REQUIRE(l.positions <= (1 << 22), "hn_segment_attention: %lld key positions (at most 2^22)", (long long)l.positions);
  HN_REQUIRE(workspace_bytes >= l.bytes && ((uintptr_t)workspace & 255) == 0,
             "hn_segment_attention: workspace of %lld bytes (256-byte aligned), %lld needed", (long long)workspace_bytes,
             (long long)l.bytes);
  for (int g = 0; g < n_groups; g++) {
    const int64_t* w = groups + 4 * g;
    HN_REQUIRE(w[0] >= 0 && w[1] >= 0 && w[2] >= 0 && w[3] >= 0 && w[0] + w[1] <= 0x7fffffff && w[2] + w[3] <= 0x7fffffff,
               "hn_segment_attention: bad group %d", g);
    HN_REQUIRE(w[1] == 0 || shared + w[3] > 0, "hn_segment_attention: no keys for group %d", g);
  }
  HN_REQUIRE(n_groups > 0 || Lq == 0 || shared > 0, "hn_segment_attention: no keys");
  if (B == 0 || Lq == 0) return HN_OK;

  char* ws = (char*)workspace;
  AttnArgs a{};
  PackArgs p{};
  a.q = (const uint16_t*)q; a.sqb = sqb; a.sqh = sqh; a.sqi = sqi;
  a.vt = (const uint16_t*)ws;
  a.svd = l.positions; a.svh = kHeadDim * l.positions; a.svb = H * a.svh;
  a.o = (uint16_t*)out; a.sob = sob; a.soh = soh; a.soi = soi;
  a.H = (int)H;
  p.vt = (uint16_t*)ws; p.svb = a.svb; p.svh = a.svh; p.svd = a.svd; p.H = (int)H; p.Lq = Lq;
  int64_t tile = 0;
  for (int i = 0; i < n_parts; i++) {
    const int64_t* w = parts + 9 * i;
    a.seg[i] = AttnSeg{(const uint16_t*)w[0], w[1], w[2], w[3], w[8], tile * kBK};
    p.part[i] = PackPart{(const uint16_t*)w[4], w[5], w[6], w[7], w[8], tile};
    tile += tiles_of(w[8]);
  }
  a.nseg = p.nparts = n_parts;
  p.text_tile0 = tile;
  a.tvpos = tile * kBK;
  p.tiles = l.positions / kBK;
  a.t_rows = p.t_rows = l.t_rows;
  a.ngroups = 1;
  a.group[0] = AttnGroup{0, 0, (int)Lq, 0, 0};
  if (n_groups) {
    a.tk = p.tk = (uint16_t*)(ws + l.tk);
    a.owner = p.owner = (int*)(ws + l.owner);
    a.rows = p.rows = rows;
    p.text_off = text_off;
    p.tk_src = (const uint16_t*)text[0]; p.tkb = text[1]; p.tkh = text[2]; p.tkj = text[3];
    p.tv_src = (const uint16_t*)text[4]; p.tvb = text[5]; p.tvh = text[6]; p.tvj = text[7];
    a.ngroups = p.ngroups = n_groups;
    int64_t pos = 0;
    for (int g = 0; g < n_groups; g++) {
      const int64_t* w = groups + 4 * g;
      a.group[g] = p.group[g] = AttnGroup{0, (int)w[0], (int)w[1], (int)w[3], (int)pos};
      p.t_off[g] = (int)w[2];
      pos += tiles_of(w[3]) * kBK;
    }
  }
  const dim3 grid((unsigned)(p.tiles + (n_groups ? 1 : 0)), (unsigned)(B * H));
  hipLaunchKernelGGL(attention_pack_kernel, grid, dim3(kPackThreads), 0, (hipStream_t)stream, p);
  const int rc = HN_LAUNCH_CHECK("attention_pack_kernel");
  return rc != HN_OK ? rc : launch_attention(a, B, scale, l.split, ws + l.partials, (hipStream_t)stream);
}
