// Prefill (chunked) attention over the cache, every mode.
//
// Replaces mlx_rs::fast::scaled_dot_product_attention for L > 1
// (src/model/gemma4_attention.rs:84-104) with the causal mask of
// create_attention_mask and the sliding band of create_sliding_mask
// (src/model/mod.rs:682-753): query position p sees key positions j with
// lo(p) <= j <= p, lo(p) = max(trim, p - W + 1) on sliding layers.
//
// One work-group = 64 query rows (a row is one (position, q head) of the
// KV head's GQA group: 64 / G consecutive positions) of one KV head; a step
// covers 32 keys (two head-blocks). head_dim is split over the waves: wave g
// of the D / 64 owns the 64 dims of group g for all 64 rows, in both
// products, so every stored code is read from memory and turned into a
// matrix-core operand by exactly one wave of the work-group, straight into
// registers (no LDS staging), and is used for four 16-row tiles. (One pair of
// waves per 16 rows, every pair decoding every block, took 7.78 ms for a
// 2048-token chunk after 32768 positions, 16 q / 2 KV heads of 512 dims, 8
// bits; this split takes 5.2 ms, and 0.147 against 0.227 ms for a 2048-token
// chunk on a 1024-position ring, 16 / 8 heads of 256 dims, 4 bits.) Small grids
// at head_dim 128 and 256 share the rows among eight waves, RW = 4 and 2 per 64
// dims (prefill_plan).
//
// What bounds it: the issue of matrix and vector instructions together. A
// 16x16x32 MFMA alone takes 8.7 ns of a SIMD, with four independent FMAs after
// it 12.4 ns (the FMAs alone: 5): they hardly overlap, also between the two
// waves of a SIMD. Of the 2.5 us of a step of a SIMD (8 bits, head_dim 512)
// its 128 MFMAs are 1.1 us, the conversion of codes and weights, the scales
// and the softmax the rest. Hence the packed f16 arithmetic on the weights
// (v_pk_* 1.9 ns for two elements; v_fma_mixlo_f16 3.7 ns for one).
//
//   QK^T  S_g^T[32 key x 64 row] = K_g . Q_g^T per wave: a partial score over
//         its 64 dims, handed through LDS to the wave that sums the row's
//         partials;
//   softmax of 64 / (number of waves) rows per wave: sum, mask, running max, weights
//         P to LDS, and the factor by which every wave rescales its row
//         accumulators when a row's reference max moved;
//   PV    O_g^T[64 dim x 64 row] += V_g^T[64 dim x 32 key] . P^T[32 key x 64
//         row] per wave.
//
// The three stages run as a pipeline, one barrier per step: between two
// barriers a wave issues the QK of step i + 1, the softmax of step i and the
// PV of step i - 1, which depend on nothing of one another (score and weight
// buffers alternate), so the two waves of a SIMD overlap one's matrix-core
// work with the other's vector work. Codes are loaded a step ahead.
//
// Operands, affine caches: K and V codes as exact f16 integers, q_rot as an
// f16 high part and an f16 residual (~22 bits), the residual's products
// first, then the high part's, in one accumulator; then s_g = scale * acc +
// bias * sum(q_group); P' = p * v_scale likewise as f16 high part and residual
// (two MFMAs), the bias terms summed on the side in f32. (Codes as f16
// subnormals, code * 2^-24, would save the subtract of the conversion, but
// the matrix cores keep 2 bits less of such products: relative error 1.7e-7
// against 5e-8 over 32 products.)
// Codebook (TurboQuant) caches: the indices become f16 centroid operands
// through the decode kernel's LDS lookup table (fmkv_cb_common.h). 2 and 3
// bits: the exact integer operands 1000 * centroid, S^T = C . q_lo + C . q_hi,
// scaled per key by norm / (1000 sqrt(D)); O^T likewise with P' = p * norm /
// (1000 sqrt(D)) as f16 high part and residual (two MFMAs each). 4 bits: the
// centroids' f16 high part and residual, S^T = C_hi . q_hi + C_lo . q_hi +
// C_hi . q_lo and O^T likewise (three MFMAs each: the fourth product is below
// f32 rounding).
// Plain (bf16) caches read K rows and V columns as bf16 operands
// (v_mfma_f32_16x16x32_bf16) against the raw bf16 q (exact products; the
// softmax scale applies after), P as bf16 high part and residual; no rotation.
//
// The 32 keys of a PV product are ordered [4j .. 4j+3 of the first block,
// 4j .. 4j+3 of the second] for lane group j on both operands: V codes as
// stored for one block's 16-key tile feed the 32-key instruction, which has
// twice the 16-key one's rate.
//
// A paged pool runs one sequence per grid z with its own start position and
// block table (linear sequences: the append goes first).
//
// A grid that would leave CUs idle is split over the keys as well (units > 0):
// grid z then counts (sequence, key range) units instead of sequences, each
// sequence getting a number of ranges that follows its length
// (prefill_unit), and a second kernel merges the ranges' partial rows. Four
// 77-token chunks after 700 .. 8000 positions (16 q / 2 KV heads of 512 dims,
// 3-bit codebook: 80 work-groups, the longest of 253 steps): 0.19 ms against
// 0.575 unsplit.
//
// Keys come from two stores: positions below p_split from old_st (the ring
// of a sliding layer, read before the chunk's own append can overwrite
// positions early queries still need), the rest from new_st (a staging
// copy of the chunk, or the cache itself for linear caches). A block that
// straddles p_split is visited once per store with the other part masked.
#include <type_traits>

#include "fmkv_device.h"
#include "fmkv_internal.h"
#include "fmkv_attn_common.h"
#include "fmkv_cb_common.h"

namespace fmkv {
namespace {

constexpr int kPfRows = 64;   // query rows per work-group, four matrix-core tiles
constexpr int kPfTiles = kPfRows / 16;
constexpr int kPfKeys = 2 * kBlockTokens;  // keys per step
constexpr int kPfQuads = kPfKeys / 4;      // groups of four keys of a step
constexpr int kPfMinSteps = 4;             // steps of the shortest key range of a split call
constexpr int kPfFewSteps = 32;            // a call of sequences shorter than this is short
// How far (base 2) a score may exceed its row's reference maximum before the
// row is rescaled. Weights stay below 2^7, and a weight times a V scale that an
// affine cache's attention documents as valid (below 511) within f16. The
// matrix cores would take an infinite high part and residual to NaN. (MODE's
// FP16_OVFL clamps such results to 65504 at no cost, but the matrix cores heed
// it too and turn infinite products and sums into finite ones.)
constexpr float kPfSlack = 7.0f;

// 2- and 3-bit codebook caches weigh V by p * norm / (1000 sqrt(D)), mostly
// below 2^-8, where an f16 residual is subnormal and ends at 2^-25: their
// weights carry a factor 32 that the accumulated row loses again (norm is an
// f16, so p <= 2^7 and D >= 128 keep them below 2.4e4). Relative error against
// 64 bits over 3000 .. 6000 positions, 3 bits, head_dim 512 / 256 / 128: 2.0e-5 /
// 1.9e-4 / 1.6e-6; 2.8e-4 / 2.8e-4 / 1.7e-4 without it, weights cut toward zero.
template <int BITS>
constexpr float kPvScale = kCbExact<BITS> ? 32.0f : 1.0f;

// RW: ways that the 64 rows are shared among the waves (each dim group's
// waves), 1 or as many as make eight waves
template <int D, int BITS, int MODE, int RW>
struct PfPlan {
  static constexpr BlockLayout L = make_layout(D, BITS, MODE);
  static constexpr int NG = D / 64;
  static constexpr int NW = NG * RW;  // waves: RW per 64 dims
  static constexpr int PT = kPfTiles / RW;  // row tiles per wave
  static_assert(RW == 1 || NW == 8, "eight waves where rows are shared");
  // The softmax stage: with 8 waves a wave sums 8 rows, lane l holding key
  // quad l >> 3 of row l & 7. With 4 (2) waves it sums one (two) whole row
  // tiles in the QK accumulators' own layout, so its own partial stays in
  // registers.
  static constexpr bool kOwn = NW < 8;
  static constexpr int NRS = NW == 2 ? 2 : 1;  // row sets per lane
  static constexpr int NQ = kOwn ? 2 : 1;      // key quads per lane and row set
  static constexpr int kSrc = kOwn ? NG - 1 : NG;  // partials of a tile in LDS
  static constexpr int kXs = kPfTiles * kSrc * 2 * 1024;  // one score buffer
  static constexpr int kPb = kPfQuads * kPfRows * 16;     // one weight buffer
  static constexpr int kPbOff = 2 * kXs;
  static constexpr int kAlOff = kPbOff + 2 * kPb;
  static constexpr int kLutOff = kAlOff + 2 * kPfRows * 4;
  static constexpr int kLutBytes = MODE == kCodebook ? CbLut<BITS == 16 ? 2 : BITS>::kBytes : 0;
  static constexpr int kQStride = D + 8;  // 16-bit values per q-table row (padding against bank conflicts)
  // q table: high and residual parts of q_rot (affine: and group sums);
  // plain: the raw bf16 rows
  static constexpr int kQTab = (MODE == kPlain ? 1 : 2) * kPfRows * kQStride * 2 +
                               (MODE == kAffine ? kPfRows * NG * 4 : 0);
  static constexpr int kRStride = D + 4;  // f32 per output row
  static constexpr int kRows = kPfRows * kRStride * 4;
  static constexpr int kRegion = cmax(cmax(kLutOff + kLutBytes, kQTab), kRows);
  // words per lane of one block's codes of the wave's 64 dims
  static constexpr int KW = MODE == kAffine ? BITS / 2 : MODE == kPlain ? 8 : BITS == 3 ? 4 : 2;
  static constexpr int VW = MODE == kAffine ? BITS / 2 : MODE == kPlain ? 8 : BITS == 3 ? 8 : 4;
};

// K operand of MFMA s of group g as the plain codes (exact f16 integers);
// w: the lane's words of the group.
template <int BITS>
__device__ inline half8_t k_operand_plain(const uint32_t* w, int s) {
  if constexpr (BITS == 8) {
    const uint32_t w0 = w[2 * s], w1 = w[2 * s + 1];
    return cat8(u8x2_to_h2(w0, 0x04010400u), u8x2_to_h2(w0, 0x04030402u),
                u8x2_to_h2(w1, 0x04010400u), u8x2_to_h2(w1, 0x04030402u));
  } else {
    return cat8(u4x2_to_h2(w[s], 0), u4x2_to_h2(w[s], 1), u4x2_to_h2(w[s], 2), u4x2_to_h2(w[s], 3));
  }
}

// V operand of column tile ct: tokens 4j .. 4j+3 of two blocks, as the plain
// codes; wa, wb: the lane's words of the group in either block.
template <int BITS>
__device__ inline half8_t v_operand_plain(const uint32_t* wa, const uint32_t* wb, int ct) {
  if constexpr (BITS == 8) {
    return cat8(u8x2_to_h2(wa[ct], 0x04010400u), u8x2_to_h2(wa[ct], 0x04030402u),
                u8x2_to_h2(wb[ct], 0x04010400u), u8x2_to_h2(wb[ct], 0x04030402u));
  } else {
    const int k0 = (ct & 1) * 2;
    return cat8(u4x2_to_h2(wa[ct >> 1], k0), u4x2_to_h2(wa[ct >> 1], k0 + 1),
                u4x2_to_h2(wb[ct >> 1], k0), u4x2_to_h2(wb[ct >> 1], k0 + 1));
  }
}

typedef __bf16 bf16x8_t __attribute__((ext_vector_type(8)));
__device__ inline uint32_t pack_bf16x2(float a, float b) {
  return (uint32_t)f32_to_bf16(a) | ((uint32_t)f32_to_bf16(b) << 16);
}

// A uniform address in memory and loads at a lane's offset from it. (Global
// address space: a generic pointer's flat loads also count as LDS operations,
// and every wait for LDS data or at a barrier would wait for memory too.)
typedef const uint8_t __attribute__((address_space(1)))* gptr_t;
typedef uint32_t u32x2 __attribute__((ext_vector_type(2)));
typedef u32x2 u32x2_a4 __attribute__((aligned(4)));  // two words at a 4-byte boundary
template <class T>
__device__ inline T load_at(gptr_t p, uint32_t off, int imm = 0) {
  return *reinterpret_cast<const T __attribute__((address_space(1)))*>(p + off + imm);
}

// 2 N consecutive bf16 in one load a lane (aligned to one of them only).
template <int N>
__device__ inline void load_words(const uint16_t* src, uint32_t (&w)[N]) {
  if constexpr (N == 1) {
    typedef uint32_t word __attribute__((aligned(2)));
    w[0] = *reinterpret_cast<const word*>(src);
  } else {
    typedef uint32_t vec __attribute__((ext_vector_type(N), aligned(2)));
    const vec v = *reinterpret_cast<const vec*>(src);
#pragma unroll
    for (int i = 0; i < N; i++) w[i] = v[i];
  }
}

// E consecutive outputs at element o_idx, in one store a lane (the caller's
// buffer is aligned to its elements only).
template <int E>
__device__ inline void store_out(const PrefillArgs& a, int64_t o_idx, const float (&v)[E]) {
  if (a.out_f32) {
    typedef float vec __attribute__((ext_vector_type(E), aligned(4)));
    vec o;
#pragma unroll
    for (int i = 0; i < E; i++) o[i] = v[i];
    *reinterpret_cast<vec*>(reinterpret_cast<float*>(a.out) + o_idx) = o;
  } else {
    typedef uint16_t vec __attribute__((ext_vector_type(E), aligned(2)));
    vec o;
#pragma unroll
    for (int i = 0; i < E; i++) o[i] = f32_to_bf16(v[i]);
    *reinterpret_cast<vec*>(reinterpret_cast<uint16_t*>(a.out) + o_idx) = o;
  }
}

// LDS of this wave written, every wave of the work-group here. Loads from
// memory stay in flight across it.
__device__ inline void lds_barrier() {
  asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
}

// Steps (32 keys) that a row tile of a sequence may need, from its start.
__device__ inline int prefill_steps(const PrefillArgs& a, int64_t p0) {
  const int64_t lo = a.vis_begin > 0 ? a.vis_begin : 0;
  int64_t keys = p0 + a.n_q - lo;
  if (a.window > 0 && keys > a.window + kPfRows) keys = a.window + kPfRows;
  if (keys > ((int64_t)1 << 25)) keys = (int64_t)1 << 25;  // (64 sequences' steps add up in 32 bits)
  return (int)((keys > 0 ? keys : 0) / kPfKeys) + 2;
}

// Scalar loads of what every lane reads alike.
typedef const int32_t __attribute__((address_space(4)))* cint_ptr;

// The sums of lanes 0 .. l, in every lane l: DPP row shifts, then the last
// lanes of rows broadcast over the rows after them.
__device__ inline int scan_add(int v) {
  v += __builtin_amdgcn_update_dpp(0, v, 0x111, 0xf, 0xf, true);   // row_shr:1
  v += __builtin_amdgcn_update_dpp(0, v, 0x112, 0xf, 0xf, true);   // row_shr:2
  v += __builtin_amdgcn_update_dpp(0, v, 0x114, 0xf, 0xf, true);   // row_shr:4
  v += __builtin_amdgcn_update_dpp(0, v, 0x118, 0xf, 0xf, true);   // row_shr:8
  v += __builtin_amdgcn_update_dpp(0, v, 0x142, 0xa, 0xf, false);  // row_bcast:15 into rows 1, 3
  v += __builtin_amdgcn_update_dpp(0, v, 0x143, 0xc, 0xf, false);  // row_bcast:31 into rows 2, 3
  return v;
}

// What unit u of the grid is: its sequence, the sequence's first unit and its
// number of key ranges. The range length c is the smallest (to a sixteenth)
// for which all sequences' ranges fit the units: the longest work-group, and
// with it the call, gets as short as the chip allows. Lane s computes
// sequence s (at most 64); every wave that asks gets the same answer. u < 0:
// the unit of range 0 of sequence `seq`.
struct PrefillUnit {
  int seq, first, ranges;
};
__device__ inline PrefillUnit prefill_unit(const PrefillArgs& a, int u, int seq, int lane) {
  // key ranges of a sequence of st steps, c steps each
  auto count = [&](int st, int c) { return st < a.min_split ? 1 : (st + c - 1) / c; };
  if (a.n_seqs == 1) {  // (the same, in scalar arithmetic)
    const int st = prefill_steps(a, a.start_pos ? (int64_t)((cint_ptr)(uintptr_t)a.start_pos)[0] : a.p0);
    int c = (st + a.units - 1) / a.units;
    if (c < kPfMinSteps) c = kPfMinSteps;
    const int n = count(st, c);
    return PrefillUnit{u < n ? 0 : -1, 0, n};
  }
  const int64_t p0 = lane < a.n_seqs ? (a.start_pos ? (int64_t)a.start_pos[lane] : a.p0) : 0;
  const int st = prefill_steps(a, p0);
  auto sum = [&](int v) { return (int)__builtin_amdgcn_readlane(scan_add(v), 63); };
  int n = lane < a.n_seqs ? 1 : 0;
  const uint64_t here = a.n_seqs < 64 ? (1ull << a.n_seqs) - 1 : ~0ull;
  if (__ballot(st >= a.min_split) & here) {
    int c = (sum(n ? st : 0) + a.units - 1) / a.units;
    if (c < kPfMinSteps) c = kPfMinSteps;
    n = n ? count(st, c) : 0;
    while (sum(n) > a.units) {  // ends: at c >= every st a sequence has one range, n_seqs <= units
      c += 1 + c / 16;
      n = n ? count(st, c) : 0;
    }
  }
  const int upto = scan_add(n);  // units of sequences 0 .. lane
  PrefillUnit r;
  if (u >= 0) {
    const uint64_t past = __ballot(upto > u);
    seq = past ? __builtin_ctzll(past) : -1;  // -1: a unit that nothing needs
  }
  r.seq = __builtin_amdgcn_readfirstlane(seq);
  const int s = r.seq < 0 ? 0 : r.seq;
  r.ranges = __builtin_amdgcn_readlane(n, s);
  r.first = __builtin_amdgcn_readlane(upto, s) - r.ranges;
  return r;
}

template <int D, int BITS, int MODE, int RW>
__global__ __launch_bounds__(D * RW)  // RW waves per 64 dims
__attribute__((amdgpu_waves_per_eu(RW == 4 ? 4 : 2, RW == 4 ? 4 : 2)))
void prefill_attn_kernel(PrefillArgs a) {
  using P = PfPlan<D, BITS, MODE, RW>;
  constexpr BlockLayout L = P::L;
  constexpr int NG = P::NG, NW = P::NW, PT = P::PT, E = D / 64, LPG = 64 / E;
  constexpr int NRS = P::NRS, NQ = P::NQ, KW = P::KW, VW = P::VW;
  constexpr bool kOwn = P::kOwn;
  constexpr int QS = P::kQStride, RS = P::kRStride;
  // codebook index width (the template's BITS; other modes never use it)
  constexpr int CB = MODE == kCodebook ? BITS : 2;

  __shared__ __align__(16) uint8_t region[P::kRegion];
  __shared__ float lrow[kPfRows], mrow[kPfRows];
  __shared__ int not_finite;

  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int dg = RW > 1 ? wave % NG : wave, rt0 = RW > 1 ? wave / NG * PT : 0;  // dim group, first row tile
  const int j = lane >> 4, c = lane & 15;
  const int G = a.group;
  const int QP = kPfRows / G;  // query positions per work-group
  const uint32_t g_inv = 65536u / (uint32_t)G + 1;
  auto pos_of = [&](int r) __attribute__((always_inline)) {  // r / G for rows r < 64, G <= 64
    return (int)((uint32_t)r * g_inv >> 16);
  };
  const int kvh = blockIdx.y;
  int seq = blockIdx.z, range = 0, ranges = 1;
  if (a.units > 0) {
    const PrefillUnit un = prefill_unit(a, blockIdx.z, 0, lane);
    if (un.seq < 0) return;
    seq = un.seq, range = (int)blockIdx.z - un.first, ranges = un.ranges;
  }
  const int qi0 = blockIdx.x * QP;
  // paged: the sequence's start, through a scalar load (everything derived
  // from it stays in scalar registers)
  const int64_t p0 = a.start_pos ? (int64_t)((cint_ptr)(uintptr_t)a.start_pos)[seq] : a.p0;
  const int nq = a.n_q - qi0 < QP ? a.n_q - qi0 : QP;  // valid positions of the tile

  // visible keys of position p: [lo(p), p]
  auto lo_of = [&](int64_t p) -> int64_t {
    int64_t lo = a.vis_begin;
    if (a.window > 0 && p - a.window + 1 > lo) lo = p - a.window + 1;
    return lo < 0 ? 0 : lo;
  };

  // ---- virtual blocks of the work-group: [lo(first), last] in 16-key
  // blocks, the part below p_split from old_st, the rest from new_st ----
  const int64_t pA = p0 + qi0, pB = p0 + qi0 + nq - 1;
  const int64_t wg_lo = lo_of(pA), wg_hi = pB;
  const int64_t b_lo = wg_lo / kBlockTokens, b_hi = wg_hi / kBlockTokens;
  const int64_t ps = a.p_split;
  int64_t old_last = (ps + kBlockTokens - 1) / kBlockTokens - 1;  // last block with keys < ps
  if (old_last > b_hi) old_last = b_hi;
  const int64_t n_old = old_last >= b_lo ? old_last - b_lo + 1 : 0;
  int64_t new_first = ps / kBlockTokens;
  if (new_first < b_lo) new_first = b_lo;
  const int64_t n_new = b_hi >= new_first ? b_hi - new_first + 1 : 0;
  const int nvb = (int)(n_old + n_new);
  const int nst = (nvb + 1) / 2;  // steps of two virtual blocks
  // Positions below are 32-bit and relative to the first block's first key
  // (a cache holds less than 2^31 positions). Virtual block i holds keys
  // 16 rb .. of block rb = i (old store) or i + vb_shift, of which those in
  // [vlo, vhi) are its own; past the last one the range is empty.
  const int64_t bl16 = b_lo * kBlockTokens;
  auto rel = [&](int64_t x) __attribute__((always_inline)) -> int {
    x -= bl16;
    return (int)(x < -(1 << 30) ? -(1 << 30) : x > INT32_MAX ? INT32_MAX : x);
  };
  const int b_lo_i = (int)b_lo, n_old_i = (int)n_old, vb_shift = (int)(new_first - b_lo) - n_old_i;
  const int ps_r = rel(ps), vis_r = rel(lo_of(0)), pA_r = rel(pA);
  const int win = (int)(a.window < INT32_MAX ? a.window : INT32_MAX);
  auto lo_rel = [&](int p) __attribute__((always_inline)) -> int {  // lo(p), relative
    return win > 0 && p - win + 1 > vis_r ? p - win + 1 : vis_r;
  };
  auto vb_range = [&](int i, int& vlo, int& vhi) __attribute__((always_inline)) {
    const bool old = i < n_old_i;
    const int t0 = (old ? i : i + vb_shift) * kBlockTokens, t1 = t0 + kBlockTokens;
    vlo = old ? t0 : t0 > ps_r ? t0 : ps_r;
    vhi = old ? (t1 < ps_r ? t1 : ps_r) : i < nvb ? t1 : vlo;
  };
  // Virtual block i's head-block (past the last one: the last one's), in
  // scalar arithmetic. A ring's slot block of virtual block i is ring0 + i
  // modulo its nrb blocks (the old keys lie in the last W positions before
  // p_split: n_old <= nrb + 1, so two conditional subtractions reduce it).
  const int nrb = a.ring_slots > 0 ? (int)(a.ring_slots / kBlockTokens) : 0;
  const int ring0 = nrb > 0 ? (int)(b_lo % nrb) : 0;
  const int32_t n_pool = (int32_t)(a.new_st.n_blocks < INT32_MAX ? a.new_st.n_blocks : INT32_MAX);
  const uint64_t base_old = reinterpret_cast<uint64_t>(a.old_st.base) + kvh * a.old_st.head_stride;
  const uint64_t base_new = reinterpret_cast<uint64_t>(a.new_st.base) + kvh * a.new_st.head_stride;
  const uint32_t t_width = a.new_st.block_table ? (uint32_t)a.new_st.table_stride : 0;
  const cint_ptr table =
      (cint_ptr)(uintptr_t)(a.new_st.block_table + (int64_t)seq * a.new_st.table_stride);
  auto blk_ptr = [&](int i) __attribute__((always_inline)) -> gptr_t {
    i = i < nvb ? i : nvb > 0 ? nvb - 1 : 0;
    if (i < n_old_i) {
      uint32_t phys = (uint32_t)(b_lo_i + i);
      if (nrb > 0) {
        int r = ring0 + i;
        r -= r >= nrb ? nrb : 0;
        r -= r >= nrb ? nrb : 0;
        phys = (uint32_t)r;
      }
      return (gptr_t)(base_old + (uint64_t)phys * (uint64_t)a.old_st.block_stride);
    }
    const uint32_t b = (uint32_t)(b_lo_i + i + vb_shift);
    uint32_t phys = b - (uint32_t)a.new_blk0;
    if (a.new_st.block_table) {
      // a table entry outside the pool (or a position past the table's
      // width) reads a valid block rather than faulting
      const int32_t e = b < t_width ? table[b] : 0;
      phys = (uint32_t)(e < 0 ? 0 : (e >= n_pool ? n_pool - 1 : e));
    }
    return (gptr_t)(base_new + (uint64_t)phys * (uint64_t)a.new_st.block_stride);
  };
  // every key of virtual block i is visible to every row: at or past the
  // largest lower bound, at or before the first position, not cut by p_split
  const int lo_max = lo_rel(pA_r + nq - 1);
  auto blk_full = [&](int i) __attribute__((always_inline)) -> bool {
    int vlo, vhi;
    vb_range(i, vlo, vhi);
    return vhi - vlo == kBlockTokens && vlo >= lo_max && vhi - 1 <= pA_r;
  };

  // ---- this wave's loads: the codes (and scale / bias) of its 64 dims in
  // the two blocks of a step ----
  uint32_t kr[2][KW], vr[2][VW];
  u32x4 km[2], vm[2];
  const int kbit = (c * (D / 2) + (dg % (NG / 2)) * 64 + 8 * j) * CB;
  const int vbit = (c * 16 + 4 * j) * CB;
  const uint32_t ksh = kbit & 31, vsh = vbit & 31;
  uint32_t k_off =
      (int)L.k_codes +
      (MODE == kAffine     ? (BITS == 8 ? dg * 1024 + lane * 16 : (dg >> 1) * 1024 + lane * 16 + (dg & 1) * 8)
       : MODE == kCodebook ? (dg / (NG / 2)) * (D * CB) + (kbit >> 5) * 4
                           : (c * D + dg * 64 + 8 * j) * 2);
  uint32_t v_off =
      (int)L.v_codes +
      (MODE == kAffine     ? (BITS == 8 ? dg * 1024 + lane * 16 : (dg >> 1) * 1024 + lane * 16 + (dg & 1) * 8)
       : MODE == kCodebook ? dg * (128 * CB) + (vbit >> 5) * 4
                           : ((dg * 64 + c) * kBlockTokens + 4 * j) * 2);
  uint32_t km_off = (int)L.k_meta + dg * 64 + j * 16;  // affine
  uint32_t vm_off = (int)L.v_meta + dg * 64 + j * 16;
  // Opaque in each step, or their extension to 64 bits leaves the loop, and
  // with it the form of the loads that adds a 32-bit offset to a scalar base:
  // 8 registers and 8 additions a step, in a loop that is short of both.
  auto fresh_offsets = [&]() __attribute__((always_inline)) {
    asm volatile("" : "+v"(k_off), "+v"(v_off));
    if constexpr (MODE == kAffine) asm volatile("" : "+v"(km_off), "+v"(vm_off));
  };
  auto load_k = [&](const gptr_t (&bp)[2]) __attribute__((always_inline)) {
#pragma unroll
    for (int kt = 0; kt < 2; kt++) {
      if constexpr (MODE == kAffine) {
        if constexpr (BITS == 8) {
          const u32x4 w = load_at<u32x4>(bp[kt], k_off);
#pragma unroll
          for (int i = 0; i < 4; i++) kr[kt][i] = w[i];
        } else {
          const u32x2 w = load_at<u32x2>(bp[kt], k_off);
          kr[kt][0] = w[0];
          kr[kt][1] = w[1];
        }
        km[kt] = load_at<u32x4>(bp[kt], km_off);
      } else if constexpr (MODE == kCodebook) {
#pragma unroll
        for (int s = 0; s < 2; s++) {
          if constexpr (CB == 3) {
            const u32x2 w = load_at<u32x2_a4>(bp[kt], k_off, s * 4 * CB);
            kr[kt][2 * s] = w[0];
            kr[kt][2 * s + 1] = w[1];
          } else {
            kr[kt][s] = load_at<uint32_t>(bp[kt], k_off, s * 4 * CB);
          }
        }
      } else {
#pragma unroll
        for (int s = 0; s < 2; s++) {
          const u32x4 w = load_at<u32x4>(bp[kt], k_off, s * 64);
#pragma unroll
          for (int i = 0; i < 4; i++) kr[kt][4 * s + i] = w[i];
        }
      }
    }
  };
  auto load_v = [&](const gptr_t (&bp)[2]) __attribute__((always_inline)) {
#pragma unroll
    for (int kt = 0; kt < 2; kt++) {
      if constexpr (MODE == kAffine) {
        if constexpr (BITS == 8) {
          const u32x4 w = load_at<u32x4>(bp[kt], v_off);
#pragma unroll
          for (int i = 0; i < 4; i++) vr[kt][i] = w[i];
        } else {
          const u32x2 w = load_at<u32x2>(bp[kt], v_off);
          vr[kt][0] = w[0];
          vr[kt][1] = w[1];
        }
        vm[kt] = load_at<u32x4>(bp[kt], vm_off);
      } else {
#pragma unroll
        for (int n = 0; n < 4; n++) {
          if constexpr (MODE == kCodebook && CB != 3) {
            vr[kt][n] = load_at<uint32_t>(bp[kt], v_off, n * 32 * CB);
          } else {
            const u32x2 w =
                MODE == kCodebook ? (u32x2)load_at<u32x2_a4>(bp[kt], v_off, n * 32 * CB)
                                  : load_at<u32x2>(bp[kt], v_off, n * 16 * kBlockTokens * 2);
            vr[kt][2 * n] = w[0];
            vr[kt][2 * n + 1] = w[1];
          }
        }
      }
    }
  };
  // codebook: the key norms of a step's softmax stage (K and V), the lane's
  // own quads
  u32x2 kn[NQ], vn[NQ];
  const int quad0 = kOwn ? j : lane >> 3;  // the lane's first key quad (then quad0 + 4)
  auto load_n = [&](const gptr_t (&bp)[2]) __attribute__((always_inline)) {
    if constexpr (MODE == kCodebook) {
#pragma unroll
      for (int u = 0; u < NQ; u++) {
        const gptr_t p = (kOwn ? u == 0 : quad0 < 4) ? bp[0] : bp[1];
        kn[u] = load_at<u32x2>(p, (uint32_t)L.k_meta + 8 * (quad0 & 3));
        vn[u] = load_at<u32x2>(p, (uint32_t)L.v_meta + 8 * (quad0 & 3));
      }
    }
  };

  // ---- the n steps from s_begin on ----
  // (with several ranges, this one's share; possibly none)
  const int per = ranges > 1 ? (nst + ranges - 1) / ranges : nst;
  const int s_begin = range * per < nst ? range * per : nst;
  // (a range that is left with none, and a sequence without keys: one step, all masked)
  const int n = nst - s_begin < per ? (nst > s_begin ? nst - s_begin : 1) : per > 0 ? per : 1;
  gptr_t cur[2], nxt[2], after[2];  // the blocks of steps i, i + 1, i + 2
  bool f_cur = false, f_nxt = false, f_after = false;
  // the blocks of step s_begin + i (past the end: of the last one)
  auto blocks_of = [&](int i, gptr_t (&bp)[2], bool& f) __attribute__((always_inline)) {
    if (i >= n) i = n - 1;
    const int v = 2 * (s_begin + i);
    bp[0] = blk_ptr(v);
    bp[1] = blk_ptr(v + 1);
    f = blk_full(v) && blk_full(v + 1);
  };
  // ---- q_rot of the 64 rows: rows wave + NW k, high / residual halves
  // (plain: the raw bf16 rows) ----
  _Float16* const qhi = reinterpret_cast<_Float16*>(region);
  _Float16* const qlo = qhi + kPfRows * QS;
  float* const qsum = reinterpret_cast<float*>(qlo + kPfRows * QS);  // [row][NG] (affine)
  if (tid == 0) not_finite = 0;
  const uint32_t sbits = lane_sign_bits<D>(a.sign_bits, lane);
  const float cs_lane = fwht_lane_sign(lane) * a.c;
  const int rows = nq * G;  // of the chunk
  // Two rows at a time, the next two on their way meanwhile. (One at a time,
  // the loads' latency made a 107-token chunk of head_dim 128, 32 rows a wave,
  // twice as slow; eight unrolled take longer to fetch than to run.)
  uint32_t raw[2][E / 2], ahead[2][E / 2];
  auto load_q = [&](int k0) __attribute__((always_inline)) {
#pragma unroll
    for (int k = 0; k < 2; k++) {
      const int rr = wave + NW * (k0 + k), r = rr < rows ? rr : rows - 1, rq = pos_of(r);
      const int64_t row = ((int64_t)seq * a.n_q + qi0 + rq) * a.n_q_heads + (int64_t)kvh * G + (r - rq * G);
      load_words<E / 2>(a.q + row * D + lane * E, ahead[k]);
    }
  };
  auto zero_rows = [&](int k0) __attribute__((always_inline)) {  // the wave's from its k0th on
    for (int r = wave + NW * k0; r < kPfRows; r += NW) {
      const _Float16 z[E] = {};
      store_halves<E>(reinterpret_cast<uint8_t*>(qhi + r * QS + lane * E), z);
      if constexpr (MODE != kPlain)
        store_halves<E>(reinterpret_cast<uint8_t*>(qlo + r * QS + lane * E), z);
      if constexpr (MODE == kAffine)
        if ((lane & (LPG - 1)) == 0) qsum[r * NG + ((lane * E) >> 6)] = 0.0f;
    }
  };
  load_q(0);
  // the first step's codes come in while the query rows are rotated (V's for
  // the second time where they are used, but no more from memory)
  blocks_of(0, cur, f_cur);
  load_k(cur);
  load_n(cur);
#pragma unroll 1
  for (int k0 = 0; k0 < kPfRows / NW; k0 += 2) {
    if (wave + NW * k0 >= rows) {  // the rest is past the chunk: zeros
      zero_rows(k0);
      break;
    }
#pragma unroll
    for (int k = 0; k < 2; k++)
#pragma unroll
      for (int i = 0; i < E / 2; i++) raw[k][i] = ahead[k][i];
    load_q(k0 + 2);  // (past the wave's last: a row of the chunk again)
#pragma unroll
    for (int k = 0; k < 2; k++) {
      const int r = wave + NW * (k0 + k);
      if constexpr (MODE == kPlain) {
        uint32_t* dst = reinterpret_cast<uint32_t*>(qhi + r * QS + lane * E);
#pragma unroll
        for (int i = 0; i < E / 2; i++) dst[i] = raw[k][i];
        continue;
      }
      float x[E];
#pragma unroll
      for (int i = 0; i < E / 2; i++) {
        x[2 * i] = __uint_as_float(raw[k][i] << 16) * a.qscale;
        x[2 * i + 1] = __uint_as_float(raw[k][i] & 0xffff0000u) * a.qscale;
      }
      // the sign-tracking FWHT: a -0 for +0 changes no score or sum
      wave_fwht_signed<E>(x, lane);
      float gs = 0.0f;
      _Float16 hv[E], lv[E];
#pragma unroll
      for (int i = 0; i < E; i++) {
        const float v = apply_sign(x[i] * cs_lane, sbits, i);
        gs += v;
        hv[i] = (_Float16)v;
        lv[i] = (_Float16)(v - (float)hv[i]);
      }
      gs = group_sum<LPG>(gs, lane);
      store_halves<E>(reinterpret_cast<uint8_t*>(qhi + r * QS + lane * E), hv);
      store_halves<E>(reinterpret_cast<uint8_t*>(qlo + r * QS + lane * E), lv);
      if constexpr (MODE == kAffine)
        if ((lane & (LPG - 1)) == 0) qsum[r * NG + ((lane * E) >> 6)] = gs;
    }
  }
  __syncthreads();

  // this wave's B operands: its 64 dims of every row tile; the lane (j, c)
  // holds 8 consecutive dims of row 16 rt + c at the K-code placement
  // (codebook and plain: slice s, dims 64 wave + 32 s + 8 j ..; plain B
  // operands are the bf16 bits)
  half8_t bqh[PT][2], bql[PT][2];
  float qs[PT];
#pragma unroll
  for (int rt = 0; rt < PT; rt++) {
    const int row = (rt0 + rt) * 16 + c;
#pragma unroll
    for (int s = 0; s < 2; s++) {
      const int d0 = dg * 64 + (MODE == kAffine && BITS == 8 ? j * 16 + s * 8 : s * 32 + j * 8);
      bqh[rt][s] = *reinterpret_cast<const half8_t*>(qhi + row * QS + d0);
      if constexpr (MODE != kPlain) bql[rt][s] = *reinterpret_cast<const half8_t*>(qlo + row * QS + d0);
    }
    qs[rt] = MODE == kAffine ? qsum[row * NG + dg] : 0.0f;
  }
  __syncthreads();  // the table is consumed: the region becomes the buffers
  uint8_t* const lut = region + P::kLutOff;
  const uint32_t lut_l = lds_addr(lut) + (lane & (kLutCopies - 1)) * 4;
  if constexpr (MODE == kCodebook) {
    cb_fill_lut<CB>(lut, tid, NW * 64);
    __syncthreads();
  }

  // ---- the three stages ----
  float4_t o[PT][4];  // [row tile][dim tile]: dims 16 ct + 4 j .., row 16 rt + c
  float bacc[PT];
#pragma unroll
  for (int rt = 0; rt < PT; rt++) {
    bacc[rt] = 0.0f;
#pragma unroll
    for (int ct = 0; ct < 4; ct++) o[rt][ct] = (float4_t){0.f, 0.f, 0.f, 0.f};
  }
  float m_run[NRS], l_run[NRS];
#pragma unroll
  for (int u = 0; u < NRS; u++) m_run[u] = -1e30f, l_run[u] = 0.0f;
  float4_t own[NRS][2];  // this wave's partial of the rows it sums (kOwn)
  // row of softmax row set u
  auto sm_row = [&](int u) __attribute__((always_inline)) { return kOwn ? (wave * NRS + u) * 16 + c : wave * 8 + (lane & 7); };

  // a row's position (past the chunk: the last one, which sees nothing that
  // no row does)
  auto pos_at = [&](int r) __attribute__((always_inline)) {
    const int rq = pos_of(r);
    return pA_r + (rq < nq ? rq : nq - 1);
  };
  int p_row[NRS];
#pragma unroll
  for (int u = 0; u < NRS; u++) p_row[u] = pos_at(sm_row(u));

  float4_t* const xs = reinterpret_cast<float4_t*>(region);
  u32x4* const pb = reinterpret_cast<u32x4*>(region + P::kPbOff);
  float* const al = reinterpret_cast<float*>(region + P::kAlOff);

  auto qk = [&](int buf) __attribute__((always_inline)) {
    float4_t* const xb = xs + buf * (P::kXs / 16) + lane;
#pragma unroll
    for (int kt = 0; kt < 2; kt++) {
      float4_t acc[PT];
#pragma unroll
      for (int rt = 0; rt < PT; rt++) acc[rt] = (float4_t){0.f, 0.f, 0.f, 0.f};
      if constexpr (MODE == kPlain) {
#pragma unroll
        for (int s = 0; s < 2; s++) {
          const bf16x8_t ak = __builtin_bit_cast(
              bf16x8_t, (u32x4){kr[kt][4 * s], kr[kt][4 * s + 1], kr[kt][4 * s + 2], kr[kt][4 * s + 3]});
#pragma unroll
          for (int rt = 0; rt < PT; rt++)
            acc[rt] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(
                ak, __builtin_bit_cast(bf16x8_t, bqh[rt][s]), acc[rt], 0, 0, 0);
        }
      } else {
        half8_t ah[2], alo[2];
#pragma unroll
        for (int s = 0; s < 2; s++) {
          if constexpr (MODE == kAffine) {
            ah[s] = k_operand_plain<BITS>(kr[kt], s);
          } else {
            uint32_t f;
            if constexpr (CB == 3)
              f = __builtin_amdgcn_alignbit(kr[kt][2 * s + 1], kr[kt][2 * s], ksh);
            else
              f = kr[kt][s] >> ksh;
            if constexpr (kCbExact<CB>) {
              ah[s] = __builtin_bit_cast(
                  half8_t, (u32x4){cb_pair_exact<CB, 0>(lut_l, f), cb_pair_exact<CB, 1>(lut_l, f),
                                   cb_pair_exact<CB, 2>(lut_l, f), cb_pair_exact<CB, 3>(lut_l, f)});
            } else {
              uint32_t h4[4], l4[4];
              cb_pair_hl4<0>(lut_l, f, h4[0], l4[0]);
              cb_pair_hl4<1>(lut_l, f, h4[1], l4[1]);
              cb_pair_hl4<2>(lut_l, f, h4[2], l4[2]);
              cb_pair_hl4<3>(lut_l, f, h4[3], l4[3]);
              ah[s] = __builtin_bit_cast(half8_t, (u32x4){h4[0], h4[1], h4[2], h4[3]});
              alo[s] = __builtin_bit_cast(half8_t, (u32x4){l4[0], l4[1], l4[2], l4[3]});
            }
          }
        }
        // the residual products first, then the high parts, in one accumulator
#pragma unroll
        for (int s = 0; s < 2; s++)
#pragma unroll
          for (int rt = 0; rt < PT; rt++)
            acc[rt] = __builtin_amdgcn_mfma_f32_16x16x32_f16(ah[s], bql[rt][s], acc[rt], 0, 0, 0);
        if constexpr (MODE == kCodebook && !kCbExact<CB>) {
#pragma unroll
          for (int s = 0; s < 2; s++)
#pragma unroll
            for (int rt = 0; rt < PT; rt++)
              acc[rt] = __builtin_amdgcn_mfma_f32_16x16x32_f16(alo[s], bqh[rt][s], acc[rt], 0, 0, 0);
        }
#pragma unroll
        for (int s = 0; s < 2; s++)
#pragma unroll
          for (int rt = 0; rt < PT; rt++)
            acc[rt] = __builtin_amdgcn_mfma_f32_16x16x32_f16(ah[s], bqh[rt][s], acc[rt], 0, 0, 0);
      }
#pragma unroll
      for (int rt = 0; rt < PT; rt++) {
        float4_t sv = acc[rt];
        if constexpr (MODE == kAffine) {
#pragma unroll
          for (int i = 0; i < 4; i++)
            sv[i] = fmaf(lo16(km[kt][i]), acc[rt][i], hi16(km[kt][i]) * qs[rt]);
        }
        if constexpr (kOwn) {
          const int owner = rt / NRS;  // the wave that sums this row tile
          if (owner == wave)
            own[rt % NRS][kt] = sv;
          else
            xb[((rt * P::kSrc + (wave < owner ? wave : wave - 1)) * 2 + kt) * 64] = sv;
        } else {
          xb[((dg * 2 + kt) * kPfTiles + rt0 + rt) * 64] = sv;
        }
      }
    }
  };

  auto softmax = [&](int buf, int step, const float4_t (&mine)[NRS][2], bool full) __attribute__((always_inline)) {
#pragma unroll
    for (int u = 0; u < NRS; u++) {
      const int row = sm_row(u);
      float s[NQ][4];
      if constexpr (kOwn) {
        const float4_t* xr = xs + buf * (P::kXs / 16) + (wave * NRS + u) * P::kSrc * 128 + lane;
#pragma unroll
        for (int t = 0; t < NQ; t++) {
          float4_t v = mine[u][t];
#pragma unroll
          for (int g = 0; g < P::kSrc; g++) v += xr[(g * 2 + t) * 64];
#pragma unroll
          for (int i = 0; i < 4; i++) s[t][i] = v[i];
        }
      } else {
        const float4_t* xr = xs + buf * (P::kXs / 16) +
                             ((quad0 >> 2) * kPfTiles + (wave >> 1)) * 64 + (quad0 & 3) * 16 +
                             (wave & 1) * 8 + (lane & 7);
        float4_t v = xr[0];
#pragma unroll
        for (int g = 1; g < NG; g++) v += xr[g * 2 * kPfTiles * 64];
#pragma unroll
        for (int i = 0; i < 4; i++) s[0][i] = v[i];
      }
      // codebook: the keys' norms / sqrt(D); plain: the softmax scale
      float vscale[NQ][4];
      if constexpr (MODE == kCodebook) {
        // (1 / sqrt(D) in the table operands' units)
        const float cu = a.c * kCbOperandScale<CB>;
#pragma unroll
        for (int t = 0; t < NQ; t++) {
          const float ks[4] = {lo16(kn[t][0]), hi16(kn[t][0]), lo16(kn[t][1]), hi16(kn[t][1])};
          const float vs[4] = {lo16(vn[t][0]), hi16(vn[t][0]), lo16(vn[t][1]), hi16(vn[t][1])};
#pragma unroll
          for (int i = 0; i < 4; i++) {
            s[t][i] = s[t][i] * (ks[i] * cu);
            vscale[t][i] = vs[i] * (cu * kPvScale<CB>);
          }
        }
      } else if constexpr (MODE == kPlain) {
#pragma unroll
        for (int t = 0; t < NQ; t++)
#pragma unroll
          for (int i = 0; i < 4; i++) s[t][i] = s[t][i] * a.qscale;
      }
      if (!full) {
        const int p = p_row[u], lo = lo_rel(p);
#pragma unroll
        for (int t = 0; t < NQ; t++) {
          const int vi = 2 * step + (kOwn ? t : quad0 >> 2);
          int vlo, vhi;
          vb_range(vi, vlo, vhi);
          vlo = vlo > lo ? vlo : lo;
          vhi = vhi < p + 1 ? vhi : p + 1;
          const int kp = (vi < n_old_i ? vi : vi + vb_shift) * kBlockTokens + 4 * (quad0 & 3);
#pragma unroll
          for (int i = 0; i < 4; i++)
            if (!(kp + i >= vlo && kp + i < vhi)) {
              s[t][i] = -INFINITY;
              if constexpr (MODE == kCodebook) vscale[t][i] = 0.0f;  // (a norm may be infinite)
            }
        }
      }
      float mb = -INFINITY;
#pragma unroll
      for (int t = 0; t < NQ; t++)
        mb = fmaxf(mb, fmaxf(fmaxf(s[t][0], s[t][1]), fmaxf(s[t][2], s[t][3])));
      if constexpr (!kOwn) mb = fmaxf(mb, row_ror8(mb));
      mb = xor16_max(mb);
      mb = xor32_max(mb);
      const float m_new = fmaxf(m_run[u], mb);
      const float m_old = m_run[u];
      m_run[u] = __any(m_new > m_old + kPfSlack) ? m_new : m_old;
      const float alpha = __builtin_amdgcn_exp2f(m_old - m_run[u]);  // 1 when it stays
      l_run[u] *= alpha;
      if (kOwn ? j == 0 : lane < 8) al[buf * kPfRows + (row & 15) * 4 + (row >> 4)] = alpha;
#pragma unroll
      for (int t = 0; t < NQ; t++) {
        float p[4];
#pragma unroll
        for (int i = 0; i < 4; i++) p[i] = __builtin_amdgcn_exp2f(s[t][i] - m_run[u]);
        l_run[u] += (p[0] + p[1]) + (p[2] + p[3]);
        asm volatile("" : "+v"(l_run[u]));
        u32x4 w;
        if constexpr (MODE != kPlain) {
          // f16 high part and residual of P (affine) or of P' = p * norm /
          // sqrt D (codebook)
          half4_t h, r;
          float rest[4];
#pragma unroll
          for (int i = 0; i < 4; i++) {
            float x = MODE == kCodebook ? p[i] * vscale[t][i] : p[i];
            // (one rounded product for both parts: fused into either conversion
            // it can round the high part to its other neighbour)
            asm("" : "+v"(x));
            // (4 bits: norm / sqrt(D) has no bound. At most 65504 and a residual
            // of as much, cut: infinite parts would meet as NaN. What is
            // infinite or NaN before stays so, in the residual.)
            if constexpr (MODE == kCodebook && !kCbExact<CB>) {
              h[i] = (_Float16)fminf(x, 65504.0f);
              rest[i] = x - (float)h[i];
            } else {
              h[i] = (_Float16)x;
              r[i] = (_Float16)(x - (float)h[i]);
            }
          }
          if constexpr (MODE == kCodebook && !kCbExact<CB>)
            r = cat4(pkrtz(rest[0], rest[1]), pkrtz(rest[2], rest[3]));
          const uint2 hw = __builtin_bit_cast(uint2, h), rw = __builtin_bit_cast(uint2, r);
          w = (u32x4){hw.x, hw.y, rw.x, rw.y};
        } else {
          // P as bf16 high part and residual
          float r[4];
#pragma unroll
          for (int i = 0; i < 4; i++) r[i] = p[i] - bf16_to_f32(f32_to_bf16(p[i]));
          w = (u32x4){pack_bf16x2(p[0], p[1]), pack_bf16x2(p[2], p[3]), pack_bf16x2(r[0], r[1]),
                      pack_bf16x2(r[2], r[3])};
        }
        pb[buf * (P::kPb / 16) + (quad0 + 4 * t) * kPfRows + row] = w;
      }
    }
  };

  auto rescale = [&](int buf) __attribute__((always_inline)) {
    typedef float av_t __attribute__((ext_vector_type(PT)));  // (one load)
    const av_t av = *reinterpret_cast<const av_t*>(al + buf * kPfRows + c * 4 + rt0);
    bool moved = false;
#pragma unroll
    for (int rt = 0; rt < PT; rt++) moved = moved || av[rt] != 1.0f;
    if (__any(moved)) {
#pragma unroll
      for (int rt = 0; rt < PT; rt++) {
#pragma unroll
        for (int ct = 0; ct < 4; ct++) o[rt][ct] *= av[rt];
        bacc[rt] *= av[rt];
      }
    }
  };
  auto pv = [&](int buf, auto hide) __attribute__((always_inline)) {
    half2_t vsc[4], vbi[4];  // affine: scales and biases of the lane's key pairs
    if constexpr (MODE == kAffine) {
#pragma unroll
      for (int e = 0; e < 4; e++) {
        const uint32_t m0 = vm[e >> 1][(e & 1) * 2], m1 = vm[e >> 1][(e & 1) * 2 + 1];
        vsc[e] = __builtin_bit_cast(half2_t, __builtin_amdgcn_perm(m1, m0, 0x05040100u));
        vbi[e] = __builtin_bit_cast(half2_t, __builtin_amdgcn_perm(m1, m0, 0x07060302u));
      }
    }
    // V operands of the four dim tiles (codebook 4 bits: high parts and residuals)
    half8_t va[4], vl[4];
#pragma unroll
    for (int ct = 0; ct < 4; ct++) {
      if constexpr (MODE == kAffine) {
        va[ct] = v_operand_plain<BITS>(vr[0], vr[1], ct);
      } else if constexpr (MODE == kPlain) {
        va[ct] = __builtin_bit_cast(
            half8_t, (u32x4){vr[0][2 * ct], vr[0][2 * ct + 1], vr[1][2 * ct], vr[1][2 * ct + 1]});
      } else {
        uint32_t f[2], h[4], l[4];
#pragma unroll
        for (int kt = 0; kt < 2; kt++) {
          if constexpr (CB == 3)
            f[kt] = __builtin_amdgcn_alignbit(vr[kt][2 * ct + 1], vr[kt][2 * ct], vsh);
          else
            f[kt] = vr[kt][ct] >> vsh;
          if constexpr (kCbExact<CB>) {
            h[2 * kt] = cb_pair_exact<CB, 0>(lut_l, f[kt]);
            h[2 * kt + 1] = cb_pair_exact<CB, 1>(lut_l, f[kt]);
          } else {
            cb_pair_hl4<0>(lut_l, f[kt], h[2 * kt], l[2 * kt]);
            cb_pair_hl4<1>(lut_l, f[kt], h[2 * kt + 1], l[2 * kt + 1]);
          }
        }
        va[ct] = __builtin_bit_cast(half8_t, (u32x4){h[0], h[1], h[2], h[3]});
        if constexpr (!kCbExact<CB>)
          vl[ct] = __builtin_bit_cast(half8_t, (u32x4){l[0], l[1], l[2], l[3]});
      }
    }
#pragma unroll
    for (int rt = 0; rt < PT; rt++) {
      const u32x4 w0 = pb[buf * (P::kPb / 16) + j * kPfRows + (rt0 + rt) * 16 + c];
      const u32x4 w1 = pb[buf * (P::kPb / 16) + (j + 4) * kPfRows + (rt0 + rt) * 16 + c];
      half8_t bh, bl;
      if constexpr (MODE == kAffine) {
        // P' = p * v_scale in packed f16: the high part P_hi * s rounded, then
        // what that left out plus P_lo * s, rounded in turn (its grid ends at
        // 2^-24). HIDE: from 32 bits, toward zero, so that a scale beyond the
        // documented ones ends in 65504 and a residual of as much at most.
#pragma unroll
        for (int e = 0; e < 4; e++) {
          const half2_t ph = __builtin_bit_cast(half2_t, e < 2 ? w0[e] : w1[e - 2]);
          const half2_t pl = __builtin_bit_cast(half2_t, e < 2 ? w0[e + 2] : w1[e]);
          half2_t h = ph * vsc[e];
          half2_t l = __builtin_elementwise_fma(
              pl, vsc[e], __builtin_elementwise_fma(ph, vsc[e], -h));
          if constexpr (decltype(hide)::value) {
            const float x0 = ((float)ph[0] + (float)pl[0]) * (float)vsc[e][0];
            const float x1 = ((float)ph[1] + (float)pl[1]) * (float)vsc[e][1];
            h = pkrtz(x0, x1);
            l = pkrtz(x0 - (float)h[0], x1 - (float)h[1]);
          }
          bh[2 * e] = h[0];
          bh[2 * e + 1] = h[1];
          bl[2 * e] = l[0];
          bl[2 * e + 1] = l[1];
          bacc[rt] = __builtin_amdgcn_fdot2(pl, vbi[e], bacc[rt], false);
          bacc[rt] = __builtin_amdgcn_fdot2(ph, vbi[e], bacc[rt], false);
        }
        // (here, not sunk past the barrier with every weight and bias kept for it)
        asm volatile("" : "+v"(bacc[rt]));
      } else {
        bh = __builtin_bit_cast(half8_t, (u32x4){w0[0], w0[1], w1[0], w1[1]});
        bl = __builtin_bit_cast(half8_t, (u32x4){w0[2], w0[3], w1[2], w1[3]});
      }
#pragma unroll
      for (int ct = 0; ct < 4; ct++) {
        if constexpr (MODE == kPlain) {
          const bf16x8_t v = __builtin_bit_cast(bf16x8_t, va[ct]);
          o[rt][ct] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(v, __builtin_bit_cast(bf16x8_t, bh),
                                                              o[rt][ct], 0, 0, 0);
          o[rt][ct] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(v, __builtin_bit_cast(bf16x8_t, bl),
                                                              o[rt][ct], 0, 0, 0);
        } else {
          o[rt][ct] = __builtin_amdgcn_mfma_f32_16x16x32_f16(va[ct], bh, o[rt][ct], 0, 0, 0);
          if constexpr (MODE == kCodebook && !kCbExact<CB>)
            o[rt][ct] = __builtin_amdgcn_mfma_f32_16x16x32_f16(vl[ct], bh, o[rt][ct], 0, 0, 0);
          o[rt][ct] = __builtin_amdgcn_mfma_f32_16x16x32_f16(va[ct], bl, o[rt][ct], 0, 0, 0);
        }
      }
    }
  };

  // V values (affine: scales and biases) that are not finite, in a step whose
  // keys some rows do not see: a hidden key's weight 0 makes NaN of them. They
  // become 0, and infinite (or NaN) the accumulators of the rows that do see
  // them. (In arithmetic without compares: their masks would crowd the scalar
  // registers of the whole kernel, and the loop ran up to 10% slower.)
  auto hide_not_finite = [&](int step) __attribute__((always_inline)) {
    // 1 in each half of w that is not finite: its exponent is all ones
    auto bad_of = [&](uint32_t w) __attribute__((always_inline)) -> uint32_t {
      constexpr uint32_t kExp = MODE == kPlain ? 0x7f807f80u : 0x7c007c00u;
      constexpr uint32_t kOne = MODE == kPlain ? 0x00800080u : 0x04000400u;
      return ((w & kExp) + kOne) >> 15 & 0x00010001u;
    };
    // 1 for the keys 4 j + i of block kt that row 16 (rt0 + rt) + c sees, else 0
    auto seen_of = [&](int rt, int kt, int i) __attribute__((always_inline)) -> uint32_t {
      const int p = pos_at((rt0 + rt) * 16 + c), lo = lo_rel(p), vi = 2 * step + kt;
      int vlo, vhi;
      vb_range(vi, vlo, vhi);
      vlo = vlo > lo ? vlo : lo;
      vhi = vhi < p + 1 ? vhi : p + 1;
      const int kp = (vi < n_old_i ? vi : vi + vb_shift) * kBlockTokens + 4 * j + i;
      return ~(uint32_t)((kp - vlo) | (vhi - 1 - kp)) >> 31;
    };
    auto poison = [](float x, float n) __attribute__((always_inline)) -> float {  // n = 0: x
      return fmaf(n * 0x1p127f, 0x1p127f, x);
    };
    if constexpr (MODE == kPlain) {
#pragma unroll
      for (int rt = 0; rt < PT; rt++) {
        // how many of them a row sees, per dim: a product of ones
        u32x4 seen;
#pragma unroll
        for (int e = 0; e < 4; e++)
          seen[e] = seen_of(rt, e >> 1, (e & 1) * 2) * 0x3f80u |
                    seen_of(rt, e >> 1, (e & 1) * 2 + 1) * 0x3f800000u;
#pragma unroll
        for (int ct = 0; ct < 4; ct++) {
          u32x4 bad;
#pragma unroll
          for (int e = 0; e < 4; e++) bad[e] = bad_of(vr[e >> 1][2 * ct + (e & 1)]) * 0x3f80u;
          const float4_t n = __builtin_amdgcn_mfma_f32_16x16x32_bf16(
              __builtin_bit_cast(bf16x8_t, bad), __builtin_bit_cast(bf16x8_t, seen),
              (float4_t){0.f, 0.f, 0.f, 0.f}, 0, 0, 0);
#pragma unroll
          for (int i = 0; i < 4; i++) o[rt][ct][i] = poison(o[rt][ct][i], n[i]);
        }
      }
#pragma unroll
      for (int w = 0; w < VW; w++) {
        vr[0][w] &= ~(bad_of(vr[0][w]) * 0xffffu);
        vr[1][w] &= ~(bad_of(vr[1][w]) * 0xffffu);
      }
    } else if constexpr (MODE == kAffine) {
#pragma unroll
      for (int kt = 0; kt < 2; kt++)
#pragma unroll
        for (int i = 0; i < 4; i++) {
          const uint32_t b = bad_of(vm[kt][i]), bad = (b | b >> 16) & 1u;
          vm[kt][i] &= bad - 1u;
#pragma unroll
          for (int rt = 0; rt < PT; rt++)  // (the lanes' sums join the row at the end)
            bacc[rt] = poison(bacc[rt], (float)(bad & seen_of(rt, kt, i)));
        }
    }
  };

  // ---- the pipeline ----
  float4_t mine[NRS][2];
  auto keep_own = [&]() __attribute__((always_inline)) {
    if constexpr (kOwn) {
#pragma unroll
      for (int u = 0; u < NRS; u++) mine[u][0] = own[u][0], mine[u][1] = own[u][1];
    }
  };
  auto advance = [&](int i) __attribute__((always_inline)) {  // cur = step i, nxt, after
#pragma unroll
    for (int t = 0; t < 2; t++) cur[t] = nxt[t], nxt[t] = after[t];
    f_cur = f_nxt, f_nxt = f_after;
    blocks_of(i + 2, after, f_after);
  };
  blocks_of(1, nxt, f_nxt);
  blocks_of(2, after, f_after);
  // the first interval's PV is of zero weights and codes
#pragma unroll
  for (int kt = 0; kt < 2; kt++) {
#pragma unroll
    for (int w = 0; w < VW; w++) vr[kt][w] = 0;
    vm[kt] = (u32x4){0, 0, 0, 0};
  }
  for (int i = tid; i < P::kPb / 16; i += NW * 64) pb[P::kPb / 16 + i] = (u32x4){0, 0, 0, 0};
  if (tid < kPfRows) al[kPfRows + tid] = 1.0f;
  qk(0);
  keep_own();
  load_k(nxt);
  lds_barrier();
  // an interval between two barriers: QK of step i + 1, softmax of step i, PV of
  // step i - 1; the last one has no QK (a tenth of a call of one or two steps)
#pragma unroll 1
  for (int i = 0; i < n - 1; i++) {
    fresh_offsets();
    rescale((i - 1) & 1);
    qk((i + 1) & 1);
    load_k(after);
    softmax(i & 1, s_begin + i, mine, f_cur);
    keep_own();
    load_n(nxt);
    pv((i - 1) & 1, std::false_type{});
    load_v(cur);
    lds_barrier();
    advance(i + 1);
  }
  rescale((n - 2) & 1);
  softmax((n - 1) & 1, s_begin + n - 1, mine, f_cur);
  if (n > 1) pv((n - 2) & 1, std::false_type{});
  load_v(cur);
  lds_barrier();
  rescale((n - 1) & 1);
  pv((n - 1) & 1, std::false_type{});

  // A sum that is not finite: some V value was not (or some score), and a row
  // that does not see it may have it all the same, as 0 * inf; or a V scale
  // took a weight past f16. The steps again, one stage after the other, with
  // such values kept from those rows and such weights saturated. (Tested here
  // and not where V is read: a test in the steps with hidden keys alone cost
  // 2% of every call.)
  // (Codebook caches: the norms are in the weights, 0 for a hidden key.)
  if constexpr (MODE != kCodebook) {
    float zero = 0.0f;
#pragma unroll
    for (int rt = 0; rt < PT; rt++) {
      if constexpr (MODE == kAffine) zero = fmaf(bacc[rt], 0.0f, zero);
#pragma unroll
      for (int ct = 0; ct < 4; ct++)
#pragma unroll
        for (int i = 0; i < 4; i++) zero = fmaf(o[rt][ct][i], 0.0f, zero);
    }
    if (__any(zero != 0.0f)) not_finite = 1;
  }
  lds_barrier();  // the buffers are free
  if (MODE != kCodebook && not_finite) {
#pragma unroll
    for (int rt = 0; rt < PT; rt++) {
      bacc[rt] = 0.0f;
#pragma unroll
      for (int ct = 0; ct < 4; ct++) o[rt][ct] = (float4_t){0.f, 0.f, 0.f, 0.f};
    }
#pragma unroll
    for (int u = 0; u < NRS; u++) m_run[u] = -1e30f, l_run[u] = 0.0f;
#pragma unroll 1
    for (int i = 0; i < n; i++) {
      blocks_of(i, cur, f_cur);
      load_k(cur);
      load_n(cur);
      load_v(cur);
      qk(0);
      keep_own();
      lds_barrier();
      softmax(0, s_begin + i, mine, f_cur);
      lds_barrier();
      rescale(0);
      if (!f_cur) hide_not_finite(s_begin + i);
      pv(0, std::true_type{});
    }
    lds_barrier();
  }

  // ---- epilogue: normalise, inverse rotation, store ----
#pragma unroll
  for (int u = 0; u < NRS; u++) {
    if constexpr (!kOwn) l_run[u] += row_ror8(l_run[u]);
    l_run[u] = xor16_sum(l_run[u]);
    l_run[u] = xor32_sum(l_run[u]);
    if (kOwn ? j == 0 : lane < 8) lrow[sm_row(u)] = l_run[u], mrow[sm_row(u)] = m_run[u];
  }
  float* const Rr = reinterpret_cast<float*>(region);
#pragma unroll
  for (int rt = 0; rt < PT; rt++) {
    if constexpr (MODE == kAffine) bacc[rt] = xor32_sum(xor16_sum(bacc[rt]));
#pragma unroll
    for (int ct = 0; ct < 4; ct++)
      *reinterpret_cast<float4_t*>(&Rr[((rt0 + rt) * 16 + c) * RS + dg * 64 + ct * 16 + 4 * j]) =
          MODE == kAffine     ? o[rt][ct] + bacc[rt]
          : MODE == kCodebook ? o[rt][ct] * (1.0f / kPvScale<CB>)
                              : o[rt][ct];
  }
  __syncthreads();
  if (ranges > 1) {  // partial rows, as accumulated, with their (m, l)
    const int64_t slot =
        (((int64_t)blockIdx.z * gridDim.y + kvh) * gridDim.x + blockIdx.x) * kPfRows;
#pragma unroll 2
    for (int k = 0; k < kPfRows / NW; k++) {
      const int r = wave + NW * k;
      float* dst = a.part_o + (slot + r) * D + lane * E;
#pragma unroll
      for (int i = 0; i < E; i++) dst[i] = Rr[r * RS + lane * E + i];
    }
    if (tid < kPfRows)
      *reinterpret_cast<float2*>(a.part_ml + (slot + tid) * 2) = make_float2(mrow[tid], lrow[tid]);
    return;
  }
#pragma unroll 1
  for (int k0 = 0; k0 < kPfRows / NW && wave + NW * k0 < rows; k0 += 4) {
    float x[4][E];  // four rows at a time, past the chunk too (not stored)
#pragma unroll
    for (int k = 0; k < 4; k++) {
      const int r = wave + NW * (k0 + k);
#pragma unroll
      for (int i = 0; i < E; i++) x[k][i] = Rr[r * RS + lane * E + i];
      if constexpr (MODE != kPlain) {  // (plain: no rotation, the row as accumulated)
#pragma unroll
        for (int i = 0; i < E; i++) x[k][i] = apply_sign(x[k][i], sbits, i);
        wave_fwht_signed<E>(x[k], lane);
      }
    }
#pragma unroll
    for (int k = 0; k < 4; k++) {
      const int r = wave + NW * (k0 + k);
      const int rq_ = pos_of(r), rh_ = r - rq_ * G;
      if (rq_ >= nq) continue;
      const float l = lrow[r];
#pragma unroll
      for (int i = 0; i < E; i++)
        x[k][i] = l > 0.0f ? (x[k][i] * (MODE == kPlain ? 1.0f : cs_lane)) / l : 0.0f;
      store_out<E>(a, (((int64_t)seq * a.n_q + qi0 + rq_) * a.n_q_heads + (int64_t)kvh * G + rh_) * D +
                          lane * E, x[k]);
    }
  }
}

// Merges the key ranges of a split sequence's rows: a wave per row, lane l
// holding dims E l .., out = sum_k 2^(m_k - M) O_k / sum_k 2^(m_k - M) l_k,
// rotated back. Reads each partial once (bound by that: D * 4 bytes a row and
// range). A work-group takes 16 rows of a tile.
constexpr int kPfMergeRows = 16;
template <int D, bool ROT>
__global__ __launch_bounds__(256) void prefill_merge_kernel(PrefillArgs a, int tiles) {
  constexpr int E = D / 64;
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int seq = blockIdx.z, kvh = blockIdx.y;
  const int tile = blockIdx.x / (kPfRows / kPfMergeRows);
  const int r0 = (blockIdx.x % (kPfRows / kPfMergeRows)) * kPfMergeRows;
  const PrefillUnit un = prefill_unit(a, -1, seq, lane);
  if (un.ranges <= 1) return;
  const int G = a.group, QP = kPfRows / G;
  const int nq = a.n_q - tile * QP < QP ? a.n_q - tile * QP : QP;
  const uint32_t sbits = lane_sign_bits<D>(a.sign_bits, lane);
  const float cs = ROT ? fwht_lane_sign(lane) * a.c : 1.0f;
#pragma unroll 1
  for (int r = r0 + wave; r < r0 + kPfMergeRows; r += 4) {
    const int rq = r / G, rh = r - rq * G;
    if (rq >= nq) break;
    const int64_t step = (int64_t)gridDim.y * tiles * kPfRows;  // rows from range to range
    const int64_t row = (((int64_t)un.first * gridDim.y + kvh) * tiles + tile) * kPfRows + r;
    float M = -1e30f;
    for (int k = lane; k < un.ranges; k += 64) M = fmaxf(M, a.part_ml[(row + k * step) * 2]);
    M = group_max<64>(M, lane);
    float x[E], l = 0.0f;
#pragma unroll
    for (int i = 0; i < E; i++) x[i] = 0.0f;
#pragma unroll 2
    for (int k = 0; k < un.ranges; k++) {
      const float2 ml = *reinterpret_cast<const float2*>(a.part_ml + (row + k * step) * 2);
      const float w = __builtin_amdgcn_exp2f(ml.x - M);
      const float* src = a.part_o + (row + k * step) * D + lane * E;
      l = fmaf(w, ml.y, l);
#pragma unroll
      for (int i = 0; i < E; i++) x[i] = fmaf(w, src[i], x[i]);
    }
    if constexpr (ROT) {
#pragma unroll
      for (int i = 0; i < E; i++) x[i] = apply_sign(x[i], sbits, i);
      wave_fwht_signed<E>(x, lane);
    }
#pragma unroll
    for (int i = 0; i < E; i++) x[i] = l > 0.0f ? (x[i] * cs) / l : 0.0f;
    store_out<E>(a, (((int64_t)seq * a.n_q + tile * QP + rq) * a.n_q_heads + (int64_t)kvh * G + rh) * D +
                        lane * E, x);
  }
}

template <int D, int BITS, int MODE, int RW>
hipError_t launch_rw(const PrefillArgs& a, hipStream_t s) {
  const int qp = kPfRows / a.group;
  const int tiles = (a.n_q + qp - 1) / qp, H = a.new_st.n_kv_heads;
  dim3 grid(tiles, H, a.units > 0 ? a.units : a.n_seqs);
  hipLaunchKernelGGL((prefill_attn_kernel<D, BITS, MODE, RW>), grid, dim3(D * RW), 0, s, a);
  if (a.units > 0) {
    dim3 mgrid(tiles * (kPfRows / kPfMergeRows), H, a.n_seqs);
    hipLaunchKernelGGL((prefill_merge_kernel<D, MODE != kPlain>), mgrid, dim3(256), 0, s, a, tiles);
  }
  return hipGetLastError();
}
template <int D, int BITS, int MODE>
hipError_t launch_t(const PrefillArgs& a, hipStream_t s) {
  if constexpr (D < 512)
    if (a.share_rows) return launch_rw<D, BITS, MODE, 512 / D>(a, s);
  return launch_rw<D, BITS, MODE, 1>(a, s);
}

}  // namespace

namespace {
int64_t prefill_places(int D, bool share_rows, int cus) {
  return (int64_t)cus * (D == 512 ? 1 : D == 256 ? (share_rows ? 1 : 2) : share_rows ? 2 : 3);
}
size_t prefill_part_bytes(int64_t work_groups, int D) {
  return (size_t)(work_groups * kPfRows) * (D + 2) * sizeof(float);
}
}  // namespace

size_t prefill_scratch_bytes(int cus) {
  size_t most = 0;
  for (int D : {128, 256, 512}) {
    const size_t b = prefill_part_bytes(prefill_places(D, false, cus), D);
    if (b > most) most = b;
  }
  return most;
}

// How a call runs. `total` counts its work-groups, one per (tile, KV head,
// sequence); times are us per call with its append, 107 tokens after 50 written
// 107@50.
//
// share_rows: the tile of a small grid at head_dim 128 and 256 goes to eight
// waves instead of two and four. What a wave does once per row (rotations) then
// takes a quarter or half of the time, and a step less, but each code is decoded
// by four or two waves. Of short sequences that wins while every work-group has
// a CU: 107@50, head_dim 128, affine 25 against 46, 256: 31 against 40; 4 x
// 300@200 (160 work-groups), 128: 46 against 74; 800@100 (200), 256, 3-bit
// codebook: 86 against 79, hence half the CUs there. Of long ones, which the key
// ranges spread anyway, only a few rows win: 3@8000, 128: 47 against 52; 300@4000
// of two sequences (80), 128: 92 against 86 (3-bit), 87 against 93 (affine);
// 400@8000 (104), 256: 288 against 201. Head_dim 512 has eight waves in any case.
//
// places: work-groups that run at once. Registers allow two waves a SIMD (four
// where a wave has one row tile): at head_dim 128 unshared that is four
// work-groups a CU, of which three are counted, as the 3-bit codebook's 42 KB
// of LDS allow no more.
//
// min_split: shorter sequences stay one range, and a call without longer ones
// has no merge launch (about 4 us, also where it finds nothing to merge). At
// 107@50 (7 steps), 512: 46 one range, 51 two. Eight waves a work-group at 128
// and 256 need 9 steps that an average row sees: 400@0 (8 of 14), 128: 38 one
// range, 42 two; 8 x 40@276..483 (10 to 16), 128: 53 and 38; and more where
// the grid fills part of the chip: 4 x 300@200 (160 work-groups, 13 of 17),
// 128: 46 one range, 56 three each. From 8 steps on gain 512 (400@0: 66 one, 62
// two), fewer waves (256, 600@10: 75 and 60) and calls with a long bound, where
// the merge is launched anyway (a wide table's 2 x 150@100, 256: 53 and 47).
size_t prefill_plan(PrefillArgs& a, int cus, int64_t max_steps, bool may_split) {
  const int D = a.new_st.layout.head_dim, qp = kPfRows / a.group;
  const int64_t wgs = (int64_t)((a.n_q + qp - 1) / qp) * a.new_st.n_kv_heads;  // per unit
  const int64_t total = wgs * a.n_seqs;
  may_split = may_split && a.n_seqs <= 64;
  const bool few = !may_split || max_steps < kPfFewSteps;
  a.units = 0;
  a.share_rows = D < 512 && total <= (!few ? cus / 4 : D == 128 ? cus : cus / 2);
  const int64_t places = prefill_places(D, a.share_rows, cus);
  const int mean = a.n_q / (2 * kPfKeys);  // steps that a row has less than the last, on average
  a.min_split = D == 512 || (total <= cus && !(few && a.share_rows)) ? 8
                : total <= cus / 4                                   ? 9 + mean
                                                                     : (int)(5 + 16 * total / cus) + mean;
  if (!may_split || max_steps < a.min_split) return 0;
  int64_t units = places / wgs;
  const int64_t most = a.n_seqs * ((max_steps + kPfMinSteps - 1) / kPfMinSteps);
  if (units > most) units = most;
  if (2 * units < 3 * a.n_seqs) return 0;
  a.units = (int)units;
  return prefill_part_bytes(units * wgs, D);
}

hipError_t launch_prefill_attention(const PrefillArgs& a, hipStream_t s) {
  if (a.n_q <= 0) return hipSuccess;
  const BlockLayout& L = a.new_st.layout;
  if (L.mode == kAffine) {
    switch (L.head_dim * 16 + L.bits) {
      case 128 * 16 + 4: return launch_t<128, 4, kAffine>(a, s);
      case 128 * 16 + 8: return launch_t<128, 8, kAffine>(a, s);
      case 256 * 16 + 4: return launch_t<256, 4, kAffine>(a, s);
      case 256 * 16 + 8: return launch_t<256, 8, kAffine>(a, s);
      case 512 * 16 + 4: return launch_t<512, 4, kAffine>(a, s);
      case 512 * 16 + 8: return launch_t<512, 8, kAffine>(a, s);
    }
  } else if (L.mode == kCodebook) {
    switch (L.head_dim * 16 + L.bits) {
      case 128 * 16 + 2: return launch_t<128, 2, kCodebook>(a, s);
      case 128 * 16 + 3: return launch_t<128, 3, kCodebook>(a, s);
      case 128 * 16 + 4: return launch_t<128, 4, kCodebook>(a, s);
      case 256 * 16 + 2: return launch_t<256, 2, kCodebook>(a, s);
      case 256 * 16 + 3: return launch_t<256, 3, kCodebook>(a, s);
      case 256 * 16 + 4: return launch_t<256, 4, kCodebook>(a, s);
      case 512 * 16 + 2: return launch_t<512, 2, kCodebook>(a, s);
      case 512 * 16 + 3: return launch_t<512, 3, kCodebook>(a, s);
      case 512 * 16 + 4: return launch_t<512, 4, kCodebook>(a, s);
    }
  } else if (L.mode == kPlain) {
    switch (L.head_dim) {
      case 128: return launch_t<128, 16, kPlain>(a, s);
      case 256: return launch_t<256, 16, kPlain>(a, s);
      case 512: return launch_t<512, 16, kPlain>(a, s);
    }
  }
  return hipErrorInvalidValue;
}

}  // namespace fmkv
