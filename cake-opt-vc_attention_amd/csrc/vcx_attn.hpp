// The fused attention's device building blocks: tile loads, scores, softmax bytes, PV. See
// vcx_attn.hip for the algorithm and the numerical contract; included by the kernels there
// (blocks that stream every tile) and in vcx_attn_piece.hip (tiles split over waves).
#pragma once
#include "vcx_common.hpp"

#include <type_traits>

namespace vcx {

struct AttnArgs {
  const int8_t* q8;
  const int8_t* k8;
  const uint8_t* v8;
  const float* qs;
  const float* ks;
  const float* vs;
  const uint16_t* means;
  void* out;
  int64_t osb, osh, osn;
  int64_t H, Nq, Nk, tiles, qblocks, qs_len;
  float sm;
  uint8_t* pdump;
  int64_t prow0, prow1;
  // Block list: nfull 128-row blocks, dealt to the 8 XCDs as contiguous ranges; the last kconv
  // blocks of every XCD's range run as two 64-row blocks each, after all its 128-row blocks.
  int64_t nfull, kconv;
  int out_bf16;  // split pieces: the output type (attn_kernel's is a template argument)
};

// vcx_attn_piece.hip
int piece_groups(int64_t BH, int64_t Nq, int64_t tiles, int64_t D, int vm, int mode, int qf);
int launch_pieces(const AttnArgs& a, int64_t BH, int64_t D, int groups, int vm, int mode, int qf, hipStream_t st);

namespace {

typedef int v4i __attribute__((ext_vector_type(4)));
typedef int v8i __attribute__((ext_vector_type(8)));
typedef float v4f __attribute__((ext_vector_type(4)));

constexpr int kThreadsPerBlock = 256;
constexpr int kRowsPerBlock = 128;

// LDS placement of the K and V^T tiles. Both operands are read as lane (G = l/16,
// li = l%16) -> LDS row 16b + li, physical 16-byte chunk X ^ x(li), where X is what the
// lane group needs (QK: 4ds + G; PV: 4h + G) and x(li) = li & 7 for 128-byte rows,
// (li >> 1) & 3 for the 64-byte K rows of D64. On gfx950 this read pattern runs at the
// conflict-free ds_read_b128 rate (4.55 clocks per wave instruction per CU, measured);
// XORs keyed on the key row instead of the reading lane ran 2-way conflicted (8.2).
//  K:   LDS row p holds key 16(p/16) + kr(p%16) (kr: the MFMA row order, whose lane
//       group G gets Sage K-scale group (key%8)/2 == G); chunk q holds channel chunk
//       q ^ x(p).
//  V^T: LDS row = channel; physical chunk q holds token chunk 2(q' & 3) + q'/4 with
//       q' = q ^ (channel & 7), so lane group G finds its chunks 2G, 2G + 1 at 4h + G.
__device__ inline int key_row(int p) {
  const int r = p & 15;
  return (p & ~15) + 8 * ((r & 3) >> 1) + 2 * (r >> 2) + (r & 1);
}
template <int D>
__device__ inline int chunk_xor(int p) { return D == 128 ? (p & 7) : ((p >> 1) & 3); }

typedef __attribute__((address_space(3))) void lds_void;
typedef const __attribute__((address_space(1))) void global_void;

// Direct-to-LDS loads of one key tile. Each of the 4 waves issues D/32
// instructions for K and D/32 for V^T; instruction n of wave w fills the 64
// consecutive 16-byte slots (w*(D/32) + n)*64 + lane. Slot s is LDS row s/(D/16) (K)
// or s/8 (V^T) at physical chunk s%(D/16) or s%8; the source row and chunk follow the
// placement above.
// Lane-constant parts of the addresses are precomputed once per kernel.
// Raw buffer resource over [base, base + bytes): out-of-range lanes read zeros.
__device__ inline __amdgpu_buffer_rsrc_t make_rsrc(const void* base, uint32_t bytes) {
  return __builtin_amdgcn_make_buffer_rsrc(const_cast<void*>(base), 0, static_cast<int>(bytes), 0x00020000);
}

// Value modes: VM 0 = no smoothing (per-channel V scale in the epilogue),
// 1 = block-mean smoothing with per-channel scales, 2 = block-mean smoothing
// with per-block scales (applied to every tile's contribution).
// VM 1 and 2 defer the block-mean restore: the fp16 means of tile t land in slot t % NR of
// an LDS ring, and every kChunk tiles one f16 MFMA per channel block adds
// sum_t mean_t (x) w_t to O (w_t: the row's tile mass, rescaled like O). VM 2 also rings
// the tile's fp32 V scales and feeds RN_f16(vs_t * mean_t) to that MFMA instead.
constexpr int kChunk = 16, kRing = 32;

template <int D, int VM, int QF = 0>
struct TileLoader {
  static constexpr bool SMOOTH = VM >= 1, BSCALE = VM == 2, RING = VM >= 1;
  // Ring slots: the DMA of tile t+1 is in flight while a flush reads tiles t-15..t, so a
  // ring needs kChunk + 1 slots; VM 1 keeps 32 (power of two), VM 2 (which also rings
  // 4*D bytes of V scales per tile) the minimum, to stay within two blocks' LDS per CU.
  static constexpr int NR = BSCALE ? kChunk + 1 : kRing;
  // Slot strides of the rings, padded by 16 bytes: a flush reads slots 4 apart in the four
  // lane groups, and 4 x (2D + 16) = 64 mod 256 puts those reads in four different 64-byte
  // bank windows (unpadded, 4 x 2D is a multiple of 256: four-way bank conflicts).
  static constexpr int RS = 2 * D + 16, VS = 4 * D + 16;
  // Meta region of a buffer: the tile's K scales (INT8: 4 Sage key-group scales, 16 bytes;
  // FP8 block: one scale, 4 bytes), loaded by wave 0 with the means; V scales by wave 1.
  static constexpr int MR = SMOOTH ? (2 * D) / 16 : 0;  // lanes that load the tile's means
  static constexpr int VL = BSCALE ? (4 * D) / 16 : 0;  // lanes that load the tile's V scales
  static constexpr int KS_OFF = 0;
  static constexpr int META_BYTES = 16;
  static constexpr int N = D / 32;  // instructions per wave per operand
  uint32_t koff[N];                 // lane byte offset inside the K tile (row*D + chunk*16)
  uint32_t voff[N];                 // lane byte offset inside the V^T tile columns
  uint32_t moff;                    // lane byte offset of the meta load (wave 0)
  __amdgpu_buffer_rsrc_t rk, rv, rm, rs, rb;
  uint8_t* ring;                    // RING: LDS ring of NR tiles x D fp16 means
  uint8_t* vsring;                  // BSCALE: LDS ring of NR tiles x D fp32 V scales
  int wave;

  __device__ inline void init(const AttnArgs& a, int64_t bh) {
    wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int lane = threadIdx.x & 63;
    const int64_t npad = a.tiles * kTile;
#pragma unroll
    for (int n = 0; n < N; ++n) {
      const int s = (wave * N + n) * 64 + lane;
      const int p = s / (D / 16), phys = s % (D / 16);
      koff[n] = static_cast<uint32_t>(key_row(p) * D + ((phys ^ chunk_xor<D>(p)) * 16));
      const int ch = s >> 3, q = (s & 7) ^ (ch & 7);
      voff[n] = static_cast<uint32_t>(ch * static_cast<int>(npad) + (2 * (q & 3) + (q >> 2)) * 16);
    }
    // Per-head resources. K rows past Nk read zeros (their logits are masked anyway).
    rk = make_rsrc(a.k8 + bh * a.Nk * D, static_cast<uint32_t>(a.Nk * D));
    rv = make_rsrc(a.v8 + bh * D * npad, static_cast<uint32_t>(D * npad));
    if constexpr (QF == 1) rs = make_rsrc(a.ks + bh * a.tiles, static_cast<uint32_t>(a.tiles * 4));
    else rs = make_rsrc(a.ks + bh * a.tiles * 4, static_cast<uint32_t>(a.tiles * 16));
    if constexpr (SMOOTH) rm = make_rsrc(a.means + bh * a.tiles * D, static_cast<uint32_t>(a.tiles * D * 2));
    if constexpr (BSCALE) rb = make_rsrc(a.vs + bh * a.tiles * D, static_cast<uint32_t>(a.tiles * D * 4));
    moff = static_cast<uint32_t>(lane * 16);
  }

  // All addresses are a wave-uniform soffset (the tile) plus lane-constant
  // voffsets: no per-lane address arithmetic in the loop.
  static constexpr int kParts = 2 * N;
  __device__ inline void issue(int64_t t, uint8_t* lk, uint8_t* lv, uint8_t* lm) const {
#pragma unroll
    for (int i = 0; i < kParts; ++i) part(i, t, lk, lv, lm);
  }
  // One instruction's worth of the tile's loads (0 <= i < kParts).
  __device__ __forceinline__ void part(int i, int64_t t, uint8_t* lk, uint8_t* lv, uint8_t* lm) const {
    if (i == 0) meta(t, lm);
    if (i < N)
      __builtin_amdgcn_raw_ptr_buffer_load_lds(rk, (lds_void*)(lk + (wave * N + i) * 1024), 16, koff[i],
                                               static_cast<int>(t * kTile * D), 0, 0);
    else
      __builtin_amdgcn_raw_ptr_buffer_load_lds(rv, (lds_void*)(lv + (wave * N + i - N) * 1024), 16, voff[i - N],
                                               static_cast<int>(t * kTile), 0, 0);
  }
  __device__ __forceinline__ void meta(int64_t t, uint8_t* lm) const {
    const int lane = threadIdx.x & 63;
    if (wave == 0) {
      if constexpr (SMOOTH) {
        uint8_t* dst = ring + (t % NR) * RS;
        if (lane < MR)
          __builtin_amdgcn_raw_ptr_buffer_load_lds(rm, (lds_void*)dst, 16, moff, static_cast<int>(t * D * 2), 0, 0);
      }
      if (lane == 0) {
        if constexpr (QF == 1)
          __builtin_amdgcn_raw_ptr_buffer_load_lds(rs, (lds_void*)(lm + KS_OFF), 4, 0, static_cast<int>(t * 4), 0, 0);
        else
          __builtin_amdgcn_raw_ptr_buffer_load_lds(rs, (lds_void*)(lm + KS_OFF), 16, 0, static_cast<int>(t * 16), 0, 0);
      }
    }
    if constexpr (BSCALE) {
      if (wave == 1 && lane < VL)
        __builtin_amdgcn_raw_ptr_buffer_load_lds(rb, (lds_void*)(vsring + (t % NR) * VS), 16, moff,
                                                 static_cast<int>(t * D * 4), 0, 0);
    }
  }
};

__device__ inline v4f mfma_fp8(const v8i& a, const v8i& b, const v4f& c) {
  return __builtin_amdgcn_mfma_scale_f32_16x16x128_f8f6f4(a, b, c, 0, 0, 0, 0, 0, 0);
}
// Row mass: A = 16 x 128 ones in FP4 E2M1 (0x2 = 1.0; 16 bytes per lane, so the compiler
// keeps four registers instead of eight), B = the E4M3 probabilities. Same 8-pass timing as
// the E4M3 x E4M3 product (measured) and the same sums: every product is exactly P.
__device__ inline v4f mfma_mass(const v4i& ones4, const v8i& b, const v4f& c) {
  const v8i a = {ones4[0], ones4[1], ones4[2], ones4[3], 0, 0, 0, 0};  // upper half unread
  return __builtin_amdgcn_mfma_scale_f32_16x16x128_f8f6f4(a, b, c, 4, 0, 0, 0, 0, 0);
}

// v_max_f32 / v_max3_f32 as single instructions: fmaxf lowers to maxnum, around which the
// compiler inserts NaN-quieting copies of values coming out of the permlane swaps. The
// operands here are finite or -inf.
__device__ inline float vmax(float a, float b) {
  float r;
  asm("v_max_f32 %0, %1, %2" : "=v"(r) : "v"(a), "v"(b));
  return r;
}
__device__ inline float vmax3(float a, float b, float c) {
  float r;
  asm("v_max3_f32 %0, %1, %2, %3" : "=v"(r) : "v"(a), "v"(b), "v"(c));
  return r;
}

// Row reductions over the four lane groups that hold one query row: gfx950
// permlane swaps give each lane the values of lanes l^16 and l^32 without an LDS
// round trip. Every lane of the row ends with the same value (the adds commute).
// running_max returns max(m, row maximum of x).
__device__ inline float running_max(float m, float x) {
  const auto x16 = __builtin_amdgcn_permlane16_swap(__float_as_uint(x), __float_as_uint(x), false, false);
  x = vmax(__uint_as_float(x16[0]), __uint_as_float(x16[1]));
  const auto x32 = __builtin_amdgcn_permlane32_swap(__float_as_uint(x), __float_as_uint(x), false, false);
  return vmax3(m, __uint_as_float(x32[0]), __uint_as_float(x32[1]));
}

// running_max2 gives mn[g] = max(m[g], row maximum of x[g]) for both row groups of a wave
// in one reduction. With the wave's 16-lane rows R0..R3 (lane group G = row RG): the 16-lane
// swap of x[0] against x[1] and a maximum leave (x0 of R0|R1, x1 of R0|R1, x0 of R2|R3,
// x1 of R2|R3) in R0..R3; the 32-lane swap and a maximum complete each group's maximum
// (R0, R2: group 0; R1, R3: group 1); a last 16-lane swap hands every lane both.
__device__ inline void running_max2(const float (&m)[2], const float (&x)[2], float (&mn)[2]) {
  const auto a = __builtin_amdgcn_permlane16_swap(__float_as_uint(x[0]), __float_as_uint(x[1]), false, false);
  const float c = vmax(__uint_as_float(a[0]), __uint_as_float(a[1]));
  const auto b = __builtin_amdgcn_permlane32_swap(__float_as_uint(c), __float_as_uint(c), false, false);
  const float d = vmax(__uint_as_float(b[0]), __uint_as_float(b[1]));
  const auto e = __builtin_amdgcn_permlane16_swap(__float_as_uint(d), __float_as_uint(d), false, false);
  mn[0] = vmax(m[0], __uint_as_float(e[0]));
  mn[1] = vmax(m[1], __uint_as_float(e[1]));
}

// Whether `pred` holds on some active lane (a scalar test of the lane mask).
__device__ inline bool wave_any(bool pred) { return __builtin_amdgcn_ballot_w64(pred) != 0; }

__device__ inline float row_sum(float x) {
  const auto x16 = __builtin_amdgcn_permlane16_swap(__float_as_uint(x), __float_as_uint(x), false, false);
  x = __uint_as_float(x16[0]) + __uint_as_float(x16[1]);
  const auto x32 = __builtin_amdgcn_permlane32_swap(__float_as_uint(x), __float_as_uint(x), false, false);
  return __uint_as_float(x32[0]) + __uint_as_float(x32[1]);
}

// Sage's FP8 offset: the control path's row maximum is lowered by 8.807 so that the
// largest probability is 2^8.807 ~ 448, the E4M3 maximum (sal/csrc/qattn/attn_utils.cuh:30).
constexpr float kFp8Offset = 8.807f;
// The folded path starts its QK accumulators at the bits of 1.5 * 2^23: with |acc| < 2^22
// they read as the float 12582912 + acc, so float(acc) is one exact subtraction.
constexpr int kBias = 0x4B400000;
constexpr float kBiasF = 12582912.0f;

// Mask of the active lanes whose x is a positive normal number: one v_cmp_class_f32 into an
// SGPR pair (the ballot of __builtin_amdgcn_classf adds a select and a compare).
__device__ inline uint64_t pos_normal_lanes(float x) {
  uint64_t r;
  asm("v_cmp_class_f32_e64 %0, %1, %2" : "=s"(r) : "v"(x), "s"(1 << 8));
  return r;
}

// Score of accumulator element r: FP8 scores are floats already; the folded path's
// INT8 accumulators carry the kBias offset.
__device__ inline float acc_value(const v4f& acc, int r) { return acc[r]; }
__device__ inline float acc_value(const v4i& acc, int r) { return __int_as_float(acc[r]) - kBiasF; }

// NQG: 16-row groups per wave (2: a 128-row block of 4 waves; 1: a 64-row block, the
// finer work pieces that end each XCD's list of blocks).
template <int D, int VM, bool DUMP, int PM, int QF = 0, int NQG = 2>
struct Wave {
  static constexpr bool EC = PM != 0;  // ExpCast bytes (1 unfused, 2 folded) or the control path (0)
  // Biased INT8 accumulators (float(acc) = one v_sub_f32): the folded path, the unfused
  // path at D128 with channel-scale smoothing (same-box: smoothing 11.13 -> 11.06 ms, long
  // 43.24 -> 43.00 ms) and the control path at D128 (but its per-block-scale diagnostic
  // variant). D64 (168 VGPRs at three waves per SIMD) and the unfused path with per-block V
  // scales keep v_cvt_f32_i32: the bias register costs them spills.
  static constexpr bool IB = QF == 0 && (PM == 2 || (PM == 1 && D == 128 && VM == 1) ||
                                         (PM == 0 && D == 128 && !(VM == 2 && DUMP)));
  static constexpr int kD = D, kPM = PM;
  // Whether the next tile's loads are spread over the QK steps (see tile) or all issued before
  // them. A D64 tile has half the loads and half the MFMA time: spread, the last load lands too
  // late for a tile without block values, the shortest one. Same box, us, issued first / spread: FP8
  // [1,2,40001,64] 653 / 706, [1,24,16001,64] 1102 / 1169, [1,16,8192,64] unfused 253 / 259, control 328 /
  // 338; INT8 [1,24,16001,64] 932 / 939, [2,16,4097,64] 107.3 / 107.7.
  static constexpr bool kSpread = D == 128 || VM > 0;
  // Control path: whether the copy of the loop without small probabilities pays (see bytes). At
  // D128 with per-block V scales two copies spill (527 scalars and 178 vector registers against
  // 296 and 170 in one): [1,16,8192,128] 1194 us with both, 800 us with the general one.
  static constexpr bool kCheapTest = D == 64 || VM < 2;
  static constexpr int DS = D / 64;  // 64-deep QK steps
  static constexpr int CB = D / 16;  // 16-channel output blocks
  static constexpr bool SMOOTH = VM >= 1, BSCALE = VM == 2;
  typedef TileLoader<D, VM, QF> LD;
  typedef std::conditional_t<QF == 1, v4f, v4i> Acc;  // 16x16 score accumulator

  // The exact float value of one INT8 score accumulator element.
  __device__ static inline float acc_float(int x) {
    if constexpr (IB) return __int_as_float(x) - kBiasF;
    else return static_cast<float>(x);
  }

  // DACC: the row mass accumulates in the C operand of the all-ones MFMA (element 0 is the
  // row's denominator; the history rescale scales only that element, the other three are
  // never read) instead of a zero-started MFMA and one addition per tile: ExpCast without
  // block values at D128 (D64's three waves per SIMD have no registers for it).
  static constexpr bool DACC = EC && VM == 0 && D == 128;
  v4i qf[NQG][DS];
  float qsv[NQG];
  int64_t row[NQG];
  float m[NQG], den[NQG];
  v4f dacc[NQG];
  // Folded encode: fmaf(-m, A, B) of the running maximum, refreshed only when m moves
  float fbias[NQG];
  v4f O[NQG][CB];
  float wts[NQG][4];  // VM 1, 2: pending mean weights of chunk tiles 4G..4G+3 (row li)
  int koff[DS], voff[2];
  v4i ones;  // all-ones FP4 (E2M1) A operand of the row-mass MFMA
  v4i bacc;  // kBias in every element: the initial QK accumulator of the biased paths
  // Folded encode (INT8 QK): the per-tile fold conditions are known to hold on every tile
  // but the last (set once per wave by fold_precheck; wave-uniform)
  int fold_ok;
  int wide;  // control path: the wave has met a vanishing probability
  int G, li;
  int64_t bh_;

  // The folded encode's conditions on a tile before the last (scale = RN(sm * RN(qs * ks))
  // and gain = RN(scale * A) positive normal, |m'| <= 128) hold on every such tile when
  //  - RN(sm * RN(qs * ks)) is a positive normal at the head's smallest and largest K scale
  //    and RN(scale * A) is one at the largest (RN and multiplication by positive factors
  //    are monotone, so every tile's scale and gain lie between these; the K scales are
  //    compared as bit patterns, which orders positive floats and sends zero, negative,
  //    NaN and infinite scales to an end that fails), and
  //  - |logit| <= RN(128 * sum|q8| * scale_hi) <= 128 for the lane's row: every score's
  //    |acc| <= 128 * sum|q8|, so every logit, each tile's maximum and from the first tile on
  //    the running maximum stay within it.
  // fold_ok is the AND over the wave; when it fails the tiles test the conditions.
  __device__ inline void fold_precheck(const AttnArgs& a, int lane) {
    const uint32_t* kb = reinterpret_cast<const uint32_t*>(a.ks) + bh_ * a.tiles * 4;
    uint32_t kmin = 0xffffffffu, kmax = 0u;
    // 16 loads per lane in flight before any is used (one round trip per 1024 scales)
    constexpr int kBatch = 16;
    const int64_t n = a.tiles * 4;
    for (int64_t i0 = lane; i0 < n; i0 += 64 * kBatch) {
      uint32_t u[kBatch];
#pragma unroll
      for (int b = 0; b < kBatch; ++b) u[b] = i0 + 64 * b < n ? kb[i0 + 64 * b] : kb[i0];
      __builtin_amdgcn_sched_barrier(0);  // all loads issued before the first use
#pragma unroll
      for (int b = 0; b < kBatch; ++b) {
        kmin = u[b] < kmin ? u[b] : kmin;
        kmax = u[b] > kmax ? u[b] : kmax;
      }
    }
#pragma unroll
    for (int sh = 32; sh >= 1; sh >>= 1) {
      const uint32_t lo = __shfl_xor(kmin, sh), hi = __shfl_xor(kmax, sh);
      kmin = lo < kmin ? lo : kmin;
      kmax = hi > kmax ? hi : kmax;
    }
    uint64_t ok = __builtin_amdgcn_read_exec();
#pragma unroll
    for (int qg = 0; qg < NQG; ++qg) {
      int asum = 0;
#pragma unroll
      for (int ds = 0; ds < DS; ++ds)
#pragma unroll
        for (int e = 0; e < 4; ++e)
#pragma unroll
          for (int by = 0; by < 4; ++by) {
            const int x = static_cast<int8_t>((static_cast<uint32_t>(qf[qg][ds][e]) >> (8 * by)) & 0xffu);
            asum += x < 0 ? -x : x;
          }
      asum += __shfl_xor(asum, 16);
      asum += __shfl_xor(asum, 32);
      const float s_lo = a.sm * (qsv[qg] * __uint_as_float(kmin));
      const float s_hi = a.sm * (qsv[qg] * __uint_as_float(kmax));
      const float bound = static_cast<float>(128 * asum) * s_hi;
      ok &= pos_normal_lanes(s_lo) & pos_normal_lanes(s_hi) & pos_normal_lanes(s_hi * kExpA) &
            __builtin_amdgcn_ballot_w64(bound <= 128.0f);
    }
    fold_ok = __builtin_amdgcn_readfirstlane(ok == __builtin_amdgcn_read_exec() ? 1 : 0);
  }

  __device__ inline v8i load_v(const uint8_t* lv, int cb) const {
    const v4i lo = *reinterpret_cast<const v4i*>(lv + cb * 16 * kTile + voff[0]);
    const v4i hi = *reinterpret_cast<const v4i*>(lv + cb * 16 * kTile + voff[1]);
    return v8i{lo[0], lo[1], lo[2], lo[3], hi[0], hi[1], hi[2], hi[3]};
  }

  // Phase 1 of a tile for row group qg: the values the encode reads (PM 2 and 0: float(acc),
  // on the last tile float(acc) * dq or -inf past Nk; PM 1: the logits), the logit scale
  // (PM 2) or log2-domain factor (PM 0), and the maximum over this lane's keys.
  template <bool LAST>
  __device__ __forceinline__ float logits(const AttnArgs& a, int64_t t, int qg, const Acc (&Sq)[8], float ksv,
                                          float (&bs)[8][4], float& scl) const {
    float tmo;
    const float dq = qsv[qg] * ksv;
    if constexpr (PM == 2) {
      const float scale = LAST ? a.sm : a.sm * dq;
      scl = scale;
      if constexpr (!LAST && QF == 1) {
        // scale > 0, so RN(max(base) * scale) is the maximum of the rounded logits
        float bm = -INFINITY;
#pragma unroll
        for (int j = 0; j < 8; ++j)
#pragma unroll
          for (int r = 0; r < 4; ++r) {
            bs[j][r] = Sq[j][r];
            bm = fmaxf(bm, bs[j][r]);
          }
        tmo = bm * scale;
      } else if constexpr (!LAST) {
        // float(acc) is exact and monotone: the row maximum is taken on the integers
        int im = Sq[0][0];
#pragma unroll
        for (int j = 0; j < 8; ++j)
#pragma unroll
          for (int r = 0; r < 4; ++r) {
            im = im > Sq[j][r] ? im : Sq[j][r];
            bs[j][r] = __int_as_float(Sq[j][r]) - kBiasF;
          }
        // the biased bits read as 12582912 + max: one exact subtraction gives float(max)
        tmo = (__int_as_float(im) - kBiasF) * scale;
      } else {
        float bm = -INFINITY;
#pragma unroll
        for (int j = 0; j < 8; ++j)
#pragma unroll
          for (int r = 0; r < 4; ++r) {
            const int64_t key = t * kTile + 16 * j + 8 * (r >> 1) + 2 * G + (r & 1);
            const float f = acc_value(Sq[j], r);
            bs[j][r] = key < a.Nk ? f * dq : -INFINITY;
            bm = fmaxf(bm, bs[j][r]);
          }
        tmo = bm * scale;
      }
    } else if constexpr (PM == 1) {
      float tm = -INFINITY;
      if constexpr (!LAST) {
        const float c = a.sm * dq;
#pragma unroll
        for (int j = 0; j < 8; ++j)
#pragma unroll
          for (int r = 0; r < 4; ++r) {
            bs[j][r] = acc_float(Sq[j][r]) * c;
            tm = fmaxf(tm, bs[j][r]);
          }
      } else {
#pragma unroll
        for (int j = 0; j < 8; ++j)
#pragma unroll
          for (int r = 0; r < 4; ++r) {
            const int64_t key = t * kTile + 16 * j + 8 * (r >> 1) + 2 * G + (r & 1);
            float x = (acc_float(Sq[j][r]) * dq) * a.sm;
            bs[j][r] = key < a.Nk ? x : -INFINITY;
            tm = fmaxf(tm, bs[j][r]);
          }
      }
      tmo = tm;
    } else {
      // Sage FP8 control path: log2-domain logits (a.sm carries RN(sm * RN(log2 e))),
      // running maximum with the upstream 8.807 offset, P = E4M3(exp2(.)) and an
      // unrounded mass.
      const float f = LAST ? a.sm : a.sm * dq;
      scl = f;
      float tm;
      if constexpr (!LAST) {
        // f > 0, so fmaf(b, f, -offset) is monotone in b: the maximum is taken on the
        // scores (on the integers for INT8 accumulators), then shifted once
        if constexpr (QF == 0) {
          int im = Sq[0][0];
#pragma unroll
          for (int j = 0; j < 8; ++j)
#pragma unroll
            for (int r = 0; r < 4; ++r) {
              im = im > Sq[j][r] ? im : Sq[j][r];
              bs[j][r] = acc_float(Sq[j][r]);
            }
          tm = __builtin_fmaf(acc_float(im), f, -kFp8Offset);
        } else {
          float bm = -INFINITY;
#pragma unroll
          for (int j = 0; j < 8; ++j)
#pragma unroll
            for (int r = 0; r < 4; ++r) {
              bs[j][r] = Sq[j][r];
              bm = vmax(bm, bs[j][r]);
            }
          tm = __builtin_fmaf(bm, f, -kFp8Offset);
        }
        // f = +inf (an extreme sm_scale) with a zero maximum gives NaN where the maximum of
        // the shifted terms (each -inf or NaN) is -inf
        if (tm != tm) tm = -INFINITY;
      } else {
        tm = -INFINITY;
#pragma unroll
        for (int j = 0; j < 8; ++j)
#pragma unroll
          for (int r = 0; r < 4; ++r) {
            float b;
            if constexpr (QF == 1) b = Sq[j][r];
            else b = acc_float(Sq[j][r]);
            const int64_t key = t * kTile + 16 * j + 8 * (r >> 1) + 2 * G + (r & 1);
            b = key < a.Nk ? b * dq : -INFINITY;
            bs[j][r] = b;
            tm = fmaxf(tm, __builtin_fmaf(b, f, -kFp8Offset));
          }
      }
      tmo = tm;
    }
    return tmo;
  }

  // Rescale the history of row group qg, in which some maximum moved (dm = m - m' on each
  // lane): alpha = exp(dm) (exp2 of the log2-domain difference on the control path) is
  // exactly 1 on the other lanes, and O, den (and the pending mean weights) are scaled before
  // the tile's PV adds in.
  __device__ __forceinline__ void rescale(int qg, float dm) {
    const float alpha = EC ? __builtin_amdgcn_exp2f(dm * 1.44269504088896341f) : __builtin_amdgcn_exp2f(dm);
#pragma unroll
    for (int cb = 0; cb < CB; ++cb) O[qg][cb] *= alpha;
    if constexpr (DACC) dacc[qg][0] *= alpha;
    else den[qg] *= alpha;
    if constexpr (SMOOTH) {
#pragma unroll
      for (int j = 0; j < 4; ++j) wts[qg][j] *= alpha;
    }
  }

  // Control path: whether probabilities of this wave's rows are likely to vanish, by the scales
  // alone: the score (in bits) of a row and a key of the first tile whose entries are all their
  // group's largest. N(0,1) inputs give 19 (D64) to 21, and as much more as Q is scaled by; from about
  // 14 times on some probability of almost every block vanishes in the first tiles, which such a wave
  // would do twice before it leaves the copy with the cheap test (see bytes). Only the copy of the
  // tile loop depends on it, not a result. Same box, us, both neighbours' bytes of every probability /
  // leaving alone / this, Q scaled by 1, 14 and 25: [1,32,2048 x 512,128] 27.7 / 24.9 / 24.9, 25.4 / 27.8 /
  // 25.7, 25.1 / 28.4 / 22.9; [1,32,2048 x 1024,64] 33.2 / 29.4 / 29.7, 32.4 / 31.2 / 30.7, 32.5 / 34.3 / 29.7;
  // [1,16,3000,128] with smoothing 97.2 / 87.4 / 87.5, 92.9 / 95.2 / 90.4, 93.0 / 91.2 / 86.5;
  // [1,28,8192,128] 729 / 661 / 656, 698 / 667 / 655, 697 / 650 / 632.
  __device__ inline bool wide_scores(const AttnArgs& a) const {
    constexpr float kWide = 280.0f, kMax = QF == 1 ? 448.0f : 127.0f, kRootD = D == 128 ? 11.313708f : 8.0f;
    const float ks0 = a.ks[QF == 1 ? bh_ * a.tiles : bh_ * a.tiles * 4 + G];
    bool any = false;
#pragma unroll
    for (int qg = 0; qg < NQG; ++qg) any |= row[qg] < a.Nq && qsv[qg] * ks0 * a.sm * (kMax * kMax * kRootD) > kWide;
    return wave_any(any);
  }

  // Phase 3 of a tile for row group qg: the P bytes against the running maximum mx (and on
  // the control path the row's unrounded mass tmq).
  template <bool LAST, bool PRE>
  __device__ __forceinline__ void bytes(const AttnArgs& a, const float (&bs)[8][4], float scl, float mx, float fb,
                                        v8i& Pq, float& tmq) {
    if constexpr (PM == 2) {
      // Folded ExpCast encode (the reference's default kernel modes without block
      // values, sal/csrc/vc/vc_math.cuh:16-111): code = RNE(fmaf(base, gain, bias)) with
      // gain = RN(scale * A) and bias = fmaf(-m', A, B), unless some row of this 16-row
      // group has |m'| > 128 or a lane's scale underflows or its gain overflows; then the
      // whole group takes the unfused code RNE(fmaf(RN(RN(base * scale) - m'), A, B)).
      const float scale = scl;
      const float gain = scale * kExpA;
      // every lane admits the fold: scale a positive normal (so gain is a positive normal
      // or +inf) and gain a positive normal (finite), |m'| <= 128; lane masks combined on
      // the scalar unit
      bool fold = true;
      if constexpr (!PRE) {
        const uint64_t safe = pos_normal_lanes(scale) & pos_normal_lanes(gain) &
                              __builtin_amdgcn_ballot_w64(fabsf(mx) <= 128.0f);
        fold = safe == __builtin_amdgcn_read_exec();
      }
      if (fold) {
        const float bias = fb;  // fmaf(-mx, A, B), kept with the running maximum
#pragma unroll
        for (int j = 0; j < 8; ++j) {
          uint32_t w = 0;
#pragma unroll
          for (int r = 0; r < 4; ++r) w = __builtin_amdgcn_cvt_pk_u8_f32(__builtin_fmaf(bs[j][r], gain, bias), r, w);
          Pq[j] = static_cast<int>(w);
        }
      } else {
#pragma unroll
        for (int j = 0; j < 8; ++j) {
          uint32_t w = 0;
#pragma unroll
          for (int r = 0; r < 4; ++r) {
            const float lgt = bs[j][r] * scale;
            w = __builtin_amdgcn_cvt_pk_u8_f32(__builtin_fmaf(lgt - mx, kExpA, kExpB), r, w);
          }
          Pq[j] = static_cast<int>(w);
        }
      }
    } else if constexpr (PM == 1) {
#pragma unroll
      for (int j = 0; j < 8; ++j) {
        uint32_t w = 0;
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          const float u = __builtin_fmaf(bs[j][r] - mx, kExpA, kExpB);
          w = __builtin_amdgcn_cvt_pk_u8_f32(u, r, w);
        }
        Pq[j] = static_cast<int>(w);
      }
    } else {
      // E4M3 of the hardware exp2, unless a probability of the span (a tile, at D64 four: its
      // three waves per SIMD have no registers for more) may lie within two ulps of an E4M3
      // midpoint by fp8_exp2_gap (a few in a hundred thousand): then the lane redoes the span
      // from the scores, which stay live, with both neighbours' bytes, and in binary64 where
      // these differ. One branch per tile keeps the loop one block that the MFMAs interleave with.
      // A vanishing probability (a score more than about 103 nats below the row maximum) always
      // fails the test: PRE takes none into account but sets wide, upon which the wave leaves for
      // the copy of the loop that lifts small probabilities over it, one more instruction per
      // probability; a wave whose scales let it expect one (wide_scores) starts there. Same box, us,
      // both neighbours' bytes of every probability / lifted / this: smoothing [1,7,37741,128] 3830 /
      // 3703 / 3528, [1,8,16000,64] 696 / 638 / 601, [1,16,3000,128] 94.4 / 92.1 / 87.3.
      const float f = scl;
      float ls = -0.0f;  // -0 + p = p: the first addition folds away
      constexpr int kSpan = D == 128 ? 8 : 1;
#pragma unroll
      for (int j0 = 0; j0 < 8; j0 += kSpan) {
        const float ls0 = ls;
        uint32_t gap = 0xffffffffu;
#pragma unroll
        for (int j = j0; j < j0 + kSpan; ++j) {
          float pr[4];
#pragma unroll
          for (int r = 0; r < 4; ++r) pr[r] = __builtin_amdgcn_exp2f(__builtin_fmaf(bs[j][r], f, -mx));
#pragma unroll
          for (int r = 0; r < 4; ++r) ls += pr[r];
          Pq[j] = static_cast<int>(fp8_exp2_quick<!PRE>(pr, gap));
        }
        if (__builtin_expect(gap <= kFp8Gap, 0)) {
          ls = ls0;
          float low = 1.0f;
#pragma unroll
          for (int j = j0; j < j0 + kSpan; ++j) {
            float xs[4], pr[4];
#pragma unroll
            for (int r = 0; r < 4; ++r) {
              float b = bs[j][r];
              asm volatile("" : "+v"(b));  // recomputed here, not kept live from the loop above
              xs[r] = __builtin_fmaf(b, f, -mx);
              pr[r] = __builtin_amdgcn_exp2f(xs[r]);
              low = fminf(low, pr[r]);
            }
            Pq[j] = static_cast<int>(fp8_exp2_word(xs, pr));
#pragma unroll
            for (int r = 0; r < 4; ++r) ls += pr[r];
          }
          if constexpr (PRE) wide |= low < 0x1p-100f ? 1 : 0;
        }
      }
      tmq = row_sum(ls);
    }
  }

  // DUMP: the P bytes of rows prow0..prow1 to pdump in logical key order.
  __device__ __forceinline__ void dump_p(const AttnArgs& a, int64_t t, int qg, const v8i& Pq) const {
    if constexpr (DUMP) {
      if (row[qg] >= a.prow0 && row[qg] < a.prow1 && row[qg] < a.Nq) {
        const int64_t npad = a.tiles * kTile;
        uint8_t* dst = a.pdump + (bh_ * (a.prow1 - a.prow0) + (row[qg] - a.prow0)) * npad + t * kTile;
#pragma unroll
        for (int j = 0; j < 8; ++j)
#pragma unroll
          for (int r = 0; r < 4; ++r)
            dst[16 * j + 8 * (r >> 1) + 2 * G + (r & 1)] = static_cast<uint8_t>((static_cast<uint32_t>(Pq[j]) >> (8 * r)) & 0xffu);
      }
    }
  }

  // Scores of one 16-key block against one 16-row group.
  __device__ __forceinline__ Acc score(const v4i (&k)[DS], const v4i (&q)[DS]) const {
    if constexpr (QF == 1) {
      // E4M3 x E4M3 over all D channels in one 128-deep step; lane group G holds the
      // channel sets {16G..16G+15} and {64+16G..64+16G+15} for both operands.
      const v8i ka = DS == 2 ? v8i{k[0][0], k[0][1], k[0][2], k[0][3], k[DS - 1][0], k[DS - 1][1], k[DS - 1][2], k[DS - 1][3]}
                             : v8i{k[0][0], k[0][1], k[0][2], k[0][3], 0, 0, 0, 0};
      const v8i qb = DS == 2 ? v8i{q[0][0], q[0][1], q[0][2], q[0][3], q[DS - 1][0], q[DS - 1][1], q[DS - 1][2], q[DS - 1][3]}
                             : v8i{q[0][0], q[0][1], q[0][2], q[0][3], 0, 0, 0, 0};
      return mfma_fp8(ka, qb, v4f{0.0f, 0.0f, 0.0f, 0.0f});
    } else {
      v4i acc = IB ? bacc : v4i{0, 0, 0, 0};
#pragma unroll
      for (int ds = 0; ds < DS; ++ds) acc = __builtin_amdgcn_mfma_i32_16x16x64_i8(k[ds], q[ds], acc, 0, 0, 0);
      return acc;
    }
  }

  // PRE: the fold conditions hold on this tile (fold_precheck), so it does not test them.
  // next(j), j = 0..7, issues a part of the next tile's loads after each key block's MFMAs. All
  // of them at the tile's start held the waves' issue until the address unit had taken 512
  // clocks of them; spread out they hide behind the MFMAs. Same box: smoothing 10.65 -> 10.51 ms,
  // control [1,7,37741,128] 3.89 -> 3.83 ms, main 9.45 -> 9.31 ms, FP8 QK call
  // 9.51 -> 9.12 ms, and where a CU runs one
  // 64-row block, [1,8,1024 x 8192,128], 62 -> 52 us.
  template <bool LAST, bool PRE = false, class Next>
  __device__ __forceinline__ void tile(const AttnArgs& a, int64_t t, const uint8_t* lk, const uint8_t* lv, const uint8_t* lm,
                                       Next next) {
    const float ksv = *reinterpret_cast<const float*>(lm + LD::KS_OFF + (QF == 1 ? 0 : 4 * G));

    // ---- S^T = K Q^T
    Acc S[NQG][8];
    v4i kf[8][DS];
#pragma unroll
    for (int j = 0; j < 2; ++j)
#pragma unroll
      for (int ds = 0; ds < DS; ++ds) kf[j][ds] = *reinterpret_cast<const v4i*>(lk + j * 16 * D + koff[ds]);
#pragma unroll
    for (int j = 0; j < 8; ++j) {
      if (j + 2 < 8) {
#pragma unroll
        for (int ds = 0; ds < DS; ++ds) kf[j + 2][ds] = *reinterpret_cast<const v4i*>(lk + (j + 2) * 16 * D + koff[ds]);
      }
#pragma unroll
      for (int qg = 0; qg < NQG; ++qg) S[qg][j] = score(kf[j], qf[qg]);
      next(j);
      __builtin_amdgcn_sched_barrier(0);
    }

    // ---- logits, online max, P bytes (ExpCast codes, or E4M3 probabilities on the control path)
    v8i P[NQG];
    float tmass[NQG], bs[NQG][8][4], tmax[NQG], scl[NQG];
    // The history of a row group in which some maximum moved is rescaled before this tile's
    // PV adds in. At D64 the scaling sits inside the branches where a maximum can move, so
    // the common tile carries no rescale state (two instructions per tile; same-box D64 with
    // smoothing 0.4-0.7 % faster); at D128 that placement costs the main kernel 0.3 % (its
    // register allocation moves), so there the flags resc / dm carry it to one place after
    // the bytes.
    constexpr bool kEarly = D == 64;
    bool resc[NQG];
    float dm[NQG];
#pragma unroll
    for (int qg = 0; qg < NQG; ++qg) resc[qg] = false;
    auto moved = [&](int qg, float mn) {
      if constexpr (kEarly) {
        if (wave_any(m[qg] != mn)) rescale(qg, m[qg] - mn);
      } else {
        resc[qg] = wave_any(m[qg] != mn);
        dm[qg] = m[qg] - mn;
      }
    };
    if constexpr (PM == 0) {
      // Control path, one row group at a time (D64's three waves per SIMD have no registers
      // for both groups' probabilities at once).
#pragma unroll
      for (int qg = 0; qg < NQG; ++qg) {
        tmax[qg] = logits<LAST>(a, t, qg, S[qg], ksv, bs[qg], scl[qg]);
        const float mn = running_max(m[qg], tmax[qg]);
        moved(qg, mn);
        m[qg] = mn;
        bytes<LAST, PRE>(a, bs[qg], scl[qg], m[qg], 0.0f, P[qg], tmass[qg]);
        if constexpr (DUMP) dump_p(a, t, qg, P[qg]);
      }
    } else {
#pragma unroll
      for (int qg = 0; qg < NQG; ++qg) tmax[qg] = logits<LAST>(a, t, qg, S[qg], ksv, bs[qg], scl[qg]);
      // Both row groups' running maxima in one cross-lane reduction, skipped when no lane's
      // maximum exceeds its row's running maximum (then no row maximum moves).
      uint64_t up = __builtin_amdgcn_ballot_w64(tmax[0] > m[0]);
      if constexpr (NQG == 2) up |= __builtin_amdgcn_ballot_w64(tmax[1] > m[1]);
      if (up != 0) {
        float mn[NQG];
        if constexpr (NQG == 2) running_max2(m, tmax, mn);
        else mn[0] = running_max(m[0], tmax[0]);
#pragma unroll
        for (int qg = 0; qg < NQG; ++qg) {
          moved(qg, mn[qg]);
          m[qg] = mn[qg];
          if constexpr (PM == 2) fbias[qg] = __builtin_fmaf(-mn[qg], kExpA, kExpB);
        }
      }
#pragma unroll
      for (int qg = 0; qg < NQG; ++qg) {
        bytes<LAST, PRE>(a, bs[qg], scl[qg], m[qg], fbias[qg], P[qg], tmass[qg]);
        if constexpr (DUMP) dump_p(a, t, qg, P[qg]);
      }
    }

    if constexpr (!kEarly) {
#pragma unroll
      for (int qg = 0; qg < NQG; ++qg)
        if (resc[qg]) rescale(qg, dm[qg]);
    }

    // ---- O^T += V^T P^T, mass = 1^T P^T
    const v4f zero = {0.0f, 0.0f, 0.0f, 0.0f};
    float mass[NQG];
    if constexpr (BSCALE) {
      // Per-block V scales: O += vs_t * PV_t per channel, one FMA per element on the PV
      // temporary of each channel block; the mean term vs_t * mean_t * mass joins the
      // deferred restore below.
#pragma unroll
      for (int qg = 0; qg < NQG; ++qg) {
        if constexpr (EC) mass[qg] = mfma_mass(ones, P[qg], zero)[0];
        else mass[qg] = tmass[qg];
        den[qg] += mass[qg];
      }
      const uint8_t* vsl = vsring + (t % LD::NR) * LD::VS;
      v8i vc = load_v(lv, 0), vn;
#pragma unroll
      for (int cb = 0; cb < CB; ++cb) {
        if (cb + 1 < CB) vn = load_v(lv, cb + 1);
        const float4 vsb = *reinterpret_cast<const float4*>(vsl + 4 * (16 * cb + 4 * G));
        const float sc[4] = {vsb.x, vsb.y, vsb.z, vsb.w};
#pragma unroll
        for (int qg = 0; qg < NQG; ++qg) {
          const v4f pv = mfma_fp8(vc, P[qg], zero);
#pragma unroll
          for (int r = 0; r < 4; ++r) O[qg][cb][r] = __builtin_fmaf(pv[r], sc[r], O[qg][cb][r]);
        }
        vc = vn;
        __builtin_amdgcn_sched_barrier(0);
      }
    } else {
      v8i vf[CB];
      vf[0] = load_v(lv, 0);
      if (CB > 1) vf[1] = load_v(lv, 1);
#pragma unroll
      for (int cb = 0; cb < CB; ++cb) {
        if (cb + 2 < CB) vf[cb + 2] = load_v(lv, cb + 2);
#pragma unroll
        for (int qg = 0; qg < NQG; ++qg) O[qg][cb] = mfma_fp8(vf[cb], P[qg], O[qg][cb]);
        __builtin_amdgcn_sched_barrier(0);
      }
#pragma unroll
      for (int qg = 0; qg < NQG; ++qg) {
        if constexpr (DACC) {
          dacc[qg] = mfma_mass(ones, P[qg], dacc[qg]);
        } else {
          if constexpr (EC) mass[qg] = mfma_mass(ones, P[qg], zero)[0];
          else mass[qg] = tmass[qg];
          den[qg] += mass[qg];
        }
      }
    }
    if constexpr (SMOOTH) {
      // Deferred block-mean restore: tile t is position c of its chunk; lane group
      // G = c / 4 keeps the row's mass in slot c % 4 (the MFMA's k = c). At the chunk's
      // end (or the last tile) O^T[ch][row] += sum_k mean_k[ch] * w_k[row] over the
      // chunk, as v_mfma_f32_16x16x16f16 (A: means from the ring, exact in fp16, or with
      // per-block scales RN_f16(vs_k[ch] * mean_k[ch]); B: the weights as fp16 hi and lo
      // parts).
      // Slots of tiles past the last hold w = 0.
      const int c = static_cast<int>(t & (kChunk - 1));
      // one select per row group: the slot c & 3 is wave-uniform (a scalar branch), only the
      // lane-group test G == c / 4 is per lane
      const bool mine = G == (c >> 2);
      switch (c & 3) {
        case 0: set_weight<0>(mine, mass); break;
        case 1: set_weight<1>(mine, mass); break;
        case 2: set_weight<2>(mine, mass); break;
        default: set_weight<3>(mine, mass); break;
      }
      if (LAST || c == kChunk - 1) flush_means(ring, t - c);
    }
  }

  template <int J>
  __device__ __forceinline__ void set_weight(bool mine, const float (&mass)[NQG]) {
#pragma unroll
    for (int qg = 0; qg < NQG; ++qg) wts[qg][J] = mine ? mass[qg] : wts[qg][J];
  }

  // O += means (x) weights over a chunk of pending tiles (VM 1, 2). Each weight goes in as two
  // fp16 parts, hi = RN_f16(w) and lo = RN_f16(w - hi) (w - hi is exact in binary32), so the
  // mean term carries about 22 bits of the weight instead of 11. mean(pos, ch) is the fp16 mean
  // of the chunk's tile pos in channel ch, vscale(pos, ch) its fp32 V scale (VM 2).
  template <class MeanFn, class ScaleFn>
  __device__ __forceinline__ void flush_weights(MeanFn mean, ScaleFn vscale) {
    typedef _Float16 v4h __attribute__((ext_vector_type(4)));
    v4h b[NQG], bl[NQG];
#pragma unroll
    for (int qg = 0; qg < NQG; ++qg) {
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        b[qg][j] = static_cast<_Float16>(wts[qg][j]);
        bl[qg][j] = static_cast<_Float16>(wts[qg][j] - static_cast<float>(b[qg][j]));
        wts[qg][j] = 0.0f;
      }
    }
#pragma unroll
    for (int cb = 0; cb < CB; ++cb) {
      v4h av;
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        const _Float16 mh = mean(4 * G + j, 16 * cb + li);
        if constexpr (BSCALE) av[j] = static_cast<_Float16>(static_cast<float>(mh) * vscale(4 * G + j, 16 * cb + li));
        else av[j] = mh;
      }
#pragma unroll
      for (int qg = 0; qg < NQG; ++qg) {
        O[qg][cb] = __builtin_amdgcn_mfma_f32_16x16x16f16(av, bl[qg], O[qg][cb], 0, 0, 0);
        O[qg][cb] = __builtin_amdgcn_mfma_f32_16x16x16f16(av, b[qg], O[qg][cb], 0, 0, 0);
      }
    }
  }
  // The chunk of tiles base .. base + 15, from the LDS rings.
  __device__ inline void flush_means(const uint8_t* ring, int64_t base) {
    const uint8_t* col = ring;
    auto slot = [&](int pos) { return (static_cast<uint32_t>(base) + pos) % LD::NR; };
    flush_weights([&](int pos, int ch) { return *reinterpret_cast<const _Float16*>(col + slot(pos) * LD::RS + 2 * ch); },
                  [&](int pos, int ch) { return *reinterpret_cast<const float*>(vsring + slot(pos) * LD::VS + 4 * ch); });
  }
  const uint8_t* ring = nullptr;
  const uint8_t* vsring = nullptr;
};

// Four channels ch .. ch + 3 of one output row: normalised, times the per-channel V scale
// (per-block scales were applied tile by tile), rounded and stored.
template <int D, int OUT, bool BSCALE>
__device__ __forceinline__ void store_row(const AttnArgs& a, int64_t bh, uint16_t* out, int ch, const v4f& o, float inv) {
  const float4 sc = BSCALE ? make_float4(1.0f, 1.0f, 1.0f, 1.0f) : *reinterpret_cast<const float4*>(a.vs + bh * D + ch);
  const float y0 = o[0] * inv * sc.x, y1 = o[1] * inv * sc.y, y2 = o[2] * inv * sc.z, y3 = o[3] * inv * sc.w;
  uint2 packed;
  if constexpr (OUT == VCX_BFLOAT16) {
    packed.x = f32_to_bf16_bits(y0) | (f32_to_bf16_bits(y1) << 16);
    packed.y = f32_to_bf16_bits(y2) | (f32_to_bf16_bits(y3) << 16);
  } else {
    packed.x = f32_to_f16_bits(y0) | (f32_to_f16_bits(y1) << 16);
    packed.y = f32_to_f16_bits(y2) | (f32_to_f16_bits(y3) << 16);
  }
  *reinterpret_cast<uint2*>(out + ch) = packed;
}

}  // namespace
}  // namespace vcx
