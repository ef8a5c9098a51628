// Fused sageattn_vc forward for gfx950 (MI355X).
//
// One workgroup = 4 waves = 128 query rows; each wave owns 32 rows as two
// 16-row groups. Per 128-key tile:
//   S^T = K Q^T       v_mfma_i32_16x16x64_i8   (A = K rows from LDS, B = Q^T in VGPRs)
//   logits, online max, ExpCast codes         VALU, one query row per lane
//   O^T += V^T P^T    v_mfma_f32_16x16x128_f8f6f4 (A = V^T from LDS, B = codes in VGPRs)
//   row mass          the same MFMA with an all-ones A operand
// The 16x16 accumulator layout (lane l holds rows 4*(l/16)+r, column l%16)
// puts the 32 scores of one query row of a 16-key block in the 4 lanes
// l%16 + 16*G; the codes of block j, rows r=0..3 form byte 4j+r of the lane's
// PV B operand, so P never leaves the registers. K rows are loaded into the
// A operand in the order key(j, 4G+r) = 16j + 8(r/2) + 2G + r%2, which gives
// every lane group G exactly the keys of Sage K-scale group (key%8)/2 == G;
// the V payload is stored in the matching order (vcx_value_token).
//
// K and V^T tiles stream through LDS with gfx950 direct-to-LDS loads
// (global_load_lds_dwordx4), double buffered, placed so that the operand reads
// run at the conflict-free ds_read_b128 rate (key_row / chunk_xor below).
//
// Numerical contract (reference sal/csrc/vc/vc_sm90.cu:284-612, vc_math.cuh:268-474):
//   tiles before the last: logit = RN(float(acc) * RN(sm * RN(qs*ks)))
//   last tile:             logit = RN(RN(float(acc) * RN(qs*ks)) * sm), keys >= Nk -> -inf
//   m' = max(m, rowmax), code = sat_u8(RNE(fmaf(RN(logit-m'), A, B)))
//   alpha = exp2((m - m') * log2(e)) (hardware exp2; alpha == 1 exactly when m' == m)
//   O = alpha*O + PV (+ mass*mean), den = alpha*den + mass, out = O/den * vs.
// The P bytes follow the contract exactly; alpha, O and den only feed the
// bf16/fp16 output, whose tolerance covers the exp2 approximation. With per-channel
// V scales (VM 1) the mass*mean term is deferred: every 16 tiles one f16 MFMA per
// channel block adds sum_t mean_t (x) w_t, w_t the tile mass rescaled with O.
//
// PM = 2 (expcast = 2, no block values) is the folded encode of the reference's default
// kernel modes (vc_math.cuh:16-111): code = sat_u8(RNE(fmaf(base, RN(scale*A), fmaf(-m', A, B))))
// with scale = RN(sm*RN(qs*ks)) (last tile: base = RN(float(acc)*dq), scale = sm), and the
// unfused code above for a whole 16-row group in a tile where some |m'| > 128, a scale
// underflows or a gain overflows (the reference's warp-wide fallback).
//
// QF = 1 is the block-scaled FP8 QK format (the reference's experimental vc27,
// sal/sageattention_local/vc_fp8.py, fp8_dispatch.cuh): E4M3 Q/K with one scale per
// 64 query rows and one per 128-key tile, scores from v_mfma_f32_16x16x128_f8f6f4 (the
// same K/Q fragment loads, two 16-byte halves per lane; D64 pads the second half with
// zeros), V per-channel E4M3 with no block values, and the PM 0/1/2 probability paths.
//
// PM = 0 is the Sage FP8 control path (expcast=False; vc_sm90.cu:177,
// attn_utils.cuh:355-455): a.sm = RN(sm * RN(log2 e)), base/factor as above,
// m' = max(m, max fmaf(base, factor, -8.807)), P = E4M3(exp2(fmaf(base, factor, -m'))) with
// the correctly rounded binary32 exp2 (fp8_exp2_quick: v_exp_f32, and next to an E4M3 rounding
// midpoint, which fp8_exp2_gap looks for, fp8_exp2_word: rechecked in binary64); den and the mean restore use the unrounded sum of P.
#include "vcx_attn.hpp"

#include <functional>
#include <map>
#include <mutex>
#include <utility>
#include <vector>

namespace vcx {
namespace {

// D64 without per-block V scales runs three workgroups per CU (at most 168 VGPRs; its
// 37 KB of LDS allows four): the VALU-bound D64 loop gains from the third wave per SIMD
// (same-box: smoothing D64 8.15 -> 7.75 ms). D128 is held to two by its 64-74 KB of LDS.
template <int D, int VM>
constexpr int kBlocksPerCU = (D == 64 && VM < 2) ? 3 : 2;


// Tiles 0 .. tiles-2, two per iteration so each buffer is a fixed LDS object; on return t is
// the last tile, whose K/V the DMA has been issued for (buffer t & 1).
template <bool PRE, class W, class LD, class TI>
__device__ __forceinline__ void body_tiles(W& w, const LD& ld, const AttnArgs& a, TI& t, uint8_t* lds0,
                                           uint8_t* lds1, uint8_t* meta0, uint8_t* meta1) {
  constexpr int KB = kTile * W::kD;
  const TI body = static_cast<TI>(a.tiles) - 1;
  constexpr bool kLeaves = PRE && W::kPM == 0;  // a wave may leave this copy for the other one
  TI end = body;
  for (; t + 2 <= end; t += 2) {
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    __syncthreads();
    if constexpr (!W::kSpread) ld.issue(t + 1, lds1, lds1 + KB, meta1);
    w.template tile<false, PRE>(a, t, lds0, lds0 + KB, meta0, [&](int i) {
      if (W::kSpread && i < LD::kParts) ld.part(i, t + 1, lds1, lds1 + KB, meta1);
    });
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    __syncthreads();
    if constexpr (!W::kSpread) ld.issue(t + 2, lds0, lds0 + KB, meta0);
    w.template tile<false, PRE>(a, t + 1, lds1, lds1 + KB, meta1, [&](int i) {
      if (W::kSpread && i < LD::kParts) ld.part(i, t + 2, lds0, lds0 + KB, meta0);
    });
    if constexpr (kLeaves) end = wave_any(w.wide != 0) ? 0 : body;
  }
  if (kLeaves ? t + 1 == body : t < body) {  // odd count of body tiles: one more from buffer 0, last tile lands in buffer 1
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    __syncthreads();
    if constexpr (!W::kSpread) ld.issue(t + 1, lds1, lds1 + KB, meta1);
    w.template tile<false, PRE>(a, t, lds0, lds0 + KB, meta0, [&](int i) {
      if (W::kSpread && i < LD::kParts) ld.part(i, t + 1, lds1, lds1 + KB, meta1);
    });
    ++t;
  }
}

// One block's rows [row0, row0 + 64 * NQG) of head bh: 4 waves of 16 * NQG rows.
template <int D, int VM, bool DUMP, int OUT, int PM, int QF, int NQG>
__device__ __forceinline__ void attn_block(const AttnArgs& a, int64_t bh, int64_t row0, uint8_t* lds0, uint8_t* lds1,
                                           uint8_t* meta0, uint8_t* meta1, uint8_t* ring, uint8_t* vsring) {
  typedef TileLoader<D, VM, QF> LD;
  typedef Wave<D, VM, DUMP, PM, QF, NQG> W;
  constexpr int KB = kTile * D;
  constexpr int RING_BYTES = LD::RING ? LD::NR * LD::RS : 16;
  constexpr int VSRING_BYTES = LD::BSCALE ? LD::NR * LD::VS : 16;
  const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
  W w;
  w.G = lane >> 4;
  w.li = lane & 15;
  w.bh_ = bh;
  // Lane-constant LDS offsets.
#pragma unroll
  for (int ds = 0; ds < W::DS; ++ds) w.koff[ds] = w.li * D + ((((D == 128) ? 4 * ds : 0) + w.G) ^ chunk_xor<D>(w.li)) * 16;
#pragma unroll
  for (int h = 0; h < 2; ++h) w.voff[h] = w.li * kTile + (((4 * h + w.G) ^ (w.li & 7)) * 16);

  // Q fragments (B operand) and per-row scales.
#pragma unroll
  for (int qg = 0; qg < NQG; ++qg) {
    const int64_t r = row0 + wave * (16 * NQG) + qg * 16 + w.li;
    w.row[qg] = r;
    // Q scale: Sage per-thread INT8 index (row/16)*8 + row%8, or the FP8 row block row/64
    const int64_t si = QF == 1 ? r / 64 : (r / 16) * 8 + r % 8;
    w.qsv[qg] = si < a.qs_len ? a.qs[bh * a.qs_len + si] : 1.0f;
#pragma unroll
    for (int ds = 0; ds < W::DS; ++ds) {
      if (r < a.Nq) w.qf[qg][ds] = *reinterpret_cast<const v4i*>(a.q8 + (bh * a.Nq + r) * D + ds * 64 + w.G * 16);
      else w.qf[qg][ds] = v4i{0, 0, 0, 0};
    }
    w.m[qg] = -5000000.0f;
    w.den[qg] = 0.0f;
    w.dacc[qg] = v4f{0.0f, 0.0f, 0.0f, 0.0f};
    w.fbias[qg] = __builtin_fmaf(5000000.0f, kExpA, kExpB);
#pragma unroll
    for (int j = 0; j < 4; ++j) w.wts[qg][j] = 0.0f;
#pragma unroll
    for (int cb = 0; cb < W::CB; ++cb) w.O[qg][cb] = v4f{0.0f, 0.0f, 0.0f, 0.0f};
  }

  // Without block values the opaque copy keeps the compiler from rebuilding the constant
  // operand every tile; the smoothing variants have no registers to spare for it.
  w.ones = v4i{0x22222222, 0x22222222, 0x22222222, 0x22222222};
  if constexpr (VM == 0 && (D == 128 || PM == 2)) asm volatile("" : "+v"(w.ones));
  w.bacc = v4i{kBias, kBias, kBias, kBias};
  if constexpr (W::IB && VM == 0 && D == 128) asm volatile("" : "+v"(w.bacc));
  w.fold_ok = 0;
  if constexpr (PM == 2 && QF == 0) w.fold_precheck(a, lane);

  LD ld;
  ld.init(a, bh);
  if constexpr (LD::RING) {
    // The last chunk's flush reads ring slots of tiles past the last one (weight 0):
    // they must hold finite values, so the rings start zeroed.
    for (int i = threadIdx.x; i < RING_BYTES / 16; i += kThreadsPerBlock)
      reinterpret_cast<uint4*>(ring)[i] = make_uint4(0, 0, 0, 0);
    if constexpr (LD::BSCALE) {
      for (int i = threadIdx.x; i < VSRING_BYTES / 16; i += kThreadsPerBlock)
        reinterpret_cast<uint4*>(vsring)[i] = make_uint4(0, 0, 0, 0);
    }
    __syncthreads();
    ld.ring = ring;
    w.ring = ring;
    ld.vsring = vsring;
    w.vsring = vsring;
  }
  ld.issue(0, lds0, lds0 + KB, meta0);
  // Tiles before the last; a wave whose fold conditions were prechecked runs the copy of
  // the loop without the tests.
  // 32-bit tile index (tiles < 2^23), so the loop test stays on the scalar unit; the
  // per-block-scale variants keep 64 bits (with 32 their register allocation spills)
  typedef std::conditional_t<VM == 2, int64_t, int> TI;
  TI t = 0;
  w.wide = 0;
  if constexpr (PM == 0) {
    // the cheap midpoint test until a vanishing probability; after an early end the rest
    if constexpr (W::kCheapTest) {
      if (!w.wide_scores(a)) body_tiles<true>(w, ld, a, t, lds0, lds1, meta0, meta1);
    }
    body_tiles<false>(w, ld, a, t, lds0, lds1, meta0, meta1);
  } else if constexpr (PM == 2 && QF == 0) {
    if (w.fold_ok) body_tiles<true>(w, ld, a, t, lds0, lds1, meta0, meta1);
    else body_tiles<false>(w, ld, a, t, lds0, lds1, meta0, meta1);
  } else {
    body_tiles<false>(w, ld, a, t, lds0, lds1, meta0, meta1);
  }
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
  __syncthreads();
  if (t & 1) w.template tile<true>(a, t, lds1, lds1 + KB, meta1, [](int) {});
  else w.template tile<true>(a, t, lds0, lds0 + KB, meta0, [](int) {});

  // ---- epilogue: normalise, per-channel V scale, store 4 channels per lane and block
  const int64_t b = bh / a.H, h = bh % a.H;
#pragma unroll
  for (int qg = 0; qg < NQG; ++qg) {
    if (w.row[qg] >= a.Nq) continue;
    const float inv = 1.0f / (W::DACC ? w.dacc[qg][0] : w.den[qg]);
    uint16_t* out = static_cast<uint16_t*>(a.out) + b * a.osb + h * a.osh + w.row[qg] * a.osn;
#pragma unroll
    for (int cb = 0; cb < W::CB; ++cb) {
      store_row<D, OUT, W::BSCALE>(a, bh, out, 16 * cb + 4 * w.G, w.O[qg][cb], inv);
    }
  }
}

template <int D, int VM, bool DUMP, int OUT, int PM, int QF = 0>
__global__ __launch_bounds__(kThreadsPerBlock, (kBlocksPerCU<D, VM>)) void attn_kernel(AttnArgs a) {
#if defined(__HIP_DEVICE_COMPILE__)  // device code; the host pass only emits the launch stub
  typedef TileLoader<D, VM, QF> LD;
  constexpr int KB = kTile * D, VB = D * kTile;
  __shared__ __attribute__((aligned(16))) uint8_t lds0[KB + VB];
  __shared__ __attribute__((aligned(16))) uint8_t lds1[KB + VB];
  __shared__ __attribute__((aligned(16))) uint8_t meta0[LD::META_BYTES];
  __shared__ __attribute__((aligned(16))) uint8_t meta1[LD::META_BYTES];
  constexpr int RING_BYTES = LD::RING ? LD::NR * LD::RS : 16;
  __shared__ __attribute__((aligned(16))) uint8_t ring[RING_BYTES];
  constexpr int VSRING_BYTES = LD::BSCALE ? LD::NR * LD::VS : 16;
  __shared__ __attribute__((aligned(16))) uint8_t vsring[VSRING_BYTES];

  // XCD-aware order: the hardware deals blocks round-robin over 8 XCDs; give each XCD a
  // contiguous range of (head, query block) so its L2 serves one head. The j-th block of XCD
  // x is the j-th entry of its list: the range's first n_x - kconv 128-row blocks, then each
  // of its last kconv blocks as two 64-row halves, so that the XCD's last round is made of
  // half-length pieces (the grid has nfull + 8 * kconv blocks; kconv <= nfull / 8).
  const int64_t p = blockIdx.x;
  const int64_t per = a.nfull / 8, rem = a.nfull % 8, xcd = p % 8, j = p / 8;
  const int64_t start = xcd < rem ? xcd * (per + 1) : rem * (per + 1) + (xcd - rem) * per;
  const int64_t nfx = per + (xcd < rem ? 1 : 0) - a.kconv;
  if (j < nfx) {
    const int64_t logical = start + j;
    const int64_t bh = logical / a.qblocks, qb = logical % a.qblocks;
    attn_block<D, VM, DUMP, OUT, PM, QF, 2>(a, bh, qb * kRowsPerBlock, lds0, lds1, meta0, meta1, ring, vsring);
  } else {
    const int64_t hj = j - nfx, logical = start + nfx + hj / 2;
    const int64_t bh = logical / a.qblocks, qb = logical % a.qblocks;
    attn_block<D, VM, DUMP, OUT, PM, QF, 1>(a, bh, qb * kRowsPerBlock + (hj & 1) * (kRowsPerBlock / 2), lds0, lds1,
                                           meta0, meta1, ring, vsring);
  }
#else
  (void)a;
#endif
}

// Explicit instantiation of every launch variant: hipcc's host pass otherwise
// emitted the kernel handle of only the first variant named in each ternary.
template __global__ void attn_kernel<64, 0, false, 0, 2>(AttnArgs);
template __global__ void attn_kernel<64, 0, false, 1, 2>(AttnArgs);
template __global__ void attn_kernel<64, 0, true, 0, 2>(AttnArgs);
template __global__ void attn_kernel<64, 0, true, 1, 2>(AttnArgs);
template __global__ void attn_kernel<128, 0, false, 0, 2>(AttnArgs);
template __global__ void attn_kernel<128, 0, false, 1, 2>(AttnArgs);
template __global__ void attn_kernel<128, 0, true, 0, 2>(AttnArgs);
template __global__ void attn_kernel<128, 0, true, 1, 2>(AttnArgs);
template __global__ void attn_kernel<64, 0, false, 0, 1>(AttnArgs);
template __global__ void attn_kernel<64, 0, false, 1, 1>(AttnArgs);
template __global__ void attn_kernel<64, 0, true, 0, 1>(AttnArgs);
template __global__ void attn_kernel<64, 0, true, 1, 1>(AttnArgs);
template __global__ void attn_kernel<64, 1, false, 0, 1>(AttnArgs);
template __global__ void attn_kernel<64, 1, false, 1, 1>(AttnArgs);
template __global__ void attn_kernel<64, 1, true, 0, 1>(AttnArgs);
template __global__ void attn_kernel<64, 1, true, 1, 1>(AttnArgs);
template __global__ void attn_kernel<64, 2, false, 0, 1>(AttnArgs);
template __global__ void attn_kernel<64, 2, false, 1, 1>(AttnArgs);
template __global__ void attn_kernel<64, 2, true, 0, 1>(AttnArgs);
template __global__ void attn_kernel<64, 2, true, 1, 1>(AttnArgs);
template __global__ void attn_kernel<128, 0, false, 0, 1>(AttnArgs);
template __global__ void attn_kernel<128, 0, false, 1, 1>(AttnArgs);
template __global__ void attn_kernel<128, 0, true, 0, 1>(AttnArgs);
template __global__ void attn_kernel<128, 0, true, 1, 1>(AttnArgs);
template __global__ void attn_kernel<128, 1, false, 0, 1>(AttnArgs);
template __global__ void attn_kernel<128, 1, false, 1, 1>(AttnArgs);
template __global__ void attn_kernel<128, 1, true, 0, 1>(AttnArgs);
template __global__ void attn_kernel<128, 1, true, 1, 1>(AttnArgs);
template __global__ void attn_kernel<128, 2, false, 0, 1>(AttnArgs);
template __global__ void attn_kernel<128, 2, false, 1, 1>(AttnArgs);
template __global__ void attn_kernel<128, 2, true, 0, 1>(AttnArgs);
template __global__ void attn_kernel<128, 2, true, 1, 1>(AttnArgs);
template __global__ void attn_kernel<64, 0, false, 0, 0>(AttnArgs);
template __global__ void attn_kernel<64, 0, false, 1, 0>(AttnArgs);
template __global__ void attn_kernel<64, 0, true, 0, 0>(AttnArgs);
template __global__ void attn_kernel<64, 0, true, 1, 0>(AttnArgs);
template __global__ void attn_kernel<64, 1, false, 0, 0>(AttnArgs);
template __global__ void attn_kernel<64, 1, false, 1, 0>(AttnArgs);
template __global__ void attn_kernel<64, 1, true, 0, 0>(AttnArgs);
template __global__ void attn_kernel<64, 1, true, 1, 0>(AttnArgs);
template __global__ void attn_kernel<64, 2, false, 0, 0>(AttnArgs);
template __global__ void attn_kernel<64, 2, false, 1, 0>(AttnArgs);
template __global__ void attn_kernel<64, 2, true, 0, 0>(AttnArgs);
template __global__ void attn_kernel<64, 2, true, 1, 0>(AttnArgs);
template __global__ void attn_kernel<128, 0, false, 0, 0>(AttnArgs);
template __global__ void attn_kernel<128, 0, false, 1, 0>(AttnArgs);
template __global__ void attn_kernel<128, 0, true, 0, 0>(AttnArgs);
template __global__ void attn_kernel<128, 0, true, 1, 0>(AttnArgs);
template __global__ void attn_kernel<128, 1, false, 0, 0>(AttnArgs);
template __global__ void attn_kernel<128, 1, false, 1, 0>(AttnArgs);
template __global__ void attn_kernel<128, 1, true, 0, 0>(AttnArgs);
template __global__ void attn_kernel<128, 1, true, 1, 0>(AttnArgs);
template __global__ void attn_kernel<128, 2, false, 0, 0>(AttnArgs);
template __global__ void attn_kernel<128, 2, false, 1, 0>(AttnArgs);
template __global__ void attn_kernel<128, 2, true, 0, 0>(AttnArgs);
template __global__ void attn_kernel<128, 2, true, 1, 0>(AttnArgs);

template __global__ void attn_kernel<64, 0, false, 0, 2, 1>(AttnArgs);
template __global__ void attn_kernel<64, 0, false, 1, 2, 1>(AttnArgs);
template __global__ void attn_kernel<64, 0, true, 0, 2, 1>(AttnArgs);
template __global__ void attn_kernel<64, 0, true, 1, 2, 1>(AttnArgs);
template __global__ void attn_kernel<128, 0, false, 0, 2, 1>(AttnArgs);
template __global__ void attn_kernel<128, 0, false, 1, 2, 1>(AttnArgs);
template __global__ void attn_kernel<128, 0, true, 0, 2, 1>(AttnArgs);
template __global__ void attn_kernel<128, 0, true, 1, 2, 1>(AttnArgs);
template __global__ void attn_kernel<64, 0, false, 0, 1, 1>(AttnArgs);
template __global__ void attn_kernel<64, 0, false, 1, 1, 1>(AttnArgs);
template __global__ void attn_kernel<64, 0, true, 0, 1, 1>(AttnArgs);
template __global__ void attn_kernel<64, 0, true, 1, 1, 1>(AttnArgs);
template __global__ void attn_kernel<128, 0, false, 0, 1, 1>(AttnArgs);
template __global__ void attn_kernel<128, 0, false, 1, 1, 1>(AttnArgs);
template __global__ void attn_kernel<128, 0, true, 0, 1, 1>(AttnArgs);
template __global__ void attn_kernel<128, 0, true, 1, 1, 1>(AttnArgs);
template __global__ void attn_kernel<64, 0, false, 0, 0, 1>(AttnArgs);
template __global__ void attn_kernel<64, 0, false, 1, 0, 1>(AttnArgs);
template __global__ void attn_kernel<64, 0, true, 0, 0, 1>(AttnArgs);
template __global__ void attn_kernel<64, 0, true, 1, 0, 1>(AttnArgs);
template __global__ void attn_kernel<128, 0, false, 0, 0, 1>(AttnArgs);
template __global__ void attn_kernel<128, 0, false, 1, 0, 1>(AttnArgs);
template __global__ void attn_kernel<128, 0, true, 0, 0, 1>(AttnArgs);
template __global__ void attn_kernel<128, 0, true, 1, 0, 1>(AttnArgs);

// Makespan, in units of one 128-row block's time, of one XCD's block list on S slots served
// in list order, each block to the slot that frees first: n - k full blocks, then 2k halves
// of relative length h.
double list_makespan(int64_t n, int64_t k, int S, double h) {
  std::vector<double> slot(static_cast<size_t>(S), 0.0);
  const int64_t nf = n - k, r = nf / S, f = nf % S;
  for (int i = 0; i < S; ++i) slot[static_cast<size_t>(i)] = static_cast<double>(r + (i < f ? 1 : 0));
  std::make_heap(slot.begin(), slot.end(), std::greater<double>());
  for (int64_t i = 0; i < 2 * k; ++i) {
    std::pop_heap(slot.begin(), slot.end(), std::greater<double>());
    slot.back() += h;
    std::push_heap(slot.begin(), slot.end(), std::greater<double>());
  }
  return *std::max_element(slot.begin(), slot.end());
}

// Relative length of a 64-row block: half the MFMA and encode work, the same K/V streaming.
constexpr double kHalfBlockTime = 0.6;

// How many of each XCD's last 128-row blocks run as two 64-row blocks: the k in [0, min(nfull/8,
// 2 S)] with the smallest modelled makespan of the fullest XCD (the smallest such k), S = the
// XCD's block slots (CUs / 8 x blocks per CU). Cached per (nfull, S).
int64_t tail_split(int64_t nfull, int blocks_per_cu) {
  static std::mutex mu;
  static std::map<std::pair<int64_t, int>, int64_t> cache;
  int dev = 0, cus = 0;
  if (hipGetDevice(&dev) != hipSuccess || hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess ||
      cus < 8)
    return 0;
  const int S = cus / 8 * blocks_per_cu;
  std::lock_guard<std::mutex> lock(mu);
  const auto key = std::make_pair(nfull, S);
  const auto it = cache.find(key);
  if (it != cache.end()) return it->second;
  const int64_t per = nfull / 8, n = per + (nfull % 8 ? 1 : 0);
  int64_t best = 0;
  double best_t = list_makespan(n, 0, S, kHalfBlockTime);
  for (int64_t k = 1; k <= std::min<int64_t>(per, 2 * S); ++k) {
    const double t = list_makespan(n, k, S, kHalfBlockTime);
    if (t < best_t - 1e-9) { best_t = t; best = k; }
  }
  if (cache.size() >= 4096) cache.clear();  // a serving process sees a bounded set of shapes; stay small
  cache.emplace(key, best);
  return best;
}

template <int D, int VM, bool DUMP, int OUT, int PM, int QF>
int launch(const AttnArgs& a, hipStream_t st) {
  AttnArgs b = a;
  b.kconv = tail_split(a.nfull, kBlocksPerCU<D, VM>);
  const int64_t grid = b.nfull + 8 * b.kconv;
  attn_kernel<D, VM, DUMP, OUT, PM, QF><<<dim3(static_cast<unsigned>(grid)), kThreadsPerBlock, 0, st>>>(b);
  return check_launch("attn_kernel");
}

template <int D, int VM, int PM, int QF>
int launch_out(const AttnArgs& a, bool dump, int out_dtype, hipStream_t st) {
  if (dump) {
    return out_dtype == VCX_BFLOAT16 ? launch<D, VM, true, VCX_BFLOAT16, PM, QF>(a, st)
                                     : launch<D, VM, true, VCX_FLOAT16, PM, QF>(a, st);
  }
  return out_dtype == VCX_BFLOAT16 ? launch<D, VM, false, VCX_BFLOAT16, PM, QF>(a, st)
                                   : launch<D, VM, false, VCX_FLOAT16, PM, QF>(a, st);
}

template <int D, int VM, int QF = 0>
int launch_mode(const AttnArgs& a, bool dump, int out_dtype, int mode, hipStream_t st) {
  if constexpr (VM == 0) {
    if (mode == 2) return launch_out<D, VM, 2, QF>(a, dump, out_dtype, st);
  }
  return mode == 1 ? launch_out<D, VM, 1, QF>(a, dump, out_dtype, st)
                   : launch_out<D, VM, 0, QF>(a, dump, out_dtype, st);
}

// Argument checks shared by the INT8 and FP8 block entry points.
int check_common(int64_t B, int64_t H, int64_t Nq, int64_t Nk, int64_t D, int expcast, int out_dtype,
                 float sm_scale, void* out, int64_t o_sb, int64_t o_sh, int64_t o_sn, const uint8_t* p_dump,
                 int64_t p_row_begin, int64_t p_row_end) {
  VCX_REQUIRE(B >= 1 && H >= 1 && Nq >= 1 && Nk >= 1, "B, H, Nq, Nk must be positive");
  VCX_REQUIRE(D == 64 || D == 128, "D must be 64 or 128");
  VCX_REQUIRE(B * H <= 65535, "B*H exceeds 65535");
  VCX_REQUIRE(Nq < (int64_t(1) << 30) && Nk < (int64_t(1) << 30), "sequence too long");
  VCX_REQUIRE(cdiv(Nk, kTile) * kTile * D < (int64_t(1) << 31), "K/V payload of one head must be below 2 GiB");
  VCX_REQUIRE(expcast >= 0 && expcast <= 2, "expcast must be 0, 1 or 2");
  VCX_REQUIRE(out_dtype == VCX_FLOAT16 || out_dtype == VCX_BFLOAT16, "out_dtype must be float16 or bfloat16");
  VCX_REQUIRE(std::isfinite(sm_scale) && sm_scale > 0.0f, "sm_scale must be positive and finite FP32");
  VCX_REQUIRE(aligned(out, 8) && o_sb % 4 == 0 && o_sh % 4 == 0 && o_sn % 4 == 0 && o_sn >= D && o_sb >= 0 &&
                  o_sh >= 0,
              "out must be 8-byte aligned with strides that are multiples of 4 elements and sn >= D");
  if (p_dump) {
    VCX_REQUIRE(p_row_begin >= 0 && p_row_begin < p_row_end && p_row_end <= Nq, "invalid P dump row range");
  }
  return VCX_OK;
}

}  // namespace
}  // namespace vcx

using namespace vcx;

extern "C" int vcx_attention_fwd(const int8_t* q8, const int8_t* k8, const uint8_t* v8, const float* qs,
                                 const float* ks, const float* vs, const uint16_t* means, int64_t B,
                                 int64_t H, int64_t Nq, int64_t Nk, int64_t D, int expcast,
                                 int block_values, int channel_scale, float sm_scale, int out_dtype,
                                 void* out, int64_t o_sb, int64_t o_sh, int64_t o_sn, uint8_t* p_dump,
                                 int64_t p_row_begin, int64_t p_row_end, void* stream) {
  if (int rc = check_common(B, H, Nq, Nk, D, expcast, out_dtype, sm_scale, out, o_sb, o_sh, o_sn, p_dump,
                            p_row_begin, p_row_end))
    return rc;
  VCX_REQUIRE(expcast != 2 || !block_values, "the folded ExpCast encode (expcast = 2) is defined without block values");
  VCX_REQUIRE(block_values || channel_scale, "per-block V scales require block values (smoothing)");
  VCX_REQUIRE(q8 && k8 && v8 && qs && ks && vs && out, "null tensor pointer");
  VCX_REQUIRE(!block_values || means, "means must be non-null with block values");
  VCX_REQUIRE(aligned(q8, 16) && aligned(k8, 16) && aligned(v8, 16), "q8/k8/v8 must be 16-byte aligned");
  VCX_REQUIRE(aligned(qs, 4) && aligned(ks, 4) && aligned(vs, 16), "scale pointer alignment (vs needs 16 bytes)");
  VCX_REQUIRE(!block_values || aligned(means, 8), "means must be 8-byte aligned");
  AttnArgs a{};
  a.q8 = q8; a.k8 = k8; a.v8 = v8; a.qs = qs; a.ks = ks; a.vs = vs; a.means = means; a.out = out;
  a.osb = o_sb; a.osh = o_sh; a.osn = o_sn;
  a.H = H; a.Nq = Nq; a.Nk = Nk; a.tiles = cdiv(Nk, kTile); a.qblocks = cdiv(Nq, kRowsPerBlock);
  a.qs_len = cdiv(Nq, 64) * 32;
  // The control path works in the log2 domain: RN(sm * RN(log2 e)) (sal/csrc/vc/vc_sm90.cu:177).
  a.sm = expcast != 0 ? sm_scale : sm_scale * 1.4426950408889634f;
  a.pdump = p_dump; a.prow0 = p_row_begin; a.prow1 = p_row_end;
  const int64_t nblocks = B * H * a.qblocks;
  VCX_REQUIRE(nblocks < (int64_t(1) << 30), "too many blocks");
  a.nfull = nblocks;
  hipStream_t st = static_cast<hipStream_t>(stream);
  const bool dump = p_dump != nullptr;
  a.out_bf16 = out_dtype == VCX_BFLOAT16;
  const int vm = block_values ? (channel_scale ? 1 : 2) : 0;
  if (const int groups = piece_groups(B * H, Nq, a.tiles, D, vm, expcast, 0))
    return launch_pieces(a, B * H, D, groups, vm, expcast, 0, st);
  if (D == 128) {
    if (!block_values) return launch_mode<128, 0>(a, dump, out_dtype, expcast, st);
    return channel_scale ? launch_mode<128, 1>(a, dump, out_dtype, expcast, st)
                         : launch_mode<128, 2>(a, dump, out_dtype, expcast, st);
  }
  if (!block_values) return launch_mode<64, 0>(a, dump, out_dtype, expcast, st);
  return channel_scale ? launch_mode<64, 1>(a, dump, out_dtype, expcast, st)
                       : launch_mode<64, 2>(a, dump, out_dtype, expcast, st);
}

extern "C" int vcx_attention_fwd_fp8(const uint8_t* q8, const uint8_t* k8, const uint8_t* v8, const float* qs,
                                     const float* ks, const float* vs, int64_t B, int64_t H, int64_t Nq,
                                     int64_t Nk, int64_t D, int expcast, float sm_scale, int out_dtype, void* out,
                                     int64_t o_sb, int64_t o_sh, int64_t o_sn, uint8_t* p_dump,
                                     int64_t p_row_begin, int64_t p_row_end, void* stream) {
  if (int rc = check_common(B, H, Nq, Nk, D, expcast, out_dtype, sm_scale, out, o_sb, o_sh, o_sn, p_dump,
                            p_row_begin, p_row_end))
    return rc;
  VCX_REQUIRE(q8 && k8 && v8 && qs && ks && vs && out, "null tensor pointer");
  VCX_REQUIRE(aligned(q8, 16) && aligned(k8, 16) && aligned(v8, 16), "q8/k8/v8 must be 16-byte aligned");
  VCX_REQUIRE(aligned(qs, 4) && aligned(ks, 4) && aligned(vs, 16), "scale pointer alignment (vs needs 16 bytes)");
  AttnArgs a{};
  a.q8 = reinterpret_cast<const int8_t*>(q8); a.k8 = reinterpret_cast<const int8_t*>(k8); a.v8 = v8;
  a.qs = qs; a.ks = ks; a.vs = vs; a.means = nullptr; a.out = out;
  a.osb = o_sb; a.osh = o_sh; a.osn = o_sn;
  a.H = H; a.Nq = Nq; a.Nk = Nk; a.tiles = cdiv(Nk, kTile); a.qblocks = cdiv(Nq, kRowsPerBlock);
  a.qs_len = cdiv(Nq, 64);
  a.sm = expcast != 0 ? sm_scale : sm_scale * 1.4426950408889634f;
  a.pdump = p_dump; a.prow0 = p_row_begin; a.prow1 = p_row_end;
  const int64_t nblocks = B * H * a.qblocks;
  VCX_REQUIRE(nblocks < (int64_t(1) << 30), "too many blocks");
  a.nfull = nblocks;
  hipStream_t st = static_cast<hipStream_t>(stream);
  const bool dump = p_dump != nullptr;
  a.out_bf16 = out_dtype == VCX_BFLOAT16;
  if (const int groups = piece_groups(B * H, Nq, a.tiles, D, 0, expcast, 1))
    return launch_pieces(a, B * H, D, groups, 0, expcast, 1, st);
  return D == 128 ? launch_mode<128, 0, 1>(a, dump, out_dtype, expcast, st)
                  : launch_mode<64, 0, 1>(a, dump, out_dtype, expcast, st);
}

namespace vcx {
namespace {
// One thread per four inputs: the control path's probability bytes as Wave::bytes forms them
// (LIFT: in the general copy of the tile loop and in pieces; else in the copy with the cheap
// midpoint test).
template <bool LIFT>
__global__ void fp8_exp2_probe_kernel(const float* x, uint8_t* y, int64_t n) {
  const int64_t i = (static_cast<int64_t>(blockIdx.x) * blockDim.x + threadIdx.x) * 4;
  if (i >= n) return;
  float xs[4], pr[4];
#pragma unroll
  for (int r = 0; r < 4; ++r) {
    xs[r] = i + r < n ? x[i + r] : -INFINITY;
    pr[r] = __builtin_amdgcn_exp2f(xs[r]);
  }
  uint32_t gap = 0xffffffffu, w = fp8_exp2_quick<LIFT>(pr, gap);
  if (gap <= kFp8Gap) w = fp8_exp2_word(xs, pr);
#pragma unroll
  for (int r = 0; r < 4; ++r)
    if (i + r < n) y[i + r] = static_cast<uint8_t>(w >> (8 * r));
}
}  // namespace
}  // namespace vcx

extern "C" int vcx_fp8_exp2_codes(const float* x, uint8_t* y, int64_t n, int form, void* stream) {
  VCX_REQUIRE(n >= 0 && (n == 0 || (x != nullptr && y != nullptr)), "invalid probe arguments");
  VCX_REQUIRE(form == 0 || form == 1, "form must be 0 or 1");
  VCX_REQUIRE(aligned(x, 4), "x must be 4-byte aligned");
  if (n == 0) return VCX_OK;
  const int64_t threads = cdiv(n, 4), blocks = cdiv(threads, 256);
  VCX_REQUIRE(blocks < (int64_t(1) << 31), "n too large");
  if (form) fp8_exp2_probe_kernel<true><<<dim3(static_cast<unsigned>(blocks)), 256, 0, static_cast<hipStream_t>(stream)>>>(x, y, n);
  else fp8_exp2_probe_kernel<false><<<dim3(static_cast<unsigned>(blocks)), 256, 0, static_cast<hipStream_t>(stream)>>>(x, y, n);
  return check_launch("fp8_exp2_probe_kernel");
}

namespace {
int resources_of(const void* fn, int64_t* out) {
  hipFuncAttributes attr{};
  hipError_t e = hipFuncGetAttributes(&attr, fn);
  if (e != hipSuccess) return fail(VCX_EHIP, "hipFuncGetAttributes: %s", hipGetErrorString(e));
  out[0] = attr.numRegs;
  out[1] = 0;
  out[2] = static_cast<int64_t>(attr.sharedSizeBytes);
  out[3] = 0;
  out[4] = attr.maxThreadsPerBlock;
  out[5] = static_cast<int64_t>(attr.localSizeBytes);
  return VCX_OK;
}
}  // namespace

extern "C" int vcx_kernel_resources(int64_t D, int block_values, int64_t* out) {
  VCX_REQUIRE(out != nullptr, "out is null");
  VCX_REQUIRE(D == 64 || D == 128, "D must be 64 or 128");
  const void* fn;
  if (D == 128) fn = block_values ? reinterpret_cast<const void*>(&attn_kernel<128, 1, false, VCX_BFLOAT16, 1>)
                                  : reinterpret_cast<const void*>(&attn_kernel<128, 0, false, VCX_BFLOAT16, 2>);
  else fn = block_values ? reinterpret_cast<const void*>(&attn_kernel<64, 1, false, VCX_BFLOAT16, 1>)
                         : reinterpret_cast<const void*>(&attn_kernel<64, 0, false, VCX_BFLOAT16, 2>);
  return resources_of(fn, out);
}

namespace {
template <int D, int VM, int PM, int OUT>
const void* kernel_of() { return reinterpret_cast<const void*>(&attn_kernel<D, VM, false, OUT, PM>); }

template <int D, int OUT>
const void* kernel_of(int vm, int pm) {
  if (vm == 0) return pm == 2 ? kernel_of<D, 0, 2, OUT>() : pm == 1 ? kernel_of<D, 0, 1, OUT>() : kernel_of<D, 0, 0, OUT>();
  if (vm == 1) return pm == 1 ? kernel_of<D, 1, 1, OUT>() : kernel_of<D, 1, 0, OUT>();
  return pm == 1 ? kernel_of<D, 2, 1, OUT>() : kernel_of<D, 2, 0, OUT>();
}
}  // namespace

extern "C" int vcx_kernel_resources_mode(int64_t D, int value_mode, int expcast, int out_dtype, int64_t* out) {
  VCX_REQUIRE(out != nullptr, "out is null");
  VCX_REQUIRE(D == 64 || D == 128, "D must be 64 or 128");
  VCX_REQUIRE(value_mode >= 0 && value_mode <= 2, "value_mode must be 0, 1 or 2");
  VCX_REQUIRE(expcast >= 0 && expcast <= 2, "expcast must be 0, 1 or 2");
  VCX_REQUIRE(expcast != 2 || value_mode == 0, "the folded ExpCast encode (expcast = 2) is defined without block values");
  VCX_REQUIRE(out_dtype == VCX_FLOAT16 || out_dtype == VCX_BFLOAT16, "out_dtype must be float16 or bfloat16");
  const void* fn = D == 128 ? (out_dtype == VCX_BFLOAT16 ? kernel_of<128, VCX_BFLOAT16>(value_mode, expcast)
                                                         : kernel_of<128, VCX_FLOAT16>(value_mode, expcast))
                            : (out_dtype == VCX_BFLOAT16 ? kernel_of<64, VCX_BFLOAT16>(value_mode, expcast)
                                                         : kernel_of<64, VCX_FLOAT16>(value_mode, expcast));
  if (int rc = resources_of(fn, out)) return rc;
  int blocks = 0;
  hipError_t e = hipOccupancyMaxActiveBlocksPerMultiprocessor(&blocks, fn, kThreadsPerBlock, 0);
  if (e != hipSuccess) return fail(VCX_EHIP, "hipOccupancyMaxActiveBlocksPerMultiprocessor: %s", hipGetErrorString(e));
  out[6] = blocks;
  return VCX_OK;
}

extern "C" int vcx_kernel_resources_fp8(int64_t D, int expcast, int64_t* out) {
  VCX_REQUIRE(out != nullptr, "out is null");
  VCX_REQUIRE(D == 64 || D == 128, "D must be 64 or 128");
  const void* fn;
  if (D == 128) fn = expcast ? reinterpret_cast<const void*>(&attn_kernel<128, 0, false, VCX_BFLOAT16, 2, 1>)
                             : reinterpret_cast<const void*>(&attn_kernel<128, 0, false, VCX_BFLOAT16, 0, 1>);
  else fn = expcast ? reinterpret_cast<const void*>(&attn_kernel<64, 0, false, VCX_BFLOAT16, 2, 1>)
                    : reinterpret_cast<const void*>(&attn_kernel<64, 0, false, VCX_BFLOAT16, 0, 1>);
  return resources_of(fn, out);
}
