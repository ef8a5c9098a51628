// Preprocessing kernels for sageattn_vc on gfx950: K channel mean, Sage
// per-thread INT8 Q/K, V E4M3 (per-channel amax or 128-token block-mean
// smoothing), ExpCast and conversion probes, plus their C-ABI entry points.
//
// All kernels are HBM-bound streaming passes. A 128-token tile is handled by
// 256 threads: thread (kk = tid/16, c = tid%16) owns channels [c*CPT, c*CPT+CPT)
// (CPT = D/16) of the keys kk + 16*i, i = 0..7, loaded as one 16-byte (D128)
// or 8-byte (D64) vector per key. Every fp64 tile sum uses the same fixed
// tree: sequential over i, then lanes xor 16, xor 32, then (w0+w1)+(w2+w3).
#include "vcx_common.hpp"

#include <mutex>

namespace vcx {
namespace {

constexpr int kThreads = 256;

// A [B,H,N,D] tensor: pointer and element strides.
struct Strided {
  const void* p;
  int64_t sb, sh, sn;
};

template <int D>
struct Row {
  static constexpr int CPT = D / 16;  // channels per thread
  uint32_t w[CPT / 2];                // packed 16-bit inputs
};

// Load CPT 16-bit values of token `tok` (already permuted) for chunk c. NT: a
// non-temporal load, for a tensor read once (Q), so that it does not displace one that is
// read again soon (K between its statistics and quantization passes) from the
// memory-side cache.
template <int D, bool NT = false>
__device__ inline void load_row(const uint16_t* base, int64_t sn, int64_t tok, int c, Row<D>& r) {
  const uint16_t* p = base + tok * sn + c * Row<D>::CPT;
  typedef uint32_t v4u __attribute__((ext_vector_type(4)));
  typedef uint32_t v2u __attribute__((ext_vector_type(2)));
  if constexpr (D == 128) {
    const v4u v = NT ? __builtin_nontemporal_load(reinterpret_cast<const v4u*>(p)) : *reinterpret_cast<const v4u*>(p);
    r.w[0] = v.x; r.w[1] = v.y; r.w[2] = v.z; r.w[3] = v.w;
  } else {
    const v2u v = NT ? __builtin_nontemporal_load(reinterpret_cast<const v2u*>(p)) : *reinterpret_cast<const v2u*>(p);
    r.w[0] = v.x; r.w[1] = v.y;
  }
}

template <int DT, int D>
__device__ inline float row_val(const Row<D>& r, int j) {
  uint32_t bits = (r.w[j >> 1] >> ((j & 1) * 16)) & 0xffffu;
  return in_to_f32<DT>(bits);
}

__device__ inline int64_t source_token(const int64_t* perm, int64_t bh, int64_t n, int64_t key) {
  return perm ? perm[bh * n + key] : key;
}

// Rows of the NR keys key0 + 16*i (i < NR) of one head, for channel chunk c.
// All permutation lookups are issued first, then all row loads, so that their
// latencies overlap; a key past n loads row 0 and reads as zero.
template <int D, int NR>
__device__ inline void load_key_rows_packed(const uint16_t* base, int64_t sn, const int64_t* perm, int64_t bh,
                                            int64_t n, int64_t key0, int c, Row<D> (&r)[NR]) {
  int64_t src[NR];
#pragma unroll
  for (int i = 0; i < NR; ++i) {
    const int64_t key = key0 + 16 * i;
    src[i] = key < n ? source_token(perm, bh, n, key) : 0;
  }
#pragma unroll
  for (int i = 0; i < NR; ++i) load_row<D>(base, sn, src[i], c, r[i]);
}

// Per-head base pointer of a strided [B,H,N,D] tensor.
__device__ inline const uint16_t* head_base(const void* x, int64_t bh, int64_t H, int64_t sb, int64_t sh) {
  int64_t b = bh / H, h = bh % H;
  return reinterpret_cast<const uint16_t*>(x) + b * sb + h * sh;
}

// Fixed fp64 tree over the 16 key-lanes of a tile (see file header). `red` is
// LDS [4][D]; the result for channel ch is returned to threads tid < D.
template <int D>
__device__ inline void tile_tree(double (&a)[D / 16], double* red, double* out_ch) {
  constexpr int CPT = D / 16;
  int tid = threadIdx.x, lane = tid & 63, w = tid >> 6, c = tid & 15;
#pragma unroll
  for (int j = 0; j < CPT; ++j) {
    a[j] = add_xor32(add_xor16(a[j]));
  }
  if (lane < 16)
#pragma unroll
    for (int j = 0; j < CPT; ++j) red[w * D + c * CPT + j] = a[j];
  __syncthreads();
  if (tid < D) *out_ch = (red[tid] + red[D + tid]) + (red[2 * D + tid] + red[3 * D + tid]);
}

// One thread's INT8 (or FP8) payload piece (CPT bytes) as a non-temporal store: the payload goes to
// HBM now instead of staying dirty in the memory-side cache, where the next streaming pass's
// reads would pay for evicting it.
template <int CPT>
__device__ inline void store_payload_nt(void* dst, const uint32_t* packed) {
  typedef uint32_t v2u __attribute__((ext_vector_type(2)));
  if constexpr (CPT == 8) __builtin_nontemporal_store(v2u{packed[0], packed[1]}, reinterpret_cast<v2u*>(dst));
  else __builtin_nontemporal_store(packed[0], reinterpret_cast<uint32_t*>(dst));
}

// ---------------------------------------------------------------- tile statistics

enum StatsMode { kKSum = 0, kVAmax = 1, kVSmooth = 2 };

// grid (tiles, B*H), 256 threads.
//  kKSum:    sum[bh][tile][ch] = fp64 tile-tree sum of K
//  kVAmax:   amax[bh][tile][ch] = max |V|
//  kVSmooth: mean[bh][tile][ch] = RN_f32(tile-tree sum / count),
//            peak[bh][tile][ch] = max |RN(V - mean)| over valid tokens
template <int DT, int D, int MODE>
__device__ __forceinline__ void tile_stats_body(const Strided& t, int64_t H, int64_t n, const int64_t* perm,
                                                double* sum_out, float* f_out0, float* f_out1, int64_t tile,
                                                int64_t bh, int64_t tiles) {
  const void* x = t.p;
  const int64_t sb = t.sb, sh = t.sh, sn = t.sn;
  constexpr int CPT = D / 16;
  __shared__ double red[4 * D];
  __shared__ float fred[4 * D];
  __shared__ float mean_sh[D];
  const int tid = threadIdx.x, kk = tid >> 4, c = tid & 15, lane = tid & 63, w = tid >> 6;
  const uint16_t* base = head_base(x, bh, H, sb, sh);
  // the rows stay packed (16-bit values) and are widened where used: the smoothing
  // statistics read them twice, and packed they take half the registers
  Row<D> rows[8];
  load_key_rows_packed<D, 8>(base, sn, perm, bh, n, tile * kTile + kk, c, rows);
  // Keys past n, which only the last tile has, read as zero. The smoothing statistics, which read
  // every value twice, clear the packed rows of such a tile and spare the others the selects
  // ([1,28,20000,64] fp16 prepare_v with block scales 42.2 -> 39.1 us); one pass is shorter with them.
  const bool full = (tile + 1) * kTile <= n;
  if (MODE == kVSmooth && !full) {
#pragma unroll
    for (int i = 0; i < 8; ++i)
#pragma unroll
      for (int k = 0; k < CPT / 2; ++k) rows[i].w[k] = tile * kTile + kk + 16 * i < n ? rows[i].w[k] : 0u;
  }
  auto v = [&](int i, int j) -> float {
    return MODE == kVSmooth || tile * kTile + kk + 16 * i < n ? row_val<DT, D>(rows[i], j) : 0.0f;
  };
  const int64_t meta = (bh * tiles + tile) * D;
  if constexpr (MODE == kVAmax) {
    float m[CPT];
#pragma unroll
    for (int j = 0; j < CPT; ++j) {
      m[j] = 0.0f;
#pragma unroll
      for (int i = 0; i < 8; ++i) m[j] = fmaxf(m[j], fabsf(v(i, j)));
      m[j] = max_xor32(max_xor16(m[j]));
    }
    if (lane < 16)
#pragma unroll
      for (int j = 0; j < CPT; ++j) fred[w * D + c * CPT + j] = m[j];
    __syncthreads();
    if (tid < D) f_out0[meta + tid] = fmaxf(fmaxf(fred[tid], fred[D + tid]), fmaxf(fred[2 * D + tid], fred[3 * D + tid]));
    return;
  } else {
    double a[CPT];
#pragma unroll
    for (int j = 0; j < CPT; ++j) {
      a[j] = 0.0;
#pragma unroll
      for (int i = 0; i < 8; ++i) a[j] = __dadd_rn(a[j], static_cast<double>(v(i, j)));
    }
    double total;
    tile_tree<D>(a, red, &total);
    if constexpr (MODE == kKSum) {
      if (tid < D) sum_out[meta + tid] = total;
      return;
    } else {
      const int64_t count = n - tile * kTile < kTile ? n - tile * kTile : kTile;
      if (tid < D) {
        float mu = static_cast<float>(__ddiv_rn(total, static_cast<double>(count)));
        mean_sh[tid] = mu;
        f_out0[meta + tid] = mu;
      }
      __syncthreads();
      // widen the packed rows again rather than keep the first pass's floats live
#pragma unroll
      for (int i = 0; i < 8; ++i)
#pragma unroll
        for (int k = 0; k < CPT / 2; ++k) asm volatile("" : "+v"(rows[i].w[k]));
      float pk[CPT];
      auto peaks = [&](auto masked) {
#pragma unroll
        for (int j = 0; j < CPT; ++j) {
          float mu = mean_sh[c * CPT + j];
          pk[j] = 0.0f;
#pragma unroll
          for (int i = 0; i < 8; ++i)
            if (!decltype(masked)::value || tile * kTile + kk + 16 * i < n)
              pk[j] = fmaxf(pk[j], fabsf(__fsub_rn(v(i, j), mu)));
        }
      };
      if (full) peaks(std::false_type());
      else peaks(std::true_type());
#pragma unroll
      for (int j = 0; j < CPT; ++j) pk[j] = max_xor32(max_xor16(pk[j]));
      if (lane < 16)
#pragma unroll
        for (int j = 0; j < CPT; ++j) fred[w * D + c * CPT + j] = pk[j];
      __syncthreads();
      if (tid < D)
        f_out1[meta + tid] = fmaxf(fmaxf(fred[tid], fred[D + tid]), fmaxf(fred[2 * D + tid], fred[3 * D + tid]));
    }
  }
}

template <int DT, int D, int MODE>
__global__ __launch_bounds__(kThreads) void tile_stats_kernel(Strided x, int64_t H, int64_t n, const int64_t* perm,
                                                              double* sum_out, float* f_out0, float* f_out1) {
  tile_stats_body<DT, D, MODE>(x, H, n, perm, sum_out, f_out0, f_out1, blockIdx.x, blockIdx.y, gridDim.x);
}

// The statistics of K (z = 0) and V (z = 1) in one launch: grid (tiles, B*H, 2).
template <int DT, int D, int VMODE>
__global__ __launch_bounds__(kThreads) void kv_stats_kernel(Strided k, Strided v, int64_t H, int64_t n,
                                                            const int64_t* perm, double* ksum, float* v0, float* v1) {
  if (blockIdx.z == 0)
    tile_stats_body<DT, D, kKSum>(k, H, n, perm, ksum, nullptr, nullptr, blockIdx.x, blockIdx.y, gridDim.x);
  else
    tile_stats_body<DT, D, VMODE>(v, H, n, perm, nullptr, v0, v1, blockIdx.x, blockIdx.y, gridDim.x);
}

// ---------------------------------------------------------------- finalize

// One thread per channel of head bh. km = RN_in(RN_f32(sum over tiles / n)); also the
// widened value for the K quantizer and, optionally, the caller's km_out.
// RAW (FP8 block path, vc27): km = RN_f32(sum / n), written to km_f32 and, as binary32,
// to the caller's km_out.
template <int DT, bool RAW = false>
__device__ inline void k_mean_body(const double* sums, int64_t tiles, int64_t n, int D, float* km_f32,
                                   void* km_out, int64_t bh, int ch) {
  const double* col = sums + bh * tiles * D + ch;
  // Sequential fp64 sum over tiles (the contract's order); the loads of a batch
  // of tiles are issued together so that their latencies overlap.
  constexpr int kBatch = 16;
  double s = 0.0;
  int64_t t = 0;
  for (; t + kBatch <= tiles; t += kBatch) {
    double v[kBatch];
#pragma unroll
    for (int i = 0; i < kBatch; ++i) v[i] = col[(t + i) * D];
#pragma unroll
    for (int i = 0; i < kBatch; ++i) s = __dadd_rn(s, v[i]);
  }
  if (t < tiles) {  // the partial last batch, its loads issued together too
    double v[kBatch];
#pragma unroll
    for (int i = 0; i < kBatch; ++i) v[i] = col[(t + i < tiles ? t + i : t) * D];
#pragma unroll
    for (int i = 0; i < kBatch; ++i)
      if (t + i < tiles) s = __dadd_rn(s, v[i]);
  }
  float mean = static_cast<float>(__ddiv_rn(s, static_cast<double>(n)));
  if constexpr (RAW) {
    km_f32[bh * D + ch] = mean;
    if (km_out) static_cast<float*>(km_out)[bh * D + ch] = mean;
  } else {
    uint32_t bits = f32_to_in<DT>(mean);
    km_f32[bh * D + ch] = in_to_f32<DT>(bits);
    if (km_out) static_cast<uint16_t*>(km_out)[bh * D + ch] = static_cast<uint16_t>(bits);
  }
}

// grid (B*H), D * S threads (S = 1024 / D slices of the tiles). Smoothing off: vs =
// RN(amax/448), recip = RN(448/amax) (0 for a zero channel). Smoothing on (channel scale):
// vs = max(P>0 ? RN(P/448) : 1, RN(M/65504)). Every quantity is a maximum, which no order
// changes: each thread takes the maximum over its slice of tiles (loads batched), and slice 0
// combines the slices from LDS.
constexpr int kScaleThreads = 1024;
template <bool SMOOTH, int THREADS>
__device__ __forceinline__ void v_scale_body(const float* a0, const float* a1, int64_t tiles, int D, float* vs,
                                             float* recip, int64_t bh) {
  __shared__ float red[2][THREADS];
  const int ch = threadIdx.x % D, sl = threadIdx.x / D, S = THREADS / D;
  const float* c0 = a0 + bh * tiles * D + ch;
  const float* c1 = SMOOTH ? a1 + bh * tiles * D + ch : nullptr;
  constexpr int kBatch = 8;
  float m0 = 0.0f, m1 = 0.0f;  // smoothing off: amax; on: M (|mean|) and P (peak)
  // batches of kBatch tiles of this slice, the last one partial (a missing tile repeats the
  // batch's first, which no maximum changes), all loads issued together
  for (int64_t t = sl; t < tiles; t += kBatch * S) {
    float v0[kBatch], v1[kBatch];
#pragma unroll
    for (int i = 0; i < kBatch; ++i) {
      const int64_t ti = t + i * S < tiles ? t + i * S : t;  // a missing tile repeats tile t
      v0[i] = c0[ti * D];
      if constexpr (SMOOTH) v1[i] = c1[ti * D];
    }
#pragma unroll
    for (int i = 0; i < kBatch; ++i) {
      if constexpr (SMOOTH) {
        m0 = fmaxf(m0, fabsf(v0[i]));
        m1 = fmaxf(m1, v1[i]);
      } else {
        m0 = fmaxf(m0, v0[i]);
      }
    }
  }
  red[0][threadIdx.x] = m0;
  red[1][threadIdx.x] = m1;
  __syncthreads();
  if (sl != 0) return;
  for (int k = 1; k < S; ++k) {
    m0 = fmaxf(m0, red[0][k * D + ch]);
    m1 = fmaxf(m1, red[1][k * D + ch]);
  }
  if constexpr (!SMOOTH) {
    vs[bh * D + ch] = m0 > 0.0f ? __fdiv_rn(m0, 448.0f) : 0.0f;
    recip[bh * D + ch] = m0 > 0.0f ? __fdiv_rn(448.0f, m0) : 0.0f;
  } else {
    const float sc = m1 > 0.0f ? __fdiv_rn(m1, 448.0f) : 1.0f;
    vs[bh * D + ch] = fmaxf(sc, __fdiv_rn(m0, 65504.0f));
  }
}

template <bool SMOOTH>
__global__ __launch_bounds__(kScaleThreads) void v_scale_kernel(const float* a0, const float* a1, int64_t tiles,
                                                                int D, float* vs, float* recip) {
  v_scale_body<SMOOTH, kScaleThreads>(a0, a1, tiles, D, vs, recip, blockIdx.x);
}

// ---------------------------------------------------------------- Q INT8

// grid (ceil(n/64), B*H), 256 threads. Groups of rows {16g+t, 16g+t+8}; each
// group is 32 lanes (16 per row) of one wave; 4 passes of 8 groups.
// ROT: the rows are rotated by the normalized Hadamard transform (hadamard_row, norm =
// RN_f32(1/sqrt(D))) in binary32 before the group maximum and the codes.
// quant_q_kernel's blocks (0, bh) instead compute head bh's K mean (k_mean_body, from the K tile
// sums of the statistics launch before), so that this latency-bound walk runs beside the
// streaming Q blocks instead of in a launch of its own; the Q blocks are (1 + blk, bh). The K
// quantization launch that follows reads the mean.
struct KMeanArgs {
  const double* sums;
  int64_t tiles, n;
  float* km;
  void* km_out;
};

template <int DT, int D, bool ROT>
__device__ __forceinline__ void quant_q_body(const Strided& q, int64_t H, int64_t n, int8_t* q8, float* qs, float norm,
                                             int64_t blk, int64_t bh) {
  constexpr int CPT = D / 16;
  const int tid = threadIdx.x, lane = tid & 63, w = tid >> 6, c = lane & 15, sel = (lane >> 4) & 1;
  const int64_t sn = q.sn;
  const uint16_t* base = head_base(q.p, bh, H, q.sb, q.sh);
  const int64_t qs_len = (n + 63) / 64 * 32;
  // The four rows of the thread are loaded together before any is used.
  Row<D> rows[4];
#pragma unroll
  for (int pass = 0; pass < 4; ++pass) {
    const int grp = pass * 8 + w * 2 + (lane >> 5);
    const int64_t row = blk * 64 + 16 * (grp >> 3) + (grp & 7) + 8 * sel;
    load_row<D, true>(base, sn, row < n ? row : 0, c, rows[pass]);
  }
#pragma unroll
  for (int pass = 0; pass < 4; ++pass) {
    const int grp = pass * 8 + w * 2 + (lane >> 5);  // 0..31 inside the 64-row block
    const int g = grp >> 3, t = grp & 7;
    const int64_t row = blk * 64 + 16 * g + t + 8 * sel;
    float x[CPT];
#pragma unroll
    for (int j = 0; j < CPT; ++j) x[j] = row < n ? row_val<DT, D>(rows[pass], j) : 0.0f;
    if constexpr (ROT) hadamard_row<CPT, 16>(x, c, norm);
    float amax = 0.0f;
#pragma unroll
    for (int j = 0; j < CPT; ++j) amax = fmaxf(amax, fabsf(x[j]));
    amax = half_wave_max(amax);
    const float s = int8_scale(amax), rs = recip_rn(s);
    if (row < n) {
      uint32_t packed[CPT / 4];
#pragma unroll
      for (int j = 0; j < CPT / 4; ++j) packed[j] = int8_codes4(&x[4 * j], s, rs);
      int8_t* dst = q8 + (bh * n + row) * D + c * CPT;
      store_payload_nt<CPT>(dst, packed);
    }
    if ((lane & 31) == 0) qs[bh * qs_len + (blk * 4 + g) * 8 + t] = s;
  }
}

template <int DT, int D, bool ROT>
__global__ __launch_bounds__(kThreads) void quant_q_kernel(Strided q, int64_t H, int64_t n, int8_t* q8, float* qs,
                                                           float norm, KMeanArgs kma) {
  if (blockIdx.x == 0) {
    if (threadIdx.x < D) k_mean_body<DT>(kma.sums, kma.tiles, kma.n, D, kma.km, kma.km_out, blockIdx.y, threadIdx.x);
    return;
  }
  quant_q_body<DT, D, ROT>(q, H, n, q8, qs, norm, blockIdx.x - 1, blockIdx.y);
}

// ---------------------------------------------------------------- FP8 block Q/K (vc27)

// grid (ceil(n/ROWS), B*H), 256 threads; one block of ROWS rows x D channels shares one
// scale. Thread (rr = tid/16, c = tid%16) holds channels [c*CPT, c*CPT+CPT) of the rows
// blk*ROWS + rr + 16*i. x' = CENTER ? RN(x - km) : x (binary32); s = max(RN(amax/448), 1e-12);
// code = E4M3_satfinite(RN(x'/s)). Rows past n are not part of the block.
// Reference: quantize_qk_fp8, sal/csrc/vc/qk_fp8.cu:38-74 (Q: 64 rows; K: 128 rows, centred).
// The Q launch's blocks (0, h) instead compute head h's K mean km = RN_f32(sum / n) from the K
// statistics (the FP8 path's unrounded mean), so that walk runs beside the Q blocks.
template <int DT, int D, int ROWS, bool CENTER>
__device__ __forceinline__ void quant_fp8_body(const Strided& x, int64_t H, int64_t n, const float* km, uint8_t* codes,
                                               float* scales, int64_t blk, int64_t bh, int64_t blocks) {
  constexpr int CPT = D / 16, NR = ROWS / 16;
  __shared__ float wmax[kThreads / 64];
  const int tid = threadIdx.x, rr = tid >> 4, c = tid & 15, lane = tid & 63, w = tid >> 6;
  const int64_t sn = x.sn;
  const uint16_t* base = head_base(x.p, bh, H, x.sb, x.sh);
  // Every row of the thread is loaded before any is used; Q (read once) non-temporally, so
  // that K stays in the memory-side cache for its own pass.
  Row<D> rows[NR];
#pragma unroll
  for (int i = 0; i < NR; ++i) {
    const int64_t row = blk * ROWS + rr + 16 * i;
    load_row<D, !CENTER>(base, sn, row < n ? row : 0, c, rows[i]);
  }
  // The compiler moves some of bf16 D128's loads behind the first uses without this (other types and
  // widths are as fast or faster without): prepare_qk_fp8 [1,28,20000,128] 103.7 us so, 100.8 with it.
  if constexpr (D == 128 && DT == VCX_BFLOAT16) __builtin_amdgcn_sched_barrier(0);
  float mean[CPT];
#pragma unroll
  for (int j = 0; j < CPT; ++j) mean[j] = CENTER ? km[bh * D + c * CPT + j] : 0.0f;
  float v[NR][CPT];
  float amax = 0.0f;
#pragma unroll
  for (int i = 0; i < NR; ++i) {
    const bool valid = blk * ROWS + rr + 16 * i < n;
#pragma unroll
    for (int j = 0; j < CPT; ++j) {
      float y = valid ? row_val<DT, D>(rows[i], j) : 0.0f;
      if constexpr (CENTER) y = valid ? __fsub_rn(y, mean[j]) : 0.0f;
      v[i][j] = y;
      amax = fmaxf(amax, fabsf(y));
    }
  }
  amax = max_xor32(half_wave_max(amax));
  if (lane == 0) wmax[w] = amax;
  __syncthreads();
  amax = fmaxf(fmaxf(wmax[0], wmax[1]), fmaxf(wmax[2], wmax[3]));
  const float s = fmaxf(__fdiv_rn(amax, 448.0f), 1e-12f);
  if (tid == 0) scales[bh * blocks + blk] = s;
#pragma unroll
  for (int i = 0; i < NR; ++i) {
    const int64_t row = blk * ROWS + rr + 16 * i;
    if (row >= n) continue;
    uint32_t packed[CPT / 4];
#pragma unroll
    for (int j = 0; j < CPT / 4; ++j) {
      float y[4];
#pragma unroll
      for (int e = 0; e < 4; ++e) y[e] = fminf(448.0f, fmaxf(-448.0f, __fdiv_rn(v[i][4 * j + e], s)));
      int wv = __builtin_amdgcn_cvt_pk_fp8_f32(y[0], y[1], 0, false);
      packed[j] = static_cast<uint32_t>(__builtin_amdgcn_cvt_pk_fp8_f32(y[2], y[3], wv, true));
    }
    uint8_t* dst = codes + (bh * n + row) * D + c * CPT;
    store_payload_nt<CPT>(dst, packed);
  }
}

template <int DT, int D>
__global__ __launch_bounds__(kThreads) void quant_fp8_q_kernel(Strided q, int64_t H, int64_t n, uint8_t* codes,
                                                               float* scales, KMeanArgs kma) {
  if (blockIdx.x == 0) {
    if (threadIdx.x < D) k_mean_body<DT, true>(kma.sums, kma.tiles, kma.n, D, kma.km, kma.km_out, blockIdx.y, threadIdx.x);
    return;
  }
  quant_fp8_body<DT, D, 64, false>(q, H, n, nullptr, codes, scales, blockIdx.x - 1, blockIdx.y, gridDim.x - 1);
}
template <int DT, int D>
__global__ __launch_bounds__(kThreads) void quant_fp8_k_kernel(Strided k, int64_t H, int64_t n, const float* km,
                                                               uint8_t* codes, float* scales) {
  quant_fp8_body<DT, D, 128, true>(k, H, n, km, codes, scales, blockIdx.x, blockIdx.y, gridDim.x);
}

// ---------------------------------------------------------------- generic Q/K preprocessing

// The reference's preprocess_qk (csrc/bindings.cpp:87-116, kernels.cu:104-123): fp32/fp16/bf16
// [B,H,N,D] with D <= 128 (any), widened to binary32; K centred by its binary32 channel mean;
// Q and K optionally rotated (width W = next power of two >= D, zero padded).
template <int DT>
__device__ inline float elem(const void* x, int64_t i) {
  if constexpr (DT == VCX_FLOAT32) return static_cast<const float*>(x)[i];
  else return in_to_f32<DT>(static_cast<const uint16_t*>(x)[i]);
}

// Four adjacent elements from element index i (on a four-element boundary), widened.
template <int DT>
__device__ inline void load_quad(const void* x, int64_t i, float (&v)[4]) {
  if constexpr (DT == VCX_FLOAT32) {
    const float4 q = *reinterpret_cast<const float4*>(static_cast<const float*>(x) + i);
    v[0] = q.x, v[1] = q.y, v[2] = q.z, v[3] = q.w;
  } else {
    const uint2 q = *reinterpret_cast<const uint2*>(static_cast<const uint16_t*>(x) + i);
    v[0] = in_to_f32<DT>(q.x & 0xffffu), v[1] = in_to_f32<DT>(q.x >> 16);
    v[2] = in_to_f32<DT>(q.y & 0xffffu), v[3] = in_to_f32<DT>(q.y >> 16);
  }
}

// Blocks of pre_rows_kernel along the grid's x; more of them go on along z, as the threads along
// one axis stay below 2^32.
constexpr int64_t kRowsGridX = int64_t(1) << 22;

// grid (tiles, B*H), D threads: binary64 sum of channel d over the tile's keys in key order, the
// loads of 16 keys in flight. One-wave blocks of four channels per thread, which move 8 or 16 bytes per
// load, are no faster at any size (centring and rotation at [1,28,37741,128] bf16: 332 us with either)
// and slower the fewer the tiles, as a lane's chain of additions is four times as long ([1,2,1000,64]
// 13.9 us with these, 8.6 us so; [1,24,16001,64] 64.8 and 59.3 us).
template <int DT>
__global__ __launch_bounds__(128) void pre_tile_sum_kernel(const void* x, int64_t H, int64_t n, int64_t sb,
                                                           int64_t sh, int64_t sn, double* part) {
  const int64_t t = blockIdx.x, bh = blockIdx.y, tiles = gridDim.x;
  const int d = threadIdx.x, D = blockDim.x;
  const int64_t off = (bh / H) * sb + (bh % H) * sh + d;
  const int64_t r0 = t * kTile, r1 = r0 + kTile < n ? r0 + kTile : n;
  constexpr int kBatch = 16;
  double s = 0.0;
  int64_t r = r0;
  for (; r + kBatch <= r1; r += kBatch) {
    float v[kBatch];
#pragma unroll
    for (int i = 0; i < kBatch; ++i) v[i] = elem<DT>(x, off + (r + i) * sn);
#pragma unroll
    for (int i = 0; i < kBatch; ++i) s = __dadd_rn(s, static_cast<double>(v[i]));
  }
  for (; r < r1; ++r) s = __dadd_rn(s, static_cast<double>(elem<DT>(x, off + r * sn)));
  part[(bh * tiles + t) * D + d] = s;
}

// grid (ceil(n / RPB) (+ 1 with KM), B*H): out = x - mean (mean nullable), rotated with ROT,
// [B*H][n][ROT ? W : D] binary32. L = min(W, 16) lanes hold a row, CPT = W / L entries each (two
// groups of four at W = 128, see hadamard_row), and a thread takes NR rows of the block's RPB, their
// loads issued before any is used; the mean's entries are loaded once.
// WIDE: D = W and every row starts on four elements, so entries move four at a time (8 or 16
// byte loads, 16-byte stores), without it one by one. The kernel streams: at [1,28,37741,128]
// bf16 one row and one-entry loads per thread took 230 us for Q and 442 us with the mean, this
// form 148 and 139 us (5.8 TB/s).
// Outputs in 16-byte pieces go past the caches (non-temporal), so that K stays in the memory-side
// cache between its sums and this pass. One by one without rotation, adjacent lanes take adjacent
// entries ([1,24,37741,72] bf16: 382 us with four adjacent entries per lane, 198 us so).
// KM (Q's launch): blocks (0, bh) form head bh's K mean instead, beside the Q rows.
template <int DT, int W, bool ROT, bool WIDE, bool KM, int NR>
__global__ __launch_bounds__(kThreads) void pre_rows_kernel(const void* x, int64_t H, int64_t n, int D, int64_t sb,
                                                            int64_t sh, int64_t sn, const float* mean, float* out,
                                                            float norm, KMeanArgs kma) {
  int64_t blk = blockIdx.z * kRowsGridX + blockIdx.x;
  if constexpr (KM) {
    if (blk-- == 0) {
      if (static_cast<int>(threadIdx.x) < D)
        k_mean_body<VCX_BFLOAT16, true>(kma.sums, kma.tiles, kma.n, D, kma.km, nullptr, blockIdx.y, threadIdx.x);
      return;
    }
  }
  constexpr int L = W < 16 ? W : 16, CPT = W / L, RPB = kThreads / L * NR;
  constexpr bool SPLIT = W == 128;
  const int tid = threadIdx.x, c = tid % L;
  const int64_t bh = blockIdx.y, r0 = blk * RPB + tid / L;
  const int64_t head = (bh / H) * sb + (bh % H) * sh;
  auto channel = [&](int j) { return !ROT && !WIDE ? c + L * j : SPLIT ? 4 * c + (j & 3) + 64 * (j >> 2) : c * CPT + j; };
  float v[NR][CPT];
#pragma unroll
  for (int i = 0; i < NR; ++i) {
    const int64_t r = r0 + i * (kThreads / L), off = head + (r < n ? r : 0) * sn;
    if constexpr (WIDE) {
#pragma unroll
      for (int j = 0; j < CPT; j += 4) load_quad<DT>(x, off + channel(j), reinterpret_cast<float(&)[4]>(v[i][j]));
    } else {
#pragma unroll
      for (int j = 0; j < CPT; ++j) v[i][j] = channel(j) < D ? elem<DT>(x, off + channel(j)) : 0.0f;
    }
  }
  if (mean != nullptr) {
    float mu[CPT];
#pragma unroll
    for (int j = 0; j < CPT; ++j) mu[j] = channel(j) < D ? mean[bh * D + channel(j)] : 0.0f;
#pragma unroll
    for (int i = 0; i < NR; ++i)
#pragma unroll
      for (int j = 0; j < CPT; ++j) v[i][j] = __fsub_rn(v[i][j], mu[j]);
  }
  const int64_t width = ROT ? W : D;
#pragma unroll
  for (int i = 0; i < NR; ++i) {
    if constexpr (ROT) hadamard_row<CPT, L, SPLIT>(v[i], c, norm);
    const int64_t r = r0 + i * (kThreads / L);
    if (r >= n) continue;
    float* dst = out + (bh * n + r) * width;
    if constexpr (WIDE) {
#pragma unroll
      for (int j = 0; j < CPT; j += 4) {
        typedef float v4f __attribute__((ext_vector_type(4)));
        __builtin_nontemporal_store(v4f{v[i][j], v[i][j + 1], v[i][j + 2], v[i][j + 3]},
                                    reinterpret_cast<v4f*>(dst + channel(j)));
      }
    } else {
#pragma unroll
      for (int j = 0; j < CPT; ++j)
        if (channel(j) < width) dst[channel(j)] = v[i][j];
    }
  }
}

// ---------------------------------------------------------------- K INT8

// grid (tiles, B*H), 256 threads. Thread (kk, c) holds keys kk+16i, all in
// scale group g = (kk%8)/2; a group is lanes 0-31 or 32-63 of waves w and w+2.
// ROT: each centred key row k'' is rotated (hadamard_row) in binary32 before quantizing.
template <int DT, int D, bool ROT>
__device__ __forceinline__ void quant_k_body(const Strided& k, int64_t H, int64_t n, const int64_t* perm,
                                             const float* km, int8_t* k8, float* ks, float norm, int64_t tile,
                                             int64_t bh, int64_t tiles) {
  constexpr int CPT = D / 16;
  __shared__ float gred[4][2];
  const int tid = threadIdx.x, kk = tid >> 4, c = tid & 15, lane = tid & 63, w = tid >> 6;
  const int64_t sn = k.sn;
  const uint16_t* base = head_base(k.p, bh, H, k.sb, k.sh);
  float mean[CPT];
#pragma unroll
  for (int j = 0; j < CPT; ++j) mean[j] = km[bh * D + c * CPT + j];
  Row<D> rows[8];
  load_key_rows_packed<D, 8>(base, sn, perm, bh, n, tile * kTile + kk, c, rows);
  float v[8][CPT];
  float amax = 0.0f;
#pragma unroll
  for (int i = 0; i < 8; ++i) {
    const uint32_t keep = tile * kTile + kk + 16 * i < n ? ~0u : 0u;  // keys past n read as zero
#pragma unroll
    for (int j = 0; j < CPT; ++j)
      v[i][j] = __uint_as_float(__float_as_uint(round_in<DT>(__fsub_rn(row_val<DT, D>(rows[i], j), mean[j]))) & keep);
    if constexpr (ROT) hadamard_row<CPT, 16>(v[i], c, norm);
#pragma unroll
    for (int j = 0; j < CPT; ++j) amax = fmaxf(amax, fabsf(v[i][j]));
  }
  amax = half_wave_max(amax);
  if ((lane & 31) == 0) gred[w][lane >> 5] = amax;
  __syncthreads();
  amax = fmaxf(gred[w][lane >> 5], gred[w ^ 2][lane >> 5]);
  const float s = int8_scale(amax), rs = recip_rn(s);
  const int g = (kk & 7) >> 1;
  if (w < 2 && (lane & 31) == 0) ks[bh * tiles * 4 + tile * 4 + g] = s;
#pragma unroll
  for (int i = 0; i < 8; ++i) {
    int64_t key = tile * kTile + kk + 16 * i;
    if (key >= n) continue;
    uint32_t packed[CPT / 4];
#pragma unroll
    for (int j = 0; j < CPT / 4; ++j) packed[j] = int8_codes4(&v[i][4 * j], s, rs);
    int8_t* dst = k8 + (bh * n + key) * D + c * CPT;
    store_payload_nt<CPT>(dst, packed);
  }
}

// (head, tile) in the reverse order of the statistics pass, so that the rows that pass read
// last are still in the memory-side cache when this pass starts.
template <int DT, int D, bool ROT>
__global__ __launch_bounds__(kThreads) void quant_k_kernel(Strided k, int64_t H, int64_t n, const int64_t* perm,
                                                           const float* km, int8_t* k8, float* ks, float norm) {
  quant_k_body<DT, D, ROT>(k, H, n, perm, km, k8, ks, norm, gridDim.x - 1 - blockIdx.x, gridDim.y - 1 - blockIdx.y,
                           gridDim.x);
}

// ---------------------------------------------------------------- V E4M3

// grid (tiles, B*H), 256 threads. Bytes are staged in LDS as [D][128] storage
// positions, then written as 16-byte rows of the [D][tiles*128] payload.
// Thread (m, cg) owns storage dword m (positions 4m..4m+3, i.e. the four tokens
// 16(m%8) + 2(m/8) + {0, 1, 8, 9}) for the D/8 channels of group cg, so it
// packs four bytes per channel into one LDS dword; 16-byte chunks of a staged
// row are XOR-swizzled by the channel group to spread the stores over banks.
//  SMOOTH = 0: byte = e4m3(RN(x * recip[ch])), zero channel -> 0.
//  SMOOTH = 1: byte = e4m3(RN(RN(x - mean_t) / s)), with s the channel scale
//              (CHANNEL) or the tile's block scale, written with the fp16 means.
template <int DT, int D, int SMOOTH, int CHANNEL>
__device__ __forceinline__ void quant_v_body(const Strided& vin, int64_t H, int64_t n, const int64_t* perm,
                                             const float* scale_or_recip, const float* tile_mean,
                                             const float* tile_peak, uint8_t* v8, float* vs_block, uint16_t* means,
                                             int64_t tile, int64_t bh, int64_t tiles) {
  constexpr int CPG = D / 8;  // channels per thread
  __shared__ __attribute__((aligned(16))) uint8_t stage[D * kTile];
  __shared__ float sc_sh[D], mu_sh[D];
  const int tid = threadIdx.x, m = tid >> 3, cg = tid & 7;
  const int64_t sn = vin.sn;
  const uint16_t* base = head_base(vin.p, bh, H, vin.sb, vin.sh);
  // Row loads first, so that they overlap the scale/mean stage below.
  uint32_t w[4][CPG / 2];
  bool valid[4];
  {
    int64_t src[4];
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      const int64_t key = tile * kTile + 16 * (m & 7) + 2 * (m >> 3) + (q & 1) + 8 * (q >> 1);
      valid[q] = key < n;
      src[q] = valid[q] ? source_token(perm, bh, n, key) : 0;
    }
    // Two vector loads per row: 16 bytes each for D = 128, 8 bytes for D = 64
    // (the alignment the input checks guarantee).
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      const uint16_t* p = base + src[q] * sn + cg * CPG;
#pragma unroll
      for (int h = 0; h < 2; ++h) {
        if constexpr (D == 128) {
          const uint4 v = *reinterpret_cast<const uint4*>(p + 8 * h);
          w[q][4 * h] = v.x;
          w[q][4 * h + 1] = v.y;
          w[q][4 * h + 2] = v.z;
          w[q][4 * h + 3] = v.w;
        } else {
          const uint2 v = *reinterpret_cast<const uint2*>(p + 4 * h);
          w[q][2 * h] = v.x;
          w[q][2 * h + 1] = v.y;
        }
      }
    }
  }
  if (tid < D) {
    const int64_t meta = (bh * tiles + tile) * D + tid;
    if constexpr (SMOOTH) {
      float mu = tile_mean[meta], s;
      if constexpr (CHANNEL) {
        s = scale_or_recip[bh * D + tid];
      } else {
        float pk = tile_peak[meta];
        s = pk > 0.0f ? __fdiv_rn(pk, 448.0f) : 1.0f;
        s = fmaxf(s, __fdiv_rn(fabsf(mu), 65504.0f));
        vs_block[meta] = s;
      }
      mu_sh[tid] = mu;
      sc_sh[tid] = s;
      means[meta] = static_cast<uint16_t>(f32_to_f16_bits(__fdiv_rn(mu, s)));
    } else {
      sc_sh[tid] = scale_or_recip[bh * D + tid];
    }
  }
  __syncthreads();
  const int chunk = ((m >> 2) ^ cg) * 16 + 4 * (m & 3);
#pragma unroll
  for (int j = 0; j < CPG; ++j) {
    const int ch = cg * CPG + j;
    float y[4];
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      const float x = in_to_f32<DT>((w[q][j >> 1] >> (16 * (j & 1))) & 0xffffu);
      float t;
      if constexpr (SMOOTH) {
        t = __fdiv_rn(__fsub_rn(x, mu_sh[ch]), sc_sh[ch]);
      } else {
        const float rc = sc_sh[ch];
        t = rc == 0.0f ? 0.0f : __fmul_rn(x, rc);  // a zero channel gives +0 bytes
      }
      // padding tokens are +0; E4M3 saturates at +-448
      y[q] = valid[q] ? fminf(448.0f, fmaxf(-448.0f, t)) : 0.0f;
    }
    uint32_t packed = static_cast<uint32_t>(__builtin_amdgcn_cvt_pk_fp8_f32(y[0], y[1], 0, false));
    packed = static_cast<uint32_t>(__builtin_amdgcn_cvt_pk_fp8_f32(y[2], y[3], static_cast<int>(packed), true));
    *reinterpret_cast<uint32_t*>(&stage[ch * kTile + chunk]) = packed;
  }
  __syncthreads();
  const int64_t npad = tiles * kTile;
  for (int s = tid; s < D * 8; s += kThreads) {
    const int ch = s >> 3, part = s & 7;
    uint4 val = *reinterpret_cast<const uint4*>(&stage[ch * kTile + ((part ^ (ch / CPG)) * 16)]);
    typedef uint32_t v4u __attribute__((ext_vector_type(4)));
    __builtin_nontemporal_store(v4u{val.x, val.y, val.z, val.w},
                                reinterpret_cast<v4u*>(v8 + (bh * D + ch) * npad + tile * kTile + part * 16));
  }
}

// (head, tile) in the reverse order of the statistics pass (see quant_k_kernel).
template <int DT, int D, int SMOOTH, int CHANNEL>
__global__ __launch_bounds__(kThreads) void quant_v_kernel(Strided v, int64_t H, int64_t n, const int64_t* perm,
                                                           const float* scale_or_recip, const float* tile_mean,
                                                           const float* tile_peak, uint8_t* v8, float* vs_block,
                                                           uint16_t* means) {
  quant_v_body<DT, D, SMOOTH, CHANNEL>(v, H, n, perm, scale_or_recip, tile_mean, tile_peak, v8, vs_block, means,
                                       gridDim.x - 1 - blockIdx.x, gridDim.y - 1 - blockIdx.y, gridDim.x);
}

// ---------------------------------------------------------------- Q, K and V together

// The whole preparation in three launches (kv_stats_kernel before these two; prepare_together),
// where the separate stages take six: the short launches of a small call end to end cost more
// than their work, and the V scales' walk hides beside the Q blocks. Same box, whole call in us,
// six launches and three: [1,2,2048,128] 39 / 30, [1,4,1024 x 8192,128] with smoothing 119 / 108,
// [1,28,8192,128] FP8 541 / 531, [1,7,37741,128] 2472 / 2456, [1,28,37741,128] 9408 / 9395 (there K
// no longer waits in the memory-side cache between its two passes, and the saved launches
// make up for it). FMT: 0 INT8, 1 INT8
// rotated, 2 FP8 blocks. VS: 0 per-channel amax, 1 smoothing with channel scales, 2 with block scales.
struct PrepOut {
  void *q8, *k8;
  uint8_t* v8;
  float *qs, *ks, *vs;
  uint16_t* means;
};

// grid (1 + (VS < 2) + ceil(Nq/64), B*H): the K mean, the V scales, then the Q blocks.
template <int DT, int D, int FMT, int VS>
__global__ __launch_bounds__(kThreads) void prep_q_kernel(Strided q, int64_t H, int64_t n, PrepOut o, float norm,
                                                          KMeanArgs kma, const float* a0, const float* a1,
                                                          float* recip) {
  constexpr int kFirst = VS == 2 ? 1 : 2;
  const int64_t bh = blockIdx.y;
  if (blockIdx.x == 0) {
    if (threadIdx.x < D) k_mean_body<DT, FMT == 2>(kma.sums, kma.tiles, kma.n, D, kma.km, kma.km_out, bh, threadIdx.x);
    return;
  }
  if constexpr (VS < 2) {
    if (blockIdx.x == 1) {
      v_scale_body<VS == 1, kThreads>(a0, a1, kma.tiles, D, o.vs, recip, bh);
      return;
    }
  }
  const int64_t blk = static_cast<int64_t>(blockIdx.x) - kFirst;
  if constexpr (FMT == 2)
    quant_fp8_body<DT, D, 64, false>(q, H, n, nullptr, static_cast<uint8_t*>(o.q8), o.qs, blk, bh, gridDim.x - kFirst);
  else
    quant_q_body<DT, D, FMT == 1>(q, H, n, static_cast<int8_t*>(o.q8), o.qs, norm, blk, bh);
}

// grid (tiles, B*H, 2): K (z = 0) and V (z = 1).
template <int DT, int D, int FMT, int VS>
__global__ __launch_bounds__(kThreads) void prep_kv_kernel(Strided k, Strided v, int64_t H, int64_t n,
                                                           const int64_t* perm, PrepOut o, float norm,
                                                           const float* km, const float* a0, const float* a1,
                                                           const float* recip) {
  const int64_t tile = blockIdx.x, bh = blockIdx.y, tiles = gridDim.x;
  if (blockIdx.z == 0) {
    if constexpr (FMT == 2)
      quant_fp8_body<DT, D, 128, true>(k, H, n, km, static_cast<uint8_t*>(o.k8), o.ks, tile, bh, tiles);
    else
      quant_k_body<DT, D, FMT == 1>(k, H, n, perm, km, static_cast<int8_t*>(o.k8), o.ks, norm, tile, bh, tiles);
  } else {
    quant_v_body<DT, D, VS != 0, VS != 2>(v, H, n, perm, VS == 0 ? recip : o.vs, a0, a1, o.v8, o.vs, o.means, tile, bh,
                                          tiles);
  }
}

// ---------------------------------------------------------------- probes

__global__ void expcast_kernel(const float* x, uint8_t* y, int64_t n) {
  int64_t i = static_cast<int64_t>(blockIdx.x) * blockDim.x + threadIdx.x;
  if (i >= n) return;
  // Same FMA + saturating RNE byte conversion as the fused kernel; the clamps
  // reproduce the reference's fminf(120, fmaxf(0, u)) for arbitrary inputs.
  float u = __builtin_fmaf(x[i], kExpA, kExpB);
  u = fminf(120.0f, fmaxf(0.0f, u));
  y[i] = static_cast<uint8_t>(__builtin_amdgcn_cvt_pk_u8_f32(u, 0, 0u) & 0xffu);
}

__global__ void convert_probe_kernel(const float* x, uint8_t* u8, uint8_t* f8, int64_t n) {
  int64_t i = static_cast<int64_t>(blockIdx.x) * blockDim.x + threadIdx.x;
  if (i >= n) return;
  u8[i] = static_cast<uint8_t>(__builtin_amdgcn_cvt_pk_u8_f32(x[i], 0, 0u) & 0xffu);
  f8[i] = static_cast<uint8_t>(e4m3_sat(x[i]));
}

// Every block writes one word: whether any of its elements has all exponent bits set. Per 16-bit
// element the exponent field plus its lowest bit carries into the sign position exactly then.
// VCX_FINITE_BLOCKS blocks, 16-byte pieces dealt to the threads in order, four in flight. One
// read of the inputs and one word per block to fetch: three torch.isfinite(x).all() took five
// elementwise passes, a reduction and a wait each (three [1,7,37741,128] bf16 inputs, host wait
// included: 500 us, this 55 us).
struct FiniteArgs {
  const uint4* p[3];
  int64_t n[3];  // 16-byte pieces
};
__global__ __launch_bounds__(256) void finite_kernel(FiniteArgs a, uint32_t mask, uint32_t step, int32_t* out) {
  constexpr int kBatch = 4;
  uint32_t bad = 0;
  const int64_t stride = static_cast<int64_t>(gridDim.x) * blockDim.x;
#pragma unroll
  for (int t = 0; t < 3; ++t) {
    for (int64_t i = static_cast<int64_t>(blockIdx.x) * blockDim.x + threadIdx.x; i < a.n[t]; i += kBatch * stride) {
      uint4 v[kBatch];
#pragma unroll
      for (int b = 0; b < kBatch; ++b) v[b] = a.p[t][i + b * stride < a.n[t] ? i + b * stride : i];
#pragma unroll
      for (int b = 0; b < kBatch; ++b) {
        const uint32_t w[4] = {v[b].x, v[b].y, v[b].z, v[b].w};
#pragma unroll
        for (int e = 0; e < 4; ++e) bad |= (w[e] & mask) + step;
      }
    }
  }
  const bool any = __syncthreads_or((bad & 0x80008000u) != 0);
  if (threadIdx.x == 0) out[blockIdx.x] = any ? 1 : 0;
}

// ---------------------------------------------------------------- host helpers

int check_input(const char* name, const void* p, int64_t B, int64_t H, int64_t N, int64_t D,
                int64_t sb, int64_t sh, int64_t sn) {
  VCX_REQUIRE(p != nullptr, "%s is null", name);
  VCX_REQUIRE(aligned(p, D == 128 ? 16 : 8), "%s pointer alignment: need %d bytes", name, D == 128 ? 16 : 8);
  const int64_t vec = D / 16;  // elements per vector load
  VCX_REQUIRE(sb % vec == 0 && sh % vec == 0 && sn % vec == 0,
              "%s strides must be multiples of %lld elements", name, (long long)vec);
  VCX_REQUIRE(sb >= 0 && sh >= 0 && sn >= D, "%s strides invalid (need sn >= D, last dim contiguous)", name);
  (void)B; (void)H; (void)N;
  return VCX_OK;
}

int check_shape(int64_t B, int64_t H, int64_t N, int64_t D) {
  VCX_REQUIRE(B >= 1 && H >= 1 && N >= 1, "B, H, N must be positive");
  VCX_REQUIRE(D == 64 || D == 128, "D must be 64 or 128");
  VCX_REQUIRE(B * H <= 65535, "B*H exceeds 65535");
  VCX_REQUIRE(N < (int64_t(1) << 31) / 2, "N too large");
  return VCX_OK;
}

template <typename F>
int dispatch(int dtype, int64_t D, F&& f) {
  if (dtype == VCX_BFLOAT16) {
    if (D == 128) return f(std::integral_constant<int, VCX_BFLOAT16>(), std::integral_constant<int, 128>());
    return f(std::integral_constant<int, VCX_BFLOAT16>(), std::integral_constant<int, 64>());
  }
  if (D == 128) return f(std::integral_constant<int, VCX_FLOAT16>(), std::integral_constant<int, 128>());
  return f(std::integral_constant<int, VCX_FLOAT16>(), std::integral_constant<int, 64>());
}

size_t align_up(size_t x) { return (x + 255) & ~size_t(255); }

}  // namespace

// Workspace layouts (all 256-byte aligned slices).
size_t ws_prepare_qk(int64_t BH, int64_t N, int64_t D) {
  int64_t tiles = cdiv(N, kTile);
  return align_up(sizeof(double) * BH * tiles * D) + align_up(sizeof(float) * BH * D);
}
size_t ws_preprocess_qk(int64_t BH, int64_t N, int64_t D) {
  return align_up(sizeof(double) * BH * cdiv(N, kTile) * D) + align_up(sizeof(float) * BH * D);
}
size_t ws_prepare_v(int64_t BH, int64_t N, int64_t D) {
  int64_t tiles = cdiv(N, kTile);
  return 2 * align_up(sizeof(float) * BH * tiles * D) + align_up(sizeof(float) * BH * D);
}

}  // namespace vcx

using namespace vcx;

namespace {
int prepare_qk_int8(const void* q, const void* k, int dtype, int64_t B, int64_t H, int64_t Nq, int64_t Nk,
                    int64_t D, int64_t q_sb, int64_t q_sh, int64_t q_sn, int64_t k_sb, int64_t k_sh, int64_t k_sn,
                    const int64_t* perm, int8_t* q8, float* qs, int8_t* k8, float* ks, void* km_out,
                    void* workspace, size_t workspace_bytes, void* stream, bool rotate) {
  if (int rc = check_shape(B, H, Nq, D)) return rc;
  if (int rc = check_shape(B, H, Nk, D)) return rc;
  VCX_REQUIRE(dtype == VCX_FLOAT16 || dtype == VCX_BFLOAT16, "dtype must be float16 or bfloat16");
  if (int rc = check_input("q", q, B, H, Nq, D, q_sb, q_sh, q_sn)) return rc;
  if (int rc = check_input("k", k, B, H, Nk, D, k_sb, k_sh, k_sn)) return rc;
  VCX_REQUIRE(q8 && qs && k8 && ks, "output pointers must be non-null");
  VCX_REQUIRE(aligned(q8, 8) && aligned(k8, 8), "q8/k8 must be 8-byte aligned");
  VCX_REQUIRE(aligned(perm, 8) && aligned(km_out, 2), "perm/km_out misaligned");
  const int64_t BH = B * H, tiles = cdiv(Nk, kTile);
  VCX_REQUIRE(workspace != nullptr && aligned(workspace, 256), "workspace must be non-null and 256-byte aligned");
  VCX_REQUIRE(workspace_bytes >= ws_prepare_qk(BH, Nk, D), "workspace too small: need %zu bytes",
              ws_prepare_qk(BH, Nk, D));
  auto* ws = static_cast<char*>(workspace);
  double* ksum = reinterpret_cast<double*>(ws);
  float* km = reinterpret_cast<float*>(ws + align_up(sizeof(double) * BH * tiles * D));
  hipStream_t st = static_cast<hipStream_t>(stream);
  const float norm = static_cast<float>(1.0 / std::sqrt(static_cast<double>(D)));
  // K statistics, then the Q quantization with the K mean in its first blocks, then the K
  // quantization.
  const KMeanArgs kma{ksum, tiles, Nk, km, km_out};
  const Strided qt{q, q_sb, q_sh, q_sn}, kt{k, k_sb, k_sh, k_sn};
  return dispatch(dtype, D, [&](auto dt, auto dd) -> int {
    constexpr int DT = decltype(dt)::value, DD = decltype(dd)::value;
    tile_stats_kernel<DT, DD, kKSum><<<dim3(tiles, BH), kThreads, 0, st>>>(kt, H, Nk, perm, ksum, nullptr, nullptr);
    VCX_LAUNCHED("tile_stats_kernel<K>");
    auto quant = [&](auto rot) -> int {
      constexpr bool ROT = decltype(rot)::value;
      quant_q_kernel<DT, DD, ROT><<<dim3(cdiv(Nq, 64) + 1, BH), kThreads, 0, st>>>(qt, H, Nq, q8, qs, norm, kma);
      VCX_LAUNCHED("quant_q_kernel");
      quant_k_kernel<DT, DD, ROT><<<dim3(tiles, BH), kThreads, 0, st>>>(kt, H, Nk, perm, km, k8, ks, norm);
      VCX_LAUNCHED("quant_k_kernel");
      return VCX_OK;
    };
    return rotate ? quant(std::true_type()) : quant(std::false_type());
  });
}
}  // namespace

extern "C" int vcx_prepare_qk_int8(const void* q, const void* k, int dtype, int64_t B, int64_t H,
                                   int64_t Nq, int64_t Nk, int64_t D, int64_t q_sb, int64_t q_sh,
                                   int64_t q_sn, int64_t k_sb, int64_t k_sh, int64_t k_sn,
                                   const int64_t* perm, int8_t* q8, float* qs, int8_t* k8, float* ks,
                                   void* km_out, void* workspace, size_t workspace_bytes,
                                   void* stream) {
  return prepare_qk_int8(q, k, dtype, B, H, Nq, Nk, D, q_sb, q_sh, q_sn, k_sb, k_sh, k_sn, perm, q8, qs, k8, ks,
                         km_out, workspace, workspace_bytes, stream, false);
}

extern "C" int vcx_prepare_qk_int8_rotated(const void* q, const void* k, int dtype, int64_t B, int64_t H,
                                           int64_t Nq, int64_t Nk, int64_t D, int64_t q_sb, int64_t q_sh,
                                           int64_t q_sn, int64_t k_sb, int64_t k_sh, int64_t k_sn,
                                           const int64_t* perm, int8_t* q8, float* qs, int8_t* k8, float* ks,
                                           void* km_out, void* workspace, size_t workspace_bytes,
                                           void* stream) {
  return prepare_qk_int8(q, k, dtype, B, H, Nq, Nk, D, q_sb, q_sh, q_sn, k_sb, k_sh, k_sn, perm, q8, qs, k8, ks,
                         km_out, workspace, workspace_bytes, stream, true);
}

// Q, K and V of one call in three launches. Outputs and results are those of
// vcx_prepare_qk_int8(_rotated) or vcx_prepare_qk_fp8, and vcx_prepare_v_fp8. ksum: K's tile sums
// (may lie over v8: the first launch writes them, the second reads them, the third writes v8);
// km: K's mean; v_scratch: vcx_prepare_v_fp8's workspace.
namespace vcx {
int prepare_together(const vcx_call& c, const int64_t* perm, void* q8, float* qs, void* k8, float* ks, uint8_t* v8,
                     float* vs, uint16_t* means, double* ksum, float* km, void* v_scratch, void* stream) {
  if (int rc = check_shape(c.B, c.H, c.Nq, c.D)) return rc;
  if (int rc = check_shape(c.B, c.H, c.Nk, c.D)) return rc;
  VCX_REQUIRE(c.dtype == VCX_FLOAT16 || c.dtype == VCX_BFLOAT16, "dtype must be float16 or bfloat16");
  if (int rc = check_input("q", c.q, c.B, c.H, c.Nq, c.D, c.q_sb, c.q_sh, c.q_sn)) return rc;
  if (int rc = check_input("k", c.k, c.B, c.H, c.Nk, c.D, c.k_sb, c.k_sh, c.k_sn)) return rc;
  if (int rc = check_input("v", c.v, c.B, c.H, c.Nk, c.D, c.v_sb, c.v_sh, c.v_sn)) return rc;
  VCX_REQUIRE(aligned(perm, 8), "perm misaligned");
  const int64_t BH = c.B * c.H, tiles = cdiv(c.Nk, kTile);
  auto* ws = static_cast<char*>(v_scratch);
  const size_t slice = align_up(sizeof(float) * BH * tiles * c.D);
  float* a0 = reinterpret_cast<float*>(ws);
  float* a1 = reinterpret_cast<float*>(ws + slice);
  float* recip = reinterpret_cast<float*>(ws + 2 * slice);
  const KMeanArgs kma{ksum, tiles, c.Nk, km, nullptr};
  const Strided q{c.q, c.q_sb, c.q_sh, c.q_sn}, k{c.k, c.k_sb, c.k_sh, c.k_sn}, v{c.v, c.v_sb, c.v_sh, c.v_sn};
  const PrepOut o{q8, k8, v8, qs, ks, vs, means};
  const float norm = static_cast<float>(1.0 / std::sqrt(static_cast<double>(c.D)));
  hipStream_t st = static_cast<hipStream_t>(stream);
  return dispatch(static_cast<int>(c.dtype), c.D, [&](auto dt, auto dd) -> int {
    constexpr int DT = decltype(dt)::value, DD = decltype(dd)::value;
    auto run = [&](auto fmt, auto value) -> int {
      constexpr int FMT = decltype(fmt)::value, VS = decltype(value)::value;
      const dim3 both(static_cast<unsigned>(tiles), static_cast<unsigned>(BH), 2);
      kv_stats_kernel<DT, DD, VS == 0 ? kVAmax : kVSmooth><<<both, kThreads, 0, st>>>(k, v, c.H, c.Nk, perm, ksum, a0, a1);
      VCX_LAUNCHED("kv_stats_kernel");
      prep_q_kernel<DT, DD, FMT, VS><<<dim3(static_cast<unsigned>(cdiv(c.Nq, 64) + (VS == 2 ? 1 : 2)),
                                            static_cast<unsigned>(BH)), kThreads, 0, st>>>(q, c.H, c.Nq, o, norm, kma,
                                                                                           a0, a1, recip);
      VCX_LAUNCHED("prep_q_kernel");
      prep_kv_kernel<DT, DD, FMT, VS><<<both, kThreads, 0, st>>>(k, v, c.H, c.Nk, perm, o, norm, km, a0, a1, recip);
      VCX_LAUNCHED("prep_kv_kernel");
      return VCX_OK;
    };
    auto format = [&](auto fmt) -> int {
      if (!c.smooth) return run(fmt, std::integral_constant<int, 0>());
      return c.channel_scale ? run(fmt, std::integral_constant<int, 1>()) : run(fmt, std::integral_constant<int, 2>());
    };
    if (c.qk_fp8) return run(std::integral_constant<int, 2>(), std::integral_constant<int, 0>());
    return c.rotate ? format(std::integral_constant<int, 1>()) : format(std::integral_constant<int, 0>());
  });
}
}  // namespace vcx

// ---------------------------------------------------------------- allocation-free variant

namespace {
// Scratch of vcx_prepare_qk_int8_noalloc: the fp64 K tile sums and the binary32 K mean
// (ws_prepare_qk bytes) of shapes up to this size. Each GPU the library runs on holds one
// copy until the process ends; every call on that GPU shares it, so calls that overlap on
// one GPU race. Every byte a call reads it first writes, so nothing needs clearing.
constexpr size_t kNoAllocScratchBytes = VCX_NOALLOC_SCRATCH_BYTES;
static __device__ __align__(256) uint8_t scratch[kNoAllocScratchBytes];

constexpr int kScratchDevices = 64;
std::mutex g_scratch_mutex;
void* g_scratch_address[kScratchDevices];  // device address of `scratch`, per device ordinal

// The current device's address of `scratch`, resolved once per device (with that device
// current) by hipGetSymbolAddress; the host-side name is not a device address.
int scratch_address(void** out) {
  int dev = -1;
  hipError_t e = hipGetDevice(&dev);
  if (e != hipSuccess) return fail(VCX_EHIP, "hipGetDevice: %s", hipGetErrorString(e));
  VCX_REQUIRE(dev >= 0 && dev < kScratchDevices, "device ordinal %d is beyond the scratch table", dev);
  std::lock_guard<std::mutex> lock(g_scratch_mutex);
  if (g_scratch_address[dev] == nullptr) {
    void* p = nullptr;
    e = hipGetSymbolAddress(&p, HIP_SYMBOL(scratch));
    if (e != hipSuccess || p == nullptr)
      return fail(VCX_EHIP, "hipGetSymbolAddress(scratch): %s", hipGetErrorString(e));
    g_scratch_address[dev] = p;
  }
  *out = g_scratch_address[dev];
  return VCX_OK;
}
}  // namespace

extern "C" int vcx_prepare_qk_int8_noalloc(const void* q, const void* k, int dtype, int64_t B, int64_t H,
                                           int64_t Nq, int64_t Nk, int64_t D, int64_t q_sb, int64_t q_sh,
                                           int64_t q_sn, int64_t k_sb, int64_t k_sh, int64_t k_sn,
                                           const int64_t* perm, int8_t* q8, float* qs, int8_t* k8, float* ks,
                                           void* km_out, void* stream) {
  if (int rc = check_shape(B, H, Nk, D)) return rc;
  const size_t need = ws_prepare_qk(B * H, Nk, D);
  VCX_REQUIRE(need <= kNoAllocScratchBytes,
              "vcx_prepare_qk_int8_noalloc: B*H=%lld, Nk=%lld, D=%lld needs %zu scratch bytes, above its %zu; "
              "call vcx_prepare_qk_int8 with a workspace", static_cast<long long>(B * H),
              static_cast<long long>(Nk), static_cast<long long>(D), need, kNoAllocScratchBytes);
  void* ws = nullptr;
  if (int rc = scratch_address(&ws)) return rc;
  return prepare_qk_int8(q, k, dtype, B, H, Nq, Nk, D, q_sb, q_sh, q_sn, k_sb, k_sh, k_sn, perm, q8, qs, k8, ks,
                         km_out, ws, kNoAllocScratchBytes, stream, false);
}

extern "C" int vcx_prepare_qk_fp8(const void* q, const void* k, int dtype, int64_t B, int64_t H,
                                  int64_t Nq, int64_t Nk, int64_t D, int64_t q_sb, int64_t q_sh,
                                  int64_t q_sn, int64_t k_sb, int64_t k_sh, int64_t k_sn, uint8_t* q8,
                                  float* qs, uint8_t* k8, float* ks, float* km_out, void* workspace,
                                  size_t workspace_bytes, void* stream) {
  if (int rc = check_shape(B, H, Nq, D)) return rc;
  if (int rc = check_shape(B, H, Nk, D)) return rc;
  VCX_REQUIRE(dtype == VCX_FLOAT16 || dtype == VCX_BFLOAT16, "dtype must be float16 or bfloat16");
  if (int rc = check_input("q", q, B, H, Nq, D, q_sb, q_sh, q_sn)) return rc;
  if (int rc = check_input("k", k, B, H, Nk, D, k_sb, k_sh, k_sn)) return rc;
  VCX_REQUIRE(q8 && qs && k8 && ks, "output pointers must be non-null");
  VCX_REQUIRE(aligned(q8, 8) && aligned(k8, 8), "q8/k8 must be 8-byte aligned");
  VCX_REQUIRE(aligned(km_out, 4), "km_out misaligned");
  const int64_t BH = B * H, tiles = cdiv(Nk, kTile);
  VCX_REQUIRE(workspace != nullptr && aligned(workspace, 256), "workspace must be non-null and 256-byte aligned");
  VCX_REQUIRE(workspace_bytes >= ws_prepare_qk(BH, Nk, D), "workspace too small: need %zu bytes",
              ws_prepare_qk(BH, Nk, D));
  auto* ws = static_cast<char*>(workspace);
  double* ksum = reinterpret_cast<double*>(ws);
  float* km = reinterpret_cast<float*>(ws + align_up(sizeof(double) * BH * tiles * D));
  hipStream_t st = static_cast<hipStream_t>(stream);
  return dispatch(dtype, D, [&](auto dt, auto dd) -> int {
    constexpr int DT = decltype(dt)::value, DD = decltype(dd)::value;
    // K statistics, then the Q quantization with the K mean in its first blocks (Q read
    // non-temporally, so K stays in the memory-side cache), then the K quantization.
    const Strided qt{q, q_sb, q_sh, q_sn}, kt{k, k_sb, k_sh, k_sn};
    tile_stats_kernel<DT, DD, kKSum><<<dim3(tiles, BH), kThreads, 0, st>>>(kt, H, Nk, nullptr, ksum, nullptr, nullptr);
    VCX_LAUNCHED("tile_stats_kernel<K>");
    const KMeanArgs kma{ksum, tiles, Nk, km, km_out};
    quant_fp8_q_kernel<DT, DD><<<dim3(cdiv(Nq, 64) + 1, BH), kThreads, 0, st>>>(qt, H, Nq, q8, qs, kma);
    VCX_LAUNCHED("quant_fp8_q_kernel");
    quant_fp8_k_kernel<DT, DD><<<dim3(tiles, BH), kThreads, 0, st>>>(kt, H, Nk, km, k8, ks);
    VCX_LAUNCHED("quant_fp8_k_kernel");
    return VCX_OK;
  });
}

extern "C" int vcx_prepare_v_fp8(const void* v, int dtype, int64_t B, int64_t H, int64_t N, int64_t D,
                                 int64_t v_sb, int64_t v_sh, int64_t v_sn, const int64_t* perm,
                                 int smooth, int channel_scale, uint8_t* v8, float* vs,
                                 uint16_t* means, void* workspace, size_t workspace_bytes,
                                 void* stream) {
  if (int rc = check_shape(B, H, N, D)) return rc;
  VCX_REQUIRE(dtype == VCX_FLOAT16 || dtype == VCX_BFLOAT16, "dtype must be float16 or bfloat16");
  if (int rc = check_input("v", v, B, H, N, D, v_sb, v_sh, v_sn)) return rc;
  VCX_REQUIRE(v8 && vs, "v8/vs must be non-null");
  VCX_REQUIRE(aligned(v8, 16), "v8 must be 16-byte aligned");
  VCX_REQUIRE(!smooth || means != nullptr, "means must be non-null when smoothing");
  VCX_REQUIRE(aligned(perm, 8), "perm misaligned");
  const int64_t BH = B * H, tiles = cdiv(N, kTile);
  VCX_REQUIRE(workspace != nullptr && aligned(workspace, 256), "workspace must be non-null and 256-byte aligned");
  VCX_REQUIRE(workspace_bytes >= ws_prepare_v(BH, N, D), "workspace too small: need %zu bytes",
              ws_prepare_v(BH, N, D));
  auto* ws = static_cast<char*>(workspace);
  const size_t slice = align_up(sizeof(float) * BH * tiles * D);
  float* a0 = reinterpret_cast<float*>(ws);
  float* a1 = reinterpret_cast<float*>(ws + slice);
  float* recip = reinterpret_cast<float*>(ws + 2 * slice);
  hipStream_t st = static_cast<hipStream_t>(stream);
  return dispatch(dtype, D, [&](auto dt, auto dd) -> int {
    constexpr int DT = decltype(dt)::value, DD = decltype(dd)::value;
    const dim3 grid(tiles, BH);
    const Strided vt{v, v_sb, v_sh, v_sn};
    if (!smooth) {
      tile_stats_kernel<DT, DD, kVAmax><<<grid, kThreads, 0, st>>>(vt, H, N, perm, nullptr, a0, nullptr);
      VCX_LAUNCHED("tile_stats_kernel<Vamax>");
      v_scale_kernel<false><<<dim3(BH), kScaleThreads / DD * DD, 0, st>>>(a0, nullptr, tiles, DD, vs, recip);
      VCX_LAUNCHED("v_scale_kernel");
      quant_v_kernel<DT, DD, 0, 1><<<grid, kThreads, 0, st>>>(vt, H, N, perm, recip, nullptr, nullptr, v8, nullptr,
                                                              nullptr);
      VCX_LAUNCHED("quant_v_kernel");
      return VCX_OK;
    }
    tile_stats_kernel<DT, DD, kVSmooth><<<grid, kThreads, 0, st>>>(vt, H, N, perm, nullptr, a0, a1);
    VCX_LAUNCHED("tile_stats_kernel<Vsmooth>");
    if (channel_scale) {
      v_scale_kernel<true><<<dim3(BH), kScaleThreads / DD * DD, 0, st>>>(a0, a1, tiles, DD, vs, nullptr);
      VCX_LAUNCHED("v_scale_kernel");
      quant_v_kernel<DT, DD, 1, 1><<<grid, kThreads, 0, st>>>(vt, H, N, perm, vs, a0, a1, v8, nullptr, means);
    } else {
      quant_v_kernel<DT, DD, 1, 0><<<grid, kThreads, 0, st>>>(vt, H, N, perm, nullptr, a0, a1, v8, vs, means);
    }
    VCX_LAUNCHED("quant_v_kernel");
    return VCX_OK;
  });
}

extern "C" int vcx_expcast_codes(const float* x, uint8_t* y, int64_t n, void* stream) {
  VCX_REQUIRE(n >= 0, "n must be non-negative");
  if (n == 0) return VCX_OK;
  VCX_REQUIRE(x && y, "null pointer");
  expcast_kernel<<<cdiv(n, 256), 256, 0, static_cast<hipStream_t>(stream)>>>(x, y, n);
  VCX_LAUNCHED("expcast_kernel");
  return VCX_OK;
}

extern "C" int vcx_convert_probe(const float* x, uint8_t* u8, uint8_t* f8, int64_t n, void* stream) {
  VCX_REQUIRE(n >= 0, "n must be non-negative");
  if (n == 0) return VCX_OK;
  VCX_REQUIRE(x && u8 && f8, "null pointer");
  convert_probe_kernel<<<cdiv(n, 256), 256, 0, static_cast<hipStream_t>(stream)>>>(x, u8, f8, n);
  VCX_LAUNCHED("convert_probe_kernel");
  return VCX_OK;
}

extern "C" int vcx_check_finite(const void* a, int64_t na, const void* b, int64_t nb, const void* c, int64_t nc,
                                int dtype, int32_t* out, void* stream) {
  VCX_REQUIRE(dtype == VCX_FLOAT16 || dtype == VCX_BFLOAT16, "dtype must be float16 or bfloat16");
  VCX_REQUIRE(out != nullptr && aligned(out, 4), "out must be non-null and 4-byte aligned");
  const void* p[3] = {a, b, c};
  const int64_t n[3] = {na, nb, nc};
  FiniteArgs args{};
  for (int t = 0; t < 3; ++t) {
    VCX_REQUIRE(n[t] >= 0 && n[t] % 8 == 0 && (n[t] == 0 || (p[t] != nullptr && aligned(p[t], 16))),
                "inputs must be 16-byte aligned with a multiple of 8 elements");
    args.p[t] = static_cast<const uint4*>(p[t]);
    args.n[t] = n[t] / 8;
  }
  const uint32_t mask = dtype == VCX_BFLOAT16 ? 0x7f807f80u : 0x7c007c00u;
  const uint32_t step = dtype == VCX_BFLOAT16 ? 0x00800080u : 0x04000400u;
  finite_kernel<<<VCX_FINITE_BLOCKS, 256, 0, static_cast<hipStream_t>(stream)>>>(args, mask, step, out);
  return check_launch("finite_kernel");
}

namespace {
template <int DT>
int preprocess_launch(const void* q, const void* k, int64_t BH, int64_t H, int64_t Nq, int64_t Nk, int64_t D,
                      int64_t q_sb, int64_t q_sh, int64_t q_sn, int64_t k_sb, int64_t k_sh, int64_t k_sn,
                      int k_smooth, int hadamard, float* q_out, float* k_out, double* part, float* mean,
                      hipStream_t st) {
  const int64_t tiles = cdiv(Nk, kTile);
  // rows of four-element pieces: D 64 or 128 and every row on a four-element boundary
  constexpr int kQuad = DT == VCX_FLOAT32 ? 16 : 8;
  auto quads = [&](const void* x, int64_t sb, int64_t sh, int64_t sn) {
    return (D == 64 || D == 128) && aligned(x, kQuad) && sb % 4 == 0 && sh % 4 == 0 && sn % 4 == 0;
  };
  const bool q_wide = quads(q, q_sb, q_sh, q_sn) && aligned(q_out, 16);
  const bool k_wide = quads(k, k_sb, k_sh, k_sn) && aligned(k_out, 16);
  KMeanArgs kma{};
  if (k_smooth) {
    kma = KMeanArgs{part, tiles, Nk, mean, nullptr};
    pre_tile_sum_kernel<DT><<<dim3(tiles, BH), static_cast<unsigned>(D), 0, st>>>(k, H, Nk, k_sb, k_sh, k_sn, part);
    VCX_LAUNCHED("pre_tile_sum_kernel");
  }
  int W = 1;
  while (W < D) W <<= 1;
  const float norm = static_cast<float>(1.0 / std::sqrt(static_cast<double>(W)));
  // Q, with the K mean in its first blocks, then K
  auto run = [&](auto wc, auto rot) -> int {
    constexpr int WW = decltype(wc)::value, L = WW < 16 ? WW : 16;
    constexpr bool ROT = decltype(rot)::value;
    auto rows = [&](auto wide, auto km, auto nr, const void* x, int64_t n, int64_t sb, int64_t sh, int64_t sn, const float* mu,
                    float* out) {
      constexpr bool KM = decltype(km)::value;
      constexpr int NR = decltype(nr)::value, RPB = kThreads / L * NR;
      const int64_t blocks = cdiv(n, RPB) + (KM ? 1 : 0), gx = std::min(blocks, kRowsGridX);
      pre_rows_kernel<DT, WW, ROT, decltype(wide)::value, KM, NR>
          <<<dim3(static_cast<unsigned>(gx), static_cast<unsigned>(BH), static_cast<unsigned>(cdiv(blocks, gx))), kThreads,
             0, st>>>(x, H, n, static_cast<int>(D), sb, sh, sn, mu, out, norm, kma);
    };
    const float* none = nullptr;
    auto launch = [&](bool wide, auto km, auto centre, const void* x, int64_t n, auto... args) {
      constexpr bool MEAN = decltype(centre)::value;
      auto nr = [&](auto w) {
        constexpr bool WIDE = decltype(w)::value;
        // Four rows per thread share a load of the mean and leave more loads in flight, one row more
        // waves: four from about two blocks of them per CU on, and one wherever entries move one
        // by one and four would gain nothing (no mean, or a plain difference of wide rows). Q and K,
        // whole call in us, one row / four rows: [1,2,1000,128] rotated 4.6 / 6.8, [1,8,4000,128] centred and
        // rotated 23.6 / 21.7, [1,28,37741,16] centred 99.9 / 80.9, [1,28,37741,72] centred 298 / 323.
        if constexpr (WIDE || (MEAN && (ROT || WW <= 32))) {
          if (BH * cdiv(n, 4 * kThreads / L) >= (WIDE && MEAN ? 256 : 512))
            return rows(w, km, std::integral_constant<int, 4>(), x, n, args...);
        }
        rows(w, km, std::integral_constant<int, 1>(), x, n, args...);
      };
      if constexpr (WW == 64 || WW == 128) {
        if (wide) return nr(std::true_type());
      }
      nr(std::false_type());
    };
    if (k_smooth) launch(q_wide, std::true_type(), std::false_type(), q, Nq, q_sb, q_sh, q_sn, none, q_out);
    else launch(q_wide, std::false_type(), std::false_type(), q, Nq, q_sb, q_sh, q_sn, none, q_out);
    VCX_LAUNCHED("pre_rows_kernel<Q>");
    if (k_smooth)
      launch(k_wide, std::false_type(), std::true_type(), k, Nk, k_sb, k_sh, k_sn, static_cast<const float*>(mean), k_out);
    else launch(k_wide, std::false_type(), std::false_type(), k, Nk, k_sb, k_sh, k_sn, none, k_out);
    VCX_LAUNCHED("pre_rows_kernel<K>");
    return VCX_OK;
  };
  auto width = [&](auto rot) -> int {
    switch (W) {
      case 1: return run(std::integral_constant<int, 1>(), rot);
      case 2: return run(std::integral_constant<int, 2>(), rot);
      case 4: return run(std::integral_constant<int, 4>(), rot);
      case 8: return run(std::integral_constant<int, 8>(), rot);
      case 16: return run(std::integral_constant<int, 16>(), rot);
      case 32: return run(std::integral_constant<int, 32>(), rot);
      case 64: return run(std::integral_constant<int, 64>(), rot);
      default: return run(std::integral_constant<int, 128>(), rot);
    }
  };
  return hadamard ? width(std::true_type()) : width(std::false_type());
}
}  // namespace

extern "C" int vcx_preprocess_qk(const void* q, const void* k, int dtype, int64_t B, int64_t H, int64_t Nq,
                                 int64_t Nk, int64_t D, int64_t q_sb, int64_t q_sh, int64_t q_sn, int64_t k_sb,
                                 int64_t k_sh, int64_t k_sn, int k_smooth, int hadamard, float* q_out,
                                 float* k_out, void* workspace, size_t workspace_bytes, void* stream) {
  VCX_REQUIRE(B >= 1 && H >= 1 && Nq >= 1 && Nk >= 1, "B, H, Nq, Nk must be positive");
  VCX_REQUIRE(D >= 1 && D <= 128, "Q/K preprocessing supports head dimensions 1..128");
  VCX_REQUIRE(B * H <= 65535, "B*H exceeds 65535");
  VCX_REQUIRE(Nq < (int64_t(1) << 30) && Nk < (int64_t(1) << 30), "sequence too long");
  VCX_REQUIRE(dtype == VCX_FLOAT16 || dtype == VCX_BFLOAT16 || dtype == VCX_FLOAT32,
              "dtype must be float16, bfloat16 or float32");
  VCX_REQUIRE(q && k && q_out && k_out, "null tensor pointer");
  const int esz = dtype == VCX_FLOAT32 ? 4 : 2;
  VCX_REQUIRE(aligned(q, esz) && aligned(k, esz) && aligned(q_out, 4) && aligned(k_out, 4), "pointer alignment");
  VCX_REQUIRE(q_sb >= 0 && q_sh >= 0 && q_sn >= D && k_sb >= 0 && k_sh >= 0 && k_sn >= D,
              "strides invalid (need sn >= D, last dim contiguous)");
  const int64_t BH = B * H;
  double* part = nullptr;
  float* mean = nullptr;
  if (k_smooth) {
    VCX_REQUIRE(workspace != nullptr && aligned(workspace, 256), "workspace must be non-null and 256-byte aligned");
    VCX_REQUIRE(workspace_bytes >= ws_preprocess_qk(BH, Nk, D), "workspace too small: need %zu bytes",
                ws_preprocess_qk(BH, Nk, D));
    part = static_cast<double*>(workspace);
    mean = reinterpret_cast<float*>(static_cast<char*>(workspace) + align_up(sizeof(double) * BH * cdiv(Nk, kTile) * D));
  }
  hipStream_t st = static_cast<hipStream_t>(stream);
  if (dtype == VCX_FLOAT32)
    return preprocess_launch<VCX_FLOAT32>(q, k, BH, H, Nq, Nk, D, q_sb, q_sh, q_sn, k_sb, k_sh, k_sn, k_smooth,
                                          hadamard, q_out, k_out, part, mean, st);
  if (dtype == VCX_BFLOAT16)
    return preprocess_launch<VCX_BFLOAT16>(q, k, BH, H, Nq, Nk, D, q_sb, q_sh, q_sn, k_sb, k_sh, k_sn, k_smooth,
                                           hadamard, q_out, k_out, part, mean, st);
  return preprocess_launch<VCX_FLOAT16>(q, k, BH, H, Nq, Nk, D, q_sb, q_sh, q_sn, k_sb, k_sh, k_sn, k_smooth,
                                        hadamard, q_out, k_out, part, mean, st);
}
