// Fused attention where the rows do not fill the chip: the key tiles of 16, 32 or 64 rows split
// over the waves of a block. A call with few rows lasts as long as one block's chain of tiles
// (about 1 us a tile, whatever the chip has idle); a split runs a half to an eighth of it.
// Algorithm and numerical contract: vcx_attn.hip.
#include "vcx_attn.hpp"

namespace vcx {
namespace {

// LDS-only workgroup barrier: __syncthreads() would also wait for the K/V loads in flight.
__device__ inline void lds_barrier() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup", "local");
  __builtin_amdgcn_s_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup", "local");
}

// Direct-to-LDS loads of one key tile by the RG waves that share it (wave g of them issues
// every RG-th KB), in the placement of TileLoader. The loads are written as asm: the compiler
// would drain loads it knows of at every LDS read that might alias them, and here V^T of a
// tile is in flight while its K is read, and the other way round. Each wave waits for its own
// loads (wait) before the barrier that hands the region to its readers. The compiler does not
// place wait states inside asm: s_nop 4 gives the five that an address or resource register
// needs when a VALU instruction (the read of a spilled scalar, say) has just written it, and the
// one that M0 needs.
template <int D, int QF, int RG>
struct PieceLoader {
  static constexpr int kOps = D / 8;  // 1 KB instructions per operand tile
  static constexpr int BYTES = 2 * kTile * D + 16;
  static constexpr int kPart = kOps / RG;  // a wave's share
  static_assert(D == 64 || RG % 2 == 0, "a wave's K instructions repeat one lane pattern");
  v4i rk, rv, rs;
  uint32_t koff, voff, base;  // base: LDS byte address of the region
  int tiles, npad, g;

  __device__ inline static v4i rsrc(const void* p, uint32_t bytes) {
    const uint64_t u = reinterpret_cast<uint64_t>(p);
    return v4i{__builtin_amdgcn_readfirstlane(static_cast<int>(u)),
               __builtin_amdgcn_readfirstlane(static_cast<int>((u >> 32) & 0xffffu)), static_cast<int>(bytes), 0x00020000};
  }
  __device__ inline void init(const AttnArgs& a, int64_t bh, uint8_t* region, int group, int lane) {
    tiles = static_cast<int>(a.tiles);
    npad = tiles * kTile;
    g = group;
    base = static_cast<uint32_t>(__builtin_amdgcn_readfirstlane(static_cast<int>(reinterpret_cast<uintptr_t>((lds_void*)region))));
    // Instruction n fills slots 64 n + lane: K rows p = (64 n + lane) / (D / 16). At D128 the
    // even and the odd instructions each repeat one lane pattern 16 rows further on, and a
    // wave's instructions g, g + RG, ... are all of one kind.
    const int p = (64 * (D == 128 ? g & 1 : 0) + lane) / (D / 16), phys = lane % (D / 16);
    koff = static_cast<uint32_t>(key_row(p) * D + ((phys ^ chunk_xor<D>(p)) * 16));
    const int ch = lane >> 3, q = (lane & 7) ^ (ch & 7);
    voff = static_cast<uint32_t>(ch * npad + (2 * (q & 3) + (q >> 2)) * 16);
    rk = rsrc(a.k8 + bh * a.Nk * D, static_cast<uint32_t>(a.Nk * D));
    rv = rsrc(a.v8 + bh * D * npad, static_cast<uint32_t>(D * npad));
    if constexpr (QF == 1) rs = rsrc(a.ks + bh * a.tiles, static_cast<uint32_t>(a.tiles * 4));
    else rs = rsrc(a.ks + bh * a.tiles * 4, static_cast<uint32_t>(a.tiles * 16));
  }
  __device__ inline static void load16(uint32_t lds, uint32_t voff, const v4i& r, int soff) {
    asm volatile("s_nop 4\n\tbuffer_load_dwordx4 %1, %2, %3 offen lds"
                 ::"{m0}"(lds), "v"(voff), "s"(r), "s"(soff) : "memory");
  }
  // One of the wave's kPart loads of an operand of tile t into the buffer at byte offset buf.
  // Tiles past the last read the last one again, so that no load stands behind a branch.
  __device__ __forceinline__ void part_k(int i, int t, uint32_t buf) const {
    t = t < tiles ? t : tiles - 1;
    constexpr int kPer = D == 128 ? 2 : 1;
    const int n = g + RG * i;
    load16(base + buf + n * 1024, koff, rk, t * kTile * D + (n / kPer) * 16 * D);
    if (i == 0 && g == 0 && (threadIdx.x & 63) == 0) {
      const uint32_t dst = base + buf + 2 * kTile * D;
      if constexpr (QF == 1)
        asm volatile("s_nop 4\n\tbuffer_load_dword %1, %2, %3 offen lds"
                     ::"{m0}"(dst), "v"(0), "s"(rs), "s"(t * 4) : "memory");
      else load16(dst, 0, rs, t * 16);
    }
  }
  __device__ __forceinline__ void part_v(int i, int t, uint32_t buf) const {
    t = t < tiles ? t : tiles - 1;
    const int n = g + RG * i;
    load16(base + buf + kTile * D + n * 1024, voff, rv, t * kTile + 8 * n * npad);
  }
  __device__ inline void issue_k(int t, uint32_t buf) const {
#pragma unroll
    for (int i = 0; i < kPart; ++i) part_k(i, t, buf);
  }
  __device__ inline void issue_v(int t, uint32_t buf) const {
#pragma unroll
    for (int i = 0; i < kPart; ++i) part_v(i, t, buf);
  }
  __device__ inline static void wait() { asm volatile("s_waitcnt vmcnt(0)" ::: "memory"); }
};

// A piece: 16 RG rows [row0, ...) of head bh on RG * KS waves. Wave (g, u) takes the 16 rows of
// group g and the key tiles u, u + KS, ..., with its own O, mass and maximum.
// The P bytes depend on the running maximum at every tile, so the waves exchange their tiles'
// row maxima through LDS once per step of KS tiles: the running maximum at tile KS s + u is the
// maximum of the steps before and of waves 0..u, exactly what the sequential blocks use. At
// the end each wave's sums are rescaled to the final maximum and added in split order.
// The RG waves of a tile share its K and V^T in LDS, one region per split, loaded between the
// MFMAs of the QK (and PV) steps. DB (two buffers): the next tile loads during this one, and a
// barrier per step hands it over. Else one buffer: the barrier at the top of a step makes K
// readable and V^T free to load, the one of the maxima V^T readable and K free, so that each
// operand loads while the other is in use.
template <int D, int VM, int PM, int QF, int RG, int KS, bool DB>
__device__ __forceinline__ void attn_piece(const AttnArgs& a, int64_t bh, int64_t row0, uint8_t* lds, float* xch) {
  typedef Wave<D, VM, true, PM, QF, 1> W;
  typedef PieceLoader<D, QF, RG> LD;
  constexpr int DS = W::DS, CB = W::CB, kRows = 16 * RG;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63;
  const int g = wave % RG, u = wave / RG;
  W w;
  w.G = lane >> 4;
  w.li = lane & 15;
  w.bh_ = bh;
  const int64_t r = row0 + 16 * g + w.li;
  w.row[0] = r;
  const int64_t si = QF == 1 ? r / 64 : (r / 16) * 8 + r % 8;
  w.qsv[0] = si < a.qs_len ? a.qs[bh * a.qs_len + si] : 1.0f;
#pragma unroll
  for (int ds = 0; ds < DS; ++ds) {
    if (r < a.Nq) w.qf[0][ds] = *reinterpret_cast<const v4i*>(a.q8 + (bh * a.Nq + r) * D + ds * 64 + w.G * 16);
    else w.qf[0][ds] = v4i{0, 0, 0, 0};
    w.koff[ds] = w.li * D + ((((D == 128) ? 4 * ds : 0) + w.G) ^ chunk_xor<D>(w.li)) * 16;
  }
#pragma unroll
  for (int h = 0; h < 2; ++h) w.voff[h] = w.li * kTile + (((4 * h + w.G) ^ (w.li & 7)) * 16);
  w.m[0] = -5000000.0f;
  w.den[0] = 0.0f;
  w.dacc[0] = v4f{0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
  for (int j = 0; j < 4; ++j) w.wts[0][j] = 0.0f;
#pragma unroll
  for (int cb = 0; cb < CB; ++cb) w.O[0][cb] = v4f{0.0f, 0.0f, 0.0f, 0.0f};
  w.ones = v4i{0x22222222, 0x22222222, 0x22222222, 0x22222222};
  w.bacc = v4i{kBias, kBias, kBias, kBias};

  const int tiles = static_cast<int>(a.tiles);
  constexpr uint32_t kBuf = DB ? KS * LD::BYTES : 0;
  LD ld;
  ld.init(a, bh, lds + u * LD::BYTES, g, lane);
  ld.issue_k(u, 0);
  if constexpr (DB) ld.issue_v(u, 0);
  float run = -5000000.0f;  // the row's running maximum over all steps so far
  int c = 0;                // position in the chunk of pending mean weights (VM 1, 2)
  // One step. TAIL: the split may have no tile left, or the last one.
  auto step = [&](int s, auto tail) __attribute__((always_inline)) {
    constexpr bool TAIL = decltype(tail)::value;
    const int t = s + u;
    const bool mine = !TAIL || t < tiles, last = TAIL && t == tiles - 1;  // wave-uniform
    LD::wait();
    lds_barrier();  // K of this step has landed; V^T of the last step is read
    const uint32_t buf = DB ? ((s / KS) & 1) * kBuf : 0;
    const uint8_t* lk = lds + u * LD::BYTES + buf;
    const uint8_t* lv = lk + kTile * D;
    float bs[8][4], scl = 0.0f, tmax = -INFINITY;
    if (mine) {
      typename W::Acc Sq[8];
      v4i kf[8][DS];
      const float ksv = *reinterpret_cast<const float*>(lv + kTile * D + (QF == 1 ? 0 : 4 * w.G));
#pragma unroll
      for (int j = 0; j < 2; ++j)
#pragma unroll
        for (int ds = 0; ds < DS; ++ds) kf[j][ds] = *reinterpret_cast<const v4i*>(lk + j * 16 * D + w.koff[ds]);
#pragma unroll
      for (int j = 0; j < 8; ++j) {
        if (j + 2 < 8) {
#pragma unroll
          for (int ds = 0; ds < DS; ++ds) kf[j + 2][ds] = *reinterpret_cast<const v4i*>(lk + (j + 2) * 16 * D + w.koff[ds]);
        }
        Sq[j] = w.score(kf[j], w.qf[0]);
        // this step's share of the loads: V^T of this tile, or all of the next tile's
        constexpr int kLoads = (DB ? 2 : 1) * LD::kPart;
#pragma unroll
        for (int i = j * kLoads / 8; i < (j + 1) * kLoads / 8; ++i) {
          if constexpr (!DB) ld.part_v(i, t, 0);
          else if (i < LD::kPart) ld.part_k(i, t + KS, kBuf - buf);
          else ld.part_v(i - LD::kPart, t + KS, kBuf - buf);
        }
        __builtin_amdgcn_sched_barrier(0);
      }
      if (TAIL && last) tmax = w.template logits<true>(a, t, 0, Sq, ksv, bs, scl);
      else tmax = w.template logits<false>(a, t, 0, Sq, ksv, bs, scl);
      tmax = running_max(tmax, tmax);
    }
    // Slots alternate, so a wave's next write comes after every wave has read this step's.
    float* slot = xch + ((s / KS) & 1) * KS * kRows + 16 * g + w.li;
    if (w.G == 0) slot[u * kRows] = tmax;
    if constexpr (!DB) LD::wait();
    lds_barrier();  // the maxima are there; V^T has landed; K is read
    float mn = run, x[KS];
#pragma unroll
    for (int i = 0; i < KS; ++i) x[i] = slot[i * kRows];
#pragma unroll
    for (int i = 0; i < KS; ++i) {
      run = vmax(run, x[i]);
      mn = i <= u ? vmax(mn, x[i]) : mn;
    }
    if (mine) {
      if (wave_any(w.m[0] != mn)) w.rescale(0, w.m[0] - mn);
      w.m[0] = mn;
      v8i P;
      float tmass, mass[1];
      w.template bytes<false, false>(a, bs, scl, mn, __builtin_fmaf(-mn, kExpA, kExpB), P, tmass);
      const v4f zero = {0.0f, 0.0f, 0.0f, 0.0f};
      v8i vf[CB];
      vf[0] = w.load_v(lv, 0);
      vf[1] = w.load_v(lv, 1);
#pragma unroll
      for (int cb = 0; cb < CB; ++cb) {
        if (cb + 2 < CB) vf[cb + 2] = w.load_v(lv, cb + 2);
        if constexpr (W::BSCALE) {
          const float4 sc = *reinterpret_cast<const float4*>(a.vs + (bh * a.tiles + t) * D + 16 * cb + 4 * w.G);
          const v4f pv = mfma_fp8(vf[cb], P, zero);
          w.O[0][cb][0] = __builtin_fmaf(pv[0], sc.x, w.O[0][cb][0]);
          w.O[0][cb][1] = __builtin_fmaf(pv[1], sc.y, w.O[0][cb][1]);
          w.O[0][cb][2] = __builtin_fmaf(pv[2], sc.z, w.O[0][cb][2]);
          w.O[0][cb][3] = __builtin_fmaf(pv[3], sc.w, w.O[0][cb][3]);
        } else {
          w.O[0][cb] = mfma_fp8(vf[cb], P, w.O[0][cb]);
        }
        if constexpr (!DB) {
#pragma unroll
          for (int i = cb * LD::kPart / CB; i < (cb + 1) * LD::kPart / CB; ++i) ld.part_k(i, t + KS, 0);
        }
        __builtin_amdgcn_sched_barrier(0);
      }
      if constexpr (W::DACC) {
        w.dacc[0] = mfma_mass(w.ones, P, w.dacc[0]);
      } else {
        if constexpr (W::EC) mass[0] = mfma_mass(w.ones, P, zero)[0];
        else mass[0] = tmass;
        w.den[0] += mass[0];
      }
      if (a.pdump) w.dump_p(a, t, 0, P);
      if constexpr (W::SMOOTH) {
        const bool group = w.G == (c >> 2);
        switch (c & 3) {
          case 0: w.template set_weight<0>(group, mass); break;
          case 1: w.template set_weight<1>(group, mass); break;
          case 2: w.template set_weight<2>(group, mass); break;
          default: w.template set_weight<3>(group, mass); break;
        }
        if (c == kChunk - 1 || t + KS >= tiles) {
          // positions past c hold no weight: they read the chunk's tile c
          const int t0 = t - KS * c;
          auto at = [&](int pos, int ch) { return (bh * a.tiles + t0 + KS * (pos < c ? pos : c)) * D + ch; };
          w.flush_weights([&](int pos, int ch) { return reinterpret_cast<const _Float16*>(a.means)[at(pos, ch)]; },
                          [&](int pos, int ch) { return a.vs[at(pos, ch)]; });
          c = 0;
        } else {
          ++c;
        }
      }
    }
  };
  int s = 0;
  for (; s + KS <= tiles - 1; s += KS) step(s, std::false_type());
  for (; s < tiles; s += KS) step(s, std::true_type());

  // ---- the splits' sums at the final maximum, added in split order; wave (g, u) takes the
  // channel blocks u, u + KS, ... of its rows
  LD::wait();
  lds_barrier();  // the tile regions are free (no load is in flight, every wave is done reading)
  v4f* part = reinterpret_cast<v4f*>(lds);  // [KS][RG][CB][64]
  float* dens = xch + 2 * KS * kRows;       // [KS][kRows]
  const float dm = w.m[0] - run;
  const float alpha = W::EC ? __builtin_amdgcn_exp2f(dm * 1.44269504088896341f) : __builtin_amdgcn_exp2f(dm);
#pragma unroll
  for (int cb = 0; cb < CB; ++cb) part[(wave * CB + cb) * 64 + lane] = w.O[0][cb] * alpha;
  if (w.G == 0) dens[u * kRows + 16 * g + w.li] = (W::DACC ? w.dacc[0][0] : w.den[0]) * alpha;
  lds_barrier();
  if (r >= a.Nq) return;
  float den = dens[16 * g + w.li];
#pragma unroll
  for (int i = 1; i < KS; ++i) den += dens[i * kRows + 16 * g + w.li];
  const int64_t b = bh / a.H, h = bh % a.H;
  uint16_t* out = static_cast<uint16_t*>(a.out) + b * a.osb + h * a.osh + r * a.osn;
#pragma unroll
  for (int k = 0; k < (CB + KS - 1) / KS; ++k) {
    const int cb = u + KS * k;
    if (cb >= CB) break;
    v4f o = part[(g * CB + cb) * 64 + lane];
#pragma unroll
    for (int i = 1; i < KS; ++i) o += part[((i * RG + g) * CB + cb) * 64 + lane];
    if (a.out_bf16) store_row<D, VCX_BFLOAT16, W::BSCALE>(a, bh, out, 16 * cb + 4 * w.G, o, 1.0f / den);
    else store_row<D, VCX_FLOAT16, W::BSCALE>(a, bh, out, 16 * cb + 4 * w.G, o, 1.0f / den);
  }
}

// Eight waves, two per SIMD: 8 / RG splits, whose tiles of 32 KB (D128) or 16 KB (D64) the 160
// KB of LDS hold once (RG 2 at D128, RG 1 at D64) or twice.
template <int RG>
constexpr int kSplits = 8 / RG;
constexpr int kPieceThreads = 512;
constexpr int kWarm = 4;  // loads per thread of warm_l2

// One 128-byte line per load of the head's first tiles, shared out over the n pieces of the head
// on this XCD (this is the i-th): the pieces walk the tiles together, so without it every step
// waits for its tile from memory; with it for the XCD's L2. Nothing waits for these loads but
// the first tile's wait, which runs beside them. In calls that have just written K and V: [1,4,1024
// x 8192,128] with smoothing 51.9 -> 39.2 us, [1,2,2048,128] 15.0 -> 13.9 us.
template <int D>
__device__ __forceinline__ void warm_l2(const AttnArgs& a, int64_t bh, int64_t i, int64_t n, uint32_t (&sink)[kWarm]) {
  const int64_t npad = a.tiles * kTile, lines = a.tiles * 2 * D, valid = a.Nk * D / 128;
  const uint8_t* k = reinterpret_cast<const uint8_t*>(a.k8) + bh * a.Nk * D;
  const uint8_t* v = a.v8 + bh * D * npad;
#pragma unroll
  for (int e = 0; e < kWarm; ++e) {
    // lines in the order of the tiles: D of K, then D of V^T (one per channel)
    const int64_t l = (e * n + i) * kPieceThreads + threadIdx.x, t = l / (2 * D), r = l % (2 * D);
    const int64_t kl = t * D + r;
    const uint8_t* p = r < D ? k + (kl < valid ? kl : 0) * 128 : v + (r - D) * npad + t * kTile;
    sink[e] = *reinterpret_cast<const uint32_t*>(l < lines ? p : v);
  }
}

template <int D, int VM, int PM, int QF, int RG>
__global__ __launch_bounds__(kPieceThreads, 1) void attn_piece_kernel(AttnArgs a) {
#if defined(__HIP_DEVICE_COMPILE__)
  constexpr int kRows = 16 * RG, KS = kSplits<RG>;
  constexpr bool DB = 2 * KS * PieceLoader<D, QF, RG>::BYTES + 4096 < 160 * 1024;
  __shared__ __attribute__((aligned(16))) uint8_t lds[(DB ? 2 : 1) * KS * PieceLoader<D, QF, RG>::BYTES];
  __shared__ float xch[3 * KS * kRows];
  // contiguous (head, row) ranges per XCD, as in attn_kernel
  const int64_t per = gridDim.x / 8, rem = gridDim.x % 8, xcd = blockIdx.x % 8, j = blockIdx.x / 8;
  const int64_t logical = (xcd < rem ? xcd * (per + 1) : rem * (per + 1) + (xcd - rem) * per) + j;
  const int64_t pieces = (a.Nq + kRows - 1) / kRows, bh = logical / pieces;
  // this XCD's pieces of the head
  const int64_t lo0 = logical - j, hi0 = lo0 + per + (xcd < rem ? 1 : 0);
  const int64_t lo = lo0 > bh * pieces ? lo0 : bh * pieces, hi = hi0 < (bh + 1) * pieces ? hi0 : (bh + 1) * pieces;
  uint32_t sink[kWarm];
  warm_l2<D>(a, bh, logical - lo, hi - lo, sink);
  attn_piece<D, VM, PM, QF, RG, KS, DB>(a, bh, logical % pieces * kRows, lds, xch);
#pragma unroll
  for (int e = 0; e < kWarm; ++e) asm volatile("" ::"v"(sink[e]));  // the loads are used
#else
  (void)a;
#endif
}

template <int D, int VM, int PM, int QF>
int launch(const AttnArgs& a, int64_t BH, int groups, hipStream_t st) {
  auto go = [&](auto rg) {
    constexpr int RG = decltype(rg)::value;
    const unsigned grid = static_cast<unsigned>(BH * cdiv(a.Nq, 16 * RG));
    attn_piece_kernel<D, VM, PM, QF, RG><<<dim3(grid), kPieceThreads, 0, st>>>(a);
  };
  if constexpr (D == 64) {
    if (groups == 1) {
      go(std::integral_constant<int, 1>());
      return check_launch("attn_piece_kernel");
    }
  }
  if (groups == 2) go(std::integral_constant<int, 2>());
  else go(std::integral_constant<int, 4>());
  return check_launch("attn_piece_kernel");
}

template <int D, int VM, int QF>
int launch_mode(const AttnArgs& a, int64_t BH, int groups, int mode, hipStream_t st) {
  if constexpr (VM == 0) {
    if (mode == 2) return launch<D, VM, 2, QF>(a, BH, groups, st);
  }
  return mode == 1 ? launch<D, VM, 1, QF>(a, BH, groups, st) : launch<D, VM, 0, QF>(a, BH, groups, st);
}

template <int D>
int launch_values(const AttnArgs& a, int64_t BH, int groups, int vm, int mode, int qf, hipStream_t st) {
  if (qf) return launch_mode<D, 0, 1>(a, BH, groups, mode, st);
  if (vm == 0) return launch_mode<D, 0, 0>(a, BH, groups, mode, st);
  return vm == 1 ? launch_mode<D, 1, 0>(a, BH, groups, mode, st) : launch_mode<D, 2, 0>(a, BH, groups, mode, st);
}

}  // namespace

// 16-row groups per piece: the fewest whose pieces all run at once, one per CU, else 0 (a call
// with more rows fills the chip with attn_kernel's blocks, which stream a tile for 64 or 128
// rows). Fewer rows per piece mean more splits of the tiles and so a shorter chain. At D128 a
// 16-row piece would need eight 32 KB tiles in LDS; with four waves of one tile each it lost to
// two groups (36 against 33 us at [1,4,1024 x 8192,128] with smoothing). Same box, kernel time
// in us, attn_kernel and 1 / 2 / 4 groups:
//   [1,2,2048,128]                  18.7    - / 12.6 / 17.9
//   [1,4,1024 x 8192,128] smoothing 61.0    - / 33.1 / 57.2, control 83.3  - / 47.2 / 86.1
//   [1,8,1024 x 8192,128]           54.1    - / 35.0 / 51.5
//   [1,8,2048 x 8192,128]           59.2    - / 66.4 (512 pieces) / 54.0
//   [1,4,1024 x 8192,64] smoothing  47.7  20.7 / 28.8 / 44.9
//   [1,8,2048 x 8192,64] smoothing  48.5    - / 55.6 (512 pieces) / 45.7
// And 0 where the keys are too few for the splits to pay, as a piece starts and ends more slowly
// than a block (pieces' time over attn_kernel's in replayed graphs, by key tiles; the folded
// encode of INT8 scores / the other modes):
//   1 or 2 groups, D64   1: 1.03-1.07 / 1.26-1.46, 2: 0.93-0.98 / 1.04-1.26, 3: 0.90 / 0.89-1.14,
//                        4: 0.83 / 0.76-1.01, 8: 0.70-0.83 / 0.57-0.89
//   2 groups, D128       1: 1.00 / 1.18-1.28, 2: 0.91 / 0.93-1.11, 4: 0.82 / 0.77-0.96, 8: 0.78 / 0.70-0.85
// With four groups the two splits stand against attn_kernel's 64-row blocks, which the same rows
// fill the chip with if the 128-row blocks deal out evenly over the XCDs (tail_split halves equally
// many on each). There the splits pay late, or not at all at D128 (64 tiles: folded 1.00, control
// 1.04-1.09), but for per-block V scales (8 tiles 0.91-0.99, 64 tiles 0.73-0.89) and the folded encode
// of D64 or FP8 scores (8 tiles 0.89-0.98, 64 tiles 0.68-0.97); the rest of D64: 8 tiles 1.00-1.10, 24 tiles
// 0.91-1.00, 64 tiles 0.89-1.04; at D128 without the control path 256 tiles 0.80-1.02, the less the
// more heads (K and V past the caches). Where they don't, attn_kernel keeps 128-row blocks, and pieces take
// 0.55-0.73 of its time at [1,9,1100 x 1024..8192].
// Up to eight pieces, one per XCD, each pays for its own code's way to the caches, which is
// shorter for pieces: [1,1,64 x 77,128] 6.5-7.5 against 9.6-10.6 us, [1,1,64 x 256,64] 5.8-6.4 against 8.3-9.0.
int piece_groups(int64_t BH, int64_t Nq, int64_t tiles, int64_t D, int vm, int mode, int qf) {
  int dev = 0, cus = 0;
  if (hipGetDevice(&dev) != hipSuccess ||
      hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess)
    return 0;
  for (int rg = D == 128 ? 2 : 1; rg <= 4; rg *= 2) {
    const int64_t pieces = BH * cdiv(Nq, 16 * rg);
    if (pieces > cus) continue;
    if (pieces <= 8) return tiles >= (D == 128 ? 1 : 2) ? rg : 0;
    const bool folded = mode == 2;
    if (rg < 4 || BH * cdiv(Nq, kRowsPerBlock) % 8 != 0) return tiles >= (folded && !qf ? 2 : 4) ? rg : 0;
    if (vm == 2 || (folded && (D == 64 || qf))) return tiles >= 8 ? rg : 0;
    return D == 64 ? (tiles >= 24 ? rg : 0) : (mode != 0 && tiles >= 192 ? rg : 0);
  }
  return 0;
}

int launch_pieces(const AttnArgs& a, int64_t BH, int64_t D, int groups, int vm, int mode, int qf, hipStream_t st) {
  return D == 128 ? launch_values<128>(a, BH, groups, vm, mode, qf, st)
                  : launch_values<64>(a, BH, groups, vm, mode, qf, st);
}

}  // namespace vcx
