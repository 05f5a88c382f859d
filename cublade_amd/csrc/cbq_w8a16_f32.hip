// cbq_w8a16_f32.hip - W8A16 linear with fp32 activations on the matrix cores of
// gfx950 (K % 64 == 0, no outlier columns).
//
// The weights are int8 codes, exact in fp16 and bf16, so the products of x with
// them are exact in fp32 if x is a sum of 16-bit numbers. k_f32_planes writes each
// row of x as two fp16 planes, x 2^e = hi + 2^-11 lo, with e such that the largest
// magnitude is in [2^14, 2^15): 22 significant bits for elements down to 2^-29 of the
// largest (lo is held 2^11 up, so that it stays a normal number as long as hi
// does), 16 or more down to 2^-34. Infinities and NaN are hi, with lo = 0.
//
// Elements outside that band of 35 powers of two (the band is where most of the
// row's elements are, if the row spans more) are far elements: 0 in the planes, and
// their 64-k step noted in a mask of the row. k_gemm_f32 takes them from x itself,
// as three bf16 numbers (24 bits: exact), in the steps that a wave's 32 rows note.
//
// So no element's precision depends on what else its row holds, and the time
// depends on the values only where there are far elements: M = 500, N = 11008, K = 4096
// takes 95 us for N(0, 1), for outlier columns, NaN and subnormal rows, 108 with a
// feature of 1e20 in every row, 145 for the SiLU of N(0, 6^2) (far elements in 30% of
// a tile's steps), 377 with far elements in every step of every tile.
//
// k_gemm_f32 adds the planes' products in fp32, each plane in accumulators of its
// own, and finishes with y[m, n] = s[n] (2^-e[m] (hi + 2^-11 lo) + far) + bias[n]. For
// N(0, 1) at K = 4096 the result is 1.7e-7 from the 64-bit one (relative, 2-norm).
//
// Two fp16 products cost 2 units of matrix-core time. Three int8 digits of x
// against the row's largest element cost 1.5 (the call above took 77 us), but
// lose the small elements of a row next to large ones, whole where the weights are
// zero at the large ones.
#include <algorithm>
#include <type_traits>

#include "cbq_device.h"
#include "cbq_host.h"
#include "cbq_lds_dma.h"
#include "cbq_mfma.h"
#include "cbq_w8a16_f32.h"

namespace cbq {
namespace {

constexpr int kBand = 34;   // a band: the largest exponent and this many below it
// 64-k steps after which the first plane's sums go to a second set of registers: the
// sums in the accumulators stay small and so do their roundings (distance from the
// 64-bit result at K = 4096 4.1e-7 without, 1.7e-7 with; 1% of the time).
constexpr int kRun = 12;

struct F32Args {
  const float* x;          // [M, K]
  const uint16_t* xp;      // [2][M, K] planes
  const int* exps;         // [M] e of the row (low 16 bits), and g: its far elements count times 2^g
  const uint64_t* far;     // [M] bit i: far elements in 64-k steps [i << far_shift, (i + 1) << far_shift)
  const int8_t* wq;        // [N, K]
  const float* scales;     // [N]
  const float* bias;       // [N] or null
  float* y;                // [M, N]
  float* part;             // SPLIT: [splits][M, N] fp32 sums
  int M, N, K;
  int tiles_m, tiles_n;
  int splits, split_steps; // k-ranges of split_steps 64-k steps
  int far_shift;
};

// floor(log2) of a positive finite float given as its bits (subnormals too).
__device__ __forceinline__ int exp2_floor(uint32_t b) {
  return b >= 0x00800000u ? static_cast<int>(b >> 23) - 127 : 31 - __builtin_clz(b) - 149;
}

// The largest exponent of the band that holds most of the row's finite non-zero
// elements. Subnormal numbers count as exponent -127, which
// their magnitude stays below.
template <int V>
__device__ int fullest_band(const float4* x4, int n4, float4 (&r)[V]) {
  static_assert(kBlock == 256, "one exponent per thread");
  __shared__ unsigned int hist[256];
  __shared__ unsigned long long s_best[kBlock / kWave];
  const int t = threadIdx.x;
  hist[t] = 0u;
  __syncthreads();
  for (int i0 = 0; i0 < n4; i0 += V * kBlock)
#pragma unroll
    for (int v = 0; v < V; ++v) {
      const int i = i0 + v * kBlock + t;
      if (i >= n4) continue;
      const float4 q = n4 > V * kBlock ? x4[i] : r[v];
      const float f[4] = {q.x, q.y, q.z, q.w};
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const uint32_t b = __float_as_uint(f[e]) & 0x7fffffffu;
        if (b != 0u && b < 0x7f800000u) atomicAdd(&hist[b >> 23], 1u);
      }
    }
  __syncthreads();
  unsigned long long best = 0;
  for (int j = max(0, t - kBand); j <= t; ++j) best += hist[j];
  best = best << 8 | (255 - t);   // of equal ones the lowest, whose largest exponent occurs
#pragma unroll
  for (int o = 1; o < kWave; o <<= 1) best = max(best, __shfl_xor(best, o));
  if (t % kWave == 0) s_best[t / kWave] = best;
  __syncthreads();
#pragma unroll
  for (int w = 0; w < kBlock / kWave; ++w) best = max(best, s_best[w]);
  return 255 - static_cast<int>(best & 255u) - 127;
}

// Whether finite non-zero x (else false) lies outside the band whose largest
// exponent is top: [low, high).
struct Band {
  float low, high;
  __device__ __forceinline__ explicit Band(int top)
      : low(__builtin_ldexpf(1.0f, top - kBand)), high(__builtin_ldexpf(1.0f, top + 1)) {}
  __device__ __forceinline__ bool outside(float x) const {
    const float a = __builtin_fabsf(x);
    return (a < low || a >= high) && a > 0.0f && a < __builtin_inff();
  }
};

// One workgroup per row: its smallest and largest magnitude, the band, then the planes.
// Rows of up to 1024 V elements stay in registers between the two. Bound: memory
// (x read, as many bytes written).
template <int V>   // float4 per thread and step
__global__ __launch_bounds__(kBlock) void k_f32_planes(F32Args a, uint16_t* __restrict__ xp,
                                                       int* __restrict__ exps,
                                                       uint64_t* __restrict__ far) {
  __shared__ uint32_t s_max[kBlock / kWave], s_min[kBlock / kWave];
  __shared__ unsigned int s_far[2];
  const int m = blockIdx.x, t = threadIdx.x;
  const int n4 = a.K >> 2;
  const int64_t base = static_cast<int64_t>(m) * a.K;
  const float4* const x4 = reinterpret_cast<const float4*>(a.x + base);
  float4 r[V];
  uint32_t mx = 0u, mn = 0xffffffffu;   // of |x|'s bits, and of those less one (0: the largest)
  if (t < 2) s_far[t] = 0u;
  for (int i0 = 0; i0 < n4; i0 += V * kBlock) {
#pragma unroll
    for (int v = 0; v < V; ++v) {
      const int i = i0 + v * kBlock + t;
      r[v] = i < n4 ? x4[i] : make_float4(0.0f, 0.0f, 0.0f, 0.0f);
    }
#pragma unroll
    for (int v = 0; v < V; ++v) {
      const float f[4] = {r[v].x, r[v].y, r[v].z, r[v].w};
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const uint32_t b = __float_as_uint(f[e]) & 0x7fffffffu;
        const uint32_t fin = b < 0x7f800000u ? b : 0u;
        mx = max(mx, fin);
        mn = min(mn, fin - 1u);
      }
    }
  }
#pragma unroll
  for (int o = 1; o < kWave; o <<= 1) {
    mx = max(mx, static_cast<uint32_t>(__shfl_xor(static_cast<int>(mx), o)));
    mn = min(mn, static_cast<uint32_t>(__shfl_xor(static_cast<int>(mn), o)));
  }
  if (t % kWave == 0) {
    s_max[t / kWave] = mx;
    s_min[t / kWave] = mn;
  }
  __syncthreads();
#pragma unroll
  for (int w = 0; w < kBlock / kWave; ++w) {
    mx = max(mx, s_max[w]);
    mn = min(mn, s_min[w]);
  }
  int top = mx ? exp2_floor(mx) : 14;
  const bool wide = mx && exp2_floor(mn + 1u) < top - kBand;
  if (wide) top = fullest_band<V>(x4, n4, r);
  const Band band(top);
  const int e = 14 - top;
  // up to 1 where the sums stay far from the largest number: subnormal bf16 parts lose bits
  const int g = wide ? max(0, min(kBand - top, 100 - exp2_floor(mx))) : 0;

  const int64_t plane = static_cast<int64_t>(a.M) * a.K;
  for (int i0 = 0; i0 < n4; i0 += V * kBlock) {
#pragma unroll
    for (int v = 0; v < V; ++v) {
      const int i = i0 + v * kBlock + t;
      if (i >= n4) continue;
      if (n4 > V * kBlock) r[v] = x4[i];
      const float f[4] = {r[v].x, r[v].y, r[v].z, r[v].w};
      uint32_t hi[4], lo[4];
      bool any = false;
#pragma unroll
      for (int k = 0; k < 4; ++k) {
        const bool out = wide && band.outside(f[k]);
        any |= out;
        const float z = out ? 0.0f : __builtin_ldexpf(f[k], e);
        const _Float16 h = static_cast<_Float16>(z);
        const bool fin = __builtin_fabsf(z) < __builtin_inff();
        const float rest = fin ? (z - static_cast<float>(h)) * 2048.0f : 0.0f;   // exact
        hi[k] = __builtin_bit_cast(uint16_t, h);
        lo[k] = __builtin_bit_cast(uint16_t, static_cast<_Float16>(rest));
      }
      if (any) {
        const int bit = (i >> 4) >> a.far_shift;   // 16 float4 per 64-k step
        atomicOr(&s_far[bit >> 5], 1u << (bit & 31));
      }
      uint16_t* const p = xp + base + 4 * i;
      *reinterpret_cast<uint2*>(p) = make_uint2(hi[0] | (hi[1] << 16), hi[2] | (hi[3] << 16));
      *reinterpret_cast<uint2*>(p + plane) = make_uint2(lo[0] | (lo[1] << 16), lo[2] | (lo[3] << 16));
    }
  }
  __syncthreads();
  if (t == 0) {
    exps[m] = (e & 0xffff) | g << 16;
    far[m] = static_cast<uint64_t>(s_far[1]) << 32 | s_far[0];
  }
}

// 8 floats times scale (a power of two), those inside the band as 0, as hi + mid + lo
// (bf16, truncated: exact).
__device__ __forceinline__ void split_far(const float (&x)[8], const Band& band, float scale,
                                          u32x4 (&out)[3]) {
#pragma unroll
  for (int w = 0; w < 4; ++w) {
    uint32_t part[3][2];
#pragma unroll
    for (int k = 0; k < 2; ++k) {
      float rest = band.outside(x[2 * w + k]) ? x[2 * w + k] * scale : 0.0f;
#pragma unroll
      for (int q = 0; q < 3; ++q) {
        part[q][k] = __float_as_uint(rest) & 0xffff0000u;
        rest -= __uint_as_float(part[q][k]);
      }
    }
#pragma unroll
    for (int q = 0; q < 3; ++q) out[q][w] = part[q][1] | (part[q][0] >> 16);
  }
}

// Tile of 32 WM rows of x (both planes) by 32 TN (8 / WM) weight rows, 8 waves (two
// per SIMD), each 32 x 32 TN: 32 TN accumulators. 64-k steps through three LDS
// stages filled by LDS DMA (two steps in flight), one barrier per step between
// its two halves; per half a wave reads TN + 4 fragments for 4 TN MFMAs. A
// weight fragment is widened once for both planes, the next tile's one word after
// each MFMA; the reads and the DMA of step t + 3 are spread between the MFMAs too
// (as in k_gemm_dma). LDS reads: 73 bytes per clock of MFMA time at TN = 3 (128
// available). x rows of 128 bytes (chunk c of row r at c ^ ((r >> 1) & 7)), weight
// rows of 64 (c ^ ((r >> 2) & 3)): no bank conflicts. Rows past M or N are clamped
// for the loads and not stored. MFMA A = x, B = weights: lane l holds n = l % 32
// and m = 8 (v / 4) + 4 (l / 32) + v % 4, so a store writes two 128-byte runs.
//
// Far elements (in the steps noted by any of a wave's 32 rows) follow the k loop, from
// x and the weight in global memory, one step at a time (loads of the next half in
// flight: level, 4.6 us per step either way).
template <int TN, int WM, bool SPLIT>
__global__ __launch_bounds__(512) void k_gemm_f32(F32Args a) {
  constexpr int WN = 8 / WM, BM = 32 * WM, BN = 32 * TN * WN, NS = 3;
  constexpr int XP = BM / 8, XI = 2 * XP, TI = XI + BN / 16;   // 1 KiB DMA instructions per step
  constexpr int XB = XI * 1024;
  constexpr int L = (TI + 7) / 8;                      // per wave (the last one: waves < TI % 8)
  constexpr int SB = TI * 1024;
  constexpr int WREM = TI % 8;                         // waves that issue L (0: all)
  static_assert(XP % 8 == 0, "an instruction slot is of one plane or the weights for all waves");
  static_assert(NS * SB <= 160 * 1024, "stages fit in LDS");
  __shared__ __attribute__((aligned(1024))) uint8_t smem[NS * SB];

  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int wm = wave % WM, wn = wave / WM;
  // XCD b % 8 takes a contiguous run of tiles, in groups of 8 tile rows
  const int total = a.tiles_m * a.tiles_n * (SPLIT ? a.splits : 1), per = total >> 3;
  int b = static_cast<int>(blockIdx.x);
  if (b < per * 8) b = (b & 7) * per + (b >> 3);
  const int split = SPLIT ? b / (a.tiles_m * a.tiles_n) : 0;
  const int lt = SPLIT ? b % (a.tiles_m * a.tiles_n) : b;
  constexpr int G = 8;
  const int group = lt / (G * a.tiles_n), gm = min(a.tiles_m - group * G, G);
  const int m0 = (group * G + lt % (G * a.tiles_n) % gm) * BM;
  const int n0 = lt % (G * a.tiles_n) / gm * BN;
  const int kb = SPLIT ? split * a.split_steps : 0;
  const int nk = SPLIT ? min(a.split_steps, a.K / 64 - kb) : a.K / 64;
  const uint32_t sbase = __builtin_amdgcn_readfirstlane(lds_addr(smem));

  // DMA instruction u of this wave is instruction 8 u + wave of the step: 8 rows of
  // the first plane, of the second, then 16 weight rows.
  uint32_t off[L];
  const uint8_t* src[L];
#pragma unroll
  for (int u = 0; u < L; ++u) {
    const int q = u * 8 + wave;
    if (u * 8 < XI) {
      const int row = (q % XP) * 8 + (lane >> 3), c = (lane & 7) ^ ((row >> 1) & 7);
      off[u] = static_cast<uint32_t>(min(m0 + row, a.M - 1)) * static_cast<uint32_t>(a.K) * 2u + c * 16u;
      src[u] = uniform_ptr(reinterpret_cast<const uint8_t*>(
          a.xp + static_cast<int64_t>(u * 8 / XP) * a.M * a.K + kb * 64));
    } else {
      const int row = (q - XI) * 16 + (lane >> 2), c = (lane & 3) ^ ((row >> 2) & 3);
      off[u] = static_cast<uint32_t>(min(n0 + row, a.N - 1)) * static_cast<uint32_t>(a.K) + c * 16u;
      src[u] = uniform_ptr(reinterpret_cast<const uint8_t*>(a.wq) + kb * 64);
    }
  }
  auto issue_one = [&](int t, int stage, int u) {
    if (WREM == 0 || u < L - 1 || wave < WREM)
      lds_dma16(off[u], uniform_ptr(src[u] + t * (u * 8 < XI ? 128 : 64)),
                sbase + stage * SB + (u * 8 + wave) * 1024);
  };
  // At most T tiles' DMA of this wave outstanding, then the barrier.
  auto wait_tiles = [&](auto tiles) {
    constexpr int T = decltype(tiles)::value;
    if (WREM == 0 || wave < WREM) dma_wait_barrier<T * L>();
    else dma_wait_barrier<T * (L - 1)>();
  };

  const int r32 = lane & 31, h = lane >> 5;
  uint32_t xr[2][2], wr[2];   // half e, slice s: x chunk 4 h + 2 e + s, weight chunk 2 h + e
#pragma unroll
  for (int e = 0; e < 2; ++e) {
#pragma unroll
    for (int s = 0; s < 2; ++s)
      xr[e][s] = (wm * 32 + r32) * 128 + (((4 * h + 2 * e + s) ^ ((r32 >> 1) & 7)) << 4);
    wr[e] = XB + (wn * 32 * TN + r32) * 64 + (((2 * h + e) ^ ((r32 >> 2) & 3)) << 4);
  }
  struct Frags {
    u32x4 x[2][2], w[TN];   // x: [plane][slice]
  };
  auto read_one = [&](int stage, int e, Frags& f, int r) {
    const uint8_t* st = smem + stage * SB;
    if (r < TN) f.w[r] = *reinterpret_cast<const u32x4*>(st + wr[e] + r * 2048);
    else f.x[(r - TN) >> 1][(r - TN) & 1] =
        *reinterpret_cast<const u32x4*>(st + xr[e][(r - TN) & 1] + ((r - TN) >> 1) * (BM * 128));
  };
  using std::integral_constant;
  using yes = std::true_type;
  using no = std::false_type;

  f16x acc[2][TN], sum[TN];   // sum: what acc[0] held at the ends of earlier runs of steps
#pragma unroll
  for (int i = 0; i < TN; ++i) acc[0][i] = acc[1][i] = sum[i] = f16x{};
  constexpr int Q = 4 * TN, R = TN + 4;
  Frags f0, f1;
  u32x4 wa[2], wb[2];         // widened weights: this and the next tile
  auto widen = [&](const Frags& f, int i, int c, u32x4 (&w)[2]) {
    const uint32_t word = c == 0 ? f.w[i].x : c == 1 ? f.w[i].y : c == 2 ? f.w[i].z : f.w[i].w;
    uint32_t lo, hi;
    i8x4_to_act<kF16>(word, lo, hi);
    w[c >> 1][(c & 1) * 2] = lo;
    w[c >> 1][(c & 1) * 2 + 1] = hi;
  };
  // One half of a step from f, widening fnext's first tile at its end (more); slots of
  // one MFMA, each followed by extra(slot). par: which of wa and wb holds tile 0.
  auto half = [&](const Frags& f, const Frags& fnext, auto more, int par, auto&& extra) {
    constexpr bool MORE = decltype(more)::value;
#pragma unroll
    for (int i = 0; i < TN; ++i) {
      u32x4(&cur)[2] = ((i + par) & 1) ? wb : wa;
      u32x4(&nxt)[2] = ((i + par) & 1) ? wa : wb;
#pragma unroll
      for (int p = 0; p < 4; ++p) {
        acc[p & 1][i] = mfma32x32x16<kF16>(f.x[p & 1][p >> 1], cur[p >> 1], acc[p & 1][i]);
        if constexpr (TN == 1) {   // the next half's tile is read at slot 0
#pragma unroll
          for (int c = 0; c < 4; ++c)
            if (MORE && (c + 1 < 4 ? c + 1 : 3) == p) widen(fnext, 0, c, nxt);
        } else {
          if (i + 1 < TN) widen(f, i + 1, p, nxt);
          else if (MORE) widen(fnext, 0, p, nxt);
        }
        extra(i * 4 + p);
        __builtin_amdgcn_sched_barrier(0);
      }
    }
  };
  // Step t: f0 holds half 0 of tile t and wa its first weights, widened; its
  // MFMAs run with the reads of half 1 between them, then the wait for tile t + 1
  // and the barrier (every wave is done with tile t's stage), then half 1 with the
  // DMA of tile t + 3 into that stage and the reads of tile t + 1's half 0. SC: t %
  // NS where known (the stage folds into the instructions' offsets), else -1.
  auto step = [&](int t, auto dma, auto ahead, auto sc) {
    constexpr int SC = decltype(sc)::value;
    const int cur = SC >= 0 ? SC : t % NS, nxt = SC >= 0 ? (SC + 1) % NS : (t + 1) % NS;
    half(f0, f1, yes{}, 0, [&](int q) {
#pragma unroll
      for (int r = q; r < R; r += Q) read_one(cur, 1, f1, r);
    });
    wait_tiles(ahead);
    __builtin_amdgcn_sched_barrier(0);
    half(f1, f0, yes{}, TN & 1, [&](int q) {
      if constexpr (decltype(dma)::value)
#pragma unroll
        for (int u = q; u < L; u += Q) issue_one(t + NS, cur, u);
#pragma unroll
      for (int r = q; r < R; r += Q) read_one(nxt, 0, f0, r);
    });
  };
#pragma unroll
  for (int t = 0; t < NS; ++t)
    if (t < nk)
#pragma unroll
      for (int u = 0; u < L; ++u) issue_one(t, t, u);
  if (nk > 2) wait_tiles(integral_constant<int, 2>{});
  else if (nk > 1) wait_tiles(integral_constant<int, 1>{});
  else wait_tiles(integral_constant<int, 0>{});
#pragma unroll
  for (int r = 0; r < R; ++r) read_one(0, 0, f0, r);
#pragma unroll
  for (int c = 0; c < 4; ++c) widen(f0, 0, c, wa);
  using one = integral_constant<int, 1>;
  using any = integral_constant<int, -1>;
  int t = 0;
  for (; t + NS + 2 < nk; t += NS) {
    step(t, yes{}, one{}, integral_constant<int, 0>{});
    step(t + 1, yes{}, one{}, integral_constant<int, 1>{});
    step(t + 2, yes{}, one{}, integral_constant<int, 2>{});
    if (t % kRun == kRun - NS) {
#pragma unroll
      for (int i = 0; i < TN; ++i) {
        sum[i] += acc[0][i];
        acc[0][i] = f16x{};
      }
    }
  }
  for (; t + NS < nk; ++t) step(t, yes{}, one{}, any{});
  if (t + 2 < nk) step(t++, no{}, one{}, any{});
  if (t + 1 < nk) step(t++, no{}, integral_constant<int, 0>{}, any{});
  half(f0, f1, yes{}, 0, [&](int q) {
#pragma unroll
    for (int r = q; r < R; r += Q) read_one((nk - 1) % NS, 1, f1, r);
  });
  half(f1, f0, no{}, TN & 1, [&](int) {});

  const int mw = m0 + wm * 32, nw = n0 + wn * 32 * TN;
  const int ml = min(mw + r32, a.M - 1);
  uint64_t far = a.far[ml];   // of this wave's 32 rows
  int ex[16];
#pragma unroll
  for (int v = 0; v < 16; ++v) {
    ex[v] = a.exps[min(mw + 8 * (v >> 2) + 4 * h + (v & 3), a.M - 1)];
#pragma unroll
    for (int i = 0; i < TN; ++i)
      sum[i][v] = __builtin_ldexpf(
          __builtin_fmaf(acc[1][i][v], 0x1p-11f, sum[i][v] + acc[0][i][v]),
          -static_cast<int16_t>(ex[v]));
  }
  if (__any(far != 0)) {
#pragma unroll
    for (int o = 1; o < 32; o <<= 1) far |= __shfl_xor(static_cast<unsigned long long>(far), o);
    const uint32_t flo = __builtin_amdgcn_readfirstlane(static_cast<uint32_t>(far));
    const uint32_t fhi = __builtin_amdgcn_readfirstlane(static_cast<uint32_t>(far >> 32));
    const int eg = a.exps[ml];
    const Band band(14 - static_cast<int16_t>(eg));
    const float scale = __builtin_ldexpf(1.0f, eg >> 16);
    const float* const xrow = a.x + static_cast<int64_t>(ml) * a.K + 32 * h;
#pragma unroll
    for (int i = 0; i < TN; ++i) acc[0][i] = f16x{};
    for (int k64 = kb; k64 < kb + nk; ++k64) {
      const int bit = k64 >> a.far_shift;
      if (!(((bit & 32 ? fhi : flo) >> (bit & 31)) & 1u)) continue;
#pragma unroll
      for (int e = 0; e < 2; ++e) {
        u32x4 wf[TN], xs[2][3];
#pragma unroll
        for (int i = 0; i < TN; ++i)
          wf[i] = *reinterpret_cast<const u32x4*>(
              a.wq + static_cast<int64_t>(min(nw + 32 * i + r32, a.N - 1)) * a.K + k64 * 64 +
              32 * h + 16 * e);
#pragma unroll
        for (int s = 0; s < 2; ++s) {
          const float4* const p = reinterpret_cast<const float4*>(xrow + k64 * 64 + 16 * e + 8 * s);
          const float4 u = p[0], v = p[1];
          const float x8[8] = {u.x, u.y, u.z, u.w, v.x, v.y, v.z, v.w};
          split_far(x8, band, scale, xs[s]);
        }
#pragma unroll
        for (int i = 0; i < TN; ++i)
#pragma unroll
          for (int s = 0; s < 2; ++s) {
            uint32_t o[4];
            i8x4_to_act<kBF16>(s ? wf[i].z : wf[i].x, o[0], o[1]);
            i8x4_to_act<kBF16>(s ? wf[i].w : wf[i].y, o[2], o[3]);
#pragma unroll
            for (int q = 0; q < 3; ++q)
              acc[0][i] = mfma32x32x16<kBF16>(xs[s][q], u32x4{o[0], o[1], o[2], o[3]}, acc[0][i]);
          }
      }
    }
#pragma unroll
    for (int v = 0; v < 16; ++v)
#pragma unroll
      for (int i = 0; i < TN; ++i) sum[i][v] += __builtin_ldexpf(acc[0][i][v], -(ex[v] >> 16));
  }

  float* const out = SPLIT ? a.part + static_cast<int64_t>(split) * a.M * a.N : a.y;
#pragma unroll
  for (int i = 0; i < TN; ++i) {
    const int n = nw + 32 * i + r32;
    const float sc = SPLIT || n >= a.N ? 1.0f : a.scales[n];
    const float bs = SPLIT || n >= a.N || !a.bias ? 0.0f : a.bias[n];
#pragma unroll
    for (int v = 0; v < 16; ++v) {
      const int m = mw + 8 * (v >> 2) + 4 * h + (v & 3);
      float f = sum[i][v];
      if constexpr (!SPLIT) f = a.bias ? f * sc + bs : f * sc;
      if (m < a.M && n < a.N) out[static_cast<int64_t>(m) * a.N + n] = f;
    }
  }
}

// y = s[n] * (the k-ranges' sums in order) + bias[n]; four outputs per thread
// (N % 4 == 0) or one.
template <int E>
__global__ __launch_bounds__(kBlock) void k_f32_reduce(F32Args a) {
  const int64_t mn = static_cast<int64_t>(a.M) * a.N;
  const int64_t i = (static_cast<int64_t>(blockIdx.x) * kBlock + threadIdx.x) * E;
  if (i >= mn) return;
  typedef float fe __attribute__((ext_vector_type(E)));
  fe sum = *reinterpret_cast<const fe*>(a.part + i);
  for (int s = 1; s < a.splits; ++s) sum += *reinterpret_cast<const fe*>(a.part + s * mn + i);
  const int n = static_cast<int>(i % a.N);
#pragma unroll
  for (int e = 0; e < E; ++e) {
    float f = sum[e] * a.scales[n + e];
    if (a.bias) f += a.bias[n + e];
    a.y[i + e] = f;
  }
}

struct F32Plan {
  int wm, tn, splits, steps;   // waves along M, weight tiles per wave, k-ranges, 64-k steps each
};

// The tile and k-ranges with the lowest modelled time (0.01 us), fitted on
// MI355X over 27 shapes (M = 1 .. 4096, N and K = 256 .. 14336): a 64-k step
// costs more the more CUs are busy (0.82 + 0.55 us x their share for 128 x 192
// tiles, 0.48 + 0.50 for 128 x 128, 0.33 + 0.29 for 128 x 64; M <= 64: 0.73 +
// 0.53, 0.48 + 0.32 and 0.20 + 0.27 for 64 x 384, 256 and 128), a split 0.3 us
// + 0.33 us per range and 1.8 us per 4 MiB of partial sums. Within 4% of the
// best plan measured. M = 256, N = 11008, K = 4096: 128 x 128 whole 57.1 us, 128 x
// 192 in two ranges 61.6; M = 128: 128 x 64 whole 39.2, 128 x 128 in two 39.5.
F32Plan f32_plan(int64_t M, int64_t N, int64_t K) {
  const int64_t cus = device_cus(), nk = K / 64;
  const int wm = M <= 64 ? 2 : 4;
  constexpr int64_t kBase[2][4] = {{0, 20, 48, 73}, {0, 33, 48, 82}};
  constexpr int64_t kBusy[2][4] = {{0, 27, 32, 53}, {0, 29, 50, 55}};
  F32Plan best{wm, 1, 1, static_cast<int>(nk)};
  int64_t best_cost = INT64_MAX;
  for (const int tn : {3, 2, 1}) {
    const int64_t tiles = cdiv(M, 32LL * wm) * cdiv(N, 32LL * tn * (8 / wm));
    for (int64_t sp = 1; sp <= 16; ++sp) {
      if (sp > 1 && (tiles * sp > cus || nk / sp < 4)) break;
      const int64_t steps = cdiv(nk, sp), full = tiles * sp / cus, rest = tiles * sp % cus;
      const int64_t base = kBase[wm == 4][tn], busy = kBusy[wm == 4][tn];
      int64_t cost = steps * (full * (base + busy) + (rest > 0 ? base + busy * rest / cus : 0));
      if (sp > 1) cost += 30 + 33 * sp + 180 * sp * M * N / (1 << 20);
      if (cost < best_cost) {
        best_cost = cost;
        best = {wm, tn, static_cast<int>(cdiv(nk, steps)), static_cast<int>(steps)};
      }
    }
  }
  return best;
}

// Rows per launch: the planes of a chunk stay within kChunkBytes.
constexpr int64_t kChunkBytes = int64_t(192) << 20;

int64_t chunk_rows(int64_t M, int64_t K) {
  const int64_t r = std::max<int64_t>(256, kChunkBytes / (4 * K) / 256 * 256);
  return M <= r + 64 ? M : r;   // a short remainder joins its chunk
}

int64_t align256(int64_t v) { return (v + 255) / 256 * 256; }

// Scratch of a chunk: the planes, the rows' exponents and masks, the k-ranges' sums.
int64_t exps_at(int64_t M, int64_t K) { return align256(4 * M * K); }
int64_t far_at(int64_t M, int64_t K) { return exps_at(M, K) + align256(4 * M); }
int64_t part_at(int64_t M, int64_t K) { return far_at(M, K) + align256(8 * M); }

int64_t chunk_bytes(int64_t M, int64_t N, int64_t K) {
  const F32Plan p = f32_plan(M, N, K);
  return part_at(M, K) + (p.splits > 1 ? p.splits * M * N * 4 : 0);
}

template <int TN, int WM>
void launch(const F32Args& a, hipStream_t s) {
  const dim3 g(static_cast<unsigned>(a.tiles_m * a.tiles_n * a.splits)), blk(512);
  if (a.splits > 1) k_gemm_f32<TN, WM, true><<<g, blk, 0, s>>>(a);
  else k_gemm_f32<TN, WM, false><<<g, blk, 0, s>>>(a);
}

}  // namespace

namespace f32lin {

bool applies(int64_t M, int64_t N, int64_t K, int64_t n_out) {
  constexpr int64_t kLim = (1LL << 32) - 4096;
  return n_out == 0 && K % 64 == 0 && M * K * 2 < kLim && N * K < kLim &&
         2 * cdiv(M, 128) * cdiv(N, 256) < (1LL << 30) && (M > 64 || N * K >= (8LL << 20));
}

int64_t ws_bytes(int64_t M, int64_t N, int64_t K) {
  int64_t most = 0;
  for (int64_t m0 = 0; m0 < M;) {
    const int64_t mr = chunk_rows(M - m0, K);
    most = std::max(most, chunk_bytes(mr, N, K));
    m0 += mr;
  }
  return most;
}

int run(const float* x, const int8_t* wq, const float* scales, const float* bias, int64_t M,
        int64_t N, int64_t K, void* scratch, float* y, hipStream_t s, const char* what) {
  for (int64_t m0 = 0; m0 < M;) {
    const int64_t mr = chunk_rows(M - m0, K);
    const F32Plan p = f32_plan(mr, N, K);
    uint8_t* const base = static_cast<uint8_t*>(scratch);
    uint16_t* const xp = reinterpret_cast<uint16_t*>(base);
    int* const exps = reinterpret_cast<int*>(base + exps_at(mr, K));
    F32Args a{};
    a.x = x + m0 * K;
    a.xp = xp;
    a.exps = exps;
    uint64_t* const far = reinterpret_cast<uint64_t*>(base + far_at(mr, K));
    a.far = far;
    while ((K / 64 - 1) >> a.far_shift > 63) ++a.far_shift;
    a.wq = wq;
    a.scales = scales;
    a.bias = bias;
    a.y = y + m0 * N;
    a.part = reinterpret_cast<float*>(base + part_at(mr, K));
    a.M = static_cast<int>(mr);
    a.N = static_cast<int>(N);
    a.K = static_cast<int>(K);
    a.tiles_m = static_cast<int>(cdiv(mr, 32LL * p.wm));
    a.tiles_n = static_cast<int>(cdiv(N, 32LL * p.tn * (8 / p.wm)));
    a.splits = p.splits;
    a.split_steps = p.steps;
    const dim3 pg(static_cast<unsigned>(mr)), pb(kBlock);
    if (K <= 4 * 4 * kBlock) k_f32_planes<4><<<pg, pb, 0, s>>>(a, xp, exps, far);
    else k_f32_planes<16><<<pg, pb, 0, s>>>(a, xp, exps, far);
    if (p.wm == 4) {
      if (p.tn == 3) launch<3, 4>(a, s);
      else if (p.tn == 2) launch<2, 4>(a, s);
      else launch<1, 4>(a, s);
    } else {
      if (p.tn == 3) launch<3, 2>(a, s);
      else if (p.tn == 2) launch<2, 2>(a, s);
      else launch<1, 2>(a, s);
    }
    if (p.splits > 1) {
      const int64_t mn = mr * N;
      if (N % 4 == 0)
        k_f32_reduce<4><<<dim3(static_cast<unsigned>(cdiv(mn, 4LL * kBlock))), dim3(kBlock), 0, s>>>(a);
      else
        k_f32_reduce<1><<<dim3(static_cast<unsigned>(cdiv(mn, static_cast<int64_t>(kBlock)))), dim3(kBlock), 0, s>>>(a);
    }
    m0 += mr;
  }
  return launch_status(what);
}

}  // namespace f32lin
}  // namespace cbq
