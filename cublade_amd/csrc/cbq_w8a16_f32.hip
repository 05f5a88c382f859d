// cbq_w8a16_f32.hip - W8A16 linear with fp32 activations on the matrix cores of
// gfx950 (K % 64 == 0, no outlier columns).
//
// The weights are int8 codes, exact in fp16 and bf16, so the products of x with
// them are exact in fp32 if x is a sum of 16-bit numbers. k_f32_planes writes two
// 16-bit planes of x, in one of two forms per row:
//   narrow  x 2^e = hi + 2^-11 lo with hi and lo fp16, the row's largest magnitude
//           in [2^14, 2^15). Taken where the smallest non-zero magnitude is at
//           least 2^-34 of the largest: 22 significant bits for elements down to
//           2^-29 of the largest (lo is held 2^11 up, so that it stays a normal
//           number as long as hi does), 16 or more for all. Infinities and NaN
//           are hi, with lo = 0.
//   wide    the upper and lower halves of the fp32 number itself. k_gemm_f32 takes
//           them apart into three bf16 numbers, 24 bits: exact.
// Either way no element's precision depends on what else the row holds, and the
// time does not depend on the values, but for tiles with wide rows (the
// N(0, 1), M = 500, N = 11008, K = 4096 call takes 92 us, 177 with every row
// wide, 240 with one in each tile).
//
// k_gemm_f32 adds the planes' products in fp32, each plane in accumulators of its
// own, and finishes with y[m, n] = s[n] 2^-e[m] (hi + 2^-11 lo) + bias[n]. For
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

constexpr int kWideRow = INT32_MIN;
// 64-k steps after which the first plane's sums go to a second set of registers: the
// sums in the accumulators stay small and so do their roundings (distance from the
// 64-bit result at K = 4096 4.1e-7 without, 1.7e-7 with; 1% of the time).
constexpr int kRun = 12;

struct F32Args {
  const float* x;          // [M, K]
  const uint16_t* xp;      // [2][M, K] planes
  const int* exps;         // [M] e of a narrow row, or kWideRow
  const int8_t* wq;        // [N, K]
  const float* scales;     // [N]
  const float* bias;       // [N] or null
  float* y;                // [M, N]
  float* part;             // SPLIT: [splits][M, N] fp32 sums (scaled by 2^-e)
  int M, N, K;
  int tiles_m, tiles_n;
  int splits, split_steps; // k-ranges of split_steps 64-k steps
};

// floor(log2) of a positive finite float given as its bits (subnormals too).
__device__ __forceinline__ int exp2_floor(uint32_t b) {
  return b >= 0x00800000u ? static_cast<int>(b >> 23) - 127 : 31 - __builtin_clz(b) - 149;
}

// One workgroup per row: its smallest and largest magnitude, then the planes.
// Rows of up to 1024 V elements stay in registers between the two. Bound: memory
// (x read, as many bytes written).
template <int V>   // float4 per thread and step
__global__ __launch_bounds__(kBlock) void k_f32_planes(F32Args a, uint16_t* __restrict__ xp,
                                                       int* __restrict__ exps) {
  __shared__ uint32_t s_max[kBlock / kWave], s_min[kBlock / kWave];
  const int m = blockIdx.x, t = threadIdx.x;
  const int n4 = a.K >> 2;
  const int64_t base = static_cast<int64_t>(m) * a.K;
  const float4* const x4 = reinterpret_cast<const float4*>(a.x + base);
  float4 r[V];
  uint32_t mx = 0u, mn = 0xffffffffu;   // of |x|'s bits, and of those less one (0: the largest)
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
  const int top = mx ? exp2_floor(mx) : 14;
  const bool wide = mx && exp2_floor(mn + 1u) < top - 34;
  const int e = 14 - top;
  if (t == 0) exps[m] = wide ? kWideRow : e;

  const int64_t plane = static_cast<int64_t>(a.M) * a.K;
  for (int i0 = 0; i0 < n4; i0 += V * kBlock) {
#pragma unroll
    for (int v = 0; v < V; ++v) {
      const int i = i0 + v * kBlock + t;
      if (i >= n4) continue;
      if (n4 > V * kBlock) r[v] = x4[i];
      const float f[4] = {r[v].x, r[v].y, r[v].z, r[v].w};
      uint32_t hi[4], lo[4];
#pragma unroll
      for (int k = 0; k < 4; ++k) {
        const uint32_t b = __float_as_uint(f[k]);
        const bool fin = (b & 0x7fffffffu) < 0x7f800000u;
        if (wide) {
          const bool nan = (b & 0x7fffffffu) > 0x7f800000u;
          hi[k] = nan ? 0x7fc0u : b >> 16;
          lo[k] = fin ? b & 0xffffu : 0u;
        } else {
          const float z = __builtin_ldexpf(f[k], e);
          const _Float16 h = static_cast<_Float16>(z);
          const float rest = fin ? (z - static_cast<float>(h)) * 2048.0f : 0.0f;   // exact
          hi[k] = __builtin_bit_cast(uint16_t, h);
          lo[k] = __builtin_bit_cast(uint16_t, static_cast<_Float16>(rest));
        }
      }
      uint16_t* const p = xp + base + 4 * i;
      *reinterpret_cast<uint2*>(p) = make_uint2(hi[0] | (hi[1] << 16), hi[2] | (hi[3] << 16));
      *reinterpret_cast<uint2*>(p + plane) = make_uint2(lo[0] | (lo[1] << 16), lo[2] | (lo[3] << 16));
    }
  }
}

// Two elements of a wide row (halves h of the upper, l of the lower plane) as
// hi + mid + lo: hi is h itself.
__device__ __forceinline__ void split_wide(uint32_t h, uint32_t l, uint32_t& mid, uint32_t& lo) {
  float r[2], q[2];
#pragma unroll
  for (int k = 0; k < 2; ++k) {
    const uint32_t hb = k ? h & 0xffff0000u : h << 16;
    const uint32_t full = hb | (k ? l >> 16 : l & 0xffffu);
    const bool fin = (hb & 0x7f800000u) != 0x7f800000u;
    r[k] = fin ? __uint_as_float(full) - __uint_as_float(hb) : 0.0f;
    q[k] = r[k] - __uint_as_float(__float_as_uint(r[k]) & 0xffff0000u);   // 8 bits or fewer
  }
  mid = (__float_as_uint(r[1]) & 0xffff0000u) | (__float_as_uint(r[0]) >> 16);
  lo = (__float_as_uint(q[1]) & 0xffff0000u) | (__float_as_uint(q[0]) >> 16);
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
// A row of an MFMA's result depends on that row of A alone. A tile with rows of
// both forms runs its k loop twice, as fp16 and as bf16, and stores of each the rows
// that are of that form.
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
  auto issue_first = [&]() {
#pragma unroll
    for (int t = 0; t < NS; ++t)
      if (t < nk)
#pragma unroll
        for (int u = 0; u < L; ++u) issue_one(t, t, u);
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

  // The tile's k loop in one of the two forms, and the store of the rows of that form.
  auto pass = [&](auto form) __attribute__((always_inline)) {
    constexpr bool W = decltype(form)::value;
    constexpr int ACT = W ? kBF16 : kF16;
    constexpr int NP = W ? 3 : 2;                 // products per element
    constexpr int S = 2 * NP, Q = S * TN, R = TN + 4;
    f16x acc[2][TN];
#pragma unroll
    for (int p = 0; p < 2; ++p)
#pragma unroll
      for (int i = 0; i < TN; ++i) acc[p][i] = f16x{};
    f16x sum[TN];   // !W: what acc[0] held at the ends of earlier runs of steps
#pragma unroll
    for (int i = 0; i < TN; ++i) sum[i] = f16x{};
    Frags f0, f1;
    u32x4 wa[2], wb[2];                           // widened weights: this and the next tile
    u32x4 xw[2][2];                               // W: mid and lo of the half's slices
    auto widen = [&](const Frags& f, int i, int c, u32x4 (&w)[2]) {
      const uint32_t word = c == 0 ? f.w[i].x : c == 1 ? f.w[i].y : c == 2 ? f.w[i].z : f.w[i].w;
      uint32_t lo, hi;
      i8x4_to_act<ACT>(word, lo, hi);
      w[c >> 1][(c & 1) * 2] = lo;
      w[c >> 1][(c & 1) * 2 + 1] = hi;
    };
    // One half of a step from f, widening fnext's first tile at its end (more); slots of
    // one MFMA, each followed by extra(slot). par: which of wa and wb holds tile 0.
    auto half = [&](const Frags& f, const Frags& fnext, auto more, int par, auto&& extra) {
      constexpr bool MORE = decltype(more)::value;
      if constexpr (W) {
#pragma unroll
        for (int s = 0; s < 2; ++s)
#pragma unroll
          for (int k = 0; k < 4; ++k) {
            uint32_t mid, lo;
            split_wide(f.x[0][s][k], f.x[1][s][k], mid, lo);
            xw[0][s][k] = mid;
            xw[1][s][k] = lo;
          }
      }
#pragma unroll
      for (int i = 0; i < TN; ++i) {
        u32x4(&cur)[2] = ((i + par) & 1) ? wb : wa;
        u32x4(&nxt)[2] = ((i + par) & 1) ? wa : wb;
#pragma unroll
        for (int p = 0; p < S; ++p) {
          const int s = p / NP, q = p % NP;
          const u32x4 xs = q == 0 ? f.x[0][s] : W ? xw[q - 1][s] : f.x[1][s];
          acc[q > 0][i] = mfma32x32x16<ACT>(xs, cur[s], acc[q > 0][i]);
          if constexpr (TN == 1) {   // the next half's tile is read at slot 0
#pragma unroll
            for (int c = 0; c < 4; ++c)
              if (MORE && (c + 1 < S ? c + 1 : S - 1) == p) widen(fnext, 0, c, nxt);
          } else if (p < 4) {
            if (i + 1 < TN) widen(f, i + 1, p, nxt);
            else if (MORE) widen(fnext, 0, p, nxt);
          }
          extra(i * S + p);
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
    if constexpr (!W) {
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
    float* const out = SPLIT ? a.part + static_cast<int64_t>(split) * a.M * a.N : a.y;
    int ex[16];
#pragma unroll
    for (int v = 0; v < 16; ++v) ex[v] = a.exps[min(mw + 8 * (v >> 2) + 4 * h + (v & 3), a.M - 1)];
#pragma unroll
    for (int i = 0; i < TN; ++i) {
      const int n = nw + 32 * i + r32;
      const float sc = SPLIT || n >= a.N ? 1.0f : a.scales[n];
      const float bs = SPLIT || n >= a.N || !a.bias ? 0.0f : a.bias[n];
#pragma unroll
      for (int v = 0; v < 16; ++v) {
        const int m = mw + 8 * (v >> 2) + 4 * h + (v & 3);
        float f;
        if constexpr (W) f = acc[0][i][v] + acc[1][i][v];
        else f = __builtin_ldexpf(__builtin_fmaf(acc[1][i][v], 0x1p-11f, sum[i][v] + acc[0][i][v]), -ex[v]);
        if constexpr (!SPLIT) f = a.bias ? f * sc + bs : f * sc;
        if (m < a.M && n < a.N && (ex[v] == kWideRow) == W)
          out[static_cast<int64_t>(m) * a.N + n] = f;
      }
    }
  };

  issue_first();
  bool narrow = false, wide = false;   // rows of each form in the tile, by every wave
#pragma unroll
  for (int i = 0; i < BM; i += kWave) {
    const bool w = a.exps[min(m0 + i + lane, a.M - 1)] == kWideRow;
    narrow |= __any(!w);
    wide |= __any(w);
  }
  if (narrow) pass(no{});
  if (wide) {
    if (narrow) {
      dma_wait_barrier<0>();   // every wave has read its last fragments
      issue_first();
    }
    pass(yes{});
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
// + 0.33 us per range and 1.8 us per 4 MiB of partial sums. Within 2.5% of the
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

// Scratch of a chunk: the planes, the rows' exponents, the k-ranges' sums.
int64_t exps_at(int64_t M, int64_t K) { return align256(4 * M * K); }
int64_t part_at(int64_t M, int64_t K) { return exps_at(M, K) + align256(4 * M); }

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
    if (K <= 4 * 4 * kBlock) k_f32_planes<4><<<pg, pb, 0, s>>>(a, xp, exps);
    else k_f32_planes<16><<<pg, pb, 0, s>>>(a, xp, exps);
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
