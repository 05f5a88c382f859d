// cbq_w8a16_f32.hip - W8A16 linear with fp32 activations on the int8 matrix
// cores of gfx950 (K % 64 == 0, no outlier columns).
//
// The weights are int8 codes, so x . w needs no widening if x is int8 too.
// k_f32_digits writes each row of x as fixed-point numbers of 24 bits
// against the row's largest magnitude, in three balanced base-256 digits:
//   x[m, k] ~ sx[m] * (65536 d2 + 256 d1 + d0),   sx[m] = max_k |x[m, k]| / 8355711
// (8355711 = 127 (65536 + 256 + 1), the largest such number). k_gemm_f32 takes
// the three int8 products with v_mfma_i32_32x32x32_i8, exact in int32
// (127 * 128 * K < 2^31 for K <= 131072), and adds them up in fp32:
//   y[m, n] = s[n] * (sx[m] * (65536 a2 + 256 a1 + a0) + spikes) + bias[n]
// Spikes: elements above 128 times the row's mean magnitude, infinities and
// NaN. They stay out of the digits and of the maximum, and their products
// are added in fp32 one by one (at most one element in 128 can be that large;
// a row with more, of non-finite values, or whose largest other magnitude is
// below 2^-80 is summed whole that way).
//
// Error per element: half a unit, at most 6e-8 max|x| <= 2^-17 mean|x|, where
// the two bf16 planes of x this replaces kept 16 significant bits (2^-17 |x|
// on average); for N(0, 1) at K = 4096 the whole result is 2e-7 from the
// 64-bit one (relative, 2-norm), with the planes 4.9e-6. k-ranges of more than
// kMaxSeg have a scale of their own.
//
// Three int8 products cost 1.5 times one bf16 product on the matrix cores
// where the two planes cost twice, and the partial tiles of the planes (90 MB
// written and read back at M = 500, N = 11008) are gone: all three digits
// meet in one workgroup's accumulators.
#include <algorithm>
#include <type_traits>

#include "cbq_device.h"
#include "cbq_host.h"
#include "cbq_lds_dma.h"
#include "cbq_w8a16_f32.h"

namespace cbq {
namespace {

typedef int i4v __attribute__((ext_vector_type(4)));
typedef int i16x __attribute__((ext_vector_type(16)));

constexpr float kDigitMax = 8355711.0f;   // 127 * (65536 + 256 + 1)
constexpr float kDigitTiny = 8.2718061e-25f;   // 2^-80

struct F32Args {
  const float* x;          // [M, K]
  const uint8_t* xd;       // [3][M, K] int8 digits, d2 first
  const float* sx;         // [segs][M] row scales
  const int* cnt;          // [segs][M] spikes of the row: none, their count, or kWholeRow
  const int* idx;          // [segs][M][kMaxSpikes] their k, in order
  const int8_t* wq;        // [N, K]
  const float* scales;     // [N]
  const float* bias;       // [N] or null
  float* y;                // [M, N]
  float* part;             // SPLIT: [splits][M, N] fp32 sums (scaled by sx)
  int M, N, K;
  int tiles_m, tiles_n;
  int splits, split_steps; // k-ranges of split_steps 64-k steps
  int segs, seg_len;       // row scales: one (K <= kMaxSeg), or one per k-range
};

constexpr int kMaxSpikes = f32lin::kMaxSeg / 128;
constexpr int kWholeRow = -1;

// One workgroup per row and scale (blockIdx.x, blockIdx.y), held in
// registers: mean magnitude, largest magnitude without the spikes, the digits,
// and the list of spikes where there are any.
template <int V>   // float4 per thread at most
__global__ __launch_bounds__(kBlock) void k_f32_digits(F32Args a, uint8_t* __restrict__ xd,
                                                       float* __restrict__ sx,
                                                       int* __restrict__ cnt,
                                                       int* __restrict__ idx) {
  __shared__ float red[kBlock / kWave];
  __shared__ float s_sum[kBlock / kWave];
  __shared__ int counts[kBlock];
  const int m = blockIdx.x, k0 = blockIdx.y * a.seg_len;
  const int t = threadIdx.x;
  const int n4 = min(a.seg_len, a.K - k0) >> 2;
  const int64_t base = static_cast<int64_t>(m) * a.K + k0;
  const int64_t row = static_cast<int64_t>(blockIdx.y) * a.M + m;
  float4 r[V];
  float sum = 0.0f;
  auto mag = [](float f) { return __builtin_fabsf(f); };
  auto finite = [](float f) { return __builtin_fabsf(f) < __builtin_inff(); };   // NaN: false
#pragma unroll
  for (int v = 0; v < V; ++v) {
    const int i = v * kBlock + t;
    r[v] = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
    if (v * kBlock < n4) {
      if (i < n4) r[v] = *reinterpret_cast<const float4*>(a.x + base + 4 * i);
      const float f[4] = {r[v].x, r[v].y, r[v].z, r[v].w};
#pragma unroll
      for (int e = 0; e < 4; ++e) sum += finite(f[e]) ? mag(f[e]) : 0.0f;
    }
  }
#pragma unroll
  for (int o = 1; o < kWave; o <<= 1) sum += __shfl_xor(sum, o);
  if (t % kWave == 0) s_sum[t / kWave] = sum;
  __syncthreads();
  sum = 0.0f;
#pragma unroll
  for (int w = 0; w < kBlock / kWave; ++w) sum += s_sum[w];
  const float limit = sum * (128.0f / (4.0f * static_cast<float>(n4)));   // inf if the sum overflowed
  auto spike = [&](float f) { return !(mag(f) <= limit) || !finite(f); };
  float amax = 0.0f;
  int mine = 0;
#pragma unroll
  for (int v = 0; v < V; ++v)
    if (v * kBlock < n4) {
      const float f[4] = {r[v].x, r[v].y, r[v].z, r[v].w};
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const bool sp = spike(f[e]);
        amax = fmaxf(amax, sp ? 0.0f : mag(f[e]));
        mine += sp;
      }
    }
  amax = block_max(amax, red);
  const int any = __syncthreads_or(mine);
  const bool tiny = amax > 0.0f && amax < kDigitTiny;
  int n = tiny ? kWholeRow : 0;
  if (any && !tiny) {
    counts[t] = mine;
    __syncthreads();
    int at = 0, total = 0;
    for (int j = 0; j < kBlock; ++j) {
      at += j < t ? counts[j] : 0;
      total += counts[j];
    }
    n = total <= kMaxSpikes ? total : kWholeRow;
    if (n > 0) {
#pragma unroll
      for (int v = 0; v < V; ++v) {
        const float f[4] = {r[v].x, r[v].y, r[v].z, r[v].w};
#pragma unroll
        for (int e = 0; e < 4; ++e)
          if (v * kBlock + t < n4 && spike(f[e])) idx[row * kMaxSpikes + at++] = k0 + 4 * (v * kBlock + t) + e;
      }
    }
  }
  const float inv = n == kWholeRow || amax == 0.0f ? 0.0f : kDigitMax / amax;
  if (t == 0) {
    sx[row] = n == kWholeRow ? 0.0f : amax / kDigitMax;
    cnt[row] = n;
  }
  const int64_t plane = static_cast<int64_t>(a.M) * a.K;
#pragma unroll
  for (int v = 0; v < V; ++v) {
    const int i = v * kBlock + t;
    if (v * kBlock < n4 && i < n4) {
      const float f[4] = {r[v].x, r[v].y, r[v].z, r[v].w};
      int d0[4], d1[4], d2[4];
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const float z = __builtin_rintf((spike(f[e]) ? 0.0f : f[e]) * inv);
        const int q = static_cast<int>(fminf(fmaxf(z, -kDigitMax), kDigitMax));
        d0[e] = static_cast<int8_t>(q);
        const int q1 = (q - d0[e]) >> 8;
        d1[e] = static_cast<int8_t>(q1);
        d2[e] = (q1 - d1[e]) >> 8;
      }
      uint8_t* p = xd + base + 4 * i;
      *reinterpret_cast<uint32_t*>(p) = pack4_low_bytes(d2[0], d2[1], d2[2], d2[3]);
      *reinterpret_cast<uint32_t*>(p + plane) = pack4_low_bytes(d1[0], d1[1], d1[2], d1[3]);
      *reinterpret_cast<uint32_t*>(p + 2 * plane) = pack4_low_bytes(d0[0], d0[1], d0[2], d0[3]);
    }
  }
}

// fix[r][c] = the spikes' products of output (m0 + r, n0 + c), r < 32, c <
// cols: by one wave, rows without spikes 0.
__device__ void add_spikes(const F32Args& a, int seg, int m0, int n0, int cols, int lane, int kb,
                           int ke, float* fix) {
  for (int r = 0; r < 32; ++r) {
    const int m = min(m0 + r, a.M - 1);
    const int64_t row = static_cast<int64_t>(seg) * a.M + m;
    const int n = a.cnt[row];
    const float* x = a.x + static_cast<int64_t>(m) * a.K;
    for (int c = lane; c < cols; c += kWave) {
      const int8_t* w = a.wq + static_cast<int64_t>(min(n0 + c, a.N - 1)) * a.K;
      float sum = 0.0f;
      if (n == kWholeRow) {
        for (int k = kb; k < ke; ++k) sum += x[k] * static_cast<float>(w[k]);
      } else {
        for (int j = 0; j < n; ++j) {
          const int k = a.idx[row * kMaxSpikes + j];
          if (k >= kb && k < ke) sum += x[k] * static_cast<float>(w[k]);
        }
      }
      fix[r * cols + c] = sum;
    }
  }
}

// Tile of 32 WM rows of x (all three digits) by 32 TN (8 / WM) weight rows, 8
// waves (two per SIMD), each 32 x 32 TN: 48 TN accumulators. 64-k steps
// through three LDS stages filled by LDS DMA (two steps in flight), one
// barrier per step between its two 32-k halves; per half a wave reads TN + 3
// fragments for 3 TN MFMAs, the next half's reads and the DMA of step t + 3
// spread between them. A weight fragment serves the three digits, so a
// workgroup reads 83 bytes of LDS per clock of MFMA time at TN = 3 (128
// available). Rows of 64 bytes, 16-byte chunk c of row r at c ^ ((r >> 2) & 3)
// (no bank conflicts); rows past M or N are clamped for the loads and not
// stored. MFMA A = x digits, B = weights: lane l holds n = l % 32 and m = 8
// (v / 4) + 4 (l / 32) + v % 4, so a store writes two 128-byte runs.
template <int TN, int WM, bool SPLIT>
__global__ __launch_bounds__(512) void k_gemm_f32(F32Args a) {
  constexpr int WN = 8 / WM, BM = 32 * WM, BN = 32 * TN * WN, NS = 3;
  constexpr int XI = 3 * BM / 16, TI = XI + BN / 16;   // 1 KiB DMA instructions per step
  constexpr int L = (TI + 7) / 8;                      // per wave (the last one: waves < TI % 8)
  constexpr int SB = TI * 1024;
  constexpr int WREM = TI % 8;                         // waves that issue L (0: all)
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

  // DMA instruction u of this wave is instruction q = 8 u + wave of the
  // step: 16 rows of a digit plane, then 16 weight rows.
  uint32_t off[L];
  const uint8_t* src[L];
#pragma unroll
  for (int u = 0; u < L; ++u) {
    const int q = u * 8 + wave;
    const bool isx = q < XI;
    const int row = (isx ? q % (BM / 16) : q - XI) * 16 + (lane >> 2);
    const int c = (lane & 3) ^ ((row >> 2) & 3);
    const int rr = isx ? min(m0 + row, a.M - 1) : min(n0 + row, a.N - 1);
    off[u] = static_cast<uint32_t>(rr) * static_cast<uint32_t>(a.K) + c * 16u;
    src[u] = uniform_ptr((isx ? a.xd + static_cast<int64_t>(q / (BM / 16)) * a.M * a.K
                              : reinterpret_cast<const uint8_t*>(a.wq)) + kb * 64);
  }
  auto issue_one = [&](int t, int stage, int u) {
    if (WREM == 0 || u < L - 1 || wave < WREM)
      lds_dma16(off[u], uniform_ptr(src[u] + t * 64), sbase + stage * SB + (u * 8 + wave) * 1024);
  };
  // At most T tiles' DMA of this wave outstanding, then the barrier.
  auto wait_tiles = [&](auto tiles) {
    constexpr int T = decltype(tiles)::value;
    if (WREM == 0 || wave < WREM) dma_wait_barrier<T * L>();
    else dma_wait_barrier<T * (L - 1)>();
  };

  const int r32 = lane & 31, h = lane >> 5;
  uint32_t xr[2], wr[2];
#pragma unroll
  for (int e = 0; e < 2; ++e) {
    const uint32_t slot = static_cast<uint32_t>((2 * h + e) ^ ((r32 >> 2) & 3)) << 4;
    xr[e] = (wm * 32 + r32) * 64 + slot;
    wr[e] = XI * 1024 + (wn * 32 * TN + r32) * 64 + slot;
  }
  i16x acc[3][TN];
#pragma unroll
  for (int p = 0; p < 3; ++p)
#pragma unroll
    for (int i = 0; i < TN; ++i) acc[p][i] = i16x{};

  struct Frags {
    u32x4 x[3], w[TN];
  };
  auto read_one = [&](int stage, int e, Frags& f, int r) {
    const uint8_t* st = smem + stage * SB;
    if (r < TN) f.w[r] = *reinterpret_cast<const u32x4*>(st + wr[e] + r * 2048);
    else f.x[r - TN] = *reinterpret_cast<const u32x4*>(st + xr[e] + (r - TN) * (BM * 64));
  };
  auto mma_one = [&](const Frags& f, int q) {
    const int p = q / TN, i = q % TN;
    acc[p][i] = __builtin_amdgcn_mfma_i32_32x32x32_i8(__builtin_bit_cast(i4v, f.x[p]),
                                                      __builtin_bit_cast(i4v, f.w[i]), acc[p][i],
                                                      0, 0, 0);
  };
  Frags f0, f1;
  using std::integral_constant;
  using yes = std::true_type;
  using no = std::false_type;
  constexpr int Q = 3 * TN, R = TN + 3;
  // Step t: f0 holds half 0 of tile t; its MFMAs run with the reads of half 1
  // between them, then the wait for tile t + 1 and the barrier (every wave is
  // done with tile t's stage), then half 1 with the DMA of tile t + 3 into that
  // stage and the reads of tile t + 1's half 0.
  auto step = [&](int t, auto dma, auto ahead) {
    const int cur = t % NS, nxt = (t + 1) % NS;
#pragma unroll
    for (int q = 0; q < Q; ++q) {
      mma_one(f0, q);
      for (int r = q; r < R; r += Q) read_one(cur, 1, f1, r);
      __builtin_amdgcn_sched_barrier(0);
    }
    wait_tiles(ahead);
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int q = 0; q < Q; ++q) {
      mma_one(f1, q);
      if constexpr (decltype(dma)::value)
        for (int u = q; u < L; u += Q) issue_one(t + NS, cur, u);
      for (int r = q; r < R; r += Q) read_one(nxt, 0, f0, r);
      __builtin_amdgcn_sched_barrier(0);
    }
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
  int t = 0;
  for (; t + NS < nk; ++t) step(t, yes{}, integral_constant<int, 1>{});
  if (t + 2 < nk) step(t++, no{}, integral_constant<int, 1>{});
  if (t + 1 < nk) step(t++, no{}, integral_constant<int, 0>{});
#pragma unroll
  for (int q = 0; q < Q; ++q) {
    mma_one(f0, q);
    for (int r = q; r < R; r += Q) read_one((nk - 1) % NS, 1, f1, r);
    __builtin_amdgcn_sched_barrier(0);
  }
#pragma unroll
  for (int q = 0; q < Q; ++q) mma_one(f1, q);

  const int mw = m0 + wm * 32, nw = n0 + wn * 32 * TN;
  const int seg = a.segs > 1 ? split : 0;
  const int64_t srow = static_cast<int64_t>(seg) * a.M;
  float* const out = SPLIT ? a.part + static_cast<int64_t>(split) * a.M * a.N : a.y;
  // Every wave is past its operand reads; rows with spikes anywhere in the tile?
  const bool spikes = __syncthreads_or(a.cnt[srow + min(mw + r32, a.M - 1)] != 0);
  float* const fix = reinterpret_cast<float*>(smem) + wave * (32 * 32 * TN);
  static_assert(8 * 32 * 32 * TN * 4 <= NS * SB, "the waves' corrections fit in LDS");
  if (spikes) add_spikes(a, seg, mw, nw, 32 * TN, lane, kb * 64, (kb + nk) * 64, fix);
  float rs[16];
#pragma unroll
  for (int v = 0; v < 16; ++v) rs[v] = a.sx[srow + min(mw + 8 * (v >> 2) + 4 * h + (v & 3), a.M - 1)];
  auto finish = [&](auto fixed) {
#pragma unroll
    for (int i = 0; i < TN; ++i) {
      const int n = nw + 32 * i + r32;
      const float sc = SPLIT || n >= a.N ? 1.0f : a.scales[n];
      const float bs = SPLIT || n >= a.N || !a.bias ? 0.0f : a.bias[n];
#pragma unroll
      for (int v = 0; v < 16; ++v) {
        const int ml = 8 * (v >> 2) + 4 * h + (v & 3), m = mw + ml;
        float f = __builtin_fmaf(static_cast<float>(acc[0][i][v]), 65536.0f,
                                 __builtin_fmaf(static_cast<float>(acc[1][i][v]), 256.0f,
                                                static_cast<float>(acc[2][i][v]))) * rs[v];
        if constexpr (decltype(fixed)::value) f += fix[ml * 32 * TN + 32 * i + r32];
        if constexpr (!SPLIT) f = a.bias ? f * sc + bs : f * sc;
        if (m < a.M && n < a.N) out[static_cast<int64_t>(m) * a.N + n] = f;
      }
    }
  };
  if (spikes) finish(yes{});
  else finish(no{});
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
// MI355X over 24 shapes (M = 1 .. 4096, N and K = 256 .. 12096): a 64-k step
// costs more the more CUs are busy (0.55 + 0.58 us x their share for 128 x 192
// tiles, 0.36 + 0.46 for 128 x 128, 0.35 + 0.28 for 128 x 64; M <= 64: 0.60 +
// 0.80, 0.42 + 0.62 and 0.15 + 0.50 for 64 x 384, 256 and 128), a split 4.5 us
// + 0.4 us per range for the reduce pass and 1 us per 4 MiB of partial sums.
// Within 4% of the best plan measured. M = 256, N = 11008, K = 4096: 128 x 128
// whole 52.7 us, 128 x 192 in two ranges 59.6; M = 128: 39.4 and 39.5 (four).
F32Plan f32_plan(int64_t M, int64_t N, int64_t K) {
  const int64_t cus = device_cus(), nk = K / 64;
  const int64_t min_sp = cdiv(K, static_cast<int64_t>(f32lin::kMaxSeg));
  const int wm = M <= 64 ? 2 : 4;
  constexpr int64_t kBase[2][4] = {{0, 15, 42, 60}, {0, 35, 36, 55}};
  constexpr int64_t kBusy[2][4] = {{0, 50, 62, 80}, {0, 28, 46, 58}};
  F32Plan best{wm, 1, static_cast<int>(min_sp), static_cast<int>(cdiv(nk, min_sp))};
  int64_t best_cost = INT64_MAX;
  for (const int tn : {3, 2, 1}) {
    const int64_t tiles = cdiv(M, 32LL * wm) * cdiv(N, 32LL * tn * (8 / wm));
    for (int64_t sp = min_sp; sp <= 16 || sp == min_sp; ++sp) {
      if (sp > min_sp && (tiles * sp > cus || nk / sp < 4)) break;
      const int64_t steps = cdiv(nk, sp), full = tiles * sp / cus, rest = tiles * sp % cus;
      const int64_t base = kBase[wm == 4][tn], busy = kBusy[wm == 4][tn];
      int64_t cost = steps * (full * (base + busy) + (rest > 0 ? base + busy * rest / cus : 0));
      if (sp > 1) cost += 450 + 40 * sp + 100 * sp * M * N / (1 << 20);
      if (cost < best_cost) {
        best_cost = cost;
        best = {wm, tn, static_cast<int>(cdiv(nk, steps)), static_cast<int>(steps)};
      }
    }
  }
  return best;
}

// Row scales: one, or one per k-range where a row is longer than kMaxSeg.
int f32_segs(int64_t K, const F32Plan& p) { return K > f32lin::kMaxSeg ? p.splits : 1; }

// Rows per launch: the digits of a chunk stay below 3/4 of kChunkBytes.
constexpr int64_t kChunkBytes = int64_t(256) << 20;

int64_t chunk_rows(int64_t M, int64_t K) {
  const int64_t r = std::max<int64_t>(256, kChunkBytes / (4 * K) / 256 * 256);
  return M <= r + 64 ? M : r;   // a short remainder joins its chunk
}

int64_t align256(int64_t v) { return (v + 255) / 256 * 256; }

int64_t chunk_bytes(int64_t M, int64_t N, int64_t K) {
  const F32Plan p = f32_plan(M, N, K);
  const int64_t need = align256(3 * M * K) + align256(f32_segs(K, p) * M * (2 + kMaxSpikes) * 4) +
                       (p.splits > 1 ? p.splits * M * N * 4 : 0);
  // The size never falls below what earlier versions of the library asked for,
  // so that workspaces shared with a caller's other buffers keep their layout:
  // two 16-bit planes of x and, at M <= 64, fp32 tiles of 128 x 256 for each
  // plane and k-range (as many ranges as fill the CUs, at most 8).
  int64_t before = 2 * align256(2 * M * K) + 256;
  if (M <= 64) {
    const int64_t tiles = cdiv(N, 256LL), nk = K / 64;
    const int64_t ks = std::max<int64_t>(1, std::min<int64_t>({device_cus() / (2 * tiles), 8, nk / 4}));
    before += tiles * 2 * cdiv(nk, cdiv(nk, ks)) * 128 * 256 * 4 - 256;
  }
  return std::max(need, before);
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
    float* const sx = reinterpret_cast<float*>(base + align256(3 * mr * K));
    F32Args a{};
    a.x = x + m0 * K;
    a.xd = base;
    a.sx = sx;
    a.wq = wq;
    a.scales = scales;
    a.bias = bias;
    a.y = y + m0 * N;
    int* const cnt = reinterpret_cast<int*>(sx + f32_segs(K, p) * mr);
    int* const idx = cnt + f32_segs(K, p) * mr;
    a.cnt = cnt;
    a.idx = idx;
    a.part = reinterpret_cast<float*>(base + align256(3 * mr * K) +
                                      align256(f32_segs(K, p) * mr * (2 + kMaxSpikes) * 4));
    a.M = static_cast<int>(mr);
    a.N = static_cast<int>(N);
    a.K = static_cast<int>(K);
    a.tiles_m = static_cast<int>(cdiv(mr, 32LL * p.wm));
    a.tiles_n = static_cast<int>(cdiv(N, 32LL * p.tn * (8 / p.wm)));
    a.splits = p.splits;
    a.split_steps = p.steps;
    a.segs = f32_segs(K, p);
    a.seg_len = a.segs > 1 ? p.steps * 64 : static_cast<int>(K);
    const dim3 dg(static_cast<unsigned>(mr), static_cast<unsigned>(a.segs)), db(kBlock);
    if (a.seg_len <= 4 * 4 * kBlock) k_f32_digits<4><<<dg, db, 0, s>>>(a, base, sx, cnt, idx);
    else k_f32_digits<f32lin::kMaxSeg / (4 * kBlock)><<<dg, db, 0, s>>>(a, base, sx, cnt, idx);
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
