// True 32-bit matrix product: C[M][N] (+)= A[M][K] * W[N][K]^T (+ bias[N]).
// out[t][o] = dot(W[o][:], x[t][:]) + b[o], as src/graph/cpu_backend.rs:214-248 of
// yusiwen/minfer.  32-bit operands, products and sums throughout, no reduced-precision matrix mode: this is the
// path that shows faults bfloat16 hides.  Any M, N, K; vector loads only where they are aligned.
//
// Three kernels:
//  * `rows_f32_kernel`: at most 8 rows, K in 4s (and not short for many weight rows): the weight stream, a wave a few weight rows.
//  * `tile_f32_kernel`: aligned operands and K in 32s: 64 x 64 tiles on the 32-bit matrix instruction (an FMA a product,
//    twice the vector units' rate), K split over blocks where the tiles leave CUs idle.
//  * `gemm_f32_kernel`: everything else, from LDS with vector FMA.
// A dot product is summed in chains of 128 terms whose sums are then added up: the rounding
// error of one long chain grows with the root of its length (18944 terms in the down product;
// the reference's scalar path sums in 64 bits, src/vec_ops.rs:31-35), that of short chains with the
// roots of a chain's and of the number of chains.  (`rows_f32_kernel`: 128 chains of K / 128 terms, which errs less
// than chains of 128 at any K.)
#include <algorithm>
#include <type_traits>

#include "common.h"

namespace {

constexpr int BM = 64, BN = 64, BK = 16, PAD = 4;

// Loads 4 consecutive k of one row into a float4, zero beyond the row count or K.
__device__ __forceinline__ float4 load4(const float* __restrict__ base, int ld, int row, int rows,
                                        int k, int K, bool vec_ok) {
  float4 v = make_float4(0.f, 0.f, 0.f, 0.f);
  if (row < rows) {
    const float* p = base + (size_t)row * ld + k;
    if (vec_ok && k + 4 <= K) {
      v = *reinterpret_cast<const float4*>(p);
    } else {
      if (k + 0 < K) v.x = p[0];
      if (k + 1 < K) v.y = p[1];
      if (k + 2 < K) v.z = p[2];
      if (k + 3 < K) v.w = p[3];
    }
  }
  return v;
}

template <bool ACCUMULATE>
__global__ __launch_bounds__(256) void gemm_f32_kernel(const float* __restrict__ A, int lda,
                                                       const float* __restrict__ W, int ldw,
                                                       const float* __restrict__ bias,
                                                       float* __restrict__ C, int ldc, int M, int N,
                                                       int K, int vec_ok) {
  __shared__ float As[BK][BM + PAD];
  __shared__ float Ws[BK][BN + PAD];
  const int tid = threadIdx.x;
  const int m0 = blockIdx.y * BM, n0 = blockIdx.x * BN;
  const int lrow = tid >> 2, lk = (tid & 3) * 4;   // 64 rows x 4 chunks of 4 k
  const int ty = tid >> 4, tx = tid & 15;
  constexpr int FLUSH = 128 / BK;                   // chunks per block of the sum
  float acc[4][4] = {}, tot[4][4] = {};
  int chunk = 0;
  for (int k0 = 0; k0 < K; k0 += BK) {
    const float4 a = load4(A, lda, m0 + lrow, M, k0 + lk, K, vec_ok);
    const float4 w = load4(W, ldw, n0 + lrow, N, k0 + lk, K, vec_ok);
    __syncthreads();
    As[lk + 0][lrow] = a.x; As[lk + 1][lrow] = a.y; As[lk + 2][lrow] = a.z; As[lk + 3][lrow] = a.w;
    Ws[lk + 0][lrow] = w.x; Ws[lk + 1][lrow] = w.y; Ws[lk + 2][lrow] = w.z; Ws[lk + 3][lrow] = w.w;
    __syncthreads();
#pragma unroll
    for (int k = 0; k < BK; ++k) {
      const float4 av = *reinterpret_cast<const float4*>(&As[k][ty * 4]);
      const float4 wv = *reinterpret_cast<const float4*>(&Ws[k][tx * 4]);
      const float ar[4] = {av.x, av.y, av.z, av.w};
      const float wr[4] = {wv.x, wv.y, wv.z, wv.w};
#pragma unroll
      for (int i = 0; i < 4; ++i)
#pragma unroll
        for (int j = 0; j < 4; ++j) acc[i][j] = fmaf(ar[i], wr[j], acc[i][j]);
    }
    if (++chunk == FLUSH) {
      chunk = 0;
#pragma unroll
      for (int i = 0; i < 4; ++i)
#pragma unroll
        for (int j = 0; j < 4; ++j) {
          tot[i][j] += acc[i][j];
          acc[i][j] = 0.f;
        }
    }
  }
#pragma unroll
  for (int i = 0; i < 4; ++i)
#pragma unroll
    for (int j = 0; j < 4; ++j) acc[i][j] += tot[i][j];
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const int m = m0 + ty * 4 + i;
    if (m >= M) continue;
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const int n = n0 + tx * 4 + j;
      if (n >= N) continue;
      float v = acc[i][j];
      if (bias) v += bias[n];
      float* c = C + (size_t)m * ldc + n;
      *c = ACCUMULATE ? *c + v : v;
    }
  }
}

// ---- many rows on the matrix cores
// A 64 x 64 tile on 4 waves of 32 x 32 (16x16x4 products).  k tiles of 32 (a row is a 128-byte line) travel global -> LDS
// in two stages, chunk c of row r at position c ^ ((r >> 1) & 7); a lane reads four neighbouring k of its row at once
// and the e-th of them goes into the e-th product, so a product's four k are 4 apart (the order of a sum's terms within
// sixteen).  The products are what bounds it (1,024 cycles a k tile for 256 of LDS reads); 32 KB of LDS let five
// blocks share a CU, whose waves cover each other's waits (three stages and three blocks: level to 3 % slower).
// 4,096^3 runs at 136 TFLOP/s.  611 rows (0.5B widths): gate|up 9,728 x 896 104 us (95 with the weights in the memory-side
// cache; 640 rows at 136 TFLOP/s are 82), with vector FMA 152; q|k|v 1,152 x 896 74 and 21 (K in 4 parts);
// down 896 x 4,864 61 (in 5).
constexpr int T_BM = 64, T_BK = 32, T_STAGES = 2, T_ROW = T_BK * 4, T_STAGE = 2 * T_BM * T_ROW;

__device__ __forceinline__ void dma16(const float* base, unsigned off, unsigned lds_byte) {
  asm volatile("s_mov_b32 m0, %2\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %0, %1" ::"v"(off), "s"(base), "s"(lds_byte)
               : "memory", "m0");
}

// SPLIT: sums without bias into this part's slab of C, [parts][M][N]; else the product's own epilogue
// by_xcd: every XCD takes one contiguous eighth of the tiles of all parts (`tiles_by_xcd`)
// PAIR: W is N gate rows and N up rows behind them, a tile takes 32 of each (16 gates and their 16 ups in turns, so that a lane holds
// both sums of its outputs) and leaves silu(gate) up, or the clamped form with `limit`: no [M][2 N] intermediate and no kernel to read
// it (611 rows of 4,864 x 896: 102 + 7.4 us as two kernels, 102 so).
template <bool ACCUMULATE, bool SPLIT, bool PAIR = false>
__global__ __launch_bounds__(256) void tile_f32_kernel(const float* __restrict__ A, int lda, const float* __restrict__ W, int ldw,
                                                       const float* __restrict__ bias, float* __restrict__ C, int ldc, int M, int N,
                                                       int K, int tiles_m, int k_per_split, int by_xcd, float limit = 0.f) {
  __shared__ __attribute__((aligned(16))) unsigned char smem[T_STAGES * T_STAGE];
  int at = blockIdx.y * gridDim.x + blockIdx.x;
  if (by_xcd) {
    const int n = gridDim.x * gridDim.y, per = n / 8, rem = n % 8, x = at % 8;
    at = x * per + min(x, rem) + at / 8;
  }
  const int part = at / (int)gridDim.x, tile = at - part * (int)gridDim.x;
  if (SPLIT) {
    const int kb = part * k_per_split;
    A += kb;
    W += kb;
    K = min(k_per_split, K - kb);
    C += (size_t)part * M * N;
  }
  const int m0 = (tile % tiles_m) * T_BM, n0 = (tile / tiles_m) * (PAIR ? T_BM / 2 : T_BM);
  const int lane = threadIdx.x & 63, wid = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int wm = (wid & 1) * 32, wn = (wid >> 1) * 32;
  const int fr = lane & 15, fk = lane >> 4;
  const unsigned lds0 = (unsigned)(uintptr_t)smem;
  // a wave copies pieces of 8 rows: 2 of A's 8 and 2 of W's 8
  unsigned ga[2], gw[2];
#pragma unroll
  for (int q = 0; q < 2; ++q) {
    const int r = (q * 4 + wid) * 8 + (lane >> 3), c = ((lane & 7) ^ ((r >> 1) & 7)) * 4;
    ga[q] = ((unsigned)min(m0 + r, M - 1) * (unsigned)lda + c) * 4u;
    const int row = PAIR ? min(n0 + (r >> 5) * 16 + (r & 15), N - 1) + ((r >> 4) & 1) * N : min(n0 + r, N - 1);
    gw[q] = ((unsigned)row * (unsigned)ldw + c) * 4u;
  }
  const int nkt = K / T_BK;
  auto copy = [&](int kt, int st) {               // (past the last tile: that one again, never read)
    const int k = min(kt, nkt - 1) * T_BK;
    const unsigned base = lds0 + st * T_STAGE + wid * 1024;
#pragma unroll
    for (int q = 0; q < 2; ++q) dma16(A + k, ga[q], __builtin_amdgcn_readfirstlane(base + q * 4096));
#pragma unroll
    for (int q = 0; q < 2; ++q) dma16(W + k, gw[q], __builtin_amdgcn_readfirstlane(base + T_BM * T_ROW + q * 4096));
  };
  floatx4 acc[2][2], tot[2][2];
#pragma unroll
  for (int i = 0; i < 2; ++i)
#pragma unroll
    for (int j = 0; j < 2; ++j) acc[i][j] = tot[i][j] = floatx4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
  for (int t = 0; t < T_STAGES - 1; ++t) copy(t, t);
  const int sw = (fr >> 1) & 7;
  int st = 0;
  for (int kt = 0; kt < nkt; ++kt) {
    // tile kt has landed for this wave (the younger ones' four copies each may be in flight), and behind the barrier for all;
    // the stage of tile kt - 1, which every wave holds in registers by then, takes the next one
    asm volatile("s_waitcnt vmcnt(%0)" ::"n"(4 * (T_STAGES - 2)) : "memory");
    __syncthreads();
    copy(kt + T_STAGES - 1, st == 0 ? T_STAGES - 1 : st - 1);
    const unsigned char* s = smem + st * T_STAGE;
    float4 a[2][2], w[2][2];
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      const int pos = ((4 * h + fk) ^ sw) * 16;
#pragma unroll
      for (int i = 0; i < 2; ++i) {
        a[h][i] = *reinterpret_cast<const float4*>(s + (wm + i * 16 + fr) * T_ROW + pos);
        w[h][i] = *reinterpret_cast<const float4*>(s + T_BM * T_ROW + (wn + i * 16 + fr) * T_ROW + pos);
      }
    }
#pragma unroll
    for (int h = 0; h < 2; ++h)
#pragma unroll
      for (int e = 0; e < 4; ++e)
#pragma unroll
        for (int i = 0; i < 2; ++i)
#pragma unroll
          for (int j = 0; j < 2; ++j)
            acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x4f32((&w[h][j].x)[e], (&a[h][i].x)[e], acc[i][j], 0, 0, 0);
    if ((kt & 3) == 3) {                          // 128 terms
#pragma unroll
      for (int i = 0; i < 2; ++i)
#pragma unroll
        for (int j = 0; j < 2; ++j) {
          tot[i][j] += acc[i][j];
          acc[i][j] = floatx4{0.f, 0.f, 0.f, 0.f};
        }
    }
    st = st == T_STAGES - 1 ? 0 : st + 1;
  }
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
  // D: the lane's row is lane % 16, its columns 4 (lane / 16) + e
  // (what a short K takes is the stores: 1,500 rows against 24,000 of 32 92 us with 4-byte ones, 45 so)
  const bool vec = ldc % 4 == 0 && (uintptr_t)C % 16 == 0;
#pragma unroll
  for (int i = 0; i < 2; ++i) {
    const int m = m0 + wm + i * 16 + fr;
    if (m >= M) continue;
    if constexpr (PAIR) {
      const int n = n0 + wn / 2 + fk * 4;
      const floatx4 g = acc[i][0] + tot[i][0], u = acc[i][1] + tot[i][1];
      floatx4 v;
#pragma unroll
      for (int e = 0; e < 4; ++e) v[e] = limit > 0.f ? clamped_gate(g[e], u[e], limit) : g[e] / (1.0f + expf(-g[e])) * u[e];
      float* c = C + (size_t)m * ldc + n;
      if (vec && n + 4 <= N) *reinterpret_cast<floatx4*>(c) = v;
      else
#pragma unroll
        for (int e = 0; e < 4; ++e)
          if (n + e < N) c[e] = v[e];
      continue;
    }
#pragma unroll
    for (int j = 0; j < 2; ++j) {
      const int n = n0 + wn + j * 16 + fk * 4;
      floatx4 v = acc[i][j] + tot[i][j];
      float* c = C + (size_t)m * ldc + n;
      if (!SPLIT && bias) {
#pragma unroll
        for (int e = 0; e < 4; ++e) v[e] += n + e < N ? bias[n + e] : 0.f;
      }
      if (vec && n + 4 <= N) {
        if (ACCUMULATE) v = *reinterpret_cast<const floatx4*>(c) + v;
        *reinterpret_cast<floatx4*>(c) = v;
        continue;
      }
#pragma unroll
      for (int e = 0; e < 4; ++e)
        if (n + e < N) c[e] = ACCUMULATE ? c[e] + v[e] : v[e];
    }
  }
}

// adds the parts of a K split in their order, then the bias, then (ACCUMULATE) what C held
template <bool ACCUMULATE>
__global__ __launch_bounds__(256) void add_parts_f32_kernel(const float* __restrict__ part, const float* __restrict__ bias,
                                                            float* __restrict__ C, int ldc, int M, int N, int splits) {
  const size_t x = (size_t)blockIdx.x * 256 + threadIdx.x, mn = (size_t)M * N;
  if (x >= mn) return;
  const int m = x / N, n = x % N;
  float v = 0.f;
  for (int s0 = 0; s0 < splits; s0 += 8) {        // eight parts' loads in flight together
    float p[8];
#pragma unroll
    for (int s = 0; s < 8; ++s) p[s] = s0 + s < splits ? part[(size_t)(s0 + s) * mn + x] : 0.f;
#pragma unroll
    for (int s = 0; s < 8; ++s) v += p[s];
  }
  if (bias) v += bias[n];
  float* c = C + (size_t)m * ldc + n;
  *c = ACCUMULATE ? *c + v : v;
}

// The same with the RMS norm of the new rows beside it (C / sqrt(mean(C^2) + eps) g): a block a row, which it holds in registers
// between the sum of squares and the scaling.  The additions in their order, the norm in that of rmsnorm_kernel.  One launch for two,
// and the rows are not read again (611 rows of 896 in 5 parts: 4.9 + 5.0 us as two kernels).
template <int KEEP>
__global__ __launch_bounds__(256) void add_norm_f32_kernel(const float* __restrict__ part, const float* __restrict__ bias,
                                                           float* __restrict__ C, int ldc, int M, int N, int splits, int accumulate,
                                                           const float* __restrict__ g, float eps, float* __restrict__ normed) {
  __shared__ float scratch[4];
  const int m = blockIdx.x;
  const size_t mn = (size_t)M * N;
  const float* p = part + (size_t)m * N;
  float* c = C + (size_t)m * ldc;
  float4 v[KEEP];
  float ss = 0.f;
#pragma unroll
  for (int q = 0; q < KEEP; ++q) {
    const int n = (q * 256 + threadIdx.x) * 4;
    v[q] = float4{0.f, 0.f, 0.f, 0.f};
    if (n < N) {
      const float4 old = accumulate ? *reinterpret_cast<const float4*>(c + n) : v[q];
      for (int s0 = 0; s0 < splits; s0 += 8) {
        float4 x[8];
#pragma unroll
        for (int s = 0; s < 8; ++s)
          x[s] = s0 + s < splits ? *reinterpret_cast<const float4*>(p + (size_t)(s0 + s) * mn + n) : float4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int s = 0; s < 8; ++s) { v[q].x += x[s].x; v[q].y += x[s].y; v[q].z += x[s].z; v[q].w += x[s].w; }
      }
      if (bias) {
        const float4 b = *reinterpret_cast<const float4*>(bias + n);
        v[q] = float4{v[q].x + b.x, v[q].y + b.y, v[q].z + b.z, v[q].w + b.w};
      }
      if (accumulate) v[q] = float4{old.x + v[q].x, old.y + v[q].y, old.z + v[q].z, old.w + v[q].w};
      *reinterpret_cast<float4*>(c + n) = v[q];
    }
    ss = fmaf(v[q].x, v[q].x, ss);
    ss = fmaf(v[q].y, v[q].y, ss);
    ss = fmaf(v[q].z, v[q].z, ss);
    ss = fmaf(v[q].w, v[q].w, ss);
  }
  ss = block_sum<256>(ss, scratch);
  const float scale = 1.0f / sqrtf(ss / (float)N + eps);
#pragma unroll
  for (int q = 0; q < KEEP; ++q) {
    const int n = (q * 256 + threadIdx.x) * 4;
    if (n < N) {
      const float4 w = *reinterpret_cast<const float4*>(g + n);
      *reinterpret_cast<float4*>(normed + (size_t)m * N + n) =
          float4{v[q].x * scale * w.x, v[q].y * scale * w.y, v[q].z * scale * w.z, v[q].w * scale * w.w};
    }
  }
}
constexpr int ADD_NORM_MAX = 256 * 4 * 16;        // a row's values that a block holds

// How many blocks share a tile's K.  The chip's time is that of the CU with the most tiles, times their k tiles (and some four
// more a tile for its start), at 0.46 us a k tile where three or more share a CU and somewhat more where two or one do; the
// parts' way to memory and back and the second kernel come on top.  (611 rows against 896 of 4,864, 140 tiles: 4 parts, 560 on
// 256 CUs, 71 us; 5 parts 54.  The constants are those with the least loss over 233 shapes of 9 to 4,000 rows timed at up to 11
// numbers of parts each: 6 % above the best of each on the average, and nowhere more than 3 % above cutting in parts of 256 until
// every CU has two tiles.)
int tile_splits(int M, int N, int K, int n_cu) {
  const long tiles = (long)((M + T_BM - 1) / T_BM) * ((N + T_BM - 1) / T_BM), nkt = K / T_BK;
  long best = 1;
  double best_us = 1e30;
  for (long parts = 1; parts <= std::min<long>(std::max<long>(1, nkt / 7), 16); ++parts) {
    const long per = (nkt + parts - 1) / parts, most = (tiles * parts + n_cu - 1) / n_cu;
    if ((nkt + per - 1) / per != parts) continue;
    const double step_us = most >= 3 ? 0.46 : most == 2 ? 0.54 : 0.7;
    const double us = (double)(most * (per + 4)) * step_us + (parts > 1 ? 3. + (double)(parts + 1) * M * N * 4. / 3.5e6 : 0.);
    if (us < best_us) {
      best_us = us;
      best = parts;
    }
  }
  return (int)best;
}

// An eighth of the tiles an XCD, each with an L2 of 4 MB: whole products whose activations stay in it beside the weights (each XCD
// then reads an eighth of these: 611 rows against 9,728 of 896 109 us and 104, 400 against 17,920 of 1,536 219 and 202; 2,000
// against 9,728 of 896 274 and 284), and parts of activations that would not (an XCD then reads a part or two: 400 x 1,536 x
// 8,960 119 us and 112; 611 x 1,152 x 896 24 and 25).
int tiles_by_xcd(int M, int K, int splits) {
  const size_t bytes = (size_t)M * K * 4;
  return splits > 1 ? bytes > (4u << 20) : bytes <= (3u << 20);
}

bool tile_takes(int M, int N, int K, int lda, int ldw, const void* A, const void* W) {
  return K % T_BK == 0 && lda % 4 == 0 && ldw % 4 == 0 && (uintptr_t)A % 16 == 0 && (uintptr_t)W % 16 == 0 &&
         (size_t)M * lda * 4 < (1ull << 32) && (size_t)N * ldw * 4 < (1ull << 32);
}

// ---- few rows: the weight stream
// The sums of a wave's lanes: a lane's N sums meet those of the lane O away, which keeps the one half of them and hands over the
// other while there are several: the additions of a `wave_sum` for each, in their order, with a sixth of the shuffles for
// 32 sums (8 rows against 24,000 of 64 16.5 us with a `wave_sum` each, 6.6 so).  Sum s ends in the lanes s 64 / N on.
template <int N, int O>
__device__ __forceinline__ void meet(float* sum, int lane) {
  if constexpr (N > 1) {
    const bool upper = lane & O;
#pragma unroll
    for (int x = 0; x < N / 2; ++x) {
      const float lo = sum[x], hi = sum[x + N / 2];
      sum[x] = (upper ? hi : lo) + __shfl_xor(upper ? lo : hi, O, MF_WAVE);
    }
  } else {
    sum[0] += __shfl_xor(sum[0], O, MF_WAVE);
  }
  if constexpr (O > 1) meet<(N > 1 ? N / 2 : 1), O / 2>(sum, lane);
}

// A wave takes NR weight rows (four where the matrix is tall enough to keep every SIMD busy all the same: the activations
// are then read once for four rows) and walks K in runs of 256, a float4 a lane; its sums meet by shuffles.
// The head of the 0.5B widths (151,936 x 896, one row): 204 us before, 92 now, 5.9 TB/s.
template <int MR, int NR, bool ACCUMULATE>
__global__ __launch_bounds__(256) void rows_f32_kernel(const float* __restrict__ A, int lda, const float* __restrict__ W, int ldw,
                                                       const float* __restrict__ bias, float* __restrict__ C, int ldc, int M, int N,
                                                       int K) {
  const int lane = threadIdx.x & 63;
  const int n0 = (blockIdx.x * 4 + (threadIdx.x >> 6)) * NR;
  if (n0 >= N) return;
  const float* w[NR];
#pragma unroll
  for (int j = 0; j < NR; ++j) w[j] = W + (size_t)min(n0 + j, N - 1) * ldw;
  float acc[MR][NR][2] = {};
  // Eight sums or more: U runs of 256 at a time, all their loads on their way before the first is waited for (left to the
  // scheduler the loads of eight rows are waited for one by one: 8 rows against 1,536 of 8,960 26 us so, 78).  Fewer: the
  // scheduler's order, which mixes the next run's loads with this one's products (4 rows against 512 of 8,960 10.0 us in runs
  // of two, 8.4 so; four rows against four weight rows each the other way round: 24,000 of 260 6.4 and 8.0).
  constexpr bool ORDERED = MR * NR >= 8;
  constexpr int U = MR * NR >= 16 ? 1 : 2;
  auto runs = [&](auto COUNT, int k) {
    constexpr int C = decltype(COUNT)::value;
    float4 x[C][NR], a[C][MR];
#pragma unroll
    for (int u = 0; u < C; ++u) {
#pragma unroll
      for (int j = 0; j < NR; ++j) x[u][j] = *reinterpret_cast<const float4*>(w[j] + k + 256 * u);
#pragma unroll
      for (int i = 0; i < MR; ++i) a[u][i] = *reinterpret_cast<const float4*>(A + (size_t)min(i, M - 1) * lda + k + 256 * u);
    }
    if (ORDERED) __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int u = 0; u < C; ++u)
#pragma unroll
      for (int i = 0; i < MR; ++i)
#pragma unroll
        for (int j = 0; j < NR; ++j) {
          acc[i][j][0] = fmaf(a[u][i].y, x[u][j].y, fmaf(a[u][i].x, x[u][j].x, acc[i][j][0]));
          acc[i][j][1] = fmaf(a[u][i].w, x[u][j].w, fmaf(a[u][i].z, x[u][j].z, acc[i][j][1]));
        }
  };
  int k = lane * 4;
  if constexpr (ORDERED) {
    for (; k + 256 * (U - 1) < K; k += 256 * U) runs(std::integral_constant<int, U>{}, k);
    if (U > 1 && k < K) runs(std::integral_constant<int, 1>{}, k);
  } else {
#pragma unroll 2
    for (; k < K; k += 256) runs(std::integral_constant<int, 1>{}, k);
  }
  constexpr int SUMS = MR * NR;
  float sum[SUMS];
#pragma unroll
  for (int i = 0; i < MR; ++i)
#pragma unroll
    for (int j = 0; j < NR; ++j) sum[i * NR + j] = acc[i][j][0] + acc[i][j][1];
  meet<SUMS, 32>(sum, lane);
  constexpr int EACH = 64 / SUMS;
  const int i = lane / EACH / NR, n = n0 + lane / EACH % NR;
  if (lane % EACH == 0 && i < M && n < N) {
    const float v = bias ? sum[0] + bias[n] : sum[0];
    float* c = C + (size_t)i * ldc + n;
    *c = ACCUMULATE ? *c + v : v;
  }
}

template <int MR, int NR>
int launch_rows(const float* A, int lda, const float* W, int ldw, const float* bias, float* C, int ldc, int M, int N, int K,
                int accumulate, hipStream_t stream) {
  const int grid = (N + 4 * NR - 1) / (4 * NR);
  if (accumulate) rows_f32_kernel<MR, NR, true><<<grid, 256, 0, stream>>>(A, lda, W, ldw, bias, C, ldc, M, N, K);
  else rows_f32_kernel<MR, NR, false><<<grid, 256, 0, stream>>>(A, lda, W, ldw, bias, C, ldc, M, N, K);
  return mf_launch_status();
}

constexpr int TALL = 16384;                       // weight rows from which a wave takes four of them
template <int MR>
int launch_rows_n(const float* A, int lda, const float* W, int ldw, const float* bias, float* C, int ldc, int M, int N, int K,
                  int accumulate, hipStream_t stream) {
  return N >= TALL ? launch_rows<MR, 4>(A, lda, W, ldw, bias, C, ldc, M, N, K, accumulate, stream)
                   : launch_rows<MR, 1>(A, lda, W, ldw, bias, C, ldc, M, N, K, accumulate, stream);
}

// At most 8 rows, K in 4s, except many weight rows of a short K: a wave's time does not fall with K below 256 (fewer of its lanes
// have work, and its sums meet all the same), a tile's does.  As tiles / so: 8 rows against 100,000 of 48 11.4 us / 16.9, of
// 80 17.0 / 17.9, one row of 16 5.2 / 6.7; 8 rows against 9,728 of 16 4.3 / 5.9, against 2,048 of 16 5.1 / 3.9.
bool rows_take(int M, int N, int K) {
  if (M > 8 || K % 4) return false;
  const int mr = M <= 2 ? M : M <= 4 ? 4 : 8;
  return K > (N >= TALL ? 8 * mr + (mr > 1 ? 16 : 8) : N >= 8192 ? 4 * mr : 0);
}

}  // namespace

// How many parts K is cut into (1: none): `mf_gemm_f32` with more than one needs part [parts][M][N].
// `aligned`: 16-byte aligned operands with row strides in multiples of 4.
MF_API int mf_gemm_f32_splits(int M, int N, int K, int aligned, int n_cu) {
  if (M <= 8 || N <= 0 || K < T_BK || n_cu <= 0 || !aligned || K % T_BK || (size_t)M * K * 4 >= (1ull << 32) || (size_t)N * K * 4 >= (1ull << 32)) return 1;
  return tile_splits(M, N, K, n_cu);
}

static const int NOT_BUILT = -2;     // an entry point's answer for a shape it has no kernel for; nothing was launched

// The parts of a K split alone, [splits][M][N] without bias, for a kernel behind the product that adds them; `splits` (2 and more) as
// `mf_gemm_f32_splits` gives it.
MF_API int mf_gemm_f32_parts(const float* A, int lda, const float* W, int ldw, float* part, int M, int N, int K, int splits,
                             hipStream_t stream) {
  if (M <= 0 || N <= 0) return 0;
  if (K <= 0 || lda < K || ldw < K || splits < 2 || !part) return (int)hipErrorInvalidValue;
  if (!tile_takes(M, N, K, lda, ldw, A, W)) return NOT_BUILT;
  const int tiles_m = (M + T_BM - 1) / T_BM, tiles = tiles_m * ((N + T_BM - 1) / T_BM);
  const int per = (K / T_BK + splits - 1) / splits * T_BK;
  if ((long)(splits - 1) * per >= K) return (int)hipErrorInvalidValue;
  tile_f32_kernel<false, true><<<dim3(tiles, splits), 256, 0, stream>>>(A, lda, W, ldw, nullptr, part, N, M, N, K, tiles_m, per,
                                                                        tiles_by_xcd(M, K, splits));
  return mf_launch_status();
}

// The product cut over K into C (stored or added to), with the RMS norm of the new rows beside it, normed [M][N].  N in fours, at most
// 16,384, every operand 16-byte aligned; NOT_BUILT (nothing launched) for any other.
MF_API int mf_gemm_f32_norm(const float* A, int lda, const float* W, int ldw, const float* bias, float* C, int ldc, float* part, int M,
                            int N, int K, int splits, int accumulate, const float* g, float eps, float* normed, hipStream_t stream) {
  if (M <= 0 || N <= 0) return 0;
  if (ldc < N || !g || !normed) return (int)hipErrorInvalidValue;
  if (N % 4 || N > ADD_NORM_MAX || ldc % 4 || (uintptr_t)C % 16 || (uintptr_t)part % 16 || (uintptr_t)bias % 16 || (uintptr_t)g % 16 ||
      (uintptr_t)normed % 16)
    return NOT_BUILT;
  const int rc = mf_gemm_f32_parts(A, lda, W, ldw, part, M, N, K, splits, stream);
  if (rc) return rc;
  auto run = [&](auto KEEP) {
    add_norm_f32_kernel<decltype(KEEP)::value><<<M, 256, 0, stream>>>(part, bias, C, ldc, M, N, splits, accumulate, g, eps, normed);
  };
  if (N <= 1024) run(std::integral_constant<int, 1>{});
  else if (N <= 2048) run(std::integral_constant<int, 2>{});
  else if (N <= 4096) run(std::integral_constant<int, 4>{});
  else if (N <= 8192) run(std::integral_constant<int, 8>{});
  else run(std::integral_constant<int, 16>{});
  return mf_launch_status();
}

// C [M][N] = silu(gate) up (limit > 0: the clamped form) of A and W, N gate rows and N up rows behind them; K whole.  NOT_BUILT (nothing
// launched) where the tiles do not take the operands.
MF_API int mf_gemm_f32_swiglu(const float* A, int lda, const float* W, int ldw, float* C, int ldc, int M, int N, int K, float limit,
                              hipStream_t stream) {
  if (M <= 0 || N <= 0) return 0;
  if (K <= 0 || lda < K || ldw < K || ldc < N) return (int)hipErrorInvalidValue;
  if (!tile_takes(M, 2 * N, K, lda, ldw, A, W)) return NOT_BUILT;
  const int tiles_m = (M + T_BM - 1) / T_BM, tiles = tiles_m * ((N + T_BM / 2 - 1) / (T_BM / 2));
  tile_f32_kernel<false, false, true><<<tiles, 256, 0, stream>>>(A, lda, W, ldw, nullptr, C, ldc, M, N, K, tiles_m, 0, tiles_by_xcd(M, K, 1),
                                                                 limit);
  return mf_launch_status();
}

MF_API int mf_gemm_f32(const float* A, int lda, const float* W, int ldw, const float* bias, float* C, int ldc, float* part,
                       int M, int N, int K, int splits, int accumulate, hipStream_t stream) {
  if (M <= 0 || N <= 0) return 0;
  if (K <= 0 || lda < K || ldw < K || ldc < N) return (int)hipErrorInvalidValue;
  const int vec_ok = (lda % 4 == 0) && (ldw % 4 == 0) && ((uintptr_t)A % 16 == 0) &&
                     ((uintptr_t)W % 16 == 0);
  if (vec_ok && rows_take(M, N, K)) {
    if (M == 1) return launch_rows_n<1>(A, lda, W, ldw, bias, C, ldc, M, N, K, accumulate, stream);
    if (M == 2) return launch_rows_n<2>(A, lda, W, ldw, bias, C, ldc, M, N, K, accumulate, stream);
    if (M <= 4) return launch_rows_n<4>(A, lda, W, ldw, bias, C, ldc, M, N, K, accumulate, stream);
    return launch_rows_n<8>(A, lda, W, ldw, bias, C, ldc, M, N, K, accumulate, stream);
  }
  if (tile_takes(M, N, K, lda, ldw, A, W)) {
    const int tiles_m = (M + T_BM - 1) / T_BM, tiles = tiles_m * ((N + T_BM - 1) / T_BM);
    if (splits > 1) {
      const int rc = mf_gemm_f32_parts(A, lda, W, ldw, part, M, N, K, splits, stream);
      if (rc) return rc;
      const unsigned blocks = (unsigned)(((size_t)M * N + 255) / 256);
      if (accumulate) add_parts_f32_kernel<true><<<blocks, 256, 0, stream>>>(part, bias, C, ldc, M, N, splits);
      else add_parts_f32_kernel<false><<<blocks, 256, 0, stream>>>(part, bias, C, ldc, M, N, splits);
      return mf_launch_status();
    }
    const int by_xcd = tiles_by_xcd(M, K, 1);
    if (accumulate) tile_f32_kernel<true, false><<<tiles, 256, 0, stream>>>(A, lda, W, ldw, bias, C, ldc, M, N, K, tiles_m, 0, by_xcd);
    else tile_f32_kernel<false, false><<<tiles, 256, 0, stream>>>(A, lda, W, ldw, bias, C, ldc, M, N, K, tiles_m, 0, by_xcd);
    return mf_launch_status();
  }
  dim3 grid((N + BN - 1) / BN, (M + BM - 1) / BM);
  if (accumulate)
    gemm_f32_kernel<true><<<grid, 256, 0, stream>>>(A, lda, W, ldw, bias, C, ldc, M, N, K, vec_ok);
  else
    gemm_f32_kernel<false><<<grid, 256, 0, stream>>>(A, lda, W, ldw, bias, C, ldc, M, N, K, vec_ok);
  return mf_launch_status();
}
