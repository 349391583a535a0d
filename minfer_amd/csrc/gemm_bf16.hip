// bfloat16 matrix products on the gfx950 matrix cores, 32-bit accumulation:
//   C[M][N] (+)= A[M][K] * W[N][K]^T (+ bias[N])
// (out[t][o] = dot(W[o][:], x[t][:]) + b[o], src/graph/cpu_backend.rs:214-248 of
// yusiwen/minfer; the reference's own matrix kernels are quantised and are not followed.)
//
// The kernels:
//  * `tile_dma_kernel`: many rows (prompts), aligned operands: tiles of 256 x 256, 256 x 192, 256 x 128 or 128 x 256 with
//    their k tiles copied straight into LDS, 16x16x32 MFMA, two groups of four waves a quarter product apart.
//  * `tile_step_kernel`: the same copies for tiles of 128 x 128 and 64 x 64 (fewer rows, and 17 to 64 rows against a short
//    K), one barrier a k tile.
//  * `tile_stream_kernel`: more than 128 rows whose tiles are all on the chip at once, weights from the tiled copy straight into MFMA
//    operands.
//  * `tile_kernel`: many rows of any alignment, through registers and double-buffered LDS, 32x32x16 MFMA.
//  * `reduce_norm_kernel`: adds the parts of a K split into the stream and norms the new rows.
//  * `stationary16_kernel`: at most 16 rows and K of 896, 1536, 2048, 3584, 4096, 5120 or 8192 (decode):
//    one block per CU keeps the activations in registers and walks over weight tiles.
//  * `rolling16_kernel`, `skinny16_kernel`: at most 16 rows, any K (decode).  The time is the
//    weight stream: the waves of a block split K, each reads weights and activations straight
//    into MFMA operands (16x16x32) and the partial sums meet in LDS.
//  * `panel_kernel`: 17 to 64 rows against a wide matrix: one block per CU over the whole of K; `panel_dma_kernel`: the same for up to
//    128 rows with copies straight into LDS, where all its tiles are on the chip at once.
//  * `whole_kernel`: 17 to 64 rows with a norm folded in on either side, a short K: one kernel over the whole of K.
//  * `skinny_ring_kernel`, `skinny_kernel` (any alignment): 17 to 64 rows.  Each wave owns 16
//    weight rows and reads them from HBM straight into MFMA operands, the activation rows are
//    staged in LDS and shared by the block, K may be split over blocks with a fixed-order
//    reduction afterwards.
// Both operands have K contiguous, which is exactly the MFMA operand layout (8 consecutive
// k per lane), so nothing is transposed.  The kernels for at most 64 rows (all but the guarded
// skinny16_kernel) can read the weights from a tiled copy instead (`w_operand`), where the
// caller has one.
//
// Epilogues: 0 store fp32, 1 add into fp32 (residual stream), 2 store bf16, 3 SwiGLU, 4 xIELU and 5 the square of relu (both bf16).
// SwiGLU (y = silu(g) * u, silu(z) = z / (1 + exp(-z)), src/graph/cpu_backend.rs:323-329):
// the weight rows come interleaved in groups of 64, 32 gate rows then the 32 up rows of the
// same outputs (the last group padded with zero rows), so a gate column and its up column
// are 32 apart inside one wave's tile; the epilogue writes bfloat16 y[M][ldc], ldc = number
// of outputs, straight from the 32-bit accumulators and the [M][2 nf] intermediate is never
// stored.  Its products have no bias; where `bias` is given all the same, it points to one number,
// the limit of the clamped form y = g sigmoid(1.702 g) (u + 1), g = min(gate, limit),
// u = clamp(up, -limit, limit), which takes silu's place.
#include <stdio.h>
#include <stdlib.h>

#include "common.h"

namespace {

// EPI_XIELU: bfloat16 output of the xIELU activation of (sum + bias); the activation's two constants
// (a_pos, a_neg: z > 0 -> a_pos z^2 + z/2, else a_neg (e^z - 1 - z) + z/2) stand behind the N biases.
// EPI_RELU2: bfloat16 output of max(sum + bias, 0)^2.
enum { EPI_F32 = 0, EPI_ACC_F32 = 1, EPI_BF16 = 2, EPI_SWIGLU = 3, EPI_XIELU = 4, EPI_RELU2 = 5, EPI_LAST = EPI_RELU2 };

__device__ __forceinline__ float xielu_f(float z, float a_pos, float a_neg) {
  return z > 0.f ? fmaf(a_pos * z, z, 0.5f * z) : fmaf(a_neg, expm1f(z) - z, 0.5f * z);
}

__device__ __forceinline__ float relu2_f(float z) {
  z = fmaxf(z, 0.f);
  return z * z;
}

__device__ __forceinline__ void store_out(void* C, int ldc, int m, int n, float v, int epi,
                                          const float* __restrict__ bias = nullptr, int N = 0) {
  if (epi == EPI_XIELU) {
    ((bf16*)C)[(size_t)m * ldc + n] = (bf16)xielu_f(v, bias[N], bias[N + 1]);
  } else if (epi == EPI_RELU2) {
    ((bf16*)C)[(size_t)m * ldc + n] = (bf16)relu2_f(v);
  } else if (epi == EPI_BF16) {
    ((bf16*)C)[(size_t)m * ldc + n] = (bf16)v;
  } else {
    float* c = (float*)C + (size_t)m * ldc + n;
    *c = (epi == EPI_ACC_F32) ? *c + v : v;
  }
}

__device__ __forceinline__ float swiglu_f(float g, float u, const float* __restrict__ limit) {
  if (limit) return clamped_gate(g, u, *limit);
  return g / (1.0f + expf(-g)) * u;
}

// 8 consecutive k of one row, zero at and beyond k_end.  Rows are clamped by the caller to a
// row that exists (results of such rows are never stored), so the fast form has no branch:
// VEC needs 16-byte aligned rows and K a multiple of 8, so a chunk is inside or outside whole.
template <bool VEC>
__device__ __forceinline__ bf16x8 load8(const bf16* __restrict__ base, int ld, int row, int k, int k_end) {
  const bf16x8 zero = {0, 0, 0, 0, 0, 0, 0, 0};
  if (VEC) {
    const int kk = min(k, k_end - 8);
    const bf16x8 v = *reinterpret_cast<const bf16x8*>(base + (size_t)row * ld + kk);
    return k + 8 <= k_end ? v : zero;
  } else {
    bf16x8 v = zero;
    const bf16* p = base + (size_t)row * ld + k;
#pragma unroll
    for (int e = 0; e < 8; ++e)
      if (k + e < k_end) v[e] = p[e];
    return v;
  }
}

// 8 consecutive k with no guard at all: the caller knows the chunk lies inside the row.
__device__ __forceinline__ bf16x8 load8_inside(const bf16* __restrict__ base, int ld, int row, int k) {
  return *reinterpret_cast<const bf16x8*>(base + (size_t)row * ld + k);
}

// Weights that no other workgroup reads, marked as read once (ONCE) or not.  From the tiled copy a load takes whole lines and is marked as read once: what the step reads
// again stays in the caches (microseconds without / with the mark, 8 rows, weights from memory: 152,064 x 6,144 326 / 292, 152,064 x
// 3,584 194 / 175, 37,888 x 3,584 49.8 / 47.7, 4,608 x 3,584 10.5 / 9.7, 3,584 x 18,944 26.6 / 25.8; 64 rows, 37,888 x 3,584 53.4 / 48.7).  From the
// matrix a load takes half a line of each of 16 rows, and the next step takes the other half: marked, the line is fetched twice (marked / not, 8 rows:
// 152,064 x 6,144 392 / 344, 8,192 x 29,568 117 / 102, 3,584 x 18,944 35.8 / 31.4, 37,888 x 3,584 56.1 / 52.3; 64 rows:
// 152,064 x 3,584 277 / 245), except with a short K (`launch_stationary16`).  Not for what several tiles of rows read (`whole_kernel`, the prompts' tiles).
template <bool ONCE>
__device__ __forceinline__ bf16x8 load_weights(const bf16* p) {
  if constexpr (ONCE) return __builtin_nontemporal_load(reinterpret_cast<const bf16x8*>(p));
  else return *reinterpret_cast<const bf16x8*>(p);
}

// The epilogue of a wave's TM x TN tiles of 32 x 32 (D[m][n]: lane holds n = lane % 32,
// m = 8 (r / 4) + 4 (lane / 32) + r % 4): bias, then store / accumulate / round / SwiGLU.
template <int TM, int TN>
__device__ __forceinline__ void tile_epilogue(floatx16 (&acc)[TM][TN], const float* __restrict__ bias,
                                              void* __restrict__ C, int ldc, int M, int N, int epi, int m0,
                                              int wm, int n0, int wn, int lane) {
  const int fr = lane & 31;
  // D[m][n]: lane holds n = lane % 32, m = 8 (r / 4) + 4 (lane / 32) + r % 4
  if (epi == EPI_SWIGLU) {
    if constexpr (TN % 2 == 0) {
      auto gated = [&](auto act) {
#pragma unroll
        for (int i = 0; i < TM; ++i)
#pragma unroll
          for (int j = 0; j < TN; j += 2) {
            const int ng = n0 + wn + j * 32 + fr;            // gate column; its up column is ng + 32
            const int col = (ng >> 6) * 32 + (ng & 63);
            if (col >= ldc) continue;
#pragma unroll
            for (int r = 0; r < 16; ++r) {
              const int m = m0 + wm + i * 32 + (r >> 2) * 8 + (lane >> 5) * 4 + (r & 3);
              if (m < M) ((bf16*)C)[(size_t)m * ldc + col] = (bf16)act(acc[i][j][r], acc[i][j + 1][r]);
            }
          }
      };
      if (bias) {
        const float limit = *bias;
        gated([=](float g, float u) { return clamped_gate(g, u, limit); });
      } else {
        gated([](float g, float u) { return swiglu_f(g, u, nullptr); });
      }
    }
    return;
  }
#pragma unroll
  for (int i = 0; i < TM; ++i)
#pragma unroll
    for (int j = 0; j < TN; ++j) {
      const int n = n0 + wn + j * 32 + fr;
      if (n >= N) continue;
      const float b = bias ? bias[n] : 0.f;
#pragma unroll
      for (int r = 0; r < 16; ++r) {
        const int m = m0 + wm + i * 32 + (r >> 2) * 8 + (lane >> 5) * 4 + (r & 3);
        if (m < M) store_out(C, ldc, m, n, acc[i][j][r] + b, epi, bias, N);
      }
    }
}

// Tile number -> (row of tiles, column of tiles).  The tiles are numbered in bands of 8 rows of
// tiles, down a band's rows first: 32 neighbouring numbers (what an XCD has in flight, see the
// kernels) are then 8 x 4 tiles, which share 12 operand panels between them (a whole column of
// 32 tile rows would share 33).
__device__ __forceinline__ void tile_position(int tile, int tiles_m, int tiles_n, int& bm, int& bn) {
  constexpr int BAND = 8;
  const int band = tile / (BAND * tiles_n), first = band * BAND;
  const int rows = min(tiles_m - first, BAND);
  const int in_band = tile - band * BAND * tiles_n;
  bn = in_band / rows;
  bm = first + in_band - bn * rows;
}

// The tile and the part of K that a block of a grid of (tiles, parts) takes.  Workgroups go to the 8 XCDs in turn, each with an
// L2 of its own: every XCD gets one contiguous eighth of the tiles, so that what it has in flight are neighbours and share their
// operands' rows in its L2 (ORDER_TILES: the same eighth of every part); or of the tiles of all parts, part by part
// (ORDER_PARTS), so that an XCD brings in the activations of one part of K or two, and not those of all of K: for activations
// that an L2 does not hold (`tile_order`).
enum { ORDER_PLAIN = 0, ORDER_TILES = 1, ORDER_PARTS = 2 };
__device__ __forceinline__ void block_work(int order, int& tile, int& part) {
  int at = blockIdx.x, n = gridDim.x;
  if (order == ORDER_PARTS) {
    at += blockIdx.y * gridDim.x;
    n *= gridDim.y;
  }
  if (order != ORDER_PLAIN) {
    const int per = n / 8, rem = n % 8, x = at % 8;
    at = x * per + min(x, rem) + at / 8;
  }
  part = order == ORDER_PARTS ? at / (int)gridDim.x : blockIdx.y;
  tile = order == ORDER_PARTS ? at - part * (int)gridDim.x : at;
}
// Part by part where the activations of all of K are half as much again as an XCD's L2 of 4 MB and all parts' tiles are at most two a
// CU.  (rows x weight rows x K, microseconds with the kernel behind it, the same eighth of every part / part by part: 800 x 1,536 x
// 8,960 41.7 / 38.8, 1,000 x 1,024 x 8,192 38.9 / 32.2, 2,048 x 2,048 x 11,008 101.3 / 90.0, 2,048 x 896 x 4,864 38.5 / 32.8; less than
// an L2: 604 x 2,048 x 2,048 22.2 / 24.8.)  In between what an XCD reads again is little, and so it pays only for few weight rows
// of a long K: 300 x 1,024 x 8,192 24.5 / 23.2, 256 x 1,536 x 8,960 23.2 / 22.7, but 604 x 896 x 4,864 20.1 / 21.4, 129 x 3,584 x
// 18,944 46.9 / 48.6.  With more tiles the XCDs stand in different parts of K at one time: level at 462 tiles (2,600 x 3,584 x 18,944
// 312.6 / 313), slower beyond: 3,300 x 5,120 x 13,824 (780) 455 / 469, 5,754 x 3,584 x 18,944 (966) 647 / 664, 8,192 x 5,120 x 13,824
// (1,280) 913 / 932.
static int cu_count();
int tile_order(int tiles, int splits, int M, int N, int K) {
  const size_t bytes = (size_t)M * K * 2;
  const bool pays = bytes > (6u << 20) || (bytes > (4u << 20) && N <= 2048 && K >= 8192);
  if (splits > 1 && pays && (long)tiles * splits <= 2L * cu_count()) return ORDER_PARTS;
  return tiles >= 16 ? ORDER_TILES : ORDER_PLAIN;
}

// Rows of a product that belong to one of several matrices: `rows` of them (at most a tile's) from row `first` on.
struct RowGroup { int first, rows, matrix, unused; };

// ------------------------------------------------------------------ tiled kernel
// LDS row stride is BK + 8 elements (144 bytes for BK 64, 80 for BK 32): conflict-free b128 reads
template <int BM, int BN, int WM, int WN, int BK, bool VEC>
__global__ __launch_bounds__(64 * (BM / WM) * (BN / WN)) void tile_kernel(const bf16* __restrict__ A, int lda,
                                                   const bf16* __restrict__ W, int ldw,
                                                   const float* __restrict__ bias, void* __restrict__ C,
                                                   int ldc, int M, int N, int K, int epi, int tiles_m,
                                                   int order, int k_per_split) {
  constexpr int NTHR = 64 * (BM / WM) * (BN / WN);
  constexpr int LDS_LD = BK + 8;
  int tile, part;
  block_work(order, tile, part);
  if (k_per_split > 0) {
    // K cut into parts: this block multiplies k_per_split of K and stores its sums, 32-bit
    // and without bias, into its own [M][N] slab of C; another kernel adds the slabs
    const int kb = part * k_per_split;
    A += kb;
    W += kb;
    K = min(k_per_split, K - kb);
    C = (float*)C + (size_t)part * M * N;
  }
  constexpr int TM = WM / 32, TN = WN / 32;
  constexpr int RP = NTHR / (BK / 8);         // rows per load pass
  constexpr int PA = BM / RP, PW = BN / RP;
  static_assert(BM % RP == 0 && BN % RP == 0, "load passes cover the tile");
  extern __shared__ __attribute__((aligned(16))) unsigned char smem[];
  bf16* As = reinterpret_cast<bf16*>(smem);               // [2][BM][LDS_LD]
  bf16* Ws = As + 2 * BM * LDS_LD;                        // [2][BN][LDS_LD]

  int bm, bn;
  tile_position(tile, tiles_m, gridDim.x / tiles_m, bm, bn);
  const int m0 = bm * BM, n0 = bn * BN;
  const int tid = threadIdx.x, lane = tid & 63, wid = tid >> 6;
  const int wm = (wid % (BM / WM)) * WM, wn = (wid / (BM / WM)) * WN;
  const int lrow = tid / (BK / 8), lk = (tid % (BK / 8)) * 8;
  const int fr = lane & 31, fk = (lane >> 5) * 8;

  floatx16 acc[TM][TN];
#pragma unroll
  for (int i = 0; i < TM; ++i)
#pragma unroll
    for (int j = 0; j < TN; ++j)
#pragma unroll
      for (int r = 0; r < 16; ++r) acc[i][j][r] = 0.f;

  bf16x8 ra[PA], rw[PW];
  int arow[PA], wrow[PW];                       // rows past the matrix read its last row
#pragma unroll
  for (int p = 0; p < PA; ++p) arow[p] = min(m0 + p * RP + lrow, M - 1);
#pragma unroll
  for (int p = 0; p < PW; ++p) wrow[p] = min(n0 + p * RP + lrow, N - 1);
  const int nkt = (K + BK - 1) / BK;
  const int nkt_inside = VEC ? K / BK : 0;      // k tiles that need no guard (the loop's fast form:
                                                // a guard's select would wait for the load at once)
  auto load_tile = [&](int kt) {
    const int k = kt * BK + lk;
    if (kt < nkt_inside) {
#pragma unroll
      for (int p = 0; p < PA; ++p) ra[p] = load8_inside(A, lda, arow[p], k);
#pragma unroll
      for (int p = 0; p < PW; ++p) rw[p] = load8_inside(W, ldw, wrow[p], k);
    } else {
#pragma unroll
      for (int p = 0; p < PA; ++p) ra[p] = load8<VEC>(A, lda, arow[p], k, K);
#pragma unroll
      for (int p = 0; p < PW; ++p) rw[p] = load8<VEC>(W, ldw, wrow[p], k, K);
    }
  };
  load_tile(0);
#pragma unroll
  for (int p = 0; p < PA; ++p)
    *reinterpret_cast<bf16x8*>(&As[(p * RP + lrow) * LDS_LD + lk]) = ra[p];
#pragma unroll
  for (int p = 0; p < PW; ++p)
    *reinterpret_cast<bf16x8*>(&Ws[(p * RP + lrow) * LDS_LD + lk]) = rw[p];
  __syncthreads();

  for (int kt = 0; kt < nkt; ++kt) {
    const int cur = kt & 1;
    const bool more = kt + 1 < nkt;
    if (more) load_tile(kt + 1);
    const bf16* as = As + cur * BM * LDS_LD;
    const bf16* ws = Ws + cur * BN * LDS_LD;
    // The fragments of k-step ks + 1 are asked for before the products of k-step ks are issued,
    // into the other half of fa / fw, so the matrix cores do not wait for LDS inside a tile.
    bf16x8 fa[2][TM], fw[2][TN];
    auto read_frags = [&](int ks, int h) {
#pragma unroll
      for (int i = 0; i < TM; ++i)
        fa[h][i] = *reinterpret_cast<const bf16x8*>(&as[(wm + i * 32 + fr) * LDS_LD + ks * 16 + fk]);
#pragma unroll
      for (int j = 0; j < TN; ++j)
        fw[h][j] = *reinterpret_cast<const bf16x8*>(&ws[(wn + j * 32 + fr) * LDS_LD + ks * 16 + fk]);
    };
    read_frags(0, 0);
#pragma unroll
    for (int ks = 0; ks < BK / 16; ++ks) {
      if (ks + 1 < BK / 16) read_frags(ks + 1, (ks + 1) & 1);
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int i = 0; i < TM; ++i)
#pragma unroll
        for (int j = 0; j < TN; ++j)
          acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(fa[ks & 1][i], fw[ks & 1][j], acc[i][j], 0, 0, 0);
      __builtin_amdgcn_sched_barrier(0);
    }
    if (more) {
      bf16* an = As + (cur ^ 1) * BM * LDS_LD;
      bf16* wn_ = Ws + (cur ^ 1) * BN * LDS_LD;
#pragma unroll
      for (int p = 0; p < PA; ++p)
        *reinterpret_cast<bf16x8*>(&an[(p * RP + lrow) * LDS_LD + lk]) = ra[p];
#pragma unroll
      for (int p = 0; p < PW; ++p)
        *reinterpret_cast<bf16x8*>(&wn_[(p * RP + lrow) * LDS_LD + lk]) = rw[p];
    }
    __syncthreads();
  }

  tile_epilogue<TM, TN>(acc, bias, C, ldc, M, N, epi, m0, wm, n0, wn, lane);
}

// ------------------------------------------------------------------ tiled kernel, loads straight into LDS
// BM x BN tiles on 8 waves whose k tiles of 64 travel global -> LDS without passing registers
// (global_load_lds_dwordx4: lane i's 16 bytes land at the wave's LDS base + 16 i).  A row of a k tile is one
// 128-byte line, fetched by 8 adjacent lanes: what a CU can have in flight towards L2 is counted in requests, so every
// request should be a whole line.  There is no room for padding in such a copy, so a row's eight 16-byte chunks are
// stored permuted: chunk c of row r sits at position c ^ ((r >> 1) & 7), which spreads the rows that one pass of a
// 16-byte fragment read covers over all banks.  Which chunk a lane fetches is free (its global address), so the
// permutation costs nothing on the way in.
//
// What bounds a large product here is the chip's power: with the same schedule, zeros run at 2.0 PFLOP/s and random
// values at 1.5 (8192^3), so what counts is energy a product and matrix cores that never wait.
//  * 16x16x32 MFMA.  The 32x32x16 form at the same tiles and schedule: 486 us for 413 at 2,048 rows against 37,888 of
//    3,584, 775 for 708 at 8192^3 (the same machine, random values).
//  * The two waves of a SIMD take turns: one reads its fragments while the other multiplies.  A wave's part of a k tile
//    is four products of a half of its rows with a half of its columns (A0 W0, A1 W0, A1 W1, A0 W1: one half changes at
//    a time); between two of them it reads the half that comes new (slot of the other wave's products), and a barrier
//    ends every slot.  Waves 4..7 run one slot behind waves 0..3.
//  * A half of a stage is set out again in the slot after its last read (STAGES tiles ahead), so that nearly all of LDS
//    is always on its way: at two stages of 256 x 256 a copy has seven of a k tile's eight slots to land.  The waits
//    count copies (vmcnt), they never drain them.
// At the widths of the 7B model (2,048 rows, random values): q|k|v (256 x 192) 77 us before, 61 now; o (256 x 128) 62 and
// 50; gate|up (256 x 256) 540 and 430; 8192^3 890 and 715.  (Before: 32x32x16 MFMA, a k tile's fragments read in two halves
// by all waves at once, one barrier and one wait a tile, 2-byte stores.)
//
// The order of the copies of a tile, W0 A0 A1 W1, is the order of the reads; LA, LW0 and LW1 copies a wave.  At the end
// of a product's read slot the half that the next slot but one reads must have landed for this wave (the barrier makes
// it everyone's): the number of younger copies allowed in flight stands at each wait.  Why a half may be overwritten:
// both groups have its last read back (lgkmcnt(0) in front of a barrier) at the latest one slot before the first
// group sets the new copy out.
// The compiler does not know that these loads write LDS and so does not wait for them.
// Needs 16-byte aligned rows and K a multiple of 64, and operands below 4 GB (32-bit byte offsets).
constexpr int DMA_BK = 64;

__device__ __forceinline__ void dma16(const bf16* base, unsigned off, unsigned lds_byte) {
  asm volatile("s_mov_b32 m0, %2\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %0, %1" ::"v"(off), "s"(base), "s"(lds_byte)
               : "m0");
}
// The lanes of a mask, of weights that no other workgroup reads (ONCE, see `load_weights`: a copy takes whole lines from the matrix too; SwiGLU of
// 37,888 x 3,584 from the matrix, 64 rows, 54.0 / 48.5 us) or of anything else
template <bool ONCE>
__device__ __forceinline__ void dma16_lanes(const bf16* base, unsigned off, unsigned lds_byte, unsigned long long lanes) {
  if constexpr (ONCE)
    asm volatile("s_mov_b32 m0, %2\n\ts_mov_b64 exec, %3\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %0, %1 nt\n\ts_mov_b64 exec, -1" ::"v"(off), "s"(base),
                 "s"(lds_byte), "s"(lanes)
                 : "m0");
  else
    asm volatile("s_mov_b32 m0, %2\n\ts_mov_b64 exec, %3\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %0, %1\n\ts_mov_b64 exec, -1" ::"v"(off), "s"(base),
                 "s"(lds_byte), "s"(lanes)
                 : "m0");
}
// at most N of this wave's youngest copies are in flight, and all its LDS reads are back
template <int N>
__device__ __forceinline__ void dma_wait() {
  static_assert(N >= 0 && N < 64, "vmcnt has six bits");
  asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)" ::"n"(N) : "memory");
}
__device__ __forceinline__ void dma_meet() {
  __builtin_amdgcn_sched_barrier(0);
  __builtin_amdgcn_s_barrier();
  __builtin_amdgcn_sched_barrier(0);
}

// Where chunk c (eight k) of weight row n begins in a k tile of 64, in bytes: in the matrix, or in its tiled copy (`w_operand`), where a
// k tile is two tiles of 32 k, a kilobyte apart, and the next one stands 2 KB on.
__device__ __forceinline__ unsigned w_copy_at(int n, int ldw, int c, bool tiled) {
  return tiled ? (unsigned)(n >> 4) * (unsigned)(ldw >> 5) * 1024u + (c >> 2) * 1024u + (n & 15) * 64u + (c & 3) * 16u
               : ((unsigned)n * (unsigned)ldw + c * 8) * 2u;
}

// How the 8 waves of a block share a BM x BN tile, in blocks of 16 x 16 results.
template <int BM, int BN>
struct DmaTile {
  static constexpr int WAVES_M = BM == 256 && BN != 256 ? 4 : 2, WAVES_N = 8 / WAVES_M;
  static constexpr int ROWS = BM / WAVES_M, COLS = BN / WAVES_N;      // of a wave
  static constexpr int I = ROWS / 16, IH = I / 2;                     // row blocks of a wave, of a half of A
  static constexpr int J = COLS / 16, J0 = BN == 192 ? 4 : J / 2, J1 = J - J0;      // column blocks, of the halves of W
  // a wave's column block j is the tile's block first(n) + j * STEP: neighbours, except where a wave's columns would not
  // hold whole pairs of a gate block and its up block (two blocks further)
  static constexpr bool PAIRED = J % 4 != 0;
  static constexpr int STEP = PAIRED ? 2 : 1;
  static __device__ __forceinline__ int first(int n) {
    return PAIRED ? n : n * J;
  }
  // copies per wave: a half of A; the halves of W
  static constexpr int LA = BM / 128, LW0 = J0 * WAVES_N / 4, LW1 = J1 * WAVES_N / 4;
  static constexpr int T = LW0 + 2 * LA + LW1;
  static constexpr int STAGE = (BM + BN) * DMA_BK * 2;
  static constexpr int OWN = 16 * 1024;       // LDS bytes of a wave in the epilogue
  template <int STAGES> static constexpr int lds() { return STAGES * STAGE > 8 * OWN ? STAGES * STAGE : 8 * OWN; }
  static_assert(ROWS % 32 == 0 && BM % 128 == 0 && (J0 * WAVES_N) % 4 == 0 && (J1 * WAVES_N) % 4 == 0, "whole copies per wave");
  static_assert(32 * (COLS + 4) * 4 <= OWN && 32 * (COLS + 8) * 2 <= OWN, "the epilogue's rows fit");
};

// A wave's results, acc[i][j]: the lane's row is 16 i + lane % 16, its columns 16 j + 4 (lane / 16) + e.  They go through the
// wave's own LDS in runs of 32 rows and leave in rows of 16 bytes a lane: straight from the registers every store would be
// pieces of lines, 2 bytes a lane (506 us for 469 at 2,048 x 37,888 x 3,584).
// Gate and up rows as they stand, all gates and then all ups (`Halves`; a plain product has none): what a tile takes as its
// interleaved weight row n, and the activation in the epilogue, y = act(gate, up), times sigmoid(z) of the row where there is one.
struct Halves {
  int width;               // gate rows, and up rows behind them; outputs
  int silu;                // y = silu(gate) up, else the clamped form
  float limit;
  const float* z;          // [M] ldz apart, or null
  int ldz;
  __device__ __forceinline__ int row(int n) const { return min((n >> 6) * 32 + (n & 31), width - 1) + ((n >> 5) & 1) * width; }
  __device__ __forceinline__ float act(float g, float u) const {
    return silu ? g * (1.0f / (1.0f + expf(-g))) * u : clamped_gate(g, u, limit);
  }
};

template <typename TT, bool HALVES = false>
__device__ __forceinline__ void dma_epilogue(floatx4 (&acc)[TT::I][TT::J], unsigned char* __restrict__ own,
                                             const float* __restrict__ bias, void* __restrict__ C, int ldc, int M, int N, int epi,
                                             int mw, int n0, int wn, int lane, const Halves& halves = Halves{}) {
  constexpr int J = TT::J, STEP = TT::STEP, COLS = TT::COLS;
  const int row = lane & 15, sub = (lane >> 4) * 4;
  const int b0 = TT::first(wn);
  auto column = [&](int c) { return n0 + (b0 + (c >> 4) * STEP) * 16 + (c & 15); };      // of the wave's column c
  if (epi == EPI_F32 || epi == EPI_ACC_F32) {
    constexpr int LD = COLS + 4, CH = COLS / 4;              // floats a staged row takes; chunks of four in it
    float* st = reinterpret_cast<float*>(own);
    const bool vec = ldc % 4 == 0 && (uintptr_t)C % 16 == 0;
#pragma unroll
    for (int h = 0; h < TT::I / 2; ++h) {
#pragma unroll
      for (int i = 0; i < 2; ++i)
#pragma unroll
        for (int j = 0; j < J; ++j) {
          const floatx4 v = acc[h * 2 + i][j];
          *reinterpret_cast<float4*>(st + (i * 16 + row) * LD + j * 16 + sub) = float4{v[0], v[1], v[2], v[3]};
        }
#pragma unroll 4
      for (int x = lane; x < 32 * CH; x += 64) {
        const int r = x / CH, c = (x % CH) * 4, m = mw + h * 32 + r, n = column(c);
        float4 v = *reinterpret_cast<const float4*>(st + r * LD + c);
        if (m >= M || n >= N) continue;
        float* o = (float*)C + (size_t)m * ldc + n;
        if (vec && n + 4 <= N) {
          if (bias) v = float4{v.x + bias[n], v.y + bias[n + 1], v.z + bias[n + 2], v.w + bias[n + 3]};
          if (epi == EPI_ACC_F32) { const float4 p = *reinterpret_cast<const float4*>(o); v = float4{p.x + v.x, p.y + v.y, p.z + v.z, p.w + v.w}; }
          *reinterpret_cast<float4*>(o) = v;
        } else {
          const float e4[4] = {v.x, v.y, v.z, v.w};
#pragma unroll
          for (int e = 0; e < 4; ++e)
            if (n + e < N) {
              const float s = e4[e] + (bias ? bias[n + e] : 0.f);
              o[e] = epi == EPI_ACC_F32 ? o[e] + s : s;
            }
        }
      }
    }
    return;
  }
  constexpr int LD = COLS + 8;                               // bfloat16 values a staged row takes
  bf16* st = reinterpret_cast<bf16*>(own);
  const bool vec = ldc % 8 == 0 && (uintptr_t)C % 16 == 0;
  // 32 staged rows of WIDTH values leave in chunks of eight: chunk c of a row to column `at(c)`, below `end`
  auto leave = [&](auto WIDTH, int h, int end, auto at) {
    constexpr int CH = decltype(WIDTH)::value / 8;
#pragma unroll 4
    for (int x = lane; x < 32 * CH; x += 64) {
      const int r = x / CH, c = (x % CH) * 8, m = mw + h * 32 + r, n = at(c);
      const bf16x8 v = *reinterpret_cast<const bf16x8*>(st + r * LD + c);
      if (m >= M) continue;
      bf16* o = (bf16*)C + (size_t)m * ldc + n;
      if (vec && n + 8 <= end) {
        *reinterpret_cast<bf16x8*>(o) = v;
      } else {
#pragma unroll
        for (int e = 0; e < 8; ++e)
          if (n + e < end) o[e] = v[e];
      }
    }
  };
  if (epi == EPI_SWIGLU) {
    // the tile's blocks of 16 columns: two of gates, the two of their ups, ...; block b's outputs are 16 ((b / 4) 2 + b % 2) on.
    // A wave holds gate block and up block as j and j + 2 (neighbours) or j and j + 1 (every second block).
    auto gated = [&](auto act) {
#pragma unroll
      for (int h = 0; h < TT::I / 2; ++h) {
#pragma unroll
        for (int i = 0; i < 2; ++i) {
          float s = 1.f;
          if constexpr (HALVES) {
            const int m = mw + h * 32 + i * 16 + row;
            if (halves.z && m < M) s = 1.0f / (1.0f + expf(-halves.z[(size_t)m * halves.ldz]));
          }
#pragma unroll
          for (int p = 0; p < J / 2; ++p) {
            const int jg = TT::PAIRED ? 2 * p : (p >> 1) * 4 + (p & 1), ju = jg + 2 / STEP;
            bf16x4 v;
#pragma unroll
            for (int e = 0; e < 4; ++e) v[e] = (bf16)(HALVES ? act(acc[h * 2 + i][jg][e], acc[h * 2 + i][ju][e]) * s
                                                             : act(acc[h * 2 + i][jg][e], acc[h * 2 + i][ju][e]));
            *reinterpret_cast<bf16x4*>(st + (i * 16 + row) * LD + p * 16 + sub) = v;
          }
        }
        leave(std::integral_constant<int, COLS / 2>{}, h, ldc, [&](int c) {
          const int p = c >> 4, b = b0 + (TT::PAIRED ? 2 * p * STEP : (p >> 1) * 4 + (p & 1));
          return (n0 >> 1) + ((b >> 2) * 2 + (b & 1)) * 16 + (c & 15);
        });
      }
    };
    if constexpr (HALVES) {
      gated([&](float g, float u) { return halves.act(g, u); });
    } else if (bias) {
      const float limit = *bias;
      gated([=](float g, float u) { return clamped_gate(g, u, limit); });
    } else {
      gated([](float g, float u) { return swiglu_f(g, u, nullptr); });
    }
    return;
  }
  const float ap = epi == EPI_XIELU ? bias[N] : 0.f, an = epi == EPI_XIELU ? bias[N + 1] : 0.f;
#pragma unroll
  for (int h = 0; h < TT::I / 2; ++h) {
#pragma unroll
    for (int j = 0; j < J; ++j) {
      float b[4];
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const int n = column(j * 16 + sub + e);
        b[e] = bias && n < N ? bias[n] : 0.f;
      }
#pragma unroll
      for (int i = 0; i < 2; ++i) {
        bf16x4 v;
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          const float z = acc[h * 2 + i][j][e] + b[e];
          v[e] = (bf16)(epi == EPI_XIELU ? xielu_f(z, ap, an) : epi == EPI_RELU2 ? relu2_f(z) : z);
        }
        *reinterpret_cast<bf16x4*>(st + (i * 16 + row) * LD + j * 16 + sub) = v;
      }
    }
    leave(std::integral_constant<int, COLS>{}, h, N, column);
  }
}

template <int BM, int BN, int STAGES, bool GROUPED = false, bool HALVES = false, bool TILED = false>
__global__ __launch_bounds__(512, 2) void tile_dma_kernel(const bf16* __restrict__ A, int lda,
                                                       const bf16* __restrict__ W, int ldw,
                                                       const float* __restrict__ bias, void* __restrict__ C,
                                                       int ldc, int M, int N, int K, int epi, int tiles_m,
                                                       int order, int k_per_split,
                                                       const RowGroup* __restrict__ groups = nullptr, Halves halves = Halves{}) {
  using TT = DmaTile<BM, BN>;
  constexpr int ROW = DMA_BK * 2, A_ST = BM * ROW, W_ST = BN * ROW, W_AT = STAGES * A_ST;
  constexpr int I = TT::I, IH = TT::IH, J = TT::J, J0 = TT::J0, J1 = TT::J1, LA = TT::LA, LW0 = TT::LW0, LW1 = TT::LW1, T = TT::T;
  int tile, part;
  block_work(order, tile, part);
  if (k_per_split > 0) {
    // K cut into parts (k_per_split a multiple of 64): this block multiplies its part of K
    // and stores 32-bit sums into its own [M][N] slab of C; another kernel adds the slabs
    const int kb = part * k_per_split;
    A += kb;
    W += TILED ? kb * 16 : kb;
    K = min(k_per_split, K - kb);
    C = (float*)C + (size_t)part * M * N;
  }
  extern __shared__ __attribute__((aligned(16))) unsigned char smem[];      // [stage][BM][64] of A, [stage][BN][64] of W
  int bm, bn;
  tile_position(tile, tiles_m, gridDim.x / tiles_m, bm, bn);
  if (GROUPED) {
    const int first = __builtin_amdgcn_readfirstlane(groups[bm].first), matrix = __builtin_amdgcn_readfirstlane(groups[bm].matrix);
    M = __builtin_amdgcn_readfirstlane(groups[bm].rows);
    A += (size_t)first * lda;
    W += (size_t)matrix * (HALVES ? 2 * halves.width : N) * ldw;
    C = HALVES ? (void*)((bf16*)C + (size_t)first * ldc) : (void*)((float*)C + (size_t)first * ldc);
    bm = 0;
  }
  const int m0 = bm * BM, n0 = bn * BN;
  const int lane = threadIdx.x & 63;
  const int wid = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int grp = wid >> 2;                                  // waves w and w + 4 share a SIMD
  const int wave_m = TT::WAVES_M == 2 ? grp : wid & 3, wave_n = TT::WAVES_M == 2 ? wid & 3 : grp;
  const int fr = lane & 15, fk = lane >> 4;

  floatx4 acc[I][J];
#pragma unroll
  for (int i = 0; i < I; ++i)
#pragma unroll
    for (int j = 0; j < J; ++j) acc[i][j] = floatx4{0.f, 0.f, 0.f, 0.f};

  constexpr int wk = TILED ? 16 * DMA_BK : DMA_BK;           // weights from a k tile to the next
  // What a wave copies: pieces of 8 rows (1 KB), the lane row lane / 8 of a piece and the chunk that belongs at position
  // lane % 8.  Half h of A: the rows of the row blocks h IH .. + IH - 1 of every row of waves; half h of W: the rows of
  // the column blocks of that half of every column of waves.
  const unsigned lds0 = (unsigned)(uintptr_t)smem;
  unsigned ga[2][LA], gw[LW0 + LW1], la[2][LA], lw[LW0 + LW1];
#pragma unroll
  for (int h = 0; h < 2; ++h)
#pragma unroll
    for (int q = 0; q < LA; ++q) {
      const int p = q * 8 + wid;                             // piece of the half: 2 IH pieces a row of waves
      const int r0 = (p / (2 * IH)) * TT::ROWS + h * IH * 16 + (p % (2 * IH)) * 8, r = r0 + (lane >> 3);
      ga[h][q] = ((unsigned)min(m0 + r, M - 1) * (unsigned)lda + ((lane & 7) ^ ((r >> 1) & 7)) * 8) * 2u;
      la[h][q] = lds0 + r0 * ROW;
    }
#pragma unroll
  for (int q = 0; q < LW0 + LW1; ++q) {
    const int jh = q < LW0 ? J0 : J1, p = (q < LW0 ? q : q - LW0) * 8 + wid;       // 2 jh pieces a column of waves
    const int b = TT::first(p / (2 * jh)) + ((q < LW0 ? 0 : J0) + (p % (2 * jh)) / 2) * TT::STEP;
    const int r0 = b * 16 + (p & 1) * 8, r = r0 + (lane >> 3);
    gw[q] = w_copy_at(HALVES ? halves.row(n0 + r) : min(n0 + r, N - 1), ldw, (lane & 7) ^ ((r >> 1) & 7), TILED);
    lw[q] = lds0 + W_AT + r0 * ROW;
  }
  auto copy_a = [&](int kt, int st, auto HALF) {
    constexpr int h = decltype(HALF)::value;
#pragma unroll
    for (int q = 0; q < LA; ++q) dma16(A + kt * DMA_BK, ga[h][q], __builtin_amdgcn_readfirstlane(la[h][q] + st * A_ST));
  };
  auto copy_w = [&](int kt, int st, auto HALF) {
    constexpr int h = decltype(HALF)::value;
#pragma unroll
    for (int q = h ? LW0 : 0; q < (h ? LW0 + LW1 : LW0); ++q)
      dma16(W + kt * wk, gw[q], __builtin_amdgcn_readfirstlane(lw[q] + st * W_ST));
  };
  // fragment reads (16x16x32): row R, chunk 4 ks + fk of its 8, at position chunk ^ ((R >> 1) & 7)
  const int sw = (fr >> 1) & 7;
  unsigned pa[2], pw[2];
#pragma unroll
  for (int ks = 0; ks < 2; ++ks) {
    const unsigned pos = ((4 * ks + fk) ^ sw) * 16;
    pa[ks] = (wave_m * TT::ROWS + fr) * ROW + pos;
    pw[ks] = W_AT + (TT::first(wave_n) * 16 + fr) * ROW + pos;
  }
  bf16x8 fa[2][IH][2], fw0[J0][2], fw1[J1][2];               // [half][block][k-step], [block][k-step]
  auto read_a = [&](int st, auto HALF) {
    constexpr int h = decltype(HALF)::value;
#pragma unroll
    for (int ks = 0; ks < 2; ++ks)
#pragma unroll
      for (int i = 0; i < IH; ++i) fa[h][i][ks] = *reinterpret_cast<const bf16x8*>(smem + pa[ks] + st * A_ST + (h * IH + i) * 16 * ROW);
  };
  auto read_w0 = [&](int st) {
#pragma unroll
    for (int ks = 0; ks < 2; ++ks)
#pragma unroll
      for (int j = 0; j < J0; ++j) fw0[j][ks] = *reinterpret_cast<const bf16x8*>(smem + pw[ks] + st * W_ST + j * TT::STEP * 16 * ROW);
  };
  auto read_w1 = [&](int st) {
#pragma unroll
    for (int ks = 0; ks < 2; ++ks)
#pragma unroll
      for (int j = 0; j < J1; ++j) fw1[j][ks] = *reinterpret_cast<const bf16x8*>(smem + pw[ks] + st * W_ST + (J0 + j) * TT::STEP * 16 * ROW);
  };
  auto multiply = [&](auto HA, auto HW) {
    constexpr int ha = decltype(HA)::value, hw = decltype(HW)::value;
    __builtin_amdgcn_s_setprio(1);
#pragma unroll
    for (int ks = 0; ks < 2; ++ks)
#pragma unroll
      for (int i = 0; i < IH; ++i)
#pragma unroll
        for (int j = 0; j < (hw ? J1 : J0); ++j) {
          floatx4& d = acc[ha * IH + i][(hw ? J0 : 0) + j];
          d = __builtin_amdgcn_mfma_f32_16x16x32_bf16(hw ? fw1[j < J1 ? j : 0][ks] : fw0[j < J0 ? j : 0][ks], fa[ha][i][ks], d, 0, 0, 0);
        }
    __builtin_amdgcn_s_setprio(0);
  };
  using H0 = std::integral_constant<int, 0>;
  using H1 = std::integral_constant<int, 1>;
  const int nkt = K / DMA_BK;
#pragma unroll
  for (int t = 0; t < STAGES; ++t) {                         // (past the last tile: that one again, never read)
    const int kt = min(t, nkt - 1);
    copy_w(kt, t, H0{});
    copy_a(kt, t, H0{});
    copy_a(kt, t, H1{});
    copy_w(kt, t, H1{});
  }
  dma_wait<STAGES * T - LW0 - LA>();                         // W0 and A0 of tile 0 are here
  dma_meet();
  read_w0(0);
  dma_wait<STAGES * T - LW0 - LA>();
  dma_meet();
  if (grp == 1) dma_meet();                                  // the second group runs a slot behind the first
  auto tile_pass = [&](int kt, int st, int st_next) {
    const int ahead = min(kt + STAGES, nkt - 1);
    read_a(st, H0{});
    __builtin_amdgcn_sched_barrier(0);
    copy_w(ahead, st, H0{});
    dma_wait<STAGES * T - 2 * LA>();                         // A1
    dma_meet();
    multiply(H0{}, H0{});
    dma_meet();
    read_a(st, H1{});
    __builtin_amdgcn_sched_barrier(0);
    copy_a(ahead, st, H0{});
    dma_wait<(STAGES - 1) * T + LW0 + LA>();                 // W1
    dma_meet();
    multiply(H1{}, H0{});
    dma_meet();
    read_w1(st);
    __builtin_amdgcn_sched_barrier(0);
    copy_a(ahead, st, H1{});
    dma_wait<(STAGES - 1) * T + 2 * LA>();                   // the next tile's W0
    dma_meet();
    multiply(H1{}, H1{});
    dma_meet();
    read_w0(st_next);
    __builtin_amdgcn_sched_barrier(0);
    copy_w(ahead, st, H1{});
    dma_wait<STAGES * T - LW0 - LA>();                       // the next tile's A0
    dma_meet();
    multiply(H0{}, H1{});
    dma_meet();
  };
  if constexpr (STAGES == 2) {
    int kt = 0;
    for (; kt + 1 < nkt; kt += 2) {
      tile_pass(kt, 0, 1);
      tile_pass(kt + 1, 1, 0);
    }
    if (kt < nkt) tile_pass(kt, 0, 1);
  } else {
    int st = 0;
    for (int kt = 0; kt < nkt; ++kt) {
      const int next = st + 1 == STAGES ? 0 : st + 1;
      tile_pass(kt, st, next);
      st = next;
    }
  }
  if (grp == 0) dma_meet();
  dma_wait<0>();
  dma_meet();
  dma_epilogue<TT, HALVES>(acc, smem + wid * TT::OWN, bias, C, ldc, M, N, HALVES ? EPI_SWIGLU : epi, m0 + wave_m * TT::ROWS, n0, wave_n, lane, halves);
}

// The sum of a row's `parts` numbers by LANES lanes that stand side by side (l: the lane's place among them), in two steps so that a
// kernel asks early and adds late: every lane asks for Q x 4 of them at once, one value a load (with 16-byte loads beside them where
// the rows allow it the compiler waited for each row's first before the next: a trip to memory for every row of a lane, in front of the
// product's first copies; gate|up of 37 rows with 84 parts a row 11.2 us so, 9.8 now), and for what is left of a longer row when it
// adds up.  ALL: no load stands behind a condition (a place past the row's end asks for the last one again), for a kernel whose own
// loads the compiler counts: behind one it counts with the way that has fewer in flight.  Elsewhere places past the end ask for nothing.
// A row without parts (p null, for all lanes alike) asks for nothing and gives 0.
template <int LANES, int Q, bool ALL = false>
struct LanesSum {
  float x[Q][4];
  __device__ __forceinline__ void ask(const float* __restrict__ p, int parts, int l) {
    if constexpr (!ALL) {
#pragma unroll
      for (int q = 0; q < Q; ++q)
#pragma unroll
        for (int e = 0; e < 4; ++e) x[q][e] = 0.f;
      if (!p) return;
    }
#pragma unroll
    for (int q = 0; q < Q; ++q)
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const int i = (q * 4 + e) * LANES + l;
        if constexpr (ALL) x[q][e] = p ? p[min(i, parts - 1)] : 0.f;
        else if (i < parts) x[q][e] = p[i];
      }
  }
  __device__ __forceinline__ float add(const float* __restrict__ p, int parts, int l) const {
    float t = 0.f;
    if (p) {
      auto of = [&](int q, int e) { return (q * 4 + e) * LANES + l < parts ? x[q][e] : 0.f; };
#pragma unroll
      for (int q = 0; q < Q; ++q) t += (of(q, 0) + of(q, 1)) + (of(q, 2) + of(q, 3));
      for (int i = Q * LANES * 4 + l; i < parts; i += LANES) t += p[i];
    }
#pragma unroll
    for (int o = LANES / 2; o > 0; o >>= 1) t += __shfl_xor(t, o, MF_WAVE);
    return t;
  }
};

// ---- the smaller tiles: one barrier a k tile
// 128 x 128 on 8 waves and 64 x 64 on 4, for products whose larger tiles would leave most of the chip idle: a block's time
// is then its own chain of k tiles, whatever the others do, and a k tile's chain is what is kept short: wait for the copies
// of the next k tile, meet, set out the copies STAGES - 1 tiles on, read the next tile's fragments, multiply this one's.  (The quarter products of
// `tile_dma_kernel` meet eight times a k tile, which 128 x 128 cannot fill: 203 rows against 9,728 of 896 15.5 us so, 12.6
// here; 2,048 x 2,048 x 2,048 27.2 and 23.3.  At 256 x 128 the two are level.)  64 x 64: 203 rows against 1,152 of 896 (the
// narrowest model's q|k|v) 11.6 us as 128 x 128, 6.4 so.
template <int BM, int BN, int WAVES_M_, int WAVES_N_>
struct StepTile {
  static constexpr int WAVES_M = WAVES_M_, WAVES_N = WAVES_N_, WAVES = WAVES_M * WAVES_N;
  static constexpr int ROWS = BM / WAVES_M, COLS = BN / WAVES_N, I = ROWS / 16, J = COLS / 16;
  // a wave's two column blocks are a gate block and its up block (see DmaTile)
  static constexpr bool PAIRED = true;
  static constexpr int STEP = 2;
  static __device__ __forceinline__ int first(int n) { return (n >> 1) * 4 + (n & 1); }
  static constexpr int LA = BM / 8 / WAVES, LW = BN / 8 / WAVES;       // copies per wave
  static constexpr int OWN = 32 * (COLS + 4) * 4;
  template <int STAGES> static constexpr int lds() {
    return STAGES * (BM + BN) * DMA_BK * 2 > WAVES * OWN ? STAGES * (BM + BN) * DMA_BK * 2 : WAVES * OWN;
  }
  static_assert(J == 2 && I % 2 == 0 && BM % (8 * WAVES) == 0 && BN % (8 * WAVES) == 0, "pairs of blocks, whole copies per wave");
};

// SCALED: the rows' sums are multiplied by 1 / sqrt(mean + eps) of the row, `in_parts` partial sums of squares of which stand
// in in_ssq [M][in_parts] (FusedNorm::in_*; one launch, K whole).
template <int BM, int BN, int WAVES_M, int WAVES_N, int STAGES, bool GROUPED = false, bool SCALED = false, bool HALVES = false,
          bool TILED = false>
__global__ __launch_bounds__(64 * WAVES_M * WAVES_N) void tile_step_kernel(const bf16* __restrict__ A, int lda,
                                                       const bf16* __restrict__ W, int ldw,
                                                       const float* __restrict__ bias, void* __restrict__ C,
                                                       int ldc, int M, int N, int K, int epi, int tiles_m,
                                                       int order, int k_per_split,
                                                       const RowGroup* __restrict__ groups = nullptr,
                                                       const float* __restrict__ in_ssq = nullptr, int in_parts = 0,
                                                       float in_eps = 0.f, Halves halves = Halves{}) {
  using TT = StepTile<BM, BN, WAVES_M, WAVES_N>;
  constexpr int ROW = DMA_BK * 2, ST = (BM + BN) * ROW, WAVES = TT::WAVES, I = TT::I, J = TT::J, LA = TT::LA, LW = TT::LW;
  int tile, part;
  block_work(order, tile, part);
  if (k_per_split > 0) {                                     // as in tile_dma_kernel
    const int kb = part * k_per_split;
    A += kb;
    W += TILED ? kb * 16 : kb;
    K = min(k_per_split, K - kb);
    C = (float*)C + (size_t)part * M * N;
  }
  extern __shared__ __attribute__((aligned(16))) unsigned char smem[];      // [stage][BM rows of A, BN rows of W][64]
  int bm, bn;
  tile_position(tile, tiles_m, gridDim.x / tiles_m, bm, bn);
  if (GROUPED) {
    const int first = __builtin_amdgcn_readfirstlane(groups[bm].first), matrix = __builtin_amdgcn_readfirstlane(groups[bm].matrix);
    M = __builtin_amdgcn_readfirstlane(groups[bm].rows);
    A += (size_t)first * lda;
    W += (size_t)matrix * (HALVES ? 2 * halves.width : N) * ldw;
    C = HALVES ? (void*)((bf16*)C + (size_t)first * ldc) : (void*)((float*)C + (size_t)first * ldc);
    bm = 0;
  }
  const int m0 = bm * BM, n0 = bn * BN;
  const int lane = threadIdx.x & 63;
  const int wid = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int wave_m = wid % WAVES_M, wave_n = wid / WAVES_M;
  const int fr = lane & 15, fk = lane >> 4;
  floatx4 acc[I][J];
#pragma unroll
  for (int i = 0; i < I; ++i)
#pragma unroll
    for (int j = 0; j < J; ++j) acc[i][j] = floatx4{0.f, 0.f, 0.f, 0.f};
  const unsigned lds0 = (unsigned)(uintptr_t)smem;
  unsigned ga[LA], gw[LW];                                   // a wave copies pieces wid, WAVES + wid, ... of 8 rows
#pragma unroll
  for (int q = 0; q < LA; ++q) {
    const int r = (q * WAVES + wid) * 8 + (lane >> 3);
    ga[q] = ((unsigned)min(m0 + r, M - 1) * (unsigned)lda + ((lane & 7) ^ ((r >> 1) & 7)) * 8) * 2u;
  }
#pragma unroll
  for (int q = 0; q < LW; ++q) {
    const int r = (q * WAVES + wid) * 8 + (lane >> 3);
    gw[q] = w_copy_at(HALVES ? halves.row(n0 + r) : min(n0 + r, N - 1), ldw, (lane & 7) ^ ((r >> 1) & 7), TILED);
  }
  const int nkt = K / DMA_BK;
  auto copy = [&](int kt, int st) {                          // (past the last tile: that one again, never read)
    const int k = min(kt, nkt - 1) * DMA_BK, kw = TILED ? k * 16 : k;
    const unsigned base = lds0 + st * ST + wid * 1024;
#pragma unroll
    for (int q = 0; q < LW; ++q) dma16(W + kw, gw[q], __builtin_amdgcn_readfirstlane(base + BM * ROW + q * (WAVES * 1024)));
#pragma unroll
    for (int q = 0; q < LA; ++q) dma16(A + k, ga[q], __builtin_amdgcn_readfirstlane(base + q * (WAVES * 1024)));
  };
  const int sw = (fr >> 1) & 7;
  // the rows' partial sums are asked for in front of the first copies and added up behind the products, eight lanes a row
  constexpr int GROUPS = (BM + WAVES * 8 - 1) / (WAVES * 8);
  LanesSum<8, 4> sums[SCALED ? GROUPS : 1];
  auto part_row = [&](int q) {
    const int r = m0 + (q * WAVES + wid) * 8 + (lane >> 3);  // (rows past M ask for nothing: 9,728 x 896 SwiGLU of 17 rows 8.65 us so and 9.1)
    return r < M ? in_ssq + (size_t)r * in_parts : nullptr;
  };
  if constexpr (SCALED) {
#pragma unroll
    for (int q = 0; q < GROUPS; ++q) sums[q].ask(part_row(q), in_parts, lane & 7);
    __builtin_amdgcn_sched_barrier(0);
  }
#pragma unroll
  for (int t = 0; t < STAGES - 1; ++t) copy(t, t);
  bf16x8 fa[2][2][I], fw[2][2][J];                           // [set][k-step][block]
  auto read = [&](int st, auto SET) {
    constexpr int set = decltype(SET)::value;
    const unsigned char* s = smem + st * ST;
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      const int pos = ((4 * h + fk) ^ sw) * 16;
#pragma unroll
      for (int i = 0; i < I; ++i) fa[set][h][i] = *reinterpret_cast<const bf16x8*>(s + (wave_m * TT::ROWS + i * 16 + fr) * ROW + pos);
#pragma unroll
      for (int j = 0; j < J; ++j)
        fw[set][h][j] = *reinterpret_cast<const bf16x8*>(s + (BM + (TT::first(wave_n) + j * TT::STEP) * 16 + fr) * ROW + pos);
    }
  };
  auto multiply = [&](auto SET) {
    constexpr int set = decltype(SET)::value;
#pragma unroll
    for (int h = 0; h < 2; ++h)
#pragma unroll
      for (int i = 0; i < I; ++i)
#pragma unroll
        for (int j = 0; j < J; ++j)
          acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(fw[set][h][j], fa[set][h][i], acc[i][j], 0, 0, 0);
  };
  using S0 = std::integral_constant<int, 0>;
  using S1 = std::integral_constant<int, 1>;
  constexpr int L = LA + LW;
  dma_wait<(STAGES - 2) * L>();
  dma_meet();
  read(0, S0{});
  int st = 0;                                                // of tile kt
  // one k tile: its fragments are in set NOW; those of the next one are read into the other set under its products
  auto pass = [&](int kt, auto NOW, auto OTHER) {
    // tile kt + 1 has landed for this wave, and behind the barrier for all; the stage of tile kt - 1, whose fragments every
    // wave's products have used by then, takes tile kt + STAGES - 1
    dma_wait<(STAGES - 3) * L>();
    dma_meet();
    copy(kt + STAGES - 1, st == 0 ? STAGES - 1 : st - 1);
    st = st == STAGES - 1 ? 0 : st + 1;
    read(st, OTHER);                                         // (behind the last tile: that one again, never used)
    multiply(NOW);
  };
  int kt = 0;
  for (; kt + 1 < nkt; kt += 2) {
    pass(kt, S0{}, S1{});
    pass(kt + 1, S1{}, S0{});
  }
  if (kt < nkt) multiply(S0{});
  dma_wait<0>();
  dma_meet();
  if constexpr (SCALED) {
    static_assert(WAVES * TT::OWN + BM * 4 <= TT::template lds<STAGES>(), "the factors stand behind the waves' own LDS");
    float* fac = reinterpret_cast<float*>(smem + WAVES * TT::OWN);
#pragma unroll
    for (int q = 0; q < GROUPS; ++q) {
      const float t = sums[q].add(part_row(q), in_parts, lane & 7);
      const int r = (q * WAVES + wid) * 8 + (lane >> 3);
      if ((lane & 7) == 0 && r < BM) fac[r] = 1.0f / sqrtf(t / (float)K + in_eps);
    }
    __syncthreads();
#pragma unroll
    for (int i = 0; i < I; ++i) {
      const float f = fac[wave_m * TT::ROWS + i * 16 + fr];
#pragma unroll
      for (int j = 0; j < J; ++j) acc[i][j] *= f;
    }
  }
  dma_epilogue<TT, HALVES>(acc, smem + wid * TT::OWN, bias, C, ldc, M, N, HALVES ? EPI_SWIGLU : epi, m0 + wave_m * TT::ROWS, n0, wave_n, lane, halves);
}

template <int BM, int BN, int WAVES_M, int WAVES_N, int STAGES, bool GROUPED, bool SCALED = false, bool HALVES = false, bool TILED = false>
int launch_tile_step(const bf16* A, int lda, const bf16* W, int ldw, const float* bias, void* C, int ldc, int M, int N, int K, int epi,
                     hipStream_t stream, int splits, int k_per_split, const RowGroup* groups, int n_groups,
                     const float* in_ssq = nullptr, int in_parts = 0, float in_eps = 0.f, const Halves& halves = Halves{}) {
  using TT = StepTile<BM, BN, WAVES_M, WAVES_N>;
  auto kern = tile_step_kernel<BM, BN, WAVES_M, WAVES_N, STAGES, GROUPED, SCALED, HALVES, TILED>;
  static bool configured = false;
  if (!configured) {
    const hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void*>(kern), hipFuncAttributeMaxDynamicSharedMemorySize,
                                             TT::template lds<STAGES>());
    if (e != hipSuccess) return (int)e;
    configured = true;
  }
  const int tiles_m = GROUPED ? n_groups : (M + BM - 1) / BM, tiles_n = (N + BN - 1) / BN;
  kern<<<dim3(tiles_m * tiles_n, splits), 64 * TT::WAVES, TT::template lds<STAGES>(), stream>>>(
      A, lda, W, ldw, bias, C, ldc, M, N, K, epi, tiles_m, tile_order(tiles_m * tiles_n, splits, M, N, K), k_per_split, groups, in_ssq, in_parts, in_eps, halves);
  return mf_launch_status();
}

// 64 x 64: five stages, so that two blocks fit a CU (ten for blocks that have a CU to themselves: level)
template <bool SCALED, bool TILED>
int launch_tile64(const bf16* A, int lda, const bf16* W, int ldw, const float* bias, void* C, int ldc, int M, int N, int K, int epi,
                  hipStream_t stream, int splits, int k_per_split, const float* in_ssq = nullptr, int in_parts = 0, float in_eps = 0.f) {
  return launch_tile_step<64, 64, 2, 2, 5, false, SCALED, false, TILED>(A, lda, W, ldw, bias, C, ldc, M, N, K, epi, stream, splits, k_per_split,
                                                                        nullptr, 0, in_ssq, in_parts, in_eps);
}

// ---- tiles that are all on the chip at once: weights straight into MFMA operands
// What bounds products of some hundred rows is neither the matrix cores nor LDS but a chain of waits in each block: a k tile of 64 is 28 KB of
// weights and activations for 96 x 128 and takes 0.46 us, 32 KB and 0.53 us for 128 x 128, with 30 blocks on the chip as with 256 and four k
// tiles ahead as with six, 60 GB/s a CU; plain loads bring a CU 75 to 95 GB/s from memory with 30 blocks on the chip (24 with 256: all
// of them share 6 TB/s) and 140 from an L2 (115 with 256).  A block's time goes with its tile, so the rows of a tile are what the product has, in
// 16s, and not 128 or 256; weights, whose tiled copy holds them as the MFMA operands they are, go to registers, four k tiles ahead, each wave its own 32
// columns; the activations of a k tile go through registers into one of two LDS buffers, and their fragments are read three
// ahead of the products.  A short way in and out (no LDS at all in the epilogue) makes few parts of a K split pay.  Products as the plan runs
// them, without / with this kernel, in microseconds, weights and activations from memory: with the norm behind them 203 x 3,584 x 3,584 23.8 in 7
// parts / 21.4 in 3, 150 x 4,096 x 4,096 24.1 in 8 / 20.4 in 4, 900 x 2,048 x 2,048 29.3 in 4 / 24.2 in 2, 150 x 2,048 x 11,008 27.8 in 15 /
// 23.4 in 8; with the rotation 150 x 4,608 x 3,584 25.8 in 7 / 22.3 in 3; alone 300 x 8,192 x 4,096 42.2 in 2 / 37.7 whole.  SwiGLU products
// were level at best (300 x 9,728 x 896 12.2 and 12.9) and have none.
// Tried: 256 columns, weights marked as read once where other rows' tiles read them (slower: 13.7 and 15.3), fragments seven ahead with four
// LDS buffers (level).
template <int I>
__global__ __launch_bounds__(256, 2) void tile_stream_kernel(const bf16* __restrict__ A, int lda, const bf16* __restrict__ Wt,
                                                                          const float* __restrict__ bias, void* __restrict__ C, int ldc, int M,
                                                                          int N, int K, int epi, int tiles_m, int tiles, int k_per_split) {
  constexpr int J = 2, AHEAD = 4, BM = 16 * I, BN = 64 * J, ROW = DMA_BK * 2, BUF = BM * ROW, LA = (I + 1) / 2, STEPS = 2 * I, D = 3, R = 4;
  static_assert(AHEAD * STEPS % R == 0 && LA < STEPS - D && I + J <= STEPS, "fragments keep their places, a k tile is written before the barrier");
  __shared__ __attribute__((aligned(16))) unsigned char smem[2 * BUF];      // [buffer][BM rows of A][64]
  int at = blockIdx.x;
  {
    const int n = gridDim.x, per = n / 8, rem = n % 8, x = at % 8;          // (neighbours on one die: a part's tiles of the same weights)
    at = x * per + min(x, rem) + at / 8;
  }
  const int part = at / tiles, tile = at - part * tiles;
  const int bm = tile % tiles_m, bn = tile / tiles_m;
  const int k_tiles = K >> 5;                                // tiles of 32 k of a block of weight rows
  if (k_per_split > 0) {                                     // as in tile_dma_kernel
    const int kb = part * k_per_split;
    A += kb;
    Wt += (size_t)(kb >> 5) * 512;
    K = min(k_per_split, K - kb);
    C = (float*)C + (size_t)part * M * N;
  }
  const int nkt = K / DMA_BK;
  const int m0 = bm * BM, n0 = bn * BN;
  const int tid = threadIdx.x, lane = tid & 63, wid = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int fr = lane & 15, fk = lane >> 4;
  floatx4 acc[I][J];
#pragma unroll
  for (int i = 0; i < I; ++i)
#pragma unroll
    for (int j = 0; j < J; ++j) acc[i][j] = floatx4{0.f, 0.f, 0.f, 0.f};
  unsigned wo[J], ao[LA], aw[LA];                            // bytes: weights, activations, and where the latter go in LDS
#pragma unroll
  for (int j = 0; j < J; ++j)
    wo[j] = (unsigned)min((n0 >> 4) + wid * J + j, (N - 1) >> 4) * (unsigned)k_tiles * 1024u + fr * 64 + fk * 16;
#pragma unroll
  for (int q = 0; q < LA; ++q) {
    const int r = min(q * 32 + (tid >> 3), BM - 1), c = tid & 7;
    ao[q] = ((unsigned)min(m0 + r, M - 1) * (unsigned)lda + c * 8) * 2u;
    aw[q] = r * ROW + (c ^ ((r >> 1) & 7)) * 16;
  }
  const bool last = I % 2 == 0 || tid < 128;                 // whether the last of a thread's chunks is a row's of the tile
  bf16x8 w[AHEAD][2][J], a[2][LA], f[R];
  // (the offsets stay 32 bits wide beside a scalar base only where the compiler cannot take them out of the loop as addresses)
  auto load = [](const void* base, size_t at, unsigned off) {
    asm volatile("" : "+v"(off));
    return *reinterpret_cast<const bf16x8*>((const char*)base + at + off);
  };
  auto load_w = [&](int kt, int u, int h, int j) { w[u][h][j] = load(Wt, (size_t)(unsigned)(min(kt, nkt - 1) * 2 + h) * 1024, wo[j]); };
  auto load_a = [&](int kt, int s, int q) { a[s][q] = load(A, (size_t)(unsigned)min(kt, nkt - 1) * ROW, ao[q]); };
  auto write_a = [&](int s, int q) {
    if (q + 1 < LA || last) *reinterpret_cast<bf16x8*>(smem + s * BUF + aw[q]) = a[s][q];
  };
  unsigned po[2];
#pragma unroll
  for (int h = 0; h < 2; ++h) po[h] = fr * ROW + ((4 * h + fk) ^ ((fr >> 1) & 7)) * 16;
  // step s of a k tile: row block s % I, half s / I of its k
  auto read = [&](int s, int st, int to) { f[to] = *reinterpret_cast<const bf16x8*>(smem + st * BUF + po[s / I] + (s % I) * 16 * ROW); };
  auto load_tile = [&](int u) {
#pragma unroll
    for (int h = 0; h < 2; ++h)
#pragma unroll
      for (int j = 0; j < J; ++j) load_w(u, u, h, j);
  };
#pragma unroll
  for (int q = 0; q < LA; ++q) load_a(0, 0, q);
  load_tile(0);
#pragma unroll
  for (int q = 0; q < LA; ++q) load_a(1, 1, q);
#pragma unroll
  for (int u = 1; u < AHEAD; ++u) load_tile(u);
  __builtin_amdgcn_sched_barrier(0);
#pragma unroll
  for (int q = 0; q < LA; ++q) write_a(0, q);
#pragma unroll
  for (int q = 0; q < LA; ++q) load_a(2, 0, q);
  auto meet = [&]() {                                        // this wave's reads and writes of LDS are done, then everyone's
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    dma_meet();
  };
  meet();
#pragma unroll
  for (int s = 0; s < D; ++s) read(s, 0, s);
  // k tile kt in buffer u % 2, its weights in set u.  The next one's activations are written to the other buffer, which every wave
  // has read to its end by the barrier before; behind this tile's barrier, D steps before its end, the next one's are read.
  auto pass = [&](int kt, auto U) {
    constexpr int u = decltype(U)::value, st = u & 1, off = u * STEPS;
#pragma unroll
    for (int s = 0; s < STEPS; ++s) {
      if (s == STEPS - D) meet();
      read((s + D) % STEPS, s + D < STEPS ? st : st ^ 1, (off + s + D) % R);
      if (s >= 1 && s <= LA) write_a(st ^ 1, s - 1);
      if (s >= 2 && s <= LA + 1) load_a(kt + 3, st ^ 1, s - 2);
      if (s >= I && s < I + J) load_w(kt + AHEAD, u, 0, s - I);
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int j = 0; j < J; ++j)
        acc[s % I][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(w[u][s / I][j], f[(off + s) % R], acc[s % I][j], 0, 0, 0);
      __builtin_amdgcn_sched_barrier(0);
    }
#pragma unroll
    for (int j = 0; j < J; ++j) load_w(kt + AHEAD, u, 1, j);
  };
  using U0 = std::integral_constant<int, 0>;
  using U1 = std::integral_constant<int, 1>;
  using U2 = std::integral_constant<int, 2>;
  using U3 = std::integral_constant<int, 3>;
  int kt = 0;
  for (; kt + AHEAD <= nkt; kt += AHEAD) {
    pass(kt, U0{});
    pass(kt + 1, U1{});
    pass(kt + 2, U2{});
    pass(kt + 3, U3{});
  }
  if (kt < nkt) {
    pass(kt, U0{});
    if (kt + 1 < nkt) {
      pass(kt + 1, U1{});
      if (kt + 2 < nkt) pass(kt + 2, U2{});
    }
  }
  // D: the lane's row is lane % 16, its columns 4 (lane / 16) + e of a block
  const bool half = epi == EPI_BF16 || epi == EPI_XIELU || epi == EPI_RELU2;
  const bool vec = ldc % 4 == 0 && (uintptr_t)C % (half ? 8 : 16) == 0;
  const float ap = epi == EPI_XIELU ? bias[N] : 0.f, an = epi == EPI_XIELU ? bias[N + 1] : 0.f;
#pragma unroll
  for (int j = 0; j < J; ++j) {
    const int n = n0 + (wid * J + j) * 16 + fk * 4;
    float b[4];
#pragma unroll
    for (int e = 0; e < 4; ++e) b[e] = bias && n + e < N ? bias[n + e] : 0.f;
#pragma unroll
    for (int i = 0; i < I; ++i) {
      const int m = m0 + i * 16 + fr;
      if (m >= M || n >= N) continue;
      const float v[4] = {acc[i][j][0] + b[0], acc[i][j][1] + b[1], acc[i][j][2] + b[2], acc[i][j][3] + b[3]};
      if (!vec || n + 4 > N) {
#pragma unroll
        for (int e = 0; e < 4; ++e)
          if (n + e < N) store_out(C, ldc, m, n + e, v[e], epi, bias, N);
      } else if (half) {
        bf16x4 o;
#pragma unroll
        for (int e = 0; e < 4; ++e) o[e] = (bf16)(epi == EPI_XIELU ? xielu_f(v[e], ap, an) : epi == EPI_RELU2 ? relu2_f(v[e]) : v[e]);
        *reinterpret_cast<bf16x4*>((bf16*)C + (size_t)m * ldc + n) = o;
      } else {
        float4* o = reinterpret_cast<float4*>((float*)C + (size_t)m * ldc + n);
        const float4 old = epi == EPI_ACC_F32 ? *o : float4{0.f, 0.f, 0.f, 0.f};
        *o = float4{old.x + v[0], old.y + v[1], old.z + v[2], old.w + v[3]};
      }
    }
  }
}

// (variant: VARIANT_STREAM + I)
constexpr int VARIANT_STREAM = 20;
int launch_tile_stream(int variant, const bf16* A, int lda, const bf16* Wt, const float* bias, void* C, int ldc, int M, int N, int K, int epi,
                       hipStream_t stream, int splits = 1, int k_per_split = 0) {
  if (!Wt || epi == EPI_SWIGLU) return (int)hipErrorInvalidValue;
  const int bm = (variant - VARIANT_STREAM) * 16, tiles_m = (M + bm - 1) / bm, tiles = tiles_m * ((N + 127) / 128);
#define MF_STREAM(I_) \
  case VARIANT_STREAM + I_: \
    tile_stream_kernel<I_><<<tiles * splits, 256, 0, stream>>>(A, lda, Wt, bias, C, ldc, M, N, K, epi, tiles_m, tiles, k_per_split); \
    return mf_launch_status();
  switch (variant) {
    MF_STREAM(6)
    MF_STREAM(8)
  }
#undef MF_STREAM
  return (int)hipErrorInvalidValue;
}

template <int BM, int BN, int STAGES, bool GROUPED, bool HALVES = false, bool TILED = false>
int configure_tile_dma() {
  static bool configured = false;
  if (configured) return 0;
  const hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void*>(tile_dma_kernel<BM, BN, STAGES, GROUPED, HALVES, TILED>),
                                           hipFuncAttributeMaxDynamicSharedMemorySize, DmaTile<BM, BN>::template lds<STAGES>());
  configured = e == hipSuccess;
  return (int)e;
}

template <int BM, int BN, int STAGES, bool TILED>
int launch_tile_dma(const bf16* A, int lda, const bf16* W, int ldw, const float* bias, void* C, int ldc, int M,
                    int N, int K, int epi, hipStream_t stream, int splits, int k_per_split) {
  if (const int e = configure_tile_dma<BM, BN, STAGES, false, false, TILED>()) return e;
  const int tiles_m = (M + BM - 1) / BM, tiles_n = (N + BN - 1) / BN;
  tile_dma_kernel<BM, BN, STAGES, false, false, TILED><<<dim3(tiles_m * tiles_n, splits), 512, DmaTile<BM, BN>::template lds<STAGES>(), stream>>>(
      A, lda, W, ldw, bias, C, ldc, M, N, K, epi, tiles_m, tile_order(tiles_m * tiles_n, splits, M, N, K), k_per_split, nullptr);
  return mf_launch_status();
}

template <int BM, int BN, int WM, int WN, int BK, bool VEC>
int launch_tile_v(const bf16* A, int lda, const bf16* W, int ldw, const float* bias, void* C, int ldc,
                  int M, int N, int K, int epi, hipStream_t stream, int splits = 1, int k_per_split = 0) {
  constexpr int smem = 2 * (BM + BN) * (BK + 8) * (int)sizeof(bf16);
  constexpr int NTHR = 64 * (BM / WM) * (BN / WN);
  static bool configured = false;
  auto kern = tile_kernel<BM, BN, WM, WN, BK, VEC>;
  if (!configured) {
    hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void*>(kern),
                                       hipFuncAttributeMaxDynamicSharedMemorySize, smem);
    if (e != hipSuccess) return (int)e;
    configured = true;
  }
  const int tiles_m = (M + BM - 1) / BM, tiles_n = (N + BN - 1) / BN;
  kern<<<dim3(tiles_m * tiles_n, splits), NTHR, smem, stream>>>(A, lda, W, ldw, bias, C, ldc, M, N, K, epi,
                                                                tiles_m, tile_order(tiles_m * tiles_n, splits, M, N, K), k_per_split);
  return mf_launch_status();
}

template <int BM, int BN, int WM, int WN, int BK = 64>
int launch_tile(const bf16* A, int lda, const bf16* W, int ldw, const float* bias, void* C, int ldc,
                int M, int N, int K, int epi, int vec_ok, hipStream_t stream, int splits = 1,
                int k_per_split = 0) {
  return vec_ok ? launch_tile_v<BM, BN, WM, WN, BK, true>(A, lda, W, ldw, bias, C, ldc, M, N, K, epi, stream,
                                                          splits, k_per_split)
                : launch_tile_v<BM, BN, WM, WN, BK, false>(A, lda, W, ldw, bias, C, ldc, M, N, K, epi, stream,
                                                           splits, k_per_split);
}

// The grouped forms: a tile row per entry of `groups` (int32 [n_groups][4] on the device), 32-bit sums stored; or, of matrices of gate
// and up rows (HALVES), the activation's values in bfloat16.
template <int BM, int BN, int STAGES, bool HALVES = false>
int launch_grouped_dma(const bf16* A, int lda, const bf16* W, int ldw, void* C, int ldc, const RowGroup* groups, int n_groups,
                       int N, int K, hipStream_t stream, const Halves& halves = Halves{}) {
  if (const int e = configure_tile_dma<BM, BN, STAGES, true, HALVES>()) return e;
  const int tiles_n = (N + BN - 1) / BN;
  tile_dma_kernel<BM, BN, STAGES, true, HALVES><<<dim3(n_groups * tiles_n), 512, DmaTile<BM, BN>::template lds<STAGES>(), stream>>>(
      A, lda, W, ldw, nullptr, C, ldc, 0, N, K, EPI_F32, n_groups, n_groups * tiles_n >= 16, 0, groups, halves);
  return mf_launch_status();
}

// one product of gate and up rows
template <int BM, int BN, int STAGES>
int launch_halves_dma(const bf16* A, int lda, const bf16* W, int ldw, bf16* C, int M, int N, int K, const Halves& halves, hipStream_t stream) {
  if (const int e = configure_tile_dma<BM, BN, STAGES, false, true>()) return e;
  const int tiles_m = (M + BM - 1) / BM, tiles_n = (N + BN - 1) / BN;
  tile_dma_kernel<BM, BN, STAGES, false, true><<<dim3(tiles_m * tiles_n), 512, DmaTile<BM, BN>::template lds<STAGES>(), stream>>>(
      A, lda, W, ldw, nullptr, C, halves.width, M, N, K, EPI_SWIGLU, tiles_m, tile_order(tiles_m * tiles_n, 1, M, N, K), 0, nullptr, halves);
  return mf_launch_status();
}

// ------------------------------------------------------------------ skinny kernel
constexpr int KC = 256;          // k per staging step
constexpr int SK_LD = KC + 8;    // LDS row stride in elements

// The tiled copy of a weight matrix (K a multiple of 32, rows padded to a multiple of 16):
// [rows / 16][K / 32][16 rows][32 k], 1 KB a tile.  A wave's load of an MFMA operand (lane ->
// row lane % 16, eight k at 8 (lane / 16)) is one tile: a contiguous kilobyte of whole 128-byte
// lines, where the row-major matrix gives it sixteen halves of lines K elements apart, and a
// wave that walks along K reads tile after tile.  The kernels for at most 64 rows, which take their
// weights straight from memory into MFMA operands, read this copy where the caller has one (the
// down product at 8 rows: 26.7 us from 34.1).  WSTEP: elements from one step of 32 k to the next.
template <bool TILED>
__device__ __forceinline__ const bf16* w_operand(const bf16* W, int ldw, int K, int row, int k) {
  if constexpr (TILED) return W + ((size_t)(row >> 4) * (K >> 5) + (k >> 5)) * 512 + (row & 15) * 32 + (k & 31);
  else return W + (size_t)row * ldw + k;
}

// 17 to 64 rows.  A block of 8 waves owns 128 weight rows; each wave streams its 16 rows from
// HBM straight into MFMA operands, a chunk (256 k) ahead; the activation rows of a chunk are
// staged in LDS once per block (double-buffered: the next chunk travels global -> registers
// while this one is multiplied, and is written to the other buffer afterwards, so there is
// one barrier per chunk).  Partial sums go to part[split][M][N]; with one split the epilogue
// runs in place.
template <int MT, bool VEC, bool TILED>
__global__ __launch_bounds__(512) void skinny_kernel(const bf16* __restrict__ A, int lda,
                                                     const bf16* __restrict__ W, int ldw,
                                                     const float* __restrict__ bias, void* __restrict__ C,
                                                     int ldc, float* __restrict__ part, int M, int N,
                                                     int K, int k_per_split, int epi) {
  extern __shared__ __attribute__((aligned(16))) unsigned char smem[];
  bf16* As = reinterpret_cast<bf16*>(smem);                     // [2][MT * 16][SK_LD]
  constexpr int ROWS = MT * 16;
  const int tid = threadIdx.x, lane = tid & 63, wid = tid >> 6;
  const int n_row = blockIdx.x * 128 + wid * 16 + (lane & 15);  // weight row of this lane
  const int n_ld = min(n_row, N - 1);                           // the row it reads
  const int kq = (lane >> 4) * 8;                               // k offset inside a 32-step
  const int k_begin = blockIdx.y * k_per_split;
  const int k_end = min(K, k_begin + k_per_split);

  floatx4 acc[MT];
#pragma unroll
  for (int i = 0; i < MT; ++i) acc[i] = floatx4{0.f, 0.f, 0.f, 0.f};

  // staging slots of this thread: MT chunks of 8 k; chunk c -> row c / 32, k (c % 32) * 8
  int srow[MT], sk[MT];
#pragma unroll
  for (int i = 0; i < MT; ++i) {
    const int c = i * 512 + tid;
    srow[i] = c / (KC / 8);
    sk[i] = (c % (KC / 8)) * 8;
  }
  bf16x8 wcur[KC / 32], wnext[KC / 32], stage[MT];
  auto load_chunk = [&](int k0, bf16x8 (&wd)[KC / 32]) {
    if (VEC && k0 + KC <= k_end) {                     // inside: no guards, nothing waits
#pragma unroll
      for (int s = 0; s < KC / 32; ++s)
        wd[s] = *reinterpret_cast<const bf16x8*>(w_operand<TILED>(W, ldw, K, n_ld, k0 + s * 32 + kq));
#pragma unroll
      for (int i = 0; i < MT; ++i) stage[i] = load8_inside(A, lda, min(srow[i], M - 1), k0 + sk[i]);
    } else {
#pragma unroll
      for (int s = 0; s < KC / 32; ++s) {
        const int k = k0 + s * 32 + kq;
        if constexpr (TILED) {          // K in whole steps of 32: eight elements are all inside or all outside
          const bf16x8 v = *reinterpret_cast<const bf16x8*>(w_operand<true>(W, ldw, K, n_ld, min(k, K - 8)));
          wd[s] = k + 8 <= k_end ? v : bf16x8{0, 0, 0, 0, 0, 0, 0, 0};
        } else {
          wd[s] = load8<VEC>(W, ldw, n_ld, k, k_end);
        }
      }
#pragma unroll
      for (int i = 0; i < MT; ++i) stage[i] = load8<VEC>(A, lda, min(srow[i], M - 1), k0 + sk[i], k_end);
    }
  };
  auto store_stage = [&](int buf) {
#pragma unroll
    for (int i = 0; i < MT; ++i)
      *reinterpret_cast<bf16x8*>(&As[(buf * ROWS + srow[i]) * SK_LD + sk[i]]) = stage[i];
  };
  load_chunk(k_begin, wcur);
  store_stage(0);
  __syncthreads();
  int buf = 0;
  for (int k0 = k_begin; k0 < k_end; k0 += KC) {
    const bool more = k0 + KC < k_end;
    if (more) load_chunk(k0 + KC, wnext);
    const bf16* as = As + buf * ROWS * SK_LD;
#pragma unroll
    for (int s = 0; s < KC / 32; ++s) {
#pragma unroll
      for (int i = 0; i < MT; ++i) {
        const bf16x8 a = *reinterpret_cast<const bf16x8*>(&as[(i * 16 + (lane & 15)) * SK_LD + s * 32 + kq]);
        acc[i] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, wcur[s], acc[i], 0, 0, 0);
      }
    }
    if (more) {
      store_stage(buf ^ 1);
#pragma unroll
      for (int s = 0; s < KC / 32; ++s) wcur[s] = wnext[s];
    }
    __syncthreads();
    buf ^= 1;
  }

  // D[m][n]: lane holds n = lane % 16, m = 4 (lane / 16) + r
  if (n_row >= N) return;
#pragma unroll
  for (int i = 0; i < MT; ++i)
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const int m = i * 16 + (lane >> 4) * 4 + r;
      if (m >= M) continue;
      if (part) {
        part[((size_t)blockIdx.y * M + m) * N + n_row] = acc[i][r];
      } else {
        store_out(C, ldc, m, n_row, acc[i][r] + (bias ? bias[n_row] : 0.f), epi, bias, N);
      }
    }
}

// The same product where every chunk is whole (K and the splits in multiples of 256, aligned rows),
// as a ring: each wave keeps its 8 weight fragments of a chunk in registers and refills one right
// behind the MFMA that used it, with the next chunk's, so the loads in flight never run dry at a
// chunk's end as they do above; the sums leave through an LDS tile, in rows of 512 bytes.
constexpr int SR_LD = 128 + 4;      // row stride of that tile (floats)

template <int MT, bool TILED>
__global__ __launch_bounds__(512) void skinny_ring_kernel(const bf16* __restrict__ A, int lda,
                                                          const bf16* __restrict__ W, int ldw,
                                                          const float* __restrict__ bias,
                                                          void* __restrict__ C, int ldc,
                                                          float* __restrict__ part, int M, int N, int K,
                                                          int k_per_split, int epi) {
  extern __shared__ __attribute__((aligned(16))) unsigned char smem[];
  constexpr int ROWS = MT * 16;
  bf16* As = reinterpret_cast<bf16*>(smem);                                            // [2][ROWS][SK_LD]
  float* ot = reinterpret_cast<float*>(smem + 2 * ROWS * SK_LD * sizeof(bf16));        // [ROWS][SR_LD]
  const int tid = threadIdx.x, lane = tid & 63, wid = tid >> 6;
  const int r16 = lane & 15, kq = (lane >> 4) * 8;
  const int n0 = blockIdx.x * 128;
  constexpr int WSTEP = TILED ? 512 : 32;
  const bf16* wrow = w_operand<TILED>(W, ldw, K, min(n0 + wid * 16 + r16, N - 1), kq);
  const int k_begin = blockIdx.y * k_per_split;
  const int k_end = min(K, k_begin + k_per_split);
  const int sk = (tid & 31) * 8;
  const bf16* src[MT];
#pragma unroll
  for (int i = 0; i < MT; ++i) src[i] = A + (size_t)min(i * 16 + (tid >> 5), M - 1) * lda + sk;
  bf16x8 stage[MT], wr[KC / 32];
#pragma unroll
  for (int i = 0; i < MT; ++i) stage[i] = *reinterpret_cast<const bf16x8*>(src[i] + k_begin);
#pragma unroll
  for (int s = 0; s < KC / 32; ++s) wr[s] = load_weights<TILED>(wrow + ((k_begin >> 5) + s) * WSTEP);
#pragma unroll
  for (int i = 0; i < MT; ++i)
    *reinterpret_cast<bf16x8*>(&As[(i * 16 + (tid >> 5)) * SK_LD + sk]) = stage[i];
  __syncthreads();
  floatx4 acc[MT];
#pragma unroll
  for (int i = 0; i < MT; ++i) acc[i] = floatx4{0.f, 0.f, 0.f, 0.f};
  int buf = 0;
  // a chunk's products, the next chunk asked for beside them (behind the last chunk nothing is: 64 KB of weights a block)
  auto chunk = [&](int kn, auto REFILL) {
    constexpr bool refill = decltype(REFILL)::value;
    if constexpr (refill) {
#pragma unroll
      for (int i = 0; i < MT; ++i) stage[i] = *reinterpret_cast<const bf16x8*>(src[i] + kn);
      __builtin_amdgcn_sched_barrier(0);
    }
    const bf16* as = As + buf * ROWS * SK_LD;
#pragma unroll
    for (int s = 0; s < KC / 32; ++s) {
#pragma unroll
      for (int i = 0; i < MT; ++i) {
        const bf16x8 a = *reinterpret_cast<const bf16x8*>(&as[(i * 16 + r16) * SK_LD + s * 32 + kq]);
        acc[i] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, wr[s], acc[i], 0, 0, 0);
      }
      if constexpr (refill) {
        wr[s] = load_weights<TILED>(wrow + ((kn >> 5) + s) * WSTEP);
        __builtin_amdgcn_sched_barrier(0);    // use a register, then refill it, in this order
      }
    }
    if constexpr (refill) {
      buf ^= 1;
#pragma unroll
      for (int i = 0; i < MT; ++i)
        *reinterpret_cast<bf16x8*>(&As[(buf * ROWS + i * 16 + (tid >> 5)) * SK_LD + sk]) = stage[i];
      __syncthreads();
    }
  };
  for (int kn = k_begin + KC; kn < k_end; kn += KC) chunk(kn, std::true_type{});
  chunk(0, std::false_type{});
  // D[m][n]: n = lane % 16, m = 4 (lane / 16) + r
#pragma unroll
  for (int i = 0; i < MT; ++i)
#pragma unroll
    for (int r = 0; r < 4; ++r) ot[(i * 16 + (lane >> 4) * 4 + r) * SR_LD + wid * 16 + r16] = acc[i][r];
  __syncthreads();
  const int c = tid & 127, n = n0 + c;
  if (n >= N) return;
  if (part) {
    for (int m = tid >> 7; m < M; m += 4) part[((size_t)blockIdx.y * M + m) * N + n] = ot[m * SR_LD + c];
  } else {
    const float b = bias ? bias[n] : 0.f;
    for (int m = tid >> 7; m < M; m += 4) store_out(C, ldc, m, n, ot[m * SR_LD + c] + b, epi, bias, N);
  }
}

// At most 16 rows: no LDS staging at all.  A block owns 16 NT weight rows; its NW waves split
// K between them, each streaming its slice of the weights from HBM and the matching slice of
// the few activation rows from L2 straight into MFMA operands, S steps (32 S k) of loads in
// flight ahead of the matrix cores.  The waves' sums meet in LDS and wave 0 adds them in a
// fixed order and runs the epilogue, so there is no second kernel and no atomics.
template <int NW, int NT, int S, bool VEC, bool PAIR = false>
__global__ __launch_bounds__(NW * 64) void skinny16_kernel(const bf16* __restrict__ A, int lda,
                                                           const bf16* __restrict__ W, int ldw,
                                                           const float* __restrict__ bias,
                                                           void* __restrict__ C, int ldc, int M, int N,
                                                           int K, int k_per_wave, int epi) {
  __shared__ float red[NW][NT][64][4];
  const int lane = threadIdx.x & 63, wid = threadIdx.x >> 6;
  // PAIR (SwiGLU, NT = 2): block b owns 16 gate rows of group b / 2 and the 16 up rows of
  // the same outputs, 32 rows further on
  constexpr int TSTRIDE = PAIR ? 32 : 16;
  const int n_base = (PAIR ? (blockIdx.x >> 1) * 64 + (blockIdx.x & 1) * 16 : blockIdx.x * 16 * NT) + (lane & 15);
  const int m_row = min(lane & 15, M - 1);               // rows past M read row M - 1; never stored
  int n_ld[NT];
#pragma unroll
  for (int j = 0; j < NT; ++j) n_ld[j] = min(n_base + TSTRIDE * j, N - 1);
  const int kq = (lane >> 4) * 8;
  const int k_begin = wid * k_per_wave;
  const int k_end = min(K, k_begin + k_per_wave);
  floatx4 acc[NT];
#pragma unroll
  for (int j = 0; j < NT; ++j) acc[j] = floatx4{0.f, 0.f, 0.f, 0.f};
  bf16x8 wc[NT][S], ac[S], wn[NT][S], an[S];
  // a batch that lies inside [k_begin, k_end) is loaded without guards (a guard's select
  // would make the wave wait for the load right away, and nothing would be in flight)
  auto load_batch = [&](int k0, bf16x8 (&wd)[NT][S], bf16x8 (&ad)[S]) {
    if (VEC && k0 + S * 32 <= k_end) {
#pragma unroll
      for (int s = 0; s < S; ++s) {
#pragma unroll
        for (int j = 0; j < NT; ++j) wd[j][s] = load8_inside(W, ldw, n_ld[j], k0 + s * 32 + kq);
        ad[s] = load8_inside(A, lda, m_row, k0 + s * 32 + kq);
      }
    } else {
      // the slice's last batch: whole steps still go unguarded, the rest is guarded or zero
#pragma unroll
      for (int s = 0; s < S; ++s) {
        const int k = k0 + s * 32;
        if (VEC && k + 32 <= k_end) {
#pragma unroll
          for (int j = 0; j < NT; ++j) wd[j][s] = load8_inside(W, ldw, n_ld[j], k + kq);
          ad[s] = load8_inside(A, lda, m_row, k + kq);
        } else {
#pragma unroll
          for (int j = 0; j < NT; ++j) wd[j][s] = load8<VEC>(W, ldw, n_ld[j], k + kq, k_end);
          ad[s] = load8<VEC>(A, lda, m_row, k + kq, k_end);
        }
      }
    }
  };
  if (k_begin < k_end) load_batch(k_begin, wc, ac);
  for (int k0 = k_begin; k0 < k_end; k0 += S * 32) {
    const bool more = k0 + S * 32 < k_end;
    if (more) load_batch(k0 + S * 32, wn, an);
#pragma unroll
    for (int s = 0; s < S; ++s)
#pragma unroll
      for (int j = 0; j < NT; ++j)
        acc[j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(ac[s], wc[j][s], acc[j], 0, 0, 0);
    if (more) {
#pragma unroll
      for (int s = 0; s < S; ++s) {
#pragma unroll
        for (int j = 0; j < NT; ++j) wc[j][s] = wn[j][s];
        ac[s] = an[s];
      }
    }
  }
#pragma unroll
  for (int j = 0; j < NT; ++j)
#pragma unroll
    for (int r = 0; r < 4; ++r) red[wid][j][lane][r] = acc[j][r];
  __syncthreads();
  if (wid != 0) return;
  if (epi == EPI_SWIGLU) {       // tile 0 gate, tile 1 up
    if constexpr (PAIR && NT == 2) {
      const int col = blockIdx.x * 16 + (lane & 15);
      if (col < ldc) {
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          const int m = (lane >> 4) * 4 + r;
          if (m >= M) continue;
          float g = 0.f, u = 0.f;
#pragma unroll
          for (int w = 0; w < NW; ++w) { g += red[w][0][lane][r]; u += red[w][1][lane][r]; }
          ((bf16*)C)[(size_t)m * ldc + col] = (bf16)swiglu_f(g, u, bias);
        }
      }
    }
    return;
  }
#pragma unroll
  for (int j = 0; j < NT; ++j) {
    const int n = n_base + 16 * j;
    if (n >= N) continue;
    const float b = bias ? bias[n] : 0.f;
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const int m = (lane >> 4) * 4 + r;      // D[m][n]: n = lane % 16, m = 4 (lane / 16) + r
      if (m >= M) continue;
      float v = 0.f;
#pragma unroll
      for (int w = 0; w < NW; ++w) v += red[w][j][lane][r];
      store_out(C, ldc, m, n, v + b, epi, bias, N);
    }
  }
}

// compute units of the current device (0 on error)
static int cu_count() {
  static int n_cu = 0;
  if (n_cu == 0) {
    int dev = 0;
    hipDeviceProp_t prop;
    if (hipGetDevice(&dev) != hipSuccess || hipGetDeviceProperties(&prop, dev) != hipSuccess) return 0;
    n_cu = prop.multiProcessorCount;
  }
  return n_cu;
}

// ---- which shapes each decode kernel takes (the launchers and `mf_gemm_bf16_plan` both ask here)

// K = 256 NS for which the register-resident kernel is instantiated
#define MF_STATIONARY_NS(X) X(4) X(6) X(8) X(10) X(12) X(14) X(16) X(20) X(24) X(28) X(32)

// weights in flight per wave of the register-resident kernel: a whole slice up to NS 16, else the
// largest divisor of NS that leaves the activations (4 NS registers) and the ring within budget
constexpr int stationary_ring(int NS, int NT) {
  if (NS <= 16) return NS;
  for (int r = 10; r > 1; --r)
    if (NS % r == 0 && 4 * NS + 4 * NT * r <= 176) return r;
  return 1;
}

constexpr int STATIONARY_K7 = 896;       // the one K that runs as 7 waves of 4 steps
constexpr int STATIONARY_PLAIN_K = 5120; // the longest K without a norm or SwiGLU

bool stationary_takes(int M, int N, int K, int epi, bool normed) {
  if (epi == EPI_SWIGLU && N % 64 != 0) return false;
  // (a model that narrow has few weight rows as well, and its steps are their kernels' starts, not
  // the stream: there the fold of the norm is what this kernel is taken for, from 64 tiles on)
  if (K == STATIONARY_K7) return M <= 16 && (N + 15) / 16 >= 64;
  if (M > 16 || (N + 15) / 16 < 128) return false;
  if (K % 256 != 0) return false;
  // a K above STATIONARY_PLAIN_K without a norm or SwiGLU to fold in (the o product of the widest models): the
  // rolling kernel is the faster one there
  if (K > STATIONARY_PLAIN_K && !normed && epi != EPI_SWIGLU) return false;
  switch (K / 256) {
#define MF_X(NS_) case NS_:
    MF_STATIONARY_NS(MF_X)
#undef MF_X
    return true;
  }
  return false;
}

// one block per CU over the whole of K, for 17 to 64 rows against a matrix that gives every CU at
// least 8 tiles of 16 weight rows
bool panel_takes(int M, int N, int K, bool aligned, int epi, int n_cu) {
  if (M <= 16 || M > 64 || K % 256 != 0 || !aligned) return false;
  if (epi == EPI_SWIGLU && N % 64 != 0) return false;
  return (N + 31) / 32 >= 4 * n_cu;
}

// the ring form of the K-split kernel needs whole chunks of 256 in every split
bool ring_takes(bool aligned, int K, int splits, int k_per_split) {
  return aligned && K % 256 == 0 && (long)(splits - 1) * k_per_split < K;
}

// The RMS norm folded around the products of at most 64 rows, across two kernels (y = x /
// sqrt(mean(x^2) + eps) * g, src/vec_ops.rs:500-522):
//  * a product that adds into the residual stream x and knows the weight g of the norm that reads
//    the stream next leaves, beside the stream's new rows, xg = bf16(x g) and for every row the
//    sums of x^2 in parts (`out_*`): over runs of 256 columns where the kernel that adds the parts
//    of a K split does it (17 to 64 rows: it has every new value of x in its hands), one part per
//    block where a one-kernel product does it in its epilogue (at most 16 rows, or `whole_kernel`: every block
//    owns some columns; `out_parts` places a row, the ones past the grid set to zero);
//  * the product that follows takes xg as its activations and multiplies its own sums by the
//    row's 1 / sqrt(sum / K + eps) in its epilogue (`in_*`), the partial sums of squares added up
//    in a fixed tree.
// No norm kernel, no pass over the stream between the two products.  The same arithmetic as the
// fold of the register-resident kernel above (bf16(x g) to the matrix cores, the row's factor in
// the epilogue).
constexpr int MF_NOT_BUILT = -2;     // an entry point's answer for a shape it has no kernel for; nothing was launched

struct FusedNorm {
  const float* in_ssq;     // [M][in_parts] partial sums of squares of the rows this product reads (null: none)
  int in_parts;
  float in_eps;
  const float* out_g;      // [N] weight of the norm that reads the output next (null: none)
  bf16* out_xg;            // [M][N]
  float* out_ssq;          // [M][out_parts]: a part for every run of 256 columns, or from a one-kernel product for every block; then zeros
  int out_parts;
};

// 1 / sqrt(mean(x^2) + eps) of NR rows from their partial sums, K the rows' length, in two steps
// so that a kernel can ask for the sums early and use them late; all lanes of a wave call both with
// the same rows (a row outside [0, M) gives 1).  The lanes take the partial sums between them, all
// rows' loads in flight together, and add up in a fixed tree.  None of the first loads stands behind a condition but `in_ssq` itself
// (see LanesSum; with a condition a load the 7B shape's gate|up of 8 rows waited two trips to memory before it asked for weights).
template <int NR>
struct RowSums {
  static constexpr int AT_ONCE = 4;      // of a row, asked for at once (as many as a product of one block a CU leaves)
  float x[NR][AT_ONCE];
  __device__ __forceinline__ void ask(const FusedNorm& f, const int (&rows)[NR], int M, int lane) {
#pragma unroll
    for (int i = 0; i < NR; ++i)
#pragma unroll
      for (int q = 0; q < AT_ONCE; ++q)
        x[i][q] = f.in_ssq ? f.in_ssq[(size_t)min(max(rows[i], 0), M - 1) * f.in_parts + min(lane + q * 64, f.in_parts - 1)] : 0.f;
  }
  __device__ __forceinline__ void factors(const FusedNorm& f, const int (&rows)[NR], int M, int K, int lane, float (&t)[NR]) const {
#pragma unroll
    for (int i = 0; i < NR; ++i) {
      const bool row = f.in_ssq && rows[i] >= 0 && rows[i] < M;
      t[i] = 0.f;
#pragma unroll
      for (int q = 0; q < AT_ONCE; ++q) t[i] += row && lane + q * 64 < f.in_parts ? x[i][q] : 0.f;
      if (row)
        for (int p = lane + AT_ONCE * 64; p < f.in_parts; p += 64) t[i] += f.in_ssq[(size_t)rows[i] * f.in_parts + p];
#pragma unroll
      for (int o = 32; o > 0; o >>= 1) t[i] += __shfl_xor(t[i], o, MF_WAVE);
      t[i] = row ? 1.0f / sqrtf(t[i] / (float)K + f.in_eps) : 1.f;
    }
  }
};


// End of a one-kernel product of at most 16 rows that prepares the next norm (FusedNorm::out_*):
// every lane has the squares of its own outputs of row e_m in `sq` (0 where it has none), the
// COLS lanes of a row sit side by side; their sum is this block's part of the row.  Block 0 also
// sets the places past the grid to zero.
template <int COLS>
__device__ __forceinline__ void norm_part_out(const FusedNorm& f, float sq, int e_m, int e_c, int M) {
#pragma unroll
  for (int o = COLS / 2; o > 0; o >>= 1) sq += __shfl_xor(sq, o, MF_WAVE);
  if (e_c == 0 && e_m < M) f.out_ssq[(size_t)e_m * f.out_parts + blockIdx.x] = sq;
  if (blockIdx.x == 0) {
    const int spare = f.out_parts - (int)gridDim.x;
    for (int i = threadIdx.x; i < M * spare; i += blockDim.x)
      f.out_ssq[(size_t)(i / spare) * f.out_parts + gridDim.x + i % spare] = 0.f;
  }
}

// The same split of the work as skinny16_kernel (a block owns up to 16 weight rows, its waves split
// K), for aligned operands and K a multiple of 32, with the loads rolling: a wave holds S steps
// of weights and activations in registers, and the refill of a register is issued right behind
// the MFMA that read it, so S steps of loads stay in flight the whole time in half the
// registers of the two-buffer scheme above.  With K of many thousands and few weight rows
// (the down projection) the chip is filled by loads in flight, not by blocks, and this is
// what the time depends on.
template <int NW, int S, bool ALL, bool TILED>
__global__ __launch_bounds__(NW * 64) void rolling16_kernel(const bf16* __restrict__ A, int lda,
                                                            const bf16* __restrict__ W, int ldw,
                                                            const float* __restrict__ bias,
                                                            void* __restrict__ C, int ldc, int M, int N,
                                                            int K, int steps_per_wave, int epi, int rpb,
                                                            FusedNorm fused) {
  constexpr int COLS = 16;
  constexpr int RS = COLS + 4;
  constexpr int WSTEP = TILED ? 512 : 32;
  __shared__ float red[NW][16][RS];
  const int lane = threadIdx.x & 63;
  const int wid = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);     // the same in the whole wave
  const int r16 = lane & 15;
  // rpb: weight rows per block (at most 16; fewer when that spreads the rows over every CU:
  // a CU draws only so much from memory, so an idle CU is bandwidth lost).  Lanes past the
  // block's rows read its last row again, from the CU's own cache.
  const int n0 = blockIdx.x * rpb;
  const int total = K / 32;
  const int T = min(steps_per_wave, total - wid * steps_per_wave);       // steps of this wave (none: not above 0)
  const int first = T > 0 ? wid * steps_per_wave : 0;
  const int kq = first * 32 + (lane >> 4) * 8;
  const bf16* arow = A + (size_t)min(r16, M - 1) * lda + kq;
  const bf16* wrow = w_operand<TILED>(W, ldw, K, min(n0 + min(r16, rpb - 1), N - 1), kq);
  floatx4 acc = floatx4{0.f, 0.f, 0.f, 0.f};
  // The epilogue's place of this lane: wave w adds up the sums of activation rows
  // [w 64 / COLS, (w + 1) 64 / COLS), every wave one pass at the same time.  Where the product is
  // added to what the output holds, the old value is asked for here, in front of the whole stream:
  // behind it, its way from memory would be the kernel's tail, once per pass.
  constexpr int ROWS_PER_PASS = 64 / COLS;
  static_assert(NW * ROWS_PER_PASS >= 16, "a pass for every activation row");
  const int e_c = lane % COLS;
  const int e_n = n0 + e_c;
  const int e_m = wid * ROWS_PER_PASS + lane / COLS;
  const bool e_mine = e_m < M && e_n < N && e_c < rpb;
  float c_old = 0.f, e_g = 0.f;
  if (epi == EPI_ACC_F32 && e_mine) c_old = ((const float*)C)[(size_t)e_m * ldc + e_n];
  if (fused.out_g && e_mine) e_g = fused.out_g[e_n];       // the next norm's weight, where this product prepares it
  bf16x8 a[S], w[S];
  auto load = [&](int s, int at) {
    w[s] = load_weights<TILED>(wrow + at * WSTEP);
    a[s] = *reinterpret_cast<const bf16x8*>(arow + at * 32);
  };
  auto multiply = [&](int s) { acc = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a[s], w[s], acc, 0, 0, 0); };
  // ALL: a slice that the registers hold, all of it asked for at once (in a loop over the slice's length the
  // compiler waits for every step: a decode step of one sequence at the 0.5B widths 775 us so, 749 at once).  A kernel of its own, for
  // 4, 8, 12 and 16 steps: with the rounds beside it in one kernel for 16 steps, 16 rows, tiled copy, microseconds together / apart: 1,280 x 2,048
  // 5.7 / 5.1, 1,152 x 3,584 7.6 / 7.1, 1,536 x 2,560 6.3 / 5.7, 1,024 x 1,024 3.8 / 3.65; 8 rows 4.9 / 4.4, 5.9 / 5.8, 5.0 / 4.8, 3.45 / 3.3.
  if constexpr (ALL) {
#pragma unroll
    for (int s = 0; s < S; ++s)
      if (s < T) load(s, s);
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int s = 0; s < S; ++s)
      if (s < T) multiply(s);
  } else {
    // Rounds of S steps, a register refilled behind its product.  Every refill is there without a condition, so that the compiler can
    // count what is in flight: past the slice's end it is the last step again (`rolling_steps` chooses S so that there are few).
    const int last = max(T, 1) - 1;
#pragma unroll
    for (int s = 0; s < S; ++s) {
      load(s, min(s, last));
      __builtin_amdgcn_sched_barrier(0);         // in the order of their use (left to the compiler: 3,584 x 18,944 of 8 rows 26.2 us, 25.4 so)
    }
    int base = 0;
    for (; base + 2 * S <= T; base += S) {
#pragma unroll
      for (int s = 0; s < S; ++s) {
        multiply(s);
        load(s, base + S + s);
        __builtin_amdgcn_sched_barrier(0);
      }
    }
    if (base + S < T) {
#pragma unroll
      for (int s = 0; s < S; ++s) {
        multiply(s);
        load(s, min(base + S + s, last));
        __builtin_amdgcn_sched_barrier(0);
      }
      base += S;
    }
#pragma unroll
    for (int s = 0; s < S; ++s)
      if (base + s < T) multiply(s);
  }
  // D[m][n]: n = lane % 16, m = 4 (lane / 16) + r
#pragma unroll
  for (int r = 0; r < 4; ++r) red[wid][(lane >> 4) * 4 + r][r16] = acc[r];
  __syncthreads();
  float sq = 0.f;
  if (e_mine) {
    float v = bias ? bias[e_n] : 0.f;
#pragma unroll
    for (int ww = 0; ww < NW; ++ww) v += red[ww][e_m][e_c];
    if (epi == EPI_ACC_F32) v += c_old;
    if (epi == EPI_ACC_F32) ((float*)C)[(size_t)e_m * ldc + e_n] = v;
    else store_out(C, ldc, e_m, e_n, v, epi, bias, N);
    if (fused.out_g) {
      fused.out_xg[(size_t)e_m * ldc + e_n] = (bf16)(v * e_g);
      sq = v * v;
    }
  }
  if (fused.out_g) norm_part_out<COLS>(fused, sq, e_m, e_c, M);
}

// How many steps `rolling16_kernel` holds for slices of `steps` above 16: at most 16, the one whose rounds have the fewest steps past the end.  Every length
// from 10 to 15 has shapes that it pays for (8 rows, tiled copy, weights from memory, microseconds with 16 steps only / 10, 12 and 16 / all):
// 896 x 4,864 9.25 / 6.8 / 6.8 (10 steps), 2,048 x 5,632 11.0 / 9.4 / 9.1 (11), 2,048 x 11,008 15.8 / 15.7 / 14.9 (11), 1,536 x 8,960 14.0 / 11.65 /
// 11.65 (12), 2,560 x 9,728 15.4 / 13.9 / 13.5 (13), 8,192 x 29,568 90 / 86 / 84.7 (13), 4,096 x 14,336 24.3 / 23.5 / 22.5 (14), 3,584 x 18,944
// 29.0 / 29.4 / 27.5 (15).
int rolling_steps(int steps) {
  int best = 16;
  for (int s = 15; s >= 10; --s)
    if ((steps + s - 1) / s * s < (steps + best - 1) / best * best) best = s;
  return best;
}

template <bool TILED>
int launch_rolling16(const bf16* A, int lda, const bf16* W, int ldw, const float* bias, void* C, int ldc,
                     int M, int N, int K, int epi, hipStream_t stream, const FusedNorm& fused = FusedNorm{}) {
  constexpr int NW = 8;
  const int steps_per_wave = (K / 32 + NW - 1) / NW;
  const int n_cu = cu_count();
  if (n_cu <= 0) return (int)hipErrorUnknown;
  int rpb = (N + n_cu - 1) / n_cu;                 // one block per CU when the rows are few
  rpb = rpb < 1 ? 1 : (rpb > 16 ? 16 : rpb);
  const int blocks = (N + rpb - 1) / rpb;
  if (fused.out_g && blocks > fused.out_parts) return MF_NOT_BUILT;
  auto run = [&](auto S, auto ALL) {
    rolling16_kernel<NW, decltype(S)::value, decltype(ALL)::value, TILED><<<blocks, NW * 64, 0, stream>>>(A, lda, W, ldw, bias, C, ldc, M, N, K,
                                                                                              steps_per_wave, epi, rpb, fused);
  };
#define MF_ROLLING(S_) case S_: run(std::integral_constant<int, S_>{}, std::false_type{}); break;
  if (steps_per_wave <= 4) run(std::integral_constant<int, 4>{}, std::true_type{});
  else if (steps_per_wave <= 8) run(std::integral_constant<int, 8>{}, std::true_type{});
  else if (steps_per_wave <= 12) run(std::integral_constant<int, 12>{}, std::true_type{});
  else if (steps_per_wave <= 16) run(std::integral_constant<int, 16>{}, std::true_type{});
  else switch (rolling_steps(steps_per_wave)) {
    MF_ROLLING(10) MF_ROLLING(11) MF_ROLLING(12) MF_ROLLING(13) MF_ROLLING(14) MF_ROLLING(15)
    default: run(std::integral_constant<int, 16>{}, std::false_type{});
  }
#undef MF_ROLLING
  return mf_launch_status();
}

template <int NW, int NT, int S, bool PAIR = false>
int launch_skinny16(const bf16* A, int lda, const bf16* W, int ldw, const float* bias, void* C, int ldc,
                    int M, int N, int K, int epi, int vec_ok, hipStream_t stream) {
  const int k_per_wave = ((K + NW - 1) / NW + 31) / 32 * 32;      // even shares; a slice's last batch may be short
  const int blocks = (N + 16 * NT - 1) / (16 * NT);
  if (vec_ok)
    skinny16_kernel<NW, NT, S, true, PAIR><<<blocks, NW * 64, 0, stream>>>(A, lda, W, ldw, bias, C, ldc, M, N,
                                                                           K, k_per_wave, epi);
  else
    skinny16_kernel<NW, NT, S, false, PAIR><<<blocks, NW * 64, 0, stream>>>(A, lda, W, ldw, bias, C, ldc, M,
                                                                            N, K, k_per_wave, epi);
  return mf_launch_status();
}

// ---- 17 to 64 rows over the whole of K, with a norm folded in
// The K-split kernels (below) need a second one to add their parts, 4 to 5 us of every product, and against a short K that is as
// much as the product itself.  Here a block takes 16 MT rows and up to 16 NT weight rows over the whole of K, its waves share K and
// read both operands straight into MFMA operands, the whole slice or S steps of it in flight (nothing is staged: no wave reads what
// another does), their sums meet in LDS, and the epilogue takes the norm's factors, adds to the stream and prepares the next norm.
// What bounds it is how many of these gathered loads (16 rows of 64 bytes) a CU gets through, activations above all: some 3.1 us
// and 0.175 us for each of a wave's loads, blocks of a CU added up (measured over 12 shapes of 896 to 18,944, 20 to 64 rows).
// Hence the choice of `whole_plan`.  q|k|v and o of 32 rows, this / K split or 64 x 64 tiles: 1,152 x 896 3.8 / 8.5 us, 896 x 896
// 4.3 / 10.2, 2,048 x 1,536 4.7 / 10.5, 2,560 x 2,048 5.9 / 10.7; 896 x 4,864 9.2 / 11.0.
template <int MT, int NT, int S, bool ONCE, bool TILED>
__global__ __launch_bounds__(512) void whole_kernel(const bf16* __restrict__ A, int lda, const bf16* __restrict__ W, int ldw,
                                                    const float* __restrict__ bias, float* __restrict__ C, int ldc, int M, int N, int K,
                                                    int accumulate, int rpb, FusedNorm fused) {
  constexpr int NW = 8, COLS = 16 * NT, RS = COLS + 4, ROWS = 16 * MT, WSTEP = TILED ? 512 : 32;
  __shared__ float red[NW][ROWS][RS];
  const int lane = threadIdx.x & 63, r16 = lane & 15;
  const int wid = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int m0 = blockIdx.y * ROWS, n0 = blockIdx.x * rpb;             // rpb: weight rows of a block, as in rolling16_kernel
  const int total = K / 32, share = (total + NW - 1) / NW;
  const int T = min(share, total - wid * share);                       // steps of this wave (none: not above 0)
  const int first = T > 0 ? wid * share : 0, last = max(T, 1) - 1;
  const int kq = first * 32 + (lane >> 4) * 8;
  const bf16 *arow[MT], *wrow[NT];
#pragma unroll
  for (int i = 0; i < MT; ++i) arow[i] = A + (size_t)min(m0 + i * 16 + r16, M - 1) * lda + kq;
#pragma unroll
  for (int j = 0; j < NT; ++j) wrow[j] = w_operand<TILED>(W, ldw, K, min(n0 + min(j * 16 + r16, rpb - 1), N - 1), kq);
  // the epilogue's places of this lane, what it needs of them asked for in front of the stream
  constexpr int PER_WAVE = 64 / COLS, PASS = NW * PER_WAVE, PASSES = (ROWS + PASS - 1) / PASS;
  const int e_c = lane % COLS, e_n = n0 + e_c;
  const bool e_col = e_c < rpb && e_n < N;
  const float e_g = fused.out_g && e_col ? fused.out_g[e_n] : 0.f, e_b = bias && e_col ? bias[e_n] : 0.f;
  float old[PASSES];
  LanesSum<COLS, 2, true> sums[PASSES];                                      // of the lane's own row
  auto part_row = [&](int p) {
    const int m = m0 + p * PASS + wid * PER_WAVE + lane / COLS;
    return fused.in_ssq ? fused.in_ssq + (size_t)min(m, M - 1) * fused.in_parts : nullptr;      // (rows past M: not stored)
  };
#pragma unroll
  for (int p = 0; p < PASSES; ++p) {
    const int r = p * PASS + wid * PER_WAVE + lane / COLS, m = m0 + r;
    old[p] = accumulate && r < ROWS && m < M && e_col ? C[(size_t)m * ldc + e_n] : 0.f;
  }
  floatx4 acc[MT][NT];
#pragma unroll
  for (int i = 0; i < MT; ++i)
#pragma unroll
    for (int j = 0; j < NT; ++j) acc[i][j] = floatx4{0.f, 0.f, 0.f, 0.f};
  bf16x8 a[S][MT], w[S][NT];
  auto load = [&](int s, int at) {
#pragma unroll
    for (int j = 0; j < NT; ++j) w[s][j] = *reinterpret_cast<const bf16x8*>(wrow[j] + (size_t)at * WSTEP);      // (the other tiles of rows read them too)
#pragma unroll
    for (int i = 0; i < MT; ++i) a[s][i] = *reinterpret_cast<const bf16x8*>(arow[i] + at * 32);
  };
  auto multiply = [&](int s) {
#pragma unroll
    for (int i = 0; i < MT; ++i)
#pragma unroll
      for (int j = 0; j < NT; ++j) acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a[s][i], w[s][j], acc[i][j], 0, 0, 0);
  };
  // All of the slice at once (ONCE: it has at most S steps), or S steps of it and the rest behind their products; no load of a slice that is longer than S stands
  // behind a condition (see `rolling16_kernel`).
  if constexpr (ONCE) {
#pragma unroll
    for (int s = 0; s < S; ++s)
      if (s < T) load(s, s);
  } else {
#pragma unroll
    for (int s = 0; s < S; ++s) load(s, min(s, last));
  }
#pragma unroll
  for (int p = 0; p < PASSES; ++p) sums[p].ask(part_row(p), fused.in_parts, e_c);
  __builtin_amdgcn_sched_barrier(0);
  if constexpr (ONCE) {
#pragma unroll
    for (int s = 0; s < S; ++s)
      if (s < T) multiply(s);
  } else {
    int base = 0;
    for (; base + S < T; base += S) {
#pragma unroll
      for (int s = 0; s < S; ++s) {
        multiply(s);
        load(s, min(base + S + s, last));
        __builtin_amdgcn_sched_barrier(0);
      }
    }
#pragma unroll
    for (int s = 0; s < S; ++s)
      if (base + s < T) multiply(s);
  }
  // D[m][n]: n = lane % 16, m = 4 (lane / 16) + r
#pragma unroll
  for (int i = 0; i < MT; ++i)
#pragma unroll
    for (int j = 0; j < NT; ++j)
#pragma unroll
      for (int r = 0; r < 4; ++r) red[wid][i * 16 + (lane >> 4) * 4 + r][j * 16 + r16] = acc[i][j][r];
  float fac[PASSES];
#pragma unroll
  for (int p = 0; p < PASSES; ++p)
    fac[p] = fused.in_ssq ? 1.0f / sqrtf(sums[p].add(part_row(p), fused.in_parts, e_c) / (float)K + fused.in_eps) : 1.f;
  __syncthreads();
#pragma unroll
  for (int p = 0; p < PASSES; ++p) {
    const int r = p * PASS + wid * PER_WAVE + lane / COLS, m = m0 + r;
    const bool mine = r < ROWS && m < M && e_col;
    float sq = 0.f;
    if (mine) {
      float v = 0.f;
#pragma unroll
      for (int ww = 0; ww < NW; ++ww) v += red[ww][r][e_c];
      v *= fac[p];
      v = v + e_b + old[p];
      C[(size_t)m * ldc + e_n] = v;
      if (fused.out_g) {
        fused.out_xg[(size_t)m * N + e_n] = (bf16)(v * e_g);
        sq = v * v;
      }
    }
    if (fused.out_g) {                                                 // this block's part of the row
#pragma unroll
      for (int o = COLS / 2; o > 0; o >>= 1) sq += __shfl_xor(sq, o, MF_WAVE);
      if (e_c == 0 && r < ROWS && m < M) {
        fused.out_ssq[(size_t)m * fused.out_parts + blockIdx.x] = sq;
        if (blockIdx.x == 0)                                           // (a row's places past the grid: zero)
          for (int x = gridDim.x; x < fused.out_parts; ++x) fused.out_ssq[(size_t)m * fused.out_parts + x] = 0.f;
      }
    }
  }
}

// How `whole_kernel` cuts a product: tiles of rows and of weight rows a block, weight rows a block, blocks; `loads`: a wave's loads
// by the cost above, those of the blocks that share a CU added up.  Every CU gets a block where there are rows enough.
struct WholePlan { int mt, nt, rpb, gx, gy; long loads; };
WholePlan whole_plan(int M, int N, int K, int n_cu) {
  WholePlan best{0, 0, 0, 0, 0, 1L << 40};
  for (int mt = 1; mt <= 2; ++mt)
    for (int nt = 1; nt <= 2; ++nt) {
      const int gy = (M + 16 * mt - 1) / (16 * mt), columns = std::max(1, n_cu / gy);
      const int rpb = std::min(16 * nt, (N + columns - 1) / columns), gx = (N + rpb - 1) / rpb;
      if (nt == 2 && rpb <= 16) continue;                              // (nothing to gain)
      const long loads = ((long)gx * gy + n_cu - 1) / n_cu * (mt + nt) * ((K / 32 + 7) / 8);
      if (loads < best.loads) best = WholePlan{mt, nt, rpb, gx, gy, loads};
    }
  return best;
}
// Up to 38 loads.  K split and added / this, 17, 32, 48 and 64 rows, 17 matrices: up to 38 loads 0.53 to 0.96 of the time (896 x 4,864, 38: 9.3 / 8.9 us
// at 17 rows, 11.5 / 9.6 at 64), with 40 to 48 0.78 to 1.0 (2,560 x 2,560 at 64 rows 13.8 / 12.2, 3,584 x 3,584 at 32 12.7 / 11.9, 3,072 x 3,072 at 64
// 13.9 / 13.9), with 56 0.99 to 1.11, from 70 on 1.13 and more (1,536 x 8,960 at 17 rows 13.1 / 14.9): the line is on the safe side of where they
// meet, some 45 to 50.  At least 512 weight rows, in 16s: not for the kernel's sake, which clamps its rows and would gain there too (500 x 896
// 6.9 / 4.2 at 17 rows, 384 x 2,048 7.4 / 5.5); widths that no model of this library's has keep the kernels that they had.
// (With the tiled copy or without, the same sums: the choice does not ask for it.)
bool whole_takes(int M, int N, int K, bool aligned, int epi, int n_cu) {
  if (M <= 16 || M > 64 || !aligned || N < 512 || N % 16 || K % 32 || n_cu <= 0 || (epi != EPI_F32 && epi != EPI_ACC_F32)) return false;
  return whole_plan(M, N, K, n_cu).loads <= 38;
}

template <bool TILED>
int launch_whole(const bf16* A, int lda, const bf16* W, int ldw, const float* bias, float* C, int ldc, int M, int N, int K, int epi,
                 const FusedNorm& fused, hipStream_t stream) {
  const WholePlan p = whole_plan(M, N, K, cu_count());
  const int share = (K / 32 + 7) / 8;
  auto run = [&](auto MT, auto NT) {
    auto held = [&](auto S, auto ONCE) {
      whole_kernel<decltype(MT)::value, decltype(NT)::value, decltype(S)::value, decltype(ONCE)::value, TILED>
          <<<dim3(p.gx, p.gy), 512, 0, stream>>>(A, lda, W, ldw, bias, C, ldc, M, N, K, epi == EPI_ACC_F32, p.rpb, fused);
    };
    // a slice of up to ten steps at once, or in two rounds (a longer one in more) with few steps past its end
    if (share <= 4) held(std::integral_constant<int, 4>{}, std::true_type{});
    else if (share <= 10) held(std::integral_constant<int, 10>{}, std::true_type{});
    else if (share <= 12) held(std::integral_constant<int, 6>{}, std::false_type{});
    else if (share <= 16) held(std::integral_constant<int, 8>{}, std::false_type{});
    else held(std::integral_constant<int, 10>{}, std::false_type{});
  };
  using One = std::integral_constant<int, 1>;
  using Two = std::integral_constant<int, 2>;
  if (p.mt == 1) p.nt == 1 ? run(One{}, One{}) : run(One{}, Two{});
  else p.nt == 1 ? run(Two{}, One{}) : run(Two{}, Two{});
  return mf_launch_status();
}

// At most 16 rows and K = 256 NS (NS steps of 32 k for each of 8 waves): the activations are
// read once per block and stay in registers.  The grid is one block per CU; a block walks
// over its share of the 16-row weight tiles (items), and the load of the next item's
// weights is issued right behind the MFMA that frees the register, so the weight stream
// never pauses between items.  After an item the waves' sums meet in LDS (two buffers, one
// barrier per item) and the waves take turns at adding them and running the epilogue.
// Against the kernel above this removes the per-tile re-read of the activations (which
// cost a quarter of the time at 8 rows) and the start-up of a block per tile.
//
// NORM: the activations are rows of the 32-bit residual stream, to be RMS-normalised on the way
// in (y = x / sqrt(mean(x^2) + eps) * g, src/vec_ops.rs:500-522).  The 1 / sqrt(..) is one
// number per row, so it can wait for the epilogue: the matrix cores get bf16(x * g), every
// wave sums x^2 over its own slice of K while it converts, and the epilogue multiplies the
// row's sums by 1 / sqrt(total / K + eps).  No pass over the row beforehand, no kernel and no
// activation buffer between the norm and the product.
struct NormArgs {
  const float* g;          // [K] norm weight
  const int* row_idx;      // activation row m is residual row row_idx[m] (null: m)
  float eps;
};

//
// RING: how many of a slice's NS steps of weights a wave keeps in flight (a divisor of NS).  With
// RING = NS the registers hold a whole item; for a long K (5120, 8192) the activations alone take
// up to half the registers, so the weights go through a shorter ring, and a register is refilled
// with the step RING further on, of this item or of the next one.
// NW: waves of a block, each with a slice of NS steps of K: 8, K = 256 NS; or 7 with NS = 4 for a K
// of 896 (14 heads of 64, the narrowest model of the family), which is no multiple of 256.
// ONCE: the weights are marked as read once (`load_weights`).
template <int NS, int RING, int NT, bool PAIR, bool NORM, bool TILED, int NW, bool ONCE>
__global__ __launch_bounds__(NW * 64) void stationary16_kernel(const void* __restrict__ Av, int lda,
                                                               const bf16* __restrict__ W, int ldw,
                                                               const float* __restrict__ bias,
                                                               void* __restrict__ C, int ldc, int M, int N,
                                                               int cols_total, int unit, int share, int extra, int epi,
                                                               NormArgs norm, FusedNorm fused) {
  constexpr int KK = NW * NS * 32;         // K
  constexpr int WSTEP = TILED ? 512 : 32;  // elements from one step's weights to the next's
  constexpr int COLS = 16 * NT;            // weight rows (output columns) of an item
  constexpr int RS = COLS + 4;             // row stride of the sums in LDS: conflict-free writes
  __shared__ float red[2][NW][16][RS];     // [buffer][wave][activation row][weight row of the item]
  __shared__ float ssq[NW][16];            // NORM: sum of x^2 over a wave's slice, per activation row
  __shared__ float rfac[16];               // not NORM: the rows' factors of a norm prepared by the product before (1 where none)
  extern __shared__ __attribute__((aligned(16))) float gs[];   // NORM: the norm's weight, K floats
  static_assert(NS % RING == 0, "the ring divides a slice");
  static_assert(PAIR ? NW * 4 >= 16 : NW * (64 / COLS) >= 16, "an epilogue pass for every activation row");
  const int lane = threadIdx.x & 63, wid = threadIdx.x >> 6;
  const int r16 = lane & 15;
  const int k0 = wid * NS * 32 + (lane >> 4) * 8;         // this lane's k in step 0 of its slice
  // The block's share: output columns [c_begin, c_end), the same number for every block up to
  // one `unit`, so that every CU streams the same bytes (a CU draws only so much from memory;
  // whole items per block would leave some with a fifth more than others).  PAIR: a column is
  // a gate row and the up row 32 further on, in groups of 64 weight rows.  An item is CH
  // columns; lanes past c_end read the share's last row again, from the CU's own cache.
  // (`share` units a block and one more for the first `extra` blocks: the host has divided, so
  // that a block's first loads do not wait behind a division in software)
  constexpr int CH = PAIR ? 16 : COLS;
  const int b = blockIdx.x;
  const int c_begin = (b * share + min(b, extra)) * unit;
  const int c_end = min(((b + 1) * share + min(b + 1, extra)) * unit, cols_total);
  const int n_items = (c_end - c_begin + CH - 1) / CH;
  auto lane_wrow = [&](int c0, int j) {      // weight row of this lane in tile j of the item at c0
    if (PAIR) {
      const int col = min(c0 + r16, c_end - 1);
      return (col >> 5) * 64 + (col & 31) + 32 * j;
    }
    return min(c0 + 16 * j + r16, c_end - 1);
  };
  const bf16* Wp = W;            // the weights, through a name whose use can be held back
  bf16x8 w[NT][RING];
  const bf16* wrow[NT];          // this lane's rows in the next item
  const bf16* wcur[NT];          // and in the current one (used when RING < NS)
  // The first item's loads are asked for without a condition (every block has an item: the grid is
  // no larger than the units to share): a load behind a branch makes the compiler count, for every
  // wait after it, with the path that has fewer loads in flight, and the prologue would wait for
  // the activations until most of the first weights have arrived as well.
  auto first_loads = [&](int j) {
    wcur[j] = w_operand<TILED>(Wp, ldw, KK, lane_wrow(c_begin, j), k0);
#pragma unroll
    for (int s = 0; s < RING; ++s) w[j][s] = load_weights<ONCE>(wcur[j] + s * WSTEP);
  };
  // The epilogue's place of this lane in an item: wave w adds up the sums of activation rows
  // [w 64 / COLS, (w + 1) 64 / COLS), all waves at once.  What the epilogue needs from memory (the
  // bias, and the output's old value where the product is added to it) is asked for an item ahead, in
  // front of the refills and without a condition (a lane with no place, or no such
  // operand, reads the head of the weights and drops it): behind the barrier it would make
  // the wave wait for every load it has in flight, and the kernel's last item for memory; asked for in the item itself and held
  // there, it made every item wait for the weights in flight before it (gate|up of 8 rows at the 7B widths).
  // The place is made anew each time: left alone, the compiler carries an address from item to item for every operand and for
  // every kind of output, and with a K from 5,120 on spilled them; a reload is counted with the weights' loads and comes back behind
  // them, so every item waited for the weights in flight (8 rows with the norm folded in, tiled copy, microseconds with spills / so:
  // 152,064 x 6,144 320 / 292, 128,000 x 7,168 306 / 284, 9,216 x 7,168 34.4 / 32.9; level where nothing was spilled).
  const int e_c = lane % COLS;
  auto place = [&](int c0, int& m, int& n) {
    m = PAIR ? wid * 4 + (lane >> 4) : wid * (64 / COLS) + lane / COLS;
    n = c0 + (PAIR ? r16 : e_c);
    asm volatile("" : "+v"(m), "+v"(n));
  };
  float next_old = 0.f, next_bias = 0.f, next_g = 0.f;
  auto ask_epilogue = [&](int c0) {
    if constexpr (!PAIR) {
      int e_m, e_n;
      place(c0, e_m, e_n);
      const bool mine = e_n < c_end && e_m < M;
      const float* none = reinterpret_cast<const float*>(W);
      next_old = *((mine && epi == EPI_ACC_F32) ? (const float*)C + (size_t)e_m * ldc + e_n : none);
      next_bias = *((mine && bias) ? bias + e_n : none);
      next_g = *((mine && fused.out_g) ? fused.out_g + e_n : none);
    }
  };
  bf16x8 afr[NS];
  float ss = 0.f;
  if constexpr (NORM) {
    const int m_src = min(r16, M - 1);
    const float* xrow = (const float*)Av + (size_t)(norm.row_idx ? norm.row_idx[m_src] : m_src) * lda + k0;
    // step s of the slice: sum of squares, and bf16(x * g) into the operand registers
    auto convert_step = [&](int s, const float4 x0, const float4 x1) {
      const float4 g0 = *reinterpret_cast<const float4*>(&gs[k0 + s * 32]);
      const float4 g1 = *reinterpret_cast<const float4*>(&gs[k0 + s * 32 + 4]);
      ss = fmaf(x0.x, x0.x, ss); ss = fmaf(x0.y, x0.y, ss); ss = fmaf(x0.z, x0.z, ss); ss = fmaf(x0.w, x0.w, ss);
      ss = fmaf(x1.x, x1.x, ss); ss = fmaf(x1.y, x1.y, ss); ss = fmaf(x1.z, x1.z, ss); ss = fmaf(x1.w, x1.w, ss);
      afr[s][0] = (bf16)(x0.x * g0.x); afr[s][1] = (bf16)(x0.y * g0.y);
      afr[s][2] = (bf16)(x0.z * g0.z); afr[s][3] = (bf16)(x0.w * g0.w);
      afr[s][4] = (bf16)(x1.x * g1.x); afr[s][5] = (bf16)(x1.y * g1.y);
      afr[s][6] = (bf16)(x1.z * g1.z); afr[s][7] = (bf16)(x1.w * g1.w);
      // the packed value is wanted here and now (left alone, the compiler keeps x and g
      // alive and converts in front of the first MFMA, at twice the registers)
      // (and for a long row the sum as well: put off, it keeps x alive in 32 bits)
      if constexpr (NS <= 16) asm volatile("" : "+v"(afr[s]));
      else asm volatile("" : "+v"(afr[s]), "+v"(ss));
    };
    if constexpr (NS <= 16) {
      // Everything the prologue needs is asked for at once, oldest first in the order it is
      // used: the norm's weight (staged in LDS for all waves), this lane's x, and the first
      // item's tile 0, which keeps HBM at work while the activations are converted.  The order is
      // pinned: left alone, the compiler asks for the weights first and then waits for them
      // before it stages g.
      static_assert(NS > 16 || NW * NS * 32 <= 2 * NW * 64 * 4, "two float4 of g per thread cover K");
      const int ge0 = min((int)threadIdx.x * 4, NW * NS * 32 - 4);                 // the last ones twice
      const int ge1 = min((NW * 64 + (int)threadIdx.x) * 4, NW * NS * 32 - 4);
      const float4 gt0 = *reinterpret_cast<const float4*>(norm.g + ge0);
      const float4 gt1 = *reinterpret_cast<const float4*>(norm.g + ge1);
      float4 x[NS][2];
#pragma unroll
      for (int s = 0; s < NS; ++s) {
        x[s][0] = *reinterpret_cast<const float4*>(xrow + s * 32);
        x[s][1] = *reinterpret_cast<const float4*>(xrow + s * 32 + 4);
      }
      __builtin_amdgcn_sched_barrier(0);
      ask_epilogue(c_begin);
      first_loads(0);
      __builtin_amdgcn_sched_barrier(0);
      *reinterpret_cast<float4*>(&gs[ge0]) = gt0;
      *reinterpret_cast<float4*>(&gs[ge1]) = gt1;
      __syncthreads();
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int s = 0; s < NS; ++s) convert_step(s, x[s][0], x[s][1]);
    } else {
      // A long row does not fit the registers in 32 bits beside its own bf16 copy: x comes in
      // sets of XC steps, the next set asked for before this one is converted, and the first
      // weights wait until the activations are in place.
      constexpr int XC = 4, SETS = NS / XC;
      static_assert(NS % XC == 0, "whole sets");
      float4 x[2][XC][2];
      const float* xp = xrow;
      auto load_set = [&](int c, int b) {
#pragma unroll
        for (int i = 0; i < XC; ++i) {
          x[b][i][0] = *reinterpret_cast<const float4*>(xp + (c * XC + i) * 32);
          x[b][i][1] = *reinterpret_cast<const float4*>(xp + (c * XC + i) * 32 + 4);
        }
      };
      load_set(0, 0);
      for (int e = (int)threadIdx.x * 4; e < NW * NS * 32; e += NW * 64 * 4)
        *reinterpret_cast<float4*>(&gs[e]) = *reinterpret_cast<const float4*>(norm.g + e);
      __syncthreads();
#pragma unroll
      for (int c = 0; c < SETS; ++c) {
        if (c + 1 < SETS) load_set(c + 1, (c + 1) & 1);
#pragma unroll
        for (int i = 0; i < XC; ++i) convert_step(c * XC + i, x[c & 1][i][0], x[c & 1][i][1]);
        // the address of the sets further on hangs on this set's last operand: asked for all at
        // once (which is what the compiler does with loads off one pointer) the row in 32 bits
        // would not fit the registers
        asm volatile("" : "+v"(xp), "+v"(afr[c * XC + XC - 1]));
        __builtin_amdgcn_sched_barrier(0);
      }
      asm volatile("" : "+s"(Wp), "+v"(afr[NS - 1]));     // no weights before the activations are in place
      ask_epilogue(c_begin);
      first_loads(0);
    }
    ss += __shfl_xor(ss, 16);
    ss += __shfl_xor(ss, 32);
    if (lane < 16) ssq[wid][lane] = ss;    // read behind the first item's barrier
    __builtin_amdgcn_sched_barrier(0);
  } else {
    const bf16* arow = (const bf16*)Av + (size_t)min(r16, M - 1) * lda + k0;
#pragma unroll
    for (int s = 0; s < NS; ++s) afr[s] = *reinterpret_cast<const bf16x8*>(arow + s * 32);
  }
  // Not NORM: the activations may be bf16(x g) of rows whose sums of squares the product before has
  // left in parts (FusedNorm::in_*): wave w adds up rows w, w + NW, ..., asked for here, between the
  // activations and the first weights, and used behind them; the epilogue multiplies by the factors.
  constexpr int FR = (16 + NW - 1) / NW;
  int frow[FR];
  float ffac[FR];
  RowSums<FR> fsums;
#pragma unroll
  for (int i = 0; i < FR; ++i) frow[i] = (!NORM && fused.in_ssq && wid + NW * i < 16) ? wid + NW * i : -1;
  if constexpr (!NORM) {
    fsums.ask(fused, frow, M, lane);
    ask_epilogue(c_begin);
    __builtin_amdgcn_sched_barrier(0);
    first_loads(0);
  }
#pragma unroll
  for (int j = 1; j < NT; ++j) first_loads(j);
  if constexpr (!NORM) {
    fsums.factors(fused, frow, M, KK, lane, ffac);
    if (lane == 0)
#pragma unroll
      for (int i = 0; i < FR; ++i)
        if (wid + NW * i < 16) rfac[wid + NW * i] = ffac[i];       // read behind the first item's barrier
  }
  float sq = 0.f;                      // a product that prepares the next norm: squares of this lane's outputs
  // An item.  Its body has no branch, so that the compiler can count the loads in flight and wait for the oldest one only; the last
  // item, which refills nothing, has a body of its own (loads that went to the head of the matrix there, to be dropped, were
  // every block's to the same few lines: with `load_weights` 1 us of the 4.8 that q|k|v of 1,152 x 896 took).
  auto item = [&](int it, auto NEXT) {
    constexpr bool next = decltype(NEXT)::value;
    const int c0 = c_begin + it * CH;
    if constexpr (next) {
#pragma unroll
      for (int j = 0; j < NT; ++j) wrow[j] = w_operand<TILED>(Wp, ldw, KK, lane_wrow(c0 + CH, j), k0);
    }
    floatx4 acc[NT];
#pragma unroll
    for (int j = 0; j < NT; ++j) acc[j] = floatx4{0.f, 0.f, 0.f, 0.f};
    const float c_old = next_old, e_bias = next_bias, e_g = next_g;
    if constexpr (next) ask_epilogue(c0 + CH);
#pragma unroll
    for (int s = 0; s < NS; ++s) {
#pragma unroll
      for (int j = 0; j < NT; ++j) {
        acc[j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(afr[s], w[j][s % RING], acc[j], 0, 0, 0);
        // the step RING further on: of this item, or of the next one.  (The load stays behind
        // the MFMA: moved in front of it, it needs a register of its own.)
        if constexpr (RING < NS) {
          asm volatile("" : "+v"(acc[j]) : : "memory");
          __builtin_amdgcn_sched_barrier(0);
        }
        if (s + RING < NS) w[j][s % RING] = load_weights<ONCE>(wcur[j] + (s + RING) * WSTEP);
        else if (next) w[j][s % RING] = load_weights<ONCE>(wrow[j] + (s + RING - NS) * WSTEP);
        __builtin_amdgcn_sched_barrier(0);      // keep "use a register, then refill it" in this order
      }
    }
    if constexpr (next) {
#pragma unroll
      for (int j = 0; j < NT; ++j) wcur[j] = wrow[j];
    }
    // D[m][n]: n = lane % 16, m = 4 (lane / 16) + r
    const int buf = it & 1;
#pragma unroll
    for (int j = 0; j < NT; ++j)
#pragma unroll
      for (int r = 0; r < 4; ++r) red[buf][wid][(lane >> 4) * 4 + r][j * 16 + r16] = acc[j][r];
    __syncthreads();
    // The buffer is written again two items on, behind the next barrier, which this wave
    // reaches only after it has read its sums here.
    auto row_scale = [&](int m) {          // NORM: 1 / sqrt(mean(x^2) + eps) of activation row m
      float t = 0.f;
#pragma unroll
      for (int ww = 0; ww < NW; ++ww) t += ssq[ww][m];
      return 1.0f / sqrtf(t / (float)(NW * NS * 32) + norm.eps);
    };
    if constexpr (PAIR) {
      static_assert(NT == 2, "a gate tile and an up tile");
      int col, m;
      place(c0, m, col);
      if (epi == EPI_SWIGLU && col < c_end && col < ldc && m < M) {
        float g = 0.f, u = 0.f;
#pragma unroll
        for (int ww = 0; ww < NW; ++ww) { g += red[buf][ww][m][r16]; u += red[buf][ww][m][16 + r16]; }
        const float sc = NORM ? row_scale(m) : rfac[m];
        g *= sc;
        u *= sc;
        ((bf16*)C)[(size_t)m * ldc + col] = (bf16)swiglu_f(g, u, bias);
      }
    } else {
      int e_m, e_n;
      place(c0, e_m, e_n);
      if (e_n < c_end && e_m < M) {
        float v = 0.f;
#pragma unroll
        for (int ww = 0; ww < NW; ++ww) v += red[buf][ww][e_m][e_c];
        v *= NORM ? row_scale(e_m) : rfac[e_m];
        v += (bias ? e_bias : 0.f);
        if (epi == EPI_ACC_F32) v += c_old;
        if (epi == EPI_ACC_F32) ((float*)C)[(size_t)e_m * ldc + e_n] = v;
        else store_out(C, ldc, e_m, e_n, v, epi, bias, N);
        if (fused.out_g) {
          fused.out_xg[(size_t)e_m * ldc + e_n] = (bf16)(v * e_g);
          sq = fmaf(v, v, sq);
        }
      }
    }
  };
  for (int it = 0; it + 1 < n_items; ++it) item(it, std::true_type{});
  item(n_items - 1, std::false_type{});
  if constexpr (!PAIR)
    if (fused.out_g) norm_part_out<COLS>(fused, sq, wid * (64 / COLS) + lane / COLS, lane % COLS, M);
}

// true when the shape is one the register-resident kernel is built for
template <int NS, int NT, bool PAIR, bool TILED, int NW = 8>
int launch_stationary16(const void* A, int lda, const bf16* W, int ldw, const float* bias, void* C, int ldc,
                        int M, int N, int epi, const NormArgs* norm, const FusedNorm& fused, hipStream_t stream) {
  const int n_cu = cu_count();
  if (n_cu <= 0) return (int)hipErrorUnknown;
  const int cols_total = PAIR ? N / 2 : N;
  // shares in whole 128-byte lines of 32-bit output where the output is large enough for the
  // cost of partial lines to show; else in pairs of columns
  const int unit = (!PAIR && cols_total / 32 >= 8 * n_cu) ? 32 : 2;
  const int units = (cols_total + unit - 1) / unit;
  const int grid = units < n_cu ? units : n_cu;
  // registers: 4 NS for the activations and 4 NT RING for the weights in flight, of 256.  A long
  // K keeps 8 to 10 loads of 1 KB in flight per wave, far more than a CU has outstanding anyway.
  constexpr int RING = stationary_ring(NS, NT);
  static_assert(NS % RING == 0 && 4 * NS + 4 * NT * RING <= 200, "activations and weight ring fit the registers");
  auto run = [&](auto ONCE) {
    if (norm) {
      constexpr int smem = NW * NS * 32 * (int)sizeof(float);      // the norm's weight
      auto kern = stationary16_kernel<NS, RING, NT, PAIR, true, TILED, NW, decltype(ONCE)::value>;
      static bool configured = false;
      if (!configured) {
        hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void*>(kern),
                                           hipFuncAttributeMaxDynamicSharedMemorySize, smem);
        if (e != hipSuccess) return (int)e;
        configured = true;
      }
      if (fused.in_ssq || fused.out_g) return MF_NOT_BUILT;
      kern<<<grid, NW * 64, smem, stream>>>(A, lda, W, ldw, bias, C, ldc, M, N, cols_total, unit, units / grid, units % grid,
                                            epi, *norm, FusedNorm{});
    } else if constexpr (PAIR || NS * NW * 32 <= STATIONARY_PLAIN_K) {
      if (fused.out_g && (PAIR || grid > fused.out_parts)) return MF_NOT_BUILT;
      stationary16_kernel<NS, RING, NT, PAIR, false, TILED, NW, decltype(ONCE)::value><<<grid, NW * 64, 0, stream>>>(
          A, lda, W, ldw, bias, C, ldc, M, N, cols_total, unit, units / grid, units % grid, epi, NormArgs{nullptr, nullptr, 0.f}, fused);
    } else {
      return MF_NOT_BUILT;
    }
    return mf_launch_status();
  };
  // Weights marked as read once: from the tiled copy, and from the matrix where a product that is not SwiGLU has a K of up to 2,048 and a block at
  // most eight items (of four and of 19 the marked loads are the faster and the slower ones).  Marked / not, weights from memory, no copy,
  // microseconds, 8 and 16 rows: 2,560 x 896 3.7 / 4.4 and 3.7 / 4.3, 9,216 x 1,024 6.2 / 6.8 and 6.7 / 7.1, 2,048 x 1,536 3.9 / 4.3 and level, 2,560 x 2,048
  // 4.7 / 5.1 and 5.3 / 5.2, 28,672 x 2,048 27.2 / 28.5 and 28.2 / 29.8, with the norm folded in 2,048 x 1,536 4.8 / 5.2 and 5.7 / 5.8; but
  // 151,936 x 1,536 with the norm 98.1 / 96.8 and 106.6 / 104.0 (one row 93.6 / 85.9), 3,072 x 2,560 6.2 / 5.9, 4,608 x 3,584 10.1 / 9.85, SwiGLU
  // 9,728 x 896 6.3 / 6.2, 17,920 x 1,536 13.7 / 13.1 and 14.2 / 13.4.
  if constexpr (TILED) {
    return run(std::true_type{});
  } else {
    if constexpr (!PAIR && NW * NS * 32 <= 2048)
      if ((units / grid + 1) * unit <= 8 * 16 * NT) return run(std::true_type{});
    return run(std::false_type{});
  }
}

// 17 to 64 rows against a wide matrix (at least 8 tiles of 16 weight rows for every CU): one block
// per CU with an equal share of the matrix, the whole of K, no partial sums between blocks and no
// second kernel.  The share is cut into passes of at most 16 tiles; wave w multiplies tiles w and
// w + 8 of the pass.  A slot with no tile multiplies the matrix's first bytes, read by all lanes
// alike, and its sums are dropped: every wave runs the same instructions, so the loads in flight
// can be counted, and such a load is one look-up where a tile's (64 lanes in 16 rows) is 64 -- repeating
// a real tile there made the cache's tag rate the limit.  They are marked as read once like the others (tiled copy, all loads marked / none /
// all but the second tile's of a wave, where the slots with no tile are, microseconds: 152,064 x 3,584 17 rows 184 / 197 / 196, 64 rows 211 / 230 / 231; 151,936 x 2,048
// 48 rows 116 / 130 / 130; SwiGLU 43,008 x 5,120 64 rows 84 / 93 / 92; 151,936 x 896 level).  A body of its own for the last step,
// with nothing asked for to be dropped, costs the others more than it saves: 184 / 186, 211 / 217, 116 / 121, 84 / 87.  Weights go
// from HBM straight into MFMA operands through a ring of 16 fragments a wave: the load of the
// next chunk's fragment is issued right behind the MFMA that frees the register, and runs on
// into the next pass (a ring of two chunks measured the same).  The activations of a chunk
// (256 k) are staged in LDS once per block, double-buffered, as in skinny_kernel; a pass re-reads
// them from L2.  At the end of a pass the sums go through an LDS tile so that rows are stored in
// whole lines, and SwiGLU pairs a gate tile with its up tile there.  (Folding the RMS norm into
// the staging, as the 16-row kernel does, measured slower here: every block would re-read the
// activations in 32 bits.)
constexpr int PANEL_TILES = 16;                 // tiles of a pass
constexpr int OT_LD = PANEL_TILES * 16 + 4;     // row stride of the output tile in LDS (floats)

template <int MT, bool TILED>
__global__ __launch_bounds__(512) void panel_kernel(const bf16* __restrict__ A, int lda,
                                                    const bf16* __restrict__ W, int ldw,
                                                    const float* __restrict__ bias, void* __restrict__ C,
                                                    int ldc, int M, int N, int K, int units_total, int epi,
                                                    FusedNorm fused) {
  extern __shared__ __attribute__((aligned(16))) unsigned char smem[];
  constexpr int ROWS = MT * 16;
  bf16* As = reinterpret_cast<bf16*>(smem);                                            // [2][ROWS][SK_LD]
  float* ot = reinterpret_cast<float*>(smem + 2 * ROWS * SK_LD * sizeof(bf16));        // [ROWS][OT_LD]
  __shared__ float rfac[ROWS];                 // the rows' norm factors (1 where no norm is folded in)
  const int tid = threadIdx.x, lane = tid & 63, wid = tid >> 6;

  const int r16 = lane & 15, kq = (lane >> 4) * 8;
  constexpr int WSTEP = TILED ? 512 : 32;
  const bool pair = epi == EPI_SWIGLU;
  // a unit is 32 weight rows: 32 outputs, or (pair) 16 gate rows and the 16 up rows of the same outputs
  const int u_begin = (int)((long)blockIdx.x * units_total / gridDim.x);
  const int u_end = (int)((long)(blockIdx.x + 1) * units_total / gridDim.x);
  const int n_u = u_end - u_begin;
  if (n_u <= 0) return;
  const int n_pass = (2 * n_u + PANEL_TILES - 1) / PANEL_TILES;
  const int per_u = (n_u + n_pass - 1) / n_pass;          // units of a pass (the last may have fewer)
  const int nch = K / KC;
  // what this lane reads for slot j of pass p, as a pointer at chunk 0
  auto slot_ptr = [&](int p, int j) -> const bf16* {
    if (p >= n_pass) return W;                             // behind the last pass: dropped
    const int cnt = 2 * min(per_u, n_u - p * per_u);       // tiles of the pass
    const int t = wid + 8 * j;
    if (t >= cnt) return W;                                // no tile
    const int u = u_begin + p * per_u + (t >> 1), which = t & 1;
    const int row0 = pair ? (u >> 1) * 64 + (u & 1) * 16 + 32 * which : u * 32 + 16 * which;
    return w_operand<TILED>(W, ldw, K, min(row0 + r16, N - 1), kq);
  };
  // staging: this thread handles rows i * 16 + tid / 32, k (tid % 32) * 8 of a chunk
  const int sk = (tid & 31) * 8;
  const bf16* src[MT];
#pragma unroll
  for (int i = 0; i < MT; ++i) src[i] = A + (size_t)min(i * 16 + (tid >> 5), M - 1) * lda + sk;
  bf16x8 stage[MT];
  auto load_stage = [&](int k0) {
#pragma unroll
    for (int i = 0; i < MT; ++i) stage[i] = *reinterpret_cast<const bf16x8*>(src[i] + k0);
  };
  auto store_stage = [&](int buf) {
#pragma unroll
    for (int i = 0; i < MT; ++i)
      *reinterpret_cast<bf16x8*>(&As[(buf * ROWS + i * 16 + (tid >> 5)) * SK_LD + sk]) = stage[i];
  };

  const bf16* wp[2] = {slot_ptr(0, 0), slot_ptr(0, 1)};
  bf16x8 wr[2][KC / 32];
  load_stage(0);
  // the rows' norm factors: wave w has rows w, w + 8, ...  Their partial sums are asked for between
  // the first activations and the first weights and used behind the activations' staging, so that
  // nothing the weight stream needs waits for them.
  int frow[2 * MT];
  float ffac[2 * MT];
#pragma unroll
  for (int i = 0; i < 2 * MT; ++i) frow[i] = fused.in_ssq ? wid + 8 * i : -1;
  RowSums<2 * MT> fsums;
  fsums.ask(fused, frow, M, lane);
  __builtin_amdgcn_sched_barrier(0);
#pragma unroll
  for (int s = 0; s < KC / 32; ++s) {
    wr[0][s] = load_weights<TILED>(wp[0] + s * WSTEP);
    wr[1][s] = load_weights<TILED>(wp[1] + s * WSTEP);
  }
  __builtin_amdgcn_sched_barrier(0);
  store_stage(0);
  fsums.factors(fused, frow, M, K, lane, ffac);
  if (lane == 0)
#pragma unroll
    for (int i = 0; i < 2 * MT; ++i) rfac[wid + 8 * i] = ffac[i];
  __syncthreads();
  floatx4 acc[2][MT];
#pragma unroll
  for (int j = 0; j < 2; ++j)
#pragma unroll
    for (int i = 0; i < MT; ++i) acc[j][i] = floatx4{0.f, 0.f, 0.f, 0.f};
  int buf = 0, pass = 0, kc = 0;
  const int total = n_pass * nch;
  for (int t = 0; t < total; ++t) {
    // the next step: the pass's next chunk, or chunk 0 of the next pass
    const bool last_chunk = kc + 1 == nch;
    const int kn = last_chunk ? 0 : (kc + 1) * KC;
    const bf16* wnext[2];
#pragma unroll
    for (int j = 0; j < 2; ++j) wnext[j] = last_chunk ? slot_ptr(pass + 1, j) : wp[j];
    load_stage(kn);
    __builtin_amdgcn_sched_barrier(0);
    const bf16* as = As + buf * ROWS * SK_LD;
#pragma unroll
    for (int s = 0; s < KC / 32; ++s) {
      bf16x8 a[MT];
#pragma unroll
      for (int i = 0; i < MT; ++i)
        a[i] = *reinterpret_cast<const bf16x8*>(&as[(i * 16 + r16) * SK_LD + s * 32 + kq]);
#pragma unroll
      for (int j = 0; j < 2; ++j) {
#pragma unroll
        for (int i = 0; i < MT; ++i)
          acc[j][i] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a[i], wr[j][s], acc[j][i], 0, 0, 0);
        wr[j][s] = load_weights<TILED>(wnext[j] + ((kn >> 5) + s) * WSTEP);
        __builtin_amdgcn_sched_barrier(0);      // use a register, then refill it, in this order
      }
    }
    store_stage(buf ^ 1);
    buf ^= 1;
    __syncthreads();        // the next chunk is staged
    if (!last_chunk) {
      ++kc;
      continue;
    }
    // ---- end of a pass
    const int cnt = 2 * min(per_u, n_u - pass * per_u);
    // D[m][n]: n = lane % 16, m = 4 (lane / 16) + r
#pragma unroll
    for (int j = 0; j < 2; ++j) {
      const int tl = wid + 8 * j;
      if (tl < cnt) {
#pragma unroll
        for (int i = 0; i < MT; ++i)
#pragma unroll
          for (int r = 0; r < 4; ++r)
            ot[(i * 16 + (lane >> 4) * 4 + r) * OT_LD + tl * 16 + r16] = acc[j][i][r];
      }
#pragma unroll
      for (int i = 0; i < MT; ++i) acc[j][i] = floatx4{0.f, 0.f, 0.f, 0.f};
    }
    __syncthreads();        // the tile is whole; the next pass writes it behind its own barriers
    {
      const int c = tid & 255;
      const int u0 = u_begin + pass * per_u;
      if (pair) {
        const int col = u0 * 16 + c;                       // unit c / 16 holds gate at 32 (c / 16), up 16 further
        if (c < cnt * 8 && col < ldc) {
          const int o = (c >> 4) * 32 + (c & 15);
          for (int m = tid >> 8; m < M; m += 2)
            ((bf16*)C)[(size_t)m * ldc + col] = (bf16)swiglu_f(ot[m * OT_LD + o] * rfac[m], ot[m * OT_LD + o + 16] * rfac[m],
                                                                    bias);
        }
      } else {
        const int col = u0 * 32 + c;
        if (c < cnt * 16 && col < N) {
          const float b = bias ? bias[col] : 0.f;
          for (int m = tid >> 8; m < M; m += 2) store_out(C, ldc, m, col, ot[m * OT_LD + c] * rfac[m] + b, epi, bias, N);
        }
      }
    }
    wp[0] = wnext[0];
    wp[1] = wnext[1];
    ++pass;
    kc = 0;
  }
}

// ---- one tile row against a wide matrix, a block per CU over the whole of K
// A block takes RA rows (at least M) and 32 J weight rows and copies k tiles of both straight into LDS, STAGES of them: what
// bounds it is the stream of weights and, from 100 rows on, how much a CU's copies bring in at once (some 55 GB/s of weights from
// memory and activations from L2 together), so rows past M are not copied (lanes switched off; the copies still count), the
// weight rows are cut to the number of CUs (tiles of 160 for 37,888: 237 blocks where tiles of 256 make 148), and the results of
// a block meet in LDS, where gates and ups of a SwiGLU pair up whichever waves held them.
// TURNS: the two waves of a SIMD in turns, one reading a k tile's fragments while the other multiplies (one group of waves a half
// k tile behind the other); without, all read and all multiply.
// PAIR: SwiGLU, in a kernel of its own: every block runs its epilogue once, so what it takes is also the fetch of its code.
// SwiGLU of 37,888 x 3,584: 64 rows 50.8 us (5.3 TB/s of weights; `panel_kernel` 58.7), 100 rows 55.6 (tiles of 128 x 256 66.7),
// without TURNS 2 us more.  33,000 x 512, bfloat16 results, 128 rows: 17.8 us with 2-byte stores, 15.7 with 8-byte ones.
template <int I, int J, int RA, int STAGES>
struct PanelTile {
  static constexpr int WM = 4, WN = 2, BN = 32 * J, P = (RA + BN) / 8, L = (P + 7) / 8, ST = (RA + BN) * DMA_BK * 2, OLD = BN + 4;
  static constexpr int LDS = STAGES * ST > RA * OLD * 4 ? STAGES * ST : RA * OLD * 4;
  static_assert(RA <= 16 * I * WM && RA % 8 == 0 && LDS <= 160 * 1024, "the rows fit the waves, the stages LDS");
};

template <int I, int J, int RA, int STAGES, bool TURNS, bool PAIR>
__global__ __launch_bounds__(512, 2) void panel_dma_kernel(const bf16* __restrict__ A, int lda, const bf16* __restrict__ W, int ldw,
                                                           const float* __restrict__ bias, void* __restrict__ C, int ldc, int M, int N,
                                                           int K, int epi, bool tiled, const float* __restrict__ in_ssq, int in_parts,
                                                           float in_eps) {
  using T = PanelTile<I, J, RA, STAGES>;
  constexpr int WM = T::WM, BN = T::BN, P = T::P, L = T::L, ST = T::ST, ROW = DMA_BK * 2;
  extern __shared__ __attribute__((aligned(16))) unsigned char smem[];      // [stage][RA rows of A, BN rows of W][64]
  int at = blockIdx.x;
  {
    const int n = gridDim.x, per = n / 8, rem = n % 8, x = at % 8;          // (neighbours on one die)
    at = x * per + min(x, rem) + at / 8;
  }
  const int lane = threadIdx.x & 63, wid = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int wm = wid % WM, wn = wid / WM, fr = lane & 15, fk = lane >> 4;
  // the block's weight rows: units u0 .. u0 + J - 1 of 32; of a pair (16 gate rows and the 16 up rows of the same outputs) the gates
  // of all units first, then the ups
  const int u0 = at * J;
  auto weight_row = [&](int r) {
    if (!PAIR) return u0 * 32 + r;
    const int c = r >> 4, u = u0 + c % J;
    return (u >> 1) * 64 + (u & 1) * 16 + (c / J) * 32 + (r & 15);
  };
  floatx4 acc[I][J];
#pragma unroll
  for (int i = 0; i < I; ++i)
#pragma unroll
    for (int j = 0; j < J; ++j) acc[i][j] = floatx4{0.f, 0.f, 0.f, 0.f};
  // the rows' partial sums of squares are asked for here and added up behind the products, eight lanes a row (products of more than 64
  // rows have none)
  constexpr int SUMS = (RA + 63) / 64;
  LanesSum<8, SUMS == 1 ? 4 : 1> sums[SUMS];
  auto part_row = [&](int q) {
    return in_ssq ? in_ssq + (size_t)min(q * 64 + wid * 8 + (lane >> 3), M - 1) * in_parts : nullptr;      // (rows past M: not stored)
  };
#pragma unroll
  for (int q = 0; q < SUMS; ++q) sums[q].ask(part_row(q), in_parts, lane & 7);
  __builtin_amdgcn_sched_barrier(0);
  // what a wave copies: pieces wid, 8 + wid, ... of 8 rows (chunk c of a row at position c ^ ((row >> 1) & 7))
  const unsigned lds0 = (unsigned)(uintptr_t)smem;
  unsigned g[L], dst[L];
  unsigned long long lanes[L];
#pragma unroll
  for (int q = 0; q < L; ++q) {
    const int p = q * 8 + wid, r = p * 8 + (lane >> 3), c = (lane & 7) ^ ((r >> 1) & 7);
    const bool of_a = p * 8 < RA;
    const int row = of_a ? r : weight_row(r - RA);
    lanes[q] = __builtin_amdgcn_ballot_w64(p < P && row < (of_a ? M : N));
    g[q] = of_a ? ((unsigned)min(row, M - 1) * (unsigned)lda + c * 8) * 2u : w_copy_at(min(row, N - 1), ldw, c, tiled);
    dst[q] = lds0 + min(p, P - 1) * 1024;
  }
  const int nkt = K / DMA_BK;
  auto copy = [&](int kt, int st) {
    const int k = kt * DMA_BK, kw = tiled ? k * 16 : k;
    const bool on = kt < nkt;                                // (else the copies count, and move nothing)
#pragma unroll
    for (int q = 0; q < L; ++q) {
      const unsigned to = __builtin_amdgcn_readfirstlane(dst[q] + st * ST);
      if ((q * 8 + wid) * 8 < RA) dma16_lanes<false>(A + k, g[q], to, on ? lanes[q] : 0);
      else dma16_lanes<true>(W + kw, g[q], to, on ? lanes[q] : 0);
    }
  };
  const int sw = (fr >> 1) & 7;
  bf16x8 fa[2][I], fw[2][J];
  auto read = [&](int st) {
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      const int pos = ((4 * h + fk) ^ sw) * 16;
      const unsigned char* s = smem + st * ST + fr * ROW + pos;
#pragma unroll
      for (int i = 0; i < I; ++i) fa[h][i] = *reinterpret_cast<const bf16x8*>(s + min((wm * I + i) * 16, RA - 16) * ROW);
#pragma unroll
      for (int j = 0; j < J; ++j) fw[h][j] = *reinterpret_cast<const bf16x8*>(s + (RA + (wn * J + j) * 16) * ROW);
    }
  };
  auto multiply = [&]() {
#pragma unroll
    for (int h = 0; h < 2; ++h)
#pragma unroll
      for (int i = 0; i < I; ++i)
#pragma unroll
        for (int j = 0; j < J; ++j) acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(fw[h][j], fa[h][i], acc[i][j], 0, 0, 0);
  };
#pragma unroll
  for (int t = 0; t < STAGES - 1; ++t) copy(t, t);
  int st = 0;
  if constexpr (TURNS) {
    // Waves w and w + 4 share a SIMD.  A stage is set out again in a group's read slot of the tile behind it: both groups have
    // its fragments in registers then (lgkmcnt(0) in front of the barriers between).  Tile kt + 1 has landed for every wave at
    // the end of the second group's read slot of tile kt, which is the first one's product slot.
    const bool second = wid >= 4;
    dma_wait<(STAGES - 2) * L>();
    dma_meet();
    if (second) dma_meet();
    for (int kt = 0; kt < nkt; ++kt) {
      read(st);
      __builtin_amdgcn_sched_barrier(0);
      copy(kt + STAGES - 1, st == 0 ? STAGES - 1 : st - 1);
      st = st == STAGES - 1 ? 0 : st + 1;
      if (second) dma_wait<(STAGES - 2) * L>();
      else asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
      dma_meet();
      __builtin_amdgcn_s_setprio(1);
      multiply();
      __builtin_amdgcn_s_setprio(0);
      if (!second) dma_wait<(STAGES - 2) * L>();
      dma_meet();
    }
    if (!second) dma_meet();
  } else {
    for (int kt = 0; kt < nkt; ++kt) {
      dma_wait<(STAGES - 2) * L>();                          // tile kt is here, and the one before in every wave's registers
      dma_meet();
      copy(kt + STAGES - 1, st == 0 ? STAGES - 1 : st - 1);
      read(st);
      multiply();
      st = st == STAGES - 1 ? 0 : st + 1;
    }
  }
  dma_wait<0>();
  dma_meet();
  // the results, [RA][BN + 4]; D: the lane's row is lane % 16, its columns 4 (lane / 16) + e
  float* out = reinterpret_cast<float*>(smem);
  __shared__ float fac[RA];
#pragma unroll
  for (int q = 0; q < SUMS; ++q) {
    const int r = q * 64 + wid * 8 + (lane >> 3);
    const float t = sums[q].add(part_row(q), in_parts, lane & 7);
    if ((lane & 7) == 0 && r < RA) fac[r] = in_ssq ? 1.0f / sqrtf(t / (float)K + in_eps) : 1.0f;
  }
#pragma unroll
  for (int i = 0; i < I; ++i)
#pragma unroll
    for (int j = 0; j < J; ++j)
      if ((wm * I + i) * 16 < RA) {
        const floatx4 v = acc[i][j];
        *reinterpret_cast<float4*>(out + ((wm * I + i) * 16 + fr) * T::OLD + (wn * J + j) * 16 + fk * 4) = float4{v[0], v[1], v[2], v[3]};
      }
  __syncthreads();
  if constexpr (PAIR) {
    const bool vec = ldc % 4 == 0 && (uintptr_t)C % 8 == 0;
    auto gated = [&](auto act) {
      for (int x = threadIdx.x; x < M * 4 * J; x += 512) {
        const int r = x / (4 * J), c = (x % (4 * J)) * 4, col = u0 * 16 + c;
        const float4 gt = *reinterpret_cast<const float4*>(out + r * T::OLD + c), up = *reinterpret_cast<const float4*>(out + r * T::OLD + BN / 2 + c);
        const float f = fac[r];
        const bf16x4 v = {(bf16)act(gt.x * f, up.x * f), (bf16)act(gt.y * f, up.y * f), (bf16)act(gt.z * f, up.z * f), (bf16)act(gt.w * f, up.w * f)};
        bf16* o = (bf16*)C + (size_t)r * ldc + col;
        if (vec && col + 4 <= ldc) *reinterpret_cast<bf16x4*>(o) = v;
        else
#pragma unroll
          for (int e = 0; e < 4; ++e)
            if (col + e < ldc) o[e] = v[e];
      }
    };
    if (bias) {
      const float limit = *bias;
      gated([=](float gt, float up) { return clamped_gate(gt, up, limit); });
    } else {
      gated([](float gt, float up) { return swiglu_f(gt, up, nullptr); });
    }
    return;
  }
  const bool half = epi == EPI_BF16 || epi == EPI_XIELU || epi == EPI_RELU2;
  const bool vec = ldc % 4 == 0 && (uintptr_t)C % (half ? 8 : 16) == 0;
  for (int x = threadIdx.x; x < M * (BN / 4); x += 512) {
    const int r = x / (BN / 4), c = (x % (BN / 4)) * 4, n = u0 * 32 + c;
    if (n >= N) continue;
    const float4 v4 = *reinterpret_cast<const float4*>(out + r * T::OLD + c);
    float v[4] = {v4.x, v4.y, v4.z, v4.w};
#pragma unroll
    for (int e = 0; e < 4; ++e) v[e] = v[e] * fac[r] + (bias && n + e < N ? bias[n + e] : 0.f);
    if (vec && n + 4 <= N && half) {
      bf16x4 h;
#pragma unroll
      for (int e = 0; e < 4; ++e) h[e] = (bf16)(epi == EPI_XIELU ? xielu_f(v[e], bias[N], bias[N + 1]) : epi == EPI_RELU2 ? relu2_f(v[e]) : v[e]);
      *reinterpret_cast<bf16x4*>((bf16*)C + (size_t)r * ldc + n) = h;
    } else if (vec && n + 4 <= N) {
      float4* o = reinterpret_cast<float4*>((float*)C + (size_t)r * ldc + n);
      float4 old = epi == EPI_ACC_F32 ? *o : float4{0.f, 0.f, 0.f, 0.f};
      *o = float4{old.x + v[0], old.y + v[1], old.z + v[2], old.w + v[3]};
    } else {
#pragma unroll
      for (int e = 0; e < 4; ++e)
        if (n + e < N) store_out(C, ldc, r, n + e, v[e], epi, bias, N);
    }
  }
}

template <int I, int J, int RA, int STAGES, bool TURNS>
int launch_panel_dma(const bf16* A, int lda, const bf16* W, int ldw, const float* bias, void* C, int ldc, int M, int N, int K, int epi,
                     const FusedNorm& fused, bool tiled, hipStream_t stream) {
  using T = PanelTile<I, J, RA, STAGES>;
  auto run = [&](auto PAIR) {
    auto kern = panel_dma_kernel<I, J, RA, STAGES, TURNS, decltype(PAIR)::value>;
    static bool configured = false;
    if (!configured) {
      const hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void*>(kern), hipFuncAttributeMaxDynamicSharedMemorySize, T::LDS);
      if (e != hipSuccess) return (int)e;
      configured = true;
    }
    kern<<<((N + 31) / 32 + J - 1) / J, 512, T::LDS, stream>>>(A, lda, W, ldw, bias, C, ldc, M, N, K, epi, tiled, fused.in_ssq, fused.in_parts,
                                                                   fused.in_eps);
    return mf_launch_status();
  };
  return epi == EPI_SWIGLU ? run(std::true_type{}) : run(std::false_type{});
}

// The parts of a split are added in rounds of up to eight, a round's loads in flight together, in
// the order of the splits (a plain loop over a count that is not known here is left to run split
// by split, a trip to memory each).
template <int CNT>
__device__ __forceinline__ float add_parts(float v, const float* __restrict__ p, size_t stride) {
  float x[CNT];
#pragma unroll
  for (int j = 0; j < CNT; ++j) x[j] = p[(size_t)j * stride];
#pragma unroll
  for (int j = 0; j < CNT; ++j) v += x[j];
  return v;
}

__device__ __forceinline__ float sum_of_parts(const float* __restrict__ part, size_t stride, size_t at, int splits) {
  float v = 0.f;
  for (int s0 = 0; s0 < splits; s0 += 8) {
    const float* p = part + (size_t)s0 * stride + at;
    switch (min(8, splits - s0)) {
      case 8: v = add_parts<8>(v, p, stride); break;
      case 7: v = add_parts<7>(v, p, stride); break;
      case 6: v = add_parts<6>(v, p, stride); break;
      case 5: v = add_parts<5>(v, p, stride); break;
      case 4: v = add_parts<4>(v, p, stride); break;
      case 3: v = add_parts<3>(v, p, stride); break;
      case 2: v = add_parts<2>(v, p, stride); break;
      default: v = add_parts<1>(v, p, stride); break;
    }
  }
  return v;
}

__global__ __launch_bounds__(256) void skinny_reduce_kernel(const float* __restrict__ part,
                                                            const float* __restrict__ bias,
                                                            void* __restrict__ C, int ldc, int M, int N, int K,
                                                            int splits, int epi, FusedNorm fused) {
  const int n = blockIdx.x * 256 + threadIdx.x, m = blockIdx.y;
  const size_t stride = (size_t)M * N;
  const int frow[1] = {fused.in_ssq ? m : -1};
  float ffac[1];
  RowSums<1> fsums;
  fsums.ask(fused, frow, M, threadIdx.x & 63);
  fsums.factors(fused, frow, M, K, threadIdx.x & 63, ffac);
  const float rf = ffac[0];
  if (epi == EPI_SWIGLU) {       // n runs over the ldc outputs
    if (n >= ldc) return;
    const int ng = (n >> 5) * 64 + (n & 31);
    const float g = sum_of_parts(part, stride, (size_t)m * N + ng, splits);
    const float u = sum_of_parts(part, stride, (size_t)m * N + ng + 32, splits);
    ((bf16*)C)[(size_t)m * ldc + n] = (bf16)swiglu_f(g * rf, u * rf, bias);
    return;
  }
  float v = 0.f;                 // the output's new value (0 beyond the row's end)
  if (n < N) {
    v = sum_of_parts(part, stride, (size_t)m * N + n, splits) * rf + (bias ? bias[n] : 0.f);
    if (epi == EPI_XIELU) {
      ((bf16*)C)[(size_t)m * ldc + n] = (bf16)xielu_f(v, bias[N], bias[N + 1]);
    } else if (epi == EPI_BF16 || epi == EPI_RELU2) {
      ((bf16*)C)[(size_t)m * ldc + n] = (bf16)(epi == EPI_RELU2 ? relu2_f(v) : v);
    } else {
      float* c = (float*)C + (size_t)m * ldc + n;
      if (epi == EPI_ACC_F32) v += *c;
      *c = v;
    }
  }
  if (fused.out_g) {
    // for the norm that reads these rows next: bf16(x g), and this block's sum of x^2, the waves'
    // sums added in their order
    if (n < N) fused.out_xg[(size_t)m * N + n] = (bf16)(v * fused.out_g[n]);
    __shared__ float wsum[4];
    float sq = v * v;
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) sq += __shfl_xor(sq, o, MF_WAVE);
    if ((threadIdx.x & 63) == 0) wsum[threadIdx.x >> 6] = sq;
    __syncthreads();
    if (threadIdx.x == 0) fused.out_ssq[(size_t)m * fused.out_parts + blockIdx.x] = ((wsum[0] + wsum[1]) + wsum[2]) + wsum[3];
    // (a row's places past the runs, where it has more of them: zero)
    if (blockIdx.x == 0)
      for (int p = gridDim.x + threadIdx.x; p < fused.out_parts; p += blockDim.x) fused.out_ssq[(size_t)m * fused.out_parts + p] = 0.f;
  }
}

// The same for rows whose length is a multiple of 4 (16-byte aligned parts, bias and output): a
// thread adds up four neighbouring outputs, a wave a run of 256 columns (so that a run's sum of
// squares is one wave's and needs no barrier), a block four runs.  A quarter of the blocks and of
// the loads of the kernel above, which is what its time is made of.
__global__ __launch_bounds__(256) void skinny_reduce4_kernel(const float* __restrict__ part,
                                                             const float* __restrict__ bias,
                                                             void* __restrict__ C, int ldc, int M, int N, int K,
                                                             int splits, int epi, FusedNorm fused) {
  const int run = blockIdx.x * 4 + (threadIdx.x >> 6);       // of 256 columns
  const int n = run * 256 + (threadIdx.x & 63) * 4, m = blockIdx.y;
  if (run * 256 >= N) return;                                // (whole waves leave: the shuffles below stay among those that stay)
  const size_t stride = (size_t)M * N;
  const int frow[1] = {fused.in_ssq ? m : -1};
  float ffac[1];
  RowSums<1> fsums;
  fsums.ask(fused, frow, M, threadIdx.x & 63);
  float4 v = float4{0.f, 0.f, 0.f, 0.f};
  const bool in = n < N;                                     // N in fours: all four inside, or none
  if (in) {
    const float* p = part + (size_t)m * N + n;
    for (int s0 = 0; s0 < splits; s0 += 8) {                 // eight parts' loads in flight together, added in their order
      float4 x[8];
#pragma unroll
      for (int j = 0; j < 8; ++j)
        x[j] = s0 + j < splits ? *reinterpret_cast<const float4*>(p + (size_t)(s0 + j) * stride) : float4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int j = 0; j < 8; ++j) { v.x += x[j].x; v.y += x[j].y; v.z += x[j].z; v.w += x[j].w; }
    }
  }
  fsums.factors(fused, frow, M, K, threadIdx.x & 63, ffac);
  if (in) {
    const float rf = ffac[0];
    const float4 b = bias ? *reinterpret_cast<const float4*>(bias + n) : float4{0.f, 0.f, 0.f, 0.f};
    v = float4{v.x * rf + b.x, v.y * rf + b.y, v.z * rf + b.z, v.w * rf + b.w};
    if (epi == EPI_XIELU) {
      const float ap = bias[N], an = bias[N + 1];
      bf16* c = (bf16*)C + (size_t)m * ldc + n;
      c[0] = (bf16)xielu_f(v.x, ap, an); c[1] = (bf16)xielu_f(v.y, ap, an);
      c[2] = (bf16)xielu_f(v.z, ap, an); c[3] = (bf16)xielu_f(v.w, ap, an);
    } else if (epi == EPI_RELU2) {
      bf16* c = (bf16*)C + (size_t)m * ldc + n;
      c[0] = (bf16)relu2_f(v.x); c[1] = (bf16)relu2_f(v.y); c[2] = (bf16)relu2_f(v.z); c[3] = (bf16)relu2_f(v.w);
    } else if (epi == EPI_BF16) {
      bf16* c = (bf16*)C + (size_t)m * ldc + n;
      c[0] = (bf16)v.x; c[1] = (bf16)v.y; c[2] = (bf16)v.z; c[3] = (bf16)v.w;
    } else {
      float4* c = reinterpret_cast<float4*>((float*)C + (size_t)m * ldc + n);
      if (epi == EPI_ACC_F32) { const float4 o = *c; v = float4{v.x + o.x, v.y + o.y, v.z + o.z, v.w + o.w}; }
      *c = v;
    }
  }
  if (fused.out_g) {
    if (in) {
      const float4 g = *reinterpret_cast<const float4*>(fused.out_g + n);
      bf16* xg = fused.out_xg + (size_t)m * N + n;
      xg[0] = (bf16)(v.x * g.x); xg[1] = (bf16)(v.y * g.y); xg[2] = (bf16)(v.z * g.z); xg[3] = (bf16)(v.w * g.w);
    }
    float sq = ((v.x * v.x + v.y * v.y) + v.z * v.z) + v.w * v.w;
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) sq += __shfl_xor(sq, o, MF_WAVE);
    if ((threadIdx.x & 63) == 0 && run < (N + 255) / 256) fused.out_ssq[(size_t)m * fused.out_parts + run] = sq;
    if (blockIdx.x == 0 && threadIdx.x < 64)                 // (a row's places past its runs, where it has more of them: zero)
      for (int p = (N + 255) / 256 + threadIdx.x; p < fused.out_parts; p += 64) fused.out_ssq[(size_t)m * fused.out_parts + p] = 0.f;
  }
}

// The kernel that adds the parts of a K split into the residual stream and norms the new rows for the product that reads
// them next (more than 64 rows, where that product takes them normed): a block a row, which it holds in registers between
// the sum of squares and the scaling.  The additions are those of `skinny_reduce4_kernel` and the norm that of
// `rmsnorm_kernel`, in their order.  One launch for two, and the rows are not read again: 203 rows of 3,584 values in 9
// parts 6.6 + 4.7 us as two kernels, 7.5 as this one; 2,048 rows in two parts 20.9 + 10.2 and 23.4.
template <int KEEP, int NT>
__global__ __launch_bounds__(NT) void reduce_norm_kernel(const float* __restrict__ part, const float* __restrict__ bias,
                                                          float* __restrict__ C, int ldc, int M, int N, int splits, int accumulate,
                                                          const float* __restrict__ g, float eps, bf16* __restrict__ normed) {
  __shared__ float scratch[NT / 64];
  extern __shared__ __attribute__((aligned(16))) float row[];      // [N] (more than 256 threads)
  const int m = blockIdx.x;
  const size_t stride = (size_t)M * N;
  const float* p = part + (size_t)m * N;
  float* c = C + (size_t)m * ldc;
  float4 v[KEEP];
  float ss = 0.f;
  auto squares = [&](const float4& x) {
    ss = fmaf(x.x, x.x, ss);
    ss = fmaf(x.y, x.y, ss);
    ss = fmaf(x.z, x.z, ss);
    ss = fmaf(x.w, x.w, ss);
  };
#pragma unroll
  for (int q = 0; q < KEEP; ++q) {
    const int n = (q * NT + threadIdx.x) * 4;
    v[q] = float4{0.f, 0.f, 0.f, 0.f};
    if (n < N) {
      const float4 old = accumulate ? *reinterpret_cast<const float4*>(c + n) : v[q];
      for (int s0 = 0; s0 < splits; s0 += 8) {               // eight parts' loads in flight together, added in their order
        float4 x[8];
#pragma unroll
        for (int j = 0; j < 8; ++j)
          x[j] = s0 + j < splits ? *reinterpret_cast<const float4*>(p + (size_t)(s0 + j) * stride + n) : float4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int j = 0; j < 8; ++j) { v[q].x += x[j].x; v[q].y += x[j].y; v[q].z += x[j].z; v[q].w += x[j].w; }
      }
      if (bias) {
        const float4 b = *reinterpret_cast<const float4*>(bias + n);
        v[q] = float4{v[q].x + b.x, v[q].y + b.y, v[q].z + b.z, v[q].w + b.w};
      }
      if (accumulate) v[q] = float4{v[q].x + old.x, v[q].y + old.y, v[q].z + old.z, v[q].w + old.w};
      *reinterpret_cast<float4*>(c + n) = v[q];
    }
    if (NT == 256) squares(v[q]);
    else if (n < N) *reinterpret_cast<float4*>(row + n) = v[q];
  }
  if constexpr (NT > 256) {                                  // in the order in which 256 threads add them up
    __syncthreads();
    if (threadIdx.x < 256)
      for (int n = threadIdx.x * 4; n < N; n += 1024) squares(*reinterpret_cast<const float4*>(row + n));
  }
  ss = block_sum<NT>(ss, scratch);
  const float scale = 1.0f / sqrtf(ss / (float)N + eps);
#pragma unroll
  for (int q = 0; q < KEEP; ++q) {
    const int n = (q * NT + threadIdx.x) * 4;
    if (n < N) {
      const float4 w = *reinterpret_cast<const float4*>(g + n);
      *reinterpret_cast<bf16x4*>(normed + (size_t)m * N + n) =
          bf16x4{(bf16)(v[q].x * scale * w.x), (bf16)(v[q].y * scale * w.y), (bf16)(v[q].z * scale * w.z), (bf16)(v[q].w * scale * w.w)};
    }
  }
}

constexpr int REDUCE_NORM_MAX = 256 * 4 * 16;                // a row's values that a block holds

int launch_reduce_norm(const float* part, const float* bias, float* C, int ldc, int M, int N, int splits, int accumulate,
                       const float* g, float eps, bf16* normed, hipStream_t stream) {
  auto run = [&](auto KEEP, auto NT) {
    reduce_norm_kernel<decltype(KEEP)::value, decltype(NT)::value>
        <<<M, decltype(NT)::value, NT > 256 ? N * sizeof(float) : 0, stream>>>(part, bias, C, ldc, M, N, splits, accumulate, g, eps, normed);
  };
  auto with = [&](auto NT) {                                 // the values of a row that a thread holds, in fours
    const int keep = (N + NT * 4 - 1) / (NT * 4);
    if (keep <= 1) run(std::integral_constant<int, 1>{}, NT);
    else if (keep <= 2) run(std::integral_constant<int, 2>{}, NT);
    else if (keep <= 4) run(std::integral_constant<int, 4>{}, NT);
    else if (NT == 256 && keep <= 8) run(std::integral_constant<int, NT == 256 ? 8 : 4>{}, NT);
    else run(std::integral_constant<int, NT == 256 ? 16 : 4>{}, NT);
  };
  // Where no CU has two rows, a row's loads should all be on their way at once: 203 rows of 3,584 in 9 parts 9.9 us with 256
  // threads a row, 7.5 with 1,024.  With more rows the blocks of a CU do that for each other: 604 rows of 2,048 in 6 parts 8.1
  // and 8.5, 2,048 rows of 3,584 in 2 23.4 and 25.0; and of at most 1,024 values 256 threads ask for all at once as well (65 rows of
  // 896 with their product 9.4 us and 9.9).  1,024 threads hold the row in LDS, which a launch gives 64 KB of without being asked.
  const bool fits = N * sizeof(float) + 1024 / 64 * sizeof(float) <= 64 * 1024;
  if (M <= cu_count() && N > 1024 && fits) with(std::integral_constant<int, 1024>{});
  else with(std::integral_constant<int, 256>{});
  return mf_launch_status();
}

// adds the parts of a K split and runs the epilogue: the kernel in fours where the operands allow it
int launch_reduce(const float* part, const float* bias, void* C, int ldc, int M, int N, int K, int splits, int epi,
                  const FusedNorm& fused, hipStream_t stream) {
  const bool fours = epi != EPI_SWIGLU && N % 4 == 0 && ldc % 4 == 0 && (uintptr_t)part % 16 == 0 &&
                     (uintptr_t)bias % 16 == 0 && (uintptr_t)C % 16 == 0 && (uintptr_t)fused.out_g % 16 == 0 &&
                     (uintptr_t)fused.out_xg % 8 == 0;
  if (fours) {
    dim3 g4((N + 1023) / 1024, M);
    skinny_reduce4_kernel<<<g4, 256, 0, stream>>>(part, bias, C, ldc, M, N, K, splits, epi, fused);
  } else {
    dim3 g2(((epi == EPI_SWIGLU ? ldc : N) + 255) / 256, M);
    skinny_reduce_kernel<<<g2, 256, 0, stream>>>(part, bias, C, ldc, M, N, K, splits, epi, fused);
  }
  return mf_launch_status();
}

template <int MT, bool VEC>
int launch_skinny_v(const bf16* A, int lda, const bf16* W, const bf16* Wt, int ldw, const float* bias, void* C,
                    int ldc, float* part, int M, int N, int K, int splits, int k_per_split, int epi,
                    const FusedNorm& fused, hipStream_t stream) {
  constexpr int smem = 2 * MT * 16 * SK_LD * (int)sizeof(bf16);
  static bool configured = false;
  const bool tiled = VEC && Wt != nullptr;
  auto kern = tiled ? skinny_kernel<MT, VEC, VEC> : skinny_kernel<MT, VEC, false>;
  if (!configured) {
    hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void*>(skinny_kernel<MT, VEC, false>),
                                       hipFuncAttributeMaxDynamicSharedMemorySize, smem);
    if (e == hipSuccess)
      e = hipFuncSetAttribute(reinterpret_cast<const void*>(skinny_kernel<MT, VEC, VEC>),
                              hipFuncAttributeMaxDynamicSharedMemorySize, smem);
    if (e != hipSuccess) return (int)e;
    configured = true;
  }
  dim3 grid((N + 127) / 128, splits);
  const bool two_pass = splits > 1 || epi == EPI_SWIGLU;   // gate and up columns sit in different waves
  if (!two_pass && (fused.in_ssq || fused.out_g)) return MF_NOT_BUILT;     // the second kernel is what folds the norm in
  if (ring_takes(VEC, K, splits, k_per_split)) {
    constexpr int smem_ring = smem + MT * 16 * SR_LD * (int)sizeof(float);
    static bool ring_configured = false;
    if (!ring_configured) {
      hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void*>(skinny_ring_kernel<MT, false>),
                                         hipFuncAttributeMaxDynamicSharedMemorySize, smem_ring);
      if (e == hipSuccess)
        e = hipFuncSetAttribute(reinterpret_cast<const void*>(skinny_ring_kernel<MT, true>),
                                hipFuncAttributeMaxDynamicSharedMemorySize, smem_ring);
      if (e != hipSuccess) return (int)e;
      ring_configured = true;
    }
    if (Wt)
      skinny_ring_kernel<MT, true><<<grid, 512, smem_ring, stream>>>(A, lda, Wt, ldw, bias, C, ldc, two_pass ? part : nullptr,
                                                                     M, N, K, k_per_split, epi);
    else
      skinny_ring_kernel<MT, false><<<grid, 512, smem_ring, stream>>>(A, lda, W, ldw, bias, C, ldc, two_pass ? part : nullptr,
                                                                      M, N, K, k_per_split, epi);
  } else {
    kern<<<grid, 512, smem, stream>>>(A, lda, tiled ? Wt : W, ldw, bias, C, ldc, two_pass ? part : nullptr, M, N, K,
                                      k_per_split, epi);
  }
  int rc = mf_launch_status();
  if (rc == 0 && two_pass) rc = launch_reduce(part, bias, C, ldc, M, N, K, splits, epi, fused, stream);
  return rc;
}

template <int MT>
int launch_skinny(const bf16* A, int lda, const bf16* W, const bf16* Wt, int ldw, const float* bias, void* C,
                  int ldc, float* part, int M, int N, int K, int splits, int k_per_split, int epi, int vec_ok,
                  const FusedNorm& fused, hipStream_t stream) {
  return vec_ok ? launch_skinny_v<MT, true>(A, lda, W, Wt, ldw, bias, C, ldc, part, M, N, K, splits, k_per_split,
                                            epi, fused, stream)
                : launch_skinny_v<MT, false>(A, lda, W, nullptr, ldw, bias, C, ldc, part, M, N, K, splits,
                                             k_per_split, epi, fused, stream);
}

// The whole-K kernel for 17 to 64 rows, where the matrix is wide enough to give every CU at least
// 8 tiles; MF_NOT_BUILT (nothing launched) for any other shape.
template <int MT, bool TILED>
int launch_panel_mt(const bf16* A, int lda, const bf16* W, int ldw, const float* bias, void* C, int ldc, int M,
                    int N, int K, int epi, int grid, int units, const FusedNorm& fused, hipStream_t stream) {
  constexpr int smem = 2 * MT * 16 * SK_LD * (int)sizeof(bf16) + MT * 16 * OT_LD * (int)sizeof(float);
  static bool configured = false;
  if (!configured) {
    hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void*>(panel_kernel<MT, TILED>),
                                       hipFuncAttributeMaxDynamicSharedMemorySize, smem);
    if (e != hipSuccess) return (int)e;
    configured = true;
  }
  panel_kernel<MT, TILED><<<grid, 512, smem, stream>>>(A, lda, W, ldw, bias, C, ldc, M, N, K, units, epi, fused);
  return mf_launch_status();
}

int launch_panel(const bf16* A, int lda, const bf16* W, const bf16* Wt, int ldw, const float* bias, void* C, int ldc,
                 int M, int N, int K, int epi, const FusedNorm& fused, hipStream_t stream) {
  const int n_cu = cu_count();
  if (n_cu <= 0) return (int)hipErrorUnknown;
  const bool aligned = ldw % 8 == 0 && (uintptr_t)W % 16 == 0 && lda % 8 == 0 && (uintptr_t)A % 16 == 0;
  if (!panel_takes(M, N, K, aligned, epi, n_cu) || fused.out_g) return MF_NOT_BUILT;
  const int units = (N + 31) / 32;
  switch ((M + 15) / 16) {
    case 2:
      return Wt ? launch_panel_mt<2, true>(A, lda, Wt, ldw, bias, C, ldc, M, N, K, epi, n_cu, units, fused, stream)
                : launch_panel_mt<2, false>(A, lda, W, ldw, bias, C, ldc, M, N, K, epi, n_cu, units, fused, stream);
    case 3:
      return Wt ? launch_panel_mt<3, true>(A, lda, Wt, ldw, bias, C, ldc, M, N, K, epi, n_cu, units, fused, stream)
                : launch_panel_mt<3, false>(A, lda, W, ldw, bias, C, ldc, M, N, K, epi, n_cu, units, fused, stream);
    case 4:
      return Wt ? launch_panel_mt<4, true>(A, lda, Wt, ldw, bias, C, ldc, M, N, K, epi, n_cu, units, fused, stream)
                : launch_panel_mt<4, false>(A, lda, W, ldw, bias, C, ldc, M, N, K, epi, n_cu, units, fused, stream);
  }
  return MF_NOT_BUILT;
}

// ---- which tile kernel a product of many rows takes
// Variants: 2: 128 x 128 tiles through registers (two blocks a CU), 3: 64 x 64, 9: 256 x 256 through
// registers, and the direct-to-LDS kernel (aligned operands, K in 64s): 12 the largest tiles (256 x 256; SwiGLU products
// 256 x 192 where their rounds are the shorter), 15 256 x 192 (no SwiGLU), 13 the smaller ones (256 x 128, 128 x 256,
// 128 x 128 or 64 x 64).  With `splits` > 1 the K dimension is cut over blocks (variants 12 and 2, the latter with the smaller
// direct-to-LDS tiles where the operands allow) and skinny_reduce_kernel adds the parts.
struct TilePlan { int variant, splits, k_per_split; double us; };

// The direct-to-LDS kernels' tiles: blocks a CU, microseconds a k tile of 64 with every CU busy (random values, 2,048 rows
// at the 7B widths), and what a chip that is nearly empty takes of it (the smaller tiles are their own chains of waits).
struct DmaForm { int bm, bn, per_cu; double step_us, low; };
enum { FORM_256, FORM_192, FORM_128, FORM_128T, FORM_SMALL, FORM_TINY, N_FORMS };
constexpr DmaForm DMA_FORMS[N_FORMS] = {{256, 256, 1, 1.36, 0.7}, {256, 192, 1, 1.08, 0.7}, {256, 128, 1, 0.84, 0.9},
                                        {128, 256, 1, 0.84, 0.9}, {128, 128, 1, 0.62, 0.9}, {64, 64, 2, 0.56, 0.55}};
constexpr double ROUND_US = 5.;
constexpr int TINY_K = 3264;          // the longest K whose 64 x 64 tiles have the price of `form_us`

// The estimate behind the choice: a kernel's tiles go over its slots (blocks that fit the chip at
// once) in rounds; a round takes the product's k tiles of 64 times the variant's time per k tile, a last round that is
// not full somewhat less (fewer blocks pull on the fabric and on the power); a start, the epilogue's traffic, and for a K
// split the parts' way to memory and back come on top.
double rounds_us(long blocks, long slots, double step_us, long nkt, double round_us, double low = 0.7) {
  const long full = blocks / slots;
  const double fill = (double)(blocks % slots) / (double)slots;
  return ((double)nkt * step_us) * ((double)full + (fill > 0. ? low + (1. - low) * fill : 0.)) + round_us * (double)(full + (fill > 0.));
}

// (nkt: k tiles of a part; K: the whole product's)
double form_us(int form, int M, int N, int K, long nkt, int splits, long cu) {
  const DmaForm& f = DMA_FORMS[form];
  const long tiles = (long)((M + f.bm - 1) / f.bm) * ((N + f.bn - 1) / f.bn);
  if (form == FORM_TINY && K <= TINY_K) {
    // Blocks of four waves that start at once, two a CU: 0.27 us a k tile while no CU has two, soon 0.52
    // where some have, no more than the start that every plan pays, and 6 us for a round behind the first; of a K split the
    // second blocks' stores come late as well.  (Weights from memory, 64 x 64 whole, estimate / measured: 300 x 2,048 x 2,048
    // 13.6 / 12.1 us, 604 of them 22.5 / 18.9, 604 x 1,536 x 1,536 12.0 / 10.8, 604 x 1,152 x 896 8.9 / 6.7.  Priced like the large tiles
    // they lost to K split: 300 x 2,048 x 2,048 17.9, 65 x 8,192 x 2,048 15.7 where 64 x 64 take 12.6.)  The line is the product's own K, the same for whole and
    // cut: a line by the k tiles of all parts together gave this price to the whole product of 3,136 to 3,264 and the other one to its
    // cuts, which K in chunks of 256 takes past the line.  142 products at 3,136 and 3,264 so: 0.94 of the time of what that chose on
    // the average (88 x 896 x 3,200 13.1 us whole, 9.3 in 5 parts; SwiGLU of 203 x 1,536 x 3,136 the other way, 12.4 and 14.7), 0.86 of what
    // the large tiles' price for both chose.  Past it both have the large tiles' price.
    const long slots = cu * f.per_cu, blocks = tiles * splits, rest = blocks % slots;
    const double last = rest == 0 ? 0. : rest <= cu ? 0.27 : 0.36 + 0.16 * std::min(1., (double)(rest - cu) / 64.);
    return (double)nkt * ((double)(blocks / slots) * 0.53 + last) - 0.7 + 6. * (double)((blocks - 1) / slots) +
           (splits > 1 && blocks > cu ? 2.5 : 0.);
  }
  return rounds_us(tiles * splits, cu * f.per_cu, f.step_us, nkt, ROUND_US, f.low);
}

// the cheapest of the forms first .. last
int best_form(int first, int last, int M, int N, int K, long nkt, int splits, long cu) {
  int best = first;
  for (int f = first + 1; f <= last; ++f)
    if (form_us(f, M, N, K, nkt, splits, cu) < form_us(best, M, N, K, nkt, splits, cu)) best = f;
  return best;
}

// which tiles variant 12, 13 or 15, or variant 2 cut over K, runs
int dma_form(int variant, int M, int N, int K, int epi, long nkt, int splits, long cu) {
  switch (variant) {
    case 12: return epi == EPI_SWIGLU && splits == 1 ? best_form(FORM_256, FORM_192, M, N, K, nkt, 1, cu) : FORM_256;
    case 15: return FORM_192;
  }
  return best_form(FORM_128, FORM_TINY, M, N, K, nkt, splits, cu);
}

// A product's weights for the kernels that copy straight into LDS: the matrix, and its tiled copy where the caller has one (null: none).
// A copy of 8 rows by 64 k is eight whole lines of the one, K elements apart, and of the other two runs of four lines, with the runs of
// the neighbouring rows and k beside them, which memory gives faster (weights from memory, row-major / tiled: SwiGLU of 22,016 x 2,048, 40 rows
// 26.1 / 21.8 us, 64 rows 24.0 / 20.5, 100 rows 27.0 / 24.7; 37,888 x 3,584, 64 rows 53.5 / 51.0, 203 rows 73.3 / 72.1, 604 rows 166.1 / 163.1;
// 3,584 x 18,944, 604 rows in three parts 98.4 / 93.9; 4,608 x 3,584, 2,048 rows 63.9 / 61.2; level where many rows share the weights).
// Of 330 other products of 65 to 1,100 rows 0.975 of the time on average, 13 more than 2 % slower, none more than 6 % (6,144 x 8,192, 80
// rows 30.8 / 32.6), with no line between them; of 260 in 64 x 64 tiles 0.974, one shape slower (28,672 x 512, 17 rows 9.9 / 10.7).
// Not so 64 x 64 tiles of which no CU has two: their time is a chain of waits, with longer addresses in front of it
// (2,560 x 2,048, 100 rows 7.4 / 7.7 us, 203 rows 10.0 / 10.4; 1,152 x 896, 604 rows 6.8 / 7.0).
struct Weights {
  const bf16* w;
  const bf16* tiled;
  int ldw, K;
  Weights(const void* w_, const void* wt, int ldw_, int K_)
      : w((const bf16*)w_), tiled(wt && (uintptr_t)wt % 16 == 0 && K_ % DMA_BK == 0 ? (const bf16*)wt : nullptr), ldw(ldw_), K(K_) {}
  // from weight row n on (in 16s)
  Weights from(int n) const { return Weights(w + (size_t)n * ldw, tiled ? tiled + (size_t)n * K : nullptr, ldw, K); }
  const bf16* at(bool t) const { return t ? tiled : w; }
  int ld(bool t) const { return t ? K : ldw; }
};
bool tile64_reads_tiled(const Weights& w, int M, int N, int splits) {
  return w.tiled && (long)((M + 63) / 64) * ((N + 63) / 64) * splits > cu_count();
}

template <bool T>
int launch_form_of(int form, const bf16* A, int lda, const Weights& w, const float* bias, void* C, int ldc, int M, int N, int K,
                   int epi, hipStream_t stream, int splits, int k_per_split) {
  const bf16* W = w.at(T);
  const int ldw = w.ld(T);
  switch (form) {
    case FORM_256: return launch_tile_dma<256, 256, 2, T>(A, lda, W, ldw, bias, C, ldc, M, N, K, epi, stream, splits, k_per_split);
    case FORM_192: return launch_tile_dma<256, 192, 2, T>(A, lda, W, ldw, bias, C, ldc, M, N, K, epi, stream, splits, k_per_split);
    case FORM_128: return launch_tile_dma<256, 128, 3, T>(A, lda, W, ldw, bias, C, ldc, M, N, K, epi, stream, splits, k_per_split);
    case FORM_128T: return launch_tile_dma<128, 256, 3, T>(A, lda, W, ldw, bias, C, ldc, M, N, K, epi, stream, splits, k_per_split);
  }
  return form == FORM_SMALL ? launch_tile_step<128, 128, 2, 4, 4, false, false, false, T>(A, lda, W, ldw, bias, C, ldc, M, N, K, epi, stream, splits,
                                                                                          k_per_split, nullptr, 0)
                            : launch_tile64<false, T>(A, lda, W, ldw, bias, C, ldc, M, N, K, epi, stream, splits, k_per_split);
}
// (which of the two is known to the compiler: as an argument it cost products from the matrix 0.1 to 0.2 us, 896 x 896 of 100 rows 6.35 and 6.5)
int launch_form(int form, const bf16* A, int lda, const Weights& w, const float* bias, void* C, int ldc, int M, int N, int K,
                int epi, hipStream_t stream, int splits = 1, int k_per_split = 0) {
  return (form == FORM_TINY ? tile64_reads_tiled(w, M, N, splits) : w.tiled != nullptr)
             ? launch_form_of<true>(form, A, lda, w, bias, C, ldc, M, N, K, epi, stream, splits, k_per_split)
             : launch_form_of<false>(form, A, lda, w, bias, C, ldc, M, N, K, epi, stream, splits, k_per_split);
}

// A few weight rows past whole tiles (a gate beside q|k|v, a low-rank factor) can cost a whole round of them: 2,048 rows against
// 8,192 of 2,048 are 256 tiles of 256 x 256, a CU each, against 8,224 264.  Up to 64 of them are then a product of their own, in
// small tiles behind the large ones (variant 16).  The weight rows of the first product, or 0: none are left over, or the
// epilogue takes its columns together (SwiGLU) or its constants from behind the biases (xIELU).  (The square of relu, 2,048 x 8,200 x 4,096: 137 us
// in 256 x 192 tiles, 113 so.)
int main_rows(int N, int epi) {
  const int rest = N % 256;
  return N > 256 && rest > 0 && rest <= 64 && (epi == EPI_F32 || epi == EPI_ACC_F32 || epi == EPI_BF16 || epi == EPI_RELU2) ? N - rest : 0;
}

// by their columns where the tile has 256 rows
const char* form_name(int form, bool split) {
  static const char* names[N_FORMS][2] = {{"tile_dma_kernel<256>", "tile_dma_kernel<256>(split K)"},
                                          {"tile_dma_kernel<192>", "tile_dma_kernel<192>(split K)"},
                                          {"tile_dma_kernel<128>", "tile_dma_kernel<128>(split K)"},
                                          {"tile_dma_kernel<128,256>", "tile_dma_kernel<128,256>(split K)"},
                                          {"tile_step_kernel<128,128>", "tile_step_kernel<128,128>(split K)"},
                                          {"tile_step_kernel<64,64>", "tile_step_kernel<64,64>(split K)"}};
  return names[form][split];
}

int panel_dma_units(int M, int N, int K, int epi, int n_cu);

// What a product with a K of up to 3,072 whole costs beside its own kernel, where the parts of a split would be added by a kernel that
// runs in any case (`behind`): 1 the rotation, whose second way from memory a split saves, 2 the norm, else a kernel of its own
// (rmsnorm_kernel: 70 x 896 2.6 us, 604 x 2,048 4.2, 1,200 x 3,584 6.4).  (A longer K is priced without; so are more than 2.2 million
// results, whose parts cost more than they save: with the norm 1,700 x 2,048 x 1,024 24.0 us whole and 29.5 split.)
double whole_more(int M, int N, int K, int behind) {
  const double mn = (double)M * (double)N;
  return K > 3072 || mn > 2.2e6 || behind == 0 ? 0. : behind == 1 ? 4.5 : 3.2 + mn / 1e6;
}

// `tile_stream_kernel`'s tiles of 16 I rows, in microseconds with the kernel behind it: a k tile, what it takes more for the share of the chip and
// every 10,000 of K, a million results' way to memory and back for every part, and the rest of a whole product and of a cut one, alone, in front of
// the rotation and in front of the norm (least squares over 3,771 timings at 697 products of 129 to 2,048 rows against 512 to 11,008 of 896 to
// 28,672, weights and activations from memory: 4 % off on average).
struct StreamForm { int i; double step_us, wide_us, store_us, whole_us[3], cut_us[3]; };
constexpr StreamForm STREAM_FORMS[2] = {{6, 0.46, 0.025, 2.3, {3.4, 8.5, 8.3}, {7.5, 8.8, 7.6}},
                                        {8, 0.53, 0.035, 2.1, {4.6, 10.1, 10.4}, {8.6, 10.2, 8.9}}};
// The other plans' times over their prices at the same products, from the tiled copy with the kernel behind them, 3 to 8 % off: whole and cut;
// tiles of 256 and 256 x 128, of 128 x 128, of 64 x 64; alone, rotation, norm.
constexpr double OF_PRICE[2][3][3] = {{{0.88, 1.07, 0.98}, {0.78, 1.07, 0.89}, {0.95, 1.02, 0.93}},
                                      {{0.97, 1.03, 1.02}, {0.85, 0.90, 0.86}, {0.95, 1.00, 0.95}}};

TilePlan plan_tiles(int M, int N, int K, bool dma_ok, int epi, int n_cu, int behind = 0, bool tiled = false) {
  const long cu = n_cu > 0 ? n_cu : 1;
  const long nkt = (K + 63) / 64, chunks = (K + 255) / 256;
  const double mn = (double)M * (double)N;
  const double epi_us = (epi == EPI_ACC_F32 ? 8. : epi == EPI_F32 ? 4. : (epi == EPI_BF16 || epi == EPI_XIELU || epi == EPI_RELU2) ? 2. : 1.) * mn / 4e6;
  // The kernels through registers have costs of their own: a launch's epilogue is a chain (SwiGLU's stores 4 us, of 16 or 32
  // bits 7, a read and a store 25), the second kernel of a SwiGLU product adds its parts one value at a time, and rows that are
  // no whole 16 bytes are read in eights of single values.  1,888 products of K not in 64s, from 65 x 192 x 100 on: the choice is
  // 0.5 % from the best kernel on average; with the costs of the direct-to-LDS kernels 1.3 %, and SwiGLU of 200 rows against
  // 8,000 of 1,000 34.7 us in two parts for 21.2 whole.
  const double more_us = dma_ok ? whole_more(M, N, K, behind) : 0.;
  const double start_us = more_us + (dma_ok ? 4. : epi == EPI_ACC_F32 ? 25. : epi == EPI_SWIGLU ? 4. : 7.);
  const double slow = K % 8 ? 4. : 1.;
  auto tiles = [&](int bm, int bn) { return (long)((M + bm - 1) / bm) * ((N + bn - 1) / bn); };
  auto cut = [&](long parts, int& splits, int& per) {          // K in `parts` runs of whole chunks of 256
    const long c = (chunks + parts - 1) / parts;
    splits = (int)((chunks + c - 1) / c);
    per = (int)(c * 256);
  };
  auto parts_us = [&](int splits) {                            // the start of both kernels and the parts' way
    const double bytes = (double)(splits + 2) * mn * 4.;
    return dma_ok ? bytes / 6e6 + 8. : bytes / (epi == EPI_SWIGLU ? 3e6 : 8e6) + 14.25;
  };
  TilePlan best{0, 1, K, 1e30};
  auto offer = [&](int variant, int splits, int per, double us) {
    if (us < best.us) best = TilePlan{variant, splits, per, us};
  };
  auto form = [&](int variant, int splits, long steps) {
    return form_us(dma_form(variant, M, N, K, epi, steps, splits, cu), M, N, K, steps, splits, cu);
  };
  if (dma_ok) {
    if (M > 64 && panel_dma_units(M, N, K, epi, n_cu)) return TilePlan{13, 1, K, 0.};
    offer(12, 1, K, form(12, 1, nkt) + start_us + epi_us);
    offer(13, 1, K, form(13, 1, nkt) + start_us + epi_us);
    if (epi != EPI_SWIGLU) offer(15, 1, K, form(15, 1, nkt) + start_us + epi_us);
    if (const int n0 = main_rows(N, epi))
      offer(16, 1, K, form_us(best_form(0, N_FORMS - 1, M, n0, K, nkt, 1, cu), M, n0, K, nkt, 1, cu) +
                          form_us(best_form(FORM_128, FORM_TINY, M, N - n0, K, nkt, 1, cu), M, N - n0, K, nkt, 1, cu) + 2 * start_us - more_us + epi_us);
    // many rows against few weight rows and a long K (the down product of a prompt): K cut over
    // the big tiles, each part at least 2,048 of K
    if (epi != EPI_SWIGLU && M >= 768)
      for (long parts = 2; parts <= std::min<long>(8, K / 2048); ++parts) {
        int splits, per;
        cut(parts, splits, per);
        if (splits < 2) continue;
        offer(12, splits, per, form(12, splits, per / 64) + parts_us(splits));
      }
  } else {
    offer(9, 1, K, rounds_us(tiles(256, 256), cu, 2.1 * slow, nkt, 0.) + start_us + epi_us);
    offer(M <= 64 && tiles(128, 128) < 64 && epi != EPI_SWIGLU ? 3 : 2, 1, K,
          rounds_us(tiles(128, 128), 2 * cu, 1.45 * slow, nkt, 0.) + start_us + epi_us);
  }
  // a few hundred rows against a few thousand weight rows (some 50 tiles of 128 x 128, bound by
  // the weight stream): K over the chip, each part at least 512 of K
  const long t128 = tiles(128, 128);
  if (t128 < cu)
    for (long parts = 2; parts <= std::min(chunks / 2, (2 * cu) / std::max(1L, t128)); ++parts) {
      int splits, per;
      cut(parts, splits, per);
      if (splits < 2 || splits * t128 > 2 * cu) continue;
      const double us = dma_ok ? form(2, splits, per / 64) : rounds_us(t128 * splits, 2 * cu, 1.45 * slow, per / 64, 0.);
      offer(2, splits, per, us + parts_us(splits));
    }
  // `tile_stream_kernel`, while all its tiles are on the chip at once, in at most eight parts (more were level) of four k tiles and more on
  // average: where it takes 3 % less than the plan so far, both as they were timed.  160 of the 697
  // products go to it (see STREAM_FORMS), 0.980 of the time on average over all, eight of them 1 to 8 % slower than without; 420 others that the prices were not
  // made from: 0.987, 18 more than 2 % slower, none more than 6 %.  Whole prompts of 37 to 2,048 tokens, 896 to 3,584 wide: within 2 % of lines that
  // were drawn after such prompts.
  // Beyond the rows that the prices were made from a whole product in front of the norm has 2.6 us more for every 1,000 rows past 2,200: the norm's own
  // kernel, a workgroup a row (3,169 rows of 896 x 4,864 52.1 us in parts / 54.1 whole, 4,000 of 768 x 3,072 39.9 / 41.9, 3,372 of 1,000 x 2,816 40.7 /
  // 45.6; without the term 3 to 6 us under what they take).  Of 60 products of 2,049 to 5,710 rows against 512 to 1,024 of 768 to 4,864 that go to the kernel: 0.915
  // of the time on average, all but two faster; 2,161 x 640 x 2,560 20.6 / 22.8.
  // Not in the place of 64 x 64 tiles of a K past TINY_K (their price is another: 23 of the 697, level at best, 896 x 4,864 of 150 rows 13.1 and 15.0); in
  // front of the rotation a split only in the place of another split (level, and prompts of 450 tokens 1,536 wide 3,225 whole and 3,348 cut); not
  // for up to 128 rows (level: the weights' stream); not for a K below 768, which the prices were not made from and where they are mostly their rests
  // (1,400 x 1,536, with the norm: K 320 15.75 without and 17.15 with, 512 17.4 and 18.2, 768 19.1 and 18.2).
  const int used = !dma_ok ? -1 : best.variant == 16 ? FORM_128 : dma_form(best.variant, M, N, K, epi, best.k_per_split / 64, best.splits, cu);
  if (dma_ok && tiled && epi != EPI_SWIGLU && M > 128 && K >= 768 && !(used == FORM_TINY && K > TINY_K)) {
    const bool was_cut = best.splits > 1;
    double us = 0.97 * best.us * OF_PRICE[was_cut][used == FORM_TINY ? 2 : used == FORM_SMALL ? 1 : 0][behind];
    for (const StreamForm& f : STREAM_FORMS) {
      const long t = tiles(16 * f.i, 128);
      for (long parts = 1; parts <= 8 && t * parts <= cu && (parts == 1 || nkt >= 4 * parts); ++parts) {
        const long steps = (nkt + parts - 1) / parts, splits = (nkt + steps - 1) / steps;
        if (splits != parts || (splits > 1 && behind == 1 && !was_cut)) continue;
        const double own = (f.step_us + f.wide_us * (double)(t * splits) / (double)cu * (double)K / 1e4) * (double)steps +
                           f.store_us * (double)splits * mn / 1e6 + (splits > 1 ? f.cut_us : f.whole_us)[behind] +
                           (splits == 1 && behind == 2 && M > 2200 ? 0.0026 * (double)(M - 2200) : 0.);
        if (own < us) best = TilePlan{VARIANT_STREAM + f.i, (int)splits, splits > 1 ? (int)steps * 64 : K, us = own};
      }
    }
  }
  return best;
}

// Where `panel_dma_kernel` runs: J of its tiles (32 J weight rows), or 0.  All tiles are on the chip at once.
//  * 17 to 64 rows: in `panel_kernel`'s place up to 160 weight rows a CU (SwiGLU of 37,888 x 3,584, 17 / 48 / 64 rows 50.5 / 53.9 /
//    58.7 us there and 48.9 / 49.8 / 50.8 so; 40,960 x 512 17.2 and 11.9); beyond, that kernel's blocks go on from pass to pass.
//    (Timed at 32,768 to 40,960 weight rows of 512 to 8,192, all epilogues: 0.53 to 1.01 of its time, except 17 to 40 rows against
//    34,816 to 37,888 of 6,144 or 8,192, which begin 12 or 16 KB apart: up to 1.06, 36,864 x 8,192 122.5 and 129.1.)
//  * 51 to 64 rows, SwiGLU, more than 64 and up to 96 weight rows a CU against a K of up to 2,048, where 64 x 64 tiles are two a CU:
//    22,016 x 2,048, 64 rows 27.6 and 23.9; 17,920 x 1,536 20.7 and 16.3.  (17 to 50 rows would gain there too, 33 rows 25.5 and 23.2,
//    and still run as tiles.  With 64 weight rows a CU and fewer the tiles are the faster: 9,728 x 896 6.0 and 7.7.)
//  * 65 to 128 rows, more than 128 and up to 160 weight rows a CU, where tiles of 128 x 128 take two rounds and tiles of 128 x 256
//    leave a third of the CUs idle: SwiGLU of 37,888 x 3,584, 65 / 100 / 128 rows 63.5 / 66.7 / 68.9 and 52.6 / 55.6 / 58.7.  No other
//    plan is asked for its price there: at 32,800 to 40,960 weight rows of 512 to 8,192, all epilogues, 0.80 to 1.0 of the tiles' time.
//    (32,768 x 2,048, a round of 128 x 128: 36.2 and 38.5; 208 rows, in tiles of 208 x 160: level with 256 x 192.)
int panel_dma_units(int M, int N, int K, int epi, int n_cu) {
  const int units = (N + 31) / 32;
  if (M <= 16 || M > 128 || K % DMA_BK || n_cu <= 0 || units > 5 * n_cu) return 0;
  if (units > 4 * n_cu || (M <= 64 && units == 4 * n_cu)) return 5;
  return M > 50 && M <= 64 && epi == EPI_SWIGLU && K <= 2048 && units > 2 * n_cu && units <= 3 * n_cu ? 3 : 0;
}

int launch_panel_rows(int J, const bf16* A, int lda, const Weights& w, const float* bias, void* C, int ldc, int M, int N, int K,
                      int epi, const FusedNorm& fused, hipStream_t stream) {
  const bool t = w.tiled != nullptr;
#define MF_PANEL(I_, J_, RA_, STAGES_, TURNS_) \
  launch_panel_dma<I_, J_, RA_, STAGES_, TURNS_>(A, lda, w.at(t), w.ld(t), bias, C, ldc, M, N, K, epi, fused, t, stream)
  if (M > 64) return MF_PANEL(2, 5, 128, 4, true);
  return J == 5 ? MF_PANEL(1, 5, 64, 5, false) : MF_PANEL(1, 3, 64, 6, false);
#undef MF_PANEL
}

// Which kernel a product of at most 64 rows takes (SK_NONE: none has a place for the norms to be folded in).
enum SkinnyChoice {
  SK_STATIONARY, SK_ROLLING, SK_GUARDED_PAIR, SK_GUARDED_4X2, SK_GUARDED_8X2, SK_GUARDED_8X1, SK_PANEL, SK_RING,
  SK_STAGED, SK_TILE, SK_PANEL_SHORT, SK_WHOLE, SK_NONE
};
// Norms folded in: the activations come with a prepared one, the next one is prepared; of the latter's sums there are places for those
// over runs of 256 columns alone.
enum { FOLD_IN = 1, FOLD_OUT = 2, FOLD_RUNS = 4 };

// 17 to 64 rows against a short K: a tile of 64 x 64 over the whole of K, with the norm's factors, the bias and SwiGLU in its
// epilogue, where the K-split kernels need a second one (32 to 40 rows, K-split and added / one tile kernel: gate|up 9,728 x 896
// 15.0 / 9.0 us, 17,920 x 1,536 19.9 / 19.2, 22,016 x 2,048 28.3 / 26.6; q|k|v 1,152 x 896 11.6 / 9.0, 2,048 x 1,536 level).
// At most two tiles a CU, all at once; fewer than eight tiles are a launch whichever kernel it is.  A tile's chain over K is the
// same however few rows and tiles there are, while the K-split kernels' two launches get shorter with them in the ring form with
// the tiled copy to read: SwiGLU of 17 rows of 2,048 against 512 to 2,048 9.3 us so and 7.6 split, level where rows times weight
// rows reach some 110,000 at that K and 22,000 at 1,536; with a second tile a CU and no SwiGLU to save, 17 rows against 24,576
// of 768 10.9 us and 8.9, 48 rows 12.4 and 13.1 (12.2 so and 18.1 split without the copy).
bool tile64_takes(int M, int N, int K, bool aligned, bool tiled, int epi, int n_cu) {
  if (M <= 16 || !aligned || K % DMA_BK || N < 512 || (N + 63) / 64 > 2 * n_cu) return false;
  const bool fast_split = tiled && K % 256 == 0;             // (`ring_takes`)
  if (epi == EPI_SWIGLU) return K <= 2048 && (!fast_split || (long)M * N >= 176L * (K - 1408));
  return K <= 1024 && (!fast_split || M > 32 || K <= 512 || N <= 64 * n_cu);
}

SkinnyChoice skinny_choice(int M, int N, int K, bool aligned, bool tiled, int epi, int splits, int k_per_split, int n_cu, int folds) {
  if (folds && !(folds & FOLD_RUNS) && whole_takes(M, N, K, aligned, epi, n_cu)) return SK_WHOLE;
  if (M <= 16 && splits == 1) {
    // the register-resident kernel where it is built; other aligned shapes the rolling K-split
    // kernel; the rest (and SwiGLU outside the first) the guarded kernel.  The first takes a prepared norm and prepares
    // the next one, the second prepares the next one.
    if (aligned && stationary_takes(M, N, K, epi, false)) return SK_STATIONARY;
    if (aligned && K % 32 == 0 && epi != EPI_SWIGLU) return folds & FOLD_IN ? SK_NONE : SK_ROLLING;
    if (folds) return SK_NONE;
    if (epi == EPI_SWIGLU) return SK_GUARDED_PAIR;
    // many weight rows: 4 waves with two 16-row tiles each (less activation traffic per weight
    // byte); a row count that would leave a short second round of 16-row blocks: 8 waves with
    // two tiles; otherwise 8 waves, one tile
    const int blocks16 = (N + 15) / 16;
    if (blocks16 >= 1024) return SK_GUARDED_4X2;
    if (blocks16 > 256 && blocks16 <= 512) return SK_GUARDED_8X2;
    return SK_GUARDED_8X1;
  }
  // (the panel and the tile kernels take a prepared norm and prepare none; of the K-split kernels the second folds norms in)
  if (M > 16 && panel_takes(M, N, K, aligned, epi, n_cu)) return folds & FOLD_OUT ? SK_NONE : SK_PANEL;
  if (!(folds & FOLD_OUT)) {
    if (aligned && panel_dma_units(M, N, K, epi, n_cu) == 3) return SK_PANEL_SHORT;
    if (tile64_takes(M, N, K, aligned, tiled, epi, n_cu)) return SK_TILE;
  }
  if (folds && splits == 1 && epi != EPI_SWIGLU) return SK_NONE;
  return ring_takes(aligned, K, splits, k_per_split) ? SK_RING : SK_STAGED;
}

}  // namespace

// Products of rows that stand in groups with a matrix each: rows first .. first + rows - 1 of A (a row group's, at most
// the variant's tile rows) with matrix `matrix` of the stack W [matrices][N][K], 32-bit sums into the same rows of C.
// variant 2: tiles of 128 x 128, 12: 256 x 256, 13: 256 x 128; K in 64s.
MF_API int mf_gemm_bf16_grouped(const void* A, const void* W, float* C, const int* groups, int n_groups, int N, int K,
                                int variant, hipStream_t stream) {
  if (n_groups <= 0 || N <= 0) return 0;
  if (K <= 0 || K % DMA_BK || !groups || (uintptr_t)A % 16 || (uintptr_t)W % 16 || (size_t)N * K * 2 >= (1ull << 32))
    return (int)hipErrorInvalidValue;
  const bf16* a = (const bf16*)A;
  const bf16* w = (const bf16*)W;
  const RowGroup* g = (const RowGroup*)groups;
  switch (variant) {
    case 2: return launch_tile_step<128, 128, 2, 4, 4, true>(a, K, w, K, nullptr, C, N, 0, N, K, EPI_F32, stream, 1, 0, g, n_groups);
    case 12: return launch_grouped_dma<256, 256, 2>(a, K, w, K, C, N, g, n_groups, N, K, stream);
    case 13: return launch_grouped_dma<256, 128, 3>(a, K, w, K, C, N, g, n_groups, N, K, stream);
  }
  return (int)hipErrorInvalidValue;
}

static bool halves_ok(const Halves& h, const void* C, int K, size_t rows, int ld) {
  return h.width > 0 && C && K > 0 && K % DMA_BK == 0 && rows * (size_t)ld * 2 < (1ull << 32);
}

// The same of matrices whose rows are `width` gates and then `width` ups (W [matrices][2 width][K]): C [rows][width] =
// act(gate, up) in bfloat16 from the 32-bit sums, the activations being those of `mf_moe_act` (act 1: silu(gate) up, 0: the clamped
// form with `limit`; any other is refused).  No 32-bit intermediate and no kernel of its own for the activation: 2,048 rows over 8 matrices of 8,192 x
// 2,048 117 + 24 us as two kernels, 120 so (what the smaller stores save, the exponentials take).
MF_API int mf_gemm_bf16_grouped_gated(const void* A, const void* W, void* C, const int* groups, int n_groups, int width, int K,
                                      int variant, int act, float limit, hipStream_t stream) {
  if (n_groups <= 0 || width <= 0) return 0;
  const Halves h{width, act == 1, limit, nullptr, 0};
  if (act < 0 || act > 1 || !halves_ok(h, C, K, 2 * (size_t)width, K) || !groups || (uintptr_t)A % 16 || (uintptr_t)W % 16) return (int)hipErrorInvalidValue;
  const bf16* a = (const bf16*)A;
  const bf16* w = (const bf16*)W;
  const RowGroup* g = (const RowGroup*)groups;
  const int N = (width + 31) / 32 * 64;
  switch (variant) {
    case 2:
      return launch_tile_step<128, 128, 2, 4, 4, true, false, true>(a, K, w, K, nullptr, C, width, 0, N, K, EPI_SWIGLU, stream, 1, 0, g, n_groups,
                                                                    nullptr, 0, 0.f, h);
    case 12: return launch_grouped_dma<256, 256, 2, true>(a, K, w, K, C, width, g, n_groups, N, K, stream, h);
    case 13: return launch_grouped_dma<256, 128, 3, true>(a, K, w, K, C, width, g, n_groups, N, K, stream, h);
  }
  return (int)hipErrorInvalidValue;
}

// which of the tiles that have the form (256 x 256, 256 x 128, 128 x 128) one product of it takes
static int gated_form(int M, int N, int K, long cu) {
  const long nkt = K / DMA_BK;
  int form = FORM_256;
  for (int f : {FORM_128, FORM_SMALL})
    if (form_us(f, M, N, K, nkt, 1, cu) < form_us(form, M, N, K, nkt, 1, cu)) form = f;
  return form;
}

// Whether `mf_gemm_bf16_gated`, behind a product of its own for the rows' logits, is the faster way through a matrix of `rows` rows (2 width
// gates and ups, and the logit's behind them): 1, or 0 where one product of them all and the activation's kernel are.  The estimates of
// the plans for each of the products, the kernel at 5.5 TB/s; 8 us for what a plan counts as starts and rounds beside them.
// (The gated form has no 64 x 64 tile, and the logits are a launch or two: 8,208 x 2,048, apart / so: 65 rows 19.0 / 30.5 us, 128 23.9 / 33.1, 203
// 28.7 / 30.9, 384 29.9 / 33.2, 512 38.6 / 33.1, 2,048 83.9 / 64.6; 2,064 x 2,048: 768 19.6 / 27.2, 2,048 36.7 / 29.7.  245 shapes of 100 to 8,192
// gates and 256 to 4,096, 65 to 4,096 rows: the choice is 0.5 % above the better way on the average, at most 5 % above two kernels (1,300 rows of
// 12,304 x 3,072 135 and 142) and 7 % above one (333 of them 54.9 and 51.1).)
MF_API int mf_gemm_bf16_gated_pays(int M, int width, int rows, int K, int n_cu) {
  if (M <= 64 || width <= 0 || rows < 2 * width || K <= 0 || K % DMA_BK || n_cu <= 0) return 0;
  const int N = (width + 31) / 32 * 64, logits = rows - 2 * width;
  const double act_us = 2.5 + ((double)rows * 4. + (double)width * 2.) * M / 5.5e6;
  const double apart = plan_tiles(M, rows, K, true, EPI_F32, n_cu).us + act_us;
  const double joined = form_us(gated_form(M, N, K, n_cu), M, N, K, K / DMA_BK, 1, n_cu) +
                        (logits ? plan_tiles(M, logits, K, true, EPI_F32, n_cu).us : 0.) + 8.;
  return joined < apart;
}

// One product of that form, M rows, with a factor sigmoid(z) of every row (z [M], ldz apart; null: none): C [M][width].  The clamped form
// needs a limit above 0.  2,048 rows of
// 8,192 x 2,048: 62 + 19 us as two kernels, 64 so.
MF_API int mf_gemm_bf16_gated(const void* A, int lda, const void* W, int ldw, void* C, int M, int width, int K, int act, float limit,
                              const float* z, int ldz, hipStream_t stream) {
  if (M <= 0 || width <= 0) return 0;
  const Halves h{width, act == 1, limit, z, ldz};
  if (act < 0 || act > 1 || (act == 0 && !(limit > 0.f)) || lda < K || ldw < K || lda % 8 || ldw % 8 || !halves_ok(h, C, K, 2 * (size_t)width, ldw) || (size_t)M * lda * 2 >= (1ull << 32) ||
      (uintptr_t)A % 16 || (uintptr_t)W % 16)
    return (int)hipErrorInvalidValue;
  const bf16* a = (const bf16*)A;
  const bf16* w = (const bf16*)W;
  bf16* c = (bf16*)C;
  const int N = (width + 31) / 32 * 64, cu = cu_count();
  if (cu <= 0) return (int)hipErrorUnknown;
  const int form = gated_form(M, N, K, cu);
  if (form == FORM_256) return launch_halves_dma<256, 256, 2>(a, lda, w, ldw, c, M, N, K, h, stream);
  if (form == FORM_128) return launch_halves_dma<256, 128, 3>(a, lda, w, ldw, c, M, N, K, h, stream);
  return launch_tile_step<128, 128, 2, 4, 4, false, false, true>(a, lda, w, ldw, nullptr, c, width, M, N, K, EPI_SWIGLU, stream, 1, 0, nullptr, 0,
                                                                 nullptr, 0, 0.f, h);
}

// `variant`: 0 picks by shape among the whole-K kernels; 1: 256x256 tile with 4 waves, 2: 128x128,
// 3: 64x64, 6: 256x128 with 8 waves, 9: 256x256 with 8 waves; through the direct-to-LDS pipeline, K in
// 64s: 12: 256x256 (SwiGLU: or 256x192), 13: the cheapest of 256x128, 128x256, 128x128 and 64x64 (or the
// panel kernel where it runs), 15: 256x192 (tests name them),
// 16: the cheapest of all for the weight rows up to a multiple of 256, and of the small ones for up to 64 behind them; 17: the panel
// kernel with copies straight into LDS.
MF_API int mf_gemm_bf16(const void* A, int lda, const void* W, const void* Wt, int ldw, const float* bias, void* C,
                        int ldc, int M, int N, int K, int epi, int variant, hipStream_t stream) {
  if (M <= 0 || N <= 0) return 0;
  if (K <= 0 || lda < K || ldw < K || epi < 0 || epi > EPI_LAST || (epi == EPI_XIELU && !bias)) return (int)hipErrorInvalidValue;
  if (epi == EPI_SWIGLU ? (N % 64 != 0 || ldc > N / 2 || ldc <= N / 2 - 32) : ldc < N)
    return (int)hipErrorInvalidValue;
  const int vec_ok = (lda % 8 == 0) && (ldw % 8 == 0) && ((uintptr_t)A % 16 == 0) &&
                     ((uintptr_t)W % 16 == 0) && (K % 8 == 0);
  const bf16* a = (const bf16*)A;
  const bf16* w = (const bf16*)W;
  // the direct-to-LDS kernel addresses its operands with 32-bit byte offsets
  const bool dma_ok = vec_ok && K % DMA_BK == 0 && (size_t)M * lda * 2 < (1ull << 32) && (size_t)N * ldw * 2 < (1ull << 32);
  if (variant == 0) {
    const TilePlan plan = plan_tiles(M, N, K, dma_ok, epi, cu_count());
    if (plan.splits > 1) return (int)hipErrorInvalidValue;       // a K split needs the caller's workspace
    variant = plan.variant;
  }
  const Weights wt(w, Wt, ldw, K);
  if (variant == 17 || (variant == 13 && M > 64 && dma_ok && panel_dma_units(M, N, K, epi, cu_count()))) {
    const int J = panel_dma_units(M, N, K, epi, cu_count());
    if (!J || !dma_ok) return (int)hipErrorInvalidValue;
    return launch_panel_rows(J, a, lda, wt, bias, C, ldc, M, N, K, epi, FusedNorm{}, stream);
  }
  if (variant == 16) {
    const int n0 = main_rows(N, epi), cu = cu_count();
    if (!n0 || !dma_ok || cu <= 0) return (int)hipErrorInvalidValue;
    const long nkt = K / DMA_BK;
    const int rc = launch_form(best_form(0, N_FORMS - 1, M, n0, K, nkt, 1, cu), a, lda, wt, bias, C, ldc, M, n0, K, epi, stream);
    if (rc) return rc;
    void* rest = (char*)C + (size_t)n0 * (epi == EPI_BF16 || epi == EPI_RELU2 ? 2 : 4);
    return launch_form(best_form(FORM_128, FORM_TINY, M, N - n0, K, nkt, 1, cu), a, lda, wt.from(n0), bias ? bias + n0 : nullptr,
                       rest, ldc, M, N - n0, K, epi, stream);
  }
  if (variant > VARIANT_STREAM)
    return dma_ok ? launch_tile_stream(variant, a, lda, wt.tiled, bias, C, ldc, M, N, K, epi, stream) : (int)hipErrorInvalidValue;
  if (epi == EPI_SWIGLU && variant == 3) variant = 2;      // needs two 32-column tiles per wave
  switch (variant) {
    case 1: return launch_tile<256, 256, 128, 128>(a, lda, w, ldw, bias, C, ldc, M, N, K, epi, vec_ok, stream);
    case 2: return launch_tile<128, 128, 64, 64>(a, lda, w, ldw, bias, C, ldc, M, N, K, epi, vec_ok, stream);
    case 3: return launch_tile<64, 64, 32, 32>(a, lda, w, ldw, bias, C, ldc, M, N, K, epi, vec_ok, stream);
    case 6: return launch_tile<256, 128, 64, 64, 32>(a, lda, w, ldw, bias, C, ldc, M, N, K, epi, vec_ok, stream);
    case 9: return launch_tile<256, 256, 128, 64, 64>(a, lda, w, ldw, bias, C, ldc, M, N, K, epi, vec_ok, stream);
    case 12: case 13: case 15:
      if (!dma_ok || (variant == 15 && epi == EPI_SWIGLU)) return (int)hipErrorInvalidValue;
      return launch_form(dma_form(variant, M, N, K, epi, K / DMA_BK, 1, cu_count()), a, lda, wt, bias, C, ldc, M, N, K, epi, stream);
  }
  return (int)hipErrorInvalidValue;
}

// Few rows for the tile kernel (a prompt of a few hundred tokens against 3584 weight rows makes
// some 50 tiles for 256 CUs): K is split over `splits` blocks per tile, which store 32-bit sums
// into part[splits][M][N] (`mf_gemm_bf16_parts`), and skinny_reduce_kernel adds them and runs the epilogue.
// k_per_split is a multiple of 64.
MF_API int mf_gemm_bf16_parts(const void* A, int lda, const void* W, const void* Wt, int ldw, float* part, int M, int N, int K, int splits,
                              int k_per_split, int variant, hipStream_t stream) {
  if (M <= 0 || N <= 0) return 0;
  if (K <= 0 || lda < K || ldw < K || splits < 2 || !part || k_per_split % 64 != 0 || (long)splits * k_per_split < K ||
      (long)(splits - 1) * k_per_split >= K)
    return (int)hipErrorInvalidValue;
  const int vec_ok = (lda % 8 == 0) && (ldw % 8 == 0) && ((uintptr_t)A % 16 == 0) &&
                     ((uintptr_t)W % 16 == 0) && (K % 8 == 0);
  // variant 12: 256 x 256 tiles through the direct-to-LDS pipeline (many rows against few weight
  // rows and a long K: the down product of a prompt); 2: the smaller tiles (few rows)
  // (and VARIANT_STREAM + I: `tile_stream_kernel`)
  if (variant != 12 && variant != 2 && variant <= VARIANT_STREAM) return (int)hipErrorInvalidValue;
  const bool dma_ok = vec_ok && K % DMA_BK == 0 && (size_t)M * lda * 2 < (1ull << 32) && (size_t)N * ldw * 2 < (1ull << 32);
  if (variant != 2 && !dma_ok) return (int)hipErrorInvalidValue;
  if (variant > VARIANT_STREAM)
    return launch_tile_stream(variant, (const bf16*)A, lda, Weights(W, Wt, ldw, K).tiled, nullptr, part, N, M, N, K, EPI_F32, stream, splits,
                              k_per_split);
  return dma_ok ? launch_form(dma_form(variant, M, N, K, EPI_F32, k_per_split / DMA_BK, splits, cu_count()), (const bf16*)A, lda,
                              Weights(W, Wt, ldw, K), nullptr, part, N, M, N, K, EPI_F32, stream, splits, k_per_split)
                : launch_tile<128, 128, 64, 64>((const bf16*)A, lda, (const bf16*)W, ldw, nullptr, part, N, M,
                                                N, K, EPI_F32, vec_ok, stream, splits, k_per_split);
}

MF_API int mf_gemm_bf16_splitk(const void* A, int lda, const void* W, const void* Wt, int ldw, const float* bias, void* C,
                               int ldc, float* part, int M, int N, int K, int splits, int k_per_split,
                               int epi, int variant, hipStream_t stream) {
  if (M <= 0 || N <= 0) return 0;
  if (epi < 0 || epi > EPI_LAST || (epi == EPI_XIELU && !bias)) return (int)hipErrorInvalidValue;
  if (epi == EPI_SWIGLU ? (N % 64 != 0 || ldc > N / 2 || ldc <= N / 2 - 32) : ldc < N)
    return (int)hipErrorInvalidValue;
  const int rc = mf_gemm_bf16_parts(A, lda, W, Wt, ldw, part, M, N, K, splits, k_per_split, variant, stream);
  if (rc) return rc;
  return launch_reduce(part, bias, C, ldc, M, N, K, splits, epi, FusedNorm{}, stream);
}

// The same into the residual stream (32-bit C, stored or added to), with the RMS norm of the new rows beside it: normed =
// bfloat16 C / sqrt(mean(C^2) + eps) g, [M][N].  N in fours, at most 16,384, every operand 16-byte aligned; MF_NOT_BUILT
// (nothing launched) for any other.
MF_API int mf_gemm_bf16_splitk_norm(const void* A, int lda, const void* W, const void* Wt, int ldw, const float* bias, float* C, int ldc,
                                    float* part, int M, int N, int K, int splits, int k_per_split, int accumulate, int variant,
                                    const float* g, float eps, void* normed, hipStream_t stream) {
  if (M <= 0 || N <= 0) return 0;
  if (N % 4 || N > REDUCE_NORM_MAX || ldc % 4 || (uintptr_t)C % 16 || (uintptr_t)part % 16 || (uintptr_t)bias % 16 ||
      (uintptr_t)g % 16 || (uintptr_t)normed % 8 || !g || !normed)
    return MF_NOT_BUILT;
  if (ldc < N) return (int)hipErrorInvalidValue;
  const int rc = mf_gemm_bf16_parts(A, lda, W, Wt, ldw, part, M, N, K, splits, k_per_split, variant, stream);
  if (rc) return rc;
  return launch_reduce_norm(part, bias, C, ldc, M, N, splits, accumulate, g, eps, (bf16*)normed, stream);
}

// The register-resident kernel for the shapes it is built for (K = 256 NS with enough tiles to
// go round); MF_NOT_BUILT for any other, and nothing is launched.
static int stationary16(const void* a, int lda, const bf16* w, const bf16* wt, int ldw, const float* bias, void* C,
                        int ldc, int M, int N, int K, int epi, const NormArgs* norm, hipStream_t stream,
                        const FusedNorm& fused = FusedNorm{}) {
  if (!stationary_takes(M, N, K, epi, norm != nullptr)) return MF_NOT_BUILT;
  // two tiles an item where a block's share is more than one: 128-byte rows of 32-bit output
  const int n_cu = cu_count();
  if (n_cu <= 0) return (int)hipErrorUnknown;
  const bool two = (N + n_cu - 1) / n_cu > 16;
#define MF_STATIONARY_T(NS_, T_, W_)                                                                          \
  (epi == EPI_SWIGLU ? launch_stationary16<NS_, 2, true, T_>(a, lda, W_, ldw, bias, C, ldc, M, N, epi, norm, fused, stream) \
   : two             ? launch_stationary16<NS_, 2, false, T_>(a, lda, W_, ldw, bias, C, ldc, M, N, epi, norm, fused, stream) \
                     : launch_stationary16<NS_, 1, false, T_>(a, lda, W_, ldw, bias, C, ldc, M, N, epi, norm, fused, stream))
#define MF_STATIONARY(NS_) \
  case NS_: return wt ? MF_STATIONARY_T(NS_, true, wt) : MF_STATIONARY_T(NS_, false, w);
  if (K == STATIONARY_K7) {
    // seven waves: one tile an item outside SwiGLU (the epilogue gives every wave 64 / (16 NT) rows)
#define MF_STATIONARY_7(T_, W_)                                                                                  \
  (epi == EPI_SWIGLU ? launch_stationary16<4, 2, true, T_, 7>(a, lda, W_, ldw, bias, C, ldc, M, N, epi, norm, fused, stream) \
                     : launch_stationary16<4, 1, false, T_, 7>(a, lda, W_, ldw, bias, C, ldc, M, N, epi, norm, fused, stream))
    return wt ? MF_STATIONARY_7(true, wt) : MF_STATIONARY_7(false, w);
#undef MF_STATIONARY_7
  }
  switch (K / 256) { MF_STATIONARY_NS(MF_STATIONARY) }
#undef MF_STATIONARY
#undef MF_STATIONARY_T
  return MF_NOT_BUILT;
}

static int skinny_product(const void* A, int lda, const void* W, const void* Wt, int ldw, const float* bias,
                          void* C, int ldc, float* part, int M, int N, int K, int splits, int k_per_split, int epi,
                          const FusedNorm& fused, hipStream_t stream) {
  if (M <= 0 || N <= 0) return 0;
  if (M > 64 || K <= 0 || lda < K || ldw < K || epi < 0 || epi > EPI_LAST || (epi == EPI_XIELU && !bias) || splits < 1 ||
      k_per_split % KC != 0 || (long)splits * k_per_split < K || (splits > 1 && !part))
    return (int)hipErrorInvalidValue;
  if (epi == EPI_SWIGLU ? (N % 64 != 0 || ldc > N / 2 || ldc <= N / 2 - 32 || (M > 16 && !part))
                        : ldc < N)
    return (int)hipErrorInvalidValue;
  const int vec_ok = (lda % 8 == 0) && (ldw % 8 == 0) && ((uintptr_t)A % 16 == 0) &&
                     ((uintptr_t)W % 16 == 0) && (K % 8 == 0);
  const bf16* a = (const bf16*)A;
  const bf16* w = (const bf16*)W;
  const bf16* wt = (K % 32 == 0 && (uintptr_t)Wt % 16 == 0) ? (const bf16*)Wt : nullptr;
  // (a caller with places for the sums over runs alone gets those, from the K-split kernels)
  const bool runs = fused.out_g && M > 16 && whole_takes(M, N, K, vec_ok, epi, cu_count()) && fused.out_parts < whole_plan(M, N, K, cu_count()).gx;
  const int folds = (fused.in_ssq ? FOLD_IN : 0) | (fused.out_g ? FOLD_OUT : 0) | (runs ? FOLD_RUNS : 0);
  const SkinnyChoice choice = skinny_choice(M, N, K, vec_ok, wt != nullptr, epi, splits, k_per_split, cu_count(), folds);
  switch (choice) {
    case SK_NONE: return MF_NOT_BUILT;
    case SK_WHOLE:
      return wt ? launch_whole<true>(a, lda, wt, ldw, bias, (float*)C, ldc, M, N, K, epi, fused, stream)
                : launch_whole<false>(a, lda, w, ldw, bias, (float*)C, ldc, M, N, K, epi, fused, stream);
    case SK_STATIONARY: return stationary16(a, lda, w, wt, ldw, bias, C, ldc, M, N, K, epi, nullptr, stream, fused);
    case SK_ROLLING:
      return wt ? launch_rolling16<true>(a, lda, wt, ldw, bias, C, ldc, M, N, K, epi, stream, fused)
                : launch_rolling16<false>(a, lda, w, ldw, bias, C, ldc, M, N, K, epi, stream, fused);
    case SK_GUARDED_PAIR: return launch_skinny16<4, 2, 4, true>(a, lda, w, ldw, bias, C, ldc, M, N, K, epi, vec_ok, stream);
    case SK_GUARDED_4X2: return launch_skinny16<4, 2, 4>(a, lda, w, ldw, bias, C, ldc, M, N, K, epi, vec_ok, stream);
    case SK_GUARDED_8X2: return launch_skinny16<8, 2, 4>(a, lda, w, ldw, bias, C, ldc, M, N, K, epi, vec_ok, stream);
    case SK_GUARDED_8X1: return launch_skinny16<8, 1, 8>(a, lda, w, ldw, bias, C, ldc, M, N, K, epi, vec_ok, stream);
    case SK_PANEL:
    case SK_PANEL_SHORT: {
      // (32-bit byte offsets)
      const int J = (size_t)N * ldw * 2 < (1ull << 32) ? panel_dma_units(M, N, K, epi, cu_count()) : 0;
      if (J) return launch_panel_rows(J, a, lda, Weights(w, wt, ldw, K), bias, C, ldc, M, N, K, epi, fused, stream);
      if (choice == SK_PANEL_SHORT) break;
      return launch_panel(a, lda, w, wt, ldw, bias, C, ldc, M, N, K, epi, fused, stream);
    }
    case SK_TILE: {
      if ((size_t)N * ldw * 2 >= (1ull << 32)) break;          // (operands beyond 4 GB go to the K-split kernels)
      const Weights both(w, wt, ldw, K);
      auto run = [&](auto SCALED, auto T) {
        constexpr bool t = decltype(T)::value;
        return launch_tile64<decltype(SCALED)::value, t>(a, lda, both.at(t), both.ld(t), bias, C, ldc, M, N, K, epi, stream, 1, 0, fused.in_ssq,
                                                         fused.in_parts, fused.in_eps);
      };
      using Yes = std::true_type;
      using No = std::false_type;
      if (tile64_reads_tiled(both, M, N, 1)) return fused.in_ssq ? run(Yes{}, Yes{}) : run(No{}, Yes{});
      return fused.in_ssq ? run(Yes{}, No{}) : run(No{}, No{});
    }
    default: break;
  }
  switch ((M + 15) / 16) {
    case 1: return launch_skinny<1>(a, lda, w, wt, ldw, bias, C, ldc, part, M, N, K, splits, k_per_split, epi, vec_ok, fused, stream);
    case 2: return launch_skinny<2>(a, lda, w, wt, ldw, bias, C, ldc, part, M, N, K, splits, k_per_split, epi, vec_ok, fused, stream);
    case 3: return launch_skinny<3>(a, lda, w, wt, ldw, bias, C, ldc, part, M, N, K, splits, k_per_split, epi, vec_ok, fused, stream);
    case 4: return launch_skinny<4>(a, lda, w, wt, ldw, bias, C, ldc, part, M, N, K, splits, k_per_split, epi, vec_ok, fused, stream);
  }
  return (int)hipErrorInvalidValue;
}

// M <= 64.  `part` holds splits*M*N floats when splits > 1; k_per_split is a multiple of 256.
// `Wt`: the tiled copy of W (see w_operand), or null; the kernels that have a form for it read it
// instead of W.
MF_API int mf_gemm_bf16_skinny(const void* A, int lda, const void* W, const void* Wt, int ldw, const float* bias,
                               void* C, int ldc, float* part, int M, int N, int K, int splits,
                               int k_per_split, int epi, hipStream_t stream) {
  return skinny_product(A, lda, W, Wt, ldw, bias, C, ldc, part, M, N, K, splits, k_per_split, epi, FusedNorm{}, stream);
}

// The same with an RMS norm folded in on either side (see FusedNorm), for the shapes whose kernels
// have a place for it (17 to 64 rows: `whole_kernel`, or the K-split kernels with more than one split, on both sides, the tile
// and the panel kernels on the reading one; at most 16 rows: the register-resident kernel on both sides,
// the rolling kernel on the writing side); MF_NOT_BUILT (-2), having launched nothing, for any other.
//  * in_ssq [M][in_parts], in_eps: A holds bf16(x g) of rows x whose sums of squares these are; the
//    product's sums are multiplied by the row's 1 / sqrt(sum / K + eps) before bias and epilogue.
//  * out_g [N], out_xg [M][N] bf16, out_ssq [M][out_parts]: beside C (32-bit, stored or added
//    to), bf16(C g) and the sums of C^2 in parts are written: over runs of 256 columns (out_parts =
//    ceil(N / 256)) for 17 to 64 rows, or one part per block where `whole_kernel` takes them and there are places for that (out_parts at
//    least `mf_gemm_bf16_whole_parts`, the places past it set to zero; with fewer the K-split kernels run); for at most 16 rows one part per block of the product's one
//    kernel, out_parts at least the number of CUs (the places past the grid are set to zero).
MF_API int mf_gemm_bf16_skinny_fused(const void* A, int lda, const void* W, const void* Wt, int ldw,
                                     const float* bias, void* C, int ldc, float* part, int M, int N, int K,
                                     int splits, int k_per_split, int epi, const float* in_ssq, int in_parts,
                                     float in_eps, const float* out_g, void* out_xg, float* out_ssq,
                                     int out_parts, hipStream_t stream) {
  if (in_ssq && in_parts < 1) return (int)hipErrorInvalidValue;
  if (out_g && (!out_xg || !out_ssq || out_parts < 1 || ldc != N || (epi != EPI_F32 && epi != EPI_ACC_F32)))
    return (int)hipErrorInvalidValue;
  if (out_g && out_parts < (N + 255) / 256) return (int)hipErrorInvalidValue;
  const FusedNorm fused{in_ssq, in_parts, in_eps, out_g, (bf16*)out_xg, out_ssq, out_parts};
  return skinny_product(A, lda, W, Wt, ldw, bias, C, ldc, part, M, N, K, splits, k_per_split, epi, fused, stream);
}

// The partial sums of squares a row that `mf_gemm_bf16_skinny_fused` leaves with out_* where one kernel over the whole of K takes
// the product of 17 to 64 rows (aligned operands): one for each of its blocks; 0 where it does not.
MF_API int mf_gemm_bf16_whole_parts(int M, int N, int K, int n_cu) {
  if (M <= 0 || N <= 0 || K <= 0 || n_cu <= 0) return 0;
  return whole_takes(M, N, K, K % 8 == 0, EPI_ACC_F32, n_cu) ? whole_plan(M, N, K, n_cu).gx : 0;
}

// RMS norm of rows of the 32-bit residual stream x (row m of the product is x[row_idx[m]]), then
// the product with W, in one kernel.  Returns MF_NOT_BUILT (-2), having launched nothing, for
// shapes the register-resident kernel does not cover: the caller then runs the norm and the
// product one after the other.
MF_API int mf_gemm_bf16_normed(const float* x, int ldx, const int* row_idx, const float* g, float eps,
                               const void* W, const void* Wt, int ldw, const float* bias, void* C, int ldc, int M,
                               int N, int K, int epi, hipStream_t stream) {
  if (M <= 0 || N <= 0) return 0;
  if (K <= 0 || epi < 0 || epi > EPI_LAST || (epi == EPI_XIELU && !bias)) return (int)hipErrorInvalidValue;
  if (ldx % 4 != 0 || ldw % 8 != 0 || (uintptr_t)x % 16 != 0 || (uintptr_t)g % 16 != 0 || (uintptr_t)W % 16 != 0)
    return MF_NOT_BUILT;
  const NormArgs norm{g, row_idx, eps};
  const bf16* wt = (uintptr_t)Wt % 16 == 0 ? (const bf16*)Wt : nullptr;
  return stationary16(x, ldx, (const bf16*)W, wt, ldw, bias, C, ldc, M, N, K, epi, &norm, stream);
}

// How a product of more than 64 rows is run: out[0] the variant for mf_gemm_bf16, or with out[1] > 1
// for mf_gemm_bf16_splitk with out[1] splits of out[2] of K each.  `aligned`: 16-byte aligned
// operands with row strides and K in multiples of 8; `tiled`: the product is given the tiled copy, 16-byte aligned.  `behind`: 1 where the
// kernel behind the product adds its parts on the way (the rotation), 2 where that kernel is the norm of the rows as well, else 0.
MF_API int mf_gemm_bf16_tile_plan(int M, int N, int K, int aligned, int tiled, int epi, int n_cu, int behind, int* out) {
  if (!out || behind < 0 || behind > 2 || M <= 0 || N <= 0 || K <= 0 || epi < 0 || epi > EPI_LAST || n_cu <= 0) return (int)hipErrorInvalidValue;
  const bool dma_ok = aligned && K % DMA_BK == 0 && (size_t)M * K * 2 < (1ull << 32) && (size_t)N * K * 2 < (1ull << 32);
  const TilePlan plan = plan_tiles(M, N, K, dma_ok, epi, n_cu, behind, tiled != 0);
  out[0] = plan.variant;
  out[1] = plan.splits;
  out[2] = plan.k_per_split;
  return 0;
}

// The name of the kernel that a product of this shape takes, without launching anything: `rows`
// activation rows against `N` weight rows of length `K`; `aligned`: 16-byte aligned operands with
// row strides and K in multiples of 8; `tiled`: there is the tiled copy; for at most 64 rows `splits`, `k_per_split`: the caller's K
// split (1, K for none); `normed`: the RMS norm is to be folded in (an empty name then means "no
// such kernel": norm and product run one after the other); `folds`, at most 64 rows: norms folded in on either side as
// `mf_gemm_bf16_skinny_fused` does it, 1 a prepared one is taken, 2 the next one is prepared (with places for as many sums a row as the
// kernels leave; 4 beside it: for those over runs of 256 columns alone); an empty name where it returns MF_NOT_BUILT; `behind`, more rows: as in
// `mf_gemm_bf16_tile_plan`; `variant`: of the tile kernels, as `mf_gemm_bf16` takes it (0: the
// plan's own choice, K split or whole); `n_cu`: compute units of the device.
MF_API int mf_gemm_bf16_plan(int M, int N, int K, int aligned, int tiled, int epi, int splits, int k_per_split,
                             int normed, int folds, int behind, int variant, int n_cu, char* name, int cap) {
  if (folds < 0 || folds > 7 || (folds && (normed || M > 64)) || ((folds & FOLD_OUT) && epi != EPI_F32 && epi != EPI_ACC_F32) || behind < 0 ||
      behind > 2)
    return (int)hipErrorInvalidValue;
  if (!name || cap < 48 || M <= 0 || N <= 0 || K <= 0 || epi < 0 || epi > EPI_LAST || n_cu <= 0) return (int)hipErrorInvalidValue;
  const char* what = "";
  if (normed) {
    what = (aligned && stationary_takes(M, N, K, epi, true)) ? "stationary16_kernel(norm)" : "";
  } else if (M <= 64 && !variant) {
    switch (skinny_choice(M, N, K, aligned != 0, tiled != 0 && K % 32 == 0, epi, splits, k_per_split, n_cu, folds)) {
      case SK_STATIONARY: what = "stationary16_kernel"; break;
      case SK_ROLLING: what = "rolling16_kernel"; break;
      case SK_GUARDED_PAIR: case SK_GUARDED_4X2: case SK_GUARDED_8X2: case SK_GUARDED_8X1: what = "skinny16_kernel"; break;
      case SK_PANEL: what = "panel_kernel"; break;           // (either form: `panel_dma_units`)
      case SK_PANEL_SHORT: what = "panel_dma_kernel"; break;
      case SK_RING: what = "skinny_ring_kernel"; break;
      case SK_STAGED: what = "skinny_kernel"; break;
      case SK_TILE: what = "tile_step_kernel<64,64>"; break;
      case SK_WHOLE: what = "whole_kernel"; break;
      case SK_NONE: break;
    }
  } else {
    const bool dma_ok = aligned && K % DMA_BK == 0 && (size_t)M * K * 2 < (1ull << 32) && (size_t)N * K * 2 < (1ull << 32);
    const TilePlan plan = variant ? TilePlan{variant, 1, K, 0.} : plan_tiles(M, N, K, dma_ok, epi, n_cu, behind, tiled != 0);
    const bool split = plan.splits > 1;
    if (variant >= 12 && !dma_ok) return (int)hipErrorInvalidValue;
    switch (plan.variant) {
      case 12: case 13: case 15:
        if (plan.variant == 13 && M > 64 && panel_dma_units(M, N, K, epi, n_cu)) what = "panel_dma_kernel";
        else what = form_name(dma_form(plan.variant, M, N, K, epi, (split ? plan.k_per_split : K) / DMA_BK, plan.splits, n_cu), split);
        break;
      case 16: what = "tile kernels (the last weight rows apart)"; break;
      case 17: what = "panel_dma_kernel"; break;
      case 9: what = "tile_kernel<256,256>"; break;
      case 2:
        what = split && dma_ok ? form_name(dma_form(2, M, N, K, EPI_F32, plan.k_per_split / DMA_BK, plan.splits, n_cu), true)
               : split         ? "tile_kernel<128,128>(split K)" : "tile_kernel<128,128>";
        break;
      case 3: what = "tile_kernel<64,64>"; break;
      case VARIANT_STREAM + 6: what = split ? "tile_stream_kernel<96>(split K)" : "tile_stream_kernel<96>"; break;
      case VARIANT_STREAM + 8: what = split ? "tile_stream_kernel<128>(split K)" : "tile_stream_kernel<128>"; break;
      default: return (int)hipErrorInvalidValue;
    }
  }
  snprintf(name, (size_t)cap, "%s", what);
  return 0;
}
