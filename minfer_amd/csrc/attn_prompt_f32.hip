// Attention of many query tokens per sequence (prompts) in the 32-bit run type, on the 32-bit matrix instruction
// (16x16x4: an FMA a product), over the paged cache.
//
// Semantics as `attn_tokens_impl.h` (src/graph/cpu_backend.rs:437-494 of yusiwen/minfer): a query at position p sees cache
// rows lo..p of its own sequence, lo = 0 or p - window + 1; s = q.k scale, softmax (accurate expf), sum of v; query head h
// reads kv head h / (nh / nk).
//
// The query heads of a group read the same keys, so the rows of the problem are (token, head of the group) pairs; a block
// takes 16 neighbouring ones of a sequence and kv head, and its 8 waves take the keys in runs of 16 in turn, each with
// statistics and sums of its own, which meet in LDS at the end.  (With rows of their own the waves would walk all keys one
// after the other, and 611 tokens of 14 heads on 2 would be 134 blocks.)  Keys and values come straight into MFMA operands, a
// run ahead of their use:
//   S^T[key][row] = K Q^T     A: lane -> key lane % 16, four neighbouring values of its row, the e-th of which go into the e-th
//                             product (the order of a sum's terms, alike on both sides); B = Q, held in registers
//   lane <-> row lane % 16: its keys of a run are 4 (lane / 16) + e, the operand layout of
//   O^T[d][row]  += V^T P^T   A: lane -> row 4 (lane / 16) + e of V, E neighbouring values, the d-th of which go into the d-th
//                             tile of results: the lane's results are values E (4 (lane / 16) + r) + d of its row
// The sums are kept in short chains, so that a result is no further from one in 64 bits than that of the kernel of a wave a
// token (1.2e-7 both at 611 tokens; chains of a whole score or a run of 32 keys: 1.5e-7): a score in chains of 4 QI terms, a
// run's weighted values in two chains of 8, the runs one after another.
// What bounds it: 16 E products of 32 cycles a run of a wave, some 25 vector instructions a score, and a trip to memory a run
// and wave (two blocks a CU cover each other's).  Two row tiles a wave (half the reads of keys): 21 us for 22 at 611 tokens, 36
// for 40 at 1,000, 23 for 17 where 20 tokens see 5,000 keys.
// 14 heads of 64 on 2, a wave a token (vector FMA) and now: 611 tokens 73 us and 21, 1,000 tokens 149 and 40, four times 180
// tokens on up to 5,000 keys 581 and 125; 12 heads of 128 on 2, 611 tokens: 91 and 29.  Heads of more than 128 stay with the
// kernel of a wave a token: their registers leave a wave a SIMD (300 tokens, 4 heads of 256 on 2: 45 us so, 48 here).
#include "attn_tokens_impl.h"

namespace {

constexpr int NW = 8;                                // waves of a block
constexpr int ROWS = 16;                             // rows of a block
constexpr int KU = 16;                               // keys of a run
constexpr int MAX_HEAD = 128;

template <int E>
struct PromptF32 {
  static constexpr int HD = 16 * E, VALUES = E * 4;  // a lane's results
  static constexpr int QI = E <= 4 ? 1 : 2;          // places of a score's chains (four chains a place)
  static constexpr int SMEM = NW * (VALUES * 64 + 2 * ROWS) * 4;
};

template <int E>
__global__ __launch_bounds__(64 * NW) void attn_prompt_f32_kernel(
    const float* __restrict__ q, const float* __restrict__ kc, const float* __restrict__ vc, const int* __restrict__ page_table,
    int pt_stride, const int* __restrict__ cu_seqlens, const int* __restrict__ start_pos, const int* __restrict__ tile_seq,
    const int* __restrict__ tile_row, float* __restrict__ out, float* __restrict__ part, int nh, int nk, float scale, int window,
    int split_len) {
  using S = PromptF32<E>;
  constexpr int HD = S::HD, QI = S::QI;
  const floatx4 zero = {0.f, 0.f, 0.f, 0.f};
  __shared__ __attribute__((aligned(16))) float sm[S::SMEM / 4];  // [wave][value][lane], then [wave][m, l][row]
  const int G = nh / nk;
  const int tile = blockIdx.x / nk, hk = blockIdx.x % nk;
  const int split = blockIdx.y, n_splits = gridDim.y;
  const int b = tile_seq[tile], r0 = tile_row[tile];
  const int tok0 = cu_seqlens[b], n_rows = (cu_seqlens[b + 1] - tok0) * G, start = start_pos[b];
  const int* pt = page_table + (size_t)b * pt_stride;
  const int lane = threadIdx.x & 63, wid = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int row = lane & 15, c = lane >> 4;
  // positions of the block's first and last row, and its keys
  const int p_lo = start + r0 / G, p_hi = start + min(r0 + ROWS - 1, n_rows - 1) / G;
  const int j_begin = max(window > 0 ? max(0, p_lo - window + 1) : 0, split * split_len);
  const int j_end = min(p_hi + 1, (split + 1) * split_len);
  // the lane's row (behind the last one: that one again, not stored)
  const int r = min(r0 + row, n_rows - 1), tl = r / G;
  const bool ok = r0 + row < n_rows;
  const int pos = start + tl;
  const size_t at = ((size_t)(tok0 + tl) * nh + hk * G + (r - tl * G)) * HD;
  floatx4 qf[E], o[E];
#pragma unroll
  for (int i = 0; i < E; ++i) {
    qf[i] = *reinterpret_cast<const floatx4*>(q + at + 16 * i + 4 * c);
    o[i] = zero;
  }
  float m = -INFINITY, l = 0.f;

  floatx4 kf[E];
  float vf[4][E];
  auto run_at = [&](int u) { return (((size_t)pt[u * KU / MF_PAGE] * nk + hk) * MF_PAGE + u * KU % MF_PAGE) * HD; };
  auto load_k = [&](int u) {
    const float* p = kc + run_at(u) + row * HD + 4 * c;
#pragma unroll
    for (int i = 0; i < E; ++i) kf[i] = *reinterpret_cast<const floatx4*>(p + 16 * i);
  };
  auto load_v = [&](int u) {
    const float* p = vc + run_at(u) + 4 * c * HD + E * row;
#pragma unroll
    for (int e = 0; e < 4; ++e) attn_tokens::load_raw<float, E>(p + e * HD, vf[e]);
  };
  const int u_end = j_begin < j_end ? (j_end + KU - 1) / KU : 0;
  int u = j_begin / KU + wid;
  if (u < u_end) {
    load_k(u);
    load_v(u);
  }
  for (; u < u_end; u += NW) {
    const bool more = u + NW < u_end;
    constexpr int PLACES = (E + QI - 1) / QI;
    floatx4 place[PLACES];
#pragma unroll
    for (int i = 0; i < PLACES; ++i) {
      floatx4 chain[4];
#pragma unroll
      for (int x = i * QI; x < E && x < (i + 1) * QI; ++x)
#pragma unroll
        for (int e = 0; e < 4; ++e)
          chain[e] = __builtin_amdgcn_mfma_f32_16x16x4f32(kf[x][e], qf[x][e], x == i * QI ? zero : chain[e], 0, 0, 0);
      place[i] = (chain[0] + chain[1]) + (chain[2] + chain[3]);
    }
#pragma unroll
    for (int step = 1; step < PLACES; step *= 2)
#pragma unroll
      for (int i = 0; i + step < PLACES; i += 2 * step) place[i] += place[i + step];
    floatx4 s = place[0];
    if (more) load_k(u + NW);
    const int key0 = u * KU;
    const bool whole = key0 + KU - 1 <= p_lo && key0 >= j_begin && (window <= 0 || key0 > p_hi - window);      // every row sees all of it
    auto sees = [&](int key) { return key >= j_begin && key <= pos && (window <= 0 || key > pos - window); };
    float top = -INFINITY, sum = 0.f;
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      s[e] = whole || sees(key0 + 4 * c + e) ? s[e] * scale : -INFINITY;
      top = fmaxf(top, s[e]);
    }
    top = fmaxf(top, __shfl_xor(top, 16, MF_WAVE));
    top = fmaxf(top, __shfl_xor(top, 32, MF_WAVE));
    const float m_new = fmaxf(m, top), m_use = m_new == -INFINITY ? 0.f : m_new;
    const float corr = m_new == -INFINITY ? 1.f : expf(m - m_new);
    m = m_new;
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      s[e] = expf(s[e] - m_use);                     // exp(-inf) = 0 for masked keys
      sum += s[e];
    }
    l = l * corr + sum;                              // of this lane's keys; the four lanes of a row meet at the end
    bool apart = false;
    if (!whole) {
      // Keys that the block does not take may never have been written (0 * garbage could be NaN): their values become zero.
      // And a value that is no number, of a key that only some rows see, must not reach the others.
      float any = 0.f;
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const int key = key0 + 4 * c + e;
        const bool there = key >= j_begin && key < j_end;
#pragma unroll
        for (int d = 0; d < E; ++d) {
          vf[e][d] = there ? vf[e][d] : 0.f;
          any = fmaf(vf[e][d], 0.f, any);
        }
      }
      apart = __builtin_amdgcn_ballot_w64(any != 0.f) != 0;        // (NaN: unequal)
    }
    floatx4 now[E];
    if (!apart) {
#pragma unroll
      for (int d = 0; d < E; ++d) {
        const floatx4 even = __builtin_amdgcn_mfma_f32_16x16x4f32(vf[0][d], s[0], zero, 0, 0, 0);
        const floatx4 odd = __builtin_amdgcn_mfma_f32_16x16x4f32(vf[1][d], s[1], zero, 0, 0, 0);
        now[d] = __builtin_amdgcn_mfma_f32_16x16x4f32(vf[2][d], s[2], even, 0, 0, 0) +
                 __builtin_amdgcn_mfma_f32_16x16x4f32(vf[3][d], s[3], odd, 0, 0, 0);
      }
    } else {
      // key by key: a row takes the products of the keys it sees
#pragma unroll
      for (int d = 0; d < E; ++d) now[d] = zero;
#pragma unroll
      for (int e = 0; e < 4; ++e)
#pragma unroll 1
        for (int k = 0; k < 4; ++k) {
          const bool mine = sees(key0 + 4 * k + e);
          const float p = c == k ? s[e] : 0.f;
#pragma unroll
          for (int d = 0; d < E; ++d) {
            const floatx4 one = __builtin_amdgcn_mfma_f32_16x16x4f32(c == k ? vf[e][d] : 0.f, p, zero, 0, 0, 0);
            if (mine) now[d] += one;
          }
        }
    }
    if (more) load_v(u + NW);
#pragma unroll
    for (int d = 0; d < E; ++d) o[d] = o[d] * corr + now[d];
  }

  // the waves' parts meet
  float* ml = sm + NW * S::VALUES * 64;
  l += __shfl_xor(l, 16, MF_WAVE);
  l += __shfl_xor(l, 32, MF_WAVE);
#pragma unroll
  for (int d = 0; d < E; ++d)
#pragma unroll
    for (int e = 0; e < 4; ++e) sm[(wid * S::VALUES + e * E + d) * 64 + lane] = o[d][e];
  if (c == 0) {
    ml[(wid * 2 + 0) * 16 + row] = m;
    ml[(wid * 2 + 1) * 16 + row] = l;
  }
  __syncthreads();
  // wave x adds up values e = x of every lane
  if (wid >= 4 || !ok) return;
  float w[NW], top = -INFINITY, sum = 0.f;
#pragma unroll
  for (int k = 0; k < NW; ++k) {
    w[k] = ml[(k * 2) * 16 + row];
    top = fmaxf(top, w[k]);
  }
#pragma unroll
  for (int k = 0; k < NW; ++k) {
    w[k] = top == -INFINITY ? 0.f : expf(w[k] - top);
    sum += ml[(k * 2 + 1) * 16 + row] * w[k];
  }
  float a[E];
#pragma unroll
  for (int d = 0; d < E; ++d) {
    a[d] = 0.f;
#pragma unroll
    for (int k = 0; k < NW; ++k) a[d] += sm[(k * S::VALUES + wid * E + d) * 64 + lane] * w[k];
  }
  const int d0 = E * (4 * c + wid);
  if (n_splits == 1) {
    const float inv = sum > 0.f ? 1.0f / sum : 0.f;
    float* to = out + at + d0;
#pragma unroll
    for (int d = 0; d < E; ++d) to[d] = a[d] * inv;
  } else {
    float* to = part + (at / HD * n_splits + split) * (HD + 2);
#pragma unroll
    for (int d = 0; d < E; ++d) to[d0 + d] = a[d];
    if (c == 0 && wid == 0) { to[HD] = top; to[HD + 1] = sum; }
  }
}

template <int E>
int launch(const float* q, const float* kc, const float* vc, const int* page_table, int pt_stride, const int* cu_seqlens,
           const int* start_pos, const int* tile_seq, const int* tile_row, float* out, float* part, int n_tiles, int n_tok, int nh,
           int nk, float scale, int window, int n_splits, int split_len, hipStream_t stream) {
  attn_prompt_f32_kernel<E><<<dim3(n_tiles * nk, n_splits), 64 * NW, 0, stream>>>(q, kc, vc, page_table, pt_stride, cu_seqlens, start_pos,
                                                                                  tile_seq, tile_row, out, part, nh, nk, scale, window,
                                                                                  split_len);
  int rc = mf_launch_status();
  if (rc == 0 && n_splits > 1) {
    attn_tokens::attn_combine_kernel<float><<<n_tok * nh, 64 * ((16 * E + 63) / 64), 0, stream>>>(part, out, 16 * E, n_splits);
    rc = mf_launch_status();
  }
  return rc;
}

}  // namespace

// (token, head of the group) rows that a block takes at this head size; 0: heads that this kernel does not take
MF_API int mf_attn_prompt_f32_rows(int hd) { return hd % 16 == 0 && hd >= 16 && hd <= MAX_HEAD ? ROWS : 0; }
// keys that the waves of a block take at once
MF_API int mf_attn_prompt_f32_keys() { return NW * KU; }

// tile_seq[i], tile_row[i]: sequence (index in the step's batch) and first row of the i-th run of mf_attn_prompt_f32_rows(hd)
// rows; row x of a sequence is head x % (nh / nk) of each group at its new token x / (nh / nk).  n_splits > 1: the keys are
// cut into runs of split_len (whole pages) and part [n_tok][nh][n_splits][hd + 2] takes the parts.
MF_API int mf_attn_prompt_f32(const float* q, const float* kc, const float* vc, const int* page_table, int pt_stride,
                              const int* cu_seqlens, const int* start_pos, const int* tile_seq, const int* tile_row, float* out,
                              float* part, int n_tiles, int n_tok, int nh, int nk, int hd, float scale, int window, int n_splits,
                              int split_len, hipStream_t stream) {
  if (n_tiles <= 0) return 0;
  if (mf_attn_prompt_f32_rows(hd) == 0 || nk <= 0 || nh % nk != 0 || n_splits < 1 || n_splits > 64 || split_len < MF_PAGE ||
      split_len % MF_PAGE != 0 || (n_splits > 1 && part == nullptr))
    return (int)hipErrorInvalidValue;
#define MF_CASE(E)                                                                                                          \
  case E:                                                                                                                   \
    return launch<E>(q, kc, vc, page_table, pt_stride, cu_seqlens, start_pos, tile_seq, tile_row, out, part, n_tiles, n_tok, \
                     nh, nk, scale, window, n_splits, split_len, stream);
  switch (hd / 16) {
    MF_CASE(1) MF_CASE(2) MF_CASE(3) MF_CASE(4) MF_CASE(5) MF_CASE(6) MF_CASE(7) MF_CASE(8)
  }
#undef MF_CASE
  return (int)hipErrorInvalidValue;
}
