// The ordered, weighted sum of one token's expert outputs (the MoE layer's
// unpermute), shared by moe_unpermute_kernel (hn_route.hip) and the fused
// unpermute + residual add + RMSNorm of the decoder (hn_decoder.hip), so both
// give the same bits.
//
// Reference arithmetic (model/mixtral.py:327-368): the experts a token was
// routed to are visited in ascending expert id (torch.unique order); each
// expert's output row y is scaled by its routing weight in fp16 and added
// into an fp16 accumulator: acc = fp16(acc + fp16(y * w)).
#pragma once
#include "hn_common.h"
#include "hn_topk.h"

// The token's assignments (position in the permuted rows, expert, weight)
// sorted by expert id; returns their number (assignments with inv < 0 are
// dropped).  Loads are unconditional (index clamped to k - 1): a load under
// `if (s < k)` ends its own block, and the compiler then waits for each in
// turn.
__device__ __forceinline__ int unp_select(int t, const int* __restrict__ inv,
                                          const int* __restrict__ idx,
                                          const h16* __restrict__ w, int k,
                                          int pos[kMaxTopK], float wt[kMaxTopK]) {
  int ex[kMaxTopK];
  int pv[kMaxTopK], ev[kMaxTopK];
  h16 wv[kMaxTopK];
#pragma unroll
  for (int s = 0; s < kMaxTopK; ++s) {
    const int j = t * k + (s < k ? s : k - 1);
    pv[s] = inv[j];
    ev[s] = idx[j];
    wv[s] = w[j];
  }
  int n = 0;
#pragma unroll
  for (int s = 0; s < kMaxTopK; ++s) {
    if (s >= k) break;
    const int p = pv[s];
    if (p < 0) continue;
    const int e = ev[s];
    // insertion by expert id (ascending)
    int q = n;
    while (q > 0 && ex[q - 1] > e) {
      ex[q] = ex[q - 1];
      pos[q] = pos[q - 1];
      wt[q] = wt[q - 1];
      --q;
    }
    ex[q] = e;
    pos[q] = p;
    wt[q] = (float)wv[s];
    ++n;
  }
  return n;
}

// Columns c .. c + 7 of the token's weighted sum over its n sorted
// assignments, whose rows are given as KS fp32 partial sums part[j * ks_stride
// + row * ld_y] (a K-split down projection), added in slice order and rounded
// to fp16 once.  The rows of two assignments are loaded before any is used.
template <int KS>
__device__ __forceinline__ half8_t unp_cols_split(const float* __restrict__ part, long ks_stride,
                                                  long ld_y, const int pos[kMaxTopK],
                                                  const float wt[kMaxTopK], int n, int c) {
  constexpr int B = 2;
  half8_t acc = {0, 0, 0, 0, 0, 0, 0, 0};
  for (int s0 = 0; s0 < n; s0 += B) {
    half8_t v[B];
#pragma unroll
    for (int u = 0; u < B; ++u) {
      const int s = s0 + u < n ? s0 + u : n - 1;
      float f[8];
#pragma unroll
      for (int q = 0; q < 8; ++q) f[q] = 0.f;
#pragma unroll
      for (int j = 0; j < KS; ++j) {
        const float* pp = part + j * ks_stride + (long)pos[s] * ld_y + c;
        const float4_t a = *reinterpret_cast<const float4_t*>(pp);
        const float4_t b = *reinterpret_cast<const float4_t*>(pp + 4);
#pragma unroll
        for (int q = 0; q < 4; ++q) {
          f[q] += a[q];
          f[4 + q] += b[q];
        }
      }
#pragma unroll
      for (int q = 0; q < 8; ++q) v[u][q] = (h16)f[q];
    }
#pragma unroll
    for (int u = 0; u < B; ++u) {
      if (s0 + u >= n) break;
      const float ws = wt[s0 + u];
#pragma unroll
      for (int j = 0; j < 8; ++j) {
        const h16 prod = (h16)((float)v[u][j] * ws);
        acc[j] = (h16)((float)acc[j] + (float)prod);
      }
    }
  }
  return acc;
}

// The same list for a whole wave with one token: lane s holds assignment s,
// counts those that sort before it (equal ids stay in assignment order), and
// the sorted list is read back lane by lane, so pos and wt are scalars at
// positions known when compiling (past n: the last one again).  unp_select
// indexes its arrays by run-time values: with up to 8 assignments of fp16 rows
// behind it, 301 tokens of 4096 columns took 20 us, so 9 (the rows' bytes: 5).
// With two assignments and rows in fp32 slices, a decode step's, unp_select is
// the faster one (decoder of 64 tokens, two layers: 626 and 632 us).
__device__ __forceinline__ int unp_select_wave(int t, const int* __restrict__ inv,
                                               const int* __restrict__ idx,
                                               const h16* __restrict__ w, int k,
                                               int pos[kMaxTopK], float wt[kMaxTopK]) {
  const int lane = threadIdx.x & 63;
  const int j = t * k + (lane < k ? lane : k - 1);
  const int p = inv[j], e = idx[j];
  const float wv = (float)w[j];
  const bool ok = lane < k && p >= 0;
  const unsigned long long valid = __ballot(ok);
  int rank = 0;
  for (int u = 0; u < k; ++u) {
    const int eu = __builtin_amdgcn_readlane(e, u);
    if ((valid >> u & 1) && (eu < e || (eu == e && u < lane))) ++rank;
  }
  const int n = __popcll(valid);
  int src = 0;
#pragma unroll
  for (int q = 0; q < kMaxTopK; ++q) {  // past n: the last one again
    const unsigned long long m = __ballot(ok && rank == q);
    src = m ? __builtin_ctzll(m) : src;
    pos[q] = __builtin_amdgcn_readlane(p, src);
    wt[q] = __builtin_bit_cast(float, __builtin_amdgcn_readlane(__builtin_bit_cast(int, wv), src));
  }
  return n;
}

// acc += the batch of B assignments from S0 on of fp16 rows y (those
// below n), in order; all their loads go out before any is used.
template <int S0, int B>
__device__ __forceinline__ void unp_batch(const h16* __restrict__ y, long ld_y,
                                          const int pos[kMaxTopK], const float wt[kMaxTopK],
                                          int n, int c, half8_t& acc) {
  half8_t v[B];
#pragma unroll
  for (int u = 0; u < B; ++u)
    v[u] = *reinterpret_cast<const half8_t*>(y + (long)pos[S0 + u] * ld_y + c);
#pragma unroll
  for (int u = 0; u < B; ++u) {
    // a select, not a branch: a load used only under a branch moves into it,
    // after the others' waits
    const float ws = wt[S0 + u];
    half8_t sum;
#pragma unroll
    for (int j = 0; j < 8; ++j) {
      const h16 prod = (h16)((float)v[u][j] * ws);
      sum[j] = (h16)((float)acc[j] + (float)prod);
    }
    acc = S0 + u < n ? sum : acc;
  }
}

// Columns c .. c + 7 of the token's weighted sum over its n assignments listed
// by unp_select_wave, rows of y in fp16.
__device__ __forceinline__ half8_t unp_cols(const h16* __restrict__ y, long ld_y,
                                            const int pos[kMaxTopK], const float wt[kMaxTopK],
                                            int n, int c) {
  static_assert(kMaxTopK == 16, "the batches cover 16 assignments");
  half8_t acc = {0, 0, 0, 0, 0, 0, 0, 0};
  if (n == 0) return acc;
  if (n <= 2) {
    unp_batch<0, 2>(y, ld_y, pos, wt, n, c, acc);
    return acc;
  }
  unp_batch<0, 8>(y, ld_y, pos, wt, n, c, acc);
  if (n > 8) unp_batch<8, 8>(y, ld_y, pos, wt, n, c, acc);
  return acc;
}
