// Prefill attention: many query tokens over the KV cache, grouped-query heads,
// scores, softmax and the value product in one kernel (the reference's
// Attention, model/mixtral.py:193-207, whose scores matrix is never written).
//
// One workgroup of 4 waves takes 128 rows of one (sequence, KV head), a row
// being a (query head of the group, token) pair, so the heads that share a KV
// head share its tiles also where there are few tokens.  Each wave owns 32
// rows and walks the positions in tiles of 64:
//   S^T = K Q^T   v_mfma_f32_32x32x16_f16, A = K from LDS, B = Q in registers;
//   softmax       a lane holds 32 scores of one row (the other 32 in lane ^ 32):
//                 running fp32 maximum and sum, exponentials as fp16;
//   O^T += V^T P  the score accumulators' own layout is a B operand whose 8
//                 values are positions {0-3, 8-11} (lanes below 32) and
//                 {4-7, 12-15} (the others) of 16, so P never leaves the
//                 registers: V is laid out in LDS in that order instead.
// K is cached as [hd][position] and V as [position][hd]: the operands want
// both the other way round, so both tiles are transposed in registers on their
// way into LDS (4 x 4 blocks of byte permutes), 16-byte loads one tile ahead.
//
// The mask is read once per call by mask_kernel, which keeps for each 32 rows
// x 64 positions whether all are -inf (the tile is not computed: half of a
// causal mask), all are 0 (no mask work), or only 0 and -inf (one 64-bit word
// per token and tile); other values are added as the torch formulation rounds
// them.
//
// At 8 sequences of 333 tokens, 32 heads over 8 KV heads, causal: 33 us + 5 us
// for the mask, where two products, the softmax between them and the copy of
// the heads' outputs into rows took 195 us.  What bounds it: each wave's chain
// of a tile (LDS reads, 32 MFMAs of 32 cycles, about 300 VALU instructions of
// softmax), which two waves per SIMD overlap only in part; alone on a CU, a
// workgroup takes 1.9 us per tile, half of it the latency of the next tile's
// loads.
#include "hn_common.h"

namespace {

typedef float float16_t __attribute__((ext_vector_type(16)));
typedef _Float16 half4_t __attribute__((ext_vector_type(4)));
typedef uint32_t u32x2 __attribute__((ext_vector_type(2)));

constexpr int kHd = 128;    // head dim
constexpr int kRows = 128;  // rows per workgroup
constexpr int kPos = 64;    // positions per tile
constexpr float kLog2e = 1.4426950408889634f;

// mask tile classes, one byte per (tile of 64 positions, 32 rows)
enum : uint32_t { kSkip = 0, kClear = 1, kBits = 2, kValues = 3 };

// One wave per (32 rows, 64 positions), lane = position, all 32 loads out
// together: the class byte, and the word of -inf positions of each token (rows
// past S are further heads' rows of the same tokens).
__global__ __launch_bounds__(256) void mask_kernel(const h16* __restrict__ mask, long ld_m, int S,
                                                   int R, int L, int nblk,
                                                   uint8_t* __restrict__ cls,
                                                   unsigned long long* __restrict__ bits) {
  const int lane = threadIdx.x & 63;
  const int blk = blockIdx.x * 4 + (threadIdx.x >> 6), tile = blockIdx.y;
  if (blk >= nblk) return;
  const int pos = tile * kPos + lane, row0 = blk * 32;
  h16 m[32];
  int s = row0 % S;
#pragma unroll
  for (int i = 0; i < 32; ++i) {
    m[i] = mask[(long)s * ld_m + (pos < L ? pos : L - 1)];  // unconditional: all in flight
    if (++s == S) s = 0;
  }
  bool any_fin = false, any_hid = false, any_val = false;
  unsigned long long mine = 0;  // lane i: the word of row i
#pragma unroll
  for (int i = 0; i < 32; ++i) {
    const bool in = row0 + i < R && pos < L;
    const bool hid = in && (float)m[i] == -__builtin_inff();
    const unsigned long long w = __ballot(hid);
    if (lane == i) mine = w;
    any_hid |= hid;
    any_fin |= in && !hid;
    any_val |= in && !hid && (float)m[i] != 0.f;  // also NaN and +inf
  }
  if (lane < 32 && row0 + lane < S) bits[(long)tile * S + row0 + lane] = mine;
  const bool hidden = __any(any_hid), fin = __any(any_fin), val = __any(any_val);
  if (lane == 0)
    cls[(long)tile * nblk + blk] = !fin ? kSkip : val ? kValues : hidden ? kBits : kClear;
}

__device__ __forceinline__ uint32_t perm_lo(uint32_t a, uint32_t b) {  // (a.lo, b.lo)
  return __builtin_amdgcn_perm(b, a, 0x05040100u);
}
__device__ __forceinline__ uint32_t perm_hi(uint32_t a, uint32_t b) {  // (a.hi, b.hi)
  return __builtin_amdgcn_perm(b, a, 0x07060302u);
}

// Four rows of 8 halves -> eight columns of 4 halves.
__device__ __forceinline__ void transpose4x8(const u32x4 r[4], u32x2 c[8]) {
#pragma unroll
  for (int d = 0; d < 4; ++d) {
    c[2 * d] = u32x2{perm_lo(r[0][d], r[1][d]), perm_lo(r[2][d], r[3][d])};
    c[2 * d + 1] = u32x2{perm_hi(r[0][d], r[1][d]), perm_hi(r[2][d], r[3][d])};
  }
}

// K tile in LDS: [64 positions][128 hd], 16-byte chunks of a position's 256
// bytes at chunk ^ k_key(position); V tile: [128 hd][64 positions], 16-byte
// chunk 2 u + h of a row's 128 bytes holding the 4-position groups 4 u + h and
// 4 u + 2 + h (the order P has them), at chunk ^ v_key(hd).  Both keys spread a
// wave's reads (one chunk of 32 rows) and writes over the banks.
__device__ __forceinline__ int k_key(int p) { return (p ^ (p >> 3)) & 15; }
__device__ __forceinline__ int v_key(int d) { return (d ^ (d >> 3)) & 7; }

// Thread t: hd rows 4 (t / 8) + j at positions 8 (t % 8) of K; positions 4 (t /
// 16) + j at hd 8 (t % 16) of V.  Positions past L are not read: V's are zero
// (their probabilities are, and stale values may be NaN), K's scores are
// replaced.  max_len is a multiple of 8, so a K load that starts below L ends
// inside the row.
__device__ __forceinline__ void load_k(u32x4 r[4], const h16* kt, long max_len, int p0, int L,
                                       int tid) {
  const int p = p0 + 8 * (tid & 7);
#pragma unroll
  for (int j = 0; j < 4; ++j) {
    r[j] = u32x4{0, 0, 0, 0};
    if (p < L)
      r[j] = *reinterpret_cast<const u32x4*>(kt + (long)(4 * (tid >> 3) + j) * max_len + p);
  }
}

__device__ __forceinline__ void load_v(u32x4 r[4], const h16* v, int p0, int L, int tid) {
  const int p = p0 + 4 * (tid >> 4);
#pragma unroll
  for (int j = 0; j < 4; ++j) {
    r[j] = u32x4{0, 0, 0, 0};
    if (p + j < L)
      r[j] = *reinterpret_cast<const u32x4*>(v + (long)(p + j) * kHd + 8 * (tid & 15));
  }
}

__device__ __forceinline__ void store_k(const u32x4 r[4], h16* ks, int tid) {
  u32x2 c[8];
  transpose4x8(r, c);
  // position p = 8 (t % 8) + i: k_key(p) = k_key(8 (t % 8)) ^ i; hd 4 (t / 8) is
  // half (t / 8) % 2 of chunk t / 16
  const int p = 8 * (tid & 7);
  const int a = (((tid >> 4) ^ k_key(p)) << 3) + (((tid >> 3) & 1) << 2);
#pragma unroll
  for (int i = 0; i < 8; ++i) *reinterpret_cast<u32x2*>(ks + (p + i) * kHd + (a ^ (i << 3))) = c[i];
}

__device__ __forceinline__ void store_v(const u32x4 r[4], h16* vs, int tid) {
  u32x2 c[8];
  transpose4x8(r, c);
  const int d = 8 * (tid & 15), g = tid >> 4;  // g: group of 4 positions
  const int a = (((2 * (g >> 2) + (g & 1)) ^ v_key(d)) << 3) + (((g >> 1) & 1) << 2);
#pragma unroll
  for (int i = 0; i < 8; ++i)
    *reinterpret_cast<u32x2*>(vs + (d + i) * kPos + (a ^ (i << 3))) = c[i];
}

// The rows of one KV head are units of Rh: each of its rep query heads by
// itself (S >= 128 tokens: Rh = S, the causal mask hides most per tile), or all
// together (Rh = rep * S, fewer empty rows).  Grid (B * nkv, units * ceil(Rh /
// 128)): the workgroups of one KV head are B * nkv apart, on one XCD (and its
// L2) whenever B * nkv is a multiple of 8, and the last tokens' tiles, the
// longest under a causal mask, start first.
// __launch_bounds__(256, 2): two workgroups per CU (64 KiB of LDS each), one's
// staging under the other's arithmetic.
template <bool MASK>
__global__ __launch_bounds__(256, 2) void prefill_kernel(
    const h16* __restrict__ q, const h16* __restrict__ ktc, const h16* __restrict__ vc,
    long max_len, int nkv, int rep, int S, int L, int units, const h16* __restrict__ mask,
    long ld_m, const uint8_t* __restrict__ cls, const unsigned long long* __restrict__ bits, int nblk,
    float inv_scale, h16* __restrict__ out, long ld_o) {
  __shared__ h16 ks[2][kPos * kHd];
  __shared__ h16 vs[2][kHd * kPos];
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int lq = lane & 31, h = lane >> 5;
  const int R = rep / units * S;  // rows per unit
  const int bg = blockIdx.x, unit = blockIdx.y % units;
  const int qt = (int)(gridDim.y / units) - 1 - (int)(blockIdx.y / units);
  const int row0 = qt * kRows + 32 * wave, row = row0 + lq;
  const h16* kt = ktc + (long)bg * kHd * max_len;
  const h16* v = vc + (long)bg * max_len * kHd;
  const int ntile = (L + kPos - 1) / kPos;
  const int s = row < R ? row % S : 0;  // token of this lane's row

  half8_t qr[8];
#pragma unroll
  for (int u = 0; u < 8; ++u) {
    u32x4 w = {0, 0, 0, 0};
    if (row < R)
      w = *reinterpret_cast<const u32x4*>(q + (((long)bg * units + unit) * R + row) * kHd + 16 * u + 8 * h);
    qr[u] = __builtin_bit_cast(half8_t, w);
  }

  // Tiles that some wave computes: class bytes of this workgroup's four row
  // blocks, 64 tiles at a time (lane = tile), and the set that is not
  // all-skipped.
  int base = 0;
  uint32_t cw = 0;
  unsigned long long todo = 0;
  auto fetch = [&]() {
    const int t = base + lane;
    uint32_t w = 0;
    if (t < ntile) {
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const int blk = qt * 4 + i;
        uint32_t c = kSkip;
        if (blk < nblk) c = MASK ? (uint32_t)cls[(long)t * nblk + blk] : (uint32_t)kClear;
        w |= c << (8 * i);
      }
    }
    cw = w;
    todo = __ballot(w != 0);
  };
  // the next tile (or -1) and this wave's class of it
  auto next = [&](uint32_t& c) -> int {
    while (todo == 0) {
      base += 64;
      if (base >= ntile) return -1;
      fetch();
    }
    const int i = __builtin_ctzll(todo);
    todo &= todo - 1;
    c = ((uint32_t)__builtin_amdgcn_readlane((int)cw, i) >> (8 * wave)) & 0xffu;
    return base + i;
  };

  float16_t o[4];
#pragma unroll
  for (int d = 0; d < 4; ++d) o[d] = (float16_t)(0.f);
  float mx = -__builtin_inff(), sum = 0.f;
  const float scale = inv_scale * kLog2e;

  fetch();
  uint32_t cur_c = kSkip, nxt_c = kSkip;
  int cur = next(cur_c);
  u32x4 st[4];
  if (cur >= 0) {
    load_k(st, kt, max_len, cur * kPos, L, tid);
    store_k(st, ks[0], tid);
    load_v(st, v, cur * kPos, L, tid);
    store_v(st, vs[0], tid);
  }
  // LDS chunk of this lane's operands: (2 u + h) ^ key, and k_key(32 b + lq) =
  // k_key(lq) ^ 4 b, v_key(32 d + lq) = v_key(lq) ^ 4 (d % 2)
  const int ka = lq * kHd + ((h ^ k_key(lq)) << 3), va = lq * kPos + ((h ^ v_key(lq)) << 3);
  __syncthreads();
  for (int buf = 0; cur >= 0; buf ^= 1) {
    const int nxt = next(nxt_c);
    // the next tile's keys under the score product, its values under the
    // softmax and the value product: 16 staging registers, not 32
    if (nxt >= 0) load_k(st, kt, max_len, nxt * kPos, L, tid);
    float16_t sc[2];
    if (cur_c != kSkip) {  // wave-uniform
#pragma unroll
      for (int b = 0; b < 2; ++b) {
        sc[b] = (float16_t)(0.f);
#pragma unroll
        for (int u = 0; u < 8; ++u) {
          const half8_t a =
              *reinterpret_cast<const half8_t*>(ks[buf] + 32 * b * kHd + (ka ^ ((2 * u ^ 4 * b) << 3)));
          sc[b] = __builtin_amdgcn_mfma_f32_32x32x16_f16(a, qr[u], sc[b], 0, 0, 0);
        }
      }
    }
    if (nxt >= 0) {
      store_k(st, ks[buf ^ 1], tid);
      load_v(st, v, nxt * kPos, L, tid);
    }
    if (cur_c != kSkip) {
      // element r of block b: position 32 b + 8 (r / 4) + 4 h + r % 4 of the tile
      const int p0 = cur * kPos;
      if (MASK && cur_c == kValues) {
        // the torch formulation's rounding steps: fp16 scores, scaled, masked
        const h16* mr = mask + (long)s * ld_m;
#pragma unroll
        for (int b = 0; b < 2; ++b)
#pragma unroll
          for (int r = 0; r < 16; ++r) {
            const int p = p0 + 32 * b + 8 * (r >> 2) + 4 * h + (r & 3);
            const float m = p < L ? (float)mr[p] : -__builtin_inff();
            const h16 a = (h16)((float)(h16)sc[b][r] * inv_scale);
            sc[b][r] = p < L ? (float)(h16)((float)a + m) * kLog2e : -__builtin_inff();
          }
      } else {
#pragma unroll
        for (int b = 0; b < 2; ++b) sc[b] *= scale;
        if ((MASK && cur_c == kBits) || p0 + kPos > L) {
          unsigned long long w = 0;
          if (MASK && cur_c == kBits) w = bits[(long)cur * S + s];
          if (p0 + kPos > L) w |= ~0ull << (L - p0);
#pragma unroll
          for (int b = 0; b < 2; ++b) {
            const uint32_t wb = (uint32_t)(w >> (32 * b + 4 * h));
#pragma unroll
            for (int r = 0; r < 16; ++r)
              if ((wb >> (8 * (r >> 2) + (r & 3))) & 1u) sc[b][r] = -__builtin_inff();
          }
        }
      }
      float tm = sc[0][0];
#pragma unroll
      for (int b = 0; b < 2; ++b)
#pragma unroll
        for (int r = 0; r < 16; ++r) tm = fmaxf(tm, sc[b][r]);
      tm = fmaxf(tm, __shfl_xor(tm, 32, 64));
      const float nm = fmaxf(mx, tm);
      // a row with nothing visible yet keeps sum 0 (and ends as 0 / 0, the
      // softmax of a fully masked row)
      const float ref = nm == -__builtin_inff() ? 0.f : nm;
      if (__any(nm != mx)) {
        const float al = __builtin_amdgcn_exp2f(mx - ref);
        sum *= al;
#pragma unroll
        for (int d = 0; d < 4; ++d) o[d] *= al;
        mx = nm;
      }
      half8_t p[4];
#pragma unroll
      for (int b = 0; b < 2; ++b)
#pragma unroll
        for (int r = 0; r < 16; ++r) {
          const float e = __builtin_amdgcn_exp2f(sc[b][r] - ref);
          sum += e;
          p[2 * b + (r >> 3)][r & 7] = (h16)e;
        }
#pragma unroll
      for (int d = 0; d < 4; ++d) {
#pragma unroll
        for (int u = 0; u < 4; ++u) {
          const half8_t a =
              *reinterpret_cast<const half8_t*>(vs[buf] + 32 * d * kPos + (va ^ ((2 * u ^ 4 * (d & 1)) << 3)));
          o[d] = __builtin_amdgcn_mfma_f32_32x32x16_f16(a, p[u], o[d], 0, 0, 0);
        }
      }
    }
    if (nxt >= 0) store_v(st, vs[buf ^ 1], tid);
    __syncthreads();
    cur = nxt;
    cur_c = nxt_c;
  }

  // O^T / sum, through LDS (each wave its own 8 KiB) to whole rows: 16-byte
  // chunks of a row's 256 bytes at chunk ^ (row & 15)
  sum += __shfl_xor(sum, 32, 64);
  const float is = 1.f / sum;
  h16* os = &ks[0][0] + wave * (32 * kHd);
#pragma unroll
  for (int d = 0; d < 4; ++d)
#pragma unroll
    for (int r = 0; r < 16; r += 4) {
      const int dd = 32 * d + 2 * r + 4 * h;
      half4_t w;
#pragma unroll
      for (int i = 0; i < 4; ++i) w[i] = (h16)(o[d][r + i] * is);
      *reinterpret_cast<half4_t*>(os + lq * kHd + (((dd >> 3) ^ (lq & 15)) << 3) + (dd & 7)) = w;
    }
  __syncthreads();
  const int b = bg / nkv, g = bg - b * nkv;
#pragma unroll
  for (int i = 0; i < 8; ++i) {
    const int lr = 4 * i + (lane >> 4), c = lane & 15, rw = row0 + lr;
    if (rw < R) {
      const int head = rw / S, tok = rw - head * S;  // head of the unit
      const u32x4 w = *reinterpret_cast<const u32x4*>(os + lr * kHd + ((c ^ (lr & 15)) << 3));
      *reinterpret_cast<u32x4*>(out + ((long)b * S + tok) * ld_o +
                                (g * rep + unit + head) * kHd + 8 * c) = w;
    }
  }
}

bool al16(const void* p) { return ((uintptr_t)p & 15) == 0; }
long unit_rows(long S, long rep) { return S >= kRows ? S : rep * S; }
long round16(long n) { return (n + 15) / 16 * 16; }

}  // namespace

// Mask words, then class bytes.  See include/hn_int4.h.
extern "C" long hn_attn_prefill_workspace_bytes(long S, long rep, long L) {
  if (S <= 0 || rep <= 0 || L <= 0) return 0;
  const long tiles = (L + kPos - 1) / kPos, nblk = (unit_rows(S, rep) + 31) / 32;
  return round16(tiles * S * 8) + tiles * nblk;
}

// Attention of S query tokens per sequence over the KV cache.  See
// include/hn_int4.h.
extern "C" int hn_attn_prefill(const void* q, const void* kt, const void* v, long max_len, long B,
                               long nkv, long rep, long hd, long S, long L, const void* mask,
                               long ld_m, float inv_scale, void* out, long ld_o, void* work,
                               void* stream) {
  HN_ARG_CHECK(B >= 0 && S >= 0 && nkv > 0 && rep > 0 && hd == kHd,
               "hn_attn_prefill: need head_dim 128 and nkv, rep > 0");
  HN_ARG_CHECK(L >= 1 && L <= max_len && max_len % 8 == 0 && max_len < (1L << 31) - kPos,
               "hn_attn_prefill: need 1 <= L <= max_len, max_len %% 8 == 0");
  HN_ARG_CHECK(rep * S < (1L << 22) && B * nkv < (1L << 31),
               "hn_attn_prefill: rep * S or B * nkv too large");
  if (B == 0 || S == 0) return 0;
  HN_ARG_CHECK(al16(q) && al16(kt) && al16(v) && al16(out) && ld_o % 8 == 0 &&
                   ld_o >= nkv * rep * hd,
               "hn_attn_prefill: operands must be 16-byte aligned, ld_o >= heads * 128");
  HN_ARG_CHECK(!mask || (work && al16(work) && ld_m >= L),
               "hn_attn_prefill: a mask needs work and ld_m >= L");
  const long R = unit_rows(S, rep), units = S >= kRows ? rep : 1, tiles = (L + kPos - 1) / kPos, nblk = (R + 31) / 32;
  HN_ARG_CHECK(!mask || tiles <= 65535, "hn_attn_prefill: too many positions for a mask");
  hipStream_t st = (hipStream_t)stream;
  const dim3 grid((unsigned)(B * nkv), (unsigned)(units * ((R + kRows - 1) / kRows)));
  unsigned long long* bits = (unsigned long long*)work;
  uint8_t* cls = mask ? (uint8_t*)work + round16(tiles * S * 8) : nullptr;
  if (mask) {
    hipLaunchKernelGGL(mask_kernel, dim3((unsigned)((nblk + 3) / 4), (unsigned)tiles), dim3(256),
                       0, st, (const h16*)mask, ld_m, (int)S, (int)R, (int)L, (int)nblk, cls,
                       bits);
    HN_LAUNCH_CHECK("hn_attn_prefill");
  }
#define HN_PREFILL(M)                                                                            \
  hipLaunchKernelGGL(prefill_kernel<M>, grid, dim3(256), 0, st, (const h16*)q, (const h16*)kt,   \
                     (const h16*)v, max_len, (int)nkv, (int)rep, (int)S, (int)L, (int)units,     \
                     (const h16*)mask, ld_m, cls, bits, (int)nblk, inv_scale, (h16*)out, ld_o)
  if (mask)
    HN_PREFILL(true);
  else
    HN_PREFILL(false);
#undef HN_PREFILL
  HN_LAUNCH_CHECK("hn_attn_prefill");
  return 0;
}
