// W4A16 GEMM for a middle number of tokens per weight matrix (about 17 to a
// few hundred), gfx950: too many for the streaming decode kernels' whole-K
// activation staging (hn_stream.hip), too few to fill the prefill GEMM's
// 256-token tiles (hn_gemm.hip).
//
//   out[m, n] = sum_k x[m, k] * W[n, k],   W[n, k] = (nibble - 8) * scale[n, k / group]
//
// Replaces the Triton int4_matmul_kernel (kernels/int4_gemm.py:25-121) and its
// SwiGLU epilogue (kernels/int4_gemm.py:175-193) at these sizes, single or
// grouped over the active experts of a MoE layer (model/mixtral.py:327-368,
// model/glm4.py:421-466).
//
// Up to about 100 tokens per matrix the weight bytes bound the product, so the
// kernel is built to keep HBM reads in flight:
//  * Tile = 256 weight rows x up to 16 RBM tokens, one workgroup of four waves,
//    two workgroups per CU.  A wave owns 64 weight rows (four 16-row tiles of
//    one matrix, or two of gate and the same two of up, so the SwiGLU epilogue
//    finds both values of an output in one lane).
//  * Weights go HBM -> VGPR: each weight is used by one wave only, so LDS would
//    add a trip and nothing else.  One load instruction covers 16 rows x 64
//    bytes (128 k), lane (row l % 16, 16 bytes at 16 (l / 16)): the B operand of
//    four v_mfma_f32_16x16x32_f16.  Two register buffers: stage s + 1
//    is in flight while stage s (128 k) computes.
//  * Activations go L2 -> LDS directly (buffer_load ... lds) into two stage
//    slots, rows XOR-swizzled by 16-byte chunk (1.4 to 2.5 bank conflict cycles per
//    LDS instruction are left); one barrier per stage.
//  * Where the tiles alone would leave CUs idle, K is split over the waves of a
//    workgroup (mid_kwave_kernel), or over workgroups where that does not apply: the
//    splits store fp32 partials, and the last of a tile to arrive (per wave,
//    hn_arrive) sums them in split order and writes the result, all of a
//    thread's loads in flight; grouped launches leave them to the MoE unpermute.
//  * Group scales: SC multiplies the fp32 partial of each 128-k group (group a
//    multiple of 128); otherwise each unpacked weight is multiplied in fp16 and
//    rounded once, the reference's dequantised weight.
#include "hn_lds_dma.h"

namespace {

constexpr int kWaves = 4;
constexpr int kTN = 4;                       // 16-row weight tiles per wave
constexpr int kBN = kWaves * kTN * 16;       // weight rows per workgroup tile
constexpr int kStageK = 128;
constexpr int kRowB = kStageK * 2;           // bytes of one staged activation row
constexpr int kMaxProb = 256;
constexpr uint32_t kOOB = 0x7ffffff0u;
// Workspace: tagged counters (hn_arrive) first, partials past the counter
// regions of the other split kernels, which share the buffer.
constexpr long kPartOffset = 2u << 20;
constexpr long kMaxCounters = 1L << 16;

struct MExpert {
  const uint8_t* gate_q; const h16* gate_s;
  const uint8_t* up_q;   const h16* up_s;
  const uint8_t* down_q; const h16* down_s;
};

struct MidArgs {
  const h16* x; long ld_x; int M;
  const uint8_t* q[2];
  const h16* s[2];
  h16* out; long ld_o;
  int phase;          // grouped: 0 gate/up + SiLU (N = I, K = H); 1 down (N = H, K = I)
  int E;
  int N, K, group;
  int ld_q;           // packed row stride (bytes)
  int ld_s;           // scale row stride (elements)
  int ks;             // K splits per tile
  int sv;             // scales per load when staging them (8, 2 or 1, by alignment)
  float* part;        // PART: [ks][MATS][part_rows][N] fp32
  long part_rows;
  unsigned long long* ctr;  // SUM: [tiles][kWaves] tagged counters, left zero
  unsigned long long tag;
  uint32_t m_pair, magic;
};

// Eight exact fp16 (n_k - 8), k = 0..7 in order, from one packed dword; with
// MUL also times the fp16 scale pair (rounded once).
template <bool MUL>
__device__ __forceinline__ half8_t unpack8(uint32_t w, const DeqRegs& c, half2_t s2) {
  u32x4 r;
  uint32_t t[4];
#pragma unroll
  for (int j = 0; j < 4; ++j) t[j] = __builtin_amdgcn_perm(w, w, 0x01010101u * j);  // byte j, 4 times
#pragma unroll
  for (int j = 0; j < 4; ++j) {
    const half2_t v = hn_bits_h2((t[j] & c.m_pair) | c.magic);  // (1024+n, 1024+16n')
    half2_t d = __builtin_elementwise_fma(v, hn_bits_h2(c.mul), hn_bits_h2(c.add));
    if (MUL) d = d * s2;
    r[j] = __builtin_bit_cast(uint32_t, d);
  }
  return __builtin_bit_cast(half8_t, r);
}

// The weights of one 128-k stage for this wave: lane (r = l % 16, c = l / 16)
// holds row 16 b + r, k 32 c .. + 32 of tile b.
struct WStage {
  u32x4 w[kTN];
};

// One tile, or a K split of it: stages [sb, se) of a problem's rows against 256 /
// MATS output columns from n-tile ntile.
struct Item {
  const h16* x;
  h16* out;
  const uint8_t* q[2];
  const h16* s[2];
  long prow;   // first row in the partial planes
  int rows;    // valid rows of this m-tile
  int nrb;     // 16-row blocks holding them
  int ntile, ks, sb, se;
  int id;      // tile number (counters)
};

// What a tile's loads need.
struct TileSrc {
  const void* px; int nx;     // activation rows of the tile, from k = 0; their bytes
  const void* pq[2]; int nq;  // packed matrices
  uint32_t vq[kTN];           // lane byte offsets (out-of-range rows: kOOB)
};

template <int MATS>
__device__ __forceinline__ int tile_mat(int b) { return MATS == 2 ? b / (kTN / 2) : 0; }

// Weight loads of stage g (k 128 g ..): the row and chunk are in voffset (what
// the range check covers), the stage in soffset.  real false: the same number
// of loads against an empty range (nothing is read, zeros come back).
template <int MATS>
__device__ __forceinline__ void issue_w(WStage& ws, const TileSrc& t, int g, bool real) {
#pragma unroll
  for (int b = 0; b < kTN; ++b) {
    const __amdgpu_buffer_rsrc_t r = rsrc(t.pq[tile_mat<MATS>(b)], real ? t.nq : 0);
    ws.w[b] = __builtin_bit_cast(
        u32x4, __builtin_amdgcn_raw_buffer_load_b128(r, t.vq[b], 64 * g, 0));
  }
}
constexpr int kWLoads = kTN;  // per wave and stage

// The scales of the wave's 64 weight rows, copied to LDS in runs of kMaxScales per
// row ([row][kScalePitch] fp16, the wave's own region): read per stage from memory
// they are one 2-byte gather over 16 rows per tile and stage, which costs the
// CU's L1 about 65 clocks against 35 for a 1 KiB weight load (measured, L2-resident;
// the grouped gate/up of 8 experts x 25 rows 183 -> 145 us without them).  A run is
// loaded when the stages of the one before are done, which waits for the loads of
// one stage; with K split so that one run covers a split instead (2 splits at group 64
// and 4 at group 32 of K = 4096, whatever the tiles), the partials cost more: us
// by splits / by runs, 1500 x 4096 x 4096 group 64 117 / 71, group 32 128 / 73;
// 512 x 14336 x 4096 group 32 171 / 77.  The pitch spreads 16 rows over the banks.
constexpr int kMaxScales = 32;
constexpr int kScalePitch = kMaxScales + 2;
constexpr int kScaleBytes = kTN * 16 * kScalePitch * 2;  // per wave

template <int V> struct ScaleVec;
template <> struct ScaleVec<1> { typedef uint16_t T; };
template <> struct ScaleVec<2> { typedef uint32_t T; };
template <> struct ScaleVec<8> { typedef u32x4 T; };

// V scales per load; cnt scales per row from element e0 of the row.
template <int MATS, int V, int PITCH = kScalePitch>
__device__ __forceinline__ void stage_scales_v(const void* const (&ps)[2], int ns, int N, int ld_s,
                                               int nw, int e0, int cnt, uint32_t dst, int lane) {
  const int per_row = (cnt + V - 1) / V;
  for (int i = lane; i < kTN * 16 * per_row; i += 64) {
    const int r = i / per_row, c = (i - r * per_row) * V;
    const int b = r >> 4;
    const int row = nw + 16 * (MATS == 2 ? b % (kTN / 2) : b) + (r & 15);
    const uint32_t off = row < N ? (uint32_t)(2 * (row * ld_s + e0 + c)) : kOOB;
    const __amdgpu_buffer_rsrc_t r0 = rsrc(ps[0], ns);
    const __amdgpu_buffer_rsrc_t r1 = rsrc(ps[MATS - 1], ns);
    const bool second = MATS == 2 && b >= kTN / 2;
    typename ScaleVec<V>::T v;
    const uint32_t off0 = second ? kOOB : off, off1 = second ? off : kOOB;
    __attribute__((address_space(3))) char* p =
        (__attribute__((address_space(3))) char*)nullptr + dst + r * (PITCH * 2) + 2 * c;
    if constexpr (V == 8) {
      u32x4 v4 = __builtin_bit_cast(u32x4, __builtin_amdgcn_raw_buffer_load_b128(r0, off0, 0, 0));
      if (MATS == 2)
        v4 |= __builtin_bit_cast(u32x4, __builtin_amdgcn_raw_buffer_load_b128(r1, off1, 0, 0));
#pragma unroll
      for (int j = 0; j < 4; ++j)
        *reinterpret_cast<__attribute__((address_space(3))) uint32_t*>(p + 4 * j) = v4[j];
    } else if constexpr (V == 2) {
      uint32_t v2 = __builtin_amdgcn_raw_buffer_load_b32(r0, off0, 0, 0);
      if (MATS == 2) v2 |= __builtin_amdgcn_raw_buffer_load_b32(r1, off1, 0, 0);
      *reinterpret_cast<__attribute__((address_space(3))) uint32_t*>(p) = v2;
    } else {
      uint16_t v1 = __builtin_amdgcn_raw_buffer_load_b16(r0, off0, 0, 0);
      if (MATS == 2) v1 |= __builtin_amdgcn_raw_buffer_load_b16(r1, off1, 0, 0);
      *reinterpret_cast<__attribute__((address_space(3))) uint16_t*>(p) = v1;
    }
  }
}

// Activation loads of a stage: NRB loads of 1 KiB per wave.  LDS chunk L =
// (row r, slot c') holds 16-byte chunk c' ^ (r % 16) of row r; rows past the
// valid ones repeat the last one (their results are never stored).
template <int NRB>
__device__ __forceinline__ void a_offsets(uint32_t (&va)[NRB], int wave, int lane, int rows,
                                          long ld_x) {
#pragma unroll
  for (int j = 0; j < NRB; ++j) {
    const int L = (wave * NRB + j) * 64 + lane;
    const int r = L >> 4, c = (L & 15) ^ (r & 15);
    va[j] = (uint32_t)(min(r, rows - 1) * (int)ld_x * 2 + 16 * c);
  }
}

template <int NRB>
__device__ __forceinline__ void issue_a(const uint32_t (&va)[NRB], const TileSrc& t, int s,
                                        uint32_t st, int wave, bool real) {
  const __amdgpu_buffer_rsrc_t r = rsrc(t.px, real ? t.nx : 0);
#pragma unroll
  for (int j = 0; j < NRB; ++j)
    dma_b128(r, va[j], kRowB * s, st + (wave * NRB + j) * 1024);
}

// One stage: NRB x kTN blocks of 16 tokens x 16 weight rows over 128 k.  Lane
// (t = l % 16, c = l / 16) supplies A[token t][k 32 c + 8 d ..] at step d.
// sc: LDS address of the scale of the lane's row in tile 0.
template <int NRB, bool SC, int PITCH = kScalePitch>
__device__ __forceinline__ void compute_stage(const WStage& ws, uint32_t st, uint32_t sc, int col,
                                              int q, const DeqRegs& dr,
                                              float4_t (&acc)[NRB][kTN]) {
  const float4_t zero = {0.f, 0.f, 0.f, 0.f};
  float4_t tmp[NRB][kTN];
  uint32_t sv[kTN];
#pragma unroll
  for (int b = 0; b < kTN; ++b) sv[b] = lds_read<uint16_t>(sc + b * 16 * PITCH * 2);
  half8_t a[2][NRB];  // step d + 1's A reads go out before step d's MFMAs
  const uint32_t row = st + col * kRowB;
#pragma unroll
  for (int rb = 0; rb < NRB; ++rb)
    a[0][rb] = lds_read<half8_t>(row + rb * 16 * kRowB + ((4 * q ^ col) << 4));
#pragma unroll
  for (int d = 0; d < 4; ++d) {
    if (d < 3) {
#pragma unroll
      for (int rb = 0; rb < NRB; ++rb)
        a[(d + 1) & 1][rb] =
            lds_read<half8_t>(row + rb * 16 * kRowB + (((4 * q + d + 1) ^ col) << 4));
    }
#pragma unroll
    for (int b = 0; b < kTN; ++b) {
      half8_t w;
      if (SC) {
        w = unpack8<false>(ws.w[b][d], dr, half2_t{});
      } else {
        w = unpack8<true>(ws.w[b][d], dr, hn_bits_h2(sv[b] | (sv[b] << 16)));
      }
#pragma unroll
      for (int rb = 0; rb < NRB; ++rb) {
        if (SC)
          tmp[rb][b] = __builtin_amdgcn_mfma_f32_16x16x32_f16(
              a[d & 1][rb], w, d == 0 ? zero : tmp[rb][b], 0, 0, 0);
        else
          acc[rb][b] =
              __builtin_amdgcn_mfma_f32_16x16x32_f16(a[d & 1][rb], w, acc[rb][b], 0, 0, 0);
      }
    }
    __builtin_amdgcn_sched_barrier(0);
  }
  if (SC) {
#pragma unroll
    for (int b = 0; b < kTN; ++b) {
      const float sf = (float)__builtin_bit_cast(h16, (uint16_t)sv[b]);
#pragma unroll
      for (int rb = 0; rb < NRB; ++rb)
#pragma unroll
        for (int r = 0; r < 4; ++r)
          acc[rb][b][r] = __builtin_fmaf(sf, tmp[rb][b][r], acc[rb][b][r]);
    }
  }
}

// The stages of an item, two slots.  At stage s: wait for its own activation
// loads (only s's weight loads, issued after them, may still be in flight),
// meet the other waves, request stage s + 1 into the slot that stage s - 1 has
// left, compute.  Past the end the requests go out against empty ranges, so
// the count of loads after a stage's activations is fixed.
template <int MATS, int NRB, int RBM, bool SC>
__device__ __forceinline__ void k_loop(const MidArgs& A, const Item& it, const TileSrc& t, int nw,
                                       uint32_t lds0, const uint32_t (&va)[NRB], int wave,
                                       int lane, const DeqRegs& dr, float4_t (&acc)[NRB][kTN]) {
  constexpr uint32_t kStageB = NRB * 16 * kRowB;
  const int col = lane & 15, q = lane >> 4;
  const int s0 = it.sb, s1 = it.se;
  WStage ws0, ws1;
  stage_barrier();  // the previous item's last LDS reads are done
  issue_a<NRB>(va, t, s0, lds0, wave, true);
  __builtin_amdgcn_sched_barrier(0);
  issue_w<MATS>(ws0, t, s0, true);
  __builtin_amdgcn_sched_barrier(0);
  const int sps = kStageK / A.group, run = kMaxScales / sps;  // scales, stages per run: even
  const uint32_t scw = lds0 + (uint32_t)(2 * RBM * 16 * kRowB) + wave * kScaleBytes;
  uint32_t sc = 0;
  auto stage = [&](int s, const WStage& cur, WStage& nxt, uint32_t stc, uint32_t stn) {
    wait_vmcnt<kWLoads>();
    stage_barrier();
    const bool more = s + 1 < s1;  // uniform
    issue_a<NRB>(va, t, s + 1, stn, wave, more);
    __builtin_amdgcn_sched_barrier(0);
    issue_w<MATS>(nxt, t, s + 1, more);
    __builtin_amdgcn_sched_barrier(0);
    compute_stage<NRB, SC>(cur, stc, sc, col, q, dr, acc);
    sc += 2 * sps;
  };
  int s = s0;
  for (int r0 = s0; r0 < s1; r0 += run) {
    // the run's scales, the first behind the first stage's loads
    const int r1 = min(r0 + run, s1);
    const void* const ps[2] = {it.s[0], it.s[MATS - 1]};
    const int ns = A.N * A.ld_s * 2, cnt = (r1 - r0) * sps, e0 = r0 * sps;
    if (A.sv == 8)  // uniform
      stage_scales_v<MATS, 8>(ps, ns, A.N, A.ld_s, nw, e0, cnt, scw, lane);
    else if (A.sv == 2)
      stage_scales_v<MATS, 2>(ps, ns, A.N, A.ld_s, nw, e0, cnt, scw, lane);
    else
      stage_scales_v<MATS, 1>(ps, ns, A.N, A.ld_s, nw, e0, cnt, scw, lane);
    sc = scw + col * (kScalePitch * 2) + 2 * (q * sps / 4);
    for (; s + 2 <= r1; s += 2) {
      stage(s, ws0, ws1, lds0, lds0 + kStageB);
      stage(s + 1, ws1, ws0, lds0 + kStageB, lds0);
    }
  }
  if (s < s1) {  // the last of an odd number: nothing left to request
    wait_vmcnt<kWLoads>();
    stage_barrier();
    compute_stage<NRB, SC>(ws0, lds0, sc, col, q, dr, acc);
  }
  // the requests past the end have landed before another item's may be issued
  wait_vmcnt<0>();
}

__device__ __forceinline__ h16 swiglu16(float g, float u) {
  return (h16)(hn_silu((float)(h16)g) * (float)(h16)u);
}

// Launch-wide lookup of items (LDS).
struct Lookup {
  const int* mt_off;  // m-tiles per problem, prefix
  const int* s_row;   // first row, rows and expert of each problem
  const int* s_cnt;
  const int* s_exp;
  int nprob, NT;
};

template <bool GROUPED>
__device__ __forceinline__ Item find_item(const MidArgs& A, const Lookup& lk,
                                          const MExpert* __restrict__ table, int i) {
  // item -> (problem, n-tile, k split, m-tile), m-tiles fastest
  const int per_mt = lk.NT * A.ks;
  int p = 0;
  if (GROUPED) {
    const int key = i / per_mt;  // mt_off[p] <= key < mt_off[p + 1]
    int lo = 0, hi = lk.nprob - 1;
    while (lo < hi) {
      const int mid = (lo + hi + 1) >> 1;
      if (lk.mt_off[mid] <= key) lo = mid; else hi = mid - 1;
    }
    p = __builtin_amdgcn_readfirstlane(lo);
  }
  const int mt0 = __builtin_amdgcn_readfirstlane(lk.mt_off[p]);
  const int nmt = __builtin_amdgcn_readfirstlane(lk.mt_off[p + 1]) - mt0;
  const int loc = i - mt0 * per_mt;
  const int rest = loc / nmt, mtile = loc - rest * nmt;
  Item it;
  it.ntile = rest / A.ks;
  it.ks = rest - it.ntile * A.ks;
  it.id = (mt0 + mtile) * lk.NT + it.ntile;
  const int T = A.K / kStageK;
  it.sb = (int)((long)T * it.ks / A.ks);
  it.se = (int)((long)T * (it.ks + 1) / A.ks);
  int rows_p, row0 = 0;
  if (GROUPED) {
    const int e = __builtin_amdgcn_readfirstlane(lk.s_exp[p]);
    row0 = __builtin_amdgcn_readfirstlane(lk.s_row[p]);
    rows_p = __builtin_amdgcn_readfirstlane(lk.s_cnt[p]);
    const MExpert ew = table[e];
    if (A.phase == 0) {
      it.q[0] = ew.gate_q; it.s[0] = ew.gate_s;
      it.q[1] = ew.up_q;   it.s[1] = ew.up_s;
    } else {
      it.q[0] = it.q[1] = ew.down_q;
      it.s[0] = it.s[1] = ew.down_s;
    }
  } else {
    rows_p = A.M;
    it.q[0] = A.q[0]; it.s[0] = A.s[0];
    it.q[1] = A.q[1]; it.s[1] = A.s[1];
  }
  // a problem's rows are dealt evenly to its m-tiles in blocks of 16
  const int blocks = (rows_p + 15) >> 4;
  const int b0 = blocks * mtile / nmt, b1 = blocks * (mtile + 1) / nmt;
  it.nrb = b1 - b0;
  it.rows = min(16 * it.nrb, rows_p - 16 * b0);
  it.x = A.x + (long)(row0 + 16 * b0) * A.ld_x;
  it.out = A.out + (long)(row0 + 16 * b0) * A.ld_o;
  it.prow = row0 + 16 * b0;
  return it;
}

// Where an item's results go: fp16 out; fp32 partials of its K split, left to
// the caller; or the same summed by the tile's last split to arrive.
enum { kOut = 0, kPart = 1, kSum = 2 };

// The wave's output columns of a tile, summed over its K splits in order: a
// thread takes four columns of a row at a time, two such and eight splits' loads
// in flight together.
template <int MATS>
__device__ __forceinline__ void sum_tile(const MidArgs& A, const Item& it, int nw, int lane) {
  constexpr int kCols = kTN * 16 / MATS, kC4 = kCols / 4;
  const long plane = A.part_rows * (long)A.N;
  const int n_e = it.rows * kC4;
  for (int e0 = lane; e0 < n_e; e0 += 128) {
    float4_t v[2][MATS];
    const float* p[2];
#pragma unroll
    for (int u = 0; u < 2; ++u) {
      const int e = min(e0 + 64 * u, n_e - 1);
      const int n = min(nw + 4 * (e % kC4), A.N - 4);
      p[u] = A.part + (it.prow + e / kC4) * A.N + n;
#pragma unroll
      for (int mt = 0; mt < MATS; ++mt) v[u][mt] = float4_t{0.f, 0.f, 0.f, 0.f};
    }
    for (int kb = 0; kb < A.ks; kb += 8) {
      float4_t t[2][8][MATS];
#pragma unroll
      for (int u = 0; u < 2; ++u)
#pragma unroll
        for (int j = 0; j < 8; ++j)
#pragma unroll
          for (int mt = 0; mt < MATS; ++mt)
            t[u][j][mt] = *reinterpret_cast<const float4_t*>(
                p[u] + ((long)min(kb + j, A.ks - 1) * MATS + mt) * plane);
#pragma unroll
      for (int u = 0; u < 2; ++u)
#pragma unroll
        for (int j = 0; j < 8; ++j)
#pragma unroll
          for (int mt = 0; mt < MATS; ++mt)
            if (kb + j < A.ks) v[u][mt] += t[u][j][mt];
    }
#pragma unroll
    for (int u = 0; u < 2; ++u) {
      const int e = e0 + 64 * u;
      const int n = nw + 4 * (e % kC4);
      if (e < n_e && n < A.N) {
        h16* o = it.out + (long)(e / kC4) * A.ld_o + n;
#pragma unroll
        for (int j = 0; j < 4; ++j)
          o[j] = MATS == 2 ? swiglu16(v[u][0][j], v[u][MATS - 1][j]) : (h16)v[u][0][j];
      }
    }
  }
}

template <int MATS, int NRB, int RBM, bool SC, int OUT>
__device__ __forceinline__ void run_item(const MidArgs& A, const Item& it, uint32_t lds0,
                                         int wave, int lane, const DeqRegs& dr) {
  constexpr int kCols = kTN * 16 / MATS;  // output columns per wave
  const int col = lane & 15, q = lane >> 4;
  const int N = A.N;
  TileSrc t;
  t.px = it.x;
  t.nx = (int)(((long)(it.rows - 1) * A.ld_x + A.K) * 2);
  t.nq = N * A.ld_q;
  const int nw = it.ntile * (kWaves * kCols) + wave * kCols;  // the wave's first output column
#pragma unroll
  for (int m = 0; m < 2; ++m) t.pq[m] = it.q[MATS == 2 ? m : 0];
#pragma unroll
  for (int b = 0; b < kTN; ++b) {
    const int row = nw + 16 * (MATS == 2 ? b % (kTN / 2) : b) + col;
    t.vq[b] = row < N ? (uint32_t)(row * A.ld_q + 16 * q) : kOOB;
  }
  uint32_t va[NRB];
  a_offsets<NRB>(va, wave, lane, it.rows, A.ld_x);
  float4_t acc[NRB][kTN];
#pragma unroll
  for (int rb = 0; rb < NRB; ++rb)
#pragma unroll
    for (int b = 0; b < kTN; ++b) acc[rb][b] = float4_t{0.f, 0.f, 0.f, 0.f};
  k_loop<MATS, NRB, RBM, SC>(A, it, t, nw, lds0, va, wave, lane, dr, acc);

  // lane: weight row 16 b + col, tokens 16 rb + 4 q + r
  const long plane = A.part_rows * (long)N;
#pragma unroll
  for (int rb = 0; rb < NRB; ++rb)
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const int m = 16 * rb + 4 * q + r;
      if (m < it.rows) {
#pragma unroll
        for (int b = 0; b < (OUT != kOut ? kTN : kTN / MATS); ++b) {
          const int n = nw + 16 * (MATS == 2 ? b % (kTN / 2) : b) + col;
          if (n < N) {
            float* const pp = A.part +
                (long)(it.ks * MATS + tile_mat<MATS>(b)) * plane + (it.prow + m) * N + n;
            if (OUT == kPart)
              *pp = acc[rb][b][r];
            else if (OUT == kSum)
              __hip_atomic_store(pp, acc[rb][b][r], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            else
              it.out[(long)m * A.ld_o + n] =
                  MATS == 2 ? swiglu16(acc[rb][b][r], acc[rb][(b + kTN / 2) % kTN][r])
                            : (h16)acc[rb][b][r];
          }
        }
      }
    }
  if constexpr (OUT == kSum) {
    hn_publish_partials();
    unsigned long long* c = A.ctr + (long)it.id * kWaves + wave;
    int n = 0;
    if (lane == 0) n = hn_arrive(c, A.tag);
    n = __builtin_amdgcn_readfirstlane(n);
    if (n != A.ks - 1) return;
    hn_acquire_agent();
    if (lane == 0) hn_counter_reset(c);
    sum_tile<MATS>(A, it, nw, lane);
  }
}

// RBM: 16-token blocks per tile at most (2: more weight loads per register, 4:
// fewer passes over the weights).
template <bool GROUPED, int MATS, int RBM, bool SC, int OUT>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(2, 2))) void mid_kernel(
    MidArgs A, const MExpert* __restrict__ table, const int* __restrict__ active,
    const int* __restrict__ n_active, const int* __restrict__ offsets) {
  static_assert(RBM == 2 || RBM == 4, "tiles of 32 or 64 tokens");
  __shared__ __align__(16) unsigned char lds[2 * RBM * 16 * kRowB + kWaves * kScaleBytes];
  __shared__ int mt_off[(GROUPED ? kMaxProb : 1) + 1];
  __shared__ int s_row[GROUPED ? kMaxProb : 1], s_cnt[GROUPED ? kMaxProb : 1];
  __shared__ int s_exp[GROUPED ? kMaxProb : 1];
  __shared__ int s_wsum[kWaves];
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const uint32_t lds0 = (uint32_t)(uintptr_t)(lds_void_t*)lds;
  DeqRegs dr;
  dr.m_pair = A.m_pair;
  dr.magic = hn_vgpr(A.magic);
  dr.mul = hn_vgpr(0x2C003C00u);  // half2(1, 0.0625)
  dr.add = hn_vgpr(0xD480E408u);  // half2(-1032, -72)
  constexpr int TM = 16 * RBM;
  constexpr int kColsWg = kBN / MATS;

  Lookup lk;
  lk.NT = (A.N + kColsWg - 1) / kColsWg;
  lk.mt_off = mt_off;
  lk.s_row = s_row;
  lk.s_cnt = s_cnt;
  lk.s_exp = s_exp;
  lk.nprob = 1;
  if (GROUPED) {
    static_assert(kMaxProb <= kWaves * 64, "one thread per problem");
    lk.nprob = min(*n_active, min(A.E, kMaxProb));
    int v = 0;
    if (tid < lk.nprob) {
      const int e = active[tid];
      const int r0 = offsets[e], n = offsets[e + 1] - r0;
      s_exp[tid] = e;
      s_row[tid] = r0;
      s_cnt[tid] = n;
      v = (n + TM - 1) / TM;
    }
    int incl = v;
#pragma unroll
    for (int off = 1; off < 64; off <<= 1) {
      const int o = __shfl_up(incl, off, 64);
      if (lane >= off) incl += o;
    }
    if (lane == 63) s_wsum[wave] = incl;
    __syncthreads();
    for (int w = 0; w < wave; ++w) incl += s_wsum[w];
    if (tid < kMaxProb) mt_off[tid + 1] = incl;
    if (tid == 0) mt_off[0] = 0;
  } else if (tid == 0) {
    mt_off[0] = 0;
    mt_off[1] = (A.M + TM - 1) / TM;
  }
  __syncthreads();
  if (lk.nprob <= 0) return;
  const int items = __builtin_amdgcn_readfirstlane(mt_off[lk.nprob]) * lk.NT * A.ks;
  const int nwg = gridDim.x;
  // workgroups are dealt round-robin to the 8 XCDs: consecutive item numbers
  // (m-tiles of one n-tile, which share its weights) run on one XCD
  const int bid = blockIdx.x;
  const int vid = (nwg % 8 == 0) ? (bid % 8) * (nwg / 8) + bid / 8 : bid;
  if (vid >= items) return;
  Item it = find_item<GROUPED>(A, lk, table, vid);
  for (int i = vid; i < items; i += nwg) {
    // the next item's lookup (its table loads) ahead of this item's K loop
    const Item nx = i + nwg < items ? find_item<GROUPED>(A, lk, table, i + nwg) : it;
    if (it.nrb == 1) run_item<MATS, 1, RBM, SC, OUT>(A, it, lds0, wave, lane, dr);
    else if (RBM == 2 || it.nrb == 2) run_item<MATS, 2, RBM, SC, OUT>(A, it, lds0, wave, lane, dr);
    else if (it.nrb == 3) run_item<MATS, RBM == 4 ? 3 : 1, RBM, SC, OUT>(A, it, lds0, wave, lane, dr);
    else run_item<MATS, RBM == 4 ? 4 : 1, RBM, SC, OUT>(A, it, lds0, wave, lane, dr);
    it = nx;
  }
}

// ---------------------------------------------------------------------------
// One problem of few tiles: K split over the eight waves of a workgroup.
//
// A K split over workgroups costs about 8 us of its own (partials out to memory,
// counter, read back: 17 x 4096 x 512 in two splits 15.5 us, whole 7.6), and a
// workgroup of a short K has little in flight.  So a workgroup takes a tile of 64 weight rows x 32 tokens whole and its waves a K
// range each: every wave stages its own activations (no barrier in the K loop, two
// slots as above) and the partials meet in LDS, summed in K order.  The
// activations are read once per 64 weight rows instead of once per 256, from L2.
// us with K over workgroups (32-token tiles) / over waves: 64 x 6144 x 4096 19.5 /
// 11.3, 64 x 4096 x 1408 15.0 / 6.8, 333 x 4096 x 4096 group 64 (whole) 36.9 / 30.3, 37
// x 4096 x 14336 27.8 / 30.0.  Bound by the stages' latency: 27 us for the 14 of a wave
// at 37 x 4096 x 14336, in which waves issue vector instructions for 28 % of their
// cycles, wait for 63 %, and the matrix cores are busy for 6 %; a third register
// buffer of weights, two stages ahead, gave nothing (32.9 against 32.7 at 128 x 4096 x
// 14336, 12.6 against 11.9 at 64 x 6144 x 4096).
// ---------------------------------------------------------------------------
constexpr int kKWaves = 8;
constexpr int kKScales = 16;                       // scales per row of a wave's K range at most
constexpr int kKPitch = kKScales + 2;
constexpr int kKSlots = 2 * 2 * 16 * kRowB;        // per wave: two slots of 32 tokens
constexpr int kKScaleBytes = kTN * 16 * kKPitch * 2;
static_assert(kKSlots >= 2 * kTN * 4 * 64 * 4, "a wave's partials fit its slots");

template <int MATS, int NRB, bool SC>
__device__ __forceinline__ void kwave_tile(const MidArgs& A, const Item& it, uint32_t lds0,
                                           int wave, int lane, const DeqRegs& dr) {
  constexpr uint32_t kStageB = NRB * 16 * kRowB;
  constexpr int kLoads = 4 * NRB;  // 1 KiB activation loads of a wave and stage
  const int col = lane & 15, q = lane >> 4;
  const int N = A.N, s0 = it.sb, s1 = it.se;
  const int nw = it.ntile * (kTN * 16 / MATS);
  TileSrc t;
  t.px = it.x;
  t.nx = (int)(((long)(it.rows - 1) * A.ld_x + A.K) * 2);
  t.nq = N * A.ld_q;
#pragma unroll
  for (int m = 0; m < 2; ++m) t.pq[m] = it.q[MATS == 2 ? m : 0];
#pragma unroll
  for (int b = 0; b < kTN; ++b) {
    const int row = nw + 16 * (MATS == 2 ? b % (kTN / 2) : b) + col;
    t.vq[b] = row < N ? (uint32_t)(row * A.ld_q + 16 * q) : kOOB;
  }
  // wave-private rows: the layout of a_offsets with one wave's loads covering all
  uint32_t va[kLoads];
#pragma unroll
  for (int j = 0; j < kLoads; ++j) {
    const int L = j * 64 + lane, r = L >> 4, c = (L & 15) ^ (r & 15);
    va[j] = (uint32_t)(min(r, it.rows - 1) * (int)A.ld_x * 2 + 16 * c);
  }
  const uint32_t st0 = lds0 + wave * kKSlots;
  auto issue_rows = [&](int s, uint32_t st, bool real) {
    const __amdgpu_buffer_rsrc_t r = rsrc(t.px, real ? t.nx : 0);
#pragma unroll
    for (int j = 0; j < kLoads; ++j) dma_b128(r, va[j], kRowB * s, st + j * 1024);
  };
  float4_t acc[NRB][kTN];
#pragma unroll
  for (int rb = 0; rb < NRB; ++rb)
#pragma unroll
    for (int b = 0; b < kTN; ++b) acc[rb][b] = float4_t{0.f, 0.f, 0.f, 0.f};

  WStage ws0, ws1;
  issue_rows(s0, st0, true);
  __builtin_amdgcn_sched_barrier(0);
  issue_w<MATS>(ws0, t, s0, true);
  __builtin_amdgcn_sched_barrier(0);
  const int sps = kStageK / A.group;
  const uint32_t scw = lds0 + (uint32_t)(kKWaves * kKSlots) + wave * kKScaleBytes;
  {
    const void* const ps[2] = {it.s[0], it.s[MATS - 1]};
    const int ns = N * A.ld_s * 2, cnt = (s1 - s0) * sps, e0 = s0 * sps;
    if (A.sv == 8)  // uniform
      stage_scales_v<MATS, 8, kKPitch>(ps, ns, N, A.ld_s, nw, e0, cnt, scw, lane);
    else if (A.sv == 2)
      stage_scales_v<MATS, 2, kKPitch>(ps, ns, N, A.ld_s, nw, e0, cnt, scw, lane);
    else
      stage_scales_v<MATS, 1, kKPitch>(ps, ns, N, A.ld_s, nw, e0, cnt, scw, lane);
  }
  uint32_t sc = scw + col * (kKPitch * 2) + 2 * (q * sps / 4);
  // as k_loop's stage, the slots being the wave's own: its loads landed and its
  // LDS reads returned are all that a slot's reuse needs
  auto stage = [&](int s, const WStage& cur, WStage& nxt, uint32_t stc, uint32_t stn) {
    wait_vmcnt<kWLoads>();
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    const bool more = s + 1 < s1;  // uniform
    issue_rows(s + 1, stn, more);
    __builtin_amdgcn_sched_barrier(0);
    issue_w<MATS>(nxt, t, s + 1, more);
    __builtin_amdgcn_sched_barrier(0);
    compute_stage<NRB, SC, kKPitch>(cur, stc, sc, col, q, dr, acc);
    sc += 2 * sps;
  };
  int s = s0;
  for (; s + 2 <= s1; s += 2) {
    stage(s, ws0, ws1, st0, st0 + kStageB);
    stage(s + 1, ws1, ws0, st0 + kStageB, st0);
  }
  if (s < s1) {
    wait_vmcnt<kWLoads>();
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    compute_stage<NRB, SC, kKPitch>(ws0, st0, sc, col, q, dr, acc);
  }
  wait_vmcnt<0>();  // requests past the end have landed: the slots are free
  asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");

  // partials by (register, lane) into the wave's slots; wave w sums register r =
  // w % 4 of two tiles (a gate and up pair with MATS 2)
  auto cell = [&](int w, int rb, int b, int r) {
    return (__attribute__((address_space(3))) float*)(
        (__attribute__((address_space(3))) char*)nullptr + lds0 + w * kKSlots +
        (((rb * kTN + b) * 4 + r) * 64 + lane) * 4);
  };
#pragma unroll
  for (int rb = 0; rb < NRB; ++rb)
#pragma unroll
    for (int b = 0; b < kTN; ++b)
#pragma unroll
      for (int r = 0; r < 4; ++r) *cell(wave, rb, b, r) = acc[rb][b][r];
  __syncthreads();
  const int r = wave & 3, h = wave >> 2;
#pragma unroll
  for (int rb = 0; rb < NRB; ++rb) {
    float v[2];
#pragma unroll
    for (int u = 0; u < 2; ++u) {
      const int b = MATS == 2 ? h + u * (kTN / 2) : 2 * h + u;
      v[u] = 0.f;
#pragma unroll
      for (int w = 0; w < kKWaves; ++w) v[u] += *cell(w, rb, b, r);
    }
    const int m = 16 * rb + 4 * q + r;
    if (m < it.rows) {
#pragma unroll
      for (int u = 0; u < 2 / MATS; ++u) {
        const int n = nw + 16 * (MATS == 2 ? h : 2 * h + u) + col;
        if (n < N)
          it.out[(long)m * A.ld_o + n] = MATS == 2 ? swiglu16(v[0], v[1]) : (h16)v[u];
      }
    }
  }
}

// One tile per workgroup: n-tile bid / mtiles, m-tiles fastest on one XCD.
template <int MATS, bool SC>
__global__ __launch_bounds__(512) __attribute__((amdgpu_waves_per_eu(2, 2))) void mid_kwave_kernel(
    MidArgs A) {
  __shared__ __align__(16) unsigned char lds[kKWaves * (kKSlots + kKScaleBytes)];
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const uint32_t lds0 = (uint32_t)(uintptr_t)(lds_void_t*)lds;
  DeqRegs dr;
  dr.m_pair = A.m_pair;
  dr.magic = hn_vgpr(A.magic);
  dr.mul = hn_vgpr(0x2C003C00u);  // half2(1, 0.0625)
  dr.add = hn_vgpr(0xD480E408u);  // half2(-1032, -72)
  const int nwg = gridDim.x, bid = blockIdx.x;
  const int vid = (nwg % 8 == 0) ? (bid % 8) * (nwg / 8) + bid / 8 : bid;
  const int nmt = (A.M + 31) >> 5;
  Item it;
  it.ntile = vid / nmt;
  const int mtile = vid - it.ntile * nmt;
  const int T = A.K / kStageK;
  it.sb = T * wave / kKWaves;
  it.se = T * (wave + 1) / kKWaves;
  it.q[0] = A.q[0]; it.s[0] = A.s[0];
  it.q[1] = A.q[1]; it.s[1] = A.s[1];
  // rows dealt evenly to the m-tiles in blocks of 16
  const int blocks = (A.M + 15) >> 4;
  const int b0 = blocks * mtile / nmt, b1 = blocks * (mtile + 1) / nmt;
  it.nrb = b1 - b0;
  it.rows = min(16 * it.nrb, A.M - 16 * b0);
  it.x = A.x + (long)(16 * b0) * A.ld_x;
  it.out = A.out + (long)(16 * b0) * A.ld_o;
  if (it.nrb == 1) kwave_tile<MATS, 1, SC>(A, it, lds0, wave, lane, dr);
  else kwave_tile<MATS, 2, SC>(A, it, lds0, wave, lane, dr);
}

// out[m, n] = the ks partials of (m, n) summed in split order; four columns per
// thread, all of its loads in flight.
__global__ __launch_bounds__(256) void mid_reduce_kernel(const float* __restrict__ part,
                                                         long plane, int ks, int M, int N,
                                                         h16* __restrict__ out, long ld_o) {
  const int n4 = N >> 2;
  const long i = (long)blockIdx.x * 256 + threadIdx.x;
  if (i >= (long)M * n4) return;
  const int m = (int)(i / n4), n = 4 * (int)(i - (long)m * n4);
  const float* p = part + (long)m * N + n;
  float4_t v = {0.f, 0.f, 0.f, 0.f};
  for (int kb = 0; kb < ks; kb += 8) {
    float4_t t[8];
#pragma unroll
    for (int j = 0; j < 8; ++j)
      t[j] = *reinterpret_cast<const float4_t*>(p + (long)min(kb + j, ks - 1) * plane);
#pragma unroll
    for (int j = 0; j < 8; ++j)
      if (kb + j < ks) v += t[j];
  }
  h16* o = out + (long)m * ld_o + n;
#pragma unroll
  for (int j = 0; j < 4; ++j) o[j] = (h16)v[j];
}

}  // namespace

// ---------------------------------------------------------------------------
// host side
// ---------------------------------------------------------------------------
namespace {

bool aligned16(const void* p) { return ((uintptr_t)p & 15) == 0; }

// Resident workgroups of mid_kernel: two per CU.
int slots() { return 2 * hn_device_cus(); }

// Single problems that mid_kernel takes.  Work in units of one tile's stage.  Measured
// on MI355X (graph replays over rotating weights, us, 32- / 64-token tiles, the
// 256-token GEMM or, at 64 tokens, the split-K kernels; M x N x K):
//     64 x  6144 x  4096     20 /  28    39      64 x 4096 x 14336       29 /  43   102
//    128 x  4096 x 14336     39 /  43    64     333 x 4096 x 14336       90 /  84   128
//   1024 x  4096 x 14336    174 / 151   152     200 x 14336 x 4096 x2    98 /  77    98
//    333 x 14336 x 4096 x2  146 / 146   139    1024 x 4096 x 1408        25 /  29    48
//    512 x  4096 x 4096 g64  38 /  44    75    1024 x 1408 x 4096        32 /  43    75
//    300 x 14336 x 4096      92 /  71   106     600 x 4096 x 4096        48 /  48    81
// so: 32-token tiles up to 8192 units (16 stages per resident workgroup), then
// 64-token tiles while they fit one round of workgroups and 16384 units, past
// which the weights' re-reads and unpacks cost more than the GEMM's tile
// padding and idle CUs.
constexpr long kUnits32 = 8192, kUnits64 = 16384;

constexpr long kLongK = 64, kSplitStages = 16;

// Where the kernels beside these are faster (us here, theirs; M x N x K, group 128
// unless said):
//  * a short K, under kShort stages: K is not split (64 x 4096 x 512 in 2 splits 17.7,
//    whole 8.3), up to 32 rows the decode kernels win (17 x 4096 x 512 7.6, 5.7; 32 x
//    4096 x 768 12.4, 12.6; 33: 9.8, 13.4), up to 64 below half of that (64 x 8192 x
//    256 6.6, 6.1); past 64 the GEMM where there are two tiles and more for a resident
//    workgroup (4096 x 4096 x 512 37, 34; 512 x 14336 x 512 gate and up 43, 32; 2048 x
//    4096 x 512 23, 35), or one up to its 128-token tile (65 x 65536 x 512 19.2, 18.5);
//  * up to kFewRows rows the decode kernels hold a long K's activations in few K
//    chunks: one matrix of K > 4096 over the waves, tiles for less than half of the
//    CUs (17 x 1024 x 7680 18.7, 15.8; 20 x 4096 x 14336 32.2, 28.7), apart from even
//    ranges of 5 to 8 stages over 64 tiles (17 x 4096 x 8192 16.4, 18.8);
//  * up to 32 rows a product too small for the reduction across workgroups (K beyond
//    what the waves' ranges take; mats * N * K against kFewWork): 20 x 5120 x 13824
//    group 64 32.5, 30.3; 21 x 14336 x 7680 group 32 43.5, 43.5; 24 x 4096 x 8192 group
//    32 24.7, 21.8; 24 x 4096 x 10240 group 64 27.0, 27.8.
constexpr long kShort = 8, kFewRows = 21, kFewWork = 100'000'000;

struct MidPlan {
  bool ok;
  int rbm;  // 16-token blocks per tile
  int ks;   // K splits
  bool kw;  // K over the waves of a workgroup (mid_kwave_kernel)
};

long kwave_tiles(int mats, long M, long N) {
  return (M + 31) / 32 * ((N * mats + kTN * 16 - 1) / (kTN * 16));
}

// Where mid_kwave_kernel takes a problem: a stage for every wave, the scales of a
// wave's range in LDS, and up to two rounds of workgroups (one per CU).  Beyond, its
// 32-token tiles unpack the weights too often, but for one matrix up to three while
// an XCD's L2 holds the activations, which every 64 weight rows read again; past K =
// 8192, which the kernel below splits, under two.  us, this kernel and the one below
// (rounds: M x N x K, group 128 unless said):
//   1.1: 490 x 1024 x 4096          12 / 27     1.7: 640 x 1408 x 4096          24 / 35
//   1.9: 700 x 1408 x 4096          23 / 33     1.8: 200 x 4096 x 1408          12 / 18
//   2.3: 260 x 4096 x 4096          29 / 33     2.3: 850 x 1408 x 4096          36 / 33
//   2.8: 333 x 4096 x 4096 group 64 32 / 38     2.9: 1500 x 1024 x 4096         40 / 34
//   2.8: 333 x 4096 x 2048          21 / 20     2.8: the same, group 32         22 / 24
//   3.3: 400 x 4096 x 4096          40 / 34     3.5: 100 x 14336 x 4096 group 64  41 / 37
//   1.8: 200 x 4096 x 11008         51 / 60     1.9: 480 x 2048 x 10240         47 / 57
//   2.0: 1024 x 1024 x 14336        75 / 68     2.4: 600 x 2048 x 11008         73 / 68
//   gate and up (the whole expert): 1.8: 17 x 14336 x 4096 58 / 66; 2.8: 500 x 1408 x
//     4096 49 / 49; 3.5: 37 x 14336 x 4096 73 / 66; 3.8: 700 x 1408 x 4096 67 / 55
constexpr long kL2Bytes = 4 << 20;  // per XCD

bool kwave_ok(int mats, long M, long N, long T, long sps) {
  if (T < kKWaves || (T + kKWaves - 1) / kKWaves * sps > kKScales) return false;
  const long round = hn_device_cus(), tiles = kwave_tiles(mats, M, N);
  if (T > kLongK) return tiles < 2 * round;
  if (mats == 1 && M * T * kRowB <= kL2Bytes && (T >= 32 || (T >= 2 * kKWaves && sps > 1)))
    return tiles <= 3 * round;
  return tiles <= 2 * round;
}

MidPlan mid_plan(int mats, long M, long N, long K, long group) {
  MidPlan p{};
  if (M < 1 || N < 1 || K % kStageK != 0 || group < 32 || (group & (group - 1)) || group > kStageK)
    return p;
  const long T = K / kStageK, sps = kStageK / group;
  if (T < kShort && (M <= 32 || (M <= 64 && T < kShort / 2))) return p;
  const long nt = (N * mats + kBN - 1) / kBN, tk = kwave_tiles(mats, M, N);
  if (kwave_ok(mats, M, N, T, sps)) {
    if (mats == 1 && M <= kFewRows && T > 32 && tk < 128 && (tk < 64 || T > kLongK || T % kKWaves != 0))
      return p;
    p.kw = p.ok = true;
    p.rbm = 2;
    p.ks = 1;
    return p;
  }
  const long t32 = (M + 31) / 32 * nt, t64 = (M + 63) / 64 * nt;
  const bool small = t32 * T <= kUnits32 || t32 == t64;
  if (!small && (t64 > slots() || t64 * T > kUnits64)) return p;
  if (T < kShort && M > 64 && t32 > (M <= 128 ? 1 : 2) * slots()) return p;
  p.rbm = small ? 2 : 4;
  const long tiles = small ? t32 : t64;
  // K splits to one workgroup per CU (at two per CU the splits' reduction costs more
  // than they give: the expert of 4096 x 14336 at 37 rows 74.0 us, 66.0 with gate/up
  // whole; 37 x 4096 x 14336 group 32 40.7 / 37.1), of at least two stages each; an
  // even split (whole scale vectors per load) where one comes within half of that
  long lim = hn_device_cus() / tiles;
  if (lim > T / 2) lim = T / 2;
  if (N % 4 != 0) {  // the reduction reads four columns at a time
    if (T > 32) return p;
    lim = 1;
  }
  if (lim < 1 || T < kShort) lim = 1;
  long ks = lim;
  for (long d = lim; d >= 1 && 2 * d >= lim; --d)
    if (T % d == 0) { ks = d; break; }
  // past K = 8192, splits of at most kSplitStages stages, as long as all are resident at
  // once, an even split where there is one nearby (us by one split per CU / so: 560 x
  // 1024 x 14336 group 64 65 / 49; 333 x 4096 x 12288 group 64 94 / 74; but up to 64
  // rows 64 x 8192 x 28672 70 / 82)
  if (T > kLongK && M > 64) {
    const long m = std::min((T + kSplitStages - 1) / kSplitStages, std::max(slots() / tiles, 1L));
    long d = m;
    while (4 * d > 3 * m && T % d != 0) --d;
    if (4 * d <= 3 * m) d = m;
    if (ks < d) ks = d;
  }
  if (M <= 32 && ks > 1 && mats * N * K < (M <= kFewRows ? kFewWork : kFewWork * 2 / 5)) return p;
  p.ks = (int)ks;
  p.ok = true;
  return p;
}

// Scales per load: whole vectors when every split of every row starts aligned (below
// group 128 a stage's scales are whole pairs).
int scale_vec(long K, long ld_s, long group, long ks, const void* s0, const void* s1) {
  const long T = K / kStageK, sps = kStageK / group;
  const long per = T % ks == 0 ? T / ks * sps : sps;
  if (ld_s % 8 == 0 && per % 8 == 0 && aligned16(s0) && aligned16(s1)) return 8;
  if (ld_s % 2 == 0 && per % 2 == 0 && (((uintptr_t)s0 | (uintptr_t)s1) & 3) == 0) return 2;
  return 1;
}

void fill_common(MidArgs& A, long N, long K, long group, long ld_q, long ld_s, int ks, int sv) {
  A.N = (int)N;
  A.K = (int)K;
  A.group = (int)group;
  A.ld_q = (int)ld_q;
  A.ld_s = (int)ld_s;
  A.ks = ks;
  A.sv = sv;
  A.m_pair = 0x00F0000Fu;
  A.magic = 0x64006400u;
}

#define HN_MID_LAUNCH(GROUPED, MATS, RBM, SC, OUT)                                           \
  hipLaunchKernelGGL((mid_kernel<GROUPED, MATS, RBM, SC, OUT>), dim3(grid), dim3(256), 0, s, \
                     A, tb, active, n_active, offsets)

template <int MATS, int OUT>
void launch_single(const MidArgs& A, const MidPlan& p, int grid, hipStream_t s) {
  const MExpert* tb = nullptr;
  const int *active = nullptr, *n_active = nullptr, *offsets = nullptr;
  if (A.group == kStageK) {
    if (p.rbm == 2) HN_MID_LAUNCH(false, MATS, 2, true, OUT);
    else HN_MID_LAUNCH(false, MATS, 4, true, OUT);
  } else {
    if (p.rbm == 2) HN_MID_LAUNCH(false, MATS, 2, false, OUT);
    else HN_MID_LAUNCH(false, MATS, 4, false, OUT);
  }
}

// Grouped launches, group 128: 32-token tiles up to this many rows per expert on
// average, 64-token tiles above (us, gate/up + down, 8 experts of 4096 x 14336: 24
// rows each 129 + 66 against 136 + 74; 48 rows 211 + 106 against 157 + 82; 25 on
// average, 58 at most, 166 + 107 against 150 + 89; 128 experts of 4096 x 1408 with 19
// rows 196 + 120 against 205 + 129).
constexpr long kRows32 = 20;
constexpr long kGroupedStages = 32;  // of an item at most: the sizes that were measured

}  // namespace

// How a single problem is run here: 0 not at all, -1 K over the waves of a workgroup,
// else the tile's tokens << 16 | the number of K splits over workgroups (1: whole).
extern "C" int hn_mid_linear_plan(int mats, long M, long N, long K, long group) {
  const MidPlan p = mid_plan(mats, M, N, K, group);
  return !p.ok ? 0 : p.kw ? -1 : p.rbm << 20 | p.ks;
}

// Workspace bytes (after kPartOffset) a single problem's K splits need; 0 when
// not handled or not split.
extern "C" long hn_mid_part_bytes(int mats, long M, long N, long K) {
  long b = 0;
  for (long g = 32; g <= kStageK; g *= 2) {
    const MidPlan p = mid_plan(mats, M, N, K, g);
    if (p.ok && p.ks > 1 && (long)p.ks * mats * M * N * 4 > b) b = (long)p.ks * mats * M * N * 4;
  }
  return b;
}

// Single problem: out[M, N] = x @ deq(W)^T (mats 1) or the SwiGLU h (mats 2).
// Returns HN_NOT_HANDLED when the shape (or the workspace) is not handled here,
// 0 after the launches, a HIP error code when one failed.
extern "C" int hn_mid_linear_impl(int mats, const void* x, long ld_x, const void* q0,
                                  const void* s0, const void* q1, const void* s1, long ld_q,
                                  long ld_s, void* out, long ld_o, long M, long N, long K,
                                  long group, void* work, long work_bytes, void* stream) {
  const MidPlan p = mid_plan(mats, M, N, K, group);
  if (!p.ok) return HN_NOT_HANDLED;
  if (!aligned16(x) || ld_x % 8 != 0 || !aligned16(q0) || !aligned16(q1) || ld_q % 16 != 0)
    return HN_NOT_HANDLED;
  if (ld_x * 2 * 64 >= (long)kOOB || N * ld_q >= (long)kOOB || N * ld_s * 2 >= (long)kOOB)
    return HN_NOT_HANDLED;
  if (p.ks > 1 && (!work || !aligned16(work) ||
                   work_bytes < kPartOffset + (long)p.ks * mats * M * N * 4))
    return HN_NOT_HANDLED;
  MidArgs A = {};
  A.x = (const h16*)x;
  A.ld_x = ld_x;
  A.M = (int)M;
  A.q[0] = (const uint8_t*)q0; A.s[0] = (const h16*)s0;
  A.q[1] = (const uint8_t*)q1; A.s[1] = (const h16*)s1;
  A.out = (h16*)out;
  A.ld_o = ld_o;
  fill_common(A, N, K, group, ld_q, ld_s, p.ks,
              scale_vec(K, ld_s, group, p.kw ? kKWaves : p.ks, s0, s1));
  A.part = work ? (float*)((char*)work + kPartOffset) : nullptr;
  A.part_rows = M;
  hipStream_t s = (hipStream_t)stream;
  if (p.kw) {
    const dim3 grid((unsigned)kwave_tiles(mats, M, N)), block(64 * kKWaves);
    if (mats == 2) {
      if (group == kStageK) hipLaunchKernelGGL((mid_kwave_kernel<2, true>), grid, block, 0, s, A);
      else hipLaunchKernelGGL((mid_kwave_kernel<2, false>), grid, block, 0, s, A);
    } else {
      if (group == kStageK) hipLaunchKernelGGL((mid_kwave_kernel<1, true>), grid, block, 0, s, A);
      else hipLaunchKernelGGL((mid_kwave_kernel<1, false>), grid, block, 0, s, A);
    }
    HN_LAUNCH_CHECK("hn_mid_linear");
    return 0;
  }
  const long tm = 16 * p.rbm;
  const long tiles = (M + tm - 1) / tm * ((N * mats + kBN - 1) / kBN);
  const long items = tiles * p.ks;
  if (p.ks > 1) {
    if (tiles * kWaves > kMaxCounters || p.ks > kHnMaxArrivals) return HN_NOT_HANDLED;
    A.ctr = (unsigned long long*)work;
    A.tag = hn_next_tag();
  }
  const int grid = (int)(items < slots() ? items : slots());
  if (mats == 2) {
    if (p.ks > 1) launch_single<2, kSum>(A, p, grid, s);
    else launch_single<2, kOut>(A, p, grid, s);
  } else {
    if (p.ks > 1) launch_single<1, kSum>(A, p, grid, s);
    else launch_single<1, kOut>(A, p, grid, s);
  }
  HN_LAUNCH_CHECK("hn_mid_linear");
  return 0;
}

// Grouped over the active experts of one MoE layer (rows sorted by expert, as
// hn_grouped_expert_mlp_int4), group 128.  phase 0: gate/up + SiLU into out [rows,
// I]; phase 1: down, whole into out [rows, H] (part NULL), or as ks K slices in fp32
// part[j][rows][H].  dry_run: only say whether the shape is handled.
extern "C" int hn_mid_grouped_impl(int phase, const void* x, long ld_x, const void* table,
                                   const int* active, const int* n_active, const int* offsets,
                                   long E, long rows, long H, long I, long group, void* out,
                                   long ld_o, float* part, int ks, void* stream, int dry_run) {
  const long K = phase == 0 ? H : I, N = phase == 0 ? I : H;
  if (E < 1 || E > kMaxProb || group != kStageK || K % kStageK != 0 || ks < 1 ||
      (K / kStageK) % ks != 0 || K / kStageK / ks > kGroupedStages)
    return HN_NOT_HANDLED;
  if ((phase == 0 && part) || N * (K / 2) >= (long)kOOB || N * (K / group) * 2 >= (long)kOOB ||
      ld_x * 2 * 64 >= (long)kOOB || ld_x % 8 != 0)
    return HN_NOT_HANDLED;
  if (dry_run) return 0;
  if (rows <= 0) return 0;
  MidArgs A = {};
  A.x = (const h16*)x;
  A.ld_x = ld_x;
  A.out = (h16*)out;
  A.ld_o = ld_o;
  A.phase = phase;
  A.E = (int)E;
  // table pointers are 16-byte aligned (the grouped entry points' contract)
  fill_common(A, N, K, group, K / 2, K / group, ks,
              scale_vec(K, K / group, group, ks, nullptr, nullptr));
  A.part = part;
  A.part_rows = rows;
  const bool r32 = rows <= kRows32 * E;
  const int mats = phase == 0 ? 2 : 1;
  const long tm = r32 ? 32 : 64;
  const long items = (rows / tm + (E < rows ? E : rows)) * ((N * mats + kBN - 1) / kBN) * ks;
  const int grid = (int)(items < slots() ? items : slots());
  const MExpert* tb = (const MExpert*)table;
  hipStream_t s = (hipStream_t)stream;
  if (phase == 0) {
    if (r32) HN_MID_LAUNCH(true, 2, 2, true, kOut);
    else HN_MID_LAUNCH(true, 2, 4, true, kOut);
  } else if (part) {
    if (r32) HN_MID_LAUNCH(true, 1, 2, true, kPart);
    else HN_MID_LAUNCH(true, 1, 4, true, kPart);
  } else {
    if (r32) HN_MID_LAUNCH(true, 1, 2, true, kOut);
    else HN_MID_LAUNCH(true, 1, 4, true, kOut);
  }
  HN_LAUNCH_CHECK("hn_mid_grouped");
  return 0;
}

// out[rows, N] = the ks fp32 planes part[j][rows][N] summed in order.
extern "C" int hn_mid_reduce_impl(const float* part, int ks, long rows, long N, void* out,
                                  long ld_o, void* stream) {
  if (rows <= 0) return 0;
  hipLaunchKernelGGL(mid_reduce_kernel, dim3(hn_cdiv(rows * (N / 4), 256)), dim3(256), 0,
                     (hipStream_t)stream, part, rows * N, ks, (int)rows, (int)N, (h16*)out, ld_o);
  HN_LAUNCH_CHECK("hn_mid_reduce");
  return 0;
}
