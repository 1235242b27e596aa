// g4v_w4a8.hip -- W4A8 (int4 weights x per-group int8 activations) for gfx950.
//
// Restates engine/w4a8_avx2.h: quant (A8:30-42) and tile<MT> (A8:46-61), driven over all rows
// as i8_task does (E:303-309).  Per activation row m and 32-group g:
//   sx = amax / 127, inv = sx > 0 ? 1 / sx : 0, q_i = RNE(x_i * inv) (int8), sum = sum_i q_i
//   a32[m][n][g] = sum_i u[n][i] q[m][i] - 8 sum[m][g]               (exact integer)
//   y[m][n] = fma chain over g in order of  row = fma((float)a32, sw[n][g] * sx[m][g], row)
//
// The integer dot runs on the matrix cores: v_mfma_f32_16x16x32_bf16 over one group (K = 32).
// Operands: q as bf16 (|q| <= 127 is exact in bf16) and the weight nibble u as bf16(128 + u)
// (bit pattern 0x4300 | u, no arithmetic to decode); the accumulator input is -136 sum, so
//   D = sum_i q_i (128 + u_i) - 136 sum = sum_i q_i u_i - 8 sum = a32.
// Every product (<= 143 * 128) and every partial sum (< 2^21) is an integer that fp32 holds
// exactly, so D is exact whatever order the unit adds in.  The fp32 chain over groups then
// runs on the VALU in the reference's order, one fma per (row, output, group).
//
// q never saturates: |x_i| <= amax and amax * RN(1 / RN(amax / 127)) < 127.5, so |q_i| <= 127
// and the reference's int16/int8 saturation (A8:40) and its sum of the unsaturated integers
// agree; q is still clamped to [-128, 127] as A8:40 does.
//
// Weights are re-laid once per matrix (k_tile_a8): per tile of 16 output rows and chunk of
// 4 groups, the 64 lanes of a wave hold 16 contiguous bytes each (one coalesced 1 KB load):
// lane (r = lane % 16, h = lane / 16) gets bytes 4h .. 4h+3 of groups 4c .. 4c+3 of row 16t + r,
// i.e. elements 8h .. 8h+7 of each group: the MFMA's B operand for column r, k-slice h.
#include "g4v_internal.h"

namespace g4v {

typedef __attribute__((ext_vector_type(8))) __bf16 bf16x8_t;
typedef __attribute__((ext_vector_type(4))) float f32x4_t;
typedef __attribute__((ext_vector_type(4))) uint32_t u32x4_t;

// within each 8-element k-slice the operands hold elements in the order 0,2,4,6,1,3,5,7 (a8_slot: low
// nibbles first, then high nibbles), which keeps the weight decode to byte permutes

// orig w [N][K/2] (low nibble = even k), s [N][K/32] bf16  ->
// tw [N/16][G/4][64] uint4, ts [N/16][G/8][16] uint4 (8 scales of one row)
__global__ void k_tile_a8(const uint8_t* __restrict__ w, const uint16_t* __restrict__ s, uint4* __restrict__ tw,
                          uint4* __restrict__ ts, int N, int K) {
  const int G = K / 32, GC = G / 4, G8 = G / 8;
  const size_t total = (size_t)(N / 16) * GC * 64;
  for (size_t u = (size_t)blockIdx.x * blockDim.x + threadIdx.x; u < total; u += (size_t)gridDim.x * blockDim.x) {
    const int lane = (int)(u & 63);
    const size_t tc = u >> 6;
    const int c = (int)(tc % GC);
    const size_t t = tc / GC;
    const int r = lane & 15, h = lane >> 4;
    const uint8_t* row = w + (size_t)(t * 16 + r) * (K / 2);
    uint32_t d[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) d[i] = *reinterpret_cast<const uint32_t*>(row + (4 * c + i) * 16 + 4 * h);
    tw[u] = make_uint4(d[0], d[1], d[2], d[3]);
    if (h == 0 && c < G8 * 2 && (c & 1) == 0) {
      const uint4* sr = reinterpret_cast<const uint4*>(s + (size_t)(t * 16 + r) * G);
      ts[(t * G8 + c / 2) * 16 + r] = sr[c / 2];
    }
  }
}

void launch_tile_a8(const uint8_t* w, const uint16_t* s, uint4* tw, uint4* ts, int N, int K, hipStream_t st) {
  const size_t total = (size_t)(N / 16) * (K / 128) * 64;
  int grid = (int)((total + 255) / 256);
  if (grid > 65536) grid = 65536;
  hipLaunchKernelGGL(k_tile_a8, dim3(grid), dim3(256), 0, st, w, s, tw, ts, N, K);
}

// A8:30-42: a thread takes 8 consecutive values, four neighbouring lanes a group (with a thread per
// group the lanes' 128-byte rows cost 78 us for 6,841 x 6,144 values).  Optional q [M][K] int8 (plain
// order), sx / sum [M][G] for the quant entry point.
__global__ __launch_bounds__(256) void k_w4a8_quant(const float* __restrict__ x, int M, int K, A8Rows o,
                                                    int8_t* __restrict__ qo, float* __restrict__ sxo,
                                                    int32_t* __restrict__ sumo) {
  const size_t u = (size_t)blockIdx.x * 256 + threadIdx.x;
  const int K8 = K / 8;
  if (u >= (size_t)M * K8) return;  // whole groups: M K / 8 is a multiple of 4
  const int m = (int)(u / K8), i = (int)(u - (size_t)m * K8);
  const float4 a = *reinterpret_cast<const float4*>(x + 8 * u), b = *reinterpret_cast<const float4*>(x + 8 * u + 4);
  const float v[8] = {a.x, a.y, a.z, a.w, b.x, b.y, b.z, b.w};
  a8_store8(o, m, K, i, v);
  if (qo) {  // (uniform)
    float amax = 0.f, sum = 0.f, q[8];
#pragma unroll
    for (int k = 0; k < 8; ++k) amax = fmaxf(amax, fabsf(v[k]));
    amax = fmaxf(amax, dpp_f(amax, 2));
    amax = fmaxf(amax, dpp_f(amax, 3));
    const float sx = amax / 127.0f, inv = sx > 0.f ? 1.0f / sx : 0.0f;
#pragma unroll
    for (int k = 0; k < 8; ++k) q[k] = a8_q(v[k], inv, sum);
    sum += dpp_f(sum, 2);
    sum += dpp_f(sum, 3);
    uint32_t w[2] = {0, 0};
#pragma unroll
    for (int k = 0; k < 8; ++k) w[k >> 2] |= ((uint32_t)(int)q[k] & 0xFFu) << (8 * (k & 3));
    *reinterpret_cast<uint2*>(qo + 8 * u) = make_uint2(w[0], w[1]);
    if ((i & 3) == 0) {
      sxo[u >> 2] = sx;
      sumo[u >> 2] = (int32_t)sum;
    }
  }
}

void launch_w4a8_quant(const float* x, int M, int Mpad, int K, uint16_t* xqb, float* sxt, float* corr, int8_t* qo,
                       float* sxo, int32_t* sumo, hipStream_t st) {
  const size_t n = (size_t)M * (K / 8);
  hipLaunchKernelGGL(k_w4a8_quant, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, st, x, M, K,
                     A8Rows{xqb, sxt, corr, Mpad}, qo, sxo, sumo);
}

// bf16(128 + u) for the four low (sel 0x04010400 / 0x04030402 of the lo word) or high nibbles
__device__ __forceinline__ bf16x8_t a8_decode(uint32_t d) {
  const uint32_t lo = d & 0x0F0F0F0Fu, hi = (d >> 4) & 0x0F0F0F0Fu, c = 0x43434343u;
  uint4 o;
  o.x = __builtin_amdgcn_perm(c, lo, 0x04010400u);  // elements 0, 2
  o.y = __builtin_amdgcn_perm(c, lo, 0x04030402u);  // 4, 6
  o.z = __builtin_amdgcn_perm(c, hi, 0x04010400u);  // 1, 3
  o.w = __builtin_amdgcn_perm(c, hi, 0x04030402u);  // 5, 7
  return __builtin_bit_cast(bf16x8_t, o);
}

// Products of more than 8 rows.  A block of 4 waves covers 16 MT rows and 4 NT tiles of 16 outputs
// (wave w the tiles NT w ..); lane (r, h): B column r, A row r, k-slice h; D element i = row 4h + i,
// column r.  The block's operand rows, corrections and row scales of a step of CG groups are loaded
// once per block a step ahead into registers and written to the other half of a double-buffered
// LDS stage, one LDS barrier per step (the weights, each wave's own, stay in flight across it).
// PAIR: the NT tiles are NT / 2 gate tiles (matrix 0) and the same outputs' up tiles (matrix 1), and
// the activation r16(r16(gelu8(r16 g)) * r16 u) leaves as down's quantised rows (A8Gemm::yq).
template <int MT, int NT, int CG, bool PAIR>
__global__ __launch_bounds__(256, MT * NT >= 16 ? 2 : 3) void k_w4a8_gemm(A8Gemm q, const uint16_t* __restrict__ xqb,
                                                   const float* __restrict__ sxt, const float* __restrict__ corr,
                                                   int M, int Mpad, int K) {
  constexpr int RB = 16 * MT;  // rows of a block
  constexpr int NP = MT * CG / 4;                   // 16-byte pieces per thread and step
  constexpr int NC = CG * RB, NCT = (NC + 255) / 256;
  static_assert(MT * CG % 4 == 0 && (CG == 4 || CG == 8), "whole pieces, whole chunks of 4 groups");
  __shared__ __align__(16) u32x4_t As[2][64 * MT * CG];  // [MT][CG][16 rows][4 pieces], as in memory
  __shared__ __align__(16) float Cs[2][CG][RB], Ss[2][CG][RB];
  const int lane = threadIdx.x & 63, tid = threadIdx.x, w = threadIdx.x >> 6;
  constexpr int TPW = PAIR ? NT / 2 : NT;           // tiles of a matrix per wave
  const int tg = (blockIdx.x * 4 + w) * TPW;        // first of the wave's tiles over the matrices
  const bool active = tg < q.t0[PAIR ? 1 : 3];      // idle waves still stage and wait
  const int tw = active ? tg : 0;
  const int mi = PAIR ? 0 : ((tw >= q.t0[1]) + (tw >= q.t0[2]));
  const int t0 = tw - (mi == 0 ? 0 : (mi == 1 ? q.t0[1] : q.t0[2]));
  const int m0 = blockIdx.y * RB;
  const int r = lane & 15, h = lane >> 4;
  const int G = K / 32, NS = G / CG;
  const uint4 *wp[NT], *sp[NT];  // chunk c of 4 groups at wp + 64 c, scales of 8 groups at sp + 16 c8
#pragma unroll
  for (int u = 0; u < NT; ++u) {
    const int t = t0 + (PAIR ? u % TPW : u);
    const uint4 *tww = q.tw[0], *tss = q.ts[0];
    if constexpr (PAIR) {
      if (u >= TPW) tww = q.tw[1], tss = q.ts[1];
    } else {
      if (mi == 1) tww = q.tw[1], tss = q.ts[1];
      if (mi == 2) tww = q.tw[2], tss = q.ts[2];
    }
    wp[u] = tww + (size_t)t * (G / 4) * 64 + lane;
    sp[u] = tss + (size_t)t * (G / 8) * 16 + r;
  }
  f32x4_t acc[MT][NT];
#pragma unroll
  for (int mt = 0; mt < MT; ++mt)
#pragma unroll
    for (int u = 0; u < NT; ++u) acc[mt][u] = f32x4_t{0.f, 0.f, 0.f, 0.f};
  u32x4_t ap[NP];
  float crn[NCT], sxn[NCT];
  auto issue = [&](int st) {
#pragma unroll
    for (int k = 0; k < NP; ++k) {
      const int i = tid + 256 * k;  // 16 bytes i % (64 CG) of the step's groups of row block i / (64 CG)
      ap[k] = *reinterpret_cast<const u32x4_t*>(xqb + a8_at(K, m0 + 16 * (i / (64 * CG)), CG * st) + 8 * (i % (64 * CG)));
    }
#pragma unroll
    for (int k = 0; k < NCT; ++k) {
      const int i = (tid + 256 * k) & (NC - 1), g = i / RB, m = i % RB;
      crn[k] = corr[(size_t)(CG * st + g) * Mpad + m0 + m];
      sxn[k] = sxt[(size_t)(CG * st + g) * Mpad + m0 + m];
    }
  };
  auto commit = [&](int b) {
#pragma unroll
    for (int k = 0; k < NP; ++k) As[b][tid + 256 * k] = ap[k];
#pragma unroll
    for (int k = 0; k < NCT; ++k) {  // (with fewer than 256 entries several threads store the same)
      const int i = (tid + 256 * k) & (NC - 1);
      Cs[b][i / RB][i % RB] = crn[k];
      Ss[b][i / RB][i % RB] = sxn[k];
    }
  };
  static_assert((NC & (NC - 1)) == 0, "a power of two of corrections");
  // weight words (chunks of 4 groups) of the current and the next step in two register sets that swap
  // roles, the 8 scales of a row likewise (one word serves a step of 8 groups, or two of 4)
  constexpr int CW = CG / 4;
  u32x4_t wA[NT][CW], wB[NT][CW], sA[NT], sB[NT];
  auto issue_w = [&](u32x4_t (&wx)[NT][CW], int st) {
#pragma unroll
    for (int u = 0; u < NT; ++u)
#pragma unroll
      for (int k = 0; k < CW; ++k)
        wx[u][k] = *reinterpret_cast<const u32x4_t*>(wp[u] + (size_t)(CW * st + k) * 64);
  };
  auto issue_s = [&](u32x4_t (&sx)[NT], int c8) {
#pragma unroll
    for (int u = 0; u < NT; ++u) sx[u] = *reinterpret_cast<const u32x4_t*>(sp[u] + (size_t)c8 * 16);
  };
  auto products = [&](const int b, const u32x4_t (&wc)[NT][CW], const u32x4_t (&sc8)[NT]) {
#pragma unroll
    for (int i = 0; i < CG; ++i) {
      const int e = CG == 4 ? 4 * b + i : i;  // group within the 8 scales
      bf16x8_t B[NT];
      float sw[NT];
#pragma unroll
      for (int u = 0; u < NT; ++u) {
        B[u] = a8_decode(wc[u][i >> 2][i & 3]);
        const uint32_t s2 = sc8[u][e >> 1];
        sw[u] = as_f32((e & 1) ? (s2 & 0xFFFF0000u) : (s2 << 16));
      }
#pragma unroll
      for (int mt = 0; mt < MT; ++mt) {
        const u32x4_t av = As[b][((mt * CG + i) * 16 + r) * 4 + h];
        const f32x4_t cin = *reinterpret_cast<const f32x4_t*>(&Cs[b][i][16 * mt + 4 * h]);
        const f32x4_t sx = *reinterpret_cast<const f32x4_t*>(&Ss[b][i][16 * mt + 4 * h]);
        const bf16x8_t A = __builtin_bit_cast(bf16x8_t, av);
#pragma unroll
        for (int u = 0; u < NT; ++u) {
          const f32x4_t a = __builtin_amdgcn_mfma_f32_16x16x32_bf16(A, B[u], cin, 0, 0, 0);
#pragma unroll
          for (int k = 0; k < 4; ++k) acc[mt][u][k] = fmaf(a[k], sw[u] * sx[k], acc[mt][u][k]);  // A8:59
        }
      }
    }
  };
  issue(0);
  issue_w(wA, 0);
  issue_s(sA, 0);
  commit(0);
  lds_barrier();
  // (NS is even with steps of 4 groups: K % 256 == 0; with 8 it may be odd; the prefetch past the last
  // step reads that step again and is not used)
  for (int st = 0; st < NS; st += 2) {
    issue(min(st + 1, NS - 1));
    issue_w(wB, min(st + 1, NS - 1));
    issue_s(sB, CG == 4 ? min(st / 2 + 1, NS / 2 - 1) : min(st + 1, NS - 1));
    products(0, wA, sA);
    commit(1);
    lds_barrier();
    if (CG == 8 && st + 1 >= NS) break;  // uniform
    issue(min(st + 2, NS - 1));
    issue_w(wA, min(st + 2, NS - 1));
    if constexpr (CG == 4) {
      products(1, wB, sA);
#pragma unroll
      for (int u = 0; u < NT; ++u) sA[u] = sB[u];
    } else {
      issue_s(sA, min(st + 2, NS - 1));
      products(1, wB, sB);
    }
    commit(0);
    lds_barrier();
  }
  if (!active) return;
  if constexpr (PAIR) {
    // TPW = 2: the wave's two tiles are one 32-group of the activation, quantised here for down; the
    // sixteen lanes r hold two of its values each
    static_assert(TPW == 2, "a wave owns whole groups");
    const int g = t0 >> 1;  // (t0 is even)
    const int N = 16 * q.t0[1];
#pragma unroll
    for (int mt = 0; mt < MT; ++mt)
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const int m = m0 + 16 * mt + 4 * h + i;
        float v[2];
#pragma unroll
        for (int u = 0; u < 2; ++u) v[u] = r16(r16(gelu8(r16(acc[mt][u][i]))) * r16(acc[mt][u + 2][i]));
        const float amax = row16_all_max(fmaxf(fabsf(v[0]), fabsf(v[1])));
        const float sx = amax / 127.0f, inv = sx > 0.f ? 1.0f / sx : 0.0f;
        float sum = 0.f;
        const float q0 = a8_q(v[0], inv, sum), q1 = a8_q(v[1], inv, sum);
        sum = row16_all_sum(sum);
        if (m < M) {
          uint16_t* d = q.yq.q + a8_at(N, m, g) + a8_slot(r);
          d[0] = (uint16_t)(as_u32(q0) >> 16);
          d[16] = (uint16_t)(as_u32(q1) >> 16);
          if (r == 0) {
            q.yq.sx[(size_t)g * q.yq.ld + m] = sx;
            q.yq.corr[(size_t)g * q.yq.ld + m] = -136.0f * sum;
          }
        }
      }
  } else {
    float* y = mi == 0 ? q.y[0] : (mi == 1 ? q.y[1] : q.y[2]);
    const int ldy = mi == 0 ? q.ldy[0] : (mi == 1 ? q.ldy[1] : q.ldy[2]);
#pragma unroll
    for (int mt = 0; mt < MT; ++mt)
#pragma unroll
      for (int u = 0; u < NT; ++u)
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          const int m = m0 + 16 * mt + 4 * h + i;
          if (m < M) y[(size_t)m * ldy + 16 * (t0 + u) + r] = acc[mt][u][i];
        }
  }
}

// The same products where they leave SIMDs idle (few tiles of 16 x 16): a block of eight waves per
// tile.  Only the chain over the groups is ordered, so waves 0..3 form a phase's 16 group dots and
// factors sw * sx (a chunk of 4 groups each, operands loaded two phases ahead) into LDS while waves
// 4..7 run the previous phase's chains, D element i of every lane on wave 4 + i.  A lone wave issues an
// instruction every ~6 cycles, and in k_w4a8_gemm's loop a tile's group took it ~300 cycles (40 rows,
// K = 6144: 24 us on 288 waves); here a phase costs its four groups of dots (17 us; K = 1536, 160 tiles x
// 3 row blocks: 8.4).
constexpr int SP_G = 16;  // groups of a phase
__global__ __launch_bounds__(512) void k_w4a8_split(A8Gemm q, const uint16_t* __restrict__ xqb,
                                                    const float* __restrict__ sxt, const float* __restrict__ corr,
                                                    int M, int Mpad, int K) {
  __shared__ __align__(16) float2 S[2][SP_G][4][64];  // (a32, sw * sx) of D element i, lane
  const int lane = threadIdx.x & 63, w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int tg = blockIdx.x, mi = (tg >= q.t0[1]) + (tg >= q.t0[2]);
  const int t = tg - (mi == 0 ? 0 : (mi == 1 ? q.t0[1] : q.t0[2]));
  const int m0 = blockIdx.y * 16, r = lane & 15, h = lane >> 4;
  const int G = K / 32, NC = G / 4, NPH = ((G + SP_G - 1) / SP_G + 1) & ~1;  // phases, by twos
  const uint4 *tww = q.tw[0], *tss = q.ts[0];
  if (mi == 1) tww = q.tw[1], tss = q.ts[1];
  if (mi == 2) tww = q.tw[2], tss = q.ts[2];
  if (w < 4) {
    const __amdgpu_buffer_rsrc_t wr = buf_rsrc(tww + (size_t)t * NC * 64, (uint32_t)NC * 1024);
    const __amdgpu_buffer_rsrc_t sr = buf_rsrc(tss + (size_t)t * (G / 8) * 16, (uint32_t)(G / 8) * 256);
    const __amdgpu_buffer_rsrc_t ar = buf_rsrc(xqb + (size_t)m0 * K, 32u * K);
    const __amdgpu_buffer_rsrc_t cr = buf_rsrc(corr, (uint32_t)G * Mpad * 4), xr = buf_rsrc(sxt, (uint32_t)G * Mpad * 4);
    const uint32_t ao = 64 * r + 16 * h, co = 4u * (m0 + 4 * h);
    auto ld = [](__amdgpu_buffer_rsrc_t rs, uint32_t o) { return __builtin_bit_cast(u32x4_t, buf_load16(rs, o)); };
    struct Ops {
      u32x4_t w, s, a[4];
      f32x4_t c[4], x[4];
    };
    // (No branch between the loads and their uses: a wait behind a join is for every load in flight,
    // and the phases then took a trip to memory each, 23 us for K = 6144.)
    auto load = [&](Ops& o, int p) {  // chunk 4 p + w (past the last: that one again, not read)
      const uint32_t c = min(4 * p + w, NC - 1);
      o.w = ld(wr, c * 1024 + lane * 16);
      o.s = ld(sr, (c >> 1) * 256 + r * 16);
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const uint32_t g = 4 * c + i;
        o.a[i] = ld(ar, ao + 1024 * g);
        o.c[i] = __builtin_bit_cast(f32x4_t, ld(cr, co + 4 * g * Mpad));
        o.x[i] = __builtin_bit_cast(f32x4_t, ld(xr, co + 4 * g * Mpad));
      }
    };
    auto form = [&](const Ops& o, int p) {
      const bool hi = w & 1;  // (the chunk's parity)
      const uint32_t s01 = hi ? o.s[2] : o.s[0], s23 = hi ? o.s[3] : o.s[1];
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const uint32_t s2 = i < 2 ? s01 : s23;
        const float sw = as_f32((i & 1) ? (s2 & 0xFFFF0000u) : (s2 << 16));
        const f32x4_t d = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8_t, o.a[i]),
                                                                 a8_decode(o.w[i]), o.c[i], 0, 0, 0);
#pragma unroll
        for (int k = 0; k < 4; ++k) S[p & 1][4 * w + i][k][lane] = make_float2(d[k], sw * o.x[i][k]);
      }
      __builtin_amdgcn_sched_barrier(0);
      lds_barrier();
    };
    Ops A, B;
    load(A, 0);
    asm volatile("" ::: "memory");  // (A's loads before B's also through the IR passes)
    __builtin_amdgcn_sched_barrier(0);
    load(B, 1);
    __builtin_amdgcn_sched_barrier(0);
    for (int p = 0; p < NPH; p += 2) {
      form(A, p);
      load(A, p + 2);
      __builtin_amdgcn_sched_barrier(0);
      form(B, p + 1);
      load(B, p + 3);
      __builtin_amdgcn_sched_barrier(0);
    }
    return;
  }
  const int i = w - 4;
  float acc = 0.f;
  for (int p = 0; p < NPH; ++p) {
    lds_barrier();  // phase p is formed; the producers go on to the other half
    const float2* s = &S[p & 1][0][i][lane];
    const int ng = min(SP_G, G - SP_G * p);  // 8 or 16 (K % 256 == 0), or none in a last odd phase
    for (int g8 = 0; g8 < ng; g8 += 8)
#pragma unroll
      for (int g = 0; g < 8; ++g) {
        const float2 v = s[(g8 + g) * 256];
        acc = fmaf(v.x, v.y, acc);  // A8:59
      }
  }
  const int m = m0 + 4 * h + i;
  float* y = mi == 0 ? q.y[0] : (mi == 1 ? q.y[1] : q.y[2]);
  const int ldy = mi == 0 ? q.ldy[0] : (mi == 1 ? q.ldy[1] : q.ldy[2]);
  if (m < M) y[(size_t)m * ldy + 16 * t + r] = acc;
}

// y [M][ldy] from the quantised rows; Mpad = M rounded up to 16 MT for the chosen MT
// Decode rows (M <= 8, Mpad 16): one block per 16-column tile t.  The tile's K walk is split by
// phases of DEC_PG groups: the sixteen waves compute the phase's group dots (exact integers, the
// same MFMA and operands as k_w4a8_gemm<1>) and the factors sc = sw * sx, and store them for
// rows 0..7 in LDS; after a barrier lane (m, r) of the first 128 threads continues its chain
// row = fma(a32, sc, row) over the phase's groups in group order (A8:59).  Every value and every
// rounding is the one k_w4a8_gemm<1> computes; the group dots of a phase run on sixteen waves at
// once instead of one after another.  K % 256 == 0 (whole chunks of 4 groups, scale blocks of 8).
// Up to three matrices of the same input in one launch (i8_task over nj matrices, E:303-309):
// block b runs tile b - t0[j] of matrix j, t0[j] <= b < t0[j + 1], t0[j + 1] - t0[j] = N_j / 16.
constexpr int DEC_PG = 64;
__global__ __launch_bounds__(1024) void k_w4a8_dec(A8Dec m, const uint16_t* __restrict__ xqb,
                                                  const float* __restrict__ sxt, const float* __restrict__ corr,
                                                  int M, int Mpad, int K) {
  __shared__ float2 S[DEC_PG][32][4];  // [group in phase][lane of rows 0..7][D register]: (a32, sc)
  const int tid = threadIdx.x, lane = tid & 63, w = tid >> 6;
  const int b = blockIdx.x;  // gridDim.x == t0[n]
  const int j = b < m.t0[1] ? 0 : (b < m.t0[2] ? 1 : 2);
  const int t = b - m.t0[j];
  const uint4* __restrict__ tw = m.tw[j];
  const uint4* __restrict__ ts = m.ts[j];
  float* __restrict__ y = m.y[j];
  const int ldy = m.ldy[j];
  const int r = lane & 15, h = lane >> 4;
  const int G = K / 32;
  const uint4* wp = tw + (size_t)t * (G / 4) * 64 + lane;  // chunk c at + 64 c
  const uint4* sp = ts + (size_t)t * (G / 8) * 16 + r;     // scales of groups 8 c8 .. at + 16 c8
  const uint16_t* ap = xqb + a8_at(K, r, 0) + 8 * h;        // group g at + 512 g
  const int mrow = 4 * h;
  const int cm = tid >> 4, cr = tid & 15;                   // chain lane: row cm, column cr
  const int cl = ((cm >> 2) << 4) | cr, ci = cm & 3;
  float acc = 0.f;
  for (int p = 0; p < G; p += DEC_PG) {
    const int nc = min(DEC_PG, G - p) / 4;  // chunks in this phase
    for (int q = w; q < nc; q += 16) {
      const int c = p / 4 + q;
      const uint4 wcur = wp[(size_t)c * 64];
      const uint4 scur = sp[(size_t)(c >> 1) * 16];
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const int g = 4 * c + i;
        const uint32_t d = i == 0 ? wcur.x : (i == 1 ? wcur.y : (i == 2 ? wcur.z : wcur.w));
        const bf16x8_t B = a8_decode(d);
        const int gi = 4 * (c & 1) + i;
        const uint32_t s2 = gi < 2 ? scur.x : (gi < 4 ? scur.y : (gi < 6 ? scur.z : scur.w));
        const float sw = as_f32((gi & 1) ? (s2 & 0xFFFF0000u) : (s2 << 16));
        const uint4 av = *reinterpret_cast<const uint4*>(ap + 512 * (size_t)g);
        const float4 crv = *reinterpret_cast<const float4*>(corr + (size_t)g * Mpad + mrow);
        const float4 sx = *reinterpret_cast<const float4*>(sxt + (size_t)g * Mpad + mrow);
        const f32x4_t cin = {crv.x, crv.y, crv.z, crv.w};
        const f32x4_t a = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8_t, av), B, cin, 0, 0, 0);
        if (h < 2) {
          float2* o = S[g - p][lane];
          o[0] = make_float2(a[0], sw * sx.x);
          o[1] = make_float2(a[1], sw * sx.y);
          o[2] = make_float2(a[2], sw * sx.z);
          o[3] = make_float2(a[3], sw * sx.w);
        }
      }
    }
    __syncthreads();
    if (tid < 128) {
      const int ng = nc * 4;
#pragma unroll 8
      for (int gi = 0; gi < ng; ++gi) {
        const float2 v = S[gi][cl][ci];
        acc = fmaf(v.x, v.y, acc);
      }
    }
    __syncthreads();
  }
  if (tid < 128 && cm < M) y[(size_t)cm * ldy + 16 * t + cr] = acc;
}

int w4a8_mpad(int M) {  // rows of the quantised operand: whole blocks of every shape used for M rows
  const int bm = M <= 16 ? 16 : (M <= 64 ? 32 : 64);
  return (M + bm - 1) / bm * bm;
}

template <int MT, int NT, int CG, bool PAIR>
static void launch_gemm(const A8Gemm& q, const uint16_t* xqb, const float* sxt, const float* corr, int M, int K,
                        hipStream_t st) {
  const int tpw = PAIR ? NT / 2 : NT, tiles = q.t0[PAIR ? 1 : 3];
  const dim3 grid((tiles + 4 * tpw - 1) / (4 * tpw), (M + 16 * MT - 1) / (16 * MT));
  hipLaunchKernelGGL((k_w4a8_gemm<MT, NT, CG, PAIR>), grid, dim3(256), 0, st, q, xqb, sxt, corr, M, w4a8_mpad(M), K);
}

int launch_w4a8_gemm_multi(const A8Gemm& q_in, int n, bool pair, const uint16_t* xqb, const float* sxt,
                           const float* corr, int M, int K, hipStream_t st) {
  A8Gemm q = q_in;
  if (n < 1 || n > 3 || M < 1 || K % 256 || (pair && (n != 2 || q.N[0] != q.N[1] || q.N[0] % 32 || !q.yq.q))) return 0;
  q.t0[0] = 0;
  bool by4 = true;
  int tiles = 0;
  for (int j = 0; j < 3; ++j) {
    if (j < n && q.N[j] % 16) return 0;
    tiles += j < n ? q.N[j] / 16 : 0;
    by4 = by4 && (j >= n || q.N[j] % 64 == 0);
    q.t0[j + 1] = tiles;
  }
  if (pair) q.t0[1] = q.N[0] / 16;
  const long waves1 = (long)tiles * ((M + 15) / 16);  // waves with a tile each
  if (pair) {
    if (by4 && M > 64 && waves1 > 8192) launch_gemm<4, 4, 4, true>(q, xqb, sxt, corr, M, K, st);
    else launch_gemm<1, 4, 4, true>(q, xqb, sxt, corr, M, K, st);
    return 1;
  }
  // A tile per block of eight waves while every block has a place at once (two a CU at 128 VGPRs, 64 KB
  // of LDS): prompts of 32 / 64 rows 3.1 / 3.6 ms with every product on it, 3.7 / 3.8 with none; of 96 /
  // 128 / 160 rows (576 to 960 blocks for o and down) 4.3 / 4.5 / 5.1 ms with, 4.0 / 4.2 / 4.2 without.
  if (by4 && M > 64 && waves1 > 8192) launch_gemm<4, 4, 4, false>(q, xqb, sxt, corr, M, K, st);
  else if (waves1 <= 512)
    hipLaunchKernelGGL(k_w4a8_split, dim3(tiles, (M + 15) / 16), dim3(512), 0, st, q, xqb, sxt, corr, M, w4a8_mpad(M), K);
  else launch_gemm<1, 1, 8, false>(q, xqb, sxt, corr, M, K, st);
  return 1;
}

void launch_w4a8_gemm(const uint4* tw, const uint4* ts, const uint16_t* xqb, const float* sxt, const float* corr,
                      float* y, int M, int N, int K, int ldy, hipStream_t st) {
  if (M <= 8) {  // decode rows: group dots split over the block's waves
    A8Dec m{};
    m.tw[0] = tw;
    m.ts[0] = ts;
    m.y[0] = y;
    m.ldy[0] = ldy;
    m.t0[1] = m.t0[2] = m.t0[3] = N / 16;
    hipLaunchKernelGGL(k_w4a8_dec, dim3(N / 16), dim3(1024), 0, st, m, xqb, sxt, corr, M, w4a8_mpad(M), K);
    return;
  }
  A8Gemm q{};
  q.tw[0] = tw, q.ts[0] = ts, q.y[0] = y, q.ldy[0] = ldy, q.N[0] = N;
  (void)launch_w4a8_gemm_multi(q, 1, false, xqb, sxt, corr, M, K, st);
}

int launch_w4a8_dec(const A8Dec& m, int n, const uint16_t* xqb, const float* sxt, const float* corr, int M, int K,
                    hipStream_t st) {
  if (n < 1 || n > 3 || M < 1 || M > 8 || K % 256) return 0;
  hipLaunchKernelGGL(k_w4a8_dec, dim3(m.t0[n]), dim3(1024), 0, st, m, xqb, sxt, corr, M, w4a8_mpad(M), K);
  return 1;
}

}  // namespace g4v
