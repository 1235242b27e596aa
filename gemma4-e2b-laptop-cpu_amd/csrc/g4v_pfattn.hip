// g4v_pfattn.hip -- prompt attention (more than MAXM rows) on the fp32 matrix cores.
//
// The arithmetic of g4v_prefill.hip's attention (attn_tile E:1063-1083, run_mh E:1338-1349), chain
// for chain.  The fp32 matrix instructions add their products one after the other, each with one
// rounding (the order and the roundings of fmaf, subnormals kept; g4v_gemmx.hip), so they run the
// reference's chains 16 x 16 or 32 x 32 at a time:
//   scores: v_mfma_f32_16x16x1_4b, four chains of 2 prompt rows x 8 heads x 16 keys an instruction
//     (k_pfa_scores); the chains of a score meet in one lane, in hsum's order;
//   output: v_mfma_f32_32x32x2, 4 prompt rows x 8 heads x 32 dims; O = fma(w, v, O) over the
//     positions, two an instruction (k_pfa_out).
// What bounds it: the matrix unit's 31 fp32 FMAs a cycle and SIMD (VALU fp32 work reaches 22 and adds
// to it).  The VALU kernels this replaces read an LDS word per 1 (scores) or 4 (output) FMAs and
// reached half of the VALU rate.  The rows of a tile share every key and value word; a block's waves
// split rows (scores) or dims (output), so no partial sums meet.
// Measured, prompt of 6,841 rows (28 window and 7 global layers): scores 19.8 -> 13.1 ms, output
// 22.3 -> 11.9 ms.  The o product's input is quantised by a launch of its own: from the output's
// registers (32 lanes a group) it cost 27 us a layer where that launch takes 22, and 9 for 3.5 at 40
// rows.
//
// Scores go through memory as tiles [row quad][32 keys][32 rows x 32 keys] with each wave's row
// maxima beside them: exp needs the row maximum first, and den the weights in position order.
#include <algorithm>

#include "g4v_layer.h"

namespace g4v {

typedef __attribute__((ext_vector_type(16))) float f32x16_t;
typedef __attribute__((ext_vector_type(4))) float f32x4v_t;
typedef __attribute__((ext_vector_type(4))) uint32_t u32x4_t;

namespace {

__constant__ uint64_t c_expf_tab_p[32] = G4V_EXPF_TABLE;
constexpr int WSTRIDE = 18;  // tiles of a window quad: 515 positions at any alignment
// attention path of row r (E:1305, 1328, 1337): its block [b pfb, ...) of M rows at p0
__device__ __forceinline__ bool pfa_tiled(int r, const PfGeom& g) {
  const int b = r / g.pfb, M = min(g.pfb, g.n - b * g.pfb), p0 = g.pos0 + b * g.pfb;
  return M >= 4 && p0 + M > 64;
}
__device__ __forceinline__ int pfa_lo(int P, int sliding) { return sliding ? max(0, P - 511) : 0; }
// sum over i < n of (a + 4 i) / 32, rounded down
__host__ __device__ inline long long quad_tiles_before(int a, int n) {
  const long long A = a >> 5, s = (a & 31) >> 2, k = s + n, t = k >> 3;
  return A * n + 4 * t * (t - 1) + t * (k - 8 * t);
}
// first tile of quad q of a segment at position Pb (global layers: quad i has (Pb + 4 i + 3) / 32 + 1)
__host__ __device__ inline long long quad_tile0(int q, int Pb, int sliding) {
  return sliding ? (long long)q * WSTRIDE : quad_tiles_before(Pb + 3, q) + q;
}

// Block: 8 prompt rows x a span of `spt` tiles of 32 keys; wave w rows 2 w, 2 w + 1 with their 8 heads.
// v_mfma_f32_16x16x1_4b_f32 (1024 FMAs in 33 cycles) runs four independent 16 x 16 chains a step:
// block b = lane / 16 is chain n = 4 cg + b of element 16 tt + n, so the 16 chains of a score are four
// accumulators, they meet in one lane (15 adds per output), and a row's operands are 64 (128)
// registers, two waves a SIMD.  run_mh's chain l takes the same operands in the order tt, s.
// Keys: a step of NK positions widened to fp32 in LDS in operand order [cg][tt / 4][b][key][4], the
// four waves sharing them, the next step's words in flight.  (On 32x32x2 tiles the operands and
// sums of one 4-row tile are 210 registers: with the rows in LDS and each wave reading its own keys
// from global memory, a 16-byte word of 32 rows an instruction, a global layer of 6,841 rows took
// 1213 us; with the rows in registers, one wave a SIMD, 1786 us.)
template <int D>
__global__ __launch_bounds__(256, 2) void k_pfa_scores(const float* __restrict__ q, const uint16_t* __restrict__ KC,
                                                       float* __restrict__ S, float* __restrict__ PM, PfGeom g, int r0,
                                                       int M, int sliding, int spt, int nspan) {
  constexpr int TT = D / 16, T4 = TT / 4, NK = D == 256 ? 32 : 16;  // chain steps, keys of a step
  constexpr int WD = D / 8, NP = WD * NK / 256;                      // 16-byte words of a key; of a step per thread
  constexpr int RS = 4 * NK + 4;                                     // floats of an operand row (+ pad)
  __shared__ __align__(16) float KT[2][4 * T4 * 4 * RS];
  const int rb = gridDim.x - 1 - (int)blockIdx.x;  // the longest ranges first
  const int lane = threadIdx.x & 63, w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int k16 = lane & 15, bl = lane >> 4;
  const int Pb = g.pos0 + r0, rw = 8 * rb + 2 * w, nr = min(2, M - rw);  // the wave's first row, its rows
  const int qd = rw >> 2;                                                // its quad
  const int P0 = Pb + rw, Pl = P0 + nr - 1;
  const int kb0 = pfa_lo(Pb + 8 * rb, sliding) >> 5, kbn = ((Pb + min(8 * rb + 7, M - 1)) >> 5) + 1;
  const int ka = kb0 + (int)blockIdx.y * spt, ke = min(ka + spt, kbn);  // the block's tiles [ka, ke)
  const int kt0 = pfa_lo(Pb + 4 * qd, sliding) >> 5;                    // the quad's first tile
  float* pm = PM + ((size_t)qd * nspan + blockIdx.y) * 32 + 16 * (w & 1);
  if (ka >= ke) {  // uniform
    if (nr > 0 && lane < 16) pm[lane] = -1e30f;
    return;
  }
  const int row = r0 + rw + min(lane >> 5, max(nr, 1) - 1);  // this lane's output row
  bool any_t = false, any_m = false;
  for (int t = 0; t < nr; ++t) (pfa_tiled(r0 + rw + t, g) ? any_t : any_m) = true;
  const bool tl = nr > 0 && pfa_tiled(row, g);
  const int P = P0 + (lane >> 5), lo = pfa_lo(P, sliding);
  float qr[TT][4];  // operand row k16 (prompt row k16 / 8, head k16 % 8): element 16 tt + 4 cg + bl
  if (nr > 0) {
    const float* qm = q + (size_t)(r0 + rw + min(k16 >> 3, nr - 1)) * NQ * D + (k16 & 7) * D + bl;
#pragma unroll
    for (int tt = 0; tt < TT; ++tt)
#pragma unroll
      for (int cg = 0; cg < 4; ++cg) qr[tt][cg] = qm[16 * tt + 4 * cg];
  }
  float mx[4] = {-1e30f, -1e30f, -1e30f, -1e30f};
  u32x4_t st[NP];
  auto fetch = [&](int ks) {
#pragma unroll
    for (int k = 0; k < NP; ++k)
      st[k] = *reinterpret_cast<const u32x4_t*>(KC + (size_t)ks * NK * D + 8 * (threadIdx.x + 256 * k));
  };
  auto stage = [&](int b) {  // word wd: 8 steps of chain n from step tt on
#pragma unroll
    for (int k = 0; k < NP; ++k) {
      const int i = threadIdx.x + 256 * k, key = i / WD, wd = i % WD;
      int n, t8;
      if constexpr (D == 512) n = 8 * (wd >> 5) + (wd & 7), t8 = (wd >> 3) & 3;
      else n = 8 * ((wd >> 1) & 1) + (wd >> 2), t8 = wd & 1;
      float* d = KT[b] + (((n >> 2) * T4 + 2 * t8) * 4 + (n & 3)) * RS + 4 * key;
      f32x4v_t v0, v1;
#pragma unroll
      for (int c = 0; c < 2; ++c) {
        v0[2 * c] = as_f32(st[k][c] << 16), v0[2 * c + 1] = as_f32(st[k][c] & 0xFFFF0000u);
        v1[2 * c] = as_f32(st[k][2 + c] << 16), v1[2 * c + 1] = as_f32(st[k][2 + c] & 0xFFFF0000u);
      }
      *reinterpret_cast<f32x4v_t*>(d) = v0;
      *reinterpret_cast<f32x4v_t*>(d + 4 * RS) = v1;
    }
  };
  const int sa = ka * (32 / NK), se = ke * (32 / NK);  // steps of the span
  fetch(sa);
  stage(0);
  lds_barrier();
  for (int ks = sa; ks < se; ++ks) {
    const int b = (ks - sa) & 1;
    fetch(min(ks + 1, se - 1));
    if (nr > 0 && NK * ks + NK > pfa_lo(P0, sliding) && NK * ks <= Pl) {  // (uniform over the wave)
#pragma unroll
      for (int sub = 0; sub < NK / 16; ++sub) {
        const float* kl = KT[b] + bl * RS + 4 * (16 * sub + k16);
        float sum[4];
        if (any_t) {  // attn_tile: 16 chains, v_l = (l, 0) + (l, 1)
          f32x16_t a[4] = {f32x16_t{}, f32x16_t{}, f32x16_t{}, f32x16_t{}};
#pragma unroll
          for (int t4 = 0; t4 < T4; ++t4) {
            f32x4v_t kv[4];
#pragma unroll
            for (int cg = 0; cg < 4; ++cg) kv[cg] = *reinterpret_cast<const f32x4v_t*>(kl + (cg * T4 + t4) * 4 * RS);
#pragma unroll
            for (int c = 0; c < 4; ++c)
#pragma unroll
              for (int cg = 0; cg < 4; ++cg)
                a[cg] = __builtin_amdgcn_mfma_f32_16x16x1f32(qr[4 * t4 + c][cg], kv[cg][c], a[cg], 0, 0, 0);
          }
          a[0] += a[2];  // [4 b + r]: l = b; a[1]: l = 4 + b
          a[1] += a[3];
          a[0] += a[1];
#pragma unroll
          for (int r = 0; r < 4; ++r) sum[r] = (a[0][r] + a[0][4 + r]) + (a[0][8 + r] + a[0][12 + r]);
        }
        if (any_m) {  // run_mh: 8 chains, element 8 t + l in order of t = 2 tt + s
          f32x16_t a[2] = {f32x16_t{}, f32x16_t{}};
#pragma unroll
          for (int t4 = 0; t4 < T4; ++t4) {
            f32x4v_t kv[4];
#pragma unroll
            for (int cg = 0; cg < 4; ++cg) kv[cg] = *reinterpret_cast<const f32x4v_t*>(kl + (cg * T4 + t4) * 4 * RS);
#pragma unroll
            for (int c = 0; c < 4; ++c)
#pragma unroll
              for (int cg = 0; cg < 4; ++cg)
                a[cg & 1] = __builtin_amdgcn_mfma_f32_16x16x1f32(qr[4 * t4 + c][cg], kv[cg][c], a[cg & 1], 0, 0, 0);
          }
          a[0] += a[1];
#pragma unroll
          for (int r = 0; r < 4; ++r) {
            const float v = (a[0][r] + a[0][4 + r]) + (a[0][8 + r] + a[0][12 + r]);
            sum[r] = any_t && tl ? sum[r] : v;
          }
        }
        // register r: row 2 w + lane / 32, head 4 (lane / 16 % 2) + r, key lane % 16
        const int p = NK * ks + 16 * sub + k16;
        float* St = S + (quad_tile0(qd, Pb, sliding) + ((NK * ks) >> 5) - kt0) * 1024 + (p & 31) +
                    32 * (16 * (w & 1) + 4 * bl);
        const bool ok = p <= P && p >= lo;
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          St[32 * r] = sum[r];
          mx[r] = fmaxf(mx[r], ok ? sum[r] : -1e30f);
        }
      }
    }
    stage(b ^ 1);  // last read a step ago
    lds_barrier();
  }
  if (nr <= 0) return;
#pragma unroll
  for (int r = 0; r < 4; ++r) {
    float v = mx[r];
#pragma unroll
    for (int o = 8; o >= 1; o >>= 1) v = fmaxf(v, __shfl_xor(v, o));
    if (k16 == 0) pm[4 * bl + r] = v;
  }
}

// One block per quad, D threads: wave w the dims 64 w .. 64 w + 63 (two tiles).  Weights of CP
// positions at a time in LDS in operand order [8 positions][half][row][4], double-buffered: the next
// step's are formed (by thread (row, 8 positions)) after this step's products are issued.
template <int D>
__global__ __launch_bounds__(D, 2) void k_pfa_out(const float* __restrict__ S, const float* __restrict__ PM,
                                               const uint16_t* __restrict__ VC, float* __restrict__ att, PfGeom g,
                                               int r0, int M, int sliding, int nspan) {
  constexpr int G8 = D / 32, CP = 8 * G8;  // groups of 8 positions, positions of a step
  __shared__ __align__(16) float W[2][G8][2][32][4];
  __shared__ uint64_t T[32];
  __shared__ float dens[32];
  const int nq = gridDim.x, qd = nq - 1 - (int)blockIdx.x;
  const int Pb = g.pos0 + r0, P0 = Pb + 4 * qd, nr = min(4, M - 4 * qd), Pl = P0 + nr - 1;
  const int lom = pfa_lo(P0, sliding), lol = pfa_lo(Pl, sliding);  // first keys of the first and last row
  const int kt0 = lom >> 5, ktn = (Pl >> 5) - kt0 + 1, pk = 32 * kt0;
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6, c32 = lane & 31, half = lane >> 5;
  const int nstep = (Pl - pk) / CP + 1;
  const float* Sq = S + quad_tile0(qd, Pb, sliding) * 1024;
  if (threadIdx.x < 32) T[threadIdx.x] = c_expf_tab_p[threadIdx.x];
  // this thread's weights: row wm (prompt row wm / 8, head wm % 8), positions 8 wg .. of a step
  const int wm = threadIdx.x & 31, wg = threadIdx.x >> 5;
  const int wP = (wm >> 3) < nr ? P0 + (wm >> 3) : -1, wlo = pfa_lo(wP, sliding);
  const bool wt = pfa_tiled(r0 + 4 * qd + min(wm >> 3, nr - 1), g);
  bool any_m = false;
  for (int t = 0; t < nr; ++t) any_m = any_m || !pfa_tiled(r0 + 4 * qd + t, g);
  float mx = -1e30f;  // order free
  for (int i = 0; i < nspan; ++i) mx = fmaxf(mx, PM[((size_t)qd * nspan + i) * 32 + wm]);
  float4 sa, sb;
  auto load_s = [&](int c) {  // (steps past the last tile read it again; their weights are 0)
    const int p = c * CP + 8 * wg, kt = min(p >> 5, ktn - 1);
    const float4* s4 = reinterpret_cast<const float4*>(Sq + (size_t)kt * 1024 + wm * 32 + (p & 31));
    sa = s4[0];
    sb = s4[1];
  };
  float den1 = 0.f;  // run_mh: the row's sum, formed before the weights
  auto weights = [&](int c, bool raw) {
    const int p = pk + c * CP + 8 * wg;
    const float s8[8] = {sa.x, sa.y, sa.z, sa.w, sb.x, sb.y, sb.z, sb.w};
    float e[8];
#pragma unroll
    for (int k = 0; k < 8; ++k) {
      const bool ok = p + k <= wP && p + k >= wlo;
      const float d = s8[k] - mx;
      float v = 0.f;
      if (ok) {
        if (wt) v = raw ? 0.f : exp8(d);
        else v = raw ? libm_expf_neg(d, T) : libm_expf_neg(d, T) / den1;
      }
      e[k] = v;
    }
    float4* d4 = reinterpret_cast<float4*>(&W[c & 1][wg][0][wm][0]);
    d4[0] = make_float4(e[0], e[2], e[4], e[6]);
    d4[32] = make_float4(e[1], e[3], e[5], e[7]);
  };
  float den = 0.f;  // wave dw, lane m < 32: row m's sum in position order
  const int dw = blockIdx.x & (D / 64 - 1);  // (spread over the SIMDs)
  auto add_den = [&](int b) {
    if (w == dw) {
#pragma unroll
      for (int k = 0; k < G8; ++k) {
        const float4 a = *reinterpret_cast<const float4*>(&W[b][k][0][c32][0]);
        const float4 o = *reinterpret_cast<const float4*>(&W[b][k][1][c32][0]);
        den = den + a.x;
        den = den + o.x;
        den = den + a.y;
        den = den + o.y;
        den = den + a.z;
        den = den + o.z;
        den = den + a.w;
        den = den + o.w;
      }
    }
  };
  __syncthreads();  // T
  if (any_m) {  // uniform: run_mh rows divide by their sum before the value pass
    for (int c = 0; c < nstep; ++c) {
      load_s(c);
      weights(c, true);
      __syncthreads();
      add_den(c & 1);
      // (the other half is written next; this half again after the next barrier)
    }
    if (w == dw && lane < 32) dens[lane] = den;
    __syncthreads();
    den1 = dens[wm];
    den = 0.f;
    __syncthreads();
  }
  f32x16_t acc0 = f32x16_t{}, acc1 = f32x16_t{};
  // the value words of 8 positions of dims 64 w + c32 and + 32, VR groups in flight; groups past
  // the part that holds the last position read zeros
  constexpr int VR = 4;
  static_assert(G8 % VR == 0, "whole rings a step");
  const __amdgpu_buffer_rsrc_t vrs = buf_rsrc(VC, (uint32_t)((Pl >> 5) + 1) * (32 * D * 2));
  const uint32_t vo = (uint32_t)(64 * w + c32) * 16u;
  uint4 v0[VR], v1[VR];
#pragma unroll
  for (int i = 0; i < VR; ++i) {
    v0[i] = buf_load16(vrs, (uint32_t)(pk / 8 + i) * (16u * D) + vo);
    v1[i] = buf_load16(vrs, (uint32_t)(pk / 8 + i) * (16u * D) + vo + 512u);
    __builtin_amdgcn_sched_barrier(0);
  }
  load_s(0);
  weights(0, false);
  lds_barrier();
  for (int c = 0; c < nstep; ++c) {
    if (c + 1 < nstep) load_s(c + 1);
    const int b = c & 1, p0 = pk + c * CP;
    const int ng = min(G8, ((Pl - p0) >> 3) + 1);
    for (int kb = 0; kb < ng; kb += VR) {
#pragma unroll
      for (int i = 0; i < VR; ++i) {
        const int k = kb + i, p = p0 + 8 * k;
        const uint32_t a4[4] = {v0[i].x, v0[i].y, v0[i].z, v0[i].w}, b4[4] = {v1[i].x, v1[i].y, v1[i].z, v1[i].w};
        float fa[4], fb[4];  // this half's position of each pair
#pragma unroll
        for (int j = 0; j < 4; ++j) {
          fa[j] = as_f32((a4[j] << (half ? 0 : 16)) & 0xFFFF0000u);
          fb[j] = as_f32((b4[j] << (half ? 0 : 16)) & 0xFFFF0000u);
        }
        bool plain = true;
        if (p < lol || p + 7 > P0) {
          // positions some row does not attend: their weight 0 leaves the row's sum as it is unless
          // the value is not finite or the sum is -0; those take the row-by-row form
          bool odd = false;
#pragma unroll
          for (int j = 0; j < 4; ++j) {
            odd |= (as_u32(fa[j]) & 0x7F800000u) == 0x7F800000u;
            odd |= (as_u32(fb[j]) & 0x7F800000u) == 0x7F800000u;
          }
#pragma unroll
          for (int r = 0; r < 16; ++r) odd |= as_u32(acc0[r]) == 0x80000000u || as_u32(acc1[r]) == 0x80000000u;
          plain = !__any(odd);
          if (!plain) {  // uniform
            for (int j = 0; j < 8; ++j) {
              const uint32_t ua = j < 2 ? a4[0] : (j < 4 ? a4[1] : (j < 6 ? a4[2] : a4[3]));
              const uint32_t ub = j < 2 ? b4[0] : (j < 4 ? b4[1] : (j < 6 ? b4[2] : b4[3]));
              const float va = as_f32((j & 1) ? (ua & 0xFFFF0000u) : (ua << 16));
              const float vb = as_f32((j & 1) ? (ub & 0xFFFF0000u) : (ub << 16));
#pragma unroll
              for (int t = 0; t < 4; ++t) {
                if (t >= nr || p + j > P0 + t || p + j < pfa_lo(P0 + t, sliding)) continue;  // uniform
#pragma unroll
                for (int q = 0; q < 4; ++q) {
                  const float x = W[b][k][j & 1][8 * t + 4 * half + q][j >> 1];
                  acc0[4 * t + q] = fmaf(x, va, acc0[4 * t + q]);
                  acc1[4 * t + q] = fmaf(x, vb, acc1[4 * t + q]);
                }
              }
            }
          }
        }
        __builtin_amdgcn_sched_barrier(0);
        v0[i] = buf_load16(vrs, (uint32_t)(p / 8 + VR) * (16u * D) + vo);
        v1[i] = buf_load16(vrs, (uint32_t)(p / 8 + VR) * (16u * D) + vo + 512u);
        __builtin_amdgcn_sched_barrier(0);
        if (plain) {  // uniform
          const float4 wv = *reinterpret_cast<const float4*>(&W[b][k][half][c32][0]);
          const float ww[4] = {wv.x, wv.y, wv.z, wv.w};
#pragma unroll
          for (int j = 0; j < 4; ++j) {
            acc0 = __builtin_amdgcn_mfma_f32_32x32x2f32(ww[j], fa[j], acc0, 0, 0, 0);
            acc1 = __builtin_amdgcn_mfma_f32_32x32x2f32(ww[j], fb[j], acc1, 0, 0, 0);
          }
        }
      }
    }
    add_den(b);
    if (c + 1 < nstep) weights(c + 1, false);  // into the half read two steps ago
    lds_barrier();
  }
  if (w == dw && lane < 32) dens[lane] = den;
  __syncthreads();
#pragma unroll
  for (int r = 0; r < 16; ++r) {
    const int t = r >> 2, m = 8 * t + 4 * half + (r & 3);
    if (t >= nr) continue;  // uniform
    const bool tl = pfa_tiled(r0 + 4 * qd + t, g);
    const float ih = 1.0f / dens[m];
    const float v[2] = {tl ? r16(acc0[r] * ih) : r16(acc0[r]), tl ? r16(acc1[r] * ih) : r16(acc1[r])};
    float* orow = att + (size_t)(r0 + 4 * qd + t) * NQ * D + (4 * half + (r & 3)) * D + 64 * w + c32;
    orow[0] = v[0];
    orow[32] = v[1];
  }
}

// key tiles a block: 8 (the query operands' loads are a tenth of that) while that gives four blocks a
// CU, else fewer.  A block of 8 rows spans a window of at most 18 tiles (518 positions).
int pfa_spt(int M, int Pb, int sliding, int* nspan) {
  const int rb = (M + 7) / 8, kt = ((Pb + M - 1) >> 5) + 1, ktm = sliding ? std::min(WSTRIDE, kt) : kt;
  int spt = 8;
  while (spt > 1 && (long)rb * ((ktm + spt - 1) / spt) < 1024) --spt;
  *nspan = (ktm + spt - 1) / spt;
  return spt;
}
long long pfa_tiles(int M, int Pb, int sliding) { return quad_tile0((M + 3) / 4, Pb, sliding); }

}  // namespace

// score tiles, then the partial maxima [quad][span][32 rows], of either layer type
long long pfa_scratch_floats(int M, int Pb) {
  long long n = 0;
  for (int sliding = 0; sliding < 2; ++sliding) {
    int ns;
    (void)pfa_spt(M, Pb, sliding, &ns);
    n = std::max(n, pfa_tiles(M, Pb, sliding) * 1024 + (long long)((M + 3) / 4) * ns * 32);
  }
  return n;
}

void launch_pfa(const float* q, const uint16_t* KC, const uint16_t* VC, float* S, float* att, const PfGeom& g, int r0,
                int M, int sliding, hipStream_t st, int hd) {
  const int Pb = g.pos0 + r0, nq = (M + 3) / 4;
  int ns;
  const int spt = pfa_spt(M, Pb, sliding, &ns);
  float* PM = S + pfa_tiles(M, Pb, sliding) * 1024;
  if (hd == 512) {
    hipLaunchKernelGGL(k_pfa_scores<512>, dim3((M + 7) / 8, ns), dim3(256), 0, st, q, KC, S, PM, g, r0, M, sliding, spt, ns);
    hipLaunchKernelGGL(k_pfa_out<512>, dim3(nq), dim3(512), 0, st, S, PM, VC, att, g, r0, M, sliding, ns);
  } else {
    hipLaunchKernelGGL(k_pfa_scores<HD>, dim3((M + 7) / 8, ns), dim3(256), 0, st, q, KC, S, PM, g, r0, M, sliding, spt, ns);
    hipLaunchKernelGGL(k_pfa_out<HD>, dim3(nq), dim3(HD), 0, st, S, PM, VC, att, g, r0, M, sliding, ns);
  }
}

}  // namespace g4v
