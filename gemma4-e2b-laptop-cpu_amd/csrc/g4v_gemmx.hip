// g4v_gemmx.hip -- exact-order W4G32 product of many rows (prompt blocks) on the fp32 matrix cores.
//
// Same arithmetic as g4v_gemv.hip (w4::gemm_rows_tile, engine/w4g32_avx2.h:64-96): eight lane
// chains per output, in each 32-group a = the fma chain of lane j's four weights, row_j =
// fma(a, sc, row_j), off = fma(sc, gsum, off), y = hsum8(row) - 8 off.
//
// v_mfma_f32_32x32x2_f32 adds its two products to the accumulator one after the other, each with
// one rounding (D = fma(a1, b1, fma(a0, b0, C)), subnormals kept: equal to fmaf in that order on
// every one of 8192 outputs tried, in normal, subnormal-result and subnormal-operand ranges), so
// two of them chained from 0 form a lane chain's four-term a for 32 rows x 32 outputs.  (From +0
// instead of the reference's plain first product only the sign of a zero a can differ, and
// fma(+-0, sc, row) leaves row as it is: row starts at +0, and it is -0 only after a product a sc
// below 2^-150 of negative sign, where the sign of an output that is zero is all that can change.)
// Operands need no shuffling: instruction k = lane / 32 takes x[32g + 16k + 2j] (then + 1) and
// nibble lo (then hi) of byte 8k + j, so a lane holds consecutive floats of its row and
// consecutive bytes of its output's group, as the W4A8 operand tiles (k_tile_a8) store them.
//
// What bounds it: an instruction of 2048 FMAs takes 66 cycles of its SIMD and fp32 VALU work does
// not overlap with it (measured: 8 added fmas add 23 cycles at 4 waves a SIMD), so a group of a
// 32 x 32 tile costs 16 instructions and 8 x 16 fold fmas, ~1450 cycles; the decode, once per
// 32 outputs, adds ~10%.  The 8-row VALU GEMV spends 41 operations per (row, output, group) plus
// an LDS read per fma.  A block is one tile (two with gate / up) whose eight chains sit on eight
// waves: they only meet in the final sum, so a tile's latency is an eighth of its work and small
// prompts still fill the SIMDs.  The block's rows go through LDS four groups at a time (the eight
// waves read different floats of the same lines), double-buffered, one LDS barrier per step.
// Measured (333-row prompt, 35 layers, exact float): q/k/v, o and down 69 us, gate / up 181 us on
// average, the prompt 212.5 -> 18.6 ms (16.5 with its attention on the matrix cores; the 8-row GEMV took 42 launches of 8 to 42 us a product).
// Row pitch 130 floats: the 32 rows of an 8-byte read fall on 64 different banks.
#include "g4v_internal.h"

namespace g4v {

typedef __attribute__((ext_vector_type(16))) float f32x16_t;

// gs[m][g] = x[m][32g] + ... + x[m][32g + 31] in order (W:22)
__global__ __launch_bounds__(256) void k_group_sums(const float* __restrict__ x, float* __restrict__ gs, int n) {
  const int u = blockIdx.x * 256 + threadIdx.x;
  if (u >= n) return;
  const float4* p = reinterpret_cast<const float4*>(x + (size_t)u * 32);
  float4 v[8];
#pragma unroll
  for (int i = 0; i < 8; ++i) v[i] = p[i];
  float s = 0.f;
#pragma unroll
  for (int i = 0; i < 8; ++i) {
    s += v[i].x;
    s += v[i].y;
    s += v[i].z;
    s += v[i].w;
  }
  gs[u] = s;
}

// NT tiles of 32 outputs: NT = 2 is the gate / up pair (matrices 0 and 1, the same outputs), whose
// epilogue writes the activation.  Wave w is chain w of every output.
constexpr int GX_PITCH = 130;  // floats of a staged row: 4 groups + 2
template <int NT>
__global__ __launch_bounds__(512, NT == 1 ? 6 : 4) void k_gemm_x(GemmXArgs a) {
  __shared__ __align__(16) float X[2][32 * GX_PITCH];  // later the chains' sums [8][16][64]
  __shared__ __align__(8) float S[2][4][32];           // the step's group sums
  __shared__ float O[32][32];
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
  const int c32 = lane & 31, half = lane >> 5;
  const int K = a.K, G = K / 32, NC = G / 4;
  const int m0 = blockIdx.y * 32;
  const int mi = NT == 2 ? 0 : (((int)blockIdx.x >= a.t0[1]) + ((int)blockIdx.x >= a.t0[2]));
  const int nb = NT == 2 ? (int)blockIdx.x * 32 : ((int)blockIdx.x - a.t0[mi]) * 32;
  // staging: 8 floats of row tid / 16 (rows past M repeat the last one and are not stored)
  const int srow = threadIdx.x >> 4, scol = 8 * (threadIdx.x & 15);
  // (32-bit byte offsets from the uniform bases: M K floats stay below 4 GB, checked at the launch)
  const char *xb = reinterpret_cast<const char*>(a.x), *gb = reinterpret_cast<const char*>(a.gs);
  const uint32_t xo = ((uint32_t)min(m0 + srow, a.M - 1) * (uint32_t)a.ldx + (uint32_t)scol) * 4u;
  // this lane's two offset chains: rows om, om + 1, output c32
  const int om = 4 * w + 2 * half;
  // the step's 32 x 4 group sums, stored by every wave pair alike (a branch here would cost registers)
  const int grow = (threadIdx.x >> 2) & 31, gcol = threadIdx.x & 3;
  const uint32_t go = ((uint32_t)min(m0 + grow, a.M - 1) * (uint32_t)G + (uint32_t)gcol) * 4u;
  const int hb = 2 * half + (w >> 2), sh = 8 * (w & 3);  // 4-byte slice of the group, the byte in it
  const char *wb[NT], *sb[NT];
  uint32_t wo, so;
#pragma unroll
  for (int u = 0; u < NT; ++u) {
    const int q = NT == 2 ? u : mi;
    const uint4* tw = q == 0 ? a.tw[0] : (q == 1 ? a.tw[1] : a.tw[2]);
    const uint4* ts = q == 0 ? a.ts[0] : (q == 1 ? a.ts[1] : a.ts[2]);
    const int N = q == 0 ? a.N[0] : (q == 1 ? a.N[1] : a.N[2]);
    const int t = min((nb + c32) >> 4, N / 16 - 1), r = c32 & 15;  // outputs past N read the last tile
    wb[u] = reinterpret_cast<const char*>(tw);
    sb[u] = reinterpret_cast<const char*>(ts);
    wo = (uint32_t)(t * (G / 4) * 64 + hb * 16 + r) * 16u;  // (the same for both matrices of a pair)
    so = (uint32_t)(t * (G / 8) * 16 + r) * 16u;
  }
  auto load_w = [&](int u, int c) { return *reinterpret_cast<const uint4*>(wb[u] + (wo + 1024u * c)); };
  auto load_s = [&](int u, int c8) { return *reinterpret_cast<const uint4*>(sb[u] + (so + 256u * c8)); };
  f32x16_t row[NT];
  float off[NT][2];
#pragma unroll
  for (int u = 0; u < NT; ++u) {
    row[u] = f32x16_t{};
    off[u][0] = off[u][1] = 0.f;
  }
  float4 x0 = *reinterpret_cast<const float4*>(xb + xo), x1 = *reinterpret_cast<const float4*>(xb + (xo + 16u));
  uint4 wn[NT], sv[NT];
  float gn = *reinterpret_cast<const float*>(gb + go);
#pragma unroll
  for (int u = 0; u < NT; ++u) {
    wn[u] = load_w(u, 0);
    sv[u] = load_s(u, 0);
  }
  auto stage = [&](int b) {  // 8-byte stores: the pitch keeps rows 8-byte aligned only
    float2* p = reinterpret_cast<float2*>(X[b] + srow * GX_PITCH + scol);
    p[0] = make_float2(x0.x, x0.y), p[1] = make_float2(x0.z, x0.w);
    p[2] = make_float2(x1.x, x1.y), p[3] = make_float2(x1.z, x1.w);
    S[b][gcol][grow] = gn;
  };
  stage(0);
  lds_barrier();
  for (int c = 0; c < NC; ++c) {
    const int cn = min(c + 1, NC - 1);  // the next step's operands in flight (the last step's are not used)
    uint4 wc[NT], sc8[NT];
#pragma unroll
    for (int u = 0; u < NT; ++u) wc[u] = wn[u], sc8[u] = sv[u];
    x0 = *reinterpret_cast<const float4*>(xb + (xo + 512u * cn));
    x1 = *reinterpret_cast<const float4*>(xb + (xo + 512u * cn + 16u));
#pragma unroll
    for (int u = 0; u < NT; ++u) {
      wn[u] = load_w(u, cn);
      sv[u] = load_s(u, cn >> 1);
    }
    gn = *reinterpret_cast<const float*>(gb + (go + 16u * cn));
    const float* xl = X[c & 1] + c32 * GX_PITCH + 16 * half + 2 * w;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const float2 xv = *reinterpret_cast<const float2*>(xl + 32 * i);
      const float2 gc = *reinterpret_cast<const float2*>(&S[c & 1][i][om]);
#pragma unroll
      for (int u = 0; u < NT; ++u) {
        const uint32_t d = i == 0 ? wc[u].x : (i == 1 ? wc[u].y : (i == 2 ? wc[u].z : wc[u].w));
        const float b0 = (float)((d >> sh) & 15u), b1 = (float)((d >> (sh + 4)) & 15u);
        const uint32_t e = (c & 1) ? (i < 2 ? sc8[u].z : sc8[u].w) : (i < 2 ? sc8[u].x : sc8[u].y);
        const float sc = as_f32((i & 1) ? (e & 0xFFFF0000u) : (e << 16));
        f32x16_t t = __builtin_amdgcn_mfma_f32_32x32x2f32(xv.x, b0, f32x16_t{}, 0, 0, 0);
        t = __builtin_amdgcn_mfma_f32_32x32x2f32(xv.y, b1, t, 0, 0, 0);
        off[u][0] = fmaf(sc, gc.x, off[u][0]);
        off[u][1] = fmaf(sc, gc.y, off[u][1]);
#pragma unroll
        for (int r = 0; r < 16; ++r) row[u][r] = fmaf(t[r], sc, row[u][r]);
        __builtin_amdgcn_sched_barrier(0);  // one product in registers at a time: 3 blocks a CU
      }
    }
    stage((c & 1) ^ 1);  // last read a step ago
    lds_barrier();
  }
  // D register r of lane (half, c32) is row 8 (r / 4) + 4 half + r % 4, output c32
  float(*R)[16][64] = reinterpret_cast<float(*)[16][64]>(&X[0][0]);
  static_assert(sizeof(X) >= 8 * 16 * 64 * 4, "the chains' sums fit the staging buffer");
  float g[2];
#pragma unroll
  for (int u = 0; u < NT; ++u) {
    if (u) __syncthreads();
#pragma unroll
    for (int r = 0; r < 16; ++r) R[w][r][lane] = row[u][r];
    O[om][c32] = off[u][0];
    O[om + 1][c32] = off[u][1];
    __syncthreads();
#pragma unroll
    for (int q = 0; q < 2; ++q) {
      const int idx = threadIdx.x + q * 512, r = idx >> 6, l = idx & 63;
      float v[8];
#pragma unroll
      for (int j = 0; j < 8; ++j) v[j] = R[j][r][l];
      const int ml = 8 * (r >> 2) + 4 * (l >> 5) + (r & 3), m = m0 + ml, n = nb + (l & 31);
      const float y = hsum8(v) - 8.f * O[ml][l & 31];
      if (NT == 2 && u == 0) {
        g[q] = y;
        continue;
      }
      const int N = mi == 0 ? a.N[0] : (mi == 1 ? a.N[1] : a.N[2]);
      if (m < a.M && n < N) {
        float* yb = mi == 0 ? a.y[0] : (mi == 1 ? a.y[1] : a.y[2]);
        const int ld = mi == 0 ? a.ldy[0] : (mi == 1 ? a.ldy[1] : a.ldy[2]);
        yb[(size_t)m * ld + n] = NT == 2 ? r16(r16(gelu8(r16(g[q]))) * r16(y)) : y;  // E:292-299
      }
    }
  }
}

int launch_gemm_x(const GemmXArgs& a_in, int nmat, bool gateup, hipStream_t st) {
  GemmXArgs a = a_in;
  if (a.M < 1 || (long)a.M * a.K >= (1L << 30) || a.K % 256 || nmat < 1 || nmat > 3) return 0;
  if (gateup && (nmat != 2 || a.N[0] != a.N[1])) return 0;
  for (int i = 0; i < nmat; ++i)
    if (a.N[i] % 16 || (long)a.N[i] * a.K >= (1L << 32) || !a.tw[i] || !a.ts[i]) return 0;
  a.t0[0] = 0;
  for (int i = 0; i < 3; ++i) a.t0[i + 1] = a.t0[i] + (i < nmat ? (a.N[i] + 31) / 32 : 0);
  const int n = a.M * (a.K / 32);
  hipLaunchKernelGGL(k_group_sums, dim3((n + 255) / 256), dim3(256), 0, st, a.x, const_cast<float*>(a.gs), n);
  const int mt = (a.M + 31) / 32;
  if (gateup) hipLaunchKernelGGL(k_gemm_x<2>, dim3(a.t0[1], mt), dim3(512), 0, st, a);
  else hipLaunchKernelGGL(k_gemm_x<1>, dim3(a.t0[3], mt), dim3(512), 0, st, a);
  return 1;
}

}  // namespace g4v
