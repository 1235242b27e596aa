// g4v_mtp.hip -- the MTP drafter step (draft_step, E:1534-1563) on gfx950.
//
// One draft step on the device, so that a chain of drafts runs without host round trips:
//   comb = [r16(E[tok] * sqrt(1536)), h]  ->  dx = r16(pre . comb)                   (E:1537-1539)
//   4 layers: da = rms(dx, in_ln); q = q_proj . da; per head r16-norm + RoPE at pos;
//     attention over the target's KV cache (layer 13, the global drafter layer: 14), split-KV
//     with T splits, keys [lo, P]; o = r16(o_proj . att); dx = r16(dx + r16(rms(o, post_attn)));
//     da = r16(rms(dx, pre_ff)); act = r16(r16(gelu8(r16 gate)) * r16 up); o = r16(down . act);
//     dx = r16(dx + r16(rms(o, post_ff))); dx = r16(dx * scalar)                    (E:1540-1550)
//   dh = r16(rms(dx, norm)); b_out = r16(post . dh); centroid scores = cent . dh  (E:1551-1553)
//   top-32 centroids (descending score, earlier index first), their 32 x 128 tokens scored
//   against dh, the first maximum is the draft; the runner-up follows the engine's scan
//   (E:1554-1559).
// Every bf16 product is b16_rows (E:586-614): per output, two 8-lane FMA chains over k in steps
// of 16 (k = 16 s + l and 16 s + 8 + l), summed lane-wise, then hsum.  Here 16 lanes of a wave
// hold the 16 chains of one output, so a 256-thread block computes 16 outputs.
#include "g4v_layer.h"

namespace g4v {

namespace {

// input prologue: x; rms(x, nw); r16(rms(x, nw)); [r16(E[*tok] sqrt H), x]; and the residual
// blocks of a drafter layer folded in front of the next product (K = 256, x = dx):
//   RES0 (E:1545-1546): v = r16(x + r16(rms(r16(yin), w1))); input r16(rms(v, nw))
//   RES1 (E:1548-1550): v = r16(r16(x + r16(rms(r16(yin), w1))) * scalar); input rms(v, nw)
//   RES1_R16: as RES1, input r16(rms(v, nw))
// block 0 stores v to dxout (a different buffer from x: other blocks still read x)
enum { B16_PLAIN = 0, B16_RMS = 1, B16_RMS_R16 = 2, B16_COMB = 3, B16_RES0 = 4, B16_RES1 = 5, B16_RES1_R16 = 6 };
enum { B16_STORE = 0, B16_R16 = 1, B16_GATEUP = 2 };                  // output epilogue

struct B16Args {
  const uint16_t* W;   // [rows][K] bf16, chain-major
  const uint16_t* W2;  // B16_GATEUP: the up matrix
  const int* rows;     // row of output n, or null: row n (or, with top: order[top[n / 128] 128 + n % 128])
  const int* top;
  const int* order;
  int N;
  const float* x;      // input [K], or the prologue's source
  const float* nw;     // norm weights (B16_RMS*)
  const uint16_t* E;   // B16_COMB: token embedding [V][1536] ...
  const int* tok;      // ... of token *tok, followed by x [1536]
  float* y;
  float* xout;         // optional: block 0 stores the staged input
  const float* yin;    // RES*: the previous product's output [256]
  const float* w1;     // RES*: post_attn / post_ff
  float* dxout;        // RES*: the updated residual (block 0)
  float scalar;        // RES1*: the layer scalar
};

typedef __attribute__((ext_vector_type(4))) uint32_t u32x4_t;

// [rows][K] to chain-major, a block per row, in place
constexpr int B16_MAXK = 3072;
__global__ __launch_bounds__(256) void k_b16_chains(uint16_t* __restrict__ W, int K) {
  __shared__ uint16_t row[B16_MAXK];
  uint16_t* w = W + (size_t)blockIdx.x * K;
  for (int i = threadIdx.x; i < K; i += 256) row[i] = w[i];
  __syncthreads();
  for (int i = threadIdx.x; i < K; i += 256) w[(i & 15) * (K / 16) + (i >> 4)] = row[i];
}
constexpr int DR_MAXC = 4096;  // centroids

// Weights are kept chain-major (launch_b16_chains): row r's element 16 s + l at r K + l (K / 16) + s, so
// lane l's chain is K / 16 consecutive values, 16-byte loads that are all issued before the prologue
// (with 2-byte loads after it a product took 5.0 us, with its K of 256 or 2048 against a launch of
// 4.5).  The input is staged the same way, a pad of 4 floats per chain.
template <int PRO, int EPI, int KT>
__global__ __launch_bounds__(256) void k_b16(B16Args a) {
  constexpr int CH = KT / 16, CP = CH + 4, NV = CH / 8;  // values of a chain, its LDS stride, its 16-byte words
  constexpr bool NORM = PRO == B16_RMS || PRO == B16_RMS_R16 || PRO >= B16_RES0;
  static_assert(!NORM || KT == 256, "a thread per element of a norm's input");
  __shared__ __align__(16) float xp[16 * CP];
  __shared__ float xs[NORM ? KT : 1];
  __shared__ double red[16];
  const int n = blockIdx.x * 16 + (threadIdx.x >> 4), l = threadIdx.x & 15;
  const bool live = n < a.N;
  const size_t row = !live ? 0
                     : a.rows ? (size_t)a.rows[n]
                     : a.top  ? (size_t)a.order[(size_t)a.top[n >> 7] * 128 + (n & 127)]
                              : (size_t)n;
  u32x4_t wv[NV], wv2[EPI == B16_GATEUP ? NV : 1];
  const u32x4_t* w4 = reinterpret_cast<const u32x4_t*>(a.W + row * KT + l * CH);
#pragma unroll
  for (int v = 0; v < NV; ++v) wv[v] = w4[v];
  if constexpr (EPI == B16_GATEUP) {
    const u32x4_t* u4 = reinterpret_cast<const u32x4_t*>(a.W2 + row * KT + l * CH);
#pragma unroll
    for (int v = 0; v < NV; ++v) wv2[v] = u4[v];
  }
  auto put = [&](int i, float v) { xp[(i & 15) * CP + (i >> 4)] = v; };
  const int i = threadIdx.x;
  if constexpr (PRO == B16_COMB) {
    const int tk = *a.tok;
    const float sqh = sqrtf((float)H);
    for (int e = i; e < H; e += 256) {
      put(e, r16(bf2f(a.E[(size_t)tk * H + e]) * sqh));  // E:1537
      put(H + e, a.x[e]);
    }
  } else if constexpr (!NORM) {
    for (int e = i; e < KT; e += 256) {
      const float v = a.x[e];
      put(e, v);
      if (a.xout && blockIdx.x == 0) a.xout[e] = v;
    }
  } else {  // thread i owns element i
    const float nw = a.nw[i];
    float v = a.x[i];
    if constexpr (PRO >= B16_RES0) {
      const float w1 = a.w1[i], o = r16(a.yin[i]);
      xs[i] = o;
      __syncthreads();
      const float r1 = rms_inv(block_sumsq(xs, 256, red), 256);
      v = r16(v + r16((o * r1) * w1));
      if (PRO != B16_RES0) v = r16(v * a.scalar);
      if (a.dxout && blockIdx.x == 0) a.dxout[i] = v;
      __syncthreads();  // every thread is done with xs
    }
    xs[i] = v;
    __syncthreads();
    const bool rnd = PRO == B16_RMS_R16 || PRO == B16_RES0 || PRO == B16_RES1_R16;
    const float r = rms_inv(block_sumsq(xs, 256, red), 256);
    const float y = (v * r) * nw;  // E:345: (x * r) * w
    v = rnd ? r16(y) : y;
    put(i, v);
    if (a.xout && blockIdx.x == 0) a.xout[i] = v;
  }
  __syncthreads();
  float acc = 0.f, acc2 = 0.f;
  if (live) {  // chain l: elements l, 16 + l, ... in order
    const float4* x4 = reinterpret_cast<const float4*>(xp + l * CP);
#pragma unroll
    for (int v = 0; v < NV; ++v) {
      const float4 x0 = x4[2 * v], x1 = x4[2 * v + 1];
      const float x[8] = {x0.x, x0.y, x0.z, x0.w, x1.x, x1.y, x1.z, x1.w};
#pragma unroll
      for (int k = 0; k < 8; ++k) {
        const uint32_t u = wv[v][k >> 1];
        acc = fmaf(as_f32((k & 1) ? (u & 0xFFFF0000u) : (u << 16)), x[k], acc);
        if constexpr (EPI == B16_GATEUP) {
          const uint32_t u2 = wv2[v][k >> 1];
          acc2 = fmaf(as_f32((k & 1) ? (u2 & 0xFFFF0000u) : (u2 << 16)), x[k], acc2);
        }
      }
    }
  }
  // lanes 0..7 of each 16-lane group: v_l = a_l + b_l, then ((v0+v4)+(v1+v5))+((v2+v6)+(v3+v7))
  auto hsum16 = [](float v) {
    v = v + __shfl_down(v, 8, 16);
    v = v + __shfl_down(v, 4, 16);
    v = v + __shfl_down(v, 1, 16);
    return v + __shfl_down(v, 2, 16);
  };
  const float s = hsum16(acc);
  const float s2 = EPI == B16_GATEUP ? hsum16(acc2) : 0.f;
  if (live && l == 0) {
    if (EPI == B16_STORE) a.y[n] = s;
    else if (EPI == B16_R16) a.y[n] = r16(s);
    else a.y[n] = r16(r16(gelu8(r16(s))) * r16(s2));  // E:669-672
  }
}

// per head (4): x = r16((x * r) * qn), then NeoX RoPE at the step's position (E:1542): P + 1 + j,
// or P + 1 for every step with ENGINE_DRAFT_SAMEPOS (Pp[2] set, E:1516, 1633); D the layer's head
// dim (256, or 512 for the global layer of a drafter checkpoint)
template <int D>
__global__ __launch_bounds__(D) void k_dr_qnorm(float* __restrict__ q, const float* __restrict__ qn,
                                                const float* __restrict__ cs, const float* __restrict__ sn,
                                                const int* __restrict__ Pp, int j) {
  constexpr int NV = 4;
  const int pos = Pp[0] + 1 + (Pp[2] ? 0 : j);
  __shared__ float xv[NV][D];
  __shared__ double part[NV][16];
  __shared__ float rinv[NV];
  const int e = threadIdx.x;
#pragma unroll
  for (int h = 0; h < NV; ++h) xv[h][e] = q[h * D + e];
  __syncthreads();
  if (e < NV * 16) {  // ss_avx2 order (E:326-343): lane t16 sums x[16 i + t16]^2 over i
    const int row = e >> 4, t16 = e & 15;
    double s = 0;
#pragma unroll
    for (int i = 0; i < D / 16; ++i) {
      const double d = (double)xv[row][16 * i + t16];
      s = fma(d, d, s);
    }
    part[row][t16] = s;
  }
  __syncthreads();
  if (e < NV) {
    const double* p = part[e];
    double a[4];
#pragma unroll
    for (int k = 0; k < 4; ++k) a[k] = (p[k] + p[4 + k]) + (p[8 + k] + p[12 + k]);
    rinv[e] = rms_inv((a[0] + a[2]) + (a[1] + a[3]), D);
  }
  __syncthreads();
  float y[NV];
#pragma unroll
  for (int h = 0; h < NV; ++h) y[h] = r16((xv[h][e] * rinv[h]) * qn[e]);
  __syncthreads();
#pragma unroll
  for (int h = 0; h < NV; ++h) xv[h][e] = y[h];
  __syncthreads();
  const int i2 = e & (D / 2 - 1);
  const float c = cs[(size_t)pos * (D / 2) + i2], sv = sn[(size_t)pos * (D / 2) + i2];
#pragma unroll
  for (int h = 0; h < NV; ++h)
    q[h * D + e] = e < D / 2 ? fmaf(xv[h][e], c, -(xv[h][e + D / 2] * sv)) : fmaf(xv[h][e], c, xv[h][e - D / 2] * sv);
}

// a chain's inputs (E:1631-1633): the hidden state, the first token and, per step j, the
// attention geometry (M = 1, keys [lo, P], lo = pos - 511 clamped at 0 on sliding layers,
// pos = P + 1 + j, E:1543, or P + 1 with ENGINE_DRAFT_SAMEPOS: in[3] set, E:1633)
__global__ __launch_bounds__(256) void k_dr_setup(const int* __restrict__ in, const float* __restrict__ hbase,
                                                  float* __restrict__ hin, int* __restrict__ tok,
                                                  AttnGeom* __restrict__ geo, int k, int T) {
  const int t0 = in[0], P = in[1], hrow = in[2], same = in[3];
  const float* src = hrow >= 0 ? hbase + (size_t)hrow * H : reinterpret_cast<const float*>(in + 4);
  for (int i = threadIdx.x; i < H; i += 256) hin[i] = src[i];
  if (threadIdx.x == 0) tok[0] = t0;
  if (threadIdx.x < 2 * k) {
    const int j = threadIdx.x >> 1, sl = (threadIdx.x & 1) == 0;
    AttnGeom g{};
    g.M = 1;
    g.T = T;
    g.pos[0] = P;
    g.lo[0] = sl ? max(0, P + 1 + (same ? 0 : j) - 511) : 0;
    g.skip_lo[0] = 1;
    g.skip_hi[0] = 0;
    g.kmin = g.lo[0];
    g.kmax = P;
    geo[threadIdx.x] = g;
  }
}

// E:1554-1555 top-32 centroids (descending, equal scores in index order): centroid c's place is
// the count of scores above it plus the equal scores before it.  A block ranks 16 centroids, 16
// threads each counting over every 16th group of 4 scores (64 a block, a quarter of the scores a
// thread, took 22.4 us for 2,048 centroids on 32 blocks).
__global__ __launch_bounds__(256) void k_dr_rank(const float* __restrict__ score, int C, int* __restrict__ top) {
  __shared__ __align__(16) float s[DR_MAXC];
  __shared__ int part[16][16];
  for (int j = threadIdx.x; j < C; j += 256) s[j] = score[j];
  __syncthreads();
  const int cl = threadIdx.x & 15, q = threadIdx.x >> 4, c = blockIdx.x * 16 + cl;  // C % 16 == 0
  const float v = s[c];
  int rank = 0;
#pragma unroll 4
  for (int j = 4 * q; j < C; j += 64) {
    const float4 u = *reinterpret_cast<const float4*>(&s[j]);
    rank += (u.x > v) || (u.x == v && j < c);
    rank += (u.y > v) || (u.y == v && j + 1 < c);
    rank += (u.z > v) || (u.z == v && j + 2 < c);
    rank += (u.w > v) || (u.w == v && j + 3 < c);
  }
  part[q][cl] = rank;
  __syncthreads();
  if (q == 0) {
    rank = 0;
#pragma unroll
    for (int k = 0; k < 16; ++k) rank += part[k][cl];
    if (rank < 32) top[rank] = c;
  }
}

// E:1557-1559: the first maximum of the candidate scores is the draft.  The engine's scan keeps
// a runner-up: at the maximum's first index i* it becomes the best before i* (or cand[0] at
// -1e30 when i* = 0), then any later score above it replaces it.  So the runner-up is the first
// maximum after i* if that beats the best before i*, else the best before i*.
__global__ __launch_bounds__(1024) void k_dr_best(const float* __restrict__ cs, const int* __restrict__ top,
                                                  const int* __restrict__ order, int nc, int* __restrict__ tok,
                                                  int* __restrict__ sec, float* __restrict__ gap) {
  auto cand = [&](int i) { return order[(size_t)top[i >> 7] * 128 + (i & 127)]; };  // E:1556
  __shared__ float rv[32];
  __shared__ int ri[32];
  auto argmax = [&](int lo, int hi, float& bv, int& bi) {  // first index of the maximum of [lo, hi)
    float v = -INFINITY;
    int idx = 0x7fffffff;
    for (int i = lo + (int)threadIdx.x; i < hi; i += 1024) {
      const float u = cs[i];
      if (u > v) {  // ascending i per thread: keeps the first
        v = u;
        idx = i;
      }
    }
#pragma unroll
    for (int o = 32; o >= 1; o >>= 1) {
      const float v2 = __shfl_xor(v, o);
      const int i2 = __shfl_xor(idx, o);
      if (v2 > v || (v2 == v && i2 < idx)) {
        v = v2;
        idx = i2;
      }
    }
    __syncthreads();
    if ((threadIdx.x & 63) == 0) {
      rv[threadIdx.x >> 6] = v;
      ri[threadIdx.x >> 6] = idx;
    }
    __syncthreads();
    v = rv[0];
    idx = ri[0];
    for (int w = 1; w < 16; ++w)
      if (rv[w] > v || (rv[w] == v && ri[w] < idx)) {
        v = rv[w];
        idx = ri[w];
      }
    bv = v;
    bi = idx;
  };
  float M, M1 = -1e30f, M2 = -INFINITY;
  int is, i1 = 0, i2 = -1;
  argmax(0, nc, M, is);
  if (is > 0) argmax(0, is, M1, i1);
  if (is + 1 < nc) argmax(is + 1, nc, M2, i2);
  if (threadIdx.x == 0) {
    const bool later = i2 >= 0 && M2 > M1;
    *tok = cand(is);
    *sec = later ? cand(i2) : cand(i1);
    *gap = M - (later ? M2 : M1);
  }
}

}  // namespace

void launch_b16(const B16Launch& L, hipStream_t st) {
  B16Args a{L.W, L.W2, L.rows, L.top, L.order, L.N, L.x, L.nw, L.E, L.tok, L.y, L.xout, L.yin, L.w1, L.dxout,
            L.scalar};
  const dim3 grid((L.N + 15) / 16), block(256);
#define G4V_B16(P, E, K) hipLaunchKernelGGL((k_b16<P, E, K>), grid, block, 0, st, a)
  switch (L.pro * 3 + L.epi) {  // the drafter's products: K 256, o's 4 hd, down's 2048, the pre-projection's 3072
    case B16_PLAIN * 3 + B16_STORE:
      if (L.K == 256) G4V_B16(B16_PLAIN, B16_STORE, 256);
      else if (L.K == 1024) G4V_B16(B16_PLAIN, B16_STORE, 1024);
      else if (L.K == 2048) G4V_B16(B16_PLAIN, B16_STORE, 2048);
      break;
    case B16_RMS * 3 + B16_STORE: G4V_B16(B16_RMS, B16_STORE, 256); break;
    case B16_COMB * 3 + B16_R16: G4V_B16(B16_COMB, B16_R16, 2 * H); break;
    case B16_RES0 * 3 + B16_GATEUP: G4V_B16(B16_RES0, B16_GATEUP, 256); break;
    case B16_RES1 * 3 + B16_STORE: G4V_B16(B16_RES1, B16_STORE, 256); break;
    case B16_RES1_R16 * 3 + B16_STORE: G4V_B16(B16_RES1_R16, B16_STORE, 256); break;
    case B16_RES1_R16 * 3 + B16_R16: G4V_B16(B16_RES1_R16, B16_R16, 256); break;
    default: break;  // not used by the drafter
  }
#undef G4V_B16
}

void launch_b16_chains(uint16_t* W, int rows, int K, hipStream_t st) {
  hipLaunchKernelGGL(k_b16_chains, dim3(rows), dim3(256), 0, st, W, K);
}

void launch_dr_qnorm(float* q, const float* qn, const float* cs, const float* sn, const int* Pp, int j, int hd,
                     hipStream_t st) {
  if (hd == 512) hipLaunchKernelGGL(k_dr_qnorm<512>, dim3(1), dim3(512), 0, st, q, qn, cs, sn, Pp, j);
  else hipLaunchKernelGGL(k_dr_qnorm<HD>, dim3(1), dim3(HD), 0, st, q, qn, cs, sn, Pp, j);
}
void launch_dr_setup(const int* in, const float* hbase, float* hin, int* tok, AttnGeom* geo, int k, int T,
                     hipStream_t st) {
  hipLaunchKernelGGL(k_dr_setup, dim3(1), dim3(256), 0, st, in, hbase, hin, tok, geo, k, T);
}
void launch_dr_rank(const float* score, int C, int* top, hipStream_t st) {
  hipLaunchKernelGGL(k_dr_rank, dim3(C / 16), dim3(256), 0, st, score, C, top);
}
void launch_dr_best(const float* cs, const int* top, const int* order, int nc, int* tok, int* sec, float* gap,
                    hipStream_t st) {
  hipLaunchKernelGGL(k_dr_best, dim3(1), dim3(1024), 0, st, cs, top, order, nc, tok, sec, gap);
}

}  // namespace g4v
