// Prompt prefill: the L rows of a prompt through the talker's bf16 layers, keys and values into the decode cache.
//
// The reference runs the prompt through the talker's modules (qwen3/fast.py:251-263): about forty small launches per layer,
// each of which reads and writes the rows. Here a layer is six: qkv GEMM, per-head norm + RoPE + cache append, causal
// attention, o GEMM, gate/up GEMM, down GEMM. A prompt is a few dozen to a few hundred rows, so the weights (31 MB per
// 0.6B layer) are read about once and each launch is bound by its own latency: every kernel loads what it can at the top.
//
// A prompt of 45 rows through four 0.6B layers and its first code: 1316 us through the modules, 285 now (of which the head,
// the sampling on torch's path and the copies are 150); per launch qkv 5.2 us, norm and RoPE 2.8, attention 7.5, o and down
// 5.5 each, gate/up 6.8. Error of the hidden states, keys and values against 64 bits: 0.010 before, 0.007 now.
//
// Numerics: weights and the GEMMs' inputs are bf16, as in the modules; sums, the residual, q/k/v before their norms and the
// softmax stay in fp32 (the modules round each of them to bf16), and the softmax weights enter P V as two bf16 terms.
//
// Layouts: rows are padded to Mp, a multiple of 64, and rows past L hold zeros or are never used. GEMM inputs are kept in
// the order in which the matrix cores take them (frag_index): 1 KiB per 16 rows and 32 columns, lane m + 16 j holding
// x[m][32 c + 8 j .. + 8]. RMSNorm: the kernel that updates the residual writes bf16(h ⊙ w_next) and, per 16 columns, the
// partial sums of squares; the consumer scales its sums by rsqrt(Σh²/H + eps) (qwen3/kernels.py:180-186).
#include "common.h"
#include "internal.h"

namespace {

constexpr int kWaves = 8, kGemmThreads = kWaves * SK_WAVE;
constexpr int kC = 4;  // 32-wide chunks a wave holds in flight
constexpr float kInvSqrtHd = 0.08838834764831845f;

__device__ __forceinline__ size_t frag_index(int m, int k, int K) {
  return ((size_t)(m >> 4) * (K >> 5) + (k >> 5)) * 512 + (((k >> 3) & 3) * 16 + (m & 15)) * 8 + (k & 7);
}

enum { kQkv = 0, kSwiglu = 1, kAcc = 2 };

struct PGemm {
  const bf16_t* x;         // input fragments, Mp rows of K
  const bf16_t* w[3];      // kQkv: q, k, v; kSwiglu: gate, up; kAcc: one matrix, [rows][K]
  int rows[3];             // kQkv: rows of each
  int K, N, M, Mp;         // N: output columns (kSwiglu: of each matrix)
  const float* ssp;        // [np][Mp] partial sums of squares behind x (NULL: none)
  int np;
  float eps;
  float* out;              // kQkv: [Mp][N]; kAcc: residual [Mp][N], updated in place
  bf16_t* xo;              // kSwiglu: fragments of N columns; kAcc: fragments of bf16(h ⊙ nw)
  const bf16_t* nw;        // kAcc: the next norm's weights
  float* ssp_out;          // kAcc: [N / 16][Mp]
};

// Workgroup (column block, row block): CG groups of 16 output columns (16 of gate and of up each) for MT tiles of 16 rows. Its
// eight waves split K (kC chunks of 32 in flight each), and their sums meet in LDS.
template <int OUT, int MT, int CG>
__global__ __launch_bounds__(kGemmThreads) void k_pgemm(PGemm p) {
  constexpr int kMat = OUT == kSwiglu ? 2 : 1, RG = CG * kMat, kStrips = MT * RG * 4;  // weight group r: columns r / kMat, matrix r % kMat
  __shared__ float red[kWaves][kStrips][64];
  __shared__ float ssq[kGemmThreads / (16 * MT)][16 * MT];
  __shared__ float inv_s[16 * MT];
  const int tid = threadIdx.x, w = __builtin_amdgcn_readfirstlane(tid >> 6), lane = tid & 63, nl = lane & 15, j = lane >> 4;
  const int g = blockIdx.x * CG, m0 = blockIdx.y * 16 * MT, C = p.K >> 5;
  const bf16_t* wr[RG];
#pragma unroll
  for (int r = 0; r < RG; r++) {
    int row = (g + r / kMat) * 16;
    const bf16_t* b = p.w[r % kMat];
    if constexpr (OUT == kQkv)
      if (row >= p.rows[0]) { row -= p.rows[0]; b = p.w[1]; if (row >= p.rows[1]) { row -= p.rows[1]; b = p.w[2]; } }
    wr[r] = b + (size_t)(row + nl) * p.K + 8 * j;
  }
  const bf16_t* xr = p.x + (size_t)(m0 >> 4) * C * 512 + lane * 8;
  f32x4 acc[MT][RG];
#pragma unroll
  for (int m = 0; m < MT; m++)
#pragma unroll
    for (int r = 0; r < RG; r++) acc[m][r] = f32x4{0.f, 0.f, 0.f, 0.f};
  float ssv = 0.f;
  constexpr int kRows = 16 * MT;
  const bool ssl = p.ssp && tid < kGemmThreads / kRows * kRows;
  auto pass = [&](int c0) __attribute__((always_inline)) {
    uint4 wq[kC][RG], xq[kC][MT];
#pragma unroll
    for (int c = 0; c < kC; c++)
#pragma unroll
      for (int r = 0; r < RG; r++) wq[c][r] = gload4((const uint4*)(wr[r] + (c0 + c) * 32));
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int c = 0; c < kC; c++)
#pragma unroll
      for (int m = 0; m < MT; m++) xq[c][m] = gload4((const uint4*)(xr + ((size_t)m * C + c0 + c) * 512));
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int c = 0; c < kC; c++)
#pragma unroll
      for (int m = 0; m < MT; m++)
#pragma unroll
        for (int r = 0; r < RG; r++)
          acc[m][r] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(as_bf16x8(xq[c][m]), as_bf16x8(wq[c][r]), acc[m][r], 0, 0, 0);
  };
  const int per = C / kWaves;  // a multiple of kC
  constexpr int kOut = MT * CG * 4, kOwn = (kOut + kWaves - 1) / kWaves;  // output strips (4 (CG m + c) + i), of a wave
  float hv[kOwn];
  uint32_t nv[kOwn];
  if constexpr (OUT == kAcc) {  // what the epilogue needs
#pragma unroll
    for (int o = 0; o < kOwn; o++) {
      const int st = min(w + o * kWaves, kOut - 1), n = (g + (st >> 2) % CG) * 16 + nl;
      nv[o] = gload(p.nw + n);
      hv[o] = gload(p.out + (size_t)(m0 + 16 * ((st >> 2) / CG) + 4 * j + (st & 3)) * p.N + n);
    }
  }
  constexpr int kSs = 8, kSg = kGemmThreads / kRows;
  float sq[kSs];
  if (ssl) {
#pragma unroll
    for (int u = 0; u < kSs; u++) sq[u] = gload(p.ssp + (size_t)min(tid / kRows + u * kSg, p.np - 1) * p.Mp + m0 + tid % kRows);
  }
  pass(w * per);  // (outside the loop: before a loop's loads the compiler waits for every earlier one)
  for (int c = kC; c < per; c += kC) pass(w * per + c);
  if (ssl) {
#pragma unroll
    for (int u = 0; u < kSs; u++) ssv += tid / kRows + u * kSg < p.np ? sq[u] : 0.f;
    for (int q = tid / kRows + kSs * kSg; q < p.np; q += kSg) ssv += gload(p.ssp + (size_t)q * p.Mp + m0 + tid % kRows);
    ssq[tid / kRows][tid % kRows] = ssv;
  }
  // D[m][n] sits in lane n + 16 (m / 4), element m % 4
#pragma unroll
  for (int m = 0; m < MT; m++)
#pragma unroll
    for (int r = 0; r < RG; r++)
#pragma unroll
      for (int i = 0; i < 4; i++) red[w][((m * CG + r / kMat) * 4 + i) * kMat + r % kMat][lane] = acc[m][r][i];
  __syncthreads();
  if (p.ssp && tid < kRows) {
    float s = 0.f;
    for (int q = 0; q < kGemmThreads / kRows; q++) s += ssq[q][tid];
    inv_s[tid] = rsqrtf(s / p.K + p.eps);
  }
  __syncthreads();
#pragma unroll
  for (int o = 0; o < kOwn; o++) {
    const int st = w + o * kWaves;
    if (st >= kOut) break;
    const int ml = 16 * ((st >> 2) / CG) + 4 * j + (st & 3), m = m0 + ml, gc = g + (st >> 2) % CG, n = gc * 16 + nl;
    const float inv = p.ssp ? inv_s[ml] : 1.f;
    float y = 0.f, u = 0.f;
#pragma unroll
    for (int q = 0; q < kWaves; q++) {
      y += red[q][st * kMat][lane];
      if constexpr (kMat == 2) u += red[q][st * kMat + 1][lane];
    }
    if constexpr (OUT == kQkv) {
      p.out[(size_t)m * p.N + n] = y * inv;
    } else if constexpr (OUT == kSwiglu) {
      p.xo[frag_index(m, n, p.N)] = f2bf(silu_mul(y * inv, u * inv));
    } else {
      const float h = hv[o] + y;
      p.out[(size_t)m * p.N + n] = h;
      p.xo[frag_index(m, n, p.N)] = f2bf(h * bf2f(nv[o]));
      const float ss = row16_sum(h * h);
      if (nl == 0) p.ssp_out[(size_t)gc * p.Mp + m] = ss;
    }
  }
}

// Block m: the prompt's row m (zero past M) as the fp32 residual, its normed fragments and sums of squares (one partial).
__global__ __launch_bounds__(256) void k_pin(const bf16_t* emb, const bf16_t* nw, int M, int Mp, int H, float* h, bf16_t* x, float* ssp) {
  __shared__ float red[4];
  const int m = blockIdx.x, t = threadIdx.x;
  float ss = 0.f;
  for (int k = t; k < H; k += 256) {
    const float v = m < M ? bf2f(gload(emb + (size_t)m * H + k)) : 0.f;
    h[(size_t)m * H + k] = v;
    x[frag_index(m, k, H)] = f2bf(v * bf2f(gload(nw + k)));
    ss = __builtin_fmaf(v, v, ss);
  }
  ss = wave_sum(ss);
  if ((t & 63) == 0) red[t >> 6] = ss;
  __syncthreads();
  if (t == 0) ssp[m] = (red[0] + red[1]) + (red[2] + red[3]);
}

// Block m: the final norm of row m as bf16.
__global__ __launch_bounds__(256) void k_pout(const float* h, const float* ssp, int np, int Mp, const bf16_t* nw, float eps, int H, bf16_t* out) {
  __shared__ float red[4];
  const int m = blockIdx.x, t = threadIdx.x;
  float s = 0.f;
  for (int q = t; q < np; q += 256) s += gload(ssp + (size_t)q * Mp + m);
  s = wave_sum(s);
  if ((t & 63) == 0) red[t >> 6] = s;
  __syncthreads();
  const float inv = rsqrtf(((red[0] + red[1]) + (red[2] + red[3])) / H + eps);
  for (int k = t; k < H; k += 256) out[(size_t)m * H + k] = f2bf(h[(size_t)m * H + k] * inv * bf2f(gload(nw + k)));
}

// Wave (row m, head of q | k | v): per-head RMSNorm and rotate-half RoPE of q (bf16, times 1/sqrt(128)) and k, k and v into
// the cache at position m, v also transposed ([kv head][dim][Mp], zero past M) for the attention's P V.
struct PRope {
  const float* qkv;   // [Mp][(nq + 2 nkv) * 128]
  const bf16_t* qn;
  const bf16_t* kn;
  float eps;
  const float* rope;  // [>= M][cos 64 | sin 64]
  int M, Mp, nq, nkv, max_len;
  bf16_t* q;          // [nq][Mp][128]
  bf16_t* kc;         // [nkv][max_len][128]
  bf16_t* vc;
  bf16_t* vt;         // [nkv][128][Mp]
};
__global__ __launch_bounds__(256) void k_prope(PRope a) {
  const int m = blockIdx.x, hd = blockIdx.y * 4 + (threadIdx.x >> 6), lane = threadIdx.x & 63;
  const bool live = m < a.M;
  const float* src = a.qkv + (size_t)m * (a.nq + 2 * a.nkv) * SK_HD + hd * SK_HD;
  float x0 = gload(src + lane), x1 = gload(src + lane + 64);
  if (hd >= a.nq + a.nkv) {
    const int g = hd - a.nq - a.nkv;
    const bf16_t v0 = live ? f2bf(x0) : (bf16_t)0, v1 = live ? f2bf(x1) : (bf16_t)0;
    bf16_t* vt = a.vt + ((size_t)g * SK_HD + lane) * a.Mp + m;
    vt[0] = v0;
    vt[(size_t)64 * a.Mp] = v1;
    if (live) {
      bf16_t* v = a.vc + ((size_t)g * a.max_len + m) * SK_HD + lane;
      v[0] = v0;
      v[64] = v1;
    }
    return;
  }
  if (!live) return;
  const bool isq = hd < a.nq;
  const bf16_t* nw = isq ? a.qn : a.kn;
  const float inv = rsqrtf(wave_sum(x0 * x0 + x1 * x1) / SK_HD + a.eps);
  x0 = x0 * inv * bf2f(gload(nw + lane));
  x1 = x1 * inv * bf2f(gload(nw + lane + 64));
  const float c = gload(a.rope + (size_t)m * SK_HD + lane), s = gload(a.rope + (size_t)m * SK_HD + 64 + lane);
  const float r0 = x0 * c - x1 * s, r1 = x1 * c + x0 * s;
  bf16_t* o = isq ? a.q + ((size_t)hd * a.Mp + m) * SK_HD : a.kc + ((size_t)(hd - a.nq) * a.max_len + m) * SK_HD;
  o[lane] = f2bf(r0);
  o[lane + 64] = f2bf(r1);
}

// Block (16 queries, kv head): causal attention of both q heads. Wave w takes head w % 2 and the key tiles (32 keys) w / 2,
// w / 2 + 2, ... to its own maxima, sums and Σ p v; the two waves of a head meet in LDS. Scores and P V on the matrix
// cores (D[query][key], then A = the weights as two bf16 terms after a trip through LDS that only this wave uses).
struct PAttn {
  const bf16_t* q;
  const bf16_t* kc;
  const bf16_t* vt;
  int M, Mp, nkv, max_len;
  bf16_t* att;   // fragments of nq * 128 columns
};
__global__ __launch_bounds__(256) void k_pattn(PAttn a) {
  __shared__ __align__(16) bf16_t ps[4][2][16][40];  // [wave][term][query][32 keys, padded]
  __shared__ float om[2][64][32 + 1];
  __shared__ float mlx[2][2][16];
  const int q0 = blockIdx.x * 16, kvh = blockIdx.y, t = threadIdx.x, w = __builtin_amdgcn_readfirstlane(t >> 6), lane = t & 63;
  const int nl = lane & 15, j = lane >> 4, hd = 2 * kvh + (w & 1);
  const bf16_t* K = a.kc + (size_t)kvh * a.max_len * SK_HD;
  const bf16_t* V = a.vt + (size_t)kvh * SK_HD * a.Mp;
  bf16x8 qa[4];
  const bf16_t* qr = a.q + ((size_t)hd * a.Mp + min(q0 + nl, a.M - 1)) * SK_HD + 8 * j;
#pragma unroll
  for (int c = 0; c < 4; c++) qa[c] = as_bf16x8(gload4((const uint4*)(qr + 32 * c)));
  f32x4 acc[8];
  float mx[4], l[4];
#pragma unroll
  for (int d = 0; d < 8; d++) acc[d] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
  for (int i = 0; i < 4; i++) { mx[i] = -INFINITY; l[i] = 0.f; }
  const int last = min(q0 + 15, a.M - 1);
  for (int k0 = 32 * (w >> 1); k0 <= last; k0 += 64) {
    uint4 kr[2][4], vr[8];
#pragma unroll
    for (int i = 0; i < 2; i++)
#pragma unroll
      for (int c = 0; c < 4; c++) kr[i][c] = gload4((const uint4*)(K + (size_t)min(k0 + 16 * i + nl, a.M - 1) * SK_HD + 32 * c + 8 * j));
#pragma unroll
    for (int d = 0; d < 8; d++) vr[d] = gload4((const uint4*)(V + (size_t)(16 * d + nl) * a.Mp + k0 + 8 * j));
    __builtin_amdgcn_sched_barrier(0);
    f32x4 s[2];
#pragma unroll
    for (int i = 0; i < 2; i++) {
      s[i] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int c = 0; c < 4; c++) s[i] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(qa[c], as_bf16x8(kr[i][c]), s[i], 0, 0, 0);
    }
#pragma unroll
    for (int i = 0; i < 4; i++) {  // query q0 + 4 j + i, keys k0 + nl and k0 + 16 + nl
      const int q = q0 + 4 * j + i;
      const bool u0 = k0 + nl <= q && k0 + nl < a.M, u1 = k0 + 16 + nl <= q && k0 + 16 + nl < a.M;
      const float s0 = u0 ? s[0][i] * kInvSqrtHd : -INFINITY, s1 = u1 ? s[1][i] * kInvSqrtHd : -INFINITY;
      const float mn = fmaxf(mx[i], row16_max(fmaxf(s0, s1)));
      const float e0 = u0 ? expf(s0 - mn) : 0.f, e1 = u1 ? expf(s1 - mn) : 0.f;
      const float f = mx[i] == -INFINITY ? 0.f : expf(mx[i] - mn);
      l[i] = l[i] * f + row16_sum(e0 + e1);
      mx[i] = mn;
#pragma unroll
      for (int d = 0; d < 8; d++) acc[d][i] *= f;
      const bf16_t h0 = f2bf_hw(e0), h1 = f2bf_hw(e1);
      ps[w][0][4 * j + i][nl] = h0;
      ps[w][0][4 * j + i][16 + nl] = h1;
      ps[w][1][4 * j + i][nl] = f2bf_hw(e0 - bf2f(h0));
      ps[w][1][4 * j + i][16 + nl] = f2bf_hw(e1 - bf2f(h1));
    }
    wave_sync();
    const bf16x8 p0 = as_bf16x8(*(const uint4*)&ps[w][0][nl][8 * j]), p1 = as_bf16x8(*(const uint4*)&ps[w][1][nl][8 * j]);
#pragma unroll
    for (int d = 0; d < 8; d++) {
      acc[d] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(p0, as_bf16x8(vr[d]), acc[d], 0, 0, 0);
      acc[d] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(p1, as_bf16x8(vr[d]), acc[d], 0, 0, 0);
    }
    wave_sync();
  }
  // the second wave of a head hands over; the first merges and writes
  if (w >= 2) {
#pragma unroll
    for (int d = 0; d < 8; d++)
#pragma unroll
      for (int i = 0; i < 4; i++) om[w & 1][lane][4 * d + i] = acc[d][i];
    if (nl == 0)
#pragma unroll
      for (int i = 0; i < 4; i++) { mlx[w & 1][0][4 * j + i] = mx[i]; mlx[w & 1][1][4 * j + i] = l[i]; }
  }
  __syncthreads();
  if (w >= 2) return;
#pragma unroll
  for (int i = 0; i < 4; i++) {
    const int q = q0 + 4 * j + i;
    const float m2 = mlx[w][0][4 * j + i], l2 = mlx[w][1][4 * j + i], mm = fmaxf(mx[i], m2);
    const float f1 = mx[i] == -INFINITY ? 0.f : expf(mx[i] - mm), f2 = m2 == -INFINITY ? 0.f : expf(m2 - mm);
    const float r = 1.f / (l[i] * f1 + l2 * f2);
#pragma unroll
    for (int d = 0; d < 8; d++) {
      const float o = (acc[d][i] * f1 + om[w][lane][4 * d + i] * f2) * r;
      a.att[frag_index(q, hd * SK_HD + 16 * d + nl, 2 * a.nkv * SK_HD)] = q < a.M ? f2bf(o) : (bf16_t)0;
    }
  }
}

int64_t up256(int64_t v) { return (v + 255) / 256 * 256; }
struct PWs {
  int64_t h, x, xb, ssa, ssb, qkv, q, vt, att, act, total;
};
PWs pws(int H, int I, int nq, int nkv, int L) {
  PWs w;
  int64_t o = 0;
  const int64_t Mp = (L + 63) / 64 * 64;
  auto take = [&](int64_t bytes) { const int64_t at = o; o += up256(bytes); return at; };
  w.h = take(Mp * H * 4);
  w.x = take(Mp * H * 2);
  w.xb = take(Mp * H * 2);
  w.ssa = take(H / 16 * Mp * 4);
  w.ssb = take(H / 16 * Mp * 4);
  w.qkv = take(Mp * (nq + 2 * nkv) * SK_HD * 4);
  w.q = take(Mp * nq * SK_HD * 2);
  w.vt = take(Mp * nkv * SK_HD * 2);
  w.att = take(Mp * nq * SK_HD * 2);
  w.act = take(Mp * I * 2);
  w.total = o;
  return w;
}
bool shape_ok(int H, int I, int nq, int nkv, int L) {
  return H > 0 && I > 0 && nkv > 0 && nq == 2 * nkv && nkv % 2 == 0 && L > 0 && L <= 65536 && H % 1024 == 0 && I % 1024 == 0 && nq * SK_HD % 1024 == 0;
}

// The tile of a workgroup: the largest of 4 x 4, 4 x 2, 4 x 1 (16-row tiles x column groups; gate/up's groups are two
// matrices wide, so up to 4 x 2), fewer rows for shorter prompts, that leaves kMinWg workgroups: large tiles read the rows and
// weights fewer times from the caches, small ones fill the chip. Against one column group everywhere, four row tiles where a row
// of workgroups has 128 and one elsewhere (whole prompts, us): 0.6B four layers 250 rows 446 -> 389, two layers 1900 rows
// 1152 -> 912; 1.7B two layers 33 rows 273 -> 255, 250 rows 447 -> 382, 900 rows 1140 -> 931.
constexpr int kMinWg = 192;
template <int OUT, int MT, int CG>
hipError_t run(const PGemm& p, int tiles, hipStream_t st) {
  hipLaunchKernelGGL((k_pgemm<OUT, MT, CG>), dim3(p.N / 16 / CG, (tiles + MT - 1) / MT), dim3(kGemmThreads), 0, st, p);
  return hipGetLastError();
}
template <int OUT>
hipError_t go(const PGemm& p, hipStream_t st) {
  const int tiles = (p.M + 15) / 16, G = p.N / 16;
  auto wgs = [&](int mt, int cg) { return (tiles + mt - 1) / mt * (G / cg); };
  if constexpr (OUT != kSwiglu)
    if (tiles > 3 && wgs(4, 4) >= kMinWg) return run<OUT, 4, 4>(p, tiles, st);
  if (tiles > 3) {
    if (wgs(4, 2) >= kMinWg) return run<OUT, 4, 2>(p, tiles, st);
    if (wgs(4, 1) >= kMinWg) return run<OUT, 4, 1>(p, tiles, st);
  }
  if (tiles == 3) {
    if (wgs(3, 2) >= kMinWg) return run<OUT, 3, 2>(p, tiles, st);
    if (wgs(3, 1) >= kMinWg) return run<OUT, 3, 1>(p, tiles, st);
  }
  if (tiles >= 2) {
    if (wgs(2, 2) >= kMinWg) return run<OUT, 2, 2>(p, tiles, st);
    if (wgs(2, 1) >= kMinWg) return run<OUT, 2, 1>(p, tiles, st);
  }
  return run<OUT, 1, 1>(p, tiles, st);
}

}  // namespace

extern "C" int64_t sk_prefill_workspace_size(int hidden, int inter, int nq, int nkv, int rows) {
  return shape_ok(hidden, inter, nq, nkv, rows) ? pws(hidden, inter, nq, nkv, rows).total : 0;
}

extern "C" int sk_prefill(const sk_prefill_desc* d, void* stream) {
  if (!d) return sk_set_error(SK_EINVAL, "sk_prefill: null descriptor");
  const int H = d->hidden, I = d->inter, nq = d->nq, nkv = d->nkv, M = d->rows;
  if (!shape_ok(H, I, nq, nkv, M))
    return sk_set_error(SK_EINVAL, "sk_prefill: needs hidden, inter and nq*128 multiples of 1024, nq == 2 nkv, 1..65536 rows");
  if (d->n_layers <= 0 || !d->layers || !d->embeds || !d->norm || !d->rope || !d->out || !d->workspace || M > d->max_len)
    return sk_set_error(SK_EINVAL, "sk_prefill: null pointer, no layers, or more rows than the cache holds");
  if (!SK_ALIGNED16(d->workspace) || !SK_ALIGNED16(d->embeds) || !SK_ALIGNED16(d->out))
    return sk_set_error(SK_EINVAL, "sk_prefill: workspace, embeds and out must be 16-byte aligned");
  if (d->workspace_bytes < sk_prefill_workspace_size(H, I, nq, nkv, M)) return sk_set_error(SK_EWORKSPACE, "sk_prefill: workspace too small");
  for (int l = 0; l < d->n_layers; l++) {
    const sk_prefill_layer& y = d->layers[l];
    const void* ptr[] = {y.q, y.k, y.v, y.o, y.gate, y.up, y.down, y.in_norm, y.post_norm, y.qn, y.kn, y.kc, y.vc};
    for (const void* q : ptr)
      if (!q || !SK_ALIGNED16(q)) return sk_set_error(SK_EINVAL, "sk_prefill: null or unaligned pointer in a layer");
  }
  hipStream_t st = (hipStream_t)stream;
  char* ws = (char*)d->workspace;
  const PWs w = pws(H, I, nq, nkv, M);
  const int Mp = (M + 63) / 64 * 64, nqkv = (nq + 2 * nkv) * SK_HD;
  float *h = (float*)(ws + w.h), *ssa = (float*)(ws + w.ssa), *ssb = (float*)(ws + w.ssb), *qkv = (float*)(ws + w.qkv);
  bf16_t *x = (bf16_t*)(ws + w.x), *xb = (bf16_t*)(ws + w.xb), *q = (bf16_t*)(ws + w.q), *vt = (bf16_t*)(ws + w.vt);
  bf16_t *att = (bf16_t*)(ws + w.att), *act = (bf16_t*)(ws + w.act);
  auto bw = [](const void* p) { return (const bf16_t*)p; };
  hipLaunchKernelGGL(k_pin, dim3(Mp), dim3(256), 0, st, bw(d->embeds), bw(d->layers[0].in_norm), M, Mp, H, h, x, ssa);
  hipError_t e = hipGetLastError();
  for (int l = 0; l < d->n_layers && e == hipSuccess; l++) {
    const sk_prefill_layer& y = d->layers[l];
    const PGemm g1{x, {bw(y.q), bw(y.k), bw(y.v)}, {nq * SK_HD, nkv * SK_HD, nkv * SK_HD}, H, nqkv, M, Mp, ssa, l ? H / 16 : 1, d->eps, qkv,
                   nullptr, nullptr, nullptr};
    if ((e = go<kQkv>(g1, st)) != hipSuccess) break;
    const PRope r{qkv, bw(y.qn), bw(y.kn), d->eps, d->rope, M, Mp, nq, nkv, d->max_len, q, (bf16_t*)y.kc, (bf16_t*)y.vc, vt};
    hipLaunchKernelGGL(k_prope, dim3(Mp, (nq + 2 * nkv) / 4), dim3(256), 0, st, r);
    if ((e = hipGetLastError()) != hipSuccess) break;
    const PAttn a{q, (const bf16_t*)y.kc, vt, M, Mp, nkv, d->max_len, att};
    hipLaunchKernelGGL(k_pattn, dim3((M + 15) / 16, nkv), dim3(256), 0, st, a);
    if ((e = hipGetLastError()) != hipSuccess) break;
    const PGemm g2{att, {bw(y.o), nullptr, nullptr}, {}, nq * SK_HD, H, M, Mp, nullptr, 0, d->eps, h, xb, bw(y.post_norm), ssb};
    if ((e = go<kAcc>(g2, st)) != hipSuccess) break;
    const PGemm g3{xb, {bw(y.gate), bw(y.up), nullptr}, {}, H, I, M, Mp, ssb, H / 16, d->eps, nullptr, act, nullptr, nullptr};
    if ((e = go<kSwiglu>(g3, st)) != hipSuccess) break;
    const void* nw = l + 1 < d->n_layers ? d->layers[l + 1].in_norm : d->norm;
    const PGemm g4{act, {bw(y.down), nullptr, nullptr}, {}, I, H, M, Mp, nullptr, 0, d->eps, h, x, bw(nw), ssa};
    e = go<kAcc>(g4, st);
  }
  if (e == hipSuccess) {
    hipLaunchKernelGGL(k_pout, dim3(M), dim3(256), 0, st, h, ssa, H / 16, Mp, bw(d->norm), d->eps, H, (bf16_t*)d->out);
    e = hipGetLastError();
  }
  return sk_check_launch(e, "sk_prefill");
}
