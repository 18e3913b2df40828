// Batched talker decode: up to 16 streams per step, the projections as M=16 skinny GEMMs on the matrix cores.
//
// The reference decodes one stream (qwen3/fast.py:146 asserts batch 1) with M=1 GEMVs (qwen3/kernels.py:143-310).
// With 16 streams the projections are dense [16 x K] x [K x N] contractions, so they go to
// v_mfma_f32_16x16x32_bf16: int8 weights are exact in bf16 (|q| <= 127 has 7 significant bits), and each
// activation is split into kTerms bf16 terms (x = t0 + t1 + ..., t_i = bf16 of what the earlier terms left), so
// the products are exact and the sum keeps fp32 input precision; one bf16 term alone loses ~1e-2 of relative
// accuracy over 28 layers.
//
// Data layout (all activations have 16 rows; rows of inactive streams stay zero):
//   * weights: int8 in 1 KiB tiles. Tile (g, c) holds rows 16g..16g+15, columns 64c..64c+63; lane L = n + 16 j of
//     a wave reads bytes [16 L, 16 L + 16) = W[16 g + n][64 c + 16 j .. + 16] with one 16-byte load, so a wave's
//     load is one contiguous KiB. Within a chunk the contraction index is permuted identically for both operands
//     (MFMA h = 0, 1 of the chunk takes bytes 8h..8h+7 of every lane), which leaves the dot product unchanged.
//   * GEMM inputs: bf16 planes [kTerms][16][K], row-major at the C interface; the planes that stay inside the batched
//     step are kept in the order in which the matrix cores take them (plane_index).
//   * RMSNorm: the kernel that updates the residual h also writes the planes of bf16(h ⊙ w_next) and, per
//     16-column tile, the partial sums of squares of h; the consuming GEMM adds the partials of its row in a fixed
//     order and applies rsqrt(Σh²/K + eps) after the dot product (qwen3/kernels.py:180-186, 224).
//
// Per layer: qkv GEMM -> ragged split-K attention -> o GEMM (+= h, norm planes) -> gate/up GEMM (SwiGLU planes)
// -> down GEMM (+= h, norm planes of the next layer). Then the head GEMM and a greedy pick that also embeds the
// chosen token for the next step. Every kernel is deterministic: fixed reduction orders, no float atomics.
#include "common.h"
#include "internal.h"

namespace {

typedef __attribute__((ext_vector_type(4))) uint32_t u32x4;

constexpr int kM = 16;         // rows of every activation buffer (streams)
#ifndef SK_BATCH_TERMS
#define SK_BATCH_TERMS 3
#endif
constexpr int kTerms = SK_BATCH_TERMS;
constexpr int kThreads = 256;
constexpr int kMaxSlices = 4;  // K slices of one GEMM (plan)
constexpr int kOutF32 = 0, kOutSwiglu = 1, kOutAcc = 2;

// ---- conversions ----------------------------------------------------------------------------------------------
// two floats whose low 16 bits are zero (small integers) -> packed bf16 pair, lo in the low half
__device__ __forceinline__ uint32_t pack_hi16(float lo, float hi) {
  return __builtin_amdgcn_perm(__float_as_uint(hi), __float_as_uint(lo), 0x07060302u);
}
// 8 int8 (two dwords) -> 8 bf16, exactly
__device__ __forceinline__ bf16x8 i8x8_bf16(uint32_t a, uint32_t b) {
  u32x4 r;
  r.x = pack_hi16((float)(int8_t)a, (float)(int8_t)(a >> 8));
  r.y = pack_hi16((float)(int8_t)(a >> 16), (float)(int8_t)(a >> 24));
  r.z = pack_hi16((float)(int8_t)b, (float)(int8_t)(b >> 8));
  r.w = pack_hi16((float)(int8_t)(b >> 16), (float)(int8_t)(b >> 24));
  return __builtin_bit_cast(bf16x8, r);
}
// v as kTerms bf16 terms written to planes [kTerms][plane] at index i
__device__ __forceinline__ void store_terms(bf16_t* __restrict__ planes, size_t plane, size_t i, float v) {
#pragma unroll
  for (int t = 0; t < kTerms; t++) {
    const bf16_t b = f2bf_hw(v);
    planes[t * plane + i] = b;
    v -= bf2f(b);
  }
}

// rotation (in fours) of staging segment s = 2 (j & 1) + h, s = 0..3
__device__ __forceinline__ int sq_rot(int s) { return 2 * ((s >> 1) & 1) + (s & 1); }

// Index of x[m][k] in a plane of K columns: row-major at the C interface; inside the batched step (TILED) in the order in
// which the matrix cores take it, 1 KiB per (64-wide chunk, half h): lane m + 16 j holds x[m][64 c + 16 j + 8 h .. + 8].
template <bool TILED>
__device__ __forceinline__ size_t plane_index(int m, int k, int K) {
  return TILED ? (size_t)((k >> 6) * 2 + ((k >> 3) & 1)) * 512 + (((k >> 4) & 3) * 16 + m) * 8 + (k & 7) : (size_t)m * K + k;
}

struct GemmArgs {
  const bf16_t* x;      // input planes [kTerms][16][K]
  const float* ssp;     // [np][16] partial sums of squares behind x (NULL: no RMSNorm scale)
  int np;
  float eps;
  const uint8_t* w;     // tiled int8 weights
  const uint16_t* s;    // [N] bf16 row scales
  int N, K;
  float* out;           // F32: [16][N]; ACC: residual [16][N], updated in place
  bf16_t* act;          // SWIGLU: planes [kTerms][16][N/2]
  bf16_t* xn;           // ACC: planes [kTerms][16][N] of bf16(h ⊙ nw)
  const float* nw;      // ACC: next RMSNorm weight [N]
  float* ssp_out;       // ACC: [N/16][16] partial sums of squares of the updated residual
  int S = 1;            // K slices (workgroups per row block)
  float* part = nullptr;          // S > 1: [S][N / 16][256] partial sums
  unsigned* counters = nullptr;   // S > 1: [row blocks] arrivals, zero between launches
};

// Workgroup (nb, slice) computes RG row groups (16 output rows each) for all 16 streams over K slice `slice`, which its
// kWaves waves split once more (wave w takes KW chunks of 64), each for all RG groups; the waves' sums meet once in LDS
// and are added in wave order. What bounds it is latency, not a rate: the launch (2.2-2.6 us measured with every load
// and MFMA taken out), then one memory round trip, since every load a wave will make goes out at the top: the weights
// (from HBM) first, then the activation planes (from L2). Weights first measured 5.7 against 6.2 us (qkv 4096 x 2048),
// 4.8 against 5.5 (o 2048 x 2048) and 5.8 against 7.1 (down 1024 x 3072) for chunk by chunk.
//   * Up to K = 2048 a workgroup takes all of K, so nothing is exchanged between workgroups. Splitting K over workgroups
//     for every shape (partial sums stored, acknowledged, counted and reloaded before the epilogue) took 9.2 / 7.5 /
//     16.6 us (qkv / o / gate-up 12288 x 2048) against 5.8 / 4.9 / 9.0 now.
//   * Beyond, reading all of the planes (96 K bytes) takes a CU longer than the exchange: K is cut into slices of 1536 or
//     2048, the workgroups of a row block publish their sums (device-coherent stores) and the last to arrive adds them
//     in slice order, so the result does not depend on arrival order. Down 2048 x 6144: 10.1 us with 12 slices of 512,
//     12.3 with the whole of K, 7.2 with 4 of 1536.
//   * TILED planes (plane_index) are loaded as whole fragments, 1 KiB per instruction. Row-major planes, the C
//     interface's, are loaded four lanes per row (64 contiguous bytes) and turned into fragments by a trip through 6 KB
//     of LDS that only this wave uses, so no barrier; the trip costs 1.4 us at K = 2048 (LDS bandwidth).
template <int OUT, bool TILED, int kWaves, int RG, int KW>
__global__ __launch_bounds__(64 * kWaves) void k_bgemm(GemmArgs p) {
  constexpr int kGemmThreads = 64 * kWaves;
  constexpr int kStrips = RG * 4, kOwn = (kStrips + kWaves - 1) / kWaves;  // 64-element output strips, per wave
  __shared__ uint4 stage[kWaves][TILED ? kStrips * 16 : kTerms * 128];  // [term][half][lane m + 16 j], one chunk per wave
  __shared__ int last_s;
  __shared__ float ssq[kGemmThreads / 16][kM];
  __shared__ float inv_s[kM];
  static_assert(kWaves * kStrips * 64 * 4 <= (int)sizeof(stage), "the waves' sums alias the staging area");
  float(*red)[kStrips][64] = (float(*)[kStrips][64])&stage[0][0];  // [wave][strip 4 r + i][lane]
  const int tid = threadIdx.x, wv = tid >> 6, lane = tid & 63;
  const int C = p.K / 64;                 // 64-wide chunks per row
  const int G = p.N / 16;                 // row groups
  const int g0 = blockIdx.x * RG;
  const size_t plane = (size_t)kM * p.K;
  const int slice = blockIdx.y;
  const int c0 = (slice * kWaves + wv) * KW;
  // activation loads: lane 4 m + s takes 16-byte segments s and 4 + s of row m's chunk, per term
  const bf16_t* xw = TILED ? p.x + (size_t)c0 * 1024 + lane * 8 : p.x + (size_t)(lane >> 2) * p.K + (size_t)c0 * 64 + 8 * (lane & 3);
  const uint4* wp[RG];
#pragma unroll
  for (int r = 0; r < RG; r++)  // a row group past the matrix loads the last one (never stored)
    wp[r] = (const uint4*)p.w + ((size_t)min(g0 + r, G - 1) * C + c0) * 64 + lane;
  uint4 wq[KW][RG], xq[KW][kTerms][2];
#pragma unroll
  for (int c = 0; c < KW; c++)
#pragma unroll
    for (int r = 0; r < RG; r++) wq[c][r] = ld_stream(wp[r] + c * 64);
  __builtin_amdgcn_sched_barrier(0);  // keep the weights ahead of the planes
#pragma unroll
  for (int c = 0; c < KW; c++)
#pragma unroll
    for (int t = 0; t < kTerms; t++)
#pragma unroll
      for (int i = 0; i < 2; i++) xq[c][t][i] = gload4((const uint4*)(xw + t * plane + (TILED ? 1024 * c + 512 * i : 64 * c + 32 * i)));
  float ssv = 0.f;  // this thread's share of the RMSNorm partial sums
  if (p.ssp)
    for (int q = tid >> 4; q < p.np; q += kGemmThreads / 16) ssv += gload(p.ssp + q * kM + (tid & 15));
  // what the epilogue needs of this thread's outputs
  const int nl = lane & 15;
  float sc[kOwn], hv[kOwn], nv[kOwn];
#pragma unroll
  for (int o = 0; o < kOwn; o++) {
    const int st = min(wv + o * kWaves, kStrips - 1), g = min(g0 + st / 4, G - 1), n = g * 16 + nl, m = 4 * (lane >> 4) + st % 4;
    sc[o] = bf2f(gload(p.s + n));
    if constexpr (OUT == kOutAcc) {
      hv[o] = gload(p.out + (size_t)m * p.N + n);
      nv[o] = gload(p.nw + n);
    }
  }
  f32x4 acc[RG], acc2[RG];  // first term, later terms (kept apart: the small terms accumulate at their own scale)
#pragma unroll
  for (int r = 0; r < RG; r++) { acc[r] = f32x4{0.f, 0.f, 0.f, 0.f}; acc2[r] = acc[r]; }
  uint4* my = &stage[wv][0];
  // segment q = 2 j + h of row m sits at slot 16 j + (m rotated by 4 (2 (j & 1) + h)) of half h: the 8 lanes of a
  // store beat and the 8 of a read beat each touch distinct bank groups
  const int sm = lane >> 2, sq = lane & 3, wslot = (sq & 1) * 64 + 16 * (sq >> 1) + ((sm + 4 * sq_rot(sq)) & 15);
  const int rj = lane >> 4, rs0 = 16 * rj + ((nl + 8 * (rj & 1)) & 15), rs1 = 64 + 16 * rj + ((nl + 8 * (rj & 1) + 4) & 15);
#pragma unroll
  for (int c = 0; c < KW; c++) {
    bf16x8 xa[kTerms][2];
    if constexpr (TILED) {
#pragma unroll
      for (int t = 0; t < kTerms; t++)
#pragma unroll
        for (int i = 0; i < 2; i++) xa[t][i] = as_bf16x8(xq[c][t][i]);
    } else {
#pragma unroll
      for (int t = 0; t < kTerms; t++)
#pragma unroll
        for (int i = 0; i < 2; i++) my[t * 128 + wslot + 32 * i] = xq[c][t][i];
      wave_sync();
#pragma unroll
      for (int t = 0; t < kTerms; t++) {
        xa[t][0] = as_bf16x8(my[t * 128 + rs0]);
        xa[t][1] = as_bf16x8(my[t * 128 + rs1]);
      }
      wave_sync();
    }
#pragma unroll
    for (int h = 0; h < 2; h++)
#pragma unroll
      for (int r = 0; r < RG; r++) {
        const uint4 q = wq[c][r];
        const bf16x8 b = h ? i8x8_bf16(q.z, q.w) : i8x8_bf16(q.x, q.y);
        acc[r] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(xa[0][h], b, acc[r], 0, 0, 0);
#pragma unroll
        for (int t = 1; t < kTerms; t++) acc2[r] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(xa[t][h], b, acc2[r], 0, 0, 0);
      }
  }
  if (p.ssp) ssq[tid >> 4][tid & 15] = ssv;
  __syncthreads();  // every wave is done with its staging area
  // D[m][n] sits in lane n + 16 (m / 4), element m % 4
#pragma unroll
  for (int r = 0; r < RG; r++)
#pragma unroll
    for (int i = 0; i < 4; i++) red[wv][4 * r + i][lane] = acc[r][i] + acc2[r][i];
  if (p.ssp && tid < kM) {
    float s = 0.f;
#pragma unroll
    for (int q = 0; q < kGemmThreads / 16; q++) s += ssq[q][tid];
    inv_s[tid] = rsqrtf(s / p.K + p.eps);
  }
  __syncthreads();
  float vs[kOwn];
#pragma unroll
  for (int o = 0; o < kOwn; o++) {
    const int st = min(wv + o * kWaves, kStrips - 1);
    vs[o] = red[0][st][lane];
#pragma unroll
    for (int w = 1; w < kWaves; w++) vs[o] += red[w][st][lane];
  }
  if (p.S > 1) {
    // partial of (slice, row group g): 256 floats, element i of lane L at 64 i + L
    const uint32_t stride = (uint32_t)G * 256u;
#pragma unroll
    for (int o = 0; o < kOwn; o++) {
      const int st = wv + o * kWaves;
      if (st < kStrips && g0 + st / 4 < G)
        buf_stf(p.part, ((uint32_t)slice * stride + (uint32_t)(g0 * 4 + st) * 64u + lane) * 4u, vs[o]);
    }
    __builtin_amdgcn_s_waitcnt(0);
    __syncthreads();
    if (tid == 0) {
      const unsigned prev = __hip_atomic_fetch_add(&p.counters[blockIdx.x], 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      last_s = prev == (unsigned)(p.S - 1);
    }
    __syncthreads();
    if (!last_s) return;
    // every slice's partial at once (one round trip), then the sum in slice order
    float pv[kMaxSlices][kOwn];
#pragma unroll
    for (int q = 0; q < kMaxSlices; q++)
      if (q < p.S)
#pragma unroll
        for (int o = 0; o < kOwn; o++) {
          const int st = min(wv + o * kWaves, kStrips - 1), g = min(g0 + st / 4, G - 1);
          pv[q][o] = buf_ldf(p.part, ((uint32_t)q * stride + (uint32_t)(g * 4 + st % 4) * 64u + lane) * 4u);
        }
#pragma unroll
    for (int o = 0; o < kOwn; o++) {
      vs[o] = pv[0][o];
#pragma unroll
      for (int q = 1; q < kMaxSlices; q++)
        if (q < p.S) vs[o] += pv[q][o];
    }
    if (tid == 0) __hip_atomic_store(&p.counters[blockIdx.x], 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  }
#pragma unroll
  for (int o = 0; o < kOwn; o++) {
    const int st = wv + o * kWaves;
    if (st >= kStrips || g0 + st / 4 >= G) break;
    const float v = vs[o];
    const int g = g0 + st / 4, n = g * 16 + nl, m = 4 * (lane >> 4) + st % 4;
    const float y = v * sc[o] * (p.ssp ? inv_s[m] : 1.f);
    if constexpr (OUT == kOutF32) {
      p.out[(size_t)m * p.N + n] = y;
    } else if constexpr (OUT == kOutSwiglu) {
      const float u = dpp<0xB1>(y);  // lane L ^ 1: the up row next to this gate row
      if (!(nl & 1)) store_terms(p.act, (size_t)kM * (p.N / 2), plane_index<TILED>(m, n / 2, p.N / 2), silu_mul(y, u));
    } else {
      const float hn = hv[o] + y;
      p.out[(size_t)m * p.N + n] = hn;
      store_terms(p.xn, (size_t)kM * p.N, plane_index<TILED>(m, n, p.N), hn * nv[o]);
      const float ss = row16_sum(hn * hn);
      if (nl == 0) p.ssp_out[g * kM + m] = ss;
    }
  }
}

// ---- weight tiling -----------------------------------------------------------------------------------------
__global__ void k_tile(const int8_t* __restrict__ w, int8_t* __restrict__ tiled, int N, int K) {
  // one thread per 16-byte lane slot: tile t = g * C + c, lane L = n + 16 j
  const size_t slot = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
  const int C = K / 64;
  if (slot >= (size_t)N * K / 16) return;
  const int L = (int)(slot & 63);
  const size_t t = slot >> 6;
  const int g = (int)(t / C), c = (int)(t % C);
  const int n = L & 15, j = L >> 4;
  const uint4 v = *(const uint4*)(w + (size_t)(16 * g + n) * K + 64 * c + 16 * j);
  *(uint4*)(tiled + slot * 16) = v;
}

// ---- ragged split-K decode attention -----------------------------------------------------------------------
// Block (stream b, kv head g, split s) covers positions [128 s, 128 s + 128) of stream b's cache up to its current
// position; the split that holds the position also normalises, rotates and appends this step's K and V. Each of its four
// waves takes 32 positions, all of whose K and V rows are loaded at the top, and works alone to its own maximum, sum and
// Σ p v; the four meet once in LDS. The block's partial (max, sum, Σ p v) goes to the workspace and a second launch
// (k_bmerge, one block per (b, g)) merges the splits in order and writes the attention output as bf16 term planes; a
// stream whose cache fits one split writes its output directly. The partials need no device-coherent stores and no
// arrival counter this way (the launch boundary orders them). Numerics as sk_attn (qwen3/kernels.py:338-414).
//   * Scores on the matrix cores: q of both heads is kept as kTerms bf16 terms in rows 4 head + term of the MFMA's A, so
//     the products are exact and a lane (16 head + position) finds its score's terms in its own registers: no sum over
//     lanes, and the softmax statistics are 16-lane DPP reductions of two values. Σ p v stays on the vector units (fp32
//     weights, 24 instructions per four rows), where a row of V is one contiguous load.
//   * What bounds it is the memory rate: with all arithmetic taken out it takes as long. Per call (with the merge) of 16
//     streams of 64..2048 positions, 82 MB: 27.4 us in two passes of 64 positions with the softmax statistics and the sums
//     over lanes shared by the block (ten barriers), 22.5 with waves alone, 20.1 (5.4 TB/s behind the launches) with
//     nontemporal loads, 19.8 for the loads alone; 133 MB 35.8 / 31.2 / 26.6. Five streams of 8..200: 10.0 -> 7.1, one
//     of 1500 11.5 -> 7.3, sixteen of 20..128 8.9 -> 7.0 (latency and the launches).
constexpr int kWavePos = 32;                       // positions of one wave
constexpr int kAttnChunk = kWavePos * 4;           // positions of a split where a cache has several (four waves)
constexpr int kAttnSplitMax = 32;  // max_len <= 4096
constexpr int kPart = SK_HD + 2;
constexpr float kInvSqrtHd = 0.08838834764831845f;

struct AttnArgs {
  const float* qkv;     // [16][(nq + 2 nkv) * 128]
  const float* qn;
  const float* kn;
  float eps;
  const float* rope;    // [max_len][cos 64 | sin 64]
  bf16_t* Kc;           // [batch][nkv][max_len][128]
  bf16_t* Vc;
  const int64_t* pos;   // [batch]
  int max_len, nq, nkv;
  bf16_t* att;          // planes [kTerms][16][nq * 128]
  float* part;          // [batch * nkv][2][kAttnSplitMax][kPart]
  int* err;
  bool tiled;           // layout of att (plane_index)
};
__device__ __forceinline__ size_t att_index(const AttnArgs& a, int b, int k) {
  return a.tiled ? plane_index<true>(b, k, a.nq * SK_HD) : plane_index<false>(b, k, a.nq * SK_HD);
}

template <int kWaves>
__global__ __launch_bounds__(SK_WAVE * kWaves) void k_battn(AttnArgs a) {
  constexpr int kChunk = kWavePos * kWaves;
  static_assert(kTerms <= 4, "a head's terms fill four rows of the MFMA");
  __shared__ __align__(16) bf16_t qt[8][SK_HD + 8];  // row 4 head + term
  __shared__ __align__(16) bf16_t ksh[SK_HD];        // this step's K and V rows as the cache holds them
  __shared__ __align__(16) bf16_t vsh[SK_HD];
  __shared__ float es[kWaves][kWavePos][2];          // softmax weights of a wave's positions, both heads
  __shared__ __align__(16) float op[kWaves][2][SK_HD];
  __shared__ float ml[kWaves][2][2];
  const int bg = blockIdx.x, b = bg / a.nkv, kvh = bg % a.nkv, split = blockIdx.y;
  const int t = threadIdx.x, p = (t >> 7) & 1, d = t & (SK_HD - 1), w = __builtin_amdgcn_readfirstlane(t >> 6), lane = t & 63, gq = lane >> 4, sl = lane & 15;
  const int qs = (a.nq + 2 * a.nkv) * SK_HD;
  const int64_t pos64 = a.pos[b];
  const size_t ap = (size_t)kM * a.nq * SK_HD;
  if (pos64 < 0 || pos64 >= a.max_len) {  // a stream past its cache: zero output, error word set
    if (split == 0 && t < 2 * SK_HD) {
      store_terms(a.att, ap, att_index(a, b, (2 * kvh + p) * SK_HD + d), 0.f);
      if (t == 0) atomicCAS(a.err, 0, 5);
    }
    return;
  }
  const int pos = (int)pos64, T = pos + 1, ns = (T + kChunk - 1) / kChunk;
  if (split >= ns) return;
  const int t0 = split * kChunk, n = min(kChunk, T - t0);
  const bool has_pos = split == ns - 1;  // only this split can have fewer than kChunk positions
  bf16_t* Kh = a.Kc + ((size_t)b * a.nkv + kvh) * a.max_len * SK_HD;
  bf16_t* Vh = a.Vc + ((size_t)b * a.nkv + kvh) * a.max_len * SK_HD;
  // this step's inputs first (the wait for them must not also wait for the cache rows): wave 0 q of head 2 g, wave 1 q of
  // head 2 g + 1, wave 2 k, wave 3 v, dims lane and lane + 64 per lane
  const int wq = w & 3;
  const float* src = a.qkv + (size_t)b * qs + (wq < 2 ? (2 * kvh + wq) * SK_HD : a.nq * SK_HD + ((wq - 2) * a.nkv + kvh) * SK_HD);
  const float* nw = wq < 2 ? a.qn : a.kn;
  const float* rp = a.rope + (size_t)pos * SK_HD;
  const float x0 = gload(src + lane), x1 = gload(src + lane + 64), n0 = gload(nw + lane), n1 = gload(nw + lane + 64);
  const float cs = gload(rp + lane), sn = gload(rp + lane + 64);
  __builtin_amdgcn_sched_barrier(0);
  // every cache row of the wave: lane (gq, sl) holds K of positions 16 i + sl, dims 32 c + 8 gq .. + 8 (the MFMA's B), and V
  // of positions 4 i + gq, dims 8 sl .. + 8. Rows past the split's range read row t0 instead.
  uint4 kr[2][4], vr[8];
#pragma unroll
  for (int i = 0; i < 2; i++) {
    const int jj = kWavePos * w + 16 * i + sl, row = jj < n ? t0 + jj : t0;
#pragma unroll
    for (int c = 0; c < 4; c++) kr[i][c] = ld_stream((const uint4*)(Kh + (uint32_t)(row * SK_HD + 32 * c + 8 * gq)));
  }
#pragma unroll
  for (int i = 0; i < 8; i++) {
    const int jj = kWavePos * w + 4 * i + gq, row = jj < n ? t0 + jj : t0;
    vr[i] = ld_stream((const uint4*)(Vh + (uint32_t)(row * SK_HD + 8 * sl)));
  }
  __builtin_amdgcn_sched_barrier(0);
  if (w < 3) {  // per-head RMSNorm, RoPE
    const float inv = rsqrtf(wave_sum(x0 * x0 + x1 * x1) / SK_HD + a.eps);
    const float y0 = x0 * inv * n0, y1 = x1 * inv * n1;
    const float r0 = y0 * cs + -y1 * sn, r1 = y1 * cs + y0 * sn;
    if (w < 2) {
      store_terms(&qt[4 * w][0], SK_HD + 8, lane, r0 * kInvSqrtHd);
      store_terms(&qt[4 * w][0], SK_HD + 8, lane + 64, r1 * kInvSqrtHd);
    } else if (has_pos) {
      const bf16_t k0 = f2bf(r0), k1 = f2bf(r1);
      ksh[lane] = k0;
      ksh[lane + 64] = k1;
      Kh[(size_t)pos * SK_HD + lane] = k0;
      Kh[(size_t)pos * SK_HD + lane + 64] = k1;
    }
  } else if (w == 3 && has_pos) {
    const bf16_t v0 = f2bf(x0), v1 = f2bf(x1);
    vsh[lane] = v0;
    vsh[lane + 64] = v1;
    Vh[(size_t)pos * SK_HD + lane] = v0;
    Vh[(size_t)pos * SK_HD + lane + 64] = v1;
  }
  __syncthreads();
  if (has_pos) {  // the row at pos from LDS; zero V past it (its weight is zero, the memory may hold anything)
#pragma unroll
    for (int i = 0; i < 2; i++)
      if (t0 + kWavePos * w + 16 * i + sl == pos)
#pragma unroll
        for (int c = 0; c < 4; c++) kr[i][c] = *(const uint4*)&ksh[32 * c + 8 * gq];
#pragma unroll
    for (int i = 0; i < 8; i++) {
      const int jj = kWavePos * w + 4 * i + gq;
      if (t0 + jj == pos) vr[i] = *(const uint4*)&vsh[8 * sl];
      else if (jj >= n) vr[i] = make_uint4(0, 0, 0, 0);
    }
  }
  const bool used = sl < 8 && (sl & 3) < kTerms;
  bf16x8 qa[4];
#pragma unroll
  for (int c = 0; c < 4; c++) {
    const uint4 v = *(const uint4*)&qt[4 * ((sl >> 2) & 1) + min(sl & 3, kTerms - 1)][32 * c + 8 * gq];
    qa[c] = as_bf16x8(used ? v : make_uint4(0, 0, 0, 0));
  }
  // scores: lane 16 head + sl (the lower half of the wave) holds positions sl and 16 + sl
  float sv[2], e[2];
#pragma unroll
  for (int i = 0; i < 2; i++) {
    f32x4 acc = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int c = 0; c < 4; c++) acc = __builtin_amdgcn_mfma_f32_16x16x32_bf16(qa[c], as_bf16x8(kr[i][c]), acc, 0, 0, 0);
    float s = acc[kTerms - 1];
#pragma unroll
    for (int q = kTerms - 2; q >= 0; q--) s += acc[q];
    sv[i] = kWavePos * w + 16 * i + sl < n ? s : -INFINITY;
  }
  const float mw = row16_max(fmaxf(sv[0], sv[1]));
#pragma unroll
  for (int i = 0; i < 2; i++) e[i] = kWavePos * w + 16 * i + sl < n ? expf(sv[i] - mw) : 0.f;
  const float lw = row16_sum(e[0] + e[1]);
  if (gq < 2) {
    es[w][sl][gq] = e[0];
    es[w][16 + sl][gq] = e[1];
    if (sl == 0) {
      ml[w][gq][0] = mw;
      ml[w][gq][1] = lw;
    }
  }
  wave_sync();
  float a0[8], a1[8];
#pragma unroll
  for (int k = 0; k < 8; k++) { a0[k] = 0.f; a1[k] = 0.f; }
#pragma unroll
  for (int i = 0; i < 8; i++) {
    const float2 ew = *(const float2*)&es[w][4 * i + gq][0];
    float v8[8];
    unpack_bf8(vr[i], v8);
#pragma unroll
    for (int k = 0; k < 8; k++) { a0[k] = __builtin_fmaf(ew.x, v8[k], a0[k]); a1[k] = __builtin_fmaf(ew.y, v8[k], a1[k]); }
  }
  *(float4*)&op[w][gq >> 1][8 * sl + 4 * (gq & 1)] = rows_sum(a0, a1);
  __syncthreads();
  if (t >= 2 * SK_HD) return;
  // the waves' partials of head p, dim d
  float m = ml[0][p][0], l = 0.f, o = 0.f;
#pragma unroll
  for (int q = 1; q < kWaves; q++) m = fmaxf(m, ml[q][p][0]);
#pragma unroll
  for (int q = 0; q < kWaves; q++) {
    const float f = ml[q][p][0] == -INFINITY ? 0.f : expf(ml[q][p][0] - m);
    l = __builtin_fmaf(f, ml[q][p][1], l);
    o = __builtin_fmaf(f, op[q][p][d], o);
  }

  if (ns == 1) {  // the whole cache in this block: the output directly, nothing to merge
    store_terms(a.att, ap, att_index(a, b, (2 * kvh + p) * SK_HD + d), l > 0.f ? o / l : 0.f);
    return;
  }
  // publish the partial for k_bmerge
  float* pp = a.part + ((bg * 2 + p) * kAttnSplitMax + split) * kPart;  // plain stores: k_bmerge is another launch
  if (d == 0) { pp[0] = m; pp[1] = l; }
  pp[2 + d] = o;
}

// Block (stream b, kv head g): the log-sum-exp merge of k_battn's partials of (b, g) (thread (p, d): q head 2 g + p, dim
// d), written as bf16 term planes. Streams past their cache and streams of one split were handled by k_battn. Bound by
// the launch and one memory round trip: the partials of every split that the cache could have are loaded together with
// the position, those past it are not used, and one wave finds the splits' weights for all.
__global__ __launch_bounds__(kThreads) void k_bmerge(AttnArgs a) {
  static_assert(2 * kAttnSplitMax == SK_WAVE, "one lane per head and split");
  __shared__ __align__(16) float fs[2][kAttnSplitMax];  // a split's weight, negative where it has none
  __shared__ float ls[2];
  const int bg = blockIdx.x, b = bg / a.nkv, kvh = bg % a.nkv;
  const int t = threadIdx.x, p = t >> 7, d = t & (SK_HD - 1);
  const int nmax = (a.max_len + kAttnChunk - 1) / kAttnChunk;  // at most kAttnSplitMax
  const int cc = t % kAttnSplitMax;
  const float2 st = *(const float2*)(a.part + (bg * 2 * kAttnSplitMax + t % SK_WAVE) * kPart);
  float oc[kAttnSplitMax];
  const float* po = a.part + (bg * 2 + p) * kAttnSplitMax * kPart + 2 + d;
#pragma unroll
  for (int k0 = 0; k0 < kAttnSplitMax; k0 += 8)
    if (k0 < nmax)
#pragma unroll
      for (int k = k0; k < k0 + 8; k++) oc[k] = gload(po + k * kPart);
  const int64_t pos64 = a.pos[b];
  if (pos64 < 0 || pos64 >= a.max_len) return;
  const int ns = ((int)pos64 + kAttnChunk) / kAttnChunk;
  if (ns == 1) return;
  if (t < SK_WAVE) {  // lane 32 head + split
    const float m = cc < ns ? st.x : -INFINITY;
    const float r = row16_max(m);
    const float ma = fmaxf(lane_value(r, 0), lane_value(r, 16));
    const float mb = fmaxf(lane_value(r, 32), lane_value(r, 48));
    const bool has = cc < ns && m != -INFINITY;
    const float f = has ? expf(m - (t < kAttnSplitMax ? ma : mb)) : -1.f;
    fs[t / kAttnSplitMax][cc] = f;
    const float q = row16_sum(has ? f * st.y : 0.f);
    const float la = lane_value(q, 0) + lane_value(q, 16);
    const float lb = lane_value(q, 32) + lane_value(q, 48);
    if (t < 2) ls[t] = t ? lb : la;
  }
  __syncthreads();
  const float L = ls[p];
  float O = 0.f;
#pragma unroll
  for (int k0 = 0; k0 < kAttnSplitMax; k0 += 8) {
    if (k0 >= ns) break;
#pragma unroll
    for (int k = k0; k < k0 + 8; k++) {
      const float f = fs[p][k], x = __builtin_fmaf(f, oc[k], O);
      O = f < 0.f ? O : x;
    }
  }
  const size_t ap = (size_t)kM * a.nq * SK_HD;
  store_terms(a.att, ap, att_index(a, b, (2 * kvh + p) * SK_HD + d), L > 0.f ? O / L : 0.f);
}

// ---- greedy pick + embedding of the next input ---------------------------------------------------------------
// Block b: argmax of logits row b (largest value, lowest index on ties, NaN never wins; qwen3/sampler.py:114-149)
// when pick != 0, else the stored id; then h[b] = emb[id] (bf16 -> fp32), the input planes of bf16(h ⊙ nw0) and
// the row's sum of squares (one partial) for the first layer's RMSNorm.
struct PickArgs {
  const float* logits;  // [16][V]
  int V, H, pick, max_frames;
  int64_t* ids;         // [batch]
  int64_t* pos;         // [batch]
  int64_t* codes;       // [max_frames][16]
  int64_t* nstep;       // [batch]
  const bf16_t* emb;    // [V][H]
  const float* nw0;     // [H]
  float* h;             // [16][H]
  bf16_t* xa;           // planes [kTerms][16][H]
  float* ssa;           // [1][16]
  int* err;
};

// Bound by the launch and two dependent memory round trips (the logits, then the embedding row of the pick): 1024 threads
// with four logits each in flight and the largest found by DPP maxima: 10.9 -> 4.3 us per step of 16 streams (V 3072, H 2048)
// against 256 threads that took twelve logits one after the other and met in eight LDS steps.
constexpr int kPickThreads = 1024, kPickPer = 4;
__global__ __launch_bounds__(kPickThreads) void k_bpick(PickArgs a) {
  constexpr int kWaves = kPickThreads / SK_WAVE;
  static_assert(kWaves == 16, "one wave's result per lane of a row");
  __shared__ uint32_t wkey[kWaves], widx[kWaves];
  __shared__ float red[kWaves];
  const int b = blockIdx.x, t = threadIdx.x, lane = t & 63, w = t >> 6;
  int id;
  if (a.pick) {
    const float* lg = a.logits + (size_t)b * a.V;
    const int64_t f = a.nstep[b], pos = a.pos[b];
    uint32_t best = 0, bi = 0xffffffffu;  // key 0 is below every value's
    for (int k0 = 0; k0 < a.V; k0 += kPickThreads * kPickPer) {
      float v[kPickPer];
#pragma unroll
      for (int j = 0; j < kPickPer; j++) v[j] = gload(lg + min(k0 + j * kPickThreads + t, a.V - 1));
#pragma unroll
      for (int j = 0; j < kPickPer; j++) {
        const int k = k0 + j * kPickThreads + t;
        const uint32_t key = k < a.V && v[j] == v[j] ? order_key(v[j] == 0.f ? 0.f : v[j]) : 0u;  // -0 equals +0, NaN never wins
        if (key > best) { best = key; bi = (uint32_t)k; }
      }
    }
    const uint32_t top = wave_umax(best);
    const uint32_t ti = ~wave_umax(best == top ? ~bi : 0u);
    if (lane == 0) { wkey[w] = top; widx[w] = ti; }
    __syncthreads();
    const uint32_t k2 = wkey[lane & 15], tk = wave_umax(k2);  // every wave finds the pick
    const uint32_t pick = ~wave_umax(k2 == tk ? ~widx[lane & 15] : 0u);
    id = pick >= (uint32_t)a.V ? 0 : (int)pick;
    if (t == 0) {
      a.ids[b] = id;
      if (f >= 0 && f < a.max_frames) a.codes[f * kM + b] = id;
      else atomicCAS(a.err, 0, 6);
      a.nstep[b] = f + 1;
      a.pos[b] = pos + 1;
    }
  } else {
    const int64_t i = a.ids[b];
    if (t == 0 && (i < 0 || i >= a.V)) atomicCAS(a.err, 0, 5);
    id = i < 0 || i >= a.V ? 0 : (int)i;
  }
  const bf16_t* row = a.emb + (size_t)id * a.H;
  float ss = 0.f;
  for (int k0 = 0; k0 < a.H; k0 += 2 * kPickThreads) {
    float v[2], nv[2];
#pragma unroll
    for (int j = 0; j < 2; j++) {
      const int k = min(k0 + j * kPickThreads + t, a.H - 1);
      v[j] = bf2f(gload(row + k));
      nv[j] = gload(a.nw0 + k);
    }
#pragma unroll
    for (int j = 0; j < 2; j++) {
      const int k = k0 + j * kPickThreads + t;
      if (k >= a.H) break;
      a.h[(size_t)b * a.H + k] = v[j];
      store_terms(a.xa, (size_t)kM * a.H, plane_index<true>(b, k, a.H), v[j] * nv[j]);
      ss = __builtin_fmaf(v[j], v[j], ss);
    }
  }
  ss = wave_sum(ss);
  if (lane == 0) red[w] = ss;
  __syncthreads();
  const float tot = row16_sum(red[lane & 15]);
  if (t == 0) a.ssa[b] = tot;
}

// ---- dispatch ------------------------------------------------------------------------------------------------
// Launch plan: S slices of K (one up to K = 2048, else slices of 1536 or 2048), RG row groups per workgroup (as many as
// keep the grid near one workgroup per CU, up to 3), NW waves. Best of a sweep over 4, 8 and 16 waves, 1 to 6 groups and
// 1 to 12 slices on the 1.7B and 0.6B shapes; what the rule's neighbours took, in us: qkv 4096 x 2048 5.8 (2 groups 6.7,
// 2 slices 7.0), o 2048 x 2048 4.9 (2 slices 5.5), gate/up 12288 x 2048 9.0 with 16 waves and 3 groups (8 waves 10.0, 4
// groups 9.9), down 2048 x 6144 7.2 (3 slices 7.8, 6 slices 8.0), gate/up 6144 x 1024 5.2 (1 group 6.0, 3 groups 5.8),
// down 1024 x 3072 5.7 (6 slices and 2 groups 5.4).
struct Plan {
  int S, RG, NW;
};
Plan plan(int N, int K, bool tiled) {
  Plan pl;
  pl.S = K <= 2048 ? 1 : K % 2048 == 0 && K % 1536 != 0 ? K / 2048 : K / 1536;
  const int g = N / 16 * pl.S;
  pl.RG = g <= 256 ? 1 : g <= 512 ? 2 : 3;
  // 16 waves halve what each of three row groups' waves waits for; row-major planes would need 96 KB of LDS
  pl.NW = tiled && pl.RG == 3 && K / pl.S % 1024 == 0 ? 16 : 8;
  return pl;
}
int64_t part_floats(int N, int K) {
  const int S = plan(N, K, true).S;
  return S > 1 ? (int64_t)S * (N / 16) * 256 : 0;
}
template <int OUT, bool TILED, int NW, int RG, int KW>
void launch_one(const GemmArgs& p, hipStream_t st) {
  hipLaunchKernelGGL((k_bgemm<OUT, TILED, NW, RG, KW>), dim3((p.N / 16 + RG - 1) / RG, p.S), dim3(64 * NW), 0, st, p);
}
template <int OUT, bool TILED, int RG>
hipError_t launch_kw(const GemmArgs& p, int NW, hipStream_t st) {
  const int C = p.K / p.S / 64;  // chunks of a slice
  if constexpr (TILED && RG == 3) {
    if (NW == 16) {
      if (C == 16) launch_one<OUT, TILED, 16, RG, 1>(p, st);
      else launch_one<OUT, TILED, 16, RG, 2>(p, st);
      return hipGetLastError();
    }
  }
  switch (C) {
    case 8: launch_one<OUT, TILED, 8, RG, 1>(p, st); break;
    case 16: launch_one<OUT, TILED, 8, RG, 2>(p, st); break;
    case 24: launch_one<OUT, TILED, 8, RG, 3>(p, st); break;
    case 32: launch_one<OUT, TILED, 8, RG, 4>(p, st); break;
    default: return hipErrorInvalidValue;
  }
  return hipGetLastError();
}
template <int OUT, bool TILED>
hipError_t launch_rg(const GemmArgs& p, const Plan& pl, hipStream_t st) {
  switch (pl.RG) {
    case 1: return launch_kw<OUT, TILED, 1>(p, pl.NW, st);
    case 2: return launch_kw<OUT, TILED, 2>(p, pl.NW, st);
    default: return launch_kw<OUT, TILED, 3>(p, pl.NW, st);
  }
}
bool k_supported(int K) { return K == 512 || K == 1024 || K == 2048 || K == 3072 || K == 4096 || K == 6144; }

template <bool TILED>
hipError_t launch_gemm(GemmArgs p, int mode, hipStream_t st) {
  const Plan pl = plan(p.N, p.K, TILED);
  p.S = pl.S;
  switch (mode) {
    case kOutF32: return launch_rg<kOutF32, TILED>(p, pl, st);
    case kOutSwiglu: return launch_rg<kOutSwiglu, TILED>(p, pl, st);
    default: return launch_rg<kOutAcc, TILED>(p, pl, st);
  }
}

// The attention of the batch: one block per stream and head that holds the whole cache up to 256 positions (eight waves,
// four up to 128), else splits of 128 positions and the merge. Five streams in caches of 205: 6.9 us per call with two
// splits, 6.5 in one block without the merge's launch; one block of sixteen waves up to 512 positions took 12.3 against 9.8 with
// splits (sixteen streams), since one CU then loads what four had.
hipError_t launch_attn(const AttnArgs& a, int batch, hipStream_t st) {
  const int bh = batch * a.nkv;
  if (a.max_len <= kWavePos * 4) {
    hipLaunchKernelGGL(k_battn<4>, dim3(bh), dim3(SK_WAVE * 4), 0, st, a);
  } else if (a.max_len <= kWavePos * 8) {
    hipLaunchKernelGGL(k_battn<8>, dim3(bh), dim3(SK_WAVE * 8), 0, st, a);
  } else {
    hipLaunchKernelGGL(k_battn<4>, dim3(bh, (a.max_len + kAttnChunk - 1) / kAttnChunk), dim3(SK_WAVE * 4), 0, st, a);
    const hipError_t e = hipGetLastError();
    if (e != hipSuccess) return e;
    hipLaunchKernelGGL(k_bmerge, dim3(bh), dim3(kThreads), 0, st, a);
  }
  return hipGetLastError();
}

int check_gemm(const GemmArgs& p, int mode) {
  if (!p.x || !p.w || !p.s || (!p.out && mode != kOutSwiglu)) return SK_EINVAL;
  if (p.N <= 0 || p.N % 16 || !k_supported(p.K)) return SK_EINVAL;
  if (p.ssp && p.np < 1) return SK_EINVAL;
  if (mode == kOutSwiglu && (!p.act || p.N % 32)) return SK_EINVAL;
  if (mode == kOutAcc && (!p.xn || !p.nw || !p.ssp_out)) return SK_EINVAL;
  if (mode < 0 || mode > kOutAcc) return SK_EINVAL;
  if (!SK_ALIGNED16(p.x) || !SK_ALIGNED16(p.w)) return SK_EINVAL;
  return SK_OK;
}

// workspace layout
struct Ws {
  int64_t err, h, xa, xb, ssa, ssb, qkv, att, act, logits, part, gpart, gctr, total;
};
int64_t up256(int64_t v) { return (v + 255) / 256 * 256; }
Ws ws_layout(int H, int I, int nq, int nkv, int V) {
  Ws w;
  int64_t o = 0;
  auto take = [&](int64_t bytes) { const int64_t at = o; o += up256(bytes); return at; };
  w.err = take(256);
  w.h = take((int64_t)kM * H * 4);
  w.xa = take((int64_t)kTerms * kM * H * 2);
  w.xb = take((int64_t)kTerms * kM * H * 2);
  w.ssa = take((int64_t)(H / 16) * kM * 4);
  w.ssb = take((int64_t)(H / 16) * kM * 4);
  w.qkv = take((int64_t)kM * (nq + 2 * nkv) * SK_HD * 4);
  w.att = take((int64_t)kTerms * kM * nq * SK_HD * 2);
  w.act = take((int64_t)kTerms * kM * I * 2);
  w.logits = take((int64_t)kM * V * 4);
  w.part = take((int64_t)kM * nkv * 2 * kAttnSplitMax * kPart * 4);
  const int nqkv = (nq + 2 * nkv) * SK_HD;
  int64_t pf = 0, nmax = 0;
  const int shapes[5][2] = {{nqkv, H}, {H, nq * SK_HD}, {2 * I, H}, {H, I}, {V, H}};
  for (const auto& sh : shapes) {
    pf = pf > part_floats(sh[0], sh[1]) ? pf : part_floats(sh[0], sh[1]);
    nmax = nmax > sh[0] ? nmax : sh[0];
  }
  w.gpart = take(pf * 4);
  w.gctr = take(nmax / 16 * 4);
  w.total = o;
  return w;
}

}  // namespace

extern "C" int sk_tile_weights(const void* w, void* tiled, int N, int K, void* stream) {
  if (!w || !tiled || N <= 0 || K <= 0 || N % 16 || K % 64) return sk_set_error(SK_EINVAL, "sk_tile_weights: bad arguments");
  if (!SK_ALIGNED16(w) || !SK_ALIGNED16(tiled)) return sk_set_error(SK_EINVAL, "sk_tile_weights: pointers must be 16-byte aligned");
  const size_t slots = (size_t)N * K / 16;
  hipLaunchKernelGGL(k_tile, dim3((unsigned)((slots + 255) / 256)), dim3(256), 0, (hipStream_t)stream,
                     (const int8_t*)w, (int8_t*)tiled, N, K);
  return sk_check_launch(hipGetLastError(), "sk_tile_weights");
}

extern "C" int64_t sk_bgemm_workspace_size(int N, int K) {
  if (N <= 0 || N % 16 || !k_supported(K)) return 0;
  return up256(part_floats(N, K) * 4) + up256((int64_t)N / 16 * 4);
}

extern "C" int sk_bgemm(const void* x, const float* ssp, int np, float eps, const void* w_tiled, const uint16_t* s, int N,
                        int K, int mode, float* out, void* act, void* xn, const float* nw, float* ssp_out,
                        void* workspace, int64_t workspace_bytes, void* stream) {
  GemmArgs p{(const bf16_t*)x, ssp, np, eps, (const uint8_t*)w_tiled, s, N, K, out, (bf16_t*)act, (bf16_t*)xn, nw, ssp_out};
  if (check_gemm(p, mode)) return sk_set_error(SK_EINVAL, "sk_bgemm: bad shape, mode or pointer");
  if (!workspace || !SK_ALIGNED16(workspace)) return sk_set_error(SK_EINVAL, "sk_bgemm: workspace must be 16-byte aligned");
  if (workspace_bytes < sk_bgemm_workspace_size(N, K)) return sk_set_error(SK_EWORKSPACE, "sk_bgemm: workspace too small");
  p.part = (float*)workspace;
  p.counters = (unsigned*)((char*)workspace + up256(part_floats(N, K) * 4));
  return sk_check_launch(launch_gemm<false>(p, mode, (hipStream_t)stream), "sk_bgemm");
}

extern "C" int sk_batch_terms(void) { return kTerms; }

extern "C" int64_t sk_batch_workspace_size(int hidden, int inter, int nq, int nkv, int vocab) {
  if (hidden <= 0 || inter <= 0 || nq <= 0 || nkv <= 0 || vocab <= 0) return 0;
  return ws_layout(hidden, inter, nq, nkv, vocab).total;
}

namespace {
int check_batch(const sk_batch_desc* d) {
  if (!d) return sk_set_error(SK_EINVAL, "sk_batch: null descriptor");
  const int H = d->hidden, I = d->inter;
  if (d->batch < 1 || d->batch > kM) return sk_set_error(SK_EINVAL, "sk_batch: batch must be 1..16");
  if (d->nkv <= 0 || d->nq != 2 * d->nkv) return sk_set_error(SK_EINVAL, "sk_batch: needs nq == 2 nkv (head_dim 128)");
  if (!k_supported(H) || !k_supported(I) || !k_supported(d->nq * SK_HD) || H % 16)
    return sk_set_error(SK_EINVAL, "sk_batch: hidden / inter / nq*128 must be 512, 1024, 2048, 3072, 4096 or 6144");
  if (d->vocab <= 0 || d->vocab % 16) return sk_set_error(SK_EINVAL, "sk_batch: vocab must be a positive multiple of 16");
  if (d->max_len <= 0 || d->max_len > kAttnChunk * kAttnSplitMax) return sk_set_error(SK_EINVAL, "sk_batch: max_len must be 1..4096");
  if (d->n_layers <= 0 || !d->layers || !d->norm || !d->head_w || !d->head_s || !d->emb || !d->rope || !d->ids || !d->pos ||
      !d->codes || !d->nstep || d->max_frames <= 0 || !d->workspace)
    return sk_set_error(SK_EINVAL, "sk_batch: null pointer or bad count");
  if (!SK_ALIGNED16(d->workspace)) return sk_set_error(SK_EINVAL, "sk_batch: workspace must be 16-byte aligned");
  if (d->workspace_bytes < sk_batch_workspace_size(H, I, d->nq, d->nkv, d->vocab))
    return sk_set_error(SK_EWORKSPACE, "sk_batch: workspace too small");
  for (int l = 0; l < d->n_layers; l++) {
    const sk_layer_desc& L = d->layers[l];
    if (!L.qkv_w || !L.qkv_s || !L.o_w || !L.o_s || !L.gu_w || !L.gu_s || !L.down_w || !L.down_s || !L.in_norm ||
        !L.post_norm || !L.qn || !L.kn || !L.kc || !L.vc)
      return sk_set_error(SK_EINVAL, "sk_batch: null pointer in a layer descriptor");
    if (!SK_ALIGNED16(L.kc) || !SK_ALIGNED16(L.vc)) return sk_set_error(SK_EINVAL, "sk_batch: caches must be 16-byte aligned");
  }
  return SK_OK;
}

hipError_t embed_launch(const sk_batch_desc* d, int pick, const float* logits, hipStream_t st) {
  char* ws = (char*)d->workspace;
  const Ws w = ws_layout(d->hidden, d->inter, d->nq, d->nkv, d->vocab);
  PickArgs a{logits, d->vocab, d->hidden, pick, d->max_frames, d->ids, d->pos, d->codes, d->nstep,
             (const bf16_t*)d->emb, d->layers[0].in_norm, (float*)(ws + w.h), (bf16_t*)(ws + w.xa), (float*)(ws + w.ssa),
             (int*)(ws + w.err)};
  hipLaunchKernelGGL(k_bpick, dim3(d->batch), dim3(kPickThreads), 0, st, a);
  return hipGetLastError();
}
}  // namespace

extern "C" int64_t sk_batch_attn_workspace_size(int nkv) {
  if (nkv <= 0) return 0;
  return up256(256) + up256((int64_t)kM * nkv * 2 * kAttnSplitMax * kPart * 4);
}

extern "C" int sk_batch_attn(const float* qkv, const float* qn, const float* kn, float eps, const float* rope, void* Kc,
                             void* Vc, const int64_t* pos, int batch, int max_len, int nq, int nkv, void* att,
                             void* workspace, int64_t workspace_bytes, void* stream) {
  if (!qkv || !qn || !kn || !rope || !Kc || !Vc || !pos || !att || !workspace)
    return sk_set_error(SK_EINVAL, "sk_batch_attn: null pointer");
  if (batch < 1 || batch > kM || nkv <= 0 || nq != 2 * nkv || max_len <= 0 || max_len > kAttnChunk * kAttnSplitMax)
    return sk_set_error(SK_EINVAL, "sk_batch_attn: needs batch 1..16, nq == 2 nkv, max_len 1..4096");
  if (!SK_ALIGNED16(Kc) || !SK_ALIGNED16(Vc) || !SK_ALIGNED16(workspace))
    return sk_set_error(SK_EINVAL, "sk_batch_attn: caches and workspace must be 16-byte aligned");
  if (workspace_bytes < sk_batch_attn_workspace_size(nkv)) return sk_set_error(SK_EWORKSPACE, "sk_batch_attn: workspace too small");
  char* ws = (char*)workspace;
  const int64_t part = up256(256);
  AttnArgs at{qkv, qn, kn, eps, rope, (bf16_t*)Kc, (bf16_t*)Vc, pos, max_len, nq, nkv, (bf16_t*)att,
              (float*)(ws + part), (int*)ws, false};
  return sk_check_launch(launch_attn(at, batch, (hipStream_t)stream), "sk_batch_attn");
}

extern "C" int sk_batch_embed(const sk_batch_desc* d, void* stream) {
  int rc = check_batch(d);
  if (rc) return rc;
  return sk_check_launch(embed_launch(d, 0, nullptr, (hipStream_t)stream), "sk_batch_embed");
}

extern "C" int sk_batch_frame(const sk_batch_desc* d, void* stream) {
  int rc = check_batch(d);
  if (rc) return rc;
  hipStream_t st = (hipStream_t)stream;
  char* ws = (char*)d->workspace;
  const int H = d->hidden, I = d->inter, nq = d->nq, nkv = d->nkv, V = d->vocab;
  const Ws w = ws_layout(H, I, nq, nkv, V);
  float* h = (float*)(ws + w.h);
  bf16_t* xa = (bf16_t*)(ws + w.xa);
  bf16_t* xb = (bf16_t*)(ws + w.xb);
  float* ssa = (float*)(ws + w.ssa);
  float* ssb = (float*)(ws + w.ssb);
  float* qkv = (float*)(ws + w.qkv);
  bf16_t* att = (bf16_t*)(ws + w.att);
  bf16_t* act = (bf16_t*)(ws + w.act);
  float* logits = d->logits ? d->logits : (float*)(ws + w.logits);  // the caller's buffer directly: no copy behind the head
  const int nqkv = (nq + 2 * nkv) * SK_HD;
  float* gpart = (float*)(ws + w.gpart);
  unsigned* gctr = (unsigned*)(ws + w.gctr);
  hipError_t e = hipSuccess;
  for (int l = 0; l < d->n_layers && e == hipSuccess; l++) {
    const sk_layer_desc& L = d->layers[l];
    const int np_a = l == 0 ? 1 : H / 16;
    GemmArgs g1{xa, ssa, np_a, d->eps, (const uint8_t*)L.qkv_w, L.qkv_s, nqkv, H, qkv, nullptr, nullptr, nullptr, nullptr,
                1, gpart, gctr};
    e = launch_gemm<true>(g1, kOutF32, st);
    if (e != hipSuccess) break;
    AttnArgs at{qkv, L.qn, L.kn, d->eps, d->rope, (bf16_t*)L.kc, (bf16_t*)L.vc, d->pos, d->max_len, nq, nkv, att,
                (float*)(ws + w.part), (int*)(ws + w.err), true};
    e = launch_attn(at, d->batch, st);
    if (e != hipSuccess) break;
    GemmArgs g2{att, nullptr, 0, d->eps, (const uint8_t*)L.o_w, L.o_s, H, nq * SK_HD, h, nullptr, xb, L.post_norm, ssb,
                1, gpart, gctr};
    e = launch_gemm<true>(g2, kOutAcc, st);
    if (e != hipSuccess) break;
    GemmArgs g3{xb, ssb, H / 16, d->eps, (const uint8_t*)L.gu_w, L.gu_s, 2 * I, H, nullptr, act, nullptr, nullptr, nullptr,
                1, gpart, gctr};
    e = launch_gemm<true>(g3, kOutSwiglu, st);
    if (e != hipSuccess) break;
    const float* nw_next = l + 1 < d->n_layers ? d->layers[l + 1].in_norm : d->norm;
    GemmArgs g4{act, nullptr, 0, d->eps, (const uint8_t*)L.down_w, L.down_s, H, I, h, nullptr, xa, nw_next, ssa,
                1, gpart, gctr};
    e = launch_gemm<true>(g4, kOutAcc, st);
    if (e != hipSuccess) break;
    if (d->layer_out)
      e = hipMemcpyAsync(d->layer_out + (size_t)l * kM * H, h, (size_t)kM * H * 4, hipMemcpyDeviceToDevice, st);
  }
  if (e == hipSuccess) {
    GemmArgs gh{xa, ssa, H / 16, d->eps, (const uint8_t*)d->head_w, d->head_s, V, H, logits, nullptr, nullptr, nullptr,
                nullptr, 1, gpart, gctr};
    e = launch_gemm<true>(gh, kOutF32, st);
  }
  if (e == hipSuccess) e = embed_launch(d, 1, logits, st);
  return sk_check_launch(e, "sk_batch_frame");
}
