// One-token GQA decode attention with fused per-head q/k RMSNorm, rotate-half RoPE and bf16 KV append.
//
// Replaces the reference's `attn` kernel (qwen3/kernels.py:338-414), which runs one 256-thread block per kv head
// (8 blocks on the whole GPU) and keeps every score of the cache in shared memory. Here the cache length is split:
// block (kvh, split) takes positions [t0, t1) of kv head kvh for both of its q heads and produces an
// unnormalised partial (max m, sum l, o = Σ exp(s - m) v). The last block of a head to arrive (a counter per head
// in the workspace) merges the partials with a log-sum-exp combine and writes the output, so the whole step is
// one launch of nkv * nsplit blocks.
//
// Decode attention moves few bytes per block, so its time is the launch and a chain of dependent memory round trips. A
// block has two before it can publish: everything whose address does not depend on the position goes out first (q, the
// new k and v, the norm weights and every K/V row of the block's first pass), together with the position; then the RoPE
// row. A cache that fits one block needs no more; else the partial is published, counted and merged (three more).
//
// Each wave works alone on its positions (32 per pass of a bf16 cache, 16 of an f32 cache) to its own maximum, sum and
// Σ p v, and the waves meet once in LDS: two barriers. Scores of a bf16 cache come from the matrix cores: q of both heads
// is kept as three bf16 terms (which give the fp32 value exactly) in rows 4 head + term of the MFMA's A, so the products
// are exact and a lane (16 head + position) finds its score's terms in its own registers; those of an f32 cache are
// 16-lane DPP sums. Σ p v stays on the vector units, where a row of V is one contiguous load of 16 lanes.
// Per call, HBM-cold, 8 kv heads (cache length / position), against blocks of 64 positions per pass whose statistics and
// sums were shared by the block: bf16 320 / 256 7.2 -> 6.6 us, 1024 / 100 8.1 -> 5.1, 1024 / 1000 10.0 -> 6.9, 2048 / 1601
// 12.9 -> 8.0, 5000 / 4000 21.6 -> 12.5; f32 320 / 256 7.5 -> 6.2, 1280 / 1023 12.7 -> 8.8, 5000 / 4000 25.1 -> 15.4 (33 MB).
// Nontemporal loads, which the batched attention uses, lose here (5000 / 4000 14.0): one stream's cache stays in the
// caches from step to step.
//
// Numerics follow the reference: K is stored as bf16 (round to nearest even) after norm and RoPE, and the
// rounded value is used for its own score; V is stored as given; q stays fp32 and is scaled by 1/sqrt(128) after
// RoPE; softmax subtracts the max and uses expf; one division at the end.
#include <type_traits>

#include "common.h"
#include "internal.h"

namespace {

constexpr int kSplitMax = 16;
constexpr int kPart = SK_HD + 2;  // m, l, o[128]
constexpr float kInvSqrtHd = 0.08838834764831845f;

// Blocks of four waves over the cache: one block per head up to 128 positions (64 of f32; nothing to publish and merge),
// else 16 splits or fewer; beyond that (2048 positions, 1024 of f32) blocks of eight waves and as many passes as 16 splits
// take. Fixed chunks (rather than the cache so far divided evenly) let a block load its first pass before it knows the
// position. Measured against the neighbours: eight waves per block at 577 and 1024 positions 7.9 and 8.3 us (four: 6.7 and
// 6.9), a single block of sixteen waves at 320 8.2 (three splits: 6.6), sixteen waves in one pass at 5000 13.7 (eight
// waves in two: 12.5).
struct SplitPlan {
  int waves, chunk, nsplit;
};
constexpr int wave_pos(int ct) { return ct == SK_CT_BF16 ? 32 : 16; }
SplitPlan split_plan(int max_len, int ct) {
  const int wp = wave_pos(ct), waves = max_len <= 4 * wp * kSplitMax ? 4 : 8, pass = waves * wp;
  const int chunk = pass * (int)(((int64_t)max_len + (int64_t)pass * kSplitMax - 1) / ((int64_t)pass * kSplitMax));
  return {waves, chunk, (max_len + chunk - 1) / chunk};
}
constexpr int64_t part_bytes(int nkv, int nsplit) { return ((int64_t)nkv * 2 * nsplit * kPart * 4 + 255) / 256 * 256; }
// Workspace: the error word (byte 0) and the per-head arrival counters (from byte 4) first, at a fixed place for
// any cache length, then the partials, so one workspace serves calls with different max_len (talker and code
// predictor) without a partial landing on a counter.
constexpr uint32_t kErrBadPos = 5;  // the position lies outside [0, max_len): nothing is read or written
constexpr int64_t counter_bytes(int nkv) { return ((int64_t)nkv * 4 + 4 + 255) / 256 * 256; }

// A wave's K and V rows of one pass. bf16: lane (gq, sl) holds K of positions 16 i + sl, dims 32 c + 8 gq .. + 8 (the MFMA's
// B), and V of positions 4 i + gq, dims 8 sl .. + 8. f32: K and V of positions 4 i + gq, dims 8 sl .. + 8.
template <int CT> struct Rows;
template <> struct Rows<SK_CT_BF16> {
  uint4 k[2][4], v[8];
  __device__ __forceinline__ void load(const bf16_t* K, const bf16_t* V, int row0, int last, int gq, int sl) {
#pragma unroll
    for (int i = 0; i < 2; i++) {
      const bf16_t* p = K + (size_t)min(row0 + 16 * i + sl, last) * SK_HD + 8 * gq;
#pragma unroll
      for (int c = 0; c < 4; c++) k[i][c] = gload4((const uint4*)(p + 32 * c));
    }
#pragma unroll
    for (int i = 0; i < 8; i++) v[i] = gload4((const uint4*)(V + (size_t)min(row0 + 4 * i + gq, last) * SK_HD + 8 * sl));
  }
  // the row at pos from LDS; zero V past it (its weight is zero, the memory may hold anything)
  __device__ __forceinline__ void fix(const bf16_t* ks, const bf16_t* vs, int row0, int pos, int gq, int sl) {
#pragma unroll
    for (int i = 0; i < 2; i++)
      if (row0 + 16 * i + sl == pos)
#pragma unroll
        for (int c = 0; c < 4; c++) k[i][c] = *(const uint4*)&ks[32 * c + 8 * gq];
#pragma unroll
    for (int i = 0; i < 8; i++) {
      if (row0 + 4 * i + gq == pos) v[i] = *(const uint4*)&vs[8 * sl];
      else if (row0 + 4 * i + gq > pos) v[i] = make_uint4(0, 0, 0, 0);
    }
  }
  __device__ __forceinline__ void value(int i, float* o) const { unpack_bf8(v[i], o); }
};
template <> struct Rows<SK_CT_F32> {
  uint4 k[4][2], v[4][2];
  __device__ __forceinline__ void load(const float* K, const float* V, int row0, int last, int gq, int sl) {
#pragma unroll
    for (int i = 0; i < 4; i++) {
      const size_t at = (size_t)min(row0 + 4 * i + gq, last) * SK_HD + 8 * sl;
#pragma unroll
      for (int c = 0; c < 2; c++) k[i][c] = gload4((const uint4*)(K + at) + c);
    }
#pragma unroll
    for (int i = 0; i < 4; i++) {
      const size_t at = (size_t)min(row0 + 4 * i + gq, last) * SK_HD + 8 * sl;
#pragma unroll
      for (int c = 0; c < 2; c++) v[i][c] = gload4((const uint4*)(V + at) + c);
    }
  }
  __device__ __forceinline__ void fix(const float* ks, const float* vs, int row0, int pos, int gq, int sl) {
#pragma unroll
    for (int i = 0; i < 4; i++)
#pragma unroll
      for (int c = 0; c < 2; c++) {
        if (row0 + 4 * i + gq == pos) {
          k[i][c] = *(const uint4*)&ks[8 * sl + 4 * c];
          v[i][c] = *(const uint4*)&vs[8 * sl + 4 * c];
        } else if (row0 + 4 * i + gq > pos) {
          v[i][c] = make_uint4(0, 0, 0, 0);
        }
      }
  }
  static __device__ __forceinline__ void get(const uint4 (&r)[2], float* o) {
    o[0] = __uint_as_float(r[0].x); o[1] = __uint_as_float(r[0].y); o[2] = __uint_as_float(r[0].z); o[3] = __uint_as_float(r[0].w);
    o[4] = __uint_as_float(r[1].x); o[5] = __uint_as_float(r[1].y); o[6] = __uint_as_float(r[1].z); o[7] = __uint_as_float(r[1].w);
  }
  __device__ __forceinline__ void value(int i, float* o) const { get(v[i], o); }
};

__device__ __forceinline__ int64_t uniform64(int64_t v) {
  const uint32_t lo = __builtin_amdgcn_readfirstlane((uint32_t)v), hi = __builtin_amdgcn_readfirstlane((uint32_t)((uint64_t)v >> 32));
  return (int64_t)(((uint64_t)hi << 32) | lo);
}

template <int CT, int NW>
__global__ __launch_bounds__(SK_WAVE * NW) void k_attn(const float* __restrict__ qkv, const float* __restrict__ qn,
                                                       const float* __restrict__ kn, float eps, const float* __restrict__ rope,
                                                       typename Cache<CT>::T* __restrict__ Kc,
                                                       typename Cache<CT>::T* __restrict__ Vc,
                                                       const int64_t* __restrict__ pos_ptr, int pos_add, int max_len, int nq,
                                                       int nkv, float* __restrict__ out, float* __restrict__ part,
                                                       unsigned* __restrict__ err, unsigned* __restrict__ counters,
                                                       int chunk, int nsplit) {
  using C = Cache<CT>;
  using T = typename C::T;
  constexpr bool kMfma = CT == SK_CT_BF16;
  constexpr int WP = wave_pos(CT), kPass = WP * NW, kTerms = 3;
  __shared__ __align__(16) bf16_t qt[kMfma ? 8 : 1][SK_HD + 8];  // bf16: row 4 head + term
  __shared__ __align__(16) float qs[kMfma ? 1 : 2][SK_HD];       // f32: both heads
  __shared__ __align__(16) T ksh[SK_HD];                         // this step's K and V rows as the cache holds them
  __shared__ __align__(16) T vsh[SK_HD];
  __shared__ float es[NW][WP][2];                                // softmax weights of a wave's positions, both heads
  __shared__ __align__(16) float op[NW][2][SK_HD];
  __shared__ float ml[NW][2][2];
  __shared__ __align__(16) float fs[2][kSplitMax];
  __shared__ float ls[2];
  __shared__ int is_last;
  const int kvh = blockIdx.x, split = blockIdx.y;
  const int t = threadIdx.x, w = __builtin_amdgcn_readfirstlane(t >> 6), lane = t & 63, gq = lane >> 4, sl = lane & 15;
  const int t0 = split * chunk;
  T* Kh = Kc + (size_t)kvh * max_len * SK_HD;
  T* Vh = Vc + (size_t)kvh * max_len * SK_HD;
  // what does not depend on the position: wave 0 takes q of head 2 kvh, wave 1 q of head 2 kvh + 1, wave 2 k, wave 3 v, dims
  // lane and lane + 64 per lane; then every cache row of the first pass (rows past the cache's end read its last row and,
  // like rows at or past the position, are never used)
  // (the position by a vector load ahead of all others: a scalar one would be waited for with the arguments; without a
  // pointer it reads the workspace and drops what it finds)
  const int64_t pv = __hip_atomic_load(pos_ptr ? pos_ptr : (const int64_t*)part, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
  const int wq = w & 3;
  const float* src = qkv + (wq < 2 ? (2 * kvh + wq) * SK_HD : nq * SK_HD + ((wq - 2) * nkv + kvh) * SK_HD);
  const float* nw = wq < 2 ? qn : kn;
  const float x0 = gload(src + lane), x1 = gload(src + lane + 64), n0 = gload(nw + lane), n1 = gload(nw + lane + 64);
  Rows<CT> r;
  if (t0 + WP * w < max_len) r.load(Kh, Vh, t0 + WP * w, max_len - 1, gq, sl);
  const int64_t pos64 = (pos_ptr ? uniform64(pv) : 0) + (int64_t)pos_add;
  if (pos64 < 0 || pos64 >= max_len) {
    // every block takes this exit (the position is uniform), so no counter moves and nothing is written
    if (kvh == 0 && split == 0 && t == 0) __hip_atomic_store(err, kErrBadPos, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    return;
  }
  const int pos = (int)pos64;
  if (t0 > pos) return;  // the splits past the position neither publish nor count
  const int ns = pos / chunk + 1;
  const int n = min(chunk, pos + 1 - t0);
  const bool has_pos = split == ns - 1;
  if (w < 4) {
    const float c = gload(rope + (size_t)pos * SK_HD + lane), sn = gload(rope + (size_t)pos * SK_HD + 64 + lane);
    if (w < 3) {  // per-head RMSNorm, RoPE
      const float inv = rsqrtf(wave_sum(x0 * x0 + x1 * x1) / SK_HD + eps);
      const float y0 = x0 * inv * n0, y1 = x1 * inv * n1;
      const float r0 = y0 * c + -y1 * sn, r1 = y1 * c + y0 * sn;
      if (w < 2) {
        if constexpr (kMfma) {
          float v0 = r0 * kInvSqrtHd, v1 = r1 * kInvSqrtHd;
#pragma unroll
          for (int q = 0; q < kTerms; q++) {
            const bf16_t b0 = f2bf_hw(v0), b1 = f2bf_hw(v1);
            qt[4 * w + q][lane] = b0;
            qt[4 * w + q][lane + 64] = b1;
            v0 -= bf2f(b0);
            v1 -= bf2f(b1);
          }
        } else {
          qs[w][lane] = r0 * kInvSqrtHd;
          qs[w][lane + 64] = r1 * kInvSqrtHd;
        }
      } else if (has_pos) {
        const T k0 = C::st(r0), k1 = C::st(r1);
        ksh[lane] = k0;
        ksh[lane + 64] = k1;
        Kh[(size_t)pos * SK_HD + lane] = k0;
        Kh[(size_t)pos * SK_HD + lane + 64] = k1;
      }
    } else if (has_pos) {
      const T v0 = C::st(x0), v1 = C::st(x1);
      vsh[lane] = v0;
      vsh[lane + 64] = v1;
      Vh[(size_t)pos * SK_HD + lane] = v0;
      Vh[(size_t)pos * SK_HD + lane + 64] = v1;
    }
  }
  __syncthreads();
  bf16x8 qa[4];
  float q0[8], q1[8];
  if constexpr (kMfma) {
    const bool used = sl < 8 && (sl & 3) < kTerms;
#pragma unroll
    for (int c = 0; c < 4; c++) {
      const uint4 v = *(const uint4*)&qt[4 * ((sl >> 2) & 1) + min(sl & 3, kTerms - 1)][32 * c + 8 * gq];
      qa[c] = as_bf16x8(used ? v : make_uint4(0, 0, 0, 0));
    }
  } else {
#pragma unroll
    for (int e = 0; e < 8; e++) { q0[e] = qs[0][8 * sl + e]; q1[e] = qs[kMfma ? 0 : 1][8 * sl + e]; }
  }
  // the wave's partial: its maximum and sum (lanes 16 head .. + 16) and Σ p v of dims 8 sl .. + 8 over its share of rows
  float mw = -INFINITY, lw = 0.f, a0[8], a1[8];
#pragma unroll
  for (int k = 0; k < 8; k++) { a0[k] = 0.f; a1[k] = 0.f; }
  auto pass = [&](int base) __attribute__((always_inline)) {  // positions t0 + base + WP w .. + WP
    const int off = base + WP * w;
    if (t0 + base + kPass > pos) r.fix(ksh, vsh, t0 + off, pos, gq, sl);
    float sv[2], e[2];
    if constexpr (kMfma) {
#pragma unroll
      for (int i = 0; i < 2; i++) {
        f32x4 acc = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int c = 0; c < 4; c++) acc = __builtin_amdgcn_mfma_f32_16x16x32_bf16(qa[c], as_bf16x8(r.k[i][c]), acc, 0, 0, 0);
        sv[i] = acc[0] + (acc[1] + acc[2]);
      }
    } else {
#pragma unroll
      for (int i = 0; i < 4; i++) {
        float k8[8], s0 = 0.f, s1 = 0.f;
        Rows<SK_CT_F32>::get(r.k[i], k8);
#pragma unroll
        for (int k = 0; k < 8; k++) { s0 = __builtin_fmaf(q0[k], k8[k], s0); s1 = __builtin_fmaf(q1[k], k8[k], s1); }
        s0 = row16_sum(s0);
        s1 = row16_sum(s1);
        if (sl < 2) es[w][4 * i + gq][sl] = sl ? s1 : s0;
      }
      wave_sync();
      sv[0] = es[w][sl][gq & 1];
      sv[1] = -INFINITY;
    }
#pragma unroll
    for (int i = 0; i < 2; i++)
      if (off + 16 * i + sl >= n) sv[i] = -INFINITY;
    const float mn = fmaxf(mw, row16_max(fmaxf(sv[0], sv[1])));
#pragma unroll
    for (int i = 0; i < 2; i++) e[i] = 16 * i < WP && off + 16 * i + sl < n ? expf(sv[i] - mn) : 0.f;
    const float le = row16_sum(e[0] + e[1]);
    if (base > 0) {
      const float fo = mw == -INFINITY ? 0.f : expf(mw - mn), f0 = lane_value(fo, 0), f1 = lane_value(fo, 16);
      lw *= fo;
#pragma unroll
      for (int k = 0; k < 8; k++) { a0[k] *= f0; a1[k] *= f1; }
    }
    lw += le;
    mw = mn;
    if (gq < 2) {
      es[w][sl][gq] = e[0];
      if constexpr (WP > 16) es[w][16 + sl][gq] = e[1];
    }
    wave_sync();
#pragma unroll
    for (int i = 0; i < WP / 4; i++) {
      const float2 ew = *(const float2*)&es[w][4 * i + gq][0];
      float v8[8];
      r.value(i, v8);
#pragma unroll
      for (int k = 0; k < 8; k++) { a0[k] = __builtin_fmaf(ew.x, v8[k], a0[k]); a1[k] = __builtin_fmaf(ew.y, v8[k], a1[k]); }
    }
    wave_sync();
  };
  if (WP * w < n) {
    pass(0);
    for (int base = kPass; base + WP * w < n; base += kPass) {
      r.load(Kh, Vh, t0 + base + WP * w, max_len - 1, gq, sl);
      pass(base);
    }
  }
  *(float4*)&op[w][gq >> 1][8 * sl + 4 * (gq & 1)] = rows_sum(a0, a1);
  if (gq < 2 && sl == 0) {
    ml[w][gq][0] = mw;
    ml[w][gq][1] = lw;
  }
  __syncthreads();
  // the waves' partials of head p, dim d (threads 0..255)
  const int p = (t >> 7) & 1, d = t & (SK_HD - 1);
  float m = ml[0][p][0], l = 0.f, o = 0.f;
  if (t < 2 * SK_HD) {
#pragma unroll
    for (int q = 1; q < NW; q++) m = fmaxf(m, ml[q][p][0]);
#pragma unroll
    for (int q = 0; q < NW; q++) {
      const float f = ml[q][p][0] == -INFINITY ? 0.f : expf(ml[q][p][0] - m);
      l = __builtin_fmaf(f, ml[q][p][1], l);
      o = __builtin_fmaf(f, op[q][p][d], o);
    }
    if (ns == 1) out[(2 * kvh + p) * SK_HD + d] = l > 0.f ? o / l : 0.f;  // the whole cache so far in this block
  }
  if (ns == 1) return;
  // ---- publish the partial (device-coherent stores), count the arrival ---------------------------------------
  if (t < 2 * SK_HD) {
    const uint32_t pofs = (uint32_t)((kvh * 2 + p) * nsplit + split) * kPart * 4;
    if (d == 0) { buf_stf(part, pofs, m); buf_stf(part, pofs + 4, l); }
    buf_stf(part, pofs + 8 + 4 * d, o);
  }
  __builtin_amdgcn_s_waitcnt(0);
  __syncthreads();
  if (t == 0) {
    const unsigned prev = __hip_atomic_fetch_add(&counters[kvh], 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    is_last = prev == (unsigned)(ns - 1);
  }
  __syncthreads();
  if (!is_last) return;
  // ---- merge: one batch of device-coherent loads; wave 0 finds the splits' weights for all ------------------
  float oc[kSplitMax];
#pragma unroll
  for (int cc = 0; cc < kSplitMax; cc++)  // (waves past the fourth repeat the first four's)
    oc[cc] = buf_ldf(part, (uint32_t)((kvh * 2 + p) * nsplit + min(cc, ns - 1)) * kPart * 4 + 8 + 4 * d);
  if (w == 0) {  // lane 16 head + split
    const uint32_t of = (uint32_t)((kvh * 2 + (gq & 1)) * nsplit + min(sl, ns - 1)) * kPart * 4;
    const float ms = buf_ldf(part, of), lp = buf_ldf(part, of + 4);
    const bool has = sl < ns && ms != -INFINITY;
    const float M = row16_max(has ? ms : -INFINITY);
    const float f = has ? expf(ms - M) : -1.f;  // negative: no such partial
    const float L = row16_sum(has ? f * lp : 0.f);
    if (gq < 2) {
      fs[gq][sl] = f;
      if (sl == 0) ls[gq] = L;
    }
    if (t == 0) __hip_atomic_store(&counters[kvh], 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  }
  __syncthreads();
  const float L = ls[p];
  float O = 0.f;
#pragma unroll
  for (int cc = 0; cc < kSplitMax; cc++) {
    const float f = fs[p][cc], x = __builtin_fmaf(f, oc[cc], O);
    O = f < 0.f ? O : x;
  }
  if (t < 2 * SK_HD) out[(2 * kvh + p) * SK_HD + d] = L > 0.f ? O / L : 0.f;
}

}  // namespace

extern "C" int64_t sk_attn_workspace_size(int nq, int nkv, int max_len) {
  if (nkv <= 0 || max_len <= 0) return 0;
  (void)nq;
  // one size past the shortest caches: a workspace also serves shorter ones, whose plans may have more splits
  return counter_bytes(nkv) + part_bytes(nkv, max_len <= 128 ? 1 : kSplitMax);
}

namespace {

// Checks shared by both entry points; SK_OK or the status already recorded.
int check_attn(const float* qkv, const float* qn, const float* kn, const float* rope, const void* Kc, const void* Vc,
               int max_len, int nq, int nkv, const float* out, int ct) {
  if (!qkv || !qn || !kn || !rope || !Kc || !Vc || !out) return sk_set_error(SK_EINVAL, "sk_attn: null pointer");
  if (nkv <= 0 || nq != 2 * nkv || max_len <= 0)
    return sk_set_error(SK_EINVAL, "sk_attn: needs nq == 2*nkv and max_len > 0 (head_dim 128)");
  if ((int64_t)nkv * 2 * kSplitMax * kPart * 4 >= (int64_t)1 << 31 || (int64_t)max_len * nkv * SK_HD * 4 >= (int64_t)1 << 40)
    return sk_set_error(SK_EINVAL, "sk_attn: sizes out of range");
  if (ct != SK_CT_BF16 && ct != SK_CT_F32) return sk_set_error(SK_EINVAL, "sk_attn: bad cache type");
  if (!SK_ALIGNED16(Kc) || !SK_ALIGNED16(Vc)) return sk_set_error(SK_EINVAL, "sk_attn: caches must be 16-byte aligned");
  return SK_OK;
}

int launch_attn(const float* qkv, const float* qn, const float* kn, float eps, const float* rope, void* Kc, void* Vc,
                const int64_t* pos_ptr, int pos_add, int max_len, int nq, int nkv, float* out, float* part,
                unsigned* err, unsigned* counters, int ct, hipStream_t st, const char* name) {
  const SplitPlan sp = split_plan(max_len, ct);
  auto go = [&](auto ctc, auto nwc) {
    constexpr int CT = decltype(ctc)::value, NW = decltype(nwc)::value;
    using T = typename Cache<CT>::T;
    hipLaunchKernelGGL((k_attn<CT, NW>), dim3(nkv, sp.nsplit), dim3(SK_WAVE * NW), 0, st, qkv, qn, kn, eps, rope, (T*)Kc, (T*)Vc,
                       pos_ptr, pos_add, max_len, nq, nkv, out, part, err, counters, sp.chunk, sp.nsplit);
  };
  auto by_waves = [&](auto ctc) {
    if (sp.waves == 4) go(ctc, std::integral_constant<int, 4>{});
    else go(ctc, std::integral_constant<int, 8>{});
  };
  if (ct == SK_CT_BF16) by_waves(std::integral_constant<int, SK_CT_BF16>{});
  else by_waves(std::integral_constant<int, SK_CT_F32>{});
  return sk_check_launch(hipGetLastError(), name);
}

}  // namespace

extern "C" int sk_attn(const float* qkv, const float* qn, const float* kn, float eps, const float* rope, void* Kc,
                       void* Vc, const int64_t* pos_ptr, int pos_add, int max_len, int nq, int nkv, float* out,
                       void* workspace, int64_t workspace_bytes, int ct, void* stream) {
  const int rc = check_attn(qkv, qn, kn, rope, Kc, Vc, max_len, nq, nkv, out, ct);
  if (rc != SK_OK) return rc;
  if (!workspace) return sk_set_error(SK_EINVAL, "sk_attn: null pointer");
  if (!SK_ALIGNED16(workspace)) return sk_set_error(SK_EINVAL, "sk_attn: workspace must be 16-byte aligned");
  if (workspace_bytes < sk_attn_workspace_size(nq, nkv, max_len))
    return sk_set_error(SK_EWORKSPACE, "sk_attn: workspace too small");
  unsigned* err = (unsigned*)workspace;
  float* part = (float*)((char*)workspace + counter_bytes(nkv));
  return launch_attn(qkv, qn, kn, eps, rope, Kc, Vc, pos_ptr, pos_add, max_len, nq, nkv, out, part, err, err + 1, ct,
                     (hipStream_t)stream, "sk_attn");
}

// ---- allocation-free variant -------------------------------------------------------------------------------------
// sk_attn_noalloc keeps its split-K scratch (error word, arrival counters, partials) in this file-scope device array
// instead of a caller workspace: at most kNoAllocMaxKv kv heads. Each device holds its own copy until the process
// ends. The host never passes the array's name to a kernel: the first call on a device looks up the device address
// with hipGetSymbolAddress and keeps it per device.
namespace {
constexpr int kNoAllocMaxKv = 16;
constexpr int64_t kNoAllocBytes = counter_bytes(kNoAllocMaxKv) + part_bytes(kNoAllocMaxKv, kSplitMax);
constexpr int kMaxDevices = 64;
}  // namespace

static __device__ __align__(256) unsigned char scratch[kNoAllocBytes];

namespace {

void* g_scratch[kMaxDevices];  // device address of `scratch` per device (null until the first call there)

// Clears the error word and the arrival counters (the first counter_bytes of the scratch): a fill kernel, not a
// memset node, so the clear is also safe inside a captured graph.
__global__ void k_clear_words(unsigned* p, int n) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) p[i] = 0u;
}

}  // namespace

extern "C" int sk_attn_noalloc(const float* qkv, const float* qn, const float* kn, float eps, const float* rope,
                               void* Kc, void* Vc, const int64_t* pos_ptr, int pos_add, int max_len, int nq, int nkv,
                               float* out, int* err, int ct, void* stream) {
  const int rc = check_attn(qkv, qn, kn, rope, Kc, Vc, max_len, nq, nkv, out, ct);
  if (rc != SK_OK) return rc;
  if (nkv > kNoAllocMaxKv)
    return sk_set_error(SK_EINVAL, "sk_attn_noalloc: at most 16 kv heads (the static scratch holds 260 KiB)");
  int dev = 0;
  if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= kMaxDevices)
    return sk_set_error(SK_EDEVICE, "sk_attn_noalloc: no current HIP device");
  hipStream_t st = (hipStream_t)stream;
  if (!g_scratch[dev]) {
    void* p = nullptr;
    const hipError_t e = hipGetSymbolAddress(&p, HIP_SYMBOL(scratch));
    if (e != hipSuccess || !p) return sk_check_launch(e != hipSuccess ? e : hipErrorInvalidSymbol,
                                                      "sk_attn_noalloc: hipGetSymbolAddress(scratch)");
    const int words = (int)(counter_bytes(kNoAllocMaxKv) / 4);
    hipLaunchKernelGGL(k_clear_words, dim3(1), dim3(words), 0, st, (unsigned*)p, words);
    const int lrc = sk_check_launch(hipGetLastError(), "sk_attn_noalloc: clearing the scratch counters");
    if (lrc != SK_OK) return lrc;
    g_scratch[dev] = p;
  }
  unsigned* base = (unsigned*)g_scratch[dev];
  float* part = (float*)((char*)base + counter_bytes(kNoAllocMaxKv));
  unsigned* errw = err ? (unsigned*)err : base;  // word 0 of the scratch when the caller takes no error word
  return launch_attn(qkv, qn, kn, eps, rope, Kc, Vc, pos_ptr, pos_add, max_len, nq, nkv, out, part, errw, base + 1, ct,
                     st, "sk_attn_noalloc");
}
