// Small kernels of the talker step (final RMSNorm, embedding rows, greedy sampling) and the library's
// error/status plumbing.
#include <stdio.h>
#include <string.h>

#include "common.h"
#include "internal.h"

namespace {

thread_local char g_err[512] = "";

// ---- RMSNorm (qwen3/kernels.py:312-319) --------------------------------------------------------------------
// One block of 1024 threads; P values per thread, all loaded (with the weights) at the top, so the launch, one memory round
// trip and one barrier bound it: 1024 values 3.4 -> 2.2 us, against 256 threads that read the input twice in loops.
constexpr int kNormThreads = 1024;
template <int P>
__global__ __launch_bounds__(kNormThreads) void k_rmsnorm(const float* __restrict__ h, const float* __restrict__ nw,
                                                           float eps, float* __restrict__ out, int K) {
  __shared__ float red[kNormThreads / SK_WAVE];
  const int t = threadIdx.x, per = (K + kNormThreads - 1) / kNormThreads;
  float hv[P], nv[P], ss = 0.f;
#pragma unroll
  for (int j = 0; j < P; j++) {
    const int i = min(t + j * kNormThreads, K - 1);
    hv[j] = h[i];
    nv[j] = nw[i];
  }
#pragma unroll
  for (int j = 0; j < P; j++) ss = t + j * kNormThreads < K ? __builtin_fmaf(hv[j], hv[j], ss) : ss;
  for (int j = P; j < per; j++) {  // longer inputs: the rest is read twice
    const int i = t + j * kNormThreads;
    if (i < K) ss = __builtin_fmaf(h[i], h[i], ss);
  }
  ss = wave_sum(ss);
  if ((t & 63) == 0) red[t >> 6] = ss;
  __syncthreads();
  const float tot = row16_sum(red[t & 15]);
  static_assert(kNormThreads / SK_WAVE == 16, "one wave's sum per lane of a row");
  const float inv = rsqrtf(tot / K + eps);
#pragma unroll
  for (int j = 0; j < P; j++) {
    const int i = t + j * kNormThreads;
    if (i < K) out[i] = hv[j] * inv * nv[j];
  }
  for (int j = P; j < per; j++) {
    const int i = t + j * kNormThreads;
    if (i < K) out[i] = h[i] * inv * nw[i];
  }
}

// ---- embedding row (qwen3/kernels.py:321-326) --------------------------------------------------------------
template <int CT>
__global__ void k_embed(const typename Cache<CT>::T* __restrict__ table, const int64_t* __restrict__ idx,
                        float* __restrict__ out, int dim) {
  const int64_t r = idx[0];
  for (int i = blockIdx.x * blockDim.x + threadIdx.x; i < dim; i += gridDim.x * blockDim.x)
    out[i] = Cache<CT>::ld(table[(size_t)r * dim + i]);
}

// ---- talker input: sum of G codebook rows + pad (qwen3/kernels.py:328-336) ----------------------------------
template <int CT>
__global__ void k_talker_in(const uint64_t* __restrict__ tabs, const int64_t* __restrict__ codes,
                            const typename Cache<CT>::T* __restrict__ pad, float* __restrict__ out, int dim, int G) {
  typedef typename Cache<CT>::T ct;
  for (int i = blockIdx.x * blockDim.x + threadIdx.x; i < dim; i += gridDim.x * blockDim.x) {
    float s = 0.f;
    for (int g = 0; g < G; g++) s += Cache<CT>::ld(((const ct*)tabs[g])[(size_t)codes[g] * dim + i]);
    out[i] = s + Cache<CT>::ld(pad[i]);
  }
}

// ---- greedy sampling with the talker processor (qwen3/sampler.py:37-159, do_sample = 0) ---------------------
constexpr int kSampleThreads = 1024;
constexpr int kPer = SK_MAX_V / kSampleThreads;

// This thread's entries t + 1024 j through the talker processor, every load at the top (entries past V read the last
// one; the caller drops them).
template <int PER>
__device__ __forceinline__ void load_entries(const float* logits, int V, const uint8_t* seen, float rep_pen, const uint8_t* suppress,
                                             const int64_t* ngen, int min_new, int eos, int talker, float (&v)[PER]) {
  const int t = threadIdx.x;
  uint8_t sn[PER], sp[PER];
#pragma unroll
  for (int j = 0; j < PER; j++) {
    v[j] = gload(logits + min(t + j * kSampleThreads, V - 1));
    sn[j] = sp[j] = 0;
  }
  if (!talker) return;
  const int64_t ng = ngen ? ngen[0] : 0;
  if (seen) {
#pragma unroll
    for (int j = 0; j < PER; j++) sn[j] = gload(seen + min(t + j * kSampleThreads, V - 1));
  }
  if (suppress) {
#pragma unroll
    for (int j = 0; j < PER; j++) sp[j] = gload(suppress + min(t + j * kSampleThreads, V - 1));
  }
  const bool block_eos = ngen && ng < min_new;
#pragma unroll
  for (int j = 0; j < PER; j++) {
    if (sn[j]) v[j] = v[j] < 0.f ? v[j] * rep_pen : v[j] / rep_pen;
    if (sp[j] || (block_eos && t + j * kSampleThreads == eos)) v[j] = -INFINITY;
  }
}

// Of the block's 16 waves, each with its largest key and the lowest index that holds it: the index of the largest, the lowest
// on ties (wave 0; uniform).
__device__ __forceinline__ uint32_t block_pick(const uint32_t* keys, const uint32_t* idx, int lane) {
  constexpr int kWaves = kSampleThreads / SK_WAVE;
  const uint32_t k = lane < kWaves ? keys[lane] : 0u, i = lane < kWaves ? idx[lane] : 0xffffffffu;
  const uint32_t top = wave_umax(k);
  return ~wave_umax(k == top ? ~i : 0u);
}

__global__ __launch_bounds__(kSampleThreads) void k_sample_greedy(const float* __restrict__ logits, int V,
                                                                  uint8_t* __restrict__ seen, float rep_pen,
                                                                  const uint8_t* __restrict__ suppress,
                                                                  int64_t* __restrict__ ngen, int min_new, int eos,
                                                                  int64_t* __restrict__ out, int talker,
                                                                  int64_t* __restrict__ id0, int64_t* __restrict__ pos) {
  __shared__ uint32_t wkey[kSampleThreads / SK_WAVE], widx[kSampleThreads / SK_WAVE];
  const int t = threadIdx.x, lane = t & 63, w = t >> 6;
  float v[kPer];
  load_entries<kPer>(logits, V, seen, rep_pen, suppress, ngen, min_new, eos, talker, v);
  uint32_t best = 0, bi = 0xffffffffu;  // key 0 is below every non-NaN value; NaN never wins
#pragma unroll
  for (int j = 0; j < kPer; j++) {
    const int i = t + j * kSampleThreads;
    const uint32_t k = i < V && v[j] == v[j] ? order_key(v[j]) : 0u;
    if (k > best) { best = k; bi = (uint32_t)i; }
  }
  const uint32_t top = wave_umax(best);
  const uint32_t ti = ~wave_umax(best == top ? ~bi : 0u);
  if (lane == 0) { wkey[w] = top; widx[w] = ti; }
  __syncthreads();
  if (w != 0) return;
  const uint32_t pick = block_pick(wkey, widx, lane);
  if (lane != 0) return;
  const int64_t id = pick >= (uint32_t)V ? 0 : (int64_t)pick;
  out[0] = id;
  if (talker) {
    if (id0) id0[0] = id;
    if (seen) seen[id] = 1;
    if (ngen) ngen[0] += 1;
    if (pos) pos[0] += 1;
  }
}

// ---- sampled pick: processor, temperature, top-k threshold, Gumbel-max (qwen3/sampler.py:37-159) -----------------
// One block of 1024 threads; thread t holds entries t + 1024 j (j < 4) in registers as processed values and their
// order keys. The threshold (the key of the top_k-th largest value, ties kept) is found without a histogram:
//  * bound: the top_k-th largest of group maxima is a lower bound of the threshold, since the maxima are themselves
//    entries. Up to top_k = 64: 64 groups (16 threads' entries each, a DPP row max), whose ranks wave 0 counts, one lane per
//    maximum. Up to 256: 256 groups of 16 consecutive entries, bisected by wave 0.
//  * candidates: the entries at or above the bound are compacted into LDS (one ballot per register and one LDS atomic
//    per wave for the wave's offset); typically twice top_k of them.
//  * up to top_k = 64 and 256 candidates, a candidate is kept iff fewer than top_k candidates have a larger key (every entry
//    above the bound is a candidate, so that is its rank among all): four lanes count for one candidate, while other
//    waves draw the Gumbel value of every candidate.
//  * else wave 0 bisects the key space over the candidates, bit by bit from the highest bit where the bound and the largest
//    key differ, counting the candidates at or above each probe with ballots. Below the bound every count reaches top_k, as
//    it does over all entries, so the result is the full-vocabulary threshold, and every thread draws for its own
//    entries.
// Larger top_k (256 < top_k < V) bisects over all entries, every wave counting its own with ballots per step.
// Entries past V carry key 0, which no probe counts (every probe is at least 1). Every entry at or above the
// threshold that is not -inf draws its Gumbel value v - log(-log(u)), u from Philox4x32-10 with counter (index,
// draw lo, draw hi, 0x51) and key (seed lo, seed hi); the largest wins, the lowest index on ties (a wave max of the
// value, then a wave max of the complemented index among the lanes holding it). Afterwards the draw counter advances.
// What bounds it is the chain: the launch, one memory round trip and four barriers' worth of serial steps. A frame's
// sixteen picks (V 2048, top_k 50, and the talker's) in a graph: 127 us with entries loaded one after the other, two
// bisections and each wave drawing for its own entries, 70 now.
constexpr int kDrawThreads = kSampleThreads, kDrawWaves = kDrawThreads / SK_WAVE, kDrawPer = kPer;
constexpr int kBoundGroups = 256;  // groups of 16 entries: SK_MAX_V / 16
constexpr int kRankK = 64, kRankCand = 256;  // what the ranked path holds: top_k, candidates

// The largest key t in [lo, hi] whose count (keys >= t) reaches K, given count(lo) >= K: the bits above the highest
// bit where lo and hi differ are common to every such key; below it the key grows one bit at a time, each bit kept
// when the count at the key with that bit set still reaches K.
template <class F>
__device__ __forceinline__ uint32_t kth_key(uint32_t lo, uint32_t hi, uint32_t K, F count) {
  if (lo >= hi) return lo;
  const int top = 31 - __builtin_clz(lo ^ hi);
  uint32_t p = top == 31 ? 0u : lo & ~((2u << top) - 1u);
  for (int b = top; b >= 0; b--) {
    const uint32_t t = p | (1u << b);
    if (count(t) >= K) p = t;
  }
  return p;
}

__global__ __launch_bounds__(kDrawThreads) void k_sample_draw(const float* __restrict__ logits, int V, float inv_temp,
                                                               int top_k, uint8_t* __restrict__ seen, float rep_pen,
                                                               const uint8_t* __restrict__ suppress,
                                                               int64_t* __restrict__ ngen, int min_new, int eos,
                                                               const uint64_t* __restrict__ seed,
                                                               uint64_t* __restrict__ counter, int64_t* __restrict__ out,
                                                               int talker, int64_t* __restrict__ id0,
                                                               int64_t* __restrict__ pos) {
  __shared__ __align__(16) uint32_t gmax[kBoundGroups];
  __shared__ __align__(16) uint32_t cand[SK_MAX_V];
  __shared__ uint16_t cidx[SK_MAX_V];
  __shared__ uint32_t crank[kRankCand];
  __shared__ float cg[kRankCand];
  __shared__ uint32_t wsum[kDrawWaves];
  __shared__ uint32_t wpick[kDrawWaves];
  __shared__ uint32_t s_n, s_lb, s_thr;
  const int t = threadIdx.x, lane = t & 63, w = t >> 6;
  const uint64_t sd = seed[0], cnt = counter[0];
  float xv[kDrawPer];
  uint32_t key[kDrawPer];
  load_entries<kDrawPer>(logits, V, seen, rep_pen, suppress, ngen, min_new, eos, talker, xv);
#pragma unroll
  for (int j = 0; j < kDrawPer; j++) {
    xv[j] *= inv_temp;
    key[j] = t + j * kDrawThreads < V ? order_key(xv[j]) : 0u;
  }
  auto finish = [&](uint32_t pick) {  // wave 0, lane 0
    const int64_t id = pick >= (uint32_t)V ? 0 : (int64_t)pick;  // nothing kept: index 0
    out[0] = id;
    counter[0] = cnt + 1;
    if (talker) {
      if (id0) id0[0] = id;
      if (seen) seen[id] = 1;
      if (ngen) ngen[0] += 1;
      if (pos) pos[0] += 1;
    }
  };
  uint32_t thr = 0;  // 0 keeps every entry (top_k <= 0 or >= V)
  if (top_k > 0 && top_k < V) {
    const uint32_t K = (uint32_t)top_k;
    if (top_k <= kBoundGroups) {
      if (t == 0) s_n = 0;
      if (top_k <= kRankK) {
        uint32_t m = key[0];
#pragma unroll
        for (int j = 1; j < kDrawPer; j++) m = max(m, key[j]);
        m = row16_umax(m);
        if ((lane & 15) == 0) gmax[4 * w + (lane >> 4)] = m;
        __syncthreads();
        if (w == 0) {  // the largest maximum that at least K of the 64 reach (zero, an empty group's, where none does)
          const uint32_t g = gmax[lane];
          uint32_t c0 = 0, c1 = 0, c2 = 0, c3 = 0;
#pragma unroll
          for (int q = 0; q < 16; q++) {
            const uint4 o = *(const uint4*)&gmax[4 * q];
            c0 += o.x >= g;
            c1 += o.y >= g;
            c2 += o.z >= g;
            c3 += o.w >= g;
          }
          const uint32_t lb = wave_umax((c0 + c1) + (c2 + c3) >= K ? g : 0u);
          if (lane == 0) s_lb = lb;
        }
      } else {
        // bound: group maxima (lanes 16 r .. 16 r + 15 hold 16 consecutive entries of each j)
#pragma unroll
        for (int j = 0; j < kDrawPer; j++) {
          const uint32_t m = row16_umax(key[j]);
          if ((lane & 15) == 0) gmax[(j * kDrawWaves + w) * 4 + (lane >> 4)] = m;
        }
        __syncthreads();
        if (w == 0) {
          uint32_t g4[4], lo = 0xffffffffu, hi = 0;
#pragma unroll
          for (int q = 0; q < 4; q++) {
            g4[q] = gmax[lane + 64 * q];
            lo = min(lo, g4[q]);
            hi = max(hi, g4[q]);
          }
          lo = ~wave_umax(~lo);
          hi = wave_umax(hi);
          const uint32_t lb = kth_key(lo, hi, K, [&](uint32_t x) {
            uint32_t c = 0;
#pragma unroll
            for (int q = 0; q < 4; q++) c += (uint32_t)__popcll(__ballot(g4[q] >= x));
            return c;
          });
          if (lane == 0) s_lb = lb;
        }
      }
      __syncthreads();
      const uint32_t lb = s_lb;
      // candidates: keys >= lb (key 0 is never a candidate: no probe counts it)
#pragma unroll
      for (int j = 0; j < kDrawPer; j++) {
        const bool take = key[j] >= lb && key[j] != 0u;
        const uint64_t msk = __ballot(take);
        uint32_t base = 0;
        if (lane == 0 && msk) base = atomicAdd(&s_n, (uint32_t)__popcll(msk));
        base = (uint32_t)__builtin_amdgcn_readfirstlane((int)base);
        if (take) {
          const uint32_t at = base + __builtin_amdgcn_mbcnt_hi((uint32_t)(msk >> 32), __builtin_amdgcn_mbcnt_lo((uint32_t)msk, 0u));
          cand[at] = key[j];
          cidx[at] = (uint16_t)(t + j * kDrawThreads);
        }
      }
      __syncthreads();
      if (const uint32_t n = s_n; top_k <= kRankK && n <= kRankCand) {
        // the last quarter of the block draws, the first ones rank: thread 4 c + q compares candidate c with every fourth quad
        if (t >= kDrawThreads - kRankCand) {
          const uint32_t c = (uint32_t)(t - (kDrawThreads - kRankCand));
          if (c < n) {
            const uint32_t k = cand[c];
            const float v = __uint_as_float(k ^ ((k >> 31) ? 0x80000000u : 0xffffffffu));
            cg[c] = v == -INFINITY ? -INFINITY : gumbel(v, cidx[c], cnt, (uint32_t)sd, (uint32_t)(sd >> 32));
          }
        }
        for (uint32_t c = (uint32_t)t >> 2; t < kDrawThreads - kRankCand && c < n; c += (kDrawThreads - kRankCand) / 4) {
          const uint32_t k = cand[c];
          uint32_t r = 0;
          for (uint32_t q = 4 * (t & 3); q < n; q += 16) {
            const uint4 o = *(const uint4*)&cand[q];  // words past n: not counted
            r += o.x > k;
            r += q + 1 < n && o.y > k;
            r += q + 2 < n && o.z > k;
            r += q + 3 < n && o.w > k;
          }
          r += dpp_u<0xB1>(r);
          r += dpp_u<0x4E>(r);
          if ((t & 3) == 0) crank[c] = r;
        }
        __syncthreads();
        if (w != 0) return;
        uint32_t mk = order_key(-INFINITY), bi = 0xffffffffu;
#pragma unroll
        for (int q = 0; q < kRankCand / SK_WAVE; q++) {
          const uint32_t c = (uint32_t)(lane + q * SK_WAVE);
          if (c < n && crank[c] < K) {
            const float g = cg[c];
            const uint32_t k = g == g ? order_key(g == 0.f ? 0.f : g) : 0u, i = cidx[c];  // NaN never wins
            if (g != -INFINITY && (k > mk || (k == mk && i < bi))) { mk = k; bi = i; }
          }
        }
        const uint32_t top = wave_umax(mk);
        const uint32_t pick = ~wave_umax(mk == top ? ~bi : 0u);
        if (lane == 0) finish(pick);
        return;
      }
      if (w == 0) {
        const uint32_t n = s_n;
        uint32_t hi = 0;
        for (uint32_t c = (uint32_t)lane; c < n; c += 64) hi = max(hi, cand[c]);
        hi = wave_umax(hi);
        uint32_t r;
        if (n <= 256) {  // the candidate keys stay in registers for the whole bisection
          uint32_t c4[4];
#pragma unroll
          for (int q = 0; q < 4; q++) c4[q] = (uint32_t)(lane + 64 * q) < n ? cand[lane + 64 * q] : 0u;
          r = kth_key(lb, hi, K, [&](uint32_t x) {
            uint32_t c = 0;
#pragma unroll
            for (int q = 0; q < 4; q++) c += (uint32_t)__popcll(__ballot(c4[q] >= x));
            return c;
          });
        } else {
          r = kth_key(lb, hi, K, [&](uint32_t x) {
            uint32_t c = 0;
            for (uint32_t b = 0; b < n; b += 64) {
              const uint32_t i = b + (uint32_t)lane;
              c += (uint32_t)__popcll(__ballot(i < n && cand[i] >= x));
            }
            return c;
          });
        }
        if (lane == 0) s_thr = r;
      }
      __syncthreads();
      thr = s_thr;
    } else {
      // every wave counts its own keys per probe; the counts meet in LDS (two barriers per bit)
      uint32_t p = 0;
      for (int b = 31; b >= 0; b--) {
        const uint32_t x = p | (1u << b);
        uint32_t c = 0;
#pragma unroll
        for (int j = 0; j < kDrawPer; j++) c += (uint32_t)__popcll(__ballot(key[j] >= x));
        if (lane == 0) wsum[w] = c;
        __syncthreads();
        uint32_t tot = 0;
#pragma unroll
        for (int q = 0; q < kDrawWaves; q++) tot += wsum[q];
        __syncthreads();
        if (tot >= K) p = x;
      }
      thr = p;
    }
  }
  // Gumbel-max over the kept entries
  float best = -INFINITY;
  uint32_t bi = 0xffffffffu;
#pragma unroll
  for (int j = 0; j < kDrawPer; j++) {
    const int i = t + j * kDrawThreads;
    if (i >= V || key[j] < thr || xv[j] == -INFINITY) continue;
    const float g = gumbel(xv[j], (uint32_t)i, cnt, (uint32_t)sd, (uint32_t)(sd >> 32));
    if (g > best || (g == best && (uint32_t)i < bi)) { best = g; bi = (uint32_t)i; }  // NaN never wins
  }
  // wave: the largest value (as an order key; -0 made +0 so equal values have equal keys), then the lowest index
  // among the lanes holding it
  const uint32_t mk = order_key(best == 0.f ? 0.f : best);
  const uint32_t bk = wave_umax(mk);
  const uint32_t bidx = ~wave_umax(mk == bk ? ~bi : 0u);
  if (lane == 0) { wsum[w] = bk; wpick[w] = bidx; }
  __syncthreads();
  if (w != 0) return;
  const uint32_t pick = block_pick(wsum, wpick, lane);
  if (lane == 0) finish(pick);
}

}  // namespace

int sk_set_error(int rc, const char* msg) {
  snprintf(g_err, sizeof g_err, "%s", msg);
  return rc;
}

int sk_check_launch(hipError_t e, const char* where) {
  if (e == hipSuccess) return SK_OK;
  snprintf(g_err, sizeof g_err, "%s: %s", where, hipGetErrorString(e));
  return SK_ELAUNCH;
}

extern "C" const char* sk_version(void) { return "sokutou_amd 0.1.0 (gfx950)"; }
extern "C" const char* sk_last_error(void) { return g_err; }

extern "C" int sk_device_check(void) {
  int dev = 0;
  if (hipGetDevice(&dev) != hipSuccess) return sk_set_error(SK_EDEVICE, "sk_device_check: no HIP device");
  hipDeviceProp_t p;
  if (hipGetDeviceProperties(&p, dev) != hipSuccess) return sk_set_error(SK_EDEVICE, "sk_device_check: no properties");
  if (strncmp(p.gcnArchName, "gfx950", 6) != 0) {
    snprintf(g_err, sizeof g_err, "sk_device_check: device is %s, this build targets gfx950", p.gcnArchName);
    return SK_EDEVICE;
  }
  return SK_OK;
}

extern "C" int sk_rmsnorm(const float* h, const float* nw, float eps, float* out, int K, void* stream) {
  if (!h || !nw || !out || K <= 0) return sk_set_error(SK_EINVAL, "sk_rmsnorm: bad arguments");
  auto* k = K <= kNormThreads ? k_rmsnorm<1> : K <= 2 * kNormThreads ? k_rmsnorm<2> : k_rmsnorm<4>;
  hipLaunchKernelGGL(k, dim3(1), dim3(kNormThreads), 0, (hipStream_t)stream, h, nw, eps, out, K);
  return sk_check_launch(hipGetLastError(), "sk_rmsnorm");
}

extern "C" int sk_embed(const void* table, const int64_t* idx, float* out, int dim, int ct, void* stream) {
  if (!table || !idx || !out || dim <= 0) return sk_set_error(SK_EINVAL, "sk_embed: bad arguments");
  hipStream_t st = (hipStream_t)stream;
  const int blocks = (dim + 255) / 256 < 8 ? (dim + 255) / 256 : 8;
  if (ct == SK_CT_BF16)
    hipLaunchKernelGGL(k_embed<SK_CT_BF16>, dim3(blocks), dim3(256), 0, st, (const bf16_t*)table, idx, out, dim);
  else if (ct == SK_CT_F32)
    hipLaunchKernelGGL(k_embed<SK_CT_F32>, dim3(blocks), dim3(256), 0, st, (const float*)table, idx, out, dim);
  else
    return sk_set_error(SK_EINVAL, "sk_embed: bad element type");
  return sk_check_launch(hipGetLastError(), "sk_embed");
}

extern "C" int sk_talker_in(const uint64_t* tabs, const int64_t* codes, const void* pad, float* out, int dim, int G,
                            int ct, void* stream) {
  if (!tabs || !codes || !pad || !out || dim <= 0 || G <= 0) return sk_set_error(SK_EINVAL, "sk_talker_in: bad arguments");
  hipStream_t st = (hipStream_t)stream;
  const int blocks = (dim + 255) / 256 < 8 ? (dim + 255) / 256 : 8;
  if (ct == SK_CT_BF16)
    hipLaunchKernelGGL(k_talker_in<SK_CT_BF16>, dim3(blocks), dim3(256), 0, st, tabs, codes, (const bf16_t*)pad, out,
                       dim, G);
  else if (ct == SK_CT_F32)
    hipLaunchKernelGGL(k_talker_in<SK_CT_F32>, dim3(blocks), dim3(256), 0, st, tabs, codes, (const float*)pad, out, dim,
                       G);
  else
    return sk_set_error(SK_EINVAL, "sk_talker_in: bad element type");
  return sk_check_launch(hipGetLastError(), "sk_talker_in");
}

extern "C" int sk_sample(const float* logits, int V, float inv_temp, int top_k, int do_sample, uint8_t* seen,
                         float rep_pen, const uint8_t* suppress, int64_t* ngen, int min_new, int eos,
                         const uint64_t* seed, uint64_t* counter, int64_t* out, int talker, int64_t* id0, int64_t* pos,
                         void* stream) {
  if (!logits || !out || V <= 0 || V > SK_MAX_V) return sk_set_error(SK_EINVAL, "sk_sample: bad arguments (V <= 4096)");
  if (talker && !ngen) return sk_set_error(SK_EINVAL, "sk_sample: talker mode needs ngen");
  if (do_sample) {
    if (!seed || !counter) return sk_set_error(SK_EINVAL, "sk_sample: sampling needs the device seed and counter");
    if (!(inv_temp > 0.f) || inv_temp == INFINITY) return sk_set_error(SK_EINVAL, "sk_sample: temperature must be > 0");
    hipLaunchKernelGGL(k_sample_draw, dim3(1), dim3(kDrawThreads), 0, (hipStream_t)stream, logits, V, inv_temp, top_k,
                       seen, rep_pen, suppress, ngen, min_new, eos, seed, counter, out, talker, id0, pos);
    return sk_check_launch(hipGetLastError(), "sk_sample");
  }
  hipLaunchKernelGGL(k_sample_greedy, dim3(1), dim3(kSampleThreads), 0, (hipStream_t)stream, logits, V, seen, rep_pen,
                     suppress, ngen, min_new, eos, out, talker, id0, pos);
  return sk_check_launch(hipGetLastError(), "sk_sample");
}
