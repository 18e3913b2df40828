// M=1 weight-only GEMV for the talker projections (qkv, o, gate/up, down, codec head): sk_rms_gemv and sk_gemv,
// replacing the reference's `rms_gemv` / `gemv` (qwen3/kernels.py:255-310; math of gemv_core 143-253).
//
// Design for CDNA4 (wave64, 256 CUs). The matrices are small (2 to 50 MB): what bounds a call is its launch (1.8 us) and
// one memory round trip, then the bytes. So every load goes out at the top and nothing is exchanged but one sum:
//  * A workgroup of NW waves owns 4 RG consecutive rows and splits K over its waves in steps of 256 inputs. A wave is four
//    16-lane groups; group g takes rows r0 + g + 4 k (k < RG), its lane q the 16-byte chunks q, q + 16, ... of a step.
//    A row's share is a 16-lane DPP sum; the waves' shares meet in LDS behind the only barrier. Small projections (1024
//    rows) launch 256 workgroups of 4 or 8 waves and fill the chip.
//  * Each wave stages its own steps of the input (one float4 per lane and step) in LDS that no other wave uses, so without
//    a barrier, in slots that leave both the writes and the reads (16 chunks, one quarter; the four groups the same)
//    without bank conflicts. The fused RMSNorm's sum of squares comes from the same registers.
//  * Per call, HBM-cold, against one wave per workgroup with the whole input staged first in a loop: int8 2048 x 6144
//    10.6 -> 4.5 us, 2048 x 2048 4.9 -> 3.2, 12288 x 2048 9.4 -> 6.5 (25 MB, 5.4 TB/s behind the launch), 4096 x 1024
//    4.1 -> 3.1, 1024 x 3072 5.7 -> 3.2; bf16 12288 x 2048 12.8 -> 9.7, 2048 x 6144 12.3 -> 5.9; f32 2048 x 6144
//    16.3 -> 9.5, 12288 x 2048 20.5 -> 16.5 (101 MB, 6.9 TB/s).
//  * Dequantisation in registers: int8 -> fp32 per byte, fp32 FMA; i8row applies the bf16 row scale after the row
//    sum, i8g32 the fp16 scale of each 32-element group per 16-element chunk; the RMSNorm factor multiplies the
//    result (the reference's order, qwen3/kernels.py:180-186, 224).
#include "common.h"
#include "internal.h"

namespace {

constexpr int kGroups = 4;  // 16-lane row groups per wave
constexpr int kStep = 256;  // inputs a wave takes at a time: one float4 per lane

template <int POL>
__device__ __forceinline__ uint4 ldw(const uint4* p) {
  if constexpr (POL == 1) return ld_stream(p);
  else return *p;
}

// Dot of one 16-byte weight chunk with its E inputs, held as E / 4 float4 quarters.
template <int WD>
__device__ __forceinline__ float chunk_dot4(uint4 v, const float4* xv) {
  if constexpr (WD == SK_WD_I8ROW || WD == SK_WD_I8G32) {
    const uint32_t w[4] = {v.x, v.y, v.z, v.w};
    float a = 0.f;
#pragma unroll
    for (int j = 0; j < 4; j++) {
      a = __builtin_fmaf((float)(int8_t)(w[j]), xv[j].x, a);
      a = __builtin_fmaf((float)(int8_t)(w[j] >> 8), xv[j].y, a);
      a = __builtin_fmaf((float)(int8_t)(w[j] >> 16), xv[j].z, a);
      a = __builtin_fmaf((float)(int8_t)(w[j] >> 24), xv[j].w, a);
    }
    return a;
  } else if constexpr (WD == SK_WD_BF16) {
    float a = bf2f(v.x & 0xffffu) * xv[0].x;
    a = __builtin_fmaf(bf2f(v.x >> 16), xv[0].y, a);
    a = __builtin_fmaf(bf2f(v.y & 0xffffu), xv[0].z, a);
    a = __builtin_fmaf(bf2f(v.y >> 16), xv[0].w, a);
    a = __builtin_fmaf(bf2f(v.z & 0xffffu), xv[1].x, a);
    a = __builtin_fmaf(bf2f(v.z >> 16), xv[1].y, a);
    a = __builtin_fmaf(bf2f(v.w & 0xffffu), xv[1].z, a);
    a = __builtin_fmaf(bf2f(v.w >> 16), xv[1].w, a);
    return a;
  } else {
    float a = __uint_as_float(v.x) * xv[0].x;
    a = __builtin_fmaf(__uint_as_float(v.y), xv[0].y, a);
    a = __builtin_fmaf(__uint_as_float(v.z), xv[0].z, a);
    a = __builtin_fmaf(__uint_as_float(v.w), xv[0].w, a);
    return a;
  }
}

// mode: 0 write, 1 accumulate into out, 2 SwiGLU over interleaved gate/up rows (out[row / 2]).
template <int WD, int RG, int POL, int NW, int NI>
__global__ __launch_bounds__(SK_WAVE * NW) void k_gemv(const float* __restrict__ x, const float* __restrict__ nw, float eps,
                                                       const uint8_t* __restrict__ W, const uint16_t* __restrict__ S,
                                                       const float* __restrict__ bias, float* __restrict__ out, int N, int K,
                                                       int mode) {
  constexpr int E = WdInfo<WD>::E, Q = E / 4;  // elements per 16-byte chunk, float4 quarters per chunk
  constexpr int CH = kStep / E / 16;           // chunks per lane, row and step
  constexpr int R = kGroups * RG;              // rows of the workgroup
  __shared__ float4 xs[NW][NI][SK_WAVE];       // each wave's own steps of the input
  __shared__ float red[NW][R];
  __shared__ float ssw[NW];
  const int tid = threadIdx.x, w = __builtin_amdgcn_readfirstlane(tid >> 6), lane = tid & 63, grp = lane >> 4, q = lane & 15;
  const int nsteps = K / kStep;
  const size_t row_bytes = (size_t)K * WdInfo<WD>::BYTES;
  const int r0 = blockIdx.x * R;
  int rows[RG];
  const uint4* wp[RG];
#pragma unroll
  for (int k = 0; k < RG; k++) {
    rows[k] = min(r0 + grp + kGroups * k, N - 1);
    wp[k] = (const uint4*)(W + (size_t)rows[k] * row_bytes) + q;
  }
  // float4 `lane` of a step is quarter j of chunk 16 i + qc; it sits at slot 16 (Q i + j) + (qc rotated by 16 j / Q), so that the
  // lanes of a write and those of a read (one j, every qc) touch distinct banks
  const int sj = lane % Q, sc = lane / Q, slot = ((sc >> 4) * Q + sj) * 16 + (((sc & 15) + 16 / Q * sj) & 15);
  // what the epilogue needs of this thread's row
  const int row = r0 + tid;
  const bool own = tid < R && row < N;
  const int rc = min(r0 + min(lane, R - 1), N - 1);
  uint32_t rs = 0;
  float bv = 0.f, ov = 0.f;
  if constexpr (WD == SK_WD_I8ROW) rs = gload(S + rc);
  if (bias) bv = gload(bias + rc);
  if (mode == 1) ov = gload(out + rc);
  float acc[RG], ss = 0.f;
#pragma unroll
  for (int k = 0; k < RG; k++) acc[k] = 0.f;
  auto pass = [&](int u0) __attribute__((always_inline)) {  // steps u0, u0 + NW, ... (NI of them)
    float4 xv[NI], nv[NI];
    uint4 wv[NI][CH][RG];
    uint16_t sv[NI][CH][RG];
#pragma unroll
    for (int i = 0; i < NI; i++) {
      const int u = u0 + NW * i < nsteps ? u0 + NW * i : u0;  // a step past the end loads the first again
      xv[i] = *(const float4*)(x + u * kStep + 4 * lane);
      if (nw) nv[i] = *(const float4*)(nw + u * kStep + 4 * lane);
    }
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int i = 0; i < NI; i++) {
      const int u = u0 + NW * i < nsteps ? u0 + NW * i : u0;
#pragma unroll
      for (int c = 0; c < CH; c++)
#pragma unroll
        for (int k = 0; k < RG; k++) {
          const int ch = (u * CH + c) * 16;
          wv[i][c][k] = ldw<POL>(wp[k] + ch);
          if constexpr (WD == SK_WD_I8G32) sv[i][c][k] = gload(S + (size_t)rows[k] * (K >> 5) + ((ch + q) >> 1));
        }
    }
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int i = 0; i < NI; i++) {
      float4 a = xv[i];
      if (nw) {
        if (u0 + NW * i < nsteps) ss += a.x * a.x + a.y * a.y + a.z * a.z + a.w * a.w;
        a = make_float4(a.x * nv[i].x, a.y * nv[i].y, a.z * nv[i].z, a.w * nv[i].w);
      }
      xs[w][i][slot] = a;
    }
    wave_sync();
#pragma unroll
    for (int i = 0; i < NI; i++) {
      if (u0 + NW * i >= nsteps) break;  // uniform over the wave
#pragma unroll
      for (int c = 0; c < CH; c++) {
        float4 xq[Q];
#pragma unroll
        for (int j = 0; j < Q; j++) xq[j] = xs[w][i][(c * Q + j) * 16 + ((q + 16 / Q * j) & 15)];
#pragma unroll
        for (int k = 0; k < RG; k++) {
          const float d = chunk_dot4<WD>(wv[i][c][k], xq);
          if constexpr (WD == SK_WD_I8G32) acc[k] = __builtin_fmaf(h2f(sv[i][c][k]), d, acc[k]);
          else acc[k] += d;
        }
      }
    }
    wave_sync();
  };
  // the first pass outside the loop: before a loop's loads the compiler waits for every earlier one
  if (w < nsteps) pass(w);
  for (int u0 = w + NW * NI; u0 < nsteps; u0 += NW * NI) pass(u0);
  if constexpr (WD == SK_WD_I8ROW) asm volatile("" : "+v"(rs));  // its conversion (so the wait for it) stays behind the loop
#pragma unroll
  for (int k = 0; k < RG; k++) {
    const float y = row16_sum(acc[k]);
    if (q == 0) red[w][grp + kGroups * k] = y;
  }
  if (nw) {
    ss = wave_sum(ss);
    if (lane == 0) ssw[w] = ss;
  }
  __syncthreads();
  if (w != 0) return;
  float y = 0.f;
  if (tid < R) {
    y = red[0][tid];
#pragma unroll
    for (int v = 1; v < NW; v++) y += red[v][tid];
  }
  if constexpr (WD == SK_WD_I8ROW) y *= bf2f(rs);
  if (nw) {
    float s = ssw[0];
#pragma unroll
    for (int v = 1; v < NW; v++) s += ssw[v];
    y *= rsqrtf(s / K + eps);
  }
  if (mode == 2) {
    const float up = dpp<0xB1>(y);  // thread t ^ 1: the up row next to this gate row
    if (own && !(tid & 1) && row + 1 < N) out[row >> 1] = silu_mul(y, up);
  } else if (own) {
    if (bias) y += bv;
    if (mode == 1) y += ov;
    out[row] = y;
  }
}

template <int WD, int RG, int POL, int NW, int NI>
hipError_t launch_one(const float* x, const float* nw, float eps, const void* W, const uint16_t* S, const float* bias,
                      float* out, int N, int K, int mode, hipStream_t st) {
  dim3 grid((N + kGroups * RG - 1) / (kGroups * RG));
  hipLaunchKernelGGL((k_gemv<WD, RG, POL, NW, NI>), grid, dim3(SK_WAVE * NW), 0, st, x, nw, eps,
                     (const uint8_t*)W, S, bias, out, N, K, mode);
  return hipGetLastError();
}

// NW waves, RG rows per 16-lane group, NI steps in flight per wave; us per call, HBM-cold, in a graph:
//   * eight waves from K = 2048, four below (1024 x 2048 int8 2.9 against 3.0; 3072 x 1024 2.8 either way).
//   * All steps of a wave at once up to 3 (int8) or 2 (bf16): 2048 x 6144 int8 4.5 with 3, 4.7 with 1; 1024 x 3072 int8 3.2
//     with 2, 3.5 with 1. More bytes a step need fewer in flight: bf16 at 6144 5.9 with 1, 6.2 with 3; f32 9.5 either way.
//   * Rows: two per group from 2048 rows in int8 (4096 x 2048 3.8 against 4.1) and from 4096 in bf16 (4096 x 2048 5.1
//     against 5.4; 2048 x 6144 6.3 with two, 6.2 with one); four from 8192 in int8, whose input costs as much LDS and cache
//     traffic as eight rows' weights (12288 x 2048 6.5 against 6.9; bf16 9.7 with two, 10.9 with four). f32 rows are bytes
//     enough one at a time (12288 x 2048 16.5 against 17.2 with two).
template <int WD, int POL, int RG>
hipError_t launch_rg(const float* x, const float* nw, float eps, const void* W, const uint16_t* S, const float* bias,
                     float* out, int N, int K, int mode, hipStream_t st) {
  constexpr int kCap = WdInfo<WD>::BYTES == 1 ? 3 : WdInfo<WD>::BYTES == 2 ? 2 : 1;
  if (K < 2048) return launch_one<WD, RG, POL, 4, 1>(x, nw, eps, W, S, bias, out, N, K, mode, st);
  const int ni = (K / kStep + 7) / 8;
  if constexpr (kCap >= 2)
    if (ni == 2) return launch_one<WD, RG, POL, 8, 2>(x, nw, eps, W, S, bias, out, N, K, mode, st);
  if constexpr (kCap >= 3)
    if (ni == 3) return launch_one<WD, RG, POL, 8, 3>(x, nw, eps, W, S, bias, out, N, K, mode, st);
  return launch_one<WD, RG, POL, 8, 1>(x, nw, eps, W, S, bias, out, N, K, mode, st);
}

template <int WD, int POL>
hipError_t launch_wd(const float* x, const float* nw, float eps, const void* W, const uint16_t* S, const float* bias,
                     float* out, int N, int K, int mode, hipStream_t st) {
  if constexpr (WdInfo<WD>::BYTES == 1)
    if (N >= 8192) return launch_rg<WD, POL, 4>(x, nw, eps, W, S, bias, out, N, K, mode, st);
  if constexpr (WdInfo<WD>::BYTES <= 2)
    if (N >= (WdInfo<WD>::BYTES == 1 ? 2048 : 4096)) return launch_rg<WD, POL, 2>(x, nw, eps, W, S, bias, out, N, K, mode, st);
  return launch_rg<WD, POL, 1>(x, nw, eps, W, S, bias, out, N, K, mode, st);
}

template <int POL>
hipError_t launch_pol(const float* x, const float* nw, float eps, const void* W, const uint16_t* S, const float* bias,
                      float* out, int N, int K, int mode, int wd, hipStream_t st) {
  switch (wd) {
    case SK_WD_I8ROW: return launch_wd<SK_WD_I8ROW, POL>(x, nw, eps, W, S, bias, out, N, K, mode, st);
    case SK_WD_I8G32: return launch_wd<SK_WD_I8G32, POL>(x, nw, eps, W, S, bias, out, N, K, mode, st);
    case SK_WD_BF16: return launch_wd<SK_WD_BF16, POL>(x, nw, eps, W, S, bias, out, N, K, mode, st);
    case SK_WD_F32: return launch_wd<SK_WD_F32, POL>(x, nw, eps, W, S, bias, out, N, K, mode, st);
  }
  return hipErrorInvalidValue;
}

int check_shape(int N, int K, int wd, const void* S) {
  if (N <= 0 || K <= 0) return SK_EINVAL;
  if (K % 512 != 0) return SK_EINVAL;  // same constraint as the reference's _Lin (qwen3/kernels.py:433)
  if (K > SK_MAX_K) return SK_EINVAL;
  if (wd < 0 || wd > SK_WD_F32) return SK_EINVAL;
  if ((wd == SK_WD_I8ROW || wd == SK_WD_I8G32) && !S) return SK_EINVAL;
  return SK_OK;
}

}  // namespace

extern "C" int sk_rms_gemv(const float* h, const float* nw, float eps, const void* W, const uint16_t* S, float* out,
                           int N, int K, int swiglu, int wd, int policy, void* stream) {
  int rc = check_shape(N, K, wd, S);
  if (rc) return sk_set_error(rc, "sk_rms_gemv: bad shape or format");
  if (!h || !nw || !W || !out) return sk_set_error(SK_EINVAL, "sk_rms_gemv: null pointer");
  if (swiglu && (N & 1)) return sk_set_error(SK_EINVAL, "sk_rms_gemv: swiglu needs an even row count");
  hipStream_t st = (hipStream_t)stream;
  hipError_t e = policy ? launch_pol<1>(h, nw, eps, W, S, nullptr, out, N, K, swiglu ? 2 : 0, wd, st)
                        : launch_pol<0>(h, nw, eps, W, S, nullptr, out, N, K, swiglu ? 2 : 0, wd, st);
  return sk_check_launch(e, "sk_rms_gemv");
}

extern "C" int sk_gemv(const float* x, const void* W, const uint16_t* S, const float* bias, float* out, int N, int K,
                       int accumulate, int wd, int policy, void* stream) {
  int rc = check_shape(N, K, wd, S);
  if (rc) return sk_set_error(rc, "sk_gemv: bad shape or format");
  if (!x || !W || !out) return sk_set_error(SK_EINVAL, "sk_gemv: null pointer");
  hipStream_t st = (hipStream_t)stream;
  hipError_t e = policy ? launch_pol<1>(x, nullptr, 0.f, W, S, bias, out, N, K, accumulate ? 1 : 0, wd, st)
                        : launch_pol<0>(x, nullptr, 0.f, W, S, bias, out, N, K, accumulate ? 1 : 0, wd, st);
  return sk_check_launch(e, "sk_gemv");
}
