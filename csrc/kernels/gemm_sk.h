// Shared parts of the two split-K tiled GEMMs (gemm_sk.hip, gemm_pipe.hip): launch
// parameters, the in-launch reduction of a tile's K chunks, and the epilogues.
#pragma once
#include "common.h"

#define SK_BK 64

enum { SK_BF16 = 0, SK_SWIGLU = 1, SK_RESID = 2, SK_GELU = 3 };   // (SK_GELU: the pipelined tiles' SK_BF16 with act 1)

struct GemmSkParams {
  const void* x; long long ldx;   // [M, K] bf16 rows
  const void* w;                  // [N, K] bf16 row-major (SwiGLU: gate rows [0, N/2), up [N/2, N))
  int M, N, K, S;                 // S: K chunks per output tile
  int epi, act;                   // act (SK_BF16): 0 none, 1 GELU (erf) after the bias
  const float* bias;              // [N] f32 or null (SK_BF16, SK_RESID)
  void* y; long long ldy;         // bf16 output (SK_RESID: the residual, updated in place)
  float* ws;                      // S > 1: [tiles][S][BM * BN] f32 partials
  int* counters;                  // S > 1: [tiles] tickets, zero on entry (left zero)
  int layout;
  int ahead_wgs;                  // workgroups behind the tiles' that only touch what follows (pipelined tiles)
  int hurry;                      // looks at a tile's word that a K chunk leaves out before it gives its share up (0, but in tests)
};
// A call: what the kernels without touching workgroups have no use for stands behind their arguments, as
// a third cache line of them is another miss before the first load (0.2 us of 12 at 80 x 11264 x 2048).
struct GemmSkCall : GemmSkParams {
  const void* ahead[2]; long long ahead_bytes[2];   // weights of later launches, null or empty: none
};

// s_waitcnt vmcnt(N) with expcnt / lgkmcnt at their maxima (gfx9 encoding:
// vmcnt[3:0] in bits 3:0, vmcnt[5:4] in bits 15:14)
template <int N>
__device__ __forceinline__ void sk_wait_vm() {
  static_assert(N >= 0 && N < 64, "vmcnt range");
  __builtin_amdgcn_s_waitcnt((N & 15) | ((N >> 4) << 14) | (7 << 4) | (15 << 8));
}

// GELU as (v + |v|) / 2 - |v| Phi(-|v|), no cancellation in the negative tail, with log2 Phi(-a) / 2
// as a polynomial of degree 12 and its power of two squared: one transcendental instruction, less issue
// time than the rational form of erfc (Abramowitz and Stegun 7.1.26) with its reciprocal - with one wave
// per SIMD nothing hides an epilogue's arithmetic. Fitted on [0, 14.2], where Phi leaves the f32 range (it
// falls without end beyond), tightest near 0; the square keeps the values that the exponential's
// own range (its results stop at 2^-126) would cut off from -12.95 on. Its argument is the f32 sum.
// Relative error against 64 bits on the GPU, erfc's form and this one, root mean square before the
// rounding to bf16: 0.3 to 1 8.4e-8, 4.4e-8; 0 to 0.3 1.4e-7, 6.9e-8; -0.3 to 0 1.8e-7, 8.4e-8; -1 to
// -0.3 2.2e-7, 9.2e-8; -2 to -1 1.2e-6, 1.9e-7; -4 to -3 2.5e-4, 1.9e-6; -6 to -5 2.6e-3, 2.4e-5; -8 to
// -7 8.4e-3, 3.0e-4; -10 to -9 0.017, 0.0021; -12 to -11 0.028, 0.0026; -13.2 to -12.9 0.037, 0.0032 (values
// of 1e-37). The bf16 result is within half an ulp (0.0039) from -5 on, 0.0043 from -8, 0.0098 from -13.2.
// Four values at a time, so that four chains of the polynomial run side by side on one set of
// constants.
__device__ __forceinline__ void sk_gelu4(float* v) {
  constexpr float C[] = {8.958461195e-10f, -2.714527447e-08f, 4.635971322e-07f, -4.886001534e-06f, 3.206257679e-05f, -1.132769830e-04f,
                         -6.210878200e-05f, 3.555311821e-03f, -2.627918683e-02f, -2.295900732e-01f, -5.755547285e-01f, -4.999999404e-01f};
  float e[4];
#pragma unroll
  for (int r = 0; r < 4; ++r) e[r] = -1.272199707e-11f;
#pragma unroll
  for (int k = 0; k < 12; ++k)
#pragma unroll
    for (int r = 0; r < 4; ++r) e[r] = e[r] * fabsf(v[r]) + C[k];
  // |v| once more, held below infinity on the positive side only: -inf is inf * 0, as with erf
#pragma unroll
  for (int r = 0; r < 4; ++r) {
    const float x = __builtin_amdgcn_exp2f(e[r]);
    v[r] = fmaxf(v[r], 0.f) - fmaxf(-v[r], fminf(v[r], 1e30f)) * x * x;
  }
}

__device__ __forceinline__ float sk_swiglu(float g, float u) {   // silu(g) u
  return g * __builtin_amdgcn_rcpf(1.f + __builtin_amdgcn_exp2f(g * -1.4426950408889634f)) * u;
}

// Publish this chunk's partial; the tile's last arriver gets the sum of all S in
// `acc` and returns true, the others return false.
template <int NW, int FN, int FM>
__device__ __forceinline__ bool sk_reduce(const GemmSkParams& p, float4v (&acc)[FN][FM], int tile, int s,
                                          int wave, int lane, int* flag) {
  const int S = p.S;
  constexpr int PER_WAVE = FN * FM * 256;      // floats per wave partial (16 B per lane per fragment)
  float* mine = p.ws + (((size_t)tile * S + s) * NW + wave) * PER_WAVE;
#pragma unroll
  for (int i = 0; i < FN; ++i)
#pragma unroll
    for (int j = 0; j < FM; ++j)
      *reinterpret_cast<float4v*>(mine + ((i * FM + j) * 64 + lane) * 4) = acc[i][j];
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
  __syncthreads();
  if (threadIdx.x == 0) {
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "agent");
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    const int t = __hip_atomic_fetch_add(p.counters + tile * TICKET, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    const int last = t == S - 1;
    if (last) __hip_atomic_store(p.counters + tile * TICKET, 0, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    *flag = last;
  }
  __syncthreads();
  if (!*flag) return false;
  if (threadIdx.x == 0) __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "agent");
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
  __syncthreads();
  // fixed chunk order 0..S-1, every partial (this workgroup's own included)
  // read back from the workspace: the sum does not depend on who arrived
  // last, and needs no second accumulator array (the 256 x 256 tile has no
  // registers for one). Loads go in groups of up to 16 fragments.
  constexpr int GI = FM >= 16 ? 1 : (16 / FM < FN ? 16 / FM : FN);
  static_assert(FN % GI == 0, "fragment groups");
  for (int c = 0; c < S; ++c) {
    const float* theirs = p.ws + (((size_t)tile * S + c) * NW + wave) * PER_WAVE;
#pragma unroll
    for (int i0 = 0; i0 < FN; i0 += GI) {
      float4v v[GI][FM];
#pragma unroll
      for (int i = 0; i < GI; ++i)
#pragma unroll
        for (int j = 0; j < FM; ++j)
          v[i][j] = *reinterpret_cast<const float4v*>(theirs + (((i0 + i) * FM + j) * 64 + lane) * 4);
#pragma unroll
      for (int i = 0; i < GI; ++i)
#pragma unroll
        for (int j = 0; j < FM; ++j) acc[i0 + i][j] = c == 0 ? v[i][j] : acc[i0 + i][j] + v[i][j];
    }
  }
  return true;
}

// acc[i][j] = C[n = nw + 16 i + 4 fq + r][m = mw + 16 j + fr] of one wave; fw: its first
// SwiGLU output feature.
template <int EPI, int FN, int FM>
__device__ __forceinline__ void sk_epilogue(const GemmSkParams& p, float4v (&acc)[FN][FM], int nw, int fw,
                                            int mw, int fr, int fq) {
  const int M = p.M;
  bf16_t* Y = reinterpret_cast<bf16_t*>(p.y);
  if constexpr (EPI == SK_SWIGLU) {
#pragma unroll
    for (int j = 0; j < FM; ++j) {
      const int m = mw + 16 * j + fr;
      if (m >= M) continue;
#pragma unroll
      for (int i = 0; i < FN / 2; ++i) {
        const int f = fw + 16 * i + 4 * fq;
        float o[4];
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          o[r] = sk_swiglu(acc[i][j][r], acc[i + FN / 2][j][r]);
        }
        *reinterpret_cast<uint2*>(Y + (size_t)m * p.ldy + f) =
            make_uint2(pack_bf16x2(o[0], o[1]), pack_bf16x2(o[2], o[3]));
      }
      __builtin_amdgcn_sched_barrier(0);   // a row block's accumulators at a time
    }
  } else if constexpr (EPI == SK_RESID) {
    float4 bv[FN];
#pragma unroll
    for (int i = 0; i < FN; ++i) {
      const int n = nw + 16 * i + 4 * fq;
      bv[i] = p.bias ? *reinterpret_cast<const float4*>(p.bias + n) : make_float4(0.f, 0.f, 0.f, 0.f);
    }
#pragma unroll
    for (int j = 0; j < FM; ++j) {
      const int m = mw + 16 * j + fr;
      if (m >= M) continue;
#pragma unroll
      for (int i = 0; i < FN; ++i) {
        const int n = nw + 16 * i + 4 * fq;
        uint2* yp = reinterpret_cast<uint2*>(Y + (size_t)m * p.ldy + n);
        const uint2 rv = *yp;
        const float o0 = bf2f(rv.x & 0xffff) + (acc[i][j][0] + bv[i].x);
        const float o1 = bf2f(rv.x >> 16) + (acc[i][j][1] + bv[i].y);
        const float o2 = bf2f(rv.y & 0xffff) + (acc[i][j][2] + bv[i].z);
        const float o3 = bf2f(rv.y >> 16) + (acc[i][j][3] + bv[i].w);
        *yp = make_uint2(pack_bf16x2(o0, o1), pack_bf16x2(o2, o3));
      }
      __builtin_amdgcn_sched_barrier(0);
    }
  } else {
    float4 bv[FN];
#pragma unroll
    for (int i = 0; i < FN; ++i) {
      const int n = nw + 16 * i + 4 * fq;
      bv[i] = p.bias ? *reinterpret_cast<const float4*>(p.bias + n) : make_float4(0.f, 0.f, 0.f, 0.f);
    }
#pragma unroll
    for (int j = 0; j < FM; ++j) {
      const int m = mw + 16 * j + fr;
      if (m >= M) continue;
#pragma unroll
      for (int i = 0; i < FN; ++i) {
        const int n = nw + 16 * i + 4 * fq;
        float o[4] = {acc[i][j][0] + bv[i].x, acc[i][j][1] + bv[i].y, acc[i][j][2] + bv[i].z,
                      acc[i][j][3] + bv[i].w};
        if (p.act == 1) sk_gelu4(o);
        *reinterpret_cast<uint2*>(Y + (size_t)m * p.ldy + n) =
            make_uint2(pack_bf16x2(o[0], o[1]), pack_bf16x2(o[2], o[3]));
      }
      __builtin_amdgcn_sched_barrier(0);
    }
  }
}

