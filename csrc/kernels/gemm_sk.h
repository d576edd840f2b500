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
  int* counters;                  // S > 1: [tiles] ints, zero on entry (left zero)
  int layout;
  int ahead_wgs;                  // workgroups behind the tiles' that only touch what follows (pipelined tiles)
  const void* ahead[2]; long long ahead_bytes[2];   // weights of later launches, null or empty: none
};

// s_waitcnt vmcnt(N) with expcnt / lgkmcnt at their maxima (gfx9 encoding:
// vmcnt[3:0] in bits 3:0, vmcnt[5:4] in bits 15:14)
template <int N>
__device__ __forceinline__ void sk_wait_vm() {
  static_assert(N >= 0 && N < 64, "vmcnt range");
  __builtin_amdgcn_s_waitcnt((N & 15) | ((N >> 4) << 14) | (7 << 4) | (15 << 8));
}

// GELU as (v + |v|) / 2 - |v| Phi(-|v|), no cancellation in the negative tail, with log2 Phi(-a) as
// a polynomial of degree 10 fitted on [0, 6.5] (largest error 6.3e-7; it falls without end beyond):
// one transcendental instruction, and a quarter less issue time than the rational form of erfc
// (Abramowitz and Stegun 7.1.26) with its reciprocal - with one wave per SIMD nothing hides an
// epilogue's arithmetic. Its argument is the f32 sum. Largest relative error of the bf16 result, erfc's
// form and this one: -7 to -6 0.0102, 0.0039; -6 to -5 0.0074, 0.0039; -5 to -4 0.0054, 0.0039; -4 to
// -3 0.0042, 0.0039; from -3 on 0.0039 both (rounding the result alone: 0.0039).
// Four values at a time, so that four chains of the polynomial run side by side on one set of
// constants.
__device__ __forceinline__ void sk_gelu4(float* v) {
  constexpr float C[] = {3.011999468e-07f, -4.531088052e-06f, 3.564885992e-05f, -1.246613683e-04f, -3.609243722e-04f,
                         7.453413680e-03f, -5.284556746e-02f, -4.590584338e-01f, -1.151129246f, -9.999993443e-01f};
  float e[4];
#pragma unroll
  for (int r = 0; r < 4; ++r) e[r] = -8.442756716e-09f;
#pragma unroll
  for (int k = 0; k < 10; ++k)
#pragma unroll
    for (int r = 0; r < 4; ++r) e[r] = e[r] * fabsf(v[r]) + C[k];
  // |v| once more, held below infinity on the positive side only: -inf is inf * 0, as with erf
#pragma unroll
  for (int r = 0; r < 4; ++r)
    v[r] = fmaxf(v[r], 0.f) - fmaxf(-v[r], fminf(v[r], 1e30f)) * __builtin_amdgcn_exp2f(e[r]);
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
    const int t = __hip_atomic_fetch_add(p.counters + tile, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    const int last = t == S - 1;
    if (last) __hip_atomic_store(p.counters + tile, 0, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
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

