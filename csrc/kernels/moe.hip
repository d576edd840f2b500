// Mixture-of-experts feed-forward: grouped top-k router, device-side grouping
// of tokens by expert, grouped expert GEMMs, weighted combine.
//
// moe_route_lanes_kernel (16 to 64 lanes per token, up to 64 router outputs) and
//   moe_route_kernel (a wave and LDS): scores = softmax(z) over all router
//   outputs; choice = score + correction; router outputs form `groups` equal
//   groups of neighbours, a group ranks by its best choice score and only the
//   `keep` best groups stay eligible (the others count as -inf); the `top`
//   best eligible choices are taken; the weights are the plain scores. Mode 1:
//   the choice is by the logit itself (+ bias) and the weights are the softmax
//   over the chosen logits only. Mode 2: scores = sigmoid(z) instead of the
//   softmax. With `grank` n > 1 a group ranks by the sum of its n best choice
//   scores. With `renorm` the chosen weights are divided by their sum (+ 1e-20);
//   `wscale` multiplies them.
// moe_pipe.hip: the bf16 grouped products wherever rows are whole 16-byte pieces; the
//   forms here serve f32 and other sizes.
// moe_plan_kernel (one workgroup): (token, k) pairs bucketed by expert without
//   a host round trip: offsets[E + 2], perm[P] (pair ids in expert order; the
//   identity bucket E last), pos[P] (where each pair sits).
// moe_grouped_gemm_kernel: C = A . W_e^T per expert segment, 64 x 64 tiles,
//   f32 accumulation over K in ascending order for every output element (so a
//   pair's result does not depend on which other pairs share its tile). Mode
//   1 gathers A rows by token and applies the SwiGLU epilogue to the (gate,
//   up) weight row pairs; mode 2 gathers A rows by token and squares the relu
//   of a single (up) weight set; mode 3 is mode 1 with the clamped gate
//   g sigmoid(1.702 g) (u + 1), g = min(gate, limit), u = clamp(up, +-limit);
//   mode 0 reads the sorted activation rows.
// moe_combine_kernel: out[t] = sum_k weight * (expert output | the input
//   itself for an identity expert), f32.
#include "seqmix.h"

#define MOE_MAX_E 1024

template <int LANES> __device__ __forceinline__ void lanes_argmax(float& v, int& i) {
#pragma unroll
  for (int o = LANES / 2; o > 0; o >>= 1) {
    const float ov = __shfl_xor(v, o, LANES);
    const int oi = __shfl_xor(i, o, LANES);
    if (ov > v || (ov == v && oi < i)) { v = ov; i = oi; }
  }
}

__global__ __launch_bounds__(64) void moe_route_kernel(
    const float* __restrict__ z, const float* __restrict__ corr, const float* __restrict__ bias,
    int mode, int E, int G, int keep, int grank, int top, int renorm, float wscale,
    int* __restrict__ idx, float* __restrict__ wt) {
  const int top_softmax = mode == 1;
  __shared__ float sc[MOE_MAX_E], ch[MOE_MAX_E], gs[MOE_MAX_E];
  const int t = blockIdx.x, lane = threadIdx.x;
  const float* zr = z + (size_t)t * E;
  float mx = -INFINITY;
  for (int e = lane; e < E; e += 64) {
    const float v = bias ? zr[e] + bias[e] : zr[e];
    gs[e] = v;                                  // the logit with its bias
    mx = fmaxf(mx, v);
  }
  mx = wave_max(mx);
  float sum = 0.f;
  for (int e = lane; e < E; e += 64) {
    const float v = mode == 2 ? sigmoid_f(gs[e]) : expf(gs[e] - mx);
    sc[e] = v;
    sum += v;
  }
  sum = wave_sum(sum);
  const float inv = mode == 2 ? 1.f : 1.f / sum;
  for (int e = lane; e < E; e += 64) {
    if (top_softmax) { ch[e] = gs[e]; continue; }      // scores stay unnormalised: see below
    const float s = sc[e] * inv;
    sc[e] = s;
    ch[e] = corr ? s + corr[e] : s;
  }
  __syncthreads();
  if (G > 1 && keep < G) {
    const int per = E / G;
    for (int g = lane; g < G; g += 64) {
      float b = -INFINITY;
      if (grank <= 1) {
        for (int j = 0; j < per; ++j) b = fmaxf(b, ch[g * per + j]);
      } else {
        // the sum of the group's n best: n passes, each taking the largest entry
        // below the previous one (by value, then index)
        float pv = INFINITY;
        int pi = -1;
        b = 0.f;
        for (int n = 0; n < min(grank, per); ++n) {
          float bv = -INFINITY;
          int bi = -1;
          for (int j = 0; j < per; ++j) {
            const float v = ch[g * per + j];
            const bool below = v < pv || (v == pv && j > pi);
            if (below && (bi < 0 || v > bv)) { bv = v; bi = j; }
          }
          if (bi < 0) break;
          b += bv;
          pv = bv;
          pi = bi;
        }
      }
      gs[g] = b;
    }
    __syncthreads();
    // the `keep` best groups are marked with +inf, then the rest is masked
    for (int k = 0; k < keep; ++k) {
      float bv = -INFINITY;
      int bi = 0x7fffffff;
      for (int g = lane; g < G; g += 64) {
        const float v = gs[g];
        if (v != INFINITY && (v > bv || bi == 0x7fffffff)) { bv = v; bi = g; }
      }
      lanes_argmax<64>(bv, bi);
      if (lane == 0 && bi < G) gs[bi] = INFINITY;
      __syncthreads();
    }
    for (int e = lane; e < E; e += 64)
      if (gs[e / per] != INFINITY) ch[e] = -INFINITY;
    __syncthreads();
  }
  float tot = 0.f;
  for (int k = 0; k < top; ++k) {
    float bv = -INFINITY;
    int bi = 0x7fffffff;
    for (int e = lane; e < E; e += 64) {
      const float v = ch[e];
      if (v != INFINITY && (v > bv || bi == 0x7fffffff)) { bv = v; bi = e; }
    }
    lanes_argmax<64>(bv, bi);
    bi = min(max(bi, 0), E - 1);
    if (lane == 0) {
      idx[(size_t)t * top + k] = bi;
      wt[(size_t)t * top + k] = sc[bi];
      tot += sc[bi];
      ch[bi] = INFINITY;                      // taken
    }
    __syncthreads();
  }
  if ((top_softmax || renorm || wscale != 1.f) && lane == 0) {
    // top_softmax: exp(z - max) of the chosen logits over their sum
    const float r = top_softmax ? wscale / tot : renorm ? wscale / (tot + 1e-20f) : wscale;
    for (int k = 0; k < top; ++k) wt[(size_t)t * top + k] *= r;
  }
}

// Up to 64 router outputs: LPT lanes a token, one output a lane, scores and
// choices in registers; the same sums and comparisons in the same order (the lanes left out above held
// zeros and nothing to choose), and the same bits. Bound by a launch, one trip to memory and the chain
// of choices. us, with a workgroup per token, LDS and a barrier per choice, and now: 2048 / 4097 tokens
// of 16 outputs, best 2 of 4 groups, 4 chosen 8.7, 5.7 / 14.4, 5.8; 64 outputs, 3 of 8 groups, 8 chosen
// 12.2, 10.5 / 21.6, 12.9; one token 7.3, 5.4 and 10.5, 9.4.
template <int LPT>
__global__ __launch_bounds__(256) void moe_route_lanes_kernel(
    const float* __restrict__ z, const float* __restrict__ corr, const float* __restrict__ bias,
    int mode, int E, int G, int keep, int grank, int top, int renorm, float wscale, int* __restrict__ idx,
    float* __restrict__ wt, int T) {
  const int t = blockIdx.x * (256 / LPT) + threadIdx.x / LPT, lane = threadIdx.x % LPT;
  const bool on = lane < E;
  float g = -INFINITY;
  if (on) g = z[(size_t)min(t, T - 1) * E + lane] + (bias ? bias[lane] : 0.f);
  float mx = g;
#pragma unroll
  for (int o = LPT / 2; o > 0; o >>= 1) mx = fmaxf(mx, __shfl_xor(mx, o, LPT));
  float s = 0.f;
  if (on) s = mode == 2 ? sigmoid_f(g) : expf(g - mx);
  float sum = s;
#pragma unroll
  for (int o = LPT / 2; o > 0; o >>= 1) sum += __shfl_xor(sum, o, LPT);
  float ch = g;
  if (mode != 1) {
    const float inv = mode == 2 ? 1.f : 1.f / sum;
    s *= inv;
    ch = corr && on ? s + corr[lane] : s;
  }
  if (G > 1 && keep < G) {                     // lane g ranks group g, as above
    const int per = E / G;
    float b = -INFINITY;
    if (grank <= 1) {
      for (int j = 0; j < per; ++j) b = fmaxf(b, __shfl(ch, min(lane * per + j, E - 1), LPT));
    } else {
      float pv = INFINITY;
      int pi = -1;
      b = 0.f;
      for (int n = 0; n < min(grank, per); ++n) {
        float bv = -INFINITY;
        int bi = -1;
        for (int j = 0; j < per; ++j) {
          const float v = __shfl(ch, min(lane * per + j, E - 1), LPT);
          const bool below = v < pv || (v == pv && j > pi);
          if (below && (bi < 0 || v > bv)) { bv = v; bi = j; }
        }
        if (bi >= 0) { b += bv; pv = bv; pi = bi; }
      }
    }
    for (int k = 0; k < keep; ++k) {
      const bool cand = lane < G && b != INFINITY;
      float bv = cand ? b : -INFINITY;
      int bi = cand ? lane : 0x7fffffff;
      lanes_argmax<LPT>(bv, bi);
      if (lane == __shfl(bi, 0, LPT)) b = INFINITY;
    }
    if (__shfl(b, min(lane / per, LPT - 1), LPT) != INFINITY) ch = -INFINITY;
  }
  bool left = on && ch != INFINITY;
  float tot = 0.f, w = 0.f;
  int mine = 0;
  for (int k = 0; k < top; ++k) {
    float bv = left ? ch : -INFINITY;
    int bi = left ? lane : 0x7fffffff;
    lanes_argmax<LPT>(bv, bi);
    bi = min(__shfl(bi, 0, LPT), E - 1);
    const float c = __shfl(s, bi, LPT);
    tot += c;
    if (lane == bi) left = false;
    if (lane == k) { mine = bi; w = c; }
  }
  if (t >= T || lane >= top) return;
  if (mode == 1) w *= wscale / tot;
  else if (renorm) w *= wscale / (tot + 1e-20f);
  else if (wscale != 1.f) w *= wscale;
  idx[(size_t)t * top + lane] = mine;
  wt[(size_t)t * top + lane] = w;
}

// One workgroup: its time is the chain count -> prefix sum -> scatter, so it is as wide as a
// workgroup gets, keeps a thread's first pairs in registers for the second pass and sums
// up 64 buckets at a time (8192 pairs, 16 experts: 17.4 -> 7.4 us).
#define MP_KEEP 8
__global__ __launch_bounds__(1024) void moe_plan_kernel(const int* __restrict__ idx, int P, int E,
                                                        int* __restrict__ plan) {
  __shared__ int cnt[MOE_MAX_E + 2];
  int* offsets = plan;                // [E + 2]
  int* perm = plan + E + 2;           // [P]
  int* pos = perm + P;                // [P]
  const int tid = threadIdx.x;
  int keep[MP_KEEP];
#pragma unroll
  for (int i = 0; i < MP_KEEP; ++i) {
    const int p = tid + 1024 * i;
    keep[i] = p < P ? min(max(idx[p], 0), E) : 0;      // identity experts share bucket E
  }
  for (int e = tid; e < E + 2; e += 1024) cnt[e] = 0;
  __syncthreads();
#pragma unroll
  for (int i = 0; i < MP_KEEP; ++i)
    if (tid + 1024 * i < P) atomicAdd(&cnt[keep[i]], 1);
  for (int p = tid + 1024 * MP_KEEP; p < P; p += 1024) atomicAdd(&cnt[min(max(idx[p], 0), E)], 1);
  __syncthreads();
  if (tid < 64) {
    int run = 0;
    for (int e0 = 0; e0 <= E; e0 += 64) {
      const int e = e0 + tid, c = e <= E ? cnt[e] : 0;
      int end = c;                                     // inclusive prefix sum over the lanes
#pragma unroll
      for (int o = 1; o < 64; o <<= 1) {
        const int v = __shfl_up(end, o, 64);
        if (tid >= o) end += v;
      }
      if (e <= E) {
        offsets[e] = run + end - c;
        cnt[e] = run + end - c;                        // becomes the fill cursor
      }
      run += __shfl(end, 63, 64);
    }
    if (tid == 0) offsets[E + 1] = run;
  }
  __syncthreads();
#pragma unroll
  for (int i = 0; i < MP_KEEP; ++i) {
    const int p = tid + 1024 * i;
    if (p < P) {
      const int s = atomicAdd(&cnt[keep[i]], 1);
      perm[s] = p;
      pos[p] = s;
    }
  }
  for (int p = tid + 1024 * MP_KEEP; p < P; p += 1024) {
    const int s = atomicAdd(&cnt[min(max(idx[p], 0), E)], 1);
    perm[s] = p;
    pos[p] = s;
  }
}

#define GG_T 64
#define GG_K 16

__device__ __forceinline__ float relu2_f(float z) { const float r = fmaxf(z, 0.f); return r * r; }
__device__ __forceinline__ float clamped_glu_f(float g, float u, float limit) {
  g = fminf(g, limit);
  return g * sigmoid_f(1.702f * g) * (fminf(fmaxf(u, -limit), limit) + 1.f);
}
// the up product's epilogue (a: gate or the only product, u: up)
template <int MODE> __device__ __forceinline__ float moe_epilogue(float a, float u, float limit) {
  if constexpr (MODE == 1) return silu_f(a) * u;
  else if constexpr (MODE == 2) return relu2_f(a);
  else if constexpr (MODE == 3) return clamped_glu_f(a, u, limit);
  else return a;
}

template <typename T, int MODE>
__global__ __launch_bounds__(256) void moe_grouped_gemm_kernel(
    const T* __restrict__ A, const T* __restrict__ Wt, const int* __restrict__ plan, int P, int E,
    int top, int K, int N, float limit, T* __restrict__ out) {
  constexpr int SWIGLU = MODE == 1 || MODE == 3;    // gate and up rows
  constexpr bool GATHER = MODE != 0;
  __shared__ float As[GG_K][GG_T + 1], Bs[GG_K][GG_T + 1], Bu[SWIGLU ? GG_K : 1][GG_T + 1];
  const int* offsets = plan;
  const int* perm = plan + E + 2;
  // which expert segment and which 64-row tile of it this workgroup owns
  int tile = blockIdx.x, e = 0, r0 = 0, r1 = 0;
  for (; e < E; ++e) {
    const int s0 = offsets[e], s1 = offsets[e + 1];
    const int nt = (s1 - s0 + GG_T - 1) / GG_T;
    if (tile < nt) { r0 = s0 + tile * GG_T; r1 = min(s1, r0 + GG_T); break; }
    tile -= nt;
  }
  if (e == E) return;
  const int n0 = blockIdx.y * GG_T;
  const int tx = threadIdx.x % 16, ty = threadIdx.x / 16;
  const int wrows = SWIGLU ? 2 * N : N;        // rows of one expert's weight
  const T* We = Wt + (size_t)e * wrows * K;
  float acc[4][4], accu[SWIGLU ? 4 : 1][4];
#pragma unroll
  for (int i = 0; i < 4; ++i)
#pragma unroll
    for (int j = 0; j < 4; ++j) { acc[i][j] = 0.f; if (SWIGLU) accu[i][j] = 0.f; }
  for (int k0 = 0; k0 < K; k0 += GG_K) {
    __syncthreads();
    for (int i = threadIdx.x; i < GG_T * GG_K; i += 256) {
      const int r = i / GG_K, kk = i % GG_K;
      float a = 0.f, b = 0.f, u = 0.f;
      if (k0 + kk < K) {
        if (r0 + r < r1) {
          const size_t src = GATHER ? (size_t)(perm[r0 + r] / top) : (size_t)(r0 + r);
          a = Act<T>::ld(A + src * K + k0 + kk);
        }
        if (n0 + r < N) {
          b = Act<T>::ld(We + (size_t)(n0 + r) * K + k0 + kk);
          if (SWIGLU) u = Act<T>::ld(We + (size_t)(N + n0 + r) * K + k0 + kk);
        }
      }
      As[kk][r] = a;
      Bs[kk][r] = b;
      if (SWIGLU) Bu[kk][r] = u;
    }
    __syncthreads();
#pragma unroll
    for (int kk = 0; kk < GG_K; ++kk) {
      float a[4], b[4], u[4];
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        a[i] = As[kk][ty * 4 + i];
        b[i] = Bs[kk][tx * 4 + i];
        if (SWIGLU) u[i] = Bu[kk][tx * 4 + i];
      }
#pragma unroll
      for (int i = 0; i < 4; ++i)
#pragma unroll
        for (int j = 0; j < 4; ++j) {
          acc[i][j] += a[i] * b[j];
          if (SWIGLU) accu[i][j] += a[i] * u[j];
        }
    }
  }
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const int r = r0 + ty * 4 + i;
    if (r >= r1) continue;
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const int n = n0 + tx * 4 + j;
      if (n < N)
        Act<T>::st(out + (size_t)r * N + n,
                   moe_epilogue<MODE>(acc[i][j], accu[SWIGLU ? i : 0][j], limit));
    }
  }
}

// The bf16 form on the matrix cores for sizes that moe_pipe.hip does not take (K a multiple
// of 32 only, rows that are no multiple of 16 bytes):
// v_mfma_f32_16x16x32_bf16 with the expert's weight rows as the A operand and
// the (gathered) token rows as B, both fragments loaded straight from global
// memory as one 16-byte load per lane (weights are [n][k] and rows [m][k], so a
// lane's 8 k-values are contiguous). A workgroup owns 64 token rows x 64
// features of one expert segment; each of its 4 waves takes 16 features (and
// the 16 matching up-rows for SwiGLU) against all 64 rows, so the row fragments
// are shared through L1. An accumulator lane holds 4 consecutive features of
// one token row. Per output element the sum over K has a fixed order.
template <int MODE>
__global__ __launch_bounds__(256) void moe_grouped_gemm_mfma_kernel(
    const bf16_t* __restrict__ A, const bf16_t* __restrict__ Wt, const int* __restrict__ plan, int P,
    int E, int top, int K, int N, float limit, bf16_t* __restrict__ out) {
  constexpr int SWIGLU = MODE == 1 || MODE == 3;    // gate and up rows
  constexpr bool GATHER = MODE != 0;
  const int* offsets = plan;
  const int* perm = plan + E + 2;
  int tile = blockIdx.x, e = 0, r0 = 0, r1 = 0;
  for (; e < E; ++e) {
    const int s0 = offsets[e], s1 = offsets[e + 1];
    const int nt = (s1 - s0 + GG_T - 1) / GG_T;
    if (tile < nt) { r0 = s0 + tile * GG_T; r1 = min(s1, r0 + GG_T); break; }
    tile -= nt;
  }
  if (e == E) return;
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int fr = lane & 15, fq = lane >> 4;
  const int nb = blockIdx.y * GG_T + wave * 16;         // this wave's 16 features
  if (nb >= N) return;
  const int wrows = SWIGLU ? 2 * N : N;
  const bf16_t* We = Wt + (size_t)e * wrows * K;
  const int nrow = min(nb + fr, N - 1);                 // clamped: loads stay in range
  const bf16_t* wg = We + (size_t)nrow * K + fq * 8;
  const bf16_t* wu = SWIGLU ? We + (size_t)(N + nrow) * K + fq * 8 : nullptr;
  const bf16_t* arow[4];
#pragma unroll
  for (int j = 0; j < 4; ++j) {
    const int r = min(r0 + 16 * j + fr, r1 - 1);
    const size_t src = GATHER ? (size_t)(perm[r] / top) : (size_t)r;
    arow[j] = A + src * K + fq * 8;
  }
  float4v acc[4], accu[SWIGLU ? 4 : 1];
#pragma unroll
  for (int j = 0; j < 4; ++j) {
    acc[j] = float4v{0.f, 0.f, 0.f, 0.f};
    if (SWIGLU) accu[j] = float4v{0.f, 0.f, 0.f, 0.f};
  }
  for (int k0 = 0; k0 < K; k0 += 32) {
    const bf16x8 a = *reinterpret_cast<const bf16x8*>(wg + k0);
    bf16x8 au;
    if (SWIGLU) au = *reinterpret_cast<const bf16x8*>(wu + k0);
    bf16x8 b[4];
#pragma unroll
    for (int j = 0; j < 4; ++j) b[j] = *reinterpret_cast<const bf16x8*>(arow[j] + k0);
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      acc[j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, b[j], acc[j], 0, 0, 0);
      if (SWIGLU) accu[j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(au, b[j], accu[j], 0, 0, 0);
    }
  }
  // acc[j][i]: feature nb + 4 fq + i of token row r0 + 16 j + fr
#pragma unroll
  for (int j = 0; j < 4; ++j) {
    const int r = r0 + 16 * j + fr;
    if (r >= r1) continue;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int n = nb + 4 * fq + i;
      if (n < N) {
        out[(size_t)r * N + n] =
            f2bf(moe_epilogue<MODE>(acc[j][i], accu[SWIGLU ? j : 0][i], limit));
      }
    }
  }
}

// R: neighbouring columns of a thread (4 where rows and bases allow: 8- or 16-byte
// accesses; 2048 tokens of 2048, 4 experts: 17.5 -> 9.2 us, the copy rate)
template <typename T, int R>
__global__ __launch_bounds__(256) void moe_combine_kernel(
    const T* __restrict__ h, const T* __restrict__ y, const int* __restrict__ idx,
    const float* __restrict__ wt, const int* __restrict__ plan, int P, int top, int E, int d,
    float* __restrict__ out) {
  const int t = blockIdx.x;
  const int* pos = plan + E + 2 + P;
  for (int c = R * (blockIdx.y * blockDim.x + threadIdx.x); c < d; c += R * gridDim.y * blockDim.x) {
    float s[R] = {};
#pragma unroll 4
    for (int k = 0; k < top; ++k) {
      const int p = t * top + k;
      float v[R];
      ld_run<T, R>(idx[p] >= E ? h + (size_t)t * d + c : y + (size_t)pos[p] * d + c, v);
#pragma unroll
      for (int r = 0; r < R; ++r) s[r] += wt[p] * v[r];
    }
    st_run<float, R>(out + (size_t)t * d + c, s);
  }
}

// 0.5 z (1 + tanh(sqrt(2 / pi) (z + 0.044715 z^3)))
__device__ __forceinline__ float gelu_tanh_f(float z) {
  return 0.5f * z * (1.f + tanhf(0.7978845608028654f * (z + 0.044715f * z * z * z)));
}

// ACT 0: SiLU, 1: the tanh form of GELU
template <typename T, int ACT>
__global__ __launch_bounds__(256) void act_mul_any_kernel(const T* __restrict__ x, int F,
                                                          T* __restrict__ y) {
  const size_t r = blockIdx.x;
  for (int c = blockIdx.y * blockDim.x + threadIdx.x; c < F; c += gridDim.y * blockDim.x) {
    const float g = Act<T>::ld(x + r * 2 * F + c);
    Act<T>::st(y + r * F + c, (ACT == 1 ? gelu_tanh_f(g) : silu_f(g)) * Act<T>::ld(x + r * 2 * F + F + c));
  }
}

// relu(x)^2 entry by entry, in place or out of place
template <typename T, int N>
__global__ __launch_bounds__(256) void relu2_any_kernel(const T* x, long n, T* y) {
  for (long i = N * ((long)blockIdx.x * 256 + threadIdx.x); i < n; i += N * 256L * gridDim.x) {
    float f[N];
    ld_run<T, N>(x + i, f);
#pragma unroll
    for (int k = 0; k < N; ++k) f[k] = relu2_f(f[k]);
    st_run<T, N>(y + i, f);
  }
}

extern "C" int loqa_relu2_any(const void* x, int dt, long n, void* y, hipStream_t st) {
  if (n <= 0) return 0;
  const size_t esz = dt == 0 ? 2 : 4;
  const bool v4 = n % 4 == 0 && (size_t)x % (4 * esz) == 0 && (size_t)y % (4 * esz) == 0;
  const long units = (n / (v4 ? 4 : 1) + 255) / 256;
  const dim3 grid((int)(units < 8192 ? units : 8192));
#define GO(TT, NN)                                                                            \
  hipLaunchKernelGGL((relu2_any_kernel<TT, NN>), grid, dim3(256), 0, st, (const TT*)x, n, (TT*)y)
  if (dt == 0) { if (v4) GO(bf16_t, 4); else GO(bf16_t, 1); }
  else { if (v4) GO(float, 4); else GO(float, 1); }
#undef GO
  return (int)hipGetLastError();
}

// y[t, c] = gelu_tanh(z[t, c]) * table[tokens[t], off + c]: a gate on the rows of
// a per-token table. TE: the table's dtype.
template <typename T, typename TE>
__global__ __launch_bounds__(256) void token_gate_kernel(const T* __restrict__ z, long ldz,
                                                         const TE* __restrict__ table, long ldt,
                                                         const int* __restrict__ tokens, int vocab,
                                                         int off, int n, T* __restrict__ y, int T_) {
  const long total = (long)T_ * n;
  for (long i = (long)blockIdx.x * 256 + threadIdx.x; i < total; i += 256L * gridDim.x) {
    const int t = (int)(i / n), c = (int)(i - (long)t * n);
    const int tok = min(max(tokens[t], 0), vocab - 1);
    Act<T>::st(y + i, gelu_tanh_f(Act<T>::ld(z + (size_t)t * ldz + c)) *
                          Act<TE>::ld(table + (size_t)tok * ldt + off + c));
  }
}

extern "C" int loqa_token_gate(const void* z, int dt, long ldz, const void* table, int t_dt, long ldt,
                               const void* tokens, int vocab, int off, int n, void* y, int T,
                               hipStream_t st) {
  if (T <= 0 || n <= 0) return 0;
  if (vocab <= 0 || off < 0 || off + n > ldt || ldz < n) return (int)hipErrorInvalidValue;
  const long units = ((long)T * n + 255) / 256;
  const dim3 grid((int)(units < 8192 ? units : 8192));
#define GO(TT, TE)                                                                            \
  hipLaunchKernelGGL((token_gate_kernel<TT, TE>), grid, dim3(256), 0, st, (const TT*)z, ldz,   \
                     (const TE*)table, ldt, (const int*)tokens, vocab, off, n, (TT*)y, T)
  if (dt == 0 && t_dt == 0) GO(bf16_t, bf16_t);
  else if (dt == 0) GO(bf16_t, float);
  else if (t_dt == 0) GO(float, bf16_t);
  else GO(float, float);
#undef GO
  return (int)hipGetLastError();
}

extern "C" int loqa_act_mul_any(const void* x, int dt, int T, int F, int act, void* y,
                                hipStream_t st) {
  if (T <= 0) return 0;
  if (act < 0 || act > 1) return (int)hipErrorInvalidValue;
  const dim3 grid(T, T >= 512 ? 1 : (F + 255) / 256);
#define GO(TT, A)                                                                             \
  hipLaunchKernelGGL((act_mul_any_kernel<TT, A>), grid, dim3(256), 0, st, (const TT*)x, F, (TT*)y)
  if (dt == 0 && act == 0) GO(bf16_t, 0);
  else if (dt == 0) GO(bf16_t, 1);
  else if (act == 0) GO(float, 0);
  else GO(float, 1);
#undef GO
  return (int)hipGetLastError();
}

extern "C" int loqa_moe_route(const void* z, const void* corr, const void* bias, int mode,
                              int E, int G, int keep, int grank, int top, int renorm, float wscale,
                              void* idx, void* wt, int T, hipStream_t st) {
  if (T <= 0) return 0;
  if (E > MOE_MAX_E || E <= 0 || G <= 0 || E % G || top <= 0 || top > E || mode < 0 || mode > 2)
    return (int)hipErrorInvalidValue;
  if (E <= 64) {                               // faster at every size measured, 1 to 4097 tokens
#define GO(LPT)                                                                                  \
  hipLaunchKernelGGL(moe_route_lanes_kernel<LPT>, dim3((T + 256 / LPT - 1) / (256 / LPT)), dim3(256), 0, st, \
                     (const float*)z, (const float*)corr, (const float*)bias, mode, E, G, keep, grank, top, \
                     renorm, wscale, (int*)idx, (float*)wt, T)
    if (E <= 16) GO(16);
    else if (E <= 32) GO(32);
    else GO(64);
#undef GO
    return (int)hipGetLastError();
  }
  hipLaunchKernelGGL(moe_route_kernel, dim3(T), dim3(64), 0, st, (const float*)z, (const float*)corr,
                     (const float*)bias, mode, E, G, keep, grank, top, renorm, wscale, (int*)idx,
                     (float*)wt);
  return (int)hipGetLastError();
}

extern "C" int loqa_moe_plan(const void* idx, int P, int E, void* plan, hipStream_t st) {
  if (E > MOE_MAX_E) return (int)hipErrorInvalidValue;
  hipLaunchKernelGGL(moe_plan_kernel, dim3(1), dim3(1024), 0, st, (const int*)idx, P, E, (int*)plan);
  return (int)hipGetLastError();
}

bool moe_pipe(const void* A, long rows, const void* W, const void* plan, int P, int E, int top, int K, int N, int mode,
              float limit, void* out, hipStream_t st);        // moe_pipe.hip

extern "C" int loqa_moe_grouped_gemm(const void* A, int dt, const void* W, const void* plan, int P,
                                     int E, int top, int K, int N, int mode, float limit, void* out,
                                     hipStream_t st) {
  if (P <= 0) return 0;
  if (mode < 0 || mode > 3) return (int)hipErrorInvalidValue;
  if (dt == 0 && moe_pipe(A, mode == 0 ? P : P / top, W, plan, P, E, top, K, N, mode, limit, out, st))
    return (int)hipGetLastError();
  const dim3 grid((P + GG_T - 1) / GG_T + E, (N + GG_T - 1) / GG_T);
#define GO_MODE(M, KERNEL, GRID, TT)                                                             \
  hipLaunchKernelGGL(KERNEL(M), GRID, dim3(256), 0, st, (const TT*)A, (const TT*)W,             \
                     (const int*)plan, P, E, top, K, N, limit, (TT*)out)
#define BY_MODE(KERNEL, GRID, TT)                                                               \
  do {                                                                                          \
    if (mode == 1) GO_MODE(1, KERNEL, GRID, TT);                                                \
    else if (mode == 2) GO_MODE(2, KERNEL, GRID, TT);                                           \
    else if (mode == 3) GO_MODE(3, KERNEL, GRID, TT);                                           \
    else GO_MODE(0, KERNEL, GRID, TT);                                                          \
  } while (0)
#define K_MFMA(M) (moe_grouped_gemm_mfma_kernel<M>)
#define K_BF16(M) (moe_grouped_gemm_kernel<bf16_t, M>)
#define K_F32(M) (moe_grouped_gemm_kernel<float, M>)
  if (dt == 0 && K >= 32 && K % 32 == 0) {
    BY_MODE(K_MFMA, grid, bf16_t);
  } else if (dt == 0) {
    BY_MODE(K_BF16, grid, bf16_t);
  } else {
    BY_MODE(K_F32, grid, float);
  }
#undef K_MFMA
#undef K_BF16
#undef K_F32
#undef BY_MODE
#undef GO_MODE
  return (int)hipGetLastError();
}

extern "C" int loqa_moe_combine(const void* h, const void* y, int dt, const void* idx,
                                const void* wt, const void* plan, int T, int top, int E, int d,
                                void* out, hipStream_t st) {
  if (T <= 0) return 0;
  const bool runs = d % 4 == 0 && (((size_t)h | (size_t)y | (size_t)out) & 15) == 0;
  const dim3 cgrid(T, T >= 512 ? 1 : ceil_div(d, 256 * (runs ? 4 : 1)));
#define GO(TT, R)                                                                                   \
  hipLaunchKernelGGL((moe_combine_kernel<TT, R>), cgrid, dim3(256), 0, st, (const TT*)h, (const TT*)y, \
                     (const int*)idx, (const float*)wt, (const int*)plan, T * top, top, E, d, (float*)out)
  if (dt == 0 && runs) GO(bf16_t, 4);
  else if (dt == 0) GO(bf16_t, 1);
  else if (runs) GO(float, 4);
  else GO(float, 1);
#undef GO
  return (int)hipGetLastError();
}
