// Token steps of the windowed paged attention (attn_window.hip), bf16, head sizes up to 128: few
// query rows against many keys, bound by the reads of K and V and, at the sizes of a step, by
// the chain from the block table over the keys and their maximum to the values and the merge.
//
// A workgroup of 16 waves serves one token and key head, or with key splits (p.ns) one of four waves a share of
// its keys. A wave takes 32 keys at a time: K rows go from the pages straight to the A operands of the score
// MFMAs (16 x 16 x 32; the group's query heads, up to 16, are the columns), V rows straight to
// its part of LDS meanwhile, whence transposed reads make them the A operands of the second
// product, whose B operand the exponentials of the scores are as they lie. All of a wave's loads
// are in flight together and maxima of 16 heads cost two exchanges. What one compute unit gets of K and V bounds a
// workgroup (60 KB/us), so beyond some 400 keys a row's keys are split and the splits join in the launch.
// The weights stay what 32 bits hold: each goes as a sum of three bf16 (24 bits), none of them
// negative or zero, so that an infinite value stays one.
// 8 tokens, 16 heads (4 key heads) of 128, window 1024: 24.5 us at first (a key on one lane
// at a time, five key splits and their merge in a second launch), 15.9 in one workgroup of 16 waves, 9.0 in eight of four;
// 4000 keys 26.9 (splits of 16 waves and the second launch), 18.9; up to 400 keys 16 waves 6 to 8; 64 tokens
// behind 2000: 168, 100.
#include "flash_pipe.h"
#include "seqmix.h"

#define WT_KEYS 32

__device__ __forceinline__ float wt_max16(float x) {   // over lanes 16 apart: all keys of a head
  typedef unsigned u2 __attribute__((ext_vector_type(2)));
  const u2 r = __builtin_amdgcn_permlane16_swap(__float_as_uint(x), __float_as_uint(x), false, false);
  return fl_max32(fmaxf(__uint_as_float(r[0]), __uint_as_float(r[1])));
}
__device__ __forceinline__ float wt_sum16(float x) {
  typedef unsigned u2 __attribute__((ext_vector_type(2)));
  const u2 r = __builtin_amdgcn_permlane16_swap(__float_as_uint(x), __float_as_uint(x), false, false);
  return fl_both32(__uint_as_float(r[0]) + __uint_as_float(r[1]));
}

// place of chunk c of V row r: a half wave reads 8 rows of two chunks
template <int DV> __device__ __forceinline__ int wt_swz(int r) { return DV == 128 ? 2 * (r & 7) : 2 * ((r >> 1) & 3); }

// Of a workgroup's partial: per head and column the sum, then (maximum, sum of the weights) per head.
__host__ __device__ __forceinline__ int wt_part_floats(int rep, int Dv) { return rep * Dv + (2 * rep + 3) / 4 * 4; }

// The workgroups of a row's key splits (p.ns of them): each leaves the joint partial of its waves (mm, ll, aa in LDS, which
// this uses up), and the last to arrive sums them up in the splits' order, whichever it is. Nobody waits for anybody.
// Written through and read past the caches (sc1).
template <int NW, int DV>
__device__ __forceinline__ void wt_join(const WinAttnParams& p, float* mm, float* ll, float* aa, int t, int g, int sp, int rep) {
  constexpr int SC1 = 16, TH = 64 * NW, BATCH = 8;
  const int tid = threadIdx.x, Dv = p.Dv, per = wt_part_floats(rep, Dv), row = t * p.G + g, quads = rep * Dv / 4;
  constexpr float LOG2E = 1.4426950408889634f;
  const __amdgpu_buffer_rsrc_t part = __builtin_amdgcn_make_buffer_rsrc(p.part + (size_t)row * p.ns * per, 0, p.ns * per * 4, 0x00020000);
  auto top = [&](int r) {
    float M = -1e30f;
#pragma unroll
    for (int w = 0; w < NW; ++w) M = fmaxf(M, mm[w * 16 + r]);
    return M;
  };
  for (int q = tid; q < quads; q += TH) {
    const int r = q * 4 / Dv, e = q * 4 - r * Dv;
    const float M = top(r);
    float4v num = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int w = 0; w < NW; ++w)
      num += __builtin_amdgcn_exp2f(mm[w * 16 + r] - M) * *reinterpret_cast<const float4v*>(aa + ((size_t)w * rep + r) * DV + e);
    __builtin_amdgcn_raw_buffer_store_b128(__builtin_bit_cast(fl_u4, num), part, (sp * per + q * 4) * 4, 0, SC1);
  }
  if (tid < rep) {
    const float M = top(tid);
    float den = 0.f;
#pragma unroll
    for (int w = 0; w < NW; ++w) den += __builtin_amdgcn_exp2f(mm[w * 16 + tid] - M) * ll[w * 16 + tid];
    typedef unsigned u2 __attribute__((ext_vector_type(2)));
    __builtin_amdgcn_raw_buffer_store_b64(u2{__float_as_uint(M), __float_as_uint(den)}, part, (sp * per + rep * Dv + 2 * tid) * 4, 0, SC1);
  }
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");           // written through: visible when acknowledged
  __syncthreads();
  int* word = p.words + (size_t)row * TICKET;
  int* flag = reinterpret_cast<int*>(mm);                    // (mm, ll and aa have been read)
  if (tid == 0) {
    *flag = __hip_atomic_fetch_add(word, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) == p.ns - 1;
    if (*flag) __hip_atomic_store(word, 0, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  }
  __syncthreads();
  if (!*flag) return;
  // (maximum, sum) of every split and head
  float* f = mm + 16;                                        // [rep][ns] factors, then [rep] 1 / sum
  float* inv = f + rep * p.ns;
  for (int i = tid; i < rep * p.ns; i += TH) {
    const int r = i / p.ns, s = i - r * p.ns;
    f[i] = __uint_as_float(__builtin_amdgcn_raw_buffer_load_b32(part, (s * per + rep * Dv + 2 * r) * 4, 0, SC1));
  }
  __syncthreads();
  if (tid < rep) {
    float M = p.sink ? p.sink[g * rep + tid] * LOG2E : -1e30f;
    for (int s = 0; s < p.ns; ++s) M = fmaxf(M, f[tid * p.ns + s]);
    float den = p.sink ? __builtin_amdgcn_exp2f(p.sink[g * rep + tid] * LOG2E - M) : 0.f;
    for (int s = 0; s < p.ns; ++s) {
      const float a = __builtin_amdgcn_exp2f(f[tid * p.ns + s] - M);
      f[tid * p.ns + s] = a;
      den += a * __uint_as_float(__builtin_amdgcn_raw_buffer_load_b32(part, (s * per + rep * Dv + 2 * tid + 1) * 4, 0, SC1));
    }
    inv[tid] = den > 0.f ? 1.f / den : 0.f;
  }
  __syncthreads();
  for (int q = tid; q < quads; q += TH) {
    const int r = q * 4 / Dv, e = q * 4 - r * Dv, h = g * rep + r;
    float4v num = {0.f, 0.f, 0.f, 0.f};
    for (int s0 = 0; s0 < p.ns; s0 += BATCH) {
      float4v v[BATCH];
#pragma unroll
      for (int k = 0; k < BATCH; ++k)                        // past the last split: zeros from past the buffer, not summed up
        v[k] = __builtin_bit_cast(float4v, __builtin_amdgcn_raw_buffer_load_b128(part, ((s0 + k) * per + q * 4) * 4, 0, SC1));
#pragma unroll
      for (int k = 0; k < BATCH; ++k)
        if (s0 + k < p.ns) num += f[r * p.ns + s0 + k] * v[k];
    }
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      float out = num[i] * inv[r];
      if (p.gate) out *= sigmoid_f(bf2f(((const bf16_t*)p.gate)[(size_t)t * p.gate_ld + (size_t)h * Dv + e + i]));
      ((bf16_t*)p.o)[(size_t)t * p.o_ld + (size_t)h * Dv + e + i] = f2bf(out);
    }
  }
}

template <int DK, int DV, int WT_WAVES>
__global__ __launch_bounds__(64 * WT_WAVES, 4) void window_attn_token_kernel(WinAttnParams p) {
  constexpr int NS = DK / 32, NDT = DV / 16, CH = DV / 8, NV = WT_KEYS * CH / 64;
  constexpr int VB = WT_KEYS * DV * 2;                       // bytes of a wave's V tile
  extern __shared__ __attribute__((aligned(16))) unsigned char lds[];
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int c = lane & 15, q4 = lane >> 4;                   // head column, key quarter
  const int t = blockIdx.x, g = blockIdx.y, sp = blockIdx.z;
  if (t >= p.cu_q[p.B]) return;
  const int b = wa_seq_of_row(p.cu_q, p.B, t);
  const int rep = p.H / p.G, D = p.D, Dv = p.Dv;
  const int pq = p.pos[t];
  const int hi = min(pq, p.ctx[b] - 1);
  const int lo = p.window > 0 ? max(0, pq - p.window + 1) : 0;
  // tiles of 32 keys: the kept first tokens before the window, then from its first key on
  const int kept = p.window > 0 ? min(p.keep_first, min(lo, hi + 1)) : 0;
  const int n1 = kept > 0 ? (kept + WT_KEYS - 1) / WT_KEYS : 0;
  const int nt = n1 + max(hi - lo + WT_KEYS, 0) / WT_KEYS;
  const int* bt = p.bt + (size_t)b * p.max_blocks;
  const bf16_t* kc = (const bf16_t*)p.kc + (size_t)g * D;
  const bf16_t* vc = (const bf16_t*)p.vc + (size_t)g * Dv;
  const size_t kst = (size_t)p.G * D, vst = (size_t)p.G * Dv;

  bf16x8 qf[NS];
  {
    const bf16_t* qr = (const bf16_t*)p.q + ((size_t)t * p.H + g * rep + min(c, rep - 1)) * D;
#pragma unroll
    for (int s = 0; s < NS; ++s) {
      const int e = 32 * s + 8 * q4;
      const uint4 v = c < rep && e < D ? *reinterpret_cast<const uint4*>(qr + e) : make_uint4(0, 0, 0, 0);
      qf[s] = *reinterpret_cast<const bf16x8*>(&v);
    }
  }
  const float slope = p.slopes ? p.slopes[g * rep + min(c, rep - 1)] : 0.f;
  float4v acc[NDT];
#pragma unroll
  for (int d = 0; d < NDT; ++d) acc[d] = float4v{0.f, 0.f, 0.f, 0.f};
  float m = -1e30f, l = 0.f;                                 // base 2
  constexpr float LOG2E = 1.4426950408889634f;
  const unsigned my = fl_lds_at(lds) + wave * VB;
  for (int wk = sp * WT_WAVES + wave; wk < nt; wk += p.ns * WT_WAVES) {
    const int k0 = wk < n1 ? wk * WT_KEYS : lo + (wk - n1) * WT_KEYS, end = wk < n1 ? kept : hi + 1;
    // lane r names the cache row of key k0 + r % 32 (past the last key: that one's)
    const int jc = min(k0 + (lane & 31), end - 1), pi = jc / p.blk;
    const int row = (int)min(max((long)bt[pi] * p.blk + (jc - pi * p.blk), 0L), p.cache_rows - 1);
    uint4 kr[2][NS];
#pragma unroll
    for (int u = 0; u < 2; ++u) {
      const bf16_t* r = kc + (size_t)__shfl(row, 16 * u + c) * kst;
#pragma unroll
      for (int s = 0; s < NS; ++s) {
        const int e = 32 * s + 8 * q4;
        kr[u][s] = e < D ? *reinterpret_cast<const uint4*>(r + e) : make_uint4(0, 0, 0, 0);
      }
    }
#pragma unroll
    for (int i = 0; i < NV; ++i) {
      const int id = lane + 64 * i, r = id / CH, ch = (id % CH) ^ wt_swz<DV>(r);
      const bf16_t* src = vc + (size_t)__shfl(row, r) * vst + ch * 8;
      if (ch * 8 < Dv) fl_load_lds(src, __builtin_amdgcn_readfirstlane(my + i * 1024));
    }
    float4v st[2];
#pragma unroll
    for (int u = 0; u < 2; ++u) {
      st[u] = float4v{0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int s = 0; s < NS; ++s)
        st[u] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(*reinterpret_cast<bf16x8*>(&kr[u][s]), qf[s], st[u], 0, 0, 0);
    }
    // score (u, r) of lane (c, q4): head c, key k0 + 16 u + 4 q4 + r
    float mx = -INFINITY;
#pragma unroll
    for (int u = 0; u < 2; ++u)
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int j = k0 + 16 * u + 4 * q4 + r;
        float sv = st[u][r] * p.scale;
        if (p.cap > 0.f) sv = p.cap * tanhf(sv / p.cap);
        sv = (sv - slope * (float)(pq - j)) * LOG2E;
        if (j >= end) sv = -INFINITY;
        st[u][r] = sv;
        mx = fmaxf(mx, sv);
      }
    const float mn = fmaxf(m, wt_max16(mx));
    const float alpha = __builtin_amdgcn_exp2f(m - mn);
    m = mn;
    l *= alpha;
    bf16x8 pw[3];
#pragma unroll
    for (int u = 0; u < 2; ++u)
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        // the weight's leading, middle and last 8 bits, cut off toward zero (exact); a part that
        // is zero would make 0 x inf of an infinite value: it is 2^-126, nothing beside weights up to 1
        float e = __builtin_amdgcn_exp2f(st[u][r] - mn);
        l += e;
#pragma unroll
        for (int w = 0; w < 3; ++w) {
          const float h = __uint_as_float(__float_as_uint(e) & 0xffff0000u);
          pw[w][4 * u + r] = (__bf16)fmaxf(h, 1.17549435e-38f);
          e -= h;
        }
      }
#pragma unroll
    for (int d = 0; d < NDT; ++d) acc[d] *= alpha;
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");         // this wave's V tile is here
#pragma unroll
    for (int d = 0; d < NDT; ++d) {
      bf16x8 a;
      short8 a8;
#pragma unroll
      for (int u = 0; u < 2; ++u) {
        const int r = 16 * u + 4 * q4 + (c >> 2), ch = (2 * d + ((c & 3) >> 1)) ^ wt_swz<DV>(r);
        const fl_v4s v = __builtin_amdgcn_ds_read_tr16_b64_v4i16(fl_lds<fl_v4s>(my + r * (DV * 2) + ch * 16 + (c & 1) * 8));
#pragma unroll
        for (int i = 0; i < 4; ++i) a8[4 * u + i] = v[i];
      }
      a = *reinterpret_cast<bf16x8*>(&a8);
#pragma unroll
      for (int w = 0; w < 3; ++w) acc[d] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, pw[w], acc[d], 0, 0, 0);
    }
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");       // read, before the next tile's loads
  }
  l = wt_sum16(l);

  // the waves' partials, in wave order: acc (d, r) of lane (c, q4) is column 16 d + 4 q4 + r of head c
  __syncthreads();
  float* mm = reinterpret_cast<float*>(lds);                 // [waves][16]
  float* ll = mm + WT_WAVES * 16;
  float* aa = ll + WT_WAVES * 16;                            // [waves][rep][DV]
  if (q4 == 0) {
    mm[wave * 16 + c] = m;
    ll[wave * 16 + c] = l;
  }
  if (c < rep)
#pragma unroll
    for (int d = 0; d < NDT; ++d)
      *reinterpret_cast<float4v*>(aa + ((size_t)wave * rep + c) * DV + 16 * d + 4 * q4) = acc[d];
  __syncthreads();
  if (p.ns > 1) {
    wt_join<WT_WAVES, DV>(p, mm, ll, aa, t, g, sp, rep);
    return;
  }
  for (int idx = threadIdx.x; idx < rep * Dv; idx += 64 * WT_WAVES) {
    const int r = idx / Dv, e = idx - r * Dv, h = g * rep + r;
    const bool snk = p.sink != nullptr;
    const float sk = snk ? p.sink[h] * LOG2E : -1e30f;
    float M = sk;
#pragma unroll
    for (int w = 0; w < WT_WAVES; ++w) M = fmaxf(M, mm[w * 16 + r]);
    float num = 0.f, den = snk ? __builtin_amdgcn_exp2f(sk - M) : 0.f;
#pragma unroll
    for (int w = 0; w < WT_WAVES; ++w) {
      const float f = __builtin_amdgcn_exp2f(mm[w * 16 + r] - M);
      num += f * aa[((size_t)w * rep + r) * DV + e];
      den += f * ll[w * 16 + r];
    }
    float out = den > 0.f ? num / den : 0.f;
    if (p.gate) out *= sigmoid_f(bf2f(((const bf16_t*)p.gate)[(size_t)t * p.gate_ld + (size_t)h * Dv + e]));
    ((bf16_t*)p.o)[(size_t)t * p.o_ld + (size_t)h * Dv + e] = f2bf(out);
  }
}

#define WT_SPLITS 64

// -1: not these sizes or places
int window_attention_token(const WinAttnParams& p, hipStream_t st) {
  const int rep = p.H / p.G;
  if (p.ns > 1) {
    if (p.ns > WT_SPLITS || !p.words || ((size_t)p.part & 15)) return -1;
    if ((long)p.T * p.G > p.tickets || (long)p.T * p.G * p.ns * wt_part_floats(rep, p.Dv) > p.part_floats) return (int)hipErrorInvalidValue;
  }
  if (p.D > 128 || p.Dv > 128 || p.D % 8 || p.Dv % 8 || rep > 16 || p.cache_rows > 0x7fffffffL ||
      (((size_t)p.q | (size_t)p.kc | (size_t)p.vc) & 15))
    return -1;
  const dim3 grid(p.T, p.G, p.ns);
  // Enough rows to fill the chip: four waves, whose workgroups share a CU and wait in turn (us,
  // 16 and 4 waves: 32 tokens of 4 key heads, 1024 keys: 21, 24; 80 tokens, 512 keys: 24, 21; 240
  // tokens of 16 key heads of 64, 1000 keys: 130, 94).
  const bool many = (long)p.T * p.G >= 256;
#define RUN(A, C, W)                                                                                    \
  do {                                                                                                  \
    const int ring = W * WT_KEYS * C * 2, end = W * (32 + rep * C) * 4;                                 \
    hipLaunchKernelGGL((window_attn_token_kernel<A, C, W>), grid, dim3(64 * W), ring > end ? ring : end, st, p); \
    return (int)hipGetLastError();                                                                      \
  } while (0)
#define GO(A, C)                                                                                        \
  do {                                                                                                  \
    if (many || p.ns > 1) RUN(A, C, 4);                                                                             \
    RUN(A, C, 16);                                                                                      \
  } while (0)
  if (p.D <= 64) {
    if (p.Dv <= 64) GO(64, 64); else GO(64, 128);
  }
  if (p.Dv <= 64) GO(128, 64); else GO(128, 128);
#undef RUN
#undef GO
}
