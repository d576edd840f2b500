// A product per head for the few rows of a token step: y[t, h, :] = x[t, h, :] W[h], W [H, K, N] bf16, K up to 512,
// f32 sums rounded once. (Latent attention's queries into the latent space and its results out of it.)
//
// Bound by the start, one trip to memory and the end. A workgroup of four waves takes 64 columns of a head and 32 rows,
// a wave a quarter of K: all of its W rows go straight to its part of LDS at once (4 KB for 32 of them), whence
// transposed reads make them the A operands of 16 x 16 x 32 MFMAs whose columns are the rows of x; the waves' sums meet
// in LDS. 8 rows, 16 heads: 128 x 512 3.5 us, the vendor's batched product 11.2; 512 x 128 5.0, 5.4. A latent token step has both and
// is bound by the host: 79.5 -> 51 us. Beyond 64 rows the weights' way through LDS for every 32 of them is no longer the lesser.
#include "flash_pipe.h"
#include "seqmix.h"

#define HP_K 32                        // rows of W a step
#define HP_N 64
#define HP_T 32

struct HeadProductParams {
  const bf16_t* x; long x_t, x_h; const bf16_t* w; int T, H, K, N; bf16_t* y; long y_t, y_h;
};

__device__ __forceinline__ int hp_swz(int r) { return 2 * ((r >> 1) & 3); }   // place of chunk c of row r: a half wave reads 8 rows of two

template <int KS>                       // steps of a wave: K = 128 KS
__global__ __launch_bounds__(256) void head_product_kernel(HeadProductParams p) {
  constexpr int STEP = HP_K * HP_N * 2, RING = 4 * KS * STEP, SUMS = 4 * HP_T * (HP_N + 4) * 4;
  __shared__ __attribute__((aligned(1024))) unsigned char lds[RING > SUMS ? RING : SUMS];
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), c = lane & 15, q4 = lane >> 4;
  const int h = blockIdx.y, n0 = blockIdx.x * HP_N, t0 = blockIdx.z * HP_T;
  const bf16_t* w = p.w + ((size_t)h * p.K + wave * KS * HP_K) * p.N + n0;
  const unsigned my = fl_lds_at(lds) + wave * KS * STEP;
  // slot 4 u + i of lane (c, q4) is entry 16 u + 4 q4 + i of a step, as the transposed reads have it
  uint2 xv[KS][2][2];
#pragma unroll
  for (int tb = 0; tb < 2; ++tb) {
    const int t = t0 + 16 * tb + c;
    const bf16_t* row = p.x + (size_t)min(t, p.T - 1) * p.x_t + (size_t)h * p.x_h + wave * KS * HP_K + 4 * q4;
#pragma unroll
    for (int s = 0; s < KS; ++s)
#pragma unroll
      for (int u = 0; u < 2; ++u) xv[s][tb][u] = *reinterpret_cast<const uint2*>(row + s * HP_K + 16 * u);
  }
#pragma unroll
  for (int s = 0; s < KS; ++s)
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int id = lane + 64 * i, r = id / 8, ch = (id % 8) ^ hp_swz(r);
      fl_load_lds(w + (size_t)(s * HP_K + r) * p.N + ch * 8, __builtin_amdgcn_readfirstlane(my + s * STEP + i * 1024));
    }
  float4v acc[4][2];
#pragma unroll
  for (int d = 0; d < 4; ++d) acc[d][0] = acc[d][1] = float4v{0.f, 0.f, 0.f, 0.f};
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");           // this wave's rows of W are here
#pragma unroll
  for (int s = 0; s < KS; ++s)
#pragma unroll
    for (int d = 0; d < 4; ++d) {
      short8 a8;
#pragma unroll
      for (int u = 0; u < 2; ++u) {
        const int r = 16 * u + 4 * q4 + (c >> 2), ch = (2 * d + ((c & 3) >> 1)) ^ hp_swz(r);
        const fl_v4s v = __builtin_amdgcn_ds_read_tr16_b64_v4i16(fl_lds<fl_v4s>(my + s * STEP + r * (HP_N * 2) + ch * 16 + (c & 1) * 8));
#pragma unroll
        for (int i = 0; i < 4; ++i) a8[4 * u + i] = v[i];
      }
#pragma unroll
      for (int tb = 0; tb < 2; ++tb) {
        const fl_u4 b = {xv[s][tb][0].x, xv[s][tb][0].y, xv[s][tb][1].x, xv[s][tb][1].y};
        acc[d][tb] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(*reinterpret_cast<bf16x8*>(&a8), __builtin_bit_cast(bf16x8, b), acc[d][tb], 0, 0, 0);
      }
    }
  // acc (d, tb, r) of lane (c, q4): column 16 d + 4 q4 + r of row 16 tb + c
  __syncthreads();
  float* sums = reinterpret_cast<float*>(lds);               // [waves][rows][columns + 4]
#pragma unroll
  for (int d = 0; d < 4; ++d)
#pragma unroll
    for (int tb = 0; tb < 2; ++tb)
      *reinterpret_cast<float4v*>(sums + (wave * HP_T + 16 * tb + c) * (HP_N + 4) + 16 * d + 4 * q4) = acc[d][tb];
  __syncthreads();
#pragma unroll
  for (int k = 0; k < HP_T * HP_N / 4 / 256; ++k) {
    const int id = threadIdx.x + 256 * k, t = id / (HP_N / 4), e = id % (HP_N / 4) * 4;
    float4v v = *reinterpret_cast<const float4v*>(sums + t * (HP_N + 4) + e);
#pragma unroll
    for (int s = 1; s < 4; ++s) v += *reinterpret_cast<const float4v*>(sums + (s * HP_T + t) * (HP_N + 4) + e);
    if (t0 + t < p.T)
      *reinterpret_cast<uint2*>(p.y + (size_t)(t0 + t) * p.y_t + (size_t)h * p.y_h + n0 + e) =
          make_uint2(pack_bf16x2(v[0], v[1]), pack_bf16x2(v[2], v[3]));
  }
}

extern "C" int loqa_head_product(const void* x, long x_t, long x_h, const void* w, int T, int H, int K, int N, void* y, long y_t, long y_h,
                                 hipStream_t st) {
  if (T <= 0 || H <= 0) return 0;
  if (K <= 0 || K % 128 || K > 512 || N <= 0 || N % HP_N || H > 65535 || T > 65535 * HP_T || (x_t | x_h | y_t | y_h) % 4 ||
      (((size_t)x | (size_t)y) & 7) || ((size_t)w & 15))
    return (int)hipErrorInvalidValue;
  const HeadProductParams p{(const bf16_t*)x, x_t, x_h, (const bf16_t*)w, T, H, K, N, (bf16_t*)y, y_t, y_h};
  const dim3 grid(N / HP_N, H, (T + HP_T - 1) / HP_T);
  switch (K / 128) {
    case 1: hipLaunchKernelGGL(head_product_kernel<1>, grid, dim3(256), 0, st, p); break;
    case 2: hipLaunchKernelGGL(head_product_kernel<2>, grid, dim3(256), 0, st, p); break;
    case 3: hipLaunchKernelGGL(head_product_kernel<3>, grid, dim3(256), 0, st, p); break;
    default: hipLaunchKernelGGL(head_product_kernel<4>, grid, dim3(256), 0, st, p);
  }
  return (int)hipGetLastError();
}
