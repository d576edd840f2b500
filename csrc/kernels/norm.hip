// Fused normalisation kernels (layer norm, rms norm).
//
// The row stays in registers between the statistics pass and the scale pass, so HBM traffic is
// exactly
//   read x (+ read residual, write residual) + write y.
// Rows are loaded as 16-byte vectors (8 bf16 per lane). A row is a wave's
// (norm_rows_kernel) or, where it is long and there are few, a 256-thread workgroup's (up to d =
// 256 * 8 * MAXV). d % 8 == 0.
#include "common.h"

#define NORM_THREADS 256
#define MAXV 4

// y = rmsnorm(x [+ residual]) * w.  If residual != nullptr, residual <- x + residual.
// Output row i normalises x row row_idx[i] (or i): the final norm of a decode
// step gathers the logit rows itself instead of a separate index_select.
__global__ __launch_bounds__(NORM_THREADS) void rmsnorm_kernel(
    const bf16_t* __restrict__ x, bf16_t* __restrict__ residual,
    const bf16_t* __restrict__ w, bf16_t* __restrict__ y, int d, float eps,
    const int64_t* __restrict__ row_idx) {
  __shared__ float scratch[NORM_THREADS / 64];
  const int row = blockIdx.x;
  const int src = row_idx ? (int)row_idx[row] : row;
  const int nvec = d >> 3;
  const uint4* xr = reinterpret_cast<const uint4*>(x + (size_t)src * d);
  uint4* rr = residual ? reinterpret_cast<uint4*>(residual + (size_t)row * d) : nullptr;
  // the norm weight does not depend on the statistics: requested with the row,
  // so the scale pass does not wait for a second memory round trip
  const uint4* wr = reinterpret_cast<const uint4*>(w);
  uint4 wpre[MAXV];
#pragma unroll
  for (int i = 0; i < MAXV; ++i) {
    const int c = threadIdx.x + i * NORM_THREADS;
    wpre[i] = c < nvec ? wr[c] : make_uint4(0, 0, 0, 0);
  }
  float v[MAXV][8];
  float ss = 0.f;
#pragma unroll
  for (int i = 0; i < MAXV; ++i) {
    const int c = threadIdx.x + i * NORM_THREADS;
    if (c < nvec) {
      unpack8(xr[c], v[i]);
      if (rr) {
        float r[8];
        unpack8(rr[c], r);
#pragma unroll
        for (int j = 0; j < 8; ++j) v[i][j] += r[j];
        // The residual stream is stored in bf16 (as the model's dtype); the norm
        // is computed from the same rounded values a bf16 reference would see.
        uint4 p = pack8(v[i]);
        rr[c] = p;
        unpack8(p, v[i]);
      }
#pragma unroll
      for (int j = 0; j < 8; ++j) ss += v[i][j] * v[i][j];
    }
  }
  ss = block_sum(ss, scratch);
  const float inv = rsqrtf(ss / (float)d + eps);
  uint4* yr = reinterpret_cast<uint4*>(y + (size_t)row * d);
#pragma unroll
  for (int i = 0; i < MAXV; ++i) {
    const int c = threadIdx.x + i * NORM_THREADS;
    if (c < nvec) {
      float wf[8], o[8];
      unpack8(wpre[i], wf);
#pragma unroll
      for (int j = 0; j < 8; ++j) o[j] = v[i][j] * inv * wf[j];
      yr[c] = pack8(o);
    }
  }
}

// y = layernorm(x [+ residual]) * w + b  (Whisper pre-LN blocks).
__global__ __launch_bounds__(NORM_THREADS) void layernorm_kernel(
    const bf16_t* __restrict__ x, bf16_t* __restrict__ residual,
    const bf16_t* __restrict__ w, const bf16_t* __restrict__ b,
    bf16_t* __restrict__ y, int d, float eps, const int64_t* __restrict__ row_idx) {
  __shared__ float scratch[NORM_THREADS / 64];
  const int row = blockIdx.x;
  const int src = row_idx ? (int)row_idx[row] : row;
  const int nvec = d >> 3;
  const uint4* xr = reinterpret_cast<const uint4*>(x + (size_t)src * d);
  uint4* rr = residual ? reinterpret_cast<uint4*>(residual + (size_t)row * d) : nullptr;
  const uint4* wr = reinterpret_cast<const uint4*>(w);
  const uint4* br = reinterpret_cast<const uint4*>(b);
  uint4 wpre[MAXV], bpre[MAXV];     // requested with the row (see rmsnorm_kernel)
#pragma unroll
  for (int i = 0; i < MAXV; ++i) {
    const int c = threadIdx.x + i * NORM_THREADS;
    wpre[i] = c < nvec ? wr[c] : make_uint4(0, 0, 0, 0);
    bpre[i] = c < nvec ? br[c] : make_uint4(0, 0, 0, 0);
  }
  float v[MAXV][8];
  float s = 0.f;
#pragma unroll
  for (int i = 0; i < MAXV; ++i) {
    const int c = threadIdx.x + i * NORM_THREADS;
    if (c < nvec) {
      unpack8(xr[c], v[i]);
      if (rr) {
        float r[8];
        unpack8(rr[c], r);
#pragma unroll
        for (int j = 0; j < 8; ++j) v[i][j] += r[j];
        uint4 p = pack8(v[i]);
        rr[c] = p;
        unpack8(p, v[i]);
      }
#pragma unroll
      for (int j = 0; j < 8; ++j) s += v[i][j];
    }
  }
  const float mean = block_sum(s, scratch) / (float)d;
  float q = 0.f;
#pragma unroll
  for (int i = 0; i < MAXV; ++i) {
    const int c = threadIdx.x + i * NORM_THREADS;
    if (c < nvec) {
#pragma unroll
      for (int j = 0; j < 8; ++j) {
        const float t = v[i][j] - mean;
        q += t * t;
      }
    }
  }
  const float inv = rsqrtf(block_sum(q, scratch) / (float)d + eps);
  uint4* yr = reinterpret_cast<uint4*>(y + (size_t)row * d);
#pragma unroll
  for (int i = 0; i < MAXV; ++i) {
    const int c = threadIdx.x + i * NORM_THREADS;
    if (c < nvec) {
      float wf[8], bf[8], o[8];
      unpack8(wpre[i], wf);
      unpack8(bpre[i], bf);
#pragma unroll
      for (int j = 0; j < 8; ++j) o[j] = (v[i][j] - mean) * inv * wf[j] + bf[j];
      yr[c] = pack8(o);
    }
  }
}

// The sum over a wave, in every lane; exchanges in the VALU as far as they go, where a shuffle
// takes a trip through LDS.
template <int CTRL> __device__ __forceinline__ float dpp_add(float v) {
  return v + __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), CTRL, 0xF, 0xF, true));
}
__device__ __forceinline__ float row_sum(float v) {
  v = dpp_add<0xB1>(v);     // lane ^ 1
  v = dpp_add<0x4E>(v);     // lane ^ 2
  v = dpp_add<0x141>(v);    // the other half of 8
  v = dpp_add<0x140>(v);    // the other half of 16
  v += __shfl_xor(v, 16, 64);
  return v + __shfl_xor(v, 32, 64);
}

// Layer norm (LN) or rms norm, a wave per row, VEC 16-byte pieces of it a lane (d <= 512 VEC), no
// barrier. With a workgroup per row two barriers and LDS sums a row stood between its loads and
// its stores, and 96 of 256 threads had nothing at 1280 columns; us a layer norm, before and now:
// 96 x 1280 3.2, 2.7; 1500 x 512 5.1, 2.5; 1500 x 1280 6.1, 3.9; 9000 x 1280 23.2, 11.5 (46 MB).
// Pieces past the row's end are loaded from its last one and not used: a load behind a condition,
// with zeros as the alternative, becomes one through a generic pointer.
// A piece is summed up by itself: one chain over a lane's entries lost more than the workgroup's sums
// of 8 or 16 a thread. Sums of squares, root mean square error, workgroup, one chain, by pieces:
// 1280 columns 4.6e-8, 4.5e-8, 4.3e-8; 3072 4.2e-8, 4.6e-8, 3.9e-8; 4096 4.5e-8, 6.1e-8, 4.5e-8.
template <int VEC, bool LN>
__global__ __launch_bounds__(NORM_THREADS) void norm_rows_kernel(
    const bf16_t* __restrict__ x, bf16_t* __restrict__ residual, const bf16_t* __restrict__ w,
    const bf16_t* __restrict__ b, bf16_t* __restrict__ y, int rows, int d, float eps,
    const int64_t* __restrict__ row_idx) {
  const int lane = threadIdx.x & 63, nvec = d >> 3;
  const int row = blockIdx.x * (NORM_THREADS / 64) + (threadIdx.x >> 6);
  if (row >= rows) return;
  const int src = row_idx ? (int)row_idx[row] : row;
  const uint4* xr = reinterpret_cast<const uint4*>(x + (size_t)src * d);
  uint4* rr = residual ? reinterpret_cast<uint4*>(residual + (size_t)row * d) : nullptr;
  uint4 xv[VEC], wv[VEC], bv[VEC];
#pragma unroll
  for (int i = 0; i < VEC; ++i) xv[i] = xr[min(lane + 64 * i, nvec - 1)];
#pragma unroll
  for (int i = 0; i < VEC; ++i) {
    wv[i] = reinterpret_cast<const uint4*>(w)[min(lane + 64 * i, nvec - 1)];
    if (LN) bv[i] = reinterpret_cast<const uint4*>(b)[min(lane + 64 * i, nvec - 1)];
  }
  if (rr) {
#pragma unroll
    for (int i = 0; i < VEC; ++i) {
      float f[8], r[8];
      unpack8(xv[i], f);
      unpack8(rr[min(lane + 64 * i, nvec - 1)], r);
#pragma unroll
      for (int j = 0; j < 8; ++j) f[j] += r[j];
      xv[i] = pack8(f);
    }
#pragma unroll
    for (int i = 0; i < VEC; ++i)
      if (lane + 64 * i < nvec) rr[lane + 64 * i] = xv[i];
  }
  float mean = 0.f, q = 0.f;
  if (LN) {
#pragma unroll
    for (int i = 0; i < VEC; ++i)
      if (lane + 64 * i < nvec) {
        float f[8];
        unpack8(xv[i], f);
        float s = 0.f;
#pragma unroll
        for (int j = 0; j < 8; ++j) s += f[j];
        mean += s;
      }
    mean = row_sum(mean) / (float)d;
  }
#pragma unroll
  for (int i = 0; i < VEC; ++i)
    if (lane + 64 * i < nvec) {
      float f[8];
      unpack8(xv[i], f);
      float s = 0.f;
#pragma unroll
      for (int j = 0; j < 8; ++j) {
        const float t = LN ? f[j] - mean : f[j];
        s += t * t;
      }
      q += s;
    }
  const float inv = rsqrtf(row_sum(q) / (float)d + eps);
  uint4* yr = reinterpret_cast<uint4*>(y + (size_t)row * d);
#pragma unroll
  for (int i = 0; i < VEC; ++i)
    if (lane + 64 * i < nvec) {
      float f[8], wf[8], bf[8];
      unpack8(xv[i], f);
      unpack8(wv[i], wf);
      if (LN) unpack8(bv[i], bf);
#pragma unroll
      for (int j = 0; j < 8; ++j) f[j] = LN ? (f[j] - mean) * inv * wf[j] + bf[j] : f[j] * inv * wf[j];
      yr[lane + 64 * i] = pack8(f);
    }
}

// A wave per row, or a workgroup? The wave's chain of pieces is longer, the workgroup has two
// barriers. Times with waves over times with workgroups, both builds' calls in turn, 1 to 9000 rows:
// up to 3072 columns 0.44 to 1.00 (rms norm) and 0.27 to 1.00 (layer norm). Beyond, one row more than fills the
// compute units with waves costs a round: 4096 columns at 1100 / 1300 / 1600 / 1800 / 2048 / 4096 rows 1.08, 1.05, 1.02,
// 0.97, 0.94, 0.87 (rms norm), 1.08, 0.86, 0.84, 0.86, 0.87, 0.82 (layer norm). A residual's rows come and go on
// the same chain: up to 1024 columns 0.49 to 0.97; 1280 and more from 2048 rows on 0.76 to 1.02 (worst: 2048 x
// 2048, 9000 x 4096), layer norm 0.62 to 0.99.
static bool wave_per_row(int rows, int d, bool residual, bool ln) {
  if (d <= 0 || d > 4096) return false;
  return residual ? d <= 1024 || rows >= 2048 : d <= 3072 || rows >= (ln ? 1300 : 1800);
}

template <bool LN>
static int norm_rows(const void* x, void* residual, const void* w, const void* b, void* y, int rows, int d, float eps,
                     const int64_t* row_idx, hipStream_t s) {
#define GO(VEC)                                                                                                     \
  case VEC:                                                                                                         \
    hipLaunchKernelGGL((norm_rows_kernel<VEC, LN>), dim3((rows + NORM_THREADS / 64 - 1) / (NORM_THREADS / 64)),     \
                       dim3(NORM_THREADS), 0, s, (const bf16_t*)x, (bf16_t*)residual, (const bf16_t*)w,             \
                       (const bf16_t*)b, (bf16_t*)y, rows, d, eps, row_idx);                                        \
    break
  switch ((d + 511) / 512) { GO(1); GO(2); GO(3); GO(4); GO(5); GO(6); GO(7); GO(8); }
#undef GO
  return (int)hipGetLastError();
}

// row_idx (int64, may be null) selects the source rows; it is not combined with
// residual (the wrapper rejects that).
extern "C" int loqa_rmsnorm(const void* x, void* residual, const void* w, void* y,
                            int rows, int d, float eps, const int64_t* row_idx, hipStream_t s) {
  if (d % 8 != 0 || d > NORM_THREADS * 8 * MAXV || rows <= 0) return (int)hipErrorInvalidValue;
  if (row_idx && residual) return (int)hipErrorInvalidValue;
  if (wave_per_row(rows, d, residual, false)) return norm_rows<false>(x, residual, w, nullptr, y, rows, d, eps, row_idx, s);
  hipLaunchKernelGGL(rmsnorm_kernel, dim3(rows), dim3(NORM_THREADS), 0, s,
                     (const bf16_t*)x, (bf16_t*)residual, (const bf16_t*)w, (bf16_t*)y, d, eps,
                     row_idx);
  return (int)hipGetLastError();
}

extern "C" int loqa_layernorm(const void* x, void* residual, const void* w, const void* b,
                              void* y, int rows, int d, float eps, const int64_t* row_idx,
                              hipStream_t s) {
  if (d % 8 != 0 || d > NORM_THREADS * 8 * MAXV || rows <= 0) return (int)hipErrorInvalidValue;
  if (row_idx && residual) return (int)hipErrorInvalidValue;
  if (wave_per_row(rows, d, residual, true)) return norm_rows<true>(x, residual, w, b, y, rows, d, eps, row_idx, s);
  hipLaunchKernelGGL(layernorm_kernel, dim3(rows), dim3(NORM_THREADS), 0, s,
                     (const bf16_t*)x, (bf16_t*)residual, (const bf16_t*)w, (const bf16_t*)b,
                     (bf16_t*)y, d, eps, row_idx);
  return (int)hipGetLastError();
}

// Decoder input embedding: out[r] = bf16(tok_embed[tokens[r]] + pos_embed[positions[r]])
// (Whisper decoder; feeds layernorm as the first residual).
__global__ void embed_pos_kernel(const int* __restrict__ tokens, const int* __restrict__ positions,
                                 const bf16_t* __restrict__ te, const bf16_t* __restrict__ pe,
                                 bf16_t* __restrict__ out, int d) {
  const int row = blockIdx.x;
  const uint4* a = reinterpret_cast<const uint4*>(te + (size_t)max(tokens[row], 0) * d);
  const uint4* b = reinterpret_cast<const uint4*>(pe + (size_t)positions[row] * d);
  uint4* o = reinterpret_cast<uint4*>(out + (size_t)row * d);
  for (int c = threadIdx.x; c < (d >> 3); c += blockDim.x) {
    float x[8], y[8];
    unpack8(a[c], x);
    unpack8(b[c], y);
#pragma unroll
    for (int j = 0; j < 8; ++j) x[j] += y[j];
    o[c] = pack8(x);
  }
}

extern "C" int loqa_embed_pos(const int* tokens, const int* positions, const void* tok_embed,
                              const void* pos_embed, void* out, int rows, int d, hipStream_t s) {
  if (rows <= 0) return 0;
  if (d % 8) return (int)hipErrorInvalidValue;
  hipLaunchKernelGGL(embed_pos_kernel, dim3(rows), dim3(128), 0, s, tokens, positions,
                     (const bf16_t*)tok_embed, (const bf16_t*)pos_embed, (bf16_t*)out, d);
  return (int)hipGetLastError();
}

// Decode-step input of the fused-GEMM path: out[r] = tok_embed[tokens[r]]
// (+ pos_embed[positions[r]], rounded to bf16 once) AND the row statistics the
// first layer's norm prologue reads as one partial tile: rowsq[r] = sum out^2,
// rowsum[r] = sum out (optional). Replaces embedding + a float copy + two
// reductions (four to five launches) with one; the sums are taken over the
// stored bf16 values, as the residual epilogues do.
__global__ __launch_bounds__(NORM_THREADS) void embed_stats_kernel(
    const int* __restrict__ tokens, const int* __restrict__ positions,
    const bf16_t* __restrict__ te, const bf16_t* __restrict__ pe, bf16_t* __restrict__ out,
    float* __restrict__ rowsq, float* __restrict__ rowsum, int d) {
  __shared__ float scratch[NORM_THREADS / 64];
  const int row = blockIdx.x;
  const int nvec = d >> 3;
  const uint4* a = reinterpret_cast<const uint4*>(te + (size_t)max(tokens[row], 0) * d);
  const uint4* b = pe ? reinterpret_cast<const uint4*>(pe + (size_t)positions[row] * d) : nullptr;
  uint4* o = reinterpret_cast<uint4*>(out + (size_t)row * d);
  float ss = 0.f, s1 = 0.f;
#pragma unroll
  for (int i = 0; i < MAXV; ++i) {
    const int c = threadIdx.x + i * NORM_THREADS;
    if (c < nvec) {
      uint4 p = a[c];
      float x[8];
      if (b) {
        float y[8];
        unpack8(p, x);
        unpack8(b[c], y);
#pragma unroll
        for (int j = 0; j < 8; ++j) x[j] += y[j];
        p = pack8(x);
      }
      o[c] = p;
      unpack8(p, x);
#pragma unroll
      for (int j = 0; j < 8; ++j) {
        ss += x[j] * x[j];
        s1 += x[j];
      }
    }
  }
  ss = block_sum(ss, scratch);
  if (threadIdx.x == 0) rowsq[row] = ss;
  if (rowsum) {
    s1 = block_sum(s1, scratch);
    if (threadIdx.x == 0) rowsum[row] = s1;
  }
}

extern "C" int loqa_embed_stats(const int* tokens, const int* positions, const void* tok_embed,
                                const void* pos_embed, void* out, float* rowsq, float* rowsum,
                                int rows, int d, hipStream_t s) {
  if (rows <= 0) return 0;
  if (d % 8 || d > NORM_THREADS * 8 * MAXV || !rowsq) return (int)hipErrorInvalidValue;
  if (pos_embed && !positions) return (int)hipErrorInvalidValue;
  hipLaunchKernelGGL(embed_stats_kernel, dim3(rows), dim3(NORM_THREADS), 0, s, tokens, positions,
                     (const bf16_t*)tok_embed, (const bf16_t*)pos_embed, (bf16_t*)out, rowsq,
                     rowsum, d);
  return (int)hipGetLastError();
}
