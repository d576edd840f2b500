// Whisper audio front-end on the GPU (log_mel, im2col of the conv1d stem).
//
// log_mel: the STFT is a GEMM. A workgroup owns 16 frames of one utterance: their samples
// come to LDS once, are windowed and folded (y[n] + y[400 - n] for the cosines, y[n] -
// y[400 - n] for the sines: the basis rows n and 400 - n are equal up to the sine's sign,
// so half the K range does), eight waves run exact-f32 MFMA (v_mfma_f32_16x16x4_f32;
// log-mel needs f32 dynamic range) against the DFT basis, two bin tiles a wave, and square
// into LDS. A mel band is a handful of neighbouring bins, so the filterbank is a short sum
// per band over the bins where its row is not zero. log10 and the
// workgroup's maximum are fused into the epilogue, which writes time-major rows; a second
// kernel takes the utterance's maximum and applies whisper's max-8
// clamp and (x + 4) / 4 scaling and emits bf16, time-major (the conv stem's rows, padded
// with zero columns) or mel-major.
// One 30 s window, 80 / 128 mels: 69 / 92 us before (32 frames a workgroup, 94 of them, the
// whole K range, the filterbank as a GEMM whose operand loads formed one chain, an atomic per
// wave), 20 / 24 us now; what is left is the chain of basis loads of one workgroup per CU.
//
// im2col: k=3, pad=1 conv1d input unfolding so the conv becomes a plain GEMM
// (hipBLASLt) followed by the fused bias+GELU(+pos) epilogue (elementwise.hip).
#include "common.h"
#include <float.h>

#define NFFT 400
#define HOP 160
#define NBINS 201
#define BASIS_LD 224
#define FPW 16              // frames of a workgroup
#define SPAN ((FPW - 1) * HOP + NFFT)
#define FOLD_LD 208         // 201 taps, padded with zeros to whole k-steps (of 4)
#define POW_LD 209          // 13 tiles of 16 bins + 1

typedef float f4v __attribute__((ext_vector_type(4)));

// audio: [B, n_samples] f32;  window: [400];  cosb/sinb: [400, 224];  filt: [n_mels, 201];
// range: [n_mels, 2] first and past-the-last bin of each band;
// out: [B, n_frames, n_mels] f32 (log10 mel);  gmax: [B, gridDim.x] maximum of each workgroup
__global__ __launch_bounds__(512) void logmel_kernel(
    const float* __restrict__ audio, int n_samples, const float* __restrict__ window,
    const float* __restrict__ cosb, const float* __restrict__ sinb,
    const float* __restrict__ filt, const int* __restrict__ range, int n_mels, float* __restrict__ out,
    int n_frames, float* __restrict__ gmax) {
  __shared__ float raw[SPAN];
  __shared__ float even[FPW][FOLD_LD + 1], odd[FPW][FOLD_LD + 1];   // odd row strides: a lane per frame
  __shared__ float power[FPW][POW_LD];
  __shared__ float top[8];
  __shared__ int lost[FPW];            // the frame has bins that are not finite
  const int b = blockIdx.y, f0 = blockIdx.x * FPW;
  const float* x = audio + (size_t)b * n_samples;
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int fr = lane & 15, kq = lane >> 4;

  // wave w < 7 has the bins 32 w .. 32 w + 31 (201 of 224 exist); 52 k-steps of 4 taps (the last
  // ones meet zeros) in four blocks of 13, whose basis values are loaded one block ahead, the
  // first before the samples: the basis comes from far away when other work ran in between
  const int bin = wave * 32 + fr;
  const float* cb = cosb + (size_t)kq * BASIS_LD + bin;
  const float* sb = sinb + (size_t)kq * BASIS_LD + bin;
  float c[2][13][2], n[2][13][2];
  auto load = [&](int blk) __attribute__((always_inline)) {
#pragma unroll
    for (int u = 0; u < 13; ++u)
#pragma unroll
      for (int t = 0; t < 2; ++t) {
        c[blk & 1][u][t] = cb[(size_t)(52 * blk + 4 * u) * BASIS_LD + 16 * t];
        n[blk & 1][u][t] = sb[(size_t)(52 * blk + 4 * u) * BASIS_LD + 16 * t];
      }
  };
  if (wave < 7) load(0);

  if (threadIdx.x < FPW) lost[threadIdx.x] = 0;
  // the samples of all frames, reflected at the ends (center = True)
  for (int i = threadIdx.x; i < SPAN; i += 512) {
    int idx = f0 * HOP + i - NFFT / 2;
    if (idx < 0) idx = -idx;
    if (idx >= n_samples) idx = max(2 * (n_samples - 1) - idx, 0);   // frames past the end: any sample
    raw[i] = x[idx];
  }
  __syncthreads();
  for (int i = threadIdx.x; i < FPW * FOLD_LD; i += 512) {
    const int f = i / FOLD_LD, n = i - f * FOLD_LD;
    const float lo = n <= NFFT / 2 ? raw[f * HOP + n] * window[n] : 0.f;
    const bool two = n > 0 && n < NFFT / 2;
    const float hi = two ? raw[f * HOP + NFFT - n] * window[NFFT - n] : 0.f;
    even[f][n] = lo + hi;
    odd[f][n] = two ? lo - hi : 0.f;
  }
  __syncthreads();

  // power spectrum
  if (wave < 7) {
    f4v re[2] = {{0.f, 0.f, 0.f, 0.f}, {0.f, 0.f, 0.f, 0.f}}, im[2] = {{0.f, 0.f, 0.f, 0.f}, {0.f, 0.f, 0.f, 0.f}};
#pragma unroll
    for (int blk = 0; blk < 4; ++blk) {
      if (blk < 3) load(blk + 1);
#pragma unroll
      for (int u = 0; u < 13; ++u) {
        const int k = 52 * blk + 4 * u + kq;
        const float e = even[fr][k], o = odd[fr][k];
#pragma unroll
        for (int t = 0; t < 2; ++t) {
          re[t] = __builtin_amdgcn_mfma_f32_16x16x4f32(e, c[blk & 1][u][t], re[t], 0, 0, 0);
          im[t] = __builtin_amdgcn_mfma_f32_16x16x4f32(o, n[blk & 1][u][t], im[t], 0, 0, 0);
        }
      }
    }
    // column = lane & 15 (bin), row = 4 (lane / 16) + r (frame)
#pragma unroll
    for (int t = 0; t < 2; ++t)
#pragma unroll
      for (int r = 0; r < 4; ++r)
        if (bin + 16 * t < NBINS) {
          const float e = re[t][r] * re[t][r] + im[t][r] * im[t][r];
          power[4 * kq + r][bin + 16 * t] = e;
          if (!(e < INFINITY)) lost[4 * kq + r] = 1;
        }
  }
  __syncthreads();

  // a thread per band and four frames; a frame with samples that are not finite, or whose power is
  // not, counts as silent: the maximum below is of the others, which keep their values
  float wmax = -FLT_MAX;
  const int mel = threadIdx.x & 127, fg = threadIdx.x >> 7;
  if (mel < n_mels) {
    float acc[4] = {0.f, 0.f, 0.f, 0.f};
    const int hi = range[2 * mel + 1];
    for (int j = range[2 * mel]; j < hi; ++j) {
      const float w = filt[(size_t)mel * NBINS + j];
#pragma unroll
      for (int r = 0; r < 4; ++r) acc[r] += power[4 * fg + r][j] * w;
    }
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const int f = f0 + 4 * fg + r;
      if (f < n_frames) {
        const float lv = log10f(lost[4 * fg + r] ? 1e-10f : fmaxf(acc[r], 1e-10f));
        out[((size_t)b * n_frames + f) * n_mels + mel] = lv;
        wmax = fmaxf(wmax, lv);
      }
    }
  }
  wmax = wave_max(wmax);
  if (lane == 0) top[wave] = wmax;
  __syncthreads();
  if (threadIdx.x == 0) {
#pragma unroll
    for (int w = 1; w < 8; ++w) wmax = fmaxf(wmax, top[w]);
    gmax[(size_t)b * gridDim.x + blockIdx.x] = wmax;
  }
}

// x [B, frames, M] f32 -> (max(x, top - 8) + 4) / 4 in bf16, top the maximum of the utterance's
// `groups` entries of gmax: rows [B, frames, cols] with zeros in the columns from M on, or
// (cols = 0) mel-major [B, M, frames]. One utterance per blockIdx.y.
__global__ __launch_bounds__(256) void logmel_finalize_kernel(const float* __restrict__ x,
                                                              const float* __restrict__ gmax, int groups,
                                                              bf16_t* __restrict__ y, int frames, int M, int cols) {
  __shared__ float top[4];
  const int b = blockIdx.y;
  float mx = -FLT_MAX;
  for (int g = threadIdx.x; g < groups; g += 256) mx = fmaxf(mx, gmax[(size_t)b * groups + g]);
  mx = wave_max(mx);
  if ((threadIdx.x & 63) == 0) top[threadIdx.x >> 6] = mx;
  __syncthreads();
  const float lo = fmaxf(fmaxf(top[0], top[1]), fmaxf(top[2], top[3])) - 8.f;
  const int width = cols ? cols : M;
  const long long total = (long long)frames * width;
  x += (size_t)b * frames * M;
  y += (size_t)b * total;
  for (long long i = blockIdx.x * 256LL + threadIdx.x; i < total; i += gridDim.x * 256LL) {
    int t, m;
    if (cols) {
      t = (int)(i / cols);
      m = (int)(i - (long long)t * cols);
    } else {
      m = (int)(i / frames);
      t = (int)(i - (long long)m * frames);
    }
    const float v = m < M ? fmaxf(x[(size_t)t * M + m], lo) : -4.f;
    y[i] = f2bf((v + 4.f) * 0.25f);
  }
}

extern "C" int loqa_log_mel(const float* audio, int B, int n_samples, const float* window,
                            const float* cosb, const float* sinb, const float* filt, const int* range, int n_mels,
                            float* work, float* gmax, void* out_bf16, int n_frames, int cols,
                            hipStream_t s) {
  if (B <= 0) return 0;
  if (n_frames <= 0 || n_mels <= 0 || n_mels > 128 || n_samples <= NFFT / 2 || (cols && cols < n_mels))
    return (int)hipErrorInvalidValue;
  dim3 grid((n_frames + FPW - 1) / FPW, B);
  hipLaunchKernelGGL(logmel_kernel, grid, dim3(512), 0, s, audio, n_samples, window, cosb, sinb,
                     filt, range, n_mels, work, n_frames, gmax);
  hipError_t e = hipGetLastError();
  if (e != hipSuccess) return (int)e;
  long long blocks = ((long long)n_frames * (cols ? cols : n_mels) + 1023) / 1024;
  if (blocks > 8192) blocks = 8192;
  hipLaunchKernelGGL(logmel_finalize_kernel, dim3((unsigned)blocks, B), dim3(256), 0, s, work, gmax, (int)grid.x,
                     (bf16_t*)out_bf16, n_frames, n_mels, cols);
  return (int)hipGetLastError();
}

// --------------------------------------------------------------------- im2col
// x element (b, c, t) at x[b*sb + c*sc + t*st]; cols[(b*Lout + to), c*3 + k] =
// x[b, c, to*stride + k - 1] (zero outside [0, L)).  Row-major [B*Lout, 3C].
__global__ void im2col_k3_kernel(const bf16_t* __restrict__ x, long long sb, long long sc,
                                 long long st, int C, int L, int Lout, int stride,
                                 bf16_t* __restrict__ cols, long long total) {
  for (long long i = blockIdx.x * (long long)blockDim.x + threadIdx.x; i < total;
       i += (long long)gridDim.x * blockDim.x) {
    const long long row = i / (3LL * C);
    const int col = (int)(i - row * 3LL * C);
    const int b = (int)(row / Lout), to = (int)(row - (long long)b * Lout);
    const int c = col / 3, k = col - c * 3;
    const int t = to * stride + k - 1;
    cols[i] = (t >= 0 && t < L) ? x[b * sb + c * sc + t * st] : (bf16_t)0;
  }
}

extern "C" int loqa_im2col_k3(const void* x, long long sb, long long sc, long long st, int B,
                              int C, int L, int stride, void* cols, hipStream_t s) {
  if (B <= 0) return 0;
  const int Lout = (L + 2 - 3) / stride + 1;
  const long long total = (long long)B * Lout * 3 * C;
  long long blocks = (total + 255) / 256;
  if (blocks > 16384) blocks = 16384;
  hipLaunchKernelGGL(im2col_k3_kernel, dim3((unsigned)blocks), dim3(256), 0, s, (const bf16_t*)x,
                     sb, sc, st, C, L, Lout, stride, (bf16_t*)cols, total);
  return (int)hipGetLastError();
}
