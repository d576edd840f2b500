// Whisper audio front-end on the GPU (log_mel, im2col of the conv1d stem).
//
// log_mel: the STFT is a GEMM. A workgroup owns 16 frames of one utterance: their samples
// come to LDS once, are windowed and folded twice. The basis rows n and 400 - n are equal up
// to the sine's sign, and so are the rows n and 200 - n up to a sign that only the bin's parity
// decides: with e[n] = y[n] + y[400 - n] and o[n] = y[n] - y[400 - n], the even bins are products
// with e[n] + e[200 - n] and o[n] - o[200 - n], the odd ones with e[n] - e[200 - n] and
// o[n] + o[200 - n], all over 101 of the 400 taps. Seven waves run exact-f32 MFMA
// (v_mfma_f32_16x16x4_f32; log-mel needs f32 dynamic range) against the DFT basis, each a tile
// of 16 even bins and one of the 16 odd bins beside them (a lane loads both at once), and square
// into LDS. A mel band is a handful of neighbouring bins, so the filterbank is a short sum
// per band over the bins where its row is not zero, its weights loaded at the start. log10 and the
// workgroup's maximum are fused into the epilogue, which writes time-major rows; a second
// kernel takes the utterance's maximum and applies whisper's max-8
// clamp and (x + 4) / 4 scaling and emits bf16, time-major (the conv stem's rows, padded
// with zero columns) or mel-major.
// What bounds one window is the basis, 182 KB that every CU reads from far away at about 50 KB / us
// (samples and basis 6 us, folding 1, MFMA 3 of 12), so a CU's workgroup keeps it in registers for
// every 256th group of frames and has the next group's samples under way.
// Both launches, caches cold, 80 mels, 1 / 6 / 16 windows of 30 s: 30 / 85 / 188 us with one fold, a
// basis read per group and a 64-bit division per output element, 21 / 48 / 95 us now.
//
// im2col: k=3, pad=1 conv1d input unfolding so the conv becomes a plain GEMM
// (hipBLASLt) followed by the fused bias+GELU(+pos) epilogue (elementwise.hip).
#include "common.h"
#include <float.h>
#include <limits.h>

#define NFFT 400
#define HOP 160
#define NBINS 201
#define BASIS_LD 224
#define FPW 16              // frames of a workgroup
#define SPAN ((FPW - 1) * HOP + NFFT)
#define TAPS 101            // of the folded frame: 0 .. 100
#define FOLD_LD 104         // padded with zeros to whole k-steps (of 4)
#define KSTEPS (FOLD_LD / 4)
#define SPT ((SPAN + 511) / 512)   // samples of a thread
#define BANDW 16            // weights of a band that are loaded ahead (80 mels: at most 15)
#define LM_WGS 256          // a CU's workgroup keeps its basis for every CUs-th group of frames
#define POW_LD 20           // frames of a bin's power, 16-byte aligned, off the bank stride

typedef float f4v __attribute__((ext_vector_type(4)));
typedef float f2v __attribute__((ext_vector_type(2)));

// audio: [B, n_samples] f32;  window: [400];  cosb/sinb: [400, 224], 8-byte aligned;  filt: [n_mels, 201];
// range: [n_mels, 2] first and past-the-last bin of each band;
// out: [B, n_frames, n_mels] f32 (log10 mel);  gmax: [B, groups] maximum of each group of FPW frames; items = B groups
__global__ __launch_bounds__(512) void logmel_kernel(
    const float* __restrict__ audio, int n_samples, const float* __restrict__ window,
    const float* __restrict__ cosb, const float* __restrict__ sinb,
    const float* __restrict__ filt, const int* __restrict__ range, int n_mels, float* __restrict__ out,
    int n_frames, float* __restrict__ gmax, int groups, int items) {
  __shared__ float raw[SPT * 512], hann[512];
  // by the bin's parity; odd row strides: a lane per frame
  __shared__ float even[2][FPW][FOLD_LD + 1], odd[2][FPW][FOLD_LD + 1];
  __shared__ __attribute__((aligned(16))) float power[NBINS][POW_LD];
  __shared__ float top[8];
  __shared__ int lost[FPW];            // the frame has bins that are not finite
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int fr = lane & 15, kq = lane >> 4;

  // the samples of an item's frames, reflected at the ends (center = True)
  float smp[SPT];
  auto fetch = [&](int item) __attribute__((always_inline)) {
    const int b = item / groups;
    const float* x = audio + (size_t)b * n_samples;
    const int first = (item - b * groups) * (FPW * HOP) - NFFT / 2;
#pragma unroll
    for (int u = 0; u < SPT; ++u) {
      int idx = first + u * 512 + threadIdx.x;
      if (idx < 0) idx = -idx;
      if (idx >= n_samples) idx = max(2 * (n_samples - 1) - idx, 0);   // past the end: any sample
      smp[u] = x[idx];
    }
  };
  fetch(blockIdx.x);
  __builtin_amdgcn_s_barrier();            // every wave's samples before any wave's basis
  const float hw = window[min((int)threadIdx.x, NFFT - 1)];
  // a thread per band and four frames
  const int mel = threadIdx.x & 127, fg = threadIdx.x >> 7;
  const int mrow = min(mel, n_mels - 1);
  const int blo = range[2 * mrow], bhi = range[2 * mrow + 1];
  // wave w < 7 has the bins 32 w .. 32 w + 31 (201 of 224 exist), a lane the bins 32 w + 2 fr and
  // the next; the last of the 26 k-steps of 4 taps meets zeros. Wave 7 loads with the others, one
  // cache line a time: a load that some waves skip would make all of them wait for the basis where
  // the samples are needed.
  const int bin = wave * 32 + 2 * fr;
  const int col = wave < 7 ? kq * BASIS_LD + bin : 0;
  f2v c[KSTEPS], n[KSTEPS];
#pragma unroll
  for (int u = 0; u < KSTEPS; ++u) {
    c[u] = *(const f2v*)(cosb + 4 * u * BASIS_LD + col);
    n[u] = *(const f2v*)(sinb + 4 * u * BASIS_LD + col);
  }
  __builtin_amdgcn_sched_barrier(0);       // all of these are in flight before the first wait
  auto put = [&]() __attribute__((always_inline)) {
#pragma unroll
    for (int u = 0; u < SPT; ++u) raw[u * 512 + threadIdx.x] = smp[u];
  };
  put();
  hann[threadIdx.x] = hw;
  float bw[BANDW];
#pragma unroll
  for (int u = 0; u < BANDW; ++u) bw[u] = filt[(size_t)mrow * NBINS + min(blo + u, NBINS - 1)];

  int item = blockIdx.x;
  do {
    const int b = item / groups, f0 = (item - b * groups) * FPW;
    __syncthreads();
    if (threadIdx.x < FPW) lost[threadIdx.x] = 0;
    fetch(item + (int)gridDim.x < items ? item + (int)gridDim.x : item);
    for (int i = threadIdx.x; i < FPW * FOLD_LD; i += 512) {
      const int f = i / FOLD_LD, n = i - f * FOLD_LD;
      const float* y = raw + f * HOP;
      auto at = [&](int j) __attribute__((always_inline)) { return y[j] * hann[j]; };
      float e = 0.f, o = 0.f, em = 0.f, om = 0.f;      // of tap n and of its mirror 200 - n
      if (n < TAPS) {
        const float a = at(n), d = at(NFFT / 2 - n);
        const float b = n > 0 ? at(NFFT - n) : 0.f, g = n > 0 ? at(NFFT / 2 + n) : 0.f;
        e = a + b;
        o = n > 0 ? a - b : 0.f;
        if (n < TAPS - 1) {                            // tap 100 is its own mirror
          em = d + g;
          om = n > 0 ? d - g : 0.f;
        }
      }
      even[0][f][n] = e + em;
      even[1][f][n] = e - em;
      odd[0][f][n] = o - om;
      odd[1][f][n] = o + om;
    }
    __syncthreads();

    // power spectrum
    if (wave < 7) {
      f4v re[2] = {{0.f, 0.f, 0.f, 0.f}, {0.f, 0.f, 0.f, 0.f}}, im[2] = {{0.f, 0.f, 0.f, 0.f}, {0.f, 0.f, 0.f, 0.f}};
#pragma unroll
      for (int u = 0; u < KSTEPS; ++u)
#pragma unroll
        for (int t = 0; t < 2; ++t) {
          re[t] = __builtin_amdgcn_mfma_f32_16x16x4f32(even[t][fr][4 * u + kq], c[u][t], re[t], 0, 0, 0);
          im[t] = __builtin_amdgcn_mfma_f32_16x16x4f32(odd[t][fr][4 * u + kq], n[u][t], im[t], 0, 0, 0);
        }
      // column = lane & 15 (bin), row = 4 (lane / 16) + r (frame)
#pragma unroll
      for (int t = 0; t < 2; ++t)
        if (bin + t < NBINS) {
          const f4v e = re[t] * re[t] + im[t] * im[t];
          *(f4v*)&power[bin + t][4 * kq] = e;
#pragma unroll
          for (int r = 0; r < 4; ++r)
            if (!(e[r] < INFINITY)) lost[4 * kq + r] = 1;
        }
    }
    put();
    __syncthreads();

    // a frame with samples that are not finite, or whose power is not, counts as silent: the maximum
    // below is of the others, which keep their values
    float wmax = -FLT_MAX;
    if (mel < n_mels) {
      f4v acc = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int u = 0; u < BANDW; ++u) {
        asm volatile("" : "+v"(bw[u]));                // the selection stays here: it waits for the load
        if (u % 4 == 0 && !__any(blo + u < bhi)) break;
        const float w = blo + u < bhi ? bw[u] : 0.f;
        acc += *(const f4v*)&power[max(min(blo + u, bhi - 1), 0)][4 * fg] * w;
      }
      for (int j = blo + BANDW; j < bhi; ++j) acc += *(const f4v*)&power[j][4 * fg] * filt[(size_t)mel * NBINS + j];
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
      gmax[item] = wmax;
    }
    item += gridDim.x;
  } while (item < items);
}

// The utterance's maximum, of its `groups` entries of gmax, less 8.
static __device__ __forceinline__ float logmel_floor(const float* __restrict__ gmax, int groups) {
  __shared__ float top[4];
  float mx = -FLT_MAX;
  for (int g = threadIdx.x; g < groups; g += 256) mx = fmaxf(mx, gmax[(size_t)blockIdx.y * groups + g]);
  mx = wave_max(mx);
  if ((threadIdx.x & 63) == 0) top[threadIdx.x >> 6] = mx;
  __syncthreads();
  return fmaxf(fmaxf(top[0], top[1]), fmaxf(top[2], top[3])) - 8.f;
}

// x [B, frames, M] f32 -> (max(x, top - 8) + 4) / 4 in bf16, mel-major [B, M, frames]. One
// utterance per blockIdx.y.
__global__ __launch_bounds__(256) void logmel_finalize_kernel(const float* __restrict__ x,
                                                              const float* __restrict__ gmax, int groups,
                                                              bf16_t* __restrict__ y, int frames, int M) {
  const float lo = logmel_floor(gmax, groups);
  const long long total = (long long)frames * M;
  x += blockIdx.y * total;
  y += blockIdx.y * total;
  for (long long i = blockIdx.x * 256LL + threadIdx.x; i < total; i += gridDim.x * 256LL) {
    const int m = (int)(i / frames);
    const int t = (int)(i - (long long)m * frames);
    y[i] = f2bf((fmaxf(x[(size_t)t * M + m], lo) + 4.f) * 0.25f);
  }
}

// The same as rows [B, frames, cols] with zeros in the columns from M on: a wave per row, V columns
// a lane (with a 64-bit division per element 16 windows took 17 us, now 9).
template <int V>
__global__ __launch_bounds__(256) void logmel_rows_kernel(const float* __restrict__ x,
                                                          const float* __restrict__ gmax, int groups,
                                                          bf16_t* __restrict__ y, int frames, int M, int cols) {
  typedef float xv __attribute__((ext_vector_type(V)));
  typedef unsigned short yv __attribute__((ext_vector_type(V)));
  const float lo = logmel_floor(gmax, groups);
  for (int t = blockIdx.x * 4 + (threadIdx.x >> 6); t < frames; t += gridDim.x * 4) {
    const size_t row = (size_t)blockIdx.y * frames + t;
    for (int m = (threadIdx.x & 63) * V; m < cols; m += 64 * V) {
      xv v = (xv)-4.f;
      if (m < M) v = *(const xv*)(x + row * M + m);
      yv o;
#pragma unroll
      for (int u = 0; u < V; ++u) o[u] = m < M ? f2bf((fmaxf(v[u], lo) + 4.f) * 0.25f) : (bf16_t)0;
      *(yv*)(y + row * cols + m) = o;
    }
  }
}

extern "C" int loqa_log_mel(const float* audio, int B, int n_samples, const float* window,
                            const float* cosb, const float* sinb, const float* filt, const int* range, int n_mels,
                            float* work, float* gmax, void* out_bf16, int n_frames, int cols,
                            hipStream_t s) {
  if (B <= 0) return 0;
  if (n_frames <= 0 || n_mels <= 0 || n_mels > 128 || n_samples <= NFFT / 2 || (cols && cols < n_mels))
    return (int)hipErrorInvalidValue;
  const int groups = (n_frames + FPW - 1) / FPW;
  const long long items = (long long)B * groups;
  if (items > INT_MAX - LM_WGS) return (int)hipErrorInvalidValue;
  hipLaunchKernelGGL(logmel_kernel, dim3((unsigned)(items < LM_WGS ? items : LM_WGS)), dim3(512), 0, s, audio,
                     n_samples, window, cosb, sinb, filt, range, n_mels, work, n_frames, gmax, groups, (int)items);
  hipError_t e = hipGetLastError();
  if (e != hipSuccess) return (int)e;
  if (cols) {
    const dim3 rows((n_frames + 15) / 16, B);
    // four columns a lane where the rows of both sides keep their alignment
    if (n_mels % 4 == 0 && cols % 4 == 0 && (uintptr_t)work % 16 == 0 && (uintptr_t)out_bf16 % 8 == 0)
      hipLaunchKernelGGL((logmel_rows_kernel<4>), rows, dim3(256), 0, s, work, gmax, groups, (bf16_t*)out_bf16,
                         n_frames, n_mels, cols);
    else
      hipLaunchKernelGGL((logmel_rows_kernel<1>), rows, dim3(256), 0, s, work, gmax, groups, (bf16_t*)out_bf16,
                         n_frames, n_mels, cols);
  } else {
    long long blocks = ((long long)n_frames * n_mels + 1023) / 1024;
    if (blocks > 8192) blocks = 8192;
    hipLaunchKernelGGL(logmel_finalize_kernel, dim3((unsigned)blocks, B), dim3(256), 0, s, work, gmax, groups,
                       (bf16_t*)out_bf16, n_frames, n_mels);
  }
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
