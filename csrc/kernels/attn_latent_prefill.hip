// Prompt-pass latent attention on the matrix cores (bf16).
//
// For passes with many query rows the folded form (attn_latent.hip) would pay
// R + Dr multiply-adds per score and R per value entry; here the keys and
// values are first materialised per head from the latent rows (latent_kv.hip), and the pipelined
// tile loop of the other prompt attentions (flash_pipe.h) runs over [key, head, DK] / [key, head, DV].
// Queries may come unrotated: a row's entries are turned as they are loaded. What is its own: DK != DV
// (rotary part only in the keys), zero-padded head sizes (DK, DV are the next instantiated sizes), the
// causal bound from each row's absolute position (with a sliding window the keys before it are neither
// gathered nor visited), a learned per-head sink in the softmax denominator, and the output gate
// sigmoid(gate), applied before the unpadded heads go to rows of any stride. Numerator and denominator
// are of the same rounded weights (flash_pipe.h has the errors).
// 2048 rows of 16 heads, 192 / 128: 99.5 us before (128 rows in four waves, tiles through
// registers, scores, exponentials and products one after the other), 55 now; 4 x that: 365, 120;
// 256 / 128: 111, 75. A single prompt is one round of the CUs, as long as its last rows (32
// tiles, 16.5 on average); smaller blocks with one wave a SIMD were no faster.
// Few rows behind many keys: parts of a block's keys in workgroups of their own, joined in the launch (fl_join).
//
// Helpers, for the sizes and alignments that latent_kv.hip does not take and queries that come turned:
// latent_gather_kernel copies the last cu_k[b + 1] - cu_k[b] latent rows
// of each sequence from its pages into contiguous [sum L, R] / [sum L, Dr] buffers; latent_kfill_kernel
// writes the shared rotary key part into every head's key row;
// rope_pairs_kernel rotates the queries' rotary part in place.
#include "flash_pipe.h"
#include "seqmix.h"

struct LatPrefillParams {
  const bf16_t* q; long q_st;       // [T, H, DK]
  const bf16_t* k;                  // [sum L, H, DK]
  const bf16_t* v;                  // [sum L, H, DV]
  bf16_t* o; long o_ld;             // [T, H * Dv], row stride o_ld
  const int* cu_q; const int* cu_k; const int* pos;
  const int* ctx;                   // [B] keys in the cache; the buffer holds the last of them
  const float* sink; float scale_log2;
  int H, Dv, window;
  const bf16_t* gate; long gate_ld; // [T, H * Dv] or null
  const float* cs; int max_pos, rot0, rot_dims;   // queries to be rotated: tables, first entry and width (null: done)
  int parts; float* part; int* words;             // parts of a block's keys at most (fl_join)
  int runs, rows16;                 // gate rows can be read in runs of four, output rows written in runs of eight
};

// QW blocks of 32 query rows, the keys in KS runs. At 192 / 128 a run's ring is 80 KB of LDS and a
// tile's working set with two waves a SIMD all of the registers; the 256-column keys take one wave.
// The bound of two stands also where LDS holds one (64 rows in two runs): from 257 registers on the
// compiler keeps MFMA results in the accumulation registers and moves them for every rescaling.
// us with 256 registers (10 spilled at 192 / 128) and with 320 (none): 300 rows x 16 heads 13.8, 14.7;
// 2048 x 8 heads 37.2, 41.8, at 128 / 128 30.6, 36.9.
// PARTS: of a block's keys, a kernel of its own (in one with the others these took 0.2 to 0.6 us more, 17 rows x 16 heads of
// 256 / 64 8.4 us, 7.8 alone).
template <int DK, int DV, int QW, int KS, bool PARTS>
__global__ __launch_bounds__(64 * QW * KS, DK > 192 ? 1 : 2) void latent_prefill_kernel(LatPrefillParams p) {
  using L = FlashLds<DK, DV>;
  constexpr int NS = DK / 16, NDT = DV / 32, NTH = 64 * QW;
  extern __shared__ __attribute__((aligned(16))) unsigned char lds[];
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int run = wave / QW, wq = wave % QW, th = threadIdx.x - run * NTH, h = lane >> 5;
  int bx, head, b, share = 0;
  {
    // row blocks with the most keys first, over all heads of an XCD where these are whole
    const int gx = gridDim.x, gy = gridDim.y, heads = gy * gridDim.z;
    const int at = xcd_remap(blockIdx.x + gx * (blockIdx.y + gy * blockIdx.z), gx * heads);
    int hd = at / gx;
    bx = at - hd * gx;
    if (heads % 8 == 0) {
      const int hp = heads / 8, xcd = at / (hp * gx), in = at - xcd * hp * gx;
      bx = in / hp;
      hd = xcd * hp + in - bx * hp;
    }
    if constexpr (PARTS) {
      const int block = bx / p.parts;
      share = bx - block * p.parts;
      bx = gx / p.parts - 1 - block;
    } else {
      bx = gx - 1 - bx;
    }
    b = hd / gy;
    head = hd - b * gy;
  }
  const int q0 = p.cu_q[b], qlen = p.cu_q[b + 1] - q0;
  const int row_lo = bx * (32 * QW);
  if (row_lo >= qlen) return;                             // whole workgroup: uniform
  const int row_hi = min(qlen - 1, row_lo + 32 * QW - 1);
  const int k0 = p.cu_k[b], klen = p.cu_k[b + 1] - k0;
  const int koff = p.ctx[b] - klen;                       // position of the buffer's first key
  const int qi = row_lo + wq * 32 + (lane & 31);
  const bool valid = qi < qlen;
  // positions relative to the buffer's first key
  const int qpos = p.pos[q0 + min(qi, row_hi)] - koff;
  int kend = min(klen, p.pos[q0 + row_hi] - koff + 1);         // positions grow along a sequence
  int kt0 = p.window > 0 ? max(0, p.pos[q0 + row_lo] - koff - p.window + 1) / FL_KEYS * FL_KEYS : 0;
  int ntiles = kend > kt0 ? (kend - kt0 + FL_KEYS - 1) / FL_KEYS : 0, parts = 1;
  if constexpr (PARTS) {
    parts = max(1, min(p.parts, ntiles / FL_CAP));
    if (share >= parts) return;                           // uniform
    const int len = (ntiles + parts - 1) / parts;
    kt0 += share * len * FL_KEYS;
    kend = min(kend, kt0 + len * FL_KEYS);
    ntiles = max(0, min(len, ntiles - share * len));
  }
  // what this wave's rows see at all
  const int wpos_lo = __builtin_amdgcn_readfirstlane(p.pos[q0 + min(row_lo + wq * 32, row_hi)]) - koff;
  const int wpos_hi = __builtin_amdgcn_readfirstlane(p.pos[q0 + min(row_lo + wq * 32 + 31, row_hi)]) - koff;
  const int per = (ntiles + KS - 1) / KS, first = run * per;

  // where a fetch stands: tiles come in order; past the last one it stays there
  const FlFetch<DK, NTH, false, false> kf(th, DK, (long long)p.H * DK);
  const FlFetch<DV, NTH, true, false> vf(th, DV, (long long)p.H * DV);
  struct At {
    const bf16_t* row;
    int kt;
  };
  const int at0 = kt0 + max(min(first, ntiles - 1), 0) * FL_KEYS;
  At ka{p.k + ((size_t)(k0 + at0) * p.H + head) * DK, at0}, va{p.v + ((size_t)(k0 + at0) * p.H + head) * DV, at0};
  auto fetch = [&](const auto& f, At& a, int cols, unsigned stage) __attribute__((always_inline)) {
    const int last = kend - 1 - a.kt;
    f.strided(stage, a.row, last);
    if (last >= FL_KEYS) {
      a.row += (size_t)FL_KEYS * p.H * cols;
      a.kt += FL_KEYS;
    }
  };
  const unsigned ring = fl_lds_at(lds) + run * L::RING;
  if (per > 0) fetch(kf, ka, DK, ring);

  bf16x8 qf[NS];
  {
    const bf16_t* qrow = p.q + (size_t)(q0 + min(qi, row_hi)) * p.q_st + (size_t)head * DK;
#pragma unroll
    for (int s = 0; s < NS; ++s) {
      uint4 v = valid ? *reinterpret_cast<const uint4*>(qrow + 16 * s + 8 * h) : make_uint4(0, 0, 0, 0);
      const int e = 16 * s + 8 * h - p.rot0;
      if (p.cs && e >= 0 && e < p.rot_dims) {
        const float* c = p.cs + (size_t)min(max(p.pos[q0 + min(qi, row_hi)], 0), p.max_pos - 1) * p.rot_dims + e;
        float t[8], f[8];
        ld_run<float, 4>(c, t);
        ld_run<float, 4>(c + 4, t + 4);
        unpack8(v, f);
#pragma unroll
        for (int i = 0; i < 8; i += 2) {
          const float a = f[i], z = f[i + 1];
          f[i] = a * t[i] - z * t[i + 1];
          f[i + 1] = z * t[i] + a * t[i + 1];
        }
        v = pack8(f);
      }
      qf[s] = *reinterpret_cast<const bf16x8*>(&v);
    }
  }
  float16v acc[NDT];
#pragma unroll
  for (int i = 0; i < NDT; ++i)
#pragma unroll
    for (int j = 0; j < 16; ++j) acc[i][j] = 0.f;
  float m = -1e30f, l = 0.f;
  const float sink = p.sink ? p.sink[head] : 0.f;
  const bool neg = !(p.scale_log2 > 0.f);                 // the loop's maxima are of growing scores
  fl_loop<DK, DV, kf.N + vf.N, true>(
      qf, acc, m, l, ring, per, neg ? 1.f : p.scale_log2, lane, true,
      // (64 columns on two runs are 3 % faster in step: 2048 rows x 32 heads, 700 x 16)
      QW * KS == 8 && (KS == 4 || DK > 64 || DV > 64) ? wave >> 2 : -1,
      [&](float16v(&st)[2], int i) __attribute__((always_inline)) {
        const int kt = kt0 + (first + i) * FL_KEYS;       // tiles past the last lie behind kend
        if (neg) {
#pragma unroll
          for (int t = 0; t < 2; ++t)
#pragma unroll
            for (int j = 0; j < 16; ++j) st[t][j] *= p.scale_log2;
        }
        // a tile that every row of this wave sees whole needs no per-score tests
        const bool whole = kt + FL_KEYS - 1 <= wpos_lo && kt + FL_KEYS <= kend && (p.window <= 0 || wpos_hi - kt < p.window);
        if (!whole) {
          const int lim = min(kend, qpos + 1) - kt - 4 * h;
          const int lo = p.window > 0 ? qpos - p.window + 1 - kt - 4 * h : -FL_KEYS;
#pragma unroll
          for (int t = 0; t < 2; ++t)
#pragma unroll
            for (int j = 0; j < 16; ++j) {
              const int c = 32 * t + (j & 3) + 8 * (j >> 2);
              if (c >= lim || c < lo) st[t][j] = -INFINITY;
            }
        }
      },
      [&](int, unsigned stage) __attribute__((always_inline)) { fetch(kf, ka, DK, stage); },
      [&](int, unsigned stage) __attribute__((always_inline)) { fetch(vf, va, DV, stage); });

  fl_sync();                                              // every wave is done with the rings
  constexpr int OWN = FlEnd<NDT, QW, KS, PARTS>::OWN;
  const bf16_t* grow = p.gate ? p.gate + (size_t)(q0 + min(qi, row_hi)) * p.gate_ld + (size_t)head * p.Dv : nullptr;
  float4v own[OWN];
  uint2 gate[OWN];
  auto ask = [&]() __attribute__((always_inline)) {       // the gates of the run's own units
#pragma unroll
    for (int s = 0; s < OWN; ++s) {
      const int d0 = fl_column<NDT, QW, KS, PARTS>(s, run, lane);
      gate[s] = make_uint2(0, 0);
      if (grow && p.runs) {
        if (d0 < p.Dv) gate[s] = *reinterpret_cast<const uint2*>(grow + d0);
      } else if (grow) {
        unsigned e[4];
#pragma unroll
        for (int i = 0; i < 4; ++i) e[i] = d0 + i < p.Dv ? grow[d0 + i] : 0u;
        gate[s] = make_uint2(e[0] | e[1] << 16, e[2] | e[3] << 16);
      }
    }
  };
  if constexpr (!PARTS) ask();                            // on their way while the runs meet
  fl_merge<NDT, QW, KS, PARTS>(acc, own, m, l, lds, run, wq, lane);
  if constexpr (PARTS) {
    if (run) return;
    const int block = (b * p.H + head) * (int)(gridDim.x / p.parts) + bx;
    if (parts > 1 && !fl_join<NDT, QW>(acc, m, l, p.part + (size_t)block * p.parts * QW * fl_join_floats(NDT),
                                       p.words + (size_t)block * TICKET, parts, share, wq, lane))
      return;
    fl_units(acc, own);
    ask();
  }
  // the sink joins the denominator only (log2 domain, like the scores)
  float f = 1.f, den = l;
  if (p.sink) {
    const float sk = sink * 1.4426950408889634f;
    const float M = fmaxf(m, sk);
    f = exp2f(m - M);
    den = l * f + exp2f(sk - M);
  }
  const float inv = den > 0.f ? f / den : 0.f;
#pragma unroll
  for (int s = 0; s < OWN; ++s) {
    const unsigned g[2] = {gate[s].x, gate[s].y};
#pragma unroll
    for (int i = 0; i < 4; ++i) own[s][i] *= grow ? inv * sigmoid_fast(__uint_as_float(i % 2 ? g[i / 2] & 0xffff0000u : g[i / 2] << 16)) : inv;
  }
  if (p.rows16) {
    fl_store<NDT, QW, KS, PARTS>(own, lds, p.o + (size_t)(q0 + row_lo + wq * 32) * p.o_ld + (size_t)head * p.Dv, p.o_ld,
                                 qlen - row_lo - wq * 32, p.Dv, run, wq, lane);
  } else if (valid) {
    bf16_t* orow = p.o + (size_t)(q0 + qi) * p.o_ld + (size_t)head * p.Dv;
#pragma unroll
    for (int s = 0; s < OWN; ++s)
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const int e = fl_column<NDT, QW, KS, PARTS>(s, run, lane) + i;
        if (e < p.Dv) orow[e] = f2bf(own[s][i]);
      }
  }
}

__global__ __launch_bounds__(256) void latent_gather_kernel(
    const bf16_t* __restrict__ cache, int blk, const int* __restrict__ bt, int max_blocks,
    const int* __restrict__ cu_k, const int* __restrict__ ctx, int R, int Dr,
    bf16_t* __restrict__ cl, bf16_t* __restrict__ kr) {
  const int b = blockIdx.y;
  const int k0 = cu_k[b], L = cu_k[b + 1] - k0, off = ctx[b] - L;
  const int W = R + Dr;
  for (int j = blockIdx.x * 4 + (threadIdx.x >> 6); j < L; j += gridDim.x * 4) {
    const int jp = off + j;
    const bf16_t* src = cache + ((size_t)bt[(size_t)b * max_blocks + jp / blk] * blk + jp % blk) * W;
    for (int c = threadIdx.x & 63; c < W; c += 64) {
      if (c < R) cl[(size_t)(k0 + j) * R + c] = src[c];
      else kr[(size_t)(k0 + j) * Dr + (c - R)] = src[c];
    }
  }
}

// k[j, h, D + i] = kr[j, i]: the shared rotary key part into every head's row.
__global__ __launch_bounds__(256) void latent_kfill_kernel(bf16_t* __restrict__ k,
                                                           const bf16_t* __restrict__ kr, int H,
                                                           int DKp, int D, int Dr) {
  const size_t j = blockIdx.x;
  for (int i = threadIdx.x; i < H * Dr; i += blockDim.x) {
    const int hh = i / Dr, c = i - hh * Dr;
    k[(j * H + hh) * DKp + D + c] = kr[j * Dr + c];
  }
}

// x[t, h, off + 2i], x[t, h, off + 2i + 1] rotated by the angle of (pos[t], i).
__global__ __launch_bounds__(256) void rope_pairs_kernel(bf16_t* __restrict__ x, long st_t, long st_h,
                                                         int H, int off, int dims,
                                                         const int* __restrict__ pos,
                                                         const float* __restrict__ cs, int max_pos) {
  const size_t t = blockIdx.x;
  const int p = min(max(pos[t], 0), max_pos - 1);
  const float* csr = cs + (size_t)p * dims;
  const int half = dims / 2;
  for (int i = threadIdx.x; i < H * half; i += blockDim.x) {
    const int hh = i / half, pr = i - hh * half;
    bf16_t* e = x + t * st_t + (size_t)hh * st_h + off + 2 * pr;
    const float c = csr[2 * pr], s = csr[2 * pr + 1];
    const float u = bf2f(e[0]), v = bf2f(e[1]);
    e[0] = f2bf(u * c - v * s);
    e[1] = f2bf(v * c + u * s);
  }
}

extern "C" int loqa_latent_gather(const void* cache, int blk, const void* bt, int max_blocks,
                                  const void* cu_k, const void* ctx, int B, int max_len, int R,
                                  int Dr, void* cl, void* kr, hipStream_t st) {
  if (B <= 0 || max_len <= 0) return 0;
  const dim3 grid(min(1024, (max_len + 3) / 4), B);
  hipLaunchKernelGGL(latent_gather_kernel, grid, dim3(256), 0, st, (const bf16_t*)cache, blk,
                     (const int*)bt, max_blocks, (const int*)cu_k, (const int*)ctx, R, Dr, (bf16_t*)cl, (bf16_t*)kr);
  return (int)hipGetLastError();
}

extern "C" int loqa_latent_kfill(void* k, const void* kr, int L, int H, int DKp, int D, int Dr,
                                 hipStream_t st) {
  if (L <= 0) return 0;
  hipLaunchKernelGGL(latent_kfill_kernel, dim3(L), dim3(256), 0, st, (bf16_t*)k, (const bf16_t*)kr, H,
                     DKp, D, Dr);
  return (int)hipGetLastError();
}

extern "C" int loqa_rope_pairs(void* x, long st_t, long st_h, int T, int H, int off, int dims,
                               const void* pos, const void* cs, int max_pos, hipStream_t st) {
  if (T <= 0 || dims <= 0) return 0;
  hipLaunchKernelGGL(rope_pairs_kernel, dim3(T), dim3(256), 0, st, (bf16_t*)x, st_t, st_h, H, off,
                     dims, (const int*)pos, (const float*)cs, max_pos);
  return (int)hipGetLastError();
}

// DK in {64, 128, 192, 256}, DV in {64, 128}: callers pad head sizes up; the
// output keeps the model's value size Dv <= DV.
extern "C" int loqa_latent_prefill(const void* q, long q_st, const void* k, const void* v, void* o,
                                   long o_ld, const void* cu_q, const void* cu_k, const void* ctx,
                                   const void* pos, const void* sink, float scale, int window,
                                   const void* gate, long gate_ld, int B, int H, int max_q, int DK,
                                   int DV, int Dv, const void* cs, int max_pos, int rot0, int rot_dims,
                                   int parts, float* part, long part_floats, int* words, long tickets,
                                   hipStream_t st) {
  if (B <= 0 || H <= 0 || max_q <= 0) return 0;
  if (cs && (max_pos <= 0 || rot0 < 0 || rot0 % 8 || rot_dims <= 0 || rot_dims % 8 || rot0 + rot_dims > DK || ((size_t)cs & 15)))
    return (int)hipErrorInvalidValue;
  if (Dv <= 0 || Dv > DV || o_ld < (long)H * Dv || !ctx) return (int)hipErrorInvalidValue;
  LatPrefillParams p;
  p.q = (const bf16_t*)q; p.q_st = q_st; p.k = (const bf16_t*)k; p.v = (const bf16_t*)v;
  p.o = (bf16_t*)o; p.o_ld = o_ld; p.cu_q = (const int*)cu_q; p.cu_k = (const int*)cu_k;
  p.pos = (const int*)pos; p.ctx = (const int*)ctx; p.Dv = Dv; p.window = window;
  p.sink = (const float*)sink; p.scale_log2 = scale * 1.4426950408889634f; p.H = H;
  p.gate = (const bf16_t*)gate; p.gate_ld = gate_ld;
  p.parts = parts; p.part = part; p.words = words;
  if (parts < 1 || parts > FL_PARTS || (parts > 1 && (!part || !words || ((size_t)part & 15)))) return (int)hipErrorInvalidValue;
  p.cs = (const float*)cs; p.max_pos = max_pos; p.rot0 = rot0; p.rot_dims = rot_dims;
  p.runs = Dv % 4 == 0 && (!gate || (gate_ld % 4 == 0 && ((size_t)gate & 7) == 0));
  p.rows16 = Dv % 8 == 0 && o_ld % 8 == 0 && ((size_t)o & 15) == 0;
  // the direct-to-LDS loads take 16-byte rows, a tile's rows within 32-bit offsets
  if ((((size_t)k | (size_t)v) & 15) || (long)H * DK >= (1L << 24)) return (int)hipErrorInvalidValue;
  // 64 rows and two runs (also where the keys are in parts; keys of 256 columns: one) while these workgroups are one round of the
  // CUs, then 128 rows and two runs (160 KB of LDS at 192 columns), or one run, whose workgroups
  // share a CU: with feeds of up to 128 rows from a second round on (us with two runs and with one,
  // 9 feeds x 32 heads: 20 rows, 192 / 128 columns: 18, 9.8; 128 rows behind 300: 41.5, 31)
  const long n64 = (long)((max_q + 63) / 64) * H * B, n128 = (long)((max_q + 127) / 128) * H * B;
  if (parts > 1 && n64 > 256) return (int)hipErrorInvalidValue;
#define RUN(A, C, QW, KS, PARTS)                                                              \
  do {                                                                                        \
    constexpr int ring = KS * FlashLds<A, C>::RING;                                           \
    constexpr int end = FlEnd<C / 32, QW, KS, PARTS>::BYTES;                                  \
    constexpr int bytes = ring > end ? ring : end;                                            \
    static_assert(bytes <= 160 * 1024, "LDS of a CU");                                        \
    const long blocks = (max_q + 32 * QW - 1) / (32 * QW), all = blocks * H * B;              \
    if (PARTS && (all > tickets || all * parts * QW * fl_join_floats(C / 32) > part_floats))  \
      return (int)hipErrorInvalidValue;                                                       \
    const dim3 grid(blocks * (PARTS ? parts : 1), H, B);                                      \
    hipLaunchKernelGGL((latent_prefill_kernel<A, C, QW, KS, PARTS>), grid, dim3(64 * QW * KS), bytes, st, p); \
    return (int)hipGetLastError();                                                            \
  } while (0)
#define GO(A, C)                                                                              \
  if (DK == A && DV == C) {                                                                   \
    constexpr int K2 = A > 192 ? 1 : 2;                                                       \
    if (parts > 1) RUN(A, C, 2, K2, true);                                                    \
    else if (n64 <= 256) RUN(A, C, 2, K2, false);                                             \
    else if (n128 <= (max_q <= 128 ? 256 : 512)) RUN(A, C, 4, K2, false);                     \
    else RUN(A, C, 4, 1, false);                                                              \
  }
  GO(64, 64) GO(128, 64) GO(192, 64) GO(256, 64) GO(64, 128) GO(128, 128) GO(192, 128) GO(256, 128)
#undef GO
#undef RUN
  return (int)hipErrorInvalidValue;
}
