// Prompt portions of the windowed paged attention (attn_window.hip) on the pipelined tile loop
// (flash_pipe.h), bf16, key and value sizes up to 128 a workgroup.
//
// A workgroup is QW KS waves: QW blocks of 32 query rows of one head (and up to 128 of its value
// columns), the key tiles that these rows see split into KS runs. Tiles that lie wholly between
// the kept first tokens and the rows' windows are skipped; a tile that every row of a wave sees
// whole takes no per-score tests. Head sizes between the built ones are padded in LDS. Numerator
// and denominator are of the same rounded weights (flash_pipe.h has the errors).
// What bounds it at 128 columns: MFMAs, LDS and L2 about alike (flash_pipe.h). 2048 rows of 16
// heads (4 key heads) of 128, window 1024: 92 us before (256 rows a workgroup, half of the CUs;
// tiles through registers; maximum, exponentials and products one after the other), 35 now; without a window 128, 50. Few rows
// behind many keys: parts of a block's keys in workgroups of their own, joined in the launch (fl_join; 16 heads of 128, 64
// rows behind 2000 42.6 -> 22.7 us, with a window of 1024 27.5 -> 21.8, 128 behind 8000 139 -> 36).
#include "flash_pipe.h"
#include "seqmix.h"

__device__ __forceinline__ float wp_tanh(float z) {
  return 1.f - 2.f * __builtin_amdgcn_rcpf(1.f + __builtin_amdgcn_exp2f(2.885390081777927f * z));
}

// GEN: a soft cap, slopes or a scale that is not positive; else scores only need masking. PARTS: of a block's keys, a kernel of
// its own (in one with the others these took 0.2 to 0.5 us more, 300 rows x 16 heads of 128 in a window of 300 15.4 us, 14.6 alone).
template <int DK, int DV, int QW, int KS, bool GEN, bool PARTS>
__global__ __launch_bounds__(64 * QW * KS, 2) void window_attn_pipe_kernel(WinAttnParams p) {
  using L = FlashLds<DK, DV>;
  constexpr int NS = DK / 16, NDT = DV / 32, NTH = 64 * QW;
  extern __shared__ __attribute__((aligned(16))) unsigned char lds[];
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int run = wave / QW, wq = wave % QW, th = threadIdx.x - run * NTH, h = lane >> 5;
  int bx, head, v0, b, share = 0;
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
    bx = gx - 1 - bx;
    if constexpr (PARTS) {
      share = bx % p.parts;
      bx /= p.parts;
    }
    b = hd / gy;
    head = (hd - b * gy) / p.vparts;
    v0 = ((hd - b * gy) - head * p.vparts) * DV;            // this workgroup's value columns
  }
  const int g = head / (p.H / p.G), Dv = min(DV, p.Dv - v0);
  const int q0 = p.cu_q[b], qlen = p.cu_q[b + 1] - q0;
  const int row_lo = bx * (32 * QW);
  if (row_lo >= qlen) return;                               // whole workgroup: uniform
  const int row_hi = min(qlen - 1, row_lo + 32 * QW - 1);
  const int qi = row_lo + wq * 32 + (lane & 31);
  const bool valid = qi < qlen;
  const int qpos = p.pos[q0 + min(qi, row_hi)];
  const int pos_lo = p.pos[q0 + row_lo];
  int kend = min(p.ctx[b], p.pos[q0 + row_hi] + 1);   // positions grow along a feed
  // key tiles: those holding kept first tokens, then from the first window on
  const int wg_lo = p.window > 0 ? max(0, pos_lo - p.window + 1) : 0;
  const int lo_t = wg_lo / FL_KEYS * FL_KEYS;
  const int n1 = p.window > 0 ? min((min(p.keep_first, wg_lo) + FL_KEYS - 1) / FL_KEYS, lo_t / FL_KEYS) : 0;
  int ntiles = kend > 0 ? n1 + max(kend - lo_t + FL_KEYS - 1, 0) / FL_KEYS : 0, parts = 1, t0 = 0;
  auto tile_at = [&](int i) { return i < n1 ? i * FL_KEYS : lo_t + (i - n1) * FL_KEYS; };
  if constexpr (PARTS) {
    parts = max(1, min(p.parts, ntiles / FL_CAP));
    if (share >= parts) return;                             // uniform
    const int len = (ntiles + parts - 1) / parts;
    t0 = share * len;
    if (t0 + len < ntiles) kend = min(kend, tile_at(t0 + len));
    ntiles = min(t0 + len, ntiles);                         // past the part's last tile
  }
  // what this wave's rows can see
  const int wpos_lo = __builtin_amdgcn_readfirstlane(p.pos[q0 + min(row_lo + wq * 32, row_hi)]);
  const int wpos_hi = __builtin_amdgcn_readfirstlane(p.pos[q0 + min(row_lo + wq * 32 + 31, row_hi)]);
  const int per = (max(ntiles - t0, 0) + KS - 1) / KS, first = t0 + run * per;

  const float scale_log2 = p.scale * 1.4426950408889634f;
  const float slope_log2 = GEN && p.slopes ? p.slopes[head] * 1.4426950408889634f : 0.f;
  const float sink = p.sink ? p.sink[head] : 0.f;
  const float cap_log2 = p.cap * 1.4426950408889634f, inv_cap = p.cap > 0.f ? p.scale / p.cap : 0.f;

  const unsigned ring = fl_lds_at(lds) + run * L::RING;
  if (p.D < DK) {                                           // the missing key columns are zero
    for (int i = th * 16; i < 2 * L::K; i += NTH * 16) *reinterpret_cast<uint4*>(lds + run * L::RING + i) = make_uint4(0, 0, 0, 0);
    fl_sync();
  }
  const FlFetch<DK, NTH, false, true> kf(th, p.D, (long long)p.G * p.D);
  const FlFetch<DV, NTH, true, true> vf(th, Dv, (long long)p.G * p.Dv);
  // where a fetch stands: tiles come in order; past the last one it stays there
  struct At {
    const bf16_t* base;
    unsigned row_bytes;
    int i;
    FlPages pages;
  };
  const int sh = 31 - __clz(p.blk), last_page = (int)(p.cache_rows / p.blk) - 1;
  auto start = [&](const void* src, int col, int heads_cols) __attribute__((always_inline)) {
    return At{(const bf16_t*)src + col, (unsigned)heads_cols * 2, first, FlPages(p.bt + (size_t)b * p.max_blocks, sh, kend)};
  };
  auto fetch = [&](const auto& f, At& a, unsigned stage) __attribute__((always_inline)) {
    const int kt = tile_at(min(a.i, ntiles - 1)), last = kend - 1 - kt;
    ++a.i;
    a.pages.hold(kt, lane);
    f.paged(stage, last, [&](int r) __attribute__((always_inline)) {
      const int key = kt + r, pg = min(max(a.pages.page(key), 0), last_page);
      return (const bf16_t*)((const char*)a.base + (unsigned long long)(unsigned)pg * ((unsigned)p.blk * a.row_bytes) +
                             (unsigned)(key & (p.blk - 1)) * a.row_bytes);
    });
  };
  At ka = start(p.kc, g * p.D, p.G * p.D), va = start(p.vc, g * p.Dv + v0, p.G * p.Dv);

  bf16x8 qf[NS];
  {
    const bf16_t* qrow = (const bf16_t*)p.q + ((size_t)(q0 + min(qi, row_hi)) * p.H + head) * p.D;
#pragma unroll
    for (int s = 0; s < NS; ++s) {
      const uint4 v = valid && 16 * s + 8 * h < p.D ? *reinterpret_cast<const uint4*>(qrow + 16 * s + 8 * h) : make_uint4(0, 0, 0, 0);
      qf[s] = *reinterpret_cast<const bf16x8*>(&v);
    }
  }
  float16v acc[NDT];
#pragma unroll
  for (int i = 0; i < NDT; ++i)
#pragma unroll
    for (int j = 0; j < 16; ++j) acc[i][j] = 0.f;
  float m = -1e30f, l = 0.f;
  if (per > 0) fetch(kf, ka, ring);
  va.pages = ka.pages;                                      // with what it holds of the table

  // Waves half a tile apart only where a tile's halves weigh alike: transformed scores add a tanh or a bias a score to the
  // second half, and every half then waits for the longer one (us a call, apart, in step: 2716 rows x 8 heads of 96, window
  // 1024, bias 57.9, 52.6; 951 x 16 of 128, cap 30 and bias 49.7, 49.4; 3493 x 8 of 64, window 512, bias 35.2, 31.0).
  fl_loop<DK, DV, vf.N, false>(
      qf, acc, m, l, ring, per, GEN ? 1.f : scale_log2, lane, p.D == DK && Dv == DV, !GEN && QW * KS == 8 && per >= FL_APART ? wave >> 2 : -1,
      [&](float16v(&st)[2], int i) __attribute__((always_inline)) {
        const int kt = tile_at(first + i), k0 = kt + 4 * h;   // tiles past the last lie behind kend
        if constexpr (GEN) {
          // the distance bias of key k0 + c for this lane's query: nb + slope * c
          const float nb = slope_log2 * (float)(k0 - qpos);
#pragma unroll
          for (int t = 0; t < 2; ++t)
#pragma unroll
            for (int j = 0; j < 16; ++j)
              st[t][j] = (p.cap > 0.f ? cap_log2 * wp_tanh(st[t][j] * inv_cap) : st[t][j] * scale_log2) +
                         (nb + slope_log2 * (float)(32 * t + (j & 3) + 8 * (j >> 2)));
        }
        const bool whole = kt + FL_KEYS - 1 <= wpos_lo && kt + FL_KEYS <= kend &&
                           (p.window <= 0 || wpos_hi - kt < p.window || kt + FL_KEYS <= p.keep_first);
        if (!whole) {
          // seen: up to lim, but not from the kept tokens to before the window
          const int lim = min(kend, qpos + 1) - k0, keep = p.keep_first - k0;
          const unsigned gap = p.window > 0 ? (unsigned)max(qpos - p.window + 1 - k0 - keep, 0) : 0u;
#pragma unroll
          for (int t = 0; t < 2; ++t)
#pragma unroll
            for (int j = 0; j < 16; ++j) {
              const int c = 32 * t + (j & 3) + 8 * (j >> 2);
              if (c >= lim || (unsigned)(c - keep) < gap) st[t][j] = -INFINITY;
            }
        }
      },
      [&](int, unsigned stage) __attribute__((always_inline)) { fetch(kf, ka, stage); },
      [&](int, unsigned stage) __attribute__((always_inline)) { fetch(vf, va, stage); });

  fl_sync();                                                // every wave is done with the rings
  constexpr int OWN = FlEnd<NDT, QW, KS, PARTS>::OWN;
  const bf16_t* grow = p.gate ? (const bf16_t*)p.gate + (size_t)(q0 + min(qi, row_hi)) * p.gate_ld + (size_t)head * p.Dv + v0 : nullptr;
  float4v own[OWN];
  uint2 gate[OWN];
  auto ask = [&]() __attribute__((always_inline)) {         // the gates of the run's own units
#pragma unroll
    for (int s = 0; s < OWN; ++s) {
      const int d0 = fl_column<NDT, QW, KS, PARTS>(s, run, lane);
      gate[s] = grow && d0 < Dv ? *reinterpret_cast<const uint2*>(grow + d0) : make_uint2(0, 0);
    }
  };
  if constexpr (!PARTS) ask();                              // on their way while the runs meet
  fl_merge<NDT, QW, KS, PARTS>(acc, own, m, l, lds, run, wq, lane);
  if constexpr (PARTS) {
    if (run) return;
    const int block = (b * (int)gridDim.y + head * p.vparts + v0 / DV) * (int)(gridDim.x / p.parts) + bx;
    if (parts > 1 && !fl_join<NDT, QW>(acc, m, l, p.part + (size_t)block * p.parts * QW * fl_join_floats(NDT),
                                       p.words + (size_t)block * TICKET, parts, share, wq, lane))
      return;
    fl_units(acc, own);
    ask();
  }
  float inv = l > 0.f ? 1.f / l : 0.f;
  if (p.sink) {
    // the running maximum and sum are in the base-2 domain
    const float sl = sink * 1.44269504088896f;
    const float mx2 = fmaxf(m, sl);
    const float a = __builtin_amdgcn_exp2f(m - mx2);
    inv = a / (l * a + __builtin_amdgcn_exp2f(sl - mx2));
  }
#pragma unroll
  for (int s = 0; s < OWN; ++s) {
    float f[4] = {inv, inv, inv, inv};
    if (grow) {
      f[0] *= sigmoid_fast(__uint_as_float(gate[s].x << 16));
      f[1] *= sigmoid_fast(__uint_as_float(gate[s].x & 0xffff0000u));
      f[2] *= sigmoid_fast(__uint_as_float(gate[s].y << 16));
      f[3] *= sigmoid_fast(__uint_as_float(gate[s].y & 0xffff0000u));
    }
#pragma unroll
    for (int i = 0; i < 4; ++i) own[s][i] *= f[i];
  }
  fl_store<NDT, QW, KS, PARTS>(own, lds, (bf16_t*)p.o + (size_t)(q0 + row_lo + wq * 32) * p.o_ld + (size_t)head * p.Dv + v0, p.o_ld,
                               qlen - row_lo - wq * 32, Dv, run, wq, lane);
}

template <int DK, int DV, int QW, int KS, bool GEN, bool PARTS = false>
static int launch(const WinAttnParams& p, int max_q, hipStream_t st) {
  constexpr int ring = KS * FlashLds<DK, DV>::RING, end = FlEnd<DV / 32, QW, KS, PARTS>::BYTES;
  constexpr int bytes = ring > end ? ring : end;
  static_assert(bytes <= 160 * 1024, "LDS of a CU");
  const long blocks = (max_q + 32 * QW - 1) / (32 * QW), all = blocks * p.H * p.vparts * p.B;
  if (PARTS && (p.parts > FL_PARTS || all > p.tickets || all * p.parts * QW * fl_join_floats(DV / 32) > p.part_floats))
    return (int)hipErrorInvalidValue;
  const dim3 grid(blocks * (PARTS ? p.parts : 1), p.H * p.vparts, p.B);
  hipLaunchKernelGGL((window_attn_pipe_kernel<DK, DV, QW, KS, GEN, PARTS>), grid, dim3(64 * QW * KS), bytes, st, p);
  return (int)hipGetLastError();
}

// 64 query rows and two key runs while these workgroups are one round of the 256 CUs, then 128
// rows and two runs, then 128 rows and one run in four waves, two or three workgroups a CU. Feeds
// of up to 128 rows, whose chain of tiles is short, take the last form from a second round on (us
// with two runs and with one, 9 feeds x 32 heads: 20 rows, 64 columns: 14.3, 7.6; 128 rows behind
// 300, 128 columns: 39, 29). Transformed scores (GEN) go without the first form, which would
// be four more kernels to build (100 rows x 8 heads of 128: 12.4, with it 11.6; 320 behind 1000
// x 16: 51, 47).
template <int DK, int DV>
static int launch_rows(const WinAttnParams& p, int max_q, hipStream_t st) {
  const long hd = (long)p.H * p.vparts * p.B, n64 = (max_q + 63) / 64 * hd, n128 = (max_q + 127) / 128 * hd;
  const bool one = n128 > (max_q <= 128 ? 256 : 512);
  if (p.cap > 0.f || p.slopes || !(p.scale > 0.f))
    return one ? launch<DK, DV, 4, 1, true>(p, max_q, st) : launch<DK, DV, 4, 2, true>(p, max_q, st);
  if (n64 <= 128 && p.parts > 1) return launch<DK, DV, 2, 2, false, true>(p, max_q, st);   // parts only of the first form
  if (n64 <= 256) return launch<DK, DV, 2, 2, false>(p, max_q, st);
  if (!one) return launch<DK, DV, 4, 2, false>(p, max_q, st);
  return launch<DK, DV, 4, 1, false>(p, max_q, st);
}

// -1: not these sizes or places (the direct-to-LDS loads and whole-row stores take 16-byte rows,
// one load's eight rows lie in one page)
int window_attention_pipe(const WinAttnParams& p, int max_q, hipStream_t st) {
  const bool rows16 = (((size_t)p.q | (size_t)p.kc | (size_t)p.vc | (size_t)p.o) & 15) == 0 && p.o_ld % 8 == 0;
  if (!rows16 || p.D > 128 || p.D % 8 || p.Dv % 8 || p.blk < 8 || (p.blk & (p.blk - 1)) ||
      (long)p.blk * p.G * max(p.D, p.Dv) >= (1L << 30) || p.cache_rows < p.blk)
    return -1;
#define GO(A, C) return launch_rows<A, C>(p, max_q, st)
  if (p.D <= 64) {
    if (p.Dv <= 64) GO(64, 64); else GO(64, 128);
  }
  if (p.Dv <= 64) GO(128, 64); else GO(128, 128);
#undef GO
}
