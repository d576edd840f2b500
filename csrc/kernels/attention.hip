// Flash attention forward for CDNA4.
//
// One kernel family covers every attention in the hub:
//   * PREFILL mode  - a block of query rows of ONE head per workgroup (Whisper encoder,
//                     Llama prompt prefill, VITS text encoder). Causal or not.
//                     attn_pipe_kernel below; rows off 16 bytes and cache blocks of
//                     other sizes than 8, 16, 32, .. take attn_prefill2_kernel.
//   * GROUPED mode  - all query heads of ONE kv head x a few query tokens per
//                     workgroup (decode / jump-forward extend, GQA), with
//                     split-K over the context and a separate combine kernel.
// K/V come either from a contiguous [T, H_kv, D] tensor (cu_k offsets) or from
// the paged KV cache [n_blocks, H_kv, BLK, D] through a block table.
//
// MFMA formulation (v_mfma_f32_32x32x16_bf16, 4 waves, 32 query rows per wave):
//   S^T = K * Q^T  : A = K rows (ds_read_b128 from a padded LDS tile),
//                    B = Q^T fragment kept in VGPRs for the whole KV loop.
//                    The query lands on the MFMA lane, so the softmax row
//                    max/sum is in-register + one lane^32 exchange.
//   O^T += V^T * P^T : the S^T accumulator, exp2'ed and packed to bf16, IS the B
//                    operand (the accumulator tile as next operand); the
//                    V^T fragment comes from ds_read_b64_tr_b16 transposed reads
//                    of the row-major V tile. O^T also has the
//                    query on the lane, so the online-softmax rescale is a
//                    per-lane scalar multiply.
// LDS rows are padded (K: +16 B, V: +64 B) so that both the b128 row reads and
// the tr_b16 reads are bank-conflict free (all but the pipelined kernel).
#include "flash_pipe.h"

#define ATT_THREADS 256
#define ATT_WAVES 4
#define KV_TILE 64

typedef short v4s __attribute__((ext_vector_type(4)));
typedef unsigned u32x4 __attribute__((ext_vector_type(4)));

struct AttnParams {
  const bf16_t* q;
  long long q_stride;  // elements between consecutive query tokens (head stride = D)
  const bf16_t* k;
  const bf16_t* v;
  long long kv_stride;  // contiguous mode: elements between tokens
  bf16_t* o;
  long long o_stride;
  const int* cu_q;          // [B+1]
  const int* cu_k;          // [B+1] contiguous mode (or [B] starts when ctx_lens given)
  const int* ctx_lens;      // [B]   paged mode
  const int* block_tables;  // [B, max_blocks]
  int max_blocks;
  int blk;
  int Hq, Hkv;
  float scale_log2;
  int causal;
  int split_keys;  // GROUPED: keys per split (multiple of KV_TILE)
  int num_splits;
  float* part_o;   // [num_splits, Tq, Hq, D]
  float* part_ml;  // [num_splits, Tq, Hq, 2]
  int total_q;
  int parts;                // prompts: parts of a row block's keys at most, (fl_join)
  float* part; int* words;
};

template <int D>
struct AttnSmem {
  bf16_t k[KV_TILE][D + 8];
  bf16_t v[KV_TILE][D + 32];
};

__device__ __forceinline__ float16v mfma32(const bf16x8& a, const bf16x8& b, const float16v& c) {
  return __builtin_amdgcn_mfma_f32_32x32x16_bf16(a, b, c, 0, 0, 0);
}

template <int D, bool PAGED>
__global__ __launch_bounds__(ATT_THREADS, 1) void attn_fwd_kernel(AttnParams p) {
  __shared__ __attribute__((aligned(16))) AttnSmem<D> sm;
  constexpr int NS = D / 16;  // k-slices of the QK^T product
  constexpr int NDT = D / 32; // 32-wide d tiles of O^T
  const int lane = threadIdx.x & 63;
  const int wave = threadIdx.x >> 6;
  const int h = lane >> 5;
  const int b = blockIdx.z;
  const int q0 = p.cu_q[b];
  const int qlen = p.cu_q[b + 1] - q0;
  int k0 = 0, klen;
  if (PAGED) {
    klen = p.ctx_lens[b];
  } else {
    // contiguous K/V: start cu_k[b]; length ctx_lens[b] if given, else cu_k[b+1]-cu_k[b]
    k0 = p.cu_k[b];
    klen = p.ctx_lens ? p.ctx_lens[b] : p.cu_k[b + 1] - k0;
  }
  const int G = p.Hq / p.Hkv;

  // ---- row mapping: this lane's query row (token index within seq, head)
  const int r = wave * 32 + (lane & 31), kvh = blockIdx.y;
  const int qi = r / G, head = kvh * G + (r - qi * G);
  const int row_hi = min(qlen, (ATT_WAVES * 32) / G) - 1;   // last token (for the causal bound)
  const bool row_valid = qi < qlen && (ATT_WAVES * 32) / G > 0 && r < (ATT_WAVES * 32 / G) * G;

  // ---- key range of this workgroup
  const int split = blockIdx.x, kbeg = split * p.split_keys;
  int kend = min(klen, kbeg + p.split_keys);
  if (p.causal) kend = min(kend, klen - qlen + row_hi + 1);

  // ---- Q^T fragments (B operand): lane (query, h) holds Q[q][16s + 8h .. +7]
  bf16x8 qf[NS];
  const bf16_t* qrow = p.q + (size_t)(q0 + (row_valid ? qi : 0)) * p.q_stride + (size_t)head * D;
#pragma unroll
  for (int s = 0; s < NS; ++s) {
    uint4 v = row_valid ? *reinterpret_cast<const uint4*>(qrow + 16 * s + 8 * h) : make_uint4(0, 0, 0, 0);
    qf[s] = *reinterpret_cast<bf16x8*>(&v);
  }

  float16v acc[NDT];
  float m_run = -1e30f, l_run = 0.f;
#pragma unroll
  for (int i = 0; i < NDT; ++i)
#pragma unroll
    for (int j = 0; j < 16; ++j) acc[i][j] = 0.f;

  const int* btab = PAGED ? p.block_tables + (size_t)b * p.max_blocks : nullptr;
  constexpr int CH = D / 8;  // 16-byte chunks per row

  for (int kt = kbeg; kt < kend; kt += KV_TILE) {
    // ---- stage K and V tile (64 keys) into LDS
    __syncthreads();
#pragma unroll
    for (int c = threadIdx.x; c < KV_TILE * CH; c += ATT_THREADS) {
      const int kr = c / CH, cc = (c - kr * CH) * 8;
      const int key = kt + kr;
      uint4 kv4 = make_uint4(0, 0, 0, 0), vv4 = make_uint4(0, 0, 0, 0);
      if (key < kend) {
        size_t off;
        if (PAGED) {
          const int bi = key / p.blk, bo = key - bi * p.blk;
          off = (((size_t)btab[bi] * p.Hkv + kvh) * p.blk + bo) * D + cc;
        } else {
          off = (size_t)(k0 + key) * p.kv_stride + (size_t)kvh * D + cc;
        }
        kv4 = *reinterpret_cast<const uint4*>(p.k + off);
        vv4 = *reinterpret_cast<const uint4*>(p.v + off);
      }
      *reinterpret_cast<uint4*>(&sm.k[kr][cc]) = kv4;
      *reinterpret_cast<uint4*>(&sm.v[kr][cc]) = vv4;
    }
    __syncthreads();

    // ---- S^T = K Q^T for the two 32-key halves
    float16v st[2];
#pragma unroll
    for (int t = 0; t < 2; ++t) {
#pragma unroll
      for (int j = 0; j < 16; ++j) st[t][j] = 0.f;
#pragma unroll
      for (int s = 0; s < NS; ++s) {
        const bf16x8 a = *reinterpret_cast<const bf16x8*>(&sm.k[32 * t + (lane & 31)][16 * s + 8 * h]);
        st[t] = mfma32(a, qf[s], st[t]);
      }
    }
    // ---- mask + online softmax (row = this lane's query)
    bf16x8 pf[2][2];
    const int qpos = klen - qlen + qi;  // absolute position for causal masking
    float mx = -INFINITY;
#pragma unroll
    for (int t = 0; t < 2; ++t)
#pragma unroll
      for (int j = 0; j < 16; ++j) {
        const int key = kt + 32 * t + (j & 3) + 8 * (j >> 2) + 4 * h;
        float sv = st[t][j] * p.scale_log2;
        if (key >= kend || (p.causal && key > qpos)) sv = -INFINITY;
        st[t][j] = sv;
        mx = fmaxf(mx, sv);
      }
    mx = fmaxf(mx, __shfl_xor(mx, 32, 64));
    const float m_new = fmaxf(m_run, mx);
    const float alpha = exp2f(m_run - m_new);
    float ls = 0.f;
#pragma unroll
    for (int t = 0; t < 2; ++t)
#pragma unroll
      for (int s2 = 0; s2 < 2; ++s2)
#pragma unroll
        for (int j = 0; j < 8; ++j) {
          const float e = exp2f(st[t][8 * s2 + j] - m_new);
          ls += e;
          pf[t][s2][j] = (__bf16)e;
        }
    ls += __shfl_xor(ls, 32, 64);
    l_run = l_run * alpha + ls;
    m_run = m_new;
#pragma unroll
    for (int i = 0; i < NDT; ++i)
#pragma unroll
      for (int j = 0; j < 16; ++j) acc[i][j] *= alpha;

    // ---- O^T += V^T P^T
    const int g = lane >> 4, li = lane & 15;
#pragma unroll
    for (int dt = 0; dt < NDT; ++dt) {
      const int c0 = 32 * dt + 16 * (g & 1) + 4 * (li & 3);
#pragma unroll
      for (int t = 0; t < 2; ++t)
#pragma unroll
        for (int s2 = 0; s2 < 2; ++s2) {
          const int kb = 32 * t + 16 * s2 + 4 * h + (li >> 2);
          const v4s lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16(
              (__attribute__((address_space(3))) v4s*)(&sm.v[kb][c0]));
          const v4s hi = __builtin_amdgcn_ds_read_tr16_b64_v4i16(
              (__attribute__((address_space(3))) v4s*)(&sm.v[kb + 8][c0]));
          short8 a8;
          a8[0] = lo[0]; a8[1] = lo[1]; a8[2] = lo[2]; a8[3] = lo[3];
          a8[4] = hi[0]; a8[5] = hi[1]; a8[6] = hi[2]; a8[7] = hi[3];
          acc[dt] = mfma32(*reinterpret_cast<bf16x8*>(&a8), pf[t][s2], acc[dt]);
        }
    }
  }

  if (!row_valid) return;
  const size_t tok = (size_t)(q0 + qi);
  if (p.num_splits > 1) {
    // unnormalised partial result + (m, l) for the combine kernel
    float* po = p.part_o + (((size_t)split * p.total_q + tok) * p.Hq + head) * D;
#pragma unroll
    for (int dt = 0; dt < NDT; ++dt)
#pragma unroll
      for (int g4 = 0; g4 < 4; ++g4) {
        const int d0 = 32 * dt + 8 * g4 + 4 * h;
        *reinterpret_cast<float4*>(po + d0) = make_float4(acc[dt][4 * g4], acc[dt][4 * g4 + 1],
                                                          acc[dt][4 * g4 + 2], acc[dt][4 * g4 + 3]);
      }
    if (h == 0) {
      float* pm = p.part_ml + (((size_t)split * p.total_q + tok) * p.Hq + head) * 2;
      pm[0] = m_run;
      pm[1] = l_run;
    }
    return;
  }
  const float inv = l_run > 0.f ? 1.f / l_run : 0.f;
  bf16_t* orow = p.o + tok * p.o_stride + (size_t)head * D;
#pragma unroll
  for (int dt = 0; dt < NDT; ++dt)
#pragma unroll
    for (int g4 = 0; g4 < 4; ++g4) {
      const int d0 = 32 * dt + 8 * g4 + 4 * h;
      uint2 w;
      w.x = pack_bf16x2(acc[dt][4 * g4] * inv, acc[dt][4 * g4 + 1] * inv);
      w.y = pack_bf16x2(acc[dt][4 * g4 + 2] * inv, acc[dt][4 * g4 + 3] * inv);
      *reinterpret_cast<uint2*>(orow + d0) = w;
    }
}

// ---------------------------------------------------------------------------
// PREFILL / ENCODER attention on the pipelined tile loop (flash_pipe.h).
//
// A workgroup is QW KS waves: QW blocks of 32 query rows of one head, the key tiles split
// into KS runs with a ring of their own; the runs' (m, l, O) meet in LDS at the end.
// One 30 s window has 1500 rows: 128 rows a workgroup are 240 workgroups at 20 heads, but 96
// at 8, where 64 rows and four runs fill the chip (launch_attn() has the rule).
// us a pass before (8 waves in step, K / V through registers, padded rows) and now: 1500 rows x 8
// heads of 64: 23.4, 15.6; x 20 heads: 24, 22.8; 6 x 1500 x 20: 133, 100; 128 columns causal from a
// paged cache: 2048 x 32 heads: 91, 60; 4 x that: 294, 198; 320 x 32 heads: 19, 19. What is left
// above the VALU's and MFMAs' time: the loads' share of LDS and L2 (a third at 128 columns with
// two runs), the barrier and the maxima, each of which all waves of a workgroup meet together.
// PAGES: 0 contiguous rows, 1 cache blocks of 64 rows or more, 2 of 8, 16 or 32.
template <int D, int PAGES, int QW, int KS, bool PARTS>
__global__ __launch_bounds__(64 * QW * KS, D == 64 && QW * KS == 4 ? 3 : 2) void attn_pipe_kernel(AttnParams p) {
  constexpr bool PAGED = PAGES > 0;
  using L = FlashLds<D, D>;
  constexpr int NS = D / 16, NDT = D / 32, NTH = 64 * QW;
  extern __shared__ __attribute__((aligned(16))) unsigned char lds[];
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int run = wave / QW, wq = wave % QW, th = threadIdx.x - run * NTH, h = lane >> 5;
  int bx, by, bz, share = 0;
  {
    const int gx = gridDim.x, gy = gridDim.y, heads = gy * gridDim.z, n = gx * heads;
    const int logical = xcd_remap(blockIdx.x + gx * (blockIdx.y + gy * blockIdx.z), n);
    int hd = logical / gx;
    bx = logical - hd * gx;
    if (p.causal) {
      // row blocks with the most keys first, over all heads of an XCD where these are whole
      if (heads % 8 == 0) {
        const int hp = heads / 8, xcd = logical / (hp * gx), at = logical - xcd * hp * gx;
        bx = at / hp;
        hd = xcd * hp + at - bx * hp;
      }
      bx = gx - 1 - bx;
    }
    if constexpr (PARTS) {
      share = bx % p.parts;
      bx /= p.parts;
    }
    by = hd % gy;
    bz = hd / gy;
  }
  const int b = bz;
  const int q0 = p.cu_q[b];
  const int qlen = p.cu_q[b + 1] - q0;
  int k0 = 0, klen;
  if (PAGED) {
    klen = p.ctx_lens[b];
  } else {
    k0 = p.cu_k[b];
    klen = p.ctx_lens ? p.ctx_lens[b] : p.cu_k[b + 1] - k0;
  }
  const int head = by, kvh = head / (p.Hq / p.Hkv);
  const int row_lo = bx * (32 * QW);
  if (row_lo >= qlen) return;                               // whole workgroup: uniform
  const int row_hi = min(qlen - 1, row_lo + 32 * QW - 1);
  const int qi = row_lo + wq * 32 + (lane & 31);
  const bool row_valid = qi < qlen;
  const int qpos_lo = klen - qlen + row_lo + wq * 32;       // wave's first query position
  int kend = klen;
  if (p.causal) kend = min(kend, klen - qlen + row_hi + 1);
  int ntiles = kend > 0 ? (kend + FL_KEYS - 1) / FL_KEYS : 0, parts = 1, t0 = 0;
  if constexpr (PARTS) {
    parts = max(1, min(p.parts, ntiles / FL_CAP));
    if (share >= parts) return;                             // uniform
    const int len = (ntiles + parts - 1) / parts;
    t0 = share * len;
    ntiles = max(0, min(len, ntiles - t0));
    kend = min(kend, (t0 + len) * FL_KEYS);
  }
  const int per = (ntiles + KS - 1) / KS;                   // tiles of a run; the last may have fewer
  const int first = t0 + run * per;
  // run 0 has the only tile: the others leave before they fetch and mask a copy of it, and nothing is merged (1500 rows behind
  // 64 keys: 8 heads of 64 5.7 -> 4.4 us, 20 heads 6.5 -> 5.0; 64 rows x 32 heads with the merge 6.6, without 6.0). A barrier
  // waits for the waves that are left.
  const bool alone = KS > 1 && !PARTS && ntiles <= 1;
  if (alone && run) return;

  const FlFetch<D, NTH, false, false> kf(th, D, PAGED ? D : p.kv_stride);
  const FlFetch<D, NTH, true, false> vf(th, D, PAGED ? D : p.kv_stride);
  // Where a fetch stands: tiles come in order, one call each; past the last tile it stays there.
  // Rows past kend read the last key again (finite scores, masked to -inf, so P = 0).
  const int kt0 = max(min(first, t0 + ntiles - 1), 0) * FL_KEYS;
  const int* btab = PAGED ? p.block_tables + (size_t)b * p.max_blocks : nullptr;
  const unsigned page_bytes = (unsigned)(p.Hkv * p.blk) * (D * 2);
  struct At {
    const bf16_t* row;               // contiguous: the tile's first row
    int kt;
    FlPages pages;
  };
  auto start = [&](const bf16_t* src) __attribute__((always_inline)) {
    return At{src + (PAGED ? (size_t)kvh * p.blk * D : (size_t)(k0 + kt0) * p.kv_stride + (size_t)kvh * D), kt0,
              FlPages(btab, PAGED ? 31 - __clz(p.blk) : 0, kend)};
  };
  auto fetch = [&](const auto& f, At& a, unsigned stage) __attribute__((always_inline)) {
    const int last = kend - 1 - a.kt;
    if constexpr (!PAGED) {
      f.strided(stage, a.row, last);
      if (last >= FL_KEYS) a.row += FL_KEYS * p.kv_stride;
    } else {
      a.pages.hold(a.kt, lane);
      auto at = [&](int r) __attribute__((always_inline)) {
        const int key = a.kt + r;
        const unsigned long long off = (unsigned long long)(unsigned)a.pages.page(key) * page_bytes;
        return (const bf16_t*)((const char*)a.row + off + (unsigned)(key & (p.blk - 1)) * (D * 2));
      };
      if constexpr (PAGES == 1)
        f.strided(stage, at(0), last);
      else
        f.paged(stage, last, at);
    }
    if (last >= FL_KEYS) a.kt += FL_KEYS;
  };
  const unsigned ring = fl_lds_at(lds) + run * L::RING;
  At ka = start(p.k), va = start(p.v);
  constexpr bool AHEAD = PAGED ? D == 128 && QW == 2 : KS == 1;   // K 0 before Q (fl_loop)
  auto fetch_first = [&]() __attribute__((always_inline)) {
    if (per > 0) fetch(kf, ka, ring);
    va.pages = ka.pages;                                    // with what it holds of the table
  };
  if constexpr (AHEAD) fetch_first();

  bf16x8 qf[NS];
  {
    const bf16_t* qrow = p.q + (size_t)(q0 + (row_valid ? qi : 0)) * p.q_stride + (size_t)head * D;
#pragma unroll
    for (int s = 0; s < NS; ++s) {
      uint4 v = row_valid ? *reinterpret_cast<const uint4*>(qrow + 16 * s + 8 * h) : make_uint4(0, 0, 0, 0);
      qf[s] = *reinterpret_cast<bf16x8*>(&v);
    }
  }
  float16v acc[NDT];
#pragma unroll
  for (int i = 0; i < NDT; ++i)
#pragma unroll
    for (int j = 0; j < 16; ++j) acc[i][j] = 0.f;
  float m = -1e30f, l = 0.f;
  if constexpr (!AHEAD) fetch_first();
  fl_loop<D, D, vf.N + (AHEAD ? kf.N : 0), AHEAD>(
      qf, acc, m, l, ring, per, p.scale_log2, lane, true,
      // half a tile apart costs 64-column heads on two runs off contiguous keys up to 4 % (1500 rows x 20 heads 20.1 -> 20.5)
      QW * KS == 8 && (PAGED || KS == 4 || D == 128) && per >= FL_APART ? wave >> 2 : -1,
      [&](float16v(&st)[2], int i) __attribute__((always_inline)) {
        // masking only where a key can be invalid for this wave (wave-uniform test)
        const int kt = (first + i) * FL_KEYS;
        if (kt + FL_KEYS > kend || (p.causal && kt + FL_KEYS - 1 > qpos_lo)) {
          const int lim = (p.causal ? min(kend, klen - qlen + qi + 1) : kend) - kt - 4 * h;
#pragma unroll
          for (int t = 0; t < 2; ++t)
#pragma unroll
            for (int j = 0; j < 16; ++j)
              if (32 * t + (j & 3) + 8 * (j >> 2) >= lim) st[t][j] = -INFINITY;
        }
      },
      [&](int, unsigned stage) __attribute__((always_inline)) { fetch(kf, ka, stage); },
      [&](int, unsigned stage) __attribute__((always_inline)) { fetch(vf, va, stage); });

  fl_sync();                                                // every wave is done with the rings
  auto finish = [&](auto all, auto& own) __attribute__((always_inline)) {
    constexpr bool ALL = decltype(all)::value != 0;
    const float inv = l > 0.f ? 1.f / l : 0.f;
#pragma unroll
    for (int s = 0; s < FlEnd<NDT, QW, KS, ALL>::OWN; ++s) own[s] *= inv;
    fl_store<NDT, QW, KS, ALL>(own, lds, p.o + (size_t)(q0 + row_lo + wq * 32) * p.o_stride + (size_t)head * D, p.o_stride,
                               qlen - row_lo - wq * 32, D, run, wq, lane);
  };
  if (alone) {
    float4v own[4 * NDT];
    fl_units(acc, own);
    finish(Fl<1>{}, own);
    return;
  }
  float4v own[FlEnd<NDT, QW, KS, PARTS>::OWN];
  fl_merge<NDT, QW, KS, PARTS>(acc, own, m, l, lds, run, wq, lane);
  if constexpr (PARTS) {
    if (run) return;
    const int block = (b * p.Hq + head) * (int)(gridDim.x / p.parts) + bx;
    if (parts > 1 && !fl_join<NDT, QW>(acc, m, l, p.part + (size_t)block * p.parts * QW * fl_join_floats(NDT),
                                       p.words + (size_t)block * TICKET, parts, share, wq, lane))
      return;
    fl_units(acc, own);
  }
  finish(Fl<PARTS>{}, own);
}

// ---------------------------------------------------------------------------
// PREFILL / ENCODER attention where the pipelined loop's loads do not go: rows that do not start
// on 16 bytes, cache blocks that are no power of two from 8 on (every chunk finds its own row).
//
// 8 waves over 128 query rows: waves 0-3 take the first half of the key tiles, waves 4-7 the
// second half (same query rows, same lane layout), so that the MFMA and VALU phases of a SIMD's
// two waves overlap. Each half streams its K / V tiles through registers into its own
// double-buffered LDS ring (the global loads of tile i + 1 are issued before tile i is computed
// and written to LDS after it), one barrier per tile. The halves merge their (m, l, O) through
// LDS at the end. LDS rows are padded (K: +16 B, V: +64 B), so that the b128 row reads and the
// tr_b16 reads are free of bank conflicts.
// us a pass, the grouped kernel's 4-wave form in its place and this one (paged, blocks of 12):
// 40 rows behind 960, 20 heads of 64: 63, 17; 2048 rows causal: 128, 45; 32 heads of 128: 69, 24
// and 158, 93; 1500 rows of 20 heads, rows 4 entries off: 83, 26.
template <int D>
struct AttnSmem2 {
  bf16_t k[2][2][KV_TILE][D + 8];   // [half][stage]
  bf16_t v[2][2][KV_TILE][D + 32];
};

template <int D, bool PAGED>
__global__ __launch_bounds__(512, 1) void attn_prefill2_kernel(AttnParams p) {
  __shared__ __attribute__((aligned(16))) AttnSmem2<D> sm;
  constexpr int NS = D / 16, NDT = D / 32, CH = D / 8;
  constexpr int NC = KV_TILE * CH / 256;      // 16-byte chunks per thread per operand
  const int lane = threadIdx.x & 63;
  const int wave = threadIdx.x >> 6;
  const int half = wave >> 2, w4 = wave & 3;
  const int th = threadIdx.x & 255;
  const int h = lane >> 5;
  int bx, by, bz;
  {
    const int gx = gridDim.x, gy = gridDim.y;
    const int n = gx * gy * gridDim.z;
    const int lin = blockIdx.x + gx * (blockIdx.y + gy * blockIdx.z);
    const int logical = xcd_remap(lin, n);
    bx = logical % gx;
    by = (logical / gx) % gy;
    bz = logical / (gx * gy);
  }
  const int b = bz;
  const int q0 = p.cu_q[b];
  const int qlen = p.cu_q[b + 1] - q0;
  int k0 = 0, klen;
  if (PAGED) {
    klen = p.ctx_lens[b];
  } else {
    k0 = p.cu_k[b];
    klen = p.ctx_lens ? p.ctx_lens[b] : p.cu_k[b + 1] - k0;
  }
  const int head = by, kvh = head / (p.Hq / p.Hkv);
  const int row_lo = bx * 128;
  if (row_lo >= qlen) return;                               // whole workgroup: uniform
  const int row_hi = min(qlen - 1, row_lo + 127);
  const int qi = row_lo + w4 * 32 + (lane & 31);
  const bool row_valid = qi < qlen;
  const int qpos_lo = klen - qlen + row_lo + w4 * 32;       // wave's first / last query position
  const int qpos_hi = qpos_lo + 31;
  int kend = klen;
  if (p.causal) kend = min(kend, klen - qlen + row_hi + 1);
  const int ntiles = kend > 0 ? (kend + KV_TILE - 1) / KV_TILE : 0;
  const int n0 = (ntiles + 1) >> 1;
  const int my_t0 = half ? n0 : 0;
  const int my_n = half ? ntiles - n0 : n0;

  bf16x8 qf[NS];
  {
    const bf16_t* qrow = p.q + (size_t)(q0 + (row_valid ? qi : 0)) * p.q_stride + (size_t)head * D;
#pragma unroll
    for (int s = 0; s < NS; ++s) {
      uint4 v = row_valid ? *reinterpret_cast<const uint4*>(qrow + 16 * s + 8 * h) : make_uint4(0, 0, 0, 0);
      qf[s] = *reinterpret_cast<bf16x8*>(&v);
    }
  }
  float16v acc[NDT];
#pragma unroll
  for (int i = 0; i < NDT; ++i)
#pragma unroll
    for (int j = 0; j < 16; ++j) acc[i][j] = 0.f;
  float m_run = -1e30f, l_run = 0.f;
  const float sl2 = p.scale_log2;

  const int* btab = PAGED ? p.block_tables + (size_t)b * p.max_blocks : nullptr;
  // Loads are unconditional (rows past kend re-read the last key - finite
  // values whose scores are masked to -inf, so P = 0 exactly; a half past its
  // last tile re-reads a valid tile): a load under a branch makes hipcc fall
  // back to vmcnt(0) at the first MFMA, serialising the prefetch.
#define ATT2_ROW_OFF(KT, i, key_, cc_)                                                \
    const int c = th + (i) * 256;                                                     \
    const int kr = c / CH, cc_ = (c - kr * CH) * 8;                                   \
    const int key_ = min((KT) + kr, kend - 1);                                        \
    size_t off;                                                                       \
    if (PAGED) {                                                                      \
      const int bi = key_ / p.blk, bo = key_ - bi * p.blk;                            \
      off = (((size_t)btab[bi] * p.Hkv + kvh) * p.blk + bo) * D + cc_;                \
    } else {                                                                          \
      off = (size_t)(k0 + key_) * p.kv_stride + (size_t)kvh * D + cc_;                \
    }
#define ATT2_LOAD1(SRC, KT, R)                                                        \
  _Pragma("clang loop unroll(full)") for (int i = 0; i < NC; ++i) {                   \
    ATT2_ROW_OFF(KT, i, key, cc)                                                      \
    R[i] = *reinterpret_cast<const u32x4*>(SRC + off);                                \
  }
#define ATT2_STORE1(DST, R)                                                           \
  _Pragma("clang loop unroll(full)") for (int i = 0; i < NC; ++i) {                   \
    const int c = th + i * 256;                                                       \
    const int kr = c / CH, cc = (c - kr * CH) * 8;                                    \
    *reinterpret_cast<u32x4*>(&DST[kr][cc]) = R[i];                                   \
  }
  // S^T = K Q^T for the tile in K stage KST (two 32-key halves; the query is
  // this lane's column)
#define ATT2_QK(KST, ST)                                                              \
  {                                                                                   \
    const bf16_t(*ks_)[D + 8] = sm.k[half][KST];                                      \
    _Pragma("unroll") for (int t = 0; t < 2; ++t) {                                   \
      _Pragma("unroll") for (int j = 0; j < 16; ++j) ST[t][j] = 0.f;                  \
      _Pragma("unroll") for (int s = 0; s < NS; ++s) {                                \
        const bf16x8 a = *reinterpret_cast<const bf16x8*>(&ks_[32 * t + (lane & 31)][16 * s + 8 * h]); \
        ST[t] = mfma32(a, qf[s], ST[t]);                                              \
      }                                                                               \
    }                                                                                 \
  }

  // online softmax of the scores ST of the tile at key KT, then O^T += V^T P^T
  // with V from V stage VST
  auto softmax_pv = [&](float16v (&st)[2], int vst, int kt) __attribute__((always_inline)) {
    // masking only where a key can be invalid for this wave (wave-uniform test)
    if (kt + KV_TILE > kend || (p.causal && kt + KV_TILE - 1 > qpos_lo)) {
      const int lim = (p.causal ? min(kend, klen - qlen + qi + 1) : kend) - kt - 4 * h;
#pragma unroll
      for (int t = 0; t < 2; ++t)
#pragma unroll
        for (int j = 0; j < 16; ++j)
          if (32 * t + (j & 3) + 8 * (j >> 2) >= lim) st[t][j] = -INFINITY;
    }
    float mx = st[0][0];
#pragma unroll
    for (int j = 1; j < 16; ++j) mx = fmaxf(mx, st[0][j]);
#pragma unroll
    for (int j = 0; j < 16; ++j) mx = fmaxf(mx, st[1][j]);
    mx = fmaxf(mx, __shfl_xor(mx, 32, 64));
    const float m_new = fmaxf(m_run, mx * sl2);
    const float alpha = __builtin_amdgcn_exp2f(m_run - m_new);
    bf16x8 pf[2][2];
#pragma unroll
    for (int t = 0; t < 2; ++t)
#pragma unroll
      for (int s2 = 0; s2 < 2; ++s2)
#pragma unroll
        for (int j = 0; j < 8; ++j)
          pf[t][s2][j] = (__bf16)__builtin_amdgcn_exp2f(fmaf(st[t][8 * s2 + j], sl2, -m_new));
    // row sums on the matrix core (ones . P^T: every output row is the sum
    // over the tile's 64 keys of the bf16 P that also feeds O), which has
    // slack here, instead of 32 VALU adds + a cross-lane exchange
    {
      bf16x8 ones;
#pragma unroll
      for (int j = 0; j < 8; ++j) ones[j] = (__bf16)1.0f;
      float16v ls = {};
#pragma unroll
      for (int t = 0; t < 2; ++t)
#pragma unroll
        for (int s2 = 0; s2 < 2; ++s2) ls = mfma32(ones, pf[t][s2], ls);
      l_run = l_run * alpha + ls[0];
    }
    m_run = m_new;
#pragma unroll
    for (int i = 0; i < NDT; ++i)
#pragma unroll
      for (int j = 0; j < 16; ++j) acc[i][j] *= alpha;
    const bf16_t(*vt_s)[D + 32] = sm.v[half][vst];
    const int g = lane >> 4, li = lane & 15;
#pragma unroll
    for (int dt = 0; dt < NDT; ++dt) {
      const int c0 = 32 * dt + 16 * (g & 1) + 4 * (li & 3);
#pragma unroll
      for (int t = 0; t < 2; ++t)
#pragma unroll
        for (int s2 = 0; s2 < 2; ++s2) {
          const int kb = 32 * t + 16 * s2 + 4 * h + (li >> 2);
          const v4s lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16(
              (__attribute__((address_space(3))) v4s*)(&vt_s[kb][c0]));
          const v4s hi = __builtin_amdgcn_ds_read_tr16_b64_v4i16(
              (__attribute__((address_space(3))) v4s*)(&vt_s[kb + 8][c0]));
          short8 a8;
          a8[0] = lo[0]; a8[1] = lo[1]; a8[2] = lo[2]; a8[3] = lo[3];
          a8[4] = hi[0]; a8[5] = hi[1]; a8[6] = hi[2]; a8[7] = hi[3];
          acc[dt] = mfma32(*reinterpret_cast<bf16x8*>(&a8), pf[t][s2], acc[dt]);
        }
    }
  };
#define ATT2_BARRIER()                                                                \
  asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");                                  \
  __builtin_amdgcn_s_barrier();                                                       \
  asm volatile("" ::: "memory");

  // two K/V stages; tile i+1 is loaded to registers while tile i is computed
  if (ntiles > 0) {
    const int kt0 = min(my_t0, ntiles - 1) * KV_TILE;
    u32x4 kreg[NC], vreg[NC];   // native vectors: HIP's uint4 struct copies stay in scratch
    ATT2_LOAD1(p.k, kt0, kreg)
    ATT2_LOAD1(p.v, kt0, vreg)
    ATT2_STORE1(sm.k[half][0], kreg)
    ATT2_STORE1(sm.v[half][0], vreg)
  }
  for (int it = 0; it < n0; ++it) {
    const int stage = it & 1;
    const int kt = (my_t0 + it) * KV_TILE;
    const int ktn = min(my_t0 + it + 1, ntiles - 1) * KV_TILE;   // next tile (clamped)
    u32x4 kreg[NC], vreg[NC];
    ATT2_LOAD1(p.k, ktn, kreg)                       // lands during this tile's math
    ATT2_LOAD1(p.v, ktn, vreg)
    ATT2_BARRIER()                                   // stage `stage` written by every wave
    if (it < my_n && !(p.causal && kt > qpos_hi)) {
      float16v st[2];
      ATT2_QK(stage, st)
      softmax_pv(st, stage, kt);
    }
    // that stage was last read before this tile's barrier; past a half's last
    // tile the write is never read
    ATT2_STORE1(sm.k[half][stage ^ 1], kreg)
    ATT2_STORE1(sm.v[half][stage ^ 1], vreg)
  }
#undef ATT2_ROW_OFF
#undef ATT2_LOAD1
#undef ATT2_STORE1
#undef ATT2_QK
#undef ATT2_BARRIER

  // ---- merge the two halves: waves 4-7 hand (m, l, O) to waves 0-3 through LDS
  asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
  __builtin_amdgcn_s_barrier();                        // every wave done with the K/V rings
  asm volatile("" ::: "memory");
  float* xo = reinterpret_cast<float*>(&sm);           // [4 waves][NDT * 16][64 lanes]
  float* xml = xo + 4 * NDT * 16 * 64;                 // [4 waves][2][64 lanes]
  if (half) {
#pragma unroll
    for (int dt = 0; dt < NDT; ++dt)
#pragma unroll
      for (int j = 0; j < 16; ++j) xo[(w4 * NDT * 16 + dt * 16 + j) * 64 + lane] = acc[dt][j];
    xml[(w4 * 2) * 64 + lane] = m_run;
    xml[(w4 * 2 + 1) * 64 + lane] = l_run;
  }
  asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
  __builtin_amdgcn_s_barrier();
  asm volatile("" ::: "memory");
  if (half || !row_valid) return;
  const float m1 = xml[(w4 * 2) * 64 + lane], l1 = xml[(w4 * 2 + 1) * 64 + lane];
  const float m = fmaxf(m_run, m1);
  const float a0 = exp2f(m_run - m), a1 = exp2f(m1 - m);
  const float l = l_run * a0 + l1 * a1;
  const float inv = l > 0.f ? 1.f / l : 0.f;
  const float s0 = a0 * inv, s1 = a1 * inv;
  bf16_t* orow = p.o + (size_t)(q0 + qi) * p.o_stride + (size_t)head * D;
#pragma unroll
  for (int dt = 0; dt < NDT; ++dt)
#pragma unroll
    for (int g4 = 0; g4 < 4; ++g4) {
      const int d0 = 32 * dt + 8 * g4 + 4 * h;
      float o[4];
#pragma unroll
      for (int r = 0; r < 4; ++r)
        o[r] = acc[dt][4 * g4 + r] * s0 + xo[(w4 * NDT * 16 + dt * 16 + 4 * g4 + r) * 64 + lane] * s1;
      *reinterpret_cast<uint2*>(orow + d0) = make_uint2(pack_bf16x2(o[0], o[1]), pack_bf16x2(o[2], o[3]));
    }
}

// Combine split-K partials: one workgroup of D threads per (token, head).
__global__ void attn_combine_kernel(const float* __restrict__ part_o,
                                    const float* __restrict__ part_ml, bf16_t* __restrict__ o,
                                    long long o_stride, int total_q, int Hq, int D,
                                    int num_splits) {
  const int tok = blockIdx.x, head = blockIdx.y, d = threadIdx.x;
  float mstar = -1e30f;
  for (int s = 0; s < num_splits; ++s)
    mstar = fmaxf(mstar, part_ml[(((size_t)s * total_q + tok) * Hq + head) * 2]);
  float l = 0.f, acc = 0.f;
  for (int s = 0; s < num_splits; ++s) {
    const size_t idx = ((size_t)s * total_q + tok) * Hq + head;
    const float w = exp2f(part_ml[idx * 2] - mstar);
    l += w * part_ml[idx * 2 + 1];
    acc += w * part_o[idx * D + d];
  }
  o[(size_t)tok * o_stride + (size_t)head * D + d] = f2bf(l > 0.f ? acc / l : 0.f);
}

template <int D, int PAGES, int QW, int KS, bool PARTS = false>
static int launch_pipe(const AttnParams& p, int B, int max_q, hipStream_t s) {
  constexpr int ring = KS * FlashLds<D, D>::RING, end = FlEnd<D / 32, QW, KS, PARTS>::BYTES;
  constexpr int bytes = ring > end ? ring : end;
  static_assert(bytes <= 160 * 1024, "LDS of a CU");
  const dim3 grid((max_q + 32 * QW - 1) / (32 * QW) * (PARTS ? p.parts : 1), p.Hq, B);
  hipLaunchKernelGGL((attn_pipe_kernel<D, PAGES, QW, KS, PARTS>), grid, dim3(64 * QW * KS), bytes, s, p);
  return (int)hipGetLastError();
}

// 64 rows and all runs that LDS holds while these workgroups are one round of the 256 CUs; then
// 128 rows and two runs; with more work, 128 rows and one run in four waves, two or three
// workgroups a CU, which are out of step with each other. us a pass (64-row form, 128 / two,
// 128 / one): 1500 x 8 heads of 64: 15.6, 20, 25; x 20 heads: 26, 22.7, 27; 6 x 1500 x 20 heads:
// 133, 124, 106; 128 columns, paged: 320 rows behind 1000 x 32 heads: 31, 32, 40; 2048 x 32 heads
// causal: 101, 60, 70; 4 x that: 349, 238, 200.
// Short prompts of 128-column heads leave two runs at a second round: their chain of tiles is
// short (128 / two, 128 / one; 9 prompts x 32 heads: 40 rows 14.7, 7.7; 128 behind 300 31.4, 22.6;
// behind 1500 72.7, 63.6).
// Long causal prompts of 64-column heads stay with two runs longer: half of the work is gone and
// the last rows' chain of tiles is what the pass lasts (128 / two, 128 / one): 1400 x 32 heads 24,
// 29; 2048 x 20 heads 40, 50; 4096 x 12 heads 68, 94, x 20 heads 116, 121; but 4 x 700 x 16 heads
// 18.0, 17.0, 3000 x 20 heads 76, 62, 4096 x 32 heads 121, 102.
template <int D, int PAGES>
static int launch_rows(const AttnParams& p, int B, int max_q, hipStream_t s) {
  const long n64 = (long)((max_q + 63) / 64) * p.Hq * B, n128 = (long)((max_q + 127) / 128) * p.Hq * B;
  const long two = D == 128 ? (max_q <= 128 ? 256 : 512) : !p.causal || max_q < 1024 ? 256 : max_q < 4096 ? 384 : 640;
  // parts only of 64-row blocks, all of them one round, and in a kernel of their own: with both in one, launches
  // without parts took 0.2 to 0.4 us more (17 rows x 32 heads of 128 7.8 us, 7.5 alone)
  if (n64 <= 128 && p.parts > 1) return launch_pipe<D, PAGES, 2, D == 64 ? 4 : 2, true>(p, B, max_q, s);
  if (n64 <= 256) return launch_pipe<D, PAGES, 2, D == 64 ? 4 : 2>(p, B, max_q, s);
  if (n128 <= two) return launch_pipe<D, PAGES, 4, 2>(p, B, max_q, s);
  return launch_pipe<D, PAGES, 4, 1>(p, B, max_q, s);
}

template <int D, bool PAGED, bool GROUPED>
static int launch_attn(const AttnParams& p, int B, int max_q, hipStream_t s) {
  dim3 grid;
  if (!GROUPED) {
    // The direct-to-LDS loads and whole-row stores take 16-byte aligned rows, a tile's rows within
    // 32-bit offsets, and cache blocks in which eight (four) rows of one load lie together.
    const bool rows16 = (((size_t)p.q | (size_t)p.k | (size_t)p.v | (size_t)p.o) & 15) == 0 &&
                        ((p.q_stride | p.kv_stride | p.o_stride) & 7) == 0 && p.kv_stride < (1 << 24);
    const bool blocks = p.blk >= 8 && (p.blk & (p.blk - 1)) == 0 && (long)p.Hkv * p.blk < (1 << 22);
    if (rows16 && !PAGED) return launch_rows<D, 0>(p, B, max_q, s);
    if (rows16 && blocks) return p.blk >= FL_KEYS ? launch_rows<D, 1>(p, B, max_q, s) : launch_rows<D, 2>(p, B, max_q, s);
  }
  if (GROUPED) {
    grid = dim3(p.num_splits, p.Hkv, B);
    hipLaunchKernelGGL((attn_fwd_kernel<D, PAGED>), grid, dim3(ATT_THREADS), 0, s, p);
  } else {
    grid = dim3((max_q + 127) / 128, p.Hq, B);
    hipLaunchKernelGGL((attn_prefill2_kernel<D, PAGED>), grid, dim3(512), 0, s, p);
  }
  return (int)hipGetLastError();
}

// mode: 0 = prefill (rows = q tokens of one head), 1 = grouped decode/extend.
extern "C" int loqa_attention(const void* q, long long q_stride, const void* k, const void* v,
                              long long kv_stride, void* o, long long o_stride, const int* cu_q,
                              const int* cu_k, const int* ctx_lens, const int* block_tables,
                              int max_blocks, int blk, int B, int max_q, int Hq, int Hkv, int D,
                              float scale, int causal, int mode, int split_keys, int num_splits,
                              float* part_o, float* part_ml, int total_q, int parts, float* part,
                              long long part_floats, int* words, long long tickets, hipStream_t s) {
  if (B <= 0) return 0;
  if (Hkv <= 0 || Hq % Hkv != 0 || (D != 64 && D != 128)) return (int)hipErrorInvalidValue;
  const bool paged = block_tables != nullptr;
  if (paged && (!ctx_lens || blk <= 0)) return (int)hipErrorInvalidValue;
  if (!paged && !cu_k) return (int)hipErrorInvalidValue;
  if (mode == 1) {
    if ((ATT_WAVES * 32) / (Hq / Hkv) < max_q) return (int)hipErrorInvalidValue;
    if (num_splits < 1 || split_keys % KV_TILE != 0) return (int)hipErrorInvalidValue;
    if (num_splits > 1 && (!part_o || !part_ml)) return (int)hipErrorInvalidValue;
  }
  AttnParams p;
  p.q = (const bf16_t*)q; p.q_stride = q_stride;
  p.k = (const bf16_t*)k; p.v = (const bf16_t*)v; p.kv_stride = kv_stride;
  p.o = (bf16_t*)o; p.o_stride = o_stride;
  p.cu_q = cu_q; p.cu_k = cu_k; p.ctx_lens = ctx_lens; p.block_tables = block_tables;
  p.max_blocks = max_blocks; p.blk = blk; p.Hq = Hq; p.Hkv = Hkv;
  p.scale_log2 = scale * 1.4426950408889634f; p.causal = causal;
  p.split_keys = split_keys; p.num_splits = num_splits; p.part_o = part_o; p.part_ml = part_ml;
  p.total_q = total_q;
  p.parts = parts; p.part = part; p.words = words;
  const long long blocks = (long long)((max_q + 63) / 64) * Hq * B;
  if (parts < 1 || parts > FL_PARTS ||
      (parts > 1 && (mode == 1 || !part || !words || ((size_t)part & 15) || blocks > tickets ||
                     blocks * parts * 2 * fl_join_floats(D / 32) > part_floats)))
    return (int)hipErrorInvalidValue;
  int rc;
#define DISPATCH(DD)                                                                    \
  if (mode == 0) rc = paged ? launch_attn<DD, true, false>(p, B, max_q, s)              \
                            : launch_attn<DD, false, false>(p, B, max_q, s);            \
  else rc = paged ? launch_attn<DD, true, true>(p, B, max_q, s)                         \
                  : launch_attn<DD, false, true>(p, B, max_q, s);
  if (D == 64) { DISPATCH(64) } else { DISPATCH(128) }
#undef DISPATCH
  if (rc != 0) return rc;
  if (mode == 1 && num_splits > 1) {
    hipLaunchKernelGGL(attn_combine_kernel, dim3(total_q, Hq), dim3(D), 0, s, part_o, part_ml,
                       (bf16_t*)o, o_stride, total_q, Hq, D, num_splits);
    rc = (int)hipGetLastError();
  }
  return rc;
}
