// Device parts of the software-pipelined flash attention (attention.hip, attn_window_pipe.hip,
// attn_latent_prefill.hip): a wave's 32 query rows over a run of 64-key tiles.
//
// S^T = K Q^T (v_mfma_f32_32x32x16_bf16: the query lands on the MFMA lane, so row maxima and
// sums are in-register plus one exchange with lane ^ 32) and O^T += V^T P^T with the exp2'ed
// S^T as the B operand as it stands, V^T by transposed LDS reads of the row-major V tile.
//
// What bounds a tile of a wave: at 64 / 64 head columns the VALU (32 exp2 of 8 cycles, fma,
// maximum, conversion, rescaling: ~700 cycles) as much as the MFMAs (640), at 128 / 128 the
// MFMAs (1024). Done one after the other they add up, and two waves of a SIMD that share a barrier
// per tile stay in step instead of filling each other's gaps (fl_loop's phase has them half a tile apart). So the scores of tile i + 1 are
// computed between the exponentials of tile i (first half of the keys), its first P V product
// between those of the second half, and the second P V product covers the row maxima of
// i + 1. O is rescaled in a branch, when a row of the wave has a new maximum.
// (Rescaling only when a maximum passes the reference point by a factor of 256 made the 64
// column form 6 % faster, but the largest weights then no longer lie just below a power of two,
// where bf16's rounding is finest: 4 to 10 % more error.)
// K and V come straight to LDS (16 bytes a lane), two stages each, K one tile ahead of V; a
// lane fetches the chunk that its LDS place holds after an XOR of chunk and row, so rows need
// no padding and both kinds of LDS reads are free of bank conflicts. Taken back: a third stage
// (nothing: the loads cost LDS and L2 time, not waiting), spreading the loads between the MFMAs,
// eight fragments in flight, the barrier between the last MFMAs of a tile (5 % slower).
#pragma once
#include "common.h"

#define FL_KEYS 64                     // keys of a tile
#define FL_PARTS 8                     // parts of a row block's keys at most
#define FL_CAP 8                       // tiles of one at least

typedef short fl_v4s __attribute__((ext_vector_type(4)));
typedef float fl_f2 __attribute__((ext_vector_type(2)));
typedef __bf16 fl_b2 __attribute__((ext_vector_type(2)));
typedef unsigned fl_u4 __attribute__((ext_vector_type(4)));

__device__ __forceinline__ float16v fl_mfma(const bf16x8& a, const bf16x8& b, const float16v& c) {
  return __builtin_amdgcn_mfma_f32_32x32x16_bf16(a, b, c, 0, 0, 0);
}

template <int V> struct Fl { static constexpr int value = V; };

// f(Fl<u>{}) for every u of A .. B - 1: indexes of registers that are constants from the start
template <int A, int B, typename F> __device__ __forceinline__ void fl_each(F&& f) {
  if constexpr (A < B) {
    f(Fl<A>{});
    fl_each<A + 1, B>(f);
  }
}

// f(Fl<run>{}) for a wave-uniform run < KS: what the runs keep in registers at different places
template <int KS, int R = 0, typename F> __device__ __forceinline__ void fl_by_run(int run, F&& f) {
  if constexpr (R + 1 == KS) f(Fl<R>{});
  else if (run == R) f(Fl<R>{});
  else fl_by_run<KS, R + 1>(run, f);
}

template <int DK, int DV> struct FlashLds {
  static constexpr int K = FL_KEYS * DK * 2, V = FL_KEYS * DV * 2;   // bytes of a stage
  static constexpr int RING = 2 * (K + V);                           // K stages, then V stages
};

// Chunk (16 bytes) c of row r lies at place c ^ swz(r). K: 16 rows of one chunk are read at
// once, V: four rows of four chunks; a 256-byte row covers the 64 banks, a 128-byte row half.
template <int D> __device__ __forceinline__ int fl_kswz(int r) { return D % 128 == 0 ? r & 15 : (r >> 1) & 7; }
template <int D> __device__ __forceinline__ int fl_vswz(int r) { return D % 128 == 0 ? (r & 3) << 2 : (r & 2) << 1; }

// LDS by its byte address, which leaves the base and the constant part of an access to one
// register and the instruction's offset.
#define FL_LDS __attribute__((address_space(3)))
__device__ __forceinline__ unsigned fl_lds_at(unsigned char* p) { return (unsigned)(size_t)(FL_LDS unsigned char*)p; }
template <typename T> __device__ __forceinline__ FL_LDS T* fl_lds(unsigned at) { return (FL_LDS T*)(size_t)at; }

// 16 bytes per lane straight to LDS (lane l at dst + 16 l, dst wave-uniform). As the builtin, each
// load made the compiler wait for all of them before the next transposed LDS read, of whose
// address it knows nothing; the waits are fl_sync()'s. No vector register is written.
// A vector memory instruction may read a scalar register 5 wait states after a vector instruction
// (v_readlane: page numbers, spilled scalars) wrote it at the earliest, and the compiler does not
// look into the asm. The scalar unit has no such limit: the base goes through a scalar copy, which
// is also the wait state that m0 asks for.
__device__ __forceinline__ void fl_load_lds(const bf16_t* base, unsigned off, unsigned dst) {   // base wave-uniform
  unsigned long long at;
  asm volatile("s_mov_b32 m0, %1\n\ts_mov_b64 %0, %3\n\tglobal_load_lds_dwordx4 %2, %0"
               : "=&s"(at) : "s"(dst), "v"(off), "s"(base) : "memory", "m0");
}
__device__ __forceinline__ void fl_load_lds(const bf16_t* at, unsigned dst) {
  asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, off" ::"s"(dst), "v"(at) : "memory", "m0");
}

// The fetch of one tile of K (ISV = false) or V rows into a stage by the NTH threads (whole
// waves) of a group, th the thread. Rows past `last` read row `last`; PAD: only cols of the D
// columns exist (the others' places in LDS are left as they are).
template <int D, int NTH, bool ISV, bool PAD> struct FlFetch {
  static constexpr int CH = D / 8, N = FL_KEYS * CH / NTH;
  static constexpr int RG = 64 % CH == 0 ? 64 / CH : 1;     // rows of one instruction of a wave, if whole
  static_assert(N * NTH == FL_KEYS * CH, "whole chunks per thread");
  int th, cols;
  unsigned st;                         // stride of the rows in bytes (64 st < 2^32)
  __device__ __forceinline__ int row(int i, int t) const { return NTH % CH == 0 ? t / CH + i * (NTH / CH) : (t + i * NTH) / CH; }
  __device__ __forceinline__ int chunk(int i, int t) const {
    const int r = row(i, t);
    return ((t + i * NTH) - r * CH) ^ (ISV ? fl_vswz<D>(r) : fl_kswz<D>(r));
  }
  // th once more, for what the last tile alone computes and no register should hold before
  __device__ __forceinline__ int late() const {
    int t = th;
    asm volatile("" : "+v"(t));
    return t;
  }
  __device__ __forceinline__ FlFetch(int th_, int cols_, long long stride) : th(th_), cols(cols_), st((unsigned)stride * 2) {}
  __device__ __forceinline__ unsigned dst(unsigned stage) const { return __builtin_amdgcn_readfirstlane(stage + (th & ~63) * 16); }
  // A whole tile has its own branch: the rows' clamp, as selects in every tile, was 20 to 40 vector instructions
  // of a tile's 180, a multiplication of four times the length per load among them.
  // rows at the stride, from the tile's first (wave-uniform)
  __device__ __forceinline__ void strided(unsigned stage, const bf16_t* base, int last) const {
    const unsigned d = dst(stage);
    if (last >= FL_KEYS - 1) {
#pragma unroll
      for (int i = 0; i < N; ++i)
        if (!PAD || chunk(i, th) * 8 < cols) fl_load_lds(base, (unsigned)row(i, th) * st + chunk(i, th) * 16, d + i * NTH * 16);
    } else {
      const int t = late();
#pragma unroll
      for (int i = 0; i < N; ++i)
        if (!PAD || chunk(i, t) * 8 < cols) fl_load_lds(base, (unsigned)min(row(i, t), last) * st + chunk(i, t) * 16, d + i * NTH * 16);
    }
  }
  // rows in pages of a multiple of RG: at(r), called with wave-uniform multiples of RG, the first of RG rows
  template <typename At> __device__ __forceinline__ void paged(unsigned stage, int last, At&& at) const {
    static_assert(64 % CH == 0, "whole rows per instruction");
    const unsigned d = dst(stage);
    const int w0 = __builtin_amdgcn_readfirstlane(th & ~63) / CH;
    if (last >= FL_KEYS - 1) {
#pragma unroll
      for (int i = 0; i < N; ++i) {
        const bf16_t* base = at(w0 + i * (NTH / CH));
        if (!PAD || chunk(i, th) * 8 < cols) fl_load_lds(base, (unsigned)((th & 63) / CH) * st + chunk(i, th) * 16, d + i * NTH * 16);
      }
    } else {
      const int t = late(), in = (t & 63) / CH;
#pragma unroll
      for (int i = 0; i < N; ++i) {
        const int r = min(w0 + i * (NTH / CH), last & ~(RG - 1));
        const bf16_t* base = at(r);
        if (!PAD || chunk(i, t) * 8 < cols) fl_load_lds(base, (unsigned)min(in, last - r) * st + chunk(i, t) * 16, d + i * NTH * 16);
      }
    }
  }
};

// A sequence's block table for pages of 1 << sh rows, 64 entries at a time (one a lane).
struct FlPages {
  const int* tab;
  int sh, last, base, held;            // last: the last page of use
  __device__ __forceinline__ FlPages(const int* t, int sh_, int keys)
      : tab(t), sh(sh_), last(max(keys - 1, 0) >> sh_), base(-64), held(0) {}
  // the table's part for keys kt .. kt + 63 (at most 64 pages)
  __device__ __forceinline__ void hold(int kt, int lane) {
    if (min((kt + FL_KEYS - 1) >> sh, last) >= base + 64) {
      base = __builtin_amdgcn_readfirstlane(kt >> sh);
      held = tab[min(base + lane, last)];
    }
  }
  __device__ __forceinline__ int page(int key) const { return __builtin_amdgcn_readlane(held, (key >> sh) - base); }
};

// every load of this wave has landed, its LDS reads are done, and so for the other waves
__device__ __forceinline__ void fl_sync() {
  asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)" ::: "memory");
  __builtin_amdgcn_s_barrier();
  asm volatile("" ::: "memory");
}

// the same for the first tile of K only, with N loads behind it
template <int N> __device__ __forceinline__ void fl_sync_first() {
  static_assert(N < 64, "vmcnt range");
  asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)" ::"n"(N) : "memory");
  __builtin_amdgcn_s_barrier();
  asm volatile("" ::: "memory");
}

// every wave is here, whatever it waits for
__device__ __forceinline__ void fl_step() {
  asm volatile("" ::: "memory");
  __builtin_amdgcn_s_barrier();
  asm volatile("" ::: "memory");
}

// LDS writes of all waves are visible; global loads stay in flight
__device__ __forceinline__ void fl_meet() {
  asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
  __builtin_amdgcn_s_barrier();
  asm volatile("" ::: "memory");
}

__device__ __forceinline__ float fl_max32(float x) {   // over lane and lane ^ 32
  typedef unsigned u2 __attribute__((ext_vector_type(2)));
  const u2 r = __builtin_amdgcn_permlane32_swap(__float_as_uint(x), __float_as_uint(x), false, false);
  return fmaxf(__uint_as_float(r[0]), __uint_as_float(r[1]));
}

__device__ __forceinline__ float fl_both32(float x) {  // lane + lane ^ 32
  typedef unsigned u2 __attribute__((ext_vector_type(2)));
  const u2 r = __builtin_amdgcn_permlane32_swap(__float_as_uint(x), __float_as_uint(x), false, false);
  return __uint_as_float(r[0]) + __uint_as_float(r[1]);
}

// The tiles 0 .. n - 1 of a group of waves that share a ring (n the same for every wave that
// meets the barriers): acc and l get sum P V and sum P relative to exp2(m), scores in units
// of sl2 (> 0). prep(st, i) masks (or transforms) the scores of tile i: register 16 t + j of
// lane (column, h) is key 32 t + (j & 3) + 8 (j >> 2) + 4 h; a wave whose rows see nothing of a
// tile masks all of it (it would wait for the others anyway, and one path through the loop
// leaves the registers where they are). load_k / load_v(i, stage) start the fetch of tile i;
// they are called for i = 1, 2, .. up to n (K) and i = 0 .. n - 1 (V); for i = n they must fetch
// something that exists (or nothing). Where n > 0 the caller has started the fetch of K tile 0 into the ring, ahead of
// its loads of Q or behind them: one trip to memory for both. V 0 is asked for before the first wait, which is for K 0, and K 1 behind
// it, or with BOTH before it as well; counted: those are BEHIND loads of every wave exactly.
// (What a form takes is what it measured: with K 0 behind Q and K 1 behind the wait, windowed prompts of 64-column heads in 512
// keys 17.0 -> 16.3 us, causal ones of 1300 rows x 32 such heads 24.7 -> 23.9; 64-row blocks of 128-column heads off pages go with K 0 ahead
// of Q and BOTH, as the other order leaves registers to scratch there, and so do latent prompts and runs of four waves off
// contiguous keys, which it cost 1 % and 0.5: 8 x 1500 rows x 8 heads of 64 52.9 us, 52.4.)
// phase: -1, or in workgroups of eight waves 0 for the first four and 1 for the others, which share the four SIMDs: each
// half of a tile then begins with a barrier of all waves, and the second four run half a tile behind, their exponentials,
// maxima and rescaling beside the scores' MFMAs of the first (in step, both waves of a SIMD want the same unit; 2048 rows of
// 16 latent heads of 192 / 128 43.7 -> 41.6 us, of 32 58.5 -> 56.7, 1500 rows x 8 heads of 64 on four runs 13.7 -> 12.9; wave priorities
// and six or eight fragments in flight beside it: the same within 1 %). The half tile more is too much for runs of few tiles
// (windows of 300 keys, four tiles a run: 2048 rows x 16 heads of 64 14.5 us in step, 15.3 apart; of 128 19.3, 19.7), so a workgroup
// takes it from FL_APART tiles a run on.
// Before the call m = -1e30, l = 0, acc = 0; ring must not be in use. After it the waves
// are not synchronised.
#define FL_APART 6

template <int DK, int DV, int BEHIND, bool BOTH, typename Prep, typename LoadK, typename LoadV>
__device__ __forceinline__ void fl_loop(const bf16x8 (&qf)[DK / 16], float16v (&acc)[DV / 32], float& m, float& l,
                                        unsigned ring, int n, float sl2, int lane, bool counted, int phase, Prep&& prep,
                                        LoadK&& load_k, LoadV&& load_v) {
  using L = FlashLds<DK, DV>;
  // The sums of a tile's P, rounded to bf16 as in the numerator, so that a row's weights add up to
  // one exactly: as one more output column block where the VALU is what is short, as dot products
  // with ones where the MFMAs are. Error against 64 bits of windowed and latent prompts, whose
  // sums were of the f32 exponentials before (1000 rows in two feeds, without and with a sink,
  // three spreads of the scores): 0.00173 - 0.00223 then, 0.00170 - 0.00220 now, less in each of
  // 24 comparisons; with f32 sums here between the two, and 192 / 128 columns behind 1000 keys
  // 40 -> 62 us.
  constexpr bool ROW = DV <= 64;
  constexpr int NS = DK / 16, NDT = DV / 32, NQ = 2 * NS, NW = NDT + ROW, NP = 2 * NW;
  const int h = lane >> 5, li = lane & 15;
  // K fragment (t, s): row 32 t + (lane & 31), chunk 2 s + h; the XOR keeps the chunk's part
  // above its 3 or 4 bits, so that part and t are constants added to a lane's base
  constexpr int KM = DK % 128 == 0 ? 8 : 4;            // fragments of a swizzled run
  unsigned kb[KM];
#pragma unroll
  for (int s = 0; s < KM; ++s) kb[s] = ring + (lane & 31) * (DK * 2) + ((2 * s + h) ^ fl_kswz<DK>(lane & 31)) * 16;
  // V fragment (t, s2, dt): rows 32 t + 16 s2 + 4 h + (li >> 2), + 8, columns 32 dt + 16 (lane / 16 & 1) + 4 (li & 3)
  unsigned vb[NDT];
#pragma unroll
  for (int d = 0; d < NDT; ++d)
    vb[d] = ring + 2 * L::K + (4 * h + (li >> 2)) * (DV * 2) +
            ((4 * d + 2 * ((lane >> 4) & 1) + ((li & 3) >> 1)) ^ fl_vswz<DV>(li >> 2)) * 16 + (li & 1) * 8;
  constexpr int KR = 4, VR = 4;                        // fragments in flight + 1
  const float16v zero = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
  bf16x8 ones;
#pragma unroll
  for (int j = 0; j < 8; ++j) ones[j] = (__bf16)1.0f;
  const fl_b2 one2 = {(__bf16)1.0f, (__bf16)1.0f};

  // Q is here, and a K 0 asked for ahead of it, before the next loads whose wait the compiler does not know
  bf16x8 qr[NS];
#pragma unroll
  for (int s = 0; s < NS; ++s) {
    qr[s] = qf[s];
    asm volatile("" : "+v"(qr[s]));
  }
  // cur: scores of tile i (SM: softmax and P V of it), nxt: of tile i + 1 (QK: compute them);
  // V of i lies in stage S, K of i + 1 in stage 1 - S
  auto body = [&](auto qk, auto sm, auto slot, float16v(&cur)[2], float16v(&nxt)[2], int i) __attribute__((always_inline)) {
    constexpr bool QK = decltype(qk)::value != 0, SM = decltype(sm)::value != 0;
    constexpr int S = decltype(slot)::value;
    bf16x8 kf[KR], vf[VR];
    fl_u4 pf[2][2];
    auto kread = [&](int u, int stage) __attribute__((always_inline)) {
      const int t = u & 1, s = u >> 1;
      kf[u % KR] = *fl_lds<bf16x8>(kb[s % KM] + (stage * L::K + 32 * t * DK * 2 + s / KM * KM * 32));
    };
    auto vread = [&](int v) __attribute__((always_inline)) {      // v = (2 t + s2) NDT + dt
      const int ts = v / NDT, d = v % NDT;
      const unsigned a = vb[d] + (S * L::V + 16 * ts * DV * 2);
      const fl_v4s lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16(fl_lds<fl_v4s>(a));
      const fl_v4s hi = __builtin_amdgcn_ds_read_tr16_b64_v4i16(fl_lds<fl_v4s>(a + 8 * DV * 2));
      short8 a8;
      a8[0] = lo[0]; a8[1] = lo[1]; a8[2] = lo[2]; a8[3] = lo[3];
      a8[4] = hi[0]; a8[5] = hi[1]; a8[6] = hi[2]; a8[7] = hi[3];
      vf[v % VR] = *reinterpret_cast<bf16x8*>(&a8);
    };
    // the exponentials of slice w of N: pairs of scores of key half t
    auto exps = [&](int t, int w, int N) __attribute__((always_inline)) {
#pragma unroll
      for (int q = w * 8 / N; q < (w + 1) * 8 / N; ++q) {
        fl_f2 e;
        e[0] = __builtin_amdgcn_exp2f(fmaf(cur[t][2 * q], sl2, -m));
        e[1] = __builtin_amdgcn_exp2f(fmaf(cur[t][2 * q + 1], sl2, -m));
        const fl_b2 b = __builtin_convertvector(e, fl_b2);
        pf[t][q >> 2][q & 3] = __builtin_bit_cast(unsigned, b);
        if constexpr (!ROW) l = __builtin_amdgcn_fdot2_f32_bf16(b, one2, l, false);
      }
    };
    float16v ls;
    auto pv = [&](int t, int w) __attribute__((always_inline)) {  // MFMA w of half t; reads three ahead
      const int s2 = w / NW, d = w % NW - ROW, v = (2 * t + s2) * NDT + d;
      const bf16x8 p8 = __builtin_bit_cast(bf16x8, pf[t][s2]);
      if (d < 0)
        ls = fl_mfma(ones, p8, t + s2 == 0 ? zero : ls);
      else {
        acc[d] = fl_mfma(vf[v % VR], p8, acc[d]);
        if (v + VR - 1 < 4 * NDT) vread(v + VR - 1);
      }
    };
    // tile i's V and i + 1's K are here, the K of i and the V of i - 1 have been read
    if constexpr (SM) {
      fl_sync();
    } else {
      load_v(0, ring + 2 * L::K);
      if constexpr (BOTH) load_k(1, ring + L::K);
      if (counted) fl_sync_first<BEHIND>();
      else fl_sync();
    }
    if constexpr (QK) {
#pragma unroll
      for (int u = 0; u < KR - 1; ++u) kread(u, 1 - S);
      if constexpr (SM) {
        load_k(i + 2, ring + S * L::K);
        load_v(i + 1, ring + 2 * L::K + (1 - S) * L::V);
      } else if constexpr (!BOTH) {
        load_k(1, ring + L::K);
      }
    }
#pragma unroll
    for (int u = 0; u < NQ; ++u) {
      if constexpr (QK) {
        const int t = u & 1, s = u >> 1;
        nxt[t] = fl_mfma(kf[u % KR], qr[s], s == 0 ? zero : nxt[t]);
        if (u + KR - 1 < NQ) kread(u + KR - 1, 1 - S);
      }
      if constexpr (SM) {
        exps(0, u, NQ);
        if (u >= NQ - (VR - 1)) vread(u - (NQ - (VR - 1)));
      }
      __builtin_amdgcn_sched_barrier(0);
    }
    // what is used in a later block stays computed in this one
    if constexpr (SM) asm volatile("" : "+v"(pf[0][0]), "+v"(pf[0][1]));
    if (phase >= 0) fl_step();
    if constexpr (QK) prep(nxt, i + 1);
    if constexpr (SM) {
#pragma unroll
      for (int w = 0; w < NP; ++w) {
        pv(0, w);
        exps(1, w, NP);
        __builtin_amdgcn_sched_barrier(0);
      }
    }
    float mx[2] = {-INFINITY, -INFINITY};
#pragma unroll
    for (int w = 0; w < NP; ++w) {
      if constexpr (SM) pv(1, w);
      if constexpr (QK) {
#pragma unroll
        for (int q = w * 16 / NP; q < (w + 1) * 16 / NP; ++q)
          mx[q & 1] = fmaxf(fmaxf(mx[q & 1], nxt[q >> 3][2 * (q & 7)]), nxt[q >> 3][2 * (q & 7) + 1]);
      }
      if constexpr (SM) __builtin_amdgcn_sched_barrier(0);
    }
    if constexpr (SM && ROW) l += ls[0];
    if constexpr (QK) {
      const float top = fl_max32(fmaxf(mx[0], mx[1])) * sl2;
      if (__any(top > m)) {
        const float m_new = fmaxf(m, top), alpha = __builtin_amdgcn_exp2f(m - m_new);
        m = m_new;
        l *= alpha;
#pragma unroll
        for (int d = 0; d < NDT; ++d) {
#pragma unroll
          for (int j = 0; j < 16; ++j) acc[d][j] *= alpha;
          asm volatile("" : "+v"(acc[d]));              // one value, so that no path copies it
        }
      }
    }
  };

  if (n <= 0) return;
  float16v sa[2], sb[2];
  if (phase == 1) fl_step();
  body(Fl<1>{}, Fl<0>{}, Fl<1>{}, sb, sa, -1);         // scores of tile 0; fetches V 0 and K 1
  int i = 0;
  for (; i + 2 < n; i += 2) {
    body(Fl<1>{}, Fl<1>{}, Fl<0>{}, sa, sb, i);
    body(Fl<1>{}, Fl<1>{}, Fl<1>{}, sb, sa, i + 1);
  }
  if (i + 1 < n) {
    body(Fl<1>{}, Fl<1>{}, Fl<0>{}, sa, sb, i);
    sa[0] = sb[0];
    sa[1] = sb[1];
#pragma unroll
    for (int d = 0; d < NDT; ++d) vb[d] += L::V;        // the last tile's V lies in the other stage
  }
  body(Fl<0>{}, Fl<1>{}, Fl<0>{}, sa, sb, n - 1);
  if (phase == 0) fl_step();
  if constexpr (!ROW) l = fl_both32(l);                 // a lane has summed its half of the keys
}

// ---- the end of a pass. The KS runs of a query block meet in LDS, and each of them finishes its share of the
// output: a unit is four columns of a lane's row (accumulators 4 g .. of block d: unit 4 d + g), a run's
// units lie side by side. With run 0 finishing all of it, as it was, half or three quarters of the waves stood idle behind the last
// tile (with K 0 fetched ahead of Q as well: 64 rows and keys x 16 heads of 192 / 128 9.4 -> 8.1 us, 1024 x 16 22.0 -> 20.8;
// 1500 rows x 8 heads of 64 behind 256 keys 6.7 -> 6.2). ALL: run 0 has all units (what other workgroups join, fl_join).
template <int NDT, int QW, int KS, bool ALL = false> struct FlEnd {
  static constexpr int U = 4 * NDT;
  static constexpr int first(int r) { return ALL ? (r ? U : 0) : r * U / KS; }
  static constexpr int count(int r) { return first(r + 1) - first(r); }
  static constexpr int OWN = ALL ? U : U / KS;
  static_assert(ALL || OWN * KS == U, "whole units for every run");
  static constexpr bool own(int r, int u) { return u >= first(r) && u < first(r + 1); }
  // the place of unit u among the others' that run r leaves in LDS, a kilobyte each per wave of rows
  static constexpr int slot(int r, int u) { return r * U - first(r) + (u < first(r) ? u : u - count(r)); }
  static constexpr int ML = (KS - 1) * U * QW * 1024;                  // where (m, l) lie
  static constexpr int MERGE = KS > 1 ? ML + KS * QW * 512 : 0;        // bytes
  static constexpr int LD = NDT * 64 + 16, ROWS = 32 * LD;             // of a row and of a wave's 32 rows as bf16, behind those
  static constexpr int BYTES = MERGE + QW * ROWS;
};

template <int U, int NDT> __device__ __forceinline__ float4v fl_unit(const float16v (&acc)[NDT]) {
  constexpr int d = U / 4, j = 4 * (U % 4);
  return float4v{acc[d][j], acc[d][j + 1], acc[d][j + 2], acc[d][j + 3]};
}

template <int NDT, int N> __device__ __forceinline__ void fl_units(const float16v (&acc)[NDT], float4v (&own)[N]) {
  static_assert(N == 4 * NDT, "all of them");
  fl_each<0, N>([&](auto c) __attribute__((always_inline)) { own[decltype(c)::value] = fl_unit<decltype(c)::value>(acc); });
}

// Called by all waves, the rings no longer in use. Afterwards m and l are the joint ones and own has the run's units;
// with ALL acc of run 0 has them, and the other runs' are of no use.
template <int NDT, int QW, int KS, bool ALL, int N>
__device__ __forceinline__ void fl_merge(float16v (&acc)[NDT], float4v (&own)[N], float& m, float& l,
                                         unsigned char* lds, int run, int wq, int lane) {
  using E = FlEnd<NDT, QW, KS, ALL>;
  if constexpr (KS == 1) {
    fl_units(acc, own);
  } else {
    unsigned char* x = lds + wq * 1024 + lane * 16;
    fl_by_run<KS>(run, [&](auto r) __attribute__((always_inline)) {
      constexpr int R = decltype(r)::value;
      fl_each<0, E::U>([&](auto c) __attribute__((always_inline)) {
        constexpr int u = decltype(c)::value;
        if constexpr (!E::own(R, u)) *reinterpret_cast<float4v*>(x + E::slot(R, u) * QW * 1024) = fl_unit<u>(acc);
      });
    });
    float2* ml = reinterpret_cast<float2*>(lds + E::ML + wq * 512 + lane * 8);
    ml[run * QW * 64] = make_float2(m, l);
    fl_meet();
    if (ALL && run) return;
    float a[KS], lr[KS];
#pragma unroll
    for (int r = 0; r < KS; ++r) {
      const float2 v = ml[r * QW * 64];
      a[r] = v.x;
      lr[r] = v.y;
    }
    m = a[0];
#pragma unroll
    for (int r = 1; r < KS; ++r) m = fmaxf(m, a[r]);
    l = 0.f;
#pragma unroll
    for (int r = 0; r < KS; ++r) {
      a[r] = exp2f(a[r] - m);
      l = r ? l + lr[r] * a[r] : lr[r] * a[r];
    }
    fl_by_run<ALL ? 1 : KS>(run, [&](auto r) __attribute__((always_inline)) {
      constexpr int R = decltype(r)::value;
      fl_each<E::first(R), E::first(R + 1)>([&](auto c) __attribute__((always_inline)) {
        constexpr int u = decltype(c)::value;
        float4v s = {0.f, 0.f, 0.f, 0.f};
        fl_each<0, KS>([&](auto kc) __attribute__((always_inline)) {
          constexpr int k = decltype(kc)::value;
          float4v v;
          if constexpr (k == R) v = fl_unit<u>(acc);
          else v = *reinterpret_cast<const float4v*>(x + E::slot(k, u) * QW * 1024);
          if constexpr (k == 0) s = v * a[k];
          else s = s + v * a[k];
        });
        if constexpr (ALL)
          fl_each<0, 4>([&](auto e) __attribute__((always_inline)) { acc[u / 4][4 * (u % 4) + decltype(e)::value] = s[decltype(e)::value]; });
        else own[u - E::first(R)] = s;
      });
    });
  }
}

// The first column of a run's s-th unit for a lane (the unit's own of ALL: run 0).
template <int NDT, int QW, int KS, bool ALL> __device__ __forceinline__ int fl_column(int s, int run, int lane) {
  return 8 * ((ALL ? 0 : run * FlEnd<NDT, QW, KS, ALL>::OWN) + s) + 4 * (lane >> 5);
}

// A run's finished units of a wave's 32 rows as bf16 to y (rows ld apart, `rows` of them exist, `cols` <= 32 NDT columns,
// a multiple of 8), turned through LDS: a lane's units are 4 columns of its row each, and 8-byte pieces of 32 rows in one
// store make every piece a line of its own. Each run stores its share of whole rows.
template <int NDT, int QW, int KS, bool ALL, int OWN>
__device__ __forceinline__ void fl_store(const float4v (&own)[OWN], unsigned char* lds, bf16_t* y, long long ld,
                                         int rows, int cols, int run, int wq, int lane) {
  using E = FlEnd<NDT, QW, KS, ALL>;
  static_assert(OWN == E::OWN, "a run's units");
  constexpr int CPR = NDT * 4, N = ALL ? 32 : 32 / KS;      // 16-byte pieces of a row, rows of a run
  unsigned char* my = lds + E::MERGE + wq * E::ROWS;
#pragma unroll
  for (int s = 0; s < E::OWN; ++s)
    *reinterpret_cast<uint2*>(my + (lane & 31) * E::LD + fl_column<NDT, QW, KS, ALL>(s, run, lane) * 2) =
        make_uint2(pack_bf16x2(own[s][0], own[s][1]), pack_bf16x2(own[s][2], own[s][3]));
  if constexpr (KS > 1 && !ALL) fl_meet();
  else __builtin_amdgcn_wave_barrier();
  const int r0 = KS > 1 && !ALL ? run * N : 0;
#pragma unroll
  for (int k = 0; k < N * CPR / 64; ++k) {
    const int id = lane + 64 * k, r = r0 + id / CPR, c = id % CPR;
    const fl_u4 v = *reinterpret_cast<const fl_u4*>(my + r * E::LD + c * 16);
    if (r < rows && c * 8 < cols) *reinterpret_cast<fl_u4*>(y + (size_t)r * ld + c * 8) = v;
  }
}

// Parts of a row block's keys in workgroups of their own (n > 1 of them): each wave of rows publishes its
// (m, l, acc), the last part to arrive gets the joint values and returns true, whichever it is summed up in
// the parts' order. part: n slots of the block, QW fl_join_floats each; words: the block's 2 QW <= TICKET
// zeroed words, zero again afterwards (arrivals, and parts that can be read: the last waits for those, whose
// owners are past everything but their own stores). Written through and read past the caches (sc1).
// Publishing and joining two parts takes 3 to 4 us (64 rows x 32 heads of 128 behind 1000 keys: 22.2 us whole, 16.7).
__host__ __device__ constexpr int fl_join_floats(int NDT) { return (NDT * 16 + 4) * 64; }

// The n <= N parts' values, LB 16-byte pieces of each part's slot asked for at a time.
template <int NDT, int QW, int N, int LB>
__device__ __forceinline__ void fl_join_sum(float16v (&acc)[NDT], float& m, float& l, const __amdgpu_buffer_rsrc_t& r, int n, int mine,
                                            int wq, int lane) {
  constexpr int PER = fl_join_floats(NDT) * 4, SC1 = 16, O = N == 2 ? 1 : N;   // of two parts one is the other
  auto load = [&](int i, int piece) __attribute__((always_inline)) {
    return __builtin_bit_cast(fl_u4, __builtin_amdgcn_raw_buffer_load_b128(r, (i * QW + wq) * PER + piece * 1024 + lane * 16, 0, SC1));
  };
  float a[N], lp[N], top = m;
  fl_u4 ml[O], o[O][LB];
  auto fetch = [&](int p0) __attribute__((always_inline)) {
#pragma unroll
    for (int i = 0; i < O; ++i)
      if (N == 2 || (i < n && i != mine))
#pragma unroll
        for (int k = 0; k < LB; ++k) o[i][k] = load(N == 2 ? 1 - mine : i, p0 + k);
  };
#pragma unroll
  for (int i = 0; i < O; ++i)
    if (N == 2 || (i < n && i != mine)) ml[i] = load(N == 2 ? 1 - mine : i, 4 * NDT);
  fetch(0);
#pragma unroll
  for (int i = 0; i < N; ++i) {
    const bool own = i == mine, there = i < n;
    a[i] = own ? m : there ? __uint_as_float(ml[N == 2 ? 0 : i][0]) : -1e30f;
    lp[i] = own ? l : there ? __uint_as_float(ml[N == 2 ? 0 : i][1]) : 0.f;
    top = fmaxf(top, a[i]);
  }
  l = 0.f;
#pragma unroll
  for (int i = 0; i < N; ++i) {
    a[i] = exp2f(a[i] - top);
    l += lp[i] * a[i];
  }
  m = top;
#pragma unroll
  for (int p0 = 0; p0 < 4 * NDT; p0 += LB) {
    if (p0) fetch(p0);
    float sum[LB * 4];
#pragma unroll
    for (int j = 0; j < LB * 4; ++j) sum[j] = 0.f;
#pragma unroll
    for (int i = 0; i < N; ++i)
      if (i < n)
#pragma unroll
        for (int j = 0; j < LB * 4; ++j)
          sum[j] = fmaf(i == mine ? acc[p0 / 4 + j / 16][(p0 % 4) * 4 + j % 16] : __uint_as_float(o[N == 2 ? 0 : i][j >> 2][j & 3]), a[i], sum[j]);
#pragma unroll
    for (int j = 0; j < LB * 4; ++j) acc[p0 / 4 + j / 16][(p0 % 4) * 4 + j % 16] = sum[j];
  }
}

template <int NDT, int QW>
__device__ __forceinline__ bool fl_join(float16v (&acc)[NDT], float& m, float& l, float* part, int* words, int n, int mine, int wq,
                                        int lane) {
  constexpr int PER = fl_join_floats(NDT) * 4, SC1 = 16;          // bytes of a wave's slot
  const __amdgpu_buffer_rsrc_t r = __builtin_amdgcn_make_buffer_rsrc(part, 0, n * QW * PER, 0x00020000);
  int* word = words + 2 * wq;
  int old = 0;
  if (lane == 0) old = __hip_atomic_fetch_add(word, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  old = __builtin_amdgcn_readfirstlane(old);
  if (old != n - 1) {
    const int at = (mine * QW + wq) * PER;
#pragma unroll
    for (int d = 0; d < NDT; ++d)
#pragma unroll
      for (int g = 0; g < 4; ++g) {
        const fl_u4 v = {__float_as_uint(acc[d][4 * g]), __float_as_uint(acc[d][4 * g + 1]), __float_as_uint(acc[d][4 * g + 2]),
                         __float_as_uint(acc[d][4 * g + 3])};
        __builtin_amdgcn_raw_buffer_store_b128(v, r, at + (4 * d + g) * 1024 + lane * 16, 0, SC1);
      }
    const fl_u4 ml = {__float_as_uint(m), __float_as_uint(l), 0u, 0u};
    __builtin_amdgcn_raw_buffer_store_b128(ml, r, at + 4 * NDT * 1024 + lane * 16, 0, SC1);
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");   // written through: visible when acknowledged
    if (lane == 0) __hip_atomic_fetch_add(word + 1, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    return false;
  }
  while (__hip_atomic_load(word + 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) != n - 1) __builtin_amdgcn_s_sleep(1);
  asm volatile("" ::: "memory");
  if (lane == 0) {
    __hip_atomic_store(word, 0, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    __hip_atomic_store(word + 1, 0, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  }
  // as many loads in flight as registers allow: the trip is what this costs
  if (n == 2) fl_join_sum<NDT, QW, 2, NDT * 4>(acc, m, l, r, n, mine, wq, lane);
  else if (n <= 4) fl_join_sum<NDT, QW, 4, 4>(acc, m, l, r, n, mine, wq, lane);
  else fl_join_sum<NDT, QW, FL_PARTS, 2>(acc, m, l, r, n, mine, wq, lane);
  return true;
}
