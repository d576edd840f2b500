// Decode attention with the keys and values streamed through LDS: the form of attn_decode.hip for up to
// 16 query rows per kv head (a GQA group times the tokens fed).
//
// A token step reads every cached key and value once, so it is bound by the bytes that a compute unit has
// under way (64 KB over 1.2 us of latency) and by what stands around the stream: metadata, the first
// trip to memory, the merge. A wave that loads a tile of 32 keys into registers, works on it and loads the
// next has nothing under way half of the time (2.4 us a tile). Here a wave's loads go straight to its own
// ring of two tiles in LDS, the next tile's on their way while it works on one. 1500 keys x 20 heads of 64, eight
// sequences (61 MB) 19.6 -> 16.2 us, one 10.3 -> 7.4; 600 keys x 8 heads of 128, eight sequences 12.8 -> 10.2;
// 4000 keys in splits of 128 61 -> 25, 32 sequences of them 249 -> 92 (5.7 TB/s):
//
//   S^T = K Q^T    : 16 x 16 x 32 MFMAs, K rows from LDS (16-byte chunks swizzled on the source address)
//   O^T += V^T P^T : V^T from LDS by transposing reads; P^T is the S^T accumulator as it stands: the keys of
//                    a lane (4 q .. 4 q + 3 of both halves of the tile) are the K slots of its V^T operand
//   merge          : every thread of the workgroup sums up four columns of a row over the waves
//   splits         : as in attn_decode.hip, the last to arrive merges; but a workgroup takes as many of the
//                    caller's splits as leave the chip filled (attn_stream below)
#include "attn_decode.h"

#define AS_ROWS 16

template <int D> constexpr int as_tile_bytes() { return DEC_TILE * D * 2; }   // of K, and of V

// 16 bytes per lane at rsrc + off straight to LDS at dst + 16 lane, zeros from out of range. As the
// builtin, the loads made the compiler wait for all of them before every transposed LDS read; here the
// waits are as_wait()'s, and the kernel has no other vector load before its last tile. No vector register
// is written. A scalar register that a vector instruction wrote may be read 5 wait states later at the
// earliest, and the compiler does not look into the asm: hence the s_nop, which also covers m0.
typedef unsigned as_u4 __attribute__((ext_vector_type(4)));
__device__ __forceinline__ as_u4 as_rsrc(const bf16_t* base, unsigned bytes) {
  const unsigned long long at = (unsigned long long)base;
  return as_u4{(unsigned)__builtin_amdgcn_readfirstlane((int)at), (unsigned)__builtin_amdgcn_readfirstlane((int)(at >> 32)),
               (unsigned)__builtin_amdgcn_readfirstlane((int)bytes), 0x00020000u};
}
__device__ __forceinline__ void as_load_lds(const as_u4& rsrc, unsigned off, unsigned dst) {
  asm volatile("s_mov_b32 m0, %0\n\ts_nop 4\n\tbuffer_load_dwordx4 %1, %2, 0 offen lds" ::"s"(dst), "v"(off), "s"(rsrc) : "memory", "m0");
}
template <int N> __device__ __forceinline__ void as_wait() { asm volatile("s_waitcnt vmcnt(%0)" ::"n"(N) : "memory"); }

#define AS_LDS __attribute__((address_space(3)))
template <typename T> __device__ __forceinline__ AS_LDS T* as_lds(unsigned at) { return (AS_LDS T*)(size_t)at; }

// metadata by the scalar unit, whatever the asm may do to memory: nothing writes it during a launch
__device__ __forceinline__ int as_scalar(const int* p) { return *(const __attribute__((address_space(4))) int*)(size_t)p; }

template <int D, int NW, int R> constexpr int as_smem() {
  constexpr int ring = NW * (2 * R * as_tile_bytes<D>() + AS_ROWS * D * 2);
  static_assert(NW * AS_ROWS * (D + 4 + 2) * 4 + 16 <= ring, "the merge must fit the rings");
  return ring;
}

// R: stages of a wave's ring; one where no wave has a second tile
template <int D, bool PAGED, int NW, int R>
__global__ __launch_bounds__(NW * 64) void attn_stream_kernel(AttnDecArgs A) {
  if (A.prio) __builtin_amdgcn_s_setprio(3);     // kernel argument: wave-uniform
  constexpr int TB = as_tile_bytes<D>(), LPR = D / 8, RPL = 64 / LPR, NL = DEC_TILE / RPL;   // lanes a row, rows a load, loads
  constexpr int NS = D / 32, ND = D / 16, LD = D + 4, NQ = AS_ROWS / RPL, STEP = NW * DEC_TILE;
  __shared__ __attribute__((aligned(1024))) unsigned char lds[as_smem<D, NW, R>()];
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int li = lane & 15, fq = lane >> 4;
  const int split = blockIdx.x, kvh = blockIdx.y, b = blockIdx.z;
  const int G = A.Hq / A.Hkv, blk = A.blk, sh = PAGED ? __builtin_ctz(blk) : 0;   // rows of a page: a power of two
  const int kbeg = split * A.split_keys;
  // block-table entries of a tile: two pages of 16 rows, or one
  const int* bt = PAGED ? A.block_tables + (size_t)b * A.max_blocks : nullptr;
  auto page_at = [&](int kt, int i) { return as_scalar(bt + min((kt >> sh) + i, A.max_blocks - 1)); };
  int pages[2][2] = {{0, 0}, {0, 0}};            // of the tile asked for next and of the one behind it
  const int kt0 = kbeg + wave * DEC_TILE;
  if constexpr (PAGED) {
    pages[0][0] = page_at(kt0, 0); pages[0][1] = page_at(kt0, 1);
    if constexpr (R > 1) { pages[1][0] = page_at(kt0 + STEP, 0); pages[1][1] = page_at(kt0 + STEP, 1); }
  }
  const int q0 = as_scalar(A.cu_q + b), qlen = as_scalar(A.cu_q + b + 1) - q0, klen = as_scalar(A.ctx_lens + b);
  const int kend = min(klen, kbeg + A.split_keys);
  const int kv0_of = PAGED ? 0 : as_scalar(A.kv_start + b);
  if (split > 0 && kbeg >= klen) return;
  const size_t kv0 = PAGED ? 0 : (size_t)kv0_of;
  const int rows = min(qlen * G, AS_ROWS);       // row r: token r / G, head r % G of the group
  const int qpos = klen - qlen + li / G;

  // lane l of load j brings chunk (l % LPR) ^ swz of row RPL j + l / LPR
  auto swz = [](int row) { return D == 64 ? (row >> 1) & 7 : row & 15; };
  const unsigned stride = PAGED ? D * 2 : (unsigned)A.kv_stride * 2;
  unsigned voff[NL];
#pragma unroll
  for (int j = 0; j < NL; ++j) {
    const int r = j * RPL + lane / LPR;
    voff[j] = (PAGED ? r % (DEC_TILE / 2) : r) * stride + (((lane % LPR) ^ swz(r)) * 16);
  }
  const unsigned ring = (unsigned)(size_t)(AS_LDS unsigned char*)lds + wave * (2 * R * TB + AS_ROWS * D * 2);
  const unsigned qrow = ring + 2 * R * TB;       // the query rows, behind the ring
  {
    const as_u4 rq = as_rsrc(A.q + (size_t)q0 * A.q_stride + (size_t)kvh * G * D, 0xfffffff0u);
#pragma unroll
    for (int j = 0; j < NQ; ++j) {
      const int r = j * RPL + lane / LPR, t = r / G;
      as_load_lds(rq, r < rows ? ((unsigned)t * (unsigned)A.q_stride + (r - t * G) * D) * 2 + (((lane % LPR) ^ swz(r)) * 16) : 0xfffffff0u,
                  qrow + j * 1024);
    }
  }
  // the tile's loads, or as many that reach nothing: the wait counts stay the same
  auto ask = [&](int kt, unsigned slot, const int (&page)[2]) {
    const int n = min(max(kend - kt, 0), DEC_TILE);
    if constexpr (PAGED) {
      // 16 rows at a time, which a page holds whole; shifts for divisions and an address for half of a tile instead of one
      // for each load: 1500 keys x 20 heads of 64 in one workgroup each 19.4 us with these, 16.4 without, 15.7 off contiguous rows
#pragma unroll
      for (int t = 0; t < 2; ++t) {
        const int at = kt + t * (DEC_TILE / 2);
        const size_t off = ((((size_t)(at >> sh == kt >> sh ? page[0] : page[1]) * A.Hkv + kvh) << sh) + (at & (blk - 1))) * D;
        const unsigned bytes = min(max(n - t * (DEC_TILE / 2), 0), DEC_TILE / 2) * (D * 2);
        const as_u4 rk = as_rsrc(A.kc + off, bytes), rv = as_rsrc(A.vc + off, bytes);
#pragma unroll
        for (int j = t * (NL / 2); j < (t + 1) * (NL / 2); ++j) {
          as_load_lds(rk, voff[j], slot + j * 1024);
          as_load_lds(rv, voff[j], slot + TB + j * 1024);
        }
      }
    } else {
      const size_t off = (kv0 + kt) * (size_t)A.kv_stride + (size_t)kvh * D;
      const unsigned bytes = n ? (n - 1) * stride + D * 2 : 0;
      const as_u4 rk = as_rsrc(A.kc + off, bytes), rv = as_rsrc(A.vc + off, bytes);
#pragma unroll
      for (int j = 0; j < NL; ++j) as_load_lds(rk, voff[j], slot + j * 1024);
#pragma unroll
      for (int j = 0; j < NL; ++j) as_load_lds(rv, voff[j], slot + TB + j * 1024);
    }
  };

  float4v acc[ND];
#pragma unroll
  for (int d = 0; d < ND; ++d) acc[d] = float4v{0.f, 0.f, 0.f, 0.f};
  float m_run = -1e30f, l_run = 0.f;
  ask(kt0, ring, pages[0]);
  if constexpr (R > 1) ask(kt0 + STEP, ring + 2 * TB, pages[1]);
  bf16x8 qf[NS];
  unsigned slot = ring;
  for (int kt = kt0; kt < kend; kt += STEP) {
    int next[2] = {0, 0};                        // wanted behind this tile's work
    if constexpr (PAGED) { next[0] = page_at(kt + R * STEP, 0); next[1] = page_at(kt + R * STEP, 1); }
    as_wait<(R - 1) * 2 * NL>();                 // this tile is here, the next one's loads may be under way
    if (kt == kt0) {
#pragma unroll
      for (int s = 0; s < NS; ++s) qf[s] = *as_lds<bf16x8>(qrow + li * (D * 2) + (((4 * s + fq) ^ swz(li)) * 16));
    }
    float4v st[2] = {float4v{0.f, 0.f, 0.f, 0.f}, float4v{0.f, 0.f, 0.f, 0.f}};
#pragma unroll
    for (int s = 0; s < NS; ++s)
#pragma unroll
      for (int t = 0; t < 2; ++t) {
        const bf16x8 kf = *as_lds<bf16x8>(slot + (16 * t + li) * (D * 2) + (((4 * s + fq) ^ swz(16 * t + li)) * 16));
        st[t] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(kf, qf[s], st[t], 0, 0, 0);
      }
    float mx = -INFINITY;
#pragma unroll
    for (int t = 0; t < 2; ++t)
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        const int key = kt + 16 * t + 4 * fq + j;
        float sv = st[t][j] * A.scale_log2;
        if (key >= kend || (A.causal && key > qpos)) sv = -INFINITY;
        st[t][j] = sv;
        mx = fmaxf(mx, sv);
      }
    mx = fmaxf(mx, __shfl_xor(mx, 16, 64));
    mx = fmaxf(mx, __shfl_xor(mx, 32, 64));
    const float m_new = fmaxf(m_run, mx), alpha = exp2f(m_run - m_new);
    m_run = m_new;
    // Weights as two bf16, 16 bits of mantissa, which the memory's time covers: relative error against 64 bits of
    // 1500 keys 0.00204 with one in runs of 64 keys, 0.00208 in these longer runs (fewer weights are exactly
    // one), 0.00165 with two. The upper one is cut off below the weight, so that the lower one is positive as well:
    // an infinite value stays infinite, where a lower part of zero or below makes it NaN.
    typedef __bf16 b2 __attribute__((ext_vector_type(2)));
    typedef float f2 __attribute__((ext_vector_type(2)));
    bf16x8 ph, pl;
    float ls = 0.f;
#pragma unroll
    for (int t = 0; t < 2; ++t)
#pragma unroll
      for (int j = 0; j < 4; j += 2) {
        const f2 e = {exp2f(st[t][j] - m_new), exp2f(st[t][j + 1] - m_new)};
        const unsigned h0 = __builtin_elementwise_sub_sat(__float_as_uint(e[0]), 1u), h1 = __builtin_elementwise_sub_sat(__float_as_uint(e[1]), 1u);
        const b2 hi = __builtin_bit_cast(b2, __builtin_amdgcn_perm(h1, h0, 0x07060302u));   // the upper halves
        const b2 lo = __builtin_convertvector((f2{e[0] - __uint_as_float(h0 & 0xffff0000u), e[1] - __uint_as_float(h1 & 0xffff0000u)}), b2);
        ls += e[0] + e[1];
        ph[4 * t + j] = hi[0];
        ph[4 * t + j + 1] = hi[1];
        pl[4 * t + j] = lo[0];
        pl[4 * t + j + 1] = lo[1];
      }
    l_run = l_run * alpha + ls;                  // of this lane's keys
#pragma unroll
    for (int d = 0; d < ND; ++d) {
      short8 a8;
#pragma unroll
      for (int t = 0; t < 2; ++t) {
        const int row = 16 * t + 4 * fq + (li >> 2), chunk = 2 * d + ((li & 3) >> 1);
        const v4s_ x = __builtin_amdgcn_ds_read_tr16_b64_v4i16(as_lds<v4s_>(slot + TB + row * (D * 2) + (chunk ^ swz(row)) * 16 + (li & 1) * 8));
#pragma unroll
        for (int j = 0; j < 4; ++j) a8[4 * t + j] = x[j];
      }
#pragma unroll
      for (int j = 0; j < 4; ++j) acc[d][j] *= alpha;
      acc[d] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(*reinterpret_cast<bf16x8*>(&a8), pl, acc[d], 0, 0, 0);
      acc[d] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(*reinterpret_cast<bf16x8*>(&a8), ph, acc[d], 0, 0, 0);
    }
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");   // the slot has been read
    ask(kt + R * STEP, slot, next);
    if constexpr (R > 1) slot = slot == ring ? ring + 2 * TB : ring;
  }
  as_wait<0>();                                  // no load into LDS outlives the loop
  l_run += __shfl_xor(l_run, 16, 64);
  l_run += __shfl_xor(l_run, 32, 64);
  __syncthreads();
  float* so = reinterpret_cast<float*>(lds);             // [wave][row][LD]
  float* sm = so + NW * AS_ROWS * LD;                    // [wave][m, l][row]
  if (li < rows) {
#pragma unroll
    for (int d = 0; d < ND; ++d) *reinterpret_cast<float4v*>(so + (wave * AS_ROWS + li) * LD + 16 * d + 4 * fq) = acc[d];
    if (fq == 0) {
      sm[(2 * wave) * AS_ROWS + li] = m_run;
      sm[(2 * wave + 1) * AS_ROWS + li] = l_run;
    }
  }
  __syncthreads();
  const int nsplit = min(A.num_splits, max(1, (klen + A.split_keys - 1) / A.split_keys));
  const auto ro = __builtin_amdgcn_make_buffer_rsrc(A.part_o, 0, (int)((size_t)A.num_splits * A.total_q * A.Hq * D * 4), 0x00020000);
  const auto rm = __builtin_amdgcn_make_buffer_rsrc(A.part_ml, 0, (int)((size_t)A.num_splits * A.total_q * A.Hq * 2 * 4), 0x00020000);
  auto put = [&](int r, int c, const float4v& o, float l) {
    const int t = r / G;
    const float inv = l > 0.f ? 1.f / l : 0.f;
    *reinterpret_cast<uint2*>(A.out + (size_t)(q0 + t) * A.o_stride + (size_t)(kvh * G + r - t * G) * D + c) =
        make_uint2(pack_bf16x2(o[0] * inv, o[1] * inv), pack_bf16x2(o[2] * inv, o[3] * inv));
  };
  for (int id = tid; id < rows * (D / 4); id += NW * 64) {
    const int r = id / (D / 4), c = id % (D / 4) * 4;
    float ms = sm[r];
#pragma unroll
    for (int w = 1; w < NW; ++w) ms = fmaxf(ms, sm[2 * w * AS_ROWS + r]);
    float l = 0.f;
    float4v o = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int w = 0; w < NW; ++w) {
      const float x = exp2f(sm[2 * w * AS_ROWS + r] - ms);
      l += sm[(2 * w + 1) * AS_ROWS + r] * x;
      const float4v v = *reinterpret_cast<const float4v*>(so + (w * AS_ROWS + r) * LD + c);
#pragma unroll
      for (int j = 0; j < 4; ++j) o[j] += x * v[j];
    }
    if (nsplit == 1) {
      put(r, c, o, l);
    } else {                                             // this split's partial, written through
      const int row = (q0 + r / G) * A.Hq + kvh * G + r % G, at = split * A.total_q * A.Hq + row;
      __builtin_amdgcn_raw_buffer_store_b128(__builtin_bit_cast(u32x4_, o), ro, (at * D + c) * 4, 0, 16);
      if (c == 0) __builtin_amdgcn_raw_buffer_store_b64(__builtin_bit_cast(u32x2_, make_float2(ms, l)), rm, at * 8, 0, 16);
    }
  }
  if (nsplit == 1) return;
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
  int* flag = reinterpret_cast<int*>(lds + NW * AS_ROWS * (LD + 2) * 4);
  __syncthreads();
  if (tid == 0) {
    int* cnt = A.counters + ((size_t)b * A.Hkv + kvh) * TICKET;
    const int t = __hip_atomic_fetch_add(cnt, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    if (t == nsplit - 1) __hip_atomic_store(cnt, 0, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    *flag = t;
  }
  __syncthreads();
  if (*flag != nsplit - 1) return;
  // the last split merges all of them, in order: past the caches, eight partials under way
  constexpr int OB = 8;
  for (int id = tid; id < rows * (D / 4); id += NW * 64) {
    const int r = id / (D / 4), c = id % (D / 4) * 4;
    const int row = (q0 + r / G) * A.Hq + kvh * G + r % G, per = A.total_q * A.Hq;
    float ms = -1e30f, l = 0.f;
    float4v o = {0.f, 0.f, 0.f, 0.f};
    for (int s0 = 0; s0 < nsplit; s0 += OB) {
      float4v v[OB];
      float2 ml[OB];
#pragma unroll
      for (int i = 0; i < OB; ++i) {
        const int at = min(s0 + i, nsplit - 1) * per + row;
        ml[i] = __builtin_bit_cast(float2, __builtin_amdgcn_raw_buffer_load_b64(rm, at * 8, 0, 16));
        v[i] = __builtin_bit_cast(float4v, __builtin_amdgcn_raw_buffer_load_b128(ro, (at * D + c) * 4, 0, 16));
      }
      // All are asked for before the first is waited for: left alone, the compiler moved each load to its use behind
      // the question whether there is such a split, a trip each (2000 keys in 16 splits x 4 kv heads of 64, four
      // sequences: 12.6 us, now 8.9; the form of attn_decode.hip 10.4).
#pragma unroll
      for (int i = 0; i < OB; ++i) asm volatile("" : "+v"(ml[i].x), "+v"(ml[i].y), "+v"(v[i]));
      float mn = ms;
#pragma unroll
      for (int i = 0; i < OB; ++i) mn = fmaxf(mn, ml[i].x);
      const float a = exp2f(ms - mn);
      ms = mn;
      l *= a;
#pragma unroll
      for (int j = 0; j < 4; ++j) o[j] *= a;
#pragma unroll
      for (int i = 0; i < OB; ++i) {
        if (s0 + i >= nsplit) break;
        const float x = exp2f(ml[i].x - ms);
        l += x * ml[i].y;
#pragma unroll
        for (int j = 0; j < 4; ++j) o[j] += x * v[i][j];
      }
    }
    put(r, c, o, l);
  }
}

template <int D, int NW, int R>
static int as_go(const AttnDecArgs& a, int B, hipStream_t st) {
  const dim3 grid(a.num_splits, a.Hkv, B);
  if (a.block_tables) hipLaunchKernelGGL((attn_stream_kernel<D, true, NW, R>), grid, dim3(NW * 64), 0, st, a);
  else hipLaunchKernelGGL((attn_stream_kernel<D, false, NW, R>), grid, dim3(NW * 64), 0, st, a);
  return (int)hipGetLastError();
}

template <int D, int NW>
static int as_launch(const AttnDecArgs& a, int B, hipStream_t st) {
  return a.split_keys <= NW * DEC_TILE ? as_go<D, NW, 1>(a, B, st) : as_go<D, NW, 2>(a, B, st);
}

// Takes the call if the kernel can: true, *err says how the launch went. A workgroup takes f of the
// caller's splits: the f with the least of a compute unit's keys, 5.6 ns each at 64 columns, and its
// further workgroups, 2 us each (their start and their part of the merges). Measured, us by f, 1500 keys x 20
// heads of 64 on contiguous rows in splits of 256: one sequence 7.4, 9.1 (2), 11.0 (3), 15.7 (6); four 11.0, 10.4, 11.8, 16.2;
// eight 19.0, 16.2, 18.5, 17.4; sixteen 34.6, 29.0, 30.1, 32.1; 4000 keys x 8 heads of 128 on pages in splits of 256, eight
// sequences 44, 34 (2), 37 (3), 29 (4), 35 (8), 32 sequences 155, 118, 113, 103, 97 (8), 92 (16).
// Left to attn_decode.hip: more workgroups than their rings fit on the chip (147 KB at 128 columns, one a compute unit; 74
// KB at 64, two), where none takes more than one split, of more than a tile a wave: its 51 KB fit
// three times. Measured there, us in this form and in that: 128 columns, 264 heads x 130 keys 16.8, 12.0, x 600 33.0,
// 27.0, 512 heads x 300 27.6, 21.8, x 1500 79.6, 76.5, 1024 heads x 600 66.9, 59.2; 64 columns, 640 heads x 130 keys 12.2,
// 10.4, x 300 18.1, 16.1. At 64 columns and more heads than three a compute unit both take rounds, and from 512 keys on
// this form is the faster one again (1280 heads x 1500 keys 91, 101). Several splits: 128 columns, 160 heads x 600 keys in three
// 19.1, 17.0, x 1500 in three 32.5, 30.2; 64 columns, 384 heads x 1000 keys in two 27.4, 24.6; of 2203 shapes with one split or
// more seven are slower than there by more than 2 %, two by 5 to 7 (560 heads of 64 x 2500 keys 77.7, 72.3).
bool attn_stream(AttnDecArgs a, int B, int max_q, int D, hipStream_t st, int* err) {
  // 32-bit offsets within a tile's rows and a sequence's queries, 16-byte pieces
  if (a.Hq / a.Hkv * max_q > AS_ROWS || ((size_t)a.q | (size_t)a.kc | (size_t)a.vc) & 15 || a.q_stride % 8 || a.q_stride < 0 ||
      a.q_stride >= 1 << 24 || a.kv_stride < 0 || a.kv_stride >= 1 << 25)
    return false;
  const long long heads = (long long)B * a.Hkv, all = heads * a.num_splits;
  int best = 1;
  double least = 0;
  for (int f = 1; f <= a.num_splits; ++f) {
    const long long n = (heads * ((a.num_splits + f - 1) / f) + 255) / 256;
    const double t = n * f * (double)a.split_keys * (D * 5.6e-3 / 64) + 2.0 * (n - 1);
    if (f == 1 || t < least) { least = t; best = f; }
  }
  if (best == 1 && a.split_keys > 4 * DEC_TILE && all > 256 * (128 / D) && (D == 128 || all <= 768 || a.split_keys <= 512)) return false;
  a.split_keys *= best;
  a.num_splits = (a.num_splits + best - 1) / best;
  *err = D == 64 ? as_launch<64, 4>(a, B, st) : as_launch<128, 4>(a, B, st);
  return true;
}
