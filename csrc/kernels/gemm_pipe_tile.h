// The kernel behind gemm_pipe.hip, for its translation units (with K chunks or whole tiles, with
// workgroups that touch later weights or without: they compile side by side).
#pragma once
#include <type_traits>
#include "gemm_sk.h"
#include "gemm_pipe.h"


#define GP_GROUP 4

template <bool AHEAD> using GpArgs = std::conditional_t<AHEAD, GemmSkCall, GemmSkParams>;

// The K chunks of a tile are summed up by all of its workgroups, each its share of the tile: the last to
// arrive alone reads 27 KB/us of partials (what a compute unit has in flight over the trip to memory),
// 14.5 us for four chunks of 128 x 192. Partials are written through and read past the caches (sc1), so
// no cache is written back or invalidated for them, and the tiles' words are a cache line apart: in one
// line they cost 5 us more. Up to SK_KEEP chunks a workgroup's own part of its own share stays in LDS: half of
// the traffic at two (1500 x 1280 x 5120 in 128 x 128 31.6 -> 29.4 us); from five on it is 3 % slower. A workgroup
// that has published its partial waits for the others for SK_POLLS looks at the word (some 30 us), no longer:
// if one of them starts late it gives its share up to the last to arrive and leaves, so a launch always
// drains whatever else holds the compute units. The word: arrivals in bits 0 - 15, given-up shares in
// 16 - 23, workgroups done in 24 - 31 for up to SK_SHARE chunks; more chunks than that are summed up by
// the last. In four chunks of 128 x 192, cold weights: 320 x 4096 x 4096 32.6 -> 23.4 us, 320 x 4096 x 14336
// 62.2 -> 51.1.
#define SK_KEEP 4
#define SK_SHARE 8
#define SK_POLLS 48
#define SK_SC1 16                     // buffer cache policy: device scope

template <int NW, int FN, int FM>
__device__ __forceinline__ __amdgpu_buffer_rsrc_t sk_part(const GemmSkParams& p, int tile, int c) {
  constexpr int TILE = NW * FN * FM * 256;             // floats of a partial
  return __builtin_amdgcn_make_buffer_rsrc(p.ws + ((size_t)tile * p.S + c) * TILE, 0, TILE * 4, 0x00020000);
}

// The shares of the tile that this workgroup sums up, a bit each. late() publishes what it has kept back. hurry: 0, or
// SK_POLLS where a test has every workgroup but the last give its share up.
template <typename Late>
__device__ __forceinline__ unsigned sk_shares(int* word, int S, int s, int hurry, int* flag, Late&& late) {
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");   // written through: visible when acknowledged
  __syncthreads();
  if (threadIdx.x == 0) {
    const unsigned old = __hip_atomic_fetch_add(word, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    unsigned mine = 0;
    if (S > SK_SHARE) {
      if ((int)old == S - 1) mine = (1u << SK_SHARE) - 1;
    } else if ((int)(old & 0xffff) == S - 1) {
      mine = 1u << s | (old >> 16 & 0xff);
    } else {
      for (int k = hurry; k < SK_POLLS && !mine; ++k)
        if ((__hip_atomic_load(word, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) & 0xffff) == S) mine = 1u << s;
        else __builtin_amdgcn_s_sleep(4);
    }
    *flag = (int)mine;
  }
  __syncthreads();
  const unsigned mine = (unsigned)__builtin_amdgcn_readfirstlane(*flag);
  if (mine || S > SK_SHARE) return mine;
  // the last to arrive takes the share, unless it has been here meanwhile
  late();
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
  __syncthreads();
  if (threadIdx.x == 0)
    *flag = (__hip_atomic_fetch_or(word, 0x10000 << s, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) & 0xffff) == S ? 1 << s : 0;
  __syncthreads();
  return (unsigned)__builtin_amdgcn_readfirstlane(*flag);
}

// Sums up units u0 .. u1 of a wave's corner (16 rows by 16 output features each, row blocks slowest) over
// the S partials, in chunk order whoever does it, and finishes them. kept: chunk s of these units in LDS,
// or null. UB units and CB chunks are asked for at a time: 32 loads in flight, the accumulators' registers
// being free. nw: the wave's first output feature.
template <int EPI, int FN, int FM, int NW, int UB, int CB>
__device__ __forceinline__ void sk_units(const GemmSkParams& p, const unsigned char* kept, int tile, int s, int u0, int u1, int wave,
                                         int lane, int mw, int nw) {
  constexpr bool PAIR = EPI == SK_SWIGLU;
  constexpr int G = PAIR ? 2 : 1, FO = FN / G, UG = UB / G;
  const int S = p.S, fr = lane & 15, fq = lane >> 4;
  for (int u = u0; u < u1; u += UG) {
    float4v sum[UG][G];
    uint2 old[UG];
    float4v bv[UG];
    bf16_t* at[UG];
#pragma unroll
    for (int b = 0; b < UG; ++b) {
      const int v = min(u + b, u1 - 1), j = v / FO, i = v % FO;
      at[b] = reinterpret_cast<bf16_t*>(p.y) + (size_t)min(mw + 16 * j + fr, p.M - 1) * p.ldy + nw + 16 * i + 4 * fq;
      if constexpr (EPI == SK_RESID) old[b] = *reinterpret_cast<const uint2*>(at[b]);
      if constexpr (!PAIR)
        bv[b] = p.bias ? *reinterpret_cast<const float4v*>(p.bias + nw + 16 * i + 4 * fq) : float4v{0.f, 0.f, 0.f, 0.f};
    }
    for (int c0 = 0; c0 < S; c0 += CB) {
      float4v v[CB][UG][G];
#pragma unroll
      for (int c = 0; c < CB; ++c)
        if (c0 + c < S) {
          const bool here = kept && c0 + c == s;
          const __amdgpu_buffer_rsrc_t part = sk_part<NW, FN, FM>(p, tile, c0 + c);
#pragma unroll
          for (int b = 0; b < UG; ++b) {
            const int w = min(u + b, u1 - 1), j = w / FO, i = w % FO;
#pragma unroll
            for (int g = 0; g < G; ++g)
              if (here) v[c][b][g] = *reinterpret_cast<const float4v*>(kept + ((w - u0) * G + g) * 1024 + lane * 16);
              else v[c][b][g] = __builtin_bit_cast(float4v, __builtin_amdgcn_raw_buffer_load_b128(
                  part, lane * 16, ((wave * FN + i + g * FO) * FM + j) * 1024, SK_SC1));
          }
        }
#pragma unroll
      for (int c = 0; c < CB; ++c)
        if (c0 + c < S) {
#pragma unroll
          for (int b = 0; b < UG; ++b)
#pragma unroll
            for (int g = 0; g < G; ++g) sum[b][g] = c0 + c == 0 ? v[c][b][g] : sum[b][g] + v[c][b][g];
        }
    }
#pragma unroll
    for (int b = 0; b < UG; ++b) {
      const int j = min(u + b, u1 - 1) / FO;
      float o[4];
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        if constexpr (PAIR) o[r] = sk_swiglu(sum[b][0][r], sum[b][G - 1][r]);
        else o[r] = sum[b][0][r] + bv[b][r];
      }
      if constexpr (EPI == SK_RESID) {
        o[0] = bf2f(old[b].x & 0xffff) + o[0]; o[1] = bf2f(old[b].x >> 16) + o[1];
        o[2] = bf2f(old[b].y & 0xffff) + o[2]; o[3] = bf2f(old[b].y >> 16) + o[3];
      }
      if constexpr (EPI == SK_GELU) sk_gelu4(o);
      if (u + b < u1 && mw + 16 * j + fr < p.M)
        *reinterpret_cast<uint2*>(at[b]) = make_uint2(pack_bf16x2(o[0], o[1]), pack_bf16x2(o[2], o[3]));
    }
  }
}

// A K chunk's way out: its partial, then this workgroup's shares of the finished tile. lds: BYTES that
// nobody reads any more, the last 16 for the flag.
template <int EPI, int FN, int FM, int NW, int BYTES>
__device__ __forceinline__ void sk_finish(const GemmSkParams& p, float4v (&acc)[FN][FM], int tile, int s, int wave, int lane,
                                          int mw, int nw, unsigned char* lds) {
  const int S = p.S, n = min(S, SK_SHARE);
  constexpr int G = EPI == SK_SWIGLU ? 2 : 1, FO = FN / G, UNITS = FM * FO;
  constexpr int KEEP = (UNITS + 1) / 2 * G * 1024;     // bytes of a wave's largest share, of two chunks
  static_assert(NW * KEEP + 16 <= BYTES, "the kept shares must fit the rings");
  const int u0 = s * UNITS / n, u1 = S > SK_KEEP ? u0 : (s + 1) * UNITS / n;
  unsigned char* kept = lds + wave * KEEP;
  const __amdgpu_buffer_rsrc_t part = sk_part<NW, FN, FM>(p, tile, s);
#pragma unroll
  for (int i = 0; i < FN; ++i) {
#pragma unroll
    for (int j = 0; j < FM; ++j) {
      const int u = j * FO + i % FO;
      if (u >= u0 && u < u1) *reinterpret_cast<float4v*>(kept + ((u - u0) * G + i / FO) * 1024 + lane * 16) = acc[i][j];
      else __builtin_amdgcn_raw_buffer_store_b128(__builtin_bit_cast(u32x4, acc[i][j]), part, lane * 16,
                                                  ((wave * FN + i) * FM + j) * 1024, SK_SC1);
    }
    __builtin_amdgcn_sched_barrier(0);
  }
  int* word = p.counters + tile * TICKET;
  const unsigned mine = sk_shares(word, S, s, p.hurry, reinterpret_cast<int*>(lds + BYTES - 16), [&]() {
    for (int u = u0; u < u1; ++u)
#pragma unroll
      for (int g = 0; g < G; ++g)
        __builtin_amdgcn_raw_buffer_store_b128(*reinterpret_cast<const u32x4*>(kept + ((u - u0) * G + g) * 1024 + lane * 16), part,
                                               lane * 16, ((wave * FN + u % FO + g * FO) * FM + u / FO) * 1024, SK_SC1);
  });
  // leaving: the last one puts the word back to zero; its answer travels with the loads below
  int before = 0;
  if (threadIdx.x == 0 && S <= SK_SHARE) before = __hip_atomic_fetch_add(word, 1 << 24, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  for (unsigned left = mine; left; left &= left - 1) {
    const int t = __builtin_ctz(left), a = t * UNITS / n, b = (t + 1) * UNITS / n;
    if (S <= SK_KEEP) sk_units<EPI, FN, FM, NW, 8, 4>(p, t == s ? kept : nullptr, tile, s, a, b, wave, lane, mw, nw);
    else sk_units<EPI, FN, FM, NW, 4, 8>(p, nullptr, tile, s, a, b, wave, lane, mw, nw);
  }
  if (threadIdx.x == 0 && (S <= SK_SHARE ? before >> 24 == S - 1 : mine != 0))
    __hip_atomic_store(word, 0, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

// SPLIT: the K chunks of a tile in workgroups of their own (p.S of them)
template <int FN, int FM, int NA, int NB, int EPI, bool AHEAD, bool SPLIT>
__global__ __launch_bounds__(256, (gp_per_cu<FN, FM, NA, NB>())) void gemm_pipe_kernel(GpArgs<AHEAD> p) {
  constexpr int NW = 4;
  constexpr int TN = 16 * FN, TM = 16 * FM;
  constexpr int BN = 2 * TN, BM = 2 * TM;
  constexpr int IA = BN / 8 / NW, IB = BM / 8 / NW;   // 1 KB direct-to-LDS loads per wave and stage
  static_assert(IA * 8 * NW == BN && IB * 8 * NW == BM, "rows must split evenly over the waves");
  constexpr int XRING = NA * BN * 128;                // where the ring of X stages starts
  __shared__ __attribute__((aligned(1024))) unsigned char lds[gp_lds_bytes<FN, FM, NA, NB>()];

  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int wn = wave & 1, wm = wave >> 1;
  const int M = p.M, N = p.N, S = SPLIT ? p.S : 1;
  const int mblocks = (M + BM - 1) / BM, nblocks = N / BN;
  int tiles = gridDim.x;
  if constexpr (AHEAD) {
    tiles -= p.ahead_wgs;
    if ((int)blockIdx.x >= tiles) {
      const int at = (blockIdx.x - tiles) * NW + wave, n = p.ahead_wgs * NW;
      gp_touch(p.ahead[0], p.ahead_bytes[0], lds + wave * 1024, at, n, lane);
      gp_touch(p.ahead[1], p.ahead_bytes[1], lds + wave * 1024, at, n, lane);
      gp_wait_vm<0>();
      return;
    }
  }
  const int id = xcd_remap(blockIdx.x, tiles);
  const int s = id % S, tile = id / S;
  const int per = GP_GROUP * nblocks, grp = tile / per, in = tile - grp * per;
  const int gm = min(GP_GROUP, mblocks - grp * GP_GROUP);
  const int mb = grp * GP_GROUP + in % gm, nb = in / gm;
  const int KT = p.K / SK_BK;
  const int kt0 = (int)(((long long)s * KT) / S), kt1 = (int)(((long long)(s + 1) * KT) / S);
  const int nt = kt1 - kt0;
  const int m0 = mb * BM, n0 = nb * BN;
  // Buffer addressing: 32-bit offsets from the tile's own corner, rows past M and stages
  // past the K chunk read as zeros without touching memory, so the loop has no tail.
  const int xrows = min(BM, M - m0);
  const bf16_t* xp = reinterpret_cast<const bf16_t*>(p.x) + (size_t)m0 * p.ldx + (size_t)kt0 * SK_BK;
  const bf16_t* wp = reinterpret_cast<const bf16_t*>(p.w) +
                     (size_t)(EPI == SK_SWIGLU ? n0 >> 1 : n0) * p.K + (size_t)kt0 * SK_BK;
  const unsigned xbytes = (unsigned)((size_t)(xrows - 1) * p.ldx + (size_t)nt * SK_BK) * 2;
  const unsigned wlast = EPI == SK_SWIGLU ? (N >> 1) + BN / 2 - 1 : BN - 1;
  const unsigned wbytes = (unsigned)((size_t)wlast * p.K + (size_t)nt * SK_BK) * 2;
  // lane l of a load brings chunk c of row 8 k + l / 8
  unsigned woff[IA], xoff[IB];
#pragma unroll
  for (int i = 0; i < IA; ++i) {
    const int r = 8 * (wave * IA + i) + (lane >> 3), c = (lane & 7) ^ ((r >> 1) & 7);
    int row = r;
    if constexpr (EPI == SK_SWIGLU) {
      const int blk = r / TN, rr = r - blk * TN;
      const int f = blk * (TN / 2) + (rr % (TN / 2));
      row = rr < TN / 2 ? f : (N >> 1) + f;
    }
    woff[i] = ((unsigned)row * (unsigned)p.K + c * 8) * 2;
  }
#pragma unroll
  for (int i = 0; i < IB; ++i) {
    const int r = 8 * (wave * IB + i) + (lane >> 3), c = (lane & 7) ^ ((r >> 1) & 7);
    xoff[i] = r < xrows ? ((unsigned)r * (unsigned)p.ldx + c * 8) * 2 : 0xfffffff0u;
  }
  // stages past the chunk: an empty range, so the wait counts stay the same without traffic
  auto load_w = [&](int i, int slot, int t) {
    const bool on = t < nt;
    gp_load_lds(wp, on ? wbytes : 0u, lds + slot * (BN * 128) + (wave * IA + i) * 1024, woff[i],
                on ? t * (SK_BK * 2) : 0);
  };
  auto load_x = [&](int i, int slot, int t) {
    const bool on = t < nt;
    gp_load_lds(xp, on ? xbytes : 0u, lds + XRING + slot * (BM * 128) + (wave * IB + i) * 1024, xoff[i],
                on ? t * (SK_BK * 2) : 0);
  };

  // What the epilogue adds is asked for before the loop: a trip to memory behind it took 1 to 2 us
  // of a launch. Bias up to 32 fragments a wave, residual rows up to 24: larger
  // tiles have no registers left.
  const int mw = m0 + wm * TM, nw = n0 + wn * TN, fq = lane >> 4;
  bf16_t* Y = reinterpret_cast<bf16_t*>(p.y) + (size_t)mw * p.ldy;
  float4v bv[FN];
  auto bias = [&]() {
#pragma unroll
    for (int i = 0; i < FN; ++i)
      bv[i] = p.bias ? *reinterpret_cast<const float4v*>(p.bias + nw + 16 * i + 4 * fq) : float4v{0.f, 0.f, 0.f, 0.f};
  };
  constexpr bool BIAS = EPI != SK_SWIGLU && FN * FM <= 32 && !SPLIT, ROWS = EPI == SK_RESID && FN * FM <= 24 && !SPLIT;
  GpRows<FN, FM> old;
  if constexpr (BIAS) bias();
  if constexpr (ROWS) old.load(Y + nw, p.ldy, M - mw, TN, lane);
  __builtin_amdgcn_sched_barrier(0);

  float4v acc[FN][FM];
  gp_loop<FN, FM, NA, NB>(acc, lds, nt, wn, wm, lane, load_w, load_x);

  if constexpr (SPLIT) {
    __syncthreads();           // the rings are free
    sk_finish<EPI, FN, FM, NW, gp_lds_bytes<FN, FM, NA, NB>()>(p, acc, tile, s, wave, lane, mw,
                                                               EPI == SK_SWIGLU ? (n0 >> 1) + wn * (TN / 2) : nw, lds);
    return;
  }
  // every wave has read its last fragments, every load has landed: the rings are free
  constexpr int WAVE_LDS = TM * (TN * 2 + 16);
  static_assert(WAVE_LDS * NW <= XRING + NB * BM * 128, "the epilogue's rows must fit the rings");
  __syncthreads();
  unsigned char* my = lds + wave * WAVE_LDS;
  if constexpr (EPI == SK_SWIGLU) {
    gp_store<FN / 2, FM, false>(my, Y + (n0 >> 1) + wn * (TN / 2), p.ldy, M - mw, TN / 2, lane, [&](int i, int j, float* o) {
#pragma unroll
      for (int r = 0; r < 4; ++r) o[r] = sk_swiglu(acc[i][j][r], acc[i + FN / 2][j][r]);
    });
  } else {
    if constexpr (!BIAS) bias();
    if constexpr (EPI == SK_RESID) {
      if constexpr (!ROWS) old.load(Y + nw, p.ldy, M - mw, TN, lane);
      old.to_lds(my, lane);
    }
    gp_store<FN, FM, EPI == SK_RESID>(my, Y + nw, p.ldy, M - mw, TN, lane, [&](int i, int j, float* o) {
#pragma unroll
      for (int r = 0; r < 4; ++r) o[r] = EPI == SK_RESID ? o[r] + (acc[i][j][r] + bv[i][r]) : acc[i][j][r] + bv[i][r];
      if constexpr (EPI == SK_GELU) sk_gelu4(o);
    });
  }
}

template <int FN, int FM, int NA, int NB, bool AHEAD, bool SPLIT>
static int gp_launch(const GemmSkCall& p, hipStream_t st) {
  constexpr int BN = 32 * FN, BM = 32 * FM;
  if (p.N % BN || p.K % SK_BK || p.S > p.K / SK_BK) return (int)hipErrorInvalidValue;
  // 32-bit buffer offsets: a tile's rows of X, and all of W (SwiGLU: its other half)
  if ((long long)BM * p.ldx * 2 >= 0x7fffffffll || (long long)p.N * p.K * 2 >= 0xfffffff0ll || p.ldx < p.K)
    return (int)hipErrorInvalidValue;
  // whole 16-byte pieces of the output rows
  if (p.ldy % 8 || ((size_t)p.y & 15) || ((size_t)p.x & 15) || ((size_t)p.w & 15)) return (int)hipErrorInvalidValue;
  for (int i = 0; i < 2; ++i)
    if (p.ahead_wgs < 0 || p.ahead_bytes[i] < 0 || p.ahead_bytes[i] > 0x7fffffff || (p.ahead_bytes[i] && !p.ahead[i]))
      return (int)hipErrorInvalidValue;
  const long long grid = (long long)((p.M + BM - 1) / BM) * (p.N / BN) * p.S + p.ahead_wgs;
  if (grid > 0x7fffffff) return (int)hipErrorInvalidValue;
  // GELU costs a wave 20 vector instructions a value, 10 us at 256 x 256, with the matrix cores idle: from
  // more tiles on than compute units, two stages of W and X instead of three fit two workgroups of 128
  // x 192 on one, whose products run beside the other's epilogue (9000 x 2048 x 512 39.7 -> 33.0 us, 12000 x
  // 3072 x 768 79.4 -> 70.5, 9000 x 5120 x 1280 129.3 -> 126.7, always against the best of the other tiles;
  // without GELU 15 to 30 % slower than those)
  if constexpr (FN == 4 && FM == 6 && NA == 3 && !AHEAD && !SPLIT)
    if (p.act == 1 && grid > 256) return gp_launch<FN, FM, 2, 2, AHEAD, SPLIT>(p, st);
#define GO(EPI) hipLaunchKernelGGL((gemm_pipe_kernel<FN, FM, NA, NB, EPI, AHEAD, SPLIT>), dim3(grid), dim3(256), 0, st, static_cast<const GpArgs<AHEAD>&>(p))
  if constexpr (FN == 4 && FM == 6 && NA == 2) GO(SK_GELU);
  else switch (p.epi) {
    case SK_SWIGLU: GO(SK_SWIGLU); break;
    case SK_RESID: GO(SK_RESID); break;
    default:
      if (p.act == 1) GO(SK_GELU); else GO(SK_BF16);
  }
#undef GO
  return (int)hipGetLastError();
}

// (features x rows), stages of W and X; the smaller tiles spend the LDS on deeper rings, as
// what they wait for is the first touch of cold weights
template <bool AHEAD, bool SPLIT> static int gp_layout(const GemmSkCall& p, int layout, hipStream_t st) {
  switch (layout) {
    case -1: return gp_launch<2, 2, 5, 5, AHEAD, SPLIT>(p, st);  // 64 x 64
    case 0: return gp_launch<8, 8, 3, 2, AHEAD, SPLIT>(p, st);   // 256 x 256
    case 1: return gp_launch<8, 6, 3, 2, AHEAD, SPLIT>(p, st);   // 256 x 192
    case 2: return gp_launch<6, 8, 3, 2, AHEAD, SPLIT>(p, st);   // 192 x 256
    case 3: return gp_launch<8, 4, 3, 3, AHEAD, SPLIT>(p, st);   // 256 x 128
    case 4: return gp_launch<4, 8, 3, 3, AHEAD, SPLIT>(p, st);   // 128 x 256
    case 5: return gp_launch<4, 6, 3, 3, AHEAD, SPLIT>(p, st);   // 128 x 192
    case 6: return gp_launch<6, 6, 3, 3, AHEAD, SPLIT>(p, st);   // 192 x 192
    case 7: return gp_launch<4, 2, 4, 4, AHEAD, SPLIT>(p, st);   // 128 x 64
    case 8: return gp_launch<4, 4, 5, 5, AHEAD, SPLIT>(p, st);   // 128 x 128
    case 9: return gp_launch<8, 5, 3, 3, AHEAD, SPLIT>(p, st);   // 256 x 160
    case 10: return gp_launch<4, 5, 3, 3, AHEAD, SPLIT>(p, st);  // 128 x 160
    default: return (int)hipErrorInvalidValue;
  }
}
