// The kernel behind gemm_pipe.hip, for its two translation units (one with workgroups that touch
// later weights, one without: they compile side by side).
#pragma once
#include <type_traits>
#include "gemm_sk.h"
#include "gemm_pipe.h"


#define GP_GROUP 4

template <bool AHEAD> using GpArgs = std::conditional_t<AHEAD, GemmSkCall, GemmSkParams>;

template <int FN, int FM, int NA, int NB, int EPI, bool AHEAD>
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
  const int M = p.M, N = p.N, S = p.S;
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
  constexpr bool BIAS = EPI != SK_SWIGLU && FN * FM <= 32, ROWS = EPI == SK_RESID && FN * FM <= 24;
  GpRows<FN, FM> old;
  if constexpr (BIAS) bias();
  if constexpr (ROWS) old.load(Y + nw, p.ldy, M - mw, TN, lane);
  __builtin_amdgcn_sched_barrier(0);

  float4v acc[FN][FM];
  gp_loop<FN, FM, NA, NB>(acc, lds, nt, wn, wm, lane, load_w, load_x);

  if (S > 1 && !sk_reduce<NW, FN, FM>(p, acc, tile, s, wave, lane, reinterpret_cast<int*>(lds))) return;
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

template <int FN, int FM, int NA, int NB, bool AHEAD>
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
#define GO(EPI) hipLaunchKernelGGL((gemm_pipe_kernel<FN, FM, NA, NB, EPI, AHEAD>), dim3(grid), dim3(256), 0, st, static_cast<const GpArgs<AHEAD>&>(p))
  switch (p.epi) {
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
template <bool AHEAD> static int gp_layout(const GemmSkCall& p, int layout, hipStream_t st) {
  switch (layout) {
    case 0: return gp_launch<8, 8, 3, 2, AHEAD>(p, st);   // 256 x 256
    case 1: return gp_launch<8, 6, 3, 2, AHEAD>(p, st);   // 256 x 192
    case 2: return gp_launch<6, 8, 3, 2, AHEAD>(p, st);   // 192 x 256
    case 3: return gp_launch<8, 4, 3, 3, AHEAD>(p, st);   // 256 x 128
    case 4: return gp_launch<4, 8, 3, 3, AHEAD>(p, st);   // 128 x 256
    case 5: return gp_launch<4, 6, 3, 3, AHEAD>(p, st);   // 128 x 192
    case 6: return gp_launch<6, 6, 3, 3, AHEAD>(p, st);   // 192 x 192
    case 7: return gp_launch<4, 2, 4, 4, AHEAD>(p, st);   // 128 x 64
    case 8: return gp_launch<4, 4, 5, 5, AHEAD>(p, st);   // 128 x 128
    default: return (int)hipErrorInvalidValue;
  }
}
