// The k = 3 conv1d of an encoder's stem on the software-pipelined tile loop (gemm_pipe.h): rows of
// Y [B * tout, N] = GELU(conv(X) + bias) (+ position rows), X time-major [B * tin, cin], padding 1.
// As a matrix product with k = tap * cin + c, an output row's K entries are the three input rows
// around it one behind the other, so the loader is the projections' with a row step of the
// stride; only where a tap falls off a window's end is a lane's offset put out of the buffer's
// range, and reads zeros. On the burst-loaded tiles of gemm_tile.hip (which keep every other size)
// 1500 x 512 x 1536 ran on 48 workgroups.
#include "gemm_sk.h"
#include "gemm_pipe.h"

struct ConvPipeParams {
  const bf16_t* x; long long ldx;   // [B * tin, cin]
  const bf16_t* w;                  // [N, 3 cin]
  int M, N, cin, tin, tout, stride;
  const float* bias;                // [N] or null
  const bf16_t* pos; int pos_rows;  // [pos_rows, N], row m % pos_rows added after GELU, or null
  bf16_t* y; long long ldy;
  int layout;
};

template <int FN, int FM, int NA, int NB, bool POS>
__global__ __launch_bounds__(256, (gp_per_cu<FN, FM, NA, NB>())) void conv_pipe_kernel(ConvPipeParams p) {
  constexpr int NW = 4, TN = 16 * FN, TM = 16 * FM, BN = 2 * TN, BM = 2 * TM;
  constexpr int IA = BN / 8 / NW, IB = BM / 8 / NW, XRING = NA * BN * 128;
  __shared__ __attribute__((aligned(1024))) unsigned char lds[gp_lds_bytes<FN, FM, NA, NB>()];
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int wn = wave & 1, wm = wave >> 1, fq = lane >> 4;
  const int M = p.M, N = p.N, K = 3 * p.cin, nt = K / GP_BK;
  const int mblocks = (M + BM - 1) / BM, id = xcd_remap(blockIdx.x, gridDim.x);
  const int mb = id % mblocks, nb = id / mblocks, m0 = mb * BM, n0 = nb * BN;
  const bf16_t* wp = p.w + (size_t)n0 * K;
  const unsigned wbytes = (unsigned)BN * K * 2;
  // offsets from the first input row that the tile's rows read
  const int b0 = m0 / p.tout, first = b0 * p.tin + max((m0 - b0 * p.tout) * p.stride - 1, 0);
  const bf16_t* xp = p.x + (size_t)first * p.ldx;
  const long long xleft = ((long long)(M / p.tout) * p.tin - first - 1) * p.ldx + p.cin;
  const unsigned xbytes = (unsigned)min(xleft * 2, (long long)0x7fffffff);
  unsigned woff[IA], xoff[IB], lo[IB], hi[IB];
#pragma unroll
  for (int i = 0; i < IA; ++i) {
    const int r = 8 * (wave * IA + i) + (lane >> 3), c = (lane & 7) ^ ((r >> 1) & 7);
    woff[i] = ((unsigned)r * (unsigned)K + c * 8) * 2;
  }
#pragma unroll
  for (int i = 0; i < IB; ++i) {
    const int r = 8 * (wave * IB + i) + (lane >> 3), c = (lane & 7) ^ ((r >> 1) & 7);
    const int m = m0 + r, b = m / p.tout, t = m - b * p.tout;
    // (tap 0 of a window's first row is off: its offset may be below zero and is not used)
    xoff[i] = (unsigned)((b * p.tin + t * p.stride - 1 - first) * (int)p.ldx + c * 8) * 2;
    lo[i] = t == 0 ? ~0u : 0u;
    hi[i] = t * p.stride + 1 >= p.tin ? ~0u : 0u;
    if (m >= M) xoff[i] = lo[i] = hi[i] = ~0u;
  }
  auto load_w = [&](int i, int slot, int t) {
    const bool on = t < nt;
    gp_load_lds(wp, on ? wbytes : 0u, lds + slot * (BN * 128) + (wave * IA + i) * 1024, woff[i], on ? t * (GP_BK * 2) : 0);
  };
  auto load_x = [&](int i, int slot, int t) {
    const bool on = t < nt;
    const int k = t * GP_BK, tap = (k >= p.cin) + (k >= 2 * p.cin);
    const unsigned off = tap == 1 ? 0u : tap == 0 ? lo[i] : hi[i];
    // the tap's row is part of the lane's offset: what is compared with the range must not wrap
    const unsigned at = (xoff[i] + (unsigned)(tap * (int)p.ldx) * 2) | off;
    gp_load_lds(xp, on ? xbytes : 0u, lds + XRING + slot * (BM * 128) + (wave * IB + i) * 1024,
                xoff[i] == ~0u ? ~0u : at, on ? (k - tap * p.cin) * 2 : 0);
  };
  const int mw = m0 + wm * TM, nw = n0 + wn * TN;
  float4v bv[FN];
#pragma unroll
  for (int i = 0; i < FN; ++i)
    bv[i] = p.bias ? *reinterpret_cast<const float4v*>(p.bias + nw + 16 * i + 4 * fq) : float4v{0.f, 0.f, 0.f, 0.f};
  using R = GpRows<FN, FM>;
  R old;
  if constexpr (POS) {
#pragma unroll
    for (int k = 0; k < R::CH; ++k) {
      const int c = lane + 64 * k, m = min(mw + c / R::CPR, M - 1);
      old.v[k] = *reinterpret_cast<const u32x4*>(p.pos + (size_t)(m % p.pos_rows) * N + nw + (c % R::CPR) * 8);
    }
  }
  __builtin_amdgcn_sched_barrier(0);

  float4v acc[FN][FM];
  gp_loop<FN, FM, NA, NB>(acc, lds, nt, wn, wm, lane, load_w, load_x);

  constexpr int WAVE_LDS = TM * (TN * 2 + 16);
  static_assert(WAVE_LDS * NW <= XRING + NB * BM * 128, "the epilogue's rows must fit the rings");
  __syncthreads();
  unsigned char* my = lds + wave * WAVE_LDS;
  if constexpr (POS) old.to_lds(my, lane);
  gp_store<FN, FM, POS>(my, p.y + (size_t)mw * p.ldy + nw, p.ldy, M - mw, TN, lane, [&](int i, int j, float* o) {
    float g[4];
#pragma unroll
    for (int r = 0; r < 4; ++r) g[r] = acc[i][j][r] + bv[i][r];
    sk_gelu4(g);
#pragma unroll
    for (int r = 0; r < 4; ++r) o[r] = POS ? o[r] + g[r] : g[r];
  });
}

template <int FN, int FM, int NA, int NB> static int cp_launch(const ConvPipeParams& p, hipStream_t st) {
  constexpr int BN = 32 * FN, BM = 32 * FM;
  // 32-bit buffer offsets of a tile's input rows (it may reach over several windows' ends) and of W
  if (p.N % BN || (long long)(BM * p.stride + 2 * (BM / p.tout + 2)) * p.ldx * 2 >= 0x7fffffffll ||
      (long long)BN * p.cin * 6 >= 0x7fffffffll)
    return (int)hipErrorInvalidValue;
  const dim3 grid((p.M + BM - 1) / BM * (p.N / BN));
  if (p.pos)
    hipLaunchKernelGGL((conv_pipe_kernel<FN, FM, NA, NB, true>), grid, dim3(256), 0, st, p);
  else
    hipLaunchKernelGGL((conv_pipe_kernel<FN, FM, NA, NB, false>), grid, dim3(256), 0, st, p);
  return (int)hipGetLastError();
}

// layout: numbers of the pipelined projections' tiles (64 x 64, 128 x 64, 128 x 128, 256 x 128)
extern "C" int loqa_conv_pipe(const ConvPipeParams* p, hipStream_t st) {
  if (!p || !p->x || !p->w || !p->y || p->M <= 0 || p->cin <= 0 || p->cin % GP_BK || p->stride < 1 || p->tin < 1 ||
      p->tout != (p->tin - 1) / p->stride + 1 || p->M % p->tout || p->ldx < p->cin || p->ldx % 8 || p->ldy % 8 ||
      (p->pos && p->pos_rows < 1) || (((size_t)p->x | (size_t)p->w | (size_t)p->y | (size_t)p->pos) & 15))
    return (int)hipErrorInvalidValue;
  switch (p->layout) {
    case 11: return cp_launch<2, 2, 5, 5>(*p, st);
    case 19: return cp_launch<4, 2, 4, 4>(*p, st);
    case 20: return cp_launch<4, 4, 5, 5>(*p, st);
    case 15: return cp_launch<8, 4, 3, 3>(*p, st);
    default: return (int)hipErrorInvalidValue;
  }
}
