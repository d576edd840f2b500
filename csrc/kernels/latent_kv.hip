// Per-head keys and values of a prompt pass from latent cache rows: [k | v] = c W^T on the
// software-pipelined tile loop (gemm_pipe.h), the rows c straight from their pages (a lane's offset
// into the cache is all that a page table changes), the rotary key part copied beside every head's
// keys on the way out. One launch where a gather, two products and a fill of the rotary part
// passed the latents and the keys through memory twice: 2048 rows of 16 heads (192 / 128, rank 512)
// 39 us then, 20 now; a layer of 5 x 64 rows, where the host's calls count, 97 and 50.
#include "seqmix.h"
#include "gemm_pipe.h"

#define LK_MAX_ROT 64              // rotary entries of a row

struct LatentKvParams {
  const bf16_t* pages; long long page_bytes; int blk, W;   // rows of W = R + Dr entries
  const int* bt; int max_blocks; const int* cu_k; const int* ctx; int B, total;
  const bf16_t* w;                 // [H DK + H DV, R]: rows of keys (zero from D of each head on), then values
  int R, NK, NV, DK, D, Dr;        // NK = H DK, NV = H DV
  bf16_t* k; bf16_t* v;            // [total, NK], [total, NV]
  int layout;
};

template <int FN, int FM, int NA, int NB>
__global__ __launch_bounds__(256, (gp_per_cu<FN, FM, NA, NB>())) void latent_kv_kernel(LatentKvParams p) {
  constexpr int NW = 4, TN = 16 * FN, TM = 16 * FM, BN = 2 * TN, BM = 2 * TM;
  constexpr int IA = BN / 8 / NW, IB = BM / 8 / NW, XRING = NA * BN * 128;
  // (one array: beside a second one the compiler waits for every direct-to-LDS load at each
  // fragment's read, 35 us instead of 17)
  __shared__ __attribute__((aligned(1024))) unsigned char lds[gp_lds_bytes<FN, FM, NA, NB>() + BM * 4];
  unsigned* rows = reinterpret_cast<unsigned*>(lds + gp_lds_bytes<FN, FM, NA, NB>());   // cache row of each of the tile's rows
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int wn = wave & 1, wm = wave >> 1, fr = lane & 15, fq = lane >> 4;
  const int mblocks = (p.total + BM - 1) / BM, id = xcd_remap(blockIdx.x, gridDim.x);
  const int mb = id % mblocks, nb = id / mblocks, m0 = mb * BM, n0 = nb * BN;
  const int xrows = min(BM, p.total - m0), nt = p.R / GP_BK;
  if ((int)threadIdx.x < BM) {
    const int j = m0 + min((int)threadIdx.x, xrows - 1);
    int b = 0, to = p.B - 1;                                // the last sequence that starts at j or before
    while (b < to) {
      const int mid = (b + to + 1) / 2;
      if (p.cu_k[mid] <= j) b = mid; else to = mid - 1;
    }
    const int jp = p.ctx[b] - p.cu_k[b + 1] + j;            // position in its sequence
    rows[threadIdx.x] = (unsigned)p.bt[(size_t)b * p.max_blocks + jp / p.blk] * p.blk + jp % p.blk;
  }
  __syncthreads();
  const bf16_t* wp = p.w + (size_t)n0 * p.R;
  const unsigned wbytes = (unsigned)BN * p.R * 2;
  unsigned woff[IA], xoff[IB];
#pragma unroll
  for (int i = 0; i < IA; ++i) {
    const int r = 8 * (wave * IA + i) + (lane >> 3), c = (lane & 7) ^ ((r >> 1) & 7);
    woff[i] = ((unsigned)r * (unsigned)p.R + c * 8) * 2;
  }
#pragma unroll
  for (int i = 0; i < IB; ++i) {
    const int r = 8 * (wave * IB + i) + (lane >> 3), c = (lane & 7) ^ ((r >> 1) & 7);
    xoff[i] = r < xrows ? (rows[r] * (unsigned)p.W + c * 8) * 2 : 0xfffffff0u;
  }
  auto load_w = [&](int i, int slot, int t) {
    const bool on = t < nt;
    gp_load_lds(wp, on ? wbytes : 0u, lds + slot * (BN * 128) + (wave * IA + i) * 1024, woff[i], on ? t * (GP_BK * 2) : 0);
  };
  auto load_x = [&](int i, int slot, int t) {
    const bool on = t < nt;
    gp_load_lds(p.pages, on ? (unsigned)p.page_bytes : 0u, lds + XRING + slot * (BM * 128) + (wave * IB + i) * 1024, xoff[i],
                on ? t * (GP_BK * 2) : 0);
  };
  const bool keys = n0 < p.NK;                             // a tile is all keys or all values
  // the rows' rotary parts, 16 bytes a lane at a time: asked for ahead of the loop (one by one
  // behind it they took longer than the loop), through LDS once its rings are free
  constexpr int RC = BM * LK_MAX_ROT / 8 / 256;
  const int cpr = p.Dr / 8, chunks = keys ? xrows * cpr : 0;
  u32x4 rot[RC];
#pragma unroll
  for (int k = 0; k < RC; ++k) {
    const int c = threadIdx.x + 256 * k;
    if (c < chunks) rot[k] = *reinterpret_cast<const u32x4*>(p.pages + (size_t)rows[c / cpr] * p.W + p.R + c % cpr * 8);
  }
  __builtin_amdgcn_sched_barrier(0);
  float4v acc[FN][FM];
  gp_loop<FN, FM, NA, NB>(acc, lds, nt, wn, wm, lane, load_w, load_x);

  constexpr int WAVE_LDS = TM * (TN * 2 + 16);
  constexpr int ROT_LD = LK_MAX_ROT * 2 + 16;
  static_assert(WAVE_LDS * NW + BM * ROT_LD <= XRING + NB * BM * 128, "the epilogue's rows must fit the rings");
  __syncthreads();
  unsigned char* side = lds + WAVE_LDS * NW;
#pragma unroll
  for (int k = 0; k < RC; ++k) {
    const int c = threadIdx.x + 256 * k;
    if (c < chunks) *reinterpret_cast<u32x4*>(side + c / cpr * ROT_LD + c % cpr * 16) = rot[k];
  }
  __syncthreads();
  const int mw = wm * TM, nw = n0 + wn * TN;
  const int ld = keys ? p.NK : p.NV, col = keys ? nw : nw - p.NK;
  bf16_t* out = (keys ? p.k : p.v) + (size_t)(m0 + mw) * ld + col;
  int at[FN];                                              // of a block of 16 features among the rotary ones
#pragma unroll
  for (int i = 0; i < FN; ++i) {
    const int e = (col + 16 * i) % p.DK - p.D;
    at[i] = keys && e >= 0 && e < p.Dr ? e : -1;
  }
  gp_store<FN, FM, false>(lds + wave * WAVE_LDS, out, ld, xrows - mw, TN, lane, [&](int i, int j, float* o) {
#pragma unroll
    for (int r = 0; r < 4; ++r) o[r] = acc[i][j][r];
    if (at[i] >= 0) {
      const uint2 t = *reinterpret_cast<const uint2*>(side + (mw + 16 * j + fr) * ROT_LD + (at[i] + 4 * fq) * 2);
      o[0] = bf2f(t.x & 0xffff); o[1] = bf2f(t.x >> 16);
      o[2] = bf2f(t.y & 0xffff); o[3] = bf2f(t.y >> 16);
    }
  });
}

template <int FN, int FM, int NA, int NB> static int lk_launch(const LatentKvParams& p, hipStream_t st) {
  constexpr int BN = 32 * FN, BM = 32 * FM;
  if (p.NK % BN || p.NV % BN) return (int)hipErrorInvalidValue;
  hipLaunchKernelGGL((latent_kv_kernel<FN, FM, NA, NB>), dim3((p.total + BM - 1) / BM * ((p.NK + p.NV) / BN)), dim3(256), 0, st, p);
  return (int)hipGetLastError();
}

// layout: numbers of the pipelined projections' tiles (256 x 192, 128 x 128, 128 x 64)
extern "C" int loqa_latent_kv(const void* pages, long page_bytes, int blk, int W, const void* bt, int max_blocks,
                              const void* cu_k, const void* ctx, int B, int total, const void* w, int R, int H, int DK,
                              int DV, int D, void* k, void* v, int layout, hipStream_t st) {
  if (B <= 0 || total <= 0) return 0;
  const int Dr = W - R;
  if (R <= 0 || R % GP_BK || Dr < 0 || Dr > LK_MAX_ROT || Dr % 16 || D % 16 || D + Dr > DK || DK % 16 || W % 8 || blk <= 0 || page_bytes <= 0 ||
      page_bytes >= 0x7fffffffl || (((size_t)pages | (size_t)w | (size_t)k | (size_t)v) & 15) || (long)H * (DK + DV) >= (1 << 20))
    return (int)hipErrorInvalidValue;
  const LatentKvParams p{(const bf16_t*)pages, page_bytes, blk, W, (const int*)bt, max_blocks, (const int*)cu_k, (const int*)ctx,
                         B, total, (const bf16_t*)w, R, H * DK, H * DV, DK, D, Dr, (bf16_t*)k, (bf16_t*)v, layout};
  switch (layout) {
    case 13: return lk_launch<8, 6, 3, 2>(p, st);
    case 20: return lk_launch<4, 4, 4, 4>(p, st);
    case 19: return lk_launch<4, 2, 4, 4>(p, st);
    default: return (int)hipErrorInvalidValue;
  }
}
