// Grouped expert GEMM on the software-pipelined tile loop of gemm_pipe.h: for every expert
// segment of the plan, C = A W_e^T with the activation as the epilogue (moe.hip names the
// modes), bf16, K a multiple of 64.
//
// A tile is up to 256 weight rows (gate and up rows in turn for the gated modes, so one
// wave holds both halves of its features) x up to 256 (token, k) pairs of one expert. Rows
// are gathered by the loads themselves: a lane's 16 bytes come from its pair's token row,
// pairs past the segment and features past N read as zeros. Workgroups past the last tile
// (the host only knows how many there can be) leave at once; the others are dealt to the
// XCDs over the real number of tiles.
//
// Bound by the way L2 -> LDS and by the last round of tiles, as in gemm_pipe.hip; with few
// tokens by the stream of cold weights, which the smallest tile's four stages keep in
// flight. Against the form without LDS for the weights it replaces (whole moe_experts call,
// 16 experts of 2048 x 1408, 4 a token): 1 token 83 -> 26 us, 64: 114 -> 61, 512: 263 -> 89,
// 2048: 537 -> 190, 4000: 894 -> 312.
#include "seqmix.h"
#include "gemm_pipe.h"

#define MP_GROUP 4

// In full 32 bits: the hardware's exp2 and reciprocal (sigmoid_fast) are off by up to |a| ulp, which
// makes the whole call's error against 64 bits larger in the fifth digit (512 tokens: 0.00234913,
// 0.00234917), for 2 to 3 % less time (16 experts of 2048 x 1408, 4 a token; 64 tokens 61.0, 59.8 us;
// 512: 87.8, 85.7; 2048: 189, 183).
template <int MODE> __device__ __forceinline__ float moe_act(float a, float u, float limit) {
  if constexpr (MODE == 1) return silu_f(a) * u;
  else if constexpr (MODE == 2) { const float r = fmaxf(a, 0.f); return r * r; }
  else if constexpr (MODE == 3) {
    const float g = fminf(a, limit);
    return g * sigmoid_f(1.702f * g) * (fminf(fmaxf(u, -limit), limit) + 1.f);
  } else return a;
}

struct MoePipeParams {
  const bf16_t* a; unsigned abytes; const bf16_t* w; const int* plan;
  int E, top, K, N; float limit; bf16_t* out;
};

template <int FN, int FM, int NA, int NB, int MODE>
__global__ __launch_bounds__(256, (gp_per_cu<FN, FM, NA, NB>())) void moe_pipe_kernel(MoePipeParams p) {
  constexpr int TN = 16 * FN, TM = 16 * FM, BN = 2 * TN, BM = 2 * TM;
  constexpr int IA = BN / 32, IB = BM / 32, XRING = NA * BN * 128;
  constexpr bool GATED = MODE == 1 || MODE == 3;
  constexpr int FO = GATED ? FN / 2 : FN, ON = 32 * FO;      // output features: of a wave / 16, of the tile
  __shared__ __attribute__((aligned(1024))) unsigned char lds[gp_lds_bytes<FN, FM, NA, NB>()];
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int wn = wave & 1, wm = wave >> 1;
  const int K = p.K, N = p.N, nblocks = (N + ON - 1) / ON;
  const int rts = __builtin_amdgcn_readfirstlane(seq_chunks_before<BM>(p.plan, p.E));
  if ((int)blockIdx.x >= rts * nblocks) return;
  const int id = xcd_remap(blockIdx.x, rts * nblocks);
  const int per = MP_GROUP * nblocks, grp = id / per, in = id - grp * per;
  const int gm = min(MP_GROUP, rts - grp * MP_GROUP);
  int e, r0, n;
  seq_chunk<BM>(p.plan, p.E, grp * MP_GROUP + in % gm, e, r0, n);
  e = __builtin_amdgcn_readfirstlane(e);
  r0 = __builtin_amdgcn_readfirstlane(r0);
  n = __builtin_amdgcn_readfirstlane(n);
  const int f0 = in / gm * ON;
  const int* perm = p.plan + p.E + 2;

  const unsigned wbytes = (unsigned)((GATED ? 2 * N : N) * K) * 2u;
  const bf16_t* wp = p.w + (size_t)e * (GATED ? 2 * N : N) * K;
  unsigned woff[IA], xoff[IB];
#pragma unroll
  for (int i = 0; i < IA; ++i) {
    const int r = 8 * (wave * IA + i) + (lane >> 3), c = (lane & 7) ^ ((r >> 1) & 7);
    int f = f0 + r, row = f;
    if constexpr (GATED) {
      const int blk = r / TN, rr = r - blk * TN;
      f = f0 + blk * (TN / 2) + rr % (TN / 2);
      row = rr < TN / 2 ? f : N + f;
    }
    woff[i] = f < N ? ((unsigned)row * (unsigned)K + c * 8) * 2 : 0xfffffff0u;
  }
#pragma unroll
  for (int i = 0; i < IB; ++i) {
    const int r = 8 * (wave * IB + i) + (lane >> 3), c = (lane & 7) ^ ((r >> 1) & 7);
    const int pair = r0 + min(r, n - 1);
    const unsigned src = MODE != 0 ? (unsigned)perm[pair] / (unsigned)p.top : (unsigned)pair;
    xoff[i] = r < n ? (src * (unsigned)K + c * 8) * 2 : 0xfffffff0u;
  }
  const int nt = K / GP_BK;
  auto load_w = [&](int i, int slot, int t) {
    const bool on = t < nt;
    gp_load_lds(wp, on ? wbytes : 0u, lds + slot * (BN * 128) + (wave * IA + i) * 1024, woff[i], on ? t * 128 : 0);
  };
  auto load_x = [&](int i, int slot, int t) {
    const bool on = t < nt;
    gp_load_lds(p.a, on ? p.abytes : 0u, lds + XRING + slot * (BM * 128) + (wave * IB + i) * 1024, xoff[i],
                on ? t * 128 : 0);
  };
  float4v acc[FN][FM];
  gp_loop<FN, FM, NA, NB>(acc, lds, nt, wn, wm, lane, load_w, load_x);

  constexpr int WAVE_LDS = TM * (FO * 32 + 16);
  static_assert(WAVE_LDS * 4 <= gp_lds_bytes<FN, FM, NA, NB>(), "the epilogue's rows must fit the rings");
  __syncthreads();
  const int col = f0 + wn * (ON / 2);
  gp_store<FO, FM, false>(lds + wave * WAVE_LDS, p.out + (size_t)(r0 + wm * TM) * N + col, N, n - wm * TM, N - col, lane,
                          [&](int i, int j, float* o) {
#pragma unroll
                            for (int r = 0; r < 4; ++r) o[r] = moe_act<MODE>(acc[i][j][r], acc[i + (GATED ? FO : 0)][j][r], p.limit);
                          });
}

// Tiles: weight rows x pairs, stages, us a K step of 64 and around a tile's K loop (as the
// plain GEMM's, ops.SK_LAYOUTS)
struct MoeTile { int bn, bm; float step, around; };
static const MoeTile MOE_TILES[] = {{256, 256, 1.20f, 10.3f}, {256, 192, 1.08f, 5.5f}, {256, 128, 0.91f, 4.0f},
                                    {128, 128, 0.50f, 3.6f}, {128, 64, 0.31f, 4.3f}};

template <int FN, int FM, int NA, int NB>
static void mp_launch(const MoePipeParams& p, int mode, int grid, hipStream_t st) {
  switch (mode) {
    case 1: hipLaunchKernelGGL((moe_pipe_kernel<FN, FM, NA, NB, 1>), dim3(grid), dim3(256), 0, st, p); break;
    case 2: hipLaunchKernelGGL((moe_pipe_kernel<FN, FM, NA, NB, 2>), dim3(grid), dim3(256), 0, st, p); break;
    case 3: hipLaunchKernelGGL((moe_pipe_kernel<FN, FM, NA, NB, 3>), dim3(grid), dim3(256), 0, st, p); break;
    default: hipLaunchKernelGGL((moe_pipe_kernel<FN, FM, NA, NB, 0>), dim3(grid), dim3(256), 0, st, p);
  }
}

// false: operands this form does not take
bool moe_pipe(const void* A, long rows, const void* W, const void* plan, int P, int E, int top, int K, int N, int mode,
              float limit, void* out, hipStream_t st) {
  const bool gated = mode == 1 || mode == 3;
  if (K % GP_BK || N % 8 || rows * K * 2 >= 0xfffffff0l || (long)N * (gated ? 2 : 1) * K * 2 >= 0xfffffff0l ||
      ((size_t)A | (size_t)W | (size_t)out) & 15)
    return false;
  if (E <= 0) return true;                                // identity experts only: nothing to multiply
  // the tile whose rounds over the compute units take least, with an expert's last tile half
  // empty on average
  const int used = E < P ? E : P;
  int best = 0;
  float best_t = 1e30f;
  for (int i = 0; i < 5; ++i) {
    const MoeTile& t = MOE_TILES[i];
    const int on = gated ? t.bn / 2 : t.bn, nb = (N + on - 1) / on;
    const float items = fmaxf(1.f, (float)P / used / t.bm + 0.5f) * used * nb;
    const float us = ceilf(items / 256.f) * (K / GP_BK * t.step + t.around);
    if (us < best_t) { best_t = us; best = i; }
  }
  const MoeTile& t = MOE_TILES[best];
  const int on = gated ? t.bn / 2 : t.bn;
  // every expert may leave a tile part empty
  const long tiles = (P / t.bm + used) * (long)((N + on - 1) / on);
  if (tiles > 0x7fffffff) return false;
  const MoePipeParams p{(const bf16_t*)A, (unsigned)(rows * K * 2), (const bf16_t*)W, (const int*)plan, E, top, K, N, limit,
                        (bf16_t*)out};
  switch (best) {
    case 0: mp_launch<8, 8, 3, 2>(p, mode, (int)tiles, st); break;
    case 1: mp_launch<8, 6, 3, 2>(p, mode, (int)tiles, st); break;
    case 2: mp_launch<8, 4, 3, 3>(p, mode, (int)tiles, st); break;
    case 3: mp_launch<4, 4, 5, 5>(p, mode, (int)tiles, st); break;
    default: mp_launch<4, 2, 4, 4>(p, mode, (int)tiles, st);
  }
  return true;
}
