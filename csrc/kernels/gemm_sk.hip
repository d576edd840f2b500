// Split-K LDS-tiled MFMA GEMM with an in-launch reduction and fused epilogues:
// Y[M, N] = X[M, K] W[N, K]^T for the projections of a prompt pass (Llama
// prefill: M = a few hundred to a few thousand rows) and the Whisper encoder.
//
// This file holds the general form (any feature count that is a multiple of 64, any row
// alignment that 16-byte loads take) and the entry point; gemm_pipe.hip has the pipelined
// form that serves everything else.
//
// Why split-K inside the launch: at M ~ 300 a projection has few output tiles
// (qkv 6144 x 4096: 240 tiles of 128 x 64; o / down 4096 wide: 160), far fewer
// than the 256 CUs x 2-3 resident workgroups, and a whole tile's K loop is one
// workgroup's serial latency. Splitting each tile's K range over S workgroups
// fills the machine; the S partial accumulators are summed by the LAST
// workgroup of the tile to finish (agent-scope release / ticket / acquire), which then runs the epilogue - no
// f32 slabs for a later kernel to re-read and no extra launch. The sum is in
// fixed chunk order over the published partials (the reducer's own included),
// so the result is bitwise identical whoever arrives last.
//
// Main loop: as gemm_tile.hip - BK = 64 stages of (BN + BM) rows x 128 B filled
// by global_load_lds with the LDS bank swizzle on the source address, NBUF - 1
// stages in flight across raw s_barriers (counted vmcnt), XCD-aware workgroup
// order with a tile's K chunks adjacent on one XCD.
//
// Epilogues (applied once per output element, by the tile's reducer):
//   SK_BF16   y = bf16(acc (+ bias)), optionally GELU (Whisper encoder fc1)
//   SK_SWIGLU y[:, f] = silu(gate_f) * up_f (a wave tile holds TN/2 gate and the
//             matching TN/2 up features, row-permuted at staging)
//   SK_RESID  y = bf16(y + (acc + bias)): the row-parallel projections (o,
//             down, encoder o / fc2) add straight into the residual stream, one
//             rounding.
#include "gemm_sk.h"

template <int WN, int WM, int FN, int FM, int NBUF, int EPI>
__global__ __launch_bounds__(64 * WN * WM) void gemm_sk_kernel(GemmSkParams p) {
  constexpr int NW = WN * WM;
  constexpr int TN = 16 * FN, TM = 16 * FM;      // wave tile: TN features x TM rows
  constexpr int BN = TN * WN, BM = TM * WM;
  constexpr int ROWS = BN + BM;
  constexpr int STAGE = ROWS * 128;             // bytes per stage
  constexpr int IPW = ROWS / 8 / NW;            // glds instructions per wave per stage
  static_assert(IPW * 8 * NW == ROWS, "stage rows must split evenly over the waves");
  static_assert(EPI != SK_SWIGLU || FN % 2 == 0, "SwiGLU pairs gate / up fragments");
  __shared__ __attribute__((aligned(1024))) unsigned char lds[NBUF * STAGE];

  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int wn = wave % WN, wm = wave / WN;
  const int M = p.M, N = p.N, S = p.S;
  const int mblocks = (M + BM - 1) / BM;
  const int id = xcd_remap(blockIdx.x, gridDim.x);
  const int s = id % S, tile = id / S;
  const int mb = tile % mblocks, nb = tile / mblocks;
  const int KT = p.K / SK_BK;
  const int kt0 = (int)(((long long)s * KT) / S), kt1 = (int)(((long long)(s + 1) * KT) / S);
  const int nt = kt1 - kt0;
  const int m0 = mb * BM, n0 = nb * BN;
  const bf16_t* __restrict__ X = reinterpret_cast<const bf16_t*>(p.x);
  const bf16_t* __restrict__ W = reinterpret_cast<const bf16_t*>(p.w);

  // per-lane source of each of this wave's stage instructions (k offset added per stage)
  const bf16_t* src[IPW];
#pragma unroll
  for (int i = 0; i < IPW; ++i) {
    const int r = 8 * (wave * IPW + i) + (lane >> 3);
    const int c = (lane & 7) ^ ((r >> 1) & 7);
    if (r < BN) {
      int row;
      if constexpr (EPI == SK_SWIGLU) {
        const int blk = r / TN, rr = r - blk * TN;
        const int f = (n0 >> 1) + blk * (TN / 2) + (rr % (TN / 2));
        row = rr < TN / 2 ? f : (N >> 1) + f;
      } else {
        row = n0 + r;
      }
      src[i] = W + (size_t)row * p.K + c * 8;
    } else {
      const int m = min(m0 + r - BN, M - 1);
      src[i] = X + (size_t)m * p.ldx + c * 8;
    }
  }

  auto stage = [&](int buf, int kt) {
    const int kc = kt * SK_BK;
#pragma unroll
    for (int i = 0; i < IPW; ++i)
      __builtin_amdgcn_global_load_lds(
          (const __attribute__((address_space(1))) void*)(src[i] + kc),
          (__attribute__((address_space(3))) void*)(lds + buf * STAGE + (wave * IPW + i) * 1024), 16, 0, 0);
  };

  float4v acc[FN][FM];
#pragma unroll
  for (int i = 0; i < FN; ++i)
#pragma unroll
    for (int j = 0; j < FM; ++j) acc[i][j] = float4v{0.f, 0.f, 0.f, 0.f};

  const int fr = lane & 15, fq = lane >> 4;
  auto frag = [&](int buf, int row, int c) -> bf16x8 {
    return *reinterpret_cast<const bf16x8*>(lds + buf * STAGE + row * 128 + 16 * (c ^ ((row >> 1) & 7)));
  };
  auto compute = [&](int buf) {
    // Half 0's fragments (activations first), then its MFMAs row by row with
    // half 1's fragment reads issued between them (sched barriers pin the
    // order), then half 1's MFMAs: only half 0's reads are exposed, and at most
    // FN + FM + 2 LDS reads are ever outstanding (the 4-bit lgkmcnt: with more
    // pending, the waitcnt pass can only wait for all of them).
    static_assert(FN + FM + 2 <= 15, "outstanding LDS reads exceed lgkmcnt");
    bf16x8 af[2][FN], bfr[2][FM];
    {
      constexpr int sub = 0;
#pragma unroll
      for (int j = 0; j < FM; ++j) bfr[0][j] = frag(buf, BN + wm * TM + 16 * j + fr, 4 * sub + fq);
#pragma unroll
      for (int i = 0; i < FN; ++i) af[0][i] = frag(buf, wn * TN + 16 * i + fr, 4 * sub + fq);
    }
    __builtin_amdgcn_sched_barrier(0);
    __builtin_amdgcn_s_setprio(1);
#pragma unroll
    for (int i = 0; i < FN; ++i) {
#pragma unroll
      for (int j = 0; j < FM; ++j)
        acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(af[0][i], bfr[0][j], acc[i][j], 0, 0, 0);
      {
        constexpr int sub = 1;
        af[1][i] = frag(buf, wn * TN + 16 * i + fr, 4 * sub + fq);
        if (i < FM) {
          const int j = i;
          bfr[1][j] = frag(buf, BN + wm * TM + 16 * j + fr, 4 * sub + fq);
        }
      }
      __builtin_amdgcn_sched_barrier(0);
    }
#pragma unroll
    for (int j = FN; j < FM; ++j) {
      constexpr int sub = 1;
      bfr[1][j] = frag(buf, BN + wm * TM + 16 * j + fr, 4 * sub + fq);
    }
#pragma unroll
    for (int i = 0; i < FN; ++i)
#pragma unroll
      for (int j = 0; j < FM; ++j)
        acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(af[1][i], bfr[1][j], acc[i][j], 0, 0, 0);
    __builtin_amdgcn_s_setprio(0);
  };

  int issued = 0;
#pragma unroll
  for (int q = 0; q < NBUF - 1; ++q)
    if (q < nt) {
      stage(q, kt0 + q);
      ++issued;
    }
  for (int t = 0; t < nt; ++t) {
    // stage t has landed once at most (issued - t - 1) newer stages are pending
    // (up to NBUF - 2 in steady state; fewer in the last iterations)
    const int newer = issued - t - 1;
    if (NBUF >= 4 && newer >= 2) sk_wait_vm<IPW * 2>();
    else if (NBUF >= 3 && newer >= 1) sk_wait_vm<IPW>();
    else sk_wait_vm<0>();
    __builtin_amdgcn_s_barrier();
    // the buffer refilled here was last read in iteration t - 1, which every
    // wave finished before the barrier above
    if (issued < nt) {
      stage(issued % NBUF, kt0 + issued);
      ++issued;
    }
    compute(t % NBUF);
  }

  if (S > 1 && !sk_reduce<NW, FN, FM>(p, acc, tile, s, wave, lane, reinterpret_cast<int*>(lds))) return;
  sk_epilogue<EPI, FN, FM>(p, acc, n0 + wn * TN, (n0 >> 1) + wn * (TN / 2), m0 + wm * TM, fr, fq);
}

template <int WN, int WM, int FN, int FM, int NBUF>
static int sk_launch(const GemmSkParams& p, hipStream_t st) {
  constexpr int BN = 16 * FN * WN, BM = 16 * FM * WM;
  if (p.N % BN || p.K % SK_BK || p.S > p.K / SK_BK) return (int)hipErrorInvalidValue;
  const long long tiles = (long long)((p.M + BM - 1) / BM) * (p.N / BN);
  const long long grid = tiles * p.S;
  if (grid > 0x7fffffff) return (int)hipErrorInvalidValue;
  dim3 block(64 * WN * WM);
  switch (p.epi) {
    case SK_SWIGLU:
      if constexpr (FN % 2 == 0) {
        hipLaunchKernelGGL((gemm_sk_kernel<WN, WM, FN, FM, NBUF, SK_SWIGLU>), dim3(grid), block, 0, st, p);
        break;
      } else {
        return (int)hipErrorInvalidValue;
      }
    case SK_RESID:
      hipLaunchKernelGGL((gemm_sk_kernel<WN, WM, FN, FM, NBUF, SK_RESID>), dim3(grid), block, 0, st, p);
      break;
    default:
      hipLaunchKernelGGL((gemm_sk_kernel<WN, WM, FN, FM, NBUF, SK_BF16>), dim3(grid), block, 0, st, p);
  }
  return (int)hipGetLastError();
}

int gemm_pipe(const GemmSkCall& p, int layout, hipStream_t st);   // gemm_pipe.hip

// layout: 1: 128 x 64 (2 x 2 waves of 64 x 32), 7: 64 x 64 (2 x 2 waves of 32 x 32), two
// stages each - the general forms, for feature counts that are no multiple of 128 and rows
// that are not 16-byte aligned; 11 on: the pipelined tiles of gemm_pipe.hip
extern "C" int loqa_gemm_sk(const GemmSkCall* p, hipStream_t st) {
  if (!p || p->M <= 0 || p->S < 1 || p->hurry < 0 || p->epi < 0 || p->epi > 2 || !p->x || !p->w || !p->y)
    return (int)hipErrorInvalidValue;
  if (p->S > 1 && (!p->ws || !p->counters)) return (int)hipErrorInvalidValue;
  if (p->ldx % 8 || p->ldy % 4) return (int)hipErrorInvalidValue;
  if ((p->epi == SK_SWIGLU && p->bias) || (p->epi != SK_BF16 && p->act)) return (int)hipErrorInvalidValue;
  if (p->ahead_wgs && p->layout < 11) return (int)hipErrorInvalidValue;
  switch (p->layout) {
    case 1: return sk_launch<2, 2, 4, 2, 2>(*p, st);
    case 7: return sk_launch<2, 2, 2, 2, 2>(*p, st);
    default: return gemm_pipe(*p, p->layout - 12, st);
  }
}

// The capture that `st` records into (unique in the process), for workspaces that its launches share.
extern "C" int loqa_capture_id(hipStream_t st, unsigned long long* id) {
  hipStreamCaptureStatus status = hipStreamCaptureStatusNone;
  const hipError_t e = hipStreamGetCaptureInfo(st, &status, id);
  if (e != hipSuccess) return (int)e;
  return status == hipStreamCaptureStatusActive ? 0 : (int)hipErrorInvalidValue;
}
