// Software-pipelined tiled MFMA GEMM for the prompt-pass and encoder projections,
// Y[M, N] = X[M, K] W[N, K]^T with the K split, reduction and epilogues of gemm_sk.h.
//
// Four waves (2 along the features, 2 along the rows), one per SIMD, own wave tiles of
// up to 128 x 128. What bounds a tile GEMM here is the way from L2 into LDS: 1 KB takes a
// CU 17 - 23 cycles when it comes as whole 128-byte lines (37 as 64-byte pieces), so a K
// step of 64 costs about 1220 cycles of loading against 2048 of MFMA at 256 x 256, 910
// against 1024 at 256 x 128 and 610 against 512 at 128 x 128. Hence the largest tile that
// fills the chip, 128-byte LDS rows, and loads spread evenly over all MFMAs: a burst
// queues up in front of the cache and stalls the wave's in-order MFMA issue.
//
// With one wave per SIMD nothing but this wave's own instruction order hides a latency:
// the fragments of the next K half are read between the MFMAs of the current one (two
// register sets). A stage of 64 K entries runs in two halves:
//
//   half 0 of stage t:  MFMAs | reads of half 1 of t     | W rows of t + NA - 1 -> LDS
//   wait: half 1 read, stage t + 1 landed; barrier (the buffers of stage t are free)
//   half 1 of stage t:  MFMAs | reads of half 0 of t + 1 | X rows of t + NB -> LDS
//
// W and X have rings of their own (NA and NB stages): at 256 x 256 three and two stages of
// 32 KB fill the 160 KB, and half of the loads get a stage and a half to arrive.
// LDS rows are 128 bytes, 16-byte chunk c of row r at place c ^ ((r >> 1) & 7) (swizzled
// on the source address): 16 neighbouring rows of one chunk fall into 16 different
// quarter-banks (no conflicts counted).
//
// Tiles go to the XCDs in contiguous runs, within a run in groups of 4 row blocks with the
// feature block slowest, so the 32 tiles an XCD works on at a time form a 4 x 8 patch:
// 12 tile edges pass its L2 per K step instead of 33 (8192^3: 1290 -> 1365 TFLOP/s against
// groups of 8).
#include "gemm_sk.h"

#define GP_GROUP 4

// In place, on the accumulation registers: left to the register allocator, the builtin's
// result and addend part ways and every MFMA is followed by register moves. Nothing but
// other MFMAs, FN FM issues away, touches the accumulators inside the loop.
__device__ __forceinline__ void gp_mfma(float4v& c, const bf16x8& a, const bf16x8& b) {
  asm volatile("v_mfma_f32_16x16x32_bf16 %0, %1, %2, %0" : "+a"(c) : "v"(a), "v"(b));
}

// 16 bytes per lane of [base, base + bytes) at off + soff, straight into LDS (lane l at
// dst + 16 l); out of range reads as zero.
__device__ __forceinline__ void gp_load_lds(const bf16_t* base, unsigned bytes, unsigned char* dst, unsigned off,
                                            unsigned soff) {
  __builtin_amdgcn_raw_ptr_buffer_load_lds(
      __builtin_amdgcn_make_buffer_rsrc(const_cast<bf16_t*>(base), 0, bytes, 0x00020000),
      (__attribute__((address_space(3))) void*)dst, 16, off, soff, 0, 0);
}

// workgroups per CU by LDS
template <int FN, int FM, int NA, int NB> constexpr int gp_per_cu() {
  return 160 * 1024 / ((NA * FN + NB * FM) * 32 * 128);
}

// Epilogue of one wave through its own part of LDS. The accumulators of an MFMA tile hold
// four neighbouring features of one row per lane, so storing them directly makes every
// 8-byte piece of an instruction a line of its own (9000 x 3840 x 1280: 26 of 96 us went
// into the stores, 38 with the residual's loads). Instead the finished bf16 pieces go to
// LDS and leave as whole rows, 16 bytes a lane; the residual comes in the same way.
template <int EPI, int FN, int FM>
__device__ __forceinline__ void gp_epilogue(const GemmSkParams& p, float4v (&acc)[FN][FM], unsigned char* my, int nw,
                                            int fw, int mw, int lane) {
  constexpr int ON = EPI == SK_SWIGLU ? 8 * FN : 16 * FN;   // output features of the wave
  constexpr int LD = ON * 2 + 16;                           // bytes of a row in LDS
  constexpr int CPR = ON / 8;                               // 16-byte chunks of a row
  constexpr int CH = 16 * FM * CPR / 64;                    // chunks per lane
  static_assert(CH * 64 == 16 * FM * CPR, "chunks must split evenly over the lanes");
  typedef unsigned u32x4 __attribute__((ext_vector_type(4)));
  const int fr = lane & 15, fq = lane >> 4;
  bf16_t* Y = reinterpret_cast<bf16_t*>(p.y) + (EPI == SK_SWIGLU ? fw : nw);
  const int rows = p.M - mw;                                // rows of the wave's tile that exist
  if constexpr (EPI == SK_RESID) {
    u32x4 v[CH];
#pragma unroll
    for (int k = 0; k < CH; ++k) {
      const int id = lane + 64 * k, r = min(id / CPR, rows - 1), c = id % CPR;
      if (rows > 0) v[k] = *reinterpret_cast<const u32x4*>(Y + (size_t)(mw + r) * p.ldy + c * 8);
    }
#pragma unroll
    for (int k = 0; k < CH; ++k) {
      const int id = lane + 64 * k;
      *reinterpret_cast<u32x4*>(my + (id / CPR) * LD + (id % CPR) * 16) = v[k];
    }
  }
  float4 bv[FN];
  if constexpr (EPI != SK_SWIGLU)
#pragma unroll
    for (int i = 0; i < FN; ++i)
      bv[i] = p.bias ? *reinterpret_cast<const float4*>(p.bias + nw + 16 * i + 4 * fq) : make_float4(0.f, 0.f, 0.f, 0.f);
  __builtin_amdgcn_wave_barrier();
#pragma unroll
  for (int j = 0; j < FM; ++j) {
    unsigned char* row = my + (16 * j + fr) * LD + fq * 8;
#pragma unroll
    for (int i = 0; i < (EPI == SK_SWIGLU ? FN / 2 : FN); ++i) {
      uint2* at = reinterpret_cast<uint2*>(row + i * 32);
      float o[4];
      if constexpr (EPI == SK_SWIGLU) {
#pragma unroll
        for (int r = 0; r < 4; ++r) o[r] = sk_swiglu(acc[i][j][r], acc[i + FN / 2][j][r]);
      } else {
        o[0] = acc[i][j][0] + bv[i].x; o[1] = acc[i][j][1] + bv[i].y;
        o[2] = acc[i][j][2] + bv[i].z; o[3] = acc[i][j][3] + bv[i].w;
        if constexpr (EPI == SK_RESID) {
          const uint2 rv = *at;
          o[0] += bf2f(rv.x & 0xffff); o[1] += bf2f(rv.x >> 16);
          o[2] += bf2f(rv.y & 0xffff); o[3] += bf2f(rv.y >> 16);
        } else if (p.act == 1) {
#pragma unroll
          for (int r = 0; r < 4; ++r) o[r] = sk_gelu(o[r]);
        }
      }
      *at = make_uint2(pack_bf16x2(o[0], o[1]), pack_bf16x2(o[2], o[3]));
    }
    __builtin_amdgcn_sched_barrier(0);   // a row block's accumulators at a time
  }
  __builtin_amdgcn_wave_barrier();
#pragma unroll
  for (int k = 0; k < CH; ++k) {
    const int id = lane + 64 * k, r = id / CPR, c = id % CPR;
    const u32x4 v = *reinterpret_cast<const u32x4*>(my + r * LD + c * 16);
    if (r < rows) *reinterpret_cast<u32x4*>(Y + (size_t)(mw + r) * p.ldy + c * 8) = v;
  }
}

template <int FN, int FM, int NA, int NB, int EPI>
__global__ __launch_bounds__(256, (gp_per_cu<FN, FM, NA, NB>())) void gemm_pipe_kernel(GemmSkParams p) {
  constexpr int NW = 4;
  constexpr int TN = 16 * FN, TM = 16 * FM;
  constexpr int BN = 2 * TN, BM = 2 * TM;
  constexpr int IA = BN / 8 / NW, IB = BM / 8 / NW;   // 1 KB direct-to-LDS loads per wave and stage
  static_assert(IA * 8 * NW == BN && IB * 8 * NW == BM, "rows must split evenly over the waves");
  constexpr int XRING = NA * BN * 128;                // where the ring of X stages starts
  __shared__ __attribute__((aligned(1024))) unsigned char lds[XRING + NB * BM * 128];

  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int wn = wave & 1, wm = wave >> 1;
  const int M = p.M, N = p.N, S = p.S;
  const int mblocks = (M + BM - 1) / BM, nblocks = N / BN;
  const int id = xcd_remap(blockIdx.x, gridDim.x);
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

  const int fr = lane & 15, fq = lane >> 4;
  // a fragment's place: rows 16 i apart keep the swizzle, the other K half is 64 bytes away
  const int swz = 16 * (fq ^ ((fr >> 1) & 7));
  const int abase = (wn * TN + fr) * 128 + swz, bbase = XRING + (wm * TM + fr) * 128 + swz;
  float4v acc[FN][FM];
#pragma unroll
  for (int i = 0; i < FN; ++i)
#pragma unroll
    for (int j = 0; j < FM; ++j) {
      acc[i][j] = float4v{0.f, 0.f, 0.f, 0.f};
      asm volatile("" : "+a"(acc[i][j]));
    }
  bf16x8 af[2][FN], bfr[2][FM];
  // read q (0 .. FN + FM - 1) of a K half into its register set
  auto read = [&](int q, int sa, int sb, int half) {
    if (q < FM)
      bfr[half][q] = *reinterpret_cast<const bf16x8*>(lds + sb * (BM * 128) + ((bbase ^ (64 * half)) + q * 2048));
    else
      af[half][q - FM] = *reinterpret_cast<const bf16x8*>(lds + sa * (BN * 128) + ((abase ^ (64 * half)) + (q - FM) * 2048));
  };
  constexpr int MF = FN * FM, R = FN + FM;
  constexpr int SPAN = MF * 7 / 8;                 // reads are spread over this many MFMAs
  // loads issued behind those of stage t + 1 when it is waited for in the middle of stage t
  constexpr int BEHIND_W = (NA - 2) * (IA + IB), BEHIND_X = (NB - 1) * IA + (NB - 2) * IB;
  constexpr int BEHIND = BEHIND_W < BEHIND_X ? BEHIND_W : BEHIND_X;

#pragma unroll
  for (int q = 0; q < NB || q < NA - 1; ++q) {
#pragma unroll
    for (int i = 0; i < IA; ++i)
      if (q < NA - 1) load_w(i, q, q);
#pragma unroll
    for (int i = 0; i < IB; ++i)
      if (q < NB) load_x(i, q, q);
  }
  sk_wait_vm<(NA - 2) * IA + (NB - 1) * IB>();     // stage 0 is here
  __builtin_amdgcn_s_barrier();
#pragma unroll
  for (int q = 0; q < R; ++q) read(q, 0, 0, 0);
  int sa = 0, sb = 0;                              // ring slots of stage t
  for (int t = 0; t < nt; ++t) {
    const int sp = sa == 0 ? NA - 1 : sa - 1;      // freed in the middle of stage t - 1
#pragma unroll
    for (int x = 0; x < MF; ++x) {
      gp_mfma(acc[x / FM][x % FM], af[0][x / FM], bfr[0][x % FM]);
#pragma unroll
      for (int q = x * R / SPAN; q < (x + 1) * R / SPAN && q < R; ++q) read(q, sa, sb, 1);
#pragma unroll
      for (int q = x * IA / MF; q < (x + 1) * IA / MF; ++q) load_w(q, sp, t + NA - 1);
      __builtin_amdgcn_sched_barrier(0);
    }
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");   // this wave has read all of stage t,
    sk_wait_vm<BEHIND>();                                // and its part of t + 1 has landed
    __builtin_amdgcn_s_barrier();
    const int na = sa + 1 == NA ? 0 : sa + 1, nb2 = sb + 1 == NB ? 0 : sb + 1;
#pragma unroll
    for (int x = 0; x < MF; ++x) {
      gp_mfma(acc[x / FM][x % FM], af[1][x / FM], bfr[1][x % FM]);
#pragma unroll
      for (int q = x * R / SPAN; q < (x + 1) * R / SPAN && q < R; ++q) read(q, na, nb2, 0);
#pragma unroll
      for (int q = x * IB / MF; q < (x + 1) * IB / MF; ++q) load_x(q, sb, t + NB);
      __builtin_amdgcn_sched_barrier(0);
    }
    sa = na;
    sb = nb2;
  }
  // no load into LDS outlives the loop; the last MFMAs' results are 16 cycles away from
  // being readable, and only this wait tells the compiler's moves so
  asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)\n s_nop 15\n s_nop 15" ::: "memory");
#pragma unroll
  for (int i = 0; i < FN; ++i)
#pragma unroll
    for (int j = 0; j < FM; ++j) asm volatile("" : "+a"(acc[i][j]));

  if (S > 1 && !sk_reduce<NW, FN, FM>(p, acc, tile, s, wave, lane, reinterpret_cast<int*>(lds))) return;
  // every wave has read its last fragments, every load has landed: the rings are free
  constexpr int WAVE_LDS = TM * (TN * 2 + 16);
  static_assert(WAVE_LDS * NW <= XRING + NB * BM * 128, "the epilogue's rows must fit the rings");
  __syncthreads();
  gp_epilogue<EPI, FN, FM>(p, acc, lds + wave * WAVE_LDS, n0 + wn * TN, (n0 >> 1) + wn * (TN / 2), m0 + wm * TM, lane);
}

template <int FN, int FM, int NA, int NB>
static int gp_launch(const GemmSkParams& p, hipStream_t st) {
  constexpr int BN = 32 * FN, BM = 32 * FM;
  if (p.N % BN || p.K % SK_BK || p.S > p.K / SK_BK) return (int)hipErrorInvalidValue;
  // 32-bit buffer offsets: a tile's rows of X, and all of W (SwiGLU: its other half)
  if ((long long)BM * p.ldx * 2 >= 0x7fffffffll || (long long)p.N * p.K * 2 >= 0xfffffff0ll || p.ldx < p.K)
    return (int)hipErrorInvalidValue;
  // whole 16-byte pieces of the output rows
  if (p.ldy % 8 || ((size_t)p.y & 15) || ((size_t)p.x & 15) || ((size_t)p.w & 15)) return (int)hipErrorInvalidValue;
  const long long grid = (long long)((p.M + BM - 1) / BM) * (p.N / BN) * p.S;
  if (grid > 0x7fffffff) return (int)hipErrorInvalidValue;
  switch (p.epi) {
    case SK_SWIGLU:
      hipLaunchKernelGGL((gemm_pipe_kernel<FN, FM, NA, NB, SK_SWIGLU>), dim3(grid), dim3(256), 0, st, p);
      break;
    case SK_RESID:
      hipLaunchKernelGGL((gemm_pipe_kernel<FN, FM, NA, NB, SK_RESID>), dim3(grid), dim3(256), 0, st, p);
      break;
    default:
      hipLaunchKernelGGL((gemm_pipe_kernel<FN, FM, NA, NB, SK_BF16>), dim3(grid), dim3(256), 0, st, p);
  }
  return (int)hipGetLastError();
}

// (features x rows), stages of W and X; the smaller tiles spend the LDS on deeper rings, as
// what they wait for is the first touch of cold weights
int gemm_pipe(const GemmSkParams& p, int layout, hipStream_t st) {
  switch (layout) {
    case 0: return gp_launch<8, 8, 3, 2>(p, st);   // 256 x 256
    case 1: return gp_launch<8, 6, 3, 2>(p, st);   // 256 x 192
    case 2: return gp_launch<6, 8, 3, 2>(p, st);   // 192 x 256
    case 3: return gp_launch<8, 4, 3, 3>(p, st);   // 256 x 128
    case 4: return gp_launch<4, 8, 3, 3>(p, st);   // 128 x 256
    case 5: return gp_launch<4, 6, 3, 3>(p, st);   // 128 x 192
    case 6: return gp_launch<6, 6, 3, 3>(p, st);   // 192 x 192
    case 7: return gp_launch<4, 2, 4, 4>(p, st);   // 128 x 64
    case 8: return gp_launch<4, 4, 5, 5>(p, st);   // 128 x 128
    default: return (int)hipErrorInvalidValue;
  }
}
