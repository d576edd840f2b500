// Device parts of the software-pipelined tile GEMM (gemm_pipe.hip; the experts' grouped
// GEMM in moe_pipe.hip): direct-to-LDS loads, the K loop of a tile, and the way of a wave's
// results through LDS.
#pragma once
#include "common.h"

typedef unsigned u32x4 __attribute__((ext_vector_type(4)));

#define GP_BK 64                       // K entries of a stage: 128-byte LDS rows

// s_waitcnt vmcnt(N), the other counters at their maxima (vmcnt[3:0] in bits 3:0,
// vmcnt[5:4] in bits 15:14)
template <int N>
__device__ __forceinline__ void gp_wait_vm() {
  static_assert(N >= 0 && N < 64, "vmcnt range");
  __builtin_amdgcn_s_waitcnt((N & 15) | ((N >> 4) << 14) | (7 << 4) | (15 << 8));
}

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

// Worker `id` of `n` waves touches its share of [base, base + bytes), kilobyte by kilobyte, so
// that the lines are in the Infinity Cache when a later launch asks for them: loads into a
// kilobyte of LDS that nobody reads, as many in flight as the counter allows.
__device__ __forceinline__ void gp_touch(const void* base, long long bytes, unsigned char* dst, int id, int n, int lane) {
  const int pieces = (int)(bytes >> 10);
  for (int k = id; k < pieces; k += n) {
    gp_load_lds(reinterpret_cast<const bf16_t*>(base), (unsigned)bytes, dst, lane * 16, (unsigned)k << 10);
    gp_wait_vm<60>();
  }
}

// workgroups per CU by LDS
template <int FN, int FM, int NA, int NB> constexpr int gp_per_cu() {
  return 160 * 1024 / ((NA * FN + NB * FM) * 32 * 128);
}

// LDS of a tile's rings: NA stages of W rows, then NB stages of X rows
template <int FN, int FM, int NA, int NB> constexpr int gp_lds_bytes() { return (NA * FN + NB * FM) * 32 * 128; }

// The K loop of a 32 FN x 32 FM tile (features x rows) in nt stages: load_w(i, slot, t) and
// load_x(i, slot, t) issue the wave's i-th kilobyte of stage t (nothing for t >= nt, but
// always one load instruction), acc[i][j] ends as C[feature 16 i + 4 (lane / 16) + r]
// [row 16 j + lane % 16] of the wave's corner.
template <int FN, int FM, int NA, int NB, typename LoadW, typename LoadX>
__device__ __forceinline__ void gp_loop(float4v (&acc)[FN][FM], const unsigned char* lds, int nt, int wn, int wm, int lane,
                                        LoadW&& load_w, LoadX&& load_x) {
  constexpr int TN = 16 * FN, TM = 16 * FM, BN = 2 * TN, BM = 2 * TM;
  constexpr int IA = BN / 32, IB = BM / 32;
  constexpr int XRING = NA * BN * 128;
  const int fr = lane & 15, fq = lane >> 4;
  // a fragment's place: rows 16 i apart keep the swizzle, the other K half is 64 bytes away
  const int swz = 16 * (fq ^ ((fr >> 1) & 7));
  const int abase = (wn * TN + fr) * 128 + swz, bbase = XRING + (wm * TM + fr) * 128 + swz;
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
  gp_wait_vm<(NA - 2) * IA + (NB - 1) * IB>();     // stage 0 is here
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
    gp_wait_vm<BEHIND>();                                // and its part of t + 1 has landed
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
}

// A wave's results to memory through its own part of LDS. An MFMA tile's accumulators hold
// four neighbouring features of one row per lane, so storing them directly makes every
// 8-byte piece of an instruction a line of its own (9000 x 3840 x 1280: 26 of 96 us went
// into the stores, 38 with a residual's loads). Instead the finished bf16 pieces go to LDS
// and leave as whole rows, 16 bytes a lane; with ADD the old rows are there already
// (GpRows) and value(i, j, o) finds them in o. FO: 16-wide feature blocks of the output; rows, cols:
// what of the wave's 16 FM x 16 FO corner exists (cols a multiple of 8).
template <int FO, int FM> struct GpRows {                  // a wave's corner as 16-byte chunks of rows
  static constexpr int LD = FO * 32 + 16;                   // bytes of a row in LDS
  static constexpr int CPR = FO * 2;                        // chunks of a row
  static constexpr int CH = 16 * FM * CPR / 64;             // chunks per lane
  static_assert(CH * 64 == 16 * FM * CPR, "chunks must split evenly over the lanes");
  u32x4 v[CH];
  __device__ __forceinline__ void load(const bf16_t* y, long ldy, int rows, int cols, int lane) {
#pragma unroll
    for (int k = 0; k < CH; ++k) {
      const int id = lane + 64 * k, r = min(id / CPR, rows - 1), c = id % CPR;
      if (rows > 0 && c * 8 < cols) v[k] = *reinterpret_cast<const u32x4*>(y + (size_t)r * ldy + c * 8);
    }
  }
  __device__ __forceinline__ void to_lds(unsigned char* my, int lane) const {
#pragma unroll
    for (int k = 0; k < CH; ++k) {
      const int id = lane + 64 * k;
      *reinterpret_cast<u32x4*>(my + (id / CPR) * LD + (id % CPR) * 16) = v[k];
    }
    __builtin_amdgcn_wave_barrier();
  }
};

template <int FO, int FM, bool ADD, typename Value>
__device__ __forceinline__ void gp_store(unsigned char* my, bf16_t* y, long ldy, int rows, int cols, int lane,
                                         Value&& value) {
  using R = GpRows<FO, FM>;
  constexpr int LD = R::LD, CPR = R::CPR, CH = R::CH;
  const int fr = lane & 15, fq = lane >> 4;
#pragma unroll
  for (int j = 0; j < FM; ++j) {
    unsigned char* row = my + (16 * j + fr) * LD + fq * 8;
#pragma unroll
    for (int i = 0; i < FO; ++i) {
      uint2* at = reinterpret_cast<uint2*>(row + i * 32);
      float o[4] = {0.f, 0.f, 0.f, 0.f};
      if constexpr (ADD) {
        const uint2 rv = *at;
        o[0] = bf2f(rv.x & 0xffff); o[1] = bf2f(rv.x >> 16);
        o[2] = bf2f(rv.y & 0xffff); o[3] = bf2f(rv.y >> 16);
      }
      value(i, j, o);
      *at = make_uint2(pack_bf16x2(o[0], o[1]), pack_bf16x2(o[2], o[3]));
    }
    __builtin_amdgcn_sched_barrier(0);   // a row block's accumulators at a time
  }
  __builtin_amdgcn_wave_barrier();
#pragma unroll
  for (int k = 0; k < CH; ++k) {
    const int id = lane + 64 * k, r = id / CPR, c = id % CPR;
    const u32x4 v = *reinterpret_cast<const u32x4*>(my + r * LD + c * 16);
    if (r < rows && c * 8 < cols) *reinterpret_cast<u32x4*>(y + (size_t)r * ldy + c * 8) = v;
  }
}
