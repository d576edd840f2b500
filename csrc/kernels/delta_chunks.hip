// The gated delta rule over a flat token batch, chunk by chunk on the f32 matrix
// cores: the long feeds of the recurrence
//
//   S <- g_t S;   u_t = beta_t (v_t - S^T k_t);   S <- S + k_t u_t^T;   o_t = S^T q_t
//
// (g_t a number per head or, CHAN, one per head and key channel) that
// delta_scan_kernel (delta_rule.hip) runs token by token. Feeds are cut into chunks
// of 16 tokens counted from their first one. Write P(i, j) for the product of the
// decays g_{j+1} .. g_i (per channel), P(i) for g_1 .. g_i, S for the state before the
// chunk. Unrolling the definition within the chunk,
//
//   u_i = beta_i (v_i - (P(i) k_i)^T S - sum_{j < i} A_ij u_j)   A_ij = sum_d k_i P(i, j) k_j
//   o_i = (P(i) q_i)^T S + sum_{j <= i} B_ij u_j                 B_ij = sum_d q_i P(i, j) k_j
//   S_end = P(16) S + sum_j (P(16, j) k_j) u_j^T
//
// The first line is a unit lower triangular system in the u_i. Forward substitution
// on its two right-hand sides separately gives u = U - W S with U from the values and
// W from the keys, and neither depends on S. So
//
// delta_local_kernel (a workgroup per chunk and head, all chunks in parallel) forms
// A and B (16 lanes per row i; the rows k_i P(i, j) and q_i P(i, j) are carried down
// from j = i by one multiplication per step, so no decay is ever divided by or taken
// to a negative power), and W, U by forward substitution, a thread per column;
//
// delta_pass_kernel (a workgroup per sequence, head and 16 value columns) walks the
// chunks in order with the state in MFMA accumulators: W S and (P q) S, u = U - W S,
// S <- P(16) S + K^T u, o = (P q) S + B u. Four waves split the key channels and
// add up W S through LDS, two more form the outputs behind them. With v_mfma_f32_16x16x4_f32 lane 16 g + m holds of an
// accumulator the rows 4 g + r (register r) of column m, and of a B operand row g of
// a step; taking the rows 4 g + r as step r's k indices makes an accumulator's
// registers the B operands of the next product as they are, and the A operand's four
// steps one 16-byte run.
//
// All products are exact f32 multiply-adds; the sums differ from the token-by-token
// kernel's in order only. Short chunks at a feed's end are filled with tokens that
// change nothing (k = q = v = 0, beta = 0, g = 1).
#include "seqmix.h"

#define DC_C 16

typedef unsigned dc_u4 __attribute__((ext_vector_type(4)));

struct DcParams {
  const float* act; long ld; int H, D, Dv, q_off, k_off, v_off, g_off, hpg;
  float* state; const int* slots; const int* cu_q; const int* pos; const float* tok;
  float* ws; float* o; int B;
  bool runs;                                                // rows of q, k and decays come in 16-byte pieces
};

// Workspace of one (chunk, head), DP the padded key size: W and P q in the order of the MFMA
// operand (per 16 channels a kilobyte: channels 4 g .. of token m at 16 g + m), (P(16, j) k_j)
// as [DP][16], P(16) [DP], U as [Dv][16], B [16][16]. The pass reads all of it, so every load
// there is a whole kilobyte: as rows of DP, W and P q came in 64-byte pieces.
__host__ __device__ __forceinline__ size_t dc_stride(int DP, int Dv) {
  return (size_t)49 * DP + 16 * Dv + 256;
}

template <int CTRL> __device__ __forceinline__ float dc_dpp(float v) {
  return __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), CTRL, 0xF, 0xF, true));
}
// the sum over each run of 16 lanes, in every lane of the run
__device__ __forceinline__ float dc_sum16(float v) {
  v += dc_dpp<0xB1>(v);
  v += dc_dpp<0x4E>(v);
  v += dc_dpp<0x141>(v);
  v += dc_dpp<0x140>(v);
  return v;
}

// What a workgroup that forms a chunk's block keeps in LDS (NT: key channels in units of 64, DP = 64 NT). A wave's
// stage is 64 columns of 16 tokens, a thread's four pieces of 16 bytes at 4 l + (piece ^ l / 4 % 4), so that neither
// the writes by columns nor the reads in order meet in a bank.
template <int NT> struct DcLocal {
  static constexpr int LD = 64 * NT + 4;
  float ks[DC_C][LD];
  union {
    struct { float qs[DC_C][LD], gs[DC_C][LD]; };
    float stage[4][64 * DC_C];                              // key columns: once qs is read (DP / 64 waves), values: gs as well
  };
  float A[DC_C][DC_C], B[DC_C][DC_C];
  float bs[DC_C];
};

// The block of head h's chunk of tokens t0 .. t0 + n - 1, by 256 threads. All of it is written in whole 64-byte runs.
// What bounds it is memory (2048 tokens, 16 heads of 128 x 128, a decay per channel: 67 MB of rows read, 70 written; 26 us
// at a large copy's rate), so the waves in flight: with the triangle's A in registers ahead of the substitution (166 a
// thread, three workgroups a CU), rows in 4-byte loads and columns stored in 16-byte pieces 64 bytes apart it took 39 us,
// with 55 registers, five workgroups and whole runs 30.
template <int NT, bool CHAN>
__device__ __forceinline__ void delta_local(const DcParams& p, DcLocal<NT>& s, float* ws, int t0, int n, int h, int tid) {
  constexpr int DP = 64 * NT;
  const int D = p.D, Dv = p.Dv, wave = __builtin_amdgcn_readfirstlane(tid >> 6), lane = tid & 63;
  const float* base = p.act + (size_t)t0 * p.ld;
  const __amdgpu_buffer_rsrc_t block = __builtin_amdgcn_make_buffer_rsrc(ws, 0, (int)(dc_stride(DP, Dv) * 4), 0x00020000);
  auto put = [&](int at, const float* v) {                  // four floats to entry at
    __builtin_amdgcn_raw_buffer_store_b128(dc_u4{__float_as_uint(v[0]), __float_as_uint(v[1]), __float_as_uint(v[2]), __float_as_uint(v[3])},
                                           block, at * 4, 0, 0);
  };
  // a thread's 16 numbers of column c0 + lane, as [column][16] from entry `to` on, of `cols` columns
  auto put_columns = [&](int to, int c0, int cols, const float (&x)[DC_C]) {
    float* st = s.stage[wave];
#pragma unroll
    for (int k = 0; k < 4; ++k) st_run<float, 4>(st + 16 * lane + 4 * (k ^ (lane >> 2 & 3)), x + 4 * k);
    __builtin_amdgcn_wave_barrier();
#pragma unroll
    for (int k = 0; k < 4; ++k) {
      const int l = 16 * k + (lane >> 2);
      float w[4];
      ld_run<float, 4>(st + 16 * l + 4 * ((lane ^ l >> 2) & 3), w);
      if (c0 + l < cols) put(to + (c0 + l) * DC_C + 4 * (lane & 3), w);
    }
    __builtin_amdgcn_wave_barrier();
  };
  {
    const float* qr = base + p.q_off + (size_t)(h / p.hpg) * D;
    const float* kr = base + p.k_off + (size_t)(h / p.hpg) * D;
    const float* gr = CHAN ? base + p.g_off + (size_t)h * D : nullptr;
    const float* tr = p.tok + ((size_t)t0 * p.H + h) * 2;
    if (p.runs) {                                           // whole rows of 16-byte pieces
#pragma unroll
      for (int j = 0; j < NT; ++j) {
        const int i = (tid + 256 * j) / (16 * NT), d = (tid + 256 * j) % (16 * NT) * 4;
        const size_t row = (size_t)(i < n ? i : 0) * p.ld;
        const bool ok = i < n && d < D;
        float q[4] = {0.f, 0.f, 0.f, 0.f}, k[4] = {0.f, 0.f, 0.f, 0.f}, g[4] = {1.f, 1.f, 1.f, 1.f};
        if (ok) {
          ld_run<float, 4>(qr + row + d, q);
          ld_run<float, 4>(kr + row + d, k);
          if constexpr (CHAN) ld_run<float, 4>(gr + row + d, g);
          else g[0] = g[1] = g[2] = g[3] = tr[(size_t)i * p.H * 2];
        }
        st_run<float, 4>(&s.qs[i][d], q);
        st_run<float, 4>(&s.ks[i][d], k);
        st_run<float, 4>(&s.gs[i][d], g);
      }
    } else {
#pragma unroll 4
      for (int j = 0; j < DC_C * DP / 256; ++j) {
        const int i = (tid + 256 * j) / DP, d = (tid + 256 * j) % DP;
        const bool ok = i < n && d < D;
        const size_t row = (size_t)(i < n ? i : 0) * p.ld;
        s.qs[i][d] = ok ? qr[row + d] : 0.f;
        s.ks[i][d] = ok ? kr[row + d] : 0.f;
        s.gs[i][d] = ok ? (CHAN ? gr[row + d] : tr[(size_t)i * p.H * 2]) : 1.f;
      }
    }
    if (tid < DC_C) s.bs[tid] = tid < n ? tr[(size_t)tid * p.H * 2 + 1] : 0.f;
  }
  __syncthreads();
  // A and B: row i on 16 lanes, lane q with the channels 64 m + 4 q ..
  const int i = tid >> 4, q = tid & 15;
  float a[NT][4], c[NT][4];
#pragma unroll
  for (int m = 0; m < NT; ++m) {
    ld_run<float, 4>(&s.ks[i][64 * m + 4 * q], a[m]);
    ld_run<float, 4>(&s.qs[i][64 * m + 4 * q], c[m]);
  }
#pragma unroll 4
  for (int j = DC_C - 1; j >= 0; --j) {
    float sa = 0.f, sb = 0.f;
    if (j <= i) {
#pragma unroll
      for (int m = 0; m < NT; ++m) {
        float k[4], g[4];
        ld_run<float, 4>(&s.ks[j][64 * m + 4 * q], k);
        ld_run<float, 4>(&s.gs[j][64 * m + 4 * q], g);
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          sa += a[m][e] * k[e];
          sb += c[m][e] * k[e];
          a[m][e] *= g[e];
          c[m][e] *= g[e];
        }
      }
    }
    sa = dc_sum16(sa);
    sb = dc_sum16(sb);
    if (q == 0) {
      s.A[i][j] = j < i ? sa : 0.f;
      s.B[i][j] = j <= i ? sb : 0.f;
    }
  }
  // a = P(i) k_i, c = P(i) q_i now
#pragma unroll
  for (int m = 0; m < NT; ++m) put(16 * DP + (4 * m + q / 4) * 256 + (16 * (q % 4) + i) * 4, c[m]);
  __syncthreads();
  // P(16, j) k_j and P(16), a thread per channel
  if (wave < NT) {
    float r = 1.f, kk[DC_C];
#pragma unroll
    for (int j = DC_C - 1; j >= 0; --j) {
      kk[j] = s.ks[j][tid] * r;
      r *= s.gs[j][tid];
    }
    put_columns(32 * DP, 64 * wave, DP, kk);
    __builtin_amdgcn_raw_buffer_store_b32(__float_as_uint(r), block, (48 * DP + tid) * 4, 0, 0);
  }
  __syncthreads();
#pragma unroll
  for (int m = 0; m < NT; ++m) st_run<float, 4>(&s.ks[i][64 * m + 4 * q], a[m]);
  if (wave == 3) {
    float w[4];
    ld_run<float, 4>(&s.B[0][0] + 4 * lane, w);
    put(49 * DP + 16 * Dv + 4 * lane, w);
  }
  __syncthreads();
  // forward substitution, a thread per column of [P k | v]
  for (int c0 = 64 * wave; c0 < DP + Dv; c0 += 256) {
    const int col = c0 + lane;
    const bool key = c0 < DP;
    float x[DC_C];
    const float* vr = base + p.v_off + (size_t)h * Dv + min(max(col - DP, 0), Dv - 1);
#pragma unroll
    for (int t = 0; t < DC_C; ++t)
      x[t] = key ? s.ks[t][col] : (t < n ? vr[(size_t)t * p.ld] : 0.f);
#pragma unroll
    for (int t = 0; t < DC_C; ++t) {
      float y = x[t];
#pragma unroll
      for (int j = 0; j < t; ++j) y -= s.A[t][j] * x[j];
      x[t] = s.bs[t] * y;
    }
    if (key) {
#pragma unroll
      for (int t = 0; t < DC_C; ++t) s.ks[t][col] = x[t];    // a column is its thread's own
    } else {
      put_columns(49 * DP, c0 - DP, Dv, x);
    }
  }
  __syncthreads();
#pragma unroll
  for (int j = 0; j < NT; ++j) {
    const int at = tid + 256 * j, l = at & 63;
    float w[4];
    ld_run<float, 4>(&s.ks[l & 15][16 * (at >> 6) + 4 * (l >> 4)], w);
    put(at * 4, w);
  }
}

template <int NT, bool CHAN>
__global__ __launch_bounds__(256) void delta_local_kernel(DcParams p) {
  __shared__ __attribute__((aligned(16))) DcLocal<NT> s;
  int b, t0, n;
  if (!seq_chunk<DC_C>(p.cu_q, p.B, blockIdx.x, b, t0, n)) return;
  delta_local<NT, CHAN>(p, s, p.ws + ((size_t)blockIdx.x * p.H + blockIdx.y) * dc_stride(64 * NT, p.Dv), t0, n, blockIdx.y, threadIdx.x);
}

// Every wave of the workgroup is here and its LDS writes are visible; global loads stay in
// flight. Called from both roles of delta_pass_kernel, the same number of times by each.
__device__ __forceinline__ void dc_barrier() {
  asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
  __builtin_amdgcn_s_barrier();
  asm volatile("" ::: "memory");
}

// The chunks of a sequence are a serial chain: X = W S, u = U - X, S <- P S + K^T u, with X
// added up over the waves in between. Nothing but that may stand in its way: waves 0 - 3 run
// the chain, with (P q) S while X travels through LDS, and leave their parts of X
// and of (P q) S there; waves 4 and 5 take every other chunk, add up, form the outputs and
// store them (DC_RING: what chunk c leaves is read before the barrier of chunk c + 2). Loads
// are buffer loads, a chunk's block as the buffer: its address is a scalar and a lane's offset
// stays. As four waves that did it all, with addresses per lane, a chunk took 1950 cycles, 800
// of them MFMAs; now 1350 (2048 tokens, 16 heads of 128 x 128: 119 -> 79 us).
#define DC_RING 3

template <int NT>
__global__ __launch_bounds__(384, 2) void delta_pass_kernel(DcParams p) {
  constexpr int DP = 64 * NT;
  __shared__ float4v xs[DC_RING][4][64], ys[DC_RING][4][64];
  const int b = blockIdx.x, h = blockIdx.y, e0 = blockIdx.z * 16;
  const int q0 = __builtin_amdgcn_readfirstlane(p.cu_q[b]);
  const int len = __builtin_amdgcn_readfirstlane(p.cu_q[b + 1]) - q0;
  if (len <= 0) return;
  const int before = __builtin_amdgcn_readfirstlane(seq_chunks_before<DC_C>(p.cu_q, b));
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int lane = threadIdx.x & 63, m = lane & 15, g = lane >> 4;
  const int D = p.D, Dv = p.Dv, nc = (len + DC_C - 1) / DC_C;
  const bool col = e0 + m < Dv;
  const int ec = min(e0 + m, Dv - 1);
  const size_t st = dc_stride(DP, Dv), step = st * p.H;
  const float* ws = p.ws + ((size_t)before * p.H + h) * st;
  const float4v zero = {0.f, 0.f, 0.f, 0.f};
  // 16 bytes a lane of a chunk's block: part (floats) and block are scalars, at (bytes) the lane's
  auto load = [&](const float* block, int part, unsigned at) {
    typedef unsigned u32x4 __attribute__((ext_vector_type(4)));
    const u32x4 v = __builtin_amdgcn_raw_buffer_load_b128(
        __builtin_amdgcn_make_buffer_rsrc(const_cast<float*>(block), 0, (int)(st * 4), 0x00020000), at, part * 4, 0);
    return __builtin_bit_cast(float4v, v);
  };
  const unsigned l16 = lane * 16, g16 = g * 16, k16 = (m * DC_C + 4 * g) * 4, u16 = (ec * DC_C + 4 * g) * 4;
  auto sum = [&](const float4v (&v)[4][64]) { return (v[0][lane] + v[1][lane]) + (v[2][lane] + v[3][lane]); };
  int slot = 0;
  auto next = [](int at) { return at + 1 == DC_RING ? 0 : at + 1; };
  if (wave < 4) {
    // state [slots, H, Dv, D]: the wave's tile t holds the channels 16 (NT wave + t) ..
    float* Sg = p.state + (((size_t)p.slots[b] * p.H + h) * Dv + ec) * D;
    const bool fresh = p.pos[q0] == 0;
    float4v S[NT];
#pragma unroll
    for (int t = 0; t < NT; ++t)
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int d = 16 * (NT * wave + t) + 4 * g + r;
        S[t][r] = !fresh && d < D ? Sg[d] : 0.f;
      }
    struct Set { float4v W[NT], Q[NT], K[NT], G[NT], U; };
    const float* block = ws;                // of the next chunk to fetch, then again the last one's:
    int more = nc - 1;                      // loads in flight are counted, so none is left out
    auto advance = [&]() {
      block += more > 0 ? step : 0;
      --more;
    };
    // A set's loads one by one: W and P q, two per tile, then K and P, then U. As a burst behind
    // the MFMAs they queued up before the cache and took 20 us of a pass of 2048 tokens.
    auto fetch = [&](Set& f, int k) {
      const int t = (k % (2 * NT)) / 2, d0 = 16 * (NT * wave + t);
      if (k == 4 * NT) f.U = load(block, 49 * DP, u16);
      else if (k < 2 * NT && k % 2 == 0) f.W[t] = load(block, 16 * d0, l16);
      else if (k < 2 * NT) f.Q[t] = load(block, 16 * DP + 16 * d0, l16);
      else if (k % 2 == 0) f.K[t] = load(block, 32 * DP + 16 * d0, k16);
      else f.G[t] = load(block, 48 * DP + d0, g16);
      __builtin_amdgcn_sched_barrier(0);
    };
    auto fetch_all = [&](Set& f) {
#pragma unroll
      for (int k = 0; k <= 4 * NT; ++k) fetch(f, k);
      advance();
    };
    // one chunk from f, and the loads of a later one into its set n
    auto chunk = [&](Set& f, Set& n) {
      float4v X = zero, Y = zero;
#pragma unroll
      for (int k = 0; k < 4 * NT; ++k) {
        X = __builtin_amdgcn_mfma_f32_16x16x4f32(f.W[k / 4][k % 4], S[k / 4][k % 4], X, 0, 0, 0);
        if (k % 2 == 1) fetch(n, k / 2);
      }
      xs[slot][wave][lane] = X;
#pragma unroll
      for (int k = 0; k < 4 * NT; ++k)
        Y = __builtin_amdgcn_mfma_f32_16x16x4f32(f.Q[k / 4][k % 4], S[k / 4][k % 4], Y, 0, 0, 0);
      __builtin_amdgcn_sched_barrier(0);
      dc_barrier();
      float4v x[4];
#pragma unroll
      for (int w = 0; w < 4; ++w) x[w] = xs[slot][w][lane];
      fetch(n, 4 * NT);
      const float4v u = f.U - ((x[0] + x[1]) + (x[2] + x[3]));
#pragma unroll
      for (int t = 0; t < NT; ++t) S[t] *= f.G[t];
#pragma unroll
      for (int k = 0; k < 4 * NT; ++k) {
        S[k % NT] = __builtin_amdgcn_mfma_f32_16x16x4f32(f.K[k % NT][k / NT], u[k / NT], S[k % NT], 0, 0, 0);
        if (k % 2 == 1) fetch(n, 2 * NT + k / 2);
      }
      advance();
      ys[slot][wave][lane] = Y;
      slot = next(slot);
    };
    // the inputs of NS - 1 chunks in flight: a chunk takes less time than a trip to memory
    constexpr int NS = NT <= 2 ? 4 : 2;
    Set f0, f1, f2, f3;
    fetch_all(f0);
    int c = 0;
    if constexpr (NS == 4) {
      fetch_all(f1);
      fetch_all(f2);
      for (; c + 3 < nc; c += 4) {
        chunk(f0, f3);
        chunk(f1, f0);
        chunk(f2, f1);
        chunk(f3, f2);
      }
      if (c < nc) chunk(f0, f3);
      if (c + 1 < nc) chunk(f1, f0);
      if (c + 2 < nc) chunk(f2, f1);
    } else {
      for (; c + 1 < nc; c += 2) {
        chunk(f0, f1);
        chunk(f1, f0);
      }
      if (c < nc) chunk(f0, f1);
    }
    dc_barrier();
    if (col)
#pragma unroll
      for (int t = 0; t < NT; ++t)
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          const int d = 16 * (NT * wave + t) + 4 * g + r;
          if (d < D) Sg[d] = S[t][r];
        }
  } else {
    const int ldo = p.H * Dv, turn = wave - 4;
    unsigned ro[4];                           // of a lane's entries in a chunk's rows; past every buffer if its column is none
#pragma unroll
    for (int r = 0; r < 4; ++r) ro[r] = col ? ((4u * g + r) * ldo + m) * 4 : 0xfffffff0u;
    struct Set { float4v U, B; };
    auto fetch = [&](Set& f, int c) {
      const float* block = ws + (size_t)min(c, nc - 1) * step;
      f.U = load(block, 49 * DP, u16);
      f.B = load(block, 49 * DP + 16 * Dv, k16);
      __builtin_amdgcn_sched_barrier(0);
    };
    int passed = 0;                           // barriers behind this wave, nc + 1 in the end
    auto pass = [&](int upto) {
      for (upto = min(upto, nc + 1); passed < upto; ++passed) dc_barrier();
    };
    auto chunk = [&](Set& f, int c) {
      pass(c + 2);                            // chunk c has left its parts
      slot = min(c, nc - 1) % DC_RING;        // (past the last chunk: that one again, unstored)
      const float4v u = f.U - sum(xs[slot]);
      float4v Y = sum(ys[slot]);
#pragma unroll
      for (int r = 0; r < 4; ++r) Y = __builtin_amdgcn_mfma_f32_16x16x4f32(f.B[r], u[r], Y, 0, 0, 0);
      // rows past the feed's end are past the buffer's, and are not stored
      const int rows = min(len - c * DC_C, DC_C);
      const auto out = __builtin_amdgcn_make_buffer_rsrc(
          p.o + (size_t)(q0 + min(c, nc - 1) * DC_C) * ldo + (size_t)h * Dv + e0, 0, rows > 0 ? ((rows - 1) * ldo + min(16, Dv - e0)) * 4 : 0,
          0x00020000);
#pragma unroll
      for (int r = 0; r < 4; ++r) __builtin_amdgcn_raw_buffer_store_b32(__float_as_uint(Y[r]), out, ro[r], 0, 0);
      fetch(f, c + 8);
    };
    Set f0, f1, f2, f3;
    fetch(f0, turn);
    fetch(f1, turn + 2);
    fetch(f2, turn + 4);
    fetch(f3, turn + 6);
    for (int c = turn; c < nc; c += 8) {
      chunk(f0, c);
      chunk(f1, c + 2);
      chunk(f2, c + 4);
      chunk(f3, c + 6);
    }
    pass(nc + 1);
  }
}

extern "C" long loqa_delta_chunks_ws(int H, int D, int Dv, int B, int T) {
  const int NT = D <= 64 ? 1 : (D <= 128 ? 2 : 4);
  return (long)(T / DC_C + B) * H * (long)dc_stride(64 * NT, Dv);
}

// The arguments of loqa_delta_scan; ws: f32, loqa_delta_chunks_ws entries.
extern "C" int loqa_delta_chunks(const void* act, long ld, int H, int D, int Dv, int q_off, int k_off,
                                 int v_off, int g_off, int hpg, void* state, const void* state_slots,
                                 const void* cu_q, const void* positions, const void* tok, void* ws,
                                 void* o, int B, int T, hipStream_t st) {
  if (T <= 0 || B <= 0) return 0;
  if (H <= 0 || D <= 0 || D > 256 || Dv <= 0 || hpg <= 0 || H % hpg || !tok || !ws)
    return (int)hipErrorInvalidValue;
  const DcParams p{(const float*)act, ld, H, D, Dv, q_off, k_off, v_off, g_off, hpg, (float*)state,
                   (const int*)state_slots, (const int*)cu_q, (const int*)positions,
                   (const float*)tok, (float*)ws, (float*)o, B,
                   D % 4 == 0 && ld % 4 == 0 && q_off % 4 == 0 && k_off % 4 == 0 && (g_off < 0 || g_off % 4 == 0) && ((size_t)act & 15) == 0};
  const dim3 gl(T / DC_C + B, H), gp(B, H, (Dv + 15) / 16);
#define GO(NT)                                                                                   \
  do {                                                                                           \
    if (g_off >= 0)                                                                              \
      hipLaunchKernelGGL((delta_local_kernel<NT, true>), gl, dim3(256), 0, st, p);               \
    else                                                                                         \
      hipLaunchKernelGGL((delta_local_kernel<NT, false>), gl, dim3(256), 0, st, p);              \
    hipLaunchKernelGGL(delta_pass_kernel<NT>, gp, dim3(384), 0, st, p);                          \
  } while (0)
  if (D <= 64) GO(1); else if (D <= 128) GO(2); else GO(4);
#undef GO
  return (int)hipGetLastError();
}
