// MFMA decode GEMM: out[M,N] = x[M,K] @ W[N,K]^T (+bias), M <= 64 per pass.
//
// A scalar GEMV is VALU-bound at M >= 4: every weight costs ~2 VALU ops per
// output row. Here one v_mfma_f32_16x16x32_bf16 covers a 16(M)x16(N)x32(K) tile
// and up to 4 M-tiles stack, so one weight read serves up to 64 batch rows.
// Fragment layout: lane l holds A[row=l&15][k=(l>>4)*8+j],
// B[col=l&15][k=(l>>4)*8+j], C[col=l&15][row=(l>>4)*4+r].
//
// x goes through LDS with coalesced full-line loads; bf16 weights are read in
// fragment shape, int8 / int4 weights in the packed layouts that give each lane
// 16 B of two (four) 32-wide steps. gridDim.y splits K (fp32 atomics into a
// scratch, combined by the consumer or by a convert/bias kernel).
#include "common.h"

namespace dnet {

using bf16x8 = __attribute__((ext_vector_type(8))) __bf16;
using f32x4 = __attribute__((ext_vector_type(4))) float;

// silu(g) * u
__device__ __forceinline__ float swiglu_of(const float g, const float u) {
  return g / (1.f + __expf(-g)) * u;
}

// bf16 weights. MT: number of stacked 16-row A tiles (M <= 16*MT). GLU: w holds
// N gate rows and N up rows, a wave computes 16 columns of both and stores
// silu(gate) * up (no splits): the activation as a kernel of its own, and its
// launch, are gone.
template <int MT, bool GLU>
__global__ void gemm_m16_kernel(const short* __restrict__ x,
                                const short* __restrict__ w,
                                const short* __restrict__ bias,
                                short* __restrict__ out,        // SPLITK==1
                                float* __restrict__ out_f32,    // SPLITK>1
                                const int M, const int K, const int N,
                                const int splitk) {
  constexpr int XT = 1024 / MT;        // k per x tile (LDS ~33 KB, 4 blocks/CU)
  constexpr int SE = XT + 8;           // row stride in bf16 elems (16B pad)
  __shared__ short x_lds[16 * MT * SE];
  const int wave = threadIdx.x / kWave;
  const int lane = threadIdx.x & (kWave - 1);
  const int n0 = (blockIdx.x * 4 + wave) * 16;
  // Block-wide barriers: OOB waves must stay alive; their stores are
  // skipped at the end.
  const int row = lane & 15;          // A row within a tile, B col
  const int ks = (lane >> 4) * 8;     // k-offset of this lane's 8-elem slice
  const int n_w = min(n0 + row, N - 1);     // this lane's W row

  const int pairs = K / 64;
  const int pp = pairs / splitk;
  const int p_begin = blockIdx.y * pp;
  const int p_end = (blockIdx.y == splitk - 1) ? pairs : p_begin + pp;

  constexpr int NW = GLU ? 2 : 1;
  f32x4 acc[NW][MT][2];
#pragma unroll
  for (int g = 0; g < NW; ++g)
#pragma unroll
    for (int t = 0; t < MT; ++t)
#pragma unroll
      for (int u = 0; u < 2; ++u) acc[g][t][u] = {0.f, 0.f, 0.f, 0.f};

  const short* wrow[NW];
#pragma unroll
  for (int g = 0; g < NW; ++g) wrow[g] = w + ((int64_t)g * N + n_w) * K;

  for (int k0 = p_begin * 64; k0 < p_end * 64; k0 += XT) {
    const int tk = min(XT, p_end * 64 - k0);
    // raw barrier (lgkmcnt only): __syncthreads() would wait vmcnt(0) and
    // drain the in-flight weight stream at EVERY x-tile boundary — at MT=4
    // (XT=256) that is a full memory-pipeline restart every 4 pairs
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    asm volatile("s_barrier" ::: "memory");
    for (int idx = threadIdx.x; idx < 16 * MT * (tk / 8); idx += 256) {
      const int r = idx / (tk / 8);
      const int vec = idx % (tk / 8);
      // rows >= M read a clamped row; their C rows are never stored
      *reinterpret_cast<short8*>(&x_lds[r * SE + vec * 8]) =
          *reinterpret_cast<const short8*>(
              &x[(int64_t)min(r, M - 1) * K + k0 + vec * 8]);
    }
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    asm volatile("s_barrier" ::: "memory");
    const short* arow = &x_lds[row * SE];
    int pl = 0;
    const int pl_end = tk / 64;
    for (; pl + 4 <= pl_end; pl += 4) {  // 4 pairs, all weight loads first
      bf16x8 wb[NW][4][2];
#pragma unroll
      for (int g = 0; g < NW; ++g)
#pragma unroll
        for (int u = 0; u < 4; ++u) {
          const int p = (k0 / 64) + pl + u;
          wb[g][u][0] =
              *reinterpret_cast<const bf16x8*>(&wrow[g][p * 64 + ks]);
          wb[g][u][1] =
              *reinterpret_cast<const bf16x8*>(&wrow[g][p * 64 + 32 + ks]);
        }
#pragma unroll
      for (int u = 0; u < 4; ++u)
#pragma unroll
        for (int t = 0; t < MT; ++t) {
          const short* at = arow + t * 16 * SE;
          const bf16x8 a0 =
              *reinterpret_cast<const bf16x8*>(&at[(pl + u) * 64 + ks]);
          const bf16x8 a1 =
              *reinterpret_cast<const bf16x8*>(&at[(pl + u) * 64 + 32 + ks]);
#pragma unroll
          for (int g = 0; g < NW; ++g) {
            acc[g][t][0] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(
                a0, wb[g][u][0], acc[g][t][0], 0, 0, 0);
            acc[g][t][1] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(
                a1, wb[g][u][1], acc[g][t][1], 0, 0, 0);
          }
        }
    }
    for (; pl < pl_end; ++pl) {
      const int p = (k0 / 64) + pl;
      bf16x8 b0[NW], b1[NW];
#pragma unroll
      for (int g = 0; g < NW; ++g) {
        b0[g] = *reinterpret_cast<const bf16x8*>(&wrow[g][p * 64 + ks]);
        b1[g] = *reinterpret_cast<const bf16x8*>(&wrow[g][p * 64 + 32 + ks]);
      }
#pragma unroll
      for (int t = 0; t < MT; ++t) {
        const short* at = arow + t * 16 * SE;
        const bf16x8 a0 = *reinterpret_cast<const bf16x8*>(&at[pl * 64 + ks]);
        const bf16x8 a1 = *reinterpret_cast<const bf16x8*>(&at[pl * 64 + 32 + ks]);
#pragma unroll
        for (int g = 0; g < NW; ++g) {
          acc[g][t][0] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(
              a0, b0[g], acc[g][t][0], 0, 0, 0);
          acc[g][t][1] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(
              a1, b1[g], acc[g][t][1], 0, 0, 0);
        }
      }
    }
  }
  // the last products' results are read below, behind a branch: past their
  // latency in any case
  asm volatile("s_nop 15" ::: "memory");

  // C write: lane covers col = n0 + (lane&15), rows (lane>>4)*4 + 0..3 of
  // each stacked tile.
  const int n = n0 + (lane & 15);
  if (n >= N) return;
#pragma unroll
  for (int t = 0; t < MT; ++t) {
    const f32x4 a2 = acc[0][t][0] + acc[0][t][1];
    f32x4 up = {0.f, 0.f, 0.f, 0.f};
    if (GLU) up = acc[NW - 1][t][0] + acc[NW - 1][t][1];
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const int m = t * 16 + (lane >> 4) * 4 + r;
      if (m >= M) continue;
      if (GLU) {
        out[(int64_t)m * N + n] = f2bits(swiglu_of(a2[r], up[r]));
      } else if (splitk > 1) {
        atomicAdd(out_f32 + (int64_t)m * N + n, a2[r]);
      } else {
        float v = a2[r];
        if (bias != nullptr) v += bits2f(bias[n]);
        out[(int64_t)m * N + n] = f2bits(v);
      }
    }
  }
}

// bf16 weights for few rows or little work: a workgroup owns 16 NC columns and
// its NW waves divide the inner dimension (the kernel above divides columns and
// needs atomics to divide the rest). No staging and no barrier before the one
// fold at the end: weights go from memory to registers, U neighbouring 64 B
// pieces of each row, x in fragment shape from L2; the next group of pieces is
// in flight while one is multiplied. Products start from zero and the vector
// unit adds them up (the matrix core's own running sum rounds less exactly).
// GLU as above (NF = 2 NC: gate columns, then up columns).
// Bound by the weight stream, below 10 MB by latency and launch. Measured,
// MI355X, one row, with the zeroing and combining kernels that the splits
// needed -> here:
// 6144 x 4096 15.7 us -> 13.1 (3.8 TB/s), 4096 x 14336 28.6 -> 24.0 (4.9 TB/s),
// 2 x 14336 x 4096 with swiglu 51.5 -> 42.7 (5.5 TB/s), 768 x 768 5.4 -> 2.7.
template <int MT, int NF, int NW, int U, bool GLU>
__global__ __launch_bounds__(NW * 64) void gemm_b16_kernel(
    const short* __restrict__ x, const short* __restrict__ w,
    const short* __restrict__ bias, short* __restrict__ out, const int M,
    const int K, const int N) {
  constexpr int NC = GLU ? NF / 2 : NF;
  __shared__ f32x4 part[NW - 1][MT * NF][64];
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int lane = threadIdx.x & 63;
  const int c = lane & 15, hi = lane >> 4;
  const int n0 = blockIdx.x * (16 * NC);
  const short* wp[NF];
#pragma unroll
  for (int f = 0; f < NF; ++f)
    wp[f] = w + ((int64_t)(f / NC) * N + min(n0 + (f % NC) * 16 + c, N - 1)) *
                    K + hi * 8;
  const short* xp[MT];      // rows >= M repeat the last one, never stored
#pragma unroll
  for (int m = 0; m < MT; ++m)
    xp[m] = x + (int64_t)min(m * 16 + c, M - 1) * K + hi * 8;
  f32x4 acc[MT][NF];
#pragma unroll
  for (int m = 0; m < MT; ++m)
#pragma unroll
    for (int f = 0; f < NF; ++f) acc[m][f] = {0.f, 0.f, 0.f, 0.f};
  struct Batch { bf16x8 w[U][NF], x[U][MT]; };
  auto load = [&](Batch& q, const int s) {
#pragma unroll
    for (int f = 0; f < NF; ++f)
#pragma unroll
      for (int u = 0; u < U; ++u)
        q.w[u][f] = *reinterpret_cast<const bf16x8*>(wp[f] + (s + u) * 32);
#pragma unroll
    for (int m = 0; m < MT; ++m)
#pragma unroll
      for (int u = 0; u < U; ++u)
        q.x[u][m] = *reinterpret_cast<const bf16x8*>(xp[m] + (s + u) * 32);
  };
  auto mul = [&](const Batch& q) {
#pragma unroll
    for (int m = 0; m < MT; ++m)
#pragma unroll
      for (int f = 0; f < NF; ++f) {
        f32x4 p = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int u = 0; u < U; ++u)
          p = __builtin_amdgcn_mfma_f32_16x16x32_bf16(q.x[u][m], q.w[u][f], p,
                                                      0, 0, 0);
#pragma unroll
        for (int r = 0; r < 4; ++r) acc[m][f][r] += p[r];
      }
  };
  const int total = K / 32;
  const int groups = total / (NW * U);
  auto place = [&](int g) { return (g * NW + wave) * U; };
  if (groups > 0) {
    Batch q0, q1;
    load(q0, place(0));
    int g = 0;
    for (; g + 2 < groups; g += 2) {
      load(q1, place(g + 1));
      __builtin_amdgcn_sched_barrier(0);
      mul(q0);
      load(q0, place(g + 2));
      __builtin_amdgcn_sched_barrier(0);
      mul(q1);
    }
    if (g + 1 < groups) {
      load(q1, place(g + 1));
      __builtin_amdgcn_sched_barrier(0);
      mul(q0);
      mul(q1);
    } else {
      mul(q0);
    }
  }
  for (int s = groups * NW * U + wave; s < total; s += NW) {
    bf16x8 xv[MT];
#pragma unroll
    for (int m = 0; m < MT; ++m)
      xv[m] = *reinterpret_cast<const bf16x8*>(xp[m] + s * 32);
#pragma unroll
    for (int f = 0; f < NF; ++f) {
      const bf16x8 wv = *reinterpret_cast<const bf16x8*>(wp[f] + s * 32);
#pragma unroll
      for (int m = 0; m < MT; ++m) {
        f32x4 p = {0.f, 0.f, 0.f, 0.f};
        p = __builtin_amdgcn_mfma_f32_16x16x32_bf16(xv[m], wv, p, 0, 0, 0);
#pragma unroll
        for (int r = 0; r < 4; ++r) acc[m][f][r] += p[r];
      }
    }
  }
  if (wave != 0)
#pragma unroll
    for (int m = 0; m < MT; ++m)
#pragma unroll
      for (int f = 0; f < NF; ++f)
        part[wave - 1][m * NF + f][lane] = acc[m][f];
  __syncthreads();
  if (wave != 0) return;
#pragma unroll
  for (int m = 0; m < MT; ++m) {
#pragma unroll
    for (int f = 0; f < NF; ++f)
#pragma unroll
      for (int v = 0; v < NW - 1; ++v) {
        const f32x4 p = part[v][m * NF + f][lane];
#pragma unroll
        for (int r = 0; r < 4; ++r) acc[m][f][r] += p[r];
      }
#pragma unroll
    for (int f = 0; f < NC; ++f) {
      const int n = n0 + f * 16 + c;
      if (n >= N) continue;
      const float bv = bias != nullptr ? bits2f(bias[n]) : 0.f;
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int row = m * 16 + hi * 4 + r;
        if (row >= M) continue;
        out[(int64_t)row * N + n] =
            f2bits(GLU ? swiglu_of(acc[m][f][r], acc[m][NC + f][r])
                       : acc[m][f][r] + bv);
      }
    }
  }
}

// Whether gemm_b16_kernel takes the product (`rows` weight rows, 2 N with glu).
// Its x comes from L2 once per 16 columns, so its line is where x outweighs
// what it saves (us, the staged kernel with its extra launches -> this one):
// 1 row 28672 x 4096 with swiglu 51.5 -> 42.7, 6144 x 4096 15.7 -> 13.1,
// 4096 x 14336 28.6 -> 24.0, 2304 x 768 5.8 -> 3.5; 16 rows 4096 x 4096 14.6 ->
// 11.5, but 6144 x 4096 17.5 -> 18.3 and 4096 x 14336 30.9 -> 34.7; 32 rows
// 768 x 3072 12.0 -> 10.3; 64 rows 768 x 768 11.3 -> 5.9, but 768 x 3072 15.5 ->
// 16.1. Many columns alone fill the chip without splits: 1 row 128256 x 4096
// 193 -> 199.
static bool on_b16(int64_t M, int64_t rows, int64_t K, bool glu) {
  if (rows > 16 * 1024) return glu && M <= 16;
  if (M <= 8) return true;
  if (M <= 16) return rows * K <= 20 * 1024 * 1024;
  return rows * K <= 6 * 1024 * 1024 && K <= (M <= 32 ? 4096 : 2048);
}

static void launch_b16(const short* x, const short* w, const short* bias,
                       short* out, int M, int K, int N, bool glu,
                       hipStream_t st) {
#define LB(MM, FF, WW, UU, GL)                                              \
  hipLaunchKernelGGL((gemm_b16_kernel<MM, FF, WW, UU, GL>),                 \
                     dim3((unsigned)cdiv(N, 16 * (GL ? FF / 2 : FF))),      \
                     dim3(WW * 64), 0, st, x, w, bias, out, M, K, N)
  // 8 waves per workgroup where the inner dimension has work for them (from 2
  // groups of pieces each) and the columns alone leave compute units idle
  const bool deep = K >= 2048;
  if (glu) {
    if (M > 32) LB(4, 2, 4, 2, true);
    else if (M > 16) LB(2, 2, 4, 2, true);
    else if (deep) LB(1, 2, 8, 4, true);
    else LB(1, 2, 4, 4, true);
  } else {
    if (M > 32) LB(4, 1, 4, 4, false);
    else if (M > 16) LB(2, 1, 4, 4, false);
    else if (deep) LB(1, 1, 8, 4, false);
    else LB(1, 1, 4, 4, false);
  }
#undef LB
}

// ---------------------------------------------------------------------------
// int8 / int4 weights (packed layouts), up to 64 rows.
//
// The weight stream bounds it; what has to stay out of its way are the
// conversion to bf16, the reads of x from LDS and the barriers.
//   * 4 waves, each with 16 NF columns of its own and all rows: a fragment of x
//     read from LDS serves NF fragments of weights.
//   * x goes through LDS in chunks of KC columns, two of them: the next chunk's
//     x and weights are loaded into registers before the products of this one,
//     x is written to the other buffer after them, one barrier per chunk. The
//     barrier waits for LDS only, the weights stay in flight across it.
//   * weights are multiplied as whole numbers (exact in bf16), their scale
//     applies to the fp32 sums of one 16 B load's width (64 or 128 columns):
//     one vector operation per four results instead of one per weight, and no
//     rounding of scale x weight.
//   * the inner dimension is split by chunks over gridDim.y where the columns
//     alone leave CUs idle (fp32 atomics into the scratch).
// Measured, MI355X, 5120 x 55296 / 27648 x 5120 / 5120 x 152064 (K x N):
// int8, 8 rows 68 -> 67, 46 -> 38, 175 -> 174 us (4.2, 3.8, 4.5 TB/s); 64 rows
// 108 -> 98, 66 -> 56, 267 -> 237 us; int4, 8 rows 56 -> 44, 40 -> 26, 134 ->
// 116 us; 64 rows 91 -> 79, 57 -> 46, 230 -> 190 us. Before: one 16-column
// fragment per wave, a drained round trip per chunk or two, weights rounded to
// bf16 after scaling (error of the fp32 sums against 64 bits 1.6e-3, now 1e-7).
// Reading a row's scales by one load per chunk instead of one per weight load
// was a third of the time. What remains is a rate per CU and chunk that does
// not depend on the number of waves.
// Columns past the end of K repeat the last ones with a scale of zero: no
// branch stands between products and the reads of their results.
// ---------------------------------------------------------------------------

using i32x4 = __attribute__((ext_vector_type(4))) int;

// NG: scales of a row and chunk, read by one load (groups of KC / NG columns, K
// a multiple of KC); 0: one scale per 16 B load, any group.
// GLU: as in gemm_m16_kernel, the two fragments of a wave are 16 gate columns
// and the 16 up columns beside them.
template <int BITS, int MT, int NF, int KC, int NG, bool GLU>
__global__ __launch_bounds__(256, MT == 4 ? 2 : 3) void gemm_q_kernel(
    const short* __restrict__ x, const void* __restrict__ w,
    const short* __restrict__ scales, const short* __restrict__ bias,
    short* __restrict__ out, float* __restrict__ out_f32, const int M,
    const int K, const int N, const int G, const int splitk) {
  constexpr int SW = BITS == 8 ? 64 : 128;   // columns of a lane group's load
  constexpr int NS = KC / SW;                // loads per row and chunk
  constexpr int NJ = SW / 32;                // products per load
  constexpr int R = 16 * MT;
  constexpr int XP = KC + 8;                 // LDS pitch: 16 rows of a 16 B
                                             // column fall into all banks
  constexpr int XL = R * KC / 8 / 256;       // 16 B of x per thread and chunk
  static_assert(XL * 256 * 8 == R * KC, "chunk");
  __shared__ __attribute__((aligned(16))) short x_lds[2][R * XP];
  const int wave = threadIdx.x >> 6;
  const int lane = threadIdx.x & 63;
  const int c = lane & 15, hi = lane >> 4;
  static_assert(!GLU || NF == 2, "gate and up");
  const int n0 = (blockIdx.x * 4 + wave) * (GLU ? 16 : 16 * NF);
  const int chunks = (K + KC - 1) / KC;
  const int per = (chunks + splitk - 1) / splitk;
  const int c0 = blockIdx.y * per, c1 = min(chunks, c0 + per);
  if (c0 >= c1) return;

  const int rb = BITS == 8 ? K : K / 2;      // bytes of a weight row
  const int gs = G / SW;                     // loads per scale
  const uint64_t ginv = ((1ull << 32) + gs - 1) / gs;
  const char* wp[NF];
  const short* sp[NF];
#pragma unroll
  for (int f = 0; f < NF; ++f) {
    const int64_t row = GLU ? (int64_t)f * N + min(n0 + c, N - 1)
                            : min(n0 + f * 16 + c, N - 1);
    wp[f] = (const char*)w + row * rb + hi * 16;
    sp[f] = scales + row * (K / G);
  }
  f32x4 acc[MT][NF];
#pragma unroll
  for (int m = 0; m < MT; ++m)
#pragma unroll
    for (int f = 0; f < NF; ++f) acc[m][f] = {0.f, 0.f, 0.f, 0.f};

  constexpr int NSC = NG ? NG : NS;          // scales of a chunk
  constexpr int UG = NS / NSC;               // loads per scale
  struct Weights {
    i32x4 w[NS][NF];
    unsigned s[NF][(NSC + 1) / 2];           // bf16 bits, two a word
  };
  const int loads = K / SW;                  // of a whole row
  auto load_w = [&](Weights& q, const int ch) {
#pragma unroll
    for (int f = 0; f < NF; ++f) {
#pragma unroll
      for (int u = 0; u < NS; ++u) {
        const int at = NG ? ch * NS + u : min(ch * NS + u, loads - 1);
        q.w[u][f] = *reinterpret_cast<const i32x4*>(wp[f] + at * 64);
      }
      if constexpr (NG == 4) {
        const uint2 v = *reinterpret_cast<const uint2*>(sp[f] + ch * 4);
        q.s[f][0] = v.x;
        q.s[f][1] = v.y;
      } else if constexpr (NG == 2) {
        q.s[f][0] = *reinterpret_cast<const unsigned*>(sp[f] + ch * 2);
      } else {
#pragma unroll
        for (int u = 0; u < NS; ++u) {
          const int at = min(ch * NS + u, loads - 1);
          const unsigned v =
              ch * NS + u < loads
                  ? (unsigned short)sp[f][((uint64_t)at * ginv) >> 32] : 0u;
          q.s[f][u / 2] = u & 1 ? q.s[f][u / 2] | v << 16 : v;
        }
      }
    }
  };
  i32x4 xr[XL];
  auto load_x = [&](const int ch) {
#pragma unroll
    for (int i = 0; i < XL; ++i) {
      const int e = i * 256 + threadIdx.x;
      const int k = min(ch * KC + e % (KC / 8) * 8, K - 8);
      // rows >= M repeat the last one; their results are never stored
      xr[i] = *reinterpret_cast<const i32x4*>(
          &x[(int64_t)min(e / (KC / 8), M - 1) * K + k]);
    }
  };
  auto store_x = [&](const int buf) {
#pragma unroll
    for (int i = 0; i < XL; ++i) {
      const int e = i * 256 + threadIdx.x;
      *reinterpret_cast<i32x4*>(
          &x_lds[buf][e / (KC / 8) * XP + e % (KC / 8) * 8]) = xr[i];
    }
    // LDS only: the weights in flight are waited for where they are used
    asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
  };
  auto mul = [&](const Weights& q, const int buf) {
#pragma unroll
    for (int g = 0; g < NSC; ++g) {
      f32x4 p[MT][NF];
#pragma unroll
      for (int m = 0; m < MT; ++m)
#pragma unroll
        for (int f = 0; f < NF; ++f) p[m][f] = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int uu = 0; uu < UG; ++uu) {
        const int u = g * UG + uu;
        bf16x8 b[NF][NJ];
#pragma unroll
        for (int f = 0; f < NF; ++f) {
          // ties the conversions to this place: moved up to the load, a
          // chunk's weights take four times the registers
          i32x4 v = q.w[u][f];
          asm volatile("" : "+v"(v));
#pragma unroll
          for (int j = 0; j < NJ; ++j)
#pragma unroll
            for (int e = 0; e < 8; ++e) {
              if (BITS == 8)
                b[f][j][e] = (__bf16)(float)(signed char)(
                    v[2 * j + e / 4] >> (8 * (e & 3)));
              else       // nibbles are stored offset by 8
                b[f][j][e] = (__bf16)(float)(
                    (int)((unsigned)(v[j] ^ 0x88888888) << (28 - 4 * e)) >>
                    28);
            }
        }
#pragma unroll
        for (int m = 0; m < MT; ++m)
#pragma unroll
          for (int j = 0; j < NJ; ++j) {
            const bf16x8 a = *reinterpret_cast<const bf16x8*>(
                &x_lds[buf][(m * 16 + c) * XP + u * SW + j * 32 + hi * 8]);
#pragma unroll
            for (int f = 0; f < NF; ++f)
              p[m][f] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(
                  a, b[f][j], p[m][f], 0, 0, 0);
          }
        // one load's conversions at a time
        __builtin_amdgcn_sched_barrier(0);
      }
#pragma unroll
      for (int f = 0; f < NF; ++f) {
        const float sc = __builtin_bit_cast(
            float, g & 1 ? q.s[f][g / 2] & 0xffff0000u : q.s[f][g / 2] << 16);
#pragma unroll
        for (int m = 0; m < MT; ++m)
#pragma unroll
          for (int r = 0; r < 4; ++r)
            acc[m][f][r] = fmaf(sc, p[m][f][r], acc[m][f][r]);
      }
    }
  };
  // every workgroup starts at another chunk: in step they would all read the
  // same columns of rows that lie a multiple of 256 B apart, a few channels
  const int n_ch = c1 - c0;
  const int turn = (int)((blockIdx.x * 5 + blockIdx.y * 3) % n_ch);
  auto place = [&](int i) {
    i += turn;
    return c0 + (i < n_ch ? i : i - n_ch);
  };
  Weights q0, q1;
  load_x(place(0));
  load_w(q0, place(0));
  store_x(0);
  int i = 0;
  for (; i + 2 < n_ch; i += 2) {
    load_x(place(i + 1));
    load_w(q1, place(i + 1));
    __builtin_amdgcn_sched_barrier(0);
    mul(q0, 0);
    store_x(1);
    load_x(place(i + 2));
    load_w(q0, place(i + 2));
    __builtin_amdgcn_sched_barrier(0);
    mul(q1, 1);
    store_x(0);
  }
  if (i + 1 < n_ch) {
    load_x(place(i + 1));
    load_w(q1, place(i + 1));
    __builtin_amdgcn_sched_barrier(0);
    mul(q0, 0);
    store_x(1);
    mul(q1, 1);
  } else {
    mul(q0, 0);
  }

  if constexpr (GLU) {
    if (n0 + c >= N) return;
#pragma unroll
    for (int m = 0; m < MT; ++m)
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int row = m * 16 + hi * 4 + r;
        if (row < M)
          out[(int64_t)row * N + n0 + c] =
              f2bits(swiglu_of(acc[m][0][r], acc[m][1][r]));
      }
    return;
  }
#pragma unroll
  for (int f = 0; f < NF; ++f) {
    const int n = n0 + f * 16 + c;
    if (n >= N) continue;
    const float bv =
        splitk == 1 && bias != nullptr ? bits2f(bias[n]) : 0.f;
#pragma unroll
    for (int m = 0; m < MT; ++m)
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int row = m * 16 + hi * 4 + r;
        if (row >= M) continue;
        if (splitk > 1)
          atomicAdd(out_f32 + (int64_t)row * N + n, acc[m][f][r]);
        else
          out[(int64_t)row * N + n] = f2bits(acc[m][f][r] + bv);
      }
  }
}

__global__ void f32_to_bf16_bias_kernel(const float* __restrict__ in,
                                        const short* __restrict__ bias,
                                        short* __restrict__ out,
                                        const int64_t total, const int N) {
  for (int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; i < total;
       i += (int64_t)gridDim.x * blockDim.x) {
    float v = in[i];
    if (bias != nullptr) v += bits2f(bias[i % N]);
    out[i] = f2bits(v);
  }
}

// One device per process (shard design): number of leading scratch
// elements holding un-zeroed partials from plain (non-deferred)
// combines. A bool is NOT enough: a small GEMM's memset after a big
// combine would clear the flag while stale partials remain beyond its
// own M*N region and corrupt the next bigger user.
static int64_t g_scratch_dirty_elems = 0;

// Scratch clears are a small fill kernel, never a memset node: the clear may
// be recorded into a captured decode graph.
__global__ __launch_bounds__(256) void zero_fill_kernel(float* __restrict__ p,
                                                        const int64_t n) {
  const int64_t n4 = (n + 3) / 4;
  for (int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; i < n4;
       i += (int64_t)gridDim.x * blockDim.x) {
    if (4 * i + 3 < n) {
      reinterpret_cast<float4*>(p)[i] = make_float4(0.f, 0.f, 0.f, 0.f);
    } else {
      for (int64_t j = 4 * i; j < n; ++j) p[j] = 0.f;
    }
  }
}

static void zero_fill(float* p, int64_t elems, hipStream_t stream) {
  if (elems <= 0) return;
  const int64_t n4 = (elems + 3) / 4;
  const int grid = (int)std::min<int64_t>((n4 + 255) / 256, 2048);
  hipLaunchKernelGGL(zero_fill_kernel, dim3(grid), dim3(256), 0, stream, p,
                     elems);
}

// Zero whatever plain combines left behind and forget it. A captured step
// starts from a clean scratch and ends with this call, so replays and eager
// launches can alternate: the host-side count above describes the device
// state at every boundary between them.
void scratch_clean(torch::Tensor scratch) {
  if (g_scratch_dirty_elems <= 0) return;
  DNET_CHECK(scratch.scalar_type() == torch::kFloat32 &&
                 scratch.is_contiguous(), "scratch fp32");
  zero_fill(scratch.data_ptr<float>(),
            std::min<int64_t>(g_scratch_dirty_elems, scratch.numel()),
            current_stream());
  g_scratch_dirty_elems = 0;
}

// Splits of the inner dimension for the bf16 kernel: ~1024 workgroups (4 per CU)
// so that wave overlap covers the memory's latency; each split keeps 8 x 64
// columns.
static int pick_splitk(int64_t N, int64_t K, int64_t M,
                       int64_t scratch_elems) {
  static const int forced = []() {
    const char* e = getenv("DNET_GEMM_SPLITK");  // debug/bench override
    return e ? atoi(e) : 0;
  }();
  const int blocks = (int)((N + 63) / 64);
  if (forced > 0)
    return (M * N > scratch_elems || (K / 64) < forced) ? 1 : forced;
  int sk = 1;
  while (sk < 32 && blocks * sk < 1024 && (K / 64) / (sk * 2) >= 8) sk *= 2;
  // a span that is no multiple of 256 ends in single steps: half as many splits
  // where that rest is >= 15 % of the span, twice the span has none and the
  // grid still covers the chip
  if (sk > 1) {
    const int64_t span = ((K / 64) / sk) * 64;
    const int64_t span2 = ((K / 64) / (sk / 2)) * 64;
    if (span % 256 != 0 && (double)(span % 256) / span >= 0.15 &&
        span2 % 256 == 0 && blocks * (sk / 2) >= 440)
      sk /= 2;
  }
  if (sk > 1 && M * N > scratch_elems) sk = 1;
  return sk;
}

constexpr int kQChunk = 256, kQCols = 128;   // of gemm_q_kernel

// Splits of the inner dimension for the int8 / int4 kernel, by a model of what
// was measured over 4096 to 55296 columns, 4096 to 27648 deep, 8 to 64 rows: a
// CU gets through its workgroups' chunks at a constant rate, whether one or
// three of them share it, so the fullest CU counts (56 column tiles, 20 chunks,
// 8 rows: 4 splits, 224 workgroups, 11.9 us; 5 splits, 280 workgroups, 15.7);
// one workgroup alone is a tenth slower, filling the pipeline costs about 0.6
// of a chunk per workgroup, and of the splits' atomics, 1.8 TB/s, a quarter
// shows, more where they exceed 0.4 of the rest (432 tiles, 64 rows: 1 split
// 94 us, 5 splits 101, 10 splits 141).
static int pick_splits_q(int64_t N, int64_t K, int64_t M,
                         int64_t scratch_elems, int bits) {
  static const int forced = []() {
    const char* e = getenv("DNET_GEMM_SPLITK");  // debug/bench override
    return e ? atoi(e) : 0;
  }();
  const int chunks = cdiv(K, kQChunk), tiles = cdiv(N, kQCols);
  if (M * N > scratch_elems) return 1;
  if (forced > 0) return std::min(forced, chunks);
  const double chunk_us =
      (M <= 16 ? 1.5 : M <= 32 ? 1.9 : 2.6) * (bits == 8 ? 1.0 : 0.8);
  int best = 1;
  double best_us = 1e30;
  for (int sk = 1; sk <= std::min(chunks, 32); ++sk) {
    const int per = cdiv(chunks, sk);
    if (cdiv(chunks, per) != sk) continue;      // the last ones would be empty
    const int full = cdiv((int64_t)tiles * sk, 256);
    const double base = chunk_us * (full == 1 ? 1.1 : full) * (per + 0.6);
    const double atom = sk > 1 ? (double)sk * M * N * 4 / 1.8e6 : 0.0;
    const double us = base + std::max(0.25 * atom, atom - 0.4 * base);
    if (us < best_us) {
      best_us = us;
      best = sk;
    }
  }
  return best;
}

static int pick_splits(int64_t N, int64_t K, int64_t M, int64_t scratch_elems,
                       int bits) {
  if (bits < 16) return pick_splits_q(N, K, M, scratch_elems, bits);
  return on_b16(M, N, K, false) ? 1 : pick_splitk(N, K, M, scratch_elems);
}

static bool launch_m16(torch::Tensor x, torch::Tensor w,
                       c10::optional<torch::Tensor> scales,
                       c10::optional<torch::Tensor> bias, torch::Tensor out,
                       c10::optional<torch::Tensor> scratch, int group,
                       int64_t m0, int M, int bits, bool defer_combine,
                       bool glu = false) {
  const int64_t K = x.size(1), N = glu ? w.size(0) / 2 : w.size(0);
  auto stream = current_stream();
  const int64_t scratch_elems = scratch.has_value() ? scratch->numel() : 0;
  const int sk = glu ? 1 : pick_splits(N, K, M, scratch_elems, bits);
  const short* bptr = bias.has_value() ? (const short*)bias->data_ptr() : nullptr;
  const dim3 grid((unsigned)((N + 63) / 64), sk);
  const short* xp = (const short*)x.data_ptr() + m0 * K;
  short* op = (short*)out.data_ptr() + m0 * N;
  float* fp = nullptr;
  if (sk > 1) {
    TORCH_CHECK(scratch.has_value() && scratch->numel() >= (int64_t)M * N,
                "split-k scratch required");
    fp = (float*)scratch->data_ptr();
    // The scratch must be zero before the atomics. Deferred-combine
    // consumers (rope/swiglu/rmsnorm f32 variants) re-zero what they
    // read, so a chain of deferred GEMMs never needs a memset; the
    // plain combine does NOT re-zero — a combine-side in[i]=0 write
    // measured a 3.5x MoE decode slowdown (the grouped expert kernels
    // dropped ~3.9 -> ~2.5 TB/s whenever the combine left dirtied
    // scratch lines behind; bisected to that single change) — so the
    // NEXT split-k launch after a combine memsets first.
    if (g_scratch_dirty_elems > 0) {
      const int64_t span = std::max<int64_t>(g_scratch_dirty_elems,
                                             (int64_t)M * N);
      zero_fill(fp, std::min<int64_t>(span, scratch->numel()), stream);
      g_scratch_dirty_elems = 0;
    }
  }
  if (bits == 16 && on_b16(M, glu ? 2 * N : N, K, glu)) {
    launch_b16(xp, (const short*)w.data_ptr(), bptr, op, M, (int)K, (int)N,
               glu, stream);
    return false;
  }
  const short* sp = bits < 16 ? (const short*)scales->data_ptr() : nullptr;
  const short* bp1 = sk > 1 ? nullptr : bptr;
#define LAUNCH(TT, GL)                                                      \
  hipLaunchKernelGGL((gemm_m16_kernel<TT, GL>), grid, dim3(256), 0, stream, \
                     xp, (const short*)w.data_ptr(), bp1, op, fp, M,        \
                     (int)K, (int)N, sk)
#define LAUNCH_QN(QQ, TT, GG, GL)                                           \
  hipLaunchKernelGGL((gemm_q_kernel<QQ, TT, 2, kQChunk, GG, GL>),           \
                     dim3((unsigned)cdiv(N, GL ? 64 : kQCols), sk),         \
                     dim3(256), 0, stream, xp, w.data_ptr(), sp, bp1, op,   \
                     fp, M, (int)K, (int)N, group, sk)
#define LAUNCH_Q(QQ, TT, GL)                                                \
  do {                                                                      \
    if (K % kQChunk == 0 && group == 128) LAUNCH_QN(QQ, TT, 2, GL);         \
    else if (QQ == 8 && K % kQChunk == 0 && group == 64)                    \
      LAUNCH_QN(QQ, TT, QQ == 8 ? 4 : 0, GL);                               \
    else LAUNCH_QN(QQ, TT, 0, GL);                                          \
  } while (0)
#define LAUNCH_M(GL)                                                        \
  do {                                                                      \
    if (bits == 8) {                                                        \
      if (M > 32) LAUNCH_Q(8, 4, GL);                                       \
      else if (M > 16) LAUNCH_Q(8, 2, GL);                                  \
      else LAUNCH_Q(8, 1, GL);                                              \
    } else if (bits == 4) {                                                 \
      if (M > 32) LAUNCH_Q(4, 4, GL);                                       \
      else if (M > 16) LAUNCH_Q(4, 2, GL);                                  \
      else LAUNCH_Q(4, 1, GL);                                              \
    } else {                                                                \
      if (M > 32) LAUNCH(4, GL);                                            \
      else if (M > 16) LAUNCH(2, GL);                                       \
      else LAUNCH(1, GL);                                                   \
    }                                                                       \
  } while (0)
  if (glu) LAUNCH_M(true);
  else LAUNCH_M(false);
#undef LAUNCH_M
#undef LAUNCH_QN
#undef LAUNCH
#undef LAUNCH_Q
#undef LAUNCH_QB
  if (sk > 1) {
    // defer_combine: the caller's next kernel reads (and re-zeroes) the
    // f32 scratch itself — skip the convert/bias pass
    if (defer_combine && bptr == nullptr) return true;
    const int64_t total = (int64_t)M * N;
    const int cgrid = (int)std::min<int64_t>((total + 255) / 256, 2048);
    hipLaunchKernelGGL(f32_to_bf16_bias_kernel, dim3(cgrid), dim3(256), 0,
                       stream, fp, bptr, op, total, (int)N);
    g_scratch_dirty_elems =
        std::max<int64_t>(g_scratch_dirty_elems, (int64_t)M * N);
  }
  return false;
}

// Would gemm_m16(defer_combine=true) actually defer for this shape?
// (Pure: lets callers decide between the fused-consumer and the
// bias-in-combine paths BEFORE launching.)
bool gemm_m16_will_defer(int64_t M, int64_t N, int64_t K, int64_t group,
                         int64_t bits, int64_t scratch_elems) {
  if (M > 64 || (bits < 16 && M <= 2)) return false;
  const int sk = pick_splits(N, K, M, scratch_elems, bits);
  return sk > 1;
}

static void check_m16(const torch::Tensor& x, const torch::Tensor& w,
                      const c10::optional<torch::Tensor>& scales,
                      int64_t group, bool packed, int64_t bits) {
  const int64_t K = x.size(1);
  DNET_CHECK(K % 64 == 0, "K % 64 == 0 required for the MFMA path");
  DNET_CHECK(x.is_contiguous() && w.is_contiguous(), "contig");
  if (bits == 16) {
    DNET_CHECK(w.size(1) == K, "w shape");
  } else {
    DNET_CHECK(packed, "quantized MFMA path expects the packed weight layout");
    DNET_CHECK(scales.has_value() && scales->is_contiguous(), "scales");
    DNET_CHECK(group % 64 == 0 && K % group == 0, "group align");
    if (bits == 8) DNET_CHECK(w.size(1) == K, "w shape (int8)");
    if (bits == 4) {
      DNET_CHECK(w.size(1) == K / 2 && K % 128 == 0 && group % 128 == 0,
                 "w shape / align (int4)");
    }
  }
}

bool gemm_m16(torch::Tensor x, torch::Tensor w,
              c10::optional<torch::Tensor> scales,
              c10::optional<torch::Tensor> bias, torch::Tensor out,
              c10::optional<torch::Tensor> scratch, int64_t group,
              bool packed, int64_t bits, bool defer_combine) {
  const int64_t M = x.size(0), N = w.size(0);
  check_m16(x, w, scales, group, packed, bits);
  DNET_CHECK(out.size(0) == M && out.size(1) == N && out.is_contiguous(),
             "shape");
  // defer only meaningful for the single-chunk (M <= 64) decode path:
  // multiple chunks could pick different sk and leave a mixed state
  const bool defer = defer_combine && M <= 64 && !bias.has_value();
  bool deferred = false;
  int64_t m0 = 0;
  while (m0 < M) {
    const int mt = (int)std::min<int64_t>(M - m0, 64);
    deferred = launch_m16(x, w, scales, bias, out, scratch, (int)group, m0,
                          mt, (int)bits, defer);
    m0 += mt;
  }
  return deferred;
}

// out[M, I] = silu(x @ Wg^T) * (x @ Wu^T), w the gate rows and the up rows
// [2 I, K] without bias, M <= 64. Where the splits of the inner dimension pay
// (pick_splits), the fp32 sums stay in the scratch (returns true: the caller's
// swiglu_f32 reads and clears them), else the activation is part of the product.
bool gemm_swiglu(torch::Tensor x, torch::Tensor w,
                 c10::optional<torch::Tensor> scales, torch::Tensor out,
                 torch::Tensor scratch, int64_t group, int64_t bits) {
  const int64_t M = x.size(0), K = x.size(1), I = out.size(1);
  check_m16(x, w, scales, group, true, bits);
  DNET_CHECK(M <= 64 && out.size(0) == M && w.size(0) == 2 * I &&
                 out.is_contiguous(), "gemm_swiglu shape");
  const bool split =
      !(bits == 16 && on_b16(M, 2 * I, K, true)) &&
      pick_splits(2 * I, K, M, scratch.numel(), (int)bits) > 1;
  return launch_m16(x, w, scales, c10::nullopt, out, scratch, (int)group, 0,
                    (int)M, (int)bits, true, !split);
}

}  // namespace dnet
