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

// bf16 weights. MT: number of stacked 16-row A tiles (M <= 16*MT).
template <int MT>
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

  f32x4 acc[MT][2];
#pragma unroll
  for (int t = 0; t < MT; ++t)
#pragma unroll
    for (int u = 0; u < 2; ++u) acc[t][u] = {0.f, 0.f, 0.f, 0.f};

  const short* wrow = w + (int64_t)n_w * K;

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
      bf16x8 wb[4][2];
#pragma unroll
      for (int u = 0; u < 4; ++u) {
        const int p = (k0 / 64) + pl + u;
        wb[u][0] = *reinterpret_cast<const bf16x8*>(&wrow[p * 64 + ks]);
        wb[u][1] = *reinterpret_cast<const bf16x8*>(&wrow[p * 64 + 32 + ks]);
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
          acc[t][0] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(
              a0, wb[u][0], acc[t][0], 0, 0, 0);
          acc[t][1] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(
              a1, wb[u][1], acc[t][1], 0, 0, 0);
        }
    }
    for (; pl < pl_end; ++pl) {
      const int p = (k0 / 64) + pl;
      const bf16x8 b0 =
          *reinterpret_cast<const bf16x8*>(&wrow[p * 64 + ks]);
      const bf16x8 b1 =
          *reinterpret_cast<const bf16x8*>(&wrow[p * 64 + 32 + ks]);
#pragma unroll
      for (int t = 0; t < MT; ++t) {
        const short* at = arow + t * 16 * SE;
        const bf16x8 a0 = *reinterpret_cast<const bf16x8*>(&at[pl * 64 + ks]);
        const bf16x8 a1 = *reinterpret_cast<const bf16x8*>(&at[pl * 64 + 32 + ks]);
        acc[t][0] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a0, b0, acc[t][0],
                                                            0, 0, 0);
        acc[t][1] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a1, b1, acc[t][1],
                                                            0, 0, 0);
      }
    }
  }

  // C write: lane covers col = n0 + (lane&15), rows (lane>>4)*4 + 0..3 of
  // each stacked tile.
  const int n = n0 + (lane & 15);
  if (n >= N) return;
#pragma unroll
  for (int t = 0; t < MT; ++t) {
    const f32x4 a2 = acc[t][0] + acc[t][1];
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const int m = t * 16 + (lane >> 4) * 4 + r;
      if (m >= M) continue;
      if (splitk > 1) {
        atomicAdd(out_f32 + (int64_t)m * N + n, a2[r]);
      } else {
        float v = a2[r];
        if (bias != nullptr) v += bits2f(bias[n]);
        out[(int64_t)m * N + n] = f2bits(v);
      }
    }
  }
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
template <int BITS, int MT, int NF, int KC, int NG>
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
  const int n0 = (blockIdx.x * 4 + wave) * (16 * NF);
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
    const int64_t row = min(n0 + f * 16 + c, N - 1);
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
  return bits < 16 ? pick_splits_q(N, K, M, scratch_elems, bits)
                   : pick_splitk(N, K, M, scratch_elems);
}

static bool launch_m16(torch::Tensor x, torch::Tensor w,
                       c10::optional<torch::Tensor> scales,
                       c10::optional<torch::Tensor> bias, torch::Tensor out,
                       c10::optional<torch::Tensor> scratch, int group,
                       int64_t m0, int M, int bits, bool defer_combine) {
  const int64_t K = x.size(1), N = w.size(0);
  auto stream = current_stream();
  const int64_t scratch_elems = scratch.has_value() ? scratch->numel() : 0;
  const int sk = pick_splits(N, K, M, scratch_elems, bits);
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
  const short* sp = bits < 16 ? (const short*)scales->data_ptr() : nullptr;
  const short* bp1 = sk > 1 ? nullptr : bptr;
#define LAUNCH(TT)                                                          \
  hipLaunchKernelGGL((gemm_m16_kernel<TT>), grid, dim3(256), 0, stream, xp, \
                     (const short*)w.data_ptr(), bp1, op, fp, M, (int)K,    \
                     (int)N, sk)
#define LAUNCH_QN(QQ, TT, FF, KK, GG)                                       \
  hipLaunchKernelGGL((gemm_q_kernel<QQ, TT, FF, KK, GG>),                   \
                     dim3((unsigned)cdiv(N, 64 * FF), sk), dim3(256), 0,    \
                     stream, xp, w.data_ptr(), sp, bp1, op, fp, M, (int)K,  \
                     (int)N, group, sk)
#define LAUNCH_Q(QQ, TT, FF, KK)                                            \
  do {                                                                      \
    if (K % 256 == 0 && group == 128) LAUNCH_QN(QQ, TT, FF, KK, 2);         \
    else if (QQ == 8 && K % 256 == 0 && group == 64)                        \
      LAUNCH_QN(QQ, TT, FF, KK, QQ == 8 ? 4 : 0);                           \
    else LAUNCH_QN(QQ, TT, FF, KK, 0);                                      \
  } while (0)
#define LAUNCH_QB(QQ)                                                       \
  do {                                                                      \
    if (M > 32) LAUNCH_Q(QQ, 4, 2, 256);                                    \
    else if (M > 16) LAUNCH_Q(QQ, 2, 2, 256);                               \
    else LAUNCH_Q(QQ, 1, 2, 256);                                           \
  } while (0)
  if (bits == 8) LAUNCH_QB(8);
  else if (bits == 4) LAUNCH_QB(4);
  else {
    if (M > 32) LAUNCH(4);
    else if (M > 16) LAUNCH(2);
    else LAUNCH(1);
  }
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
  if (M > 64 || M <= 2) return false;
  const int sk = pick_splits(N, K, M, scratch_elems, bits);
  return sk > 1;
}

bool gemm_m16(torch::Tensor x, torch::Tensor w,
              c10::optional<torch::Tensor> scales,
              c10::optional<torch::Tensor> bias, torch::Tensor out,
              c10::optional<torch::Tensor> scratch, int64_t group,
              bool packed, int64_t bits, bool defer_combine) {
  const int64_t M = x.size(0), K = x.size(1), N = w.size(0);
  DNET_CHECK(K % 64 == 0, "K % 64 == 0 required for the MFMA path");
  DNET_CHECK(out.size(0) == M && out.size(1) == N, "shape");
  DNET_CHECK(x.is_contiguous() && w.is_contiguous() && out.is_contiguous(), "contig");
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

}  // namespace dnet
