// Grouped MoE expert kernels: the decode-side dense-expert path in two
// launches per layer instead of O(E) tiny per-expert GEMVs.
//
// Motivation (measured): the per-expert python loop costs ~4000 small
// kernels per token on gpt-oss-20b (24 layers x 32 experts x 3 ops) and
// runs ~350 GB/s effective; these kernels put the whole expert bank behind
// two launches with an early per-expert skip, so a single-stream decode
// reads only the routed experts' weights (top-k/E of the bank).
//
//  - moe_gateup: act[e,m,i] = glu(x[m,:] . Wg[e,i,:], x[m,:] . Wu[e,i,:])
//    with Wg/Wu the halves of the stacked gate_up weights [E, 2I, K]
//    (bf16, or grouped-int8 with fused dequant, optionally in the MFMA
//    chunk-pair packed order), glu = SwiGLU (mixtral) or the gpt-oss
//    clamped GLU. A wave owns one (e, i) pair: two K-dots amortize the x
//    read and keep the weight read a pure 16 B/lane stream.
//  - moe_down: out[m,h] += we[m,e] * (act[e,m,:] . Wd[e,h,:] + b[e,h])
//    accumulated with f32 atomics across experts.
//
// Both kernels skip expert e entirely when we[m,e] == 0 for all m in the
// tile — data-dependent work without host syncs, so the pair stays
// hipGraph-capturable (reference counterpart: the MLX MoE gather path in
// src/dnet/core/models/gpt_oss.py).
#include "common.h"

namespace dnet {

constexpr int kMoeWaves = 4;

using i32x4 = __attribute__((ext_vector_type(4))) int;
using f32x4 = __attribute__((ext_vector_type(4))) float;
using bf16x8 = __attribute__((ext_vector_type(8))) __bf16;

template <int M>
__device__ __forceinline__ bool expert_routed(const float* __restrict__ we,
                                              const int E, const int e,
                                              const int m0) {
  bool any = false;
#pragma unroll
  for (int m = 0; m < M; ++m) any |= (we[(int64_t)(m0 + m) * E + e] != 0.f);
  return any;
}

// MXFP4: e2m1 nibble * 2^(e8m0-127) block scale -> float, via bf16 bit
// construction with the block exponent folded into the exponent field
// (no table lookup). mag==1 is the e2m1 subnormal 0.5.
__device__ __forceinline__ float mxfp4_val(const int nib, const int ebits) {
  const int mag = nib & 7;
  const int e = mag >> 1, m = mag & 1;
  int bits = ((126 + e) << 7) | (m << 6);
  bits = (mag == 1) ? 0x3F00 : bits;
  bits = (mag == 0) ? 0 : (bits + ((ebits - 127) << 7));
  bits |= (nib >> 3) << 15;
  return bits2f((short)bits);
}

// GLU = 0: silu(g) * u   GLU = 1: gpt-oss clamped (u+1) * g * sigmoid(g*a)
template <int GLU>
__device__ __forceinline__ float apply_glu(float g, float u, const float alpha,
                                           const float limit) {
  if (GLU == 1) {
    g = fminf(g, limit);
    u = fminf(fmaxf(u, -limit), limit);
    return (u + 1.f) * g / (1.f + __expf(-g * alpha));
  }
  return g / (1.f + __expf(-g)) * u;
}

// QMODE: 0 = bf16, 1 = grouped int8, 2 = mxfp4 (nibble rows + e8m0)
// Few rows, mxfp4 and odd scale groups (moe_on_cores); M <= 8 per pass at a
// 128-register budget.
template <int M, int QMODE, bool PACKED, int GLU>
__global__ __launch_bounds__(256, 4) void moe_gateup_kernel(
    const short* __restrict__ x, const void* __restrict__ w,
    const short* __restrict__ scales, const short* __restrict__ bias,
    const float* __restrict__ we, short* __restrict__ act, const int K,
    const int I, const int E, const int Mtot, const int m0, const int G,
    const float alpha, const float limit) {
  const int e = blockIdx.z;
  if (!expert_routed<M>(we, E, e, m0)) return;
  const int wid = threadIdx.x / kWave;
  const int lane = threadIdx.x & (kWave - 1);
  const int i = blockIdx.x * kMoeWaves + wid;
  if (i >= I) return;
  const int64_t grow = (int64_t)e * 2 * I + i;      // gate row index
  const int64_t urow = grow + I;                    // up row index
  float ag[M], au[M];
#pragma unroll
  for (int m = 0; m < M; ++m) ag[m] = au[m] = 0.f;
  if (QMODE == 2) {
    const uint8_t* base = static_cast<const uint8_t*>(w);
    const int4* wg = reinterpret_cast<const int4*>(base + grow * (K / 2));
    const int4* wu = reinterpret_cast<const int4*>(base + urow * (K / 2));
    const uint8_t* sb = reinterpret_cast<const uint8_t*>(scales);
    const uint8_t* sg = sb + grow * (K / 32);
    const uint8_t* su = sb + urow * (K / 32);
    const int vecs = K / 32;   // one 16 B load = one 32-value block
    for (int v = lane; v < vecs; v += kWave) {
      i32x4 gv = *reinterpret_cast<const i32x4*>(&wg[v]);
      i32x4 uv = *reinterpret_cast<const i32x4*>(&wu[v]);
      // volatile tie: stops the software pipeliner from pre-extracting
      // the NEXT iterations' nibbles (it spilled 200+ regs otherwise);
      // the loads themselves still prefetch ahead
      asm volatile("" : "+v"(gv), "+v"(uv));
      const uint8_t* gq = reinterpret_cast<const uint8_t*>(&gv);
      const uint8_t* uq = reinterpret_cast<const uint8_t*>(&uv);
      const int ge = sg[v], ue = su[v];
      // dequant per 8-value chunk, outside the M loop (whole-block
      // arrays at gateup's 2 rows = 64 floats blew past 128 VGPR; doing
      // it inside the M loop hoisted M copies -> 1000+ scratch spills).
      // c is a REAL loop (unroll 1): only one chunk's dequant + x
      // values are live at a time
#pragma unroll 1
      for (int c = 0; c < 4; ++c) {         // 4 x 8 values per block
        float gd[8], ud[8];
#pragma unroll
        for (int j = 0; j < 4; ++j) {
          const int gb = gq[c * 4 + j], ub = uq[c * 4 + j];
          gd[2 * j] = mxfp4_val(gb & 0xF, ge);
          gd[2 * j + 1] = mxfp4_val(gb >> 4, ge);
          ud[2 * j] = mxfp4_val(ub & 0xF, ue);
          ud[2 * j + 1] = mxfp4_val(ub >> 4, ue);
        }
#pragma unroll
        for (int m = 0; m < M; ++m) {
          const short8 xv = reinterpret_cast<const short8*>(
              x + (int64_t)(m0 + m) * K)[v * 4 + c];
#pragma unroll
          for (int j = 0; j < 8; ++j) {
            const float xa = bits2f(xv.x[j]);
            ag[m] = fmaf(gd[j], xa, ag[m]);
            au[m] = fmaf(ud[j], xa, au[m]);
          }
        }
      }
    }
  } else if (QMODE == 1) {
    const int4* wg = reinterpret_cast<const int4*>(
        static_cast<const int8_t*>(w) + grow * K);
    const int4* wu = reinterpret_cast<const int4*>(
        static_cast<const int8_t*>(w) + urow * K);
    const short* sg = scales + grow * (K / G);
    const short* su = scales + urow * (K / G);
    const int vecs = K / 16;
    for (int v = lane; v < vecs; v += kWave) {
      const int4 gv = wg[v], uv = wu[v];
      const int8_t* gq = reinterpret_cast<const int8_t*>(&gv);
      const int8_t* uq = reinterpret_cast<const int8_t*>(&uv);
      const float gs = bits2f(sg[(v * 16) / G]);
      const float us = bits2f(su[(v * 16) / G]);
#pragma unroll
      for (int m = 0; m < M; ++m) {
        const short8* xr =
            reinterpret_cast<const short8*>(x + (int64_t)(m0 + m) * K);
        short8 x0, x1;
        if (PACKED) {
          const int pr = v / 4, sl = v % 4;
          x0 = xr[pr * 8 + sl];
          x1 = xr[pr * 8 + sl + 4];
        } else {
          x0 = xr[2 * v];
          x1 = xr[2 * v + 1];
        }
#pragma unroll
        for (int j = 0; j < 8; ++j) {
          const float xa = bits2f(x0.x[j]), xb = bits2f(x1.x[j]);
          ag[m] = fmaf((float)gq[j] * gs, xa, ag[m]);
          ag[m] = fmaf((float)gq[8 + j] * gs, xb, ag[m]);
          au[m] = fmaf((float)uq[j] * us, xa, au[m]);
          au[m] = fmaf((float)uq[8 + j] * us, xb, au[m]);
        }
      }
    }
  } else {
    const short8* wg =
        reinterpret_cast<const short8*>(static_cast<const short*>(w) + grow * K);
    const short8* wu =
        reinterpret_cast<const short8*>(static_cast<const short*>(w) + urow * K);
    const int vecs = K / 8;
    for (int v = lane; v < vecs; v += kWave) {
      const short8 gv = wg[v], uv = wu[v];
#pragma unroll
      for (int m = 0; m < M; ++m) {
        const short8 xv = reinterpret_cast<const short8*>(
            x + (int64_t)(m0 + m) * K)[v];
#pragma unroll
        for (int j = 0; j < 8; ++j) {
          ag[m] = fmaf(bits2f(gv.x[j]), bits2f(xv.x[j]), ag[m]);
          au[m] = fmaf(bits2f(uv.x[j]), bits2f(xv.x[j]), au[m]);
        }
      }
    }
  }
#pragma unroll
  for (int m = 0; m < M; ++m) {
    float g = wave_reduce_sum(ag[m]);
    float u = wave_reduce_sum(au[m]);
    if (lane == 0) {
      if (bias != nullptr) {
        g += bits2f(bias[grow]);
        u += bits2f(bias[urow]);
      }
      act[((int64_t)e * Mtot + m0 + m) * I + i] =
          f2bits(apply_glu<GLU>(g, u, alpha, limit));
    }
  }
}

// Ungated experts (up -> squared ReLU -> down): act[e,m,i] =
// relu(x[m,:] . Wu[e,i,:])^2 with Wu the stacked up weights [E, I, K] (bf16).
// Same layout as moe_gateup_kernel's bf16 branch with one weight row per
// wave; experts nobody in the tile chose are skipped.
template <int M>
__global__ __launch_bounds__(256, 4) void moe_up_act_kernel(
    const short* __restrict__ x, const short* __restrict__ w,
    const float* __restrict__ we, short* __restrict__ act, const int K,
    const int I, const int E, const int Mtot, const int m0) {
  const int e = blockIdx.z;
  if (!expert_routed<M>(we, E, e, m0)) return;
  const int wid = threadIdx.x / kWave;
  const int lane = threadIdx.x & (kWave - 1);
  const int i = blockIdx.x * kMoeWaves + wid;
  if (i >= I) return;
  const short8* wu =
      reinterpret_cast<const short8*>(w + ((int64_t)e * I + i) * K);
  float au[M];
#pragma unroll
  for (int m = 0; m < M; ++m) au[m] = 0.f;
  const int vecs = K / 8;
  for (int v = lane; v < vecs; v += kWave) {
    const short8 uv = wu[v];
#pragma unroll
    for (int m = 0; m < M; ++m) {
      const short8 xv =
          reinterpret_cast<const short8*>(x + (int64_t)(m0 + m) * K)[v];
#pragma unroll
      for (int j = 0; j < 8; ++j)
        au[m] = fmaf(bits2f(uv.x[j]), bits2f(xv.x[j]), au[m]);
    }
  }
#pragma unroll
  for (int m = 0; m < M; ++m) {
    float u = wave_reduce_sum(au[m]);
    if (lane == 0) {
      u = fmaxf(u, 0.f);
      act[((int64_t)e * Mtot + m0 + m) * I + i] = f2bits(u * u);
    }
  }
}

template <int M, int QMODE, bool PACKED>
__global__ __launch_bounds__(256, 4) void moe_down_kernel(
    const short* __restrict__ act, const void* __restrict__ w,
    const short* __restrict__ scales, const short* __restrict__ bias,
    const float* __restrict__ we, float* __restrict__ out, const int I,
    const int H, const int E, const int Mtot, const int m0, const int G) {
  const int e = blockIdx.z;
  if (!expert_routed<M>(we, E, e, m0)) return;
  const int wid = threadIdx.x / kWave;
  const int lane = threadIdx.x & (kWave - 1);
  const int h = blockIdx.x * kMoeWaves + wid;
  if (h >= H) return;
  const int64_t row = (int64_t)e * H + h;
  float acc[M];
#pragma unroll
  for (int m = 0; m < M; ++m) acc[m] = 0.f;
  if (QMODE == 2) {
    const uint8_t* base = static_cast<const uint8_t*>(w);
    const int4* wr = reinterpret_cast<const int4*>(base + row * (I / 2));
    const uint8_t* sr = reinterpret_cast<const uint8_t*>(scales) +
                        row * (I / 32);
    const int vecs = I / 32;
    for (int v = lane; v < vecs; v += kWave) {
      i32x4 wv = *reinterpret_cast<const i32x4*>(&wr[v]);
      asm volatile("" : "+v"(wv));   // see gateup: stops pre-extraction
      const uint8_t* q = reinterpret_cast<const uint8_t*>(&wv);
      const int eb = sr[v];
#pragma unroll 1
      for (int c = 0; c < 4; ++c) {
        float qd[8];
#pragma unroll
        for (int j = 0; j < 4; ++j) {
          const int b = q[c * 4 + j];
          qd[2 * j] = mxfp4_val(b & 0xF, eb);
          qd[2 * j + 1] = mxfp4_val(b >> 4, eb);
        }
#pragma unroll
        for (int m = 0; m < M; ++m) {
          const short8 xv = reinterpret_cast<const short8*>(
              act + ((int64_t)e * Mtot + m0 + m) * I)[v * 4 + c];
#pragma unroll
          for (int j = 0; j < 8; ++j)
            acc[m] = fmaf(qd[j], bits2f(xv.x[j]), acc[m]);
        }
      }
    }
  } else if (QMODE == 1) {
    const int4* wr = reinterpret_cast<const int4*>(
        static_cast<const int8_t*>(w) + row * I);
    const short* sr = scales + row * (I / G);
    const int vecs = I / 16;
    for (int v = lane; v < vecs; v += kWave) {
      const int4 wv = wr[v];
      const int8_t* q = reinterpret_cast<const int8_t*>(&wv);
      const float s = bits2f(sr[(v * 16) / G]);
#pragma unroll
      for (int m = 0; m < M; ++m) {
        const short8* xr = reinterpret_cast<const short8*>(
            act + ((int64_t)e * Mtot + m0 + m) * I);
        short8 x0, x1;
        if (PACKED) {
          const int pr = v / 4, sl = v % 4;
          x0 = xr[pr * 8 + sl];
          x1 = xr[pr * 8 + sl + 4];
        } else {
          x0 = xr[2 * v];
          x1 = xr[2 * v + 1];
        }
#pragma unroll
        for (int j = 0; j < 8; ++j) {
          acc[m] = fmaf((float)q[j] * s, bits2f(x0.x[j]), acc[m]);
          acc[m] = fmaf((float)q[8 + j] * s, bits2f(x1.x[j]), acc[m]);
        }
      }
    }
  } else {
    const short8* wr =
        reinterpret_cast<const short8*>(static_cast<const short*>(w) + row * I);
    const int vecs = I / 8;
    for (int v = lane; v < vecs; v += kWave) {
      const short8 wv = wr[v];
#pragma unroll
      for (int m = 0; m < M; ++m) {
        const short8 xv = reinterpret_cast<const short8*>(
            act + ((int64_t)e * Mtot + m0 + m) * I)[v];
#pragma unroll
        for (int j = 0; j < 8; ++j)
          acc[m] = fmaf(bits2f(wv.x[j]), bits2f(xv.x[j]), acc[m]);
      }
    }
  }
#pragma unroll
  for (int m = 0; m < M; ++m) {
    float r = wave_reduce_sum(acc[m]);
    if (lane == 0) {
      const float wme = we[(int64_t)(m0 + m) * E + e];
      if (wme != 0.f) {
        if (bias != nullptr) r += bits2f(bias[row]);
        atomicAdd(&out[(int64_t)(m0 + m) * H + h], r * wme);
      }
    }
  }
}

// ---- routed rows on matrix cores ------------------------------------------------
// What both kernels above compute, for a batch: the weights of an expert that
// any of up to 64 rows chose are read once (the scalar kernels read them once
// per 8 rows and hold 2 M accumulators per lane). Only the rows that chose the
// expert are multiplied: their numbers are compacted (a ballot, one list in
// LDS), so 20 rows with 4 of 32 experts cost one 16-row tile per expert.
//
// grid (column tiles, K splits, E), 4 waves. Weights are the B operand of
// v_mfma_f32_16x16x32_bf16 and go from memory straight to registers, 64 B of
// every one of 16 NF rows per wave and step; the waves take neighbouring steps
// and fold their sums through LDS. Rows of x come from L2 in the A layout. The
// next group of steps is in flight while one is multiplied. int8 weights are
// multiplied as whole numbers (exact in bf16), their scale applies to the fp32
// sums of a 64-wide step.
// Measured, MI355X: 20 rows, 32 bf16 experts of 2880 x 2880 (4 chosen): gate
// and up 651 -> 180 us (5.5 TB/s), down 484 -> 106 us (4.7); 20 rows, 8 int8
// experts of 4096 x 14336 (2 chosen): 1034 -> 248 us (3.8 TB/s, bound by the
// conversions at 2 waves per SIMD), 761 -> 145 us. Error of the fp32 result
// against 64 bits 1.0e-7 (bf16, as before), 1.2e-7 (int8; 2.5e-7).
// KIND: 0 / 1 = gated (GLU 0 / 1; the first half of the NF fragments are gate
// columns, the second the up columns beside them), 2 = weighted sum of the
// experts' results by fp32 atomics.
template <int MT, int NF, bool Q8, bool PACKED, int KIND>
__device__ __forceinline__ void moe_experts_body(
    const int* list, const int rows, f32x4 (*part)[MT * NF][64],
    const short* __restrict__ x, const void* __restrict__ w,
    const short* __restrict__ scales, const short* __restrict__ bias,
    const float* __restrict__ we, void* __restrict__ out, const int K,
    const int N, const int E, const int Mtot, const int m0,
    const int64_t x_expert, const int G, const float alpha,
    const float limit) {
  constexpr bool GLU = KIND != 2;
  constexpr int NC = GLU ? NF / 2 : NF;      // column fragments of the result
  constexpr int NJ = Q8 ? 2 : 1;             // products per step
  constexpr int U = Q8 && MT > 1 ? 1 : 2;    // neighbouring steps of a wave
  constexpr int KS = Q8 ? 64 : 32;           // inner width of a step (64 B)
  const int e = blockIdx.z;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int lane = threadIdx.x & 63;
  const int c = lane & 15, hi = lane >> 4;
  const int n0 = blockIdx.x * (16 * NC);

  const int rb = Q8 ? K : 2 * K;             // bytes of a weight row
  // step / (steps per scale group): exact for fewer than 2^16 steps
  const uint64_t ginv = Q8 ? ((1ull << 32) + G / 64 - 1) / (G / 64) : 0;
  const char* wp[NF];
  const short* sp[NF];
#pragma unroll
  for (int f = 0; f < NF; ++f) {
    const int col = min(n0 + (f % NC) * 16 + c, N - 1);
    const int64_t row = GLU ? ((int64_t)e * 2 + f / NC) * N + col
                            : (int64_t)e * N + col;
    wp[f] = (const char*)w + row * rb + hi * 16;
    sp[f] = Q8 ? scales + row * (K / G) : nullptr;
  }
  const short* xp[MT];
#pragma unroll
  for (int m = 0; m < MT; ++m)
    xp[m] = x + e * x_expert +
            (int64_t)(m0 + list[min(m * 16 + c, rows - 1)]) * K +
            (Q8 && !PACKED ? hi * 16 : hi * 8);
  f32x4 acc[MT][NF];
#pragma unroll
  for (int m = 0; m < MT; ++m)
#pragma unroll
    for (int f = 0; f < NF; ++f) acc[m][f] = {0.f, 0.f, 0.f, 0.f};

  struct Batch {
    i32x4 wf[U][NF];
    bf16x8 xf[U][NJ][MT];
    float sc[U][NF];
  };
  // a step past the row's end, or the part of the last one that is, is zero
  // (K is a multiple of what one lane loads)
  auto load = [&](Batch& q, const int s, const bool whole) {
#pragma unroll
    for (int f = 0; f < NF; ++f)
#pragma unroll
      for (int u = 0; u < U; ++u) {
        const int at = (s + u) * 64;
        const bool in = whole || at + hi * 16 < rb;
        q.wf[u][f] = in ? *reinterpret_cast<const i32x4*>(wp[f] + at)
                        : i32x4{0, 0, 0, 0};
        if (Q8) q.sc[u][f] = in ? bits2f(sp[f][((uint64_t)(s + u) * ginv) >> 32]) : 0.f;
      }
#pragma unroll
    for (int m = 0; m < MT; ++m) {
#pragma unroll
      for (int u = 0; u < U; ++u) {
        const bool in = whole || (s + u) * 64 + hi * 16 < rb;
#pragma unroll
        for (int j = 0; j < NJ; ++j) {
          const i32x4 v =
              in ? *reinterpret_cast<const i32x4*>(
                       xp[m] + (s + u) * KS + j * (PACKED ? 32 : 8))
                 : i32x4{0, 0, 0, 0};
          q.xf[u][j][m] = __builtin_bit_cast(bf16x8, v);
        }
      }
    }
  };
  // products of a step (bf16: of the U steps) from zero, added to the sums by
  // the vector unit: the matrix core's own sums round less exactly
  auto mul = [&](const Batch& q) {
#pragma unroll
    for (int f = 0; f < NF; ++f) {
      if (Q8) {
#pragma unroll
        for (int u = 0; u < U; ++u) {
          bf16x8 wf[NJ];
#pragma unroll
          for (int j = 0; j < NJ; ++j)
#pragma unroll
            for (int k = 0; k < 8; ++k)
              wf[j][k] = (__bf16)(float)(signed char)(
                  q.wf[u][f][2 * j + k / 4] >> (8 * (k & 3)));
#pragma unroll
          for (int m = 0; m < MT; ++m) {
            f32x4 p = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
            for (int j = 0; j < NJ; ++j)
              p = __builtin_amdgcn_mfma_f32_16x16x32_bf16(q.xf[u][j][m], wf[j],
                                                          p, 0, 0, 0);
#pragma unroll
            for (int r = 0; r < 4; ++r)
              acc[m][f][r] = fmaf(q.sc[u][f], p[r], acc[m][f][r]);
          }
        }
      } else {
#pragma unroll
        for (int m = 0; m < MT; ++m) {
          f32x4 p = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
          for (int u = 0; u < U; ++u)
            p = __builtin_amdgcn_mfma_f32_16x16x32_bf16(
                q.xf[u][0][m], __builtin_bit_cast(bf16x8, q.wf[u][f]), p, 0, 0,
                0);
#pragma unroll
          for (int r = 0; r < 4; ++r) acc[m][f][r] += p[r];
        }
      }
    }
  };
  // this split's steps; whole groups of 4 x U steps, then the rest one by one.
  // Workgroups start at different places: weight rows are often a power of two
  // apart, in step they would all read from the same few memory channels
  const int total = (rb + 63) / 64;
  const int per = (total + gridDim.y - 1) / gridDim.y;
  const int s0 = blockIdx.y * per, s1 = min(total, s0 + per);
  const int full = max(s0, min(s1, rb / 64));     // whole steps end here
  const int groups = (full - s0) / (4 * U);
  const int turn =
      groups > 1 ? (int)((blockIdx.x * 5 + blockIdx.z * 3) % groups) : 0;
  auto place = [&](int g) {
    g += turn;
    if (g >= groups) g -= groups;
    return s0 + (g * 4 + wave) * U;
  };
  Batch q0, q1;
  if (groups > 0) {
    load(q0, place(0), true);
    int g = 0;
    for (; g + 2 <= groups; g += 2) {
      load(q1, place(g + 1), true);
      __builtin_amdgcn_sched_barrier(0);
      mul(q0);
      if (g + 2 < groups) load(q0, place(g + 2), true);
      __builtin_amdgcn_sched_barrier(0);
      mul(q1);
    }
    if (g < groups) mul(q0);
  }
  for (int s = s0 + groups * 4 * U + wave * U; s < s1; s += 4 * U) {
    load(q0, s, false);
    // a step of the next split, or past the end, counts nothing
#pragma unroll
    for (int u = 0; u < U; ++u)
      if (s + u >= s1)
#pragma unroll
        for (int f = 0; f < NF; ++f) q0.wf[u][f] = i32x4{0, 0, 0, 0};
    mul(q0);
  }

  // the last products' results are read below, behind a branch: past their
  // latency in any case
  asm volatile("s_nop 15" ::: "memory");
  // fold the four waves' sums
#pragma unroll
  for (int half = 2; half > 0; half >>= 1) {
    if (wave >= half && wave < 2 * half)
#pragma unroll
      for (int m = 0; m < MT; ++m)
#pragma unroll
        for (int f = 0; f < NF; ++f) part[wave - half][m * NF + f][lane] = acc[m][f];
    __syncthreads();
    if (wave < half)
#pragma unroll
      for (int m = 0; m < MT; ++m)
#pragma unroll
        for (int f = 0; f < NF; ++f) {
          const f32x4 p = part[wave][m * NF + f][lane];
#pragma unroll
          for (int r = 0; r < 4; ++r) acc[m][f][r] += p[r];
        }
    __syncthreads();
  }
  if (wave != 0) return;
#pragma unroll
  for (int m = 0; m < MT; ++m)
#pragma unroll
    for (int f = 0; f < NC; ++f) {
      const int i = n0 + f * 16 + c;
      if (i >= N) continue;
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int p = m * 16 + hi * 4 + r;
        if (p >= rows) continue;
        const int t = m0 + list[p];
        float v = acc[m][f][r];
        if constexpr (GLU) {
          float u = acc[m][NC + f][r];
          if (bias != nullptr) {
            v += bits2f(bias[(int64_t)e * 2 * N + i]);
            u += bits2f(bias[((int64_t)e * 2 + 1) * N + i]);
          }
          ((short*)out)[((int64_t)e * Mtot + t) * N + i] =
              f2bits(apply_glu<KIND>(v, u, alpha, limit));
        } else {
          if (bias != nullptr && blockIdx.y == 0)
            v += bits2f(bias[(int64_t)e * N + i]);
          atomicAdd(&((float*)out)[(int64_t)t * N + i],
                    v * we[(int64_t)t * E + e]);
        }
      }
    }
}

template <int MT, int NF, bool Q8, bool PACKED, int KIND>
__global__ __launch_bounds__(256, 2) void moe_experts_kernel(
    const short* __restrict__ x, const void* __restrict__ w,
    const short* __restrict__ scales, const short* __restrict__ bias,
    const float* __restrict__ we, void* __restrict__ out, const int K,
    const int N, const int E, const int Mtot, const int m0,
    const int64_t x_expert, const int G, const float alpha,
    const float limit) {
  __shared__ __attribute__((aligned(16))) char part[2 * MT * NF * 64 * 16];
  __shared__ int list[64];
  const int e = blockIdx.z;
  const int lane = threadIdx.x & 63;
  const bool hit = lane < 16 * MT && m0 + lane < Mtot &&
                   we[(int64_t)(m0 + lane) * E + e] != 0.f;
  const unsigned long long mask = __ballot(hit);
  const int rows = __popcll(mask);
  if (rows == 0) return;                     // the same in all waves
  if (threadIdx.x < 64 && hit)
    list[__popcll(mask & ((1ull << lane) - 1ull))] = lane;
  __syncthreads();
  // as many row tiles as hold anything, each number its own code: a branch
  // around a tile's products inside the loop would stand between them and the
  // reads of their results
#define ME_BODY(TT)                                                           \
  moe_experts_body<TT, NF, Q8, PACKED, KIND>(                                 \
      list, rows, reinterpret_cast<f32x4(*)[(TT) * NF][64]>(part), x, w,      \
      scales, bias, we, out, K, N, E, Mtot, m0, x_expert, G, alpha, limit)
  if (MT == 1 || rows <= 16) ME_BODY(1);
  else if (MT == 2 || rows <= 32) ME_BODY(MT == 1 ? 1 : 2);
  else ME_BODY(MT);
#undef ME_BODY
}

// x [M, K] or [E, M, K] through the experts w [E, N (gated: 2 N), K]
static void moe_experts(int kind, const torch::Tensor& x,
                        const torch::Tensor& w, const short* scales,
                        const short* bias, const torch::Tensor& we,
                        torch::Tensor& out, int64_t K, int64_t N, int64_t M,
                        int64_t x_expert, int64_t group, bool q8, bool packed,
                        float alpha, float limit) {
  const int64_t E = we.size(1);
  auto stream = current_stream();
  const int nf = M <= 4 ? 2 : 4;
  const unsigned tiles = (unsigned)cdiv(N, 16 * (kind == 2 ? nf : nf / 2));
  // the weighted sum is by atomics anyway: the inner dimension is split where
  // the chosen experts' column tiles may leave CUs idle
  unsigned ks = 1;
  while (kind == 2 && ks < 4 && tiles * ks * std::min<int64_t>(E, 2 * M) < 768 &&
         K / (ks * 2) >= 1024)
    ks *= 2;
  const dim3 grid(tiles, ks, (unsigned)E);
  for (int64_t m0 = 0; m0 < M; m0 += 64) {
    const int64_t left = M - m0;
#define ME(MM, NN, QQ, PP, KK)                                                \
  hipLaunchKernelGGL((moe_experts_kernel<MM, NN, QQ, PP, KK>), grid,          \
                     dim3(256), 0, stream, (const short*)x.data_ptr(),        \
                     w.data_ptr(), scales, bias,                              \
                     (const float*)we.data_ptr(), out.data_ptr(), (int)K,     \
                     (int)N, (int)E, (int)M, (int)m0, x_expert, (int)group,   \
                     alpha, limit)
#define ME_K(MM, NN, QQ, PP)                 \
  do {                                       \
    if (kind == 0) ME(MM, NN, QQ, PP, 0);    \
    else if (kind == 1) ME(MM, NN, QQ, PP, 1); \
    else ME(MM, NN, QQ, PP, 2);              \
  } while (0)
#define ME_Q(MM, NN)                              \
  do {                                            \
    if (q8 && packed) ME_K(MM, NN, true, true);   \
    else if (q8) ME_K(MM, NN, true, false);       \
    else ME_K(MM, NN, false, false);              \
  } while (0)
    if (nf == 2) ME_Q(1, 2);
    else if (left <= 16) ME_Q(1, 4);
    else if (left <= 32) ME_Q(2, 4);
    else ME_Q(4, 4);
#undef ME_Q
#undef ME_K
#undef ME
  }
}

// ---- routing and merging for batched expert products -----------------------
// moe_route: we[t, e] = softmax(logits[t, :])[e] * scale for the `top`
// largest probabilities of row t, 0 elsewhere (the weights are not
// renormalized; ties go to the lower index). One thread per row; fp32 with
// the accurate expf.
__global__ __launch_bounds__(256) void moe_route_kernel(
    const float* __restrict__ logits, float* __restrict__ we, const int T,
    const int E, const int top, const float scale) {
  const int t = blockIdx.x * blockDim.x + threadIdx.x;
  if (t >= T) return;
  const float* lr = logits + (int64_t)t * E;
  float* wr = we + (int64_t)t * E;
  float mx = lr[0];
  for (int e = 1; e < E; ++e) mx = fmaxf(mx, lr[e]);
  float sum = 0.f;
  for (int e = 0; e < E; ++e) {
    const float p = expf(lr[e] - mx);
    wr[e] = -p;                 // negative: not chosen yet
    sum += p;
  }
  const float k = scale / sum;
  for (int c = 0; c < top; ++c) {
    int best = -1;
    float bp = 0.f;
    for (int e = 0; e < E; ++e) {
      const float p = -wr[e];
      if (p > bp) {             // chosen entries are >= 0 and never win
        bp = p;
        best = e;
      }
    }
    if (best < 0) break;
    wr[best] = bp * k;
  }
  for (int e = 0; e < E; ++e)
    if (wr[e] < 0.f) wr[e] = 0.f;
}

// moe_weighted_sum: out[t, :] = sum_e we[t, e] * d[e, t, :] (fp32 sum of the
// experts' results as they come out of the batched product).
template <typename T>
__global__ __launch_bounds__(256) void moe_weighted_sum_kernel(
    const T* __restrict__ d, const float* __restrict__ we,
    float* __restrict__ out, const int Tn, const int E, const int W) {
  const int t = blockIdx.y;
  const int w = (blockIdx.x * blockDim.x + threadIdx.x) * 4;
  if (w >= W) return;
  float a0 = 0.f, a1 = 0.f, a2 = 0.f, a3 = 0.f;
  for (int e = 0; e < E; ++e) {
    const float c = we[(int64_t)t * E + e];
    if (c == 0.f) continue;
    const T* dp = d + ((int64_t)e * Tn + t) * W + w;
    if constexpr (sizeof(T) == 2) {
      const short4v v = *reinterpret_cast<const short4v*>(dp);
      a0 = fmaf(c, bits2f(v.x[0]), a0);
      a1 = fmaf(c, bits2f(v.x[1]), a1);
      a2 = fmaf(c, bits2f(v.x[2]), a2);
      a3 = fmaf(c, bits2f(v.x[3]), a3);
    } else {
      const float4 v = *reinterpret_cast<const float4*>(dp);
      a0 = fmaf(c, v.x, a0);
      a1 = fmaf(c, v.y, a1);
      a2 = fmaf(c, v.z, a2);
      a3 = fmaf(c, v.w, a3);
    }
  }
  *reinterpret_cast<float4*>(out + (int64_t)t * W + w) =
      make_float4(a0, a1, a2, a3);
}

template <typename LaunchFn>
static void moe_dispatch_m(int M, LaunchFn&& fn) {
  switch (M) {
    case 1: fn(std::integral_constant<int, 1>{}); break;
    case 2: fn(std::integral_constant<int, 2>{}); break;
    case 3: fn(std::integral_constant<int, 3>{}); break;
    case 4: fn(std::integral_constant<int, 4>{}); break;
    case 6: fn(std::integral_constant<int, 6>{}); break;
    case 8: fn(std::integral_constant<int, 8>{}); break;
    default: TORCH_CHECK(false, "moe: unsupported M tile ", M);
  }
}

static int moe_mtile(int64_t rem, bool mx4) {
  if (mx4 && rem >= 6) return 6;   // M=8 mxfp4 spills ~30 regs
  if (rem >= 8) return 8;
  if (rem == 7 || rem == 5) return 4;
  return (int)rem;
}

// Rows from which the matrix-core kernel is the faster one (us, gateup + down,
// scalar / matrix cores). bf16, 32 experts of 2880 x 2880, 4 chosen: 2 rows
// 66 / 80, 3 rows 121 / 126, 4 rows 160 / 132, 20 rows 1135 / 287, 64 rows
// 3376 / 315; int8, 8 experts of 4096 x 14336, 2 chosen: 2 rows 192 / 200,
// 3 rows 291 / 258, 20 rows 1795 / 393, 64 rows 5617 / 467. mxfp4, and scale
// groups that a 64-wide step does not divide into, stay with the scalar one.
static bool moe_on_cores(int64_t M, bool mx4, bool q8, int64_t group) {
  if (mx4) return false;
  return q8 ? M >= 3 && group % 64 == 0 : M >= 4;
}

void moe_gateup(torch::Tensor x, torch::Tensor w,
                c10::optional<torch::Tensor> scales,
                c10::optional<torch::Tensor> bias, torch::Tensor we,
                torch::Tensor act, int64_t group, bool packed, int64_t glu,
                double alpha, double limit) {
  const int64_t M = x.size(0), K = x.size(1);
  const int64_t E = w.size(0), I2 = w.size(1), I = I2 / 2;
  // weight dtype selects the mode: bf16, int8 (kChar), mxfp4 nibble rows
  // (kByte, [E, 2I, K/2] + e8m0 uint8 scales [E, 2I, K/32])
  const bool mx4 = w.scalar_type() == torch::kByte;
  const bool q8 = w.scalar_type() == torch::kChar;
  DNET_CHECK(w.size(2) == (mx4 ? K / 2 : K) && act.size(0) == E &&
                 act.size(1) == M && act.size(2) == I, "moe_gateup shape");
  DNET_CHECK(we.size(0) == M && we.size(1) == E, "we shape");
  DNET_CHECK(x.is_contiguous() && w.is_contiguous() && we.is_contiguous() &&
                 act.is_contiguous(), "contig");
  DNET_CHECK(K % (q8 ? 16 : (mx4 ? 32 : 8)) == 0, "K align");
  if (packed) DNET_CHECK(K % 64 == 0 && group % 64 == 0, "packed align");
  const short* sptr = nullptr;
  if (q8) {
    DNET_CHECK(scales.has_value() && group > 0 && K % group == 0, "scales");
    DNET_CHECK(scales->is_contiguous() && scales->size(0) == E &&
                   scales->size(1) == I2 && scales->size(2) == K / group,
               "scales shape");
    sptr = (const short*)scales->data_ptr();
  } else if (mx4) {
    DNET_CHECK(scales.has_value() && scales->scalar_type() == torch::kByte &&
                   scales->is_contiguous() && scales->size(0) == E &&
                   scales->size(1) == I2 && scales->size(2) == K / 32,
               "mxfp4 scales shape");
    sptr = (const short*)scales->data_ptr();
  }
  const short* bptr = bias.has_value() ? (const short*)bias->data_ptr() : nullptr;
  auto stream = current_stream();
  if (moe_on_cores(M, mx4, q8, group)) {
    moe_experts(glu == 1 ? 1 : 0, x, w, sptr, bptr, we, act, K, I, M, 0, group,
                q8, packed, (float)alpha, (float)limit);
    return;
  }
  const dim3 grid(cdiv((int)I, kMoeWaves), 1, (unsigned)E);
  int64_t m0 = 0;
  while (m0 < M) {
    const int mt = moe_mtile(M - m0, mx4);
    moe_dispatch_m(mt, [&](auto mc) {
      constexpr int MV = decltype(mc)::value;
      auto launch = [&](auto qmc, auto pkc, auto gluc) {
        hipLaunchKernelGGL(
            (moe_gateup_kernel<MV, decltype(qmc)::value, decltype(pkc)::value,
                               decltype(gluc)::value>),
            grid, dim3(kMoeWaves * kWave), 0, stream,
            (const short*)x.data_ptr(), w.data_ptr(), sptr, bptr,
            (const float*)we.data_ptr(), (short*)act.data_ptr(), (int)K,
            (int)I, (int)E, (int)M, (int)m0, (int)std::max<int64_t>(group, 16),
            (float)alpha, (float)limit);
      };
      auto with_glu = [&](auto qmc, auto pkc) {
        if (glu == 1)
          launch(qmc, pkc, std::integral_constant<int, 1>{});
        else
          launch(qmc, pkc, std::integral_constant<int, 0>{});
      };
      if (q8) {
        if (packed)
          with_glu(std::integral_constant<int, 1>{}, std::true_type{});
        else
          with_glu(std::integral_constant<int, 1>{}, std::false_type{});
      } else if (mx4) {
        with_glu(std::integral_constant<int, 2>{}, std::false_type{});
      } else if constexpr (MV < 4) {
        with_glu(std::integral_constant<int, 0>{}, std::false_type{});
      }
    });
    m0 += mt;
  }
}

void moe_up_act(torch::Tensor x, torch::Tensor w, torch::Tensor we,
                torch::Tensor act) {
  const int64_t M = x.size(0), K = x.size(1);
  const int64_t E = w.size(0), I = w.size(1);
  DNET_CHECK(x.scalar_type() == torch::kBFloat16 &&
                 w.scalar_type() == torch::kBFloat16 &&
                 act.scalar_type() == torch::kBFloat16 &&
                 we.scalar_type() == torch::kFloat, "moe_up_act dtypes");
  DNET_CHECK(w.dim() == 3 && w.size(2) == K && act.size(0) == E &&
                 act.size(1) == M && act.size(2) == I, "moe_up_act shape");
  DNET_CHECK(we.size(0) == M && we.size(1) == E, "we shape");
  DNET_CHECK(x.is_contiguous() && w.is_contiguous() && we.is_contiguous() &&
                 act.is_contiguous(), "contig");
  DNET_CHECK(K % 8 == 0, "K align");
  auto stream = current_stream();
  const dim3 grid(cdiv((int)I, kMoeWaves), 1, (unsigned)E);
  int64_t m0 = 0;
  while (m0 < M) {
    const int mt = moe_mtile(M - m0, false);
    moe_dispatch_m(mt, [&](auto mc) {
      constexpr int MV = decltype(mc)::value;
      hipLaunchKernelGGL((moe_up_act_kernel<MV>), grid,
                         dim3(kMoeWaves * kWave), 0, stream,
                         (const short*)x.data_ptr(),
                         (const short*)w.data_ptr(),
                         (const float*)we.data_ptr(), (short*)act.data_ptr(),
                         (int)K, (int)I, (int)E, (int)M, (int)m0);
    });
    m0 += mt;
  }
}

void moe_route(torch::Tensor logits, torch::Tensor we, int64_t top,
               double scale) {
  DNET_CHECK(logits.dim() == 2 && logits.scalar_type() == torch::kFloat &&
                 logits.is_contiguous() && we.scalar_type() == torch::kFloat &&
                 we.is_contiguous() && we.sizes() == logits.sizes(),
             "moe_route: logits, we fp32 [T, E]");
  const int64_t T = logits.size(0), E = logits.size(1);
  DNET_CHECK(E >= 1 && top >= 1 && top <= E, "moe_route: 1 <= top <= E");
  if (T == 0) return;
  hipLaunchKernelGGL(moe_route_kernel, dim3(cdiv(T, 256)), dim3(256), 0,
                     current_stream(), logits.data_ptr<float>(),
                     we.data_ptr<float>(), (int)T, (int)E, (int)top,
                     (float)scale);
}

void moe_weighted_sum(torch::Tensor d, torch::Tensor we, torch::Tensor out) {
  DNET_CHECK(d.dim() == 3 && d.is_contiguous() && we.is_contiguous() &&
                 we.scalar_type() == torch::kFloat && out.is_contiguous() &&
                 out.scalar_type() == torch::kFloat, "moe_weighted_sum args");
  const int64_t E = d.size(0), T = d.size(1), W = d.size(2);
  DNET_CHECK(we.size(0) == T && we.size(1) == E && out.size(0) == T &&
                 out.size(1) == W && W % 4 == 0, "moe_weighted_sum shapes");
  if (T == 0) return;
  const dim3 grid(cdiv(W / 4, 256), (unsigned)T);
  auto st = current_stream();
  if (d.scalar_type() == torch::kBFloat16)
    hipLaunchKernelGGL((moe_weighted_sum_kernel<short>), grid, dim3(256), 0,
                       st, (const short*)d.data_ptr(), we.data_ptr<float>(),
                       out.data_ptr<float>(), (int)T, (int)E, (int)W);
  else if (d.scalar_type() == torch::kFloat)
    hipLaunchKernelGGL((moe_weighted_sum_kernel<float>), grid, dim3(256), 0,
                       st, d.data_ptr<float>(), we.data_ptr<float>(),
                       out.data_ptr<float>(), (int)T, (int)E, (int)W);
  else
    DNET_CHECK(false, "moe_weighted_sum: dtype");
}

void moe_down(torch::Tensor act, torch::Tensor w,
              c10::optional<torch::Tensor> scales,
              c10::optional<torch::Tensor> bias, torch::Tensor we,
              torch::Tensor out, int64_t group, bool packed) {
  const int64_t E = w.size(0), H = w.size(1);
  const int64_t M = act.size(1), I = act.size(2);
  const bool mx4 = w.scalar_type() == torch::kByte;
  const bool q8 = w.scalar_type() == torch::kChar;
  DNET_CHECK(act.size(0) == E && w.size(2) == (mx4 ? I / 2 : I),
             "moe_down act/w shape");
  DNET_CHECK(out.size(0) == M && out.size(1) == H &&
                 out.scalar_type() == torch::kFloat, "moe_down out f32");
  DNET_CHECK(we.size(0) == M && we.size(1) == E, "we shape");
  DNET_CHECK(act.is_contiguous() && w.is_contiguous() && we.is_contiguous() &&
                 out.is_contiguous(), "contig");
  DNET_CHECK(I % (q8 ? 16 : (mx4 ? 32 : 8)) == 0, "I align");
  if (packed) DNET_CHECK(I % 64 == 0 && group % 64 == 0, "packed align");
  const short* sptr = nullptr;
  if (q8) {
    DNET_CHECK(scales.has_value() && group > 0 && I % group == 0, "scales");
    DNET_CHECK(scales->is_contiguous() && scales->size(0) == E &&
                   scales->size(1) == H && scales->size(2) == I / group,
               "scales shape");
    sptr = (const short*)scales->data_ptr();
  } else if (mx4) {
    DNET_CHECK(scales.has_value() && scales->scalar_type() == torch::kByte &&
                   scales->is_contiguous() && scales->size(0) == E &&
                   scales->size(1) == H && scales->size(2) == I / 32,
               "mxfp4 scales shape");
    sptr = (const short*)scales->data_ptr();
  }
  const short* bptr = bias.has_value() ? (const short*)bias->data_ptr() : nullptr;
  auto stream = current_stream();
  if (moe_on_cores(M, mx4, q8, group)) {
    moe_experts(2, act, w, sptr, bptr, we, out, I, H, M, M * I, group, q8,
                packed, 0.f, 0.f);
    return;
  }
  const dim3 grid(cdiv((int)H, kMoeWaves), 1, (unsigned)E);
  int64_t m0 = 0;
  while (m0 < M) {
    const int mt = moe_mtile(M - m0, mx4);
    moe_dispatch_m(mt, [&](auto mc) {
      constexpr int MV = decltype(mc)::value;
      auto launch = [&](auto qmc, auto pkc) {
        hipLaunchKernelGGL(
            (moe_down_kernel<MV, decltype(qmc)::value, decltype(pkc)::value>),
            grid, dim3(kMoeWaves * kWave), 0, stream,
            (const short*)act.data_ptr(), w.data_ptr(), sptr, bptr,
            (const float*)we.data_ptr(), (float*)out.data_ptr(), (int)I,
            (int)H, (int)E, (int)M, (int)m0,
            (int)std::max<int64_t>(group, 16));
      };
      if (q8) {
        if (packed)
          launch(std::integral_constant<int, 1>{}, std::true_type{});
        else
          launch(std::integral_constant<int, 1>{}, std::false_type{});
      } else if (mx4) {
        launch(std::integral_constant<int, 2>{}, std::false_type{});
      } else if constexpr (MV < 4) {
        launch(std::integral_constant<int, 0>{}, std::false_type{});
      }
    });
    m0 += mt;
  }
}

__global__ void dequant_mxfp4_kernel(const uint8_t* __restrict__ w,
                                     const uint8_t* __restrict__ scales,
                                     short* __restrict__ out,
                                     const int64_t nblocks, const int bpr) {
  // one thread = one 32-value block (16 B in, 64 B out)
  for (int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x;
       i < nblocks; i += (int64_t)gridDim.x * blockDim.x) {
    const int64_t row = i / bpr;
    const int blk = (int)(i % bpr);
    const int4 v = reinterpret_cast<const int4*>(w)[i];
    const uint8_t* q = reinterpret_cast<const uint8_t*>(&v);
    const int eb = scales[row * bpr + blk];
    short* o = out + (row * bpr + blk) * 32;
#pragma unroll
    for (int j = 0; j < 16; ++j) {
      o[2 * j] = f2bits(mxfp4_val(q[j] & 0xF, eb));
      o[2 * j + 1] = f2bits(mxfp4_val(q[j] >> 4, eb));
    }
  }
}

void dequant_mxfp4(torch::Tensor w, torch::Tensor scales, torch::Tensor out) {
  const int64_t rows = w.size(0), kb = w.size(1);
  DNET_CHECK(w.scalar_type() == torch::kByte &&
                 scales.scalar_type() == torch::kByte, "mxfp4 dtypes");
  DNET_CHECK(kb % 16 == 0 && scales.size(1) == kb / 16 &&
                 out.size(0) == rows && out.size(1) == kb * 2, "shapes");
  DNET_CHECK(w.is_contiguous() && scales.is_contiguous() &&
                 out.is_contiguous(), "contig");
  const int64_t nblocks = rows * (kb / 16);
  const int grid = (int)std::min<int64_t>((nblocks + 255) / 256, 4096);
  hipLaunchKernelGGL(dequant_mxfp4_kernel, dim3(grid), dim3(256), 0,
                     current_stream(), (const uint8_t*)w.data_ptr(),
                     (const uint8_t*)scales.data_ptr(),
                     (short*)out.data_ptr(), nblocks, (int)(kb / 16));
}

}  // namespace dnet
