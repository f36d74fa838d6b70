// Fused decode-step RoPE + KV-cache append.
//
// Applies neox-style rotary embedding (precomputed f32 cos/sin tables — the
// CDNA4 guide's rule for trig-heavy ops: tables on host, never sinf/cosf per
// element) to q in place and to k, then writes the rotated k and raw v into
// the KV cache at position pos[b]. Position comes from a device tensor so the
// whole decode step is hipGraph-replayable.
//
// Reference equivalent: mlx_lm RoPE + KVCache.update_and_fetch
// (reference: src/dnet/core/models/llama.py, utils/model.py make_cache).
#include "common.h"

namespace dnet {

// grid: (B, Hq + Hkv); block: D/2 lanes, lane i rotates pair (i, i + D/2).
// Q8: KV cache stored int8 with one bf16 scale per 64-dim group
// (reference: utils/model.py make_cache kv quantization, 8-bit group 64).
// F32: split-k-fused variant — q/k/v come from the UN-COMBINED f32
// split-k scratch of the qkv GEMM (layout [B, (Hq+2*Hkv)*D], row stride
// ldq), bias (bf16, optional) is applied here, the rotated q goes to a
// dedicated bf16 buffer `qout`, and every scratch element read is
// re-zeroed for the next split-k use. Removes the f32->bf16 combine
// kernel from the decode dependency chain.
template <bool Q8, bool F32 = false>
__global__ void rope_append_kernel(short* __restrict__ q,
                                   short* __restrict__ k,
                                   const short* __restrict__ v,
                                   void* __restrict__ kcache,
                                   void* __restrict__ vcache,
                                   short* __restrict__ kscale,
                                   short* __restrict__ vscale,
                                   const int* __restrict__ pos,
                                   const int* __restrict__ wpos,
                                   const float* __restrict__ cost,
                                   const float* __restrict__ sint,
                                   const int Hq, const int Hkv, const int Smax,
                                   const int D, const int ldq, const int ldk,
                                   const int ldv,
                                   float* __restrict__ src = nullptr,
                                   const short* __restrict__ biasv = nullptr,
                                   short* __restrict__ qout = nullptr,
                                   const short* __restrict__ qn = nullptr,
                                   const short* __restrict__ kn = nullptr,
                                   const float eps = 0.f) {
  const int b = blockIdx.x;
  const int h = blockIdx.y;
  const int i = threadIdx.x;  // 0 .. max(D/2,64)-1; lanes >= D/2 idle
  const int p = pos[b];
  const int half = D / 2;
  const bool act = i < half;
  const float c = act ? cost[(int64_t)p * half + i] : 0.f;
  const float s = act ? sint[(int64_t)p * half + i] : 0.f;
  // per-head RMS norm of the row (x1, x2 of the block's one wave), optional
  auto head_norm = [&](const short* w, float& x1, float& x2) {
    if (w == nullptr) return;
    float ss = act ? x1 * x1 + x2 * x2 : 0.f;
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) ss += __shfl_xor(ss, off, 64);
    const float sc = rsqrtf(ss / (float)D + eps);
    if (act) {
      x1 *= sc * bits2f(w[i]);
      x2 *= sc * bits2f(w[i + half]);
    }
  };
  if (h < Hq) {
    if (F32) {
      float* row = src + (int64_t)b * ldq + h * D;
      float x1 = 0.f, x2 = 0.f;
      if (act) {
        x1 = row[i];
        x2 = row[i + half];
        if (biasv != nullptr) {
          x1 += bits2f(biasv[h * D + i]);
          x2 += bits2f(biasv[h * D + i + half]);
        }
        row[i] = 0.f;
        row[i + half] = 0.f;
      }
      head_norm(qn, x1, x2);
      if (!act) return;
      short* qrow = qout + (int64_t)b * Hq * D + h * D;
      qrow[i] = f2bits(x1 * c - x2 * s);
      qrow[i + half] = f2bits(x2 * c + x1 * s);
      return;
    }
    short* row = q + (int64_t)b * ldq + h * D;
    float x1 = act ? bits2f(row[i]) : 0.f;
    float x2 = act ? bits2f(row[i + half]) : 0.f;
    head_norm(qn, x1, x2);
    if (!act) return;
    row[i] = f2bits(x1 * c - x2 * s);
    row[i + half] = f2bits(x2 * c + x1 * s);
    return;
  }
  const int hk = h - Hq;
  short* krow = k + (int64_t)b * ldk + hk * D;
  float k1 = 0.f, k2 = 0.f, v1 = 0.f, v2 = 0.f;
  float x1 = 0.f, x2 = 0.f;
  if (act && F32) {
    const int kcol = (Hq + hk) * D, vcol = (Hq + Hkv + hk) * D;
    float* krowf = src + (int64_t)b * ldq + kcol;
    float* vrowf = src + (int64_t)b * ldq + vcol;
    x1 = krowf[i];
    x2 = krowf[i + half];
    v1 = vrowf[i];
    v2 = vrowf[i + half];
    if (biasv != nullptr) {
      x1 += bits2f(biasv[kcol + i]);
      x2 += bits2f(biasv[kcol + i + half]);
      v1 += bits2f(biasv[vcol + i]);
      v2 += bits2f(biasv[vcol + i + half]);
    }
    krowf[i] = 0.f;
    krowf[i + half] = 0.f;
    vrowf[i] = 0.f;
    vrowf[i + half] = 0.f;
  } else if (act) {
    x1 = bits2f(krow[i]);
    x2 = bits2f(krow[i + half]);
  }
  head_norm(kn, x1, x2);
  k1 = x1 * c - x2 * s;
  k2 = x2 * c + x1 * s;
  if (act && !F32) {
    krow[i] = f2bits(k1);
    krow[i + half] = f2bits(k2);
    const short* vrow = v + (int64_t)b * ldv + hk * D;
    v1 = bits2f(vrow[i]);
    v2 = bits2f(vrow[i + half]);
  }
  // context parallelism: the cache write targets the LOCAL position
  // wpos[b] (rope still uses the global p); rows outside this rank's
  // shard are skipped (uniform per block, so the Q8 wave reductions
  // below never diverge)
  const int wp = (wpos != nullptr) ? wpos[b] : p;
  if (wp < 0 || wp >= Smax) return;
  const int64_t rowbase = ((int64_t)b * Hkv + hk) * Smax + wp;
  if (!Q8) {
    if (!act) return;
    short* kdst = (short*)kcache + rowbase * D;
    kdst[i] = f2bits(k1);
    kdst[i + half] = f2bits(k2);
    short* vdst = (short*)vcache + rowbase * D;
    vdst[i] = f2bits(v1);
    vdst[i + half] = f2bits(v2);
    return;
  }
  // int8 group-64 quantization. For D=128 (half=64): elem i is in group 0,
  // elem i+half in group 1. For D=64 (half=32): both elems in group 0.
  // One full wave participates in the reductions (idle lanes contribute 0).
  const int ng = D / 64;
  auto wave_max = [](float m) {
#pragma unroll
    for (int off = 32; off > 0; off >>= 1)
      m = fmaxf(m, __shfl_xor(m, off, 64));
    return m;
  };
  auto q8scale = [](float amax) {
    return bits2f(f2bits(fmaxf(amax, 1e-8f) / 127.f));  // bf16-rounded
  };
  {
    const float a0 = wave_max(ng == 2 ? fabsf(k1) : fmaxf(fabsf(k1), fabsf(k2)));
    const float a1 = ng == 2 ? wave_max(fabsf(k2)) : a0;
    if (act) {
      const float s1 = q8scale(a0), s2 = q8scale(a1);
      int8_t* kdst = (int8_t*)kcache + rowbase * D;
      kdst[i] = (int8_t)min(max(__float2int_rn(k1 / s1), -127), 127);
      kdst[i + half] = (int8_t)min(max(__float2int_rn(k2 / s2), -127), 127);
      short* ksrow = kscale + rowbase * ng;
      if (i == 0) ksrow[0] = f2bits(q8scale(a0));
      if (i == 0 && ng == 2) ksrow[1] = f2bits(q8scale(a1));
    }
  }
  {
    const float a0 = wave_max(ng == 2 ? fabsf(v1) : fmaxf(fabsf(v1), fabsf(v2)));
    const float a1 = ng == 2 ? wave_max(fabsf(v2)) : a0;
    if (act) {
      const float s1 = q8scale(a0), s2 = q8scale(a1);
      int8_t* vdst = (int8_t*)vcache + rowbase * D;
      vdst[i] = (int8_t)min(max(__float2int_rn(v1 / s1), -127), 127);
      vdst[i + half] = (int8_t)min(max(__float2int_rn(v2 / s2), -127), 127);
      short* vsrow = vscale + rowbase * ng;
      if (i == 0) vsrow[0] = f2bits(q8scale(a0));
      if (i == 0 && ng == 2) vsrow[1] = f2bits(q8scale(a1));
    }
  }
}

// weights of a per-head norm: the kernel's block is then one wave per head
static const short* norm_of(const c10::optional<torch::Tensor>& w, int64_t D) {
  if (!w.has_value()) return nullptr;
  DNET_CHECK(D <= 128 && w->scalar_type() == torch::kBFloat16 &&
                 w->is_contiguous() && w->numel() == D, "norm weights");
  return (const short*)w->data_ptr();
}

// Fused qkv-split-k-combine + RoPE + append: src = f32 scratch of the
// qkv GEMM (un-combined), qout receives the rotated+biased q rows.
void rope_append_f32(torch::Tensor src, c10::optional<torch::Tensor> bias,
                     torch::Tensor qout, int64_t Hkv, torch::Tensor kcache,
                     torch::Tensor vcache, torch::Tensor pos,
                     torch::Tensor cos_table, torch::Tensor sin_table,
                     c10::optional<torch::Tensor> kscale,
                     c10::optional<torch::Tensor> vscale,
                     c10::optional<torch::Tensor> wpos,
                     c10::optional<torch::Tensor> q_norm,
                     c10::optional<torch::Tensor> k_norm, double eps) {
  const int64_t B = qout.size(0), Hq = qout.size(1), D = qout.size(2);
  const short* qn = norm_of(q_norm, D);
  const short* kn = norm_of(k_norm, D);
  const int64_t Smax = kcache.size(2);
  const int64_t N = (Hq + 2 * Hkv) * D;
  DNET_CHECK(D % 2 == 0 && D / 2 <= 1024, "head_dim");
  DNET_CHECK(qout.is_contiguous() && src.is_contiguous(), "contig");
  DNET_CHECK(src.numel() >= B * N, "scratch too small");
  DNET_CHECK(cos_table.dtype() == torch::kFloat32, "cos table f32");
  auto stream = current_stream();
  const bool q8 = kcache.dtype() == torch::kInt8;
  const int* wpp = wpos.has_value() ? (const int*)wpos->data_ptr() : nullptr;
  const short* bp = bias.has_value() ? (const short*)bias->data_ptr()
                                     : nullptr;
  const unsigned thr = q8 || qn || kn ? 64u : (unsigned)(D / 2);
  if (q8)
    hipLaunchKernelGGL((rope_append_kernel<true, true>),
                       dim3((unsigned)B, (unsigned)(Hq + Hkv)), dim3(thr), 0,
                       stream, nullptr, nullptr, nullptr, kcache.data_ptr(),
                       vcache.data_ptr(), (short*)kscale->data_ptr(),
                       (short*)vscale->data_ptr(),
                       (const int*)pos.data_ptr(), wpp,
                       (const float*)cos_table.data_ptr(),
                       (const float*)sin_table.data_ptr(), (int)Hq, (int)Hkv,
                       (int)Smax, (int)D, (int)N, 0, 0,
                       (float*)src.data_ptr(), bp, (short*)qout.data_ptr(),
                       qn, kn, (float)eps);
  else
    hipLaunchKernelGGL((rope_append_kernel<false, true>),
                       dim3((unsigned)B, (unsigned)(Hq + Hkv)), dim3(thr), 0,
                       stream, nullptr, nullptr, nullptr, kcache.data_ptr(),
                       vcache.data_ptr(), nullptr, nullptr,
                       (const int*)pos.data_ptr(), wpp,
                       (const float*)cos_table.data_ptr(),
                       (const float*)sin_table.data_ptr(), (int)Hq, (int)Hkv,
                       (int)Smax, (int)D, (int)N, 0, 0,
                       (float*)src.data_ptr(), bp, (short*)qout.data_ptr(),
                       qn, kn, (float)eps);
}

void rope_append(torch::Tensor q, torch::Tensor k, torch::Tensor v,
                 torch::Tensor kcache, torch::Tensor vcache, torch::Tensor pos,
                 torch::Tensor cos_table, torch::Tensor sin_table,
                 c10::optional<torch::Tensor> kscale,
                 c10::optional<torch::Tensor> vscale,
                 c10::optional<torch::Tensor> wpos,
                 c10::optional<torch::Tensor> q_norm,
                 c10::optional<torch::Tensor> k_norm, double eps) {
  const int64_t B = q.size(0), Hq = q.size(1), D = q.size(2);
  const short* qn = norm_of(q_norm, D);
  const short* kn = norm_of(k_norm, D);
  const int64_t Hkv = k.size(1), Smax = kcache.size(2);
  DNET_CHECK(D % 2 == 0 && D / 2 <= 1024, "head_dim");
  DNET_CHECK(cos_table.dtype() == torch::kFloat32, "cos table f32");
  // q/k/v may be column slices of one fused QKV buffer: strides (ld, D, 1).
  DNET_CHECK(q.stride(2) == 1 && q.stride(1) == D, "q inner contiguous");
  DNET_CHECK(k.stride(2) == 1 && k.stride(1) == D, "k inner contiguous");
  DNET_CHECK(v.stride(2) == 1 && v.stride(1) == D, "v inner contiguous");
  auto stream = current_stream();
  const bool q8 = kcache.dtype() == torch::kInt8;
  const int* wpp = wpos.has_value() ? (const int*)wpos->data_ptr() : nullptr;
  if (q8) {
    DNET_CHECK(kscale.has_value() && vscale.has_value(), "q8 needs scales");
    DNET_CHECK(D == 64 || D == 128, "q8 kv needs D 64/128");
    hipLaunchKernelGGL(rope_append_kernel<true>,
                       dim3((unsigned)B, (unsigned)(Hq + Hkv)),
                       dim3(64), 0, stream, (short*)q.data_ptr(),
                       (short*)k.data_ptr(), (const short*)v.data_ptr(),
                       kcache.data_ptr(), vcache.data_ptr(),
                       (short*)kscale->data_ptr(), (short*)vscale->data_ptr(),
                       (const int*)pos.data_ptr(), wpp,
                       (const float*)cos_table.data_ptr(),
                       (const float*)sin_table.data_ptr(), (int)Hq, (int)Hkv,
                       (int)Smax, (int)D, (int)q.stride(0), (int)k.stride(0),
                       (int)v.stride(0), nullptr, nullptr, nullptr, qn, kn,
                       (float)eps);
  } else {
    hipLaunchKernelGGL(rope_append_kernel<false>,
                       dim3((unsigned)B, (unsigned)(Hq + Hkv)),
                       dim3(qn || kn ? 64u : (unsigned)(D / 2)), 0, stream,
                       (short*)q.data_ptr(),
                       (short*)k.data_ptr(), (const short*)v.data_ptr(),
                       kcache.data_ptr(), vcache.data_ptr(), nullptr, nullptr,
                       (const int*)pos.data_ptr(), wpp,
                       (const float*)cos_table.data_ptr(),
                       (const float*)sin_table.data_ptr(), (int)Hq, (int)Hkv,
                       (int)Smax, (int)D, (int)q.stride(0), (int)k.stride(0),
                       (int)v.stride(0), nullptr, nullptr, nullptr, qn, kn,
                       (float)eps);
  }
}

// A prompt's rotation and append: q and k of the fused projection's rows,
// optionally RMS-normalized per head (rounded to bf16 as a norm of its own
// would), rotated; q to a buffer, k and v to their cache rows. 8 lanes per
// (token, head), each with 8 neighbouring dims of both halves: every access
// 16 B, every value read and written once (before: gather, multiply, subtract,
// concatenate, convert and copy as 16 passes of their own per layer).
// Measured, MI355X: a 37-token prompt through 4 layers of 4096 wide, with the
// residual sum inside the next norm, 1310 -> 948 us; 64 x 128 tokens through 2
// layers of 5120 wide 16290 -> 14960 us.
// F32: the rows are the un-combined sums of a split product (cleared here for
// the next one), the projection's bias is added.
template <bool NORM, bool F32>
__global__ __launch_bounds__(256) void rope_prefill_kernel(
    void* __restrict__ qkv, const short* __restrict__ bias,
    const short* __restrict__ qw,
    const short* __restrict__ kw, const float* __restrict__ cost,
    const float* __restrict__ sint, short* __restrict__ qout,
    short* __restrict__ kc, short* __restrict__ vc, const int64_t kb,
    const int64_t kh, const int64_t vb, const int64_t vh, const int T,
    const int nq, const int nkv, const int D, const int p0, const float eps,
    const int64_t items) {
  const int64_t item = (int64_t)blockIdx.x * 32 + threadIdx.x / 8;
  if (item >= items) return;
  const int heads = nq + 2 * nkv;
  const int64_t row = item / heads;
  const int h = (int)(item % heads);
  const int half = D / 2;
  const int d = (threadIdx.x & 7) * 8;
  const bool act = d < half;      // lanes past the half only join the norm
  const int64_t b = row / T;
  const int p = p0 + (int)(row % T);
  const int64_t at = (row * heads + h) * D + d;
  short8 x1 = {}, x2 = {};
  if (act) {
    if (F32) {
      const float4 z = make_float4(0.f, 0.f, 0.f, 0.f);
#pragma unroll
      for (int s = 0; s < 2; ++s) {
        float4* fp = reinterpret_cast<float4*>((float*)qkv + at + s * half);
        const float4 a = fp[0], c = fp[1];
        fp[0] = z;
        fp[1] = z;
        const float f[8] = {a.x, a.y, a.z, a.w, c.x, c.y, c.z, c.w};
        short8& x = s ? x2 : x1;
#pragma unroll
        for (int j = 0; j < 8; ++j)
          x.x[j] = f2bits(bias != nullptr
                              ? f[j] + bits2f(bias[h * D + s * half + d + j])
                              : f[j]);
      }
    } else {
      x1 = *reinterpret_cast<const short8*>((const short*)qkv + at);
      x2 = *reinterpret_cast<const short8*>((const short*)qkv + at + half);
    }
  }
  short* dst;
  if (h < nq) dst = qout + (row * nq + h) * D;
  else if (h < nq + nkv) dst = kc + b * kb + (h - nq) * kh + (int64_t)p * D;
  else dst = vc + b * vb + (h - nq - nkv) * vh + (int64_t)p * D;
  if (h < nq + nkv) {
    if (NORM) {
      float ss = 0.f;
#pragma unroll
      for (int j = 0; j < 8; ++j)
        ss += bits2f(x1.x[j]) * bits2f(x1.x[j]) +
              bits2f(x2.x[j]) * bits2f(x2.x[j]);
#pragma unroll
      for (int off = 4; off > 0; off >>= 1) ss += __shfl_xor(ss, off, 8);
      const float sc = rsqrtf(ss / (float)D + eps);
      if (act) {
        const short* w = (h < nq ? qw : kw) + d;
        const short8 w1 = *reinterpret_cast<const short8*>(w);
        const short8 w2 = *reinterpret_cast<const short8*>(w + half);
#pragma unroll
        for (int j = 0; j < 8; ++j) {
          x1.x[j] = f2bits(bits2f(x1.x[j]) * sc * bits2f(w1.x[j]));
          x2.x[j] = f2bits(bits2f(x2.x[j]) * sc * bits2f(w2.x[j]));
        }
      }
    }
    if (act) {
      float cs[8], sn[8];
      const float* cp = cost + (int64_t)p * half + d;
      const float* sp = sint + (int64_t)p * half + d;
#pragma unroll
      for (int j = 0; j < 8; j += 4) {
        *reinterpret_cast<float4*>(&cs[j]) =
            *reinterpret_cast<const float4*>(cp + j);
        *reinterpret_cast<float4*>(&sn[j]) =
            *reinterpret_cast<const float4*>(sp + j);
      }
#pragma unroll
      for (int j = 0; j < 8; ++j) {
        const float a = bits2f(x1.x[j]), c = bits2f(x2.x[j]);
        x1.x[j] = f2bits(a * cs[j] - c * sn[j]);
        x2.x[j] = f2bits(c * cs[j] + a * sn[j]);
      }
    }
  }
  if (act) {
    *reinterpret_cast<short8*>(dst + d) = x1;
    *reinterpret_cast<short8*>(dst + half + d) = x2;
  }
}

// qkv: bf16 rows, or the fp32 scratch of the split product (its leading values)
void rope_prefill(torch::Tensor qkv, c10::optional<torch::Tensor> bias,
                  c10::optional<torch::Tensor> qw,
                  c10::optional<torch::Tensor> kw, torch::Tensor cos,
                  torch::Tensor sin, torch::Tensor qout, torch::Tensor kcache,
                  torch::Tensor vcache, int64_t T, int64_t p0, double eps) {
  const int64_t R = qout.size(0), nq = qout.size(1), D = qout.size(2);
  const int64_t nkv = kcache.size(1), Smax = kcache.size(2);
  const bool f32 = qkv.scalar_type() == torch::kFloat;
  for (const auto& t : {qout, kcache, vcache})
    DNET_CHECK(t.scalar_type() == torch::kBFloat16 &&
                   (uintptr_t)t.data_ptr() % 16 == 0, "bf16, 16 B");
  DNET_CHECK(D % 16 == 0 && D <= 128, "head size");
  DNET_CHECK((f32 || qkv.scalar_type() == torch::kBFloat16) &&
                 qkv.is_contiguous() && (uintptr_t)qkv.data_ptr() % 16 == 0 &&
                 (f32 ? qkv.numel() >= R * (nq + 2 * nkv) * D
                      : qkv.numel() == R * (nq + 2 * nkv) * D) &&
                 qout.is_contiguous(), "qkv rows");
  DNET_CHECK(!bias.has_value() || (f32 && bias->is_contiguous() &&
                                   bias->numel() == (nq + 2 * nkv) * D),
             "bias");
  DNET_CHECK(T > 0 && R % T == 0 && kcache.size(0) == R / T && p0 >= 0 &&
                 p0 + T <= Smax, "rows and positions");
  DNET_CHECK(kcache.size(3) == D && vcache.sizes() == kcache.sizes() &&
                 kcache.stride(3) == 1 && kcache.stride(2) == D &&
                 vcache.stride(3) == 1 && vcache.stride(2) == D &&
                 kcache.stride(0) % 8 == 0 && kcache.stride(1) % 8 == 0 &&
                 vcache.stride(0) % 8 == 0 && vcache.stride(1) % 8 == 0,
             "cache rows");
  for (const auto& t : {cos, sin})
    DNET_CHECK(t.scalar_type() == torch::kFloat && t.is_contiguous() &&
                   t.size(0) >= p0 + T && t.size(1) == D / 2, "cos, sin");
  DNET_CHECK(qw.has_value() == kw.has_value(), "both norms or none");
  if (qw.has_value())
    for (const auto& t : {*qw, *kw})
      DNET_CHECK(t.scalar_type() == torch::kBFloat16 && t.is_contiguous() &&
                     t.numel() == D && (uintptr_t)t.data_ptr() % 16 == 0,
                 "norm weights");
  if (R == 0) return;
  const int64_t items = R * (nq + 2 * nkv);
  const dim3 grid((unsigned)cdiv(items, 32));
#define LAUNCH_RP(NN, FF)                                                     \
  hipLaunchKernelGGL(                                                         \
      (rope_prefill_kernel<NN, FF>), grid, dim3(256), 0, current_stream(),    \
      qkv.data_ptr(),                                                         \
      bias.has_value() ? (const short*)bias->data_ptr() : nullptr,            \
      NN ? (const short*)qw->data_ptr() : nullptr,                            \
      NN ? (const short*)kw->data_ptr() : nullptr, cos.data_ptr<float>(),     \
      sin.data_ptr<float>(), (short*)qout.data_ptr(),                         \
      (short*)kcache.data_ptr(), (short*)vcache.data_ptr(),                   \
      kcache.stride(0), kcache.stride(1), vcache.stride(0),                   \
      vcache.stride(1), (int)T, (int)nq, (int)nkv, (int)D, (int)p0,           \
      (float)eps, items)
  if (qw.has_value() && f32) LAUNCH_RP(true, true);
  else if (qw.has_value()) LAUNCH_RP(true, false);
  else if (f32) LAUNCH_RP(false, true);
  else LAUNCH_RP(false, false);
#undef LAUNCH_RP
}

}  // namespace dnet
