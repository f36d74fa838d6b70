// Single-token (decode) attention against the KV cache, GQA-aware.
//
//   out[b,h,:] = softmax(q[b,h,:] . K[b,kv(h),:len,:]^T * scale) @ V[b,kv(h),:len,:]
//
// The read of the cache bounds it; everything else has to stay out of the
// way of the loads. One workgroup of 4 waves per (batch row, kv head, split)
// and each wave on its own: it takes every 4th tile of 32 positions, keeps its
// own online softmax and never waits for another wave before the one merge at
// the end.
//   * K goes from memory straight into the registers in the A layout of
//     v_mfma_f32_16x16x32_bf16 (16 positions x 32 dims), q (the up to 16 query
//     heads of the group) is the B operand: scores^T [position][head].
//   * In C layout a lane holds 4 positions of one head, and over two 16-row
//     tiles exactly the 8 positions that the B operand of the value product
//     wants from it (the order of the contraction index is free as long as V
//     follows it): the weights never cross lanes.
//   * V rows pass through a wave-private LDS tile and come back transposed by
//     ds_read_b64_tr_b16 (4 positions of one dim per lane). Pitch DV + 16
//     halves: the 8 rows that half a wave reads at once fall into different
//     banks.
//   * The next tile's loads are issued as soon as the registers are free
//     (before the softmax), 16 KB in flight per wave.
// Softmax weights are fp32; the matrix core takes them as two bf16 parts
// (16 significant bits), so the value product is as exact as fp32 weights
// against bf16 values. An int8 cache is multiplied as whole numbers (exact in
// bf16) and scaled in fp32.
//
// Sequence length comes from a device tensor (`pos`), so the kernel is
// hipGraph-replayable; how many of the launched splits work is decided from
// it on the device (at least `min_span` positions each), the others leave at
// once.
//
// Measured, MI355X, D 128, with the combine, before (one thread per position
// on packed dot products, both tiles staged for the whole workgroup) -> now:
// 32 rows of 1500 to 8000 positions x 8 kv heads (622 MB, 4 query heads each)
// 270 -> 126 us (5.0 TB/s); 13 rows of 900 to 4000, int8 cache (67 MB, 5
// heads) 113 -> 25 us; 8 rows of 50 to 1900 (32 MB) 55 -> 14 us; one row of
// 701 positions 20 -> 8 us. Error against 64 bits: that of the bf16 result
// (int8 cache: 3.4e-3 -> 1.7e-3, its keys and values are no longer rounded to
// bf16). At 3 waves per SIMD (168 registers) the int8 form gains a tenth over
// 2, the bf16 one nothing; head size 192 would spill there.
//
// Replaces the reference's MLX scaled_dot_product_attention decode path
// (reference: src/dnet/core/models/llama.py apply_single_layer).
#include "common.h"

namespace dnet {

using bf16x8 = __attribute__((ext_vector_type(8))) __bf16;
using s16x4 = __attribute__((ext_vector_type(4))) short;
using s16x8 = __attribute__((ext_vector_type(8))) short;
using f32x4 = __attribute__((ext_vector_type(4))) float;
using u32x4 = __attribute__((ext_vector_type(4))) unsigned;

constexpr int kTile = 32;   // positions of a wave's step

// how many splits share a row's positions (same rule in the combine)
__device__ __forceinline__ int active_splits(int span, int splits,
                                             int min_span) {
  return max(1, min(splits, (span + min_span - 1) / min_span));
}

// 8 int8 codes -> bf16 (exact)
__device__ __forceinline__ bf16x8 codes8(const int lo, const int hi) {
  bf16x8 b;
#pragma unroll
  for (int j = 0; j < 4; ++j) {
    b[j] = (__bf16)(float)(signed char)(lo >> (8 * j));
    b[4 + j] = (__bf16)(float)(signed char)(hi >> (8 * j));
  }
  return b;
}

// p -> hi + lo, each bf16
__device__ __forceinline__ void split8(const float* p, bf16x8& hi, bf16x8& lo) {
#pragma unroll
  for (int j = 0; j < 8; ++j) {
    const __bf16 h = (__bf16)p[j];
    hi[j] = h;
    lo[j] = (__bf16)(p[j] - (float)h);
  }
}

template <int D, int DV, bool Q8>
__global__ __launch_bounds__(256, D == 192 ? 2 : 3) void attn_decode_kernel(
    const short* __restrict__ q, const void* __restrict__ kc,
    const void* __restrict__ vc, const short* __restrict__ kscale,
    const short* __restrict__ vscale, const int* __restrict__ pos,
    short* __restrict__ out, const int Hq, const int Hkv, const int Smax,
    const float scale, const int ldq, const int window,
    const short* __restrict__ sinks, float* __restrict__ partials,
    const int splits, const int min_span, const bool combine) {
  constexpr int DC = D / 32;         // contraction chunks of the scores
  constexpr int NV = DV / 16;        // 16-dim blocks of the values
  constexpr int VP = DV + 16;        // LDS pitch of a V row
  constexpr int KL = Q8 ? D / 64 : D / 32;     // 16 B loads per K row and lane
  constexpr int VL = Q8 ? DV / 32 : DV / 16;   // 16 B loads per V tile and lane
  constexpr int NG = D / 64, NGV = DV / 64;    // scale groups of a row
  constexpr int VE = Q8 ? 16 : 8;              // elements of a 16 B load
  __shared__ __attribute__((aligned(16))) short smem[4 * kTile * VP];
  static_assert(sizeof(smem) >= 4 * 16 * (DV + 2) * 4, "merge area");

  const int b = blockIdx.x / Hkv;
  const int hkv = blockIdx.x % Hkv;
  const int G = Hq / Hkv;
  const int wave = threadIdx.x >> 6;
  const int lane = threadIdx.x & 63;
  const int c16 = lane & 15;
  const int hi = lane >> 4;
  const int len = min(pos[b], Smax);
  const int start = (window > 0) ? max(0, len - window) : 0;
  const int split = blockIdx.y;
  const int nact = active_splits(len - start, splits, min_span);
  if (split >= nact) return;

  const int64_t row0 = ((int64_t)b * Hkv + hkv) * Smax;
  const char* kbase = (const char*)kc + row0 * D * (Q8 ? 1 : 2);
  const char* vbase = (const char*)vc + row0 * DV * (Q8 ? 1 : 2);
  short* vt = smem + wave * kTile * VP;

  // q in B layout: lane holds head c16 (rows past the group repeat its last
  // head; what they give is never stored). int8: a 16 B load of codes covers
  // 16 dims of a 64-dim group, so the contraction runs in that order
  const short* qp =
      q + (int64_t)b * ldq + (int64_t)(hkv * G + min(c16, G - 1)) * D;
  bf16x8 qf[DC];
#pragma unroll
  for (int c = 0; c < DC; ++c)
    qf[c] = *reinterpret_cast<const bf16x8*>(
        Q8 ? &qp[(c >> 1) * 64 + hi * 16 + (c & 1) * 8] : &qp[c * 32 + hi * 8]);

  f32x4 acc[NV];
#pragma unroll
  for (int n = 0; n < NV; ++n) acc[n] = {0.f, 0.f, 0.f, 0.f};
  float m = -1e30f, l = 0.f;   // l: this lane's positions only

  u32x4 kr[2][KL], vr[VL];
  // rows past the end repeat the last one: in range, finite, masked below
  auto load = [&](const int t) {
    const int s0 = t * kTile;
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      const int row = min(s0 + h * 16 + c16, len - 1);
#pragma unroll
      for (int c = 0; c < KL; ++c)
        kr[h][c] = *reinterpret_cast<const u32x4*>(
            kbase + (int64_t)row * (D * (Q8 ? 1 : 2)) + c * 64 + hi * 16);
    }
#pragma unroll
    for (int i = 0; i < VL; ++i) {
      const int e = i * 64 + lane;
      const int row = min(s0 + e / (DV / VE), len - 1);
      vr[i] = *reinterpret_cast<const u32x4*>(
          vbase + (int64_t)row * (DV * (Q8 ? 1 : 2)) + (e % (DV / VE)) * 16);
    }
  };

  const int tend = (len + kTile - 1) / kTile;
  int t = start / kTile + split * 4 + wave;
  if (t < tend) load(t);
  for (; t < tend; t += nact * 4) {
    const int s0 = t * kTile;
    // V tile into LDS (row-major, wave-private: LDS keeps a wave's order)
#pragma unroll
    for (int i = 0; i < VL; ++i) {
      const int e = i * 64 + lane;
      short* dst = &vt[(e / (DV / VE)) * VP + (e % (DV / VE)) * VE];
      if (Q8) {
        *reinterpret_cast<bf16x8*>(dst) = codes8(vr[i].x, vr[i].y);
        *reinterpret_cast<bf16x8*>(dst + 8) = codes8(vr[i].z, vr[i].w);
      } else {
        *reinterpret_cast<u32x4*>(dst) = vr[i];
      }
    }
    f32x4 sc[2];
    float ks[2][4][NG], vs[2][4][NGV];
    if (Q8) {
#pragma unroll
      for (int h = 0; h < 2; ++h)
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          const int64_t row =
              row0 + min(s0 + h * 16 + hi * 4 + r, len - 1);
#pragma unroll
          for (int g = 0; g < NG; ++g) ks[h][r][g] = bits2f(kscale[row * NG + g]);
#pragma unroll
          for (int g = 0; g < NGV; ++g)
            vs[h][r][g] = bits2f(vscale[row * NGV + g]);
        }
    }
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      sc[h] = {0.f, 0.f, 0.f, 0.f};
      if (Q8) {
#pragma unroll
        for (int c = 0; c < KL; ++c) {
          f32x4 part = {0.f, 0.f, 0.f, 0.f};
          part = __builtin_amdgcn_mfma_f32_16x16x32_bf16(
              codes8(kr[h][c].x, kr[h][c].y), qf[2 * c], part, 0, 0, 0);
          part = __builtin_amdgcn_mfma_f32_16x16x32_bf16(
              codes8(kr[h][c].z, kr[h][c].w), qf[2 * c + 1], part, 0, 0, 0);
#pragma unroll
          for (int r = 0; r < 4; ++r)
            sc[h][r] = fmaf(ks[h][r][c], part[r], sc[h][r]);
        }
      } else {
#pragma unroll
        for (int c = 0; c < DC; ++c)
          sc[h] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(
              __builtin_bit_cast(bf16x8, kr[h][c]), qf[c], sc[h], 0, 0, 0);
      }
    }
    const int tn = t + nact * 4;
    if (tn < tend) load(tn);

    // online softmax of head c16 over this lane's 8 positions and the three
    // other lanes of the head
    float p[8];
    bool ok[8];
    float mx = -1e30f;
#pragma unroll
    for (int j = 0; j < 8; ++j) {
      const int sp = s0 + (j >> 2) * 16 + hi * 4 + (j & 3);
      ok[j] = sp < len && sp >= start;
      p[j] = ok[j] ? sc[j >> 2][j & 3] * scale : -1e30f;
      mx = fmaxf(mx, p[j]);
    }
    mx = fmaxf(mx, __shfl_xor(mx, 16, 64));
    mx = fmaxf(mx, __shfl_xor(mx, 32, 64));
    const float mn = fmaxf(m, mx);
    if (__any(mn > m)) {
      const float alpha = __expf(m - mn);
      l *= alpha;
#pragma unroll
      for (int n = 0; n < NV; ++n) acc[n] *= alpha;
    }
    m = mn;
#pragma unroll
    for (int j = 0; j < 8; ++j) {
      p[j] = ok[j] ? __expf(p[j] - mn) : 0.f;
      l += p[j];
    }
    bf16x8 phi[Q8 ? NGV : 1], plo[Q8 ? NGV : 1];
    if (Q8) {
#pragma unroll
      for (int g = 0; g < NGV; ++g) {
        float ps[8];
#pragma unroll
        for (int j = 0; j < 8; ++j) ps[j] = p[j] * vs[j >> 2][j & 3][g];
        split8(ps, phi[g], plo[g]);
      }
    } else {
      split8(p, phi[0], plo[0]);
    }
#pragma unroll
    for (int n = 0; n < NV; ++n) {
      // positions h*16 + hi*4 + 0..3 of dim n*16 + c16, h = 0, 1
      s16x8 vf;
#pragma unroll
      for (int h = 0; h < 2; ++h) {
        const s16x4 part = __builtin_amdgcn_ds_read_tr16_b64_v4i16(
            (__attribute__((address_space(3))) s16x4*)&vt
                [(h * 16 + hi * 4 + (c16 >> 2)) * VP + n * 16 + (c16 & 3) * 4]);
#pragma unroll
        for (int r = 0; r < 4; ++r) vf[h * 4 + r] = part[r];
      }
      const bf16x8 v8 = __builtin_bit_cast(bf16x8, vf);
      const int g = Q8 ? n / 4 : 0;
      acc[n] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(v8, phi[g], acc[n], 0, 0,
                                                       0);
      acc[n] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(v8, plo[g], acc[n], 0, 0,
                                                       0);
    }
  }
  l += __shfl_xor(l, 16, 64);
  l += __shfl_xor(l, 32, 64);

  // merge the four waves' states (their positions are disjoint)
  __syncthreads();
  float* mrg = reinterpret_cast<float*>(smem);   // [4][16][DV]
  float* mml = mrg + 4 * 16 * DV;                // [4][16][2]
  if (c16 < G) {
#pragma unroll
    for (int n = 0; n < NV; ++n)
      *reinterpret_cast<f32x4*>(
          &mrg[(wave * 16 + c16) * DV + n * 16 + hi * 4]) = acc[n];
    if (hi == 0) {
      mml[(wave * 16 + c16) * 2] = m;
      mml[(wave * 16 + c16) * 2 + 1] = l;
    }
  }
  __syncthreads();
  for (int i = threadIdx.x; i < G * (DV / 4); i += 256) {
    const int head = i / (DV / 4);
    const int d = (i % (DV / 4)) * 4;
    float M = -1e30f, L = 0.f;
#pragma unroll
    for (int w = 0; w < 4; ++w) M = fmaxf(M, mml[(w * 16 + head) * 2]);
    f32x4 o = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int w = 0; w < 4; ++w) {
      const float wgt = __expf(mml[(w * 16 + head) * 2] - M);
      L += mml[(w * 16 + head) * 2 + 1] * wgt;
      o += *reinterpret_cast<const f32x4*>(&mrg[(w * 16 + head) * DV + d]) * wgt;
    }
    const int64_t bh = (int64_t)b * Hq + hkv * G + head;
    if (nact > 1 || !combine) {
      float* prow = partials + (bh * splits + split) * (DV + 2);
#pragma unroll
      for (int r = 0; r < 4; ++r) prow[d + r] = o[r];
      if (d == 0) {
        prow[DV] = M;
        prow[DV + 1] = L;
      }
      continue;
    }
    float inv;
    if (sinks != nullptr) {
      // one extra learned softmax logit per q head whose probability mass is
      // dropped from the output
      const float sk = bits2f(sinks[hkv * G + head]);
      const float mx = fmaxf(M, sk);
      const float num = __expf(M - mx);
      const float denom = L * num + __expf(sk - mx);
      inv = (denom > 0.f) ? num / denom : 0.f;
    } else {
      inv = (L > 0.f) ? 1.f / L : 0.f;
    }
    short4v o4;
#pragma unroll
    for (int r = 0; r < 4; ++r) o4.x[r] = f2bits(o[r] * inv);
    *reinterpret_cast<short4v*>(&out[bh * DV + d]) = o4;
  }
}

// Merge the per-split unnormalized partials: one wave per (b, h). `pos` (with
// window, min_span): only the splits that worked on the row are read, and a
// row that one split finished is left alone; null: all of them are.
template <int D>
__global__ void attn_combine_kernel(const float* __restrict__ partials,
                                    const short* __restrict__ sinks,
                                    short* __restrict__ out, const int Hq,
                                    const int splits,
                                    const int* __restrict__ pos,
                                    const int Smax, const int window,
                                    const int min_span) {
  constexpr int DPL = D / kWave;
  const int bh = blockIdx.x;          // b * Hq + h
  const int h = bh % Hq;
  const int lane = threadIdx.x;
  int n = splits;
  if (pos != nullptr) {
    const int len = min(pos[bh / Hq], Smax);
    n = active_splits(window > 0 ? min(len, window) : len, splits, min_span);
    if (n == 1) return;
  }
  const float* base = partials + (int64_t)bh * splits * (D + 2);
  float M = -1e30f;
  for (int s = lane; s < n; s += kWave) M = fmaxf(M, base[s * (D + 2) + D]);
#pragma unroll
  for (int off = 32; off > 0; off >>= 1) M = fmaxf(M, __shfl_xor(M, off, 64));
  if (sinks != nullptr) M = fmaxf(M, bits2f(sinks[h]));
  float denom = (sinks != nullptr) ? __expf(bits2f(sinks[h]) - M) : 0.f;
  float acc[DPL];
#pragma unroll
  for (int j = 0; j < DPL; ++j) acc[j] = 0.f;
#pragma unroll 4
  for (int s = 0; s < n; ++s) {
    const float* prow = base + s * (D + 2);
    const float w = __expf(prow[D] - M);
    denom += prow[D + 1] * w;
#pragma unroll
    for (int j = 0; j < DPL; ++j) acc[j] += prow[DPL * lane + j] * w;
  }
  const float inv = denom > 0.f ? 1.f / denom : 0.f;
  short* orow = out + (int64_t)bh * D + DPL * lane;
#pragma unroll
  for (int j = 0; j < DPL; ++j) orow[j] = f2bits(acc[j] * inv);
}

// merge split/rank partials [B*Hq, splits, DV+2] -> out [B, Hq, DV]
// (cross-rank context parallelism gathers partials and calls this with
// splits = world * local_splits).
void attn_combine(torch::Tensor partials, c10::optional<torch::Tensor> sinks,
                  torch::Tensor out, int64_t splits) {
  const int64_t B = out.size(0), Hq = out.size(1), DV = out.size(2);
  DNET_CHECK(DV == 64 || DV == 128, "combine DV 64/128");
  DNET_CHECK(partials.is_contiguous() && out.is_contiguous(), "contig");
  DNET_CHECK(partials.numel() >= B * Hq * splits * (DV + 2), "partials size");
  auto stream = current_stream();
  const short* skp = sinks.has_value() ? (const short*)sinks->data_ptr()
                                       : nullptr;
  if (DV == 128)
    hipLaunchKernelGGL((attn_combine_kernel<128>), dim3((unsigned)(B * Hq)),
                       dim3(kWave), 0, stream,
                       (const float*)partials.data_ptr(), skp,
                       (short*)out.data_ptr(), (int)Hq, (int)splits,
                       (const int*)nullptr, 0, 0, 0);
  else
    hipLaunchKernelGGL((attn_combine_kernel<64>), dim3((unsigned)(B * Hq)),
                       dim3(kWave), 0, stream,
                       (const float*)partials.data_ptr(), skp,
                       (short*)out.data_ptr(), (int)Hq, (int)splits,
                       (const int*)nullptr, 0, 0, 0);
}

// q may be a column slice of a fused-QKV buffer: strides (ldq, D, 1).
void attn_decode(torch::Tensor q, torch::Tensor kcache, torch::Tensor vcache,
                 torch::Tensor pos, torch::Tensor out, double scale,
                 int64_t window, c10::optional<torch::Tensor> sinks,
                 c10::optional<torch::Tensor> kscale,
                 c10::optional<torch::Tensor> vscale,
                 c10::optional<torch::Tensor> partials, int64_t splits,
                 bool combine) {
  const int64_t B = q.size(0), Hq = q.size(1), D = q.size(2);
  const int64_t Hkv = kcache.size(1), Smax = kcache.size(2);
  const int64_t DV = vcache.size(3);
  DNET_CHECK(kcache.size(0) == B && kcache.size(3) == D, "kcache shape");
  DNET_CHECK(out.size(2) == DV, "out width = v head dim");
  DNET_CHECK(Hq % Hkv == 0 && Hq / Hkv <= 16, "GQA group <= 16");
  DNET_CHECK((D == 64 && DV == 64) || (D == 128 && DV == 128) ||
                 (D == 192 && DV == 128),
             "head dims must be 64/64, 128/128 or 192/128 (MLA)");
  DNET_CHECK(pos.dtype() == torch::kInt32, "pos int32");
  DNET_CHECK(q.stride(2) == 1 && q.stride(1) == D, "q inner dims contiguous");
  DNET_CHECK(kcache.is_contiguous() && vcache.is_contiguous() &&
                 out.is_contiguous(), "contig");
  auto stream = current_stream();
  if (splits > 1 || !combine) {
    DNET_CHECK(partials.has_value()
                   && partials->numel() >= B * Hq * splits * (DV + 2),
               "split-S partials scratch required");
  }
  const dim3 grid((unsigned)(B * Hkv), (unsigned)splits);
  const int ldq = (int)q.stride(0);
  const short* skp = sinks.has_value() ? (const short*)sinks->data_ptr()
                                       : nullptr;
  const bool q8 = kcache.dtype() == torch::kInt8;
  const short* ksp = q8 ? (const short*)kscale->data_ptr() : nullptr;
  const short* vsp = q8 ? (const short*)vscale->data_ptr() : nullptr;
  float* pp = (splits > 1 || !combine) ? (float*)partials->data_ptr()
                                       : nullptr;
  // positions below which a split is not worth its launch and its partials:
  // one tile per wave while the rows alone leave most CUs idle, two otherwise
  // (64 rows x 8 kv heads at 160 positions: one split and no partials)
  const int min_span = B * Hkv < 256 ? 4 * kTile : 8 * kTile;
#define LAUNCH_ATTN(DD, DDV, QQ)                                              \
  hipLaunchKernelGGL((attn_decode_kernel<DD, DDV, QQ>), grid, dim3(256), 0,   \
                     stream, (const short*)q.data_ptr(), kcache.data_ptr(),   \
                     vcache.data_ptr(), ksp, vsp,                             \
                     (const int*)pos.data_ptr(), (short*)out.data_ptr(),      \
                     (int)Hq, (int)Hkv, (int)Smax, (float)scale, ldq,         \
                     (int)window, skp, pp, (int)splits, min_span, combine)
  if (D == 192 && q8) LAUNCH_ATTN(192, 128, true);
  else if (D == 192) LAUNCH_ATTN(192, 128, false);
  else if (D == 128 && q8) LAUNCH_ATTN(128, 128, true);
  else if (D == 128) LAUNCH_ATTN(128, 128, false);
  else if (q8) LAUNCH_ATTN(64, 64, true);
  else LAUNCH_ATTN(64, 64, false);
#undef LAUNCH_ATTN
  if (splits > 1 && combine) {
    if (DV == 128)
      hipLaunchKernelGGL((attn_combine_kernel<128>), dim3((unsigned)(B * Hq)),
                         dim3(kWave), 0, stream, pp, skp,
                         (short*)out.data_ptr(), (int)Hq, (int)splits,
                         (const int*)pos.data_ptr(), (int)Smax, (int)window,
                         min_span);
    else
      hipLaunchKernelGGL((attn_combine_kernel<64>), dim3((unsigned)(B * Hq)),
                         dim3(kWave), 0, stream, pp, skp,
                         (short*)out.data_ptr(), (int)Hq, (int)splits,
                         (const int*)pos.data_ptr(), (int)Smax, (int)window,
                         min_span);
  }
}

}  // namespace dnet
