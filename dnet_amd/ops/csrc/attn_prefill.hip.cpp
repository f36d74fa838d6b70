// Flash attention of a prompt (gfx950): causal, sliding window, sinks.
//
// Reference counterpart: src/dnet/core/models/llama.py:76-102 (MLX SDPA).
//
// The matrix cores bound it, and what feeds them: LDS reads of the key and
// value tile and, beside them, one exponential and a handful of vector
// operations per score.
//   * A workgroup of 4 waves takes 128 rows of one kv head: a row is a (token,
//     query head of the group) pair, so one tile in LDS serves every head of
//     the group and few rows are wasted at the diagonal. Each wave owns 32 rows
//     and holds their q in registers.
//   * scores^T = K q^T on v_mfma_f32_32x32x16_bf16: a lane's 16 results belong
//     to one row (its column), and are the positions that the B operand of the
//     value product wants from this lane: the weights stay in their lane (the
//     order of the contraction index is free as long as V follows it), the
//     row's maximum takes one exchange between two lanes, its sum one at the
//     end.
//   * V is kept row-major in LDS and read transposed by ds_read_b64_tr_b16.
//   * 64 positions per tile, two tiles in LDS: the next one is loaded into
//     registers before the products of this one and written after them, one
//     barrier per tile. Pitches: K D + 8 (16 rows of a 16 B column fall into
//     all banks), V a row step of 16 or 48 banks (4 rows x 64 B of half a wave).
// Tiles from the largest row on (the longest first); kv heads vary fastest, so
// that with 8 of them each XCD's L2 holds one head's keys and values.
//
// Measured, MI355X, 2048 tokens x 32 heads (8 kv heads), D 128: first chunk
// 355 -> 76 us (454 TFLOP/s on the causal half), behind 5000 positions
// 1191 -> 264 us (765 TFLOP/s); 64 prompts of 128 tokens x 40 heads 139 -> 59
// us; 1500 tokens x 64 heads of 64 201 -> 47 us. Before: 16x16 tiles, weights
// and transposed V through LDS, one query head per workgroup, loads not
// overlapped. Error against 64 bits unchanged (weights are bf16 in both).
// With changed scores (MOD; 3 more transcendental functions per score): 5
// prompts of 1023 tokens x 32 heads of 128 773 -> 129 us.
#include "common.h"

namespace dnet {

using bf16x8 = __attribute__((ext_vector_type(8))) __bf16;
using s16x4 = __attribute__((ext_vector_type(4))) short;
using s16x8 = __attribute__((ext_vector_type(8))) short;
using u32x4 = __attribute__((ext_vector_type(4))) unsigned;
using f32x16 = __attribute__((ext_vector_type(16))) float;

constexpr int kKeys = 64;    // positions of a tile
constexpr int kRows = 128;   // rows of a workgroup

struct Strides {             // elements; the last axis is contiguous
  int64_t b, h, t;
};

// Scores changed before the softmax (MOD): factor per head, tanh cap,
// logarithmic distance penalty; rows at their own positions, slots and lengths
struct Mod {
  const int *pos, *lens, *slots;             // [B]; lens, slots or null
  const float *temp, *r1, *r2, *sinks;       // [Hq] or null
  float scale, softcap;
  int Bc;
};

template <int D, int DV, bool WINDOW, bool MOD>
__global__ __launch_bounds__(256, D == 192 ? 1 : 2) void attn_prefill_kernel(
    const short* __restrict__ q, const short* __restrict__ k,
    const short* __restrict__ v, const short* __restrict__ sinks,
    short* __restrict__ out, const Strides qs, const Strides ks,
    const Strides vs, const Strides os, const int G, const int Hkv,
    const int T, const int S, const int tiles, const int q_off0,
    const int window, const float scale2, const bool flip, const Mod md) {
  constexpr int NC = D / 16;                 // contraction steps of the scores
  constexpr int NV = DV / 32;                // 32-dim blocks of the values
  constexpr int KP = D + 8;
  constexpr int VP = DV == 96 ? 96 : DV + 32;
  constexpr int KL = kKeys * D / 8 / 256, VL = kKeys * DV / 8 / 256;
  static_assert(kKeys * D / 8 % 256 == 0 && kKeys * DV / 8 % 256 == 0, "tile");
  __shared__ __attribute__((aligned(16))) short k_lds[2][kKeys * KP];
  __shared__ __attribute__((aligned(16))) short v_lds[2][kKeys * VP];

  const int hkv = blockIdx.x % Hkv;
  const int tile = tiles - 1 - (blockIdx.x / Hkv) % tiles;
  const int b = blockIdx.x / (Hkv * tiles);
  const int wave = threadIdx.x >> 6;
  const int lane = threadIdx.x & 63;
  const int c = lane & 31;
  const int hi = lane >> 5;
  const int rows = (MOD && md.lens != nullptr ? min(md.lens[b], T) : T) * G;
  const int r0 = tile * kRows;
  const int slot = MOD && md.slots != nullptr ? md.slots[b] : b;
  if (MOD && (r0 >= rows || slot < 0 || slot >= md.Bc)) return;
  const int q_off = MOD ? md.pos[b] : q_off0;
  const int row = min(r0 + wave * 32 + c, rows - 1);
  const int t = row / G, g = row % G;
  const int qpos = q_off + t;

  // positions that any row of the workgroup sees
  const int last = q_off + min(r0 + kRows - 1, rows - 1) / G;
  const int first = WINDOW ? max(0, q_off + r0 / G - window + 1) : 0;
  const int k_end = min(S, last + 1);
  const int tile0 = first / kKeys, tile1 = (k_end + kKeys - 1) / kKeys;
  // tiles up to here are seen whole by every row of this wave (the rows of a
  // wave ascend; wave-uniform)
  const int wrow0 = min(r0 + wave * 32, rows - 1);
  const int whole_end = q_off + wrow0 / G;

  const short* qp = q + b * qs.b + (int64_t)(hkv * G + g) * qs.h + t * qs.t;
  bf16x8 qf[NC];
#pragma unroll
  for (int i = 0; i < NC; ++i)
    qf[i] = *reinterpret_cast<const bf16x8*>(&qp[i * 16 + hi * 8]);

  const short* kb = k + slot * ks.b + hkv * ks.h;
  const short* vb = v + slot * vs.b + hkv * vs.h;
  // this lane's head; the cap's exponential takes 2 log2(e) x / cap
  float factor = 0.f, r1 = 0.f, r2 = 0.f, cap_in = 0.f;
  if constexpr (MOD) {
    const int h = hkv * G + g;
    factor = md.scale * (md.temp != nullptr ? md.temp[h] : 1.f);
    if (md.softcap > 0.f) cap_in = factor * (2.f * 1.44269504f) / md.softcap;
    if (md.r1 != nullptr) {
      r1 = md.r1[h] * 0.69314718f;           // of a base 2 logarithm
      r2 = md.r2[h];
    }
  }
  u32x4 kr[KL], vr[VL];
  // positions past the end repeat the last one: in range and finite, masked
  auto load = [&](const int kt) {
#pragma unroll
    for (int i = 0; i < KL; ++i) {
      const int e = i * 256 + threadIdx.x;
      const int p = min(kt * kKeys + e / (D / 8), S - 1);
      kr[i] = *reinterpret_cast<const u32x4*>(&kb[p * ks.t + e % (D / 8) * 8]);
    }
#pragma unroll
    for (int i = 0; i < VL; ++i) {
      const int e = i * 256 + threadIdx.x;
      const int p = min(kt * kKeys + e / (DV / 8), S - 1);
      vr[i] = *reinterpret_cast<const u32x4*>(&vb[p * vs.t + e % (DV / 8) * 8]);
    }
  };
  auto store = [&](const int buf) {
#pragma unroll
    for (int i = 0; i < KL; ++i) {
      const int e = i * 256 + threadIdx.x;
      *reinterpret_cast<u32x4*>(
          &k_lds[buf][e / (D / 8) * KP + e % (D / 8) * 8]) = kr[i];
    }
#pragma unroll
    for (int i = 0; i < VL; ++i) {
      const int e = i * 256 + threadIdx.x;
      *reinterpret_cast<u32x4*>(
          &v_lds[buf][e / (DV / 8) * VP + e % (DV / 8) * 8]) = vr[i];
    }
  };

  f32x16 acc[NV];
#pragma unroll
  for (int n = 0; n < NV; ++n) acc[n] = f32x16{};
  float m = -1e30f, l = 0.f;      // of scores * scale * log2(e)

  load(tile0);
  store(tile0 & 1);
  __syncthreads();
  for (int kt = tile0; kt < tile1; ++kt) {
    const int buf = kt & 1;
    if (kt + 1 < tile1) load(kt + 1);
    f32x16 s[2];
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      s[h] = f32x16{};
      const short* kl = &k_lds[buf][(h * 32 + c) * KP + hi * 8];
#pragma unroll
      for (int i = 0; i < NC; ++i)
        s[h] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(
            *reinterpret_cast<const bf16x8*>(&kl[i * 16]), qf[i], s[h], 0, 0,
            0);
    }
    // the branch below stands between the products and the first read of
    // their results: past the products' latency in any case
    asm volatile("s_nop 15\n\ts_nop 3" : "+v"(s[0]), "+v"(s[1]));
    if (!MOD && flip) {
      s[0] = -s[0];
      s[1] = -s[1];
    }
    // position of result r of half h: kt * 64 + h * 32 + r / 4 * 8 + hi * 4 +
    // r % 4
    const int k0 = kt * kKeys;
    if constexpr (MOD) {
      if (md.softcap > 0.f) {
        // cap * tanh(x / cap) = cap - 2 cap / (e^(2 x / cap) + 1)
#pragma unroll
        for (int h = 0; h < 2; ++h)
#pragma unroll
          for (int r = 0; r < 16; ++r)
            s[h][r] = fmaf(-2.f * md.softcap,
                           __builtin_amdgcn_rcpf(
                               __builtin_amdgcn_exp2f(s[h][r] * cap_in) + 1.f),
                           md.softcap);
      } else {
        s[0] *= factor;
        s[1] *= factor;
      }
      if (md.r1 != nullptr) {
        const float back = (float)(qpos - k0 - hi * 4);   // exact
#pragma unroll
        for (int h = 0; h < 2; ++h)
#pragma unroll
          for (int r = 0; r < 16; ++r)
            s[h][r] = fmaf(-r1,
                           __builtin_amdgcn_logf(fmaf(
                               r2, fmaxf(back - (h * 32 + r / 4 * 8 + r % 4),
                                         0.f), 1.f)),
                           s[h][r]);
      }
    }
    const bool whole = k0 + kKeys - 1 <= whole_end && k0 + kKeys <= S &&
                       (!WINDOW || k0 > last - window);
    if (!whole) {
#pragma unroll
      for (int h = 0; h < 2; ++h)
#pragma unroll
        for (int r = 0; r < 16; ++r) {
          const int p = k0 + h * 32 + r / 4 * 8 + hi * 4 + r % 4;
          const bool dead = p > qpos || p >= S ||
                            (WINDOW && p <= qpos - window);
          if (dead) s[h][r] = -INFINITY;
        }
    }
    float mx = -INFINITY;
#pragma unroll
    for (int h = 0; h < 2; ++h)
#pragma unroll
      for (int r = 0; r < 16; ++r) mx = fmaxf(mx, s[h][r]);
    mx = fmaxf(mx, __shfl_xor(mx, 32, 64));
    const float mn = fmaxf(m, mx * scale2);
    if (__any(mn > m)) {
      const float alpha = __builtin_amdgcn_exp2f(m - mn);
      l *= alpha;
#pragma unroll
      for (int n = 0; n < NV; ++n) acc[n] *= alpha;
      m = mn;
    }
    bf16x8 p[2][2];
#pragma unroll
    for (int h = 0; h < 2; ++h)
#pragma unroll
      for (int r = 0; r < 16; ++r) {
        const float e =
            __builtin_amdgcn_exp2f(fmaf(s[h][r], scale2, -m));
        l += e;
        p[h][r / 8][r % 8] = (__bf16)e;
      }
#pragma unroll
    for (int n = 0; n < NV; ++n)
#pragma unroll
      for (int h = 0; h < 2; ++h)
#pragma unroll
        for (int u = 0; u < 2; ++u) {
          s16x8 vf;
#pragma unroll
          for (int x = 0; x < 2; ++x) {
            const s16x4 part = __builtin_amdgcn_ds_read_tr16_b64_v4i16(
                (__attribute__((address_space(3))) s16x4*)&v_lds[buf]
                    [(h * 32 + u * 16 + x * 8 + hi * 4 + ((lane & 15) >> 2)) *
                         VP +
                     n * 32 + (c >> 4) * 16 + (lane & 3) * 4]);
#pragma unroll
            for (int j = 0; j < 4; ++j) vf[x * 4 + j] = part[j];
          }
          acc[n] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(
              __builtin_bit_cast(bf16x8, vf), p[h][u], acc[n], 0, 0, 0);
        }
    if (kt + 1 < tile1) store(buf ^ 1);
    __syncthreads();
  }
  l += __shfl_xor(l, 32, 64);
  if (r0 + wave * 32 + c >= rows) return;
  float f = 1.f;
  if (MOD ? md.sinks != nullptr : sinks != nullptr) {
    // one extra logit per head whose mass has no value
    const float sk = 1.44269504f * (MOD ? md.sinks[hkv * G + g]
                                        : bits2f(sinks[hkv * G + g]));
    const float m2 = fmaxf(m, sk);
    f = __builtin_amdgcn_exp2f(m - m2);
    l = l * f + __builtin_amdgcn_exp2f(sk - m2);
  }
  const float inv = f / fmaxf(l, 1e-30f);
  short* op = out + b * os.b + (int64_t)(hkv * G + g) * os.h + t * os.t;
#pragma unroll
  for (int n = 0; n < NV; ++n)
#pragma unroll
    for (int r = 0; r < 16; r += 4) {
      short4v o4;
#pragma unroll
      for (int j = 0; j < 4; ++j) o4.x[j] = f2bits(acc[n][r + j] * inv);
      *reinterpret_cast<short4v*>(&op[n * 32 + r * 2 + hi * 4]) = o4;
    }
}

static Strides strides_of(const torch::Tensor& t, const char* what) {
  // 16 B accesses along the last axis (an axis of one entry may have any
  // stride, it is never stepped over)
  DNET_CHECK(t.stride(3) == 1 && (uintptr_t)t.data_ptr() % 16 == 0, what);
  for (int i = 0; i < 3; ++i)
    DNET_CHECK(t.size(i) == 1 || t.stride(i) % 8 == 0, what);
  return {t.stride(0), t.stride(1), t.stride(2)};
}

// q [B,Hq,T,D], k [B,Hkv,S,D], v [B,Hkv,S,DV], out [B,Hq,T,DV]: any strides
// with contiguous rows on 16 B boundaries
void attn_prefill(torch::Tensor q, torch::Tensor k, torch::Tensor v,
                  c10::optional<torch::Tensor> sinks, torch::Tensor out,
                  int64_t q_off, int64_t window, double scale) {
  const int B = q.size(0), Hq = q.size(1), T = q.size(2), D = q.size(3);
  const int Hkv = k.size(1), S = k.size(2), DV = v.size(3);
  DNET_CHECK(q.scalar_type() == torch::kBFloat16 &&
                 k.scalar_type() == torch::kBFloat16 &&
                 v.scalar_type() == torch::kBFloat16 &&
                 out.scalar_type() == torch::kBFloat16, "bf16");
  DNET_CHECK(Hkv > 0 && Hq % Hkv == 0, "GQA heads");
  DNET_CHECK(k.size(0) == B && v.size(0) == B && v.size(1) == Hkv &&
                 v.size(2) == S && k.size(3) == D, "k, v shape");
  DNET_CHECK(out.size(0) == B && out.size(1) == Hq && out.size(2) == T &&
                 out.size(3) == DV, "out shape");
  if (B == 0 || T == 0) return;
  DNET_CHECK(S > 0 && q_off >= 0 && (int64_t)T * (Hq / Hkv) < (1ll << 30),
             "prompt size");
  const Strides qs = strides_of(q, "q rows"), ks = strides_of(k, "k rows");
  const Strides vs = strides_of(v, "v rows"), os = strides_of(out, "out rows");
  const short* sp =
      sinks.has_value() ? (const short*)sinks->data_ptr() : nullptr;
  const int G = Hq / Hkv;
  const int tiles = cdiv((int64_t)T * G, kRows);
  const dim3 grid((unsigned)(tiles * Hkv * B));
  // the kernel's maximum is taken before the factor, which has to be positive
  const float scale2 =
      (float)(std::max(std::abs(scale), 1e-30) * 1.4426950408889634);
#define LAUNCH_AP(DD, DDV, WW)                                               \
  hipLaunchKernelGGL((attn_prefill_kernel<DD, DDV, WW, false>), grid,        \
                     dim3(256), 0, current_stream(),                         \
                     (const short*)q.data_ptr(),                             \
                     (const short*)k.data_ptr(), (const short*)v.data_ptr(), \
                     sp, (short*)out.data_ptr(), qs, ks, vs, os, G, Hkv, T,  \
                     S, tiles, (int)q_off, (int)window, scale2, scale < 0,   \
                     Mod{})
#define LAUNCH_AP_W(DD, DDV)                \
  do {                                      \
    if (window > 0) LAUNCH_AP(DD, DDV, true); \
    else LAUNCH_AP(DD, DDV, false);         \
  } while (0)
  if (D == 128 && DV == 128) LAUNCH_AP_W(128, 128);
  else if (D == 64 && DV == 64) LAUNCH_AP_W(64, 64);
  else if (D == 192 && DV == 128) LAUNCH_AP_W(192, 128);
  else if (D == 96 && DV == 96) LAUNCH_AP_W(96, 96);
  else DNET_CHECK(false, "attn_prefill: unsupported head dims");
#undef LAUNCH_AP
#undef LAUNCH_AP_W
}

// The prompts of attn_mod that have only the modifiers of Mod and a window: q
// [B T, Hq D], caches [Bc, Hkv, Smax, D], out rows out_ld apart. Returns false
// (nothing launched) for other head sizes and for rows off 16 B boundaries.
bool attn_prompt_mod(const short* q, const short* k, const short* v, short* out,
                     const int* pos, const int* lens, const int* slots,
                     const float* temp, const float* r1, const float* r2,
                     const float* sinks, float scale, float softcap, int B,
                     int T, int Bc, int Hq, int Hkv, int Smax, int D, int DV,
                     int window, int64_t out_ld) {
  const int G = Hq / Hkv;
  if (D != DV || (D != 64 && D != 96 && D != 128) || Smax < 1 ||
      (uintptr_t)q % 16 || (uintptr_t)k % 16 || (uintptr_t)v % 16 ||
      (uintptr_t)out % 8 || out_ld % 4 || (int64_t)T * G >= (1ll << 30))
    return false;
  const int tiles = cdiv((int64_t)T * G, kRows);
  if ((int64_t)tiles * Hkv * B >= (1ll << 31)) return false;
  const Strides qs{(int64_t)T * Hq * D, D, (int64_t)Hq * D};
  const Strides cs{(int64_t)Hkv * Smax * D, (int64_t)Smax * D, D};
  const Strides os{(int64_t)T * out_ld, DV, out_ld};
  const Mod md{pos, lens, slots, temp, r1, r2, sinks, scale, softcap, Bc};
#define LAUNCH_PM(DD, WW)                                                    \
  hipLaunchKernelGGL((attn_prefill_kernel<DD, DD, WW, true>),                \
                     dim3((unsigned)(tiles * Hkv * B)), dim3(256), 0,        \
                     current_stream(), q, k, v, (const short*)nullptr, out,  \
                     qs, cs, cs, os, G, Hkv, T, Smax, tiles, 0, window,      \
                     1.44269504f, false, md)
#define LAUNCH_PM_W(DD)               \
  do {                                \
    if (window > 0) LAUNCH_PM(DD, true); \
    else LAUNCH_PM(DD, false);        \
  } while (0)
  if (D == 128) LAUNCH_PM_W(128);
  else if (D == 96) LAUNCH_PM_W(96);
  else LAUNCH_PM_W(64);
#undef LAUNCH_PM
#undef LAUNCH_PM_W
  return true;
}

}  // namespace dnet
