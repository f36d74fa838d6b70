// Routed experts of a prompt (gfx950): the entries (row, choice), sorted by
// expert (moe_plan), through gate/up, activation and down in two launches.
//
//   moe_tiles         the sorted entries cut into row tiles, without host work
//   moe_prompt        one product of all experts over their tiles
//
// No host synchronisation: the grid is an upper bound of the tiles that any
// routing can need, workgroups beyond them end at once.
#include "common.h"

namespace dnet {

namespace {

using bf16x8 = __attribute__((ext_vector_type(8))) __bf16;
using f32x4 = __attribute__((ext_vector_type(4))) float;
using i32x4 = __attribute__((ext_vector_type(4))) int;

constexpr int kMaxExperts = 128;     // of one launch (kernel arguments: 3 KB)
// largest row tile; int8 needs the registers of a quarter for conversions
constexpr int tile_rows(bool q8) { return q8 ? 96 : 128; }
constexpr int kTileInts = 8;         // expert, row, rows, expert's first, its number

// one expert's weights, scales (int8) and bias (or null), by place in the bank
struct Experts {
  const void* w[kMaxExperts];
  const short* s[kMaxExperts];
  const short* b[kMaxExperts];
};

// One wave. An expert's entries are divided evenly, in 16s, over as few tiles
// of up to `tile` rows as hold them. tab[0]: the number of tiles.
__global__ __launch_bounds__(64) void moe_tiles_kernel(
    const int* __restrict__ counts, int* __restrict__ tab, const int E,
    const int n, const int tile) {
  const int lane = threadIdx.x;
  int cnt[2], need[2];
#pragma unroll
  for (int j = 0; j < 2; ++j) {
    const int e = lane * 2 + j;
    cnt[j] = e < E ? counts[e] : 0;
    need[j] = (cnt[j] + tile - 1) / tile;
  }
  int rows = cnt[0] + cnt[1], tiles = need[0] + need[1];
#pragma unroll
  for (int off = 1; off < 64; off <<= 1) {
    const int r = __shfl_up(rows, off, 64), t = __shfl_up(tiles, off, 64);
    if (lane >= off) {
      rows += r;
      tiles += t;
    }
  }
  // entries of experts that are not in the bank (number -1) stand first
  const int skip = n - __shfl(rows, 63, 64);
  if (lane == 63) tab[0] = tiles;
  int row = skip + rows - cnt[0] - cnt[1];
  int first = tiles - need[0] - need[1];
#pragma unroll
  for (int j = 0; j < 2; ++j) {
    if (need[j] == 0) continue;
    const int per = ((cnt[j] + need[j] - 1) / need[j] + 15) & ~15;
    for (int i = 0; i < need[j]; ++i) {
      int* p = tab + kTileInts * (1 + first + i);
      p[0] = lane * 2 + j;
      p[1] = row + i * per;
      p[2] = min(per, cnt[j] - i * per);
      p[3] = first;
      p[4] = need[j];
    }
    row += cnt[j];
    first += need[j];
  }
}

__device__ __forceinline__ float prompt_glu(int kind, float g, float u,
                                            float alpha, float limit) {
  if (kind == 0) return g / (1.f + __expf(-g)) * u;
  g = fminf(g, limit);
  u = fminf(fmaxf(u, -limit), limit);
  return (u + 1.f) * g / (1.f + __expf(-alpha * g));
}

// A tile of up to 16 MT rows and 64 columns per wave (four waves side by side:
// rows of x through LDS for all of them, weights from memory straight to the
// registers of the one wave that needs them). A step is 128 B of every weight
// row: 64 wide in bf16, 128 in int8; its x goes to LDS without passing
// registers, its weights to registers, both one step ahead. x lies in 128 B
// rows whose 16 B pieces are exchanged by row number, so that the 16 rows of a
// fragment hit all banks. int8 weights are scaled and rounded to bf16 in
// registers, as dequantizing them to memory does. KIND: 0 / 1 gated (silu /
// clamped; half of a wave's fragments are the up columns beside its gate
// columns), 2 plain, the result times the entry's routing weight.
//
// Bound by latency between the waits of a step: 2 workgroups fit a CU. Two
// conversions and a scaling per weight for each row tile cost the vector unit as
// much time as the products of 96 rows cost the matrix cores, so they stand
// between products; a fragment of x is read two ahead. Measured, MI355X, 700
// rows, 8 int8 experts of 4096 x 14336, 2 chosen: gate/up 540 us (610
// TFLOP/s), down 312 us (530); with reads and conversions before the products
// and 128-row tiles (which spill) 1065 us for both instead of 870. One expert
// after the other (dequantize, library product, host waits) 2916 us.
template <int MT, int NF, bool Q8, bool PAIR, int KIND>
__device__ __forceinline__ void moe_prompt_body(
    char* xs, const short* __restrict__ x, const char* __restrict__ w,
    const short* __restrict__ scales, const short* __restrict__ bias,
    const int* __restrict__ order, const float* __restrict__ val,
    short* __restrict__ out, const int row0, const int rows, const int nt,
    const int K, const int N, const int top, const int G,
    const unsigned xbytes, const float alpha, const float limit) {
  constexpr bool GLU = KIND != 2;
  constexpr int NC = GLU ? NF / 2 : NF;
  constexpr int H = Q8 ? 2 : 1;              // 64-wide halves of a step
  constexpr int kHalf = tile_rows(Q8) * 128; // bytes
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int lane = threadIdx.x & 63;
  const int c = lane & 15, hi = lane >> 4;
  const int n0 = (nt * 4 + wave) * (16 * NC);
  const int steps = K / (64 * H);

  unsigned wo[NF], so[NF];
  const int rb = Q8 ? K : 2 * K;
#pragma unroll
  for (int f = 0; f < NF; ++f) {
    const unsigned row = (GLU ? (f / NC) * N : 0) +
                         min(n0 + (f % NC) * 16 + c, N - 1);
    wo[f] = row * (unsigned)rb + hi * 16;
    so[f] = Q8 ? row * (unsigned)(2 * (K / G)) : 0;
  }
  // rows >= `rows` repeat the last one, never stored
  unsigned xo[MT / 2];               // bytes
#pragma unroll
  for (int i = 0; i < MT / 2; ++i) {
    const int r = row0 + min((wave * (MT / 2) + i) * 8 + (lane >> 3), rows - 1);
    xo[i] = (unsigned)(KIND != 2 ? order[r] / top : r) *
                (unsigned)(2 * K) + (((lane & 7) ^ (lane >> 3)) * 16);
  }
  f32x4 acc[MT][NF];
#pragma unroll
  for (int m = 0; m < MT; ++m)
#pragma unroll
    for (int f = 0; f < NF; ++f) acc[m][f] = {0.f, 0.f, 0.f, 0.f};

  // buffer descriptors: a lane's 32-bit offset stays fixed, the step is a scalar
  auto buf = [](const void* p, unsigned bytes) {
    return __builtin_amdgcn_make_buffer_rsrc(const_cast<void*>(p), 0,
                                             (int)bytes, 0x00027000);
  };
  const unsigned wrows = (GLU ? 2 : 1) * N;
  const auto xd = buf(x, xbytes), wd = buf(w, wrows * (unsigned)rb),
             sd = buf(scales, Q8 ? wrows * (unsigned)(2 * (K / G)) : 0);
  struct Weights { i32x4 q[NF][2]; unsigned s[NF]; };
  auto stage = [&](const int at, const int s) {
#pragma unroll
    for (int h = 0; h < H; ++h)
#pragma unroll
      for (int i = 0; i < MT / 2; ++i)
        __builtin_amdgcn_raw_ptr_buffer_load_lds(
            xd,
            (__attribute__((address_space(3))) void*)(
                xs + (at * H + h) * kHalf + (wave * (MT / 2) + i) * 1024),
            16, xo[i], (s * H + h) * 128, 0, 0);
  };
  auto load = [&](Weights& q, const int s) {
#pragma unroll
    for (int f = 0; f < NF; ++f) {
#pragma unroll
      for (int u = 0; u < 2; ++u)
        q.q[f][u] = __builtin_bit_cast(
            i32x4, __builtin_amdgcn_raw_buffer_load_b128(
                       wd, wo[f], s * 128 + u * 64, 0));
      if (Q8)
        q.s[f] = PAIR ? __builtin_amdgcn_raw_buffer_load_b32(sd, so[f], s * 4, 0)
                      : (unsigned)__builtin_amdgcn_raw_buffer_load_b16(
                            sd, so[f], s * 128 / G * 2, 0);
    }
  };
  // fragment f of piece kk (32 wide) of a step
  auto weight = [&](const Weights& q, const int kk, const int f) {
    if (!Q8) return __builtin_bit_cast(bf16x8, q.q[f][kk]);
    const float sc = __builtin_bit_cast(
        float, PAIR && kk >= 2 ? q.s[f] & 0xffff0000u : q.s[f] << 16);
    // converted here, not where it was loaded (4x the registers)
    int raw[2] = {q.q[f][kk / 2][2 * (kk & 1)], q.q[f][kk / 2][2 * (kk & 1) + 1]};
    asm volatile("" : "+v"(raw[0]), "+v"(raw[1]));
    bf16x8 v;
#pragma unroll
    for (int k = 0; k < 8; ++k)
      v[k] = (__bf16)(sc * (float)(signed char)(raw[k / 4] >> (8 * (k & 3))));
    return v;
  };
  // Rows of x are read kAhead fragments ahead; the next piece's weights are
  // converted in the shadow of this one's products.
  constexpr int kPieces = 2 * H, kFrags = kPieces * MT, kAhead = 2;
  auto mul = [&](const Weights& q, const int half) {
    const char* xb = xs + half * H * kHalf + c * 128;
    auto row = [&](const int i) {
      const int kk = i / MT, m = i % MT;
      return *reinterpret_cast<const bf16x8*>(
          xb + kk / 2 * kHalf + m * 2048 +
          ((((kk & 1) * 4 + hi) ^ (c & 7)) * 16));
    };
    bf16x8 xf[kAhead + 1], wf[2][NF];
#pragma unroll
    for (int i = 0; i < kAhead; ++i) xf[i] = row(i);
#pragma unroll
    for (int f = 0; f < NF; ++f) wf[0][f] = weight(q, 0, f);
#pragma unroll
    for (int i = 0; i < kFrags; ++i) {
      const int kk = i / MT, m = i % MT;
      if (i + kAhead < kFrags) xf[(i + kAhead) % (kAhead + 1)] = row(i + kAhead);
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int f = 0; f < NF; ++f)
        acc[m][f] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(
            xf[i % (kAhead + 1)], wf[kk & 1][f], acc[m][f], 0, 0, 0);
      if (kk + 1 < kPieces)
#pragma unroll
        for (int f = 0; f < NF; ++f)
          if (f * MT / NF == m) wf[(kk + 1) & 1][f] = weight(q, kk + 1, f);
    }
  };
  auto ready = [&]() {
    asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)" ::: "memory");
    asm volatile("s_barrier" ::: "memory");
  };
  Weights q0, q1;
  stage(0, 0);
  load(q0, 0);
  int s = 0;
  for (; s + 2 <= steps; s += 2) {
    ready();
    stage(1, s + 1);
    load(q1, s + 1);
    __builtin_amdgcn_sched_barrier(0);
    mul(q0, 0);
    ready();
    const int n = min(s + 2, steps - 1);     // past the end: read, not used
    stage(0, n);
    load(q0, n);
    __builtin_amdgcn_sched_barrier(0);
    mul(q1, 1);
  }
  ready();
  if (s < steps) mul(q0, 0);
  // the last products' results are read below, behind branches
  asm volatile("s_nop 15\n\ts_nop 15" ::: "memory");

#pragma unroll
  for (int m = 0; m < MT; ++m)
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const int t = m * 16 + hi * 4 + r;
      if (t >= rows) continue;
      float wt = 1.f;
      if (KIND == 2) wt = val[order[row0 + t]];
#pragma unroll
      for (int f = 0; f < NC; ++f) {
        const int n = n0 + f * 16 + c;
        if (n >= N) continue;
        float v = acc[m][f][r];
        if (bias != nullptr) v += bits2f(bias[n]);
        if constexpr (GLU) {
          float u = acc[m][NC + f][r];
          if (bias != nullptr) u += bits2f(bias[N + n]);
          v = prompt_glu(KIND, v, u, alpha, limit);
        } else {
          v = wt > 0.f ? v * wt : 0.f;
        }
        out[(int64_t)(row0 + t) * N + n] = f2bits(v);
      }
    }
}

// grid: 8 column tiles (one per XCD) x groups of them x tiles, in an order that
// keeps an expert's rows and a group's weights in L2: all groups of one expert
// before the next expert, all row tiles of one group next to each other.
template <int NF, bool Q8, bool PAIR, int KIND>
__global__ __launch_bounds__(256, 2) void moe_prompt_kernel(
    const Experts ex, const short* __restrict__ x,
    const int* __restrict__ order, const float* __restrict__ val,
    const int* __restrict__ tab, short* __restrict__ out, const int K,
    const int N, const int top, const int G, const unsigned xbytes,
    const float alpha, const float limit) {
  constexpr int H = Q8 ? 2 : 1;
  __shared__ __attribute__((aligned(1024))) char xs[2 * H * tile_rows(Q8) * 128];
  const int cols = 64 * (KIND == 2 ? NF : NF / 2);
  const int nts = (N + cols - 1) / cols;
  const int groups = (nts + 7) / 8;
  const int at = blockIdx.x / 8;
  int t = at / groups;
  if (t >= tab[0]) return;
  const int* p = tab + kTileInts * (1 + t);
  const int e = __builtin_amdgcn_readfirstlane(p[0]);
  const int first = p[3], num = p[4];
  const int local = at - first * groups;
  const int nt = local / num * 8 + blockIdx.x % 8;
  if (nt >= nts) return;
  t = first + local % num;
  p = tab + kTileInts * (1 + t);
  const int row0 = __builtin_amdgcn_readfirstlane(p[1]);
  const int rows = __builtin_amdgcn_readfirstlane(p[2]);
#define MP(MM)                                                               \
  moe_prompt_body<MM, NF, Q8, PAIR, KIND>(                                   \
      xs, x, (const char*)ex.w[e], ex.s[e], ex.b[e], order, val, out, row0,  \
      rows, nt, K, N, top, G, xbytes, alpha, limit)
  if (rows <= 32) MP(2);
  else if (rows <= 64) MP(4);
  else if (Q8 || rows <= 96) MP(6);
  else MP(Q8 ? 6 : 8);
#undef MP
}

}  // namespace

// tab (int32, 8 (1 + n / tile + E) numbers): row tiles of the n entries whose
// numbers per expert moe_plan counted
void moe_tiles(torch::Tensor counts, torch::Tensor tab, int64_t n,
               int64_t tile) {
  const int64_t E = counts.numel();
  DNET_CHECK(counts.scalar_type() == torch::kInt32 && counts.is_contiguous() &&
                 E >= 1 && E <= kMaxExperts, "moe_tiles: counts int32 [E]");
  DNET_CHECK(tab.scalar_type() == torch::kInt32 && tab.is_contiguous() &&
                 tile > 0 && tile % 16 == 0 &&
                 tab.numel() >= kTileInts * (1 + n / tile + E),
             "moe_tiles: tab");
  hipLaunchKernelGGL(moe_tiles_kernel, dim3(1), dim3(64), 0, current_stream(),
                     counts.data_ptr<int>(), tab.data_ptr<int>(), (int)E,
                     (int)n, (int)tile);
}

// kind 0 / 1: out [n, I] = glu(x[order / top] Wg^T, x[order / top] Wu^T) for w
// [2 I, K] per expert; kind 2: out [n, N] = val[order] * (x w^T) for sorted
// rows x [n, K]. Entries before the first tile are not written.
void moe_prompt(torch::Tensor x, torch::Tensor order, torch::Tensor val,
                torch::Tensor tab, std::vector<torch::Tensor> w,
                std::vector<torch::Tensor> scales,
                std::vector<torch::Tensor> bias, torch::Tensor out,
                int64_t group, int64_t tile, int64_t kind, double alpha,
                double limit) {
  const int64_t E = (int64_t)w.size(), n = order.numel();
  DNET_CHECK(E >= 1 && E <= kMaxExperts && kind >= 0 && kind <= 2,
             "moe_prompt: experts");
  DNET_CHECK(x.dim() == 2 && x.scalar_type() == torch::kBFloat16 &&
                 x.is_contiguous() && out.dim() == 2 &&
                 out.scalar_type() == torch::kBFloat16 && out.is_contiguous() &&
                 out.size(0) == n, "moe_prompt: x, out bf16");
  DNET_CHECK(order.scalar_type() == torch::kInt32 && order.is_contiguous() &&
                 val.scalar_type() == torch::kFloat32 && val.is_contiguous() &&
                 val.dim() == 2 && val.numel() == n,
             "moe_prompt: order int32 [n], val fp32 [T, top]");
  const int64_t K = x.size(1), N = out.size(1);
  const int64_t WN = kind == 2 ? N : 2 * N;
  DNET_CHECK(x.size(0) == (kind == 2 ? n : val.size(0)), "moe_prompt: rows");
  const bool q8 = w[0].scalar_type() == torch::kChar;
  DNET_CHECK(tile > 0 && tile % 16 == 0 && tile <= tile_rows(q8) &&
                 tab.scalar_type() == torch::kInt32 && tab.is_contiguous() &&
                 tab.numel() >= kTileInts * (1 + n / tile + E),
             "moe_prompt: tab");
  const bool pair = q8 && group == 64;
  DNET_CHECK(q8 ? K % 128 == 0 && group > 0 && K % group == 0 &&
                      (group == 64 || group % 128 == 0)
                : K % 64 == 0, "moe_prompt: K, group");
  DNET_CHECK((int64_t)scales.size() == (q8 ? E : 0) &&
                 (bias.empty() || (int64_t)bias.size() == E),
             "moe_prompt: scales, bias");
  const int64_t rb = q8 ? K : 2 * K;
  DNET_CHECK(WN * rb < (1ll << 32) && x.numel() * 2 < (1ll << 32) &&
                 (uintptr_t)x.data_ptr() % 16 == 0, "moe_prompt: size");
  if (n == 0 || N == 0) return;
  Experts ex;
  for (int64_t e = 0; e < E; ++e) {
    DNET_CHECK(w[e].is_contiguous() && w[e].dim() == 2 &&
                   w[e].scalar_type() == (q8 ? torch::kChar : torch::kBFloat16) &&
                   w[e].size(0) == WN && w[e].size(1) == K &&
                   (uintptr_t)w[e].data_ptr() % 16 == 0 && w[e].is_cuda(),
               "moe_prompt: weights");
    ex.w[e] = w[e].data_ptr();
    ex.s[e] = nullptr;
    ex.b[e] = nullptr;
    if (q8) {
      DNET_CHECK(scales[e].is_contiguous() &&
                     scales[e].scalar_type() == torch::kBFloat16 &&
                     scales[e].numel() == WN * (K / group) &&
                     (uintptr_t)scales[e].data_ptr() % 4 == 0,
                 "moe_prompt: scales");
      ex.s[e] = (const short*)scales[e].data_ptr();
    }
    if (!bias.empty()) {
      DNET_CHECK(bias[e].is_contiguous() && bias[e].numel() == WN &&
                     bias[e].scalar_type() == torch::kBFloat16,
                 "moe_prompt: bias");
      ex.b[e] = (const short*)bias[e].data_ptr();
    }
  }
  const int64_t tiles = n / tile + std::min(E, n);
  // 128 columns per workgroup instead of 256 where those give a CU less than 3
  // workgroups: 700 rows as above 985 -> 896 us in all, 1500 rows 1669 -> 1572
  const bool half = kind == 2 && tiles * cdiv(N, 256) < 768;
  const int64_t groups = cdiv(cdiv(N, kind == 2 && !half ? 256 : 128), 8);
  const int64_t grid = tiles * groups * 8;
  DNET_CHECK(grid < (1ll << 31), "moe_prompt: grid");
#define MP(FF, QQ, PP, KK)                                                       \
  hipLaunchKernelGGL((moe_prompt_kernel<FF, QQ, PP, KK>), dim3((unsigned)grid),  \
                     dim3(256), 0, current_stream(), ex,                     \
                     (const short*)x.data_ptr(), order.data_ptr<int>(),      \
                     val.data_ptr<float>(), tab.data_ptr<int>(),             \
                     (short*)out.data_ptr(), (int)K, (int)N,                 \
                     (int)val.size(1), (int)std::max<int64_t>(group, 64),    \
                     (unsigned)(x.numel() * 2),                              \
                     (float)alpha, (float)limit)
#define MP_K(QQ, PP)              \
  do {                            \
    if (kind == 0) MP(4, QQ, PP, 0); \
    else if (kind == 1) MP(4, QQ, PP, 1); \
    else if (half) MP(2, QQ, PP, 2); \
    else MP(4, QQ, PP, 2);        \
  } while (0)
  if (pair) MP_K(true, true);
  else if (q8) MP_K(true, false);
  else MP_K(false, false);
#undef MP_K
#undef MP
}

}  // namespace dnet
