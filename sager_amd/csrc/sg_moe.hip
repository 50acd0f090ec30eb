// sg_moe.hip - standalone router top-k, SiLU and combine launchers on gfx950
// (the per-stage operators of the reference's MoE dispatch; the fused layer
// is in sg_layer.hip).  Router moe.cu:25-85 / 165-234, SiLU
// norm_rotary.cu:133-160 with the CPU chain's fp32 order q4_avx2.cpp:187-191,
// combine moe.cu:265-280; fp16-buffer twins of SiLU and the combine, the
// shared-expert sigmoid gate (norm_rotary.cu:177-184, moe.cu:282-292) and
// the fp32 x fp16 GEMV that produces gate and router logits
// (q4_k.cu:133-149, 285-303).
#include <type_traits>

#include "sg_common.hpp"
#include "sg_router.hpp"

namespace sg {

constexpr int kMaxExperts = 1024;
constexpr int kMaxK = 32;

__host__ __device__ inline int round4(int n) { return (n + 3) & ~3; }
__host__ __device__ inline int lpr_of(int nb) {
  int l = 1;
  while (l < nb) l <<= 1;
  return l;
}

template <int PL>
__global__ void __launch_bounds__(64) router_kernel(const float* __restrict__ logits,
                                                    int* __restrict__ idx,
                                                    float* __restrict__ weight, int n_expert,
                                                    int k, int stride, float shared_w) {
  __shared__ __attribute__((aligned(16))) float ev[64 * PL];
  const long long row = blockIdx.x;
  router_wave<PL>(logits + row * n_expert, n_expert, k, shared_w, idx + row * stride,
                  weight + row * stride, ev, threadIdx.x);
}

// four SiLU products per thread through the table exp (silu_mul_tab_n),
// the prefill gate/up kernel's arithmetic
__global__ void __launch_bounds__(256) silu_kernel(float* __restrict__ out,
                                                   const float* __restrict__ g,
                                                   const float* __restrict__ u, long long n) {
  __shared__ double tab[64];
  if (threadIdx.x < 64) tab[threadIdx.x] = kExp2Tab64[threadIdx.x];
  __syncthreads();
  const long long i0 = (static_cast<long long>(blockIdx.x) * 256 + threadIdx.x) * 4;
  float gv[4], uv[4], hv[4];
#pragma unroll
  for (int j = 0; j < 4; ++j) {
    const long long i = i0 + j < n ? i0 + j : n - 1;
    gv[j] = g[i];
    uv[j] = u[i];
  }
  silu_mul_tab_n<4>(gv, uv, hv, tab);
#pragma unroll
  for (int j = 0; j < 4; ++j)
    if (i0 + j < n) out[i0 + j] = hv[j];
}

__global__ void __launch_bounds__(256) combine_kernel(float* out, const float* residual,
                                                      const float* __restrict__ ys,
                                                      const float* __restrict__ w, int n_used,
                                                      int hidden) {
  const int i = blockIdx.x * 256 + threadIdx.x;
  const long long r = blockIdx.y;
  if (i >= hidden) return;
  float acc = residual ? residual[r * hidden + i] : 0.f;
  const float* yr = ys + r * (n_used + 1) * static_cast<long long>(hidden) + i;
  const float* wr = w + r * (n_used + 1);
  for (int kk = 0; kk <= n_used; ++kk)
    acc = __builtin_fmaf(wr[kk], yr[static_cast<long long>(kk) * hidden], acc);
  out[r * hidden + i] = acc;
}


// out = f16(SiLU(g) * u) on fp16 buffers (norm_rotary.cu:133-141)
__global__ void __launch_bounds__(256) silu_f16_kernel(uint16_t* __restrict__ out,
                                                       const uint16_t* __restrict__ g,
                                                       const uint16_t* __restrict__ u,
                                                       long long n) {
  const long long i = static_cast<long long>(blockIdx.x) * 256 + threadIdx.x;
  if (i < n) out[i] = f16b(silu_mul(f16v(g[i]), f16v(u[i])));
}

// out[r][i] = f16(f32(out[r][i]) + sum_kk fma(w[r][kk], f32(y[r][kk][i])))
// in slot order on fp16 buffers (moe.cu:265-280)
__global__ void __launch_bounds__(256) combine_f16_kernel(uint16_t* out,
                                                          const uint16_t* __restrict__ ys,
                                                          const float* __restrict__ w,
                                                          int n_used, int hidden) {
  const int i = blockIdx.x * 256 + threadIdx.x;
  const long long r = blockIdx.y;
  if (i >= hidden) return;
  float acc = f16v(out[r * hidden + i]);
  const uint16_t* yr = ys + r * (n_used + 1) * static_cast<long long>(hidden) + i;
  const float* wr = w + r * (n_used + 1);
  for (int kk = 0; kk <= n_used; ++kk)
    acc = __builtin_fmaf(wr[kk], f16v(yr[static_cast<long long>(kk) * hidden]), acc);
  out[r * hidden + i] = f16b(acc);
}

// out[r][i] = f16(f32(out[r][i]) * sigmoid(g[r])) (moe.cu:282-292)
__global__ void __launch_bounds__(256) sigmoid_gate_f16_kernel(uint16_t* __restrict__ out,
                                                               const float* __restrict__ g,
                                                               int hidden) {
  const int i = blockIdx.x * 256 + threadIdx.x;
  const long long r = blockIdx.y;
  if (i >= hidden) return;
  const float s = sigmoid_sg(g[r]);
  out[r * hidden + i] = f16b(f16v(out[r * hidden + i]) * s);
}

// y[t][r] = W[r] . f32(x[t]) with W fp32 [n_rows][k], x fp16 [T][k]: two
// rows per one-wave workgroup, one per 32-lane half, in the reference's lane
// order (rowdot_f32_lanes32).  One wave per workgroup spreads a router's 256
// rows over 128 CUs.
__global__ void __launch_bounds__(64) gemv_f32_f16x_kernel(const float* __restrict__ w,
                                                           const uint16_t* __restrict__ x,
                                                           float* __restrict__ y, int n_rows,
                                                           int k) {
  const int l = threadIdx.x & 31;
  const int row = blockIdx.x * 2 + (threadIdx.x >> 5);
  const long long t = blockIdx.y;
  const int r = row < n_rows ? row : n_rows - 1;  // whole halves stay active for the shuffles
  const uint16_t* xt = x + t * k;
  const float v = rowdot_f32_lanes32(w + static_cast<long long>(r) * k,
                                     [&](int i) { return f16v(xt[i]); }, k, l);
  if (l == 0 && row < n_rows) y[t * n_rows + row] = v;
}

// The same for many tokens (a prefill chunk's router logits) on the fp32
// matrix cores, bit for bit: v_mfma_f32_16x16x1_4b_f32 is four independent
// 16 x 16 outer products, K = 1, each element one fused multiply-add.  The
// reference order's 32 lane sums of an output (elements l, l + 32, ...) are 32
// chains that never meet before the final tree, so each is a block of an
// accumulator of its own: eight MFMAs of four blocks (b) per 32 elements.  Two
// waves share a tile of 16 rows x 16 tokens: wave h takes lane sums 16 h ..
// 16 h + 15 (four MFMAs, m), lane 16 b + i reading sums 16 h + 4 b .. + 3 of row
// i (16 B) and token i (8 B), and holds those 16 sums of its four outputs; the
// tree's first level (offset 16) meets the other wave's through LDS.
//
// A workgroup is WR x WT tiles.  W and x stream through a ring of LDS buffers,
// kRgK elements of every row at a time; chunk c of row r lies at c ^ (r & 15), so
// that the sixteen rows of a read start in different banks.  A step's operands
// are read while the previous one multiplies, over the slots' barriers too.
// What bounds it is the matrix core: one of these MFMAs takes 64 cycles, the
// vector ALU's rate.  2048 tokens x 256 rows x k 2048: 229 -> 29.0 us (74
// TFLOP/s), where a half-wave per output re-read 12 KB for each.
typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef float f32x16 __attribute__((ext_vector_type(16)));
constexpr int kRgK = 128;    // elements per ring slot: 32 chunks of a W row, 16 of an x row
template <int WR, int WT, int Ring>
struct RgTile {
  static constexpr int ring = Ring;
  static constexpr int rows = 16 * WR, toks = 16 * WT, waves = 2 * WR * WT;
  static constexpr int w_inst = rows * 32 / 64, x_inst = toks * 16 / 64;  // 1-KB copies per slot
  static constexpr int n_inst = w_inst + x_inst;
  static_assert(n_inst % waves == 0, "every wave issues the same number of copies");
  static constexpr int mine = n_inst / waves;
  static constexpr int slot_words = n_inst * 256;
  static constexpr size_t lds = static_cast<size_t>(ring) * slot_words * 4;
  static_assert(lds >= waves * 8192, "the final exchange fits the ring");
};
// The tiles' time is their chain, k / 32 steps of four MFMAs (11.4 us at k =
// 2048 however few tiles), the row-per-half-wave kernel's grows with the
// outputs: 256 x 2048 at 57 tokens 8.6 us against 11.4 for the tiles, at 128
// tokens 16.6 / 11.5, 60 x 1280 at 64 tokens 3.4 / 8.2, at 509 11.6 / 8.4.
// Tiles of 32 x 32 read a third less through L2 and win once they fill
// the chip (256 x 2048 at 509 tokens 15.6 against 11.7 us for 16 x 32, at 1024
// 16.9 / 17.1, at 2048 29.0 / 31.5).
constexpr long long kTileOutputs = 96 * 256, kBigTileOutputs = 1024 * 256;

template <int WR, int WT, int kRgRing>
__global__ void __launch_bounds__(128 * WR * WT) gemv_f32_f16x_tile_kernel(
    const float* __restrict__ w, const uint16_t* __restrict__ x, float* __restrict__ y, int n_rows,
    int k, int n_tokens, int n_rt) {
  using Tile = RgTile<WR, WT, kRgRing>;
  extern __shared__ __attribute__((aligned(16))) uint32_t rg_lds[];
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int r0 = blockIdx.x % n_rt * Tile::rows, t0 = blockIdx.x / n_rt * Tile::toks;
  const int h = __builtin_amdgcn_readfirstlane(wave & 1), tile = wave >> 1, wr = tile % WR, wt = tile / WR;
  const int i = lane & 15, b = lane >> 4;

  // the wave's copies of a slot: instruction wave + waves j; LDS chunk q of
  // the W part is chunk (q % 32) ^ (row & 15) of row q / 32, of the x part
  // chunk (q % 16) ^ (t & 15) of token q / 16 (rows and tokens past the end
  // repeat the last)
  const u32x4 rw = buffer_desc(w, static_cast<uint32_t>(n_rows) * k * 4u);
  const u32x4 rx = buffer_desc(x, static_cast<uint32_t>(n_tokens) * k * 2u);
  uint32_t ofs[Tile::mine];
#pragma unroll
  for (int j = 0; j < Tile::mine; ++j) {
    const int inst = wave + Tile::waves * j;
    if (inst < Tile::w_inst) {
      const int q = inst * 64 + lane, r = q >> 5, c = (q & 31) ^ (r & 15);
      ofs[j] = static_cast<uint32_t>(min(r0 + r, n_rows - 1)) * k * 4u + 16 * c;
    } else {
      const int q = (inst - Tile::w_inst) * 64 + lane, t = q >> 4, c = (q & 15) ^ (t & 15);
      ofs[j] = static_cast<uint32_t>(min(t0 + t, n_tokens - 1)) * k * 2u + 16 * c;
    }
  }
  auto issue = [&](int c, int slot) {  // elements kRgK c .. into ring slot `slot`
#pragma unroll
    for (int j = 0; j < Tile::mine; ++j) {
      const int inst = wave + Tile::waves * j;
      uint32_t* dst = rg_lds + slot * Tile::slot_words + 256 * inst;
      if (inst < Tile::w_inst) dma16(dst, ofs[j], rw, c * kRgK * 4);
      else dma16(dst, ofs[j], rx, c * kRgK * 2);
    }
  };
  const int n_c = k / kRgK;
#pragma unroll
  for (int c = 0; c < kRgRing - 1; ++c)
    if (c < n_c) issue(c, c);

  f32x16 acc[4] = {};
  f32x4 av[2];
  uint2 hv[2];
  // Slot c has landed once only the next slots' copies are left (at the end:
  // none); after the barrier every wave's have, and slot c - 1 is free.
  int slot = 0, free = kRgRing - 1;  // of the chunk being read, of the next to issue
  auto enter = [&](int c) {
    wait_vm_sets<1, (kRgRing - 2) * Tile::mine>(c + kRgRing - 2 < n_c);
    bar();
    if (c + kRgRing - 1 < n_c) issue(c + kRgRing - 1, free);
    free = free + 1 == kRgRing ? 0 : free + 1;
  };
  // the lane's word of W and x in a slot at step j (chunk 8 j + 4 h + b and 4 j
  // + 2 h + b / 2 of its rows, placed as above)
  int aw[kRgK / 32], ax[kRgK / 32];
#pragma unroll
  for (int j = 0; j < kRgK / 32; ++j) {
    aw[j] = (16 * wr + i) * 128 + 4 * ((8 * j + 4 * h + b) ^ i);
    ax[j] = Tile::w_inst * 256 + (16 * wt + i) * 64 + 4 * ((4 * j + 2 * h + (b >> 1)) ^ i) +
            2 * (b & 1);
  }
  auto read = [&](int j, int o) {  // step j of the slot into operand set o
    const uint32_t* s = rg_lds + slot * Tile::slot_words;
    av[o] = *reinterpret_cast<const f32x4*>(s + aw[j]);
    hv[o] = *reinterpret_cast<const uint2*>(s + ax[j]);
  };
  enter(0);
  read(0, 0);
  for (int c = 0; c < n_c; ++c) {
#pragma unroll
    for (int j = 0; j < kRgK / 32; ++j) {
      const int o = j & 1;
      // the next step's reads stay in front of this one's MFMAs (the
      // compiler would move them down to their use and wait there)
      const float bv[4] = {f16v(hv[o].x & 0xFFFFu), f16v(hv[o].x >> 16), f16v(hv[o].y & 0xFFFFu),
                           f16v(hv[o].y >> 16)};
      if (j + 1 < kRgK / 32) {
        read(j + 1, o ^ 1);
      } else if (c + 1 < n_c) {
        enter(c + 1);
        slot = slot + 1 == kRgRing ? 0 : slot + 1;
        read(0, o ^ 1);
      }
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int m = 0; m < 4; ++m)
        acc[m] = __builtin_amdgcn_mfma_f32_16x16x1f32(av[o][m], bv[m], acc[m], 0, 0, 0);
      __builtin_amdgcn_sched_barrier(0);
    }
  }
  // Lane sum 16 h + 4 q + m of the lane's output r (row 4 b + r, token i) is
  // element 4 q + r of acc[m]; the tree adds at offsets 16, 8, 4, 2, 1.  Wave
  // h gives the other its sums of outputs 2 (1 - h), 2 (1 - h) + 1 and finishes
  // outputs 2 h, 2 h + 1 (the sum of two is the same in either order).
  bar();  // the ring is free
  float* ex = reinterpret_cast<float*>(rg_lds) + 2048 * wave + lane;  // [32][64] per wave
  const float* ox = reinterpret_cast<const float*>(rg_lds) + 2048 * (wave ^ 1) + lane;
  const int t = t0 + 16 * wt + i;
  auto finish = [&](auto hc) {
    constexpr int H = decltype(hc)::value;
#pragma unroll
    for (int m = 0; m < 4; ++m)
#pragma unroll
      for (int q = 0; q < 4; ++q)
#pragma unroll
        for (int u = 0; u < 2; ++u) ex[64 * (8 * m + 2 * q + u)] = acc[m][4 * q + 2 * (1 - H) + u];
    bar();
#pragma unroll
    for (int u = 0; u < 2; ++u) {
      float v[4];
#pragma unroll
      for (int m = 0; m < 4; ++m) {
        float s[4];
#pragma unroll
        for (int q = 0; q < 4; ++q) s[q] = acc[m][4 * q + 2 * H + u] + ox[64 * (8 * m + 2 * q + u)];
        v[m] = (s[0] + s[2]) + (s[1] + s[3]);
      }
      const int row = r0 + 16 * wr + 4 * b + 2 * H + u;
      if (row < n_rows && t < n_tokens)
        y[static_cast<long long>(t) * n_rows + row] = (v[0] + v[2]) + (v[1] + v[3]);
    }
  };
  if (h) finish(std::integral_constant<int, 1>{});
  else finish(std::integral_constant<int, 0>{});
}

// Router GEMV and top-k of one token in one launch (mmq.cu:459-511): the
// logits y[e] = W[e] . f32(x) in gemv_f32_f16x_kernel's lane order (so bit
// for bit sg_gemv_f32_out_f16x's), eight rows per workgroup; the workgroup
// that arrives last (a counter, no waiting) routes them with router_wave
// (sg_router_topk's semantics) and resets the counter.  Logits and counter
// are file-scope device arrays: one set per GPU, so calls that overlap on
// one GPU race.  Only the k routed slots are written (the shared slot k of
// weight is left as it is, as the reference's fused kernel does).
__device__ float g_router_logits[kMaxExperts];
__device__ unsigned int g_router_arrivals;

template <int PL>
__global__ void __launch_bounds__(256) router_fused_kernel(const float* __restrict__ w,
                                                           const uint16_t* __restrict__ x,
                                                           int* __restrict__ idx,
                                                           float* __restrict__ weight,
                                                           int n_expert, int k, int hidden) {
  __shared__ __attribute__((aligned(16))) float ev[64 * PL];
  __shared__ bool s_last;
  const int l = threadIdx.x & 31;
  const int row = blockIdx.x * 8 + (threadIdx.x >> 5);
  const int r = row < n_expert ? row : n_expert - 1;
  const float v = rowdot_f32_lanes32(w + static_cast<long long>(r) * hidden,
                                     [&](int i) { return f16v(x[i]); }, hidden, l);
  if (l == 0 && row < n_expert) g_router_logits[row] = v;
  __threadfence();  // this workgroup's logits, visible before its arrival
  __syncthreads();
  if (threadIdx.x == 0)
    s_last = atomicAdd(&g_router_arrivals, 1u) == gridDim.x - 1;
  __syncthreads();
  if (!s_last) return;
  __threadfence();  // every other workgroup's logits
  if (threadIdx.x < 64)
    router_wave<PL>(g_router_logits, n_expert, k, 0.f, idx, weight, ev, threadIdx.x, false);
  if (threadIdx.x == 0) atomicExch(&g_router_arrivals, 0u);  // for the next launch
}

}  // namespace sg

using namespace sg;

extern "C" {

int sg_router_topk_fused(const float* w, const uint16_t* x, int* idx, float* weight, int n_expert,
                         int n_expert_used, int hidden, void* stream) {
  const char* nm = "sg_router_topk_fused";
  if (!w || !x || !idx || !weight) return set_error(SG_ERR_INVALID_ARGUMENT, "%s: null pointer", nm);
  if (n_expert <= 0 || n_expert > kMaxExperts || n_expert_used <= 0 ||
      n_expert_used > n_expert || n_expert_used > 64 || hidden <= 0)
    return set_error(SG_ERR_GEOMETRY, "%s: n_expert=%d (<=%d) n_expert_used=%d hidden=%d", nm,
                     n_expert, kMaxExperts, n_expert_used, hidden);
  hipStream_t s = static_cast<hipStream_t>(stream);
  const dim3 grid((n_expert + 7) / 8);
  auto launch = [&](auto kern) {
    hipLaunchKernelGGL(kern, grid, dim3(256), 0, s, w, x, idx, weight, n_expert, n_expert_used,
                       hidden);
  };
  if (n_expert <= 64) launch(router_fused_kernel<1>);
  else if (n_expert <= 128) launch(router_fused_kernel<2>);
  else if (n_expert <= 256) launch(router_fused_kernel<4>);
  else if (n_expert <= 512) launch(router_fused_kernel<8>);
  else launch(router_fused_kernel<16>);
  return check_launch(nm);
}


int sg_router_topk(const float* logits, int* idx, float* weight, int n_expert, int n_expert_used,
                   int idx_stride, int n_rows, float shared_w, void* stream) {
  if (!logits || !idx || !weight)
    return set_error(SG_ERR_INVALID_ARGUMENT, "sg_router_topk: null pointer");
  if (n_expert <= 0 || n_expert > kMaxExperts || n_expert_used <= 0 ||
      n_expert_used > n_expert || idx_stride < n_expert_used + 1 || n_rows <= 0)
    return set_error(SG_ERR_GEOMETRY,
                     "sg_router_topk: n_expert=%d (<=%d) n_expert_used=%d idx_stride=%d n_rows=%d",
                     n_expert, kMaxExperts, n_expert_used, idx_stride, n_rows);
  hipStream_t s = static_cast<hipStream_t>(stream);
  // experts per lane: the smallest power of two that covers n_expert
  auto launch = [&](auto kern) {
    hipLaunchKernelGGL(kern, dim3(n_rows), dim3(64), 0, s, logits, idx, weight, n_expert,
                       n_expert_used, idx_stride, shared_w);
  };
  if (n_expert <= 64) launch(router_kernel<1>);
  else if (n_expert <= 128) launch(router_kernel<2>);
  else if (n_expert <= 256) launch(router_kernel<4>);
  else if (n_expert <= 512) launch(router_kernel<8>);
  else launch(router_kernel<16>);
  return check_launch("sg_router_topk");
}

int sg_silu_mul(float* out, const float* g, const float* u, int n, void* stream) {
  if (!out || !g || !u) return set_error(SG_ERR_INVALID_ARGUMENT, "sg_silu_mul: null pointer");
  if (n <= 0) return set_error(SG_ERR_GEOMETRY, "sg_silu_mul: n=%d", n);
  hipLaunchKernelGGL(silu_kernel, dim3((n + 1023) / 1024), dim3(256), 0,
                     static_cast<hipStream_t>(stream), out, g, u, static_cast<long long>(n));
  return check_launch("sg_silu_mul");
}

int sg_moe_combine(float* out, const float* residual, const float* expert_y, const float* weight,
                   int n_used, int hidden, int n_rows, void* stream) {
  if (!out || !expert_y || !weight)
    return set_error(SG_ERR_INVALID_ARGUMENT, "sg_moe_combine: null pointer");
  if (n_used < 0 || hidden <= 0 || n_rows <= 0 || n_rows > 65535)
    return set_error(SG_ERR_GEOMETRY, "sg_moe_combine: n_used=%d hidden=%d n_rows=%d", n_used,
                     hidden, n_rows);
  hipLaunchKernelGGL(combine_kernel, dim3((hidden + 255) / 256, n_rows), dim3(256), 0,
                     static_cast<hipStream_t>(stream), out, residual, expert_y, weight, n_used,
                     hidden);
  return check_launch("sg_moe_combine");
}

int sg_silu_mul_f16(uint16_t* out, const uint16_t* g, const uint16_t* u, int rows, int n_ff,
                    void* stream) {
  if (!out || !g || !u) return set_error(SG_ERR_INVALID_ARGUMENT, "sg_silu_mul_f16: null pointer");
  if (rows <= 0 || n_ff <= 0)
    return set_error(SG_ERR_GEOMETRY, "sg_silu_mul_f16: rows=%d n_ff=%d", rows, n_ff);
  const long long n = static_cast<long long>(rows) * n_ff;
  if ((n + 255) / 256 > 0x7fffffffLL)
    return set_error(SG_ERR_GEOMETRY, "sg_silu_mul_f16: rows*n_ff=%lld too large", n);
  hipLaunchKernelGGL(silu_f16_kernel, dim3(static_cast<unsigned>((n + 255) / 256)), dim3(256), 0,
                     static_cast<hipStream_t>(stream), out, g, u, n);
  return check_launch("sg_silu_mul_f16");
}

int sg_moe_combine_batched_f16(uint16_t* out, const uint16_t* expert_y, const float* weight,
                               int n_used, int hidden, int n_rows, void* stream) {
  if (!out || !expert_y || !weight)
    return set_error(SG_ERR_INVALID_ARGUMENT, "sg_moe_combine_batched_f16: null pointer");
  if (n_used < 0 || hidden <= 0 || n_rows <= 0 || n_rows > 65535)
    return set_error(SG_ERR_GEOMETRY, "sg_moe_combine_batched_f16: n_used=%d hidden=%d n_rows=%d",
                     n_used, hidden, n_rows);
  hipLaunchKernelGGL(combine_f16_kernel, dim3((hidden + 255) / 256, n_rows), dim3(256), 0,
                     static_cast<hipStream_t>(stream), out, expert_y, weight, n_used, hidden);
  return check_launch("sg_moe_combine_batched_f16");
}

int sg_sigmoid_gate_scalar_batched_f16(uint16_t* out, const float* g, int n_rows, int hidden,
                                       void* stream) {
  if (!out || !g)
    return set_error(SG_ERR_INVALID_ARGUMENT, "sg_sigmoid_gate_scalar_f16: null pointer");
  if (n_rows <= 0 || n_rows > 65535 || hidden <= 0)
    return set_error(SG_ERR_GEOMETRY, "sg_sigmoid_gate_scalar_f16: n_rows=%d hidden=%d", n_rows,
                     hidden);
  hipLaunchKernelGGL(sigmoid_gate_f16_kernel, dim3((hidden + 255) / 256, n_rows), dim3(256), 0,
                     static_cast<hipStream_t>(stream), out, g, hidden);
  return check_launch("sg_sigmoid_gate_scalar_f16");
}

int sg_sigmoid_gate_scalar_f16(uint16_t* out, const float* g, int n, void* stream) {
  return sg_sigmoid_gate_scalar_batched_f16(out, g, 1, n, stream);
}

int sg_gemv_f32_out_f16x(const float* w, const uint16_t* x, float* y, int n_rows, int k,
                         int n_tokens, void* stream) {
  if (!w || !x || !y) return set_error(SG_ERR_INVALID_ARGUMENT, "sg_gemv_f32_out_f16x: null pointer");
  if (n_rows <= 0 || k <= 0 || n_tokens <= 0 || n_tokens > 65535)
    return set_error(SG_ERR_GEOMETRY, "sg_gemv_f32_out_f16x: n_rows=%d k=%d n_tokens=%d", n_rows,
                     k, n_tokens);
  hipStream_t s = static_cast<hipStream_t>(stream);
  // The tiles copy 16-B chunks of whole kRgK-element runs through 32-bit buffer
  // offsets
  const long long outs = static_cast<long long>(n_rows) * n_tokens;
  const bool tiles = k % kRgK == 0 && reinterpret_cast<uintptr_t>(w) % 16 == 0 &&
                     reinterpret_cast<uintptr_t>(x) % 16 == 0 &&
                     static_cast<long long>(n_rows) * k * 4 < 0x80000000LL &&
                     static_cast<long long>(n_tokens) * k * 2 < 0x80000000LL;
  auto tiled = [&](auto tile, auto kern) {
    using Tile = decltype(tile);
    const int n_rt = (n_rows + Tile::rows - 1) / Tile::rows;
    const int n_tt = (n_tokens + Tile::toks - 1) / Tile::toks;
    hipLaunchKernelGGL(kern, dim3(n_rt * n_tt), dim3(64 * Tile::waves), Tile::lds, s, w, x, y,
                       n_rows, k, n_tokens, n_rt);
  };
  if (tiles && outs >= kBigTileOutputs)
    tiled(RgTile<2, 2, 3>{}, gemv_f32_f16x_tile_kernel<2, 2, 3>);
  else if (tiles && outs >= kTileOutputs)
    tiled(RgTile<1, 2, 5>{}, gemv_f32_f16x_tile_kernel<1, 2, 5>);
  else
    hipLaunchKernelGGL(gemv_f32_f16x_kernel, dim3((n_rows + 1) / 2, n_tokens), dim3(64), 0, s, w, x,
                       y, n_rows, k);
  return check_launch("sg_gemv_f32_out_f16x");
}

}  // extern "C"
