// sg_gemv.hip - the Q4_K x Q8_K GEMV family on gfx950.
//
// Work unit: a wave owns a row group of 64/lpr rows, lpr = the power of two
// >= nb (nb = k/256 super-blocks per row).  The group's bytes are contiguous
// in HBM, so the wave streams them into its own 9 KB LDS buffer with
// global_load_lds_dwordx4 (1 KB of consecutive memory per instruction, no
// registers held while in flight).  Lane l then reads super-block (l mod
// lpr) of row (l / lpr) from LDS (144-B stride: conflict-free), computes the
// eight int32 sub-block dots with v_dot4_i32_i8 against its Q8_K activation
// block kept in registers, applies the fp32 super-block epilogue, and the
// lpr block sums of a row are added in block order (the reference's
// acc += sum order, q4_avx2.cpp:130-143) with DPP lane shifts.  The next group's copy is issued
// as soon as the block is in registers, so it overlaps the arithmetic.
//
// Small matrices (up to 262144 super-blocks) take gemv_lat_kernel instead:
// four lanes per super-block, loads straight into registers, one pass.
//
// Several tokens take int8 matrix cores (gemv_mt_kernel, gemv_mtw_kernel), two to
// four of them in some large matrices the sdot4 kernel (use_batched_sdot).
//
// Reference kernels replaced: gemv_q4_k_q8 / gemv_mtok_ro_f32_kernel
// (q4_k.cu:57-91, 1360-1422, 1534-1562), gemv_q4_k_q8_batched and the mtok
// variants (q4_k.cu:218-282, 359-498), gemv_ptrs_q4_k_q8_f16out
// (q4_k.cu:184-213).
#include <algorithm>
#include <type_traits>

#include "sg_common.hpp"

namespace sg {

constexpr int kMaxNb = 64;       // k <= 16384
constexpr int kMaxTokens = 16;   // batched GEMV: the rows of an MFMA result
constexpr int kWaves = 4;        // waves per workgroup
constexpr int kBufWords = 64 * 36;  // one wave's 9216-B weight buffer
constexpr int kWgPerCu = 2;        // grid cap: workgroups per CU

struct PlainRows {
  const sg_block_q4k* w;
  int nb;
  __device__ const char* row(int r) const {
    return reinterpret_cast<const char*>(w + static_cast<long long>(r) * nb);
  }
  __device__ void stage(uint32_t*, int, int) {}
  __device__ void attach(const uint32_t*) {}
  __device__ bool contiguous(int, int) const { return true; }
  __device__ int table_words() const { return 0; }
};

// Rows of n_ptrs matrices of rows_per rows each, matrix e at ptrs[e].  With
// n_ptrs <= kMaxLdsPtrs the table is copied to LDS once per workgroup, so
// the address of a row group costs an LDS read instead of a dependent
// global load in front of every weight stream.
constexpr int kMaxLdsPtrs = 2048;
// Up to three matrices of the same K stacked: rows [0, end[0]) of w[0],
// [end[0], end[1]) of w[1], [end[1], end[2]) of w[2] (the layer's q|k|v or
// qkvz|ba projections, gemv2m/gemv3m).
struct SegRows {
  const sg_block_q4k* w[3];
  int end[3];
  int nb;
  __device__ int seg(int r) const { return r < end[0] ? 0 : (r < end[1] ? 1 : 2); }
  __device__ const char* row(int r) const {
    const int m = seg(r);
    const int lr = r - (m ? end[m - 1] : 0);
    return reinterpret_cast<const char*>(w[m] + static_cast<long long>(lr) * nb);
  }
  __device__ void stage(uint32_t*, int, int) {}
  __device__ void attach(const uint32_t*) {}
  __device__ bool contiguous(int r0, int n) const { return seg(r0) == seg(r0 + n - 1); }
  __device__ int table_words() const { return 0; }
};
typedef __attribute__((address_space(3))) const unsigned long long lds_u64;
struct TableRows {
  const sg_block_q4k* const* ptrs;
  int rows_per, nb, n_ptrs;
  int shift;  // log2(rows_per) when it is a power of two, else -1
  // the staged table, as an LDS pointer: a generic pointer would make the
  // lookup a flat load, which joins the vector-memory queue and is waited
  // for together with the weight copies in flight
  lds_u64* lds = nullptr;
  __device__ int matrix(int r) const { return shift >= 0 ? r >> shift : r / rows_per; }
  __device__ const char* row(int r) const {
    const int e = matrix(r);
    const unsigned long long base =
        lds ? lds[e] : reinterpret_cast<unsigned long long>(ptrs[e]);
    return reinterpret_cast<const char*>(base) +
           static_cast<long long>(r - e * rows_per) * nb * kQ4Bytes;
  }
  // copy the table to LDS (visible after the caller's barrier)
  __device__ void stage(uint32_t* dst, int tid, int nthreads) {
    if (n_ptrs > kMaxLdsPtrs) return;
    unsigned long long* d = reinterpret_cast<unsigned long long*>(dst);
    for (int i = tid; i < n_ptrs; i += nthreads) d[i] = reinterpret_cast<unsigned long long>(ptrs[i]);
  }
  __device__ void attach(const uint32_t* src) {
    if (n_ptrs <= kMaxLdsPtrs) lds = (lds_u64*)(src);
  }
  __device__ bool contiguous(int r0, int n) const { return matrix(r0) == matrix(r0 + n - 1); }
  // LDS words the staged table occupies (2 per pointer, when it is staged)
  __device__ int table_words() const { return n_ptrs <= kMaxLdsPtrs ? 2 * n_ptrs : 0; }
};

__host__ __device__ inline int lanes_per_row(int nb) {
  int l = 1;
  while (l < nb) l <<= 1;
  return l;
}

// Issue the copy of rows r0 .. r0+n-1 into buf.  Rows that are contiguous
// in memory (always for a plain matrix; for a table when the group does not
// straddle two matrices) stream as one range: chunk c at base + 16c, with no
// per-chunk division.
template <typename Rows>
__device__ __forceinline__ void dma_rows(const Rows& rows, int r0, int n, int nb, uint32_t* buf,
                                         int lane) {
  const int cpr = nb * 9;  // 16-B chunks per row
  if (rows.contiguous(r0, n)) {
    const char* base = rows.row(r0);
    dma_chunks<kNt>([&](int c) { return base + 16 * c; }, n * cpr, buf, lane);
  } else {
    dma_chunks<kNt>([&](int c) { return rows.row(r0 + c / cpr) + 16 * (c % cpr); }, n * cpr, buf,
               lane);
  }
}

// y[r] = W[r] . x, one token.  Wave W of the NW takes the row groups W,
// W + NW, W + 2 NW, ... (a group = 64/lpr rows, one 9 KB buffer), so that the
// chip reads one window of the matrix at a time (contiguous ranges per wave
// measured 2-4 % slower); it issues the
// next group's copy as soon as the current one has been read into
// registers, so one group is always in flight while it computes.  The row
// results stay in LDS until the wave's last group and are then written
// together: a global store between the copies would sit in the vmcnt queue
// that each copy is waited on with.  Two workgroups per CU.
// Where a row result goes: fp32 y[r] (F32Out); fp16 into the row's segment
// output (F16SegOut, gemv2m/3m); fp16 y[r] and the residual add
// res[r] = f16(f32(res[r]) + f32(y[r])) (F16ResAddOut, add_kernel's
// semantics).  fp16 conversions round to nearest even (__float2half).
struct F32Out {
  float* y;
  __device__ void store(int r, float v) const { y[r] = v; }
};
struct F16Out {
  uint16_t* y;
  __device__ void store(int r, float v) const { y[r] = f16b(v); }
};
struct F16SegOut {
  uint16_t* y[3];
  int end[3];
  __device__ void store(int r, float v) const {
    const int m = r < end[0] ? 0 : (r < end[1] ? 1 : 2);
    y[m][r - (m ? end[m - 1] : 0)] = f16b(v);
  }
};
struct F16ResAddOut {
  uint16_t* y;
  uint16_t* res;
  __device__ void store(int r, float v) const {
    const uint16_t h = f16b(v);
    y[r] = h;
    res[r] = f16b(f16v(res[r]) + f16v(h));
  }
};

template <typename Rows, typename Out, int NWV>
__global__ void __launch_bounds__(64 * NWV) gemv1_kernel(Rows rows,
                                                         const unsigned char* __restrict__ xq,
                                                         Out out, int n_rows, int nb, int lpr,
                                                         int gpw) {
  __shared__ __attribute__((aligned(16))) uint32_t wbuf[NWV][kBufWords];
  extern __shared__ __attribute__((aligned(16))) uint32_t xs_dyn[];  // nb * kXStride, table, results
  const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
  const int rpw = 64 / lpr;
  const int n_groups = (n_rows + rpw - 1) / rpw;
  const int NW = gridDim.x * NWV;
  const int g_begin = blockIdx.x * NWV + wv, g_end = n_groups;
  auto rows_of = [&](int gg) { return min(rpw, n_rows - gg * rpw); };
  // the first group's weights first: their HBM latency overlaps the staging
  if (g_begin < g_end) dma_rows(rows, g_begin * rpw, rows_of(g_begin), nb, wbuf[wv], lane);
  stage_q8k(xq, nb, xs_dyn, threadIdx.x, blockDim.x);
  uint32_t* tab = xs_dyn + nb * kXStride;  // row table, when the rows have one
  rows.stage(tab, threadIdx.x, blockDim.x);
  float* res = reinterpret_cast<float*>(tab + rows.table_words()) + wv * gpw * rpw;
  bar();
  rows.attach(tab);

  const int blk = lane & (lpr - 1);
  const int rr = lane / lpr;
  const bool active = blk < nb;
  int32_t xr[64];
  float xd = 0.f, bsf[8];
  load_x_regs(xs_dyn + (active ? blk : 0) * kXStride, xr, xd, bsf);

  for (int g = g_begin, li = 0; g < g_end; g += NW, ++li) {
    const int n = rows_of(g);
    wait_vm();  // group g has landed
    uint32_t w36[36];
    const bool live = active && rr < n;
    if (live) read_block_lds(wbuf[wv] + (rr * nb + blk) * 36, w36);
    wait_lds();
    if (g + NW < g_end) dma_rows(rows, (g + NW) * rpw, rows_of(g + NW), nb, wbuf[wv], lane);
    const float s = live ? q4k_block_dot(w36, xr, xd, bsf) : 0.f;
    const float acc = row_sum_last(s, blk, nb);
    if (blk == nb - 1 && rr < n) res[li * rpw + rr] = acc;
  }
  wait_lds();  // this wave's result writes (read back by its own lanes)
  // result li * rpw + row of the wave belongs to group g_begin + li * NW
  for (int i = lane; i < gpw * rpw; i += 64) {
    const int r = (g_begin + (i / rpw) * NW) * rpw + i % rpw;
    if (r < n_rows) out.store(r, res[i]);
  }
}

// y[r] = W[r] . x for a small matrix (latency-bound: a few MB, read in one
// pass by the whole chip).  Four lanes share a super-block, each taking one
// sub-block pair (8 qs words of weights, 16 qs words of activations), so a
// 2048 x 2048 matrix spreads over 1024 one-wave workgroups instead of 256
// waves.  Every lane loads its weight and activation words straight into
// registers at entry: no LDS, no barrier, one memory latency before the
// arithmetic.  The super-block epilogue keeps the reference's order
// (sum = fma(xd, t_s, sum) for s = 0..7, q4_avx2.cpp:30-39,134-141): the
// running sum moves from the lane of pair p to that of pair p+1 with a DPP
// row shift, and the row's block sums are then added in block order by
// row_sum_last after one lane permute.  nb <= 16 (k <= 4096).
constexpr int kLatMaxNb = 16;
constexpr int kLatWaves = 4;  // waves per workgroup
constexpr int kDppRowShr1 = 0x111;
typedef uint32_t u32x4u __attribute__((ext_vector_type(4), aligned(4)));

template <typename Rows, typename Out>
__device__ __forceinline__ void gemv_lat_body(const Rows& rows, const unsigned char* __restrict__ xq,
                                              const Out& out, int n_rows, int nb, int lg) {
  const int lpr = 1 << lg;
  const int lane = threadIdx.x & 63;
  const int wave = blockIdx.x * kLatWaves + (threadIdx.x >> 6);
  const int part = lane & 3, blk = (lane >> 2) & (lpr - 1), rr = lane >> (2 + lg);
  const int rpw = 16 >> lg;
  const int r = wave * rpw + rr;
  const bool live = blk < nb && r < n_rows;
  // every lane loads (clamped to a valid block) and dead lanes zero their
  // words afterwards: no branch, so all arguments are fetched in one round
  const u32x4* wp = reinterpret_cast<const u32x4*>(rows.row(min(r, n_rows - 1)) +
                                                   min(blk, nb - 1) * kQ4Bytes);
  u32x4 h = wp[0], qa = wp[1 + 2 * part], qb = wp[2 + 2 * part];
  const unsigned char* xb = xq + min(blk, nb - 1) * kQ8Bytes;
  const u32x4u* xp = reinterpret_cast<const u32x4u*>(xb + 4 + 64 * part);
  uint32_t xw[16];
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const u32x4u v = xp[i];
    xw[4 * i] = v.x;
    xw[4 * i + 1] = v.y;
    xw[4 * i + 2] = v.z;
    xw[4 * i + 3] = v.w;
  }
  float xd = *reinterpret_cast<const float*>(xb);
  uint32_t bs = *reinterpret_cast<const uint32_t*>(xb + 260 + 4 * part);
  if (!live) {
    h = u32x4{0u, 0u, 0u, 0u};
    qa = h;
    qb = h;
    bs = 0;
    xd = 0.f;
  }
  const uint32_t q[8] = {qa.x, qa.y, qa.z, qa.w, qb.x, qb.y, qb.z, qb.w};
  int32_t lo = 0, hi = 0;
#pragma unroll
  for (int j = 0; j < 8; ++j) {
    lo = __builtin_amdgcn_sdot4(static_cast<int>(q[j] & 0x0F0F0F0Fu), static_cast<int>(xw[j]), lo,
                                false);
    hi = __builtin_amdgcn_sdot4(static_cast<int>((q[j] >> 4) & 0x0F0F0F0Fu),
                                static_cast<int>(xw[8 + j]), hi, false);
  }
  const ScaleMins sm8 = unpack_scales(h.y, h.z, h.w);
  const float d = half_bits_to_float(h.x & 0xFFFFu);
  const float dmin = half_bits_to_float(h.x >> 16);
  const uint32_t scw = part < 2 ? sm8.sc_lo : sm8.sc_hi;
  const uint32_t mnw = part < 2 ? sm8.mn_lo : sm8.mn_hi;
  const int i0 = (2 * part) & 3;
  const float b0 = static_cast<float>(static_cast<int16_t>(bs & 0xFFFFu));
  const float b1 = static_cast<float>(static_cast<int16_t>(bs >> 16));
  const float t0 = __builtin_fmaf(d * byte_f(scw, i0), static_cast<float>(lo),
                                  -((dmin * byte_f(mnw, i0)) * b0));
  const float t1 = __builtin_fmaf(d * byte_f(scw, i0 + 1), static_cast<float>(hi),
                                  -((dmin * byte_f(mnw, i0 + 1)) * b1));
  float acc = 0.f;
#pragma unroll
  for (int j = 0; j < 4; ++j) {
    const float prev = j == 0 ? 0.f : dpp_f<kDppRowShr1>(acc);
    if (part == j) acc = __builtin_fmaf(xd, t1, __builtin_fmaf(xd, t0, prev));
  }
  // block sums (lane 4b+3 of each row) to lanes row*lpr + b
  const int c = lane & 15;
  const int src = ((c >> lg) << (2 + lg)) + 4 * (c & (lpr - 1)) + 3;
  const float sb = __builtin_bit_cast(
      float, __builtin_amdgcn_ds_bpermute(src << 2, __builtin_bit_cast(int, acc)));
  const int cb = c & (lpr - 1);
  const float row = row_sum_last(sb, cb, nb);
  const int ro = wave * rpw + (c >> lg);
  if (lane < 16 && cb == nb - 1 && ro < n_rows) out.store(ro, row);
}
template <typename Rows, typename Out>
__global__ void __launch_bounds__(64 * kLatWaves) gemv_lat_kernel(
    Rows rows, const unsigned char* __restrict__ xq, Out out, int n_rows, int nb, int lg) {
  gemv_lat_body(rows, xq, out, n_rows, nb, lg);
}
// The plain fp32 GEMV with scalar arguments only, which the code object can
// preload into SGPRs (no kernel-argument load before the first address).
__global__ void __launch_bounds__(64 * kLatWaves) gemv_lat_plain_kernel(
    const sg_block_q4k* __restrict__ w, const unsigned char* __restrict__ xq, float* y, int n_rows,
    int nb, int lg) {
  gemv_lat_body(PlainRows{w, nb}, xq, F32Out{y}, n_rows, nb, lg);
}

// y[t*n_rows + r] = W[r] . x[t] for two to four tokens of large matrices: a
// lane per super-block as in gemv1_kernel, looping over the tokens with sdot4.
// The matrix-core kernels below win outside use_batched_sdot's ranges.
template <typename Out>
__global__ void __launch_bounds__(256) gemv_batched_kernel(const sg_block_q4k* __restrict__ w,
                                                           const unsigned char* __restrict__ xq,
                                                           Out y, int n_rows,
                                                           int nb, int lpr, int n_tokens) {
  __shared__ __attribute__((aligned(16))) uint32_t wbuf[kWaves][kBufWords];
  extern __shared__ __attribute__((aligned(16))) uint32_t xs_dyn[];  // T * nb * kXStride
  const PlainRows rows{w, nb};
  const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
  const int rpw = 64 / lpr;
  const int n_groups = (n_rows + rpw - 1) / rpw;
  const int n_waves = gridDim.x * kWaves;
  int g = blockIdx.x * kWaves + wv;
  uint32_t* buf = wbuf[wv];
  if (g < n_groups) dma_rows(rows, g * rpw, min(rpw, n_rows - g * rpw), nb, buf, lane);
  stage_q8k(xq, nb * n_tokens, xs_dyn, threadIdx.x, blockDim.x);
  __syncthreads();

  const int blk = lane & (lpr - 1);
  const int rr = lane / lpr;
  const bool active = blk < nb;
  for (; g < n_groups; g += n_waves) {
    const int r0 = g * rpw;
    const int n = min(rpw, n_rows - r0);
    wait_vm();
    uint32_t w36[36];
    const bool live = active && rr < n;
    if (live) read_block_lds(buf + (rr * nb + blk) * 36, w36);
    wait_lds();
    const int gn = g + n_waves;
    if (gn < n_groups) dma_rows(rows, gn * rpw, min(rpw, n_rows - gn * rpw), nb, buf, lane);
    ScaleMins sm8{};
    if (live) sm8 = unpack_scales(w36[1], w36[2], w36[3]);
    for (int t = 0; t < n_tokens; ++t) {
      float s = 0.f;
      if (live) {
        int32_t xr[64], ip[8];
        float xd, bsf[8];
        load_x_regs(xs_dyn + (t * nb + blk) * kXStride, xr, xd, bsf);
        subblock_dots(w36 + 4, xr, ip);
        s = block_sum(w36[0], sm8, ip, xd, bsf);
      }
      const float acc = row_sum_last(s, blk, nb);
      if (blk == nb - 1 && rr < n) y.store(t * n_rows + r0 + rr, acc);
    }
  }
}

// y[t*n_rows + r] = W[r] . x[t] for up to 16 tokens on int8 matrix cores, the
// weights read once; the row result goes out through Out (fp32, or rounded to
// fp16).  One v_mfma_i32_16x16x32_i8 is one Q4_K sub-block (K = 32) of 16
// weight rows (columns) against 16 token rows, so every int32 sub-block dot
// comes out by itself and the fp32 epilogue keeps the GEMV family's order
// (block_sum, then the block sums added in block order): the same bits.  Wave
// w owns super-block w of every row, so its activation operands stay in
// registers, and the block sums of a row meet in LDS, added in block order by
// one thread per output.
constexpr int kMtBsWords = 12;  // staged per (block, token): 8 bsums as floats, d, padding
typedef int v4i __attribute__((ext_vector_type(4)));
typedef uint32_t u32x2 __attribute__((ext_vector_type(2)));

// 16-B runs a (quarters 0-1 or 2-3 of group lq & 1) to the lane's K quarter
// of both groups: even gets group 0's 8 bytes, odd group 1's
__device__ __forceinline__ void quarter_swap(const u32x4 a, u32x2& even, u32x2& odd) {
  const auto s0 = __builtin_amdgcn_permlane16_swap(a.x, a.z, false, false);
  const auto s1 = __builtin_amdgcn_permlane16_swap(a.y, a.w, false, false);
  even = u32x2{s0[0], s1[0]};
  odd = u32x2{s0[1], s1[1]};
}
__device__ __forceinline__ long pack_i64(u32x2 v) { return __builtin_bit_cast(long, v); }

// The activation operands of block b: sub-block s of token lr % TP, TP = 16 /
// NG, in the rows of group lr / TP and zero in the others' (xa[j] for group j)
template <int NG>
__device__ __forceinline__ void mt_load_x(const unsigned char* __restrict__ xq, int nb, int b,
                                          int n_tokens, int lr, int lq, u32x2 (&xa)[NG][8]) {
  constexpr int TP = 16 / NG;
  const int t = min(lr % TP, n_tokens - 1);
  const unsigned char* p = xq + (static_cast<long long>(t) * nb + b) * kQ8Bytes + 4 +
                           32 * (lq & 1) + 16 * (lq >> 1);
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    u32x2 e, o;
    quarter_swap(*reinterpret_cast<const u32x4u*>(p + 64 * i), e, o);
#pragma unroll
    for (int j = 0; j < NG; ++j) {
      const bool mine = NG == 1 || lr / TP == j;
      xa[j][2 * i] = mine ? e : u32x2{0u, 0u};
      xa[j][2 * i + 1] = mine ? o : u32x2{0u, 0u};
    }
  }
}
// d and the bsums (as floats) of every (block, token) into bst
__device__ __forceinline__ void mt_stage_bs(const unsigned char* __restrict__ xq, int nb,
                                            int n_tokens, float* bst, int tid, int nth) {
  for (int i = tid; i < nb * n_tokens; i += nth) {  // i = block * n_tokens + token
    const int b = i / n_tokens, t = i - b * n_tokens;
    const uint32_t* p =
        reinterpret_cast<const uint32_t*>(xq + (static_cast<long long>(t) * nb + b) * kQ8Bytes);
    float* o = bst + i * kMtBsWords;
#pragma unroll
    for (int s = 0; s < 4; ++s) {
      const uint32_t v = p[65 + s];
      o[2 * s] = static_cast<float>(static_cast<int16_t>(v & 0xFFFFu));
      o[2 * s + 1] = static_cast<float>(static_cast<int16_t>(v >> 16));
    }
    o[8] = __builtin_bit_cast(float, p[0]);
  }
}
// ... of block b and the four tokens of the lane's results from it
template <int TP>
__device__ __forceinline__ void mt_load_bs(const float* bst, int b, int n_tokens, int lq,
                                           float (&bs)[4][8], float (&xd)[4]) {
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const int t = min((4 * lq) % TP + i, n_tokens - 1);
    const float* p = bst + (b * n_tokens + t) * kMtBsWords;
#pragma unroll
    for (int s = 0; s < 8; ++s) bs[i][s] = p[s];
    xd[i] = p[8];
  }
}
// The block sums of one result (NG row groups of one super-block): hd the
// header of the lane's weight row, qw[j][g] its K quarter of group g's qs in
// row group j.
template <int NG>
__device__ __forceinline__ void mt_block(const u32x4 hd, const u32x2 (&qw)[NG][4],
                                         const u32x2 (&xa)[NG][8], const float (&bs)[4][8],
                                         const float (&xd)[4], float (&sum)[4]) {
  const ScaleMins sm8 = unpack_scales(hd.y, hd.z, hd.w);
  const float d = half_bits_to_float(hd.x & 0xFFFFu);
  const float dmin = half_bits_to_float(hd.x >> 16);
#pragma unroll
  for (int i = 0; i < 4; ++i) sum[i] = 0.f;
#pragma unroll
  for (int s = 0; s < 8; ++s) {
    v4i ip = {0, 0, 0, 0};
#pragma unroll
    for (int j = 0; j < NG; ++j) {
      const u32x2 q = (s & 1) ? qw[j][s >> 1] >> 4 : qw[j][s >> 1];
      ip = __builtin_amdgcn_mfma_i32_16x16x32_i8(pack_i64(xa[j][s]), pack_i64(q & 0x0F0F0F0Fu), ip,
                                                 0, 0, 0);
    }
    const float sd = d * byte_f(s < 4 ? sm8.sc_lo : sm8.sc_hi, s & 3);
    const float smv = dmin * byte_f(s < 4 ? sm8.mn_lo : sm8.mn_hi, s & 3);
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const float t = __builtin_fmaf(sd, static_cast<float>(ip[i]), -(smv * bs[i][s]));
      sum[i] = __builtin_fmaf(xd[i], t, sum[i]);
    }
  }
}

// Small matrices: a workgroup per 16 rows, loads straight into registers
// (one memory latency before the arithmetic).  A lane loads the header of row
// lr and two 16-B runs of its qs; a permlane16 swap turns two runs (quarters
// 0-1 or 2-3 of two groups) into the lane's K quarter of each group.  With
// more than 16 super-blocks per row a wave takes blocks w, w + 16, ... and the
// row sums run on over these chunks.  Bound by latency.  Six tokens, cold in a
// graph, against a wave per row group that looped over the tokens with sdot4:
// 8192 x 2048 11.8 -> 6.1 us, 2048 x 4096 17.8 -> 6.5, 64 x 2048 9.0 -> 3.8.
constexpr int kMtWaves = 16;
template <bool kChunked, typename Out>
__global__ void __launch_bounds__(64 * kMtWaves) gemv_mt_kernel(
    const sg_block_q4k* __restrict__ w, const unsigned char* __restrict__ xq, Out y, int n_rows,
    int nb, int n_tokens) {
  extern __shared__ __attribute__((aligned(16))) float mt_lds[];  // [2][waves][256], then bs
  const int tid = threadIdx.x, nth = blockDim.x, lane = tid & 63, wave = tid >> 6;
  const int nwv = nth >> 6;  // min(nb, kMtWaves)
  const int lr = lane & 15, lq = lane >> 4;
  float* bst = mt_lds + 2 * nwv * 256;
  const int n_chunks = kChunked ? (nb + nwv - 1) / nwv : 1;
  const int row0 = blockIdx.x * 16;
  const sg_block_q4k* wr = w + static_cast<long long>(min(row0 + lr, n_rows - 1)) * nb;
  u32x4 hd, q0, q1;
  auto load_w = [&](int b) {
    const char* p = reinterpret_cast<const char*>(wr + b);
    hd = *reinterpret_cast<const u32x4u*>(p);
    p += 16 + 32 * (lq & 1) + 16 * (lq >> 1);
    q0 = *reinterpret_cast<const u32x4u*>(p);
    q1 = *reinterpret_cast<const u32x4u*>(p + 64);
  };
  u32x2 xa[1][8];
  load_w(wave);  // (wave < nwv <= nb)
  mt_load_x<1>(xq, nb, wave, n_tokens, lr, lq, xa);
  mt_stage_bs(xq, nb, n_tokens, bst, tid, nth);
  bar();
  float run = 0.f;  // of output tid: token 4 (tid >> 4 & 3) + (tid >> 6), row tid & 15
  for (int c = 0; c < n_chunks; ++c) {
    const int b = c * nwv + wave;
    float* part = mt_lds + (c & 1) * nwv * 256;
    if (!kChunked || b < nb) {
      u32x2 qw[1][4];
      quarter_swap(q0, qw[0][0], qw[0][1]);
      quarter_swap(q1, qw[0][2], qw[0][3]);
      float bs[4][8], xd[4], sum[4];
      mt_load_bs<16>(bst, b, n_tokens, lq, bs, xd);
      mt_block<1>(hd, qw, xa, bs, xd, sum);
#pragma unroll
      for (int i = 0; i < 4; ++i) part[wave * 256 + 64 * i + lane] = sum[i];
      if (kChunked && b + nwv < nb) {
        load_w(b + nwv);
        mt_load_x<1>(xq, nb, b + nwv, n_tokens, lr, lq, xa);
      }
    }
    bar();  // (the other buffer is free again: its readers passed this barrier too)
    const int nbc = min(nwv, nb - c * nwv);
    if (nth >= 256) {
      if (tid < 256)
        for (int i = 0; i < nbc; ++i) run += part[i * 256 + tid];
    } else {  // fewer than four waves (one chunk): several outputs per thread
      for (int v = tid; v < 256; v += nth) {
        float acc = 0.f;
        for (int i = 0; i < nbc; ++i) acc += part[i * 256 + v];
        const int t = 4 * ((v >> 4) & 3) + (v >> 6), r = row0 + (v & 15);
        if (t < n_tokens && r < n_rows) y.store(t * n_rows + r, acc);
      }
    }
  }
  if (nth >= 256 && tid < 256) {
    const int t = 4 * ((tid >> 4) & 3) + (tid >> 6), r = row0 + (tid & 15);
    if (t < n_tokens && r < n_rows) y.store(t * n_rows + r, run);
  }
}

// Large matrices: persistent workgroups take sets of 16 RG rows in turn.
// The rows stream through a ring of three LDS buffers (two sets in flight)
// with buffer_load ... lds in 1-KB instructions; one barrier per set: set
// i's copies have landed, set i - 1's block sums are complete and its buffer
// and set i - 2's sums are free.  A row is an odd number of 16-B chunks (nb *
// 9, and one of padding where that is even), so that the 16 rows a wave reads
// together start in different banks.
//
// With up to 8 tokens a 16 x 16 result would be half padding, and its
// epilogue, four operations per result and sub-block, is most of what the
// kernel issues.  NG = 2 row groups then share a result: group j's tokens sit
// in rows 8j..8j+7 of its A operand, zero elsewhere, and the two groups' MFMAs
// accumulate into one result whose row half j is group j's.
//
// Bound by the weight stream: 248320 x 2048 x 4 tokens 77.6 -> 54.8 us (5.2
// TB/s).  With 64-row sets loaded straight to registers it took 70 us: 16-B
// pieces of a 128-B line asked for by several instructions, against whole
// lines here.
constexpr int kMtwBufs = 3;
constexpr int kMtwCopies = 5;  // copy instructions per wave and set, at most
__host__ __device__ constexpr int mtw_buf_words(int rg, int nb) {
  return (16 * rg * (9 * nb | 1) + 63) / 64 * 256;
}

template <int NG, int RG, int kMaxWv, typename Out>
__global__ void __launch_bounds__(64 * kMaxWv) gemv_mtw_kernel(
    const sg_block_q4k* __restrict__ w, const unsigned char* __restrict__ xq, Out y, int n_rows,
    int nb, int n_tokens) {
  constexpr int TP = 16 / NG;       // token rows of one row group in a result
  constexpr int kSets = RG / NG;    // results (of 4 registers) per super-block, a wave each
  constexpr int kOuts = kSets * 256;  // outputs of a set, tokens past n_tokens included
  extern __shared__ __attribute__((aligned(16))) uint32_t mtw_lds[];
  const int tid = threadIdx.x, nth = blockDim.x, lane = tid & 63, wave = tid >> 6;
  const int nwv = nth >> 6;  // = nb * kSets
  const int ws = kSets == 1 ? 0 : wave / nb, wb = wave - ws * nb;  // the wave's result, block
  const int lr = lane & 15, lq = lane >> 4;
  const int cpr = 9 * nb | 1, rw = 4 * cpr;  // chunks and words of a row in LDS
  const int bufw = mtw_buf_words(RG, nb);
  uint32_t* ring = mtw_lds;
  float* part = reinterpret_cast<float*>(ring + kMtwBufs * bufw);  // [2][nwv][256]
  float* bst = part + 2 * nwv * 256;
  const int n_sets = (n_rows + 16 * RG - 1) / (16 * RG);
  const uint32_t row_bytes = nb * kQ4Bytes;

  // copy instruction wave + nwv i of a set: its lane's chunk, from the set's
  // first row (the padding chunk re-reads the row's first)
  const int n_inst = bufw / 256;
  uint32_t ofs[kMtwCopies];
#pragma unroll
  for (int i = 0; i < kMtwCopies; ++i) {
    const int c = min((wave + nwv * i) * 64 + lane, 16 * RG * cpr - 1);
    const int r = c / cpr, p = c - r * cpr;
    ofs[i] = r * row_bytes + (p == 9 * nb ? 0 : 16 * p);
  }
  const int mine = (n_inst - wave + nwv - 1) / nwv;  // this wave's instructions per set
  auto issue = [&](int g, int slot) {
    const long long r0 = static_cast<long long>(g) * 16 * RG;
    const int rows = min(16 * RG, static_cast<int>(n_rows - r0));
    // rows past the matrix are out of the buffer's range and read as zero
    const u32x4 rs = buffer_desc(reinterpret_cast<const char*>(w) + r0 * row_bytes,
                                 rows * row_bytes);
#pragma unroll
    for (int i = 0; i < kMtwCopies; ++i)
      if (i < mine) dma16<true>(ring + slot * bufw + 256 * (wave + nwv * i), ofs[i], rs, 0);
  };
  const int g0 = blockIdx.x, gs = gridDim.x;
  if (g0 < n_sets) issue(g0, 0);
  if (g0 + gs < n_sets) issue(g0 + gs, 1);
  u32x2 xa[NG][8];
  float bs[4][8], xd[4];
  mt_load_x<NG>(xq, nb, wb, n_tokens, lr, lq, xa);
  mt_stage_bs(xq, nb, n_tokens, bst, tid, nth);
  bar();
  mt_load_bs<TP>(bst, wb, n_tokens, lq, bs, xd);

  auto finish = [&](int g, const float* pr) {  // add the block sums of set g and store
    for (int v = tid; v < kOuts; v += nth) {
      float acc = 0.f;
      const int vm = v >> 8;
      for (int i = 0; i < nb; ++i) acc += pr[(vm * nb + i) * 256 + (v & 255)];
      const int vi = (v >> 6) & 3, vq = (v >> 4) & 3;
      const int t = (4 * vq) % TP + vi;
      const int r = (g * RG + vm * NG + vq * NG / 4) * 16 + (v & 15);
      if (t < n_tokens && r < n_rows) y.store(t * n_rows + r, acc);
    }
  };
  int slot = 0, buf = 0;
  for (int g = g0; g < n_sets; g += gs) {
    // the oldest set has landed once only the next one's copies are left
    wait_vm_n(g + gs < n_sets ? mine : 0);
    bar();
    const int s2 = slot == 0 ? 2 : slot - 1;  // (slot + 2) % 3
    if (g + 2 * gs < n_sets) issue(g + 2 * gs, s2);
    if (g != g0) finish(g - gs, part + (buf ^ 1) * nwv * 256);
    const uint32_t* rb = ring + slot * bufw + 36 * wb + ws * NG * 16 * rw;
    const u32x4 hd = *reinterpret_cast<const u32x4*>(rb + (lq * NG / 4 * 16 + lr) * rw);
    u32x2 qw[NG][4];
#pragma unroll
    for (int j = 0; j < NG; ++j)
#pragma unroll
      for (int q = 0; q < 4; ++q)
        qw[j][q] = *reinterpret_cast<const u32x2*>(rb + (j * 16 + lr) * rw + 4 + 8 * q + 2 * lq);
    float sum[4];
    mt_block<NG>(hd, qw, xa, bs, xd, sum);
    float* pw = part + (buf * nwv + wave) * 256;
#pragma unroll
    for (int i = 0; i < 4; ++i) pw[64 * i + lane] = sum[i];
    slot = slot == 2 ? 0 : slot + 1;
    buf ^= 1;
  }
  bar();
  if (g0 < n_sets)
    finish(g0 + (n_sets - 1 - g0) / gs * gs, part + (buf ^ 1) * nwv * 256);
}

// dots[(r*nb + b)*8 + s] = int32 sub-block dot (test hook).
__global__ void __launch_bounds__(256) subblock_dots_kernel(const sg_block_q4k* __restrict__ w,
                                                            const unsigned char* __restrict__ xq,
                                                            int32_t* __restrict__ dots,
                                                            int n_rows, int nb, int lpr) {
  __shared__ __attribute__((aligned(16))) uint32_t wbuf[kWaves][kBufWords];
  extern __shared__ __attribute__((aligned(16))) uint32_t xs_dyn[];
  const PlainRows rows{w, nb};
  const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
  const int rpw = 64 / lpr;
  const int g = blockIdx.x * kWaves + wv;
  const int n_groups = (n_rows + rpw - 1) / rpw;
  const int r0 = g * rpw;
  const int n = g < n_groups ? min(rpw, n_rows - r0) : 0;
  if (n > 0) dma_rows(rows, r0, n, nb, wbuf[wv], lane);
  stage_q8k(xq, nb, xs_dyn, threadIdx.x, blockDim.x);
  __syncthreads();
  const int blk = lane & (lpr - 1);
  const int rr = lane / lpr;
  if (blk >= nb || rr >= n) return;
  int32_t xr[64];
  float xd, bsf[8];
  load_x_regs(xs_dyn + blk * kXStride, xr, xd, bsf);
  wait_vm();
  uint32_t w36[36];
  read_block_lds(wbuf[wv] + (rr * nb + blk) * 36, w36);
  int32_t ip[8];
  subblock_dots(w36 + 4, xr, ip);
  int32_t* o = dots + (static_cast<long long>(r0 + rr) * nb + blk) * 8;
#pragma unroll
  for (int s = 0; s < 8; ++s) o[s] = ip[s];
}

// Grid for a grid-stride row loop: every row group once, capped at two
// workgroups of four waves per CU (256 CUs) - enough copies in flight to
// stream HBM at full rate.
static unsigned gemv_grid(long long n_groups) {
  const long long wgs = (n_groups + kWaves - 1) / kWaves;
  const long long cap = 256LL * kWgPerCu;
  return static_cast<unsigned>(wgs < cap ? (wgs > 0 ? wgs : 1) : cap);
}

// gemv1_kernel's launch: waves per workgroup, grid, groups per wave and the
// LDS its per-wave results take.  (One wave per workgroup over more CUs was
// measured slower on the 2048 x 2048 matrix: each workgroup stages x again,
// with a quarter of the threads.)
struct Gemv1Launch {
  int nwv;
  unsigned grid;
  int gpw;
  size_t res_bytes;
};
static Gemv1Launch gemv1_launch(long long n_groups, int rpw) {
  Gemv1Launch l{};
  l.nwv = kWaves;
  l.grid = gemv_grid(n_groups);
  const long long waves = static_cast<long long>(l.grid) * l.nwv;
  l.gpw = static_cast<int>((n_groups + waves - 1) / waves);
  l.res_bytes = static_cast<size_t>(l.nwv) * l.gpw * rpw * 4;
  return l;
}

// Matrices of at most this many super-blocks (and nb <= 16) take
// gemv_lat_kernel.  Measured with cold matrices (graph replays over rotated
// copies), it is faster up to 32768 x 2048 (2048 x 2048: 3.35 against
// 4.84 us); from 65536 x 2048 on, the streaming kernel is (248320 x 2048:
// 52 against 57 us).
constexpr long long kLatMaxBlocks = 262144;
static bool use_lat(int n_rows, int nb) {
  return nb <= kLatMaxNb && static_cast<long long>(n_rows) * nb <= kLatMaxBlocks;
}
template <typename Rows, typename Out>
static void gemv_lat_go(hipStream_t s, Rows rows, const sg_block_q8k* x, Out out, int n_rows,
                        int nb) {
  const int lpr = lanes_per_row(nb), rpw = 16 / lpr;
  const int waves = (n_rows + rpw - 1) / rpw;
  const dim3 grid((waves + kLatWaves - 1) / kLatWaves), block(64 * kLatWaves);
  const unsigned char* xb = reinterpret_cast<const unsigned char*>(x);
  const int lg = __builtin_ctz(lpr);
  if constexpr (std::is_same_v<Rows, PlainRows> && std::is_same_v<Out, F32Out>)
    hipLaunchKernelGGL(gemv_lat_plain_kernel, grid, block, 0, s, rows.w, xb, out.y, n_rows, nb, lg);
  else
    hipLaunchKernelGGL((gemv_lat_kernel<Rows, Out>), grid, block, 0, s, rows, xb, out, n_rows, nb,
                       lg);
}

template <typename Rows, typename Out>
static void gemv1_go(const Gemv1Launch& L, size_t lds, hipStream_t s, Rows rows,
                     const sg_block_q8k* x, Out out, int n_rows, int nb, int lpr) {
  if (use_lat(n_rows, nb)) return gemv_lat_go(s, rows, x, out, n_rows, nb);
  const unsigned char* xb = reinterpret_cast<const unsigned char*>(x);
  if (L.nwv == 1)
    hipLaunchKernelGGL((gemv1_kernel<Rows, Out, 1>), dim3(L.grid), dim3(64), lds, s, rows, xb, out,
                       n_rows, nb, lpr, L.gpw);
  else
    hipLaunchKernelGGL((gemv1_kernel<Rows, Out, kWaves>), dim3(L.grid), dim3(64 * kWaves), lds, s,
                       rows, xb, out, n_rows, nb, lpr, L.gpw);
}

static int check_gemv_geometry(const char* name, int n_rows, int k) {
  if (n_rows <= 0 || k <= 0 || k % kQK != 0)
    return set_error(SG_ERR_GEOMETRY, "%s: n_rows=%d k=%d (k must be a positive multiple of 256)",
                     name, n_rows, k);
  if (k / kQK > kMaxNb)
    return set_error(SG_ERR_UNSUPPORTED, "%s: k=%d exceeds %d", name, k, kMaxNb * kQK);
  return SG_OK;
}

// LDS of a gemv1 launch (the staged activations and the waves' results)
constexpr size_t kGemv1MaxLds = 96 * 1024;
static size_t gemv1_lds(int n_rows, int nb) {
  const int rpw = 64 / lanes_per_row(nb);
  return static_cast<size_t>(nb) * kXStride * 4 +
         gemv1_launch((static_cast<long long>(n_rows) + rpw - 1) / rpw, rpw).res_bytes;
}

// one gemv1 launch over a row source and an output policy (shared by the
// fp16-output entry points)
template <typename Rows, typename Out>
static int launch_gemv1(Rows rows, const sg_block_q8k* x, Out out, int n_rows, int k,
                        hipStream_t s, const char* nm) {
  if (int st = check_gemv_geometry(nm, n_rows, k)) return st;
  const int nb = k / kQK, lpr = lanes_per_row(nb);
  const long long n_groups = (n_rows + (64 / lpr) - 1) / (64 / lpr);
  const Gemv1Launch L = gemv1_launch(n_groups, 64 / lpr);
  const size_t lds = static_cast<size_t>(nb) * kXStride * 4 + L.res_bytes;
  if (lds > kGemv1MaxLds)
    return set_error(SG_ERR_UNSUPPORTED, "%s: n_rows=%d k=%d needs %zu B of LDS", nm, n_rows, k,
                     lds);
  gemv1_go(L, lds, s, rows, x, out, n_rows, nb, lpr);
  return check_launch(nm);
}

// the pointer-table GEMV over an output policy
template <typename Out>
static int launch_ptrs(const sg_block_q4k* const* ptrs, const sg_block_q8k* x, Out y, int n_ptrs,
                       int rows_per, int k, hipStream_t s, const char* nm) {
  if (!ptrs || !x) return set_error(SG_ERR_INVALID_ARGUMENT, "%s: null pointer", nm);
  if (n_ptrs <= 0 || rows_per <= 0 || static_cast<long long>(n_ptrs) * rows_per > 0x7fffffffLL)
    return set_error(SG_ERR_GEOMETRY, "%s: n_ptrs=%d rows_per=%d", nm, n_ptrs, rows_per);
  const int n_rows = n_ptrs * rows_per;
  if (int st = check_gemv_geometry(nm, n_rows, k)) return st;
  const int nb = k / kQK, lpr = lanes_per_row(nb);
  const long long n_groups = (n_rows + (64 / lpr) - 1) / (64 / lpr);
  const Gemv1Launch L = gemv1_launch(n_groups, 64 / lpr);
  const size_t lds = static_cast<size_t>(nb) * kXStride * 4 +
                     (n_ptrs <= kMaxLdsPtrs ? static_cast<size_t>(n_ptrs) * 8 : 0) + L.res_bytes;
  if (lds > 96 * 1024)
    return set_error(SG_ERR_UNSUPPORTED, "%s: n_rows=%d k=%d needs %zu B of LDS", nm, n_rows, k,
                     lds);
  gemv1_go(L, lds, s,
           TableRows{ptrs, rows_per, nb, n_ptrs,
                     (rows_per & (rows_per - 1)) == 0 ? __builtin_ctz(rows_per) : -1},
           x, y, n_rows, nb, lpr);
  return check_launch(nm);
}

// Which several-token kernel, by super-blocks (n_rows * nb), measured cold in
// graphs (us; sdot4 / matrix cores):
// - gemv_batched_kernel, the sdot4 one:
//   - at most eight staged blocks of two to four tokens from 65536 blocks on
//     (262141 x 512, 2 tokens 17.8 / 20.4, 3 tokens 19.7 / 20.6; 4 tokens x
//     1024 23.1 / 20.3);
//   - two tokens of 6 to 8 blocks per row from 150000 on (18750 x 2048 9.7 /
//     10.0, 37449 x 1792 12.4 / 14.6, 52500 x 2048 17.0 / 17.0, 250000 x 2048
//     56.6 / 59.0, but 14285 x 1792 7.9 / 7.3), of 5 up to the streaming kernel's
//     line (46000 x 1280 12.5 / 13.3, 60000 x 1280 15.3 / 13.4);
//   - two or three tokens of 17 to 32 blocks per row, which the streaming
//     kernel does not take and for which gemv_mt_kernel needs two chunks, in
//     rounds of 4096 rows (16 per CU).  Two tokens: past three rounds (12400 x
//     5120 18.3 / 21.5, 152064 x 5120 138 / 190) and while the third is less than
//     half full (9000 x 6144 17.0 / 18.3, 11000 x 6144 19.5 / 19.1, 8192 x 8192
//     19.3 / 16.9); past 32 blocks half of its lanes idle (60606 x 8448 134 /
//     114).  Three tokens: from 786432 blocks up to 20 per row (58823 x 4352 70.1 /
//     75.8, 35000 x 5120 50.9 / 49.6), from 700000 at 32, where every lane has a
//     block (21875 x 8192 44.8 / 48.0, 18750 x 8192 42.4 / 40.4), from 1048576
//     between (41666 x 7680 73.7 / 77.5, 25000 x 7168 46.4 / 45.8, 36363 x 5632
//     54.6 / 51.4).  Four tokens: never (152064 x 5120 223 / 200);
// - gemv_mtw_kernel, the streaming one (us; gemv_mt_kernel / this one): from
//   131072 with more than 8 blocks per row (8197 x 4096 13.7 / 11.5; 4096 x 4096
//   7.4 / 8.3), from 262144 below that (32765 x 2048 15.2 / 12.9; 16381 x 2048
//   10.0 / 10.0); with more than 8 tokens, whose sets are twice the work, from
//   524288 (65533 x 2048 26.0 / 23.7; 32765 15.7 / 15.8) and only with more than
//   4 blocks per row (131069 x 1024 22.6 / 25.8);
// - gemv_mt_kernel otherwise.
static bool use_batched_sdot(int n_rows, int nb, int n_tokens) {
  const long long blocks = static_cast<long long>(n_rows) * nb;
  if (n_tokens < 2 || n_tokens > 4) return false;
  if (n_tokens * nb <= 8) return blocks >= 65536;
  if (n_tokens == 2 && nb <= 8) return blocks >= 150000 && (nb > 5 || blocks < 262144);
  if (nb <= 16 || nb > 32) return false;
  if (n_tokens == 2) return n_rows > 12288 || (n_rows > 8192 && n_rows <= 10240);
  return n_tokens == 3 && blocks >= (nb <= 20 ? 786432 : nb < 32 ? 1048576 : 700000);
}
static bool use_mtw(int n_rows, int nb, int n_tokens) {
  if (nb < 2 || nb > 16 || (n_tokens > 8 && nb <= 4)) return false;
  return static_cast<long long>(n_rows) * nb >=
         (nb > 8 ? 131072 : (n_tokens <= 8 ? 262144 : 524288));
}

template <int NG, int RG, int kMaxWv, typename Out>
static void gemv_mtw_go(hipStream_t s, const sg_block_q4k* w, const unsigned char* xb, Out y,
                        int n_rows, int nb, int n_tokens) {
  const int n_sets = (n_rows + 16 * RG - 1) / (16 * RG);
  const size_t lds = (static_cast<size_t>(kMtwBufs) * mtw_buf_words(RG, nb) +
                      2 * static_cast<size_t>(nb) * (RG / NG) * 256 +
                      static_cast<size_t>(nb) * n_tokens * kMtBsWords) * 4;
  const int per_cu = std::min<int>(160 * 1024 / lds, 32 / (nb * (RG / NG)));  // resident workgroups
  const int cap = 256 * per_cu;
  hipLaunchKernelGGL((gemv_mtw_kernel<NG, RG, kMaxWv, Out>), dim3(n_sets < cap ? n_sets : cap),
                     dim3(64 * nb * (RG / NG)), lds, s, w, xb, y, n_rows, nb, n_tokens);
}
template <typename Out>
static void gemv_mt_go(hipStream_t s, const sg_block_q4k* w, const unsigned char* xb, Out y,
                       int n_rows, int nb, int n_tokens) {
  const int nwv = nb < kMtWaves ? nb : kMtWaves;
  const size_t lds = (2 * static_cast<size_t>(nwv) * 256 +
                      static_cast<size_t>(nb) * n_tokens * kMtBsWords) * 4;
  const dim3 grid((n_rows + 15) / 16), block(64 * nwv);
  if (nb <= kMtWaves)
    hipLaunchKernelGGL((gemv_mt_kernel<false, Out>), grid, block, lds, s, w, xb, y, n_rows, nb,
                       n_tokens);
  else
    hipLaunchKernelGGL((gemv_mt_kernel<true, Out>), grid, block, lds, s, w, xb, y, n_rows, nb,
                       n_tokens);
}

// the batched GEMV over an output policy (fp32 or fp16 rows)
template <typename Out>
static int launch_batched(const sg_block_q4k* w, const sg_block_q8k* x, Out y, int n_rows, int k,
                          int n_tokens, hipStream_t s, const char* nm) {
  if (!w || !x) return set_error(SG_ERR_INVALID_ARGUMENT, "%s: null pointer", nm);
  if (int st = check_gemv_geometry(nm, n_rows, k)) return st;
  if (n_tokens <= 0 || n_tokens > kMaxTokens)
    return set_error(SG_ERR_UNSUPPORTED, "%s: n_tokens=%d not in [1,%d]", nm, n_tokens,
                     kMaxTokens);
  if (static_cast<long long>(n_rows) * n_tokens > 0x7fffffffLL)
    return set_error(SG_ERR_GEOMETRY, "%s: n_rows*n_tokens too large", nm);
  const int nb = k / kQK;
  if (static_cast<size_t>(nb) * n_tokens * kXStride * 4 > 96 * 1024)
    return set_error(SG_ERR_UNSUPPORTED, "%s: k*n_tokens too large for LDS", nm);
  const unsigned char* xb = reinterpret_cast<const unsigned char*>(x);
  if (n_tokens == 1) {  // the one-token GEMV, where its results fit LDS
    if (gemv1_lds(n_rows, nb) <= kGemv1MaxLds)
      return launch_gemv1(PlainRows{w, nb}, x, y, n_rows, k, s, nm);
  }
  if (use_batched_sdot(n_rows, nb, n_tokens)) {
    const int lpr = lanes_per_row(nb);
    const long long n_groups = (n_rows + (64 / lpr) - 1) / (64 / lpr);
    hipLaunchKernelGGL((gemv_batched_kernel<Out>), dim3(gemv_grid(n_groups)), dim3(256),
                       static_cast<size_t>(nb) * n_tokens * kXStride * 4, s, w, xb, y, n_rows, nb,
                       lpr, n_tokens);
  } else if (!use_mtw(n_rows, nb, n_tokens)) {
    gemv_mt_go(s, w, xb, y, n_rows, nb, n_tokens);
  } else if (nb > 8) {
    gemv_mtw_go<1, 1, 16>(s, w, xb, y, n_rows, nb, n_tokens);
  } else if (n_tokens <= 8) {
    gemv_mtw_go<2, 2, 8>(s, w, xb, y, n_rows, nb, n_tokens);
  } else {
    gemv_mtw_go<1, 2, 16>(s, w, xb, y, n_rows, nb, n_tokens);
  }
  return check_launch(nm);
}

}  // namespace sg

using namespace sg;

extern "C" {

int sg_gemv_q4_k_q8(const sg_block_q4k* w, const sg_block_q8k* x, float* y, int n_rows, int k,
                    void* stream) {
  const char* nm = "sg_gemv_q4_k_q8";
  if (!w || !x || !y) return set_error(SG_ERR_INVALID_ARGUMENT, "%s: null pointer", nm);
  return launch_gemv1(PlainRows{w, k / kQK}, x, F32Out{y}, n_rows, k,
                      static_cast<hipStream_t>(stream), nm);
}

int sg_gemv_ptrs_q4_k_q8(const sg_block_q4k* const* ptrs, const sg_block_q8k* x, float* y,
                         int n_ptrs, int rows_per, int k, void* stream) {
  if (!y) return set_error(SG_ERR_INVALID_ARGUMENT, "sg_gemv_ptrs_q4_k_q8: null pointer");
  return launch_ptrs(ptrs, x, F32Out{y}, n_ptrs, rows_per, k, static_cast<hipStream_t>(stream),
                     "sg_gemv_ptrs_q4_k_q8");
}

int sg_gemv_ptrs_q4_k_q8_f16out(const sg_block_q4k* const* ptrs, const sg_block_q8k* x,
                                uint16_t* y, int n_ptrs, int rows_per, int k, void* stream) {
  if (!y) return set_error(SG_ERR_INVALID_ARGUMENT, "sg_gemv_ptrs_q4_k_q8_f16out: null pointer");
  return launch_ptrs(ptrs, x, F16Out{y}, n_ptrs, rows_per, k, static_cast<hipStream_t>(stream),
                     "sg_gemv_ptrs_q4_k_q8_f16out");
}

int sg_gemv_q4_k_q8_batched(const sg_block_q4k* w, const sg_block_q8k* x, float* y, int n_rows,
                            int k, int n_tokens, void* stream) {
  if (!y) return set_error(SG_ERR_INVALID_ARGUMENT, "sg_gemv_q4_k_q8_batched: null pointer");
  return launch_batched(w, x, F32Out{y}, n_rows, k, n_tokens, static_cast<hipStream_t>(stream),
                        "sg_gemv_q4_k_q8_batched");
}

int sg_gemv_q4_k_q8_f16out_batched(const sg_block_q4k* w, const sg_block_q8k* x, uint16_t* y,
                                   int n_rows, int k, int n_tokens, void* stream) {
  if (!y) return set_error(SG_ERR_INVALID_ARGUMENT, "sg_gemv_q4_k_q8_f16out_batched: null pointer");
  return launch_batched(w, x, F16Out{y}, n_rows, k, n_tokens, static_cast<hipStream_t>(stream),
                        "sg_gemv_q4_k_q8_f16out_batched");
}

int sg_q4k_subblock_dots(const sg_block_q4k* w, const sg_block_q8k* x, int32_t* dots, int n_rows,
                         int k, void* stream) {
  if (!w || !x || !dots)
    return set_error(SG_ERR_INVALID_ARGUMENT, "sg_q4k_subblock_dots: null pointer");
  if (int st = check_gemv_geometry("sg_q4k_subblock_dots", n_rows, k)) return st;
  const int nb = k / kQK, lpr = lanes_per_row(nb);
  const long long n_groups = (n_rows + (64 / lpr) - 1) / (64 / lpr);
  hipLaunchKernelGGL(subblock_dots_kernel, dim3(static_cast<unsigned>((n_groups + 3) / 4)),
                     dim3(256), nb * kXStride * 4, static_cast<hipStream_t>(stream), w,
                     reinterpret_cast<const unsigned char*>(x), dots, n_rows, nb, lpr);
  return check_launch("sg_q4k_subblock_dots");
}

int sg_gemv_q4_k_q8_f16out(const sg_block_q4k* w, const sg_block_q8k* x, uint16_t* y, int n_rows,
                           int k, void* stream) {
  const char* nm = "sg_gemv_q4_k_q8_f16out";
  if (!w || !x || !y) return set_error(SG_ERR_INVALID_ARGUMENT, "%s: null pointer", nm);
  F16SegOut o{{y, y, y}, {n_rows, n_rows, n_rows}};
  return launch_gemv1(PlainRows{w, k / kQK}, x, o, n_rows, k, static_cast<hipStream_t>(stream),
                      nm);
}

int sg_gemv3m_q4_k_q8_f16out(const sg_block_q4k* w1, const sg_block_q4k* w2,
                             const sg_block_q4k* w3, const sg_block_q8k* x, uint16_t* y1,
                             uint16_t* y2, uint16_t* y3, int rows1, int rows2, int rows3, int k,
                             void* stream) {
  const char* nm = "sg_gemv3m_q4_k_q8_f16out";
  if (!w1 || !w2 || !x || !y1 || !y2 || (rows3 > 0 && (!w3 || !y3)))
    return set_error(SG_ERR_INVALID_ARGUMENT, "%s: null pointer", nm);
  if (rows1 <= 0 || rows2 <= 0 || rows3 < 0 ||
      static_cast<long long>(rows1) + rows2 + rows3 > 0x7fffffffLL)
    return set_error(SG_ERR_GEOMETRY, "%s: rows %d/%d/%d", nm, rows1, rows2, rows3);
  const int e0 = rows1, e1 = rows1 + rows2, e2 = e1 + rows3;
  SegRows rs{{w1, w2, rows3 > 0 ? w3 : w2}, {e0, e1, e2}, k / kQK};
  F16SegOut o{{y1, y2, rows3 > 0 ? y3 : y2}, {e0, e1, e2}};
  return launch_gemv1(rs, x, o, e2, k, static_cast<hipStream_t>(stream), nm);
}

int sg_gemv2m_q4_k_q8_f16out(const sg_block_q4k* w1, const sg_block_q4k* w2,
                             const sg_block_q8k* x, uint16_t* y1, uint16_t* y2, int rows1,
                             int rows2, int k, void* stream) {
  return sg_gemv3m_q4_k_q8_f16out(w1, w2, nullptr, x, y1, y2, nullptr, rows1, rows2, 0, k,
                                  stream);
}

int sg_gemv_q4_k_q8_f16out_resadd(const sg_block_q4k* w, const sg_block_q8k* x, uint16_t* y,
                                  uint16_t* res_inout, int n_rows, int k, void* stream) {
  const char* nm = "sg_gemv_q4_k_q8_f16out_resadd";
  if (!w || !x || !y || !res_inout) return set_error(SG_ERR_INVALID_ARGUMENT, "%s: null pointer", nm);
  return launch_gemv1(PlainRows{w, k / kQK}, x, F16ResAddOut{y, res_inout}, n_rows, k,
                      static_cast<hipStream_t>(stream), nm);
}

}  // extern "C"
