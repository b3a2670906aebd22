// RMSNorm, the fused q/k RMSNorm + RoPE + paged-KV append, the SiLU-gated
// product and greedy draft acceptance for gfx950.
//
// RMSNorm follows the reference kernel's arithmetic (src/cuda_kernels.cu:11-17)
// so that results are reproducible bit for bit:
//   * thread t of a 256-thread row accumulates v_j^2 for j = t, t+256, ... in
//     order with one FMA per term (nvcc contracts `sum += v*v` by default);
//   * the 256 partial sums are combined by the pairwise tree
//     p[t] += p[t + s] for s = 128, 64, ..., 1 (p[0] is the total);
//   * scale = rsqrt(total / width + eps), here 1 / sqrt evaluated in double
//     precision and rounded once to float (the reference calls the device's
//     approximate rsqrtf);
//   * out_j = T(rn(rn(v_j * scale) * w_j)), new_residual_j = T(v_j).
// A butterfly (v + v[lane ^ s]) over the lanes that hold the tree's partial
// sums leaves the tree's total in every lane (addition commutes and each step
// pairs exactly the tree's operands), which is how the kernels below evaluate
// the tree inside a wavefront.
//
// This file is compiled with -ffp-contract=off; every fused multiply-add is
// written out.
#include <type_traits>

#include "rope_math.hpp"

namespace feattn {

__device__ __forceinline__ float rsqrt_rn(float x) { return (float)(1.0 / __dsqrt_rn((double)x)); }

template <int CTRL>
__device__ __forceinline__ float dpp(float v) {
  return __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), CTRL, 0xf, 0xf, true));
}
constexpr int kDppHalfMirror = 0x141;   // lane i <- lane 7 - i within each 8-lane half row
constexpr int kDppQuadXor2 = 0x4e;      // quad_perm [2, 3, 0, 1]
constexpr int kDppQuadXor1 = 0xb1;      // quad_perm [1, 0, 3, 2]

constexpr int kDppRowRor8 = 0x128;      // lane ^ 8 within each 16-lane row

// ---------------------------------------------------------------------------
// fe_norm
// ---------------------------------------------------------------------------
// A stripe is 256 consecutive elements of a row: element t of stripe k is
// term k of the tree's partial sum p[t].
//
// norm_row_kernel: one wavefront per row, the whole row in registers, read
// once with 16-byte loads that are all issued before the first is used.  A
// load instruction covers two stripes, lanes 0-31 the first and 32-63 the
// second; one v_permlane32_swap per register pair then gives lane i four
// consecutive elements of each of the two, t = 8c + 4 (i / 32) + 0..3 of its
// chunk c, so that every p[t] is one lane's FMA chain.  Chunks go to lanes
// in order, the upper four of each eight reversed: the tree's partner at
// distance 32 is then the half-row mirror lane, and all its cross-lane steps
// are register exchanges.  NP: stripe pairs a row may have (loads past the
// row are redirected to its last elements and dropped).  HBM bound: 8192 x
// 4096 bf16 with the residual takes 50.4 us, 5.3 TB/s of the 268 MB it needs
// (a loop of 2-byte loads over the row, twice: 154 us; 8-byte loads without
// the exchange: 53.7 us).
__device__ __forceinline__ void swap_halves(uint32_t& a, uint32_t& b) {  // a's lanes 32-63 <-> b's lanes 0-31
  const auto r = __builtin_amdgcn_permlane32_swap(a, b, false, false);
  a = r[0];
  b = r[1];
}
// Words 0, 1 become the lane's four elements of the first stripe of the pair,
// words 2, 3 of the second; its own inverse.
__device__ __forceinline__ u32x4 exchange_pair(u32x4 v) {
  uint32_t a = v[0], b = v[2], c = v[1], d = v[3];
  swap_halves(a, b);
  swap_halves(c, d);
  return u32x4{a, c, b, d};
}

template <bool BF16, int NP, bool RES, bool STREAM>
__global__ __launch_bounds__(256) void norm_row_kernel(const uint16_t* x, const uint16_t* res,
                                                       const uint16_t* __restrict__ w, uint16_t* out,
                                                       uint16_t* new_res, int rows, int width, float eps) {
  const int lane = threadIdx.x & 63;
  const int row = blockIdx.x * (blockDim.x >> 6) + uniform(threadIdx.x >> 6);
  if (row >= rows) return;
  const int c8 = lane & 7;
  const int j0 = 8 * ((lane & 56) | (c8 < 4 ? c8 : 11 - c8));
  const size_t base = (size_t)row * width;
  auto ld = [](const uint16_t* a) {
    const u32x4* q = reinterpret_cast<const u32x4*>(a);
    return STREAM ? __builtin_nontemporal_load(q) : *q;
  };
  auto put = [](uint16_t* a, u32x4 v) {
    u32x4* q = reinterpret_cast<u32x4*>(a);
    if constexpr (STREAM) __builtin_nontemporal_store(v, q);
    else *q = v;
  };
  u32x4 xv[NP], rv[NP], wv[NP];
#pragma unroll
  for (int s = 0; s < NP; ++s) {
    const int j = min(j0 + 512 * s, width - 8);
    xv[s] = ld(x + base + j);
    if constexpr (RES) rv[s] = ld(res + base + j);
  }
#pragma unroll
  for (int s = 0; s < NP; ++s) wv[s] = *reinterpret_cast<const u32x4*>(w + min(j0 + 512 * s, width - 8));

  float v[NP][8];
  float p[4] = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
  for (int s = 0; s < NP; ++s) {
    const bool in = j0 + 512 * s < width;
    const u32x4 zero = {0u, 0u, 0u, 0u};  // elements that leave the chains as they are
    const u32x4 xs = exchange_pair(in ? xv[s] : zero);
    u32x4 rs = zero;
    if constexpr (RES) rs = exchange_pair(in ? rv[s] : zero);
#pragma unroll
    for (int e = 0; e < 8; ++e) {
      float a = (e & 1) ? hi_f32<BF16>(xs[e >> 1]) : lo_f32<BF16>(xs[e >> 1]);
      if constexpr (RES) a = __fadd_rn(a, (e & 1) ? hi_f32<BF16>(rs[e >> 1]) : lo_f32<BF16>(rs[e >> 1]));
      v[s][e] = a;
      p[e & 3] = __builtin_fmaf(a, a, p[e & 3]);
    }
  }
#pragma unroll
  for (int e = 0; e < 4; ++e) p[e] = sum_x16(p[e]);                                  // step 128
#pragma unroll
  for (int e = 0; e < 4; ++e) p[e] = __fadd_rn(p[e], dpp<kDppRowRor8>(p[e]));        // step 64
#pragma unroll
  for (int e = 0; e < 4; ++e) p[e] = __fadd_rn(p[e], dpp<kDppHalfMirror>(p[e]));     // step 32
#pragma unroll
  for (int e = 0; e < 4; ++e) p[e] = __fadd_rn(p[e], dpp<kDppQuadXor2>(p[e]));       // step 16
#pragma unroll
  for (int e = 0; e < 4; ++e) p[e] = __fadd_rn(p[e], dpp<kDppQuadXor1>(p[e]));       // step 8
#pragma unroll
  for (int e = 0; e < 4; ++e) p[e] = sum_x32(p[e]);                                  // step 4
  const float total = __fadd_rn(__fadd_rn(p[0], p[2]), __fadd_rn(p[1], p[3]));       // steps 2, 1
  const float scale = rsqrt_rn(__fadd_rn(__fdiv_rn(total, (float)width), eps));
#pragma unroll
  for (int s = 0; s < NP; ++s) {
    const int j = j0 + 512 * s;
    const u32x4 ws = exchange_pair(wv[s]);
    float o[8];
#pragma unroll
    for (int e = 0; e < 8; ++e)
      o[e] = __fmul_rn(__fmul_rn(v[s][e], scale), (e & 1) ? hi_f32<BF16>(ws[e >> 1]) : lo_f32<BF16>(ws[e >> 1]));
    const u32x4 ov = exchange_pair(pack8_rne<BF16>(o));
    u32x4 nv;
    if constexpr (RES) nv = exchange_pair(pack8_rne<BF16>(v[s]));
    if (j < width) {
      if constexpr (RES) {
        if (new_res != nullptr) put(new_res + base + j, nv);
      }
      put(out + base + j, ov);
    }
  }
}

// norm_block_kernel: one 256-thread block per row, thread t walks p[t]'s
// terms.  For few rows, where the latency of one row is the call's time and
// four wavefronts get through it sooner than one, and for rows that
// norm_row_kernel cannot read or hold.  The first KEEP stripes stay in
// registers (their loads, and the weights', all in flight together); stripes
// past them are read a second time.  64 rows of 4096: 4.0 us a call
// (norm_row_kernel 5.4, a loop of dependent loads over the row 11.0); 4096
// rows of 3001: 22.9 us against 50.4.
template <bool BF16, int KEEP>
__global__ __launch_bounds__(256) void norm_block_kernel(const uint16_t* x, const uint16_t* res,
                                                       const uint16_t* __restrict__ w, uint16_t* out,
                                                       uint16_t* new_res, int width, float eps) {
  __shared__ float part[256];
  const int t = threadIdx.x;
  const size_t base = (size_t)blockIdx.x * width;
  auto load = [&](int j) {
    float v = to_f32<BF16>(x[base + j]);
    if (res != nullptr) v = __fadd_rn(v, to_f32<BF16>(res[base + j]));
    return v;
  };
  auto store = [&](int j, float v, float scale, uint32_t wj) {
    if (new_res != nullptr) new_res[base + j] = (uint16_t)from_f32_rne<BF16>(v);
    out[base + j] = (uint16_t)from_f32_rne<BF16>(__fmul_rn(__fmul_rn(v, scale), to_f32<BF16>(wj)));
  };
  uint32_t xr[KEEP], rr[KEEP], wr[KEEP];
#pragma unroll
  for (int k = 0; k < KEEP; ++k) xr[k] = x[base + min(t + 256 * k, width - 1)];
  if (res != nullptr) {
#pragma unroll
    for (int k = 0; k < KEEP; ++k) rr[k] = res[base + min(t + 256 * k, width - 1)];
  }
#pragma unroll
  for (int k = 0; k < KEEP; ++k) wr[k] = w[min(t + 256 * k, width - 1)];
  float v[KEEP];
#pragma unroll
  for (int k = 0; k < KEEP; ++k) v[k] = to_f32<BF16>(xr[k]);
  if (res != nullptr) {
#pragma unroll
    for (int k = 0; k < KEEP; ++k) v[k] = __fadd_rn(v[k], to_f32<BF16>(rr[k]));
  }
  float sum = 0.f;
#pragma unroll
  for (int k = 0; k < KEEP; ++k) {
    if (t + 256 * k >= width) v[k] = 0.f;  // leaves the chain as it is
    sum = __builtin_fmaf(v[k], v[k], sum);
  }
  for (int j = t + 256 * KEEP; j < width; j += 256) {
    const float y = load(j);
    sum = __builtin_fmaf(y, y, sum);
  }
  // Every wavefront folds the 256 partial sums by itself (one barrier): two
  // steps on what it reads, six in registers on the chunk order of
  // norm_row_kernel.
  part[t] = sum;
  __syncthreads();
  const int c8 = t & 7;
  const int l = (t & 56) | (c8 < 4 ? c8 : 11 - c8);
  float p = __fadd_rn(__fadd_rn(part[l], part[l + 128]), __fadd_rn(part[l + 64], part[l + 192]));  // steps 128, 64
  p = sum_x32(p);                                // step 32
  p = sum_x16(p);                                // step 16
  p = __fadd_rn(p, dpp<kDppRowRor8>(p));         // step 8
  p = __fadd_rn(p, dpp<kDppHalfMirror>(p));      // step 4
  p = __fadd_rn(p, dpp<kDppQuadXor2>(p));        // step 2
  p = __fadd_rn(p, dpp<kDppQuadXor1>(p));        // step 1
  const float scale = rsqrt_rn(__fadd_rn(__fdiv_rn(p, (float)width), eps));
#pragma unroll
  for (int k = 0; k < KEEP; ++k)
    if (t + 256 * k < width) store(t + 256 * k, v[k], scale, wr[k]);
  for (int j = t + 256 * KEEP; j < width; j += 256) store(j, load(j), scale, w[j]);
}

// ---------------------------------------------------------------------------
// Fused q/k RMSNorm + RoPE + paged-KV append (head dim 128).
// ---------------------------------------------------------------------------
// Eight lanes (one 8-lane half row) own a 128-element head: lane c holds
// chunk ch = c (c < 4) or 11 - c (c >= 4) of each half, i.e. elements
// 8ch .. 8ch+7 and 64+8ch .. 64+8ch+7 -- the RoPE pairs.  With that chunk
// order the tree's partner at distance 32 is the half-row mirror lane and the
// partners at distances 16 and 8 are lane ^ 2 and lane ^ 1, so the whole
// reduction is three DPP exchanges.
template <bool BF16>
__device__ __forceinline__ void normalize_head(u32x4& x, u32x4& y, u32x4 wl, u32x4 wh, float eps) {
  float a[8], b[8], s[8];
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    a[2 * i] = lo_f32<BF16>(x[i]);
    a[2 * i + 1] = hi_f32<BF16>(x[i]);
    b[2 * i] = lo_f32<BF16>(y[i]);
    b[2 * i + 1] = hi_f32<BF16>(y[i]);
  }
  // tree step 64 (steps 128 and above add zeros): position 8ch + e
#pragma unroll
  for (int e = 0; e < 8; ++e) s[e] = __fadd_rn(__fmul_rn(a[e], a[e]), __fmul_rn(b[e], b[e]));
#pragma unroll
  for (int e = 0; e < 8; ++e) s[e] = __fadd_rn(s[e], dpp<kDppHalfMirror>(s[e]));   // step 32
#pragma unroll
  for (int e = 0; e < 8; ++e) s[e] = __fadd_rn(s[e], dpp<kDppQuadXor2>(s[e]));     // step 16
#pragma unroll
  for (int e = 0; e < 8; ++e) s[e] = __fadd_rn(s[e], dpp<kDppQuadXor1>(s[e]));     // step 8
#pragma unroll
  for (int e = 0; e < 4; ++e) s[e] = __fadd_rn(s[e], s[e + 4]);                     // step 4
#pragma unroll
  for (int e = 0; e < 2; ++e) s[e] = __fadd_rn(s[e], s[e + 2]);                     // step 2
  const float total = __fadd_rn(s[0], s[1]);                                         // step 1
  const float scale = rsqrt_rn(__fadd_rn(__fdiv_rn(total, 128.f), eps));
  float na[8], nb[8];
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    na[2 * i] = __fmul_rn(__fmul_rn(a[2 * i], scale), lo_f32<BF16>(wl[i]));
    na[2 * i + 1] = __fmul_rn(__fmul_rn(a[2 * i + 1], scale), hi_f32<BF16>(wl[i]));
    nb[2 * i] = __fmul_rn(__fmul_rn(b[2 * i], scale), lo_f32<BF16>(wh[i]));
    nb[2 * i + 1] = __fmul_rn(__fmul_rn(b[2 * i + 1], scale), hi_f32<BF16>(wh[i]));
  }
  x = pack8_rne<BF16>(na);
  y = pack8_rne<BF16>(nb);
}

// Work unit = (row, head in [0, hq + 2 hkv)): query heads are normalized with
// qw, rotated and written to q_out [rows][hq][128]; key heads are normalized
// with kw, rotated and written to the K cache at the row's slot; value heads
// are copied to the V cache.  Row r of the input holds q | k | v heads at
// qkv + r * row_stride.  Rows whose slot is outside [0, cache_slots) write
// no cache entry; rows whose position is outside [0, max_pos) are normalized
// but not rotated.  I: index type of the flat work range (uint32_t when it
// fits, which keeps the (row, head) split a 32-bit division).
template <bool BF16, typename I>
__global__ __launch_bounds__(256) void norm_rope_append_kernel(
    const uint16_t* __restrict__ qkv, int64_t row_stride, const uint16_t* __restrict__ qw,
    const uint16_t* __restrict__ kw, float eps, uint16_t* __restrict__ q_out, uint16_t* __restrict__ kc,
    uint16_t* __restrict__ vc, const int64_t* __restrict__ pos, const int64_t* __restrict__ slots,
    const float* __restrict__ cache, int rows, int hq, int hkv, int max_pos, int64_t cache_slots) {
  constexpr int D = 128, H = 64;
  const int heads = hq + 2 * hkv;
  const int64_t total = (int64_t)rows * heads * 8;   // a multiple of 8: groups never straddle the end
  const int c = threadIdx.x & 7;
  const int ch = c < 4 ? c : 11 - c;
  for (I idx = (I)blockIdx.x * blockDim.x + threadIdx.x; idx < (I)total; idx += (I)gridDim.x * blockDim.x) {
    const I unit = idx >> 3;
    const int head = (int)(unit % (I)heads);
    const int64_t row = (int64_t)(unit / (I)heads);
    int64_t slot = 0;
    if (head >= hq) {
      slot = slots[row];
      if (slot < 0 || slot >= cache_slots) continue;   // the whole 8-lane group skips together
    }
    const uint16_t* src = qkv + row * row_stride + (int64_t)head * D;
    u32x4 x = ldv(src + 8 * ch);
    u32x4 y = ldv(src + H + 8 * ch);
    if (head >= hq + hkv) {
      uint16_t* vd = vc + (slot * hkv + (head - hq - hkv)) * D;
      stv(vd + 8 * ch, x);
      stv(vd + H + 8 * ch, y);
      continue;
    }
    const uint16_t* w = head < hq ? qw : kw;
    normalize_head<BF16>(x, y, ldv(w + 8 * ch), ldv(w + H + 8 * ch), eps);
    const int64_t p = pos[row];
    if (p >= 0 && p < max_pos) {
      const float* cs = cache + p * D + 8 * ch;
      rotate8<BF16>(x, y, cs, cs + H);
    }
    uint16_t* dst = head < hq ? q_out + (row * hq + head) * D : kc + (slot * hkv + (head - hq)) * D;
    stv(dst + 8 * ch, x);
    stv(dst + H + 8 * ch, y);
  }
}

// ---------------------------------------------------------------------------
// SiLU-gated product (src/cuda_kernels.cu:18): out[r][c] = T(rn(x / (1 +
// exp(-x))) * up) with x = gu[r][c], up = gu[r][width + c].
// ---------------------------------------------------------------------------
__device__ __forceinline__ float silu_any(float x) { return __fdiv_rn(x, __fadd_rn(1.f, expf(-x))); }

// The same for |x| < kSiluFast, where neither the exponential nor 1 + exp(-x)
// nor its reciprocal can leave the normal range, so that no scaling and no
// special case is needed.  exp(-x) = 2^n 2^f with n the nearest integer to -x
// log2(e) and f the rest, taken with log2(e) in two floats.  The quotient is
// the reciprocal estimate's, corrected once by its residual; it is subnormal
// only for |x| < 2^-125 (bf16), where 1 + exp(-x) is 2 and quotient and
// residual are exact.  The residual's sign is chosen so that a quotient of -0
// stays one: q d - x is +0 there, and -0 is added (x - q d would add +0; a
// copysign for it took 7.42 us for 400 x 12288 in fp16 against 7.13).
constexpr float kSiluFast = 80.f;
__device__ __forceinline__ float silu_fast(float x) {
  constexpr float kL2e = 1.44269502162933349609375f;  // log2(e) rounded to float
  constexpr float kL2eRest = 1.92596299e-08f;         // log2(e) - kL2e
  const float n = __builtin_rintf(__fmul_rn(x, -kL2e));
  const float f = __builtin_fmaf(x, -kL2eRest, __builtin_fmaf(x, -kL2e, -n));
  const float e = __builtin_ldexpf(fast_exp2(f), (int)n);
  const float d = __fadd_rn(1.f, e);
  const float r = __builtin_amdgcn_rcpf(d);
  const float q = __fmul_rn(x, r);
  return __builtin_fmaf(-__builtin_fmaf(q, d, -x), r, q);
}

// n / d for n < 2^31 by a multiplication: mul = floor(2^(31 + l) / d) + 1 with
// l = ceil(log2 d) (d >= 2; d = 1 has mul = 0).
struct FastDiv {
  uint32_t mul, shift;
};
__device__ __forceinline__ uint32_t div31(uint32_t n, FastDiv d) {
  return d.mul != 0 ? __umulhi(n, d.mul) >> d.shift : n;
}

// Eight elements per thread: two 16-byte loads and one store.  HBM bound:
// 8192 x 12288 bf16 takes 92.5 us, 6.5 TB/s of its 604 MB (103 without the
// non-temporal hint; an element per thread with a 64-bit division for its row
// and the full-range exponential and quotient, 188).  The fast form's results
// differ from the correctly rounded ones as often as the full-range form's
// (every finite 16-bit x with 256 values of up: 4549 and 4549 of 16.7 M in
// bf16, 425 and 422 of 16.3 M in fp16) and have its error against 64 bits
// (rms relative 1.65212108047e-3 and 3.95269612522e-3, subnormal results
// included, both forms alike).
template <bool BF16, bool STREAM>
__global__ __launch_bounds__(256) void silu_mul_kernel(const uint16_t* __restrict__ gu, uint16_t* __restrict__ out,
                                                       uint32_t chunks, FastDiv by_chunks, uint32_t total) {
  const uint32_t idx = blockIdx.x * 256u + threadIdx.x;
  if (idx >= total) return;
  const uint32_t row = div31(idx, by_chunks);
  const u32x4* g = reinterpret_cast<const u32x4*>(gu) + (size_t)row * chunks + idx;  // row 2 * chunks long
  u32x4 xv, uv;
  if constexpr (STREAM) {
    xv = __builtin_nontemporal_load(g);
    uv = __builtin_nontemporal_load(g + chunks);
  } else {
    xv = g[0];
    uv = g[chunks];
  }
  float x[8], y[8];
#pragma unroll
  for (int e = 0; e < 8; ++e) {
    x[e] = (e & 1) ? hi_f32<BF16>(xv[e >> 1]) : lo_f32<BF16>(xv[e >> 1]);
    y[e] = silu_fast(x[e]);
  }
  // The largest |x| by its bits, which order infinities and NaNs last.
  typedef uint16_t u16x2 __attribute__((ext_vector_type(2)));
  u16x2 most = {0, 0};
#pragma unroll
  for (int i = 0; i < 4; ++i) most = __builtin_elementwise_max(most, __builtin_bit_cast(u16x2, xv[i] & 0x7fff7fffu));
  constexpr uint16_t kFastBits = BF16 ? 0x42a0 : 0x5500;  // kSiluFast in the 16-bit type
  if (most[0] >= kFastBits || most[1] >= kFastBits) {
#pragma unroll
    for (int e = 0; e < 8; ++e)
      if (!(fabsf(x[e]) < kSiluFast)) y[e] = silu_any(x[e]);
  }
#pragma unroll
  for (int e = 0; e < 8; ++e) y[e] = __fmul_rn(y[e], (e & 1) ? hi_f32<BF16>(uv[e >> 1]) : lo_f32<BF16>(uv[e >> 1]));
  const u32x4 o = pack8_rne<BF16>(y);
  u32x4* dst = reinterpret_cast<u32x4*>(out) + idx;
  if constexpr (STREAM) __builtin_nontemporal_store(o, dst);
  else *dst = o;
}

// Rows that cannot be read eight elements at a time (widths that are no
// multiple of 8, misaligned tensors) and calls past 2^31 chunks.
template <bool BF16, typename I>
__global__ __launch_bounds__(256) void silu_mul_any_kernel(const uint16_t* __restrict__ gu,
                                                           uint16_t* __restrict__ out, int width, int64_t total) {
  for (I idx = (I)blockIdx.x * 256 + threadIdx.x; idx < (I)total; idx += (I)gridDim.x * 256) {
    const I row = idx / (I)width;
    const size_t at = (size_t)row * width + (size_t)idx;  // row 2 * width long
    const float x = to_f32<BF16>(gu[at]);
    const float up = to_f32<BF16>(gu[at + width]);
    const float y = fabsf(x) < kSiluFast ? silu_fast(x) : silu_any(x);
    out[idx] = (uint16_t)from_f32_rne<BF16>(__fmul_rn(y, up));
  }
}

// ---------------------------------------------------------------------------
// Greedy acceptance (src/cuda_kernels.cu:25; src/scheduler.cpp:110), one
// thread per sequence: m = length of the longest prefix on which draft and
// verify agree; out[b][0..k] = verify[b][0..k] (equal to the draft on the
// accepted prefix, then the bonus token verify[m]), out[b][k+1] = m + 1.
// ---------------------------------------------------------------------------
__global__ __launch_bounds__(256) void accept_kernel(const int64_t* __restrict__ draft,
                                                     const int64_t* __restrict__ verify, int64_t* __restrict__ out,
                                                     int batch, int k) {
  const int b = blockIdx.x * blockDim.x + threadIdx.x;
  if (b >= batch) return;
  const int64_t* d = draft + (int64_t)b * k;
  const int64_t* v = verify + (int64_t)b * (k + 1);
  int64_t* o = out + (int64_t)b * (k + 2);
  int m = 0;
  while (m < k && d[m] == v[m]) ++m;
  for (int j = 0; j <= k; ++j) o[j] = v[j];
  o[k + 1] = m + 1;
}

static int grid_for(int64_t work) {
  int64_t g = (work + 255) / 256;
  if (g > 65536) g = 65536;
  if (g < 1) g = 1;
  return (int)g;
}

template <bool BF16>
static hipError_t norm_launch(const uint16_t* x, const uint16_t* res, const uint16_t* w, uint16_t* out,
                              uint16_t* new_res, int rows, int width, float eps, hipStream_t st) {
  const uintptr_t addr = (uintptr_t)x | (uintptr_t)res | (uintptr_t)w | (uintptr_t)out | (uintptr_t)new_res;
  const int stripes = (width + 255) / 256;
  // Up to two rows per compute unit: the block kernel (512 rows of 4096: 6.5
  // against 8.2 us; 1024 rows: 10.1 against 8.8).
  if (rows > 512 && width % 8 == 0 && addr % 16 == 0 && stripes <= 32 && (res != nullptr || new_res == nullptr)) {
    // Two wavefronts per workgroup (8192 x 4096: 51.2 us, 52.5 with one, 52.7
    // with four).
    constexpr int wg = 2;
    // Non-temporal accesses once a call no longer fits the XCDs' L2 (32 MiB):
    // 33 MB 7.8 against 9.9 us without, 134 MB 26.3 against 27.6, 335 MB 62.1
    // against 69.3; below, what the next kernel reads is left in L2 (a decode
    // step's layers 151.2 us without the hint, 154.4 with).  Only where rows
    // fill whole 128-byte lines: 8192 x 1000 takes 14.6 us with it, 11.0
    // without.
    const bool stream = width % 64 == 0 && (int64_t)rows * width * (res != nullptr ? 8 : 4) >= (int64_t(32) << 20);
    auto go = [&](auto kernel) {
      hipLaunchKernelGGL(kernel, dim3((rows + wg - 1) / wg), dim3(64 * wg), 0, st, x, res, w, out, new_res, rows,
                         width, eps);
    };
    auto by_res = [&](auto np) {
      constexpr int NP = decltype(np)::value;
      if (res != nullptr) stream ? go(norm_row_kernel<BF16, NP, true, true>) : go(norm_row_kernel<BF16, NP, true, false>);
      else stream ? go(norm_row_kernel<BF16, NP, false, true>) : go(norm_row_kernel<BF16, NP, false, false>);
    };
    if (stripes <= 2) by_res(std::integral_constant<int, 1>{});
    else if (stripes <= 4) by_res(std::integral_constant<int, 2>{});
    else if (stripes <= 8) by_res(std::integral_constant<int, 4>{});
    else if (stripes <= 12) by_res(std::integral_constant<int, 6>{});
    else if (stripes <= 16) by_res(std::integral_constant<int, 8>{});
    else if (stripes <= 20) by_res(std::integral_constant<int, 10>{});
    else if (stripes <= 24) by_res(std::integral_constant<int, 12>{});
    else by_res(std::integral_constant<int, 16>{});
    return hipGetLastError();
  }
  auto go = [&](auto kernel) {
    hipLaunchKernelGGL(kernel, dim3(rows), dim3(256), 0, st, x, res, w, out, new_res, width, eps);
  };
  // One stripe: 8192 rows of 11 take 6.2 us with one kept, 7.6 with four.  Rows
  // of more stripes than can be kept: while their blocks are all resident (768)
  // what counts are the loads in flight, 600 x 16384 34.3 us with 24 kept, 45.1
  // with 8; many rows need the wavefronts that fewer registers leave room for,
  // the more the longer what is read twice: 2000 x 16384 90.9 and 56.3, 800 x
  // 12288 39.7 and 36.2, but 800 x 9984 28.5 and 28.8, 1600 x 9984 39.0 and 34.5,
  // 3000 x 8704 44.9 and 48.7.
  if (stripes <= 1) go(norm_block_kernel<BF16, 1>);
  else if (stripes <= 4) go(norm_block_kernel<BF16, 4>);
  else if (stripes <= 8) go(norm_block_kernel<BF16, 8>);
  else if (stripes <= 16) go(norm_block_kernel<BF16, 16>);
  else if (stripes <= 34 || rows <= (stripes < 48 ? 1536 : 768)) go(norm_block_kernel<BF16, 24>);
  else go(norm_block_kernel<BF16, 8>);
  return hipGetLastError();
}

hipError_t launch_norm(const void* x, const void* res, const void* w, void* out, void* new_res, int rows, int width,
                       float eps, bool bf16, hipStream_t st) {
  if (rows == 0) return hipSuccess;
  auto go = [&](auto bf) {
    return norm_launch<decltype(bf)::value>((const uint16_t*)x, (const uint16_t*)res, (const uint16_t*)w,
                                            (uint16_t*)out, (uint16_t*)new_res, rows, width, eps, st);
  };
  return bf16 ? go(std::true_type{}) : go(std::false_type{});
}

hipError_t launch_norm_rope_append(const void* qkv, int64_t row_stride, const void* qw, const void* kw, float eps,
                                   void* q_out, void* kc, void* vc, const int64_t* pos, const int64_t* slots,
                                   const float* cache, int rows, int hq, int hkv, bool bf16, int max_pos,
                                   int64_t cache_slots, hipStream_t st) {
  const int64_t work = (int64_t)rows * (hq + 2 * hkv) * 8;
  if (work == 0) return hipSuccess;
  const int grid = grid_for(work);
  auto go = [&](auto kernel) {
    hipLaunchKernelGGL(kernel, dim3(grid), dim3(256), 0, st, (const uint16_t*)qkv, row_stride, (const uint16_t*)qw,
                       (const uint16_t*)kw, eps, (uint16_t*)q_out, (uint16_t*)kc, (uint16_t*)vc, pos, slots, cache,
                       rows, hq, hkv, max_pos, cache_slots);
  };
  const bool narrow = work <= INT32_MAX;  // idx + grid stride stays below 2^32
  if (bf16) narrow ? go(norm_rope_append_kernel<true, uint32_t>) : go(norm_rope_append_kernel<true, int64_t>);
  else narrow ? go(norm_rope_append_kernel<false, uint32_t>) : go(norm_rope_append_kernel<false, int64_t>);
  return hipGetLastError();
}

template <bool BF16>
static hipError_t silu_launch(const uint16_t* gu, uint16_t* out, int rows, int width, hipStream_t st) {
  const int64_t total = (int64_t)rows * width;
  if (width % 8 == 0 && ((uintptr_t)gu | (uintptr_t)out) % 16 == 0 && total / 8 < INT32_MAX - 256) {
    const uint32_t chunks = (uint32_t)width / 8, n = (uint32_t)(total / 8);
    FastDiv by{0, 0};
    if (chunks > 1) {
      const int l = 32 - __builtin_clz(chunks - 1);  // ceil(log2 chunks)
      by = FastDiv{(uint32_t)((uint64_t(1) << (31 + l)) / chunks + 1), (uint32_t)(l - 1)};
    }
    // Non-temporal accesses under fe_norm's rule (past 32 MiB, whole lines):
    // 200 MB 31.8 against 35.6 us, 50 MB 9.2 against 9.3, 16 MB 6.9 against
    // 6.75.
    const bool stream = width % 64 == 0 && 6 * total >= (int64_t(32) << 20);
    auto go = [&](auto kernel) {
      hipLaunchKernelGGL(kernel, dim3((n + 255) / 256), dim3(256), 0, st, gu, out, chunks, by, n);
    };
    stream ? go(silu_mul_kernel<BF16, true>) : go(silu_mul_kernel<BF16, false>);
  } else if (total <= INT32_MAX) {  // idx + grid stride stays below 2^32
    hipLaunchKernelGGL((silu_mul_any_kernel<BF16, uint32_t>), dim3(grid_for(total)), dim3(256), 0, st, gu, out, width,
                       total);
  } else {
    hipLaunchKernelGGL((silu_mul_any_kernel<BF16, int64_t>), dim3(grid_for(total)), dim3(256), 0, st, gu, out, width,
                       total);
  }
  return hipGetLastError();
}

hipError_t launch_silu_mul(const void* gu, void* out, int rows, int width, bool bf16, hipStream_t st) {
  if ((int64_t)rows * width == 0) return hipSuccess;
  return bf16 ? silu_launch<true>((const uint16_t*)gu, (uint16_t*)out, rows, width, st)
              : silu_launch<false>((const uint16_t*)gu, (uint16_t*)out, rows, width, st);
}

hipError_t launch_accept(const int64_t* draft, const int64_t* verify, int64_t* out, int batch, int k,
                         hipStream_t st) {
  if (batch == 0) return hipSuccess;
  hipLaunchKernelGGL(accept_kernel, dim3((batch + 255) / 256), dim3(256), 0, st, draft, verify, out, batch, k);
  return hipGetLastError();
}

}  // namespace feattn
