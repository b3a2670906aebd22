// Short-context attention: one workgroup per (<= 32 (query row, head)
// columns, kv head, token range) item, its tokens divided among the
// workgroup's wavefronts and their results combined in LDS.
#pragma once
#include "attn_types.hpp"
#include "device_util.hpp"
#include "kernel_util.hpp"

namespace feattn {

constexpr int kShortBlock = 4096;               // 16 tokens x 256 bytes
constexpr int kShortWave = 4 * kShortBlock;     // a wavefront's LDS: 64 tokens of V, then its 32 x 128 fp32 results
template <int WAVES>
constexpr size_t short_lds() {
  return (size_t)WAVES * kShortWave + (size_t)WAVES * kDecodeCols * 2 * sizeof(float);
}

typedef int32_t i32x4 __attribute__((ext_vector_type(4)));
typedef int32_t i32x8 __attribute__((ext_vector_type(8)));

// K of the wavefront's next 64 tokens goes to registers (lane 16 J + L:
// token L of a block, dims 32 s + 8 J .. +8, the A operand of S^T = K Q^T as
// it is), V to the wavefront's LDS region with the tile kernel's layout, and
// all of it is in flight at once: an item of WAVES * 64 tokens costs one
// memory round trip after its record (the record names the first 64 tokens'
// blocks of every wavefront).  Then S^T, one softmax step and O^T += V^T P^T
// over the 64 tokens as in the tile kernel.
// GRID2: a workgroup's unit is (record blockIdx.y, kv head blockIdx.x); else
// the workgroups loop over n_items units (a graph's grid covers any prepare's),
// at the price of a division (0.05 us).
template <bool BF16, int WAVES, int NCB, bool GRID2>
__device__ __forceinline__ void short_items(const AttnArgs& a, int causal, int n_items, uint8_t* dsm) {
  const int lane = threadIdx.x & 63;
  const int J = lane >> 4;
  const int L = lane & 15;
  const int wave = uniform(threadIdx.x >> 6);
  const int G = a.group;
  const int row_bytes = a.hkv * kHeadDim * 2;
  const uint32_t lbase = (uint32_t)(uintptr_t)dsm;
  const uint32_t vst = lbase + (uint32_t)(wave * kShortWave);
  const uint32_t mlbase = lbase + (uint32_t)(WAVES * kShortWave);
  typedef __attribute__((address_space(3))) float lds_f32;
  typedef __attribute__((address_space(3))) f32x4 lds_f32x4;

  const uint32_t k_goff = (uint32_t)(L * row_bytes + 16 * J);
  uint32_t v_goff[4];
#pragma unroll
  for (int r = 0; r < 4; ++r) {
    const int t = 4 * r + J;
    v_goff[r] = (uint32_t)(t * row_bytes + 16 * (L ^ ((2 * t) & 15)));
  }
  uint32_t v_lds[8];
  {
    const int k = L >> 2, m = L & 3, t = 4 * J + k;
#pragma unroll
    for (int db = 0; db < 8; ++db) {
      const int c = 2 * db + (m >> 1);
      v_lds[db] = (uint32_t)(16 * (16 * t + ((c ^ (2 * t)) & 15)) + 8 * (m & 1));
    }
  }

  for (int it = GRID2 ? 0 : blockIdx.x; it < n_items; it += gridDim.x) {
    const int ri = GRID2 ? (int)blockIdx.y : uniform(it / a.hkv);
    const int kvh = GRID2 ? (int)blockIdx.x : uniform(it) - ri * a.hkv;
    const ShortItem* rec = a.shorts + ri;
    typedef const __attribute__((address_space(4))) i32x8* c_i32x8;
    typedef const __attribute__((address_space(4))) i32x4* c_i32x4;
    const i32x8 h = *(c_i32x8)rec;
    const i32x4 first = *(c_i32x4)(rec->block + 4 * wave);
    const int q0 = h[0], nq = h[1], vis = h[2], t0 = h[3], t1 = h[4], part = h[5], page_off = h[6];
    const int ncols = nq * G;
    const int nblk = (t1 - t0 + 15) >> 4;
    const int nbw = (nblk + WAVES - 1) / WAVES;     // blocks per wavefront
    const int nact = (nblk + nbw - 1) / nbw;        // wavefronts with blocks
    const int b0 = wave * nbw;
    const int nb = min(nblk, b0 + nbw) - b0;        // this wavefront's blocks (<= 0: none)
    const int wt0 = t0 + 16 * b0;
    const int wt1 = min(t1, wt0 + 16 * nb);

    float m[NCB], lsum[NCB];
    f32x4 o[8][NCB];
#pragma unroll
    for (int cb = 0; cb < NCB; ++cb) {
      m[cb] = kNegInf;
      lsum[cb] = 0.f;
#pragma unroll
      for (int db = 0; db < 8; ++db) o[db][cb] = f32x4{0.f, 0.f, 0.f, 0.f};
    }

    if (nb > 0) {
      const char* khead = reinterpret_cast<const char*>(a.kc) + (size_t)kvh * kHeadDim * 2;
      const char* vhead = reinterpret_cast<const char*>(a.vc) + (size_t)kvh * kHeadDim * 2;
      size_t blk[4];
      u32x4 kf[4][4];
      // Blocks past the wavefront's last are read as its last one: every
      // address is one of the item's, and what they hold is masked.
      auto locate = [&](int tok, int i) {
        const int t = min(tok + 16 * i, wt0 + 16 * (nb - 1));
        const int pg = ldc(a.pages, page_off + (t >> a.page_shift));
        return (((size_t)pg << a.page_shift) + (size_t)(t & ((1 << a.page_shift) - 1))) * (size_t)row_bytes;
      };
      auto load_k = [&]() {
#pragma unroll
        for (int i = 0; i < 4; ++i)
#pragma unroll
          for (int s = 0; s < 4; ++s) kf[i][s] = *reinterpret_cast<const u32x4*>(khead + blk[i] + k_goff + 64 * s);
      };
      auto copy_v = [&](int live) {
#pragma unroll
        for (int i = 0; i < 4; ++i)
          if (i < live) {
#pragma unroll
            for (int r = 0; r < 4; ++r)
              lds_dma16(vhead + blk[i], v_goff[r], vst + (uint32_t)(i * kShortBlock + 1024 * r));
          }
      };
#pragma unroll
      for (int i = 0; i < 4; ++i) blk[i] = (size_t)(uint32_t)first[i] * (size_t)(16 * row_bytes);
      u32x4 qf[NCB][4];
      int lim[NCB];
      // (Opaque, here and below: what is derived from the lane alone would
      // otherwise be computed before the item loop and held, or spilled,
      // through all of it.)
      int lq = lane;
      asm volatile("" : "+v"(lq));
#pragma unroll
      for (int cb = 0; cb < NCB; ++cb) {
        const int n = 16 * cb + (lq & 15);
        const bool ok = n < ncols;
        const int nn = ok ? n : 0;
        const int r = nn / G;
        lim[cb] = ok ? min(causal ? vis + r : t1 - 1, wt1 - 1) : -1;
        const uint16_t* qp = a.q + ((size_t)(q0 + r) * a.hq + kvh * G + (nn - r * G)) * kHeadDim + 8 * (lq >> 4);
#pragma unroll
        for (int k = 0; k < 4; ++k) qf[cb][k] = ld16(qp + 32 * k);
      }
      load_k();
      copy_v(nb);

      for (int tok = wt0; tok < wt1; tok += 64) {
        const int live = min(4, (wt1 - tok + 15) >> 4);
        wait_vmem<0>();
        f32x4 sc[4][NCB];
#pragma unroll
        for (int tb = 0; tb < 4; ++tb) {
#pragma unroll
          for (int cb = 0; cb < NCB; ++cb) sc[tb][cb] = f32x4{0.f, 0.f, 0.f, 0.f};
          if (tb < live) {
#pragma unroll
            for (int k = 0; k < 4; ++k)
#pragma unroll
              for (int cb = 0; cb < NCB; ++cb) sc[tb][cb] = mfma16<BF16>(kf[tb][k], qf[cb][k], sc[tb][cb]);
          }
        }
        __builtin_amdgcn_sched_barrier(0);
        const bool more = tok + 64 < wt1;
        if (more) {
#pragma unroll
          for (int i = 0; i < 4; ++i) blk[i] = locate(tok + 64, i);
          if constexpr (NCB == 1) load_k();  // under the softmax (two column blocks have no registers for that)
        }

        u32x4 pf[2][NCB];
#pragma unroll
        for (int cb = 0; cb < NCB; ++cb) {
          float mx = kNegInf;
#pragma unroll
          for (int tb = 0; tb < 4; ++tb)
#pragma unroll
            for (int r = 0; r < 4; ++r) {
              if (tok + 16 * tb + 4 * J + r > lim[cb]) sc[tb][cb][r] = kNegInf;
              mx = fmaxf(mx, sc[tb][cb][r]);
            }
          mx = max_x32(max_x16(mx));
          const float mt = mx * a.scale_log2;
          const bool up = mt > m[cb] + 8.f;  // lazy reference maximum, as in the tile kernel
          const float alpha = up ? fast_exp2(m[cb] - mt) : 1.f;
          if (up) m[cb] = mt;
          const float m_use = m[cb] == kNegInf ? 0.f : m[cb];
          float x[4][4];
          float ps = 0.f;
#pragma unroll
          for (int tb = 0; tb < 4; ++tb)
#pragma unroll
            for (int r = 0; r < 4; ++r) {
              x[tb][r] = fast_exp2(__builtin_fmaf(sc[tb][cb][r], a.scale_log2, -m_use));
              ps += x[tb][r];
            }
          lsum[cb] = lsum[cb] * alpha + ps;
          if (__builtin_amdgcn_ballot_w64(up) != 0) {
#pragma unroll
            for (int db = 0; db < 8; ++db) o[db][cb] *= alpha;
          }
#pragma unroll
          for (int ks = 0; ks < 2; ++ks) {
            pf[ks][cb][0] = pack2<BF16>(x[2 * ks][0], x[2 * ks][1]);
            pf[ks][cb][1] = pack2<BF16>(x[2 * ks][2], x[2 * ks][3]);
            pf[ks][cb][2] = pack2<BF16>(x[2 * ks + 1][0], x[2 * ks + 1][1]);
            pf[ks][cb][3] = pack2<BF16>(x[2 * ks + 1][2], x[2 * ks + 1][3]);
          }
        }

        __builtin_amdgcn_sched_barrier(0);
        // V rows past the last token, up to the 32-token step they end in,
        // hold stale cache or LDS contents: zero (0 * stale must stay 0).
        const int valid = wt1 - tok;
        const int rows = live > 2 ? 64 : 32;
        if (valid < rows) {
          for (int q = 16 * valid + lane; q < 16 * rows; q += 64) lds_zero16(vst + 16 * q);
        }
#pragma unroll
        for (int ks = 0; ks < 2; ++ks)
          if (ks == 0 || live > 2) {
#pragma unroll
            for (int db = 0; db < 8; ++db) {
              const u32x2 lo = lds_read_tr16(vst + v_lds[db] + (2 * ks) * kShortBlock);
              const u32x2 hi = lds_read_tr16(vst + v_lds[db] + (2 * ks + 1) * kShortBlock);
              const u32x4 vf = {lo[0], lo[1], hi[0], hi[1]};
#pragma unroll
              for (int cb = 0; cb < NCB; ++cb) o[db][cb] = mfma16<BF16>(vf, pf[ks][cb], o[db][cb]);
            }
          }
        if (more) {
          wait_lds();  // the reads of this step's V are complete
          if constexpr (NCB > 1) load_k();
          copy_v((wt1 - tok - 64 + 15) >> 4);
        }
      }
      // fp32 results and statistics to LDS: row = column, 16-byte chunk c
      // (dims 4 c ..) at chunk position c ^ L.
      wait_lds();
      int ln = lane;
      asm volatile("" : "+v"(ln));
      const int Lo = ln & 15, Jo = ln >> 4;
#pragma unroll
      for (int cb = 0; cb < NCB; ++cb) {
        const float ls = sum_x32(sum_x16(lsum[cb]));
#pragma unroll
        for (int db = 0; db < 8; ++db)
          *(lds_f32x4*)(uintptr_t)(vst + (uint32_t)(512 * (16 * cb + Lo) + 16 * ((4 * db + Jo) ^ Lo))) = o[db][cb];
        if (Jo == 0) {
          const uint32_t ml = mlbase + (uint32_t)(8 * (wave * kDecodeCols + 16 * cb + Lo));
          *(lds_f32*)(uintptr_t)ml = m[cb];
          *(lds_f32*)(uintptr_t)(ml + 4) = ls;
        }
      }
    }
    __syncthreads();

    // Combine: a 32-lane half per column, 4 dims per lane.
    int ln = lane;
    asm volatile("" : "+v"(ln));
    const int c = ln & 31;
    for (int n = 2 * wave + (ln >> 5); n < 16 * NCB; n += 2 * WAVES) {
      if (n >= ncols) break;
      float mw[WAVES], lw[WAVES];
      float top = kNegInf;
#pragma unroll
      for (int w = 0; w < WAVES; ++w) {
        mw[w] = kNegInf;
        lw[w] = 0.f;
        if (w < nact) {
          const uint32_t ml = mlbase + (uint32_t)(8 * (w * kDecodeCols + n));
          mw[w] = *(lds_f32*)(uintptr_t)ml;
          lw[w] = *(lds_f32*)(uintptr_t)(ml + 4);
        }
        top = fmaxf(top, mw[w]);
      }
      const float base = top == kNegInf ? 0.f : top;
      float ls = 0.f;
      f32x4 acc = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int w = 0; w < WAVES; ++w)
        if (w < nact) {
          const float wt = fast_exp2(mw[w] - base);
          ls += lw[w] * wt;
          acc += *(lds_f32x4*)(uintptr_t)(lbase + (uint32_t)(w * kShortWave + 512 * n + 16 * (c ^ (n & 15)))) * wt;
        }
      const float inv = ls > 0.f ? 1.f / ls : 0.f;
      const float l2 = ls > 0.f ? top + __log2f(ls) : kNegInf;
      const int r = n / G, head = kvh * G + (n - r * G);
      const u32x2 v = {pack2<BF16>(acc[0] * inv, acc[1] * inv), pack2<BF16>(acc[2] * inv, acc[3] * inv)};
      if (part < 0) {
        const size_t oi = (size_t)(q0 + r) * a.hq + head;
        *reinterpret_cast<u32x2*>(a.out + oi * kHeadDim + 4 * c) = v;
        if (a.lse != nullptr && c == 0) a.lse[oi] = l2 * kLn2;
      } else {
        const size_t oi = (size_t)(part + r) * a.hq + head;
        *reinterpret_cast<u32x2*>(a.part_o + oi * kHeadDim + 4 * c) = v;
        if (c == 0) a.part_lse[oi] = l2;
      }
    }
    if constexpr (GRID2) break;
    if (it + (int)gridDim.x < n_items) __syncthreads();  // the regions are the next item's V
  }
}

}  // namespace feattn
