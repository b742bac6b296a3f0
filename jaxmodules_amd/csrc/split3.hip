// Masked attention at float32 accuracy on the matrix cores (split3.hpp): the
// forward and the backward of float32 inputs at D = 64, 128 and 256 and of 16-bit
// inputs at D = 256 (MATTN_PRECISE: precise.hip; D = 512: the SIMT kernels of
// simt.hip, which these replaced).  Measured against them: float32
// causal [2, 2048, 8, 64] fwd 465 -> 87 us, dK/dV 768 -> 165, dQ 596 -> 126 (the
// step 16.9 -> 86 TFLOP/s); bfloat16 causal [1, 4096, 8, 256] fwd 4322 -> 326 us,
// dK/dV 14370 -> 750, dQ 4811 -> 708 (10 -> 139 TFLOP/s).  Their error against
// float64 is no larger (float32 step: 6.6e-7 of the norm, 1.1e-6 before).
// Bound by the matrix cores and the split's VALU work together: a 32 x 32 block
// of the float32 forward at D = 64 takes 48 MFMAs (1536 cycles) and about 300
// vector instructions.
//
// Same maths and tile walk as there (/root/reference/jaxmodules/
// attention.py:52-105 forward, :266-342 backward).  Every wave owns 32 rows
// (queries in the forward and dQ, keys in dK/dV), one per lane pair, and walks
// the present tiles of its map row or column, sub-block by sub-block:
//   forward  S^T = K Q^T, online softmax, O^T += V^T P^T
//   dQ       S^T = K Q^T, dP^T = V dO^T, dS = P (dP - delta), dQ^T += K^T dS^T
//   dK/dV    S = Q K^T, dP = dO V^T, dV^T += dO^T P, dK^T += Q^T dS
// The streamed tensors are read once per workgroup, split into bfloat16 pieces
// on the way to LDS (the next sub-block's rows are in registers meanwhile);
// the wave's own rows are split in registers.  P and dS are split from the
// C registers, which are the B operand of the next product as they stand.
//
// A workgroup is WQ x WK x DS waves: WQ groups of 32 own rows; WK waves per group
// that take every WK-th 32-row block of a sub-block and sum their results through
// LDS at the end; and DS = 2 waves that each hold one half of the columns (of the
// own rows' operands and of the result), form S and dP over that half and add the
// partner's through LDS, so that a wave's operands and accumulators fit half the
// registers and two waves share a SIMD.
#include <type_traits>

#include "split3.hpp"

namespace mattn {
namespace {
using namespace s3;

// own row operands: row r of a tensor slice, k-step kd = columns c0 + 16 kd + 8 hi .. + 7
template <class T, int N>
__device__ __forceinline__ void own_rows(Frag<Pieces<T>::n> (&f)[N], const char* base, int64_t rs, int r, int c0, int hi) {
#pragma unroll
  for (int kd = 0; kd < N; ++kd) {
    Raw8<T> x;
    x.load(base + elt_bytes<T>() * ((int64_t)r * rs + c0 + 16 * kd + 8 * hi));
    f[kd] = x.split();
  }
}

// Place of this wave in its workgroup
template <int WQ, int WK, int DS>
struct Place {
  static constexpr int NTH = 64 * WQ * WK * DS, NSUB = TILE / (32 * WQ);  // workgroups per 128-row tile
  int lane, l32, hi, wave, wq, wk, ds;
  __device__ __forceinline__ Place() {
    lane = threadIdx.x & 63;
    l32 = lane & 31;
    hi = lane >> 5;
    wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    wq = wave % WQ;
    wk = wave / WQ % WK;
    ds = wave / (WQ * WK);
  }
  __device__ __forceinline__ int partner() const { return wave ^ (WQ * WK); }  // DS = 2: the other half
};

constexpr int cmax(int a, int b) { return a > b ? a : b; }

// the 32 mask bits of row `row` (of a tile) against the 32-row block `blk` of the other side
__device__ __forceinline__ uint32_t bits32(const uint64_t* bits, int mask, int blk, int row) {
  return (uint32_t)(bits[((int64_t)mask * 2 + (blk >> 1)) * TILE + row] >> (32 * (blk & 1)));
}

// The walk over n sub-blocks: with one LDS buffer a sub-block is staged between two
// barriers, with two it is staged while the one before it is computed.
template <int NBUF, class S, class C>
__device__ __forceinline__ void run_walk(int n, S&& stage, C&& compute) {
  if constexpr (NBUF == 2) {
    if (n > 0) stage(0);
    for (int s = 0; s < n; ++s) {
      __syncthreads();
      if (s + 1 < n) stage(s + 1);
      compute(s);
    }
  } else {
    for (int s = 0; s < n; ++s) {
      __syncthreads();
      stage(s);
      __syncthreads();
      compute(s);
    }
  }
}

// ---------------------------------------------------------------------------
// forward
// ---------------------------------------------------------------------------
template <int D, class IT, class OT, int BN, int WQ, int WK, int DS, int NBUF, int MINW>
__global__ __attribute__((amdgpu_flat_work_group_size(64 * WQ * WK * DS, 64 * WQ * WK * DS), amdgpu_waves_per_eu(MINW, MINW)))
void fwd_s3(KArgs a) {
  using W = Place<WQ, WK, DS>;
  constexpr int NP = Pieces<IT>::n, DW = D / DS, NKD = DW / 16, NMD = DW / 32;
  constexpr int RPW = 32 * WQ, NT = BN / (32 * WK);
  static_assert(WK == 1 || DS == 1, "");
  using St = Stage<D, IT, BN, W::NTH>;
  constexpr int BUF = 2 * St::ELTS;  // K planes, then V planes
  constexpr int XCH = DS == 1 ? 0 : W::NTH * 16 * NT * 2;  // S halves (in 16-bit elements)
  constexpr int OUT = WK == 1 ? WQ * DS * put_bytes<DW>() : WK * RPW * D * 4;
  __shared__ __attribute__((aligned(16))) uint16_t L[cmax(NBUF * BUF + XCH, OUT / 2)];
  __shared__ float Ml[2][WK == 1 ? 1 : WQ * WK][32];

  const int item = a.q_order[blockIdx.x / W::NSUB];
  if (item < 0 || item >= a.B * a.Hq * a.nqt) return;  // idle slot (or an entry out of range)
  const int qt = item % a.nqt, bh = item / a.nqt;
  const int h = bh % a.Hq, b = bh / a.Hq, hk = h / a.G;
  const int mrow = map_row(a, b, h, a.nqt, qt);
  const Walk<BN> walk(a.row_ent, a.row_ptr[mrow], a.row_ptr[mrow + 1]);
  const W w;
  const int wrow = (blockIdx.x % W::NSUB) * RPW;  // workgroup's first row in the tile
  if (qt * TILE + wrow >= a.Lq) return;           // (a ragged last tile's empty part)
  const int qloc = wrow + 32 * w.wq + w.l32;
  const int q = qt * TILE + qloc;

  const char* kb = head_base(a.k, a.ks, b, hk, elt_bytes<IT>());
  const char* vb = head_base(a.v, a.vs, b, hk, elt_bytes<IT>());
  St ks, vs;
  if (walk.n > 0) {
    ks.load(kb, a.ks[1], walk.first(0), a.Lk);
    vs.load(vb, a.vs[1], walk.first(0), a.Lk);
  }
  Frag<NP> qf[NKD];
  own_rows<IT>(qf, head_base(a.q, a.qs, b, h, elt_bytes<IT>()), a.qs[1], min(q, a.Lq - 1), w.ds * DW, w.hi);

  f32x16 acc[NMD];
#pragma unroll
  for (int i = 0; i < NMD; ++i) acc[i] = f32x16{};
  float m2 = NEG_INF, l = 0.f;
  const float c2 = a.scale_log2;
  float* X = (float*)(L + NBUF * BUF);

  auto stage = [&](int s) {  // registers -> LDS buffer of sub-block s; the next one's rows -> registers
    uint16_t* buf = L + (NBUF == 2 ? (s & 1) * BUF : 0);
    ks.store(buf);
    vs.store(buf + St::ELTS);
    if (s + 1 < walk.n) {
      ks.load(kb, a.ks[1], walk.first(s + 1), a.Lk);
      vs.load(vb, a.vs[1], walk.first(s + 1), a.Lk);
    }
  };
  auto compute = [&](int s) {
    const uint16_t* Kl = L + (NBUF == 2 ? (s & 1) * BUF : 0);
    const uint16_t* Vl = Kl + St::ELTS;
    const int mask = walk.mask(s), blk0 = (s % Walk<BN>::SPT) * (BN / 32) + w.wk * NT;
    uint32_t w32[NT];
    bool live = true;
    if (mask >= 0) {
      bool any = false;
#pragma unroll
      for (int t = 0; t < NT; ++t) {
        w32[t] = bits32(a.row_bits, mask, blk0 + t, qloc);
        any |= w32[t] != 0;
      }
      live = __any(any);  // an allowed key of the wave's rows here
    }
    f32x16 st[NT];
    if (live) {
#pragma unroll
      for (int t = 0; t < NT; ++t) {
        st[t] = f32x16{};
#pragma unroll
        for (int kd = 0; kd < NKD; ++kd)
          st[t] = mma(row_frag<D, NP, BN>(Kl, 32 * (w.wk * NT + t) + w.l32, w.ds * NKD + kd, w.hi), qf[kd], st[t]);
      }
      if constexpr (DS == 2) half_put(st, X, w.wave, w.lane);
    }
    if constexpr (DS == 2) __syncthreads();
    if (!live) return;
    if constexpr (DS == 2) half_add(st, X, w.partner(), w.lane);
    if (mask >= 0) {
#pragma unroll
      for (int t = 0; t < NT; ++t)
#pragma unroll
        for (int r = 0; r < 16; ++r) st[t][r] = mask_neg_inf(st[t][r], mask_ones(w32[t] >> (4 * w.hi), r));
    }
    float mx = NEG_INF;
#pragma unroll
    for (int t = 0; t < NT; ++t)
#pragma unroll
      for (int r = 0; r < 16; ++r) mx = fmaxf(mx, st[t][r]);
    const float mx2 = wave_max32(mx) * c2;
    // the running max is raised only when a row's grows by more than 2^8 (P <= 2^8
    // until then; the pieces keep float32's range)
    if (__any(mx2 > m2 + 8.f)) {
      const float mn = fmaxf(m2, mx2);
      const float alpha = (mn == NEG_INF) ? 1.f : fast_exp2(m2 - mn);
      l *= alpha;
#pragma unroll
      for (int i = 0; i < NMD; ++i) acc[i] *= alpha;
      m2 = mn;
    }
    const float nmu = (m2 == NEG_INF) ? 0.f : -m2;
#pragma unroll
    for (int t = 0; t < NT; ++t) {
#pragma unroll
      for (int r = 0; r < 16; ++r) {
        st[t][r] = fast_exp2(fmaf(st[t][r], c2, nmu));
        l += st[t][r];
      }
#pragma unroll
      for (int j = 0; j < 2; ++j) {
        const Frag<3> pf = c_frag(st[t], j);
#pragma unroll
        for (int mt = 0; mt < NMD; ++mt)
          acc[mt] = mma(tr_frag<D, NP, BN>(Vl, 32 * (w.wk * NT + t) + 16 * j, w.ds * NMD + mt, w.lane), pf, acc[mt]);
      }
    }
  };
  run_walk<NBUF>(walk.n, stage, compute);

  l = wave_sum32(l);
  const int nrows = a.Lq - (qt * TILE + wrow);
  const int64_t orow = (int64_t)b * a.os[0] + (int64_t)(qt * TILE + wrow) * a.os[1] + (int64_t)h * a.os[2];
  float* lse = a.lse + ((int64_t)b * a.Hq + h) * a.Lq;
  __syncthreads();  // every wave is done with the operand tiles
  if constexpr (WK == 1) {
    if (w.ds == 0 && w.hi == 0 && q < a.Lq) lse[q] = l > 0.f ? m2 + __builtin_log2f(l) : NEG_INF;
    put_rows<DW, OT>(acc, l > 0.f ? 1.f / l : 0.f, (char*)L + w.wave * put_bytes<DW>(), a.out,
                     orow + (int64_t)32 * w.wq * a.os[1] + w.ds * DW, a.os[1], nrows - 32 * w.wq, w.lane);
  } else {
    if (w.hi == 0) {
      Ml[0][w.wave][w.l32] = m2;
      Ml[1][w.wave][w.l32] = l;
    }
    __syncthreads();
    float M = NEG_INF, lt = 0.f;
#pragma unroll
    for (int k = 0; k < WK; ++k) M = fmaxf(M, Ml[0][k * WQ + w.wq][w.l32]);
#pragma unroll
    for (int k = 0; k < WK; ++k) {
      const float mk = Ml[0][k * WQ + w.wq][w.l32];
      lt += mk == NEG_INF ? 0.f : Ml[1][k * WQ + w.wq][w.l32] * fast_exp2(mk - M);
    }
    const float f = (m2 == NEG_INF || !(lt > 0.f)) ? 0.f : fast_exp2(m2 - M) / lt;
    if (w.wk == 0 && w.hi == 0 && q < a.Lq) lse[q] = lt > 0.f ? M + __builtin_log2f(lt) : NEG_INF;
    slab_put<D, WQ>(acc, f, (float*)L, w.wq, w.wk, w.lane);
    __syncthreads();
    slab_sum_store<D, OT, WQ, WK, W::NTH>((const float*)L, a.out, orow, a.os[1], nrows);
  }
}

// ---------------------------------------------------------------------------
// backward
// ---------------------------------------------------------------------------

// delta = rowsum(dO * O), summed in float64: D / 8 threads a row, the rows in the
// order of memory (head fastest where a row of O holds all heads)
template <int D, class OT>
__global__ __attribute__((amdgpu_flat_work_group_size(256, 256)))
void delta_s3(KArgs a) {
  constexpr int TPR = D / 8;
  const int64_t i = ((int64_t)blockIdx.x * 256 + threadIdx.x) / TPR;
  const int part = threadIdx.x % TPR;
  if (i >= (int64_t)a.B * a.Hq * a.Lq) return;
  int b, h, q;
  if (a.os[2] < a.os[1]) {
    h = i % a.Hq;
    q = (i / a.Hq) % a.Lq;
    b = i / ((int64_t)a.Hq * a.Lq);
  } else {
    q = i % a.Lq;
    h = (i / a.Lq) % a.Hq;
    b = i / ((int64_t)a.Hq * a.Lq);
  }
  const char* o = head_base(a.o, a.os, b, h, elt_bytes<OT>()) + elt_bytes<OT>() * ((int64_t)q * a.os[1] + 8 * part);
  const char* g = head_base(a.dO, a.dos, b, h, elt_bytes<OT>()) + elt_bytes<OT>() * ((int64_t)q * a.dos[1] + 8 * part);
  double s = 0.;
  if constexpr (std::is_same<OT, float>::value) {
#pragma unroll
    for (int j = 0; j < 2; ++j) {
      const f32x4 x = *(const f32x4*)(o + 16 * j), y = *(const f32x4*)(g + 16 * j);
#pragma unroll
      for (int e = 0; e < 4; ++e) s += (double)x[e] * (double)y[e];
    }
  } else {
    const u32x4 x = *(const u32x4*)o, y = *(const u32x4*)g;
#pragma unroll
    for (int e = 0; e < 8; ++e) s += (double)Elt<OT>::to_f32(elt16(x, e)) * (double)Elt<OT>::to_f32(elt16(y, e));
  }
#pragma unroll
  for (int m = 1; m < TPR; m <<= 1) s += __shfl_xor(s, m);
  if (part == 0) a.delta[((int64_t)b * a.Hq + h) * a.Lq + q] = (float)s;
}

template <int D, class IT, class OT, int BN, int WQ, int WK, int DS, int NBUF, int MINW>
__global__ __attribute__((amdgpu_flat_work_group_size(64 * WQ * WK * DS, 64 * WQ * WK * DS), amdgpu_waves_per_eu(MINW, MINW)))
void bwd_dq_s3(KArgs a) {
  using W = Place<WQ, WK, DS>;
  constexpr int NP = Pieces<IT>::n, NG = Pieces<OT>::n, DW = D / DS, NKD = DW / 16, NMD = DW / 32;
  constexpr int RPW = 32 * WQ, NT = BN / (32 * WK);
  static_assert(WK == 1 || DS == 1, "");
  static_assert(DS == 1 || NT == 1, "one exchange per sub-block");
  using St = Stage<D, IT, BN, W::NTH>;
  constexpr int BUF = 2 * St::ELTS;  // K planes, then V planes
  constexpr int XCH = DS == 1 ? 0 : W::NTH * 32 * 2;  // S and dP halves
  constexpr int OUT = WK == 1 ? WQ * DS * put_bytes<DW>() : WK * RPW * D * 4;
  __shared__ __attribute__((aligned(16))) uint16_t L[cmax(NBUF * BUF + XCH, OUT / 2)];

  const int item = a.q_order[blockIdx.x / W::NSUB];
  if (item < 0 || item >= a.B * a.Hq * a.nqt) return;  // idle slot (or an entry out of range)
  const int qt = item % a.nqt, bh = item / a.nqt;
  const int h = bh % a.Hq, b = bh / a.Hq, hk = h / a.G;
  const int mrow = map_row(a, b, h, a.nqt, qt);
  const Walk<BN> walk(a.row_ent, a.row_ptr[mrow], a.row_ptr[mrow + 1]);
  const W w;
  const int wrow = (blockIdx.x % W::NSUB) * RPW;
  if (qt * TILE + wrow >= a.Lq) return;
  const int qloc = wrow + 32 * w.wq + w.l32;
  const int q = qt * TILE + qloc, qc = min(q, a.Lq - 1);

  const char* kb = head_base(a.k, a.ks, b, hk, elt_bytes<IT>());
  const char* vb = head_base(a.v, a.vs, b, hk, elt_bytes<IT>());
  St ks, vs;
  if (walk.n > 0) {
    ks.load(kb, a.ks[1], walk.first(0), a.Lk);
    vs.load(vb, a.vs[1], walk.first(0), a.Lk);
  }
  Frag<NP> qf[NKD];
  Frag<NG> gf[NKD];
  own_rows<IT>(qf, head_base(a.q, a.qs, b, h, elt_bytes<IT>()), a.qs[1], qc, w.ds * DW, w.hi);
  own_rows<OT>(gf, head_base(a.dO, a.dos, b, h, elt_bytes<OT>()), a.dos[1], qc, w.ds * DW, w.hi);
  const int64_t rs = ((int64_t)b * a.Hq + h) * a.Lq + qc;
  const float lse = a.lse[rs], delta = a.delta[rs], c2 = a.scale_log2;

  f32x16 acc[NMD];
#pragma unroll
  for (int i = 0; i < NMD; ++i) acc[i] = f32x16{};
  float* X = (float*)(L + NBUF * BUF);

  auto stage = [&](int s) {
    uint16_t* buf = L + (NBUF == 2 ? (s & 1) * BUF : 0);
    ks.store(buf);
    vs.store(buf + St::ELTS);
    if (s + 1 < walk.n) {
      ks.load(kb, a.ks[1], walk.first(s + 1), a.Lk);
      vs.load(vb, a.vs[1], walk.first(s + 1), a.Lk);
    }
  };
  auto compute = [&](int s) {
    const uint16_t* Kl = L + (NBUF == 2 ? (s & 1) * BUF : 0);
    const uint16_t* Vl = Kl + St::ELTS;
    const int mask = walk.mask(s), blk0 = (s % Walk<BN>::SPT) * (BN / 32) + w.wk * NT;
#pragma unroll
    for (int t = 0; t < NT; ++t) {
      uint32_t w32 = 0xffffffffu;
      if (mask >= 0) w32 = bits32(a.row_bits, mask, blk0 + t, qloc);
      const bool live = __any(w32 != 0);
      const int r0 = 32 * (w.wk * NT + t);
      f32x16 sd[2];  // S, dP
      if (live) {
        sd[0] = sd[1] = f32x16{};
#pragma unroll
        for (int kd = 0; kd < NKD; ++kd) {
          sd[0] = mma(row_frag<D, NP, BN>(Kl, r0 + w.l32, w.ds * NKD + kd, w.hi), qf[kd], sd[0]);
          sd[1] = mma(row_frag<D, NP, BN>(Vl, r0 + w.l32, w.ds * NKD + kd, w.hi), gf[kd], sd[1]);
        }
        if constexpr (DS == 2) half_put(sd, X, w.wave, w.lane);
      }
      if constexpr (DS == 2) __syncthreads();
      if (!live) continue;
      if constexpr (DS == 2) half_add(sd, X, w.partner(), w.lane);
#pragma unroll
      for (int r = 0; r < 16; ++r) {
        float p = fast_exp2(fmaf(sd[0][r], c2, -lse));
        if (mask >= 0) p = mask_zero(p, mask_ones(w32 >> (4 * w.hi), r));
        sd[1][r] = p * (sd[1][r] - delta);
      }
#pragma unroll
      for (int j = 0; j < 2; ++j) {
        const Frag<3> df = c_frag(sd[1], j);
#pragma unroll
        for (int mt = 0; mt < NMD; ++mt)
          acc[mt] = mma(tr_frag<D, NP, BN>(Kl, r0 + 16 * j, w.ds * NMD + mt, w.lane), df, acc[mt]);
      }
    }
  };
  run_walk<NBUF>(walk.n, stage, compute);

  const int nrows = a.Lq - (qt * TILE + wrow);
  const int64_t orow = (int64_t)b * a.dqs[0] + (int64_t)(qt * TILE + wrow) * a.dqs[1] + (int64_t)h * a.dqs[2];
  __syncthreads();
  if constexpr (WK == 1) {
    put_rows<DW, IT>(acc, a.scale, (char*)L + w.wave * put_bytes<DW>(), a.dq,
                     orow + (int64_t)32 * w.wq * a.dqs[1] + w.ds * DW, a.dqs[1], nrows - 32 * w.wq, w.lane);
  } else {
    slab_put<D, WQ>(acc, a.scale, (float*)L, w.wq, w.wk, w.lane);
    __syncthreads();
    slab_sum_store<D, IT, WQ, WK, W::NTH>((const float*)L, a.dq, orow, a.dqs[1], nrows);
  }
}

// PART: 1 = dV, 2 = dK, 3 = both in one workgroup.  At D = 256 the two run in
// workgroups of their own (S is then formed twice, 1/14 of the products): both
// accumulators would take half of a wave's registers.
template <int D, class IT, class OT, int PART, int WQ, int WK, int DS, int NBUF>
__device__ __forceinline__ void dkdv_s3(const KArgs& a, uint16_t* L, float* Rl, int slot, int sub) {
  using W = Place<WQ, WK, DS>;
  constexpr int NP = Pieces<IT>::n, NG = Pieces<OT>::n, DW = D / DS, NKD = DW / 16, NMD = DW / 32;
  constexpr int RPW = 32 * WQ, BN = 32 * WK;  // BN: queries per sub-block
  constexpr bool DV = PART & 1, DK = PART & 2;
  static_assert(WK == 1 || DS == 1, "");
  using Sq = Stage<D, IT, BN, W::NTH>;
  using Sg = Stage<D, OT, BN, W::NTH>;
  constexpr int BUF = Sq::ELTS + Sg::ELTS;

  const int item = a.kv_order[slot];
  if (item < 0 || item >= a.B * a.Hkv * a.nkt) return;  // idle slot (or an entry out of range)
  const int kt = item % a.nkt, bh = item / a.nkt;
  const int hk = bh % a.Hkv, b = bh / a.Hkv;
  const W w;
  const int wrow = sub * RPW;
  if (kt * TILE + wrow >= a.Lk) return;
  const int kloc = wrow + 32 * w.wq + w.l32;
  const int kc = min(kt * TILE + kloc, a.Lk - 1);
  const float c2 = a.scale_log2;
  float* X = (float*)(L + NBUF * BUF);

  Frag<NP> kf[NKD], vf[DK ? NKD : 1];
  own_rows<IT>(kf, head_base(a.k, a.ks, b, hk, elt_bytes<IT>()), a.ks[1], kc, w.ds * DW, w.hi);
  if constexpr (DK) own_rows<IT>(vf, head_base(a.v, a.vs, b, hk, elt_bytes<IT>()), a.vs[1], kc, w.ds * DW, w.hi);
  f32x16 dk[DK ? NMD : 1], dv[DV ? NMD : 1];
#pragma unroll
  for (int i = 0; i < NMD; ++i) {
    if constexpr (DK) dk[i] = f32x16{};
    if constexpr (DV) dv[i] = f32x16{};
  }

  for (int g = 0; g < a.G; ++g) {
    const int h = hk * a.G + g;
    const int mc = map_row(a, b, h, a.nkt, kt);
    const Walk<BN> walk(a.col_ent, a.col_ptr[mc], a.col_ptr[mc + 1]);
    if (walk.n == 0) continue;
    const char* qb = head_base(a.q, a.qs, b, h, elt_bytes<IT>());
    const char* gb = head_base(a.dO, a.dos, b, h, elt_bytes<OT>());
    const int64_t rs = ((int64_t)b * a.Hq + h) * a.Lq;
    Sq sq;
    Sg sg;
    float rl = 0.f;  // lse (threads 0 .. BN - 1) or delta (the next BN) of a row
    auto load = [&](int s) {
      const int q0 = walk.first(s);
      sq.load(qb, a.qs[1], q0, a.Lq);
      sg.load(gb, a.dos[1], q0, a.Lq);
      if (threadIdx.x < 2 * BN) {
        const int64_t r = rs + min(q0 + (int)(threadIdx.x % BN), a.Lq - 1);
        rl = threadIdx.x < BN ? a.lse[r] : a.delta[r];
      }
    };
    auto stage = [&](int s) {
      uint16_t* buf = L + (NBUF == 2 ? (s & 1) * BUF : 0);
      sq.store(buf);
      sg.store(buf + Sq::ELTS);
      if (threadIdx.x < 2 * BN) Rl[(NBUF == 2 ? (s & 1) * 2 * BN : 0) + threadIdx.x] = rl;
      if (s + 1 < walk.n) load(s + 1);
    };
    auto compute = [&](int s) {
      const uint16_t* Ql = L + (NBUF == 2 ? (s & 1) * BUF : 0);
      const uint16_t* Gl = Ql + Sq::ELTS;
      const float* R = Rl + (NBUF == 2 ? (s & 1) * 2 * BN : 0) + 32 * w.wk + 4 * w.hi;
      const int mask = walk.mask(s), blk = (s % Walk<BN>::SPT) * WK + w.wk;
      uint32_t w32 = 0xffffffffu;
      if (mask >= 0) w32 = bits32(a.col_bits, mask, blk, kloc);
      const bool live = __any(w32 != 0);
      const int r0 = 32 * w.wk;
      f32x16 sd[DK ? 2 : 1];  // S, dP
      if (live) {
#pragma unroll
        for (int n = 0; n < (DK ? 2 : 1); ++n) sd[n] = f32x16{};
#pragma unroll
        for (int kd = 0; kd < NKD; ++kd) {
          sd[0] = mma(row_frag<D, NP, BN>(Ql, r0 + w.l32, w.ds * NKD + kd, w.hi), kf[kd], sd[0]);
          if constexpr (DK) sd[1] = mma(row_frag<D, NG, BN>(Gl, r0 + w.l32, w.ds * NKD + kd, w.hi), vf[kd], sd[1]);
        }
        if constexpr (DS == 2) half_put(sd, X, w.wave, w.lane);
      }
      if constexpr (DS == 2) __syncthreads();
      if (!live) return;
      if constexpr (DS == 2) half_add(sd, X, w.partner(), w.lane);
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        const f32x4 ls = *(const f32x4*)(R + 8 * j), dl = *(const f32x4*)(R + BN + 8 * j);
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          const int r = 4 * j + i;
          float p = fast_exp2(fmaf(sd[0][r], c2, -ls[i]));
          if (mask >= 0) p = mask_zero(p, mask_ones(w32 >> (4 * w.hi), r));
          sd[0][r] = p;
          if constexpr (DK) sd[1][r] = p * (sd[1][r] - dl[i]);
        }
      }
#pragma unroll
      for (int j = 0; j < 2; ++j) {
        if constexpr (DV) {
          const Frag<3> pf = c_frag(sd[0], j);
#pragma unroll
          for (int mt = 0; mt < NMD; ++mt)
            dv[mt] = mma(tr_frag<D, NG, BN>(Gl, r0 + 16 * j, w.ds * NMD + mt, w.lane), pf, dv[mt]);
        }
        if constexpr (DK) {
          const Frag<3> df = c_frag(sd[DK ? 1 : 0], j);
#pragma unroll
          for (int mt = 0; mt < NMD; ++mt)
            dk[mt] = mma(tr_frag<D, NP, BN>(Ql, r0 + 16 * j, w.ds * NMD + mt, w.lane), df, dk[mt]);
        }
      }
    };
    load(0);
    __syncthreads();  // the previous head's last sub-block is consumed
    run_walk<NBUF>(walk.n, stage, compute);
  }

  const int nrows = a.Lk - (kt * TILE + wrow);
  auto out = [&](const f32x16(&acc)[NMD], float sc, void* dst, const int64_t* st) {
    const int64_t row = (int64_t)b * st[0] + (int64_t)(kt * TILE + wrow) * st[1] + (int64_t)hk * st[2];
    __syncthreads();
    if constexpr (WK == 1) {
      put_rows<DW, IT>(acc, sc, (char*)L + w.wave * put_bytes<DW>(), dst,
                       row + (int64_t)32 * w.wq * st[1] + w.ds * DW, st[1], nrows - 32 * w.wq, w.lane);
    } else {
      slab_put<D, WQ>(acc, sc, (float*)L, w.wq, w.wk, w.lane);
      __syncthreads();
      slab_sum_store<D, IT, WQ, WK, W::NTH>((const float*)L, dst, row, st[1], nrows);
    }
  };
  if constexpr (DV) out(dv, 1.f, a.dv, a.dvs);
  if constexpr (DK) out(dk, a.scale, a.dk, a.dks);
}

template <int D, class IT, class OT, bool BOTH, int WQ, int WK, int DS, int NBUF, int MINW>
__global__ __attribute__((amdgpu_flat_work_group_size(64 * WQ * WK * DS, 64 * WQ * WK * DS), amdgpu_waves_per_eu(MINW, MINW)))
void bwd_dkdv_s3(KArgs a) {
  using W = Place<WQ, WK, DS>;
  constexpr int BN = 32 * WK;
  constexpr int BUF = Stage<D, IT, BN, W::NTH>::ELTS + Stage<D, OT, BN, W::NTH>::ELTS;
  constexpr int XCH = DS == 1 ? 0 : W::NTH * 32 * 2;
  constexpr int OUT = WK == 1 ? WQ * DS * put_bytes<D / DS>() : WK * 32 * WQ * D * 4;
  __shared__ __attribute__((aligned(16))) uint16_t L[cmax(NBUF * BUF + XCH, OUT / 2)];
  __shared__ __attribute__((aligned(16))) float Rl[NBUF * 2 * BN];
  if constexpr (BOTH) {
    dkdv_s3<D, IT, OT, 3, WQ, WK, DS, NBUF>(a, L, Rl, blockIdx.x / W::NSUB, blockIdx.x % W::NSUB);
  } else {
    const int slot = blockIdx.x / (2 * W::NSUB), sub = (blockIdx.x >> 1) % W::NSUB;
    if (blockIdx.x & 1) dkdv_s3<D, IT, OT, 1, WQ, WK, DS, NBUF>(a, L, Rl, slot, sub);
    else dkdv_s3<D, IT, OT, 2, WQ, WK, DS, NBUF>(a, L, Rl, slot, sub);
  }
}

// ---------------------------------------------------------------------------
// launchers
// ---------------------------------------------------------------------------

// <BN, WQ, WK, DS, NBUF, MINW> of the kernels per head dimension
template <int D, class IT, class OT>
struct S3 {
  static constexpr int N = Pieces<IT>::n;
  static void fwd(const KArgs& a, int grid, hipStream_t st) {
    if constexpr (D == 64) go<fwd_s3<D, IT, OT, 64, 4, 2, 1, 1, 2>, Place<4, 2, 1>>(a, grid, st);
    else if constexpr (D == 128) go<fwd_s3<D, IT, OT, 32, 4, 1, 2, 1, 2>, Place<4, 1, 2>>(a, grid, st);
    else go<fwd_s3<D, IT, OT, 32, 4, 1, 2, N == 1 ? 2 : 1, 2>, Place<4, 1, 2>>(a, grid, st);
  }
  static void bwd(const KArgs& a, int stage, int q_grid, int kv_grid, hipStream_t st) {
    if (stage == MATTN_BWD_PRE) {
      const int64_t threads = (int64_t)a.B * a.Hq * a.Lq * (D / 8);
      hipLaunchKernelGGL((delta_s3<D, OT>), dim3((threads + 255) / 256), dim3(256), 0, st, a);
    } else if (stage == MATTN_BWD_DKDV) {
      if constexpr (D == 64) go<bwd_dkdv_s3<D, IT, OT, true, 4, 2, 1, 1, 2>, Place<4, 2, 1>>(a, kv_grid, st);
      else if constexpr (D == 128) go<bwd_dkdv_s3<D, IT, OT, true, 4, 1, 2, 1, 2>, Place<4, 1, 2>>(a, kv_grid, st);
      else if constexpr (N == 1) go<bwd_dkdv_s3<D, IT, OT, false, 4, 1, 2, 1, 2>, Place<4, 1, 2>>(a, 2 * kv_grid, st);
      else go<bwd_dkdv_s3<D, IT, OT, false, 2, 1, 2, 1, 1>, Place<2, 1, 2>>(a, 2 * kv_grid, st);
    } else {
      if constexpr (D == 64) go<bwd_dq_s3<D, IT, OT, 64, 4, 2, 1, 1, 2>, Place<4, 2, 1>>(a, q_grid, st);
      else if constexpr (D == 128) go<bwd_dq_s3<D, IT, OT, 32, 4, 1, 2, 1, 2>, Place<4, 1, 2>>(a, q_grid, st);
      else if constexpr (N == 1) go<bwd_dq_s3<D, IT, OT, 32, 4, 1, 2, 1, 2>, Place<4, 1, 2>>(a, q_grid, st);
      else go<bwd_dq_s3<D, IT, OT, 32, 2, 1, 2, 1, 1>, Place<2, 1, 2>>(a, q_grid, st);
    }
  }
  template <void (*K)(KArgs), class W>
  static void go(const KArgs& a, int grid, hipStream_t st) {
    hipLaunchKernelGGL(K, dim3(grid * W::NSUB), dim3(W::NTH), 0, st, a);
  }
};

template <class F>
hipError_t dispatch(int D, int dtype, int o_dtype, F&& f) {
  const bool of32 = o_dtype == MATTN_F32;
  if (dtype == MATTN_F32) {
    if (D == 64) f(S3<64, float, float>{});
    else if (D == 128) f(S3<128, float, float>{});
    else f(S3<256, float, float>{});
  } else if (dtype == MATTN_BF16) {
    if (of32) f(S3<256, bf16_tag, float>{}); else f(S3<256, bf16_tag, bf16_tag>{});
  } else {
    if (of32) f(S3<256, f16_tag, float>{}); else f(S3<256, f16_tag, f16_tag>{});
  }
  return hipGetLastError();
}

}  // namespace

bool s3_path(int D, int dtype, bool precise) {
  return !precise && (dtype == MATTN_F32 ? D <= 256 : D == 256);
}

hipError_t launch_fwd_s3(const KArgs& a, int D, int dtype, int o_dtype, int grid, hipStream_t st) {
  return dispatch(D, dtype, o_dtype, [&](auto s) { decltype(s)::fwd(a, grid, st); });
}

hipError_t launch_bwd_s3(const KArgs& a, int D, int dtype, int o_dtype, int stage, int q_grid, int kv_grid,
                         hipStream_t st) {
  return dispatch(D, dtype, o_dtype, [&](auto s) { decltype(s)::bwd(a, stage, q_grid, kv_grid, st); });
}

}  // namespace mattn
