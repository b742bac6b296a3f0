// MATTN_PRECISE on the float64 matrix cores, D = 64, 128 and 256 (D = 512: the SIMT
// kernels of simt.hip): for kernels sharper than 1/sqrt(d), whose scores reach tens
// of units and whose rows concentrate on single keys.
//
// Every product and sum is float64 (v_mfma_f64_16x16x4_f64; the inputs convert
// exactly): the scores, which float32's rounding would carry into the weights; O and
// the row sums; and dP - delta, which is a small difference of two large dot products
// where one key dominates a row.  Weights and dS are formed in float32 from float64
// arguments.  lse and O are kept as stored value + remainder (lse_lo, o_lo: the
// residual), so the backward sees both to float64; delta = dO . (O + o_lo) is formed
// where it is used (the workspace holds no float64 value per row).
//
// Bound by the float64 matrix cores: 64 cycles per 16x16x4 product, 128 flop a clock
// and CU: the rate of the vector float64 FMA, but with the operands of 16 FMAs in one
// register.  Measured against the compensated SIMT kernels, causal steps at scale 1:
// [1, 2048, 8, 64] 4.95 -> 0.47 ms, [1, 2048, 8, 128] 10.5 -> 0.91 ms, [1, 1024, 8,
// 256] 7.06 -> 1.09 ms (the backward spills 58 to 76 of its 512 registers there).
//
// MFMA 16x16x4 layout (lane l, l16 = l % 16, g = l / 16): A row l16, k = g; B column
// l16, k = g; C column l16, register i row 4 i + g.  Operands along d are read as 4
// consecutive floats, columns 16 j + 4 g + e, so product e of step j takes the
// columns 16 j + 4 g + e of both sides; C register i is the B operand of the product
// over rows 4 i + g as it stands.
//
// A workgroup is WQ x 2 waves: WQ groups of 16 own rows (lane = row), the two waves of
// a group taking halves of every streamed sub-block and summing their float64 results
// through LDS at the end.
#include <type_traits>

#include "split3.hpp"

namespace mattn {
namespace {
using namespace s3;

typedef double f64x4 __attribute__((ext_vector_type(4)));

__device__ __forceinline__ f64x4 mfma64(double a, double b, f64x4 c) {
  return __builtin_amdgcn_mfma_f64_16x16x4f64(a, b, c, 0, 0, 0);
}

// Sub-blocks of the walk over entries [e0, e1), SPT per tile.  The entry is read at each
// step: a step has thousands of cycles of matrix work (held in lanes, as split3.hpp's
// Walk does, the step ran 1.3% slower).
template <int BN>
struct Steps {
  static constexpr int SPT = TILE / BN;
  const int* ent;
  int e0, n;
  __device__ __forceinline__ Steps(const int* ent_, int e0_, int e1_) : ent(ent_), e0(e0_), n((e1_ - e0_) * SPT) {}
  __device__ __forceinline__ int first(int s) const { return ent[2 * (e0 + s / SPT)] * TILE + (s % SPT) * BN; }
  __device__ __forceinline__ int mask(int s) const { return ent[2 * (e0 + s / SPT) + 1]; }
};

// N consecutive elements (N = 4 or 8) as floats
template <class T, int N>
__device__ __forceinline__ void get(const char* p, float* x) {
#pragma unroll
  for (int c = 0; c < N; c += 4) {
    if constexpr (std::is_same<T, float>::value) {
      const f32x4 y = *(const f32x4*)(p + 4 * c);
#pragma unroll
      for (int i = 0; i < 4; ++i) x[c + i] = y[i];
    } else {
      const u32x2 y = *(const u32x2*)(p + 2 * c);
#pragma unroll
      for (int i = 0; i < 4; ++i) x[c + i] = Elt<T>::to_f32((y[i >> 1] >> (16 * (i & 1))) & 0xffffu);
    }
  }
}

constexpr int WK = 2;
// workgroups a CU holds (launch_slot): by registers (224 to 256 a wave in dK/dV at D =
// 64 and the others at 128, twice that beyond), at D = 256 by LDS
template <int D, bool KV>
constexpr int resident() { return D == 64 ? (KV ? 2 : 3) : D == 128 && !KV ? 2 : 1; }
template <int D>
constexpr int ld() { return D + 4; }  // LDS row stride in floats: 16-byte reads of 16 rows hit 16 bank groups

// ROWS rows of a tensor as float32 rows in LDS (rows past n - 1 re-read row n - 1),
// through registers: loaded one step ahead where they are few (HELD)
template <int D, class T, int ROWS, int NTH>
struct Rows32 {
  static constexpr int CH = ROWS * D / 8 / NTH;
  static constexpr bool HELD = D == 64;
  Raw8<T> v[CH];
  __device__ __forceinline__ void load(const char* base, int64_t rs, int r0, int n) {
    constexpr int ES = elt_bytes<T>();
    each_chunk<D, ES, ROWS, NTH, false>(base, rs, r0, n, [&](int c, const char* p, uint32_t off) {
      v[c].load(p + (off + ES * 8 * (threadIdx.x % (D / 8))));
    });
  }
  __device__ __forceinline__ void store(float* dst) const {
#pragma unroll
    for (int c = 0; c < CH; ++c) {
      const int i = threadIdx.x + NTH * c, r = i / (D / 8), col = 8 * (i % (D / 8));
      float x[8];
      v[c].floats(x);
      *(f32x4*)(dst + r * ld<D>() + col) = f32x4{x[0], x[1], x[2], x[3]};
      *(f32x4*)(dst + r * ld<D>() + col + 4) = f32x4{x[4], x[5], x[6], x[7]};
    }
  }
};

// this lane's D / 4 values of row r: x[4 j + e] = column 16 j + 4 g + e
template <int D, class T>
__device__ __forceinline__ void own(float (&x)[D / 4], const char* base, int64_t rs, int r, int g) {
#pragma unroll
  for (int j = 0; j < D / 16; ++j) get<T, 4>(base + elt_bytes<T>() * ((int64_t)r * rs + 16 * j + 4 * g), x + 4 * j);
}

// the four 16-lane groups' values, combined
__device__ __forceinline__ double group_sum(double x) {
  x += __shfl_xor(x, 16);
  return x + __shfl_xor(x, 32);
}
__device__ __forceinline__ float group_max(float x) {
  x = fmaxf(x, __shfl_xor(x, 16));
  return fmaxf(x, __shfl_xor(x, 32));
}

// c += (rows of A at `row`, row stride ld) . own row, over d
template <int D>
__device__ __forceinline__ f64x4 dot_rows(const float* row, const float (&x)[D / 4], int g, f64x4 c) {
#pragma unroll
  for (int j = 0; j < D / 16; ++j) {
    const f32x4 y = *(const f32x4*)(row + 16 * j + 4 * g);
#pragma unroll
    for (int e = 0; e < 4; ++e) c = mfma64((double)y[e], (double)x[4 * j + e], c);
  }
  return c;
}

// acc[mt] (columns 16 mt .. of the own row) += sum over the 16 rows at `rows` of w[i] row[4 i + g]
template <int D>
__device__ __forceinline__ void add_rows(f64x4 (&acc)[D / 16], const float* rows, const float (&w)[4], int l16, int g) {
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const double b = (double)w[i];
#pragma unroll
    for (int mt = 0; mt < D / 16; ++mt)
      acc[mt] = mfma64((double)rows[(4 * i + g) * ld<D>() + 16 * mt + l16], b, acc[mt]);
  }
}

// The float64 results of the two waves of each row group, summed through LDS
// (slab [2][16 WQ][D + 2]) and handed over row by row: f(row, column, value) for 2
// consecutive columns a thread.
template <int D, int WQ, class F>
__device__ __forceinline__ void sum_rows(const f64x4 (&acc)[D / 16], double sc, double* slab, int wq, int wk, int l16,
                                         int g, F&& f) {
  constexpr int NTH = 64 * WQ * WK, LDS = D + 2;
  __syncthreads();  // the operand tiles (or an earlier slab) are consumed
#pragma unroll
  for (int mt = 0; mt < D / 16; ++mt)
#pragma unroll
    for (int i = 0; i < 4; ++i) slab[(wk * 16 * WQ + 16 * wq + l16) * LDS + 16 * mt + 4 * i + g] = acc[mt][i] * sc;
  __syncthreads();
#pragma unroll
  for (int c = 0; c < 16 * WQ * D / 2 / NTH; ++c) {
    const int n = threadIdx.x + NTH * c, r = n / (D / 2), col = 2 * (n % (D / 2));
    const double* s = slab + r * LDS + col;
    f(r, col, s[0] + s[16 * WQ * LDS], s[1] + s[16 * WQ * LDS + 1]);
  }
}

// two values to a tensor of type T
template <class T>
__device__ __forceinline__ void put2(void* base, int64_t i, float x, float y) {
  if constexpr (std::is_same<T, float>::value) *(f32x2*)((float*)base + i) = f32x2{x, y};
  else *(uint32_t*)((uint16_t*)base + i) = Elt<T>::pack2(x, y);
}
template <class T>
__device__ __forceinline__ float stored(float x) {  // x as T keeps it
  if constexpr (std::is_same<T, float>::value) return x;
  else return Elt<T>::to_f32(Elt<T>::pack2(x, 0.f) & 0xffffu);
}

// the 16 mask bits of row `row` against the 16-row block `blk` (0 .. 7) of the other side
__device__ __forceinline__ uint32_t bits16(const uint64_t* bits, int mask, int blk, int row) {
  return (uint32_t)(bits[((int64_t)mask * 2 + (blk >> 2)) * TILE + row] >> (16 * (blk & 3))) & 0xffffu;
}

template <int D, class IT, class OT, int WQ, int NT, int MINW>
__global__ __attribute__((amdgpu_flat_work_group_size(64 * WQ * WK, 64 * WQ * WK), amdgpu_waves_per_eu(MINW)))
void fwd_f64(KArgs a) {
  constexpr int NTH = 64 * WQ * WK, BN = 16 * NT * WK, NSUB = TILE / (16 * WQ);
  constexpr int TILES = 2 * BN * ld<D>() * 4, SLAB = WK * 16 * WQ * (D + 2) * 8;
  __shared__ __attribute__((aligned(16))) char L[TILES > SLAB ? TILES : SLAB];
  __shared__ float Mm[WQ * WK][16];
  __shared__ double Ml[WQ * WK][16];
  float* Kl = (float*)L;
  float* Vl = Kl + BN * ld<D>();

  const Slot slot = launch_slot<NSUB, resident<D, false>()>(a);
  const int item = slot.ok ? a.q_order[slot.slot] : -1;
  if (item < 0 || item >= a.B * a.Hq * a.nqt) return;  // idle slot (or an entry out of range)
  const int qt = item % a.nqt, bh = item / a.nqt;
  const int h = bh % a.Hq, b = bh / a.Hq, hk = h / a.G;
  const int mrow = map_row(a, b, h, a.nqt, qt);
  const Steps<BN> walk(a.row_ent, a.row_ptr[mrow], a.row_ptr[mrow + 1]);
  const int wrow = slot.part * 16 * WQ;
  if (qt * TILE + wrow >= a.Lq) return;
  const int lane = threadIdx.x & 63, l16 = lane & 15, g = lane >> 4;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), wq = wave % WQ, wk = wave / WQ;
  const int qloc = wrow + 16 * wq + l16, q = qt * TILE + qloc;

  float qv[D / 4];
  own<D, IT>(qv, head_base(a.q, a.qs, b, h, elt_bytes<IT>()), a.qs[1], min(q, a.Lq - 1), g);
  const char* kb = head_base(a.k, a.ks, b, hk, elt_bytes<IT>());
  const char* vb = head_base(a.v, a.vs, b, hk, elt_bytes<IT>());
  f64x4 acc[D / 16];
#pragma unroll
  for (int i = 0; i < D / 16; ++i) acc[i] = f64x4{};
  float m = NEG_INF;
  double l = 0.;
  const double c2 = (double)a.scale_log2;

  using R = Rows32<D, IT, BN, NTH>;
  R ks, vs;
  auto load = [&](int k0) {
    ks.load(kb, a.ks[1], k0, a.Lk);
    vs.load(vb, a.vs[1], k0, a.Lk);
  };
  if (R::HELD && walk.n > 0) load(walk.first(0));
  for (int s = 0; s < walk.n; ++s) {
    const int key0 = walk.first(s), mask = walk.mask(s);
    __syncthreads();
    if constexpr (R::HELD) {
      ks.store(Kl);
      vs.store(Vl);
      if (s + 1 < walk.n) load(walk.first(s + 1));
    } else {
      ks.load(kb, a.ks[1], key0, a.Lk);
      ks.store(Kl);
      vs.load(vb, a.vs[1], key0, a.Lk);
      vs.store(Vl);
    }
    __syncthreads();
    uint32_t w[NT];
    bool any = false;
#pragma unroll
    for (int t = 0; t < NT; ++t) {
      w[t] = mask >= 0 ? bits16(a.row_bits, mask, (s % Steps<BN>::SPT) * (BN / 16) + wk * NT + t, qloc) : 0xffffu;
      any |= w[t] != 0;
    }
    if (!__any(any)) continue;
    f64x4 st[NT];
    float mx = NEG_INF;
#pragma unroll
    for (int t = 0; t < NT; ++t) {
      st[t] = dot_rows<D>(Kl + (16 * (wk * NT + t) + l16) * ld<D>(), qv, g, f64x4{});
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        st[t][i] *= c2;
        if ((w[t] >> (4 * i + g)) & 1u) mx = fmaxf(mx, (float)st[t][i]);
      }
    }
    mx = group_max(mx);
    if (__any(mx > m + 8.f)) {  // raised only by more than 2^8, as in the other kernels
      const float mn = fmaxf(m, mx);
      const double al = mn == NEG_INF ? 1. : (double)exp2f(m - mn);
      l *= al;
#pragma unroll
      for (int i = 0; i < D / 16; ++i) acc[i] *= al;
      m = mn;
    }
    const double mu = m == NEG_INF ? 0. : (double)m;
#pragma unroll
    for (int t = 0; t < NT; ++t) {
      float p[4];
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        p[i] = ((w[t] >> (4 * i + g)) & 1u) ? exp2f((float)(st[t][i] - mu)) : 0.f;
        l += (double)p[i];
      }
      add_rows<D>(acc, Vl + 16 * (wk * NT + t) * ld<D>(), p, l16, g);
    }
  }

  l = group_sum(l);
  if (g == 0) {
    Mm[wave][l16] = m;
    Ml[wave][l16] = l;
  }
  __syncthreads();
  float M = NEG_INF;
  double lt = 0.;
#pragma unroll
  for (int k = 0; k < WK; ++k) M = fmaxf(M, Mm[k * WQ + wq][l16]);
#pragma unroll
  for (int k = 0; k < WK; ++k) {
    const float mk = Mm[k * WQ + wq][l16];
    if (mk != NEG_INF) lt += Ml[k * WQ + wq][l16] * (double)exp2f(mk - M);
  }
  const double f = m != NEG_INF && lt > 0. ? (double)exp2f(m - M) / lt : 0.;
  const int64_t rs0 = ((int64_t)b * a.Hq + h) * a.Lq + qt * TILE + wrow;
  if (wk == 0 && g == 0 && q < a.Lq) {
    const double full = lt > 0. ? (double)M + log2(lt) : (double)NEG_INF;
    const float hi = (float)full;
    a.lse[rs0 + 16 * wq + l16] = hi;
    a.lse_lo[rs0 + 16 * wq + l16] = lt > 0. ? (float)(full - (double)hi) : 0.f;  // lse + lse_lo = m + log2 l
  }
  const int nrows = a.Lq - (qt * TILE + wrow);
  const int64_t o0 = (int64_t)b * a.os[0] + (int64_t)(qt * TILE + wrow) * a.os[1] + (int64_t)h * a.os[2];
  sum_rows<D, WQ>(acc, f, (double*)L, wq, wk, l16, g, [&](int r, int c, double x, double y) {
    if (r >= nrows) return;
    put2<OT>(a.out, o0 + (int64_t)r * a.os[1] + c, (float)x, (float)y);
    put2<float>(a.o_lo, (rs0 + r) * D + c, (float)(x - (double)stored<OT>((float)x)),
                (float)(y - (double)stored<OT>((float)y)));  // what the stored O leaves off
  });
}

template <int D, class IT, class OT, int WQ, int NT, int MINW>
__global__ __attribute__((amdgpu_flat_work_group_size(64 * WQ * WK, 64 * WQ * WK), amdgpu_waves_per_eu(MINW)))
void bwd_dq_f64(KArgs a) {
  constexpr int NTH = 64 * WQ * WK, BN = 16 * NT * WK, NSUB = TILE / (16 * WQ);
  constexpr int TILES = 2 * BN * ld<D>() * 4, SLAB = WK * 16 * WQ * (D + 2) * 8;
  __shared__ __attribute__((aligned(16))) char L[TILES > SLAB ? TILES : SLAB];
  float* Kl = (float*)L;
  float* Vl = Kl + BN * ld<D>();

  const Slot slot = launch_slot<NSUB, resident<D, false>()>(a);
  const int item = slot.ok ? a.q_order[slot.slot] : -1;
  if (item < 0 || item >= a.B * a.Hq * a.nqt) return;  // idle slot (or an entry out of range)
  const int qt = item % a.nqt, bh = item / a.nqt;
  const int h = bh % a.Hq, b = bh / a.Hq, hk = h / a.G;
  const int mrow = map_row(a, b, h, a.nqt, qt);
  const Steps<BN> walk(a.row_ent, a.row_ptr[mrow], a.row_ptr[mrow + 1]);
  const int wrow = slot.part * 16 * WQ;
  if (qt * TILE + wrow >= a.Lq) return;
  const int lane = threadIdx.x & 63, l16 = lane & 15, g = lane >> 4;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), wq = wave % WQ, wk = wave / WQ;
  const int qloc = wrow + 16 * wq + l16, qc = min(qt * TILE + qloc, a.Lq - 1);
  const int64_t rs = ((int64_t)b * a.Hq + h) * a.Lq + qc;

  float qv[D / 4], gv[D / 4];
  own<D, IT>(qv, head_base(a.q, a.qs, b, h, elt_bytes<IT>()), a.qs[1], qc, g);
  own<D, OT>(gv, head_base(a.dO, a.dos, b, h, elt_bytes<OT>()), a.dos[1], qc, g);
  double delta = 0.;
  {
    const char* ob = head_base(a.o, a.os, b, h, elt_bytes<OT>()) + elt_bytes<OT>() * (int64_t)qc * a.os[1];
#pragma unroll
    for (int j = 0; j < D / 16; ++j) {
      float o[4], lo[4];
      get<OT, 4>(ob + elt_bytes<OT>() * (16 * j + 4 * g), o);
      get<float, 4>((const char*)(a.o_lo + rs * D + 16 * j + 4 * g), lo);
#pragma unroll
      for (int e = 0; e < 4; ++e) delta += (double)gv[4 * j + e] * ((double)o[e] + (double)lo[e]);
    }
    delta = group_sum(delta);
  }
  const double lse = (double)a.lse[rs] + (double)a.lse_lo[rs], c2 = (double)a.scale_log2;
  const char* kb = head_base(a.k, a.ks, b, hk, elt_bytes<IT>());
  const char* vb = head_base(a.v, a.vs, b, hk, elt_bytes<IT>());
  f64x4 acc[D / 16];
#pragma unroll
  for (int i = 0; i < D / 16; ++i) acc[i] = f64x4{};

  using R = Rows32<D, IT, BN, NTH>;
  R ks, vs;
  auto load = [&](int k0) {
    ks.load(kb, a.ks[1], k0, a.Lk);
    vs.load(vb, a.vs[1], k0, a.Lk);
  };
  if (R::HELD && walk.n > 0) load(walk.first(0));
  for (int s = 0; s < walk.n; ++s) {
    const int key0 = walk.first(s), mask = walk.mask(s);
    __syncthreads();
    if constexpr (R::HELD) {
      ks.store(Kl);
      vs.store(Vl);
      if (s + 1 < walk.n) load(walk.first(s + 1));
    } else {
      ks.load(kb, a.ks[1], key0, a.Lk);
      ks.store(Kl);
      vs.load(vb, a.vs[1], key0, a.Lk);
      vs.store(Vl);
    }
    __syncthreads();
#pragma unroll
    for (int t = 0; t < NT; ++t) {
      const int r0 = 16 * (wk * NT + t);
      const uint32_t w =
          mask >= 0 ? bits16(a.row_bits, mask, (s % Steps<BN>::SPT) * (BN / 16) + wk * NT + t, qloc) : 0xffffu;
      if (!__any(w != 0)) continue;
      const f64x4 st = dot_rows<D>(Kl + (r0 + l16) * ld<D>(), qv, g, f64x4{});
      const f64x4 dp = dot_rows<D>(Vl + (r0 + l16) * ld<D>(), gv, g, f64x4{});
      float ds[4];
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const float p = ((w >> (4 * i + g)) & 1u) ? exp2f((float)(st[i] * c2 - lse)) : 0.f;
        ds[i] = (float)((double)p * (dp[i] - delta));
      }
      add_rows<D>(acc, Kl + r0 * ld<D>(), ds, l16, g);
    }
  }

  const int nrows = a.Lq - (qt * TILE + wrow);
  const int64_t o0 = (int64_t)b * a.dqs[0] + (int64_t)(qt * TILE + wrow) * a.dqs[1] + (int64_t)h * a.dqs[2];
  sum_rows<D, WQ>(acc, (double)a.scale, (double*)L, wq, wk, l16, g, [&](int r, int c, double x, double y) {
    if (r < nrows) put2<IT>(a.dq, o0 + (int64_t)r * a.dqs[1] + c, (float)x, (float)y);
  });
}

template <int D, class IT, class OT, int WQ, int NT, int MINW>
__global__ __attribute__((amdgpu_flat_work_group_size(64 * WQ * WK, 64 * WQ * WK), amdgpu_waves_per_eu(MINW)))
void bwd_dkdv_f64(KArgs a) {
  constexpr int NTH = 64 * WQ * WK, BN = 16 * NT * WK, NSUB = TILE / (16 * WQ);
  constexpr int TILES = 2 * BN * ld<D>() * 4, SLAB = WK * 16 * WQ * (D + 2) * 8;
  __shared__ __attribute__((aligned(16))) char L[TILES > SLAB ? TILES : SLAB];
  __shared__ double Ls[BN], Dl[BN];  // lse and delta of the sub-block's rows
  float* Ql = (float*)L;
  float* Gl = Ql + BN * ld<D>();

  const Slot slot = launch_slot<NSUB, resident<D, true>()>(a);
  const int item = slot.ok ? a.kv_order[slot.slot] : -1;
  if (item < 0 || item >= a.B * a.Hkv * a.nkt) return;  // idle slot (or an entry out of range)
  const int kt = item % a.nkt, bh = item / a.nkt;
  const int hk = bh % a.Hkv, b = bh / a.Hkv;
  const int wrow = slot.part * 16 * WQ;
  if (kt * TILE + wrow >= a.Lk) return;
  const int lane = threadIdx.x & 63, l16 = lane & 15, g = lane >> 4;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), wq = wave % WQ, wk = wave / WQ;
  const int kloc = wrow + 16 * wq + l16, kc = min(kt * TILE + kloc, a.Lk - 1);
  const double c2 = (double)a.scale_log2;

  float kv[D / 4], vv[D / 4];
  own<D, IT>(kv, head_base(a.k, a.ks, b, hk, elt_bytes<IT>()), a.ks[1], kc, g);
  own<D, IT>(vv, head_base(a.v, a.vs, b, hk, elt_bytes<IT>()), a.vs[1], kc, g);
  f64x4 dk[D / 16], dv[D / 16];
#pragma unroll
  for (int i = 0; i < D / 16; ++i) dk[i] = dv[i] = f64x4{};

  for (int gh = 0; gh < a.G; ++gh) {
    const int h = hk * a.G + gh;
    const int mc = map_row(a, b, h, a.nkt, kt);
    const Steps<BN> walk(a.col_ent, a.col_ptr[mc], a.col_ptr[mc + 1]);
    const char* qb = head_base(a.q, a.qs, b, h, elt_bytes<IT>());
    const char* gb = head_base(a.dO, a.dos, b, h, elt_bytes<OT>());
    const char* ob = head_base(a.o, a.os, b, h, elt_bytes<OT>());
    const int64_t rs0 = ((int64_t)b * a.Hq + h) * a.Lq;
    for (int s = 0; s < walk.n; ++s) {
      const int q0 = walk.first(s), mask = walk.mask(s);
      __syncthreads();
      {
        Rows32<D, IT, BN, NTH> qr;
        qr.load(qb, a.qs[1], q0, a.Lq);
        qr.store(Ql);
      }
      // dO rows, and delta = dO . (O + o_lo) by the D / 8 threads of a row
#pragma unroll
      for (int c = 0; c < BN * D / 8 / NTH; ++c) {
        const int i = threadIdx.x + NTH * c, r = i / (D / 8), col = 8 * (i % (D / 8));
        const int q = min(q0 + r, a.Lq - 1);
        float x[8], o[8], lo[8];
        get<OT, 8>(gb + elt_bytes<OT>() * ((int64_t)q * a.dos[1] + col), x);
        get<OT, 8>(ob + elt_bytes<OT>() * ((int64_t)q * a.os[1] + col), o);
        get<float, 8>((const char*)(a.o_lo + (rs0 + q) * D + col), lo);
        *(f32x4*)(Gl + r * ld<D>() + col) = f32x4{x[0], x[1], x[2], x[3]};
        *(f32x4*)(Gl + r * ld<D>() + col + 4) = f32x4{x[4], x[5], x[6], x[7]};
        double d = 0.;
#pragma unroll
        for (int e = 0; e < 8; ++e) d += (double)x[e] * ((double)o[e] + (double)lo[e]);
#pragma unroll
        for (int m = 1; m < D / 8; m <<= 1) d += __shfl_xor(d, m);
        if (col == 0) {
          Dl[r] = d;
          Ls[r] = (double)a.lse[rs0 + q] + (double)a.lse_lo[rs0 + q];
        }
      }
      __syncthreads();
#pragma unroll
      for (int t = 0; t < NT; ++t) {
        const int r0 = 16 * (wk * NT + t);
        const uint32_t w =
            mask >= 0 ? bits16(a.col_bits, mask, (s % Steps<BN>::SPT) * (BN / 16) + wk * NT + t, kloc) : 0xffffu;
        if (!__any(w != 0)) continue;
        const f64x4 st = dot_rows<D>(Ql + (r0 + l16) * ld<D>(), kv, g, f64x4{});
        const f64x4 dp = dot_rows<D>(Gl + (r0 + l16) * ld<D>(), vv, g, f64x4{});
        float p[4], ds[4];
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          p[i] = ((w >> (4 * i + g)) & 1u) ? exp2f((float)(st[i] * c2 - Ls[r0 + 4 * i + g])) : 0.f;
          ds[i] = (float)((double)p[i] * (dp[i] - Dl[r0 + 4 * i + g]));
        }
        add_rows<D>(dv, Gl + r0 * ld<D>(), p, l16, g);
        add_rows<D>(dk, Ql + r0 * ld<D>(), ds, l16, g);
      }
    }
  }

  const int nrows = a.Lk - (kt * TILE + wrow);
  const int64_t v0 = (int64_t)b * a.dvs[0] + (int64_t)(kt * TILE + wrow) * a.dvs[1] + (int64_t)hk * a.dvs[2];
  const int64_t k0 = (int64_t)b * a.dks[0] + (int64_t)(kt * TILE + wrow) * a.dks[1] + (int64_t)hk * a.dks[2];
  sum_rows<D, WQ>(dv, 1., (double*)L, wq, wk, l16, g, [&](int r, int c, double x, double y) {
    if (r < nrows) put2<IT>(a.dv, v0 + (int64_t)r * a.dvs[1] + c, (float)x, (float)y);
  });
  sum_rows<D, WQ>(dk, (double)a.scale, (double*)L, wq, wk, l16, g, [&](int r, int c, double x, double y) {
    if (r < nrows) put2<IT>(a.dk, k0 + (int64_t)r * a.dks[1] + c, (float)x, (float)y);
  });
}

// ---------------------------------------------------------------------------
// launchers
// ---------------------------------------------------------------------------

template <int D, class IT, class OT>
struct F64 {
  static constexpr int WQ = 2, NT = D == 256 ? 1 : 2, MINW = D == 64 ? 2 : 1, MINF = D <= 128 ? 2 : 1;
  static constexpr int NSUB = TILE / (16 * WQ), NTH = 64 * WQ * WK;
  static void fwd(const KArgs& a, int grid, hipStream_t st) {
    go<fwd_f64<D, IT, OT, WQ, NT, MINF>>(a, grid, st);
  }
  static void bwd(const KArgs& a, int stage, int q_grid, int kv_grid, hipStream_t st) {
    if (stage == MATTN_BWD_DKDV)
      go<bwd_dkdv_f64<D, IT, OT, WQ, 1, MINW>>(a, kv_grid, st);
    else if (stage == MATTN_BWD_DQ)
      go<bwd_dq_f64<D, IT, OT, WQ, NT, MINF>>(a, q_grid, st);
    // MATTN_BWD_PRE: nothing (delta is formed where it is used)
  }
  template <void (*K)(KArgs)>
  static void go(KArgs a, int grid, hipStream_t st) {
    a.n_slots = grid;
    hipLaunchKernelGGL(K, dim3((grid + 7) / 8 * 8 * NSUB), dim3(NTH), 0, st, a);
  }
};

template <class IT, class OT, class F>
void dispatch_d(int D, F&& f) {
  if (D == 64) f(F64<64, IT, OT>{});
  else if (D == 128) f(F64<128, IT, OT>{});
  else f(F64<256, IT, OT>{});
}
template <class F>
hipError_t dispatch(int D, int dtype, int o_dtype, F&& f) {
  const bool of32 = o_dtype == MATTN_F32;
  if (dtype == MATTN_F32) dispatch_d<float, float>(D, f);
  else if (dtype == MATTN_BF16 && of32) dispatch_d<bf16_tag, float>(D, f);
  else if (dtype == MATTN_BF16) dispatch_d<bf16_tag, bf16_tag>(D, f);
  else if (of32) dispatch_d<f16_tag, float>(D, f);
  else dispatch_d<f16_tag, f16_tag>(D, f);
  return hipGetLastError();
}

}  // namespace

hipError_t launch_fwd_f64(const KArgs& a, int D, int dtype, int o_dtype, int grid, hipStream_t st) {
  return dispatch(D, dtype, o_dtype, [&](auto s) { decltype(s)::fwd(a, grid, st); });
}

hipError_t launch_bwd_f64(const KArgs& a, int D, int dtype, int o_dtype, int stage, int q_grid, int kv_grid,
                          hipStream_t st) {
  return dispatch(D, dtype, o_dtype, [&](auto s) { decltype(s)::bwd(a, stage, q_grid, kv_grid, st); });
}

}  // namespace mattn
