// SIMT (no MFMA) masked-attention kernels: the forward and the three backward
// stages in float32 arithmetic for D = 512 (any d in (256, 512], zero-padded by the
// host), every input dtype, with and without MATTN_PRECISE.  The other problems of
// float32 accuracy run on the matrix cores: split3.hip and, under MATTN_PRECISE,
// precise.hip; launch_fwd_simt and launch_bwd_simt hand them over.
// Same maths and tile walk as the MFMA path (/root/reference/jaxmodules/
// attention.py:52-105 forward, :266-342 backward): per 32-key (or 32-query)
// sub-block an online softmax, P = exp2(scale_log2 S - lse) in the backward,
// dS = P (dP - delta), dQ = scale dS K, dK = scale dS^T Q, dV = P^T dO.
// dP - delta is formed as dO . (V_k - O) (delta = dO . O): where one key
// dominates a row, V_k - O is small and exact to float32 rounding, while
// dO . V_k and dO . O are two large dot products whose roundings (2^-24 of
// |dO| |V|) would be all that is left of their difference.
// 16 threads share a row (query or key), each holding 32 head dims; a workgroup
// of 512 threads owns 32 rows of a 128-row map tile, so a tile takes four.
#include <type_traits>

#include "common.hpp"

namespace mattn {
namespace {

// float element access to tensors of float32 or a 16-bit Tag
template <class T>
struct Mem {
  static __device__ __forceinline__ float get(const void* p, int64_t i) { return ((const float*)p)[i]; }
  // 4 consecutive values (i a multiple of 4: 16-byte aligned)
  static __device__ __forceinline__ void get4(const void* p, int64_t i, float* x) {
    const f32x4 y = *(const f32x4*)((const float*)p + i);
    x[0] = y[0]; x[1] = y[1]; x[2] = y[2]; x[3] = y[3];
  }
  static __device__ __forceinline__ void put(void* p, int64_t i, float x) { ((float*)p)[i] = x; }
};
template <class Tag>
struct Mem16 {
  using E = Elt<Tag>;
  static __device__ __forceinline__ float get(const void* p, int64_t i) {
    return E::to_f32(((const uint16_t*)p)[i]);
  }
  // 4 consecutive values (i a multiple of 4: 8-byte aligned)
  static __device__ __forceinline__ void get4(const void* p, int64_t i, float* x) {
    const u32x2 y = *(const u32x2*)((const uint16_t*)p + i);
    x[0] = E::to_f32(y[0] & 0xffffu); x[1] = E::to_f32(y[0] >> 16);
    x[2] = E::to_f32(y[1] & 0xffffu); x[3] = E::to_f32(y[1] >> 16);
  }
  static __device__ __forceinline__ void put(void* p, int64_t i, float x) {
    ((uint16_t*)p)[i] = (uint16_t)(E::pack2(x, 0.f) & 0xffffu);  // round to nearest even
  }
};
template <>
struct Mem<bf16_tag> : Mem16<bf16_tag> {};
template <>
struct Mem<f16_tag> : Mem16<f16_tag> {};

constexpr int D = 512, TPR = 16;  // head dimension, threads per row
constexpr int DP = D / TPR;       // head dims a thread
constexpr int RPW = 512 / TPR, SPLIT = TILE / RPW;  // rows a workgroup, workgroups a tile
// keys (forward, dQ) or queries (dK/dV) per sub-block: four [SB, D] float32 LDS tiles
// (the dK/dV kernel's Q, dO, O and O's low parts) must fit 160 KiB
constexpr int SB = 16;

// mask bits of sub-block sb (SB keys or queries) of a partial tile's 128-bit
// row (or column) at `row`, one bit per element (words [mask][64-half][row])
__device__ __forceinline__ uint32_t sub_bits(const uint64_t* bits, int mask, int sb, int row) {
  const int first = sb * SB;
  return (uint32_t)(bits[((int64_t)mask * 2 + (first >> 6)) * TILE + row] >> (first & 63));
}

// sum over the TPR lanes of a row (consecutive lanes)
__device__ __forceinline__ float row_sum(float x) {
#pragma unroll
  for (int o = 1; o < TPR; o <<= 1) x += __shfl_xor(x, o);
  return x;
}

// a + b = s + e exactly (Knuth's TwoSum)
__device__ __forceinline__ void two_sum(float a, float b, float& s, float& e) {
  s = a + b;
  const float z = s - a;
  e = (a - (s - z)) + (b - z);
}

// Score of a row pair, q . y over the TPR lanes of the row (DP elements each),
// as hi + lo.  With `comp` (MATTN_PRECISE) it is the compensated dot product
// Dot2 of Ogita, Rump and Oishi (SIAM J. Sci. Comput. 26(6), 2005): every
// product's rounding error (an FMA gives it exactly) and every addition's
// (TwoSum) are summed apart, so hi + lo carries the dot product to about twice
// float32's precision.  The scores of a kernel sharper than 1/sqrt(d) reach
// tens of units (base 2 after scaling), where float32's 2^-24 relative
// rounding alone moves the weights exp2(S - lse) by 1e-5; otherwise lo = 0.
__device__ __forceinline__ void score(const float* qv, const float* y, bool comp, float& hi, float& lo) {
  if (!comp) {
    float p = 0.f;
#pragma unroll
    for (int i = 0; i < DP; ++i) p = fmaf(qv[i], y[i], p);
    hi = row_sum(p);
    lo = 0.f;
    return;
  }
  float s = 0.f, c = 0.f;
#pragma unroll
  for (int i = 0; i < DP; ++i) {
    const float pr = qv[i] * y[i];
    const float ep = fmaf(qv[i], y[i], -pr);
    float e;
    two_sum(s, pr, s, e);
    c += ep + e;
  }
#pragma unroll
  for (int o = 1; o < TPR; o <<= 1) {
    const float so = __shfl_xor(s, o), co = __shfl_xor(c, o);
    float e;
    two_sum(s, so, s, e);
    c += co + e;
  }
  hi = s;
  lo = c;
}

// rows [r0, r0 + SB) of a [rows, D] tensor slice (row stride rs) as floats in
// LDS; rows past n - 1 re-read row n - 1 (their scores are masked)
template <class T>
__device__ __forceinline__ void stage_rows(float* dst, const void* base, int64_t rs, int r0, int n) {
  for (int c = threadIdx.x; c < SB * D / 4; c += 512) {
    const int r = c / (D / 4), col = 4 * (c % (D / 4));
    Mem<T>::get4(base, (int64_t)min(r0 + r, n - 1) * rs + col, dst + r * D + col);
  }
}

// PREC (MATTN_PRECISE): compensated scores, O and the row sum accumulated in
// float64 (v_fma_f64 issues at the rate of the scalar float32 FMA on these
// CUs), and the residual keeps what the stored lse and O round off: the
// backward's dP - delta = dO . (V_k - O) then sees O to float64 accuracy,
// which a row dominated by one key needs (V_k - O is then a small fraction of
// |V|, and O's own float32 rounding a large part of it).
template <class IT, class OT, bool PREC>
__global__ __attribute__((amdgpu_flat_work_group_size(512, 512)))
void fwd_simt(KArgs a) {
  using acc_t = typename std::conditional<PREC, double, float>::type;
  constexpr int ES = std::is_same<IT, float>::value ? 4 : 2;
  __shared__ __attribute__((aligned(16))) float Ks[SB * D];
  __shared__ __attribute__((aligned(16))) float Vs[SB * D];

  const int item = a.q_order[blockIdx.x / SPLIT];
  if (item < 0 || item >= a.B * a.Hq * a.nqt) return;  // idle slot (or an entry out of range)
  const int qt = item % a.nqt;
  const int bh = item / a.nqt;
  const int h = bh % a.Hq, b = bh / a.Hq, hk = h / a.G;
  const int mrow = map_row(a, b, h, a.nqt, qt);
  const int e0 = a.row_ptr[mrow], e1 = a.row_ptr[mrow + 1];
  const int tid = threadIdx.x, part = tid % TPR;
  const int row = (blockIdx.x % SPLIT) * RPW + tid / TPR;  // row within the tile
  const int q = qt * TILE + row;
  const int qc = min(q, a.Lq - 1);

  float qv[DP];
  acc_t ov[DP];
  const int64_t qo = (int64_t)b * a.qs[0] + (int64_t)qc * a.qs[1] + (int64_t)h * a.qs[2] + part * DP;
#pragma unroll
  for (int i = 0; i < DP; i += 4) {
    Mem<IT>::get4(a.q, qo + i, qv + i);
    ov[i] = ov[i + 1] = ov[i + 2] = ov[i + 3] = 0;
  }
  const char* kb = (const char*)a.k + ES * ((int64_t)b * a.ks[0] + (int64_t)hk * a.ks[2]);
  const char* vb = (const char*)a.v + ES * ((int64_t)b * a.vs[0] + (int64_t)hk * a.vs[2]);
  float m = NEG_INF;
  acc_t l = 0;

  for (int e = e0; e < e1; ++e) {
    const int kt = a.row_ent[2 * e], mask = a.row_ent[2 * e + 1];
    for (int sb = 0; sb < TILE / SB; ++sb) {
      const int key0 = kt * TILE + sb * SB;
      if (key0 >= a.Lk) break;
      __syncthreads();
      stage_rows<IT>(Ks, kb, a.ks[1], key0, a.Lk);
      stage_rows<IT>(Vs, vb, a.vs[1], key0, a.Lk);
      __syncthreads();
      uint32_t bits = 0xffffffffu;
      if (mask >= 0)
        bits = sub_bits(a.row_bits, mask, sb, row);
      float sc[SB], sl[SB];  // scores s (scaled: s * scale_log2 = sc + sl)
      float mx = NEG_INF;
#pragma unroll
      for (int j = 0; j < SB; ++j) {
        float hi, lo;
        score(qv, Ks + j * D + part * DP, PREC, hi, lo);
        float x = hi * a.scale_log2;
        sl[j] = fmaf(hi, a.scale_log2, -x) + lo * a.scale_log2;  // rounding of x, and the low part
        if (!((bits >> j) & 1u)) x = NEG_INF;
        sc[j] = x;
        mx = fmaxf(mx, x);
      }
      const float mn = fmaxf(m, mx);
      const float mu = (mn == NEG_INF) ? 0.f : mn;
      const acc_t alpha = exp2f(m - mu);   // a power of two's neighbourhood: exact enough in float
      m = mn;
      l *= alpha;
#pragma unroll
      for (int i = 0; i < DP; ++i) ov[i] *= alpha;
#pragma unroll
      for (int j = 0; j < SB; ++j) {
        const acc_t p = exp2f((sc[j] - mu) + sl[j]);  // -inf + finite: 0 for masked keys
        l += p;
#pragma unroll
        for (int i = 0; i < DP; ++i) ov[i] = p * (acc_t)Vs[j * D + part * DP + i] + ov[i];
      }
    }
  }
  if (q >= a.Lq) return;
  const acc_t inv = l > 0 ? 1 / l : 0;
  const int64_t rs = ((int64_t)b * a.Hq + h) * a.Lq + q;
  if (part == 0) {
    float lse = NEG_INF, lo = 0.f;
    if (l > 0) {
      if constexpr (PREC) {
        const double full = (double)m + log2((double)l);
        lse = (float)full;
        lo = (float)(full - (double)lse);
      } else {
        two_sum(m, log2f(l), lse, lo);
      }
    }
    a.lse[rs] = lse;
    if constexpr (PREC) a.lse_lo[rs] = lo;  // lse + lse_lo = m + log2 l (to ~2^-48)
  }
  const int64_t oo = (int64_t)b * a.os[0] + (int64_t)q * a.os[1] + (int64_t)h * a.os[2] + part * DP;
#pragma unroll
  for (int i = 0; i < DP; ++i) {
    const acc_t o = ov[i] * inv;
    Mem<OT>::put(a.out, oo + i, (float)o);
    if constexpr (PREC)  // what the stored O (in OT) leaves off
      a.o_lo[rs * D + part * DP + i] = (float)(o - (acc_t)Mem<OT>::get(a.out, oo + i));
  }
}

template <class IT, class OT, bool PREC>
__global__ __attribute__((amdgpu_flat_work_group_size(512, 512)))
void bwd_dq_simt(KArgs a) {
  constexpr int ES = std::is_same<IT, float>::value ? 4 : 2;
  __shared__ __attribute__((aligned(16))) float Ks[SB * D];
  __shared__ __attribute__((aligned(16))) float Vs[SB * D];

  const int item = a.q_order[blockIdx.x / SPLIT];
  if (item < 0 || item >= a.B * a.Hq * a.nqt) return;  // idle slot (or an entry out of range)
  const int qt = item % a.nqt;
  const int bh = item / a.nqt;
  const int h = bh % a.Hq, b = bh / a.Hq, hk = h / a.G;
  const int mrow = map_row(a, b, h, a.nqt, qt);
  const int e0 = a.row_ptr[mrow], e1 = a.row_ptr[mrow + 1];
  const int tid = threadIdx.x, part = tid % TPR;
  const int row = (blockIdx.x % SPLIT) * RPW + tid / TPR;
  const int q = qt * TILE + row;
  const int qc = min(q, a.Lq - 1);

  float qv[DP], gv[DP], ov[DP], ol[DP], dq[DP];
  const int64_t qo = (int64_t)b * a.qs[0] + (int64_t)qc * a.qs[1] + (int64_t)h * a.qs[2] + part * DP;
  const int64_t go = (int64_t)b * a.dos[0] + (int64_t)qc * a.dos[1] + (int64_t)h * a.dos[2] + part * DP;
  const int64_t oo = (int64_t)b * a.os[0] + (int64_t)qc * a.os[1] + (int64_t)h * a.os[2] + part * DP;
  const int64_t rs = ((int64_t)b * a.Hq + h) * a.Lq + qc;
#pragma unroll
  for (int i = 0; i < DP; i += 4) {
    Mem<IT>::get4(a.q, qo + i, qv + i);
    Mem<OT>::get4(a.dO, go + i, gv + i);
    Mem<OT>::get4(a.o, oo + i, ov + i);
    if constexpr (PREC) Mem<float>::get4(a.o_lo, rs * D + part * DP + i, ol + i);
    else ol[i] = ol[i + 1] = ol[i + 2] = ol[i + 3] = 0.f;
    dq[i] = dq[i + 1] = dq[i + 2] = dq[i + 3] = 0.f;
  }
  const float lse = a.lse[rs], lse_lo = PREC ? a.lse_lo[rs] : 0.f;
  const char* kb = (const char*)a.k + ES * ((int64_t)b * a.ks[0] + (int64_t)hk * a.ks[2]);
  const char* vb = (const char*)a.v + ES * ((int64_t)b * a.vs[0] + (int64_t)hk * a.vs[2]);

  for (int e = e0; e < e1; ++e) {
    const int kt = a.row_ent[2 * e], mask = a.row_ent[2 * e + 1];
    for (int sb = 0; sb < TILE / SB; ++sb) {
      const int key0 = kt * TILE + sb * SB;
      if (key0 >= a.Lk) break;
      __syncthreads();
      stage_rows<IT>(Ks, kb, a.ks[1], key0, a.Lk);
      stage_rows<IT>(Vs, vb, a.vs[1], key0, a.Lk);
      __syncthreads();
      uint32_t bits = 0xffffffffu;
      if (mask >= 0)
        bits = sub_bits(a.row_bits, mask, sb, row);
      for (int j = 0; j < SB; ++j) {
        float g = 0.f;
#pragma unroll
        for (int i = 0; i < DP; ++i) g = fmaf(gv[i], (Vs[j * D + part * DP + i] - ov[i]) - ol[i], g);  // dP - delta
        g = row_sum(g);
        float hi, lo;
        score(qv, Ks + j * D + part * DP, PREC, hi, lo);
        float p = exp2f(fmaf(hi, a.scale_log2, -lse) + fmaf(lo, a.scale_log2, -lse_lo));
        if (!((bits >> j) & 1u)) p = 0.f;
        const float ds = p * g;
#pragma unroll
        for (int i = 0; i < DP; ++i) dq[i] = fmaf(ds, Ks[j * D + part * DP + i], dq[i]);
      }
    }
  }
  if (q >= a.Lq) return;
  const int64_t qo2 = (int64_t)b * a.dqs[0] + (int64_t)q * a.dqs[1] + (int64_t)h * a.dqs[2] + part * DP;
#pragma unroll
  for (int i = 0; i < DP; ++i) Mem<IT>::put(a.dq, qo2 + i, dq[i] * a.scale);
}

template <class IT, class OT, bool PREC>
__global__ __attribute__((amdgpu_flat_work_group_size(512, 512)))
void bwd_dkdv_simt(KArgs a) {
  constexpr int ES = std::is_same<IT, float>::value ? 4 : 2;
  constexpr int EO = std::is_same<OT, float>::value ? 4 : 2;
  __shared__ __attribute__((aligned(16))) float Qs[SB * D];
  __shared__ __attribute__((aligned(16))) float Gs[SB * D];
  __shared__ __attribute__((aligned(16))) float Os[SB * D];
  __shared__ __attribute__((aligned(16))) float Ol[PREC ? SB * D : 4];   // O's low parts (PREC)
  __shared__ float Ls[SB], Llo[SB];

  const int item = a.kv_order[blockIdx.x / SPLIT];
  if (item < 0 || item >= a.B * a.Hkv * a.nkt) return;  // idle slot (or an entry out of range)
  const int kt = item % a.nkt;
  const int bh = item / a.nkt;
  const int hk = bh % a.Hkv, b = bh / a.Hkv;
  const int tid = threadIdx.x, part = tid % TPR;
  const int row = (blockIdx.x % SPLIT) * RPW + tid / TPR;  // key within the tile
  const int key = kt * TILE + row;
  const int kcl = min(key, a.Lk - 1);

  float kv[DP], vv[DP], dk[DP], dv[DP];
  const int64_t ko = (int64_t)b * a.ks[0] + (int64_t)kcl * a.ks[1] + (int64_t)hk * a.ks[2] + part * DP;
  const int64_t vo = (int64_t)b * a.vs[0] + (int64_t)kcl * a.vs[1] + (int64_t)hk * a.vs[2] + part * DP;
#pragma unroll
  for (int i = 0; i < DP; i += 4) {
    Mem<IT>::get4(a.k, ko + i, kv + i);
    Mem<IT>::get4(a.v, vo + i, vv + i);
#pragma unroll
    for (int j = 0; j < 4; ++j) dk[i + j] = dv[i + j] = 0.f;
  }
  for (int g = 0; g < a.G; ++g) {
    const int h = hk * a.G + g;
    const int mc = map_row(a, b, h, a.nkt, kt);
    const int e0 = a.col_ptr[mc], e1 = a.col_ptr[mc + 1];
    const char* qb = (const char*)a.q + ES * ((int64_t)b * a.qs[0] + (int64_t)h * a.qs[2]);
    const char* gb = (const char*)a.dO + EO * ((int64_t)b * a.dos[0] + (int64_t)h * a.dos[2]);
    const char* ob = (const char*)a.o + EO * ((int64_t)b * a.os[0] + (int64_t)h * a.os[2]);
    for (int e = e0; e < e1; ++e) {
      const int qt = a.col_ent[2 * e], mask = a.col_ent[2 * e + 1];
      for (int sb = 0; sb < TILE / SB; ++sb) {
        const int q0 = qt * TILE + sb * SB;
        if (q0 >= a.Lq) break;
        __syncthreads();
        stage_rows<IT>(Qs, qb, a.qs[1], q0, a.Lq);
        stage_rows<OT>(Gs, gb, a.dos[1], q0, a.Lq);
        stage_rows<OT>(Os, ob, a.os[1], q0, a.Lq);
        if constexpr (PREC) stage_rows<float>(Ol, a.o_lo + ((int64_t)b * a.Hq + h) * a.Lq * D, D, q0, a.Lq);
        if (tid < SB) {
          const int64_t rs = ((int64_t)b * a.Hq + h) * a.Lq + min(q0 + tid, a.Lq - 1);
          Ls[tid] = a.lse[rs];
          Llo[tid] = PREC ? a.lse_lo[rs] : 0.f;
        }
        __syncthreads();
        uint32_t bits = 0xffffffffu;
        if (mask >= 0)
          bits = sub_bits(a.col_bits, mask, sb, row);
        for (int j = 0; j < SB; ++j) {
          float gd = 0.f;
#pragma unroll
          for (int i = 0; i < DP; ++i) {
            float dvo = vv[i] - Os[j * D + part * DP + i];  // V_k - O, then O's low part
            if constexpr (PREC) dvo -= Ol[j * D + part * DP + i];
            gd = fmaf(dvo, Gs[j * D + part * DP + i], gd);  // dP - delta
          }
          gd = row_sum(gd);
          float hi, lo;
          score(kv, Qs + j * D + part * DP, PREC, hi, lo);
          float p = exp2f(fmaf(hi, a.scale_log2, -Ls[j]) + fmaf(lo, a.scale_log2, -Llo[j]));
          if (!((bits >> j) & 1u)) p = 0.f;
          const float ds = p * gd;
#pragma unroll
          for (int i = 0; i < DP; ++i) {
            dv[i] = fmaf(p, Gs[j * D + part * DP + i], dv[i]);
            dk[i] = fmaf(ds, Qs[j * D + part * DP + i], dk[i]);
          }
        }
      }
    }
  }
  if (key >= a.Lk) return;
  const int64_t dko = (int64_t)b * a.dks[0] + (int64_t)key * a.dks[1] + (int64_t)hk * a.dks[2] + part * DP;
  const int64_t dvo = (int64_t)b * a.dvs[0] + (int64_t)key * a.dvs[1] + (int64_t)hk * a.dvs[2] + part * DP;
#pragma unroll
  for (int i = 0; i < DP; ++i) {
    Mem<IT>::put(a.dk, dko + i, dk[i] * a.scale);
    Mem<IT>::put(a.dv, dvo + i, dv[i]);
  }
}

// the stages of one (input, output) combination
template <class IT, class OT>
struct Simt {
  template <bool PREC>
  static void fwd(const KArgs& a, int grid, hipStream_t st) {
    hipLaunchKernelGGL((fwd_simt<IT, OT, PREC>), dim3(grid * SPLIT), dim3(512), 0, st, a);
  }
  template <bool PREC>
  static void bwd(const KArgs& a, int stage, int q_grid, int kv_grid, hipStream_t st) {
    if (stage == MATTN_BWD_DKDV)
      hipLaunchKernelGGL((bwd_dkdv_simt<IT, OT, PREC>), dim3(kv_grid * SPLIT), dim3(512), 0, st, a);
    else if (stage == MATTN_BWD_DQ)
      hipLaunchKernelGGL((bwd_dq_simt<IT, OT, PREC>), dim3(q_grid * SPLIT), dim3(512), 0, st, a);
    // MATTN_BWD_PRE: nothing, these kernels form dP - delta per pair from O
  }
};

// f(Simt<...>{}, precise) for the problem's combination: float32 inputs, or 16-bit
// inputs with a float32 or same-dtype output
template <class IT, class OT, class F>
void dispatch_p(bool precise, F&& f) {
  if (precise) f(Simt<IT, OT>{}, std::true_type{});
  else f(Simt<IT, OT>{}, std::false_type{});
}
template <class F>
hipError_t dispatch(int dtype, int o_dtype, bool precise, F&& f) {
  const bool of32 = o_dtype == MATTN_F32;
  if (dtype == MATTN_F32) dispatch_p<float, float>(precise, f);
  else if (dtype == MATTN_BF16 && of32) dispatch_p<bf16_tag, float>(precise, f);
  else if (dtype == MATTN_BF16) dispatch_p<bf16_tag, bf16_tag>(precise, f);
  else if (of32) dispatch_p<f16_tag, float>(precise, f);
  else dispatch_p<f16_tag, f16_tag>(precise, f);
  return hipGetLastError();
}

}  // namespace

bool s3_path(int D, int dtype, bool precise);
hipError_t launch_fwd_f64(const KArgs& a, int D, int dtype, int o_dtype, int grid, hipStream_t st);
hipError_t launch_bwd_f64(const KArgs& a, int D, int dtype, int o_dtype, int stage, int q_grid, int kv_grid,
                          hipStream_t st);
hipError_t launch_fwd_s3(const KArgs& a, int D, int dtype, int o_dtype, int grid, hipStream_t st);
hipError_t launch_bwd_s3(const KArgs& a, int D, int dtype, int o_dtype, int stage, int q_grid, int kv_grid,
                         hipStream_t st);

hipError_t launch_fwd_simt(const KArgs& a, int D, int dtype, int o_dtype, int grid, hipStream_t st) {
  if (s3_path(D, dtype, a.precise)) return launch_fwd_s3(a, D, dtype, o_dtype, grid, st);
  if (D <= 256) return launch_fwd_f64(a, D, dtype, o_dtype, grid, st);
  return dispatch(dtype, o_dtype, a.precise,
                  [&](auto s, auto p) { decltype(s)::template fwd<decltype(p)::value>(a, grid, st); });
}

hipError_t launch_bwd_simt(const KArgs& a, int D, int dtype, int o_dtype, int stage, int q_grid, int kv_grid,
                           hipStream_t st) {
  if (s3_path(D, dtype, a.precise)) return launch_bwd_s3(a, D, dtype, o_dtype, stage, q_grid, kv_grid, st);
  if (D <= 256) return launch_bwd_f64(a, D, dtype, o_dtype, stage, q_grid, kv_grid, st);
  return dispatch(dtype, o_dtype, a.precise, [&](auto s, auto p) {
    decltype(s)::template bwd<decltype(p)::value>(a, stage, q_grid, kv_grid, st);
  });
}

}  // namespace mattn
