// Products of float32 accuracy on the bfloat16 matrix cores, for the problems
// that hold their operands in float32: float32 inputs, and the weights, dS and
// dO of 16-bit inputs at the head dimensions the float16-operand kernels do
// not serve.
//
// A float32 value is the exact sum of three bfloat16 pieces (8 significant
// bits each, rounded to nearest, so of either sign), with float32's own
// exponent range: no scales, and nothing to bound beforehand.  A float16 value
// is the sum of two, a bfloat16 value is one.  A product of two such sums takes
// the piece products down to 2^-16 of the largest (six for two float32
// operands, three for float32 times bfloat16); what is left out is about 2^-25
// of a term, below the float32 accumulation's own rounding.  Six
// 32x32x16 bfloat16 MFMAs take 192 cycles of a SIMD's matrix core, the eight
// float32 32x32x2 MFMAs of the same product 512.
#pragma once

#include "common.hpp"

namespace mattn {
namespace s3 {

typedef short s16x4 __attribute__((ext_vector_type(4)));

template <class T>
struct Pieces;
template <>
struct Pieces<bf16_tag> { static constexpr int n = 1; };
template <>
struct Pieces<f16_tag> { static constexpr int n = 2; };
template <>
struct Pieces<float> { static constexpr int n = 3; };

// An MFMA operand (8 values a lane) in N pieces.
template <int N>
struct Frag { u32x4 p[N]; };

using B16 = Elt<bf16_tag>;

// c += a b: the piece products a_i b_j with i + j <= 2, the small ones first
template <int NA, int NB>
__device__ __forceinline__ f32x16 mma(const Frag<NA>& a, const Frag<NB>& b, f32x16 c) {
#pragma unroll
  for (int s = 2; s >= 0; --s)
#pragma unroll
    for (int i = 0; i < NA; ++i)
      if (s - i >= 0 && s - i < NB) c = B16::mfma(a.p[i], b.p[s - i], c);
  return c;
}

// The pieces of two values, packed (low half = x0): piece 0 is x rounded, each
// further one the rest rounded.
template <int N>
__device__ __forceinline__ void split2(float x0, float x1, uint32_t (&w)[N]) {
#pragma unroll
  for (int i = 0; i < N; ++i) {
    w[i] = B16::pack2(x0, x1);
    if (i + 1 < N) {
      x0 -= __uint_as_float(w[i] << 16);
      x1 -= __uint_as_float(w[i] & 0xffff0000u);
    }
  }
}

// C registers [8 j, 8 j + 8) of a 32x32 result as the B operand of a 16-deep k-step
__device__ __forceinline__ Frag<3> c_frag(const f32x16& c, int j) {
  Frag<3> f;
#pragma unroll
  for (int e = 0; e < 4; ++e) {
    uint32_t w[3];
    split2<3>(c[8 * j + 2 * e], c[8 * j + 2 * e + 1], w);
#pragma unroll
    for (int p = 0; p < 3; ++p) f.p[p][e] = w[p];
  }
  return f;
}

// 8 consecutive elements as loaded, and their pieces
template <class T>
struct Raw8 {
  u32x4 x;
  __device__ __forceinline__ void load(const char* p) { x = *(const u32x4*)p; }
  __device__ __forceinline__ Frag<Pieces<T>::n> split() const {
    Frag<Pieces<T>::n> f;
    if constexpr (Pieces<T>::n == 1) {
      f.p[0] = x;
    } else {
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        uint32_t w[Pieces<T>::n];
        split2(Elt<T>::to_f32(x[e] & 0xffffu), Elt<T>::to_f32(x[e] >> 16), w);
#pragma unroll
        for (int i = 0; i < Pieces<T>::n; ++i) f.p[i][e] = w[i];
      }
    }
    return f;
  }
};
template <>
struct Raw8<float> {
  f32x4 x, y;
  __device__ __forceinline__ void load(const char* p) {
    x = *(const f32x4*)p;
    y = *(const f32x4*)(p + 16);
  }
  __device__ __forceinline__ Frag<3> split() const {
    Frag<3> f;
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      uint32_t w[3];
      if (e < 2) split2<3>(x[2 * e], x[2 * e + 1], w);
      else split2<3>(y[2 * e - 4], y[2 * e - 3], w);
#pragma unroll
      for (int i = 0; i < 3; ++i) f.p[i][e] = w[i];
    }
    return f;
  }
};

template <class T>
constexpr int elt_bytes() { return Pieces<T>::n == 3 ? 4 : 2; }

// LDS tile of one piece: rows of D 16-bit values, the 16-byte chunk c of row r
// at chunk c ^ swz(r): ds_read_b128 row reads and ds_read_b64_tr_b16 reads are
// then free of bank conflicts (as the swizzle of common.hpp, D = 256 like 128:
// its rows span the banks twice and the low four chunk bits are swizzled).
template <int D>
__device__ __forceinline__ int swz3(int r) { return swz<(D == 64 ? 64 : 128)>(r); }

// ROWS rows of a [rows, D] tensor: loaded into registers, and written to LDS as
// planes of pieces, by NTH threads.
template <int D, class T, int ROWS, int NTH>
struct Stage {
  static constexpr int CH = ROWS * D / 8 / NTH;
  static constexpr int NP = Pieces<T>::n;
  static constexpr int ELTS = NP * ROWS * D;  // LDS elements
  static_assert(CH >= 1, "one chunk a thread");
  Raw8<T> v[CH];
  // rows past n - 1 re-read row n - 1 (their scores are masked)
  __device__ __forceinline__ void load(const char* base, int64_t rs, int r0, int n) {
#pragma unroll
    for (int c = 0; c < CH; ++c) {
      const int i = threadIdx.x + NTH * c, r = i / (D / 8), col = i % (D / 8);
      v[c].load(base + elt_bytes<T>() * ((int64_t)min(r0 + r, n - 1) * rs + 8 * col));
    }
  }
  __device__ __forceinline__ void store(uint16_t* lds) const {
#pragma unroll
    for (int c = 0; c < CH; ++c) {
      const int i = threadIdx.x + NTH * c, r = i / (D / 8), col = i % (D / 8);
      const Frag<NP> f = v[c].split();
#pragma unroll
      for (int p = 0; p < NP; ++p) *(u32x4*)(lds + p * ROWS * D + r * D + ((col ^ swz3<D>(r)) << 3)) = f.p[p];
    }
  }
};

// A operand, k along the columns: row r of the tile, columns 16 kd + 8 hi .. + 7
template <int D, int NP, int ROWS>
__device__ __forceinline__ Frag<NP> row_frag(const uint16_t* lds, int r, int kd, int hi) {
  Frag<NP> f;
#pragma unroll
  for (int p = 0; p < NP; ++p)
    f.p[p] = *(const u32x4*)(lds + p * ROWS * D + r * D + (((2 * kd + hi) ^ swz3<D>(r)) << 3));
  return f;
}

// A operand, k along the rows (r0 + 16 ks ..), its 32 rows the columns 32 mt ..: the
// transposed read of tr_src (common.hpp), k in the order of the C registers
template <int D, int NP, int ROWS>
__device__ __forceinline__ Frag<NP> tr_frag(const uint16_t* lds, int r0, int mt, int lane) {
  Frag<NP> f;
  const int i = lane & 15, g = lane >> 4, hi = lane >> 5;
  const int c = 4 * mt + 2 * (g & 1) + ((i & 3) >> 1);
#pragma unroll
  for (int p = 0; p < NP; ++p) {
#pragma unroll
    for (int sec = 0; sec < 2; ++sec) {
      const int r = 4 * hi + 8 * sec + (i >> 2);
      const uint16_t* src = lds + p * ROWS * D + (r0 + r) * D + ((c ^ swz3<D>(r)) << 3) + 4 * (i & 1);
      const s16x4 t = __builtin_amdgcn_ds_read_tr16_b64_v4i16((__attribute__((address_space(3))) s16x4*)src);
      const u32x2 w = __builtin_bit_cast(u32x2, t);
      f.p[p][2 * sec] = w[0];
      f.p[p][2 * sec + 1] = w[1];
    }
  }
  return f;
}

// 16-bit or float32 output of a row's values, through store_rows (common.hpp), in
// column blocks of at most 128 so that a wave stages 32 x 128 values at a time
template <int D, class T>
__device__ __forceinline__ void put_rows(const f32x16 (&acc)[D / 32], float sc, void* lds, void* out, int64_t row0,
                                         int64_t rstride, int nrows, int lane) {
  constexpr int ES = elt_bytes<T>(), DB = D > 128 ? 128 : D;
  using P = Elt<typename std::conditional<std::is_same<T, float>::value, bf16_tag, T>::type>;
#pragma unroll
  for (int c = 0; c < D / DB; ++c)
    store_rows<DB, ES, true>(*(const f32x16(*)[DB / 32])(&acc[c * (DB / 32)]), sc, lds, out, row0 + c * DB, rstride,
                             nrows, lane, P::pack2);
}
template <int D>
constexpr int put_bytes() { return 32 * (D > 128 ? 128 : D) * 4; }  // LDS of one wave

// c += the partner wave's c (waves w and w ^ pair, which each formed it over half of
// d), for N results, through LDS (4 KiB a wave and result): publish, barrier, add.
template <int N>
__device__ __forceinline__ void half_put(const f32x16 (&c)[N], float* X, int wave, int lane) {
#pragma unroll
  for (int n = 0; n < N; ++n)
#pragma unroll
    for (int j = 0; j < 4; ++j)
      *(f32x4*)(X + ((wave * N + n) * 4 + j) * 256 + 4 * lane) =
          f32x4{c[n][4 * j], c[n][4 * j + 1], c[n][4 * j + 2], c[n][4 * j + 3]};
}
template <int N>
__device__ __forceinline__ void half_add(f32x16 (&c)[N], const float* X, int wave, int lane) {
#pragma unroll
  for (int n = 0; n < N; ++n)
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const f32x4 y = *(const f32x4*)(X + ((wave * N + n) * 4 + j) * 256 + 4 * lane);
#pragma unroll
      for (int i = 0; i < 4; ++i) c[n][4 * j + i] += y[i];
    }
}

// Results of the WK waves that shared the same 32 rows (lane = row, registers =
// columns as in store_rows), summed through LDS and stored: slab [WK][WQ * 32][D]
// float32; each wave has already scaled its part.
template <int D, int WQ>
__device__ __forceinline__ void slab_put(const f32x16 (&acc)[D / 32], float sc, float* slab, int wq, int wk, int lane) {
  const int r = lane & 31, hi = lane >> 5;
  float* L = slab + (wk * WQ + wq) * 32 * D + r * D;
#pragma unroll
  for (int mt = 0; mt < D / 32; ++mt)
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const int c = (32 * mt + 8 * j + 4 * hi) >> 2;
      *(f32x4*)(L + ((c ^ (r & (D / 4 - 1))) << 2)) =
          f32x4{acc[mt][4 * j] * sc, acc[mt][4 * j + 1] * sc, acc[mt][4 * j + 2] * sc, acc[mt][4 * j + 3] * sc};
    }
}
template <int D, class T, int WQ, int WK, int NTH>
__device__ __forceinline__ void slab_sum_store(const float* slab, void* out, int64_t row0, int64_t rstride, int nrows) {
  using P = Elt<typename std::conditional<std::is_same<T, float>::value, bf16_tag, T>::type>;
#pragma unroll
  for (int i = 0; i < 32 * WQ * D / 4 / NTH; ++i) {
    const int n = threadIdx.x + NTH * i, row = n / (D / 4), c = n % (D / 4);
    f32x4 s = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int k = 0; k < WK; ++k)
      s += *(const f32x4*)(slab + ((k * WQ * 32 + row) * D) + ((c ^ (row & 31 & (D / 4 - 1))) << 2));
    if (row < nrows) {
      char* dst = (char*)out + elt_bytes<T>() * (row0 + (int64_t)row * rstride + 4 * c);
      if constexpr (std::is_same<T, float>::value) __builtin_nontemporal_store(s, (f32x4*)dst);
      else __builtin_nontemporal_store(u32x2{P::pack2(s[0], s[1]), P::pack2(s[2], s[3])}, (u32x2*)dst);
    }
  }
}

// base address of (b, h) in a tensor of element strides s
__device__ __forceinline__ const char* head_base(const void* p, const int64_t* s, int b, int h, int es) {
  return (const char*)p + es * ((int64_t)b * s[0] + (int64_t)h * s[2]);
}

// Sub-blocks of the walk over entries [e0, e1): SPT = 128 / BN per tile.
template <int BN>
struct Walk {
  static constexpr int SPT = TILE / BN;
  const int* ent;
  int e0, n;
  __device__ __forceinline__ Walk(const int* ent_, int e0_, int e1_) : ent(ent_), e0(e0_), n((e1_ - e0_) * SPT) {}
  __device__ __forceinline__ int first(int s) const { return ent[2 * (e0 + s / SPT)] * TILE + (s % SPT) * BN; }
  __device__ __forceinline__ int mask(int s) const { return ent[2 * (e0 + s / SPT) + 1]; }
};

}  // namespace s3
}  // namespace mattn
