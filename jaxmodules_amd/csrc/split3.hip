// Masked attention at float32 accuracy on the matrix cores (split3.hpp): the
// forward and the backward of float32 inputs at D = 64, 128 and 256 and of 16-bit
// inputs at D = 256 (MATTN_PRECISE: precise.hip; D = 512: the SIMT kernels of
// simt.hip, which these replaced).
//
// Same maths and tile walk as there (/root/reference/jaxmodules/
// attention.py:52-105 forward, :266-342 backward).  Every wave owns 16 rows (queries in
// the forward and dQ, keys in dK/dV; lane l % 16 = row) and walks the present tiles of
// its map row or column 32 rows of the other side at a time:
//   forward  S^T = K Q^T, online softmax, O^T += V^T P^T
//   dQ       S^T = K Q^T, dP^T = V dO^T, dS = P (dP - delta), dQ^T += K^T dS^T
//   dK/dV    S = Q K^T, dP = dO V^T, dV^T += dO^T P, dK^T += Q^T dS
// (dP - delta of weights of 1/2 and more: dO . (V - O), see HOT).
// The streamed rows are read once per workgroup and split into bfloat16 pieces on the
// way to LDS (bfloat16 rows go there directly); the wave's own rows are split in
// registers.  P and dS are split from the C registers, which are the B operand of the
// next product as they stand.
//
// Why 16 rows (v_mfma_f32_16x16x32_bf16): at D = 256 a wave of 32 rows holds its
// operands and results only by sharing them with a partner wave (each half of the
// columns, S and dP summed through LDS with a barrier, the softmax done by both) or by
// spilling; for float32 at D = 64 its dK/dV spilled at two waves a SIMD.  The price is
// LDS: a streamed operand is read per 16 rows, 125 bytes a clock and CU at the matrix
// cores' full rate.
// Measured, causal steps, kernel by kernel in a trace (with gaps between them, at another
// clock than a whole step's, so they don't add up to one): float32 [2, 2048, 8, 64]
// fwd 465 -> 97 us, dK/dV 768 -> 150, dQ 596 -> 115 against the SIMT kernels; bfloat16
// [1, 4096, 8, 256] fwd 4322 -> 204 us, dK/dV 14370 -> 588, dQ 4811 -> 264.  32-row waves
// sharing columns: 326, 750, 708 beside 192, 579, 248.  (Those before the shorter chains
// of Dot, the pairs of HOT and the check for Inf and NaN, which together cost 0 to 6%,
// 12% for float32 dK/dV at D = 256.  Logits of standard deviation 8, most rows dominated
// by one key: dK/dV 199 and 677 us, dQ 129 and 274.)
// The error against float64 is 0.6 to 1.1 times that of the SIMT kernels they replaced
// (0.7 and 0.8 of it for O and the gradients of that float32 step) over logits of standard
// deviation 1 to 32 and windows of two keys; rows of one key give dQ = dK = 0 exactly.
// Where one key of a large positive dot product has nearly all of a row's weight, O is up
// to 1.3 and dQ up to 1.4 times as far off (1e-7 of the norm).
// float32 at D = 64 is bound by vector instructions (270 a step and wave against 48 MFMAs
// of 16 cycles; half of them split the streamed rows).
//
// MFMA 16x16x32 layout (lane l, l16 = l % 16, g = l / 16): A row l16, k = 8 g .. 8 g + 7;
// B column l16, the same k; C column l16, register r row 4 g + r.  The two 16-row
// blocks t of a 32-row step leave lane (l16, g) with rows 16 t + 4 g + r, taken as the
// 8 values of the next product's B operand; its A operand (transposed reads) holds the
// same rows in the same places.
#include <type_traits>

#include "split3.hpp"

namespace mattn {
namespace {
using namespace s3;

// the two blocks' C registers as a B operand over the 32 rows
__device__ __forceinline__ Frag<3> c_frag16(const f32x4& c0, const f32x4& c1) {
  Frag<3> f;
#pragma unroll
  for (int e = 0; e < 4; ++e) {
    uint32_t w[3];
    if (e < 2) split2<3>(c0[2 * e], c0[2 * e + 1], w);
    else split2<3>(c1[2 * e - 4], c1[2 * e - 3], w);
#pragma unroll
    for (int p = 0; p < 3; ++p) f.p[p][e] = w[p];
  }
  return f;
}

constexpr int BN = 32;  // streamed rows a step

// LDS tile of one piece: 16-byte chunk c of row r at c ^ sw(r).  A row read takes one
// chunk of 16 rows, a transposed read (32 lanes) one chunk pair of 8 aligned rows: both
// hit 16 (8 pairs of) distinct 16-byte bank groups.  (A row of D = 64 is half the 64
// banks: its parity is the fourth bit.)
template <int D>
__device__ __forceinline__ int sw(int r) {
  if constexpr (D == 64) return (((r >> 1) & 3) << 1) | ((r >> 3) & 1);
  else return ((r & 7) << 1) | ((r >> 3) & 1);
}

// BN rows of a tensor to LDS as planes of pieces.  bfloat16 rows (one piece, as they are)
// go straight to LDS (DMA); others through registers and split.
template <int D, class T, int NTH, bool WIDE = false>
struct Rows {
  static constexpr int NP = Pieces<T>::n, CPR = D / 8, ELTS = NP * BN * D;
  static constexpr int CH = BN * CPR / NTH;
  static constexpr bool DMA = NP == 1;
  Raw8<T> v[DMA ? 1 : CH];
  // registers, or (DMA) LDS `dst`; rows past n - 1 re-read row n - 1 (masked)
  __device__ __forceinline__ void load(const char* base, int64_t rs, int r0, int n, uint16_t* dst) {
    each_chunk<D, elt_bytes<T>(), BN, NTH, WIDE>(base, rs, r0, n, [&](int c, const char* p, uint32_t off) {
      const int i = threadIdx.x + NTH * c, r = i / CPR, col = i % CPR;
      if constexpr (DMA) {
        const int blk = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6) + c * (NTH / 64);
        lds_load16(p + (off + 16 * (col ^ sw<D>(r))), dst + blk * 512);  // lane l of block blk: chunk 64 blk + l
      } else {
        v[c].load(p + (off + elt_bytes<T>() * 8 * col));
      }
    });
  }
  __device__ __forceinline__ void store(uint16_t* dst) const {
    if constexpr (!DMA) {
#pragma unroll
      for (int c = 0; c < CH; ++c) {
        const int i = threadIdx.x + NTH * c, r = i / CPR, col = i % CPR;
        const Frag<NP> f = v[c].split();
#pragma unroll
        for (int p = 0; p < NP; ++p) *(u32x4*)(dst + p * BN * D + r * D + ((col ^ sw<D>(r)) << 3)) = f.p[p];
      }
    }
  }
};

// LDS byte addresses of the operand reads of a tile at `base` (512-byte aligned): the
// chunk index is XORed with bits of the row alone, so column steps are XORs too
//   along d:       rows 16 t + l16, columns 32 kd + 8 g ..: row_addr ^ (64 kd), offset 16 t rows
//   along the rows: columns 16 mt .., k slot 4 t + j = row 16 t + 4 g + j: tr_addr ^ (32 mt), offset 16 t rows
template <int D>
__device__ __forceinline__ uint32_t row_addr(int l16, int g) {
  return 2 * l16 * D + ((g ^ sw<D>(l16)) << 4);
}
template <int D>
__device__ __forceinline__ uint32_t tr_addr(int l16, int g) {
  const int r = 4 * g + (l16 >> 2);
  return 2 * r * D + ((((l16 & 3) >> 1) ^ sw<D>(r)) << 4) + 8 * (l16 & 1);
}

// A dot product along d in the making (C registers of one 16-row block), over D / 32 steps.
// A 16x16x32 MFMA rounds its result four times (measured: off by 0.58 units in the last
// place in the mean square, one rounding is 0.29), so one chain of all piece products
// carries 4 x 6 roundings a step at the size the sum has reached: O of float32 problems
// with logits of 10 and more was 1.3, 1.9 and 3.1 times as far off at D = 64, 128 and 256
// as sums of 16 or 32 FMAs a lane had left it.  So the small products (2^-8 of the size
// and less) come first, or apart from the leading ones:
//   LAST    one chain, the first step's leading product at its end (D = 64, where two
//           more additions an element are 5% of the backward)
//   HALVES  a: the leading products of the first half of the steps, b: the small ones
//           and the other half; a + b (D = 128)
//   LINKS   the leading products two steps at a time in a, summed here, but for the last
//           two, which follow the small ones in b (D = 256)
//   ONE     one chain in the order of the steps
enum Chains { ONE, LAST, HALVES, LINKS };
template <int D, int NA, int NB, Chains C>
struct Dot {
  static constexpr int N = D / 32, TAIL = C == HALVES ? N / 2 : N - 2;  // leading products from TAIL on: b
  static_assert(C != LAST || N == 2, "");
  f32x4 a, b, sum;
  u32x4 x0, y0;  // LAST: the first step's leading operands
  template <int KD>
  __device__ __forceinline__ void begin() {
    if constexpr (KD == 0 || (C == LINKS && KD < TAIL && KD % 2 == 0)) a = f32x4{};
    if constexpr (C >= HALVES && KD == 0) b = f32x4{};
  }
  // product n of step KD
  template <int KD, int n>
  __device__ __forceinline__ void mma(const Frag<NA>& x, const Frag<NB>& y) {
    constexpr int ij = product_ij(NA, NB, n);
    if constexpr (C == LAST && KD == 0 && ij == 0) {
      x0 = x.p[0];
      y0 = y.p[0];
    } else {
      mfma1(x.p[ij / 4], y.p[ij % 4], C < HALVES || (ij == 0 && KD < TAIL) ? a : b);
    }
  }
  template <int KD>
  __device__ __forceinline__ void end() {
    if constexpr (C == LAST && KD == N - 1) mfma1(x0, y0, a);
    if constexpr (C == LINKS && KD < TAIL && KD % 2 == 1) {
      if constexpr (KD == 1) sum = a;
      else sum += a;
    }
  }
  __device__ __forceinline__ f32x4 total() const { return C < HALVES ? a : C == HALVES ? a + b : sum + b; }
};
// x and y's products of step KD in turn (an MFMA that adds to the result of the one before
// it waits for it)
template <int KD, int D, int NA, int NB, int NC, int ND, Chains C>
__device__ __forceinline__ void dot_step(Dot<D, NA, NB, C>& x, const Frag<NA>& a, const Frag<NB>& b,
                                         Dot<D, NC, ND, C>& y, const Frag<NC>& c, const Frag<ND>& d) {
  constexpr int P1 = products(NA, NB), P2 = products(NC, ND);
  x.template begin<KD>();
  y.template begin<KD>();
  static_for<(P1 > P2 ? P1 : P2)>([&](auto nc) {
    constexpr int n = decltype(nc)::value;
    if constexpr (n < P1) x.template mma<KD, n>(a, b);
    if constexpr (n < P2) y.template mma<KD, n>(c, d);
  });
  x.template end<KD>();
  y.template end<KD>();
}

// S = A X along d for both 16-row blocks: tile at byte address ra
template <int WANT, Chains C, int D, int NA, int NX>
__device__ __forceinline__ void one_dot(uint32_t ra, const Frag<NX> (&x)[D / 32], f32x4 (&st)[2]) {
  constexpr int PF = ahead(WANT, 2 * NA), PL = 2 * BN * D;
  Frag<NA> f0[PF + 1], f1[PF + 1];
  Dot<D, NA, NX, C> s0, s1;
  pipe<D / 32, PF, 2 * NA>(
      [&](auto ic, auto sc) {
        constexpr int kd = decltype(ic)::value, sl = decltype(sc)::value;
        rd<0, PL>(f0[sl], ra ^ (uint32_t)(64 * kd));
        rd<32 * D, PL>(f1[sl], ra ^ (uint32_t)(64 * kd));
      },
      [&](auto ic, auto sc) {
        constexpr int kd = decltype(ic)::value, sl = decltype(sc)::value;
        landed(f0[sl]);
        landed(f1[sl]);
        dot_step<kd>(s0, f0[sl], x[kd], s1, f1[sl], x[kd]);
      });
  st[0] = s0.total();
  st[1] = s1.total();
}
// S = A X and dP = A2 X2 along d for both 16-row blocks t: tiles at byte addresses ra, rb
// (block by block; ONE: both blocks at each step; LINKS: one product after the other, whose
// operands in flight then leave room for the chains: side by side, float32 at D = 256
// spilled 88 and 117 registers, dK/dV 360 -> 460 and dQ 321 -> 476 us of [1, 2048, 8])
template <int WANT, Chains C, int D, int NA, int NX, int NB, int NY>
__device__ __forceinline__ void two_dots(uint32_t ra, uint32_t rb, const Frag<NX> (&x)[D / 32], const Frag<NY> (&y)[D / 32],
                                         f32x4 (&st)[2], f32x4 (&dp)[2]) {
  if constexpr (C == LINKS) {
    one_dot<1, C, D, NA>(ra, x, st);
    one_dot<1, C, D, NB>(rb, y, dp);
    return;
  }
  constexpr int PF = ahead(WANT, NA + NB), PL = 2 * BN * D, N = D / 32;
  Frag<NA> fa[PF + 1];
  Frag<NB> fb[PF + 1];
  Dot<D, NA, NX, C> s[C == ONE ? 2 : 1];
  Dot<D, NB, NY, C> p[C == ONE ? 2 : 1];
  pipe<2 * N, PF, NA + NB>(
      [&](auto ic, auto sc) {
        constexpr int i = decltype(ic)::value, sl = decltype(sc)::value;
        constexpr int kd = C == ONE ? i / 2 : i % N, t = C == ONE ? i % 2 : i / N;
        if constexpr (C != ONE && i == N) {  // the second block's addresses are formed anew (kept: 2 N registers)
          ra = opaque(ra);
          rb = opaque(rb);
        }
        rd<32 * t * D, PL>(fa[sl], ra ^ (uint32_t)(64 * kd));
        rd<32 * t * D, PL>(fb[sl], rb ^ (uint32_t)(64 * kd));
      },
      [&](auto ic, auto sc) {
        constexpr int i = decltype(ic)::value, sl = decltype(sc)::value;
        constexpr int kd = C == ONE ? i / 2 : i % N, t = C == ONE ? i % 2 : i / N, u = C == ONE ? t : 0;
        landed(fa[sl]);
        landed(fb[sl]);
        dot_step<kd>(s[u], fa[sl], x[kd], p[u], fb[sl], y[kd]);
        if constexpr (kd == N - 1) {
          st[t] = s[u].total();
          dp[t] = p[u].total();
        }
      });
}
// (forward and backward alike where gradients are float32: P = exp2(S - lse) takes S as
// lse has it.  16-bit gradients at D = 256 hide the difference by their own rounding.)
template <int D>
constexpr Chains fwd_chains() { return D == 64 ? LAST : D == 128 ? HALVES : LINKS; }
template <int D, class IT>
constexpr Chains bwd_chains() { return D == 256 && !std::is_same<IT, float>::value ? ONE : fwd_chains<D>(); }
// acc[mt] += (tile at byte address ta)^T w, the 32 rows of the tile against w
template <int D, int NA, int WANT = 2>
__device__ __forceinline__ void add_rows(uint32_t ta, const Frag<3>& w, f32x4 (&acc)[D / 16]) {
  constexpr int PF = ahead(WANT, 4 * NA), PL = 2 * BN * D;
  Tr<NA> f0[PF + 1], f1[PF + 1];
  pipe<D / 32, PF, 4 * NA>(
      [&](auto ic, auto sc) {
        constexpr int i = decltype(ic)::value, sl = decltype(sc)::value;
        static_for<NA>([&](auto pc) {
          constexpr int p = decltype(pc)::value;
          f0[sl].lo[p] = ds_read_tr8<p * PL>(ta ^ (uint32_t)(64 * i));
          f0[sl].up[p] = ds_read_tr8<p * PL + 32 * D>(ta ^ (uint32_t)(64 * i));
          f1[sl].lo[p] = ds_read_tr8<p * PL>(ta ^ (uint32_t)(64 * i + 32));
          f1[sl].up[p] = ds_read_tr8<p * PL + 32 * D>(ta ^ (uint32_t)(64 * i + 32));
        });
      },
      [&](auto ic, auto sc) {
        constexpr int i = decltype(ic)::value, sl = decltype(sc)::value;
        const Frag<NA> a0 = landed(f0[sl]), a1 = landed(f1[sl]);
        mma_two(a0, w, acc[2 * i], a1, w, acc[2 * i + 1]);
      });
}
// B operand of the wave's own rows: row r of a tensor slice, columns 32 kd + 8 g .. + 7
template <int D, class T>
__device__ __forceinline__ void own16(Frag<Pieces<T>::n> (&f)[D / 32], const char* base, int64_t rs, int r, int g) {
#pragma unroll
  for (int kd = 0; kd < D / 32; ++kd) {
    Raw8<T> x;
    x.load(base + elt_bytes<T>() * ((int64_t)r * rs + 32 * kd + 8 * g));
    f[kd] = x.split();
  }
}

// The wave's 16 rows (lane l16 = row, acc[mt][r] = column 16 mt + 4 g + r) times sc to a
// tensor, through LDS (16 x D float32 a wave) so that rows are stored whole.
template <int D, class T>
__device__ __forceinline__ void put16(const f32x4 (&acc)[D / 16], float sc, float* L, void* out, int64_t row0,
                                      int64_t rstride, int nrows, int lane) {
  using P = Elt<typename std::conditional<std::is_same<T, float>::value, bf16_tag, T>::type>;
  const int l16 = lane & 15, g = lane >> 4;
#pragma unroll
  for (int mt = 0; mt < D / 16; ++mt)
    *(f32x4*)(L + l16 * D + (((4 * mt + g) ^ l16) << 2)) = acc[mt] * sc;
#pragma unroll
  for (int i = 0; i < 16 * D / 8 / 64; ++i) {
    const int n = 64 * i + lane, row = n / (D / 8), c = 2 * (n % (D / 8));
    const f32x4 x = *(const f32x4*)(L + row * D + ((c ^ row) << 2));
    const f32x4 y = *(const f32x4*)(L + row * D + (((c + 1) ^ row) << 2));
    if (row < nrows) {
      char* dst = (char*)out + elt_bytes<T>() * (row0 + (int64_t)row * rstride + 4 * c);
      if constexpr (std::is_same<T, float>::value) {
        __builtin_nontemporal_store(x, (f32x4*)dst);
        __builtin_nontemporal_store(y, (f32x4*)dst + 1);
      } else {
        __builtin_nontemporal_store(u32x4{P::pack2(x[0], x[1]), P::pack2(x[2], x[3]), P::pack2(y[0], y[1]),
                                          P::pack2(y[2], y[3])}, (u32x4*)dst);
      }
    }
  }
}

constexpr int cmax(int a, int b) { return a > b ? a : b; }

// the 32 mask bits of row `row` (of a tile) against the 32-row block `blk` of the other
// side, shifted so that bit 16 t + r is the one of C register r of block t
__device__ __forceinline__ uint32_t bits32(const uint64_t* bits, int mask, int blk, int row, int g) {
  return (uint32_t)(bits[((int64_t)mask * 2 + (blk >> 1)) * TILE + row] >> (32 * (blk & 1))) >> (4 * g);
}
__device__ __forceinline__ uint32_t ones16(uint32_t w, int t, int r) {
  uint32_t m = (uint32_t)__builtin_amdgcn_sbfe((int)w, 16 * t + r, 1);
  asm("" : "+v"(m));
  return m;
}

// max of x over lanes l and l ^ 16 (no LDS access)
__device__ __forceinline__ float wave_max16(float x) {
  const auto r = __builtin_amdgcn_permlane16_swap(__float_as_uint(x), __float_as_uint(x), false, false);
  return fmaxf(__uint_as_float(r[0]), __uint_as_float(r[1]));
}

// P = 0 where the mask bit is clear
__device__ __forceinline__ void zero16(f32x4 (&p)[2], uint32_t w) {
#pragma unroll
  for (int t = 0; t < 2; ++t)
#pragma unroll
    for (int r = 0; r < 4; ++r) p[t][r] = mask_zero(p[t][r], ones16(w, t, r));
}

// 4 consecutive elements as float32
template <class T>
__device__ __forceinline__ f32x4 load4(const char* p) {
  if constexpr (std::is_same<T, float>::value) {
    return *(const f32x4*)p;
  } else {
    const u32x2 x = *(const u32x2*)p;
    return f32x4{Elt<T>::to_f32(x[0] & 0xffffu), Elt<T>::to_f32(x[0] >> 16), Elt<T>::to_f32(x[1] & 0xffffu),
                 Elt<T>::to_f32(x[1] >> 16)};
  }
}
// the four 16-lane groups' values, summed (in all of them)
__device__ __forceinline__ float sum_groups(float x) {
  x += __shfl_xor(x, 16);
  return x + __shfl_xor(x, 32);
}
// The kernel's arguments read anew: what only rarely taken paths need of them would
// otherwise be read at the kernel's start and held over the walk.
__device__ __forceinline__ const KArgs& args_again() {
  uint64_t p = (uint64_t)__builtin_amdgcn_kernarg_segment_ptr();
  asm volatile("" : "+s"(p));
  return *(const KArgs*)(const __attribute__((address_space(4))) KArgs*)p;
}
// O of a problem whose gradient has type GT: float32 beside a 16-bit dO under MATTN_DO_16
template <class GT>
__device__ __forceinline__ bool o_is_f32(const KArgs& a) {
  return std::is_same<GT, float>::value || a.do16;
}
// row r of a tensor slice at lane group g's first column
template <class T>
__device__ __forceinline__ const char* row_at(const char* base, int64_t rs, int r, int g) {
  return base + elt_bytes<T>() * ((int64_t)r * rs + 4 * g);
}
// the rows a hot pair needs, at the lane's first column 4 g
struct HotRows { const char *g, *v, *o, *x; };
// dO . (V - O) of three rows, in float32 (every lane of a row's four has the sum).  U: column steps whose loads are in flight together (left alone, the compiler waits for
// each step's three before it issues the next)
template <int U, int D, class IT, class GT>
__device__ __forceinline__ float dot_vo(const HotRows& p, bool of32) {
  f32x4 s = {};
#pragma unroll 1
  for (int j = 0; j < D / 16; j += U) {
    f32x4 x[U], y[U], z[U];
#pragma unroll
    for (int u = 0; u < U; ++u) {
      x[u] = load4<GT>(p.g + 16 * elt_bytes<GT>() * (j + u));
      y[u] = load4<IT>(p.v + 16 * elt_bytes<IT>() * (j + u));
    }
    if (std::is_same<GT, float>::value || of32) {
#pragma unroll
      for (int u = 0; u < U; ++u) z[u] = load4<float>(p.o + 64 * (j + u));
    } else {
#pragma unroll
      for (int u = 0; u < U; ++u) z[u] = load4<GT>(p.o + 16 * elt_bytes<GT>() * (j + u));
    }
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int u = 0; u < U; ++u)
#pragma unroll
      for (int e = 0; e < 4; ++e) s[e] = fmaf(x[u][e], y[u][e] - z[u][e], s[e]);
    __builtin_amdgcn_sched_barrier(0);
  }
  return sum_groups((s[0] + s[1]) + (s[2] + s[3]));
}

// Pairs whose weight reaches HOT take dP - delta as dO . (V - O).  Where one key
// dominates a row its dP and delta are nearly the same number, and their roundings
// (2^-24 of |dO| |V|) would be all that is left of the difference; V - O is small there
// and exact to O's own rounding.  (Left to the difference, dQ and dK of rows with a weight
// of 0.9 or more were 2.4 to 4.9 times as far off.)
// Where no row is dominated the check and the list cost dK/dV 1 to 2% and dQ nothing that
// three traces resolve (float32 [2, 2048, 8, 64] dK/dV 148 -> 150 us, dQ 116 -> 115, at
// D = 128 255 -> 260 and 237 -> 236); at 1/4 instead of 1/2 they found no error to take away.
// A step leaves its hot pairs out of dS and notes them, up to MAX for each of the wave's
// rows; they are added after the walk, when its operands' registers are free and all 16
// rows have theirs formed at once (dK/dV of such float32 rows at D = 64, one dominant key
// each: 207 us; formed in each step, 16 rows of one pair: 236).  A query (dQ) has no more
// than two.  A key that more than eight queries lean on (the first one of a sequence,
// often) has the rest formed in their step, hot_rest().
constexpr float HOT = 0.5f;
constexpr int HOT_Q = 2, HOT_K = 8;
template <int MAX>
struct HotList {
  int n[16];
  int2 pair[16][MAX];  // streamed row, weight
};
__device__ __forceinline__ bool any_hot(const f32x4 (&p)[2]) {
  float mx = 0.f;
#pragma unroll
  for (int t = 0; t < 2; ++t)
#pragma unroll
    for (int r = 0; r < 4; ++r) mx = fmaxf(mx, p[t][r]);
  return __builtin_expect(__any(mx >= HOT), 0);  // (laid out of the walk's way)
}
// The step's pairs: p weights, d = dP - delta, r0 the first streamed row.  Returns the
// lane's hot pairs that found no place, bit 4 t + r.
template <int MAX>
__device__ __forceinline__ uint32_t note_hot(const f32x4 (&p)[2], f32x4 (&d)[2], HotList<MAX>& list, int r0) {
  // (re-defined here: what depends on the lane alone would be formed before the walk and kept)
  const int lane = opaque(threadIdx.x) & 63, l16 = lane & 15, g = lane >> 4;
  uint32_t own = 0, rest = 0;
#pragma unroll
  for (int t = 0; t < 2; ++t)
#pragma unroll
    for (int r = 0; r < 4; ++r) own |= (p[t][r] >= HOT ? 1u : 0u) << (4 * t + r);
  uint32_t m = own << (8 * g);  // the row's: bit 8 g + 4 t + r
  m |= __shfl_xor(m, 16);
  m |= __shfl_xor(m, 32);
  const int n = list.n[l16];
  int at = n + (int)__builtin_popcount(m & ((1u << (8 * g)) - 1u));  // place of this lane's next one
#pragma unroll
  for (int t = 0; t < 2; ++t)
#pragma unroll
    for (int r = 0; r < 4; ++r)
      if ((own >> (4 * t + r)) & 1u) {
        if (at < MAX) {
          list.pair[l16][at++] = make_int2(r0 + 16 * t + 4 * g + r, __float_as_int(p[t][r]));
          d[t][r] = 0.f;
        } else {
          rest |= 1u << (4 * t + r);
        }
      }
  list.n[l16] = min(n + (int)__builtin_popcount(m), MAX);
  return rest;
}
// d of the pairs note_hot had no place for, 16 at a time whatever rows they belong to.
// rows(own, i): the rows of own row `own` (0 .. 15) and streamed row i (0 .. 31) at lane group g.
template <int D, class IT, class GT, class F>
__device__ __forceinline__ void hot_rest(f32x4 (&d)[2], uint32_t rest, bool of32, F&& rows) {
  while (__any(rest != 0)) {
    const int lane = opaque(threadIdx.x) & 63, g = lane >> 4;
    const uint64_t b = __ballot(rest != 0);
    const int rank = (int)__builtin_amdgcn_mbcnt_hi((uint32_t)(b >> 32), __builtin_amdgcn_mbcnt_lo((uint32_t)b, 0u));
    const bool mine = rest != 0 && rank < 16;
    const int e = rest ? (int)__builtin_ctz(rest) : 0;
    // pair `rank` to the four lanes l16 = rank (lanes without one form pair (0, 0))
    const int pair = __builtin_amdgcn_ds_permute(4 * (mine ? rank : 63), mine ? (lane & 15) | (16 * (e >> 2) + 4 * g + (e & 3)) << 4 : 0);
    const int got = __shfl(pair, lane & 15);
    const float x = __shfl(dot_vo<2, D, IT, GT>(rows(got & 15, got >> 4, g), of32), rank & 15);
#pragma unroll
    for (int t = 0; t < 2; ++t)
#pragma unroll
      for (int r = 0; r < 4; ++r)
        if (mine && e == 4 * t + r) d[t][r] = x;
    if (mine) rest &= rest - 1;
  }
}
// acc[mt] += the noted pairs' dS times their streamed rows x; rows(i): those of streamed row i
template <int D, class IT, class GT, int MAX, class F>
__device__ __forceinline__ void add_hot(f32x4 (&acc)[D / 16], HotList<MAX>& list, int l16, bool of32, F&& rows) {
  const int nh = list.n[l16];
  for (int n = 0; __any(n < nh); ++n) {
    const bool on = n < nh;
    const int2 pw = list.pair[l16][n];
    const HotRows p = rows(on ? pw.x : 0);
    // at D = 64 every load of a round in flight at once; beyond, the registers that takes cost
    // the walk more (D = 128: 86 moves a step to and from the accumulation registers)
    constexpr int U = D == 64 ? 4 : 2;
    f32x4 x[D / 16];
    if constexpr (D == 64) {
#pragma unroll
      for (int mt = 0; mt < D / 16; ++mt) x[mt] = load4<IT>(p.x + 16 * elt_bytes<IT>() * mt);
    }
    const float ds = __int_as_float(pw.y) * dot_vo<U, D, IT, GT>(p, of32);
#pragma unroll
    for (int mt = 0; mt < D / 16; ++mt) {
      if constexpr (D != 64) x[mt] = load4<IT>(p.x + 16 * elt_bytes<IT>() * mt);
#pragma unroll
      for (int e = 0; e < 4; ++e) acc[mt][e] = on ? fmaf(ds, x[mt][e], acc[mt][e]) : acc[mt][e];
    }
  }
}

// ---- results that are not finite ---------------------------------------------------
// The pieces of an infinity do not add up to it (Inf - Inf), those of a float32 past
// bfloat16's largest value neither, an infinite piece times a zero one is NaN, and so is
// the weight 0 of a masked key times an infinite V.  All of this ends as Inf or NaN in the
// results of the rows it meets, never as a wrong finite value; so a wave that finds either
// there forms its 16 rows again in plain float32, pair by allowed pair, which gives the
// infinities and NaNs that the arithmetic of the inputs has.  Lanes as before: l16 the row,
// g its columns 16 j + 4 g .. + 3.  (g is re-defined for each pair, so that the own row's
// columns are not held over the loop.)  A pair takes a wave about 1.4 us, most of it
// waiting, so this is slow: the causal steps above 2.4 and 16 ms with an Inf in one row of
// V (0.43 and 1.1 without).  NaN stays NaN whatever is added, so a wave whose rows are NaN
// throughout is done: NaN everywhere, a diverged problem's state, 0.5 and 1.5 ms (walked
// to the end 10.6 and 91).
template <int N>
__device__ __forceinline__ bool not_finite(const f32x4 (&acc)[N]) {
  float t = 0.f;
#pragma unroll
  for (int i = 0; i < N; ++i)
#pragma unroll
    for (int e = 0; e < 4; ++e) t = fmaf(acc[i][e], 0.f, t);
  return __builtin_expect(__any(!(t == 0.f)), 0);
}
template <int N>
__device__ __forceinline__ bool all_nan(const f32x4 (&acc)[N]) {
  bool r = true;
#pragma unroll
  for (int i = 0; i < N; ++i)
#pragma unroll
    for (int e = 0; e < 4; ++e) r &= !(acc[i][e] == acc[i][e]);
  return r;
}
// f(other, on): every position `other` < n of the present tiles of a map row (or column)
// with an allowed pair in the wave, on where the lane's own row has it; looks every 16
// positions whether all lanes are done()
template <class F, class E>
__device__ __forceinline__ void each_pair(const int* ent, int e0, int e1, const uint64_t* bits, int row, int n, F&& f,
                                          E&& done) {
#pragma unroll 1
  for (int e = e0; e < e1; ++e) {
    const int first = ent[2 * e] * TILE, mask = ent[2 * e + 1];
#pragma unroll 1
    for (int half = 0; half < 2; ++half) {
      const uint64_t w = mask < 0 ? ~0ull : bits[((int64_t)mask * 2 + half) * TILE + row];
#pragma unroll 1
      for (int i = 0; i < 64 && first + 64 * half + i < n; ++i) {
        const bool on = (w >> i) & 1u;
        if (__any(on)) f(first + 64 * half + i, on);
        if (i % 16 == 15 && __all(done())) return;
      }
    }
  }
}
template <int D, class T>
__device__ __forceinline__ float dot_plain(const char* x, const char* y) {
  f32x4 s = {};
#pragma unroll 2
  for (int j = 0; j < D / 16; ++j) {
    const f32x4 u = load4<T>(x + 16 * elt_bytes<T>() * j), v = load4<T>(y + 16 * elt_bytes<T>() * j);
#pragma unroll
    for (int e = 0; e < 4; ++e) s[e] = fmaf(u[e], v[e], s[e]);
  }
  return sum_groups((s[0] + s[1]) + (s[2] + s[3]));
}
// acc += w x where on
template <int D, class T>
__device__ __forceinline__ void add_plain(f32x4 (&acc)[D / 16], float w, const char* x, bool on) {
#pragma unroll
  for (int j = 0; j < D / 16; ++j) {
    const f32x4 u = load4<T>(x + 16 * elt_bytes<T>() * j);
#pragma unroll
    for (int e = 0; e < 4; ++e) acc[j][e] = on ? fmaf(w, u[e], acc[j][e]) : acc[j][e];
  }
}
template <int N>
__device__ __forceinline__ void clear(f32x4 (&acc)[N]) {
#pragma unroll
  for (int i = 0; i < N; ++i) acc[i] = f32x4{};
}
// The wave's 16 rows from row0 (of tile qt or kt: TILE t + row0) once more.
// forward: O times the weights' sum l, and lse.  l and lse come in as the walk had them: a
// finite l says that every score was finite, and then both hold whatever V is.
template <int D, class IT>
__device__ __forceinline__ void plain_fwd(const KArgs& a, int b, int h, int qt, int row0, f32x4 (&acc)[D / 16], float& l,
                                          float& lse) {
  const int row = row0 + (opaque(threadIdx.x) & 15), qc = min(qt * TILE + row, a.Lq - 1), hk = h / a.G;
  const int mrow = map_row(a, b, h, a.nqt, qt);
  const char* qb = head_base(a.q, a.qs, b, h, elt_bytes<IT>());
  const char* kb = head_base(a.k, a.ks, b, hk, elt_bytes<IT>());
  const char* vb = head_base(a.v, a.vs, b, hk, elt_bytes<IT>());
  const float l0 = l;
  const bool held = l0 * 0.f == 0.f;
  float m = NEG_INF;
  l = 0.f;
  clear(acc);
  each_pair(a.row_ent, a.row_ptr[mrow], a.row_ptr[mrow + 1], a.row_bits, row, a.Lk, [&](int key, bool on) {
    const int g = (opaque(threadIdx.x) & 63) >> 4;
    const float s = dot_plain<D, IT>(row_at<IT>(qb, a.qs[1], qc, g), row_at<IT>(kb, a.ks[1], key, g));
    const float mn = on ? fmaxf(m, s) : m, mu = mn == NEG_INF ? 0.f : mn;
    const float alpha = on ? fast_exp2((m - mu) * a.scale_log2) : 1.f, p = fast_exp2((s - mu) * a.scale_log2);
    m = mn;
    l = on ? fmaf(l, alpha, p) : l;
#pragma unroll
    for (int i = 0; i < D / 16; ++i) acc[i] *= alpha;
    add_plain<D, IT>(acc, p, row_at<IT>(vb, a.vs[1], key, g), on);
  }, [&] { return all_nan(acc) && (held || !(l == l)); });
  if (held && all_nan(acc)) l = l0;
  else lse = l > 0.f ? fmaf(m, a.scale_log2, __builtin_log2f(l)) : NEG_INF;
}
// dQ (without its scale)
template <int D, class IT, class GT>
__device__ __forceinline__ void plain_dq(const KArgs& a, int b, int h, int qt, int row0, f32x4 (&acc)[D / 16]) {
  const int row = row0 + (opaque(threadIdx.x) & 15), qc = min(qt * TILE + row, a.Lq - 1), hk = h / a.G;
  const int mrow = map_row(a, b, h, a.nqt, qt);
  const bool of32 = o_is_f32<GT>(a);
  const char* qb = head_base(a.q, a.qs, b, h, elt_bytes<IT>());
  const char* kb = head_base(a.k, a.ks, b, hk, elt_bytes<IT>());
  const char* vb = head_base(a.v, a.vs, b, hk, elt_bytes<IT>());
  const char* gb = head_base(a.dO, a.dos, b, h, elt_bytes<GT>());
  const char* ob = head_base(a.o, a.os, b, h, of32 ? 4 : 2);
  const float lse = a.lse[((int64_t)b * a.Hq + h) * a.Lq + qc];
  clear(acc);
  each_pair(a.row_ent, a.row_ptr[mrow], a.row_ptr[mrow + 1], a.row_bits, row, a.Lk, [&](int key, bool on) {
    const int g = (opaque(threadIdx.x) & 63) >> 4;
    const char* kr = row_at<IT>(kb, a.ks[1], key, g);
    const float s = dot_plain<D, IT>(row_at<IT>(qb, a.qs[1], qc, g), kr);
    const float x = dot_vo<2, D, IT, GT>(HotRows{row_at<GT>(gb, a.dos[1], qc, g), row_at<IT>(vb, a.vs[1], key, g),
                                                 ob + (of32 ? 4 : 2) * ((int64_t)qc * a.os[1] + 4 * g), kr}, of32);
    add_plain<D, IT>(acc, fast_exp2(fmaf(s, a.scale_log2, -lse)) * x, kr, on);
  }, [&] { return all_nan(acc); });
}
// PART: 1 = dV, 2 = dK (without its scale)
template <int D, class IT, class GT, int PART>
__device__ __forceinline__ void plain_dkdv(const KArgs& a, int b, int hk, int kt, int row0, f32x4 (&acc)[D / 16]) {
  const int row = row0 + (opaque(threadIdx.x) & 15), kc = min(kt * TILE + row, a.Lk - 1);
  const bool of32 = o_is_f32<GT>(a);
  const char* kb = head_base(a.k, a.ks, b, hk, elt_bytes<IT>());
  const char* vb = head_base(a.v, a.vs, b, hk, elt_bytes<IT>());
  clear(acc);
#pragma unroll 1
  for (int h = hk * a.G; h < (hk + 1) * a.G; ++h) {
    const int mc = map_row(a, b, h, a.nkt, kt);
    const char* qb = head_base(a.q, a.qs, b, h, elt_bytes<IT>());
    const char* gb = head_base(a.dO, a.dos, b, h, elt_bytes<GT>());
    const char* ob = head_base(a.o, a.os, b, h, of32 ? 4 : 2);
    each_pair(a.col_ent, a.col_ptr[mc], a.col_ptr[mc + 1], a.col_bits, row, a.Lq, [&](int q, bool on) {
      const int g = (opaque(threadIdx.x) & 63) >> 4;
      const char *qr = row_at<IT>(qb, a.qs[1], q, g), *gr = row_at<GT>(gb, a.dos[1], q, g);
      const float s = dot_plain<D, IT>(qr, row_at<IT>(kb, a.ks[1], kc, g));
      const float p = fast_exp2(fmaf(s, a.scale_log2, -a.lse[((int64_t)b * a.Hq + h) * a.Lq + q]));
      if constexpr (PART == 1) {
        add_plain<D, GT>(acc, p, gr, on);
      } else {
        const float x = dot_vo<2, D, IT, GT>(HotRows{gr, row_at<IT>(vb, a.vs[1], kc, g),
                                                     ob + (of32 ? 4 : 2) * ((int64_t)q * a.os[1] + 4 * g), qr}, of32);
        add_plain<D, IT>(acc, p * x, qr, on);
      }
    }, [&] { return all_nan(acc); });
  }
}

// One walk: the streamed rows of step s are in LDS buffer s % NBUF when compute(s) runs.
// start(s, buf) issues their loads, finish(buf) writes what went through registers.
template <int NBUF, bool DMA, int BUF, class S, class F, class C>
__device__ __forceinline__ void walk_rows(int n, uint16_t* L, S&& start, F&& finish, C&& compute) {
  static_assert(!DMA || NBUF == 2, "");
  if (n > 0) start(0, L);
  for (int s = 0; s < n; ++s) {
    uint16_t* buf = L + (NBUF == 2 ? (s & 1) * BUF : 0);
    uint16_t* nxt = L + (NBUF == 2 ? ((s + 1) & 1) * BUF : 0);
    if constexpr (DMA) __builtin_amdgcn_s_waitcnt(0);  // this wave's loads of step s have landed
    if constexpr (NBUF == 1) __syncthreads();          // step s - 1 is consumed
    finish(s, buf);
    __syncthreads();  // every wave's part of step s is there (and, NBUF = 2, step s - 1 consumed)
    if (s + 1 < n) start(s + 1, nxt);
    compute(s, buf);
  }
}

template <int D, class IT, class OT, int NW, int MINW, int RES>
__global__ __attribute__((amdgpu_flat_work_group_size(64 * NW, 64 * NW), amdgpu_waves_per_eu(MINW, MINW)))
void fwd_s3(KArgs a) {
  constexpr int NTH = 64 * NW, NSUB = TILE / (16 * NW), NP = Pieces<IT>::n, NKD = D / 32, NMD = D / 16;
  using R = Rows<D, IT, NTH>;
  constexpr int BUF = 2 * R::ELTS, NBUF = R::DMA || 4 * BUF <= 56 * 1024 ? 2 : 1;
  __shared__ __attribute__((aligned(512))) uint16_t L[cmax(NBUF * BUF, NW * 16 * D * 2)];

  const Slot slot = launch_slot<NSUB, RES>(a);
  const int item = slot.ok ? a.q_order[slot.slot] : -1;
  if (item < 0 || item >= a.B * a.Hq * a.nqt) return;  // idle slot (or an entry out of range)
  const int qt = item % a.nqt, bh = item / a.nqt;
  const int h = bh % a.Hq, b = bh / a.Hq, hk = h / a.G;
  const int mrow = map_row(a, b, h, a.nqt, qt);
  Walk<BN> walk(a.row_ent, a.row_ptr[mrow], a.row_ptr[mrow + 1]);
  const int wrow = slot.part * 16 * NW;
  if (qt * TILE + wrow >= a.Lq) return;
  const int lane = threadIdx.x & 63, l16 = lane & 15, g = lane >> 4;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const uint32_t ra = row_addr<D>(l16, g), ta = tr_addr<D>(l16, g);
  const int qloc = wrow + 16 * wave + l16, q = qt * TILE + qloc;

  const char* kb = head_base(a.k, a.ks, b, hk, elt_bytes<IT>());
  const char* vb = head_base(a.v, a.vs, b, hk, elt_bytes<IT>());
  Frag<NP> qf[NKD];
  own16<D, IT>(qf, head_base(a.q, a.qs, b, h, elt_bytes<IT>()), a.qs[1], min(q, a.Lq - 1), g);
  f32x4 acc[NMD];
#pragma unroll
  for (int i = 0; i < NMD; ++i) acc[i] = f32x4{};
  float m = NEG_INF, l = 0.f;
  const float c2 = a.scale_log2, up = fminf(8.f / c2, 3.4e38f);  // (finite: -inf + up < any score)

  R ks, vs;
  walk_rows<NBUF, R::DMA, BUF>(walk.n, L,
      [&](int s, uint16_t* buf) {
        const int k0 = walk.first(s);
        ks.load(kb, a.ks[1], k0, a.Lk, buf);
        vs.load(vb, a.vs[1], k0, a.Lk, buf + R::ELTS);
      },
      [&](int, uint16_t* buf) {
        ks.store(buf);
        vs.store(buf + R::ELTS);
      },
      [&](int s, const uint16_t* Kl) {
        const uint16_t* Vl = Kl + R::ELTS;
        const int mask = walk.mask(s);
        uint32_t w = 0xffffffffu;
        if (mask >= 0) {
          w = bits32(a.row_bits, mask, s % Walk<BN>::SPT, qloc, g);
          if (!__any((w & 0x000f000fu) != 0)) return;  // no allowed key of the wave's rows here
        }
        f32x4 st[2];
        one_dot<2, fwd_chains<D>(), D, NP>(lds_addr(Kl) + ra, qf, st);
        if (mask >= 0) {
#pragma unroll
          for (int t = 0; t < 2; ++t)
#pragma unroll
            for (int r = 0; r < 4; ++r) st[t][r] = mask_neg_inf(st[t][r], ones16(w, t, r));
        }
        float mx = NEG_INF;
#pragma unroll
        for (int t = 0; t < 2; ++t)
#pragma unroll
          for (int r = 0; r < 4; ++r) mx = fmaxf(mx, st[t][r]);
        mx = wave_max32(wave_max16(mx));
        // the running max is raised only when a row's weights grow by more than 2^8
        if (__any(mx > m + up)) {
          const float mn = fmaxf(m, mx);
          const float alpha = (mn == NEG_INF) ? 1.f : fast_exp2((m - mn) * c2);
          l *= alpha;
#pragma unroll
          for (int i = 0; i < NMD; ++i) acc[i] *= alpha;
          m = mn;
        }
        const float mu = (m == NEG_INF) ? 0.f : m;
#pragma unroll
        for (int t = 0; t < 2; ++t)
#pragma unroll
          for (int r = 0; r < 4; ++r) {
            st[t][r] = fast_exp2((st[t][r] - mu) * c2);  // exactly 1 for the key that set m
            l += st[t][r];
          }
        add_rows<D, NP>(lds_addr(Vl) + ta, c_frag16(st[0], st[1]), acc);
      });

  l += __shfl_xor(l, 16);
  l = wave_sum32(l);
  float lse = l > 0.f ? fmaf(m, c2, __builtin_log2f(l)) : NEG_INF;
  if (not_finite(acc)) plain_fwd<D, IT>(args_again(), b, h, qt, wrow + 16 * wave, acc, l, lse);
  if (g == 0 && q < a.Lq) a.lse[((int64_t)b * a.Hq + h) * a.Lq + q] = lse;
  __syncthreads();  // every wave is done with the operand tiles
  const int r0 = qt * TILE + wrow + 16 * wave;
  put16<D, OT>(acc, l > 0.f ? 1.f / l : 0.f, (float*)L + wave * 16 * D, a.out,
               (int64_t)b * a.os[0] + (int64_t)r0 * a.os[1] + (int64_t)h * a.os[2], a.os[1], a.Lq - r0, lane);
}

template <int D, class IT, class OT, int NW, int MINW, int RES>
__global__ __attribute__((amdgpu_flat_work_group_size(64 * NW, 64 * NW), amdgpu_waves_per_eu(MINW, MINW)))
void bwd_dq_s3(KArgs a) {
  constexpr int NTH = 64 * NW, NSUB = TILE / (16 * NW), NP = Pieces<IT>::n, NG = Pieces<OT>::n;
  constexpr int NKD = D / 32, NMD = D / 16;
  using R = Rows<D, IT, NTH>;
  constexpr int BUF = 2 * R::ELTS, NBUF = R::DMA || 4 * BUF <= 56 * 1024 ? 2 : 1;
  __shared__ __attribute__((aligned(512))) uint16_t L[cmax(NBUF * BUF, NW * 16 * D * 2)];
  __shared__ HotList<HOT_Q> Hl[NW];

  const Slot slot = launch_slot<NSUB, RES>(a);
  const int item = slot.ok ? a.q_order[slot.slot] : -1;
  if (item < 0 || item >= a.B * a.Hq * a.nqt) return;  // idle slot (or an entry out of range)
  const int qt = item % a.nqt, bh = item / a.nqt;
  const int h = bh % a.Hq, b = bh / a.Hq, hk = h / a.G;
  const int mrow = map_row(a, b, h, a.nqt, qt);
  Walk<BN> walk(a.row_ent, a.row_ptr[mrow], a.row_ptr[mrow + 1]);
  const int wrow = slot.part * 16 * NW;
  if (qt * TILE + wrow >= a.Lq) return;
  const int lane = threadIdx.x & 63, l16 = lane & 15, g = lane >> 4;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const uint32_t ra = row_addr<D>(l16, g), ta = tr_addr<D>(l16, g);
  const int qloc = wrow + 16 * wave + l16, qc = min(qt * TILE + qloc, a.Lq - 1);

  const char* kb = head_base(a.k, a.ks, b, hk, elt_bytes<IT>());
  const char* vb = head_base(a.v, a.vs, b, hk, elt_bytes<IT>());
  Frag<NP> qf[NKD];
  Frag<NG> gf[NKD];
  own16<D, IT>(qf, head_base(a.q, a.qs, b, h, elt_bytes<IT>()), a.qs[1], qc, g);
  own16<D, OT>(gf, head_base(a.dO, a.dos, b, h, elt_bytes<OT>()), a.dos[1], qc, g);
  const int64_t rs = ((int64_t)b * a.Hq + h) * a.Lq + qc;
  const float lse = a.lse[rs], delta = a.delta[rs], c2 = a.scale_log2;
  if (lane < 16) Hl[wave].n[lane] = 0;
  f32x4 acc[NMD];
#pragma unroll
  for (int i = 0; i < NMD; ++i) acc[i] = f32x4{};

  R ks, vs;
  walk_rows<NBUF, R::DMA, BUF>(walk.n, L,
      [&](int s, uint16_t* buf) {
        const int k0 = walk.first(s);
        ks.load(kb, a.ks[1], k0, a.Lk, buf);
        vs.load(vb, a.vs[1], k0, a.Lk, buf + R::ELTS);
      },
      [&](int, uint16_t* buf) {
        ks.store(buf);
        vs.store(buf + R::ELTS);
      },
      [&](int s, const uint16_t* Kl) {
        const uint16_t* Vl = Kl + R::ELTS;
        const int mask = walk.mask(s), k0 = walk.first(s);
        uint32_t w = 0xffffffffu;
        if (mask >= 0) {
          w = bits32(a.row_bits, mask, s % Walk<BN>::SPT, qloc, g);
          if (!__any((w & 0x000f000fu) != 0)) return;
        }
        f32x4 st[2], dp[2];
        two_dots<D == 64 ? 2 : 1, bwd_chains<D, IT>(), D, NP, NP, NP, NG>(lds_addr(Kl) + ra, lds_addr(Vl) + ra, qf, gf, st, dp);
#pragma unroll
        for (int t = 0; t < 2; ++t)
#pragma unroll
          for (int r = 0; r < 4; ++r) st[t][r] = fast_exp2(fmaf(st[t][r], c2, -lse));
        if (mask >= 0) zero16(st, w);
#pragma unroll
        for (int t = 0; t < 2; ++t)
#pragma unroll
          for (int r = 0; r < 4; ++r) dp[t][r] -= delta;
        if (any_hot(st)) note_hot(st, dp, Hl[wave], k0);
#pragma unroll
        for (int t = 0; t < 2; ++t) dp[t] *= st[t];
        add_rows<D, NP>(lds_addr(Kl) + ta, c_frag16(dp[0], dp[1]), acc);
      });

  __syncthreads();
  const bool of32 = o_is_f32<OT>(a);
  add_hot<D, IT, OT>(acc, Hl[wave], l16, of32, [&](int key) {
    const KArgs& a = args_again();
    return HotRows{row_at<OT>(head_base(a.dO, a.dos, b, h, elt_bytes<OT>()), a.dos[1], qc, g),
                   row_at<IT>(vb, a.vs[1], key, g),
                   head_base(a.o, a.os, b, h, of32 ? 4 : 2) + (of32 ? 4 : 2) * ((int64_t)qc * a.os[1] + 4 * g),
                   row_at<IT>(kb, a.ks[1], key, g)};
  });
  if (not_finite(acc)) plain_dq<D, IT, OT>(args_again(), b, h, qt, wrow + 16 * wave, acc);
  const int r0 = qt * TILE + wrow + 16 * wave;
  put16<D, IT>(acc, a.scale, (float*)L + wave * 16 * D, a.dq,
               (int64_t)b * a.dqs[0] + (int64_t)r0 * a.dqs[1] + (int64_t)h * a.dqs[2], a.dqs[1], a.Lq - r0, lane);
}

// two LDS buffers where Q's rows are loaded to LDS directly, or they leave room for
// two workgroups a CU
template <int D, class IT, class OT>
constexpr int dkdv_bufs() {
  return 4 * (Pieces<IT>::n + Pieces<OT>::n) * BN * D <= (Pieces<IT>::n == 1 ? 158 : 56) * 1024 ? 2 : 1;
}

// PART: 3 = dV and dK; 1 = dV, 2 = dK: workgroups of their own at D = 256, where both
// accumulators, K and V would take 192 registers of a wave's 256 (S is then formed
// twice, 1/14 of the products).
template <int D, class IT, class OT, int PART, int NW>
__device__ __forceinline__ void dkdv_s3(const KArgs& a, uint16_t* L, float* Rl, HotList<HOT_K>* Hl, int sl, int sub) {
  constexpr bool DV = PART & 1, DK = PART & 2;
  constexpr int NTH = 64 * NW, NP = Pieces<IT>::n, NG = Pieces<OT>::n;
  constexpr int NKD = D / 32, NMD = D / 16;
  using Rq = Rows<D, IT, NTH>;
  using Rg = Rows<D, OT, NTH, true>;
  constexpr int BUF = Rq::ELTS + Rg::ELTS, NBUF = dkdv_bufs<D, IT, OT>();
  const int item = a.kv_order[sl];
  if (item < 0 || item >= a.B * a.Hkv * a.nkt) return;  // idle slot (or an entry out of range)
  const int kt = item % a.nkt, bh = item / a.nkt;
  const int hk = bh % a.Hkv, b = bh / a.Hkv;
  const int wrow = sub * 16 * NW;
  if (kt * TILE + wrow >= a.Lk) return;
  const int lane = threadIdx.x & 63, l16 = lane & 15, g = lane >> 4;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const uint32_t ra = row_addr<D>(l16, g), ta = tr_addr<D>(l16, g);
  const int kloc = wrow + 16 * wave + l16, kc = min(kt * TILE + kloc, a.Lk - 1);
  const float c2 = a.scale_log2;
  const bool of32 = o_is_f32<OT>(a);

  Frag<NP> kf[NKD], vf[DK ? NKD : 1];
  own16<D, IT>(kf, head_base(a.k, a.ks, b, hk, elt_bytes<IT>()), a.ks[1], kc, g);
  if constexpr (DK) own16<D, IT>(vf, head_base(a.v, a.vs, b, hk, elt_bytes<IT>()), a.vs[1], kc, g);
  f32x4 dk[DK ? NMD : 1], dv[DV ? NMD : 1];
#pragma unroll
  for (int i = 0; i < NMD; ++i) {
    if constexpr (DK) dk[i] = f32x4{};
    if constexpr (DV) dv[i] = f32x4{};
  }

  for (int gh = 0; gh < a.G; ++gh) {
    const int h = hk * a.G + gh;
    const int mc = map_row(a, b, h, a.nkt, kt);
    Walk<BN> walk(a.col_ent, a.col_ptr[mc], a.col_ptr[mc + 1]);
    const char* qb = head_base(a.q, a.qs, b, h, elt_bytes<IT>());
    const char* gb = head_base(a.dO, a.dos, b, h, elt_bytes<OT>());
    const int64_t rs = ((int64_t)b * a.Hq + h) * a.Lq;
    Rq rq;
    Rg rg;
    const auto hot_rows = [&](int key, int q, int g4) {
      const KArgs& a = args_again();
      const bool of32 = o_is_f32<OT>(a);
      return HotRows{row_at<OT>(head_base(a.dO, a.dos, b, h, elt_bytes<OT>()), a.dos[1], q, g4),
                     row_at<IT>(head_base(a.v, a.vs, b, hk, elt_bytes<IT>()), a.vs[1], key, g4),
                     head_base(a.o, a.os, b, h, of32 ? 4 : 2) + (of32 ? 4 : 2) * ((int64_t)q * a.os[1] + 4 * g4),
                     row_at<IT>(head_base(a.q, a.qs, b, h, elt_bytes<IT>()), a.qs[1], q, g4)};
    };
    if (DK && lane < 16) Hl[wave].n[lane] = 0;
    float rl = 0.f;  // lse (threads 0 .. BN - 1) or delta (the next BN) of a row
    __syncthreads();  // the previous head's last step is consumed
    walk_rows<NBUF, Rq::DMA || Rg::DMA, BUF>(walk.n, L,
        [&](int s, uint16_t* buf) {
          const int q0 = walk.first(s);
          rq.load(qb, a.qs[1], q0, a.Lq, buf);
          rg.load(gb, a.dos[1], q0, a.Lq, buf + Rq::ELTS);
          if (threadIdx.x < 2 * BN) {
            const int64_t r = rs + min(q0 + (int)(threadIdx.x % BN), a.Lq - 1);
            rl = threadIdx.x < BN ? a.lse[r] : a.delta[r];
          }
        },
        [&](int s, uint16_t* buf) {
          rq.store(buf);
          rg.store(buf + Rq::ELTS);
          if (threadIdx.x < 2 * BN) Rl[(NBUF == 2 ? s & 1 : 0) * 2 * BN + threadIdx.x] = rl;
        },
        [&](int s, const uint16_t* Ql) {
          const uint16_t* Gl = Ql + Rq::ELTS;
          const float* Rs = Rl + (NBUF == 2 ? s & 1 : 0) * 2 * BN + 4 * g;
          const int mask = walk.mask(s), q0 = walk.first(s);
          uint32_t w = 0xffffffffu;
          if (mask >= 0) {
            w = bits32(a.col_bits, mask, s % Walk<BN>::SPT, kloc, g);
            if (!__any((w & 0x000f000fu) != 0)) return;
          }
          f32x4 st[2], dp[2];
          if constexpr (!DK) one_dot<2, bwd_chains<D, IT>(), D, NP>(lds_addr(Ql) + ra, kf, st);
          else two_dots<D == 128 ? 1 : 2, bwd_chains<D, IT>(), D, NP, NP, NG, NP>(lds_addr(Ql) + ra, lds_addr(Gl) + ra, kf, vf, st, dp);
#pragma unroll
          for (int t = 0; t < 2; ++t) {
            const f32x4 ls = *(const f32x4*)(Rs + 16 * t), dl = *(const f32x4*)(Rs + BN + 16 * t);
#pragma unroll
            for (int r = 0; r < 4; ++r) {
              st[t][r] = fast_exp2(fmaf(st[t][r], c2, -ls[r]));
              if constexpr (DK) dp[t][r] -= dl[r];
            }
          }
          if (mask >= 0) zero16(st, w);
          if constexpr (DV) add_rows<D, NG>(lds_addr(Gl) + ta, c_frag16(st[0], st[1]), dv);
          if constexpr (DK) {
            if (any_hot(st))
              hot_rest<D, IT, OT>(dp, note_hot(st, dp, Hl[wave], q0), of32, [&](int own, int i, int g4) {
                return hot_rows(min(kt * TILE + wrow + 16 * wave + own, a.Lk - 1), min(q0 + i, a.Lq - 1), g4);
              });
#pragma unroll
            for (int t = 0; t < 2; ++t) dp[t] *= st[t];
          }
          if constexpr (DK) add_rows<D, NP>(lds_addr(Ql) + ta, c_frag16(dp[0], dp[1]), dk);
        });
    if constexpr (DK)
      add_hot<D, IT, OT>(dk, Hl[wave], l16, of32, [&](int q) { return hot_rows(kc, q, g); });
  }

  if constexpr (DV)
    if (not_finite(dv)) plain_dkdv<D, IT, OT, 1>(args_again(), b, hk, kt, wrow + 16 * wave, dv);
  if constexpr (DK)
    if (not_finite(dk)) plain_dkdv<D, IT, OT, 2>(args_again(), b, hk, kt, wrow + 16 * wave, dk);
  const int r0 = kt * TILE + wrow + 16 * wave;
  __syncthreads();
  if constexpr (DV)
    put16<D, IT>(dv, 1.f, (float*)L + wave * 16 * D, a.dv,
                 (int64_t)b * a.dvs[0] + (int64_t)r0 * a.dvs[1] + (int64_t)hk * a.dvs[2], a.dvs[1], a.Lk - r0, lane);
  if constexpr (DK)
    put16<D, IT>(dk, a.scale, (float*)L + wave * 16 * D, a.dk,
                 (int64_t)b * a.dks[0] + (int64_t)r0 * a.dks[1] + (int64_t)hk * a.dks[2], a.dks[1], a.Lk - r0, lane);
}

template <int D, class IT, class OT, int NW, int MINW, int RES>
__global__ __attribute__((amdgpu_flat_work_group_size(64 * NW, 64 * NW), amdgpu_waves_per_eu(MINW, MINW)))
void bwd_dkdv_s3(KArgs a) {
  constexpr int NBUF = dkdv_bufs<D, IT, OT>();
  constexpr int BUF = Rows<D, IT, 64 * NW>::ELTS + Rows<D, OT, 64 * NW>::ELTS;
  __shared__ __attribute__((aligned(512))) uint16_t L[cmax(NBUF * BUF, NW * 16 * D * 2)];
  __shared__ __attribute__((aligned(16))) float Rl[NBUF * 2 * BN];  // lse, delta of the step's rows
  __shared__ HotList<HOT_K> Hl[NW];
  constexpr int NPART = D == 256 ? 2 : 1;
  const Slot s = launch_slot<NPART * TILE / (16 * NW), RES>(a);
  if (!s.ok) return;
  if constexpr (NPART == 1) dkdv_s3<D, IT, OT, 3, NW>(a, L, Rl, Hl, s.slot, s.part);
  else if (s.part & 1) dkdv_s3<D, IT, OT, 1, NW>(a, L, Rl, Hl, s.slot, s.part >> 1);
  else dkdv_s3<D, IT, OT, 2, NW>(a, L, Rl, Hl, s.slot, s.part >> 1);
}

// delta = rowsum(dO * O), summed in float64: D / 8 threads a row, the rows in the
// order of memory (head fastest where a row of O holds all heads)
template <int D, class OT, class GT>
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
  const char* g = head_base(a.dO, a.dos, b, h, elt_bytes<GT>()) + elt_bytes<GT>() * ((int64_t)q * a.dos[1] + 8 * part);
  Raw8<OT> ro;
  Raw8<GT> rg;
  ro.load(o);
  rg.load(g);
  float x[8], y[8];
  ro.floats(x);
  rg.floats(y);
  double s = 0.;
#pragma unroll
  for (int e = 0; e < 8; ++e) s += (double)x[e] * (double)y[e];
#pragma unroll
  for (int m = 1; m < TPR; m <<= 1) s += __shfl_xor(s, m);
  if (part == 0) a.delta[((int64_t)b * a.Hq + h) * a.Lq + q] = (float)s;
}

// ---------------------------------------------------------------------------
// launchers
// ---------------------------------------------------------------------------

template <int NSUB, int NW, void (*K)(KArgs)>
void go(KArgs a, int grid, hipStream_t st) {
  a.n_slots = grid;
  hipLaunchKernelGGL(K, dim3((grid + 7) / 8 * 8 * NSUB), dim3(64 * NW), 0, st, a);
}

// <waves, waves per SIMD the registers are given for, workgroups resident on a CU>: two
// waves a SIMD where that spills nothing inside the walks, else one (a spill's reload
// also waits for the loads in flight: at D = 128 the float32 step took 697 us with 41
// spilled registers in dK/dV, 600 at one wave a SIMD).
template <int D, class IT, class OT, class GT = OT>
struct S3 {
  static constexpr int N = Pieces<IT>::n;
  template <int NW, int MINW, int RES>
  static void f(const KArgs& a, int grid, hipStream_t st) {
    go<TILE / (16 * NW), NW, fwd_s3<D, IT, OT, NW, MINW, RES>>(a, grid, st);
  }
  template <int NW, int MINW, int RES>
  static void q(const KArgs& a, int grid, hipStream_t st) {
    go<TILE / (16 * NW), NW, bwd_dq_s3<D, IT, GT, NW, MINW, RES>>(a, grid, st);
  }
  template <int NW, int MINW, int RES>
  static void kv(const KArgs& a, int grid, hipStream_t st) {
    go<(D == 256 ? 2 : 1) * TILE / (16 * NW), NW, bwd_dkdv_s3<D, IT, GT, NW, MINW, RES>>(a, grid, st);
  }
  static void fwd(const KArgs& a, int grid, hipStream_t st) {
    if constexpr (D == 64) f<4, 3, 3>(a, grid, st);
    else if constexpr (D == 128) f<4, 2, 2>(a, grid, st);
    else if constexpr (N == 1) f<4, 2, 2>(a, grid, st);
    else f<4, 1, 1>(a, grid, st);
  }
  static void bwd(const KArgs& a, int stage, int q_grid, int kv_grid, hipStream_t st) {
    if (stage == MATTN_BWD_PRE) {
      const int64_t threads = (int64_t)a.B * a.Hq * a.Lq * (D / 8);
      hipLaunchKernelGGL((delta_s3<D, OT, GT>), dim3((threads + 255) / 256), dim3(256), 0, st, a);
    } else if (stage == MATTN_BWD_DKDV) {
      if constexpr (D == 64) kv<4, 2, 2>(a, kv_grid, st);
      else if constexpr (D == 128) kv<4, 1, 1>(a, kv_grid, st);
      else if constexpr (N == 1) kv<8, 2, 1>(a, kv_grid, st);
      else kv<4, 1, 1>(a, kv_grid, st);
    } else {
      if constexpr (D == 64) q<4, 2, 2>(a, q_grid, st);
      else if constexpr (D == 128) q<8, 2, 1>(a, q_grid, st);
      else if constexpr (N == 1) q<4, 2, 2>(a, q_grid, st);
      else q<4, 1, 1>(a, q_grid, st);
    }
  }
};

// (16-bit inputs: the same-dtype O of the C interface, a float32 O, and a float32 O
// whose gradient is 16-bit)
template <class Tag, class F>
void dispatch16(bool of32, bool do16, F&& f) {
  if (!of32) f(S3<256, Tag, Tag>{});
  else if (do16) f(S3<256, Tag, float, Tag>{});
  else f(S3<256, Tag, float>{});
}
template <class F>
hipError_t dispatch(const KArgs& a, int D, int dtype, int o_dtype, F&& f) {
  const bool of32 = o_dtype == MATTN_F32;
  if (dtype == MATTN_F32) {
    if (D == 64) f(S3<64, float, float>{});
    else if (D == 128) f(S3<128, float, float>{});
    else f(S3<256, float, float>{});
  } else if (dtype == MATTN_BF16) {
    dispatch16<bf16_tag>(of32, a.do16, f);
  } else {
    dispatch16<f16_tag>(of32, a.do16, f);
  }
  return hipGetLastError();
}

}  // namespace

bool s3_path(int D, int dtype, bool precise) {
  return !precise && (dtype == MATTN_F32 ? D <= 256 : D == 256);
}

hipError_t launch_fwd_s3(const KArgs& a, int D, int dtype, int o_dtype, int grid, hipStream_t st) {
  return dispatch(a, D, dtype, o_dtype, [&](auto s) { decltype(s)::fwd(a, grid, st); });
}

hipError_t launch_bwd_s3(const KArgs& a, int D, int dtype, int o_dtype, int stage, int q_grid, int kv_grid,
                         hipStream_t st) {
  return dispatch(a, D, dtype, o_dtype, [&](auto s) { decltype(s)::bwd(a, stage, q_grid, kv_grid, st); });
}

}  // namespace mattn
