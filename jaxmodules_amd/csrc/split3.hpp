// Products of float32 accuracy on the bfloat16 matrix cores, for the problems
// that hold their operands in float32: float32 inputs, and the weights, dS and
// dO of 16-bit inputs at the head dimensions the float16-operand kernels do
// not serve.
//
// A float32 value is the exact sum of three bfloat16 pieces (8 significant
// bits each, rounded to nearest, so of either sign), with float32's own
// exponent range: no scales, and nothing to bound beforehand.  (At its ends:
// below 2^-110 the last pieces are lost to the subnormals; infinities and what
// rounds past bfloat16's largest value have no such pieces and leave Inf or NaN
// in the products, which the kernels look for and form anew.)  A float16 value
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

// 8 consecutive elements as loaded, and their pieces
template <class T>
struct Raw8 {
  u32x4 x;
  __device__ __forceinline__ void load(const char* p) { x = *(const u32x4*)p; }
  __device__ __forceinline__ void floats(float* f) const {
#pragma unroll
    for (int e = 0; e < 8; ++e) f[e] = Elt<T>::to_f32(elt16(x, e));
  }
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
  __device__ __forceinline__ void floats(float* f) const {
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      f[e] = x[e];
      f[4 + e] = y[e];
    }
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

// f(c, p, off) for this thread's chunks c of ROWS rows from r0 of a [rows, D] tensor:
// p + off is the start of row r0 + threadIdx / CPR + c RPC (rows past n - 1 are row
// n - 1: their scores are masked).  p is uniform and off 32 bits a lane, formed anew
// each time (opaque: hoisted 64-bit addresses, two registers a chunk, spilled the
// kernels): 64-bit row products were 80 vector instructions a step.  The validated
// strides (Q, K, V: 128 rows within 2^31 elements, so 64 rows of float32 within 2^32
// bytes) fit, unsigned; WIDE (dO, not validated) takes
// 64-bit offsets when its stride needs them.
template <int D, int ES, int ROWS, int NTH, bool WIDE, class F>
__device__ __forceinline__ void each_chunk(const char* base, int64_t rs, int r0, int n, F&& f) {
  constexpr int CPR = D / 8, RPC = NTH / CPR, CH = ROWS / RPC;  // rows a chunk step covers
  static_assert(NTH % CPR == 0 && ROWS % RPC == 0, "whole rows a step");
  const int first = min(r0, n - 1), last = n - 1 - first;
  const char* p = base + ES * ((int64_t)first * rs);
  const int r = opaque(threadIdx.x / CPR);
  if (!WIDE || rs < (1 << 24)) {
#pragma unroll
    for (int c = 0; c < CH; ++c) f(c, p, (uint32_t)min(r + c * RPC, last) * (uint32_t)(ES * (int)rs));
  } else {
#pragma unroll
    for (int c = 0; c < CH; ++c) f(c, p + ES * ((int64_t)min(r + c * RPC, last) * rs), 0u);
  }
}

// ---- operand reads pipelined by hand ----------------------------------------------
// The compiler keeps few LDS reads in flight and waits for each before its MFMAs, so
// that a step's reads cost their latency one by one.  pipe() issues the reads of step
// i + PF (asm, in order: common.hpp) ahead of the MFMAs of step i and waits for just
// those that step i uses.

// a transposed operand as its two 4-row reads leave it (joined after the wait)
template <int N>
struct Tr { u32x2 lo[N], up[N]; };

// pieces at LDS byte address x + OFF + i PL
template <int OFF, int PL, int N>
__device__ __forceinline__ void rd(Frag<N>& f, uint32_t x) {
  static_for<N>([&](auto ic) {
    constexpr int i = decltype(ic)::value;
    f.p[i] = ds_read128<OFF + i * PL>(x);
  });
}
template <int OFF, int PL, int N>
__device__ __forceinline__ void rd(Tr<N>& f, uint32_t x0, uint32_t x1) {
  static_for<N>([&](auto ic) {
    constexpr int i = decltype(ic)::value;
    f.lo[i] = ds_read_tr8<OFF + i * PL>(x0);
    f.up[i] = ds_read_tr8<OFF + i * PL>(x1);
  });
}
template <int N>
__device__ __forceinline__ void landed(Frag<N>& f) {
#pragma unroll
  for (int i = 0; i < N; ++i) hold(f.p[i]);
}
template <int N>
__device__ __forceinline__ Frag<N> landed(Tr<N>& t) {
  Frag<N> f;
#pragma unroll
  for (int i = 0; i < N; ++i) {
    hold(t.lo[i]);
    hold(t.up[i]);
    f.p[i] = u32x4{t.lo[i][0], t.lo[i][1], t.up[i][0], t.up[i][1]};
  }
  return f;
}

// the steps to read ahead: `want`, or as many as lgkmcnt can count (15 reads)
constexpr int ahead(int want, int rps) { return want * rps <= 15 ? want : 15 / rps; }
// N steps of RPS reads each, PF steps ahead: rd(step, slot), use(step, slot), both with
// compile-time arguments, slot = step % (PF + 1)
template <int N, int PF, int RPS, class R, class U>
__device__ __forceinline__ void pipe(R&& read, U&& use) {
  static_for<(PF < N ? PF : N)>([&](auto ic) { read(ic, std::integral_constant<int, decltype(ic)::value % (PF + 1)>{}); });
  static_for<N>([&](auto ic) {
    constexpr int i = decltype(ic)::value;
    if constexpr (i + PF < N)
      read(std::integral_constant<int, i + PF>{}, std::integral_constant<int, (i + PF) % (PF + 1)>{});
    lgkm_wait<RPS * (i + PF < N ? PF : N - 1 - i)>();
    use(ic, std::integral_constant<int, i % (PF + 1)>{});
    __builtin_amdgcn_sched_barrier(0);
  });
}

// the n-th piece product (i, j), i + j <= 2, of NA x NB pieces, small ones first (n < products())
constexpr int products(int na, int nb) {
  int c = 0;
  for (int i = 0; i < na; ++i)
    for (int j = 0; j < nb; ++j) c += i + j <= 2;
  return c;
}
constexpr int product_ij(int na, int nb, int n) {  // 4 i + j
  for (int s = 2; s >= 0; --s)
    for (int i = 0; i < na; ++i) {
      const int j = s - i;
      if (j < 0 || j >= nb) continue;
      if (n-- == 0) return 4 * i + j;
    }
  return 0;
}
__device__ __forceinline__ void mfma1(u32x4 a, u32x4 b, f32x4& c) {
  c = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, a), __builtin_bit_cast(bf16x8, b), c, 0, 0, 0);
}
// c += a b and c2 += a2 b2, their products in turn (an MFMA that adds to the result of
// the one before it waits for it)
template <int NA, int NB, int NC, int ND, class C>
__device__ __forceinline__ void mma_two(const Frag<NA>& a, const Frag<NB>& b, C& c, const Frag<NC>& a2,
                                        const Frag<ND>& b2, C& c2) {
  constexpr int P1 = products(NA, NB), P2 = products(NC, ND);
  static_for<(P1 > P2 ? P1 : P2)>([&](auto nc) {
    constexpr int n = decltype(nc)::value;
    if constexpr (n < P1) {
      constexpr int ij = product_ij(NA, NB, n);
      mfma1(a.p[ij / 4], b.p[ij % 4], c);
    }
    if constexpr (n < P2) {
      constexpr int ij = product_ij(NC, ND, n);
      mfma1(a2.p[ij / 4], b2.p[ij % 4], c2);
    }
  });
}

// Launch slot and part of this workgroup, for kernels that cut a slot of the launch
// order into NPART workgroups.  The parts of slot s stay on the XCD s % 8 the order
// means it for (workgroup i runs on XCD i % 8), in the order's sequence.  When all of
// an XCD's workgroups start at once (up to RES on each of its 32 CUs), every second
// round of 32 is taken backwards: the order is longest first, so a CU then gets a long
// and a short row instead of two of the same rank.
struct Slot {
  int slot, part;
  bool ok;
};
template <int NPART, int RES>
__device__ __forceinline__ Slot launch_slot(const KArgs& a) {
  const int x = blockIdx.x & 7, R = gridDim.x >> 3;
  int r = blockIdx.x >> 3;
  if (R <= 32 * RES && (r & 32)) {
    const int r0 = r & ~31;
    r = r0 + min(32, R - r0) - 1 - (r & 31);
  }
  const int s = (r / NPART) * 8 + x;
  return {s, r % NPART, s < a.n_slots};
}

// base address of (b, h) in a tensor of element strides s
__device__ __forceinline__ const char* head_base(const void* p, const int64_t* s, int b, int h, int es) {
  return (const char*)p + es * ((int64_t)b * s[0] + (int64_t)h * s[2]);
}

// Sub-blocks of the walk over entries [e0, e1): SPT = 128 / BN per tile.  The entries
// are held 64 at a time, one per lane, and read back at a wave-uniform index: a load
// per step would cost its latency before the step's own loads can start.
template <int BN>
struct Walk {
  static constexpr int SPT = TILE / BN;
  const int* ent;
  int e0, n, base, tile, mk;
  __device__ __forceinline__ Walk(const int* ent_, int e0_, int e1) : ent(ent_), e0(e0_), n((e1 - e0_) * SPT) {
    if (n > 0) fill(0);
  }
  __device__ __forceinline__ void fill(int i) {
    base = i;
    const int e = e0 + min(i + (int)(threadIdx.x & 63), n / SPT - 1);
    // waited for here: left to where they are next read, the wait stands in every step's
    // way, and for the rows it has in flight too (float32 step 330 -> 360 us)
    tile = opaque(ent[2 * e]);
    mk = opaque(ent[2 * e + 1]);
  }
  __device__ __forceinline__ int at(int i) {  // index of entry i in the window
    if (i < base || i >= base + 64) fill(i);  // (uniform)
    return i - base;
  }
  // (at() first, in a statement of its own: it may replace the window that is then read)
  __device__ __forceinline__ int first(int s) {
    const int i = at(s / SPT);
    return __builtin_amdgcn_readlane(tile, i) * TILE + (s % SPT) * BN;
  }
  __device__ __forceinline__ int mask(int s) {
    const int i = at(s / SPT);
    return __builtin_amdgcn_readlane(mk, i);
  }
};

}  // namespace s3
}  // namespace mattn
