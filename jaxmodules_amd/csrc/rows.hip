// Row copies between tensors of different row lengths and types (mattn_copy_rows): the
// host pads head dimensions to 64, 128, 256 or 512 columns with them and takes the
// gradients' columns back.  One launch for all tensors of a call: as framework
// operations (a fill and a copy per tensor, and their gradients) the padding of a
// [2, 1000 / 1511, 12, 80] float16 step was 13 launches, 60 us of its 230 us of kernels,
// and as much again on the host.
//
// Bound by HBM: one thread per 8 destination columns, consecutive threads along a row,
// 16-byte accesses where lengths and addresses allow them (decided per tensor on the
// host).
#include "common.hpp"

namespace mattn {

constexpr int kMaxCopies = 4;

struct CopyArgs {
  mattn_row_copy c[kMaxCopies];
  int vec[kMaxCopies];      // 1: chunks of 8 columns are whole and 16-byte aligned on both sides
  int chunks[kMaxCopies];   // 8-column chunks per destination row
};

__device__ __forceinline__ float load1(const char* p, int dt) {
  if (dt == MATTN_F32) return *(const float*)p;
  const uint32_t x = *(const uint16_t*)p;
  return dt == MATTN_BF16 ? Elt<bf16_tag>::to_f32(x) : Elt<f16_tag>::to_f32(x);
}
__device__ __forceinline__ uint32_t pack(float x, float y, int dt) {
  return dt == MATTN_BF16 ? Elt<bf16_tag>::pack2(x, y) : Elt<f16_tag>::pack2(x, y);
}

__global__ __attribute__((amdgpu_flat_work_group_size(256, 256)))
void copy_rows(CopyArgs a) {
  const mattn_row_copy& c = a.c[blockIdx.y];
  const int cpr = a.chunks[blockIdx.y];
  const int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x;
  const int64_t row = i / cpr;
  const int col = 8 * (int)(i % cpr);
  if (row >= (int64_t)c.n[0] * c.n[1] * c.n[2]) return;
  const int64_t i2 = row % c.n[2], i1 = (row / c.n[2]) % c.n[1], i0 = row / ((int64_t)c.n[2] * c.n[1]);
  const int es = c.src_dtype == MATTN_F32 ? 4 : 2, ed = c.dst_dtype == MATTN_F32 ? 4 : 2;
  const char* s = (const char*)c.src + es * (i0 * c.src_stride[0] + i1 * c.src_stride[1] + i2 * c.src_stride[2] + col);
  char* d = (char*)c.dst + ed * (i0 * c.dst_stride[0] + i1 * c.dst_stride[1] + i2 * c.dst_stride[2] + col);
  const bool vec = a.vec[blockIdx.y];
  if (vec && c.src_dtype == c.dst_dtype) {  // bits as they are
    u32x4 x = {0u, 0u, 0u, 0u}, y = {0u, 0u, 0u, 0u};
    if (col < c.src_cols) {
      x = *(const u32x4*)s;
      if (es == 4) y = *(const u32x4*)(s + 16);
    }
    *(u32x4*)d = x;
    if (es == 4) *(u32x4*)(d + 16) = y;
    return;
  }
  float v[8];
#pragma unroll
  for (int e = 0; e < 8; ++e) v[e] = col + e < c.src_cols ? load1(s + es * e, c.src_dtype) : 0.f;
  if (vec) {
    if (ed == 4) {
      *(f32x4*)d = f32x4{v[0], v[1], v[2], v[3]};
      *(f32x4*)(d + 16) = f32x4{v[4], v[5], v[6], v[7]};
    } else {
      *(u32x4*)d = u32x4{pack(v[0], v[1], c.dst_dtype), pack(v[2], v[3], c.dst_dtype), pack(v[4], v[5], c.dst_dtype),
                         pack(v[6], v[7], c.dst_dtype)};
    }
    return;
  }
#pragma unroll
  for (int e = 0; e < 8; ++e) {
    if (col + e >= c.dst_cols) return;
    if (c.src_dtype == c.dst_dtype && es == 2) {  // bits as they are
      *(uint16_t*)(d + 2 * e) = col + e < c.src_cols ? *(const uint16_t*)(s + 2 * e) : (uint16_t)0;
    } else if (ed == 4) {
      *(float*)(d + 4 * e) = v[e];
    } else {
      *(uint16_t*)(d + 2 * e) = (uint16_t)(pack(v[e], 0.f, c.dst_dtype) & 0xffffu);
    }
  }
}

}  // namespace mattn

using namespace mattn;

extern "C" int mattn_copy_rows(const mattn_row_copy* copies, int32_t n, void* stream) {
  if (!copies) return MATTN_ERR_NULL;
  if (n <= 0 || n > kMaxCopies) return MATTN_ERR_SHAPE;
  CopyArgs a{};
  int64_t most = 0;
  for (int k = 0; k < n; ++k) {
    const mattn_row_copy& c = copies[k];
    if (!c.src || !c.dst) return MATTN_ERR_NULL;
    for (int dt : {c.src_dtype, c.dst_dtype})
      if (dt != MATTN_BF16 && dt != MATTN_F16 && dt != MATTN_F32) return MATTN_ERR_DTYPE;
    if (c.src_cols <= 0 || c.dst_cols <= 0) return MATTN_ERR_SHAPE;
    const int es = c.src_dtype == MATTN_F32 ? 4 : 2, ed = c.dst_dtype == MATTN_F32 ? 4 : 2;
    bool vec = (c.src_cols % 8 == 0 || c.dst_cols <= c.src_cols) && c.dst_cols % 8 == 0 &&
               ((uintptr_t)c.src & 15u) == 0 && ((uintptr_t)c.dst & 15u) == 0;
    for (int i = 0; i < 3; ++i) {
      if (c.n[i] <= 0 || c.src_stride[i] < 0 || c.dst_stride[i] < 0) return MATTN_ERR_SHAPE;
      vec = vec && (c.src_stride[i] * es) % 16 == 0 && (c.dst_stride[i] * ed) % 16 == 0;
    }
    a.c[k] = c;
    a.vec[k] = vec;
    a.chunks[k] = (c.dst_cols + 7) / 8;
    const int64_t threads = (int64_t)c.n[0] * c.n[1] * c.n[2] * a.chunks[k];
    most = threads > most ? threads : most;
  }
  const int64_t blocks = (most + 255) / 256;
  if (blocks > (1ll << 31) - 1) return MATTN_ERR_TOO_LARGE;
  hipLaunchKernelGGL(copy_rows, dim3((uint32_t)blocks, n), dim3(256), 0, (hipStream_t)stream, a);
  return hipGetLastError() == hipSuccess ? MATTN_OK : MATTN_ERR_LAUNCH;
}
