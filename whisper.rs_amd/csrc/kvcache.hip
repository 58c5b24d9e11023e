// K3: device KV arena kernels (the storage side of
// crates/whisper/src/decoder.rs:131-264 DecoderKvCache).
//
// The arena keeps planes of [ctx][64] per (layer, slot, head) for
// self-attention and per (layer, head) for cross-attention, in f16 (default)
// or f32. These kernels convert or copy the decoder's f32 projection rows into
// that layout and move rows within / between planes; the row moves see an
// f32 row as two f16-sized rows.
#include "wrs_internal.hpp"

#include <algorithm>

namespace wrs {
namespace {

typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef _Float16 f16x8 __attribute__((ext_vector_type(8)));
typedef float f32x8 __attribute__((ext_vector_type(8)));
typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));

// K (blockIdx.y == 0) and V rows in one launch: a step's append is bound by its
// launches (five slots of a 12-layer step: 120 -> 60, ~2 us each).
// One thread per 8 values: row i, head h, 8-column group c. The source rows need
// only 4-byte alignment.
__global__ void kv_write_rows(KvRows rows, int64_t src_rs, int n, int n_heads, int64_t dst_hs,
                              int pos) {
  const int64_t t = static_cast<int64_t>(blockIdx.x) * blockDim.x + threadIdx.x;
  const int64_t total = static_cast<int64_t>(n) * n_heads * 8;
  if (t >= total) return;
  const float* src = blockIdx.y ? rows.v_src : rows.k_src;
  _Float16* dst = static_cast<_Float16*>(blockIdx.y ? rows.v_dst : rows.k_dst);
  const int c = static_cast<int>(t & 7);
  const int64_t ih = t >> 3;
  const int h = static_cast<int>(ih % n_heads);
  const int i = static_cast<int>(ih / n_heads);
  const float* s = src + static_cast<int64_t>(i) * src_rs + h * 64 + c * 8;
  f32x8 x;
#pragma unroll
  for (int e = 0; e < 8; ++e) x[e] = s[e];
  const f16x8 y = __builtin_convertvector(x, f16x8);
  *reinterpret_cast<f16x8*>(dst + h * dst_hs + static_cast<int64_t>(pos + i) * 64 + c * 8) = y;
}

// f32 planes: one thread per 4 values (row i, head h, 4-column group c). The
// source rows need only 4-byte alignment; the plane rows are 256-byte aligned.
__global__ void kv_write_rows_f32(KvRows rows, int64_t src_rs, int n, int n_heads, int64_t dst_hs,
                                  int pos) {
  const int64_t t = static_cast<int64_t>(blockIdx.x) * blockDim.x + threadIdx.x;
  const int64_t total = static_cast<int64_t>(n) * n_heads * 16;
  if (t >= total) return;
  const float* src = blockIdx.y ? rows.v_src : rows.k_src;
  float* dst = static_cast<float*>(blockIdx.y ? rows.v_dst : rows.k_dst);
  const int c = static_cast<int>(t & 15);
  const int64_t ih = t >> 4;
  const int h = static_cast<int>(ih % n_heads);
  const int i = static_cast<int>(ih / n_heads);
  const float* s = src + static_cast<int64_t>(i) * src_rs + h * 64 + c * 4;
  const f32x4 x = {s[0], s[1], s[2], s[3]};
  *reinterpret_cast<f32x4*>(dst + h * dst_hs + static_cast<int64_t>(pos + i) * 64 + c * 4) = x;
}

// One workgroup per plane. Rows move down in blocks of 32 rows (256 threads x
// 8 halves); every block is read before any thread writes it, and later blocks
// only read rows above everything written so far, so the in-place move is safe
// for any drop >= 1.
__global__ __launch_bounds__(256) void kv_slide(_Float16* k, _Float16* v, int64_t layer_stride,
                                                int64_t plane_stride, int len, int drop) {
  _Float16* p = (blockIdx.z ? v : k) + blockIdx.y * layer_stride + blockIdx.x * plane_stride;
  const int keep = len - drop;
  const int tid = threadIdx.x;
  for (int r0 = 0; r0 < keep; r0 += 32) {
    const int r = r0 + (tid >> 3);
    const int c = (tid & 7) * 8;
    u32x4 v = {0, 0, 0, 0};
    if (r < keep) v = *reinterpret_cast<const u32x4*>(p + static_cast<int64_t>(r + drop) * 64 + c);
    __syncthreads();
    if (r < keep) *reinterpret_cast<u32x4*>(p + static_cast<int64_t>(r) * 64 + c) = v;
    __syncthreads();
  }
}

// Copy rows [0, len) of every (layer, head) plane of K and V from one slot to
// another. A workgroup takes pieces of kCopyUnits 16-byte units, every parts-th,
// each read whole before it is written (one that walked a whole plane 4 KB at a
// time waited out a round trip for each). K and V in one launch, us, before / now: 12
// layers x 12 heads x 64 rows 4.0/2.5, 224 rows 6.0/3.6; 32 x 20 x 448 23.1/22.3.
constexpr int kCopyUnits = 1024;
constexpr int kCopyParts = 32767;  // of a plane, at most: K's and V's share a grid dimension
__global__ __launch_bounds__(256) void kv_copy_planes(const _Float16* k_src, _Float16* k_dst,
                                                      const _Float16* v_src, _Float16* v_dst,
                                                      int64_t layer_stride, int64_t plane_stride,
                                                      int len, int parts) {
  const int which = blockIdx.z / parts, part = blockIdx.z - which * parts;
  const int64_t off = blockIdx.y * layer_stride + blockIdx.x * plane_stride;
  const u32x4* s = reinterpret_cast<const u32x4*>((which ? v_src : k_src) + off);
  u32x4* d = reinterpret_cast<u32x4*>((which ? v_dst : k_dst) + off);
  const int64_t n = static_cast<int64_t>(len) * 8;  // 16-byte units
  for (int64_t i0 = static_cast<int64_t>(part) * kCopyUnits; i0 < n;
       i0 += static_cast<int64_t>(parts) * kCopyUnits) {
    u32x4 x[kCopyUnits / 256];
#pragma unroll
    for (int u = 0; u < kCopyUnits / 256; ++u) {
      const int64_t i = i0 + 256 * u + threadIdx.x;
      x[u] = s[i < n ? i : 0];
    }
#pragma unroll
    for (int u = 0; u < kCopyUnits / 256; ++u) {
      const int64_t i = i0 + 256 * u + threadIdx.x;
      if (i < n) d[i] = x[u];
    }
  }
}

// Zero fill of a strided [batch][head][row][cols] f32 region (replaces
// memset nodes, which must not be recorded into captured graphs): one thread
// per value.
__global__ __launch_bounds__(256) void fill_zero_rows(float* base, int64_t bs, int64_t hs,
                                                      int64_t rs, int n_heads, int n_rows,
                                                      int cols) {
  const int64_t t = static_cast<int64_t>(blockIdx.x) * blockDim.x + threadIdx.x;
  const int64_t per_batch = static_cast<int64_t>(n_heads) * n_rows * cols;
  const int b = static_cast<int>(blockIdx.y);
  if (t >= per_batch) return;
  const int c = static_cast<int>(t % cols);
  const int64_t hr = t / cols;
  const int r = static_cast<int>(hr % n_rows);
  const int h = static_cast<int>(hr / n_rows);
  base[b * bs + h * hs + r * rs + c] = 0.f;
}

__global__ __launch_bounds__(256) void fill_zero_u32(unsigned* p, int64_t n) {
  const int64_t t = static_cast<int64_t>(blockIdx.x) * blockDim.x + threadIdx.x;
  if (t < n) p[t] = 0u;
}

}  // namespace

hipError_t launch_fill_zero_rows(float* base, int64_t bs, int64_t hs, int64_t rs, int batch,
                                 int n_heads, int n_rows, int cols, hipStream_t s) {
  if (batch <= 0 || n_heads <= 0 || n_rows <= 0 || cols <= 0) return hipSuccess;
  if (batch > 65535) return hipErrorInvalidConfiguration;
  const int64_t per_batch = static_cast<int64_t>(n_heads) * n_rows * cols;
  const int64_t blocks = (per_batch + 255) / 256;
  if (blocks > 0x7fffffff) return hipErrorInvalidConfiguration;
  hipLaunchKernelGGL(fill_zero_rows, dim3(static_cast<unsigned>(blocks), batch), dim3(256), 0, s,
                     base, bs, hs, rs, n_heads, n_rows, cols);
  return hipGetLastError();
}

hipError_t launch_fill_zero_u32(unsigned* p, int64_t n, hipStream_t s) {
  if (n <= 0) return hipSuccess;
  const int64_t blocks = (n + 255) / 256;
  if (blocks > 0x7fffffff) return hipErrorInvalidConfiguration;
  hipLaunchKernelGGL(fill_zero_u32, dim3(static_cast<unsigned>(blocks)), dim3(256), 0, s, p, n);
  return hipGetLastError();
}

hipError_t launch_kv_write_rows(const KvRows& rows, bool f32, int64_t src_rs, int n, int n_heads,
                                int64_t dst_hs, int pos, hipStream_t s) {
  const int64_t total = static_cast<int64_t>(n) * n_heads * (f32 ? 16 : 8);
  if (total <= 0) return hipSuccess;
  const int64_t blocks = (total + 255) / 256;
  if (blocks > 0x7fffffff) return hipErrorInvalidConfiguration;
  const dim3 grid(static_cast<unsigned>(blocks), 2);
  if (f32)
    hipLaunchKernelGGL(kv_write_rows_f32, grid, dim3(256), 0, s, rows, src_rs, n, n_heads, dst_hs, pos);
  else
    hipLaunchKernelGGL(kv_write_rows, grid, dim3(256), 0, s, rows, src_rs, n, n_heads, dst_hs, pos);
  return hipGetLastError();
}

hipError_t launch_kv_slide(_Float16* k, _Float16* v, int64_t layer_stride, int64_t plane_stride,
                           int n_layers, int n_heads, int len, int drop, hipStream_t s) {
  if (n_layers <= 0 || n_heads <= 0 || drop <= 0 || len <= drop) return hipSuccess;
  hipLaunchKernelGGL(kv_slide, dim3(n_heads, n_layers, 2), dim3(256), 0, s, k, v, layer_stride,
                     plane_stride, len, drop);
  return hipGetLastError();
}

hipError_t launch_kv_copy_planes(const _Float16* k_src, _Float16* k_dst, const _Float16* v_src,
                                 _Float16* v_dst, int64_t layer_stride, int64_t plane_stride,
                                 int n_layers, int n_heads, int len, hipStream_t s) {
  if (n_layers <= 0 || n_heads <= 0 || len <= 0) return hipSuccess;
  const int64_t pieces = (static_cast<int64_t>(len) * 8 + kCopyUnits - 1) / kCopyUnits;
  const int parts = static_cast<int>(std::min<int64_t>(pieces, kCopyParts));
  hipLaunchKernelGGL(kv_copy_planes, dim3(n_heads, n_layers, static_cast<unsigned>(2 * parts)),
                     dim3(256), 0, s, k_src, k_dst, v_src, v_dst, layer_stride, plane_stride, len,
                     parts);
  return hipGetLastError();
}

}  // namespace wrs
