// Prompt rows over the f16 KV cache: several query rows of one slot or utterance
// against one layer's planes.
//
// K10 (attend_rows): flash attention of f32 query rows over [key][64] f16 planes
//   (replaces, for more than one row, the attention calls of
//   crates/whisper/src/decoder.rs:613-647 with a causal offset, and of
//   decoder.rs:698-708 over the encoder's keys). One workgroup of 4 or 8 waves
//   runs 32 query rows of one head; wave w takes the block's 32-key steps w, w +
//   waves, ... with its own online softmax, and the waves merge their (max, sum,
//   O) in LDS.
//   The arithmetic runs on the f16 matrix pipe with split operands: each query
//   row, times scale * log2(e) and a power of two that puts its largest element
//   into [2^14, 2^15), is split into kParts f16 parts, and so are the softmax
//   weights in units of 2^-15. Two parts in one unit (cross-attention, as the
//   split-K decode) carry 2^-22 of every query element and weight within 2^-18 of
//   the row's largest, and smaller ones to 2^-40 of it, where f16 ends. Three parts
//   (the cached self-attention, whose rows the f32 kernel ran before), each in a unit
//   2^-11 of the one before and with an accumulator of its own, carry all 24 bits down
//   to 2^-28, and smaller ones to 2^-60.
//   S^T = K Q^T puts one query per lane, and the packed weights are the B operand
//   of O^T += V^T P^T as they stand; K comes from memory in operand layout, V
//   passes through a wave's own swizzled LDS rows and is read transposed
//   (ds_read_b64_tr_b16). The next step's K and V load under the current one.
//   Bound by latency: launch, first loads, then ~1 us a step on few CUs, merge.
//   Dealing a block's steps over several workgroups that merge through memory
//   cost as much as it saved (128 rows x 1500 keys: 15.0 us in three).
//   Measured, 20 heads, queued back to back: 128 rows x 1500 keys 32.5 -> 14.2 us
//   (groups of 8 rows each read the planes again: 123 MB of L2 reads); 37 cached self
//   rows 14.5 -> 5.4 us, 224 rows past 220 37.9 -> 9.4 (f32 matrix pipe, element
//   loads). Weights in units of 1 and three parts in one unit took 14.1, 5.4 and 8.9
//   us, but a weight 2^-20 of the largest kept four bits; two parts in units of their
//   own 16.2.
#include "prefill_f32_block.hpp"

namespace wrs {
namespace {

typedef _Float16 f16x8 __attribute__((ext_vector_type(8)));
typedef _Float16 f16x2 __attribute__((ext_vector_type(2)));
typedef short s16x4 __attribute__((ext_vector_type(4)));
typedef float f32x16 __attribute__((ext_vector_type(16)));
typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef float f32x4u __attribute__((ext_vector_type(4), aligned(4)));
typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
typedef uint32_t u32x2 __attribute__((ext_vector_type(2)));
typedef __attribute__((address_space(3))) s16x4 lds_s16x4;

constexpr int kQ = 32;               // query rows per block
constexpr int kN = 32;               // keys per step
constexpr float kWeightUp = 0x1p15f;  // softmax weights, at most 1, are split in units of its inverse
constexpr int kPitch = 66;           // LDS pitch (floats) of a merge row
constexpr int kRawBuffer = 0x00020000;  // buffer resource word 3: raw, 32-bit data format

__device__ inline float pow2(int e) { return __builtin_bit_cast(float, (e + 127) << 23); }
__device__ inline int clamp_exp(int e) { return e < -126 ? -126 : (e > 127 ? 127 : e); }
__device__ inline float pair_max(float x) { return fmaxf(x, __shfl_xor(x, 32)); }

// 16-byte chunk c of V row r (128 bytes) sits at c ^ swz(r): rows 4i..4i+3
// reading an aligned chunk pair (the transposed reads) hit distinct banks.
__device__ inline int swz(int r) {
  return ((2 * (r & 3)) | ((r >> 2) & 1)) ^ (((r >> 3) & 1) << 1);
}
__device__ inline u32x2 read_tr(const char* p) {
  const uint32_t addr = static_cast<uint32_t>(
      reinterpret_cast<uintptr_t>((const __attribute__((address_space(3))) void*)p));
  return __builtin_bit_cast(u32x2,
                            __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_s16x4*)(uintptr_t)addr));
}
__device__ inline f32x16 mfma(const u32x4& a, const u32x4& b, const f32x16& c) {
  return __builtin_amdgcn_mfma_f32_32x32x16_f16(__builtin_bit_cast(f16x8, a),
                                                __builtin_bit_cast(f16x8, b), c, 0, 0, 0);
}
// Two floats, times `scale` at most 2^15, as packed f16 pairs: two parts in one unit,
// whose last ends at f16's 2^-24, or three, part p in units of kPartUnit^p: what a
// part leaves is at most 2^-11 of the value, so the next one holds 11 bits more at
// the same magnitude.
constexpr float kPartUnit = 0x1p-11f;
// The pair is formed once (v_fma_mixlo, v_fma_mixhi): with nothing to hide its origin the
// compiler rounds each element again where the next part subtracts it (23 of the 285
// instructions of a two-part step, 41 of 472 with three).
__device__ inline f16x2 pack2(float x0, float x1, float scale) {
  const f16x2 h = {static_cast<_Float16>(__builtin_fmaf(x0, scale, 0.f)),
                   static_cast<_Float16>(__builtin_fmaf(x1, scale, 0.f))};
  uint32_t w = __builtin_bit_cast(uint32_t, h);
  asm("" : "+v"(w));
  return __builtin_bit_cast(f16x2, w);
}
__device__ inline void split2(float x0, float x1, float scale, uint32_t (&out)[2]) {
  const f16x2 h = pack2(x0, x1, scale);
  const f16x2 l = {
      static_cast<_Float16>(__builtin_fmaf(x0, scale, -static_cast<float>(h[0]))),
      static_cast<_Float16>(__builtin_fmaf(x1, scale, -static_cast<float>(h[1])))};
  out[0] = __builtin_bit_cast(uint32_t, h);
  out[1] = __builtin_bit_cast(uint32_t, l);
}
__device__ inline void split2(float x0, float x1, float scale, uint32_t (&out)[3]) {
  constexpr float kUp = 1.f / kPartUnit;
  const f16x2 h = pack2(x0, x1, scale);
  x0 = __builtin_fmaf(x0, scale, -static_cast<float>(h[0]));  // exact
  x1 = __builtin_fmaf(x1, scale, -static_cast<float>(h[1]));
  const f16x2 m = pack2(x0, x1, kUp);
  x0 = __builtin_fmaf(static_cast<float>(m[0]), -kPartUnit, x0);  // exact
  x1 = __builtin_fmaf(static_cast<float>(m[1]), -kPartUnit, x1);
  const f16x2 l = {static_cast<_Float16>(__builtin_fmaf(x0, kUp * kUp, 0.f)),
                   static_cast<_Float16>(__builtin_fmaf(x1, kUp * kUp, 0.f))};
  out[0] = __builtin_bit_cast(uint32_t, h);
  out[1] = __builtin_bit_cast(uint32_t, m);
  out[2] = __builtin_bit_cast(uint32_t, l);
}
// Three parts' sums of products as one, smallest first.
__device__ inline f32x16 join(const f32x16 (&x)[3]) {
  f32x16 s = x[2];
#pragma unroll
  for (int p = 1; p >= 0; --p)
#pragma unroll
    for (int i = 0; i < 16; ++i) s[i] = __builtin_fmaf(s[i], kPartUnit, x[p][i]);
  return s;
}
__device__ inline void wave_sync() {
  // LDS operations of one wave complete in order: only the compiler must keep it.
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}
template <int kParts, int kWaves>
__global__ __launch_bounds__(64 * kWaves, 2) void attend_rows(RowsArgs a, int n_qblk) {
  __shared__ __attribute__((aligned(128))) char vs[kWaves][kN * 128];
  __shared__ float mo[kWaves][kQ * kPitch];  // a wave's O rows
  __shared__ float ml[kWaves][2][kQ];        // and their max and sum
  __shared__ int nonfinite;                  // some output of the block is inf or NaN
  static_assert(sizeof(f32blk::Tiles<2>) <= sizeof(mo), "f32 tiles fit in the merge rows");

  if (threadIdx.x == 0) nonfinite = 0;
  // The blocks of one head, which read the same planes, share an XCD's L2.
  const int lid = xcd_remap(blockIdx.x, gridDim.x);
  const int qblk = lid % n_qblk, h = lid / n_qblk;
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int r32 = lane & 31, hl = lane >> 5;
  const int q0 = qblk * kQ, qi = q0 + r32;
  // Keys visible to this lane's row, and to the block's last row.
  const int row_end = a.causal ? min(a.n_keys, a.pos0 + qi + 1) : a.n_keys;
  const int kv_end = a.causal ? min(a.n_keys, a.pos0 + min(q0 + kQ, a.n_rows)) : a.n_keys;
  const int n_steps = (kv_end + kN - 1) / kN;

  // Rows past kv_end read as zero without touching memory.
  const int64_t plane = h * a.kv_hs;
  const uint32_t range = static_cast<uint32_t>(kv_end) * 128u;
  const __amdgpu_buffer_rsrc_t krs =
      __builtin_amdgcn_make_buffer_rsrc(const_cast<_Float16*>(a.k + plane), 0, range, kRawBuffer);
  const __amdgpu_buffer_rsrc_t vrs =
      __builtin_amdgcn_make_buffer_rsrc(const_cast<_Float16*>(a.v + plane), 0, range, kRawBuffer);
  u32x4 kx[4], vx[4];
  auto load = [&](int step) __attribute__((always_inline)) {
    const uint32_t ko = static_cast<uint32_t>(kN * step + r32) * 128u + 16u * hl;
    const uint32_t vo = static_cast<uint32_t>(kN * step) * 128u + 16u * lane;
#pragma unroll
    for (int i = 0; i < 4; ++i)
      kx[i] = __builtin_bit_cast(u32x4, __builtin_amdgcn_raw_buffer_load_b128(krs, ko + 32 * i, 0, 0));
#pragma unroll
    for (int i = 0; i < 4; ++i)
      vx[i] = __builtin_bit_cast(u32x4, __builtin_amdgcn_raw_buffer_load_b128(vrs, vo + 1024 * i, 0, 0));
  };

  // This lane's share of its query row: d = 16 dk + 8 hl + 0..7.
  f32x4 qx[8];
#pragma unroll
  for (int i = 0; i < 8; ++i) qx[i] = f32x4{0.f, 0.f, 0.f, 0.f};
  if (qi < a.n_rows) {
    const float* qp = a.q + static_cast<int64_t>(qi) * a.q_rs + h * 64 + 8 * hl;
#pragma unroll
    for (int i = 0; i < 8; ++i)
      qx[i] = *reinterpret_cast<const f32x4u*>(qp + 16 * (i >> 1) + 4 * (i & 1));
  }
  int step = wave;
  if (step < n_steps) load(step);

  float amax = 0.f;
#pragma unroll
  for (int i = 0; i < 8; ++i) {
    qx[i] *= a.scale_log2;
#pragma unroll
    for (int e = 0; e < 4; ++e) amax = fmaxf(amax, fabsf(qx[i][e]));
  }
  amax = pair_max(amax);
  const int e_max = static_cast<int>((__builtin_bit_cast(uint32_t, amax) >> 23) & 0xFF);
  const int sh = e_max == 0 ? 0 : clamp_exp(141 - e_max);
  const float up = pow2(sh), down = pow2(clamp_exp(-sh));
  u32x4 qf[kParts][4];
#pragma unroll
  for (int i = 0; i < 16; ++i) {
    uint32_t w[kParts];
    split2(qx[i >> 1][2 * (i & 1)], qx[i >> 1][2 * (i & 1) + 1], up, w);
#pragma unroll
    for (int p = 0; p < kParts; ++p) qf[p][i >> 2][i & 3] = w[p];
  }

  // V^T operand of a 32-key step (as the 16-bit prefill reads it): lane group
  // lane / 16 reads rows 4 (lane / 32) + (lane % 16) / 4 [+ 8 e + 16 k2] at
  // columns 16 (lane / 16 % 2) + 4 (lane % 4) [+ 32 cc], and lane (d, hl) gets
  // keys 4 hl + 0..3 of each, the order the packed weights have.
  char* const vw = vs[wave];
  const int vr = 4 * hl + ((lane & 15) >> 2), vc = 2 * ((lane >> 4) & 1) + ((lane & 3) >> 1);
  f32x16 o[2] = {f32x16{}, f32x16{}};
  float m = -INFINITY, l = 0.f;
  for (; step < n_steps; step += kWaves) {
    f32x16 s;
    if constexpr (kParts == 3) {
      f32x16 sp[kParts];  // a chain over d per part
#pragma unroll
      for (int p = 0; p < kParts; ++p) sp[p] = f32x16{};
#pragma unroll
      for (int dk = 0; dk < 4; ++dk)
#pragma unroll
        for (int p = 0; p < kParts; ++p) sp[p] = mfma(kx[dk], qf[p][dk], sp[p]);
      s = join(sp);
    } else {
      // Two chains over d (half the latency and half the roundings of one), the
      // smaller part first, so that few of the sums round at full size.
      f32x16 s2[2] = {f32x16{}, f32x16{}};
#pragma unroll
      for (int p = kParts - 1; p >= 0; --p)
#pragma unroll
        for (int dk = 0; dk < 4; ++dk) s2[dk & 1] = mfma(kx[dk], qf[p][dk], s2[dk & 1]);
      s = s2[0] + s2[1];
    }
    wave_sync();  // the last step's transposed reads are done
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int row = 8 * i + (lane >> 3);
      *reinterpret_cast<u32x4*>(vw + row * 128 + (((lane & 7) ^ swz(row)) * 16)) = vx[i];
    }
    wave_sync();
    if (step + kWaves < n_steps) load(step + kWaves);

    // Register i holds key 8 (i / 4) + 4 hl + i % 4 of the step.
    float mx = -INFINITY;
    const bool whole = kN * step + kN <= (a.causal ? a.pos0 + q0 + 1 : a.n_keys);
#pragma unroll
    for (int i = 0; i < 16; ++i) {
      float x = s[i] * down;
      if (!whole && kN * step + 8 * (i >> 2) + 4 * hl + (i & 3) >= row_end) x = -INFINITY;
      s[i] = x;
      mx = fmaxf(mx, x);
    }
    mx = pair_max(mx);
    const float m_new = fmaxf(m, mx);
    const float alpha = m == -INFINITY ? 0.f : __builtin_amdgcn_exp2f(m - m_new);
    const float m_use = m_new == -INFINITY ? 0.f : m_new;
    m = m_new;
    float ls = 0.f;
    u32x4 pf[kParts][2];
#pragma unroll
    for (int i = 0; i < 16; i += 2) {
      const float p0 = __builtin_amdgcn_exp2f(s[i] - m_use);
      const float p1 = __builtin_amdgcn_exp2f(s[i + 1] - m_use);
      ls += p0 + p1;
      uint32_t w[kParts];
      split2(p0, p1, kWeightUp, w);
#pragma unroll
      for (int p = 0; p < kParts; ++p) pf[p][i >> 3][(i >> 1) & 3] = w[p];
    }
    l = l * alpha + ls;
#pragma unroll
    for (int cc = 0; cc < 2; ++cc) {
      u32x4 va[2];
#pragma unroll
      for (int k2 = 0; k2 < 2; ++k2) {
        u32x2 t[2];
#pragma unroll
        for (int e = 0; e < 2; ++e) {
          const int row = vr + 8 * e + 16 * k2;
          t[e] = read_tr(vw + row * 128 + (((vc + 4 * cc) ^ swz(row)) * 16) + 8 * (lane & 1));
        }
        va[k2] = u32x4{t[0].x, t[0].y, t[1].x, t[1].y};
      }
      f32x16 x = {};
      if constexpr (kParts == 3) {
        f32x16 xp[kParts];
#pragma unroll
        for (int p = 0; p < kParts; ++p) xp[p] = f32x16{};
#pragma unroll
        for (int k2 = 0; k2 < 2; ++k2)
#pragma unroll
          for (int p = 0; p < kParts; ++p) xp[p] = mfma(va[k2], pf[p][k2], xp[p]);
        x = join(xp);
      } else {
#pragma unroll
        for (int p = kParts - 1; p >= 0; --p)
#pragma unroll
          for (int k2 = 0; k2 < 2; ++k2) x = mfma(va[k2], pf[p][k2], x);
      }
#pragma unroll
      for (int i = 0; i < 16; ++i) o[cc][i] = __builtin_fmaf(o[cc][i], alpha, x[i]);
    }
  }
  l += __shfl_xor(l, 32);

  // The waves' rows meet in LDS; thread (row, 8 columns) adds them with the
  // log-sum-exp rule (exp2 domain).
#pragma unroll
  for (int cc = 0; cc < 2; ++cc)
#pragma unroll
    for (int i = 0; i < 16; ++i)
      mo[wave][r32 * kPitch + 32 * cc + 8 * (i >> 2) + 4 * hl + (i & 3)] = o[cc][i];
  if (hl == 0) {
    ml[wave][0][r32] = m;
    ml[wave][1][r32] = l;
  }
  __syncthreads();
  const int row = tid >> 3, d0 = 8 * (tid & 7);
  if (row < kQ && q0 + row < a.n_rows) {
    float M = -INFINITY, L = 0.f, acc[8];
#pragma unroll
    for (int w = 0; w < kWaves; ++w) M = fmaxf(M, ml[w][0][row]);
#pragma unroll
    for (int e = 0; e < 8; ++e) acc[e] = 0.f;
#pragma unroll
    for (int w = 0; w < kWaves; ++w) {
      const float mw = ml[w][0][row];
      const float ew = mw == -INFINITY ? 0.f : __builtin_amdgcn_exp2f(mw - M);
      L = __builtin_fmaf(ml[w][1][row], ew, L);
#pragma unroll
      for (int e = 0; e < 8; ++e)
        acc[e] = __builtin_fmaf(mo[w][row * kPitch + d0 + e], ew, acc[e]);
    }
    const float inv = (L > 0.f ? 1.f / L : 0.f) * (1.f / kWeightUp);
    if constexpr (kParts == 2) {
      // A cross row whose sum is NaN (an infinite key or query) is zero, as the split-K
      // decode has it, whose groups take the shorter prompts.
#pragma unroll
      for (int e = 0; e < 8; ++e) acc[e] = L > 0.f ? acc[e] : 0.f;
    }
    float* const op = a.o + static_cast<int64_t>(q0 + row) * a.o_rs + h * 64 + d0;
    *reinterpret_cast<f32x4u*>(op) = f32x4{acc[0], acc[1], acc[2], acc[3]} * inv;
    *reinterpret_cast<f32x4u*>(op + 4) = f32x4{acc[4], acc[5], acc[6], acc[7]} * inv;
    if (a.lse && d0 == 0) {
      float* const stat = a.lse + 2 * (static_cast<int64_t>(h) * a.n_rows + q0 + row);
      stat[0] = M;
      stat[1] = L;
    }
    if constexpr (kParts == 3) {
#pragma unroll
      for (int e = 0; e < 8; ++e)
        if (!__builtin_isfinite(acc[e] * inv)) nonfinite = 1;
    }
  }
  if constexpr (kParts == 3) {
    // An infinite score (a key value past f16's range, an infinite query) gives its
    // key all of the row's weight or none, but in parts it comes out NaN (infinity
    // times a part of zero). The block's rows are then formed again with f32
    // operands, as every cached self row was before this kernel.
    __syncthreads();
    if (nonfinite) {
      PrefillArgs p{};
      p.q = a.q;
      p.k = a.k;
      p.v = a.v;
      p.o = a.o;
      p.lq = {0, 64, a.q_rs};
      p.lk = p.lv = {0, a.kv_hs, 64};
      p.lo = {0, 64, a.o_rs};
      p.n_heads = a.n_heads;
      p.t_q = min(q0 + kQ, a.n_rows);  // the extra waves share the tiles and store nothing
      p.t_kv = a.n_keys;
      p.d_head = 64;
      p.causal = 1;
      p.q_pos_offset = a.pos0;
      p.scale = 0.125f;
      f32blk::fa2_block<float, _Float16, 2, kWaves>(
          p, q0, h, 0, *reinterpret_cast<f32blk::Tiles<2>*>(mo));
    }
  }
}

}  // namespace

hipError_t launch_attend_rows(const RowsArgs& a, hipStream_t s) {
  if (a.n_rows <= 0 || a.n_heads <= 0) return hipSuccess;
  // Byte offsets of a plane are 32-bit.
  if (a.n_keys <= 0 || static_cast<int64_t>(a.n_keys) + 4096 > (int64_t{1} << 24))
    return hipErrorInvalidValue;
  const int n_qblk = (a.n_rows + kQ - 1) / kQ;
  const int64_t wgs = static_cast<int64_t>(n_qblk) * a.n_heads;
  if (wgs > 0x7fffffff) return hipErrorInvalidConfiguration;
  const dim3 grid(static_cast<unsigned>(wgs));
  // Eight waves where they get three steps or more each (128 rows x 1500 keys: 14.2
  // us, 15.4 on four); four below (300 keys: 7.4 us, 8.0 on eight; 224 self rows past
  // 220: 9.6, 10.5).
  const bool wide = a.n_keys >= 24 * kN;
#define WRS_ROWS(P, W) \
  hipLaunchKernelGGL((attend_rows<P, W>), grid, dim3(64 * W), 0, s, a, n_qblk)
  if (a.causal) {
    if (wide)
      WRS_ROWS(3, 8);
    else
      WRS_ROWS(3, 4);
  } else {
    if (wide)
      WRS_ROWS(2, 8);
    else
      WRS_ROWS(2, 4);
  }
#undef WRS_ROWS
  return hipGetLastError();
}

}  // namespace wrs
