// Projections with f16 weights: out(t, r) = W[r] . x[t] + bias[r]
// (replaces crates/tensor/src/ops/quant.rs:415-473 f16_linear, reached through
//  LinearWeight::linear, crates/tensor/src/weight.rs:116-137, from the
//  encoder's fused QKV projection, crates/whisper/src/encoder.rs:275-277, and
//  the cross-attention K/V precompute, crates/whisper/src/decoder.rs:423-447).
//
// K6 (linear_f16w): D^T = W X^T on v_mfma_f32_32x32x16_f16. Both operands are
//   "k-contiguous" rows as stored (W [n_out][n_in] f16, X [n_tokens][k] f16),
//   so neither needs a transpose. A workgroup owns a tile of output features x
//   tokens (LinTile: 64 x 64 up to 256 x 256, picked by grid size in
//   launch_parts); k advances 32 or 64 per LDS stage through a ring of 2 to 6
//   stages: tiles move global -> LDS with buffer_load ... lds (no staging
//   registers), rows past the matrix edge read as zero through the buffer range
//   check, and one barrier separates stages. Inside a stage every 16-k step
//   issues one MFMA per slot, with the LDS reads of the next step's operands
//   and a share of the tile loads between them: left to itself the compiler
//   reads two operands, waits, multiplies, and a wave alone on its SIMD idles
//   for the LDS latency six times a stage (256 x 256 tiles, one round: 31 ->
//   25 us at n_in 1280, 208 -> 171 us at 5120 with two parts). LDS rows keep
//   their 16-byte chunks XOR-permuted by the row index, so the 32 rows read by
//   one operand fetch spread over the banks (swz). Every tile shape adds k in
//   the same order, so the shape does not change a result's bits.
//   Bound: the larger tiles by LDS reads and DMA writes against the MFMAs (a
//   128 x 64 wave reads 6 operands per 8 MFMAs) and by the f32 output, which
//   one workgroup per CU does not overlap (6000 x 5120: 24 of 89 us); the
//   small ones by the memory latency of a few stages.
//   f32 activations go to the f16 matrix pipe through a pre-pass
//   (linear_split_rows): each row is scaled by a power of two so that its
//   largest element lies in [2^14, 2^15), then split into two f16 parts
//   hi + lo that sum to it within 2^-22 relative (2^-25 of the row maximum
//   where lo is subnormal). Both parts meet each W operand in turn (read once
//   for the two); each product carries at most that 2^-22
//   relative error, below what one f32 addition of the accumulation
//   (dot_f16_f32, simd.rs:593-700) already rounds away. The epilogue multiplies by
//   the row's 2^-shift (exact), adds the f32 bias and writes the output type
//   at out + t * out_rs + (r / 64) * out_hs + r % 64: token-major rows
//   (out_hs = 64) or the arena's [head][token][64] planes. Each wave passes its
//   tile through the freed stage buffers and stores 64- to 512-byte pieces of
//   output rows, 16 bytes per lane: stored straight from the MFMA layout (pieces
//   of 32 different rows per instruction) a 16-bit tile took 2.2x as long.
//   Few rows over long k (37 x 5120 -> 1280) leave too few tiles for the chip:
//   32 x 64 tiles then split k over workgroups, merged through memory.
//   Measured (f32 x, f32 output, pre-pass included, against one 256 x 256 shape
//   for every call): 37 x 1280 x 1280 54 -> 11.4 us, 1500 x 1280 x 1280 65 ->
//   23 us, 1500 x 5120 -> 1280 208 -> 57 us, 37 x 5120 -> 1280 192 -> 16 us,
//   6000 x 1280 -> 5120 166 -> 153 us.
#include "wrs_internal.hpp"

#include <algorithm>
#include <atomic>

namespace wrs {
namespace {

typedef _Float16 f16x8 __attribute__((ext_vector_type(8)));
typedef _Float16 f16x4v __attribute__((ext_vector_type(4)));
typedef float f32x16 __attribute__((ext_vector_type(16)));
typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
typedef uint32_t u32x2 __attribute__((ext_vector_type(2)));

// Tile shape of one workgroup: FT output features x TT tokens, WM x WN of it per
// wave in 32 x 32 MFMA tiles; k advances BK per LDS stage through NS stages; P
// f16 parts of every x row share each W stage.
template <int FT_, int TT_, int WM_, int WN_, int BK_, int NS_, int P_, bool kSlots_ = true>
struct LinTile {
  static constexpr bool kSlots = kSlots_;  // 16-k steps in hand-placed slots
  static constexpr int FT = FT_, TT = TT_, WM = WM_, WN = WN_, BK = BK_, NS = NS_, P = P_;
  static constexpr int MI = WM / 32, NJ = WN / 32;       // MFMA tiles of a wave
  static constexpr int kWavesM = FT / WM;
  static constexpr int kWaves = kWavesM * (TT / WN), kThreads = 64 * kWaves;
  static constexpr int KS = BK / 16;                     // 16-k steps per stage
  static constexpr int kStage = (FT + P * TT) * BK;      // f16 elements of a stage: W rows, x rows
  static constexpr int kChunks = BK / 8;                 // 16-byte chunks of an LDS row
  static constexpr int kDmaRows = 64 / kChunks;          // rows one 1 KB DMA instruction moves
  static constexpr int kDmaA = FT / kDmaRows / kWaves;   // DMA instructions per wave and stage
  static constexpr int kDmaB = P * TT / kDmaRows / kWaves;
  static constexpr int kDma = kDmaA + kDmaB;
  static constexpr int kMfmas = P * MI * NJ, kReads = MI + P * NJ;  // of one 16-k step
  static constexpr int kGroupM = FT >= 256 ? 4 : 1024 / FT;  // feature tiles an XCD walks at a time
  static_assert(kDmaA * kDmaRows * kWaves == FT && kDmaB * kDmaRows * kWaves == P * TT,
                "every wave moves whole DMA instructions");
  static_assert(BK == 32 || BK == 64, "swizzles for 64- and 128-byte rows");
  static_assert(KS % 2 == 0, "operands alternate between two register sets");
  static_assert(kWaves * WM * 128 <= NS * kStage * 2, "32 staged f32 token rows per wave fit");
};

// 16-byte chunk c of LDS row r sits at slot c ^ f(r). An operand fetch reads
// one chunk of 32 consecutive rows; 16 lanes at a time cover the 256 bytes of
// banks, i.e. two 128-byte (four 64-byte) rows per bank line, so the rows of
// every 16 that share a place in the line must land in distinct slots; f does
// that.
template <int BK>
__device__ inline int swz(int row, int chunk) {
  return BK == 64 ? chunk ^ ((row >> 1) & 7) : chunk ^ ((row >> 2) & 3);
}

#pragma clang diagnostic push
#pragma clang diagnostic ignored "-Winline-asm"
// 16 bytes per lane from global memory into LDS at m0 + 16 * lane, through a
// buffer resource (offsets past its size read as zero). Inline asm, so the
// compiler adds no waits of its own before later LDS reads; the kernel orders
// it with explicit vmcnt waits and barriers. m0 is used by nothing else here.
__device__ inline void dma16(u32x4 rsrc, uint32_t lds, uint32_t voff) {
  asm volatile("s_mov_b32 m0, %2\n\tbuffer_load_dwordx4 %0, %1, 0 offen lds"
               :: "v"(voff), "s"(rsrc), "s"(lds) : "memory", "m0");
}
// The same with 4 bytes per lane, at m0 + 4 * lane.
__device__ inline void dma4(u32x4 rsrc, uint32_t lds, uint32_t voff) {
  asm volatile("s_mov_b32 m0, %2\n\tbuffer_load_dword %0, %1, 0 offen lds"
               :: "v"(voff), "s"(rsrc), "s"(lds) : "memory", "m0");
}
#pragma clang diagnostic pop

__device__ inline u32x4 buffer_rsrc(const void* base, uint32_t bytes) {
  const uint64_t p = reinterpret_cast<uint64_t>(base);
  u32x4 r;
  r[0] = __builtin_amdgcn_readfirstlane(static_cast<uint32_t>(p));
  r[1] = __builtin_amdgcn_readfirstlane(static_cast<uint32_t>(p >> 32) & 0xffffu);
  r[2] = __builtin_amdgcn_readfirstlane(bytes);
  r[3] = 0x00020000u;  // raw buffer, 32-bit data format
  return r;
}

__device__ inline uint32_t lds_addr(const void* p) {
  return static_cast<uint32_t>(
      reinterpret_cast<uintptr_t>((const __attribute__((address_space(3))) void*)p));
}

// At most N of this wave's DMA loads are still in flight and its LDS accesses
// are done, then all waves meet.
template <int N>
__device__ inline void stage_barrier() {
  __builtin_amdgcn_sched_barrier(0);
  asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)\n\ts_barrier" ::"n"(N) : "memory");
  __builtin_amdgcn_sched_barrier(0);
}

// Tile id -> feature and token tile: ids walk groups of kGroupM feature tiles
// with the token tiles outermost inside a group, so that the workgroups an XCD
// runs at once (a contiguous range of ids) share their operand stages in its L2.
template <int kGroupM>
__device__ inline void tile_of(int id, int n_fm, int n_tn, int& fm, int& tn) {
  const int group = id / (kGroupM * n_tn);
  const int gm = min(kGroupM, n_fm - group * kGroupM);
  const int in = id - group * kGroupM * n_tn;
  fm = group * kGroupM + in % gm;
  tn = in / gm;
}

constexpr int kLinCounterStride = 32;  // words between merge counters (one 128-byte line)
constexpr int kLinMaxSplits = 8;
constexpr int kLinPartFloats = 2048;   // partial sums of one 32 x 64 tile

template <typename OutT, class C>
__global__ __launch_bounds__(C::kThreads, 1) void linear_f16w(LinearArgs a, int n_splits) {
  constexpr int MI = C::MI, NJ = C::NJ, P = C::P, BK = C::BK, NS = C::NS, KS = C::KS;
  __shared__ __attribute__((aligned(128))) _Float16 lds[NS * C::kStage];
  __shared__ __attribute__((aligned(16))) float bias_s[(C::FT + 63) / 64 * 64];
  __shared__ int merger;

  const int tid = threadIdx.x;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6), lane = tid & 63;
  const int wm = wave % C::kWavesM, wn = wave / C::kWavesM;
  const int n_fm = (a.n_out + C::FT - 1) / C::FT, n_tn = (a.n_tokens + C::TT - 1) / C::TT;
  // Workgroup ids run over (group, k split, tile); each XCD takes a contiguous
  // range of them.
  const int id = xcd_remap(blockIdx.x, gridDim.x);
  const int tiles = n_fm * n_tn;
  const int grp = id / (tiles * n_splits);
  const int split = (id / tiles) % n_splits;
  int fm, tn;
  tile_of<C::kGroupM>(id % tiles, n_fm, n_tn, fm, tn);
  const int m0 = fm * C::FT;  // first output feature
  const int n0 = tn * C::TT;  // first token

  // Row scales of this lane's tokens, requested before the stages.
  const int orow = lane & 31, kgrp = lane >> 5;
  float rs[NJ];
#pragma unroll
  for (int j = 0; j < NJ; ++j) {
    const int t = n0 + wn * C::WN + 32 * j + orow;
    rs[j] = (a.row_scale && t < a.n_tokens) ? a.row_scale[t] : 1.0f;
  }

  // DMA sources. An instruction moves kDmaRows LDS rows; lane i lands at slot
  // i % kChunks of row i / kChunks and so fetches logical chunk swz(row, slot).
  // Rows past n_out / n_tokens fall outside the buffer ranges and read as zero.
  const u32x4 wrs = buffer_rsrc(a.w[grp], static_cast<uint32_t>(
                                              static_cast<int64_t>(a.n_out) * a.n_in * 2));
  const u32x4 xrs = buffer_rsrc(
      a.x, static_cast<uint32_t>(((static_cast<int64_t>(a.n_tokens) - 1) * a.x_rs +
                                  static_cast<int64_t>(P) * a.n_in) * 2));
  uint32_t aoff[C::kDmaA], boff[C::kDmaB];
#pragma unroll
  for (int j = 0; j < C::kDmaA; ++j) {
    const int row = (wave * C::kDmaA + j) * C::kDmaRows + lane / C::kChunks;
    const int ch = swz<BK>(row, lane % C::kChunks);
    aoff[j] = static_cast<uint32_t>((static_cast<int64_t>(m0 + row) * a.n_in + ch * 8) * 2);
  }
#pragma unroll
  for (int j = 0; j < C::kDmaB; ++j) {
    const int row = (wave * C::kDmaB + j) * C::kDmaRows + lane / C::kChunks;
    const int ch = swz<BK>(row, lane % C::kChunks);
    boff[j] = static_cast<uint32_t>((static_cast<int64_t>(n0 + row % C::TT) * a.x_rs +
                                     static_cast<int64_t>(row / C::TT) * a.n_in + ch * 8) * 2);
  }
  const uint32_t a_lds = lds_addr(lds) + wave * C::kDmaA * 1024;
  const uint32_t b_lds = lds_addr(lds) + C::FT * BK * 2 + wave * C::kDmaB * 1024;
  const int n_kt = a.n_in / BK;
  const int kt0 = n_kt * split / n_splits, kt1 = n_kt * (split + 1) / n_splits;
  // DMA instruction d of stage kt into ring slot `slot`. Stages past the last
  // are issued too, out of the buffers' ranges (spans stay below 2^31): they
  // touch no memory, and every step has the same number in flight.
  auto dma = [&](int d, int kt, int slot) __attribute__((always_inline)) {
    const uint32_t ko = kt < kt1 ? static_cast<uint32_t>(kt * BK * 2) : 0x80000000u;
    const uint32_t so = __builtin_amdgcn_readfirstlane(slot * C::kStage * 2);
    if (d < C::kDmaA)
      dma16(wrs, a_lds + so + d * 1024, aoff[d] + ko);
    else
      dma16(xrs, b_lds + so + (d - C::kDmaA) * 1024, boff[d - C::kDmaA] + ko);
  };

  f32x16 acc[MI][NJ];
#pragma unroll
  for (int i = 0; i < MI; ++i)
#pragma unroll
    for (int j = 0; j < NJ; ++j)
#pragma unroll
      for (int e = 0; e < 16; ++e) acc[i][j][e] = 0.0f;

  // Operand reads: row l % 32 of each 32-row MFMA tile (32 rows on, the same
  // swizzle), k-group l / 32 (8 consecutive k) of a 16-k step.
  const char* const ldsb = reinterpret_cast<const char*>(lds);
  int aaddr[KS], baddr[KS];
#pragma unroll
  for (int ks = 0; ks < KS; ++ks) {
    const int ch = swz<BK>(orow, 2 * ks + kgrp) * 16;
    aaddr[ks] = (wm * C::WM + orow) * BK * 2 + ch;
    baddr[ks] = (C::FT + wn * C::WN + orow) * BK * 2 + ch;
  }
  struct Frag {
    f16x8 a[MI], b[P][NJ];
  };
  auto read = [&](Frag& f, int r, int slot, int ks) __attribute__((always_inline)) {
    const char* const st = ldsb + slot * (C::kStage * 2);
    if (r < MI)
      f.a[r] = *reinterpret_cast<const f16x8*>(st + aaddr[ks] + r * (32 * BK * 2));
    else
      f.b[(r - MI) / NJ][(r - MI) % NJ] = *reinterpret_cast<const f16x8*>(
          st + baddr[ks] + ((r - MI) / NJ * C::TT + (r - MI) % NJ * 32) * (BK * 2));
  };

  // The tile's bias goes to LDS (zeros without one) ahead of the first stage:
  // the stage barriers cover it, and the epilogue reads it without a round trip.
  {
    const u32x4 brs = buffer_rsrc(a.bias[grp] ? a.bias[grp] : reinterpret_cast<const float*>(a.x),
                                  a.bias[grp] ? static_cast<uint32_t>(a.n_out * 4) : 0u);
    if (wave < (C::FT + 63) / 64)
      dma4(brs, lds_addr(bias_s) + wave * 256, static_cast<uint32_t>((m0 + wave * 64 + lane) * 4));
  }
#pragma unroll
  for (int s = 0; s < NS - 1; ++s)
#pragma unroll
    for (int d = 0; d < C::kDma; ++d) dma(d, kt0 + s, s);

  // One 16-k step: its MFMAs, one per slot, with the operand reads of the next
  // step and a share of the tile loads dealt between them, so that a wave alone
  // on its SIMD keeps the matrix pipe fed. The order of the sums is k steps
  // ascending, high part before low.
  constexpr int kM = C::kMfmas, kR = C::kReads;
  auto kstep = [&](const Frag& cur, Frag& nxt, int slot, int ks, int d0, int d1, int kt_dma,
                   int slot_dma) __attribute__((always_inline)) {
#pragma unroll
    for (int n = 0; n < kM; ++n) {
#pragma unroll
      for (int r = 0; r < kR; ++r)
        if (r * kM / kR == n) read(nxt, r, slot, ks);
#pragma unroll
      for (int d = 0; d < C::kDma; ++d)
        if (d >= d0 && d < d1 && (d - d0) * kM / (d1 - d0) == n) dma(d, kt_dma, slot_dma);
      const int p = n / (MI * NJ), i = n / NJ % MI, j = n % NJ;
      acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_f16(cur.a[i], cur.b[p][j], acc[i][j], 0, 0, 0);
      __builtin_amdgcn_sched_barrier(0);
    }
  };
  if constexpr (C::kSlots) {
    Frag f0, f1;
    stage_barrier<(NS - 2) * C::kDma>();
  #pragma unroll
    for (int r = 0; r < kR; ++r) read(f0, r, 0, 0);
    // The first share of stage kt0 + NS - 1, which a step before kt0 would issue.
  #pragma unroll
    for (int d = 0; d < C::kDma / KS; ++d) dma(d, kt0 + NS - 1, NS - 1);
    int slot = 0;
    // Stage kt, whose first operands are in `f`. In its last step stage kt + 1
    // has landed and nobody reads stage kt any more, whose buffer takes stage
    // kt + NS: its loads are dealt over that step and the next stage's others.
    auto stage = [&](int kt, Frag& f, Frag& g) __attribute__((always_inline)) {
  #pragma unroll
      for (int ks = 0; ks < KS; ++ks) {
        Frag& cur = ks % 2 == 0 ? f : g;
        Frag& nxt = ks % 2 == 0 ? g : f;
        if (ks + 1 < KS) {
          kstep(cur, nxt, slot, ks + 1, C::kDma * (ks + 1) / KS, C::kDma * (ks + 2) / KS,
                kt + NS - 1, slot == 0 ? NS - 1 : slot - 1);
        } else {
          stage_barrier<(NS - 2) * C::kDma>();
          const int freed = slot;
          slot = slot + 1 == NS ? 0 : slot + 1;
          kstep(cur, nxt, slot, 0, 0, C::kDma / KS, kt + NS, freed);
        }
      }
    };
    for (int kt = kt0; kt < kt1; ++kt) stage(kt, f0, f1);
  } else {
    // A stage at a time, in the compiler's order.
    int slot = 0;
    for (int kt = kt0; kt < kt1; ++kt) {
      stage_barrier<(NS - 2) * C::kDma>();
#pragma unroll
      for (int d = 0; d < C::kDma; ++d) dma(d, kt + NS - 1, slot == 0 ? NS - 1 : slot - 1);
      Frag f[KS];
#pragma unroll
      for (int ks = 0; ks < KS; ++ks)
#pragma unroll
        for (int r = 0; r < kR; ++r) read(f[ks], r, slot, ks);
#pragma unroll
      for (int ks = 0; ks < KS; ++ks)
#pragma unroll
        for (int n = 0; n < kM; ++n) {
          const int p = n / (MI * NJ), i = n / NJ % MI, j = n % NJ;
          acc[i][j] =
              __builtin_amdgcn_mfma_f32_32x32x16_f16(f[ks].a[i], f[ks].b[p][j], acc[i][j], 0, 0, 0);
        }
      slot = slot + 1 == NS ? 0 : slot + 1;
    }
  }
  stage_barrier<0>();  // no load in flight, nobody reads a stage any more

  if constexpr (C::FT == 32 && C::TT == 64) {
    if (n_splits > 1) {
      // Split k: every wave publishes its sums lane by lane with agent-scope
      // stores and waits for them; the workgroup that counts in last adds the
      // splits in split order (the bits do not depend on the arrival order),
      // re-arms the tile's counter and writes the tile.
      static_assert(MI == 1 && NJ == 1, "one MFMA tile per wave");
      const int unit = grp * tiles + id % tiles;
      const bool valid = n0 + wn * C::WN + orow < a.n_tokens;
      float* const base = a.part + static_cast<int64_t>(unit) * n_splits * kLinPartFloats +
                          wave * 1024 + lane;
      float* const mine = base + split * kLinPartFloats;
      if (valid) {
#pragma unroll
        for (int e = 0; e < 16; ++e) st_agent(mine + e * 64, acc[0][0][e]);
      }
      __builtin_amdgcn_s_waitcnt(0);
      __syncthreads();
      unsigned* const counter = a.counters + static_cast<int64_t>(unit) * kLinCounterStride;
      if (tid == 0)
        merger = __hip_atomic_fetch_add(counter, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) ==
                 static_cast<unsigned>(n_splits - 1);
      __syncthreads();
      if (!merger) return;
      float px[kLinMaxSplits][16];
#pragma unroll
      for (int s = 0; s < kLinMaxSplits; ++s) {
        if (s >= n_splits) break;
#pragma unroll
        for (int e = 0; e < 16; ++e)
          px[s][e] = valid && s != split ? ld_agent(base + s * kLinPartFloats + e * 64) : 0.f;
      }
      f32x16 sum = {};
#pragma unroll
      for (int s = 0; s < kLinMaxSplits; ++s) {
        if (s >= n_splits) break;
#pragma unroll
        for (int e = 0; e < 16; ++e) sum[e] += s == split ? acc[0][0][e] : px[s][e];
      }
      acc[0][0] = sum;
      if (tid == 0) __hip_atomic_store(counter, 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    }
  }

  // Epilogue: acc[i][j][e] is feature 32 i + 8 (e / 4) + 4 kgrp + e % 4 of the
  // wave's part, token 32 j + orow. A wave passes 32 tokens at a time through
  // its part of the stage buffers, as rows of its WM features (16-byte chunk c
  // of row t at c ^ (t mod chunks)), and stores whole pieces of output rows.
  constexpr int kRowBytes = C::WM * static_cast<int>(sizeof(OutT));
  constexpr int kCh = kRowBytes / 16;
  constexpr int kPer = 16 / static_cast<int>(sizeof(OutT));  // values of a chunk
  char* const ot = reinterpret_cast<char*>(lds) + wave * (32 * kRowBytes);
  OutT* const out = reinterpret_cast<OutT*>(a.out[grp]);
  const bool v16 =
      sizeof(OutT) == 4 ||
      ((reinterpret_cast<uintptr_t>(out) | (a.out_rs * 2) | (a.out_hs * 2)) & 15) == 0;
  auto wave_sync = [] {
    // LDS operations of one wave complete in order: only the compiler must keep it.
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
  };
#pragma unroll
  for (int j = 0; j < NJ; ++j) {
    wave_sync();
#pragma unroll
    for (int i = 0; i < MI; ++i)
#pragma unroll
      for (int g = 0; g < 4; ++g) {
        const int fl = i * 32 + 8 * g + 4 * kgrp;  // feature within the staged row
        const f32x16& s = acc[i][j];
        f32x4 v = {s[4 * g], s[4 * g + 1], s[4 * g + 2], s[4 * g + 3]};
        v *= rs[j];
        v += *reinterpret_cast<const f32x4*>(&bias_s[wm * C::WM + fl]);
        if (a.act == kActGelu) {
#pragma unroll
          for (int e = 0; e < 4; ++e) v[e] = gelu_tanh(v[e]);
        }
        const int at = orow * kRowBytes + (((fl / kPer) ^ (orow & (kCh - 1))) * 16);
        if constexpr (sizeof(OutT) == 4) {
          *reinterpret_cast<f32x4*>(ot + at) = v;
        } else if constexpr (__is_same(OutT, __bf16)) {
          typedef __bf16 bf16x4 __attribute__((ext_vector_type(4)));
          *reinterpret_cast<u32x2*>(ot + at + (fl & 4) * 2) =
              __builtin_bit_cast(u32x2, __builtin_convertvector(v, bf16x4));
        } else {
          *reinterpret_cast<u32x2*>(ot + at + (fl & 4) * 2) =
              __builtin_bit_cast(u32x2, __builtin_convertvector(v, f16x4v));
        }
      }
    wave_sync();
#pragma unroll
    for (int q = 0; q < kCh / 2; ++q) {
      const int row = (q * 64 + lane) / kCh, c = (q * 64 + lane) % kCh;
      const int t = n0 + wn * C::WN + 32 * j + row;
      const int r = m0 + wm * C::WM + c * kPer;
      const u32x4 h =
          *reinterpret_cast<const u32x4*>(ot + row * kRowBytes + ((c ^ (row & (kCh - 1))) * 16));
      if (t < a.n_tokens && r < a.n_out) {
        OutT* p = out + static_cast<int64_t>(t) * a.out_rs +
                  static_cast<int64_t>(r >> 6) * a.out_hs + (r & 63);
        if (sizeof(OutT) == 4 || (v16 && r + 8 <= a.n_out)) {
          *reinterpret_cast<u32x4*>(p) = h;
        } else {
          *reinterpret_cast<u32x2*>(p) = u32x2{h[0], h[1]};
          if (r + 8 <= a.n_out) *reinterpret_cast<u32x2*>(p + 4) = u32x2{h[2], h[3]};
        }
      }
    }
  }
}

// Decode-sized batches (n_tokens <= 8: the beams of one step) against f16 weights,
// f16_gemv_parallel semantics (quant.rs:343-413). The weight stream is the whole
// traffic, so every kernel below reads each 16-byte chunk of W once for all rows.
//
// K7 (gemv_f16w): one or two f16 rows.
//   One persistent workgroup of 8 waves per CU stages all of x in LDS once,
//   widened exactly, then its waves walk groups of 4 output features (1 when
//   n_out <= 4096, so that a d x d matrix still spreads over ~n_out / 8 CUs)
//   across the matrix: lane l multiplies W[r][k..k+8) for k = 8 l + 512 m by the
//   staged x of every row with f32 FMAs (the products dot_f16_f32 forms). The
//   16-byte loads of the next 2048-column batch (or of the next group) are in
//   flight while a batch is multiplied. The 64 lane partials reduce with DPP and
//   two cross-row moves, and lane b stores row b.
constexpr int kGemvWaves = 8;
constexpr int kGemvChunk = 2048;                // W columns per load batch
constexpr int kGemvSmallOut = 4096;             // one feature per wave up to this n_out
constexpr int kGemvSteps = kGemvChunk / 512;    // 16-byte W loads per row and batch

template <int CTRL>
__device__ inline float dpp(float x) {
  return __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, x), CTRL,
                                                                0xF, 0xF, false));
}
// Sum over the 64 lanes: xor 1, xor 2 (quad perms), the mirror of each half row
// of 8 and of each row of 16 (DPP), then the two cross-row moves.
__device__ inline float wave_sum64(float v) {
  v += dpp<0xB1>(v);
  v += dpp<0x4E>(v);
  v += dpp<0x141>(v);
  v += dpp<0x140>(v);
  v += __shfl_xor(v, 16);
  return v + __shfl_xor(v, 32);
}

// LayerNorm of one f32 row by one wave, in the arithmetic of layer_norm_rows
// (elementwise.hip, norm.rs:116-143): lane partials over k = 4 lane + 256 i,
// mean, then the variance around it, each reduced with wave_sum64; so the
// normalized values equal that kernel's output bit for bit.
__device__ inline void ln_row_stats(const float* xr, int d, float eps, float& mean,
                                    float& inv_std) {
  const int lane = threadIdx.x & 63;
  float s = 0.0f;
  for (int k = 4 * lane; k < d; k += 256) {
    const f32x4 v = *reinterpret_cast<const f32x4*>(xr + k);
    s += (v[0] + v[1]) + (v[2] + v[3]);
  }
  mean = wave_sum64(s) / static_cast<float>(d);
  float q = 0.0f;
  for (int k = 4 * lane; k < d; k += 256) {
    const f32x4 v = *reinterpret_cast<const f32x4*>(xr + k);
#pragma unroll
    for (int j = 0; j < 4; ++j) q = fmaf(v[j] - mean, v[j] - mean, q);
  }
  const float var = wave_sum64(q) / static_cast<float>(d);
  inv_std = 1.0f / sqrtf(var + eps);
}
// Rows of up to 256 * kLnCache values live in registers: lane l holds
// columns 4 l + 256 i in v[i] (zeros past d). The loads are issued first
// (ln_row_load), the arithmetic follows (ln_row_norm), with the arithmetic
// of ln_row_stats exactly.
constexpr int kLnCache = 5;  // 1280 columns: every Whisper d_model
__device__ inline void ln_row_load(const float* xr, const float* g, const float* b, int d,
                                   f32x4 (&v)[kLnCache], f32x4 (&gg)[kLnCache],
                                   f32x4 (&bb)[kLnCache]) {
  const int lane = threadIdx.x & 63;
  const f32x4 z = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
  for (int i = 0; i < kLnCache; ++i) {
    const int k = 4 * lane + 256 * i;
    const bool in = k < d;
    v[i] = in ? *reinterpret_cast<const f32x4*>(xr + k) : z;
    if (g) {
      gg[i] = in ? *reinterpret_cast<const f32x4*>(g + k) : z;
      bb[i] = in ? *reinterpret_cast<const f32x4*>(b + k) : z;
    }
  }
}
__device__ inline void ln_reg_stats(int d, float eps, const f32x4 (&v)[kLnCache], float& mean,
                                    float& inv_std) {
  const int lane = threadIdx.x & 63;
  float s = 0.0f;
#pragma unroll
  for (int i = 0; i < kLnCache; ++i) s += (v[i][0] + v[i][1]) + (v[i][2] + v[i][3]);
  mean = wave_sum64(s) / static_cast<float>(d);
  float q = 0.0f;
#pragma unroll
  for (int i = 0; i < kLnCache; ++i) {
    if (4 * lane + 256 * i >= d) break;
#pragma unroll
    for (int j = 0; j < 4; ++j) q = fmaf(v[i][j] - mean, v[i][j] - mean, q);
  }
  const float var = wave_sum64(q) / static_cast<float>(d);
  inv_std = 1.0f / sqrtf(var + eps);
}
__device__ inline void ln_row_norm(int d, float eps, f32x4 (&v)[kLnCache],
                                   const f32x4 (&gg)[kLnCache], const f32x4 (&bb)[kLnCache]) {
  float mean, inv_std;
  ln_reg_stats(d, eps, v, mean, inv_std);
#pragma unroll
  for (int i = 0; i < kLnCache; ++i)
#pragma unroll
    for (int j = 0; j < 4; ++j) v[i][j] = fmaf((v[i][j] - mean) * inv_std, gg[i][j], bb[i][j]);
}

template <int NT, int kGemvRowsPerWave, typename OutT, int kGroups>
__global__ __launch_bounds__(64 * kGemvWaves) void gemv_f16w(GemvArgs<kGroups> a) {
  __shared__ __attribute__((aligned(16))) float xs[kGemvXFloats];
  const int tid = threadIdx.x;
  const int wave = tid >> 6, lane = tid & 63;
  const int grp = blockIdx.y;
  const int n_in = a.n_in;
  const _Float16* w = a.w[grp];

  OutT* out = reinterpret_cast<OutT*>(a.out[grp]);
  const float* bias = a.bias[grp];
  const int n_groups4 = (a.n_out + kGemvRowsPerWave - 1) / kGemvRowsPerWave;
  const int stride = gridDim.x * kGemvWaves;
  // W loads of one 2048-column batch of one group of 4 features.
  auto load_w = [&](int g4, int c0, uint4 (&wv)[kGemvRowsPerWave][kGemvSteps]) {
#pragma unroll
    for (int i = 0; i < kGemvRowsPerWave; ++i) {
      const int r = min(g4 * kGemvRowsPerWave + i, a.n_out - 1);
      const _Float16* wr = w + static_cast<int64_t>(r) * n_in + c0;
#pragma unroll
      for (int m = 0; m < kGemvSteps; ++m) {
        const int k = 8 * lane + 512 * m;
        if (c0 + k < n_in) wv[i][m] = *reinterpret_cast<const uint4*>(wr + k);
      }
    }
  };
  int g4 = blockIdx.x * kGemvWaves + wave;
  uint4 wv[kGemvRowsPerWave][kGemvSteps];
  if (g4 < n_groups4) load_w(g4, 0, wv);  // in flight while x is staged

  // Stage x: row b at xs[b * n_in ..], 8 columns per thread and step, the
  // 16-byte loads of 4 steps in flight before their stores.
  const int n8 = NT * n_in / 8;
  for (int e0 = tid; e0 < n8; e0 += 4 * 64 * kGemvWaves) {
    uint4 v[4];
#pragma unroll
    for (int u = 0; u < 4; ++u) {
      const int e = e0 + u * 64 * kGemvWaves;
      if (e < n8) {
        const int b = (8 * e) / n_in, k = 8 * e - b * n_in;
        v[u] = *reinterpret_cast<const uint4*>(static_cast<const _Float16*>(a.x) + b * a.x_rs + k);
      }
    }
#pragma unroll
    for (int u = 0; u < 4; ++u) {
      const int e = e0 + u * 64 * kGemvWaves;
      if (e < n8) {
        const f16x8 h = __builtin_bit_cast(f16x8, v[u]);
#pragma unroll
        for (int j = 0; j < 8; ++j) xs[8 * e + j] = static_cast<float>(h[j]);
      }
    }
  }
  __syncthreads();

  for (; g4 < n_groups4; g4 += stride) {
    // The group's bias is loaded now, so that its latency hides under the
    // products instead of following the reduction.
    float bias_v[kGemvRowsPerWave];
#pragma unroll
    for (int i = 0; i < kGemvRowsPerWave; ++i) {
      const int r = min(g4 * kGemvRowsPerWave + i, a.n_out - 1);
      bias_v[i] = bias ? bias[r] : 0.0f;
    }
    float acc[kGemvRowsPerWave][NT];
#pragma unroll
    for (int i = 0; i < kGemvRowsPerWave; ++i)
#pragma unroll
      for (int b = 0; b < NT; ++b) acc[i][b] = 0.0f;
    for (int c0 = 0; c0 < n_in; c0 += kGemvChunk) {
      uint4 cur[kGemvRowsPerWave][kGemvSteps];
#pragma unroll
      for (int i = 0; i < kGemvRowsPerWave; ++i)
#pragma unroll
        for (int m = 0; m < kGemvSteps; ++m) cur[i][m] = wv[i][m];
      // the next batch (or the next group's first) is in flight during this one
      if (c0 + kGemvChunk < n_in)
        load_w(g4, c0 + kGemvChunk, wv);
      else if (g4 + stride < n_groups4)
        load_w(g4 + stride, 0, wv);
#pragma unroll
      for (int m = 0; m < kGemvSteps; ++m) {
        const int k = c0 + 8 * lane + 512 * m;
        if (k >= n_in) break;
        float xv[NT][8];
#pragma unroll
        for (int b = 0; b < NT; ++b) {
          const float4 lo = *reinterpret_cast<const float4*>(&xs[b * n_in + k]);
          const float4 hi = *reinterpret_cast<const float4*>(&xs[b * n_in + k + 4]);
          xv[b][0] = lo.x; xv[b][1] = lo.y; xv[b][2] = lo.z; xv[b][3] = lo.w;
          xv[b][4] = hi.x; xv[b][5] = hi.y; xv[b][6] = hi.z; xv[b][7] = hi.w;
        }
#pragma unroll
        for (int i = 0; i < kGemvRowsPerWave; ++i) {
          const f16x8 h = __builtin_bit_cast(f16x8, cur[i][m]);
#pragma unroll
          for (int j = 0; j < 8; ++j) {
            const float wf = static_cast<float>(h[j]);
#pragma unroll
            for (int b = 0; b < NT; ++b) acc[i][b] = fmaf(wf, xv[b][j], acc[i][b]);
          }
        }
      }
    }
#pragma unroll
    for (int i = 0; i < kGemvRowsPerWave; ++i)
#pragma unroll
      for (int b = 0; b < NT; ++b) acc[i][b] = wave_sum64(acc[i][b]);
    if (lane < NT) {
      const int r0 = g4 * kGemvRowsPerWave;
#pragma unroll
      for (int i = 0; i < kGemvRowsPerWave; ++i) {
        const int r = r0 + i;
        if (r >= a.n_out) break;
        float v = 0.0f;
#pragma unroll
        for (int b = 0; b < NT; ++b)
          if (b == lane) v = acc[i][b];
        if (bias) v += bias_v[i];
        if (a.act == kActGelu) v = gelu_tanh(v);
        out[static_cast<int64_t>(lane) * a.out_rs + static_cast<int64_t>(r >> 6) * a.out_hs +
            (r & 63)] = static_cast<OutT>(v);
      }
    }
  }
}

// K7m (gemv_f16w_mfma): the same product on the matrix pipe, for 3..8 f16 rows and
//   the f32 rows that K7f does not take.
//   W is read in tiles of T <= 16 features: lane (c, g) of a wave loads 16
//   bytes of feature c (columns 32 s + 8 g ..) per 32-column k-step s, which is
//   the A operand of a 16x16x32 f16 MFMA as loaded; lanes c >= T repeat the
//   tile's first feature (no extra traffic) and feed zeros. T = ceil(n_out /
//   n_CU) up to 16, so that a d x d matrix still spreads over every CU. The 8
//   waves of a workgroup split the k-steps of a tile; each wave keeps 5
//   k-steps (one register batch) of W in flight ahead of the MFMAs, the next
//   tile's first batch included.
//   x is staged once per workgroup into LDS as f16: row b (f32) is scaled by
//   2^sh_b (its max into [2^14, 2^15)) and split into a high part (B column
//   b) and a low part (B column 8 + b), so the products carry ~2^-22 relative
//   error; f16 x is exact in the high half alone. Rows are padded by 16 bytes,
//   which puts the 16 rows a ds_read_b128 phase touches on distinct banks.
//   The waves' 16x16 partial tiles meet in LDS (double-buffered, one barrier
//   per tile); thread (feature, b) adds the 8 waves' high and low columns,
//   scales by 2^-sh_b, adds the bias and stores.
constexpr int kGmWaves = 8;
constexpr int kGmKB = 5;          // 32-column k-steps per wave per register batch
constexpr int kGmRedPitch = 20;   // LDS pitch (floats) of one wave's 16x16 partial tile
constexpr int kGmRedFloats = 16 * kGmRedPitch;
constexpr size_t kGmStaticLds = sizeof(float) * (2 * kGmWaves * kGmRedFloats + 8);
constexpr size_t kGmMaxDynLds = 160 * 1024 - kGmStaticLds;

__device__ inline float gm_pow2(int e) { return __builtin_bit_cast(float, (e + 127) << 23); }
__device__ inline int gm_clamp_exp(int e) { return e < -126 ? -126 : (e > 127 ? 127 : e); }

__device__ inline float wave_max64(float v) {
  v = fmaxf(v, dpp<0xB1>(v));
  v = fmaxf(v, dpp<0x4E>(v));
  v = fmaxf(v, dpp<0x141>(v));
  v = fmaxf(v, dpp<0x140>(v));
  v = fmaxf(v, __shfl_xor(v, 16));
  return fmaxf(v, __shfl_xor(v, 32));
}

template <typename XT, typename OutT, bool kLn, int kGroups>
__global__ __launch_bounds__(64 * kGmWaves, 4) void gemv_f16w_mfma(GemvArgs<kGroups> a, int T) {
  extern __shared__ __attribute__((aligned(16))) _Float16 gxs[];  // [parts * nt][n_in + 8]
  __shared__ __attribute__((aligned(16))) float red[2][kGmWaves][kGmRedFloats];
  __shared__ float dn[8];

  constexpr bool kSplit = sizeof(XT) == 4;
  typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
  const int tid = threadIdx.x, wave = tid >> 6, lane = tid & 63;
  const int col = lane & 15, kg = lane >> 4;
  const int grp = blockIdx.y;
  const int nt = a.n_tokens, n_in = a.n_in, n_out = a.n_out;
  const int pitch = n_in + 8;
  const _Float16* w = a.w[grp];
  const int ks_total = n_in >> 5;
  const int s_per = (ks_total + kGmWaves - 1) / kGmWaves;
  const int ks0 = min(wave * s_per, ks_total), ks1 = min(ks0 + s_per, ks_total);
  const int n_batches = (s_per + kGmKB - 1) / kGmKB;
  const int n_tiles = (n_out + T - 1) / T;
  const bool arow = col < T;
  const u32x4 zero4 = {0, 0, 0, 0};

  // One batch of W loads; k-steps past the wave's range re-read its last
  // k-step (in bounds) and are not multiplied.
  auto load_batch = [&](int tile, int bj, u32x4 (&wv)[kGmKB]) {
    const int r = min(tile * T + (arow ? col : 0), n_out - 1);
    const _Float16* wr = w + static_cast<int64_t>(r) * n_in + 8 * kg;
#pragma unroll
    for (int u = 0; u < kGmKB; ++u) {
      const int ks = min(ks0 + bj * kGmKB + u, ks_total - 1);
      wv[u] = *reinterpret_cast<const u32x4*>(wr + 32 * ks);
    }
  };

  // f32 rows of up to 256 * kLnCache values are loaded into registers before
  // the first weight batch is issued, so that their wait does not include it
  // (loads complete in order); the arithmetic depends on a value defined after
  // both.
  int tile = blockIdx.x;
  u32x4 wv[kGmKB];
  constexpr bool reg_row = kSplit;  // n_in <= 256 * kLnCache: longer f32 rows run on K7l
  f32x4 xv[kLnCache], gg[kLnCache], bb[kLnCache];
  const float* xr32 = static_cast<const float*>(a.x) + static_cast<int64_t>(wave) * a.x_rs;
  if (reg_row && wave < nt)
    ln_row_load(xr32, kLn ? a.ln_g : nullptr, a.ln_b, n_in, xv, gg, bb);
  load_batch(tile, 0, wv);  // in flight while x is staged
  float one;
  __asm__ volatile("v_mov_b32 %0, 1.0" : "=v"(one) : : "memory");

  if (reg_row && wave < nt) {
#pragma unroll
    for (int i = 0; i < kLnCache; ++i) xv[i] *= one;
    if constexpr (kLn) ln_row_norm(n_in, a.ln_eps, xv, gg, bb);
    float amax = 0.f;
#pragma unroll
    for (int i = 0; i < kLnCache; ++i)
#pragma unroll
      for (int j = 0; j < 4; ++j) amax = fmaxf(amax, fabsf(xv[i][j]));  // zeros past n_in
    amax = wave_max64(amax);
    const int e_max = static_cast<int>((__builtin_bit_cast(uint32_t, amax) >> 23) & 0xFF);
    const int sh = e_max == 0 ? 0 : gm_clamp_exp(141 - e_max);
    const float up = gm_pow2(sh);
#pragma unroll
    for (int i = 0; i < kLnCache; ++i) {
      const int k = 4 * lane + 256 * i;
      if (k >= n_in) break;
      f16x4v hv, lv;
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        const float v = xv[i][j] * up;
        const _Float16 h = static_cast<_Float16>(v);
        hv[j] = h;
        lv[j] = static_cast<_Float16>(v - static_cast<float>(h));
      }
      *reinterpret_cast<f16x4v*>(&gxs[wave * pitch + k]) = hv;
      *reinterpret_cast<f16x4v*>(&gxs[(nt + wave) * pitch + k]) = lv;
    }
    if (lane == 0) dn[wave] = gm_pow2(gm_clamp_exp(-sh));
  }
  if constexpr (!kSplit) {
    if (wave < nt) {
      const XT* xr = static_cast<const XT*>(a.x) + static_cast<int64_t>(wave) * a.x_rs;
      for (int k = 8 * lane; k < n_in; k += 512)
        *reinterpret_cast<f16x8*>(&gxs[wave * pitch + k]) = *reinterpret_cast<const f16x8*>(xr + k);
      if (lane == 0) dn[wave] = 1.f;
    }
  }
  __syncthreads();

  // B column c < 8: high part of x row c; c >= 8: low part of row c - 8;
  // absent rows (and the low half for f16 x) are zero.
  const int beam = col & 7;
  const bool bvalid = beam < nt && (kSplit || col < 8);
  const _Float16* xb = gxs + (bvalid ? (col < 8 ? beam : nt + beam) * pitch : 0) + 8 * kg;
  const f16x8 zero8 = {0, 0, 0, 0, 0, 0, 0, 0};

  OutT* out = reinterpret_cast<OutT*>(a.out[grp]);
  const float* bias = a.bias[grp];
  int par = 0;
  for (; tile < n_tiles; tile += gridDim.x) {
    // Bias of the feature this thread stores, loaded under the MFMAs.
    float bias_v = 0.f;
    if (bias && tid < 128) bias_v = bias[min(tile * T + min(tid >> 3, T - 1), n_out - 1)];
    f32x4 acc = {0.f, 0.f, 0.f, 0.f};
    for (int bj = 0; bj < n_batches; ++bj) {
      u32x4 cur[kGmKB];
#pragma unroll
      for (int u = 0; u < kGmKB; ++u) cur[u] = arow ? wv[u] : zero4;
      if (bj + 1 < n_batches)
        load_batch(tile, bj + 1, wv);
      else if (tile + static_cast<int>(gridDim.x) < n_tiles)
        load_batch(tile + gridDim.x, 0, wv);
#pragma unroll
      for (int u = 0; u < kGmKB; ++u) {
        const int ks = ks0 + bj * kGmKB + u;
        if (ks < ks1) {  // wave-uniform
          const f16x8 bx = bvalid ? *reinterpret_cast<const f16x8*>(xb + 32 * ks) : zero8;
          acc = __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(f16x8, cur[u]), bx, acc,
                                                       0, 0, 0);
        }
      }
    }
#pragma unroll
    for (int i = 0; i < 4; ++i) red[par][wave][(4 * kg + i) * kGmRedPitch + col] = acc[i];
    __syncthreads();
    if (tid < 128) {
      const int r = tid >> 3, b = tid & 7;
      const int row = tile * T + r;
      if (r < T && b < nt && row < n_out) {
        float sacc = 0.f;
#pragma unroll
        for (int w8 = 0; w8 < kGmWaves; ++w8)
          sacc += red[par][w8][r * kGmRedPitch + b] + red[par][w8][r * kGmRedPitch + b + 8];
        float v = sacc * dn[b];
        if (bias) v += bias_v;
        if (a.act == kActGelu) v = gelu_tanh(v);
        out[static_cast<int64_t>(b) * a.out_rs + static_cast<int64_t>(row >> 6) * a.out_hs +
            (row & 63)] = static_cast<OutT>(v);
      }
    }
    par ^= 1;
  }
}

// K7l (gemv_f16w_long): K7m for f32 rows longer than its registers hold (the
//   second MLP projection). A wave needs x only at its own k-steps, so each
//   stages batches of kGlKB k-steps of every row for itself: half a wave per row
//   loads 128 columns, takes their largest element (a scale per row and batch),
//   and writes the high and low parts to the wave's own LDS rows; the batch's
//   MFMAs start from zero and are scaled back (exact) as they are added up. No
//   barrier stands before the products and the next batch of W and x is in
//   flight meanwhile. Rows staged whole by one wave each, in two passes, had cost
//   most of the launch, and eight rows of 5120 did not fit the LDS: 12.2 -> 11.2 us
//   for 5 rows of 5120 -> 1280, a size that K7f now takes; here 5 rows of 5120 ->
//   5120 take 19.1 us.
//   A fused LayerNorm takes one barrier: wave b forms row b's mean and deviation.
constexpr int kGlKB = 4;                       // k-steps per wave per batch: 128 columns
constexpr int kGlPitch = 32 * kGlKB + 8;       // f16 elements of a staged row

template <typename OutT, bool kLn, int kGroups>
__global__ __launch_bounds__(64 * kGmWaves, 4) void gemv_f16w_long(GemvArgs<kGroups> a, int T) {
  __shared__ __attribute__((aligned(16))) _Float16 xs[kGmWaves][16][kGlPitch];  // hi rows, lo rows
  __shared__ __attribute__((aligned(16))) float red[2][kGmWaves][kGmRedFloats];
  __shared__ float dn[kGmWaves][8], row_mean[8], row_inv[8];

  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int col = lane & 15, kg = lane >> 4;
  const int grp = blockIdx.y;
  const int nt = a.n_tokens, n_in = a.n_in, n_out = a.n_out;
  const _Float16* w = a.w[grp];
  const float* x = static_cast<const float*>(a.x);
  const int ks_total = n_in >> 5;
  const int s_per = (ks_total + kGmWaves - 1) / kGmWaves;
  const int ks0 = min(wave * s_per, ks_total), ks1 = min(ks0 + s_per, ks_total);
  const int n_batches = (s_per + kGlKB - 1) / kGlKB;
  const int n_tiles = (n_out + T - 1) / T;
  const bool arow = col < T;

  auto load_w = [&](int tile, int bj, u32x4 (&wv)[kGlKB]) {
    const int r = min(tile * T + (arow ? col : 0), n_out - 1);
    const _Float16* wr = w + static_cast<int64_t>(r) * n_in + 8 * kg;
#pragma unroll
    for (int u = 0; u < kGlKB; ++u)
      wv[u] = *reinterpret_cast<const u32x4*>(wr + 32 * min(ks0 + bj * kGlKB + u, ks_total - 1));
  };
  // Row 2 i + (lane / 32), columns 4 (lane % 32).. of the batch (the row's last
  // columns again past the matrix).
  const int xrow = lane >> 5, xcol = 4 * (lane & 31);
  const int pairs = (nt + 1) >> 1;
  auto load_x = [&](int bj, f32x4 (&xv)[4]) {
    const int k = min(32 * (ks0 + bj * kGlKB) + xcol, n_in - 4);
#pragma unroll
    for (int i = 0; i < 4; ++i)
      if (i < pairs)
        xv[i] = *reinterpret_cast<const f32x4*>(
            x + static_cast<int64_t>(min(2 * i + xrow, nt - 1)) * a.x_rs + k);
  };

  u32x4 wv[kGlKB];
  f32x4 xv[4], gv, bv;
  auto load_norm = [&](int bj) {
    const int k = min(32 * (ks0 + bj * kGlKB) + xcol, n_in - 4);
    gv = *reinterpret_cast<const f32x4*>(a.ln_g + k);
    bv = *reinterpret_cast<const f32x4*>(a.ln_b + k);
  };
  int tile = blockIdx.x;
  load_x(0, xv);
  if constexpr (kLn) load_norm(0);
  load_w(tile, 0, wv);
  if constexpr (kLn) {
    if (wave < nt) {
      float m, iv;
      ln_row_stats(x + static_cast<int64_t>(wave) * a.x_rs, n_in, a.ln_eps, m, iv);
      if (lane == 0) {
        row_mean[wave] = m;
        row_inv[wave] = iv;
      }
    }
    __syncthreads();
  }
  auto wave_sync = [] {
    // LDS operations of one wave complete in order: only the compiler must keep it.
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
  };
  // The batch's rows into this wave's LDS rows.
  auto stage = [&](int bj) __attribute__((always_inline)) {
    const bool in = 32 * (ks0 + bj * kGlKB) + xcol < 32 * ks1;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      if (i >= pairs) break;
      const int row = 2 * i + xrow;
      f32x4 v = xv[i];
      if constexpr (kLn) {
        const float mean = row_mean[min(row, nt - 1)], inv_std = row_inv[min(row, nt - 1)];
#pragma unroll
        for (int j = 0; j < 4; ++j) v[j] = fmaf((v[j] - mean) * inv_std, gv[j], bv[j]);
      }
      if (!in) v = f32x4{0.f, 0.f, 0.f, 0.f};
      float amax = fmaxf(fmaxf(fabsf(v[0]), fabsf(v[1])), fmaxf(fabsf(v[2]), fabsf(v[3])));
      amax = fmaxf(amax, dpp<0xB1>(amax));
      amax = fmaxf(amax, dpp<0x4E>(amax));
      amax = fmaxf(amax, dpp<0x141>(amax));
      amax = fmaxf(amax, dpp<0x140>(amax));
      float p = amax, q = amax;
      swap16(p, q);  // the other 16 lanes of this half
      amax = fmaxf(p, q);
      const int e_max = static_cast<int>((__builtin_bit_cast(uint32_t, amax) >> 23) & 0xFF);
      const int sh = e_max == 0 ? 0 : gm_clamp_exp(141 - e_max);
      const float up = gm_pow2(sh);
      f16x4v hv, lv;
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        const float s = v[j] * up;
        const _Float16 h = static_cast<_Float16>(s);
        hv[j] = h;
        lv[j] = static_cast<_Float16>(s - static_cast<float>(h));
      }
      if (row < nt) {
        *reinterpret_cast<f16x4v*>(&xs[wave][row][xcol]) = hv;
        *reinterpret_cast<f16x4v*>(&xs[wave][8 + row][xcol]) = lv;
        if ((lane & 31) == 0) dn[wave][row] = gm_pow2(gm_clamp_exp(-sh));
      }
    }
  };

  const int beam = col & 7;
  const bool bvalid = beam < nt;
  const _Float16* const xb = &xs[wave][bvalid ? col : 0][8 * kg];
  OutT* out = reinterpret_cast<OutT*>(a.out[grp]);
  const float* bias = a.bias[grp];
  const f16x8 zero8 = {0, 0, 0, 0, 0, 0, 0, 0};
  const u32x4 zero4 = {0, 0, 0, 0};
  int par = 0;
  for (; tile < n_tiles; tile += gridDim.x) {
    float bias_v = 0.f;
    if (bias && tid < 128) bias_v = bias[min(tile * T + min(tid >> 3, T - 1), n_out - 1)];
    const bool more = tile + static_cast<int>(gridDim.x) < n_tiles;
    f32x4 acc = {0.f, 0.f, 0.f, 0.f};
    for (int bj = 0; bj < n_batches; ++bj) {
      u32x4 cur[kGlKB];
#pragma unroll
      for (int u = 0; u < kGlKB; ++u) cur[u] = arow ? wv[u] : zero4;
      wave_sync();  // the last batch's operand reads are done
      stage(bj);
      const bool last = bj + 1 == n_batches;
      if (!last || more) {
        const int nb = last ? 0 : bj + 1;
        load_x(nb, xv);
        if constexpr (kLn) load_norm(nb);
        load_w(last ? tile + gridDim.x : tile, nb, wv);
      }
      wave_sync();
      const float down = bvalid ? dn[wave][beam] : 0.f;
      f32x4 part = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int u = 0; u < kGlKB; ++u) {
        if (ks0 + bj * kGlKB + u < ks1) {  // wave-uniform
          const f16x8 bx = bvalid ? *reinterpret_cast<const f16x8*>(xb + 32 * u) : zero8;
          part = __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(f16x8, cur[u]), bx, part,
                                                        0, 0, 0);
        }
      }
#pragma unroll
      for (int i = 0; i < 4; ++i) acc[i] = fmaf(part[i], down, acc[i]);
    }
#pragma unroll
    for (int i = 0; i < 4; ++i) red[par][wave][(4 * kg + i) * kGmRedPitch + col] = acc[i];
    // LDS only: the next tile's loads stay in flight.
    asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
    if (tid < 128) {
      const int r = tid >> 3, b = tid & 7;
      const int row = tile * T + r;
      if (r < T && b < nt && row < n_out) {
        float v = 0.f;
#pragma unroll
        for (int w8 = 0; w8 < kGmWaves; ++w8)
          v += red[par][w8][r * kGmRedPitch + b] + red[par][w8][r * kGmRedPitch + b + 8];
        if (bias) v += bias_v;
        if (a.act == kActGelu) v = gelu_tanh(v);
        out[static_cast<int64_t>(b) * a.out_rs + static_cast<int64_t>(row >> 6) * a.out_hs +
            (row & 63)] = static_cast<OutT>(v);
      }
    }
    par ^= 1;
  }
}

// K7f (gemv_f16w_rows): few f32 rows, by f32 FMAs on the registers the loads fill.
//   A launch of this size is a chain of waits with little arithmetic between them,
//   and what K7m and K7l add to the chain is the staging of x: timed inside the
//   kernels (5 rows), 1.1 of the 4.6 us of a 1280 x 1280 product went into scaling,
//   splitting and storing the rows and its barrier, 1 us into the matrix pipe's
//   serial k steps, and at 5120 columns 1.2 us into each of the five staged batches:
//   every workgroup stages all rows, 70 instructions a wave for four columns a lane,
//   for a tile of five features. The products themselves are 25 FMAs a lane and four
//   columns. So nothing is staged: a wave takes slices of 256 columns, lane l the
//   columns 4 l .. of each feature (8 bytes) and row (16 bytes), as loaded; both
//   slices of up to 24 are in flight from the start (kDeep). The sums over lanes are
//   formed four to a register, those over waves in LDS behind the only barrier. A
//   fused LayerNorm has wave b form row b's mean and deviation (one more barrier) and
//   every lane normalize what it holds.
//   FMAs and the LayerNorm are repeated per tile of T features and row, so rows and
//   features set where the matrix pipe wins. us, K7f / before (K7 for 1-2 rows, K7l
//   for 5120 columns, else K7m), 1, 2, 3, 5 and 8 rows:
//     1280 -> 1280       3.1/3.3  3.3/4.4  3.6/4.4  4.0/4.7  4.7/4.7
//     1280 -> 3 x 1280, LN  4.9/7.5  5.4/10.1  6.0/8.0  7.8/8.8  11.4/9.0
//     1280 -> 5120, LN   5.8/7.6  6.5/8.7  7.2/8.3  9.2/9.0  13.6/9.2
//     768 -> 3 x 768, LN  3.9/5.7  4.3/7.3  4.2/5.9  5.1/6.5  6.2/6.7
//     768 -> 3072, LN    4.3/5.2  4.8/6.2  5.0/5.4  6.1/5.7  9.1/5.6
//     512 -> 3 x 512, LN (3, 5, 8 rows)  4.1/5.4  5.1/5.7  7.8/6.0
//     5120 -> 1280       5.5/6.5  5.7/9.6  6.4/9.8  7.0/11.0  8.4/12.1
//     5120 -> 2560 (3, 5, 8 rows)  8.5/10.9  12.4/12.7  15.1/13.9
//     5120 -> 5120 (3, 5, 8 rows)  17.3/16.0  22.2/19.1  28.0/21.2
//     1280 -> 51866, LN  27.7/32.4  32.8/34.2  44.9/32.2  62.9/33.1  -
//   Error against 64 bits 0.6 to 0.95 of theirs.
constexpr int gf_rows(int n_tokens) { return n_tokens <= 2 ? 8 : 5; }  // features of a workgroup
constexpr int kGfWaves = 12;  // waves of a workgroup, at most

template <int NT, int kGfRows, bool kLn, bool kDeep, int kGroups>
__global__ __launch_bounds__(64 * kGfWaves) void gemv_f16w_rows(GemvArgs<kGroups> a, int T,
                                                                int n_kw, DType out_dt) {
  __shared__ float part[kGfWaves][kGfRows * NT + 3];
  __shared__ float row_mean[NT], row_inv[NT];
  typedef uint32_t u32x2 __attribute__((ext_vector_type(2)));
  typedef _Float16 h16x4 __attribute__((ext_vector_type(4)));

  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int grp = blockIdx.y;
  const int n_in = a.n_in, n_out = a.n_out;
  const int n_slices = (n_in + 255) >> 8;
  const int row0 = blockIdx.x * T;
  const _Float16* w = a.w[grp];
  const float* x = static_cast<const float*>(a.x);
  const float* bias = a.bias[grp];
  void* out = a.out[grp];

  struct Slice {
    f32x4 x[NT], g, b;
    u32x2 w[kGfRows];
  };
  // Slice s of the rows: columns 256 s + 4 lane .. (the last ones again past the end).
  auto load = [&](int s, Slice& v) __attribute__((always_inline)) {
    const int k = min(256 * s + 4 * lane, n_in - 4);
#pragma unroll
    for (int b = 0; b < NT; ++b)
      v.x[b] = *reinterpret_cast<const f32x4*>(x + static_cast<int64_t>(b) * a.x_rs + k);
    if constexpr (kLn) {
      v.g = *reinterpret_cast<const f32x4*>(a.ln_g + k);
      v.b = *reinterpret_cast<const f32x4*>(a.ln_b + k);
    }
#pragma unroll
    for (int i = 0; i < kGfRows; ++i) {
      const int r = min(row0 + min(i, T - 1), n_out - 1);
      v.w[i] = *reinterpret_cast<const u32x2*>(w + static_cast<int64_t>(r) * n_in + k);
    }
  };

  Slice va, vb;
  f32x4 xv[kLnCache], none[kLnCache];
  const float* xr = x + static_cast<int64_t>(min(wave, NT - 1)) * a.x_rs;
  const bool reg_row = n_in <= 256 * kLnCache;
  if constexpr (kLn) {
    if (wave < NT && reg_row) ln_row_load(xr, nullptr, nullptr, n_in, xv, none, none);
  }
  load(wave, va);
  if constexpr (kDeep) load(wave + n_kw, vb);
  const int f_row = row0 + tid / NT, f_b = tid % NT;  // the output of thread tid < T * NT
  float bias_v = 0.f;
  if (bias && tid < kGfRows * NT) bias_v = bias[min(f_row, n_out - 1)];

  float mean[NT], inv[NT];
  if constexpr (kLn) {
    if (wave < NT) {
      float m, iv;
      if (reg_row)
        ln_reg_stats(n_in, a.ln_eps, xv, m, iv);
      else
        ln_row_stats(xr, n_in, a.ln_eps, m, iv);
      if (lane == 0) {
        row_mean[wave] = m;
        row_inv[wave] = iv;
      }
    }
    // LDS only: the loads stay in flight.
    asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
#pragma unroll
    for (int b = 0; b < NT; ++b) {
      mean[b] = row_mean[b];
      inv[b] = row_inv[b];
    }
  }

  float acc[kGfRows * NT + 3];
#pragma unroll
  for (int i = 0; i < kGfRows * NT + 3; ++i) acc[i] = 0.f;
  auto add = [&](int s, Slice& v) __attribute__((always_inline)) {
    if constexpr (kLn) {
#pragma unroll
      for (int b = 0; b < NT; ++b)
#pragma unroll
        for (int j = 0; j < 4; ++j)
          v.x[b][j] = fmaf((v.x[b][j] - mean[b]) * inv[b], v.g[j], v.b[j]);
    }
    if (256 * s + 4 * lane >= n_in) {  // both: an infinite weight times 0 is not 0
#pragma unroll
      for (int b = 0; b < NT; ++b) v.x[b] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int i = 0; i < kGfRows; ++i) v.w[i] = u32x2{0, 0};
    }
#pragma unroll
    for (int i = 0; i < kGfRows; ++i) {
      if (i >= T) break;  // uniform
      const h16x4 h = __builtin_bit_cast(h16x4, v.w[i]);
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        const float wf = static_cast<float>(h[j]);
#pragma unroll
        for (int b = 0; b < NT; ++b) acc[i * NT + b] = fmaf(wf, v.x[b][j], acc[i * NT + b]);
      }
    }
  };
  if (wave < n_kw) {
    if constexpr (kDeep) {
      for (int s = wave; s < n_slices; s += 2 * n_kw) {
        add(s, va);
        if (s + 2 * n_kw < n_slices) load(s + 2 * n_kw, va);
        if (s + n_kw < n_slices) add(s + n_kw, vb);
        if (s + 3 * n_kw < n_slices) load(s + 3 * n_kw, vb);
      }
    } else {
      add(wave, va);
    }
    // Sums over the 64 lanes, four to a register: two swaps leave each row of 16
    // lanes with one of four sums, which its lanes then add up.
    constexpr int R = (kGfRows * NT + 3) / 4;
    float mine = 0.f;
#pragma unroll
    for (int j = 0; j < R; ++j) {
      swap32(acc[4 * j], acc[4 * j + 1]);
      swap32(acc[4 * j + 2], acc[4 * j + 3]);
      float p = acc[4 * j] + acc[4 * j + 1], q = acc[4 * j + 2] + acc[4 * j + 3];
      swap16(p, q);
      float v = p + q;
      v += dpp<0x128>(v);
      v += dpp<0x124>(v);
      v += dpp<0x122>(v);
      v += dpp<0x121>(v);
      if ((lane & 15) == j) mine = v;
    }
    const int o = 4 * (lane & 15) + ((lane >> 5) & 1) + 2 * ((lane >> 4) & 1);
    if (o < kGfRows * NT) part[wave][o] = mine;
  }
  asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
  if (tid < T * NT && f_row < n_out) {
    float v = 0.f;
    for (int i = 0; i < n_kw; ++i) v += part[i][tid];
    if (bias) v += bias_v;
    if (a.act == kActGelu) v = gelu_tanh(v);
    const int64_t o = static_cast<int64_t>(f_b) * a.out_rs +
                      static_cast<int64_t>(f_row >> 6) * a.out_hs + (f_row & 63);
    if (out_dt == kF32)
      static_cast<float*>(out)[o] = v;
    else if (out_dt == kF16)
      static_cast<_Float16*>(out)[o] = static_cast<_Float16>(v);
    else
      static_cast<__bf16*>(out)[o] = static_cast<__bf16>(v);
  }
}

// f32 rows -> [hi | lo] f16 rows of 2 n_in, plus each row's 2^-shift; with
// kLn the rows are normalized first (norm.rs:116-143, the layer_norm_rows
// arithmetic exactly). One wave per row. Bound by memory (4 bytes in, 4 out a
// value): rows of up to 256 kCached values are loaded once, every 16-byte load
// in flight before the maximum is taken, and leave as 8-byte stores; the
// scalar form this replaces read each row twice, one dword per lane and trip
// (1500 x 5120: 57 us; 37 x 1280: 6.4 us). x needs dword alignment only.
__device__ inline float pow2(int e) { return __builtin_bit_cast(float, (e + 127) << 23); }
__device__ inline int clamp_exp(int e) { return e < -126 ? -126 : (e > 127 ? 127 : e); }

__device__ inline f32x4 load4_dword_aligned(const float* p) {
  typedef float f32x4u __attribute__((ext_vector_type(4), aligned(4)));
  return *reinterpret_cast<const f32x4u*>(p);
}

__device__ inline float abs_max4(const f32x4& v) {
  return fmaxf(fmaxf(fabsf(v[0]), fabsf(v[1])), fmaxf(fabsf(v[2]), fabsf(v[3])));
}
// Four values scaled by `up` as f16 high parts at dst and low parts at dst + n_in.
__device__ inline void split_store4(const f32x4& x, float up, _Float16* dst, int n_in) {
  f16x4v hv, lv;
#pragma unroll
  for (int j = 0; j < 4; ++j) {
    const float v = x[j] * up;
    const _Float16 h = static_cast<_Float16>(v);
    hv[j] = h;
    lv[j] = static_cast<_Float16>(v - static_cast<float>(h));
  }
  *reinterpret_cast<f16x4v*>(dst) = hv;
  *reinterpret_cast<f16x4v*>(dst + n_in) = lv;
}

template <int kCached, bool kLn>
__global__ __launch_bounds__(256) void linear_split_rows(const float* x, int64_t x_rs,
                                                         int n_tokens, int n_in,
                                                         const float* gamma, const float* beta,
                                                         float eps, _Float16* xs,
                                                         float* row_scale) {
  static_assert(!kLn || kCached > 0, "normalized rows are held in registers");
  const int t = blockIdx.x * 4 + (threadIdx.x >> 6);
  const int lane = threadIdx.x & 63;
  if (t >= n_tokens) return;
  const float* xr = x + static_cast<int64_t>(t) * x_rs;
  _Float16* dst = xs + static_cast<int64_t>(t) * kSplitParts * n_in;
  float amax = 0.0f;
  f32x4 v[kCached > 0 ? kCached : 1];
  if constexpr (kCached > 0) {
    f32x4 gv[kLn ? kCached : 1], bv[kLn ? kCached : 1];
#pragma unroll
    for (int i = 0; i < kCached; ++i) {
      const int k = 4 * lane + 256 * i;
      const bool in = k < n_in;
      const f32x4 z = {0.f, 0.f, 0.f, 0.f};
      v[i] = in ? load4_dword_aligned(xr + k) : z;
      if constexpr (kLn) {
        gv[i] = in ? *reinterpret_cast<const f32x4*>(gamma + k) : z;
        bv[i] = in ? *reinterpret_cast<const f32x4*>(beta + k) : z;
      }
    }
    if constexpr (kLn) {
      float s = 0.0f;
#pragma unroll
      for (int i = 0; i < kCached; ++i) s += (v[i][0] + v[i][1]) + (v[i][2] + v[i][3]);
      const float mean = wave_sum64(s) / static_cast<float>(n_in);
      float q = 0.0f;
#pragma unroll
      for (int i = 0; i < kCached; ++i) {
        if (4 * lane + 256 * i >= n_in) break;
#pragma unroll
        for (int j = 0; j < 4; ++j) q = fmaf(v[i][j] - mean, v[i][j] - mean, q);
      }
      const float var = wave_sum64(q) / static_cast<float>(n_in);
      const float inv_std = 1.0f / sqrtf(var + eps);
#pragma unroll
      for (int i = 0; i < kCached; ++i) {
        if (4 * lane + 256 * i >= n_in) break;
#pragma unroll
        for (int j = 0; j < 4; ++j)
          v[i][j] = fmaf((v[i][j] - mean) * inv_std, gv[i][j], bv[i][j]);
      }
    }
#pragma unroll
    for (int i = 0; i < kCached; ++i) amax = fmaxf(amax, abs_max4(v[i]));  // zeros past n_in
  } else {
    for (int k = 4 * lane; k < n_in; k += 256)
      amax = fmaxf(amax, abs_max4(load4_dword_aligned(xr + k)));
  }
  amax = wave_max64(amax);
  const int e_max = static_cast<int>((__builtin_bit_cast(uint32_t, amax) >> 23) & 0xFF);
  const int sh = e_max == 0 ? 0 : clamp_exp(141 - e_max);
  const float up = pow2(sh);
  if constexpr (kCached > 0) {
#pragma unroll
    for (int i = 0; i < kCached; ++i) {
      const int k = 4 * lane + 256 * i;
      if (k < n_in) split_store4(v[i], up, dst + k, n_in);
    }
  } else {
    for (int k = 4 * lane; k < n_in; k += 256)
      split_store4(load4_dword_aligned(xr + k), up, dst + k, n_in);
  }
  if (lane == 0) row_scale[t] = pow2(clamp_exp(-sh));
}

}  // namespace

namespace {

// CUs of the current device, read once: asked for at each launch, this and the
// occupancy of the kernel cost 0.35 us of a 6.7 us call.
int linear_cus() {
  static const int cus = [] {
    int dev = 0, n = 256;
    if (hipGetDevice(&dev) == hipSuccess)
      (void)hipDeviceGetAttribute(&n, hipDeviceAttributeMultiprocessorCount, dev);
    return n;
  }();
  return cus;
}

}  // namespace

hipError_t launch_linear_split(const float* x, int64_t x_rs, int n_tokens, int n_in,
                               const float* ln_g, const float* ln_b, float ln_eps, _Float16* xs,
                               float* row_scale, hipStream_t s) {
  if (n_tokens <= 0) return hipSuccess;
  if (ln_g && n_in > kSplitLnMax) return hipErrorInvalidValue;
  const dim3 grid((n_tokens + 3) / 4), block(256);
#define WRS_SPLIT(C, LN)                                                                     \
  hipLaunchKernelGGL((linear_split_rows<C, LN>), grid, block, 0, s, x, x_rs, n_tokens, n_in, \
                     ln_g, ln_b, ln_eps, xs, row_scale)
  if (ln_g) {
    if (n_in <= 1280)
      WRS_SPLIT(5, true);
    else
      WRS_SPLIT(8, true);
  } else if (n_in <= 512) {
    WRS_SPLIT(2, false);
  } else if (n_in <= 1280) {
    WRS_SPLIT(5, false);
  } else if (n_in <= 5120) {
    WRS_SPLIT(20, false);
  } else {
    WRS_SPLIT(0, false);
  }
#undef WRS_SPLIT
  return hipGetLastError();
}

namespace {

// Which f32 products run on K7f (see there for both sides measured). Nothing but
// the shape of one weight group decides, so that a group of a call and a call of
// its own, and the fused and the separate LayerNorm and GELU, agree bit for bit.
bool gemv_by_fma(int n_tokens, int n_in, int n_out) {
  if (n_tokens <= 2) return true;
  // Short rows, against K7m: 3 rows up to 5120 features, 4 up to 2880, 5 up to 1843.
  // Six and more lose where a call has three groups of 512, 1024 or 1280.
  if (n_in <= 256 * kLnCache)
    return n_tokens <= 5 && static_cast<int64_t>(n_tokens) * n_tokens * n_out <= 9 * 5120;
  // Long rows, against K7l: 3 rows up to 3413 features, 5 up to 2048, 8 up to 1280.
  return static_cast<int64_t>(n_tokens) * n_out <= 10240;
}

}  // namespace

// Rows too long for a workgroup's registers, whose statistics and normalized values
// every workgroup of K7f forms again: over many features they are normalized once. us,
// in the kernel / in a launch of its own:
//   1 and 2 rows     2048 -> 5120 7.2/7.3 8.6/8.2, 2112 -> 5120 10.7/9.7 12.0/10.4
//   2 rows           3072 -> 4096 8.8/10.4, 5120 -> 5120 30.3/25.7
//   3, 4 and 5 rows  1344 -> 2560 6.6/7.3 7.3/7.9 8.4/8.8, -> 2 x 1664 7.6/7.7 8.6/8.1
//                    9.5/8.8; 2112 -> 2560 7.7/9.6 9.2/10.5 10.8/12.3, -> 2 x 1664
//                    11.6/10.2 13.1/11.1 14.1/11.9; 5120 -> 2048 19.1/15.6 20.1/17.2
//                    22.3/18.3
//   6 rows           2048 -> 3 x 1280 13.5/10.0, 2112 -> 2 x 1664 19.5/13.3
// K7l stages the rows per batch and gains up to 2048 columns only. Rows that fit gain
// from 3 rows on where a call has many groups (5 rows 384 -> 12 x 384 7.0/6.3, 768 -> 16
// x 768 14.0/10.0, 1280 -> 9 x 1280 16.5/13.6; a layer's three of 1280 7.7/7.3).
bool gemv_norms_apart(int n_tokens, int n_in, int n_out, int n_groups) {
  const int64_t features = static_cast<int64_t>(n_out) * n_groups, weights = features * n_in;
  if (n_tokens <= 2) return n_in > kGemvLnMax && features >= 5120 && weights > (10 << 20);
  if (!gemv_by_fma(n_tokens, n_in, n_out)) return false;
  return n_in > kGemvLnMax ? features >= 3072 || weights >= (10 << 20) : features >= 8192;
}

template <int kGroups>
hipError_t launch_gemv_f16w(const GemvArgs<kGroups>& a, DType x_dt, DType out_dt, hipStream_t s) {
  if (a.n_tokens <= 0 || a.n_out <= 0 || a.n_groups <= 0) return hipSuccess;
  if (a.n_tokens > kGemvMaxRows || a.n_groups > kGroups) return hipErrorInvalidValue;
  if (a.n_tokens * a.n_in > kGemvXFloats) return hipErrorInvalidValue;
  const int n_cu = linear_cus();
  int dev = 0;
  (void)hipGetDevice(&dev);
  // T features a workgroup: the CU's share, or an even part of it when that is more
  // than a workgroup takes.
  if (x_dt == kF32 && gemv_by_fma(a.n_tokens, a.n_in, a.n_out)) {
    const int n_slices = (a.n_in + 255) / 256;
    const int rounds = (n_slices + kGfWaves - 1) / kGfWaves;
    const int n_kw = (n_slices + rounds - 1) / rounds;
    const int waves = a.ln_g ? std::max(n_kw, a.n_tokens) : n_kw;
    const int64_t rows = static_cast<int64_t>(a.n_out) * a.n_groups;
    const int64_t share = std::max<int64_t>(1, (rows + n_cu - 1) / n_cu);
    const int64_t per_cu = (share + gf_rows(a.n_tokens) - 1) / gf_rows(a.n_tokens);
    const int T = static_cast<int>((share + per_cu - 1) / per_cu);
    const dim3 fgrid((a.n_out + T - 1) / T, a.n_groups), fblock(64 * waves);
#define WRS_GF_L(KERNEL)                                                   \
  {                                                                        \
    hipLaunchKernelGGL((KERNEL), fgrid, fblock, 0, s, a, T, n_kw, out_dt); \
    return hipGetLastError();                                              \
  }
#define WRS_GF_K(NT, R)                                                              \
  {                                                                                  \
    if (rounds > 1 && a.ln_g) WRS_GF_L((gemv_f16w_rows<NT, R, true, true, kGroups>)) \
    if (rounds > 1) WRS_GF_L((gemv_f16w_rows<NT, R, false, true, kGroups>))          \
    if (a.ln_g) WRS_GF_L((gemv_f16w_rows<NT, R, true, false, kGroups>))              \
    WRS_GF_L((gemv_f16w_rows<NT, R, false, false, kGroups>))                         \
  }
    switch (a.n_tokens) {
      case 1: if (T > 5) WRS_GF_K(1, 8) else WRS_GF_K(1, 5)
      case 2: if (T > 5) WRS_GF_K(2, 8) else WRS_GF_K(2, 5)
      case 3: WRS_GF_K(3, 5)
      case 4: WRS_GF_K(4, 5)
      case 5: WRS_GF_K(5, 5)
      case 6: WRS_GF_K(6, 5)
      case 7: WRS_GF_K(7, 5)
      case 8: WRS_GF_K(8, 5)
    }
#undef WRS_GF_K
#undef WRS_GF_L
  }
  // Three or more rows: the matrix-pipe kernels.
  const size_t gm_lds = static_cast<size_t>(x_dt == kF32 ? 2 : 1) * a.n_tokens * (a.n_in + 8) * 2;
  const bool long_rows = x_dt == kF32 && a.n_in > 256 * kLnCache;
  if (a.n_tokens >= 3 && (long_rows || (gm_lds <= kGmMaxDynLds && (x_dt == kF32 || x_dt == kF16)))) {
    // Tiles of T features, T chosen so that the tiles of all groups just
    // cover one workgroup per CU (a d x d matrix measured fastest that way:
    // two smaller tiles per CU stage x twice), or exactly k per CU when one
    // per CU would need more than 16 features: a 5120-row matrix in 16-feature
    // tiles gave 64 CUs two tiles and the rest one. Up to as many workgroups
    // as fit at once (LDS and registers decide) share the tiles, looping.
    const dim3 gblock(64 * kGmWaves);
    const int64_t rows = static_cast<int64_t>(a.n_out) * a.n_groups;
    const int64_t per_cu_tiles = (rows + 16 * n_cu - 1) / (16 * n_cu);
    const int T = static_cast<int>(std::max<int64_t>(
        1, std::min<int64_t>(16, (rows + per_cu_tiles * n_cu - 1) / (per_cu_tiles * n_cu))));
    const int n_tiles = (a.n_out + T - 1) / T;
    // Two workgroups of 8 waves fit a CU where their LDS does (the launch bounds
    // hold their registers to 128).
    const size_t lds = kGmStaticLds + (long_rows ? 0 : gm_lds);
    const int per_cu = long_rows || 2 * lds <= 160 * 1024 ? 2 : 1;
#define WRS_GM_K(KERNEL, LDS)                                                              \
  {                                                                                        \
    const void* fn = reinterpret_cast<const void*>(&KERNEL);                               \
    static std::atomic<uint64_t> attr_set{0};  /* one bit per device */                    \
    if (LDS > 0 && dev < 64 &&                                                             \
        !(attr_set.load(std::memory_order_acquire) & (uint64_t{1} << dev))) {              \
      const hipError_t e = hipFuncSetAttribute(                                            \
          fn, hipFuncAttributeMaxDynamicSharedMemorySize, static_cast<int>(kGmMaxDynLds)); \
      if (e != hipSuccess) return e;                                                       \
      attr_set.fetch_or(uint64_t{1} << dev, std::memory_order_acq_rel);                    \
    }                                                                                      \
    const dim3 ggrid(std::min(n_tiles, n_cu * per_cu), a.n_groups);                        \
    hipLaunchKernelGGL((KERNEL), ggrid, gblock, LDS, s, a, T);                             \
    return hipGetLastError();                                                              \
  }
#define WRS_GM(OT)                                                              \
  if (x_dt == kF16) {                                                           \
    if (a.ln_g) return hipErrorInvalidValue;  /* a fused LayerNorm takes f32 */ \
    WRS_GM_K((gemv_f16w_mfma<_Float16, OT, false, kGroups>), gm_lds)            \
  }                                                                             \
  if (long_rows && a.ln_g) WRS_GM_K((gemv_f16w_long<OT, true, kGroups>), 0)     \
  if (long_rows) WRS_GM_K((gemv_f16w_long<OT, false, kGroups>), 0)              \
  if (a.ln_g) WRS_GM_K((gemv_f16w_mfma<float, OT, true, kGroups>), gm_lds)      \
  WRS_GM_K((gemv_f16w_mfma<float, OT, false, kGroups>), gm_lds)
    switch (out_dt) {
      case kF32: WRS_GM(float)
      case kF16: WRS_GM(_Float16)
      case kBF16: WRS_GM(__bf16)
      default: return hipErrorInvalidValue;
    }
#undef WRS_GM
#undef WRS_GM_K
  }
  // What is left: one or two f16 rows. Up to kGemvSmallOut features: one feature
  // per wave, so that the matrix spreads over ~n_out / 8 CUs; beyond it 4 features
  // per wave share each staged x read.
  if (x_dt != kF16 || a.n_tokens > 2) return hipErrorInvalidValue;
  const int rpw = a.n_out <= kGemvSmallOut ? 1 : 4;
  const int groups = (a.n_out + rpw - 1) / rpw;
  const int wgs = std::min(n_cu, (groups + kGemvWaves - 1) / kGemvWaves);
  dim3 grid(std::max(wgs, 1), a.n_groups);
  dim3 block(64 * kGemvWaves);
#define WRS_GEMV(OT)                                                          \
  if (rpw == 1 && a.n_tokens == 1)                                            \
    hipLaunchKernelGGL((gemv_f16w<1, 1, OT, kGroups>), grid, block, 0, s, a); \
  else if (rpw == 1)                                                          \
    hipLaunchKernelGGL((gemv_f16w<2, 1, OT, kGroups>), grid, block, 0, s, a); \
  else if (a.n_tokens == 1)                                                   \
    hipLaunchKernelGGL((gemv_f16w<1, 4, OT, kGroups>), grid, block, 0, s, a); \
  else                                                                        \
    hipLaunchKernelGGL((gemv_f16w<2, 4, OT, kGroups>), grid, block, 0, s, a);
  switch (out_dt) {
    case kF32: WRS_GEMV(float) break;
    case kF16: WRS_GEMV(_Float16) break;
    case kBF16: WRS_GEMV(__bf16) break;
    default: return hipErrorInvalidValue;
  }
#undef WRS_GEMV
  return hipGetLastError();
}
template hipError_t launch_gemv_f16w(const GemvArgs<kFewGemvGroups>&, DType, DType, hipStream_t);
template hipError_t launch_gemv_f16w(const GemvArgs<kMaxLinearGroups>&, DType, DType, hipStream_t);

namespace {

int64_t n_tiles(const LinearArgs& a, int ft, int tt) {
  return static_cast<int64_t>((a.n_out + ft - 1) / ft) * ((a.n_tokens + tt - 1) / tt);
}

// k splits of 32 x 64 tiles: as many as fill the CUs once, each of at least 1024
// k. The merge costs a chain of memory round trips: 37 rows, f32: 5120 -> 1280
// takes 16.0 us in 5 splits, 29.6 in one pass of 64 x 64 tiles; 1280 -> 1280
// 11.6 in 6 splits and 11.4 without. By the shape of one group, so that a
// grouped call sums in the order of separate calls.
int linear_splits(const LinearArgs& a) {
  const int64_t t = n_tiles(a, 32, 64);
  const int64_t s = std::min<int64_t>({linear_cus() / std::max<int64_t>(t, 1), a.n_in / 1024,
                                       kLinMaxSplits});
  return static_cast<int>(std::max<int64_t>(s, 1));
}

template <typename OutT, class C>
hipError_t launch_tile(const LinearArgs& a, int splits, hipStream_t s) {
  const int64_t wgs = n_tiles(a, C::FT, C::TT) * splits * a.n_groups;
  if (wgs > 0x7fffffff) return hipErrorInvalidConfiguration;
  hipLaunchKernelGGL((linear_f16w<OutT, C>), dim3(static_cast<unsigned>(wgs)), dim3(C::kThreads),
                     0, s, a, splits);
  return hipGetLastError();
}

// A tile shape's time: fixed, `round` for every started round of one workgroup per
// CU, and `tile` for every workgroup, in units of us at n_in = 1280 (every shape
// grows alike with n_in, so one fit serves all), measured at 37 to 6000 rows
// and 384 to 5120 features, f32 output.
struct TileCost {
  int ft, tt;
  float fixed, round, tile;
};
float tile_cost(const LinearArgs& a, const TileCost& c) {
  const int64_t n = n_tiles(a, c.ft, c.tt) * a.n_groups, cus = linear_cus();
  return c.fixed + c.round * static_cast<float>((n + cus - 1) / cus) +
         c.tile * static_cast<float>(n);
}
template <size_t N>
int cheapest(const LinearArgs& a, const TileCost (&t)[N]) {
  int best = 0;
  for (size_t i = 1; i < N; ++i)
    if (tile_cost(a, t[i]) < tile_cost(a, t[best])) best = static_cast<int>(i);
  return best;
}

// Large tiles read the LDS least per MFMA but leave CUs idle on small grids: the
// 256 x 256 tile alone took 31 us for any call of up to 3000 x 1280 outputs over
// 1280 k (f16 x; 8 to 19 us with the shapes below).
template <typename OutT>
hipError_t launch_parts(const LinearArgs& a, int splits, hipStream_t s) {
  if (a.parts == 2) {
    // Long k on at most one workgroup per CU: nothing but the ring hides a stage's
    // way from memory, so it takes the whole LDS (weights not in any cache, us, 6
    // stages / 3: 37 x 5120 -> 1280 17.4/18.1, 200 x 5120 -> 1280 34.4/41.6, 37 x
    // 1536 -> 384 12.8/13.5). Up to 1280 k the longer fill costs what it gains (64 x
    // 384 -> 384 7.3/7.0, 64 x 1280 -> 1280 12.8/12.7), with one part too.
    const auto deep = [&](int ft, int n) {
      return a.n_in >= 1536 && n_tiles(a, ft, 64) * n * a.n_groups <= linear_cus();
    };
    if (splits > 1 && deep(32, splits))
      return launch_tile<OutT, LinTile<32, 64, 32, 32, 64, 6, 2>>(a, splits, s);
    if (splits > 1) return launch_tile<OutT, LinTile<32, 64, 32, 32, 64, 3, 2>>(a, splits, s);
    static constexpr TileCost kCosts[] = {{64, 64, 6.f, 9.3f, 0.f},
                                          {128, 64, 10.f, 13.f, 0.f},
                                          {128, 64, 12.f, 11.5f, 0.f},
                                          {256, 128, 18.f, 36.f, 0.f},
                                          {256, 256, 0.f, 42.f, 0.14f}};
    switch (cheapest(a, kCosts)) {
      case 0:
        if (deep(64, 1)) return launch_tile<OutT, LinTile<64, 64, 32, 32, 64, 6, 2>>(a, 1, s);
        return launch_tile<OutT, LinTile<64, 64, 32, 32, 64, 3, 2>>(a, 1, s);
      case 1: return launch_tile<OutT, LinTile<128, 64, 64, 32, 64, 4, 2>>(a, 1, s);
      case 2: return launch_tile<OutT, LinTile<128, 64, 64, 32, 64, 2, 2>>(a, 1, s);
      case 3: return launch_tile<OutT, LinTile<256, 128, 128, 64, 32, 2, 2>>(a, 1, s);
      default: return launch_tile<OutT, LinTile<256, 256, 128, 64, 32, 3, 2>>(a, 1, s);
    }
  }
  if (splits > 1) return launch_tile<OutT, LinTile<32, 64, 32, 32, 64, 4, 1>>(a, splits, s);
  static constexpr TileCost kCosts[] = {{64, 64, 3.f, 5.f, 0.f},
                                        {128, 64, 4.5f, 7.8f, 0.f},
                                        {128, 128, 8.5f, 11.5f, 0.f},
                                        {256, 256, 0.f, 24.f, 0.077f}};
  switch (cheapest(a, kCosts)) {
    case 0: return launch_tile<OutT, LinTile<64, 64, 32, 32, 64, 4, 1>>(a, 1, s);
    case 1: return launch_tile<OutT, LinTile<128, 64, 64, 32, 64, 3, 1>>(a, 1, s);
    case 2: return launch_tile<OutT, LinTile<128, 128, 64, 64, 64, 2, 1>>(a, 1, s);
    default:
      // Past one workgroup per CU the compiler's own order of a stage (all its
      // reads, then the MFMAs) keeps the two waves of a SIMD further apart:
      // 24000 x 3840 over 1280 k 246 against 277 us; 3000 x 3840, one round, 44.2
      // against 42.7 with slots.
      if (n_tiles(a, 256, 256) * a.n_groups > linear_cus())
        return launch_tile<OutT, LinTile<256, 256, 128, 64, 64, 2, 1, false>>(a, 1, s);
      return launch_tile<OutT, LinTile<256, 256, 128, 64, 64, 2, 1>>(a, 1, s);
  }
}

template <typename OutT>
hipError_t launch_groups(const LinearArgs& a, hipStream_t s) {
  const int splits = a.part ? linear_splits(a) : 1;
  // Groups that fit the split's scratch run together.
  int per = a.n_groups;
  if (splits > 1) {
    const int64_t t = n_tiles(a, 32, 64);
    per = static_cast<int>(std::min<int64_t>(
        {a.n_groups, static_cast<int64_t>(a.part_floats) / (t * splits * kLinPartFloats),
         static_cast<int64_t>(a.counter_words) / (t * kLinCounterStride)}));
    if (per < 1) return hipErrorInvalidValue;
  }
  if (per == a.n_groups) return launch_parts<OutT>(a, splits, s);
  for (int g0 = 0; g0 < a.n_groups; g0 += per) {
    LinearArgs b = a;
    b.n_groups = std::min(per, a.n_groups - g0);
    for (int g = 0; g < b.n_groups; ++g) {
      b.w[g] = a.w[g0 + g];
      b.bias[g] = a.bias[g0 + g];
      b.out[g] = a.out[g0 + g];
    }
    const hipError_t e = launch_parts<OutT>(b, splits, s);
    if (e != hipSuccess) return e;
  }
  return hipSuccess;
}

}  // namespace

hipError_t launch_linear_f16w(const LinearArgs& a, DType out_dt, hipStream_t s) {
  if (a.n_tokens <= 0 || a.n_out <= 0 || a.n_groups <= 0) return hipSuccess;
  switch (out_dt) {
    case kF32: return launch_groups<float>(a, s);
    case kF16: return launch_groups<_Float16>(a, s);
    case kBF16: return launch_groups<__bf16>(a, s);
    default: return hipErrorInvalidValue;
  }
}

bool linear_needs_split(const LinearArgs& a) { return linear_splits(a) > 1; }
// t tiles in s splits with t * s <= CUs and s >= 2, for four groups at once.
size_t linear_split_floats() {
  return static_cast<size_t>(4) * linear_cus() * kLinPartFloats;
}
size_t linear_split_words() {
  return static_cast<size_t>(4) * (linear_cus() / 2) * kLinCounterStride;
}

}  // namespace wrs
