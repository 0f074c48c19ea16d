// The prefill GEMM's main kernel (gemm.hip): the packed weights go from global
// memory straight into MFMA operand registers, only the activations pass
// through LDS.
//
// What bounds it: the matrix cores and, on grids that fill the chip, the power
// limit (the clock falls to ~1.85 GHz under this load), so every instruction
// and LDS byte beside the MFMAs costs clock.  A packed word is 8 consecutive k
// of one column, which is exactly one lane's B operand of
// v_mfma_f32_32x32x16_f16; with the waves of a workgroup side by side along N
// no two of them need the same word, so nothing is gained by staging B:
//   * each wave owns 64 columns (2 MFMA column tiles) and all 32 * TM rows of
//     the workgroup's tile; lane l of a wave holds the columns 2 (l % 32) and
//     2 (l % 32) + 1, one 8-byte load per 16 k, decoded in registers
//     (13 VALU ops a word) between the MFMAs of the slice before;
//   * activations are copied to LDS by LDS-DMA, a 64-k step (1 KiB per
//     instruction) at a time into a ring of 4, and read with ds_read_b128:
//     TM reads per 2 TM MFMAs;
//   * a step is four 16-k slices.  Slice s reads the activations and decodes
//     the words of slice s + 1 and issues a quarter of the loads of a later
//     step, interleaved with its own 2 TM MFMAs (sched_group_barrier);
//   * one barrier a step, before its last slice.  It orders two things: the
//     copies of the next step have landed (each wave waits for its own, vmcnt
//     leaving the younger steps' loads in flight), and every wave is past the
//     reads of the step before, whose buffer the next loads overwrite.  No
//     wave drains its LDS reads for it.
// Measured on MI355X against the kernel this replaced (producer / consumer
// waves, decoded B through LDS; same bits), weights from HBM, us: 512 x 4096 x
// 14336 (M x K x N) 71 -> 54.5, 2048 x 4096 x 14336 248 -> 197 (1.22 PFLOP/s;
// hipBLASLt's fp16 product 200), 2048 x 14336 x 4096 234 -> 193 (1.25; 216),
// 4096 x 14336 x 4096 440 -> 359 (1.34; 346).  What it took: loads spread over the slices instead of one burst a
// step, and the barrier without an LDS drain (one deeper ring), 212 -> 193 at
// 2048 x 14336 x 4096; the B words in LDS or three ring buffers lose.
#pragma once

#include <type_traits>

#include "nibble_common.h"
#include "nibble_decode.h"
#include "nibble_epilogue.h"
#include "stream_matmul.h"

namespace nibble {

namespace {

typedef float f16_t __attribute__((ext_vector_type(16)));

__device__ __forceinline__ f16_t mfma32(h8_t a, h8_t b, f16_t c) {
  return __builtin_amdgcn_mfma_f32_32x32x16_f16(a, b, c, 0, 0, 0);
}

constexpr int kDirectStep = 64;            // k per step
constexpr int kDirectRing = 4;             // activation buffers (and word sets) per team
constexpr int kDirectMaxSplitTM = 3;       // larger tiles are never split over K
constexpr int kPolicyCoherent = 16;        // sc1: the cache policy of an agent-scope access
constexpr int kDirectGroupM = 8;           // row tiles per block of the tile order

struct DirectArgs {
  const _Float16* X;
  const uint32_t* Wq;
  const _Float16* S;
  _Float16* Y;
  const _Float16* bias;  // epilogue kEpilogueBias
  float* partial;        // [splits, M, N] fp32 when splits > 1
  uint32_t* counters;    // [tiles], zero on entry and on exit
  int M, K, N;
  int tiles_m, tiles_n;
  int splits, steps_per_split;  // 64-k steps per K split
  int epilogue;
  WeightLayout L;  // where a column's words and scales live (packed or strip-major)
};

// COPIES LDS-DMA copies of 1 KiB (16 bytes a lane) to LDS byte address dst,
// 1 KiB apart; lane offsets voff (out of range: no access).  Written as
// assembly because the compiler, knowing a pending LDS-DMA, waits for it
// before every LDS read it cannot tell apart (vmcnt(1) in some slices, a whole
// memory round trip); the kernel's own waits order the copies.  No register
// is written; addresses are read at issue.
template <int COPIES>
__device__ __forceinline__ void direct_copy(const void* X, uint32_t xbytes, uint32_t dst,
                                            const uint32_t* voff, uint32_t soff) {
  const uint64_t base = reinterpret_cast<uint64_t>(X);
  const u4_t rsrc = {static_cast<uint32_t>(base), static_cast<uint32_t>(base >> 32) & 0xffffu,
                     xbytes, 0x00020000u};
#pragma unroll
  for (int j = 0; j < COPIES; ++j)
    asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tbuffer_load_dwordx4 %1, %2, %3 offen lds"
                 :
                 : "s"(dst + j * 1024u), "v"(voff[j]), "s"(rsrc), "s"(soff)
                 : "memory", "m0");
}
__device__ __forceinline__ u2_t direct_words(const void* p, uint32_t bytes, uint32_t v,
                                             uint32_t s) {
  return __builtin_bit_cast(u2_t,
                            __builtin_amdgcn_raw_buffer_load_b64(make_rsrc(p, bytes), v, s, 0));
}
__device__ __forceinline__ h2_t direct_scales(const void* p, uint32_t bytes, uint32_t v,
                                              uint32_t s) {
  return as_h2(__builtin_amdgcn_raw_buffer_load_b32(make_rsrc(p, bytes), v, s, 0));
}

// The instruction mix of one slice: per MFMA an LDS read (the first TM), a
// share of the decode, a load (the rest).
template <int TM>
__device__ __forceinline__ void direct_interleave() {
#pragma unroll
  for (int i = 0; i < 2 * TM; ++i) {
    __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);  // MFMA
    if (i < TM) __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);  // LDS read
    __builtin_amdgcn_sched_group_barrier(0x002, 13 / TM + 1, 0);    // VALU
    if (i >= TM) __builtin_amdgcn_sched_group_barrier(0x010, 1, 0);  // vector memory
  }
}

// A barrier that waits for no memory operation (the caller's explicit waits
// order what has to be).
__device__ __forceinline__ void direct_barrier() {
  __atomic_signal_fence(__ATOMIC_SEQ_CST);
  __builtin_amdgcn_sched_barrier(0);
  __builtin_amdgcn_s_barrier();
  __builtin_amdgcn_sched_barrier(0);
  __atomic_signal_fence(__ATOMIC_SEQ_CST);
}

// 16-byte unit of k-unit c of tile row r: XOR-swizzled so that the 16 rows a
// ds_read_b128 phase touches cover all 64 banks once (8 rows: 32 banks).
__device__ __forceinline__ int direct_swizzle(int r) { return (r & 7) ^ ((r >> 3) & 1); }

// exact fp16((n - 8) * s) of a word's 8 weights (decode8_scaled with the
// constants kept in registers): one MFMA B-operand lane.
__device__ __forceinline__ h8_t direct_decode(uint32_t q, _Float16 s, const DecodeConsts& k) {
  uint32_t r[4];
  decode8_raw(q, r, k);
  const h2_t s2 = {s, s};
  const h2_t bias_lo = {(_Float16)1032.0f, (_Float16)1032.0f};
  const h2_t mul_hi = {(_Float16)0.0625f, (_Float16)0.0625f};
  const h2_t bias_hi = {(_Float16)-72.0f, (_Float16)-72.0f};
  const u4_t v = {as_u32((as_h2(r[0]) - bias_lo) * s2),
                  as_u32(__builtin_elementwise_fma(as_h2(r[1]), mul_hi, bias_hi) * s2),
                  as_u32((as_h2(r[2]) - bias_lo) * s2),
                  as_u32(__builtin_elementwise_fma(as_h2(r[3]), mul_hi, bias_hi) * s2)};
  return __builtin_bit_cast(h8_t, v);
}

// Two adjacent fp16 outputs at byte offset off of a resource: one 4-byte store
// where Y is 4-byte aligned (`pairs`), else two of 2 bytes.  Offsets past the
// resource (rows past M, columns past N) store nothing.
__device__ __forceinline__ void direct_store2(__amdgpu_buffer_rsrc_t r, uint32_t off, float a,
                                              float b, bool pairs) {
  const _Float16 y0 = (_Float16)a, y1 = (_Float16)b;
  if (pairs) {
    __builtin_amdgcn_raw_buffer_store_b32(as_u32(h2_t{y0, y1}), r, off, 0, 0);
  } else {
    __builtin_amdgcn_raw_buffer_store_b16(__builtin_bit_cast(uint16_t, y0), r, off, 0, 0);
    __builtin_amdgcn_raw_buffer_store_b16(__builtin_bit_cast(uint16_t, y1), r, off + 2, 0, 0);
  }
}
__device__ __forceinline__ float direct_bias(float v, _Float16 b) {
  return static_cast<float>(static_cast<_Float16>(v)) + static_cast<float>(b);
}

// The output rows of a tile from m0 on as a resource (out_n columns a row; at
// most BM rows, so its offsets fit 32 bits whatever M).
__device__ __forceinline__ __amdgpu_buffer_rsrc_t direct_out(const DirectArgs& args, int m0,
                                                             int out_n, int bm) {
  return make_rsrc(args.Y + static_cast<size_t>(m0) * out_n,
                   static_cast<uint32_t>(min(bm, args.M - m0)) * static_cast<uint32_t>(out_n) * 2u);
}

// Last-arriver sum of a split tile by the whole workgroup: each thread takes
// chunks of VEC columns (4, or 2 where N % 4 != 0; whole 16-column blocks of
// gate and the matching up for SwiGLU), loads the chunk's partial of every
// split (up to 4 in one round) with the device-coherent policy, adds them in
// split order and writes the outputs.  Needs M * N * 4 < 2^31 (32-bit offsets;
// the plans split only grids of a few hundred tiles).
template <int VEC>
struct PartialVec;
template <>
struct PartialVec<4> {
  using type = f4_t;
  static __device__ __forceinline__ type load(const void* p, uint32_t bytes, uint32_t off) {
    return __builtin_bit_cast(
        f4_t, __builtin_amdgcn_raw_buffer_load_b128(make_rsrc(p, bytes), off, 0, kPolicyCoherent));
  }
};
typedef float f2_t __attribute__((ext_vector_type(2)));
template <>
struct PartialVec<2> {
  using type = f2_t;
  static __device__ __forceinline__ type load(const void* p, uint32_t bytes, uint32_t off) {
    return __builtin_bit_cast(
        f2_t, __builtin_amdgcn_raw_buffer_load_b64(make_rsrc(p, bytes), off, 0, kPolicyCoherent));
  }
};

template <int THREADS, int BM, int BN, int VEC>
__device__ __forceinline__ void direct_sum_splits(const DirectArgs& args, int m0, int n0) {
  using P = PartialVec<VEC>;
  using vec = typename P::type;
  constexpr int kBatch = 4, kPair = 2;
  constexpr int CHUNKS = BM * BN / VEC;
  static_assert(CHUNKS % (THREADS * kPair) == 0, "whole rounds");
  const int M = args.M, N = args.N;
  const uint32_t plane = static_cast<uint32_t>(M) * static_cast<uint32_t>(N);
  const bool swiglu = args.epilogue == kEpilogueSwiglu;
  const bool add = args.epilogue == kEpilogueBias;
  const bool pairs = (reinterpret_cast<uintptr_t>(args.Y) & 3u) == 0;
  const __amdgpu_buffer_rsrc_t ry = direct_out(args, m0, swiglu ? N / 2 : N, BM);
  // A thread takes two chunks a round: SwiGLU a gate chunk and the up chunk 16
  // columns on, otherwise chunks THREADS apart.  Chunks outside Y load zeros
  // and store nothing (out-of-range offsets).
#pragma nounroll
  for (int c0 = 0; c0 < CHUNKS / kPair; c0 += THREADS) {
    uint32_t off[kPair], dst[kPair];
    int gn[kPair];
#pragma unroll
    for (int u = 0; u < kPair; ++u) {
      const int c = c0 + static_cast<int>(threadIdx.x);
      int row, tc;  // row and column in the tile
      if (swiglu) {
        constexpr int per_row = BN / 2 / VEC;
        row = c / per_row;
        const int g = VEC * (c % per_row);
        tc = g / kSwigluBlock * 2 * kSwigluBlock + g % kSwigluBlock + u * kSwigluBlock;
      } else {
        constexpr int per_row = BN / VEC;
        const int cc = c0 * kPair + u * THREADS + static_cast<int>(threadIdx.x);
        row = cc / per_row;
        tc = VEC * (cc % per_row);
      }
      const int gm = m0 + row;
      gn[u] = n0 + tc;
      const bool in = gm < M && gn[u] < N;
      off[u] = in ? (static_cast<uint32_t>(gm) * N + gn[u]) * 4u : kOutOfRange;
      const uint32_t ocol = swiglu ? n0 / 2 + VEC * (c % (BN / 2 / VEC)) : gn[u];
      dst[u] = in ? (static_cast<uint32_t>(row) * (swiglu ? N / 2 : N) + ocol) * 2u : kOutOfRange;
    }
    vec s[kPair] = {};
    for (int sp0 = 0; sp0 < args.splits; sp0 += kBatch) {
      vec v[kBatch][kPair];
#pragma unroll
      for (int b = 0; b < kBatch; ++b) {
        const int sp = sp0 + b < args.splits ? sp0 + b : 0;
#pragma unroll
        for (int u = 0; u < kPair; ++u)
          v[b][u] = P::load(args.partial + static_cast<size_t>(sp) * plane, plane * 4u, off[u]);
      }
#pragma unroll
      for (int b = 0; b < kBatch; ++b)
        if (sp0 + b < args.splits) {
#pragma unroll
          for (int u = 0; u < kPair; ++u)
#pragma unroll
            for (int e = 0; e < VEC; ++e) s[u][e] += v[b][u][e];
        }
    }
    if (swiglu) {
#pragma unroll
      for (int e = 0; e < VEC; e += 2)
        direct_store2(ry, dst[0] + 2u * e, silu_mul(s[0][e], s[1][e]),
                      silu_mul(s[0][e + 1], s[1][e + 1]), pairs);
      continue;
    }
#pragma unroll
    for (int u = 0; u < kPair; ++u)
#pragma unroll
      for (int e = 0; e < VEC; e += 2) {
        float y0 = s[u][e], y1 = s[u][e + 1];
        if (add && dst[u] != kOutOfRange) {
          y0 = direct_bias(y0, args.bias[gn[u] + e]);
          y1 = direct_bias(y1, args.bias[gn[u] + e + 1]);
        }
        direct_store2(ry, dst[u] + 2u * e, y0, y1, pairs);
      }
  }
}

// One (32 TM) x (64 WN) output tile (and K split) per workgroup of KW teams of
// WN waves.  The teams split the workgroup's K range evenly, each with its own
// ring; their sums meet in LDS in team order at the end.  Teams pay for small
// batches: the CUs are filled with narrow tiles instead of K splits, whose
// partials cross HBM, and a second wave per SIMD hides a step's decode and
// barrier (256 x 4096 x 4096, us: TM = 2, WN = 4 with one team 29.3, with two
// 25.1; TM = 1, WN = 2 with four 14.9).  A large TM hides them behind its own
// MFMAs and reads each activation for 256 columns.  Workgroups take tiles in
// blocks of 8 row tiles, eighths of the order to each XCD.
template <int TM, int KW, int WN, int GROUP, int OCC>
__global__ __launch_bounds__(KW* WN * 64, OCC) void gemm_direct_kernel(DirectArgs args) {
  constexpr int BM = 32 * TM, BN = 64 * WN, BUF = BM * kDirectStep, RING = kDirectRing, D = RING - 1;
  constexpr int THREADS = KW * WN * 64;
  constexpr int COPIES = BM / 8 / WN;  // 1 KiB copies per wave and step
  constexpr int LOADS = COPIES + 5;  // and 4 word loads, 1 scale load
  static_assert(GROUP % kDirectStep == 0, "one scale per column per step");
  static_assert((D - 2) * LOADS + 10 + COPIES / 4 <= 63, "vmcnt range");
  static_assert(KW == 1 || BM * BN * 4 <= KW * RING * BUF * 2, "team sums fit the rings");
  __shared__ __attribute__((aligned(16))) _Float16 lds[KW * RING * BUF];
  __shared__ int s_last;
  const int M = args.M, K = args.K, N = args.N;
  const int lane = static_cast<int>(threadIdx.x) & 63;
  const int wid = __builtin_amdgcn_readfirstlane(static_cast<int>(threadIdx.x) >> 6);
  const int team = KW == 1 ? 0 : wid / WN, wave = wid % WN;
  _Float16* const As = lds + team * RING * BUF;
  const uint32_t as_base = static_cast<uint32_t>(reinterpret_cast<uintptr_t>(
      (__attribute__((address_space(3))) void*)As));

  // Workgroup -> (split, tile): XCD id % 8 takes one contiguous share of the
  // order; within it 8 row tiles share each column tile's words in L2.
  const uint32_t tiles = static_cast<uint32_t>(args.tiles_m) * args.tiles_n;
  const uint32_t total = tiles * args.splits;
  const uint32_t xcd = blockIdx.x & 7u;
  const uint32_t seq = xcd * (total >> 3) + min(xcd, total & 7u) + (blockIdx.x >> 3);
  const int split = static_cast<int>(seq / tiles);
  const uint32_t in_split = seq - split * tiles;
  const uint32_t block = in_split / (kDirectGroupM * args.tiles_n);
  const uint32_t in_block = in_split - block * (kDirectGroupM * args.tiles_n);
  const uint32_t rows_in = min(static_cast<uint32_t>(kDirectGroupM),
                               args.tiles_m - block * kDirectGroupM);
  const int tile_n = static_cast<int>(in_block / rows_in);
  const int tile_m = static_cast<int>(block * kDirectGroupM + in_block - tile_n * rows_in);
  const int m0 = tile_m * BM, n0 = tile_n * BN;

  // The split's steps, shared out to the teams (the first may take one more).
  const int first = split * args.steps_per_split;
  const int steps = min(args.steps_per_split, K / kDirectStep - first);
  const int per_team = (steps + KW - 1) / KW;
  const int step0 = first + team * per_team;
  const int ntiles = max(0, min(per_team, steps - team * per_team));

  const int c32 = lane & 31, half = lane >> 5;
  const int col = n0 + 64 * wave + 2 * c32;  // N is even: both columns inside or outside
  const uint32_t row_bytes = args.L.w_row;
  const uint32_t xbytes = static_cast<uint32_t>(M) * static_cast<uint32_t>(K) * 2u;
  const uint32_t wbytes = static_cast<uint32_t>(K / 8) * static_cast<uint32_t>(N) * 4u;
  const uint32_t sbytes = static_cast<uint32_t>(K / GROUP) * static_cast<uint32_t>(N) * 2u;
  const uint32_t voff_b = col < N ? half * row_bytes + args.L.wcol(col) : kOutOfRange;
  const uint32_t voff_s = col < N ? args.L.scol(col) : kOutOfRange;
  // Copy j of this wave fills 8 tile rows; rows past M are not read (their
  // LDS holds anything: an output row depends on its own activation row
  // alone, and those are not stored).
  uint32_t voff_a[COPIES];
#pragma unroll
  for (int j = 0; j < COPIES; ++j) {
    const int r = 8 * (wave * COPIES + j) + (lane >> 3);
    const int c = (lane & 7) ^ direct_swizzle(r);
    const int gm = m0 + r;
    voff_a[j] = gm < M ? static_cast<uint32_t>(gm) * K * 2u + c * 16u : kOutOfRange;
  }

  struct Words {
    u2_t w[4];  // per slice: columns col, col + 1 of packed row 2 slice + half
    h2_t s;
  };
  Words R[RING];
  // Part p (a quarter) of the copies of a step, and of its words: slice p's,
  // with part 0 the scales.  Steps past the last read through empty resources
  // (no access: gfx950's range check takes the scalar offset in without
  // wrapping), so every wave's count of loads in flight stays exact.
  auto copy_part = [&](auto pc, int step, int buf) {
    constexpr int p = decltype(pc)::value;
    constexpr int c0 = p * COPIES / 4, c1 = (p + 1) * COPIES / 4;
    const bool in = step < ntiles;
    const uint32_t k0 = in ? static_cast<uint32_t>(step0 + step) * kDirectStep : 0u;
    if constexpr (c1 > c0)
      direct_copy<c1 - c0>(args.X, in ? xbytes : 0u,
                           as_base + (buf * BUF + (wave * COPIES + c0) * 512) * 2u, voff_a + c0,
                           k0 * 2u);
  };
  auto word_part = [&](auto pc, Words& st, int step) {
    constexpr int p = decltype(pc)::value;
    const bool in = step < ntiles;
    const uint32_t k0 = in ? static_cast<uint32_t>(step0 + step) * kDirectStep : 0u;
    st.w[p] = direct_words(args.Wq, in ? wbytes : 0u, voff_b, (k0 / 8 + 2 * p) * row_bytes);
    if constexpr (p == 0)
      st.s = direct_scales(args.S, in ? sbytes : 0u, voff_s, (k0 / GROUP) * args.L.s_row);
  };

  f16_t acc[TM][2];
#pragma unroll
  for (int i = 0; i < TM; ++i)
#pragma unroll
    for (int j = 0; j < 2; ++j)
#pragma unroll
      for (int r = 0; r < 16; ++r) acc[i][j][r] = 0.0f;

  // Row c32 of the first row tile, k-unit 2 slice + half: rows 32 apart share
  // the swizzle, so the other row tiles and buffers are constant offsets.
  int rda[4];
#pragma unroll
  for (int ks = 0; ks < 4; ++ks)
    rda[ks] = c32 * kDirectStep + (((2 * ks + half) ^ direct_swizzle(c32)) * 8);
  const DecodeConsts dk = decode_consts();
  h8_t a[2][TM], b[2][2];
  auto read_a = [&](h8_t (&dst)[TM], int buf, int ks) {
#pragma unroll
    for (int i = 0; i < TM; ++i)
      dst[i] = *reinterpret_cast<const h8_t*>(As + buf * BUF + rda[ks] + i * 32 * kDirectStep);
  };
  using I0 = std::integral_constant<int, 0>;
  using I1 = std::integral_constant<int, 1>;
  using I2 = std::integral_constant<int, 2>;
  using I3 = std::integral_constant<int, 3>;

  // Words of steps 0 .. 3, copies of steps 0 and 1 and part 0 of step 2: where
  // the loop is when it enters slice 0 of step 0.
#pragma unroll
  for (int u = 0; u < RING; ++u) {
    word_part(I0{}, R[u], u);
    word_part(I1{}, R[u], u);
    word_part(I2{}, R[u], u);
    word_part(I3{}, R[u], u);
    __builtin_amdgcn_sched_barrier(0);
    if (u < D - 1) {
      copy_part(I0{}, u, u);
      copy_part(I1{}, u, u);
      copy_part(I2{}, u, u);
      copy_part(I3{}, u, u);
    }
    __builtin_amdgcn_sched_barrier(0);
  }
  copy_part(I0{}, D - 1, D - 1);
  __builtin_amdgcn_sched_barrier(0);
  __builtin_amdgcn_s_waitcnt(waitcnt_vm((D - 2) * LOADS + 10 + COPIES / 4));
  direct_barrier();
  read_a(a[0], 0, 0);
#pragma unroll
  for (int j = 0; j < 2; ++j) b[0][j] = direct_decode(R[0].w[0][j], R[0].s[j], dk);

  // Slice ks of step t, in buffer u.  Copies go three steps ahead, into the
  // buffer of step t - 1: part 0 of step t + 3 in slice 3, after the barrier,
  // the other parts in slices 0 to 2 of the next step.  Words go four ahead,
  // into the registers of the words just decoded: the compiler counts only the
  // word loads when it waits for one, and with a step more between them that
  // wait is never stricter than the barrier's.
  // The steps after the last whole round (`tail`) wait for every load: their
  // own loads are for steps that may not exist, whose words nobody uses, so
  // the compiler drops some and a count would let too many stay in flight.
  auto slice = [&](auto kc, auto uc, auto tail, int t) {
    constexpr int ks = decltype(kc)::value, u = decltype(uc)::value;
    constexpr int cur = ks & 1;
    constexpr int ru = ks < 3 ? u : (u + 1) % RING, rk = (ks + 1) % 4;  // the next slice
      constexpr int cu = (ks < 3 ? u + RING - 2 : u + RING - 1) % RING;   // the copies' buffer
    if constexpr (ks == 3) {
      __builtin_amdgcn_s_waitcnt(waitcnt_vm(decltype(tail)::value ? 0 : (D - 2) * LOADS));
      direct_barrier();
    }
    read_a(a[cur ^ 1], ru, rk);
#pragma unroll
    for (int j = 0; j < 2; ++j) b[cur ^ 1][j] = direct_decode(R[ru].w[rk][j], R[ru].s[j], dk);
    copy_part(std::integral_constant<int, rk>{}, (ks < 3 ? t - 1 : t) + D, cu);
    word_part(std::integral_constant<int, rk>{}, R[u], t + RING);
#pragma unroll
    for (int i = 0; i < TM; ++i)
#pragma unroll
      for (int j = 0; j < 2; ++j) acc[i][j] = mfma32(a[cur][i], b[cur][j], acc[i][j]);
    direct_interleave<TM>();
    __builtin_amdgcn_sched_barrier(0);
  };
  auto step = [&](auto uc, auto tail, int t) {
    slice(I0{}, uc, tail, t);
    slice(I1{}, uc, tail, t);
    slice(I2{}, uc, tail, t);
    slice(I3{}, uc, tail, t);
  };
  // Whole rounds of the ring with no exit in the middle (each exit would keep
  // a copy of the accumulators), then the remaining 0..3 steps.
  int t = 0;
  for (; t + RING <= ntiles; t += RING) {
    step(I0{}, std::false_type{}, t);
    step(I1{}, std::false_type{}, t + 1);
    step(I2{}, std::false_type{}, t + 2);
    step(I3{}, std::false_type{}, t + 3);
  }
  if (t < ntiles) step(I0{}, std::true_type{}, t);
  if (t + 1 < ntiles) step(I1{}, std::true_type{}, t + 1);
  if (t + 2 < ntiles) step(I2{}, std::true_type{}, t + 2);
  // Every wave of the workgroup passes the same number of barriers.
  for (int e = ntiles; e < per_team; ++e) direct_barrier();
  // No copy may land after the LDS is reused or given away.
  __builtin_amdgcn_s_waitcnt(waitcnt_vm(0));

  if constexpr (KW > 1) {
    __syncthreads();
    f4_t* xch = reinterpret_cast<f4_t*>(lds) + wave * TM * 2 * 4 * 64 + lane;
#pragma unroll
    for (int k = 1; k < KW; ++k) {
      if (team == k) {
#pragma unroll
        for (int i = 0; i < TM; ++i)
#pragma unroll
          for (int j = 0; j < 2; ++j)
#pragma unroll
            for (int q = 0; q < 4; ++q)
              xch[((i * 2 + j) * 4 + q) * 64] = f4_t{acc[i][j][4 * q], acc[i][j][4 * q + 1],
                                                     acc[i][j][4 * q + 2], acc[i][j][4 * q + 3]};
      }
      __syncthreads();
      if (team == 0) {
#pragma unroll
        for (int i = 0; i < TM; ++i)
#pragma unroll
          for (int j = 0; j < 2; ++j)
#pragma unroll
            for (int q = 0; q < 4; ++q) {
              const f4_t v = xch[((i * 2 + j) * 4 + q) * 64];
#pragma unroll
              for (int e = 0; e < 4; ++e) acc[i][j][4 * q + e] += v[e];
            }
      }
      if (k + 1 < KW) __syncthreads();
    }
  }

  // Result register r of lane l: column tile j's column l % 32 (output column
  // col + j), row 8 (r / 4) + 4 (l / 32) + r % 4 of row tile i.
  const int rq = half * 4;
  if (TM > kDirectMaxSplitTM || args.splits == 1) {
    if (team != 0) return;
    const bool pairs = (reinterpret_cast<uintptr_t>(args.Y) & 3u) == 0;
    if (args.epilogue == kEpilogueSwiglu) {
      // Gate and up columns sit 16 apart, in lanes 8 apart of a 16-lane row.
      // Of each pair of rows the gate lane finishes the first and the up lane
      // the second, after one exchange.
      const bool gate = (lane & 8) == 0;
      const uint32_t out_n = static_cast<uint32_t>(N) / 2;
      const uint32_t ocol = (n0 + 64 * wave) / 2 + (c32 >> 4) * kSwigluBlock + 2 * (c32 & 7);
      const __amdgpu_buffer_rsrc_t ry = direct_out(args, m0, N / 2, BM);
      const uint32_t base = col < N ? ((rq + (gate ? 0 : 1)) * out_n + ocol) * 2u : kOutOfRange;
      auto emit = [&](auto whole) {
#pragma unroll
        for (int i = 0; i < TM; ++i)
#pragma unroll
          for (int r = 0; r < 16; r += 2) {
            float y[2];
#pragma unroll
            for (int j = 0; j < 2; ++j) {
              const float mine = gate ? acc[i][j][r] : acc[i][j][r + 1];
              const float give = gate ? acc[i][j][r + 1] : acc[i][j][r];
              const float got = __builtin_bit_cast(
                  float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, give), 0x128, 0xf,
                                                     0xf, true));  // row_ror:8
              y[j] = silu_mul(gate ? mine : got, gate ? got : mine);
            }
            direct_store2(ry, base + (32 * i + 8 * (r >> 2) + (r & 3)) * out_n * 2u, y[0], y[1],
                          decltype(whole)::value);
          }
      };
      if (pairs)
        emit(std::true_type{});
      else
        emit(std::false_type{});
      return;
    }
    const bool in = col < N;
    const __amdgpu_buffer_rsrc_t ry = direct_out(args, m0, N, BM);
    const uint32_t base = in ? (static_cast<uint32_t>(rq) * N + col) * 2u : kOutOfRange;
    auto emit = [&](auto whole, auto add) {
      constexpr bool kAdd = decltype(add)::value;
      const _Float16 b0 = kAdd && in ? args.bias[col] : (_Float16)0.0f;
      const _Float16 b1 = kAdd && in ? args.bias[col + 1] : (_Float16)0.0f;
#pragma unroll
      for (int i = 0; i < TM; ++i)
#pragma unroll
        for (int r = 0; r < 16; ++r)
          direct_store2(ry,
                        base + static_cast<uint32_t>(32 * i + 8 * (r >> 2) + (r & 3)) * N * 2u,
                        kAdd ? direct_bias(acc[i][0][r], b0) : acc[i][0][r],
                        kAdd ? direct_bias(acc[i][1][r], b1) : acc[i][1][r],
                        decltype(whole)::value);
    };
    const bool add = args.epilogue == kEpilogueBias;
    if (pairs && !add)
      emit(std::true_type{}, std::false_type{});
    else if (pairs)
      emit(std::true_type{}, std::true_type{});
    else if (!add)
      emit(std::false_type{}, std::false_type{});
    else
      emit(std::false_type{}, std::true_type{});
    return;
  }

  // K split: publish this split's fp32 tile with device-coherent stores; the
  // last workgroup of the tile (agent-scope counter) sums the splits in split
  // order and writes Y -- deterministic, one launch.  Relies on gfx950
  // hardware ordering: see "HARDWARE ASSUMPTION" in nibble_decode.h.
  if (team == 0) {
    const __amdgpu_buffer_rsrc_t rp =
        make_rsrc(args.partial + (static_cast<size_t>(split) * M + m0) * N,
                  static_cast<uint32_t>(min(BM, M - m0)) * static_cast<uint32_t>(N) * 4u);
    const uint32_t base = col < N ? (static_cast<uint32_t>(rq) * N + col) * 4u : kOutOfRange;
#pragma unroll
    for (int i = 0; i < TM; ++i)
#pragma unroll
      for (int r = 0; r < 16; ++r) {
        const f2_t v = {acc[i][0][r], acc[i][1][r]};
        __builtin_amdgcn_raw_buffer_store_b64(
            __builtin_bit_cast(u2_t, v), rp,
            base + static_cast<uint32_t>(32 * i + 8 * (r >> 2) + (r & 3)) * N * 4u, 0,
            kPolicyCoherent);
      }
  }
  wait_vm_stores();
  __syncthreads();
  uint32_t* counter = args.counters + tile_n * args.tiles_m + tile_m;
  if (threadIdx.x == 0) {
    const uint32_t prev =
        __hip_atomic_fetch_add(counter, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    s_last = prev == static_cast<uint32_t>(args.splits - 1);
  }
  __syncthreads();
  if (!s_last) return;
  if (N % 4 == 0)
    direct_sum_splits<THREADS, BM, BN, 4>(args, m0, n0);
  else
    direct_sum_splits<THREADS, BM, BN, 2>(args, m0, n0);
  if (threadIdx.x == 0)
    __hip_atomic_store(counter, 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

}  // namespace

}  // namespace nibble
