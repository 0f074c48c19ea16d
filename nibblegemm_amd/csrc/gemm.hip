// Prefill-regime W4A16 matmul on CDNA4 MFMA: Y[M,N] = X[M,K] @ dequant(Wq, S).
//
// Reference: csrc/gemm_w4a16.cu (tile staging :66-146, kernels :151-377, host
// checks :379-429).  The reference decodes B into shared memory and feeds
// wmma / mma.sync; here the tile feeds v_mfma_f32_32x32x16_f16.
//
// Two kernels.  The direct kernel (gemm_direct.h) runs nearly everything;
// gemm_tile_kernel, described here, the operands it does not take (weights or
// scales not aligned for loads of two columns, widths past its offsets).
//
// Tile: BM x BN x 32 per workgroup of 4 wave64s (2 x 2), each wave owning a
// (BM/2) x (BN/2) block of 32 x 32 MFMA tiles.  Per 32-k step:
//   * A (X, fp16): 16-byte global loads into registers, rows past M read as
//     zero, then stored to LDS;
//   * B: each thread loads BN/64 adjacent packed words of one packed row (a
//     wave covers one packed row of the tile, 4*BN contiguous bytes).  Every
//     word is exactly 8 consecutive k of one column: it is decoded with the
//     magic-exponent trick and multiplied by the group scale (one RNE
//     rounding, so the LDS tile holds exactly dequantize()'s fp16 values, as
//     the reference's does, gemm_w4a16.cu:137-146) and stored n-major
//     (k contiguous) with one 16-byte LDS store -- one MFMA B-operand lane;
//   * the next step's global loads are issued before the current step's
//     MFMAs and written to the other LDS buffer after them: one barrier per
//     step;
//   * each wave reads its operands with ds_read_b128 (the swizzled layout of
//     lds_unit keeps reads and stores free of bank conflicts) and issues
//     (BM/64) x (BN/64) MFMAs per 16 k with fp32 accumulation.
//
// MFMA operand layout (32x32x16 f16): lane l supplies row (A) / column (B)
// l % 32 and the 8 k of block l / 32; result register r of lane l holds
// column l % 32, row 8 * (r / 4) + 4 * (l / 32) + r % 4.
#include <algorithm>
#include <type_traits>

#include "gemm_direct.h"
#include "nibble_common.h"
#include "nibble_decode.h"
#include "stream_matmul.h"

namespace nibble {

namespace {

constexpr int BK = 32;
// LDS tile layout.  A tile row (an A row or a B column) holds BK = 32 fp16
// as four 16-byte units, rows 64 bytes apart with no padding.  Rows are
// permuted within aligned groups of four and the units of a row XOR-swizzled,
// both by low row bits, so that every 16-lane phase of the three access
// patterns touches 16 distinct units -- all 64 banks once -- (and every
// 8-lane phase all of 32 banks once):
//   * operand reads: 16 consecutive rows, one unit each;
//   * A stores: 4 consecutive rows, all 4 units each;
//   * B stores: 16 rows 1 or 2 apart (a lane's 1 or 2 adjacent columns), one
//     unit each -- with a 64-byte pitch, rows of one parity alone cover only
//     half the banks, hence the row permutation.
// Found by exhaustive search over linear (XOR) maps of the row bits.
__device__ __forceinline__ int lds_unit(int r, int c) {
  const int p0 = (r ^ (r >> 3) ^ (r >> 4)) & 1;
  const int p1 = ((r >> 1) ^ (r >> 3)) & 1;
  const int f = ((r >> 1) & 1) | (((r >> 2) & 1) << 1);
  return 4 * ((r & ~3) + p0 + 2 * p1) + (c ^ f);
}
constexpr int LDK = BK;  // fp16 elements per tile row
constexpr int kGemmThreads = 256;  // 4 waves as 2 x 2
constexpr int kStages = 4;         // 32-k steps of global loads in flight

template <int BM, int BN>
struct TileCfg {
  static constexpr int WM = BM / 2, WN = BN / 2;    // wave tile
  static constexpr int TM = WM / 32, TN = WN / 32;  // 32 x 32 MFMA tiles per wave
  static constexpr int A_ITERS = BM * (BK / 8) / kGemmThreads;  // 16-byte A chunks per thread
  static constexpr int VB = BN / 64;                // packed words per thread per step
  static_assert(TM >= 1 && TN >= 1, "wave tile must hold a 32 x 32 MFMA tile");
  static_assert(A_ITERS >= 1, "A tile must give every thread a chunk");
  static_assert(VB == 1 || VB == 2, "B words per thread");
};

// VB adjacent packed words (and their fp16 scales) of one packed row, as one
// buffer load each.
template <int VB>
struct BWords;
template <>
struct BWords<2> {
  using word_t = u2_t;
  using scale_t = h2_t;
  static __device__ __forceinline__ word_t load_w(__amdgpu_buffer_rsrc_t r, uint32_t v, uint32_t s) {
    return __builtin_bit_cast(u2_t, __builtin_amdgcn_raw_buffer_load_b64(r, v, s, 0));
  }
  static __device__ __forceinline__ scale_t load_s(__amdgpu_buffer_rsrc_t r, uint32_t v, uint32_t s) {
    return __builtin_bit_cast(h2_t, __builtin_amdgcn_raw_buffer_load_b32(r, v, s, 0));
  }
  static __device__ __forceinline__ uint32_t word(word_t w, int j) { return w[j]; }
  static __device__ __forceinline__ _Float16 scale(scale_t x, int j) { return x[j]; }
};
template <>
struct BWords<1> {
  using word_t = uint32_t;
  using scale_t = _Float16;
  static __device__ __forceinline__ word_t load_w(__amdgpu_buffer_rsrc_t r, uint32_t v, uint32_t s) {
    return __builtin_amdgcn_raw_buffer_load_b32(r, v, s, 0);
  }
  static __device__ __forceinline__ scale_t load_s(__amdgpu_buffer_rsrc_t r, uint32_t v, uint32_t s) {
    return __builtin_bit_cast(_Float16, __builtin_amdgcn_raw_buffer_load_b16(r, v, s, 0));
  }
  static __device__ __forceinline__ uint32_t word(word_t w, int) { return w; }
  static __device__ __forceinline__ _Float16 scale(scale_t x, int) { return x; }
};

struct TileArgs {
  const _Float16* X;
  const uint32_t* Wq;
  const _Float16* S;
  _Float16* Y;
  int M, K, N;
  WeightLayout L;  // where a column's words and scales live (packed or strip-major)
};

template <int BM, int BN, int GROUP>
__global__ __launch_bounds__(kGemmThreads) __attribute__((amdgpu_waves_per_eu(1, 2))) void
gemm_tile_kernel(TileArgs args) {
  using C = TileCfg<BM, BN>;
  constexpr int VB = C::VB;
  __shared__ __attribute__((aligned(16))) _Float16 As[2][BM * LDK];
  __shared__ __attribute__((aligned(16))) _Float16 Bs[2][BN * LDK];
  const _Float16* __restrict__ X = args.X;
  const uint32_t* __restrict__ Wq = args.Wq;
  const _Float16* __restrict__ S = args.S;
  _Float16* __restrict__ Y = args.Y;
  const int M = args.M, K = args.K, N = args.N;

  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const int wave = tid >> 6;
  const int wm = (wave >> 1) * C::WM;
  const int wn = (wave & 1) * C::WN;
  const int m0 = blockIdx.y * BM;
  const int n0 = blockIdx.x * BN;

  f16_t acc[C::TM][C::TN];
#pragma unroll
  for (int i = 0; i < C::TM; ++i)
#pragma unroll
    for (int j = 0; j < C::TN; ++j)
#pragma unroll
      for (int r = 0; r < 16; ++r) acc[i][j][r] = 0.0f;

  // Staging registers for one 32-k step.  kStages steps are in flight at
  // once (rotating register sets, indexed only by compile-time constants);
  // the LDS holds two steps (the one being multiplied and the next).  All
  // staging is in vector values (no small arrays the compiler could move to
  // memory), and every load is an unpredicated buffer load: rows past M and
  // columns past N use an offset outside the buffer and read zero.
  using BVec = typename BWords<VB>::word_t;
  using SVec = typename BWords<VB>::scale_t;
  struct Stage {
    h8_t a[C::A_ITERS];
    BVec b;
    SVec s;
  };
  // B: thread tid loads packed row (tid / 64) of the step, columns
  // n0 + VB * (tid % 64) .. + VB - 1.
  const int b_row = tid >> 6;
  const int b_col = n0 + VB * (tid & 63);
  const int ntiles = K / BK;
  const uint32_t row_bytes = args.L.w_row;
  const __amdgpu_buffer_rsrc_t rx =
      make_rsrc(X, static_cast<uint32_t>(M) * static_cast<uint32_t>(K) * 2u);
  const __amdgpu_buffer_rsrc_t rw =
      make_rsrc(Wq, static_cast<uint32_t>(K / 8) * static_cast<uint32_t>(N) * 4u);
  const __amdgpu_buffer_rsrc_t rsc =
      make_rsrc(S, static_cast<uint32_t>(K / GROUP) * static_cast<uint32_t>(N) * 2u);
  uint32_t voff_a[C::A_ITERS];
#pragma unroll
  for (int it = 0; it < C::A_ITERS; ++it) {
    const int e = tid + it * kGemmThreads;
    const int gm = m0 + (e >> 2);
    voff_a[it] = gm < M ? (static_cast<uint32_t>(gm) * K + (e & 3) * 8) * 2u : kOutOfRange;
  }
  const bool b_ok = b_col < N;
  const uint32_t voff_b = b_ok ? b_row * row_bytes + args.L.wcol(b_col) : kOutOfRange;
  const uint32_t voff_s = b_ok ? args.L.scol(b_col) : kOutOfRange;

  // Loads of step `step`, clamped to the last step: a prefetch past the end
  // re-reads it (an L2 hit) rather than being skipped, so the loads are the
  // same on every path and the compiler's in-order wait counts stay exact.
  auto load_step = [&](Stage& st, int step) {
    const uint32_t k0 = static_cast<uint32_t>(min(step, ntiles - 1) * BK);
#pragma unroll
    for (int it = 0; it < C::A_ITERS; ++it)
      st.a[it] = __builtin_bit_cast(h8_t, __builtin_amdgcn_raw_buffer_load_b128(rx, voff_a[it], k0 * 2u, 0));
    st.b = BWords<VB>::load_w(rw, voff_b, (k0 / 8) * row_bytes);
    st.s = BWords<VB>::load_s(rsc, voff_s, (k0 / GROUP) * args.L.s_row);
  };
  // LDS offsets (fp16 elements).  Rows 64 apart share the swizzle of their
  // low 5 bits, so each offset is a per-thread constant plus a row multiple.
  // A stores: thread tid writes row tid / 4 + 64 it, unit tid % 4.
  const int a_st = lds_unit(tid >> 2, tid & 3) * 8;
  // B stores: columns VB * (tid % 64) + j, unit b_row.
  int b_st[VB];
#pragma unroll
  for (int j = 0; j < VB; ++j) b_st[j] = lds_unit(VB * (tid & 63) + j, b_row) * 8;
  auto store_step = [&](const Stage& st, int buf) {
#pragma unroll
    for (int it = 0; it < C::A_ITERS; ++it)
      *reinterpret_cast<h8_t*>(&As[buf][a_st + it * 64 * LDK]) = st.a[it];
#pragma unroll
    for (int j = 0; j < VB; ++j) {
      h2_t w[4];
      const _Float16 sj = BWords<VB>::scale(st.s, j);
      const h2_t s2 = {sj, sj};
      decode8_scaled(BWords<VB>::word(st.b, j), s2, w);
      const h8_t v = {w[0][0], w[0][1], w[1][0], w[1][1], w[2][0], w[2][1], w[3][0], w[3][1]};
      *reinterpret_cast<h8_t*>(&Bs[buf][b_st[j]]) = v;
    }
  };
  // Operand reads: row (32 i + lane % 32) of a wave's 32-row block, unit
  // 2 ks + lane / 32 (the lane's 8 k of the 16-k MFMA step ks).
  const int r32 = lane & 31;
  int rd[BK / 16];
#pragma unroll
  for (int ks = 0; ks < BK / 16; ++ks) rd[ks] = lds_unit(r32, 2 * ks + (lane >> 5)) * 8;
  auto compute = [&](int buf) {
#pragma unroll
    for (int ks = 0; ks < BK / 16; ++ks) {
      h8_t a[C::TM], b[C::TN];
#pragma unroll
      for (int i = 0; i < C::TM; ++i)
        a[i] = *reinterpret_cast<const h8_t*>(&As[buf][(wm + 32 * i) * LDK + rd[ks]]);
#pragma unroll
      for (int j = 0; j < C::TN; ++j)
        b[j] = *reinterpret_cast<const h8_t*>(&Bs[buf][(wn + 32 * j) * LDK + rd[ks]]);
#pragma unroll
      for (int i = 0; i < C::TM; ++i)
#pragma unroll
        for (int j = 0; j < C::TN; ++j) acc[i][j] = mfma32(a[i], b[j], acc[i][j]);
    }
  };

  Stage R[kStages];
#pragma unroll
  for (int i = 0; i < kStages; ++i) load_step(R[i], i);
  store_step(R[0], 0);
  __syncthreads();
  // Step t: refill the register set that held step t (already in LDS) with
  // step t + kStages, multiply step t from LDS, then move step t + 1 from its
  // registers into the other LDS buffer.
  auto iter = [&](auto u_const, int t) {
    constexpr int u = decltype(u_const)::value;
    load_step(R[u], t + kStages);
    __builtin_amdgcn_sched_barrier(0);  // keep the refill ahead of the MFMAs
    compute(t & 1);
    __builtin_amdgcn_sched_barrier(0);
    store_step(R[(u + 1) % kStages], (t + 1) & 1);
    __syncthreads();
  };
  // Whole rounds of kStages steps with no exit in the middle (an exit after
  // each step makes the compiler keep a copy of the accumulators per exit),
  // then the remaining 0..kStages-1 steps once.
  int t = 0;
  for (; t + kStages <= ntiles; t += kStages) {
    iter(std::integral_constant<int, 0>{}, t);
    iter(std::integral_constant<int, 1>{}, t + 1);
    iter(std::integral_constant<int, 2>{}, t + 2);
    iter(std::integral_constant<int, 3>{}, t + 3);
  }
  const int rem = ntiles - t;
  if (rem > 0) iter(std::integral_constant<int, 0>{}, t);
  if (rem > 1) iter(std::integral_constant<int, 1>{}, t + 1);
  if (rem > 2) iter(std::integral_constant<int, 2>{}, t + 2);

  // Epilogue: register r of lane l holds row 8*(r/4) + 4*(l/32) + r%4,
  // column l % 32 of each 32 x 32 tile.
  const int rq = (lane >> 5) * 4;
#pragma unroll
  for (int i = 0; i < C::TM; ++i) {
#pragma unroll
    for (int j = 0; j < C::TN; ++j) {
      const int gn = n0 + wn + 32 * j + r32;
      if (gn >= N) continue;
#pragma unroll
      for (int r = 0; r < 16; ++r) {
        const int gm = m0 + wm + 32 * i + 8 * (r >> 2) + rq + (r & 3);
        if (gm < M) Y[static_cast<size_t>(gm) * N + gn] = (_Float16)acc[i][j][r];
      }
    }
  }
}

template <int TM, int KW, int WN>
hipError_t launch_direct_cfg(DirectArgs a, int64_t G, hipStream_t stream) {
  // Up to 3 row tiles (4 with four waves side by side) a wave leaves registers
  // for two waves per SIMD.
  constexpr int kOcc = TM <= 2 || (TM <= 4 && KW * WN >= 4 && WN == 4) ? 2 : 1;
  a.tiles_m = static_cast<int>(ceil_div(a.M, 32 * TM));
  a.tiles_n = static_cast<int>(ceil_div(a.N, 64 * WN));
  const unsigned grid = static_cast<unsigned>(a.tiles_m) * a.tiles_n * a.splits;
  if (G == 128)
    gemm_direct_kernel<TM, KW, WN, 128, kOcc><<<grid, KW * WN * 64, 0, stream>>>(a);
  else
    gemm_direct_kernel<TM, KW, WN, 64, kOcc><<<grid, KW * WN * 64, 0, stream>>>(a);
  return hipGetLastError();
}

template <int BM, int BN>
hipError_t launch_tile(const TileArgs& a, int64_t G, hipStream_t stream) {
  dim3 grid(static_cast<unsigned>(ceil_div(a.N, BN)), static_cast<unsigned>(ceil_div(a.M, BM)));
  if (G == 128)
    gemm_tile_kernel<BM, BN, 128><<<grid, kGemmThreads, 0, stream>>>(a);
  else
    gemm_tile_kernel<BM, BN, 64><<<grid, kGemmThreads, 0, stream>>>(a);
  return hipGetLastError();
}

// Which kernel a call runs, and its tile: the direct kernel's (tm > 0: 32 tm
// rows by 64 wn columns, kw teams), else the tile kernel's bm x bn.
struct TileChoice {
  int bm, bn;
  int tm = 0, kw = 1, wn = 4;
};

// The device the plans are made for: MI355X, 256 CUs.  Planning with a fixed
// count keeps the workspace query pure host code and equal to the launch.
constexpr int kPlanCUs = 256;

// The widest B vector aligned operands of this N allow (the plan the
// workspace query assumes).
int nominal_bn_max(int64_t N) { return N % 4 == 0 ? 256 : N % 2 == 0 ? 128 : 64; }

// Widest B vector (BN / 64 packed words per thread) the operands allow.
int max_bn(int64_t N, const void* w, const void* s) {
  if (N % 4 == 0 && aligned(w, 16) && aligned(s, 8)) return 256;
  if (N % 2 == 0 && aligned(w, 8) && aligned(s, 4)) return 128;
  return 64;
}

// Tile choice of the tile kernel (the shapes the direct kernel does not
// take), measured on MI355X over M = 64..2048 at 4096 x 14336 and
// 14336 x 4096: 128 x 128 (2 waves per SIMD, so one workgroup's barrier
// wait overlaps another's MFMAs) is fastest whenever its grid gives every CU
// a workgroup; otherwise 64 x 128, whose doubled grid wins (e.g. 126 us vs
// 165 us at M = 512, 14336 x 4096).  256-wide tiles of this kernel, one
// workgroup per CU, were slower at every shape.  Narrower B vectors serve N
// not a multiple of 2 or operands without 8-byte alignment.
TileChoice choose_tile(int64_t M, int64_t N, int bn_max) {
  const int bn = std::min(128, bn_max);
  if (ceil_div(M, 128) * ceil_div(N, bn) >= kPlanCUs) return {128, bn};
  return {64, bn};
}

struct TilePlan {
  TileChoice t;
  int splits = 1;
  size_t counter_bytes = 0;
  size_t workspace_bytes = 0;
};

// The K splits a shape may use and the workspace they need -- what the
// workspace query answers, so what a caller's buffer holds -- with the tile
// that runs where the direct kernel does not.  Long reductions split where
// the tiles are few, as does 4096 <= K < 8192 with at most 160 64-row tiles.
// The direct kernel takes as many of these splits as pay (plan_tile).
TilePlan plan_split_room(int64_t M, int64_t K, int64_t N, int64_t version, int bn_max) {
  TilePlan p;
  int64_t tiles = 0;
  int splits = 1;
  int unit = 64;  // k the splits are cut in
  if (M <= kStreamMaxM && K % 64 == 0 && bn_max >= 256) {
    // Small batches that do not stream (gemm_streams): the largest of 1, 2, 4,
    // 8 ways keeping the grid of 64-row tiles within 320 workgroups.  Both
    // versions take this plan (so they agree to the bit).
    p.t = TileChoice{64, 128};
    tiles = ceil_div(M, 64) * ceil_div(N, 128);
    while (splits < 8 && tiles * splits * 2 <= 320 && K / 64 >= 2 * splits) splits *= 2;
  } else if (K % 64 == 0 && bn_max >= 256) {
    const int64_t t128 = ceil_div(M, 128) * ceil_div(N, 128);
    p.t = TileChoice{version == 7 || K >= 8192 || t128 >= 192 ? 128 : 64, 128};
    tiles = ceil_div(M, p.t.bm) * ceil_div(N, 128);
    if (K >= 8192) {
      if (tiles <= 64)
        splits = 4;
      else if (tiles <= 128)
        splits = 2;
      else if (tiles > kPlanCUs && tiles < 2 * kPlanCUs)
        splits = 2;
    } else if (p.t.bm == 64 && K >= 4096 && tiles <= 160) {
      splits = 4;
    }
  } else {
    unit = BK;
    p.t = version == 7 ? TileChoice{128, std::min(128, bn_max)} : choose_tile(M, N, bn_max);
    tiles = ceil_div(M, p.t.bm) * ceil_div(N, p.t.bn);
    if (K >= 8192 && tiles < 2 * kPlanCUs)
      splits = static_cast<int>(std::min<int64_t>(ceil_div(2 * kPlanCUs, tiles), 4));
  }
  const int64_t steps = K / unit, per = ceil_div(steps, splits);
  p.splits = static_cast<int>(ceil_div(steps, per));
  if (p.splits > 1) {
    p.counter_bytes = align_up(static_cast<size_t>(tiles) * 4, 256);
    p.workspace_bytes = p.counter_bytes + static_cast<size_t>(p.splits) * M * N * 4;
  }
  return p;
}

// Widest N the direct kernel addresses: a tile's rows within 32-bit offsets.
constexpr int64_t kDirectMaxN = int64_t(1) << 22;

// Whether the direct kernel takes these operands: two columns a load.
bool direct_supported(int64_t K, int64_t N, const void* w, const void* s) {
  return K % 64 == 0 && N % 2 == 0 && N < kDirectMaxN && aligned(w, 8) && aligned(s, 4);
}

// The direct kernel's tile, teams and splits for a shape, within the splits
// and counters of `room`.  A model of its time, fitted to MI355X measurements
// of every tile and split at some 900 shapes (M = 48..1536) and the fastest
// tiles beyond, us: 4.5 to start and drain; per 64-k step and round of the CUs
// the tile's own time, `step` in a single round and `again` over several; 0.36
// of the time the whole product takes at the power-limited 1.25 PFLOP/s; and
// for a K split 1 + 0.5 a split, 0.9 for each round of coherent loads the last
// workgroup of a tile sums it in (4 tm / kw rounds: 3 us for tm = 1, 4 teams;
// 5 to 10 for tm = 2; 9 to 13 for tm = 3, 2 teams) and 0.26 a MB of partials.
// `tail` is how much of a part-filled last round is paid for (less where two
// workgroups share a CU).  Teams are for grids of one round: alone on its CU,
// such a workgroup's ring fill and the teams' meeting overlap with nothing, so
// over several rounds its steps take up to half as long again.  The model
// names the fastest plan at most of the shapes, one within 5% at six of seven
// and within 10% at nineteen of twenty:
// 96 x 8192 x 8192 (M x K x N) tm = 2, 4 teams, 2 column waves, 2 splits
// 23.2 us (tm = 1, 2 teams, 4 column waves 26.9), 128 x 4096 x 14336 the same
// unsplit 19.0 (25.2), 256 x 4096 x 4096 tm = 1, 4 teams 14.9 (2 teams, 2
// splits 21.8), 512 x 4096 x 14336 tm = 4 52.5 (2: 61, 8: 75), 1000 x 5504 x
// 4102 tm = 3, 2 teams 48 (4: 54), 4096 x 4096 x 4096 tm = 8 108 (4: 111).
// Several rounds, the fastest tiles without teams against the fastest with:
// 700 x 4096 x 14336 tm = 6 80 (85), 1024 x 4096 x 28672 tm = 8 198 (222),
// 1024 x 4096 x 6144 tm = 4 52 (62), 2048 x 5504 x 4102 tm = 5 87 (104), 2048
// x 4096 x 14336 tm = 5 200 (222).
// Tiles of one column wave (64 columns) are for few tiles, where they make one
// round: a K split of wider tiles costs more than their narrower rows lose.
// 129 x 4096 x 2048 tm = 1, 4 teams 12.0 (tm = 2, 2 column waves, 4 splits
// 15.8), 400 x 4096 x 1024 12.4 (18.0), 700 x 4096 x 512 12.3 (14.9), 300 x
// 8192 x 2048 tm = 2 23.0 (tm = 1, 2 column waves 24.5); over two rounds they
// lose, 300 x 4096 x 2048 tm = 1 17.0 (15.3).
// Teams split K, so a K below 1024 keeps one, except from 512 in one round of
// 32-row tiles, or of 64-row tiles with 2 teams: 300 x 768 x 3072 32-row 6.5 us
// (one team 8.3), 129 / 256 x 512 x 4096 5.9 / 6.1 (6.4 / 6.7); 400 x 768 x
// 3072 64-row 7.1 (8.4), 300 x 512 x 4096 6.2 (6.9), and beyond a round 700 x
// 768 x 3072 9.7 (8.7).
TileChoice choose_direct(int64_t M, int64_t K, int64_t N, const TilePlan& room, int* splits) {
  struct Cfg {
    int tm, kw, wn;
    double step, again, tail;
  };
  static constexpr Cfg kCfgs[] = {
      {1, 4, 1, 0.108, 0.108, 1.0},  {2, 4, 1, 0.13, 0.13, 1.0},   {2, 2, 2, 0.165, 0.165, 1.0},
      {1, 4, 2, 0.127, 0.127, 0.75}, {2, 4, 2, 0.155, 0.24, 1.0},  {3, 2, 2, 0.215, 0.29, 1.0},
      {4, 2, 2, 0.275, 0.345, 1.0},  {2, 2, 4, 0.28, 0.36, 1.0},   {3, 2, 4, 0.385, 0.435, 1.0},
      {1, 1, 4, 0.36, 0.36, 0.5},    {2, 1, 4, 0.40, 0.40, 0.5},   {3, 1, 4, 0.45, 0.45, 0.5},
      {4, 1, 4, 0.515, 0.515, 0.8},  {5, 1, 4, 0.65, 0.65, 1.0},   {6, 1, 4, 0.775, 0.775, 1.0},
      {8, 1, 4, 0.98, 0.98, 1.0}};
  const int64_t steps = K / kDirectStep;
  const int64_t max_counters = static_cast<int64_t>(room.counter_bytes / 4);
  const double power = 0.36 * 2.0 * static_cast<double>(M) * K * N / 1.25e9;
  TileChoice best{0, 0};
  double best_us = 1e30;
  for (const Cfg& c : kCfgs) {
    const int64_t tiles = ceil_div(M, 32 * c.tm) * ceil_div(N, 64 * c.wn);
    const bool one_round = tiles <= kPlanCUs;
    const bool short_k_form = c.tm == 2 && c.kw == 2 && c.wn == 2;
    if (c.kw == 1) {
      if (c.tm <= 3 && K >= 1024) continue;
    } else if (K < 1024) {
      if (K < 512 || !one_round || !(c.tm == 1 || short_k_form)) continue;
    } else if (short_k_form || (c.wn == 1 && !one_round)) {
      continue;
    }
    for (int s = 1; s <= (c.tm <= kDirectMaxSplitTM ? room.splits : 1); ++s) {
      if (s > 1 && tiles > max_counters) break;
      const int64_t per = ceil_div(steps, s);
      if (ceil_div(steps, per) != s) continue;  // those steps make fewer splits
      const double fill = static_cast<double>(tiles * s) / kPlanCUs;
      const double rounds = static_cast<double>(ceil_div(tiles * s, kPlanCUs));
      const double eff = fill > 1 ? c.tail * rounds + (1.0 - c.tail) * fill : rounds;
      double us = 4.5 + eff * static_cast<double>(per) * (fill > 1 ? c.again : c.step) + power;
      if (s > 1)
        us += 1.0 + 0.5 * s + 0.9 * 4 * c.tm / c.kw + 0.26e-6 * 4 * static_cast<double>(s) * M * N;
      if (us < best_us) {
        best_us = us;
        best = TileChoice{32 * c.tm, 64 * c.wn, c.tm, c.kw, c.wn};
        *splits = s;
      }
    }
  }
  return best;
}

// The launch plan.  The direct kernel (`direct`: the operands suit it) loads
// two columns at a time whatever more their alignment allows (bn_max): its
// room is the workspace query's, so the splits, the workspace they need and
// where the counters end are what the caller was told.  The tile kernel never
// splits K: it runs only under-aligned operands, or an N whose K is short.
// The versions' plans differ only where the room does (version 7 has none for
// 4096 <= K < 8192, and other splits where N % 4 == 2); elsewhere they are the
// same, with the same bits.
TilePlan plan_tile(int64_t M, int64_t K, int64_t N, int64_t version, int bn_max, bool direct) {
  TilePlan p = plan_split_room(M, K, N, version, direct ? nominal_bn_max(N) : bn_max);
  int splits = 1;
  if (direct) p.t = choose_direct(M, K, N, p, &splits);
  p.splits = splits;
  return p;
}

hipError_t launch_direct(TileChoice t, const DirectArgs& a, int64_t G, hipStream_t stream) {
  switch (t.tm * 100 + t.kw * 10 + t.wn) {
    case 141: return launch_direct_cfg<1, 4, 1>(a, G, stream);
    case 241: return launch_direct_cfg<2, 4, 1>(a, G, stream);
    case 222: return launch_direct_cfg<2, 2, 2>(a, G, stream);
    case 142: return launch_direct_cfg<1, 4, 2>(a, G, stream);
    case 242: return launch_direct_cfg<2, 4, 2>(a, G, stream);
    case 322: return launch_direct_cfg<3, 2, 2>(a, G, stream);
    case 422: return launch_direct_cfg<4, 2, 2>(a, G, stream);
    case 224: return launch_direct_cfg<2, 2, 4>(a, G, stream);
    case 324: return launch_direct_cfg<3, 2, 4>(a, G, stream);
    case 114: return launch_direct_cfg<1, 1, 4>(a, G, stream);
    case 214: return launch_direct_cfg<2, 1, 4>(a, G, stream);
    case 314: return launch_direct_cfg<3, 1, 4>(a, G, stream);
    case 414: return launch_direct_cfg<4, 1, 4>(a, G, stream);
    case 514: return launch_direct_cfg<5, 1, 4>(a, G, stream);
    case 614: return launch_direct_cfg<6, 1, 4>(a, G, stream);
    case 814: return launch_direct_cfg<8, 1, 4>(a, G, stream);
    default: return hipErrorInvalidValue;
  }
}

hipError_t launch_choice(TileChoice t, const TileArgs& a, int64_t G, hipStream_t stream) {
  if (t.bm == 128 && t.bn == 128) return launch_tile<128, 128>(a, G, stream);
  if (t.bm == 64 && t.bn == 128) return launch_tile<64, 128>(a, G, stream);
  if (t.bm == 128 && t.bn == 64) return launch_tile<128, 64>(a, G, stream);
  return launch_tile<64, 64>(a, G, stream);
}

}  // namespace

// Mirrors the reference's host checks (csrc/gemm_w4a16.cu:381-400); pure host.
int validate_gemm(const void* X, int64_t x_rows, int64_t x_cols, const void* Wq, int64_t wq_rows,
                  int64_t wq_cols, const void* S, int64_t s_rows, int64_t s_cols, int64_t group_size,
                  int64_t version, const void* Y) {
  NIBBLE_CHECK(x_rows >= 0 && x_cols >= 0 && wq_rows >= 0 && wq_cols >= 0 && s_rows >= 0 &&
                   s_cols >= 0,
               "negative dimension");
  const int64_t M = x_rows, K = x_cols, N = wq_cols;
  NIBBLE_CHECK(wq_rows * 8 == K, "packed weight rows disagree with K");
  NIBBLE_CHECK(K % BK == 0, "K must be a multiple of %d", BK);
  NIBBLE_CHECK(N % 2 == 0, "N must be even");
  NIBBLE_CHECK(group_size == 64 || group_size == 128, "group_size must be 64 or 128");
  NIBBLE_CHECK(s_rows * group_size == K, "scale rows disagree with K/group_size");
  NIBBLE_CHECK(s_cols == N, "scale columns disagree with N");
  NIBBLE_CHECK(version == 6 || version == 7, "gemm version must be 6 or 7, got %lld",
               (long long)version);
  const int64_t lim = int64_t(1) << 31;
  NIBBLE_CHECK(M * N < lim && M * K < lim && K * N < lim,
               "shape too large for 32-bit indexing in the prefill kernel");
  NIBBLE_CHECK(ceil_div(M, 64) < 65536, "M too large");
  // Only operands that hold elements are dereferenced (empty tensors may
  // carry a null data pointer).
  const bool x_used = M * K > 0 && N > 0;
  const bool w_used = K * N > 0 && M > 0;
  const bool y_used = M * N > 0;
  NIBBLE_CHECK((!x_used || X != nullptr) && (!w_used || (Wq != nullptr && S != nullptr)) &&
                   (!y_used || Y != nullptr),
               "null pointer");
  NIBBLE_CHECK((!x_used || aligned(X, 16)) && (!w_used || (aligned(Wq, 4) && aligned(S, 2))) &&
                   (!y_used || aligned(Y, 2)),
               "misaligned pointer (X needs 16-byte alignment)");
  return NIBBLE_OK;
}

}  // namespace nibble

using namespace nibble;

namespace {
// Small batches go to the weight-streaming kernel: each pass reads every
// weight byte once and multiplies it against up to 32 rows (one or two
// 16-row MFMA tiles), where a 64/128-row tile would leave most of the device
// idle.  Measured on MI355X at K=4096, N=14336: M=16 takes 82 us through the
// tile kernel and 11 us streaming.  Above 32 rows streaming takes one pass
// per 32 rows; once those passes would move 48 MiB or more, the direct
// kernel's tiles win (plan_tile).  Measured, graph replay, streaming against
// tiles: 4096 x 14336 M = 65 / 128 25 / 41.9 us against 17.2 / 19.0; 14336 x
// 4096 M = 128 56.6 against 23.6; 8192 x 8192 M = 96 43 against 23.2.  Below
// that streaming was ahead or level when the line was drawn; the tiles of one
// column wave have come level with it since, and ahead from 65 rows: 4096 x
// 4096 M = 64 / 128 10.9 / 11.9 us against 11.6 / 11.6, 4096 x 6144 M = 64 / 65
// / 96 11.7 / 16.3 / 21.0 against 11.3 / 14.6 / 14.7.
bool gemm_streams(int64_t M, int64_t K, int64_t N, int64_t G) {
  if (!(M >= 1 && M <= kStreamMaxM && K > 0 && N > 0 && N % 4 == 0 && K % G == 0)) return false;
  const int64_t pass_bytes = K * N / 2;
  return M <= 32 || K % 64 != 0 || ceil_div(M, 32) * pass_bytes < (int64_t(48) << 20) ||
         batch_block_rows(M, K, N, G) == 64;  // 33..64 rows in one 64-row block
}
}  // namespace

namespace {
// The plan a call with these arguments runs (streaming for small batches,
// tiles otherwise), assuming operands aligned for the widest loads.
void gemm_plan_bytes(int64_t M, int64_t K, int64_t N, int64_t G, int64_t version, size_t* ws,
                     size_t* counters) {
  *ws = 0;
  *counters = 0;
  if ((version != 6 && version != 7) || (G != 64 && G != 128) || M <= 0 || N <= 0 || K <= 0 ||
      K % BK != 0 || K % G != 0)
    return;
  if (gemm_streams(M, K, N, G)) {
    StreamPlan p;
    if (plan_stream(M, K, N, G, true, 0, 0, &p) != NIBBLE_OK) return;
    *ws = p.workspace_bytes;
    *counters = p.counter_bytes;
    return;
  }
  const TilePlan p = plan_split_room(M, K, N, version, nominal_bn_max(N));
  *ws = p.workspace_bytes;
  *counters = p.counter_bytes;
}
}  // namespace

extern "C" size_t nibble_gemm_workspace_bytes(int64_t M, int64_t K, int64_t N, int64_t group_size,
                                              int64_t version, void* stream) {
  (void)stream;
  size_t ws, counters;
  gemm_plan_bytes(M, K, N, group_size, version, &ws, &counters);
  return ws;
}

extern "C" int nibble_gemm_streams(int64_t M, int64_t K, int64_t N, int64_t group_size) {
  return (group_size == 64 || group_size == 128) && K % BK == 0 && gemm_streams(M, K, N, group_size)
             ? 1
             : 0;
}

extern "C" size_t nibble_gemm_counter_bytes(int64_t M, int64_t K, int64_t N, int64_t group_size,
                                            int64_t version, void* stream) {
  (void)stream;
  size_t ws, counters;
  gemm_plan_bytes(M, K, N, group_size, version, &ws, &counters);
  return counters;
}

namespace {
// The body of nibble_gemm_w4a16 for validated operands, the weights in the
// packed layout (strip_cols 0) or the strip-major layout of that width: the
// plans depend on (M, K, N, group_size, version) and pointer alignment only,
// so both layouts run the same kernels in the same order and give the same
// bits.
int gemm_run(const void* X, int64_t M, int64_t K, int64_t N, const void* Wq, const void* S,
             int64_t group_size, int64_t version, void* Y, void* workspace,
             size_t workspace_bytes, void* stream_, int64_t strip_cols, int epilogue = 0,
             const void* bias = nullptr) {
  int rc = NIBBLE_OK;
  if (M == 0 || N == 0) return ok();
  hipStream_t stream = static_cast<hipStream_t>(stream_);
  DeviceGuard guard;
  int dev = 0;
  NIBBLE_HIP(guard.enter(stream, &dev));
  if (K == 0) {
    NIBBLE_HIP(fill_zero_f16(Y, M * N, stream));
    return ok();
  }
  if (gemm_streams(M, K, N, group_size) && stream_supported(X, Wq, S, Y, M, K, N, group_size)) {
    StreamPlan p;
    rc = plan_stream(M, K, N, group_size, true, 0, 0, &p);
    if (rc != NIBBLE_OK) return rc;
    rc = launch_stream(X, Wq, S, Y, M, K, N, group_size, p, workspace, workspace_bytes, stream,
                       "gemm (streaming) kernel launch", epilogue, bias, nullptr, 0.0f, strip_cols);
    return rc == NIBBLE_OK ? ok() : rc;
  }
  const auto* x = static_cast<const _Float16*>(X);
  auto* y = static_cast<_Float16*>(Y);
  // The tiles sum every output over k in the same order, so without a K split
  // (or two teams) they give identical bits.
  const int bn_max = max_bn(N, Wq, S);
  const bool direct = direct_supported(K, N, Wq, S);
  TilePlan p = plan_tile(M, K, N, version, bn_max, direct);
  if (epilogue != kEpilogueNone && p.t.tm == 0)
    return fail(NIBBLE_ERR_UNSUPPORTED, "no fused epilogue for this shape (nibble_gemm_fuses)");
  // The kernel addresses X through a buffer resource with 32-bit offsets:
  // tall activations are run in row blocks that stay below 2^31 bytes (such
  // grids are far too large to need a K split).
  const int64_t rows_max = std::max<int64_t>(256, ((int64_t(1) << 31) - 1) / (K * 2) / 256 * 256);
  // Row-blocked tall launches run without a split, as do small batches whose
  // pointers rule out the streaming kernel that the workspace query planned.
  if (M > rows_max || gemm_streams(M, K, N, group_size)) p.splits = 1;
  if (p.splits > 1) {
    if (workspace == nullptr || workspace_bytes < p.workspace_bytes)
      return fail(NIBBLE_ERR_WORKSPACE, "gemm needs %zu bytes of workspace, got %zu",
                  p.workspace_bytes, workspace == nullptr ? size_t(0) : workspace_bytes);
    if (!aligned(workspace, 256)) return fail(NIBBLE_ERR_WORKSPACE, "workspace must be 256-byte aligned");
  }
  auto* counters = p.splits > 1 ? static_cast<uint32_t*>(workspace) : nullptr;
  auto* partial = p.splits > 1
                      ? reinterpret_cast<float*>(static_cast<char*>(workspace) + p.counter_bytes)
                      : nullptr;
  const WeightLayout layout = layout_for(K, N, group_size, strip_cols);
  const int64_t out_n = epilogue == kEpilogueSwiglu ? N / 2 : N;
  hipError_t e = hipSuccess;
  for (int64_t m0 = 0; m0 < M && e == hipSuccess; m0 += rows_max) {
    const int rows = static_cast<int>(std::min(rows_max, M - m0));
    if (p.t.tm > 0) {
      DirectArgs a{};
      a.X = x + m0 * K;
      a.Wq = static_cast<const uint32_t*>(Wq);
      a.S = static_cast<const _Float16*>(S);
      a.Y = y + m0 * out_n;
      a.bias = static_cast<const _Float16*>(bias);
      a.partial = partial;
      a.counters = counters;
      a.M = rows;
      a.K = static_cast<int>(K);
      a.N = static_cast<int>(N);
      a.splits = p.splits;
      a.steps_per_split = static_cast<int>(ceil_div(K / kDirectStep, p.splits));
      a.epilogue = epilogue;
      a.L = layout;
      e = launch_direct(p.t, a, group_size, stream);
      continue;
    }
    TileArgs a;
    a.X = x + m0 * K;
    a.Wq = static_cast<const uint32_t*>(Wq);
    a.S = static_cast<const _Float16*>(S);
    a.Y = y + m0 * N;
    a.M = rows;
    a.K = static_cast<int>(K);
    a.N = static_cast<int>(N);
    a.L = layout;
    e = launch_choice(p.t, a, group_size, stream);
  }
  if (e != hipSuccess) return hip_fail(e, "gemm kernel launch");
  return ok();
}
}  // namespace

extern "C" int nibble_gemm_w4a16(const void* X, int64_t x_rows, int64_t x_cols, const void* Wq,
                                 int64_t wq_rows, int64_t wq_cols, const void* S, int64_t s_rows,
                                 int64_t s_cols, int64_t group_size, int64_t version, void* Y,
                                 void* workspace, size_t workspace_bytes, void* stream_) {
  const int rc = validate_gemm(X, x_rows, x_cols, Wq, wq_rows, wq_cols, S, s_rows, s_cols,
                               group_size, version, Y);
  if (rc != NIBBLE_OK) return rc;
  return gemm_run(X, x_rows, x_cols, wq_cols, Wq, S, group_size, version, Y, workspace,
                  workspace_bytes, stream_, 0);
}

// nibble_gemm_w4a16 for batches of 9 rows and more on strip-major weights
// (no counterpart in the reference): the same plans, kernels and bits as the
// packed call; batches of at most 8 rows take the strip-major GEMV.
extern "C" int nibble_gemm_w4a16_strip_major(const void* X, int64_t x_rows, int64_t x_cols,
                                             const void* Wt, const void* St, int64_t K, int64_t N,
                                             int64_t group_size, int64_t strip_cols,
                                             int64_t version, void* Y, void* workspace,
                                             size_t workspace_bytes, void* stream) {
  NIBBLE_CHECK(x_cols == K, "activation columns (%lld) disagree with K=%lld", (long long)x_cols,
               (long long)K);
  NIBBLE_CHECK(K > 0 && N > 0, "bad dimension (K and N must be positive)");
  NIBBLE_CHECK(group_size == 64 || group_size == 128, "group_size must be 64 or 128");
  NIBBLE_CHECK(K % group_size == 0, "K=%lld is not a multiple of group_size=%lld", (long long)K,
               (long long)group_size);
  NIBBLE_CHECK(strip_cols == 16 || strip_cols == 32 || strip_cols == 64,
               "strip_cols must be 16, 32 or 64, got %lld", (long long)strip_cols);
  NIBBLE_CHECK(N % strip_cols == 0, "N=%lld is not a multiple of strip_cols=%lld", (long long)N,
               (long long)strip_cols);
  NIBBLE_CHECK(strip_cols != 16 || group_size == 128, "16-column strips need group_size 128");
  NIBBLE_CHECK(x_rows == 0 || x_rows > 8,
               "batches of at most 8 rows take nibble_gemv_w4a16_strip_major (got M=%lld)",
               (long long)x_rows);
  NIBBLE_CHECK(Wt == nullptr || (aligned(Wt, 16) && aligned(St, 16)),
               "strip-major weights and scales must be 16-byte aligned");
  const int rc = validate_gemm(X, x_rows, x_cols, Wt, K / 8, N, St, K / group_size, N, group_size,
                               version, Y);
  if (rc != NIBBLE_OK) return rc;
  return gemm_run(X, x_rows, K, N, Wt, St, group_size, version, Y, workspace, workspace_bytes,
                  stream, strip_cols);
}

// nibble_gemm_w4a16 (version 6) with a fused output epilogue, on either
// layout, for the shapes the streaming or direct kernels serve (no counterpart in the
// reference, whose QuantLinear adds the bias as a separate fp16 op,
// python/nibblegemm/ops.py:131-135).  The product's plan and sums are
// nibble_gemm_w4a16's, so the outputs are the separate ops' bits.
extern "C" int nibble_gemm_fuses(int64_t M, int64_t K, int64_t N, int64_t group_size) {
  if ((group_size != 64 && group_size != 128) || M <= 8 || K <= 0 || N <= 0 || K % group_size != 0 ||
      N % 2 != 0 || N >= kDirectMaxN)
    return 0;
  if (gemm_streams(M, K, N, group_size)) return 1;
  return plan_tile(M, K, N, 6, nominal_bn_max(N), true).t.tm > 0 ? 1 : 0;
}

extern "C" int nibble_gemm_w4a16_fused(const void* X, int64_t x_rows, int64_t x_cols,
                                       const void* Wq, const void* S, int64_t K, int64_t N,
                                       int64_t group_size, int64_t strip_cols, int64_t epilogue,
                                       const void* bias, void* Y, void* workspace,
                                       size_t workspace_bytes, void* stream) {
  NIBBLE_CHECK(x_cols == K, "activation columns (%lld) disagree with K=%lld", (long long)x_cols,
               (long long)K);
  NIBBLE_CHECK(K > 0 && N > 0 && K % 8 == 0, "bad dimension (K and N must be positive)");
  NIBBLE_CHECK(group_size == 64 || group_size == 128, "group_size must be 64 or 128");
  NIBBLE_CHECK(K % group_size == 0, "K=%lld is not a multiple of group_size=%lld", (long long)K,
               (long long)group_size);
  NIBBLE_CHECK(strip_cols == 0 || strip_cols == 16 || strip_cols == 32 || strip_cols == 64,
               "strip_cols must be 0 (packed), 16, 32 or 64, got %lld", (long long)strip_cols);
  NIBBLE_CHECK(strip_cols == 0 || N % strip_cols == 0, "N=%lld is not a multiple of strip_cols=%lld",
               (long long)N, (long long)strip_cols);
  NIBBLE_CHECK(strip_cols != 16 || group_size == 128, "16-column strips need group_size 128");
  NIBBLE_CHECK(strip_cols == 0 || Wq == nullptr || (aligned(Wq, 16) && aligned(S, 16)),
               "strip-major weights and scales must be 16-byte aligned");
  NIBBLE_CHECK(epilogue == kEpilogueBias || epilogue == kEpilogueSwiglu,
               "epilogue must be 1 (bias) or 2 (swiglu), got %lld", (long long)epilogue);
  NIBBLE_CHECK(epilogue != kEpilogueSwiglu || N % (2 * kSwigluBlock) == 0,
               "swiglu needs N (gate|up interleaved in 16-column blocks) to be a multiple of 32");
  NIBBLE_CHECK(epilogue != kEpilogueBias || x_rows == 0 || (bias != nullptr && aligned(bias, 2)),
               "null or misaligned bias");
  const int rc = validate_gemm(X, x_rows, x_cols, Wq, K / 8, N, S, K / group_size, N, group_size, 6,
                               Y);
  if (rc != NIBBLE_OK) return rc;
  if (x_rows > 0 && !nibble_gemm_fuses(x_rows, K, N, group_size))
    return fail(NIBBLE_ERR_UNSUPPORTED, "no fused epilogue for M=%lld K=%lld N=%lld",
                (long long)x_rows, (long long)K, (long long)N);
  return gemm_run(X, x_rows, K, N, Wq, S, group_size, 6, Y, workspace, workspace_bytes, stream,
                  strip_cols, static_cast<int>(epilogue), bias);
}
