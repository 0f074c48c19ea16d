// Round-to-nearest group quantisation of a dense [K, N] weight on the device:
// the packed codes and fp16 scales of nibblegemm_amd.quant.quantize_device's
// tensor operations (reference python/nibblegemm/quant.py:127-161), bit for
// bit, in one pass over the weight.
//
// What bounds it: HBM, 2 (fp16) or 4 bytes read and 0.52 written a weight.  A
// workgroup holds one quant group of 128 columns in registers between the two
// uses of a value (the group's largest magnitude, then its code): thread (r, q)
// takes 8 rows -- one packed word a column -- of 8 adjacent columns, loaded as
// 16-byte pieces, 256 or 512 contiguous bytes a row; the column maxima of the
// threads meet in LDS, and a thread writes the 8 words of its rows at once.
// As separate tensor operations (fp32 copies, int64 codes, some 25 passes)
// 4096 x 14336 fp16 took 1163 us on MI355X; here 30, 4.96 TB/s of 147 MB, the
// rate of a large copy.  (With an fp32 copy of the weights in registers, an
// IEEE division a weight and 32 KiB of LDS a workgroup: 50; groups of 64 75.)
#include <algorithm>

#include "nibble_common.h"
#include "nibble_decode.h"

namespace nibble {
namespace {

constexpr int kQuantCols = 128;      // columns per workgroup
constexpr int kQuantMaxGroup = 512;  // 16 threads per 8 rows, 1024 at most
constexpr int kQuantF16 = 0, kQuantBF16 = 1, kQuantF32 = 2;

typedef float f8_t __attribute__((ext_vector_type(8)));
typedef uint32_t u8_t __attribute__((ext_vector_type(8)));
typedef unsigned short us8_t __attribute__((ext_vector_type(8)));

// Eight adjacent weights as loaded, and their magnitudes as unsigned bits:
// compared as integers those order as the magnitudes do, a NaN above
// everything (torch's amax), two 16-bit ones an instruction.
template <int DT>
struct Elem {
  using type = unsigned short;
  using vec = us8_t;
  static __device__ __forceinline__ float get(unsigned short v) {
    return DT == kQuantF16 ? static_cast<float>(__builtin_bit_cast(_Float16, v))
                           : __builtin_bit_cast(float, static_cast<uint32_t>(v) << 16);
  }
  static __device__ __forceinline__ vec load8(const type* p) {
    return __builtin_nontemporal_load(reinterpret_cast<const us8_t*>(p));
  }
  static __device__ __forceinline__ vec mag(vec v) { return v & (unsigned short)0x7fff; }
};
template <>
struct Elem<kQuantF32> {
  using type = uint32_t;
  using vec = u8_t;
  static __device__ __forceinline__ float get(uint32_t v) { return __builtin_bit_cast(float, v); }
  static __device__ __forceinline__ vec load8(const type* p) {
    const u4_t a = __builtin_nontemporal_load(reinterpret_cast<const u4_t*>(p));
    const u4_t b = __builtin_nontemporal_load(reinterpret_cast<const u4_t*>(p) + 1);
    return u8_t{a[0], a[1], a[2], a[3], b[0], b[1], b[2], b[3]};
  }
  static __device__ __forceinline__ vec mag(vec v) { return v & 0x7fffffffu; }
};

// The larger of two magnitudes, a NaN winning.
__device__ __forceinline__ float max_nan(float m, float v) { return v > m || v != v ? v : m; }

constexpr int kSlot[8] = {0, 4, 1, 5, 2, 6, 3, 7};  // nibble of each k of a word

// The code round_half_even(w / s) clamped to [-8, 7] plus 8 by division; NaN
// gives 0, as the tensor operations' conversion does.
__device__ __forceinline__ uint32_t code_by_division(float w, float s) {
  float q = rintf(w / s);
  q = q < -8.0f ? -8.0f : q > 7.0f ? 7.0f : q;
  return static_cast<uint32_t>(static_cast<int>(q + 8.0f)) & 15u;
}

// Codes without the division: t = fma(w, fl(1 / s), 1.5 * 2^23 + 8) holds
// round_half_even of the product plus 8 in its low bits.  The product is
// within 2^-22 of w / s relatively, 2^-19 below 8, so where it stays that far
// from every half the quotient rounds the same way; a column whose 8 weights
// come nearer, and scales that are not finite or whose reciprocal is
// subnormal, divide.  |w| <= 7 s (1 + 2^-23) in a group, so no clamp.
constexpr float kSureBelow = 0.49999f;
constexpr float kMagic = 12582920.0f;           // 1.5 * 2^23 + 8
constexpr uint32_t kMagicBits = 0x4b400000u;    // of 1.5 * 2^23

template <int DT, bool VEC>
__global__ __launch_bounds__(1024) void quantize_kernel(const typename Elem<DT>::type* W,
                                                        uint32_t* Wq, _Float16* S, int64_t K,
                                                        int64_t N, int G) {
  using E = Elem<DT>;
  using vec = typename E::vec;
  extern __shared__ float part[];  // [G / 8][kQuantCols]: column maxima; then scales, reciprocals
  const int tid = threadIdx.x;
  const int rg = tid >> 4;                         // which 8 rows of the group
  const int cq = (tid & 15) * 8;                   // first of 8 columns in the tile
  const int64_t n = static_cast<int64_t>(blockIdx.x) * kQuantCols + cq;
  const int64_t group = blockIdx.y;
  const int64_t row = group * G + 8 * rg;
  const int cols = n < N ? static_cast<int>(N - n < 8 ? N - n : 8) : 0;
  vec v[8];
#pragma unroll
  for (int r = 0; r < 8; ++r) {
    const typename E::type* p = W + (row + r) * N + n;
    if (VEC) {
      v[r] = cols > 0 ? E::load8(p) : vec{};
    } else {
#pragma unroll
      for (int i = 0; i < 8; ++i) v[r][i] = i < cols ? p[i] : 0;
    }
  }
  vec m = E::mag(v[0]);
#pragma unroll
  for (int r = 1; r < 8; ++r) m = __builtin_elementwise_max(m, E::mag(v[r]));
#pragma unroll
  for (int i = 0; i < 8; ++i) part[rg * kQuantCols + cq + i] = E::get(m[i]);
  __syncthreads();
  float own[kQuantCols / 16];  // a thread's columns (G >= 8: at least 16 threads)
#pragma unroll
  for (int u = 0; u < kQuantCols / 16; ++u) {
    const int c = tid + u * static_cast<int>(blockDim.x);
    if (c < kQuantCols) {
      float a = part[c];
      for (int r = 1; r < G / 8; ++r) a = max_nan(a, part[r * kQuantCols + c]);
      const float s = a / 7.0f;
      own[u] = s < 1e-8f ? 1e-8f : s;  // all-zero groups stay finite; NaN stays
    }
  }
  __syncthreads();
#pragma unroll
  for (int u = 0; u < kQuantCols / 16; ++u) {
    const int c = tid + u * static_cast<int>(blockDim.x);
    if (c < kQuantCols) {
      part[c] = own[u];
      part[kQuantCols + c] = 1.0f / own[u];
    }
  }
  __syncthreads();
  uint32_t constant = 0;
#pragma unroll
  for (int r = 0; r < 8; ++r) constant += kMagicBits << (4 * kSlot[r]);
  uint32_t word[8];
#pragma unroll
  for (int i = 0; i < 8; ++i) {
    const float s = part[cq + i], inv = part[kQuantCols + cq + i];
    float worst = 0.0f;
    word[i] = 0u - constant;
#pragma unroll
    for (int r = 0; r < 8; ++r) {
      const float w = E::get(v[r][i]);
      const float t = __builtin_fmaf(w, inv, kMagic);
      worst = fmaxf(worst, fabsf(__builtin_fmaf(w, inv, kMagic - t)));
      word[i] += __builtin_bit_cast(uint32_t, t) << (4 * kSlot[r]);
    }
    if (!(worst < kSureBelow) || !(s <= 1e37f)) {
      word[i] = 0;
#pragma unroll
      for (int r = 0; r < 8; ++r) word[i] |= code_by_division(E::get(v[r][i]), s) << (4 * kSlot[r]);
    }
  }
  uint32_t* wp = Wq + (row / 8) * N + n;
  _Float16* sp = S + group * N + n;
  if (VEC) {
    if (cols > 0) {
      const u4_t lo = {word[0], word[1], word[2], word[3]};
      const u4_t hi = {word[4], word[5], word[6], word[7]};
      __builtin_nontemporal_store(lo, reinterpret_cast<u4_t*>(wp));
      __builtin_nontemporal_store(hi, reinterpret_cast<u4_t*>(wp) + 1);
      if (rg == 0) {
        h8_t h;
#pragma unroll
        for (int i = 0; i < 8; ++i) h[i] = static_cast<_Float16>(part[cq + i]);
        *reinterpret_cast<h8_t*>(sp) = h;
      }
    }
  } else {
#pragma unroll
    for (int i = 0; i < 8; ++i)
      if (i < cols) {
        wp[i] = word[i];
        if (rg == 0) sp[i] = static_cast<_Float16>(part[cq + i]);
      }
  }
}

template <int DT>
hipError_t launch_quantize(const void* W, void* Wq, void* S, int64_t K, int64_t N, int G,
                           hipStream_t stream) {
  const dim3 grid(static_cast<unsigned>(ceil_div(N, kQuantCols)), static_cast<unsigned>(K / G));
  const auto* w = static_cast<const typename Elem<DT>::type*>(W);
  auto* q = static_cast<uint32_t*>(Wq);
  auto* s = static_cast<_Float16*>(S);
  // Column maxima, then two rows of scales and reciprocals.
  const size_t lds = static_cast<size_t>(std::max(G / 8, 2)) * kQuantCols * sizeof(float);
  // 16-byte pieces where every row starts on one.
  if (N % 8 == 0 && aligned(W, 16) && aligned(Wq, 16) && aligned(S, 16))
    quantize_kernel<DT, true><<<grid, 2 * G, lds, stream>>>(w, q, s, K, N, G);
  else
    quantize_kernel<DT, false><<<grid, 2 * G, lds, stream>>>(w, q, s, K, N, G);
  return hipGetLastError();
}

}  // namespace
}  // namespace nibble

extern "C" int nibble_quantize_rtn(const void* W, int64_t K, int64_t N, int64_t dtype,
                                   int64_t group_size, void* Wq, void* S, void* stream_) {
  using namespace nibble;
  NIBBLE_CHECK(K >= 0 && N >= 0, "negative dimension");
  NIBBLE_CHECK(group_size >= 8 && group_size <= kQuantMaxGroup && group_size % 8 == 0,
               "group_size must be a multiple of 8 up to %d, got %lld", kQuantMaxGroup,
               (long long)group_size);
  NIBBLE_CHECK(K % group_size == 0, "K=%lld is not a multiple of group_size=%lld", (long long)K,
               (long long)group_size);
  NIBBLE_CHECK(dtype == kQuantF16 || dtype == kQuantBF16 || dtype == kQuantF32,
               "dtype must be 0 (fp16), 1 (bf16) or 2 (fp32), got %lld", (long long)dtype);
  NIBBLE_CHECK(K / group_size < 65536, "more than 65535 groups");
  if (K == 0 || N == 0) return ok();
  NIBBLE_CHECK(W != nullptr && Wq != nullptr && S != nullptr, "null pointer");
  NIBBLE_CHECK(aligned(W, dtype == kQuantF32 ? 4 : 2) && aligned(Wq, 4) && aligned(S, 2),
               "misaligned pointer");
  hipStream_t stream = static_cast<hipStream_t>(stream_);
  DeviceGuard guard;
  int dev = 0;
  NIBBLE_HIP(guard.enter(stream, &dev));
  const int G = static_cast<int>(group_size);
  hipError_t e = dtype == kQuantF16    ? launch_quantize<kQuantF16>(W, Wq, S, K, N, G, stream)
                 : dtype == kQuantBF16 ? launch_quantize<kQuantBF16>(W, Wq, S, K, N, G, stream)
                                       : launch_quantize<kQuantF32>(W, Wq, S, K, N, G, stream);
  if (e != hipSuccess) return hip_fail(e, "quantize kernel launch");
  return ok();
}
