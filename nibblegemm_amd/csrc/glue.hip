// Decode-step glue of a Llama-shaped layer at batch 1, around the W4A16
// projections: RMSNorm and grouped-query attention over a KV cache.
//
// In the reference these are PyTorch / transformers operations of the model
// that bench/bench_model.py decodes token by token with its Linear layers
// swapped for QuantLinear (decode_tokens_per_s, bench/bench_model.py:177-188;
// the swap, :131-154).  Here they are kernels, so that a whole decode step --
// norms, projections, attention, residual adds -- is captured in one HIP
// graph.  The residual adds need no kernel of their own: at M = 1 the residual
// is a bias vector of the o and down projections (the fused bias epilogue of
// the matmul).
//
// Both kernels are memory-latency work of a few hundred KB; they are written
// for short, dependency-free loads (16-byte rows, no LDS staging of the
// cache) and deterministic reductions (fixed orders, no float atomics).
#include <algorithm>
#include <cmath>

#include "nibble_common.h"
#include "nibble_decode.h"
#include "nibble_reduce.h"

namespace nibble {

namespace {

constexpr int kHeadDim = 128;
constexpr int kRopeHalf = kHeadDim / 2;
constexpr int kChunk = 128;     // tokens per chunk record the workspace has room for
constexpr int kRound = 64;      // tokens an attention workgroup computes at a time
constexpr int kGlueThreads = 256;
constexpr int kRmsMaxCols = kRmsThreads * 8 * 8;
constexpr int kAttnMaxSeq = 1 << 16;
constexpr int kAttnMaxChunks = 64;     // chunks a launch uses at most
constexpr int kAttnOneChunk = 384;     // tokens one workgroup takes alone
constexpr int kAttnWorkgroups = 256;   // one round of the CUs
constexpr int64_t kAttnRereadBytes = 80 << 20;  // cache bytes read by all parts together
constexpr int64_t kAttnLlcBytes = int64_t(256) << 20;  // the last-level cache

// y = fp16(x * r * w) with r = 1 / sqrt(mean(x^2) + eps), in fp32 (the
// transformers LlamaRMSNorm computes the same in fp32 and rounds x * r to
// fp16 before the weight; this rounds once).  One workgroup per row; each
// thread holds CH 16-byte chunks of the row.  The sum of squares is reduced
// per wave (DPP rows, then rows in order) and across waves in wave order:
// deterministic.
template <int CH>
__global__ __launch_bounds__(kRmsThreads) void rmsnorm_kernel(const _Float16* __restrict__ X,
                                                              const _Float16* __restrict__ W,
                                                              _Float16* __restrict__ Y, int cols,
                                                              float eps) {
  __shared__ float part[kRmsThreads / 64];
  const int tid = threadIdx.x;
  const size_t base = static_cast<size_t>(blockIdx.x) * cols;
  h8_t v[CH], w[CH];
  float ss = 0.0f;
#pragma unroll
  for (int c = 0; c < CH; ++c) {
    const int col = (c * kRmsThreads + tid) * 8;
    v[c] = col < cols ? *reinterpret_cast<const h8_t*>(X + base + col) : h8_t{};
    w[c] = col < cols ? *reinterpret_cast<const h8_t*>(W + col) : h8_t{};  // before the reduction
    ss = sumsq_chunk(v[c], ss);
  }
  const float r = rms_scale(block256_sum(ss, part), cols, eps);
#pragma unroll
  for (int c = 0; c < CH; ++c) {
    const int col = (c * kRmsThreads + tid) * 8;
    if (col < cols) *reinterpret_cast<h8_t*>(Y + base + col) = rms_apply(v[c], w[c], r);
  }
}

struct AttnArgs {
  const _Float16* qkv;     // [n_heads * 128 | n_kv * 128 | n_kv * 128]: q, k, v of this token
  _Float16* k_cache;       // [n_kv][max_seq][128]
  _Float16* v_cache;       // [n_kv][max_seq][128]
  const float* rope_cos;   // [max_seq][64], or null: no rotary embedding
  const float* rope_sin;   // [max_seq][64]
  _Float16* out;           // [n_heads * 128]
  float* partial;          // [n_kv][chunks][qpk][2 + 128] when chunks > 1
  uint32_t* counters;      // [n_kv * parts], zero on entry and on exit
  int n_kv, max_seq, pos, qpk;
  int chunks, chunk_tokens;  // chunk c: tokens [c chunk_tokens, ..); chunk_tokens a multiple of 64
  int parts;               // workgroups sharing a kv head's query heads
};

// Element d of the rotary embedding of a 128-vector x at position pos, in the
// rotate-half pairing of transformers' apply_rotary_pos_emb (d with d +- 64),
// from xd = x[d], its partner xp = x[d ^ 64] and the position's cos / sin of
// d mod 64:
//   d <  64: x[d] cos - x[d + 64] sin;   d >= 64: x[d] cos + x[d - 64] sin.
__device__ __forceinline__ float rotate_half(_Float16 xd, _Float16 xp, float c, float s, int d) {
  const float v = static_cast<float>(xd);
  return d < kRopeHalf ? v * c - static_cast<float>(xp) * s : v * c + static_cast<float>(xp) * s;
}

// exp(x - m), 0 where x is -infinity (nothing seen) whatever m is.
__device__ __forceinline__ float exp_below(float x, float m) {
  return __expf(x - (m == -INFINITY ? 0.0f : m));
}

// Grouped-query attention of one decode token: qpk query heads share each kv
// head.  Workgroup (h, c, part) takes HPW of kv head h's query heads and
// cached tokens [c chunk_tokens, min(.. + chunk_tokens, pos + 1)).  Token pos
// is the current one: its k (rotated, rounded to fp16 as the cache holds it)
// and v come from qkv; the first part of the last chunk writes them into the
// caches.
//
// What bounds it: up to a few thousand tokens latency (launch, one round of
// loads, the exchange between workgroups), beyond that the cache stream
// (32768 tokens, 32 heads on 8: 4.4 TB/s).  Against one workgroup per kv head
// and 128 tokens, softmax through LDS and a serial combine, us: 128 tokens
// 6.0 -> 3.8, 1024 10.3 -> 7.5, 8192 29.5 -> 14.5, 32768 97.8 -> 30.7.
// 16 groups of 16 lanes each take every 16th token; lane j of a group holds
// dims 8j..8j+7 of a token's rows (one 16-byte load each).  A round is 64
// tokens, 4 a group, the next round's rows in flight while one is computed:
//   1. scores: HPW dot products a token, summed over the 16-lane group (DPP),
//      so every lane has them;
//   2. each group keeps its own running maximum, sum and P V (8 dims a lane)
//      and rescales them when the maximum moves: no LDS and no barrier;
//   3. at the end the 16 groups' maxima meet in LDS, each scales its sums to
//      the common one, and the outputs are summed in group order.
// With one chunk the output is written directly.  Otherwise each workgroup
// publishes (max, sum, unnormalised P V) with device-coherent stores and the
// last workgroup of (h, part) (agent-scope counter) combines the chunks: chunk
// weights by one wave a head, then every output sums its chunks, all loads of
// up to 16 chunks a thread issued before the weights are known.  Splitting the
// query heads over workgroups (parts) spreads a short context over the CUs
// without more partials, and shares out the combine; the cache rows are then
// read by each part, from L2 (a kv head's workgroups sit on one XCD when n_kv
// is a multiple of 8).  Deterministic, one launch.
template <int HPW>
__global__ __launch_bounds__(kGlueThreads) void attention_decode_kernel(AttnArgs a) {
  constexpr int HD = kHeadDim;
  constexpr int TPG = kRound / 16;                 // tokens per 16-lane group and round
  constexpr float kScale = 0.08838834764831845f;   // 1 / sqrt(128)
  constexpr int SUBS = HPW >= 4 ? 1 : 4 / HPW;     // thread sets of the combine
  constexpr int PAIRS = HPW * HD / 2;              // output pairs
  constexpr int PER = (PAIRS + kGlueThreads - 1) / kGlueThreads;  // pairs per thread
  constexpr int PRE = 16 / PER;                    // chunks a thread loads in one round
  __shared__ float qs[HPW][HD];
  __shared__ __attribute__((aligned(16))) _Float16 knew[HD];
  __shared__ __attribute__((aligned(16))) _Float16 vnew[HD];
  __shared__ __attribute__((aligned(16))) float red[16][HPW][HD];
  __shared__ float mgrp[16][HPW], lgrp[16][HPW];
  __shared__ float wchunk[kAttnMaxChunks][HPW];  // chunk max, then chunk weight
  __shared__ float lchunk[kAttnMaxChunks][HPW];  // chunk sum
  __shared__ float ltot[HPW];
  __shared__ int s_last;

  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const int wave = tid >> 6;
  const int h = blockIdx.x;
  const int c = blockIdx.y;
  const int part = blockIdx.z;
  const int n_heads = a.n_kv * a.qpk;
  const int head0 = h * a.qpk + part * HPW;        // this workgroup's first query head
  const int t0 = c * a.chunk_tokens;
  const int t1 = min(t0 + a.chunk_tokens, a.pos + 1);
  const size_t row0 = static_cast<size_t>(h) * a.max_seq;  // cache row of token 0
  const int g16 = tid >> 4;
  const int j = tid & 15;

  // Every load of the prologue is issued before any of them is used, so the
  // prologue costs one memory round trip: this thread's q elements with their
  // rotary partners and cos / sin, the new token's k and v, then the cached
  // rows (issued last: the rotary work waits only for the loads before them).
  // Buffer loads without branches: a lane with nothing to load passes an
  // offset beyond the resource (it reads zero), and without rotary tables the
  // cos / sin resources are empty.
  constexpr int QE = (HPW * HD + kGlueThreads - 1) / kGlueThreads;  // q elements per thread
  const bool rope = a.rope_cos != nullptr;
  const uint32_t rope_bytes = rope ? static_cast<uint32_t>(a.max_seq) * kRopeHalf * 4u : 0u;
  const auto rq = make_rsrc(a.qkv, static_cast<uint32_t>(n_heads + 2 * a.n_kv) * HD * 2u);
  const auto rcos = make_rsrc(a.rope_cos, rope_bytes);
  const auto rsin = make_rsrc(a.rope_sin, rope_bytes);
  const uint32_t rope_row = static_cast<uint32_t>(a.pos) * kRopeHalf * 4u;
  const bool has_new = t1 == a.pos + 1 && tid < HD;  // holds the new token's k and v
  auto ld16 = [&](uint32_t off) {
    return __builtin_bit_cast(_Float16, __builtin_amdgcn_raw_buffer_load_b16(rq, off, 0, 0));
  };
  auto ld32 = [](__amdgpu_buffer_rsrc_t r, uint32_t off) {
    return __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(r, off, 0, 0));
  };
  _Float16 qx[QE], qp[QE];
  float qc[QE], qn[QE];
#pragma unroll
  for (int u = 0; u < QE; ++u) {
    const int e = tid + u * kGlueThreads;
    const int d = e % HD;
    const uint32_t base = e < HPW * HD ? static_cast<uint32_t>(head0 * HD + e - d) * 2u
                                       : kOutOfRange;
    const uint32_t rot = e < HPW * HD ? rope_row + static_cast<uint32_t>(d & (kRopeHalf - 1)) * 4u
                                      : kOutOfRange;
    qx[u] = ld16(base + static_cast<uint32_t>(d) * 2u);
    qp[u] = ld16(base + static_cast<uint32_t>(d ^ kRopeHalf) * 2u);
    qc[u] = ld32(rcos, rot);
    qn[u] = ld32(rsin, rot);
  }
  const uint32_t kbase = has_new ? static_cast<uint32_t>((n_heads + h) * HD) * 2u : kOutOfRange;
  const uint32_t vbase = has_new ? static_cast<uint32_t>((n_heads + a.n_kv + h) * HD) * 2u
                                 : kOutOfRange;
  const uint32_t krot = has_new ? rope_row + static_cast<uint32_t>(tid & (kRopeHalf - 1)) * 4u
                                : kOutOfRange;
  const _Float16 kx0 = ld16(kbase + static_cast<uint32_t>(tid) * 2u);
  const _Float16 kxp = ld16(kbase + static_cast<uint32_t>(tid ^ kRopeHalf) * 2u);
  const _Float16 vx0 = ld16(vbase + static_cast<uint32_t>(tid) * 2u);
  const float kc = ld32(rcos, krot);
  const float kn_s = ld32(rsin, krot);
  // This kv head's cache rows (max_seq x 128 fp16 each, under 2^31 bytes:
  // max_seq is bounded on the host); rows outside the chunk and the current
  // token's (not written yet) read as zero.
  const uint32_t head_bytes = static_cast<uint32_t>(a.max_seq) * HD * 2u;
  const auto rk = make_rsrc(a.k_cache + row0 * HD, head_bytes);
  const auto rv = make_rsrc(a.v_cache + row0 * HD, head_bytes);
  struct Rows {
    h8_t k[TPG], v[TPG];
  };
  auto load = [&](Rows& r, int tb) {
#pragma unroll
    for (int u = 0; u < TPG; ++u) {
      const int t = tb + g16 + 16 * u;
      const uint32_t off = t < t1 && t != a.pos ? static_cast<uint32_t>(t * HD + 8 * j) * 2u
                                                : kOutOfRange;
      r.k[u] = __builtin_bit_cast(h8_t, __builtin_amdgcn_raw_buffer_load_b128(rk, off, 0, 0));
      r.v[u] = __builtin_bit_cast(h8_t, __builtin_amdgcn_raw_buffer_load_b128(rv, off, 0, 0));
    }
  };
  Rows R0, R1;
  load(R0, t0);
  load(R1, t0 + kRound);

#pragma unroll
  for (int u = 0; u < QE; ++u) {
    const int e = tid + u * kGlueThreads;
    if (e < HPW * HD) {
      const int hq = e / HD, d = e % HD;
      const float v = rope ? rotate_half(qx[u], qp[u], qc[u], qn[u], d) : static_cast<float>(qx[u]);
      qs[hq][d] = v * kScale;
    }
  }
  if (has_new) {
    const _Float16 kn = static_cast<_Float16>(
        rope ? rotate_half(kx0, kxp, kc, kn_s, tid) : static_cast<float>(kx0));
    knew[tid] = kn;
    vnew[tid] = vx0;
    if (part == 0) {
      a.k_cache[(row0 + a.pos) * HD + tid] = kn;
      a.v_cache[(row0 + a.pos) * HD + tid] = vx0;
    }
  }
  __syncthreads();

  float qr[HPW][8], acc[HPW][8], m[HPW], l[HPW];
#pragma unroll
  for (int hq = 0; hq < HPW; ++hq) {
    m[hq] = -INFINITY;
    l[hq] = 0.0f;
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      qr[hq][i] = qs[hq][8 * j + i];
      acc[hq][i] = 0.0f;
    }
  }
  auto round = [&](Rows& r, int tb) {
    float s[TPG][HPW];
#pragma unroll
    for (int u = 0; u < TPG; ++u) {
      const int t = tb + g16 + 16 * u;
      if (t == a.pos) {
        r.k[u] = *reinterpret_cast<const h8_t*>(&knew[8 * j]);
        r.v[u] = *reinterpret_cast<const h8_t*>(&vnew[8 * j]);
      }
#pragma unroll
      for (int hq = 0; hq < HPW; ++hq) {
        float d = 0.0f;
#pragma unroll
        for (int i = 0; i < 8; ++i)
          d = __builtin_fmaf(qr[hq][i], static_cast<float>(r.k[u][i]), d);
        d = row16_sum(d);
        s[u][hq] = t < t1 ? d : -INFINITY;
      }
    }
#pragma unroll
    for (int hq = 0; hq < HPW; ++hq) {
      float top = m[hq];
#pragma unroll
      for (int u = 0; u < TPG; ++u) top = fmaxf(top, s[u][hq]);
      const float keep = exp_below(m[hq], top);
      m[hq] = top;
      l[hq] *= keep;
#pragma unroll
      for (int i = 0; i < 8; ++i) acc[hq][i] *= keep;
#pragma unroll
      for (int u = 0; u < TPG; ++u) {
        const float p = exp_below(s[u][hq], top);
        l[hq] += p;
#pragma unroll
        for (int i = 0; i < 8; ++i)
          acc[hq][i] = __builtin_fmaf(p, static_cast<float>(r.v[u][i]), acc[hq][i]);
      }
    }
  };
  for (int tb = t0; tb < t1; tb += 2 * kRound) {
    round(R0, tb);
    load(R0, tb + 2 * kRound);
    if (tb + kRound >= t1) break;
    round(R1, tb + kRound);
    load(R1, tb + 3 * kRound);
  }

  // The groups' sums on the workgroup's common maximum.
  if (j == 0) {
#pragma unroll
    for (int hq = 0; hq < HPW; ++hq) mgrp[g16][hq] = m[hq];
  }
  __syncthreads();
  float top[HPW];
#pragma unroll
  for (int hq = 0; hq < HPW; ++hq) {
    top[hq] = mgrp[0][hq];
#pragma unroll
    for (int g = 1; g < 16; ++g) top[hq] = fmaxf(top[hq], mgrp[g][hq]);
    const float w = exp_below(m[hq], top[hq]);
    if (j == 0) lgrp[g16][hq] = l[hq] * w;
#pragma unroll
    for (int i = 0; i < 8; ++i) red[g16][hq][8 * j + i] = acc[hq][i] * w;
  }
  __syncthreads();

  const bool direct = a.chunks == 1;
  const size_t part_stride = static_cast<size_t>(a.qpk) * (HD + 2);  // floats per chunk
  float* const P0 = a.partial + (static_cast<size_t>(h) * a.chunks * a.qpk + part * HPW) * (HD + 2);
  for (int e = tid; e < HPW * HD; e += kGlueThreads) {
    const int hq = e / HD, d = e % HD;
    float o = 0.0f, lsum = 0.0f;
#pragma unroll
    for (int g = 0; g < 16; ++g) {
      o += red[g][hq][d];
      lsum += lgrp[g][hq];
    }
    if (direct) {
      a.out[static_cast<size_t>(head0 + hq) * HD + d] = static_cast<_Float16>(o / lsum);
    } else {
      float* P = P0 + c * part_stride + hq * (HD + 2);
      store_coherent(P + 2 + d, o);
      if (d == 0) {
        float t = mgrp[0][hq];
        for (int g = 1; g < 16; ++g) t = fmaxf(t, mgrp[g][hq]);
        store_coherent(P, t);
        store_coherent(P + 1, lsum);
      }
    }
  }
  if (direct) return;

  // Last-arriver exchange; relies on gfx950 hardware ordering: see
  // "HARDWARE ASSUMPTION" in nibble_decode.h.
  wait_vm_stores();
  __syncthreads();
  uint32_t* counter = a.counters + h * a.parts + part;
  if (tid == 0) {
    const uint32_t prev =
        __hip_atomic_fetch_add(counter, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    s_last = prev == static_cast<uint32_t>(a.chunks - 1);
  }
  __syncthreads();
  if (!s_last) return;

  // Thread (sub, pair) sums output pairs `pair` (+ kGlueThreads) over the
  // chunks sub, sub + SUBS, ...; the subs are added in order at the end.
  typedef float f2_t __attribute__((ext_vector_type(2)));
  const auto rp = make_rsrc(P0, static_cast<uint32_t>(a.chunks) * a.qpk * (HD + 2) * 4u);
  auto ld_pair = [&](int cc, int hq, int d) {  // floats d, d + 1 of a chunk's record
    const uint32_t off = cc < a.chunks
                             ? (static_cast<uint32_t>(cc) * a.qpk + hq) * (HD + 2) * 4u + d * 4u
                             : kOutOfRange;
    return __builtin_bit_cast(f2_t, __builtin_amdgcn_raw_buffer_load_b64(rp, off, 0, 16));
  };
  const int sub = SUBS > 1 ? tid / PAIRS : 0;
  const int pair = SUBS > 1 ? tid % PAIRS : tid;
  f2_t pv[PER][PRE];
#pragma unroll
  for (int k = 0; k < PER; ++k)
#pragma unroll
    for (int u = 0; u < PRE; ++u) {
      const int e = pair + k * kGlueThreads;
      pv[k][u] = ld_pair(sub + u * SUBS, e / (HD / 2), 2 + 2 * (e % (HD / 2)));
    }
  for (int e = tid; e < a.chunks * HPW; e += kGlueThreads) {
    const f2_t ml = ld_pair(e / HPW, e % HPW, 0);
    wchunk[e / HPW][e % HPW] = ml[0];
    lchunk[e / HPW][e % HPW] = ml[1];
  }
  __syncthreads();
  for (int hq = wave; hq < HPW; hq += kGlueThreads / 64) {
    float M = -INFINITY;
    for (int cc = lane; cc < a.chunks; cc += 64) M = fmaxf(M, wchunk[cc][hq]);
    M = wave_max(M);
    float L = 0.0f;
    for (int cc = lane; cc < a.chunks; cc += 64) {
      const float w = exp_below(wchunk[cc][hq], M);
      wchunk[cc][hq] = w;
      L += lchunk[cc][hq] * w;
    }
    L = wave_sum(L);
    if (lane == 0) ltot[hq] = L;
  }
  __syncthreads();
#pragma unroll
  for (int k = 0; k < PER; ++k) {
    const int e = pair + k * kGlueThreads;
    const int hq = e / (HD / 2), d = 2 * (e % (HD / 2));
    f2_t o = {0.0f, 0.0f};
#pragma unroll
    for (int u = 0; u < PRE; ++u) {
      const int cc = sub + u * SUBS;
      if (cc < a.chunks) {
        const float w = wchunk[cc][hq];
        o[0] += pv[k][u][0] * w;
        o[1] += pv[k][u][1] * w;
      }
    }
    for (int c0 = sub + PRE * SUBS; c0 < a.chunks; c0 += 8 * SUBS) {  // eight loads a round
      f2_t v[8];
#pragma unroll
      for (int u = 0; u < 8; ++u) v[u] = ld_pair(c0 + u * SUBS, hq, 2 + d);
#pragma unroll
      for (int u = 0; u < 8; ++u)
        if (c0 + u * SUBS < a.chunks) {
          const float w = wchunk[c0 + u * SUBS][hq];
          o[0] += v[u][0] * w;
          o[1] += v[u][1] * w;
        }
    }
    if (SUBS > 1) {
      red[sub][hq][d] = o[0];
      red[sub][hq][d + 1] = o[1];
    } else {
      a.out[static_cast<size_t>(head0 + hq) * HD + d] = static_cast<_Float16>(o[0] / ltot[hq]);
      a.out[static_cast<size_t>(head0 + hq) * HD + d + 1] = static_cast<_Float16>(o[1] / ltot[hq]);
    }
  }
  if (SUBS > 1) {
    __syncthreads();
    for (int e = tid; e < HPW * HD; e += kGlueThreads) {
      const int hq = e / HD, d = e % HD;
      float o = red[0][hq][d];
#pragma unroll
      for (int s2 = 1; s2 < SUBS; ++s2) o += red[s2][hq][d];
      a.out[static_cast<size_t>(head0 + hq) * HD + d] = static_cast<_Float16>(o / ltot[hq]);
    }
  }
  if (tid == 0) __hip_atomic_store(counter, 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

struct AttnPlan {
  int qpk = 0, chunks = 0, chunk_tokens = 0, parts = 1;
  size_t counter_bytes = 0, workspace_bytes = 0;
};

int plan_attention(int64_t n_heads, int64_t n_kv, int64_t head_dim, int64_t max_seq, int64_t pos,
                   AttnPlan* p) {
  NIBBLE_CHECK(head_dim == kHeadDim, "head_dim must be %d, got %lld", kHeadDim,
               (long long)head_dim);
  NIBBLE_CHECK(n_kv >= 1 && n_kv <= 65535, "n_kv_heads must be in [1, 65535], got %lld",
               (long long)n_kv);
  NIBBLE_CHECK(n_heads >= n_kv && n_heads % n_kv == 0,
               "n_heads (%lld) must be a multiple of n_kv_heads (%lld)", (long long)n_heads,
               (long long)n_kv);
  const int64_t qpk = n_heads / n_kv;
  NIBBLE_CHECK(qpk == 1 || qpk == 2 || qpk == 4 || qpk == 8,
               "query heads per kv head must be 1, 2, 4 or 8, got %lld", (long long)qpk);
  NIBBLE_CHECK(pos >= 0 && pos < max_seq, "pos (%lld) must be in [0, max_seq = %lld)",
               (long long)pos, (long long)max_seq);
  NIBBLE_CHECK(max_seq <= kAttnMaxSeq, "max_seq above %d", kAttnMaxSeq);
  p->qpk = static_cast<int>(qpk);
  const int64_t tokens = pos + 1, room = ceil_div(tokens, kChunk);
  const int64_t cache_bytes = n_kv * tokens * kHeadDim * 4;
  if (room > 1) {
    p->counter_bytes = align_up(static_cast<size_t>(n_kv) * (qpk == 8 ? 2 : 1) * 4, 256);
    p->workspace_bytes = p->counter_bytes + static_cast<size_t>(n_kv) * room * qpk *
                                                (kHeadDim + 2) * sizeof(float);
  }
  // Workgroups share a kv head's query heads between them, one head each, as
  // long as reading the cache once per part stays cheap; the tokens are cut
  // into as many chunks as make one round of the CUs (at least 128 tokens
  // each: the workspace has room for no more).  Measured on MI355X, graph
  // replay, 32 heads on 8, us: 1024 tokens 4 parts x 8 chunks 7.5 (1 part 9.5),
  // 4096 tokens 4 x 8 10.6 (2 x 16 11.6, 1 x 32 13.4), 8192 tokens 2 x 16 14.5
  // (4 x 8 15.7, 1 x 32 16.1), 32768 tokens 2 x 16 30.7 (4 x 16 45).  One chunk
  // up to 384 tokens, which saves the exchange: 129 tokens 4.2 (2 chunks 6.2),
  // 256 5.0 (6.3), 512 7.3 (4 chunks 6.7).
  // Workgroups of 8 heads hold one wave a SIMD, so 8 heads make two parts
  // while the second reading comes from the last-level cache: 64 kv heads, 256
  // / 1024 tokens 1 part 16.3 / 21.0, 2 parts 10 / 18.
  // One chunk needs no counters and takes as many parts as keep the grid within
  // a round, or a round and a half where kv heads on 8 XCDs share the rows in
  // L2: 40 / 64 kv heads of 8, 384 tokens 4 parts 8.7 / 8.9 (1 part 21); 129 of
  // 2 1 part 8.6 (2 parts 13.3), 256 of 2 11.4 (13.4).  Where the heads alone
  // make a round, one chunk goes on to 768 tokens: 64 of 8, 700 tokens 12.5 (3
  // chunks 14.2), 96 of 4, 385 tokens 9.6 (2 chunks of 1 part 12.9).
  const bool one_chunk =
      tokens <= (n_kv * qpk >= kAttnWorkgroups ? 2 * kAttnOneChunk : kAttnOneChunk);
  const int64_t least = qpk == 8 && cache_bytes <= kAttnLlcBytes ? 2 : 1;
  const int64_t most = !one_chunk || room == 1 ? 2 * kAttnWorkgroups
                       : n_kv % 8 == 0         ? kAttnWorkgroups * 3 / 2
                                               : kAttnWorkgroups;
  // (Beyond the last-level cache only the padding's worth of counters: 256 kv
  // heads of 8, 4096 tokens 1 part 172, 2 parts 202.)
  const int64_t counters = static_cast<int64_t>(
      least == 2 ? p->counter_bytes / 4 : align_up(static_cast<size_t>(n_kv), 64));
  int64_t parts = qpk;
  while (parts > least &&
         (n_kv * parts > most ||
          (!one_chunk && ((parts > 2 && parts * cache_bytes > kAttnRereadBytes) ||
                          n_kv * parts > counters))))
    parts /= 2;
  // Chunks: one round of the CUs, two where 8 heads make two parts of more than
  // a quarter round (two workgroups a CU: 40 kv heads, 4096 tokens 6 chunks
  // 34.2, 3 38.9).  Above half a round of kv heads and parts, the number up to
  // 4 that wastes the least of the last round, once a workgroup's share is
  // worth an exchange: 129 kv heads of 4, 2048 tokens 3 chunks 33.0 (1: 48), of
  // 2 27.0 (27.9), 1024 tokens of 2 18.2 (16.7); 300 of 1, 2048 tokens 4 chunks
  // 52.8 (61.8), 512 tokens of 4 26.5 (24.0).
  const int64_t groups = n_kv * parts, heads = qpk / parts;
  int64_t chunks = 1;
  if (!one_chunk && groups <= kAttnWorkgroups / 2) {
    const bool pairs = qpk == 8 && parts == 2 && groups > kAttnWorkgroups / 4;
    chunks = kAttnWorkgroups * (pairs ? 2 : 1) / groups;
  } else if (tokens >= 1024 && tokens * heads >= (groups > kAttnWorkgroups ? 1536 : 4096)) {
    auto waste = [&](int64_t c) {  // rounds of the CUs over what they hold
      return static_cast<double>(ceil_div(groups * c, kAttnWorkgroups)) / static_cast<double>(c);
    };
    for (int64_t c = 2; c <= 4; ++c)
      if (waste(c) < 0.999 * waste(chunks)) chunks = c;
  }
  chunks = std::min<int64_t>({room, kAttnMaxChunks, chunks});
  const int64_t each = align_up(static_cast<size_t>(ceil_div(tokens, chunks)), kRound);
  p->parts = static_cast<int>(parts);
  p->chunk_tokens = static_cast<int>(each);
  p->chunks = static_cast<int>(ceil_div(tokens, each));
  return NIBBLE_OK;
}

template <int HPW>
hipError_t launch_attention(const AttnArgs& a, hipStream_t stream) {
  dim3 grid(static_cast<unsigned>(a.n_kv), static_cast<unsigned>(a.chunks),
            static_cast<unsigned>(a.parts));
  attention_decode_kernel<HPW><<<grid, kGlueThreads, 0, stream>>>(a);
  return hipGetLastError();
}

template <int CH>
hipError_t launch_rmsnorm(const _Float16* X, const _Float16* W, _Float16* Y, int64_t rows,
                          int cols, float eps, hipStream_t stream) {
  rmsnorm_kernel<CH><<<dim3(static_cast<unsigned>(rows)), kGlueThreads, 0, stream>>>(X, W, Y, cols,
                                                                                    eps);
  return hipGetLastError();
}

}  // namespace

}  // namespace nibble

using namespace nibble;

extern "C" int nibble_rmsnorm_f16(const void* X, int64_t rows, int64_t cols, const void* W,
                                  float eps, void* Y, void* stream_) {
  NIBBLE_CHECK(rows >= 0 && rows <= 0x7fffffff, "rows must be in [0, 2^31), got %lld",
               (long long)rows);
  NIBBLE_CHECK(cols > 0 && cols % 8 == 0 && cols <= kRmsMaxCols,
               "cols must be a positive multiple of 8 up to %d, got %lld", kRmsMaxCols,
               (long long)cols);
  NIBBLE_CHECK(std::isfinite(eps) && eps >= 0.0f, "eps must be finite and >= 0");
  if (rows == 0) return ok();
  NIBBLE_CHECK(X != nullptr && W != nullptr && Y != nullptr, "null pointer");
  NIBBLE_CHECK(aligned(X, 16) && aligned(W, 16) && aligned(Y, 16),
               "X, W and Y must be 16-byte aligned");
  hipStream_t stream = static_cast<hipStream_t>(stream_);
  DeviceGuard guard;
  int dev = 0;
  NIBBLE_HIP(guard.enter(stream, &dev));
  const auto* x = static_cast<const _Float16*>(X);
  const auto* w = static_cast<const _Float16*>(W);
  auto* y = static_cast<_Float16*>(Y);
  const int c = static_cast<int>(cols);
  const int ch = static_cast<int>(ceil_div(cols, kGlueThreads * 8));
  hipError_t e = ch <= 1   ? launch_rmsnorm<1>(x, w, y, rows, c, eps, stream)
                 : ch <= 2 ? launch_rmsnorm<2>(x, w, y, rows, c, eps, stream)
                 : ch <= 4 ? launch_rmsnorm<4>(x, w, y, rows, c, eps, stream)
                           : launch_rmsnorm<8>(x, w, y, rows, c, eps, stream);
  NIBBLE_HIP(e);
  return ok();
}

extern "C" size_t nibble_attention_decode_workspace_bytes(int64_t n_heads, int64_t n_kv_heads,
                                                          int64_t head_dim, int64_t max_seq,
                                                          int64_t pos, void* stream) {
  (void)stream;
  AttnPlan p;
  if (plan_attention(n_heads, n_kv_heads, head_dim, max_seq, pos, &p) != NIBBLE_OK) return 0;
  return p.workspace_bytes;
}

extern "C" size_t nibble_attention_decode_counter_bytes(int64_t n_heads, int64_t n_kv_heads,
                                                        int64_t head_dim, int64_t max_seq,
                                                        int64_t pos, void* stream) {
  (void)stream;
  AttnPlan p;
  if (plan_attention(n_heads, n_kv_heads, head_dim, max_seq, pos, &p) != NIBBLE_OK) return 0;
  return p.counter_bytes;
}

extern "C" int nibble_attention_decode_f16(const void* QKV, int64_t n_heads, int64_t n_kv_heads,
                                           int64_t head_dim, void* K_cache, void* V_cache,
                                           int64_t max_seq, int64_t pos, const void* rope_cos,
                                           const void* rope_sin, void* Out, void* workspace,
                                           size_t workspace_bytes, void* stream_) {
  AttnPlan p;
  int rc = plan_attention(n_heads, n_kv_heads, head_dim, max_seq, pos, &p);
  if (rc != NIBBLE_OK) return rc;
  NIBBLE_CHECK(QKV != nullptr && K_cache != nullptr && V_cache != nullptr && Out != nullptr,
               "null pointer");
  NIBBLE_CHECK(aligned(QKV, 16) && aligned(K_cache, 16) && aligned(V_cache, 16) &&
                   aligned(Out, 16),
               "qkv, caches and output must be 16-byte aligned");
  NIBBLE_CHECK((rope_cos == nullptr) == (rope_sin == nullptr),
               "rope_cos and rope_sin must both be given or both be null");
  NIBBLE_CHECK(rope_cos == nullptr || (aligned(rope_cos, 4) && aligned(rope_sin, 4)),
               "rope tables must be 4-byte aligned");
  if (p.workspace_bytes > 0) {
    if (workspace == nullptr || workspace_bytes < p.workspace_bytes)
      return fail(NIBBLE_ERR_WORKSPACE, "attention needs %zu bytes of workspace, got %zu",
                  p.workspace_bytes, workspace == nullptr ? size_t(0) : workspace_bytes);
    if (!aligned(workspace, 256))
      return fail(NIBBLE_ERR_WORKSPACE, "workspace must be 256-byte aligned");
  }
  hipStream_t stream = static_cast<hipStream_t>(stream_);
  DeviceGuard guard;
  int dev = 0;
  NIBBLE_HIP(guard.enter(stream, &dev));
  AttnArgs a;
  a.qkv = static_cast<const _Float16*>(QKV);
  a.k_cache = static_cast<_Float16*>(K_cache);
  a.v_cache = static_cast<_Float16*>(V_cache);
  a.rope_cos = static_cast<const float*>(rope_cos);
  a.rope_sin = static_cast<const float*>(rope_sin);
  a.out = static_cast<_Float16*>(Out);
  a.counters = p.chunks > 1 ? static_cast<uint32_t*>(workspace) : nullptr;
  a.partial = p.chunks > 1
                  ? reinterpret_cast<float*>(static_cast<char*>(workspace) + p.counter_bytes)
                  : nullptr;
  a.n_kv = static_cast<int>(n_kv_heads);
  a.max_seq = static_cast<int>(max_seq);
  a.pos = static_cast<int>(pos);
  a.chunks = p.chunks;
  a.chunk_tokens = p.chunk_tokens;
  a.parts = p.parts;
  a.qpk = p.qpk;
  const int heads_per_wg = p.qpk / p.parts;
  hipError_t e = heads_per_wg == 1   ? launch_attention<1>(a, stream)
                 : heads_per_wg == 2 ? launch_attention<2>(a, stream)
                 : heads_per_wg == 4 ? launch_attention<4>(a, stream)
                                     : launch_attention<8>(a, stream);
  NIBBLE_HIP(e);
  return ok();
}
