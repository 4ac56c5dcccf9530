// kernels_prefill.h -- HIP/CDNA4 kernels of the batched prefill (gfx950, wave64).
//
// Prefill runs every layer over a chunk of T prompt tokens at once.  Each token's arithmetic
// is the decode step's, in the same order (so the KV cache and the hidden states are
// bit-identical to T single-token steps, and to the CPU path, inference.rs:4411-4425):
//   RMSNorm rows     k_rmsnorm_quant with gridDim.y = T (one workgroup per token)
//   projections      k_gemm_q8: int8 matrix cores for the per-block dots, f32 folds in block order
//   QK-norm/RoPE/KV  k_rope_kv with gridDim.y = T
//   attention        k_attn_prefill_mm: 16 (head, token) rows per workgroup, products on the matrix
//                    cores; k_attn_prefill: one workgroup per (head, token); causal over [0, pos]
//   SwiGLU           k_silu_rows
#pragma once
#include "kernels_decode.h"
#include "kernels_gemm_q8.h"

namespace cm {

typedef int v4i_t __attribute__((ext_vector_type(4)));

// ---------------------------------------------------------------------------
// Greedy argmax (inference.rs:5912-5925: first index of the max, strict '>') of T rows of n
// logits: workgroup (p, t) reduces slice p of row t to a (value, index) pair, then one
// wave per row reduces the AMR_PARTS pairs; a row with no value above -inf gives 0.
constexpr int AMR_PARTS = 64;
__global__ __launch_bounds__(256) void k_argmax_rows_part(const float* __restrict__ x, int n,
                                                          float* __restrict__ pv, uint32_t* __restrict__ pi) {
  __shared__ float rv[4];
  __shared__ uint32_t ri[4];
  const int t = blockIdx.y, p = blockIdx.x, tid = threadIdx.x;
  const int per = (n + AMR_PARTS - 1) / AMR_PARTS;
  const int lo = p * per, hi = min(n, lo + per);
  const float* row = x + (size_t)t * n;
  float bv = -INFINITY;
  uint32_t bi = 0xffffffffu;
  for (int i = lo + tid; i < hi; i += 256) {
    const float v = row[i];
    if (v > bv) {
      bv = v;
      bi = (uint32_t)i;
    }
  }
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) argmax_pair(bv, bi, __shfl_xor(bv, o), __shfl_xor(bi, o));
  if ((tid & 63) == 0) {
    rv[tid >> 6] = bv;
    ri[tid >> 6] = bi;
  }
  __syncthreads();
  if (tid == 0) {
    for (int w = 1; w < 4; ++w) argmax_pair(bv, bi, rv[w], ri[w]);
    pv[t * AMR_PARTS + p] = bv;
    pi[t * AMR_PARTS + p] = bi;
  }
}

__global__ __launch_bounds__(64) void k_argmax_rows_finish(const float* __restrict__ pv,
                                                           const uint32_t* __restrict__ pi,
                                                           uint32_t* __restrict__ out) {
  const int t = blockIdx.x, lane = threadIdx.x;
  float bv = pv[t * AMR_PARTS + lane];
  uint32_t bi = pi[t * AMR_PARTS + lane];
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) argmax_pair(bv, bi, __shfl_xor(bv, o), __shfl_xor(bi, o));
  if (lane == 0) out[t] = bi == 0xffffffffu ? 0u : bi;
}

// ---------------------------------------------------------------------------
// Y[t] = W . X[t] (+ resid[t]) for 1 <= T <= GMT_MAX tokens (the shortest verify and
// prefill chunks; k_gemv_mm above, and at four where it is faster): the single-token GEMV's arithmetic for every (row, token) -- exact int32
// block dots, terms ((float)dot * d_w) * d_x, the in-order fold over blocks -- with each
// weight chunk loaded once and dotted with all T activations (a 64-token matrix-core tile
// would leave most CUs idle at this size).  4 waves x GMT_RPW rows per workgroup.
// Dynamic LDS: gemv_multi_lds_bytes(K, T).
constexpr int GMT_MAX = 4;
constexpr int GMT_RPW = 1;
constexpr int GMT_ROWS = 4 * GMT_RPW;
// LDS: the activations [T][K] i8 and their scales [T][K/32] f32, each rounded up to whole
// 1 KB wave loads (a direct load writes all 64 lanes' 16 bytes, the last one past the data),
// then per wave the terms of one 32-block slice [GMT_RPW][T][32] f32
__host__ __device__ inline size_t gemv_multi_xq_bytes(int K, int T) {
  return (((size_t)T * K + 1023) / 1024) * 1024;
}
__host__ __device__ inline size_t gemv_multi_xs_bytes(int K, int T) {
  return (((size_t)T * (K / 32) * 4 + 1023) / 1024) * 1024;
}
__host__ __device__ inline size_t gemv_multi_lds_bytes(int K, int T) {
  return gemv_multi_xq_bytes(K, T) + gemv_multi_xs_bytes(K, T) + (size_t)GMT_ROWS * T * 32 * 4;
}

template <int K>
__global__ __launch_bounds__(256) void k_gemv_multi(const int8_t* __restrict__ wq, const uint16_t* __restrict__ wd,
                                                    int rows, const int8_t* __restrict__ xq,
                                                    const float* __restrict__ xs, int T, float* y,
                                                    const float* resid) {
  constexpr int NB = K / 32, CPR = K / 16, IT = (CPR + 63) / 64;
  static_assert(NB % 4 == 0, "compile-time GEMV widths are multiples of 128");
  extern __shared__ __align__(16) unsigned char gmt_lds[];
  int8_t* xl = reinterpret_cast<int8_t*>(gmt_lds);                    // [T][K]
  float* xsl = reinterpret_cast<float*>(gmt_lds + gemv_multi_xq_bytes(K, T));  // [T][NB]
  // this wave's slice terms [GMT_RPW][T][32]
  float* tw = reinterpret_cast<float*>(gmt_lds + gemv_multi_xq_bytes(K, T) + gemv_multi_xs_bytes(K, T)) +
              (size_t)(threadIdx.x >> 6) * GMT_RPW * T * 32;
  const int tid = threadIdx.x, wave = tid >> 6, lane = tid & 63;
  const int row0 = blockIdx.x * GMT_ROWS;
  // the activations and their scales go to LDS by direct loads (1 KB per wave load; a last
  // load may overrun into its region's rounded-up pad, re-reading the last piece)
  {
    const uint4* sx = reinterpret_cast<const uint4*>(xq);
    const uint4* ss = reinterpret_cast<const uint4*>(xs);
    uint4* dx = reinterpret_cast<uint4*>(xl);
    uint4* ds = reinterpret_cast<uint4*>(xsl);
    const int nx = T * CPR, ns = (T * NB * 4 + 15) / 16;
    for (int b = wave * 64; b < nx; b += 256)
      __builtin_amdgcn_global_load_lds(reinterpret_cast<const void*>(sx + min(b + lane, nx - 1)),
                                       (__attribute__((address_space(3))) void*)(dx + b), 16, 0, 0);
    for (int b = wave * 64; b < ns; b += 256)
      __builtin_amdgcn_global_load_lds(reinterpret_cast<const void*>(ss + min(b + lane, ns - 1)),
                                       (__attribute__((address_space(3))) void*)(ds + b), 16, 0, 0);
  }
  int4 wv[GMT_RPW][IT];
  uint16_t dv[GMT_RPW][IT];
#pragma unroll
  for (int k = 0; k < GMT_RPW; ++k) {
    const int row = min(row0 + wave * GMT_RPW + k, rows - 1);
    const int4* w4 = reinterpret_cast<const int4*>(wq + (size_t)row * K);
    const uint16_t* d = wd + (size_t)row * NB;
#pragma unroll
    for (int i = 0; i < IT; ++i) {
      const int c = min(lane + 64 * i, CPR - 1);
      wv[k][i] = ld_stream(w4 + c);
      dv[k][i] = ld_stream(d + (c >> 1));
    }
  }
  __builtin_amdgcn_s_waitcnt((7 << 4) | (15 << 8));  // vmcnt(0): this wave's direct loads have landed
  __syncthreads();
  // slice i = blocks 32 i .. 32 i + 31 of every (row, token): lane pairs form the block terms
  // into LDS, then lane f (< GMT_RPW * T) continues the in-order fold of (row f / T, token
  // f % T) over them (wave-level ordering only: the slice buffer is this wave's)
  auto wave_sync = [] {
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
  };
  float acc = 0.0f;
#pragma unroll
  for (int i = 0; i < IT; ++i) {
    const int c = lane + 64 * i;
    const int cc = min(c, CPR - 1);
#pragma unroll
    for (int k = 0; k < GMT_RPW; ++k) {
      const float dw = half_bits_to_float(dv[k][i]);
      for (int tk = 0; tk < T; ++tk) {
        int sacc = dot4x4(wv[k][i], reinterpret_cast<const int4*>(xl + (size_t)tk * K)[cc], 0);
        sacc += dpp_xor1(sacc);
        if ((lane & 1) == 0 && c < CPR)
          tw[(k * T + tk) * 32 + (lane >> 1)] = ((float)sacc * dw) * xsl[tk * NB + (c >> 1)];
      }
    }
    wave_sync();
    if (lane < GMT_RPW * T) {
      const int nb = min(32, NB - 32 * i);
      acc = fold_lds(tw + (size_t)lane * 32, nb, acc);
    }
    wave_sync();
  }
  if (lane < GMT_RPW * T) {
    const int lr = wave * GMT_RPW + lane / T, tk = lane - (lane / T) * T;
    const int row = row0 + lr;
    if (row < rows) {
      const size_t o = (size_t)tk * rows + row;
      y[o] = resid ? resid[o] + acc : acc;
    }
  }
}

// ---------------------------------------------------------------------------
// The same on the matrix cores for 1 <= T <= GMM_MAX tokens (speculative verify, short
// prefill chunks): the single-token GEMV's arithmetic for every (row, token) -- exact int32
// block dots, terms ((float)dot * d_w) * d_x, the in-order fold over blocks.
// One v_mfma_i32_16x16x64_i8 gives the dots of 16 rows with 8 tokens for TWO blocks: the weights
// are the B operand as they lie in memory (lane (n, g): bytes 16 g .. +15 of 64 of row n), the
// activations the A operand, its 16 rows being (token, block of the two), zero in the other
// block's half of K.  Row m is token 2 (m / 4) + m % 2 and block m / 2 % 2, so lane (n, g) gets
// tokens 2 g, 2 g + 1 of row n in both blocks, and every lane's four terms are wanted.
// Workgroup: 16 rows; each wave takes GMM_SEG values of K, all its loads in flight at once (8 KB
// of weights per wave, plain loads: a 128-byte line is the two halves of two loads, and streaming
// ones fetched it twice: the large shape below 106 us), and leaves its terms in LDS; then one wave
// per token of the pair adds them in block order, reading a segment ahead.  The grid is what the
// device holds: a wave's activations stay in its registers over all its row tiles, and the next
// tile's weights are on their way while this one's terms are formed and added.  More than
// GMM_WAVES segments go in slices with the sums carried along.
// Bound by HBM on large matrices, by the latency of one load, product and fold on small ones.
// Measured, weights from HBM, 8 tokens (us, k_gemv_multi / this): [16384 x 3072] 24.4 / 13.4, [5120 x
// 3072] 10.2 / 8.0, [3072 x 3072] 7.9 / 5.6, [3072 x 8192] 25.1 / 10.8, [128256 x 3072] 156 / 80 (5.2
// TB/s), [28672 x 4096] 55.6 / 31.6; two slices (the prefill GEMM / this): [4096 x 14336] 44.6 / 19.7,
// [5120 x 13824] 52 / 32.3.
// K % GMM_SEG == 0; scales of either side at any alignment of their type (16-byte loads all the same:
// global memory takes them at any byte).
constexpr int GMM_MAX = 8;
constexpr int GMM_SEG = 512;   // values of K per wave and slice: 8 chunks of two blocks
constexpr int GMM_WAVES = 16;  // waves of a workgroup at most
constexpr int GMM_ROWS = 16;
typedef uint32_t gmm_u4_t __attribute__((ext_vector_type(4), aligned(2)));  // eight f16 scales
typedef float gmm_f4_t __attribute__((ext_vector_type(4), aligned(4)));     // four f32 scales
// waves per workgroup (the last one idle in the products at K = 512: the fold wants two)
inline int gemv_mm_waves(int K) {
  const int segs = K / GMM_SEG, slices = (segs + GMM_WAVES - 1) / GMM_WAVES;
  const int w = (segs + slices - 1) / slices;
  return w < 2 ? 2 : w;
}
inline bool gemv_mm_sliced(int K) { return K / GMM_SEG > GMM_WAVES; }
// per wave: the terms of a segment, then its activation scales [two chunks][token][block]
constexpr int GMM_WAVE_LDS = 8 * 64 * 16 + GMM_MAX * (GMM_SEG / 32) * 4;
inline size_t gemv_mm_lds_bytes(int K) { return (size_t)gemv_mm_waves(K) * GMM_WAVE_LDS; }
// resident workgroups (four waves per SIMD at 128 registers; their LDS fits too)
inline int gemv_mm_grid(int rows, int K) {
  const int tiles = (rows + GMM_ROWS - 1) / GMM_ROWS, res = 256 * (16 / gemv_mm_waves(K));
  return tiles < res ? tiles : res;
}

// SLICED: rows of more than one slice (gemv_mm_sliced(K)).
template <bool SLICED>
__global__ __launch_bounds__(GMM_WAVES * 64) void k_gemv_mm(const int8_t* __restrict__ wq,
                                                            const uint16_t* __restrict__ wd, int rows, int K,
                                                            const int8_t* __restrict__ xq,
                                                            const float* __restrict__ xs, int T, float* y,
                                                            const float* resid) {
  extern __shared__ __align__(16) unsigned char gmm_lds[];
  // [segment of the slice][two chunks][token % 2][lane]: the terms of four blocks
  float4* terms = reinterpret_cast<float4*>(gmm_lds);
  const int tid = threadIdx.x, wave = tid >> 6, lane = tid & 63, W = blockDim.x >> 6;
  const int n = lane & 15, g = lane >> 4, NB = K >> 5, segs = K / GMM_SEG;
  const int tiles = (rows + GMM_ROWS - 1) / GMM_ROWS;
  // as A row n and K group g: the token, and whether this half of K is its block
  const int xt = 2 * (n >> 2) + (n & 1);
  const bool xon = xt < T && (g >> 1) == ((n >> 1) & 1);
  int4 wv[8];
  gmm_u4_t dv[2];
  v4i_t xv[8];
  float4* sl = terms + (size_t)W * 8 * 64 + wave * (GMM_MAX * GMM_SEG / 32 / 4);
  auto load_x = [&](int sg) __attribute__((always_inline)) {
    const int8_t* xp = xq + (size_t)min(xt, T - 1) * K + sg * GMM_SEG + 16 * g;
    // (lane: token lane / 4 % 8, blocks 4 (lane % 4) .. + 3)
    const gmm_f4_t sc =
        reinterpret_cast<const gmm_f4_t*>(xs + (size_t)min((lane >> 2) & 7, T - 1) * NB + sg * 16)[lane & 3];
#pragma unroll
    for (int c = 0; c < 8; ++c) xv[c] = v4i_t{0, 0, 0, 0};
    if (xon) {
#pragma unroll
      for (int c = 0; c < 8; ++c) xv[c] = *reinterpret_cast<const v4i_t*>(xp + 64 * c);
    }
    if (lane < 32) sl[(lane & 3) * GMM_MAX + (lane >> 2)] = make_float4(sc.x, sc.y, sc.z, sc.w);
    // (this wave's own LDS, read by all its lanes: wave-level ordering only)
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
  };
  auto w_at = [&](int tile, int sg) __attribute__((always_inline)) {
    return wq + (size_t)min(tile * GMM_ROWS + n, rows - 1) * K + sg * GMM_SEG + 16 * g;
  };
  auto d_at = [&](int tile, int sg) __attribute__((always_inline)) {
    return reinterpret_cast<const gmm_u4_t*>(wd + (size_t)min(tile * GMM_ROWS + n, rows - 1) * NB + sg * 16);
  };
  auto load_w = [&](const int8_t* wn, const gmm_u4_t* dn) __attribute__((always_inline)) {
#pragma unroll
    for (int c = 0; c < 8; ++c) wv[c] = *reinterpret_cast<const int4*>(wn + 64 * c);
#pragma unroll
    for (int i = 0; i < 2; ++i) dv[i] = dn[i];
  };
  // the terms of a segment; with next, a chunk's registers take the next segment's loads as soon
  // as its product is issued
  auto segment = [&](auto nextc, const int8_t* wn, const gmm_u4_t* dn) __attribute__((always_inline)) {
    constexpr bool next = decltype(nextc)::value;
    float4* tp = terms + (size_t)wave * 8 * 64 + lane;
#pragma unroll
    for (int c2 = 0; c2 < 4; ++c2) {
      float t[2][4];  // [token][block]
      const float4 sv[2] = {sl[c2 * GMM_MAX + 2 * g], sl[c2 * GMM_MAX + 2 * g + 1]};
#pragma unroll
      for (int u = 0; u < 2; ++u) {
        const int c = 2 * c2 + u;
        const v4i_t d = __builtin_amdgcn_mfma_i32_16x16x64_i8(xv[c], v4i_t{wv[c].x, wv[c].y, wv[c].z, wv[c].w},
                                                              v4i_t{0, 0, 0, 0}, 0, 0, 0);
        if constexpr (next) wv[c] = *reinterpret_cast<const int4*>(wn + 64 * c);
        const uint32_t h2[4] = {dv[c >> 2].x, dv[c >> 2].y, dv[c >> 2].z, dv[c >> 2].w};
        const float w0 = half_bits_to_float((uint16_t)(h2[c & 3] & 0xffffu));
        const float w1 = half_bits_to_float((uint16_t)(h2[c & 3] >> 16));
#pragma unroll
        for (int p = 0; p < 2; ++p) {
          t[p][2 * u] = ((float)d[p] * w0) * (u ? sv[p].z : sv[p].x);
          t[p][2 * u + 1] = ((float)d[2 + p] * w1) * (u ? sv[p].w : sv[p].y);
        }
      }
      if constexpr (next)
        if (c2 & 1) dv[c2 >> 1] = dn[c2 >> 1];
#pragma unroll
      for (int p = 0; p < 2; ++p) tp[(c2 * 2 + p) * 64] = make_float4(t[p][0], t[p][1], t[p][2], t[p][3]);
    }
  };
  int tile = blockIdx.x, s0 = 0;
  const int8_t* wn = w_at(tile, min(wave, segs - 1));
  const gmm_u4_t* dn = d_at(tile, min(wave, segs - 1));
  if (wave < segs) {
    load_w(wn, dn);
    load_x(wave);
  }
  float acc = 0.0f;  // waves 0, 1: token 2 g + wave of row n
  for (;;) {
    // what follows: the next slice of the tile, or the first of the next tile
    const bool last_slice = !SLICED || s0 + W >= segs;
    const int nt = last_slice ? tile + (int)gridDim.x : tile, ns = last_slice ? 0 : s0 + W;
    const int sn = ns + wave;
    const bool more = nt < tiles && sn < segs;  // this wave has work there
    wn = w_at(nt, min(sn, segs - 1));
    dn = d_at(nt, min(sn, segs - 1));
    if (s0 + wave < segs) {
      if (more)
        segment(std::true_type{}, wn, dn);
      else
        segment(std::false_type{}, wn, dn);
    } else if (SLICED && more) {  // idle in a short last slice, not in what follows
      load_w(wn, dn);
    }
    if (SLICED && more) load_x(sn);
    __syncthreads();
    if (wave < 2) {
      const float4* tp = terms + wave * 64 + lane;
      const int ns4 = min(W, segs - s0);
      // a segment's 16 terms are read while the one before is added
      float4 va[4], vb[4];
      auto rd = [&](float4* v, int i) __attribute__((always_inline)) {
#pragma unroll
        for (int u = 0; u < 4; ++u) v[u] = tp[(min(i, ns4 - 1) * 4 + u) * 128];
      };
      auto add = [&](const float4* v) __attribute__((always_inline)) {
#pragma unroll
        for (int u = 0; u < 4; ++u) {
          acc += v[u].x;
          acc += v[u].y;
          acc += v[u].z;
          acc += v[u].w;
        }
      };
      rd(va, 0);
#pragma unroll 1
      for (int i = 0; i < ns4; i += 2) {
        rd(vb, i + 1);
        add(va);
        rd(va, i + 2);
        if (i + 1 < ns4) add(vb);
      }
      if (last_slice) {
        const int t = 2 * g + wave, r = tile * GMM_ROWS + n;
        if (t < T && r < rows) {
          const size_t o = (size_t)t * rows + r;
          y[o] = resid ? resid[o] + acc : acc;
        }
        acc = 0.0f;
      }
    }
    if (nt >= tiles) break;
    __syncthreads();
    tile = nt;
    s0 = ns;
  }
}

// ---------------------------------------------------------------------------
// Causal attention of a prefill chunk (attention_batched, cuda_resident.rs:1994; CPU
// inference.rs:23945-24025 per token): one workgroup per (query head, token); token t of
// the chunk sits at position pos0 + t and attends positions [0, pos0 + t], all already in
// the cache.  The arithmetic is the decode kernel's: scores one lane per position with d in
// order, exact max, glibc expf, a serial fold of the exponentials, normalisation by the
// reciprocal, and out_d folded over positions in order (one lane per d).  A single position
// copies the V row (inference.rs:23564-23575).  The output row is quantized to Q8_0.
// Rows are dealt longest first.  Dynamic LDS: align4(pos0 + T) floats.
constexpr int AP_NT = 256;

template <int HD>
__global__ __launch_bounds__(AP_NT) void k_attn_prefill(const float* __restrict__ qrot, int n_heads, int n_kv,
                                                        const uint16_t* __restrict__ kc, const uint16_t* __restrict__ vc,
                                                        int layer, int kvs, int pos0, float scale,
                                                        float* __restrict__ att_out, int8_t* __restrict__ xq,
                                                        float* __restrict__ xs) {
  static_assert(HD % 64 == 0 && HD <= AP_NT, "head_dim must be 64, 128 or 256");
  constexpr int R8 = HD / 8;
  extern __shared__ __align__(16) float sc[];
  __shared__ __align__(16) float qs[HD];
  __shared__ float red[AP_NT / 64];
  __shared__ float s_inv;
  const int tid = threadIdx.x;
  const int h = blockIdx.x;
  const int t = (int)gridDim.y - 1 - (int)blockIdx.y;
  const int pos = pos0 + t, P = pos + 1;
  const int kvh = h / (n_heads / n_kv);
  const size_t hbase = kv_head_base(layer, n_kv, kvh, HD, kvs);
  const uint4* kg = reinterpret_cast<const uint4*>(kc + hbase);
  const uint4* vg = reinterpret_cast<const uint4*>(vc + hbase);
  const size_t row = (size_t)t * n_heads * HD + (size_t)h * HD;
  if (tid < HD) qs[tid] = qrot[row + tid];
  __syncthreads();
  float o = 0.0f;
  if (P == 1) {
    if (tid < HD) o = half_bits_to_float(vc[hbase + kv_v_index(HD, 0, tid)]);
  } else {
    float lmax = -INFINITY;
    for (int p = tid; p < P; p += AP_NT) {
      uint4 rk[R8];
#pragma unroll
      for (int u = 0; u < R8; ++u) rk[u] = kg[(size_t)u * kvs + p];
      float a = 0.0f;
#pragma unroll
      for (int u = 0; u < R8; ++u) {
        __builtin_amdgcn_sched_barrier(0);
        const float4 qa = reinterpret_cast<const float4*>(qs)[2 * u];
        const float4 qb = reinterpret_cast<const float4*>(qs)[2 * u + 1];
        a += mul_f16_lo(qa.x, rk[u].x);
        a += mul_f16_hi(qa.y, rk[u].x);
        a += mul_f16_lo(qa.z, rk[u].y);
        a += mul_f16_hi(qa.w, rk[u].y);
        a += mul_f16_lo(qb.x, rk[u].z);
        a += mul_f16_hi(qb.y, rk[u].z);
        a += mul_f16_lo(qb.z, rk[u].w);
        a += mul_f16_hi(qb.w, rk[u].w);
      }
      const float sv = a * scale;
      sc[p] = sv;
      lmax = fmaxf(lmax, sv);
    }
    const float mx = block_max(lmax, red);
    for (int p = tid; p < P; p += AP_NT) sc[p] = glibc_expf(sc[p] - mx);
    __syncthreads();
    if (tid == 0) s_inv = 1.0f / fold_lds(sc, P);
    __syncthreads();
    const float inv = s_inv;
    for (int p = tid; p < P; p += AP_NT) sc[p] = sc[p] * inv;
    __syncthreads();
    if (tid < HD) {
      const int ng = P >> 3;  // full granules of 8 positions (f16 V, one FMA-mix product each)
      const float4* pr4 = reinterpret_cast<const float4*>(sc);
      float a = 0.0f;
      auto granule = [&](const uint4& g, int j) {
        const float4 p0 = pr4[2 * j], p1 = pr4[2 * j + 1];
        const float r0 = mul_f16_lo(p0.x, g.x), r1 = mul_f16_hi(p0.y, g.x);
        const float r2 = mul_f16_lo(p0.z, g.y), r3 = mul_f16_hi(p0.w, g.y);
        const float r4 = mul_f16_lo(p1.x, g.z), r5 = mul_f16_hi(p1.y, g.z);
        const float r6 = mul_f16_lo(p1.z, g.w), r7 = mul_f16_hi(p1.w, g.w);
        a += r0;
        a += r1;
        a += r2;
        a += r3;
        a += r4;
        a += r5;
        a += r6;
        a += r7;
      };
      int j = 0;
      for (; j + 4 <= ng; j += 4) {
        uint4 v[4];
#pragma unroll
        for (int u = 0; u < 4; ++u) v[u] = vg[(size_t)(j + u) * HD + tid];
#pragma unroll
        for (int u = 0; u < 4; ++u) granule(v[u], j + u);
      }
      for (; j < ng; ++j) granule(vg[(size_t)j * HD + tid], j);
      for (int p = ng * 8; p < P; ++p) a += sc[p] * half_bits_to_float(vc[hbase + kv_v_index(HD, p, tid)]);
      o = a;
    }
  }
  if (tid < HD) {
    if (att_out) att_out[row + tid] = o;
    int8_t q;
    const float dd = quantize_lane32(o, &q);
    xq[row + tid] = q;
    if ((tid & 31) == 0) xs[(row + tid) >> 5] = dd;
  }
}

// ---------------------------------------------------------------------------
// Causal attention of a prefill chunk, tiled over query tokens (attention_batched and the
// flash prefill of cuda_resident.rs:1994, :2523-2757; CPU inference.rs:23945-24025 per token),
// its products formed on the matrix cores.
// Both sums of the attention are, per term, an outer product: term d of the scores of 16 rows
// and some positions is q_d[row] * k_d[position], term p of the outputs of 16 rows and some dims
// is prob_p[row] * v_p[dim].  v_mfma_f32_16x16x1_4b with a zero addend forms four such 16 x 16
// product tiles, each product rounded once to nearest even (bit for bit v_mul_f32, subnormals
// included), and the VALU then only adds, in order.  1024 products and their adds take 67-77
// clocks of a SIMD (two or more waves, four product tiles issued together) where products from
// v_fma_mix_f32 (half the rate of v_add_f32) and their adds take 111, and the operands are one
// register each instead of LDS reads of both.
//
// One workgroup per (16 rows, KV head), the KV heads of a tile in consecutive workgroups (with 8 of
// them, a head's K/V stay in one XCD's L2): row R = 16 * tile + r of the KV head's T * rep rows is
// query head R % rep of the group at token R / rep.  W = HD / 32 waves; lane l of a wave is
// l % 16 = lr in block l / 16 = lb.  A wave's product covers 16 rows x 32 columns (positions or
// dims) for two terms: blocks 0, 1 are columns 0-15, 16-31 of the first term, blocks 2, 3 of the
// second (cbsz 1: blocks 0, 1 share one A block, 2, 3 another; abid picks which of two terms'
// rows a register holds for each).  A term pair is (8 g + c, 8 g + 4 + c): four products c = 0..3
// give the 8 terms of one 16-byte granule, which the adds take in order.
//   A  wave w takes the 32-position blocks w, w + W, ...: q in HD / 4 registers, K straight from
//      global memory (8 bytes of a granule per lane); the scores (acc * scale) go to the scratch,
//      cells [row quad][position][4 rows], the row maxima (exact, any order) to LDS;
//   B  wave w takes 16 / W rows: e_p = expf(s_p - m_r), folded in position order by one lane per
//      row, and written over the scores with every 4 x 4 cell transposed;
//   C  wave w takes dims 32 w ..: prob_p = e_p * inv_r (one 16-byte load per lane and 16
//      positions, already the A operand's layout), V straight from global memory.
// Each row's arithmetic and order are k_attn_prefill's.  Positions p >= P_r contribute e = 0 to
// the sum (a non-negative sum from +0 is never -0, so +0 leaves it unchanged) and are not added
// to the outputs (selects where a row of the tile ends).  A row with P_r = 1 copies the V row
// (inference.rs:23564-23575).  Outputs as k_attn_prefill: f32 rows (optional) and Q8_0 per
// 32-value block.
// Bound by the adds and the f32 matrix issue, which share the f32 units and so do not overlap, and
// by the scratch (20 bytes per row and position) at 8K positions.  Measured (32 heads of 128 dims,
// 511-512 tokens): 72 us at positions 0.., 173 us at 512.., 746 us at 3584.., 1435 us at 7680..,
// where one workgroup per (head, token) takes 128, 319, 1625 and 4036 us and the same tiling with
// v_fma_mix products (64 rows per 1024-thread workgroup, operands in LDS) took 1281 us on average
// over the chunks of an 8191-token prompt (740 us now).
constexpr int APM_R = 16;   // rows per tile
constexpr int APM_PB = 64;  // the scratch's positions are padded to this
__host__ __device__ constexpr int apm_tiles(int rep, int T) { return (T * rep + APM_R - 1) / APM_R; }
__host__ __device__ constexpr size_t apm_pitch(size_t pmax) { return (pmax + APM_PB - 1) / APM_PB * APM_PB; }
__host__ __device__ constexpr bool apm_hd_ok(int hd) { return hd == 64 || hd == 128; }
// threads per workgroup
__host__ __device__ constexpr int apm_nt(int hd) { return hd * 2; }
// scratch floats for T tokens up to position pos_end - 1
__host__ __device__ constexpr size_t apm_scratch(int n_heads, int n_kv, int T, size_t pos_end) {
  return (size_t)n_kv * apm_tiles(n_heads / n_kv, T) * APM_R * apm_pitch(pos_end);
}

typedef float v16f_t __attribute__((ext_vector_type(16)));

// element 4 b + i of lane l: a[row 4 (l / 16) + i, held in block 2 (b / 2) + AB] * b[lane 16 b + l % 16]
template <int AB>
__device__ __forceinline__ v16f_t outer16x2(float a, float b) {
  const v16f_t z = {0.0f, 0.0f, 0.0f, 0.0f, 0.0f, 0.0f, 0.0f, 0.0f, 0.0f, 0.0f, 0.0f, 0.0f, 0.0f, 0.0f, 0.0f, 0.0f};
  return __builtin_amdgcn_mfma_f32_16x16x1f32(a, b, z, 1, AB, 0);
}

// The f32 of the f16 in either half of w.  The conversions are left to the compiler, which knows
// the wait states a matrix instruction needs after its operand is written; the shift is opaque
// to it so that the high half takes a shift and a plain conversion (7 clocks) and not one with a
// sub-word select (about 10).
__device__ __forceinline__ float half_lo(uint32_t w) { return half_bits_to_float((uint16_t)w); }
__device__ __forceinline__ float half_hi(uint32_t w) {
  uint32_t h;
  asm("v_lshrrev_b32 %0, 16, %1" : "=v"(h) : "v"(w));
  return half_bits_to_float((uint16_t)h);
}

// acc[j] (j = 4 * column block + row) += the 8 terms of a granule, in order: a[c] holds the rows'
// factors of terms c and 4 + c, f the columns' (two f16 pairs per lane: terms 0-3 in the lanes of
// blocks 0, 1, terms 4-7 in those of blocks 2, 3).  MASK: term e is added where e < left[j % 4].
template <int AB, bool MASK>
__device__ __forceinline__ void outer_terms(float (&acc)[8], const float* a, const uint2& f, const int* left) {
  const v16f_t t0 = outer16x2<AB>(a[0], half_lo(f.x)), t1 = outer16x2<AB>(a[1], half_hi(f.x));
  const v16f_t t2 = outer16x2<AB>(a[2], half_lo(f.y)), t3 = outer16x2<AB>(a[3], half_hi(f.y));
#pragma unroll
  for (int h = 0; h < 2; ++h) {
#pragma unroll
    for (int c = 0; c < 4; ++c) {
      const v16f_t& t = c == 0 ? t0 : c == 1 ? t1 : c == 2 ? t2 : t3;
#pragma unroll
      for (int j = 0; j < 8; ++j)
        acc[j] = !MASK || 4 * h + c < left[j & 3] ? acc[j] + t[8 * h + j] : acc[j];
    }
  }
}

template <int HD>
__global__ __launch_bounds__(HD * 2, 4) void k_attn_prefill_mm(
    const float* __restrict__ qrot, int n_heads, int n_kv, const uint16_t* __restrict__ kc,
    const uint16_t* __restrict__ vc, int layer, int kvs, int pos0, int T, float scale, float* __restrict__ scg,
    size_t pitch, float* __restrict__ att_out, int8_t* __restrict__ xq, float* __restrict__ xs) {
  static_assert(apm_hd_ok(HD), "tiled prefill attention: head_dim 64 or 128");
  constexpr int W = HD / 32;              // waves
  constexpr int RW = APM_R / W;           // rows per wave in phase B
  constexpr int LP = RW / 4;              // lanes per position there (4 rows each)
  constexpr int PS = 64 / LP;             // positions per step there
  constexpr int ES = PS + 4;              // row stride of its LDS block
  constexpr int NM = HD / 16;             // 16-dim stages of a score
  __shared__ __align__(16) float eb[W][RW * ES];
  __shared__ float smax[W][APM_R], sinv[APM_R];
  __shared__ __align__(16) float os[APM_R][HD + 4];
  __shared__ uint64_t etab[32];
  const int tid = threadIdx.x, wave = tid >> 6, lane = tid & 63;
  const int lr = lane & 15, lb = lane >> 4;
  const int rep = n_heads / n_kv, ntile = apm_tiles(rep, T);
  const int kvh = (int)blockIdx.x % n_kv, tile = ntile - 1 - (int)blockIdx.x / n_kv;  // longest first
  const int R0 = tile * APM_R, nr = min(APM_R, T * rep - R0);           // its rows
  const size_t hbase = kv_head_base(layer, n_kv, kvh, HD, kvs);
  const uint2* kg = reinterpret_cast<const uint2*>(kc + hbase);
  const uint2* vg = reinterpret_cast<const uint2*>(vc + hbase);
  float* sc = scg + ((size_t)kvh * ntile + tile) * APM_R * pitch;
  auto row_off = [&](int r) {  // element offset of row r in the [T][n_heads * HD] arrays
    const int R = R0 + min(r, nr - 1);  // (rows past the last repeat it and are not stored)
    return (size_t)(R / rep) * n_heads * HD + (size_t)(kvh * rep + R % rep) * HD;
  };
  auto row_p = [&](int r) { return pos0 + (R0 + min(r, nr - 1)) / rep + 1; };  // P_r
  const int pmax = row_p(nr - 1), pmin = row_p(0);
  int pr[4];  // P of rows 4 lb + i, whose values this lane holds in a product
#pragma unroll
  for (int i = 0; i < 4; ++i) pr[i] = row_p(4 * lb + i);
  if (tid < 32) etab[tid] = kExp2Tab[tid];

  // ---- A: scores and row maxima
  {
    // q of row lr: register 4 m + c holds, in block b, dim 16 m + 8 (b % 2) + 4 (b / 2) + c
    float q[4 * NM];
    const float* qp = qrot + row_off(lr) + 8 * (lb & 1) + 4 * (lb >> 1);
#pragma unroll
    for (int m = 0; m < NM; ++m) {
      const float4 v = *reinterpret_cast<const float4*>(qp + 16 * m);
      q[4 * m] = v.x;
      q[4 * m + 1] = v.y;
      q[4 * m + 2] = v.z;
      q[4 * m + 3] = v.w;
    }
    float rm[4] = {-INFINITY, -INFINITY, -INFINITY, -INFINITY};
    const int nblk = (pmax + 31) / 32;
    // this lane's halves of the K granules of a 16-dim stage, loaded KD stages ahead of their use
    constexpr int KD = 1;
    static_assert(NM % (KD + 1) == 0, "K ring");
    uint2 kr[KD + 1][2];
    auto kload = [&](uint2 (&r)[2], int b, int m) __attribute__((always_inline)) {
      const int p = min(b * 32 + 16 * (lb & 1) + lr, pmax - 1);
      const uint2* a = kg + ((size_t)(2 * m) * kvs + p) * 2 + (lb >> 1);
      r[0] = a[0];
      r[1] = a[2 * (size_t)kvs];
    };
#pragma unroll
    for (int m = 0; m < KD; ++m) kload(kr[m], min(wave, nblk - 1), m);
    for (int b = wave; b < nblk; b += W) {
      const int bn = min(b + W, nblk - 1);  // (the last block loads itself again)
      float acc[8];
#pragma unroll
      for (int j = 0; j < 8; ++j) acc[j] = 0.0f;
#pragma unroll
      for (int m = 0; m < NM; ++m) {
        kload(kr[(m + KD) % (KD + 1)], m + KD < NM ? b : bn, (m + KD) % NM);
        outer_terms<0, false>(acc, q + 4 * m, kr[m % (KD + 1)][0], nullptr);
        outer_terms<1, false>(acc, q + 4 * m, kr[m % (KD + 1)][1], nullptr);
      }
#pragma unroll
      for (int u = 0; u < 2; ++u) {
        const int p = b * 32 + 16 * u + lr;
        float s[4];
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          s[i] = acc[4 * u + i] * scale;
          if (p < pr[i]) rm[i] = fmaxf(rm[i], s[i]);
        }
        *reinterpret_cast<float4*>(sc + ((size_t)lb * pitch + p) * 4) = make_float4(s[0], s[1], s[2], s[3]);
      }
    }
    // over the 16 lanes of a block
#pragma unroll
    for (int i = 0; i < 4; ++i) {
#pragma unroll
      for (int o = 8; o >= 1; o >>= 1) rm[i] = fmaxf(rm[i], __shfl_xor(rm[i], o));
      if (lr == 0) smax[wave][4 * lb + i] = rm[i];
    }
  }
  __syncthreads();

  // ---- B: exponentials, each row's sum in position order
  {
    const int rq = RW / 4 * wave + lane % LP;  // this lane's row quad
    float m[4];
    int prb[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      m[i] = smax[0][4 * rq + i];
#pragma unroll
      for (int w = 1; w < W; ++w) m[i] = fmaxf(m[i], smax[w][4 * rq + i]);
      prb[i] = row_p(4 * rq + i);
    }
    float* ew = eb[wave];
    float sum = 0.0f;
    const int pl = lane / LP;
    const float* sp = sc + ((size_t)rq * pitch + pl) * 4;
    // the transposed cells: lane = (cell of 4 positions, row) of the wave's rows
    const int tr = lane % RW, tc = lane / RW;
    float* tp = sc + ((size_t)(RW / 4 * wave + tr / 4) * pitch + 4 * tc) * 4 + 4 * (tr & 3);
    float4 nx = *reinterpret_cast<const float4*>(sp);
    for (int p0 = 0; p0 < pmax; p0 += PS) {
      const float4 s4 = nx;
      if (p0 + PS < pmax) nx = *reinterpret_cast<const float4*>(sp + (size_t)(p0 + PS) * 4);
      const float s[4] = {s4.x, s4.y, s4.z, s4.w};
      float e[4];
#pragma unroll
      for (int i = 0; i < 4; ++i) e[i] = glibc_expf_nonpos_t(s[i] - m[i], etab);
#pragma unroll
      for (int i = 0; i < 4; ++i)
        ew[(4 * (lane % LP) + i) * ES + pl] = p0 + pl < prb[i] ? e[i] : 0.0f;
      // the LDS block is this wave's own: wave-level ordering only
      __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
      __builtin_amdgcn_wave_barrier();
      __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
      const float* er = ew + tr * ES;
#pragma unroll
      for (int k = 0; k < PS * RW / 256; ++k)  // (one cell per lane when RW = 4)
        *reinterpret_cast<float4*>(tp + (size_t)(p0 + k * (256 / RW)) * 4) =
            *reinterpret_cast<const float4*>(er + 4 * tc + k * (256 / RW));
#pragma unroll
      for (int k = 0; k < PS / 4; ++k) add4(sum, reinterpret_cast<const float4*>(er)[k]);
      __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
      __builtin_amdgcn_wave_barrier();
      __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
    }
    if (lane < RW) sinv[RW * wave + lane] = 1.0f / sum;
  }
  __syncthreads();

  // ---- C: output sums of dims 32 wave ..
  {
    const float inv = sinv[lr];
    const int n16 = (pmax + 15) >> 4;  // steps of 16 positions
    const int nfree = pmin >> 4;       // of them before any row's end
    const int glast = (pmax - 1) >> 3;
    const uint2* vp = vg + (32 * wave + 16 * (lb & 1) + lr) * 2 + (lb >> 1);
    // exponentials of row lr: register c holds, in block b, position 16 s + 8 (b % 2) + 4 (b / 2) + c
    const float* ep = sc + ((size_t)(lr >> 2) * pitch + 8 * (lb & 1) + 4 * (lb >> 1)) * 4 + 4 * (lr & 3);
    float acc[8];
#pragma unroll
    for (int j = 0; j < 8; ++j) acc[j] = 0.0f;
    constexpr int D = 3;  // steps in flight
    uint2 vr[D][2];
    float4 er[D];
    auto load = [&](int k, int s) __attribute__((always_inline)) {
      const int sl = min(s, n16 - 1);
      vr[k][0] = vp[(size_t)(2 * sl) * HD * 2];
      vr[k][1] = vp[(size_t)min(2 * sl + 1, glast) * HD * 2];
      er[k] = *reinterpret_cast<const float4*>(ep + (size_t)sl * 64);
    };
    auto step = [&](int k, int s, auto mc) __attribute__((always_inline)) {
      constexpr bool masked = decltype(mc)::value;
      const float a[4] = {er[k].x * inv, er[k].y * inv, er[k].z * inv, er[k].w * inv};
      int left[4], left8[4];
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        left[i] = pr[i] - 16 * s;
        left8[i] = left[i] - 8;
      }
      outer_terms<0, masked>(acc, a, vr[k][0], left);
      outer_terms<1, masked>(acc, a, vr[k][1], left8);
    };
#pragma unroll
    for (int k = 0; k < D; ++k) load(k, k);
    int s = 0;
    for (; s + D <= nfree; s += D) {
#pragma unroll
      for (int k = 0; k < D; ++k) {
        step(k, s + k, std::false_type{});
        load(k, s + k + D);
      }
    }
#pragma unroll 1
    for (; s < n16; ++s) {  // the last steps: rows ending inside, or fewer than D left
      step(0, s, std::true_type{});
#pragma unroll
      for (int k = 0; k + 1 < D; ++k) {
        vr[k][0] = vr[k + 1][0];
        vr[k][1] = vr[k + 1][1];
        er[k] = er[k + 1];
      }
      load(D - 1, s + D);
    }
#pragma unroll
    for (int u = 0; u < 2; ++u)
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const int d = 32 * wave + 16 * u + lr;
        // a single position copies the V row (its bits, -0 included)
        os[4 * lb + i][d] = pr[i] == 1 ? half_bits_to_float(vc[hbase + kv_v_index(HD, 0, d)]) : acc[4 * u + i];
      }
  }
  __syncthreads();
  // ---- outputs: one (row, 32-value block) per thread
  if (tid < APM_R * (HD / 32)) {
    const int r = tid / (HD / 32), blk = tid % (HD / 32);
    if (r >= nr) return;
    float y[32];
#pragma unroll
    for (int e = 0; e < 32; ++e) y[e] = os[r][32 * blk + e];
    const size_t o0 = row_off(r) + 32 * blk;
    if (att_out) {
#pragma unroll
      for (int e = 0; e < 32; e += 4)
        *reinterpret_cast<float4*>(att_out + o0 + e) = make_float4(y[e], y[e + 1], y[e + 2], y[e + 3]);
    }
    uint32_t packed[8];
    xs[o0 >> 5] = quantize_block_regs(y, packed);
    uint4* qp = reinterpret_cast<uint4*>(xq + o0);
    qp[0] = make_uint4(packed[0], packed[1], packed[2], packed[3]);
    qp[1] = make_uint4(packed[4], packed[5], packed[6], packed[7]);
  }
}

// ---------------------------------------------------------------------------
// SwiGLU + Q8_0 quantization of T rows (silu_mul_quantize, cuda_resident.rs:1315; CPU
// tensor/mod.rs:1943-1967).  Row t of gu holds 2F values: [gate | up], or, interleaved,
// groups of 32 gate values followed by the matching 32 up values.  grid (ceil(F/256), T).
__global__ __launch_bounds__(256) void k_silu_rows(const float* __restrict__ gu, int F, int interleaved,
                                                   int8_t* __restrict__ xq, float* __restrict__ xs) {
  const int i = blockIdx.x * 256 + threadIdx.x;
  if (i >= F) return;  // uniform per 32-lane group (F % 32 == 0)
  const size_t t = blockIdx.y;
  const float* r = gu + t * 2 * (size_t)F;
  const int gi = interleaved ? (i >> 5) * 64 + (i & 31) : i;
  const int ui = interleaved ? gi + 32 : F + i;
  const float a = silu_mul1(r[gi], r[ui]);
  int8_t q;
  const float d = quantize_lane32(a, &q);
  xq[t * F + i] = q;
  if ((i & 31) == 0) xs[(t * F + i) >> 5] = d;
}

}  // namespace cm
