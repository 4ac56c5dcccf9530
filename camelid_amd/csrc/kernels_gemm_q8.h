// kernels_gemm_q8.h -- the Q8_0 prefill GEMM (gfx950, wave64).
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>
#include <type_traits>

namespace cm {

// ---------------------------------------------------------------------------
// Q8_0 GEMM (q8_gemm_batched, cuda_resident.rs:1494; CPU: the row dot of
// inference.rs:19871-19905 per token):
//   y[t][n] = (resid ? resid[t][n] : 0) + fold_b (float(dot_b(W[n], X[t])) * wd[n][b]) * xs[t][b]
// with dot_b the exact int32 dot of one 32-value block and the fold in block order from 0.
// The block dots run on the matrix cores: one v_mfma_i32_{32x32x32,16x16x32}_i8 per M x M tile
// of (tokens x rows) and block; its K = 32 is exactly one Q8_0 block, so every block's int32 dot
// comes out separately (any assignment of the 32 byte positions to lanes gives the same integer,
// as long as both operands use the same one).
// The activations are the A operand and the weights the B operand: a lane's outputs are M * M / 64
// tokens of ONE weight row, so the weight scale is one register per tile and block and the
// activation scales are read from LDS 16 bytes at a time (broadcasts).
// Per output and block 3 VALU operations.  The accumulator starts from the bit pattern of
// 1.5 * 2^23: |dot| <= 32 * 128^2 = 2^19 < 2^22, so the int32 sum's bits are those of the f32
// value 1.5 * 2^23 + dot (ulp 1 in [2^23, 2^24)), and fma(f, w, -(1.5 * 2^23) w) = round(f w -
// 1.5 * 2^23 w) = round(dot w) exactly (the FMA rounds once, -(1.5 * 2^23) w is exact for every
// finite f16 w: 13 significant bits, no overflow); then * xs, then +.  The scale is widened to f32
// when it is staged: v_fma_f32 on f32 registers, v_mul_f32 and v_add_f32 alone fold 1024 outputs
// in 108 clocks of a SIMD (45 ns, and 51 ns with the whole device at it; two or four waves), the plain
// form with its conversion in 141.  An infinite w is the one value the FMA form does not give
// (dot * w = +-inf, or NaN at dot = 0): a workgroup that has staged one runs its remaining steps in
// the plain form (conversion, product), which is the same for every other value.
// Workgroup: 2 (rows) x 2 (tokens) waves of M x M each.  Operands move in steps of SB blocks: 16-byte
// global loads into registers one step ahead, at the next step's start into the other half of a
// double-buffered LDS tile [16-byte chunk][row] (planes padded so that the chunks of a row's load
// land in different banks), scales beside them as (w, -(1.5 * 2^23) w) pairs; one barrier per step.
// Tiles are dealt so that each XCD (workgroup id mod 8) runs a contiguous range of tiles, token
// tiles innermost: a row tile's weights are read once per XCD and re-read from its L2.
// Two forms.  M = 32, SB = 4 (64 x 64 tiles, four workgroups per CU) where there are tiles for the
// device; [128256 x 3072] x 512 takes 135 ns per 1024 outputs, block and SIMD, 2.7 times the bare
// fold: the matrix instruction, the LDS reads of the operands and scales and the fold share the
// issue slots, and the clock falls to 1.8-2.1 GHz under them, so it is bound by power as much as
// by issue.  M = 16,
// SB = 8, PIPE (32 x 32 tiles, 4 outputs per lane, each block's operands read and products issued
// during the previous block's fold) for short prompts and narrow matrices, where a wave has its
// SIMD to itself and its own latency per block sets the time.  Measured (us, the previous
// 64- and 32-row tiles of v_fma_mix folds at their best / now): [16384 x 3072] x 511 122 / 111,
// [3072 x 8192] x 511 76 / 74, [4096 x 14336] x 512 166 / 138, [32000 x 2048] x 512 157 / 145,
// [128256 x 3072] x 512 989 / 980, [3072 x 8192] x 100 50.5 / 34, [2048 x 2048] x 37 14.0 / 8.4,
// [2048 x 5632] x 37 34.7 / 19.
// K % 32 == 0; y may alias resid.
constexpr int32_t GM_MAGIC = 0x4B400000;
constexpr float GM_MAGIC_F = 12582912.0f;

typedef int gm_i4 __attribute__((ext_vector_type(4)));
typedef int gm_i16 __attribute__((ext_vector_type(16)));

template <int M>
struct gm_tile;
template <>
struct gm_tile<32> {
  typedef gm_i16 acc_t;
  typedef gm_i4 op_t;
  static __device__ __forceinline__ acc_t mfma(op_t a, op_t b, acc_t c) {
    return __builtin_amdgcn_mfma_i32_32x32x32_i8(a, b, c, 0, 0, 0);
  }
};
template <>
struct gm_tile<16> {
  typedef gm_i4 acc_t;
  typedef long op_t;
  static __device__ __forceinline__ acc_t mfma(op_t a, op_t b, acc_t c) {
    return __builtin_amdgcn_mfma_i32_16x16x32_i8(a, b, c, 0, 0, 0);
  }
};

constexpr int GM_NT = 256;  // threads
template <int M, int SB>
struct gm_cfg {
  static constexpr int TR = 2 * M;                                 // rows, and tokens, of a tile
  static constexpr int CH = 2 * SB;                                // 16-byte chunks of a row per step
  static constexpr int PL = TR + (SB == 4 ? 1 : SB == 8 ? 1 : 2);  // rows per chunk plane (padded)
  static constexpr int OJ = TR * CH / GM_NT;                       // operand loads per thread and step
  static constexpr int RPJ = GM_NT / CH, SPJ = GM_NT / SB;         // rows per load round, scales likewise
  static_assert(TR * CH % GM_NT == 0 && TR * SB == GM_NT, "one scale of each kind per thread and step");
};
__host__ __device__ inline int gm_tiles(int N, int T, int M) {
  return ((N + 2 * M - 1) / (2 * M)) * ((T + 2 * M - 1) / (2 * M));
}
__host__ __device__ inline int gm_grid(int N, int T, int M) { return (gm_tiles(N, T, M) + 7) / 8 * 8; }

template <int M, int SB, bool PIPE>
__global__ __launch_bounds__(GM_NT, 4) void k_gemm_q8(const int8_t* __restrict__ wq, const uint16_t* __restrict__ wd,
                                                      int N, int K, const int8_t* __restrict__ xq,
                                                      const float* __restrict__ xs, int T, float* y,
                                                      const float* resid) {
  typedef gm_cfg<M, SB> C;
  typedef gm_tile<M> MT;
  constexpr int R = M * M / 64;  // outputs per lane
  constexpr int NH = 64 / M;     // lane groups (of different operand bytes and output tokens)
  __shared__ __align__(16) gm_i4 sa[2][C::CH][C::PL];
  __shared__ __align__(16) gm_i4 sb[2][C::CH][C::PL];
  __shared__ __align__(16) float sx[2][SB][C::TR];
  __shared__ __align__(16) float2 sw[2][SB][C::TR];
  // bit b: a weight scale staged into buffer b was infinite.  A step tests its own buffer's bit while
  // the other one's may be set, so all waves of the workgroup leave the first loop at the same step.
  __shared__ uint32_t sinf;
  const int NB = K >> 5, nsteps = (NB + SB - 1) / SB;
  const int ntt = (T + C::TR - 1) / C::TR, tiles = gm_tiles(N, T, M), per = (tiles + 7) >> 3;
  const int L = (int)(blockIdx.x & 7) * per + (int)(blockIdx.x >> 3);
  if (L >= tiles) return;
  const int n_base = (L / ntt) * C::TR, t_base = (L % ntt) * C::TR;
  const int tid = threadIdx.x, wave = tid >> 6, lane = tid & 63;
  const int lr = lane % M, lh = lane / M;
  const int wn = (wave & 1) * M, wt = (wave >> 1) * M;

  // global -> register loads of one step: 16-byte chunk cc of rows crow + RPJ j of either operand,
  // and block sblk's scale of row srow
  const int crow = tid / C::CH, cc = tid % C::CH, srow = tid / SB, sblk = tid % SB;
  const int8_t* wbase = wq + (size_t)n_base * K;
  const int8_t* xbase = xq + (size_t)t_base * K;
  const int nlast = N - 1 - n_base, tlast = T - 1 - t_base;
  const uint16_t* wdrow = wd + (size_t)(n_base + min(srow, nlast)) * NB;
  const float* xsrow = xs + (size_t)(t_base + min(srow, tlast)) * NB;
  uint32_t oa[C::OJ], ob[C::OJ];
#pragma unroll
  for (int j = 0; j < C::OJ; ++j) {
    oa[j] = (uint32_t)min(crow + C::RPJ * j, tlast) * (uint32_t)K;
    ob[j] = (uint32_t)min(crow + C::RPJ * j, nlast) * (uint32_t)K;
  }
  gm_i4 ra[C::OJ], rb[C::OJ];
  float rx;
  uint32_t rw;
  auto gload = [&](int s) __attribute__((always_inline)) {
    const uint32_t co = (uint32_t)min((s * C::CH + cc) * 16, K - 16);
    const int so = min(s * SB + sblk, NB - 1);
#pragma unroll
    for (int j = 0; j < C::OJ; ++j) ra[j] = *reinterpret_cast<const gm_i4*>(xbase + (oa[j] + co));
#pragma unroll
    for (int j = 0; j < C::OJ; ++j) rb[j] = *reinterpret_cast<const gm_i4*>(wbase + (ob[j] + co));
    rx = xsrow[so];
    rw = wdrow[so];
  };
  auto put = [&](int buf) __attribute__((always_inline)) {
#pragma unroll
    for (int j = 0; j < C::OJ; ++j) {
      sa[buf][cc][crow + C::RPJ * j] = ra[j];
      sb[buf][cc][crow + C::RPJ * j] = rb[j];
    }
    sx[buf][sblk][srow] = rx;
    _Float16 h;
    __builtin_memcpy(&h, &rw, 2);
    const float w = (float)h;
    sw[buf][sblk][srow] = make_float2(w, -GM_MAGIC_F * w);
    if ((rw & 0x7fffu) == 0x7c00u) atomicOr(&sinf, 1u << buf);
  };

  float acc[R];
#pragma unroll
  for (int i = 0; i < R; ++i) acc[i] = 0.0f;
  typename MT::acc_t c0;
#pragma unroll
  for (int i = 0; i < R; ++i) c0[i] = GM_MAGIC;

  // what a block's products and fold read from LDS
  struct operands {
    typename MT::op_t a, b;
    float x[R];
    float2 w;
  };
  auto fetch = [&](operands& o, int buf, int b) __attribute__((always_inline)) {
    if constexpr (M == 32) {
      o.a = sa[buf][2 * b + lh][wt + lr];
      o.b = sb[buf][2 * b + lh][wn + lr];
    } else {
      o.a = reinterpret_cast<const long*>(&sa[buf][2 * b + (lh >> 1)][wt + lr])[lh & 1];
      o.b = reinterpret_cast<const long*>(&sb[buf][2 * b + (lh >> 1)][wn + lr])[lh & 1];
    }
    o.w = sw[buf][b][wn + lr];
#pragma unroll
    for (int q = 0; q < R / 4; ++q) {
      const float4 v = *reinterpret_cast<const float4*>(&sx[buf][b][wt + 4 * NH * q + 4 * lh]);
      o.x[4 * q] = v.x;
      o.x[4 * q + 1] = v.y;
      o.x[4 * q + 2] = v.z;
      o.x[4 * q + 3] = v.w;
    }
  };
  auto fold = [&](const typename MT::acc_t& d, const operands& o, auto plainc) __attribute__((always_inline)) {
    constexpr bool plain = decltype(plainc)::value;
#pragma unroll
    for (int i = 0; i < R; ++i) {
      const float t = plain ? (float)(d[i] - GM_MAGIC) * o.w.x : __builtin_fmaf(__int_as_float(d[i]), o.w.x, o.w.y);
      acc[i] += t * o.x[i];
    }
    // (the fold stays ahead of what follows in the source)
#pragma unroll
    for (int i = 0; i < R; ++i) asm volatile("" : "+v"(acc[i]));
  };

  // Step s computes from buffer s % 2.  At its start the operands of step s + 1 (loaded during step
  // s - 1) go to the other buffer and the loads of step s + 2 are issued.
  if (tid == 0) sinf = 0;
  gload(0);
  __syncthreads();
  put(0);
  gload(min(1, nsteps - 1));
  __syncthreads();
  auto infinite = [&]() __attribute__((always_inline)) {
    return (uint32_t)__builtin_amdgcn_readfirstlane(
        (int)__hip_atomic_load(&sinf, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP));
  };
  int s = 0;
  const int nfull = NB / SB;
#pragma unroll 1
  for (; s < nfull && !(infinite() >> (s & 1) & 1); ++s) {
    const int buf = s & 1;
    put(buf ^ 1);
    gload(min(s + 2, nsteps - 1));
    if constexpr (PIPE) {
      operands o[2];
      typename MT::acc_t d[2];
      fetch(o[0], buf, 0);
      d[0] = MT::mfma(o[0].a, o[0].b, c0);
#pragma unroll
      for (int b = 0; b < SB; ++b) {
        if (b + 1 < SB) {
          fetch(o[(b + 1) & 1], buf, b + 1);
          d[(b + 1) & 1] = MT::mfma(o[(b + 1) & 1].a, o[(b + 1) & 1].b, c0);
        }
        fold(d[b & 1], o[b & 1], std::false_type{});
      }
    } else {
#pragma unroll
      for (int b = 0; b < SB; ++b) {
        operands o;
        fetch(o, buf, b);
        fold(MT::mfma(o.a, o.b, c0), o, std::false_type{});
      }
    }
    __syncthreads();
  }
  // the partial last step; every step from an infinite scale on
#pragma unroll 1
  for (; s < nsteps; ++s) {
    const int buf = s & 1;
    put(buf ^ 1);
    gload(min(s + 2, nsteps - 1));
#pragma unroll 1
    for (int b = 0; b < min(SB, NB - s * SB); ++b) {
      operands o;
      fetch(o, buf, b);
      fold(MT::mfma(o.a, o.b, c0), o, std::true_type{});
    }
    __syncthreads();
  }
  const int n = n_base + wn + lr;
  if (n < N) {
#pragma unroll
    for (int i = 0; i < R; ++i) {
      const int t = t_base + wt + 4 * NH * (i / 4) + 4 * lh + i % 4;
      if (t < T) {
        const size_t o = (size_t)t * N + n;
        y[o] = resid ? resid[o] + acc[i] : acc[i];
      }
    }
  }
}

}  // namespace cm
