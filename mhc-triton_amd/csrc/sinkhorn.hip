// Standalone Sinkhorn-Knopp forward / backward over N independent 4x4
// matrices (reference src/mhc/_kernels.py:30-130,597-614 and
// src/mhc/_backward.py:29-262,503-530).
//
// One matrix per lane: a wave handles 64 matrices, a 256-thread workgroup
// 256.  The forward is VALU-bound at 20 rounds (40 VALU ops and 8 v_rcp per
// round in the scaling-vector form of sk_forward, 32 + 8 from the eighth round
// on with a small eps: 2^20 bf16 matrices 38.5 -> 33.3 us, fp16 39.6 -> 34.4;
// fp32, whose reads and writes also go through LDS, 40.6 -> 38.8, and fwd + bwd
// 118.8 -> 113.4, at 32 rounds 227 -> 210); the backward keeps every round's
// scaling vectors in registers for up to 20 rounds and carries the adjoint in
// scaled coordinates (sk_backward_scaled: 95-100 us at 2^20 matrices, 20
// rounds, when chosen, against 131 us for the explicit normalisation backward on the same
// states and 175 us for the checkpointed reverse sweep).  From 21 to 64
// rounds it recomputes the vectors in 16-round segments from checkpoints
// (sk_backward_segmented; fwd + bwd at 2^20 matrices: 190 against 255 us at
// 21 rounds, 436 against 818 us at 64); past 64 rounds it keeps the
// checkpointed sweep.  The unaligned (element-wise load) path runs the same
// forms (fwd + bwd at 20 rounds: 130-134 against 241-245 us with the
// checkpointed sweep it used before).
#include "sinkhorn.hpp"

namespace mhc {

// A wave's 64 fp32 matrices are one contiguous span of 4 KiB.  The forward reads and writes it 1 KiB
// per access, 16 bytes a lane, and it changes hands in the wave's own LDS tile, where lane l picks up
// the chunks of matrix l.  A lane loading its own 64 bytes touches 32 lines per access: 2^20 matrices
// at 7 rounds took 34.8 us against 26.9 so.  Of 16 bits (32 bytes a lane)
// lanes load their own: 21.4 against 22.5 us at 7 rounds, 33.3 against 33.6 at 20 in bf16, 22.2 against
// 23.8 and 34.4 against 36.3 in fp16.  Chunk c sits in slot c with its low three bits turned by c / 8,
// so that eight lanes in a row hit different banks both ways.
template <typename T>
struct WaveTile {
  static constexpr int N = Vec<T>::N;   // elements per chunk
  static constexpr int Q = 16 / N;      // chunks per matrix
  u32x4* tile;                          // 64 * Q chunks
  int lane;

  __device__ __forceinline__ static int slot(int c) { return (c & ~7) | ((c + (c >> 3)) & 7); }

  // Lanes read what other lanes of the wave wrote: keep the order.
  __device__ __forceinline__ static void order() {
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
  }

  // base: the wave's first matrix; chunks: how many 16-byte chunks of it lie inside the tensor
  __device__ __forceinline__ void fetch(const T* base, int64_t chunks, u32x4 (&r)[Q]) const {
#pragma unroll
    for (int q = 0; q < Q; ++q) {
      const int c = 64 * q + lane;
      r[q] = c < chunks ? reinterpret_cast<const u32x4*>(base)[c] : u32x4{0u, 0u, 0u, 0u};
    }
  }

  __device__ __forceinline__ void to_matrix(const u32x4 (&r)[Q], float (&m)[16]) const {
    order();
#pragma unroll
    for (int q = 0; q < Q; ++q) tile[slot(64 * q + lane)] = r[q];
    order();
#pragma unroll
    for (int q = 0; q < Q; ++q)
      RawVec<T>::unpack(__builtin_bit_cast(typename RawVec<T>::type, tile[slot(Q * lane + q)]), m + q * N);
  }

  __device__ __forceinline__ void store(T* base, int64_t chunks, const float (&m)[16]) const {
    order();
#pragma unroll
    for (int q = 0; q < Q; ++q) tile[slot(Q * lane + q)] = RawVec<T>::pack(m + q * N);
    order();
#pragma unroll
    for (int q = 0; q < Q; ++q) {
      const int c = 64 * q + lane;
      if (c < chunks) reinterpret_cast<u32x4*>(base)[c] = tile[slot(c)];
    }
  }
};

// A lane's own matrix in 16-byte vectors, or element by element for tensors that do not start on a
// 16-byte boundary.
template <typename T, bool VEC>
__device__ __forceinline__ void load_mat(const T* p, float (&m)[16]) {
  if constexpr (VEC) {
    constexpr int N = Vec<T>::N;
#pragma unroll
    for (int q = 0; q < 16 / N; ++q) Io<T>::load(p + q * N, m + q * N);
  } else {
#pragma unroll
    for (int k = 0; k < 16; ++k) m[k] = to_f32(p[k]);
  }
}

template <typename T, bool VEC>
__device__ __forceinline__ void store_mat(T* p, const float (&m)[16]) {
  if constexpr (VEC) {
    constexpr int N = Vec<T>::N;
#pragma unroll
    for (int q = 0; q < 16 / N; ++q) Io<T>::template store<false>(p + q * N, m + q * N);
  } else {
#pragma unroll
    for (int k = 0; k < 16; ++k) p[k] = from_f32<T>(m[k]);
  }
}

constexpr int kSkWaves = kThreads / 64;

template <typename T, bool VEC, bool SMALL>
__global__ __launch_bounds__(kThreads) void sinkhorn_fwd_kernel(const T* __restrict__ M, T* __restrict__ out,
                                                                int64_t n, int iters, float eps) {
  float m[16];
  if constexpr (VEC && sizeof(T) == 4) {
    using Tile = WaveTile<T>;
    __shared__ __attribute__((aligned(16))) u32x4 tiles[kSkWaves][64 * Tile::Q];
    const int64_t i0 = (int64_t)blockIdx.x * kThreads + (threadIdx.x & ~63);  // the wave's first matrix
    if (i0 >= n) return;                                                      // the whole wave
    const Tile t{tiles[threadIdx.x >> 6], (int)(threadIdx.x & 63)};
    const int64_t chunks = (n - i0) * Tile::Q;
    u32x4 r[Tile::Q];
    t.fetch(M + i0 * 16, chunks, r);
    t.to_matrix(r, m);
    sk_forward<SMALL>(m, iters, eps);
    t.store(out + i0 * 16, chunks, m);
  } else {
    const int64_t i = (int64_t)blockIdx.x * kThreads + threadIdx.x;
    if (i >= n) return;
    load_mat<T, VEC>(M + i * 16, m);
    sk_forward<SMALL>(m, iters, eps);
    store_mat<T, VEC>(out + i * 16, m);
  }
}

constexpr int kSkScaledMax = 20;  // rounds the scaling-vector backward keeps in registers
constexpr int kSkSegRounds = 16;  // rounds per segment of the segmented backward
constexpr int kSkSegs = 4;        // its segments: up to 64 rounds

// Lanes load their own matrices: the backward is bound by its VALU work, and through WaveTile it
// needs 261 registers (one wave per SIMD, 136 us over 2^20 fp32 matrices) or, held to 256, 36 moves
// to accumulator registers (87.5 us against 86.6; at 7 rounds 58.2 against 51.8).
template <typename T, typename TD, bool VEC, bool SMALL>
__global__ __launch_bounds__(kThreads) void sinkhorn_bwd_kernel(const T* __restrict__ M, const TD* __restrict__ dP,
                                                                T* __restrict__ dM, int64_t n, int iters, float eps) {
  const int64_t i = (int64_t)blockIdx.x * kThreads + threadIdx.x;
  if (i >= n) return;
  float m[16], d[16];
  load_mat<T, VEC>(M + i * 16, m);
  load_mat<TD, VEC>(dP + i * 16, d);
  // Past 64 rounds the explicit-state checkpoints: on the unaligned path five
  // keep 3 waves per SIMD (its element-wise loads need more registers; ten
  // would leave one).  The result does not depend on the checkpoint count.
  if (iters <= kSkScaledMax)
    sk_backward_scaled<kSkScaledMax, SMALL>(m, d, iters, eps);
  else if (iters <= kSkSegRounds * kSkSegs)
    sk_backward_segmented<kSkSegRounds, kSkSegs, SMALL>(m, d, iters, eps);
  else
    sk_backward<VEC ? 10 : 5>(m, d, iters, eps);
  store_mat<T, VEC>(dM + i * 16, d);
}

static int check_common(int64_t n_mat, int iters) {
  if (n_mat < 0) { set_error("sinkhorn: negative matrix count %lld", (long long)n_mat); return MHC_ERR_ARG; }
  if (iters < 0) { set_error("sinkhorn: negative iteration count %d", iters); return MHC_ERR_ARG; }
  return MHC_OK;
}

}  // namespace mhc

using namespace mhc;

extern "C" int mhc_sinkhorn_forward(const void* M, void* out, int64_t n_mat, int dtype, int iters, float eps,
                                    mhc_stream_t stream) {
  if (int rc = check_common(n_mat, iters)) return rc;
  if (n_mat == 0) return MHC_OK;
  if (!M || !out) { set_error("sinkhorn_forward: null pointer"); return MHC_ERR_ARG; }
  const bool vec = aligned16(M) && aligned16(out);
  const dim3 grid((unsigned)((n_mat + kThreads - 1) / kThreads));
  return MHC_DISPATCH_DTYPE(dtype, [&] {
    auto* k = vec ? (sk_small_eps(eps) ? sinkhorn_fwd_kernel<T, true, true> : sinkhorn_fwd_kernel<T, true, false>)
                  : (sk_small_eps(eps) ? sinkhorn_fwd_kernel<T, false, true> : sinkhorn_fwd_kernel<T, false, false>);
    k<<<grid, kThreads, 0, (hipStream_t)stream>>>((const T*)M, (T*)out, n_mat, iters, eps);
    return hip_status(hipGetLastError(), "sinkhorn_forward launch");
  });
}

extern "C" int mhc_sinkhorn_backward(const void* M, int dtype_M, const void* dP, int dtype_dP, void* dM,
                                     int64_t n_mat, int iters, float eps, mhc_stream_t stream) {
  if (int rc = check_common(n_mat, iters)) return rc;
  if (n_mat == 0) return MHC_OK;
  if (!M || !dP || !dM) { set_error("sinkhorn_backward: null pointer"); return MHC_ERR_ARG; }
  const bool vec = aligned16(M) && aligned16(dP) && aligned16(dM);
  const dim3 grid((unsigned)((n_mat + kThreads - 1) / kThreads));
  return MHC_DISPATCH_DTYPE(dtype_M, [&] {
    using TM = T;
    return MHC_DISPATCH_DTYPE(dtype_dP, [&] {
      auto* k = vec ? (sk_small_eps(eps) ? sinkhorn_bwd_kernel<TM, T, true, true>
                                         : sinkhorn_bwd_kernel<TM, T, true, false>)
                    : (sk_small_eps(eps) ? sinkhorn_bwd_kernel<TM, T, false, true>
                                          : sinkhorn_bwd_kernel<TM, T, false, false>);
      k<<<grid, kThreads, 0, (hipStream_t)stream>>>((const TM*)M, (const T*)dP, (TM*)dM, n_mat, iters, eps);
      return hip_status(hipGetLastError(), "sinkhorn_backward launch");
    });
  });
}
