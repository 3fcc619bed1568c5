// Streaming KV window cache (ring) and window-layout kernels for gfx950 (MI355X).
//
// Reference semantics: the window K/V cache of `blockForward` (DiT.swift:507-511 concat, :532-538 trim) and
// `windowPartition` / `windowReverse` (DiT.swift:113-126).
//
// Design: the reference rebuilds the whole window each chunk (concat = read cache + new, write all). Here each
// layer owns `capacity` slots of one temporal slice (s blocks x 128 tokens x C) in window order; an append writes
// only the new slices into the next free slots (pool_mean_kernel then pools the new key blocks, so selection never
// re-reads cached keys); evict moves the ring head. Attention and selection address key block j through
// slot = (head + j / s) % capacity. All kernels are pure HBM streams.
#include "common.hpp"

namespace fvsr {

// Copies 128-token blocks between layouts (16 bytes per vector): src to dst and, for gridDim.z 2, src2 to dst2 in the
// same way. Block b of the source maps to block (dst_slot0 + b / slice_blocks) % capacity of slices (identity when
// capacity == 1 and slice_blocks >= the block count); tokens inside a block may be gathered from grid order (src_grid) or
// scattered to grid order (dst_grid).
// Memory-bound, and at streaming sizes short of loads in flight: a wave moves kCopyTokens tokens with every load of up to
// 64 x kCopyVecs vectors a token issued before the first store, and a block is spread over 16 workgroups, so that a
// one-slice append of 16 blocks covers the chip. 6144 fp32 tokens of 1536 channels (75 MB moved): 53 -> 29 us against
// one run of 32 tokens a thread, 8 in flight.
constexpr int kCopyTokens = 2, kCopyVecs = 6;
constexpr int kCopyParts = kBlock / (4 * kCopyTokens);   // workgroups of 4 waves per block
template <typename T>
__global__ __launch_bounds__(256) void block_copy_kernel(const T* __restrict__ src, T* __restrict__ dst, int C,
                                                         bool src_grid, bool dst_grid, int nbh, int nbw, int dst_slot0,
                                                         int capacity, int slice_blocks, const T* __restrict__ src2,
                                                         T* __restrict__ dst2, int64_t dst_head_stride) {
  constexpr int VN = 16 / sizeof(T);
  const int b = blockIdx.x, lane = threadIdx.x & 63;
  const int t0 = (blockIdx.y * 4 + __builtin_amdgcn_readfirstlane(threadIdx.x >> 6)) * kCopyTokens;
  const T* __restrict__ from = blockIdx.z ? src2 : src;
  T* __restrict__ to = blockIdx.z ? dst2 : dst;
  const int64_t db = (int64_t)((dst_slot0 + b / slice_blocks) % capacity) * slice_blocks + (b % slice_blocks);
  const int nvec = C / VN;
  int64_t si[kCopyTokens], di[kCopyTokens];
#pragma unroll
  for (int t = 0; t < kCopyTokens; ++t) {
    si[t] = src_grid ? window_token_to_grid(b, t0 + t, nbh, nbw) : (int64_t)b * kBlock + t0 + t;
    di[t] = dst_grid ? window_token_to_grid((int)db, t0 + t, nbh, nbw) : db * kBlock + t0 + t;
  }
  for (int c0 = 0; c0 < nvec; c0 += 64 * kCopyVecs) {
    u32x4 x[kCopyTokens][kCopyVecs];
#pragma unroll
    for (int t = 0; t < kCopyTokens; ++t)
#pragma unroll
      for (int i = 0; i < kCopyVecs; ++i) {
        const int cv = c0 + 64 * i + lane;
        if (cv < nvec) x[t][i] = *(const u32x4*)(from + si[t] * C + cv * VN);
      }
#pragma unroll
    for (int t = 0; t < kCopyTokens; ++t)
#pragma unroll
      for (int i = 0; i < kCopyVecs; ++i) {
        const int cv = c0 + 64 * i + lane;
        // token-major, or head-major (a ring)
        if (cv < nvec) *(u32x4*)(to + kv_offset(di[t], cv * VN, C, dst_head_stride)) = x[t][i];
      }
  }
}

// Ring -> window order: logical block j of the held window (slot (head + j/s) % capacity) -> block j of dst.
template <typename T>
__global__ void ring_read_kernel(const T* __restrict__ rk, const T* __restrict__ rv, T* __restrict__ ok,
                                 T* __restrict__ ov, int C, int64_t head_stride, KeyMap map) {
  constexpr int VN = 16 / sizeof(T);
  typedef unsigned u4 __attribute__((ext_vector_type(4)));
  const int j = blockIdx.x;
  const int64_t sr = map.row(j), dr = (int64_t)j * kBlock;
  const int nvec = C / VN;
  for (int e = threadIdx.x; e < kBlock * nvec; e += blockDim.x) {
    const int t = e / nvec, cv = e % nvec;
    const int64_t so = kv_offset(sr + t, cv * VN, C, head_stride);
    *(u4*)(ok + (dr + t) * C + cv * VN) = *(const u4*)(rk + so);
    *(u4*)(ov + (dr + t) * C + cv * VN) = *(const u4*)(rv + so);
  }
}

// k_new / v_new into the ring slots from slot0 on
int launch_ring_append(int dtype, const void* k_new, const void* v_new, int n_blocks, int C, bool grid_layout,
                       int nbh, int nbw, int slot0, int capacity, void* ring_k, void* ring_v, int64_t head_stride,
                       hipStream_t stream) {
  if (n_blocks <= 0) return FVSR_OK;
  const int s = nbh * nbw;
  const dim3 grid(n_blocks, kCopyParts, 2);
  if (dtype == FVSR_DTYPE_BF16)
    hipLaunchKernelGGL(block_copy_kernel<bf16>, grid, dim3(256), 0, stream, (const bf16*)k_new, (bf16*)ring_k, C,
                       grid_layout, false, nbh, nbw, slot0, capacity, s, (const bf16*)v_new, (bf16*)ring_v,
                       head_stride);
  else
    hipLaunchKernelGGL(block_copy_kernel<float>, grid, dim3(256), 0, stream, (const float*)k_new, (float*)ring_k, C,
                       grid_layout, false, nbh, nbw, slot0, capacity, s, (const float*)v_new, (float*)ring_v,
                       head_stride);
  FVSR_HIP_CHECK(hipGetLastError());
  return FVSR_OK;
}

int launch_ring_read(int dtype, const void* rk, const void* rv, void* ok, void* ov, int n_blocks, int C,
                     int64_t head_stride, KeyMap map, hipStream_t stream) {
  if (n_blocks <= 0) return FVSR_OK;
  if (dtype == FVSR_DTYPE_BF16)
    hipLaunchKernelGGL(ring_read_kernel<bf16>, dim3(n_blocks), dim3(256), 0, stream, (const bf16*)rk,
                       (const bf16*)rv, (bf16*)ok, (bf16*)ov, C, head_stride, map);
  else
    hipLaunchKernelGGL(ring_read_kernel<float>, dim3(n_blocks), dim3(256), 0, stream, (const float*)rk,
                       (const float*)rv, (float*)ok, (float*)ov, C, head_stride, map);
  FVSR_HIP_CHECK(hipGetLastError());
  return FVSR_OK;
}

// natural (f, h, w) order <-> window order
int launch_window_layout(int dtype, const void* x, void* out, int f, int h, int w, int C, bool to_windows,
                         hipStream_t stream) {
  const int nbh = h / 8, nbw = w / 8;
  const int n_blocks = (f / 2) * nbh * nbw;
  if (n_blocks <= 0) return FVSR_OK;
  const int big = 1 << 30;   // identity destination mapping
  const dim3 grid(n_blocks, kCopyParts);
  if (dtype == FVSR_DTYPE_BF16)
    hipLaunchKernelGGL(block_copy_kernel<bf16>, grid, dim3(256), 0, stream, (const bf16*)x, (bf16*)out, C, to_windows,
                       !to_windows, nbh, nbw, 0, 1, big, (const bf16*)nullptr, (bf16*)nullptr, (int64_t)0);
  else
    hipLaunchKernelGGL(block_copy_kernel<float>, grid, dim3(256), 0, stream, (const float*)x, (float*)out, C,
                       to_windows, !to_windows, nbh, nbw, 0, 1, big, (const float*)nullptr, (float*)nullptr,
                       (int64_t)0);
  FVSR_HIP_CHECK(hipGetLastError());
  return FVSR_OK;
}

}  // namespace fvsr
