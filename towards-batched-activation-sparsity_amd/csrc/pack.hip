// pack.hip — packing of a weight into the tiled K-major layout of include/bsgemm.h (the reference's
// _get_prepacked_weight_block_major, kernels/shared_mask_batched_triton_min_runtime.py:3133-3163).
//
// The layout is a transposition of 16-byte pieces: tile (K-block j, 16 columns t) is 2 KiB, the
// piece of column c and channels 8q .. 8q+7 of the block at byte (16 q + c) * 16 of it.  Packing
// moves every weight byte once in and once out, so it is bound by HBM; three kernels differ in
// how the source is laid out.

#include <hip/hip_runtime.h>

#include "pack.hpp"

namespace {

typedef unsigned int u32x4 __attribute__((ext_vector_type(4)));
typedef unsigned int u32x2 __attribute__((ext_vector_type(2)));

// Rows of consecutive channels (stride_k == 1, rows 16-byte aligned: nn.Linear's [N, K]): one
// wave moves one tile.  Each of its two loads covers 8 columns x 128 bytes (whole cache lines) and
// each store eight 128-byte runs of the tile.  The waves of a work-group take consecutive K-blocks
// of the same 16 columns, so neighbouring waves read on in the same 16 rows.  180 MB in and out
// ([11008, 4096]): 31.8 us (5.7 TB/s; a plain copy reaches 5.0), where eight 16-bit loads per
// piece took 81; 2, 4 or 8 tiles per wave: 33.1, 34.7, 35.8.
__global__ __launch_bounds__(256) void bsg_pack_rows_kernel(const uint16_t* __restrict__ w, int32_t N, int32_t K,
                                                            int64_t sn, int32_t nblk, int32_t ntile,
                                                            uint16_t* __restrict__ wp) {
  const int lane = threadIdx.x & 63;
  const int64_t item = (int64_t)blockIdx.x * 4 + (threadIdx.x >> 6);
  const int t = (int)(item / nblk);
  const int j = (int)(item - (int64_t)t * nblk);
  if (t >= ntile) return;
  const int q = lane & 7, c0 = lane >> 3;
  const int k = 64 * j + 8 * q;
  u32x4 v[2];
#pragma unroll
  for (int i = 0; i < 2; ++i) {
    const int n = 16 * t + c0 + 8 * i;
    v[i] = u32x4{0u, 0u, 0u, 0u};
    if (n < N && k < K) {
      const uint16_t* src = w + (int64_t)n * sn + k;
      if (k + 8 <= K) {
        v[i] = __builtin_nontemporal_load((const u32x4*)src);
      } else {  // the last channels of a K that is not a multiple of 8
        uint32_t d[4] = {0u, 0u, 0u, 0u};
#pragma unroll
        for (int e = 0; e < 8; ++e)
          if (k + e < K) d[e >> 1] |= (uint32_t)src[e] << (16 * (e & 1));
        v[i] = u32x4{d[0], d[1], d[2], d[3]};
      }
    }
  }
  uint16_t* dst = wp + ((int64_t)j * ntile + t) * 1024 + (16 * q + c0) * 8;
#pragma unroll
  for (int i = 0; i < 2; ++i) __builtin_nontemporal_store(v[i], (u32x4*)(dst + 64 * i));
}

// Consecutive columns (stride_n == 1, rows 8-byte aligned: a [K, N] matrix): a work-group moves one
// K-block of 256 columns.  Wave q reads channels 8q .. 8q+7, 512 contiguous bytes of each, and
// transposes 4 columns x 8 channels per lane in registers; the pieces cross the work-group in LDS
// (one piece of padding per 16) so that every store covers whole contiguous KiBs.  180 MB in and
// out: 30.0 us (41-45 with 16-bit loads); 42 when each lane stores its own four pieces, 113 when
// those partial lines are also non-temporal.
__global__ __launch_bounds__(512) void bsg_pack_cols_kernel(const uint16_t* __restrict__ w, int32_t N, int32_t K,
                                                            int64_t sk, int32_t ntile, int32_t cgroups,
                                                            uint16_t* __restrict__ wp) {
  __shared__ u32x4 s_piece[8][256 + 16];
  const int lane = threadIdx.x & 63, q = threadIdx.x >> 6;
  const int j = (int)(blockIdx.x / (unsigned)cgroups);
  const int n0 = ((int)blockIdx.x - j * cgroups) * 256;
  const int n = n0 + 4 * lane;
  u32x2 v[8];
#pragma unroll
  for (int e = 0; e < 8; ++e) {
    const int k = 64 * j + 8 * q + e;
    v[e] = u32x2{0u, 0u};
    if (k < K && n < N) {
      const uint16_t* src = w + (int64_t)k * sk + n;
      if (n + 4 <= N) {
        v[e] = __builtin_nontemporal_load((const u32x2*)src);
      } else {  // the last columns of an N that is not a multiple of 4
        uint32_t d[2] = {0u, 0u};
#pragma unroll
        for (int i = 0; i < 4; ++i)
          if (n + i < N) d[i >> 1] |= (uint32_t)src[i] << (16 * (i & 1));
        v[e] = u32x2{d[0], d[1]};
      }
    }
  }
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    u32x4 o;
#pragma unroll
    for (int d = 0; d < 4; ++d) {
      const uint32_t a = i < 2 ? v[2 * d].x : v[2 * d].y, b = i < 2 ? v[2 * d + 1].x : v[2 * d + 1].y;
      o[d] = (i & 1) ? (a >> 16) | (b & 0xffff0000u) : (a & 0xffffu) | (b << 16);
    }
    s_piece[q][4 * lane + i + (lane >> 2)] = o;
  }
  __syncthreads();
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const int tl = 4 * i + (threadIdx.x >> 7), pc = threadIdx.x & 127;  // tile of the 16, piece of the 128
    const int t = (n0 >> 4) + tl;
    if (t < ntile)
      __builtin_nontemporal_store(s_piece[pc >> 4][17 * tl + (pc & 15)],
                                  (u32x4*)(wp + ((int64_t)j * ntile + t) * 1024 + pc * 8));
  }
}

// Any other strides or alignment: one thread gathers the 8 channels of one 16-byte piece.
__global__ __launch_bounds__(256) void bsg_pack_kernel(const uint16_t* __restrict__ w, int64_t N, int64_t K,
                                                       int64_t sn, int64_t skk, int64_t ntile, int64_t groups,
                                                       uint16_t* __restrict__ wp) {
  const int64_t gid = (int64_t)blockIdx.x * 256 + threadIdx.x;
  if (gid >= groups) return;
  const int64_t blk = gid / (ntile * 128);
  const int64_t rem = gid - blk * ntile * 128;
  const int64_t t = rem >> 7;
  const int r = (int)(rem & 127);
  const int h = r >> 6, g = (r >> 4) & 3, c = r & 15;
  const int64_t n = 16 * t + c;
  const int64_t k0 = 64 * blk + 32 * h + 8 * g;
  uint16_t v[8];
#pragma unroll
  for (int e = 0; e < 8; ++e) v[e] = (n < N && k0 + e < K) ? w[n * sn + (k0 + e) * skk] : (uint16_t)0;
  u32x4 o;
  o.x = v[0] | ((uint32_t)v[1] << 16);
  o.y = v[2] | ((uint32_t)v[3] << 16);
  o.z = v[4] | ((uint32_t)v[5] << 16);
  o.w = v[6] | ((uint32_t)v[7] << 16);
  *(u32x4*)(wp + gid * 8) = o;
}

int64_t cdiv(int64_t a, int64_t b) { return (a + b - 1) / b; }

}  // namespace

namespace bsgk {

int launch_pack(const void* w, int64_t N, int64_t K, int64_t stride_n, int64_t stride_k, void* wp, void* stream) {
  const int64_t ntile = cdiv(N, 16), nblk = cdiv(K, 64);
  const hipStream_t st = (hipStream_t)stream;
  const uint16_t* src = (const uint16_t*)w;
  // The wide loads need their alignment in every row; whatever lacks it keeps the gather.
  const int64_t row_groups = cdiv(ntile * nblk, 4);
  const int64_t cgroups = cdiv(16 * ntile, 256), col_groups = nblk * cgroups;
  if (stride_k == 1 && stride_n % 8 == 0 && ((uintptr_t)w & 15u) == 0 && N <= 0x7ffffff0 && row_groups <= 0x7fffffff) {
    hipLaunchKernelGGL(bsg_pack_rows_kernel, dim3((unsigned)row_groups), dim3(256), 0, st, src, (int32_t)N,
                       (int32_t)K, stride_n, (int32_t)nblk, (int32_t)ntile, (uint16_t*)wp);
  } else if (stride_n == 1 && stride_k % 4 == 0 && ((uintptr_t)w & 7u) == 0 && N <= 0x7ffffff0 &&
             col_groups <= 0x7fffffff) {
    hipLaunchKernelGGL(bsg_pack_cols_kernel, dim3((unsigned)col_groups), dim3(512), 0, st, src, (int32_t)N,
                       (int32_t)K, stride_k, (int32_t)ntile, (int32_t)cgroups, (uint16_t*)wp);
  } else {
    const int64_t groups = nblk * ntile * 128;
    const int64_t nb = cdiv(groups, 256);
    if (nb > 0x7fffffff) return -1;
    hipLaunchKernelGGL(bsg_pack_kernel, dim3((unsigned)nb), dim3(256), 0, st, src, N, K, stride_n, stride_k, ntile,
                       groups, (uint16_t*)wp);
  }
  return (int)hipGetLastError();
}

}  // namespace bsgk
