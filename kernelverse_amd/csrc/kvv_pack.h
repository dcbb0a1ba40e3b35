// Packing of a strided tensor into contiguous workspace memory, in logical
// (row-major) order, ahead of a single pair's main pass (included by kvv.hip).
//
// A pair whose layouts rule out 16-byte vectors (a transposed or channels-last
// view against a contiguous tensor, a slice at an odd offset or pitch, a step)
// took the scalar main pass: one element per lane and step with its index
// divided out per dim, and the full per-element treatment whatever the data.
// Each such tensor is now copied once into the workspace, and the vector main
// pass reads the copy: one write and one read of the tensor more, far less than
// the scalar pass's time.  Whole verdicts, scalar and packed: 4096 x 4096 bf16
// with a transposed reference 178 and 84 us (the copy 14.4, 4.7 TB/s), 4096 x
// 8192 fp8 233 and 77 us, 4096 x 8192 fp32 625 and 139 us, 16384 x 1000 bf16
// against a slice at an odd offset and pitch 124 and 73 us.
//
// Two forms:
// * transpose: another dim p is the contiguous one of the source.  A block moves
//   a 64 x 64 tile of (p, q), q the innermost logical dim, through LDS: loads
//   run along p and stores along q, a wave on 64 consecutive elements each.
// * gather: any other strides (rows at odd offsets, steps, broadcast dims).  A
//   thread assembles one 16-byte output vector from element loads; a wave's
//   loads stay within the rows it covers, which the caches serve.
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

namespace kvv {

constexpr int kPackTile = 64;

// Tensors above this many bytes are not packed: the copies would cost that much
// workspace each.
constexpr int64_t kPackMax = int64_t(1) << 30;
static_assert(kPackMax < (int64_t(1) << 31), "32-bit element indices and block counts");

struct PackArgs {
  const void* src;
  void* dst;
  int64_t n;
  int32_t nd;
  int32_t p;                    // the source's contiguous dim (transpose form), else -1
  int64_t sizes[KVV_MAX_DIMS];  // coalesced, none of size 1
  int64_t str[KVV_MAX_DIMS];    // source strides
  int64_t out[KVV_MAX_DIMS];    // logical (row-major) strides
  int64_t blocks;
};

// (One kernel per form and tensor: with both tensors' arguments in one launch,
// chosen by block, the compiler copied them to scratch and every field came from
// memory: 125 us instead of 14.4 for the first pair above.)
template <typename T>
__global__ __launch_bounds__(256) void pack_gather_kernel(PackArgs a) {
  constexpr int V = 16 / (int)sizeof(T);
  union {
    uint4 q;
    T e[V];
  } o;
  const int64_t i0 = ((int64_t)blockIdx.x * 256 + threadIdx.x) * V;
  if (i0 >= a.n) return;
  const T* src = reinterpret_cast<const T*>(a.src);
  T* dst = reinterpret_cast<T*>(a.dst);
  // source offset of element i; c: its index in the innermost dim
  auto offset_of = [&](uint32_t i, uint32_t& c) {
    int64_t off = 0;
    uint32_t r = i;
    c = r;
    for (int k = a.nd - 1; k > 0; --k) {
      const uint32_t s = (uint32_t)a.sizes[k], q = r / s, x = r - q * s;
      if (k == a.nd - 1) c = x;
      off += (int64_t)x * a.str[k];
      r = q;
    }
    return off + (int64_t)r * a.str[0];
  };
  uint32_t c_last;
  const int64_t off = offset_of((uint32_t)i0, c_last);
  const int64_t s_last = a.str[a.nd - 1];
  const int ne = a.n - i0 < V ? (int)(a.n - i0) : V;
  if (ne == V && c_last + V <= a.sizes[a.nd - 1]) {
#pragma unroll
    for (int e = 0; e < V; ++e) o.e[e] = src[off + e * s_last];
    *reinterpret_cast<uint4*>(dst + i0) = o.q;
    return;
  }
  // a vector across rows, or the tensor's last
  for (int e = 0; e < ne; ++e) dst[i0 + e] = src[offset_of((uint32_t)(i0 + e), c_last)];
}

template <typename T>
__global__ __launch_bounds__(256) void pack_transpose_kernel(PackArgs a) {
  // (a row of the tile is an odd number of words: its columns spread over the banks)
  __shared__ T tile[kPackTile][kPackTile + 4 / (sizeof(T) < 4 ? sizeof(T) : 4)];
  const int64_t blk = blockIdx.x;
  constexpr int R = kPackTile / 4;  // rows per wave
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6, q = a.nd - 1, p = a.p;
  const int64_t np = a.sizes[p], nq = a.sizes[q];
  const int64_t tp = (np + kPackTile - 1) / kPackTile, tq = (nq + kPackTile - 1) / kPackTile;
  const int64_t per = tp * tq;
  int64_t rest = blk / per;  // the other dims' index
  const int64_t t = blk - rest * per;
  const int64_t p0 = (t % tp) * kPackTile, q0 = (t / tp) * kPackTile;
  int64_t so = 0, po = 0;
  for (int k = a.nd - 2; k >= 0; --k) {
    if (k == p) continue;
    const int64_t n = rest / a.sizes[k], c = rest - n * a.sizes[k];
    so += c * a.str[k];
    po += c * a.out[k];
    rest = n;
  }
  const T* src = reinterpret_cast<const T*>(a.src) + so + p0 + q0 * a.str[q];
  T* dst = reinterpret_cast<T*>(a.dst) + po + p0 * a.out[p] + q0;
  const int64_t left_p = np - p0, left_q = nq - q0;
  T x[R];
#pragma unroll
  for (int i = 0; i < R; ++i) {
    const int row = w * R + i;
    x[i] = row < left_q && lane < left_p ? src[(int64_t)row * a.str[q] + lane] : (T)0;
  }
#pragma unroll
  for (int i = 0; i < R; ++i) tile[w * R + i][lane] = x[i];
  __syncthreads();
#pragma unroll
  for (int i = 0; i < R; ++i) {
    const int row = w * R + i;
    if (row < left_p && lane < left_q) dst[(int64_t)row * a.out[p] + lane] = tile[lane][row];
  }
}

}  // namespace kvv
