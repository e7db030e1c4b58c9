// hgpu_xfer.h -- kernels of the copies of large arrays between device and
// (pageable) host memory through a ring of pinned chunks (hgpu_ring.h).
//
// The reference's arrays hold a zone's variables together ([zone][8]), the
// device's hold a variable's zones together ([8][zone]).  The GPU turns one into
// the other as it fills or empties a pinned chunk, and the host moves the chunks
// meanwhile (up to 6 threads on the way down, the caller alone on the way up), so
// a download runs near the link's rate (57 GB/s pinned) instead of one host core's
// (transposing 336 MB on the host took 50 ms beside the copy).  Measured, 192x192x128 with ghosts
// (336 MB) to fresh numpy memory: 57 -> 8.1 ms down, 12 ms up.
#pragma once
#include "hgpu_launch.h"
#include "hgpu_ring.h"

namespace hgpu {

constexpr int XFER_B = 256;

// nz zones from zone z0 of S ([8][nt]) to out ([nz][8]); a workgroup turns 256
// zones around in LDS so that both sides are read and written in whole lines.
// The LDS rows are 264 words of 8 B apart: a wavefront's 8 variables x 8 zones
// then meet on at most two lanes per bank.
__global__ __launch_bounds__(XFER_B) void k_soa_to_aos(const double* __restrict__ S, long long nt, long long z0,
                                                       long long nz, double* __restrict__ out) {
  __shared__ double buf[NP][XFER_B + 8];
  const long long zb = (long long)blockIdx.x * XFER_B;
  const long long z = zb + threadIdx.x;
  if (z < nz) {
#pragma unroll
    for (int v = 0; v < NP; v++) buf[v][threadIdx.x] = S[v*nt + z0 + z];
  }
  __syncthreads();
  const long long n = (nz - zb < XFER_B ? nz - zb : XFER_B) * NP;
#pragma unroll
  for (int r = 0; r < NP; r++) {
    const int e = r*XFER_B + threadIdx.x;
    if (e < n) out[zb*NP + e] = buf[e % NP][e / NP];
  }
}

__global__ __launch_bounds__(XFER_B) void k_aos_to_soa(const double* __restrict__ in, long long nt, long long z0,
                                                       long long nz, double* __restrict__ S) {
  __shared__ double buf[NP][XFER_B + 8];
  const long long zb = (long long)blockIdx.x * XFER_B;
  const long long n = (nz - zb < XFER_B ? nz - zb : XFER_B) * NP;
#pragma unroll
  for (int r = 0; r < NP; r++) {
    const int e = r*XFER_B + threadIdx.x;
    if (e < n) buf[e % NP][e / NP] = in[zb*NP + e];
  }
  __syncthreads();
  const long long z = zb + threadIdx.x;
  if (z < nz) {
#pragma unroll
    for (int v = 0; v < NP; v++) S[v*nt + z0 + z] = buf[v][threadIdx.x];
  }
}

// n32 words of 4 B from src to dst, 16 B at a time; both 16 B aligned
__global__ __launch_bounds__(XFER_B) void k_copy_words(const unsigned* __restrict__ src, long long n32,
                                                       unsigned* __restrict__ dst) {
  const long long n16 = n32 / 4, stride = (long long)gridDim.x * XFER_B;
  const long long t0 = (long long)blockIdx.x * XFER_B + threadIdx.x;
  for (long long t = t0; t < n16; t += stride)
    reinterpret_cast<uint4*>(dst)[t] = reinterpret_cast<const uint4*>(src)[t];
  if (t0 < n32 - 4*n16) dst[4*n16 + t0] = src[4*n16 + t0];
}

}  // namespace hgpu
