// spmm.hpp — sparse matrix times a block of W interleaved dense vectors
// (device code shared by the batched and the unrolled/adjoint paths).
//
// The W right-hand sides of one block are stored interleaved per element
// (V[j*W + f]), so the W lanes that own one matrix segment gather one
// contiguous W*4-byte run per record and every matrix record streamed from
// HBM serves W vectors. A 256-lane workgroup walks whole tiles of segments
// (rows of the CSR or columns of the CSC) in a persistent loop, stages each
// tile's 8-byte records in LDS with coalesced loads, and gives every segment
// to a group of W lanes; lane f accumulates vector f sequentially in element
// order with separate multiply and add (this code is compiled with
// -ffp-contract=off), so every vector's result is the reference driver's
// sequential fp32 sum (mlem_seq/seqcsr4mlem.cpp:69-91 for the CSR,
// :108-120 for the CSC in ascending row order). Where that is faster, the lanes
// of a segment read its records themselves (walk_direct): the same sums.
#pragma once
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cstdint>
#include <type_traits>
#include <vector>

namespace mlem {
namespace spmm {

constexpr int kBlock = 256;
constexpr uint32_t kTile = 2048;  // records staged per tile (16 KB of LDS)
#ifndef MLEM_SPMM_UNROLL
#define MLEM_SPMM_UNROLL 16
#endif
constexpr int kUnroll = MLEM_SPMM_UNROLL;  // gathers in flight per lane

// Sequential fp32 dot product of one segment's records with vector f of an
// interleaved block. The gathers of U consecutive records are issued
// together (the segment's last group with clamped indices), the products are
// then added one by one in element order.
template <int W, int U = kUnroll>
__device__ __forceinline__ float seg_dot(const uint2* rec, uint32_t b, uint32_t e,
                                         const float* __restrict__ v, uint32_t f) {
  float acc = 0.f;
  for (uint32_t k = b; k < e; k += U) {
    float a[U], g[U];
#pragma unroll
    for (int j = 0; j < U; ++j) {
      const uint2 r = rec[min(k + j, e - 1)];
      a[j] = __uint_as_float(r.y);
      g[j] = v[(size_t)r.x * W + f];
    }
#pragma unroll
    for (int j = 0; j < U; ++j)
      if (k + j < e) acc = acc + a[j] * g[j];
  }
  return acc;
}

// Walk the tiles [0, ntiles) of a segment partition (tiles[t] = {first
// segment, first element}) and call epi(segment, f, dot) for every segment
// and vector. Tiles hold at most 256 segments and kTile records, or one
// longer segment (read from HBM, 4 records at a time: its 64-bit record
// addresses would otherwise set the kernel's register count). Workgroup b runs on XCD b % 8 (the grid is
// a multiple of 8): XCD x walks the x-th contiguous eighth of the tiles, so
// neighbouring segments (rows of one sinogram region, voxels of one brick
// range) share that XCD's L2.
template <int W, class Epi>
__device__ __forceinline__ void walk(const uint32_t* __restrict__ ptr,
                                     const uint2* __restrict__ el,
                                     const uint2* __restrict__ tiles, uint32_t ntiles,
                                     const float* __restrict__ v, Epi& epi) {
  constexpr int G = kBlock / W;
  __shared__ uint2 rec[kTile];
  __shared__ uint32_t S[kBlock + 1];
  const uint32_t t = threadIdx.x, f = t % W, grp = t / W;
  const uint32_t xcd = blockIdx.x & 7u, per_xcd = gridDim.x >> 3;
  const uint32_t t0 = (uint32_t)((uint64_t)ntiles * xcd / 8);
  const uint32_t t1 = (uint32_t)((uint64_t)ntiles * (xcd + 1) / 8);
  for (uint32_t tile = t0 + (blockIdx.x >> 3); tile < t1; tile += per_xcd) {
    const uint2 d0 = tiles[tile], d1 = tiles[tile + 1];
    const uint32_t s0 = d0.x, e0 = d0.y, nseg = d1.x - s0, count = d1.y - e0;
    __syncthreads();  // the previous tile's readers are done with rec / S
    const bool staged = count <= kTile;
    if (staged)
      for (uint32_t i = t; i < count; i += kBlock) rec[i] = el[e0 + i];
    for (uint32_t i = t; i <= nseg; i += kBlock) S[i] = ptr[s0 + i] - e0;
    __syncthreads();
    for (uint32_t sg = grp; sg < nseg; sg += G) {
      const float d = staged ? seg_dot<W>(rec, S[sg], S[sg + 1], v, f)
                             : seg_dot<W, 4>(el + e0, S[sg], S[sg + 1], v, f);
      epi(s0 + sg, f, d);
    }
  }
}

// The same sums without tiles, for W = 16 and 32: the W lanes of a segment load
// 16 records at a time themselves (one per lane; W = 32: both rows of 16 lanes the
// same ones) and broadcast them along the row, the next 16 in flight while these
// are gathered. Workgroup b takes kBlock / W neighbouring segments, numbered as
// walk() numbers its tiles. The gathered vectors are shorter than 2^32 bytes.
//
// Bound by the gathered lines (64 or 128 bytes per record). No barrier and no
// second reading of the records from LDS; but a run of 16 records is only half
// or a whole line, read by as many waves as there are segments in it. us, walk()
// first: A v, 128x128x48 voxels and 1327104 lines, W = 16 1622 > 1294, W = 32
// 2395 > 1589; 75x77x31 and 200003 138 > 135, 217 > 178. A^T v, W = 32 1964 >
// 1840, 192 > 167; but W = 16 1447 > 1635, 124 > 136, and narrower blocks 3 to
// 20 % slower in either direction: direct() leaves those to walk().
template <int j>
__device__ __forceinline__ uint32_t row_lane(uint32_t x) {  // lane j of each row of 16
  return (uint32_t)__builtin_amdgcn_mov_dpp((int)x, 0x150 + j, 0xF, 0xF, true);
}
template <int j>
__device__ __forceinline__ void row_gather(uint32_t at, uint32_t val, const char* __restrict__ v,
                                           uint32_t f4, float (&g)[16], float (&a)[16]) {
  if constexpr (j < 16) {
    g[j] = *reinterpret_cast<const float*>(v + (row_lane<j>(at) + f4));
    a[j] = __uint_as_float(row_lane<j>(val));
    row_gather<j + 1>(at, val, v, f4, g, a);
  }
}
template <int W, class Epi>
__device__ __forceinline__ void walk_direct(const uint32_t* __restrict__ ptr,
                                            const uint2* __restrict__ el, uint32_t n,
                                            const float* __restrict__ v, Epi& epi) {
  static_assert(W == 16 || W == 32, "whole rows of 16 lanes per segment");
  constexpr uint32_t G = kBlock / W;
  const uint32_t t = threadIdx.x, f = t % W, l = t % 16;
  const uint32_t nb = (n + G - 1) / G, xcd = blockIdx.x & 7u;
  const uint32_t blk = (uint32_t)((uint64_t)nb * xcd / 8) + (blockIdx.x >> 3);
  const uint64_t s = (uint64_t)blk * G + t / W;
  if (blk >= (uint32_t)((uint64_t)nb * (xcd + 1) / 8) || s >= n) return;
  const uint32_t b = ptr[s], e = ptr[s + 1];
  const char* __restrict__ vb = reinterpret_cast<const char*>(v);
  float acc = 0.f;
  uint2 next = make_uint2(0, 0);
  if (b < e) next = el[min(b + l, e - 1)];
  for (uint32_t k = b; k < e; k += 16) {
    float g[16], a[16];
    row_gather<0>(next.x * (4 * W), next.y, vb, f * 4, g, a);
    if (k + 16 < e) next = el[min(k + 16 + l, e - 1)];
    if (k + 16 <= e) {
#pragma unroll
      for (int j = 0; j < 16; ++j) acc = acc + a[j] * g[j];
    } else {
#pragma unroll
      for (int j = 0; j < 16; ++j)
        if (k + j < e) acc = acc + a[j] * g[j];
    }
  }
  epi((uint32_t)s, f, acc);
}

// count: segments (kDirect) or tiles.
template <int W, bool kDirect, class Epi>
__device__ __forceinline__ void product(const uint32_t* __restrict__ ptr,
                                        const uint2* __restrict__ el,
                                        const uint2* __restrict__ tiles, uint32_t count,
                                        const float* __restrict__ v, Epi& epi) {
  if constexpr (kDirect)
    walk_direct<W>(ptr, el, count, v, epi);
  else
    walk<W>(ptr, el, tiles, count, v, epi);
}
// Whether A v (csc = false, gathering cols runs) or A^T v (csc, rows runs) of W
// vectors takes walk_direct(); the reasons stand there.
template <int W>
constexpr bool kDirectWidth = W == 16 || W == 32;
template <int W>
inline bool direct(bool csc, uint64_t gathered) {
  return (W == 32 || (W == 16 && !csc)) && gathered * W * 4 < (1ull << 32);
}
template <int W>
inline uint32_t direct_grid(uint32_t n) {
  return ((n + kBlock / W - 1) / (kBlock / W) + 7) / 8 * 8;
}

// Greedy partition of segments [0, n) into tiles of at most T records and
// 256 segments; a segment longer than T forms a tile of its own. Returns the
// first segment of every tile plus n.
inline std::vector<uint32_t> partition(const std::vector<uint32_t>& ptr, uint32_t T) {
  const uint32_t n = (uint32_t)ptr.size() - 1;
  std::vector<uint32_t> tiles{0};
  uint32_t s = 0;
  while (s < n) {
    uint32_t e = s;
    if (ptr[s + 1] - ptr[s] > T) {
      e = s + 1;
    } else {
      uint64_t cnt = 0;
      while (e < n && e - s < (uint32_t)kBlock && cnt + (ptr[e + 1] - ptr[e]) <= T) {
        cnt += ptr[e + 1] - ptr[e];
        ++e;
      }
    }
    tiles.push_back(e);
    s = e;
  }
  return tiles;
}

}  // namespace spmm
}  // namespace mlem
