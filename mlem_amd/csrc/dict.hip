// dict.hip — load-time construction of the dictionary tiles (kernels.hip runs
// the projections over them), gfx950.
//
// Every tile of at most T elements gets the sorted distinct indices it
// gathers, and every element its 16-bit position among them. The tile's
// indices are marked in a bitmap in LDS; a prefix sum of the words' population
// counts gives every marked index its rank, which is its position. The bitmap
// holds the pages that the tile uses, one after the other (a page: at most
// 1/8192th of all indices, at least 32 of them), in slabs of 2^18 indices at a
// time.
//
// What bounds it: the LDS passes over the slabs (clear, mark, count, look up;
// about 1 us each for a 1024-lane workgroup, two of them per CU).
// Both projections' tiles of 2048 / 8192 / 16384 elements, allocation included, ms:
//   192x192x64 voxels, 1.5M lines (282M elements)     20.6 / 10.8 / 9.7
//   3M rows, 5M columns, 30M elements at random        7.8 /  7.5 / 8.6
// A bitmap of all indices, without pages, took 41 / 17 / 16 and 14 / 33 / 34 (a
// pass per slab that holds an element: up to one per element where the indices
// spread far), a bitonic sort of 8-byte keys in LDS 43 / 110 / 222 and 8.9 / 27 / 89.
#include <algorithm>
#include <initializer_list>
#include <vector>

#include "internal.hpp"
#include "mlem.h"

namespace mlem {
namespace {

constexpr int kBlock = 256;
constexpr uint32_t kWave = 64;
constexpr uint32_t kBuild = 1024;                 // lanes of a build workgroup
constexpr uint32_t kSlabBits = 18;                // indices per bitmap slab (log2)
constexpr uint32_t kWords = (1u << kSlabBits) / 32;
constexpr uint32_t kLaneWords = kWords / kBuild;  // words counted by one lane
constexpr uint32_t kPages = 1u << 14;             // pages of all indices (at most)
static_assert(kLaneWords == 8, "word() pads every lane's run of 8 words");

// Word w of the bitmap: one word of padding after every 8, so that the lanes'
// runs of 8 words start in different LDS banks.
__device__ __forceinline__ uint32_t word(uint32_t w) { return w + (w >> 3); }

void check_launch(const char* what) {
  hipError_t e = hipGetLastError();
  if (e != hipSuccess) raise(MLEM_EDEVICE, std::string(what) + ": " + hipGetErrorString(e));
}

// One tile per workgroup, at most EB elements per lane. Pass 1 (tiles4 ==
// nullptr) counts the distinct indices of every tile, and the runs of 32 indices
// (128-byte lines of the gathered vector) that they lie in; pass 2 writes the
// dictionary, padded with zeros to whole rounds of `nb` entries, and the
// {value, position} element arrays, with the tile's leading zero elements and
// padded with zeros to 64 elements. Indices are below kPages * 2^page_bits.
template <uint32_t EB, int VK>
__global__ __launch_bounds__(kBuild) void k_dict_rank(const uint2* __restrict__ el,
                                                      const uint2* __restrict__ tiles2,
                                                      const uint4* __restrict__ tiles4,
                                                      uint32_t nb, uint32_t page_bits,
                                                      uint2* __restrict__ counts,
                                                      uint32_t* __restrict__ dict,
                                                      void* __restrict__ dval,
                                                      uint16_t* __restrict__ dlix) {
  constexpr uint32_t T = kBuild * EB;
  __shared__ uint32_t bits[kWords + kWords / 8];
  __shared__ uint16_t before[kWords + kWords / 8];  // marked indices before each word
  __shared__ uint32_t pages[kPages / 32];           // pages that hold an element
  __shared__ uint16_t pbefore[kPages / 32];         // such pages before each word
  __shared__ uint32_t wsum[kBuild / kWave], lines;
  const uint32_t tile = blockIdx.x, t = threadIdx.x, lane = t % kWave, wave = t / kWave;
  uint32_t e0, e1, a0 = 0, lead = 0, g0 = 0;
  if (tiles4) {
    const uint4 a = tiles4[tile], b = tiles4[tile + 1];
    e0 = a.y;
    e1 = b.y;
    a0 = a.z & ~63u;
    lead = a.z & 63u;
    g0 = a.w;
  } else {
    e0 = tiles2[tile].y;
    e1 = tiles2[tile + 1].y;
  }
  const uint32_t count = e1 - e0;
  if (count > T || count == 0) {  // one long segment, or nothing: no dictionary
    if (!tiles4 && t == 0) counts[tile] = make_uint2(0, 0);
    return;
  }
  // Sum over the lanes before this one; all: over all of them. A barrier lies
  // between two calls.
  auto scan = [&](uint32_t mine, uint32_t& all) __attribute__((always_inline)) {
    uint32_t run = mine;  // inclusive sum over the wave
#pragma unroll
    for (uint32_t d = 1; d < kWave; d <<= 1) {
      const uint32_t o = (uint32_t)__shfl_up((int)run, d);
      if (lane >= d) run += o;
    }
    if (lane == kWave - 1) wsum[wave] = run;
    __syncthreads();
    uint32_t base = run - mine;
    all = 0;
    for (uint32_t w = 0; w < kBuild / kWave; ++w) {
      const uint32_t v = wsum[w];
      if (w < wave) base += v;
      all += v;
    }
    return base;
  };
  uint2 e[EB];
#pragma unroll
  for (uint32_t j = 0; j < EB; ++j) e[j] = el[e0 + min(t + j * kBuild, count - 1)];
  if (t < kPages / 32) pages[t] = 0;
  if (t == 0) lines = 0;
  __syncthreads();
#pragma unroll
  for (uint32_t j = 0; j < EB; ++j) {
    const uint32_t p = e[j].x >> page_bits;
    if (!((pages[p >> 5] >> (p & 31u)) & 1u)) atomicOr(&pages[p >> 5], 1u << (p & 31u));
  }
  __syncthreads();
  uint32_t used;  // pages
  const uint32_t pb = scan(t < kPages / 32 ? __popc(pages[t]) : 0u, used);
  if (t < kPages / 32) pbefore[t] = (uint16_t)pb;
  __syncthreads();
  uint32_t pos[EB];  // place in the used pages, then the index's rank
#pragma unroll
  for (uint32_t j = 0; j < EB; ++j) {
    const uint32_t p = e[j].x >> page_bits, b = p & 31u;
    const uint32_t at = pbefore[p >> 5] + __popc(pages[p >> 5] & ((1u << b) - 1u));
    pos[j] = (at << page_bits) | (e[j].x & ((1u << page_bits) - 1u));
  }
  const uint64_t places = (uint64_t)used << page_bits;
  const uint32_t slabs = (uint32_t)((places + (1u << kSlabBits) - 1) >> kSlabBits);
  uint32_t total = 0;  // distinct indices in the slabs so far (uniform)
  for (uint32_t s = 0; s < slabs; ++s) {
    // words of the slab, to a whole lane's run
    const uint64_t left = (places - ((uint64_t)s << kSlabBits) + 255) / 256 * 8;
    const uint32_t words = (uint32_t)min(left, (uint64_t)kWords);
    for (uint32_t w = t; w < words + words / 8; w += kBuild) bits[w] = 0;
    __syncthreads();
#pragma unroll
    for (uint32_t j = 0; j < EB; ++j)
      if (pos[j] >> kSlabBits == s)
        atomicOr(&bits[word((pos[j] & ((1u << kSlabBits) - 1)) >> 5)], 1u << (pos[j] & 31u));
    __syncthreads();
    uint32_t mine = 0, full = 0;
    if (t * kLaneWords < words) {
#pragma unroll
      for (uint32_t k = 0; k < kLaneWords; ++k) {
        const uint32_t w = bits[word(t * kLaneWords + k)];
        mine += __popc(w);
        full += w != 0;
      }
    }
    if (!tiles4 && full) atomicAdd(&lines, full);
    uint32_t all;
    uint32_t at = total + scan(mine, all);
    total += all;
    if (tiles4) {
      if (t * kLaneWords < words) {
#pragma unroll
        for (uint32_t k = 0; k < kLaneWords; ++k) {
          const uint32_t w = word(t * kLaneWords + k);
          before[w] = (uint16_t)at;
          at += __popc(bits[w]);
        }
      }
      __syncthreads();
#pragma unroll
      for (uint32_t j = 0; j < EB; ++j)
        // (a rank is below 2^14: it is taken for a place of slab 0 at most)
        if (pos[j] >> kSlabBits == s) {
          const uint32_t w = word((pos[j] & ((1u << kSlabBits) - 1)) >> 5), b = pos[j] & 31u;
          pos[j] = before[w] + __popc(bits[w] & ((1u << b) - 1u));
          dict[g0 + pos[j]] = e[j].x;  // equal indices write the same word
        }
    }
    __syncthreads();  // the next slab clears the bitmap
  }
  if (!tiles4) {
    if (t == 0) counts[tile] = make_uint2(total, lines);
    return;
  }
  for (uint32_t i = total + t; i < (total + nb - 1) / nb * nb; i += kBuild) dict[g0 + i] = 0;
  auto put = [&](uint32_t i, uint32_t v, uint32_t p) {  // v: fp32 bits; 16-bit kinds are exact
    dlix[a0 + i] = (uint16_t)p;
    if constexpr (VK == kF32)
      static_cast<uint32_t*>(dval)[a0 + i] = v;
    else if constexpr (VK == kF16)
      static_cast<uint16_t*>(dval)[a0 + i] =
          __builtin_bit_cast(uint16_t, (_Float16)__uint_as_float(v));
    else
      static_cast<uint16_t*>(dval)[a0 + i] = (uint16_t)(v >> 16);
  };
#pragma unroll
  for (uint32_t j = 0; j < EB; ++j)
    if (t + j * kBuild < count) put(lead + t + j * kBuild, e[j].y, pos[j]);
  const uint32_t end = lead + count, padded = (end + 63) / 64 * 64;
  if (t < lead) put(t, 0u, 0u);
  if (end + t < padded) put(end + t, 0u, 0u);
}

// Packs every 64-entry dictionary slot in place, one wave per slot: when the
// slot's ascending indices span less than 2^16 they become 16-bit offsets
// from the first (two per word, in the slot's first 32 words); meta[slot] =
// first index, with bit 31 set when the slot keeps its 32-bit indices.
// Unused entries at a tile's end hold 0 (below the first index) and become
// offset 0.
__global__ __launch_bounds__(kBlock) void k_dict_pack(uint32_t* __restrict__ dict,
                                                      uint32_t* __restrict__ meta,
                                                      uint64_t nslots) {
  const uint64_t s = (uint64_t)blockIdx.x * (kBlock / kWave) + threadIdx.x / kWave;
  if (s >= nslots) return;  // whole waves
  const uint32_t l = threadIdx.x % kWave;
  const uint32_t v = dict[s * kWave + l];
  const uint32_t base = __shfl(v, 0);
  uint32_t hi = v;
#pragma unroll
  for (int off = kWave / 2; off > 0; off >>= 1) hi = max(hi, (uint32_t)__shfl_xor(hi, off));
  const bool wide = hi - base > 0xFFFFu;
  if (!wide) {
    const uint32_t o = v >= base ? v - base : 0u;
    const uint32_t o1 = __shfl_down(o, 1);
    if ((l & 1) == 0) dict[s * kWave + (l >> 1)] = o | (o1 << 16);
  }
  if (l == 0) meta[s] = base | (wide ? 0x80000000u : 0u);
}

// Cuts the segments [s0, s1) of one tile of 16384 elements and 512 segments into
// tiles of at most T elements, leading zeros included, and `maxseg` segments
// (DictFormat): tile(first, end, leading zeros). A larger segment stays whole.
template <class Tile>
void cut_nested(const std::vector<uint32_t>& ptr, uint32_t s0, uint32_t s1, uint32_t T,
                uint32_t maxseg, Tile&& tile) {
  for (uint32_t s = s0, e; s < s1; s = e) {
    const uint32_t z = (ptr[s] - ptr[s0]) & 3u;
    e = s + 1;
    while (e < s1 && e - s < maxseg && (uint64_t)z + (ptr[e + 1] - ptr[s]) <= T) ++e;
    tile(s, e, z);
  }
}

std::vector<uint32_t> nested_tiles(const std::vector<uint32_t>& ptr, uint32_t T, uint32_t maxseg,
                                   std::vector<uint32_t>& lead) {
  const std::vector<uint32_t> big = partition_tiles(ptr, 16384, 512);
  std::vector<uint32_t> tiles;
  lead.clear();
  for (size_t i = 0; i + 1 < big.size(); ++i)
    cut_nested(ptr, big[i], big[i + 1], T, maxseg, [&](uint32_t s, uint32_t e, uint32_t z) {
      const uint32_t n = ptr[e] - ptr[s];
      // the kernels hold T products, leading zeros included
      if (n <= T && z + n > T) raise(MLEM_EINVAL, "a segment does not fit a nested tile");
      tiles.push_back(s);
      lead.push_back(n && n <= T ? z : 0);  // only tiles with stored elements
    });
  tiles.push_back((uint32_t)ptr.size() - 1);
  return tiles;
}

// Pages of at least 32 indices that cover dim of them.
uint32_t page_bits_for(uint32_t dim) {
  uint32_t b = 5;
  while (((uint64_t)kPages << b) < dim) ++b;
  return b;
}

// Build the dictionary format of one projection from its device-order
// segments (host copy of the pointers, device 8-byte records). The format
// depends on the tile size T = NB*EPT and the segment limit NB.
template <int NB, int EPT, int VK>
void build_dict(const std::vector<uint32_t>& ptr, const uint2* el, uint32_t dim, bool nested,
                DictFormat& D, hipStream_t s) {
  const uint32_t page_bits = page_bits_for(dim);
  constexpr uint32_t T = NB * EPT;
  static_assert(T % kBuild == 0, "build workgroups cover whole tiles");
  constexpr uint32_t EB = T / kBuild;  // elements per build lane
  std::vector<uint32_t> lead;  // leading zero elements of every tile
  const std::vector<uint32_t> tl =
      nested ? nested_tiles(ptr, T, NB, lead) : partition_tiles(ptr, T, NB);
  const uint32_t nt = (uint32_t)tl.size() - 1;
  lead.resize(tl.size(), 0);
  std::vector<uint2> d2(tl.size());
  for (size_t i = 0; i < tl.size(); ++i) d2[i] = make_uint2(tl[i], ptr[tl[i]]);
  struct Buf {
    void* p = nullptr;
    ~Buf() {
      if (p) (void)hipFree(p);
    }
  } t2, ndb;
  MLEM_HIP(hipMalloc(&t2.p, sizeof(uint2) * d2.size()));
  MLEM_HIP(hipMalloc(&ndb.p, sizeof(uint2) * std::max<uint32_t>(nt, 1)));
  MLEM_HIP(hipMemcpyAsync(t2.p, d2.data(), sizeof(uint2) * d2.size(), hipMemcpyHostToDevice, s));
  std::vector<uint2> nd(nt);
  if (nt) {
    hipLaunchKernelGGL((k_dict_rank<EB, VK>), dim3(nt), dim3(kBuild), 0, s, (const uint2*)el,
                       (const uint2*)t2.p, (const uint4*)nullptr, (uint32_t)NB, page_bits,
                       (uint2*)ndb.p,
                       (uint32_t*)nullptr, (void*)nullptr, (uint16_t*)nullptr);
    check_launch("dictionary count launch");
    MLEM_HIP(hipMemcpyAsync(nd.data(), ndb.p, sizeof(uint2) * nt, hipMemcpyDeviceToHost, s));
    MLEM_HIP(hipStreamSynchronize(s));
  }
  std::vector<uint4> d4(tl.size());
  uint64_t acc_a = 0, acc_g = 0;
  for (uint32_t i = 0; i <= nt; ++i) {
    d4[i] = make_uint4(tl[i], ptr[tl[i]], (uint32_t)acc_a | lead[i], (uint32_t)acc_g);
    if (i == nt) break;
    const uint32_t count = ptr[tl[i + 1]] - ptr[tl[i]];
    if (count <= T) acc_a += (lead[i] + count + 63) / 64 * 64;
    acc_g += (nd[i].x + NB - 1) / NB * NB;  // whole rounds of one slot per wave
  }
  if (acc_a + T > 0xFFFFFFFFull || acc_g > 0xFFFFFFFFull)
    raise(MLEM_EINVAL, "matrix too large for the dictionary format");
  free_dict(D);
  D.ntiles = nt;
  D.vk = VK;
  D.ndict = std::max<uint64_t>(acc_g, NB);
  D.nval = acc_a + T;  // tail: full-tile loads of the last tile stay in bounds
  const uint64_t vb = VK == kF32 ? 4 : 2;
  const uint64_t nslots = D.ndict / kWave;
  const uint64_t tail = (uint64_t)(NB / kWave) * EPT;  // rounded-up rounds of the last tile
  MLEM_HIP(hipMalloc(&D.tiles, sizeof(uint4) * d4.size()));
  MLEM_HIP(hipMalloc(&D.dict, 4ull * D.ndict));
  MLEM_HIP(hipMalloc(&D.dmeta, 4ull * (nslots + tail)));
  MLEM_HIP(hipMalloc(&D.dval, vb * D.nval));
  MLEM_HIP(hipMalloc(&D.dlix, 2ull * D.nval));
  // the tiles' kernels write everything but what follows the last tile
  if (acc_g < D.ndict) MLEM_HIP(hipMemsetAsync(D.dict, 0, 4ull * D.ndict, s));
  MLEM_HIP(hipMemsetAsync(D.dmeta + nslots, 0, 4ull * tail, s));
  MLEM_HIP(hipMemsetAsync(static_cast<char*>(D.dval) + vb * acc_a, 0, vb * T, s));
  MLEM_HIP(hipMemsetAsync(D.dlix + acc_a, 0, 2ull * T, s));
  MLEM_HIP(hipMemcpyAsync(D.tiles, d4.data(), sizeof(uint4) * d4.size(), hipMemcpyHostToDevice, s));
  if (nt) {
    hipLaunchKernelGGL((k_dict_rank<EB, VK>), dim3(nt), dim3(kBuild), 0, s, (const uint2*)el,
                       (const uint2*)nullptr, (const uint4*)D.tiles, (uint32_t)NB, page_bits,
                       (uint2*)nullptr, D.dict, D.dval, D.dlix);
    check_launch("dictionary fill launch");
  }
  const uint64_t per = kBlock / kWave;
  hipLaunchKernelGGL(k_dict_pack, dim3((unsigned)((nslots + per - 1) / per)), dim3(kBlock), 0, s,
                     D.dict, D.dmeta, nslots);
  check_launch("dictionary pack launch");
  MLEM_HIP(hipStreamSynchronize(s));
  D.nb = NB;
  D.ept = EPT;
  D.nested = nested;
}

template <int VK>
void build_dict_vk(const std::vector<uint32_t>& ptr, const uint2* el, uint32_t dim, int nb, int ept,
                   bool nested, DictFormat& D, hipStream_t s) {
  switch (nb * 1000 + ept) {
    case 256008: build_dict<256, 8, VK>(ptr, el, dim, nested, D, s); break;
    case 256016: build_dict<256, 16, VK>(ptr, el, dim, nested, D, s); break;
    case 256024: build_dict<256, 24, VK>(ptr, el, dim, nested, D, s); break;
    case 256032: build_dict<256, 32, VK>(ptr, el, dim, nested, D, s); break;
    case 256048: build_dict<256, 48, VK>(ptr, el, dim, nested, D, s); break;
    case 256064: build_dict<256, 64, VK>(ptr, el, dim, nested, D, s); break;
    case 512016: build_dict<512, 16, VK>(ptr, el, dim, nested, D, s); break;
    case 512024: build_dict<512, 24, VK>(ptr, el, dim, nested, D, s); break;
    case 512032: build_dict<512, 32, VK>(ptr, el, dim, nested, D, s); break;
    default: raise(MLEM_EINVAL, "unsupported dictionary tile size");
  }
}

}  // namespace

// Greedy partition of segments [0, n) into tiles of at most T elements and
// `maxseg` segments (one per lane); a segment longer than T forms a tile of
// its own.
std::vector<uint32_t> partition_tiles(const std::vector<uint32_t>& ptr, uint32_t T,
                                      uint32_t maxseg) {
  const uint32_t n = (uint32_t)ptr.size() - 1;
  std::vector<uint32_t> tiles{0};
  uint32_t s = 0;
  while (s < n) {
    uint32_t e = s;
    if (ptr[s + 1] - ptr[s] > T) {
      e = s + 1;
    } else {
      uint64_t cnt = 0;
      while (e < n && e - s < maxseg && cnt + (ptr[e + 1] - ptr[e]) <= T) {
        cnt += ptr[e + 1] - ptr[e];
        ++e;
      }
    }
    tiles.push_back(e);
    s = e;
  }
  return tiles;
}

void tile_lines(std::initializer_list<GatherSide*> sides, hipStream_t s) {
  constexpr uint32_t kSample = 64, T[3] = {16384, 8192, 2048}, kSeg[3] = {512, 512, 256};
  // the tiles of every size in the sampled large ones, one after the other: a
  // range of elements from each entry to the next, those in which `size` is set
  std::vector<uint2> range;
  std::vector<int> size;
  std::vector<size_t> end;  // of each side's entries
  std::vector<uint64_t> covered;
  for (GatherSide* g : sides) {
    const std::vector<uint32_t>& ptr = *g->ptr;
    const uint32_t n = (uint32_t)ptr.size() - 1;
    covered.push_back(0);
    for (uint32_t i = 0, s0 = 0, s1 = 0; i < kSample && s1 < n; ++i) {
      s0 = std::max(s1, (uint32_t)((uint64_t)n * i / kSample));
      s1 = s0 + 1;
      while (s1 < n && s1 - s0 < kSeg[0] && ptr[s1 + 1] - ptr[s0] <= T[0]) ++s1;
      covered.back() += ptr[s1] - ptr[s0];
      for (int k = 0; k < 3; ++k) {
        cut_nested(ptr, s0, s1, T[k], kSeg[k], [&](uint32_t b, uint32_t, uint32_t) {
          range.push_back(make_uint2(b, ptr[b]));
          size.push_back(k);
        });
        range.push_back(make_uint2(s1, ptr[s1]));
        size.push_back(-1);
      }
    }
    end.push_back(range.size());
  }
  if (range.empty()) return;
  struct Buf {
    void* p = nullptr;
    ~Buf() {
      if (p) (void)hipFree(p);
    }
  } buf;
  std::vector<uint2> counts(range.size());
  MLEM_HIP(hipMalloc(&buf.p, 2 * sizeof(uint2) * range.size()));
  uint2 *d_range = static_cast<uint2*>(buf.p), *d_counts = d_range + range.size();
  MLEM_HIP(hipMemcpyAsync(d_range, range.data(), sizeof(uint2) * range.size(),
                          hipMemcpyHostToDevice, s));
  size_t at = 0, i = 0;
  for (GatherSide* g : sides) {
    const size_t n = end[i++] - at;
    if (n > 1)
      hipLaunchKernelGGL((k_dict_rank<16, kF32>), dim3((unsigned)n - 1), dim3(kBuild), 0, s, g->el,
                         (const uint2*)(d_range + at), (const uint4*)nullptr, 0u,
                         page_bits_for(g->dim), d_counts + at, (uint32_t*)nullptr, (void*)nullptr,
                         (uint16_t*)nullptr);
    at += n;
  }
  check_launch("tile sample launch");
  MLEM_HIP(hipMemcpyAsync(counts.data(), d_counts, sizeof(uint2) * counts.size(),
                          hipMemcpyDeviceToHost, s));
  MLEM_HIP(hipStreamSynchronize(s));
  at = i = 0;
  for (GatherSide* g : sides) {
    for (; at < end[i]; ++at)
      if (size[at] >= 0) g->lines[(size_t)size[at]] += counts[at].y;
    if (covered[i])
      for (double& l : g->lines) l *= (double)g->ptr->back() / (double)covered[i];
    ++i;
  }
}

void ensure_dict(const std::vector<uint32_t>& ptr, const uint2* el, uint32_t dim, int nb, int ept,
                 bool nested, int vk, DictFormat& D, hipStream_t s) {
  if (D.nb == nb && D.ept == ept && D.nested == nested && D.vk == vk && D.tiles) return;
  switch (vk) {
    case kF32: build_dict_vk<kF32>(ptr, el, dim, nb, ept, nested, D, s); break;
    case kF16: build_dict_vk<kF16>(ptr, el, dim, nb, ept, nested, D, s); break;
    case kBF16: build_dict_vk<kBF16>(ptr, el, dim, nb, ept, nested, D, s); break;
    default: raise(MLEM_EINVAL, "unsupported value storage");
  }
}

void free_dict(DictFormat& d) {
  if (d.tiles) (void)hipFree(d.tiles);
  if (d.dict) (void)hipFree(d.dict);
  if (d.dmeta) (void)hipFree(d.dmeta);
  if (d.dval) (void)hipFree(d.dval);
  if (d.dlix) (void)hipFree(d.dlix);
  d = DictFormat();
}

}  // namespace mlem
