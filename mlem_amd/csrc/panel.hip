// panel.hip — products of the system matrix with blocks of W interleaved
// right-hand sides through its two-dimensional tiling (panels.hpp), gfx950.
//
// Both kernels run one 1024-lane workgroup per box, boxes launched largest
// first. They keep the rows of the dense operand that the elements pick from
// in LDS (forward: the box's slice of X, 128 KB at W = 32; backward: a chunk's
// rows of R), and every wave streams octets of pieces (voxels) from global
// memory (PanelFormat): L = W/4 lanes per piece, one per quad of frames, which
// read their 16 bytes of each element's operand row from LDS and add with fused
// multiply-adds. Elements are not staged and there is no barrier but the
// backward's two per chunk; D batches of 8 elements per piece are in flight.
//
// What bounds them: 16-byte LDS reads (8 cycles of a CU for 8 elements at
// W = 32; 120 of 128 bytes a cycle at best) together with the VALU (6
// instructions per step, 4 of them multiply-adds); at W = 16 and 32 the
// forward also writes 64 to 128 bytes per piece, twice the elements' bytes at
// W = 32. At 128x128x48 voxels and 1327104 lines (one kernel, us, before: the
// same boxes with elements staged in LDS chunk by chunk and 8 lanes per piece):
//     W          4         8        16         32
//   forward   570>324   570>443   710>597   846>824
//   backward  467>434   530>490   706>655  1158>985
//   row sums  250>124   254>158   238>260   443>440
//
// The slots of one row are added in box order by the callers' epilogue
// kernels, and a voxel's sum takes its chunks in order, so every result is
// deterministic.
#include <algorithm>
#include <chrono>
#include <cstring>
#include <memory>
#include <numeric>
#include <vector>

#include "internal.hpp"
#include "mlem.h"
#include "panels.hpp"

namespace mlem {
namespace {

constexpr int kBoxThreads = 1024;
constexpr uint32_t kWaves = kBoxThreads / 64;
constexpr uint32_t kOct = kFChunkPieces / 8;  // octets of a full forward chunk
static_assert(kFChunkPieces == kBoxThreads, "one packing thread per piece of a chunk");

void check_launch(const char* what) {
  hipError_t e = hipGetLastError();
  if (e != hipSuccess) raise(MLEM_EDEVICE, std::string(what) + ": " + hipGetErrorString(e));
}

template <class T>
void upload(T** dst, const std::vector<T>& v, hipStream_t s) {
  MLEM_HIP(hipMalloc(dst, std::max<size_t>(16, sizeof(T) * v.size())));
  if (!v.empty())
    MLEM_HIP(hipMemcpyAsync(*dst, v.data(), sizeof(T) * v.size(), hipMemcpyHostToDevice, s));
}

template <class T>
void dfree(T*& p) {
  if (p) (void)hipFree(p);
  p = nullptr;
}

// A piece (forward) or voxel (backward) belongs to L = W/4 lanes, one per quad
// of frames (16 bytes each). Its elements are added in batches of 8: element m
// of a batch goes to partial sum m / L of E = 8/L, and the E sums are added as a
// tree at the end, so the multiply-adds of a piece are E independent chains.
template <int W>
struct Quad {
  static_assert(W % 4 == 0 && W <= 32, "right-hand sides come in quads, at most 32");
  static constexpr uint32_t L = W / 4;              // lanes per piece (quads)
  static constexpr uint32_t E = 8 / L;              // partial sums; batch elements per lane
  static constexpr uint32_t P = 64 / L;             // pieces per wave
  static constexpr uint32_t kRow = 4 * W;           // bytes of one operand row
};

typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef uint32_t u32x2 __attribute__((ext_vector_type(2)));
typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));

// 16-byte store that does not allocate in the caches (partial sums are read
// once, by the next kernel).
__device__ __forceinline__ void store_nt(float4* p, const float4& v) {
  const f32x4 w = {v.x, v.y, v.z, v.w};
  __builtin_nontemporal_store(w, reinterpret_cast<f32x4*>(p));
}

__device__ __forceinline__ void fma4(float a, const float4& g, float4& acc) {
  acc.x = fmaf(a, g.x, acc.x);
  acc.y = fmaf(a, g.y, acc.y);
  acc.z = fmaf(a, g.z, acc.z);
  acc.w = fmaf(a, g.w, acc.w);
}

__device__ __forceinline__ float4 sum4(const float4& a, const float4& b) {
  return make_float4(a.x + b.x, a.y + b.y, a.z + b.z, a.w + b.w);
}

// The E partial sums of a piece, added pairwise: neighbours first.
template <uint32_t E>
__device__ __forceinline__ float4 tree(const float4 (&a)[E]) {
  if constexpr (E == 1) return a[0];
  else if constexpr (E == 2) return sum4(a[0], a[1]);
  else if constexpr (E == 4) return sum4(sum4(a[0], a[1]), sum4(a[2], a[3]));
  else return sum4(sum4(sum4(a[0], a[1]), sum4(a[2], a[3])), sum4(sum4(a[4], a[5]), sum4(a[6], a[7])));
}

// Value of lane m of this lane's run of L consecutive lanes (L = 1, 2, 4; runs
// start at multiples of L), by a quad permute. (All lanes are valid sources;
// bound_ctrl lets the compiler fold the move into the addition that uses it.)
constexpr int qperm(int a, int b, int c, int d) { return a | (b << 2) | (c << 4) | (d << 6); }
template <uint32_t L, uint32_t m>
__device__ __forceinline__ uint32_t bcast(uint32_t x) {
  static_assert(m < L && (L == 1 || L == 2 || L == 4), "runs of 1, 2 or 4 lanes");
  if constexpr (L == 1) {
    return x;
  } else if constexpr (L == 2) {
    return (uint32_t)__builtin_amdgcn_mov_dpp((int)x, qperm(m, m, 2 + m, 2 + m), 0xF, 0xF, true);
  } else {
    return (uint32_t)__builtin_amdgcn_mov_dpp((int)x, qperm(m, m, m, m), 0xF, 0xF, true);
  }
}
// The lower (0) or upper (1) quad of a run of 8 lanes, in both of its quads: row
// shifts by 4 lanes into the other quad's banks.
template <uint32_t half>
__device__ __forceinline__ uint32_t half_of(uint32_t x) {
  if constexpr (half == 0)
    return (uint32_t)__builtin_amdgcn_update_dpp((int)x, (int)x, 0x114, 0xF, 0xA, false);
  else
    return (uint32_t)__builtin_amdgcn_update_dpp((int)x, (int)x, 0x104, 0xF, 0x5, false);
}

// Steps m .. m+N-1 of a batch of 8 elements: element m is register m % E of
// lane m / E of the piece's lanes, or (strided) register m / L of lane m % L (at:
// byte offset of its operand row). Every lane reads its quad of the operand row
// from LDS, N reads in flight, and adds.
template <int W, bool kStrided, uint32_t m, uint32_t n, uint32_t N, uint32_t R>
__device__ __forceinline__ void step_reads(const uint32_t (&at)[R], const float (&val)[R],
                                           const char* __restrict__ op, float4 (&g)[N],
                                           float (&v)[N]) {
  if constexpr (n < N) {
    constexpr uint32_t L = 8 / R;
    constexpr uint32_t lane = kStrided ? (m + n) % L : (m + n) / R;
    constexpr uint32_t reg = kStrided ? (m + n) / L : (m + n) % R;
    g[n] = *reinterpret_cast<const float4*>(op + bcast<L, lane>(at[reg]));
    v[n] = __uint_as_float(bcast<L, lane>(__float_as_uint(val[reg])));
    step_reads<W, kStrided, m, n + 1, N>(at, val, op, g, v);
  }
}
// (W = 32: the run of 8 lanes is first turned into its two quads, 4 moves per
// batch, so that a step has the quad permutes of W = 16: 6 instead of 9 VALU
// instructions a step.)
template <int W, bool kStrided, uint32_t m, uint32_t N>
__device__ __forceinline__ void steps(const uint32_t (&at)[Quad<W>::E],
                                      const float (&val)[Quad<W>::E], const char* __restrict__ op,
                                      float4 (&acc)[Quad<W>::E]) {
  float4 g[N];
  float v[N];
  if constexpr (W == 32) {
    const uint32_t b = __float_as_uint(val[0]);
    const uint32_t at2[2] = {half_of<0>(at[0]), half_of<1>(at[0])};
    const float val2[2] = {__uint_as_float(half_of<0>(b)), __uint_as_float(half_of<1>(b))};
    step_reads<W, true, m, 0, N>(at2, val2, op, g, v);
  } else {
    step_reads<W, kStrided, m, 0, N>(at, val, op, g, v);
  }
#pragma unroll
  for (uint32_t n = 0; n < N; ++n) fma4(v[n], g[n], acc[(m + n) / Quad<W>::L]);
}

// Two quads (8 elements) of a piece in flight. For W >= 16 the piece's L lanes
// load E = 8/L elements each and broadcast them by DPP moves; for W <= 8 every
// lane loads both quads (the same 16 bytes for both lanes at W = 8). Loading
// whole quads at W = 16 and 32 repeats each of them for 4 and 8 lanes: no moves,
// but 465 against 393 and 775 against 723 us (at 128x128x48 voxels, 1327104
// lines, without the stores).
template <int W>
struct Batch {
  static constexpr uint32_t L = Quad<W>::L, E = Quad<W>::E;
  static constexpr bool kWhole = E >= 4;
  static constexpr uint32_t N = kWhole ? 8 : E;  // elements held by a lane
  float val[N];
  uint32_t idx[(N + 1) / 2];
  uint32_t slot;        // of this lane's piece
  uint32_t round;       // wave-uniform: number of the round among this wave's
  uint32_t base, most;  // wave-uniform: first quad of the batch, quads of the longest octet
  bool valid;           // wave-uniform

  __device__ __forceinline__ bool first() const { return base == 0; }
  __device__ __forceinline__ bool last() const { return base + 2 >= most; }

  // Loads quads `base` and base + 1 of the octet of n quads that starts at
  // quad q0; quads past its end come from the zeros at `zero`. i: piece within
  // the octet, q: lane of the piece.
  __device__ __forceinline__ void load(const float* __restrict__ v, const uint16_t* __restrict__ c,
                                       uint32_t q0, uint32_t n, uint32_t zero, uint32_t i,
                                       uint32_t q) {
    if constexpr (kWhole) {
#pragma unroll
      for (uint32_t h = 0; h < 2; ++h) {
        const size_t at = (size_t)(base + h < n ? q0 + base + h : zero) * 8 + i;
        const f32x4 a = reinterpret_cast<const f32x4*>(v)[at];
        const u32x2 d = reinterpret_cast<const u32x2*>(c)[at];
        val[4 * h] = a[0];
        val[4 * h + 1] = a[1];
        val[4 * h + 2] = a[2];
        val[4 * h + 3] = a[3];
        idx[2 * h] = d[0];
        idx[2 * h + 1] = d[1];
      }
    } else {
      const uint32_t k = base + q * E / 4;
      const size_t at = (size_t)(k < n ? q0 + k : zero) * 32 + i * 4 + q * E % 4;
      if constexpr (E == 1) {
        val[0] = v[at];
        idx[0] = c[at];
      } else {
        const float2 a = *reinterpret_cast<const float2*>(v + at);
        val[0] = a.x;
        val[1] = a.y;
        idx[0] = *reinterpret_cast<const uint32_t*>(c + at);
      }
    }
  }

  // Adds the batch to the piece's partial sums; the second quad only where an
  // octet of the wave has one.
  __device__ __forceinline__ void add(const char* __restrict__ op, float4 (&acc)[E]) const {
    uint32_t at[N];
#pragma unroll
    for (uint32_t j = 0; j < N; ++j) {
      const uint32_t x = N == 1 ? idx[0] : (j & 1u) ? idx[j / 2] >> 16 : idx[j / 2] & 0xFFFFu;
      at[j] = x * Quad<W>::kRow;
    }
    const bool both = base + 2 <= most;
    if constexpr (kWhole) {
      whole<0>(at, op, acc);
      if (both) whole<1>(at, op, acc);
    } else if (both) {
      steps<W, false, 0, 4>(at, val, op, acc);
      steps<W, false, 4, 4>(at, val, op, acc);
    } else {
      steps<W, false, 0, 4>(at, val, op, acc);
    }
  }

 private:
  template <uint32_t h>
  __device__ __forceinline__ void whole(const uint32_t (&at)[N], const char* __restrict__ op,
                                        float4 (&acc)[E]) const {
    float4 g[4];
#pragma unroll
    for (uint32_t j = 0; j < 4; ++j) g[j] = *reinterpret_cast<const float4*>(op + at[4 * h + j]);
#pragma unroll
    for (uint32_t j = 0; j < 4; ++j) fma4(val[4 * h + j], g[j], acc[(4 * h + j) / L]);
  }
};

// Batches in flight per wave of the forward. A store is waited for in order with
// the loads, so W = 32 holds 8 (3: 897 us, 5: 836, 8: 824, 12 no better); W = 16
// holds 2, which leaves registers for two workgroups per CU (64 VGPRs, 597 us;
// one workgroup with 3 in flight: 642); W = 4 and 8 have one workgroup per CU for
// their LDS, and 5 in flight are no faster than 3.
template <int W>
constexpr uint32_t kDepth = W == 32 ? 8 : W == 16 ? 2 : 3;

// Quads of the longest octet of a wave's round: the first lane's (octets are in
// order of length).
__device__ __forceinline__ uint32_t longest(uint32_t quads) {
  return __builtin_amdgcn_readfirstlane(quads);
}

// A piece's sums: whole 128-byte lines go past the caches (read once, by the
// next kernel); shorter runs are merged into lines in L2.
template <int W>
__device__ __forceinline__ void store_part(float4* p, const float4& v) {
  if constexpr (W == 32)
    store_nt(p, v);
  else
    *p = v;
}

// Forward: part[s * W + f] = sum over piece s of a * X[(c0 + col) * W + f] for
// the pieces of box border[blockIdx.x]; X in panel order. A round is 64 / L
// consecutive pieces (K octets) for one wave.
//   W >= 16: wave w takes rounds w, w + 16, ... of the box and stores every
//   piece's sums to its slot.
//   W <= 8: the waves go through the box group by group (kGroup chunks, two
//   rounds per wave, the second in reverse order: their lengths add up to about
//   the same), collect the sums in LDS and store each group's slots as one run;
//   two buffers, one barrier per group. (16- and 32-byte runs stored one by
//   one took 160 us of 430 at W = 4 and 220 of 550 at W = 8. Collecting 64-byte
//   runs, W = 16, leaves room for one workgroup per CU: 682 against 597 us.)
template <int W>
__global__ __launch_bounds__(kBoxThreads) __attribute__((amdgpu_waves_per_eu(W == 16 ? 8 : 4, W == 16 ? 8 : 4))) void k_box_fwd(
    const uint32_t* __restrict__ pstart, const uint32_t* __restrict__ border,
    const uint32_t* __restrict__ pfchunk, const uint32_t* __restrict__ cpiece,
    const uint32_t* __restrict__ fquad, const uint32_t* __restrict__ fpiece,
    const float* __restrict__ fval, const uint16_t* __restrict__ fcol, uint32_t zero,
    const float* __restrict__ X, float* __restrict__ part) {
  using Q = Quad<W>;
  constexpr uint32_t L = Q::L, E = Q::E, K = Q::P / 8, D = kDepth<W>;
  constexpr uint32_t XJ = kBoxVox * L / kBoxThreads;
  constexpr bool kCollect = W <= 8;
  constexpr uint32_t kGroup = W == 4 ? 2 : 1;                 // chunks per group
  constexpr uint32_t kPart = kCollect ? kGroup * kFChunkPieces * L : 1;  // quads of a group
  static_assert(!kCollect || kGroup * kOct == 2 * kWaves * K, "two rounds per wave and group");
  __shared__ float4 xs[(kBoxVox + 1) * L];  // one more row, of zeros
  __shared__ float4 ys[2][kPart];
  const uint32_t box = border[blockIdx.x];
  const uint32_t c0 = pstart[box], nv = pstart[box + 1] - c0;
  const uint32_t k0 = pfchunk[box], nk = pfchunk[box + 1] - k0;
  const uint32_t groups = (nk + kGroup - 1) / kGroup;
  const uint32_t t = threadIdx.x, lane = t % 64, q = lane % L, grp = lane / L;
  const uint32_t wave = __builtin_amdgcn_readfirstlane(t / 64);
  {  // the box's slice of X
    const float4* __restrict__ X4 = reinterpret_cast<const float4*>(X) + (size_t)c0 * L;
    const uint32_t n = nv * L;
    float4 xr[XJ];
#pragma unroll
    for (uint32_t j = 0; j < XJ; ++j) xr[j] = X4[min(t + j * kBoxThreads, n - 1)];
#pragma unroll
    for (uint32_t j = 0; j < XJ; ++j) xs[t + j * kBoxThreads] = xr[j];
    if (t < L) xs[kBoxVox * L + t] = make_float4(0.f, 0.f, 0.f, 0.f);
  }
  __syncthreads();
  const char* __restrict__ op = reinterpret_cast<const char*>(xs) + 16 * q;
  float4* __restrict__ part4 = reinterpret_cast<float4*>(part);

  // this wave's rounds: the one whose batches are being loaded, and the next
  // one looked up
  const uint32_t rounds = kCollect ? 2 * groups : nk * (kOct / K / kWaves);
  uint32_t r = 0, base = 0, most = 0, q0 = 0, nq = 0, slot = 0, lq0 = 0, lq1 = 0, lslot = 0;
  auto look = [&](uint32_t i) __attribute__((always_inline)) {
    uint32_t o;  // this lane's octet of round i, counted from the box's first
    if constexpr (kCollect) {
      const uint32_t w = (i & 1u) ? kWaves - 1 - wave : wave;
      o = (i * kWaves + w) * K + grp / 8;
    } else {
      o = (i * kWaves + wave) * K + grp / 8;
    }
    const bool in = o < nk * kOct;  // (an odd chunk at the end of the groups)
    const size_t at = (size_t)k0 * kOct + (in ? o : 0);
    lq0 = fquad[at];
    lq1 = in ? fquad[at + 1] : lq0;
    lslot = fpiece[at * 8 + grp % 8];
  };
  auto advance = [&]() __attribute__((always_inline)) {  // to the next round that has a quad
    while (r < rounds) {
      q0 = lq0;
      nq = lq1 - lq0;
      slot = lslot;
      look(min(r + 1, rounds - 1));
      most = longest(nq);
      if (most) break;
      ++r;
    }
    base = 0;
  };
  auto issue = [&](Batch<W>& e) __attribute__((always_inline)) {
    e.valid = r < rounds;
    if (!e.valid) return;
    e.slot = slot;
    e.round = r;
    e.base = base;
    e.most = most;
    e.load(fval, fcol, q0, nq, zero, grp % 8, q);
    base += 2;
    if (base >= most) {
      ++r;
      advance();
    }
  };
  // W <= 8: all of group g's sums are in ys[g % 2]; store them
  uint32_t done = 0, gp0 = kCollect && nk ? cpiece[k0] : 0;  // gp0: first piece of group `done`
  auto finish = [&]() __attribute__((always_inline)) {
    const uint32_t end = cpiece[k0 + min((done + 1) * kGroup, nk)];
    __syncthreads();
    const float4* __restrict__ y = ys[done % 2];
    for (uint32_t i = t; i < (end - gp0) * L; i += kBoxThreads) part4[(size_t)gp0 * L + i] = y[i];
    gp0 = end;
    ++done;
  };
  if (nk) {
    look(0);
    advance();
  } else {
    r = rounds;
  }
  float4 acc[E];
  Batch<W> qu[D];
#pragma unroll
  for (uint32_t d = 0; d < D; ++d) issue(qu[d]);
  for (bool more = true; more;) {
#pragma unroll
    for (uint32_t d = 0; d < D; ++d) {
      if (!qu[d].valid) {  // batches are issued in order: none follows
        more = false;
        break;
      }
      if constexpr (kCollect)
        while (done < qu[d].round / 2) finish();
      if (qu[d].first())
#pragma unroll
        for (uint32_t j = 0; j < E; ++j) acc[j] = make_float4(0.f, 0.f, 0.f, 0.f);
      qu[d].add(op, acc);
      if (qu[d].last() && qu[d].slot != ~0u) {
        const float4 y = tree<E>(acc);
        if constexpr (kCollect)
          ys[done % 2][(qu[d].slot - gp0) * L + q] = y;
        else
          store_part<W>(part4 + (size_t)qu[d].slot * L + q, y);
      }
      issue(qu[d]);
    }
  }
  if constexpr (kCollect)
    while (done < groups) finish();
}

// Backward: U[(c0 + v) * W + f] = sum over the box's elements of voxel v of
// a * R[row * W + f] (R in device row order), for box border[blockIdx.x].
// Every L lanes own V = L voxels, whose partial sums stay in registers for the
// whole box; per chunk they add those voxels' staged elements in order. While a
// chunk is reduced, the next chunk's runs of R, elements and voxel offsets
// are loaded into registers, and the rows of the one after it.
template <int W>
__global__ __launch_bounds__(kBoxThreads) __attribute__((amdgpu_waves_per_eu(4, 4))) void k_box_bwd(
    const uint32_t* __restrict__ pstart, const uint32_t* __restrict__ border,
    const uint32_t* __restrict__ pchunk, const uint2* __restrict__ chunk,
    const uint16_t* __restrict__ boff, const uint32_t* __restrict__ brow,
    const uint16_t* __restrict__ bpc, const float* __restrict__ bval,
    const float* __restrict__ R, float* __restrict__ U) {
  using Q = Quad<W>;
  constexpr uint32_t L = Q::L, E = Q::E, V = L;
  constexpr uint32_t kRq = (kChunkPieces * L + kBoxThreads - 1) / kBoxThreads;  // R quads
  static_assert(kChunkElems == 8 * kBoxThreads && kBoxVox == kBoxThreads && kBAlign % 8 == 0,
                "staging: eight elements per thread, 16-byte aligned chunks");
  constexpr uint32_t kZero = kRq * kBoxThreads / L;  // a row of zeros: past a voxel's end
  __shared__ float4 rs[kRq * kBoxThreads + L];
  __shared__ float4 sval4[kChunkElems / 4];
  __shared__ uint4 spc4[kChunkElems / 8];
  const float* __restrict__ sval = reinterpret_cast<const float*>(sval4);
  const uint16_t* __restrict__ spc = reinterpret_cast<const uint16_t*>(spc4);
  __shared__ uint16_t soff[kBoxVox + 1];  // soff[v + 1]: end of voxel v's elements
  const uint32_t box = border[blockIdx.x];
  const uint32_t c0 = pstart[box], nv = pstart[box + 1] - c0;
  const uint32_t t = threadIdx.x, q = t % L;
  // Voxels are numbered in octets whose 8 positions hold one voxel of every
  // eighth of the box by element count (panels.hpp). The waves are cut into E
  // classes of which class k takes positions k, 2E-1-k, 2E+k, ... of its
  // octets: in lockstep, a wave's lanes then work on voxels of about the same
  // count, and the classes on about the same sum.
  const uint32_t wave = t / 64, cls = wave / (kWaves / E);
  const uint32_t octet = (wave % (kWaves / E)) * (64 / L) + (t % 64) / L;
  auto voxel = [&](uint32_t j) { return 8 * octet + j * E + ((j & 1u) ? E - 1 - cls : cls); };
  const uint32_t k0 = pchunk[box], k1 = pchunk[box + 1];
  const float4* __restrict__ R4 = reinterpret_cast<const float4*>(R);
  const char* __restrict__ op = reinterpret_cast<const char*>(rs) + 16 * q;
  // vector registers (not arrays), so they are never placed in memory
  typedef float rq_t __attribute__((ext_vector_type(4 * kRq)));
  typedef uint32_t rr_t __attribute__((ext_vector_type(kRq)));
  rq_t rR;
  rr_t rrow;
  f32x4 rva, rvb;
  u32x4 rp;
  uint32_t rend = 0;
  auto rows_of = [&](uint32_t k) __attribute__((always_inline)) {  // rows of chunk k's R quads
    const uint2 a = chunk[k], b = chunk[k + 1];
    const uint32_t nq = (b.x - a.x) * L;
#pragma unroll
    for (uint32_t j = 0; j < kRq; ++j) rrow[j] = brow[a.x + min(t + j * kBoxThreads, nq - 1) / L];
  };
  auto fetch = [&](uint32_t k) __attribute__((always_inline)) {  // chunk k (its rows in rrow)
    const uint2 a = chunk[k];
#pragma unroll
    for (uint32_t j = 0; j < kRq; ++j) {
      const float4 g = R4[(size_t)rrow[j] * L + (t + j * kBoxThreads) % L];
      rR[4 * j] = g.x;
      rR[4 * j + 1] = g.y;
      rR[4 * j + 2] = g.z;
      rR[4 * j + 3] = g.w;
    }
    // elements 8t .. 8t+7 of the chunk (the arrays end with a chunk of
    // zeros); streamed once: non-temporal
    rva = __builtin_nontemporal_load(reinterpret_cast<const f32x4*>(bval + a.y) + 2 * t);
    rvb = __builtin_nontemporal_load(reinterpret_cast<const f32x4*>(bval + a.y) + 2 * t + 1);
    rp = __builtin_nontemporal_load(reinterpret_cast<const u32x4*>(bpc + a.y) + t);
    rend = boff[(size_t)k * (kBoxVox + 1) + t + 1];
  };
  if (k0 < k1) {
    rows_of(k0);
    fetch(k0);
    if (k0 + 1 < k1) rows_of(k0 + 1);
  }
  if (t == 0) soff[0] = 0;
  if (t < L) rs[kRq * kBoxThreads + t] = make_float4(0.f, 0.f, 0.f, 0.f);
  float4 acc[V][E];
#pragma unroll
  for (uint32_t j = 0; j < V; ++j)
#pragma unroll
    for (uint32_t e = 0; e < E; ++e) acc[j][e] = make_float4(0.f, 0.f, 0.f, 0.f);
  for (uint32_t k = k0; k < k1; ++k) {
    __syncthreads();  // the previous chunk's readers are done with the LDS arrays
#pragma unroll
    for (uint32_t j = 0; j < kRq; ++j)
      rs[t + j * kBoxThreads] = make_float4(rR[4 * j], rR[4 * j + 1], rR[4 * j + 2], rR[4 * j + 3]);
    sval4[2 * t] = make_float4(rva.x, rva.y, rva.z, rva.w);
    sval4[2 * t + 1] = make_float4(rvb.x, rvb.y, rvb.z, rvb.w);
    spc4[t] = make_uint4(rp.x, rp.y, rp.z, rp.w);
    soff[t + 1] = (uint16_t)rend;
    __syncthreads();
    if (k + 1 < k1) {
      fetch(k + 1);
      if (k + 2 < k1) rows_of(k + 2);
    }
#pragma unroll
    for (uint32_t j = 0; j < V; ++j) {
      const uint32_t v = voxel(j), e = soff[v + 1];
      for (uint32_t i = soff[v]; i < e; i += 8) {
        uint32_t at[E];
        float a[E];
#pragma unroll
        for (uint32_t n = 0; n < E; ++n) {
          const uint32_t my = i + n * L + q, ic = min(my, e - 1);
          const uint32_t pc = spc[ic];
          const float w = sval[ic];
          at[n] = (my < e ? pc : kZero) * Q::kRow;
          a[n] = my < e ? w : 0.f;
        }
        steps<W, true, 0, 4>(at, a, op, acc[j]);
        // the second four only where a voxel of the wave has them (985 us at
        // W = 32; always 8 steps: 1175, pairs: 1071; 8 reads in flight: 1190)
        if (__builtin_amdgcn_ballot_w64(i + 4 < e)) steps<W, true, 4, 4>(at, a, op, acc[j]);
      }
    }
  }
  float4* __restrict__ U4 = reinterpret_cast<float4*>(U);
#pragma unroll
  for (uint32_t j = 0; j < V; ++j)
    if (voxel(j) < nv) U4[(size_t)(c0 + voxel(j)) * L + q] = tree<E>(acc[j]);
}

// ---- octets of the forward chunks, built from the host tiling ----------------
// One workgroup per chunk, one lane per piece. fill = 0: quads of the chunk into
// nquads; fill = 1: its octets' first quads (base = the chunk's first quad), the
// pieces' slots (numbered in row order) and the elements (the arrays hold zeros
// and index kBoxVox elsewhere).
__global__ __launch_bounds__(kBoxThreads) void k_pack_fwd(
    int fill, const uint32_t* __restrict__ cpiece, const uint32_t* __restrict__ base,
    const uint32_t* __restrict__ fseg, const uint32_t* __restrict__ fslot,
    const float* __restrict__ hval, const uint16_t* __restrict__ hcol,
    uint32_t* __restrict__ nquads, uint32_t* __restrict__ fquad, uint32_t* __restrict__ fpiece,
    uint32_t* __restrict__ rowpiece, float* __restrict__ fval, uint16_t* __restrict__ fcol) {
  __shared__ uint32_t len[kBoxThreads], slot[kBoxThreads], first[kOct + 1];
  const uint32_t w = blockIdx.x, t = threadIdx.x;
  const uint32_t p0 = cpiece[w], n = cpiece[w + 1] - p0;
  const uint32_t b = t < n ? fseg[p0 + t] : 0u;
  const uint32_t l = t < n ? fseg[p0 + t + 1] - b : 0u;
  len[t] = l;
  slot[t] = t < n ? fslot[p0 + t] : ~0u;
  __syncthreads();
  if (t < kOct) {
    uint32_t m = 0;
    for (uint32_t i = 0; i < 8; ++i) m = max(m, len[8 * t + i]);
    first[t + 1] = (m + 3) / 4;
  }
  if (t == 0) first[0] = fill ? base[w] : 0u;
  __syncthreads();
  if (t == 0)
    for (uint32_t o = 0; o < kOct; ++o) first[o + 1] += first[o];
  __syncthreads();
  if (!fill) {
    if (t == 0) nquads[w] = first[kOct];
    return;
  }
  const size_t o0 = (size_t)w * kOct;
  if (t < kOct) fquad[o0 + t] = first[t];
  if (t == 0 && w + 1 == gridDim.x) fquad[o0 + kOct] = first[kOct];
  // slots in row order inside the chunk: the rank of the row-major slot
  uint32_t rank = 0;
  for (uint32_t i = 0; i < n; ++i) rank += slot[i] < slot[t] ? 1u : 0u;
  fpiece[8 * o0 + t] = t < n ? p0 + rank : ~0u;
  if (t < n) rowpiece[slot[t]] = p0 + rank;
  const uint32_t q = first[t / 8];
  for (uint32_t k = 0; k < l; ++k) {
    const size_t at = (size_t)(q + k / 4) * 32 + (t % 8) * 4 + k % 4;
    fval[at] = hval[b + k];
    fcol[at] = hcol[b + k];
  }
}

// Zero values and index kBoxVox in every position of q quads.
__global__ __launch_bounds__(256) void k_clear_quads(float4* __restrict__ val,
                                                     uint2* __restrict__ idx, uint64_t q) {
  constexpr uint32_t z = kBoxVox | (kBoxVox << 16);
  for (uint64_t i = blockIdx.x * 256ull + threadIdx.x; i < 8 * q; i += gridDim.x * 256ull) {
    val[i] = make_float4(0.f, 0.f, 0.f, 0.f);
    idx[i] = make_uint2(z, z);
  }
}

// Element arrays of `quads` quads (and two of zeros) for chunks of the given
// sizes: the chunks' first quads into dbase.
uint32_t alloc_quads(const std::vector<uint32_t>& nq, uint32_t** dbase, float** val,
                     uint16_t** idx, hipStream_t s) {
  std::vector<uint32_t> base(nq.size() + 1, 0);
  uint64_t q = 0;
  for (size_t i = 0; i < nq.size(); ++i) {
    base[i] = (uint32_t)q;
    q += nq[i];
  }
  if (q + 2 > 0x7FFFFFFFull) raise(MLEM_EINVAL, "matrix tiling: too many elements");
  base[nq.size()] = (uint32_t)q;
  upload(dbase, base, s);
  MLEM_HIP(hipMalloc(val, 128ull * (q + 2)));
  MLEM_HIP(hipMalloc(idx, 64ull * (q + 2)));
  hipLaunchKernelGGL(k_clear_quads, dim3(4096), dim3(256), 0, s, (float4*)*val, (uint2*)*idx, q + 2);
  check_launch("tiling clear launch");
  MLEM_HIP(hipStreamSynchronize(s));  // base goes out of scope
  return (uint32_t)q;
}

}  // namespace

PanelFormat::~PanelFormat() {
  dfree(pc_of_file);
  dfree(pc_of_dev);
  dfree(dev_of_pc);
  dfree(norm);
  dfree(pstart);
  dfree(border);
  dfree(rowslot);
  dfree(rowpiece);
  dfree(pfchunk);
  dfree(cpiece);
  dfree(fquad);
  dfree(fpiece);
  dfree(fval);
  dfree(fcol);
  dfree(pchunk);
  dfree(chunk);
  dfree(brow);
  dfree(boff);
  dfree(bpc);
  dfree(bval);
  dfree(colslot);
}

const PanelFormat& ensure_panels(DevMatrix& m) {
  if (m.panels) return *m.panels;
  if (m.streamed || !m.csr) raise(MLEM_EINVAL, "the tiled product needs a matrix held in HBM");
  if (m.vk != kF32) raise(MLEM_EINVAL, "the tiled product needs fp32 matrix values");
  auto t0 = std::chrono::steady_clock::now();
  hipStream_t s = m.stream;
  // device-order CSR and row pointers, device column of each file column
  std::vector<uint32_t> csr2(2 * m.nnz), rowptr((size_t)m.rows + 1), colmap(m.cols);
  std::vector<float> norm(m.cols);
  if (m.nnz)
    MLEM_HIP(hipMemcpyAsync(csr2.data(), m.csr, 8ull * m.nnz, hipMemcpyDeviceToHost, s));
  MLEM_HIP(hipMemcpyAsync(rowptr.data(), m.rowptr, 4ull * (m.rows + 1), hipMemcpyDeviceToHost, s));
  if (m.colmap && m.cols)
    MLEM_HIP(hipMemcpyAsync(colmap.data(), m.colmap, 4ull * m.cols, hipMemcpyDeviceToHost, s));
  if (m.cols)
    MLEM_HIP(hipMemcpyAsync(norm.data(), m.norm, 4ull * m.cols, hipMemcpyDeviceToHost, s));
  MLEM_HIP(hipStreamSynchronize(s));
  if (!m.colmap) std::iota(colmap.begin(), colmap.end(), 0u);

  std::vector<uint32_t> pc_of_file, pstart;
  uint32_t boxgrid[3] = {0, 0, 0};
  const bool has_grid = (uint64_t)m.grid[0] * m.grid[1] * m.grid[2] == m.cols && m.cols;
  std::vector<uint32_t> count_dev(m.cols, 0), count_file(m.cols);
  if (m.csc) {
    download_pointers(m, s);
    for (uint32_t c = 0; c < m.cols; ++c) count_dev[c] = m.h_colptr[c + 1] - m.h_colptr[c];
  } else {
    for (uint64_t k = 0; k < m.nnz; ++k) count_dev[csr2[2 * k]]++;
  }
  for (uint32_t c = 0; c < m.cols; ++c) count_file[c] = count_dev[colmap[c]];
  panel_order(m.cols, has_grid ? m.grid : nullptr, count_file.data(), &pc_of_file, &pstart,
              boxgrid);
  std::vector<uint32_t> pc_of_dev(m.cols), dev_of_pc(m.cols);
  for (uint32_t c = 0; c < m.cols; ++c) pc_of_dev[colmap[c]] = pc_of_file[c];
  for (uint32_t d = 0; d < m.cols; ++d) dev_of_pc[pc_of_dev[d]] = d;
  std::vector<float> pnorm(m.cols);
  for (uint32_t c = 0; c < m.cols; ++c) pnorm[c] = norm[dev_of_pc[c]];

  HostPanels H;
  try {
    build_host_panels(m.rows, m.cols, m.nnz, rowptr.data(), csr2.data(), pc_of_dev, pstart,
                      boxgrid, 0, &H);
  } catch (const std::invalid_argument& e) {
    raise(MLEM_EINVAL, std::string("matrix tiling: ") + e.what());
  }
  std::vector<uint32_t>().swap(csr2);
  const uint32_t nchunks = (uint32_t)H.chunk_piece.size() - 1;
  const uint32_t nfchunks = (uint32_t)H.fchunk_piece.size() - 1;
  std::vector<uint2> chunk((size_t)nchunks + 1);
  for (uint32_t k = 0; k <= nchunks; ++k) chunk[k] = make_uint2(H.chunk_piece[k], H.chunk_elem[k]);
  std::vector<uint32_t> colslot((size_t)m.cols + 1);
  std::iota(colslot.begin(), colslot.end(), 0u);

  std::unique_ptr<PanelFormat> P(new PanelFormat());
  P->rows = m.rows;
  P->cols = m.cols;
  P->npanels = H.npanels;
  P->nseg = H.fseg.size() - 1;
  upload(&P->pc_of_file, pc_of_file, s);
  upload(&P->pc_of_dev, pc_of_dev, s);
  upload(&P->dev_of_pc, dev_of_pc, s);
  upload(&P->norm, pnorm, s);
  upload(&P->pstart, H.pstart, s);
  upload(&P->border, H.border, s);
  upload(&P->rowslot, H.rowslot, s);
  upload(&P->pfchunk, H.pfchunk, s);
  upload(&P->cpiece, H.fchunk_piece, s);
  upload(&P->brow, H.brow, s);
  upload(&P->pchunk, H.pchunk, s);
  upload(&P->chunk, chunk, s);
  upload(&P->boff, H.boff, s);
  upload(&P->bpc, H.bpc, s);
  upload(&P->bval, H.bval, s);
  upload(&P->colslot, colslot, s);
  MLEM_HIP(hipMalloc(&P->rowpiece, 4 * std::max<uint64_t>(P->nseg, 4)));
  MLEM_HIP(hipMalloc(&P->fquad, 4ull * (nfchunks * (uint64_t)kOct + 1)));
  MLEM_HIP(hipMalloc(&P->fpiece, 4ull * std::max<uint64_t>(nfchunks * (uint64_t)kFChunkPieces, 4)));

  struct Temp {  // the host tiling's forward arrays on the device, for the packing only
    uint32_t *seg = nullptr, *slot = nullptr, *base = nullptr, *nq = nullptr;
    float* val = nullptr;
    uint16_t* col = nullptr;
    ~Temp() {
      dfree(seg);
      dfree(slot);
      dfree(base);
      dfree(nq);
      dfree(val);
      dfree(col);
    }
  } T;
  std::vector<uint32_t> nq(nfchunks);
  upload(&T.seg, H.fseg, s);
  upload(&T.slot, H.fslot, s);
  upload(&T.val, H.fval, s);
  upload(&T.col, H.fcol, s);
  MLEM_HIP(hipMalloc(&T.nq, 4ull * std::max(nfchunks, 4u)));
  auto pack_fwd = [&](int fill) {
    if (nfchunks)
      hipLaunchKernelGGL(k_pack_fwd, dim3(nfchunks), dim3(kBoxThreads), 0, s, fill, P->cpiece,
                         T.base, T.seg, T.slot, T.val, T.col, T.nq, P->fquad, P->fpiece,
                         P->rowpiece, P->fval, P->fcol);
    check_launch("forward tiling launch");
  };
  pack_fwd(0);
  if (nfchunks)
    MLEM_HIP(hipMemcpyAsync(nq.data(), T.nq, 4ull * nfchunks, hipMemcpyDeviceToHost, s));
  MLEM_HIP(hipStreamSynchronize(s));
  P->fzero = alloc_quads(nq, &T.base, &P->fval, &P->fcol, s);
  pack_fwd(1);
  MLEM_HIP(hipStreamSynchronize(s));  // host vectors go out of scope
  P->build_seconds = std::chrono::duration<double>(std::chrono::steady_clock::now() - t0).count();
  m.panels = P.release();
  return *m.panels;
}

void free_panels(DevMatrix& m) {
  delete m.panels;
  m.panels = nullptr;
}

template <int W>
void launch_panel_fwd(const PanelFormat& P, const float* X, float* part, hipStream_t s) {
  if (!P.npanels) return;
  hipLaunchKernelGGL((k_box_fwd<W>), dim3(P.npanels), dim3(kBoxThreads), 0, s, P.pstart, P.border,
                     P.pfchunk, P.cpiece, P.fquad, P.fpiece, P.fval, P.fcol, P.fzero, X, part);
  check_launch("tiled forward launch");
}

template <int W>
void launch_panel_bwd(const PanelFormat& P, const float* R, float* U, hipStream_t s) {
  if (!P.npanels) return;
  hipLaunchKernelGGL((k_box_bwd<W>), dim3(P.npanels), dim3(kBoxThreads), 0, s, P.pstart, P.border,
                     P.pchunk, P.chunk, P.boff, P.brow, P.bpc, P.bval, R, U);
  check_launch("tiled backward launch");
}

#define MLEM_PANEL_WIDTH(W)                                                                \
  template void launch_panel_fwd<W>(const PanelFormat&, const float*, float*, hipStream_t); \
  template void launch_panel_bwd<W>(const PanelFormat&, const float*, float*, hipStream_t);
MLEM_PANEL_WIDTH(4)
MLEM_PANEL_WIDTH(8)
MLEM_PANEL_WIDTH(16)
MLEM_PANEL_WIDTH(32)
#undef MLEM_PANEL_WIDTH

}  // namespace mlem
