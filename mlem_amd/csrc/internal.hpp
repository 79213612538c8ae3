// internal.hpp — device-side matrix/state structures and kernel launchers
// shared by the C ABI (api.cpp) and the kernels (kernels.hip).
#pragma once
#include <hip/hip_runtime.h>

#include <array>
#include <cstdint>
#include <functional>
#include <new>
#include <stdexcept>
#include <string>
#include <vector>

#include "csr4.hpp"

namespace mlem {

// Error raised inside the library; the C ABI converts it to a status code.
struct ApiError {
  int code;
  std::string msg;
};

// Every kernel runs in the fp32 mode of the reference driver, which sets
// flush-to-zero but not denormals-are-zero (mlem_seq/seqcsr4mlem.cpp:194):
// subnormal inputs are used as they are, subnormal results become zero. The
// code is built with -fdenormal-fp-math-f32=preserve-sign,ieee (MODE register
// FP32 denormal field 1, "flush outputs").
//
// fp32 division goes through div_rn: the compiler's own fp32 division would
// switch to full denormals for its fused steps and then write field 0
// (inputs flushed as well) for the rest of the kernel. div_rn divides in
// fp64 instead (fp64 keeps denormals, no mode switch): the quotient of two
// fp32 values rounded to fp64 and then to fp32 is the correctly rounded fp32
// quotient, since 53 >= 2*24 + 2. As x86 under FTZ, a quotient is flushed to
// zero when it is tiny after rounding, i.e. when its rounding to 24 bits with
// unbounded exponent is below 2^-126, which is |a/b| < 2^-126 - 2^-151.
__device__ __forceinline__ float div_rn(float a, float b) {
  const double q = (double)a / (double)b;
  constexpr double kTiny = 0x1.ffffffp-127;  // 2^-126 - 2^-151
  return (float)(__builtin_fabs(q) < kTiny ? __builtin_copysign(0.0, q) : q);
}

[[noreturn]] void raise(int code, const std::string& msg);
void hip_check(hipError_t e, const char* what);
#define MLEM_HIP(call) ::mlem::hip_check((call), #call)

// Thread-local message of the last failing C-ABI call (api.cpp).
void set_error(const std::string& msg);
void clear_error();

// Run f and translate exceptions into a C-ABI status code.
template <class F>
int guarded(F&& f) {
  try {
    f();
    clear_error();
    return 0;
  } catch (const ApiError& e) {
    set_error(e.msg);
    return e.code;
  } catch (const Csr4Error& e) {
    set_error(e.msg);
    return e.code;
  } catch (const std::bad_alloc&) {
    set_error("host allocation failed");
    return -4;
  } catch (const std::exception& e) {
    set_error(e.what());
    return -1;
  } catch (...) {
    set_error("unknown error");
    return -1;
  }
}

// FAST-mode kernel family of a projection. kDict and kDictWide are the same
// dictionary tiles run by 256-lane and 512-lane blocks.
enum KernelKind { kGroups = 0, kTiles = 1, kDict = 2, kDictWide = 3 };
inline bool is_dict(int kind) { return kind == kDict || kind == kDictWide; }
inline int dict_lanes(int kind) { return kind == kDictWide ? 512 : 256; }

// Dictionary-tile storage of one projection (built on the device at load
// time for `nb` lanes per block and `ept` elements per lane: tiles of at most
// nb*ept elements and nb segments; 0 = not built). Nested tiles are cut inside
// the tiles of 16384 elements and 512 segments and start with the 0 to 3 zero
// elements that give every element the place modulo 4 it has in the larger
// tile: a segment's sum is taken in aligned quads, so it is the same bit for
// bit with either tile size.
struct DictFormat {
  int nb = 0;
  int ept = 0;
  int vk = 0;                 // value storage (ValueKind): fp32, fp16, bf16
  uint32_t ntiles = 0;
  bool nested = false;        // tiles inside the 16384-element ones (see below)
  uint4* tiles = nullptr;     // [ntiles+1] {first segment, first element, element
                              //  start (a multiple of 64) + leading zero elements,
                              //  first dict word}
  uint32_t* dict = nullptr;   // distinct gather indices, sorted per tile, in
                              //  64-word slots of 64 entries, nb/64 per round
  uint32_t* dmeta = nullptr;  // per slot: first index | 0x80000000 if 32-bit
  void* dval = nullptr;       // element values, tile-aligned (4 or 2 bytes)
  uint16_t* dlix = nullptr;   // element positions in the tile dictionary
  uint64_t ndict = 0, nval = 0;  // dict words, element slots
};

// Storage precision of the matrix values.
enum ValueKind { kF32 = 0, kF16 = 1, kBF16 = 2 };

// Launch configuration of one projection (forward or backward).
struct GroupLaunch {
  int kind = kTiles;       // kGroups: lane group per row/column; kTiles: tiles
  int lanes = 16;          // kGroups: lanes per row (or column)
  int ept = 8;             // kTiles: elements per lane, tile = 256*ept elements
  int blocks_per_cu = 0;   // kGroups: 0 = one block per 256/lanes rows
  bool nested = false;     // dictionary tiles nested in the 16384-element ones
};

// A matrix kept in pinned host memory and streamed to the device in row
// blocks (out-of-core). Each block holds its rows as CSR (block-local row
// pointers, global columns) and their transpose as CSC (global rows); a
// projection copies its part of every block in turn through two device
// buffers, the copy of the next block overlapping the kernels of this one.
//
// The CSR part of a block of at least kPackMin elements that is not resident is
// held packed, where a sample of it says that this makes it smaller (and when the
// device has room to unpack one), chunk by chunk of kPackChunk elements:
//   row pointers | PackHead per chunk | kPackTable column steps | chunks
// A chunk is the elements' values, one code per element and the steps of the
// elements with code kPackEscape, each padded to 16 bytes: the column of an
// element is the column before it in the chunk (0 before the first) plus, modulo
// 2^32, the step of its code. A chunk that would not become smaller holds the
// 8-byte records (steps = kPackRaw).
//
// Why from 2^20 elements on: below, a block's kernels take longer than the copy of
// its 8-byte records (8 MB: 168 us against 160; 4 MB: 145 against 80), and
// unpacking would only add to them (77000 elements: 100 to 112 us a block).
// Above, the copy is what counts: 96x96x40 voxels, 700001 lines, 5 iterations take
// 51.5 ms from 64 MB blocks of records and 34.8 packed (5.1 bytes per element),
// 60.5 and 48.6 from 12 MB blocks.
constexpr uint64_t kPackMin = 1u << 20;
constexpr uint32_t kPackChunk = 4096;
constexpr uint32_t kPackTable = 256;
constexpr uint32_t kPackEscape = 255;
constexpr uint32_t kPackRaw = 0xFFFFFFFFu;
struct PackHead {
  uint32_t at;     // 16-byte units from the first chunk
  uint32_t count;  // elements
  uint32_t steps;  // escaped steps, or kPackRaw
  uint32_t pad;
};
struct StreamBlock {
  uint32_t row0 = 0, rows = 0;  // first row, rows
  uint64_t nnz = 0;
  uint64_t csr_off = 0, csr_bytes = 0;  // parts within the host buffer
  uint64_t packed_bytes = 0;            // of the packed CSR part; 0: not packed
  uint64_t csc_off = 0, csc_bytes = 0;
  char* resident = nullptr;  // device copy of both parts (CSR, then CSC), or none
};
struct StreamedMatrix {
  char* host = nullptr;  // pinned: every block's CSR part, then its CSC part
  uint64_t host_bytes = 0;
  std::vector<StreamBlock> blocks;
  uint64_t part_bytes = 0;  // largest part: the size of each device buffer
  char* dev[2] = {nullptr, nullptr};
  hipStream_t copy = nullptr;
  hipEvent_t copied[2] = {nullptr, nullptr};  // part in dev[i]
  hipEvent_t freed[2] = {nullptr, nullptr};   // kernels reading dev[i] done
  float* u = nullptr;                          // [cols] backprojection sums
  int lanes_fwd = 16, lanes_bwd = 4;           // FAST lane groups per row / column
  // A streamed block's CSC built on the device from its CSR part (colptr,
  // elements, sort scratch for the largest streamed block), so that a
  // reconstruction iteration streams each block once; null when it did not
  // fit in device memory next to the two part buffers (two passes then).
  char* csc_dev = nullptr;
  uint64_t csc_scratch_bytes = 0;
  uint64_t max_stream_nnz = 0;
  uint2* expand = nullptr;  // [max_stream_nnz] elements of the block unpacked last
  StreamedMatrix() = default;
  StreamedMatrix(const StreamedMatrix&) = delete;
  StreamedMatrix& operator=(const StreamedMatrix&) = delete;
  ~StreamedMatrix();
};

// Two-dimensional tiling of the matrix for products with W interleaved
// right-hand sides (panels.hpp; built on first use by ensure_panels). Vectors
// of those products index columns in panel order.
//
// The forward kernel reads the elements in octets: 8 pieces of a chunk, of about
// the same length, their elements in quads of 8 x 4: value and column of element
// 4j + k of piece i at (quad j) * 32 + 4i + k, so that the lanes of a wave load
// contiguous runs whatever W is. Positions past a piece's end hold value 0 and
// column kBoxVox, the row of zeros that the kernel keeps in LDS; the last two
// quads of the arrays hold only those.
struct PanelFormat {
  uint32_t rows = 0, cols = 0;
  uint32_t npanels = 0;                // boxes
  uint64_t nseg = 0;                   // pieces, one slot of partial sums each
  uint32_t* pc_of_file = nullptr;      // [cols] panel-order column of each file column
  uint32_t* pc_of_dev = nullptr;       // [cols] ... of each device column
  uint32_t* dev_of_pc = nullptr;       // [cols] device column of each panel-order column
  float* norm = nullptr;               // [cols] column sums in panel order
  uint32_t* pstart = nullptr;          // [npanels+1] first panel-order column of each box
  uint32_t* border = nullptr;          // [npanels] launch order (largest box first)
  uint32_t* rowslot = nullptr;         // [rows+1] first entry of each device row in rowpiece
  uint32_t* rowpiece = nullptr;        // [nseg] the rows' pieces (slots), box order
  uint32_t* pfchunk = nullptr;         // [npanels+1] first forward chunk of each box
  uint32_t* cpiece = nullptr;          // [chunks+1] first piece of each forward chunk
  uint32_t* fquad = nullptr;           // [chunks*128+1] first quad of each octet
  uint32_t* fpiece = nullptr;          // [chunks*1024] slot of each piece, ~0: none
  float* fval = nullptr;               // [quads+2][8][4]
  uint16_t* fcol = nullptr;            // [quads+2][8][4] column inside the box
  uint32_t fzero = 0;                  // first of the two quads of zeros
  uint32_t* brow = nullptr;            // [nseg] device row of each piece (backward order)
  uint32_t* pchunk = nullptr;          // [npanels+1] first backward chunk of each box
  uint2* chunk = nullptr;              // [chunks+1] {first piece, first element}
  uint16_t* boff = nullptr;            // [chunks*(kBoxVox+1)] voxel element offsets
  uint16_t* bpc = nullptr;             // piece of each element inside its chunk
  float* bval = nullptr;               // value of each element
  uint32_t* colslot = nullptr;         // [cols+1] slot of each panel-order column (identity)
  double build_seconds = 0.0;
  PanelFormat() = default;
  PanelFormat(const PanelFormat&) = delete;
  PanelFormat& operator=(const PanelFormat&) = delete;
  ~PanelFormat();
};

struct DevMatrix {
  uint32_t rows = 0, cols = 0;
  uint64_t nnz = 0;
  uint32_t grid[3] = {0, 0, 0};
  uint32_t symflags = 0;
  int device = 0;
  int cus = 256;
  hipStream_t stream = nullptr;

  uint32_t* rowptr = nullptr;  // [rows+1]
  uint2* csr = nullptr;        // [nnz] {column, value bits}
  uint32_t* colptr = nullptr;  // [cols+1]
  uint2* csc = nullptr;        // [nnz] {row, value bits}, rows ascending
  float* norm = nullptr;       // [cols] fp32 column sums, ascending row order

  // Locality layout (nullptr = identity): device column of each file column,
  // file row of each device row, device row of each file row.
  uint32_t* colmap = nullptr;  // [cols]
  uint32_t* rowold = nullptr;  // [rows]
  uint32_t* rowpos = nullptr;  // [rows]
  double sumnorm = 0.0;        // sequential double sum of norm (initImage)

  // Reduced-precision values: every record holds q_ij (exactly representable
  // in fp16 / bf16) and a_ij = rscale[i] * q_ij. The projections run on q;
  // the scales enter the FP64 column sums and the FP64 statistics only.
  int vk = kF32;
  float* rscale = nullptr;     // [rows] device row order, nullptr for fp32

  GroupLaunch fwd, bwd, scatter;
  GroupLaunch fwd_open, bwd_open;  // as chosen when the matrix was opened
  // Bumped whenever the launch configuration (and with it the tile and
  // dictionary buffers) may change; captured iterations are re-captured.
  uint64_t launch_gen = 0;

  // Tiled kernels: device-order pointers kept on the host, and the tile
  // partition (first segment of every tile, plus the end) for the current
  // elements-per-lane setting.
  std::vector<uint32_t> h_rowptr, h_colptr;
  uint2* tiles_fwd = nullptr;
  uint32_t ntiles_fwd = 0;
  int tiles_fwd_ept = 0;
  uint2* tiles_bwd = nullptr;
  uint32_t ntiles_bwd = 0;
  int tiles_bwd_ept = 0;
  DictFormat dfwd, dbwd;

  // per-handle scratch for the host-buffer step functions
  float* sx = nullptr;   // [cols]
  float* su = nullptr;   // [cols]
  float* sf = nullptr;   // [rows]
  float* sr = nullptr;   // [rows]
  int32_t* sy = nullptr; // [rows]
  float* tx = nullptr;   // [cols] file-order staging
  float* tf = nullptr;   // [rows] file-order staging

  StreamedMatrix* streamed = nullptr;  // out-of-core matrix (no device CSR/CSC)
  PanelFormat* panels = nullptr;       // tiling for many right-hand sides (or none)
};

// Deterministic FP64 reduction state for the forward pass: per-block partial
// (sum of y log f - f, sum of f) pairs, a completion counter, and a ring of
// per-iteration results indexed by a device-side iteration counter.
struct StatsState {
  double2* partials = nullptr;  // [max blocks]
  unsigned* counter = nullptr;  // [2]: [1] = next result slot ([0] unused)
  double2* results = nullptr;   // [ring]
  unsigned ring = 0;
  unsigned max_blocks = 0;
};

// ---- launchers (kernels.hip) -------------------------------------------
// Grid size of a statistics-carrying forward launch (partials needed).
unsigned stats_max_blocks(const DevMatrix& m);
// Copy the device-order row/column pointers to the host (once, after the
// layout is built).
void download_pointers(DevMatrix& m, hipStream_t s);
// (Re)build the tile partitions and dictionary formats the launch
// configuration needs.
void prepare_tiles(DevMatrix& m, hipStream_t s);
// Greedy partition of segments [0, n) into tiles of at most T elements and
// `maxseg` segments: the first segment of every tile, plus n.
std::vector<uint32_t> partition_tiles(const std::vector<uint32_t>& ptr, uint32_t T,
                                      uint32_t maxseg);
// Build a dictionary format (dict.hip) unless D holds it already; `el` indices
// are below `dim`.
void ensure_dict(const std::vector<uint32_t>& ptr, const uint2* el, uint32_t dim, int nb, int ept,
                 bool nested, int vk, DictFormat& D, hipStream_t s);
// Lines (32 neighbouring entries of the gathered vector) that the dictionary tiles
// of 16384, 8192 and 2048 elements of a projection touch in all, the smaller ones
// nested in the larger: estimated from up to 64 of the large tiles, exact if there
// are no more.
struct GatherSide {
  const std::vector<uint32_t>* ptr;  // first element of each segment, and the end
  const uint2* el;                   // elements, indices below dim
  uint32_t dim;
  std::array<double, 3> lines{0.0, 0.0, 0.0};
};
void tile_lines(std::initializer_list<GatherSide*> sides, hipStream_t s);
// Release a dictionary format's device memory.
void free_dict(DictFormat& d);
// Forward projection. ratio: out = (f != 0) ? y/f : 0, else out = f.
void launch_fwd(const DevMatrix& m, int mode, const float* x, const int32_t* y,
                float* out, bool ratio, const StatsState* stats, hipStream_t s);
// Backprojection through the CSC. update: x *= (n != 0) ? u/n : u written to
// `out` (which holds x), else out = u.
void launch_bwd(const DevMatrix& m, int mode, const float* r, const float* norm,
                float* out, bool update, hipStream_t s);
// One iteration: r = y / (A x), x *= (A^T r) / norm. The statistics of the
// forward projection (or nullptr) are complete after both.
void launch_iteration(const DevMatrix& m, int mode, float* x, const int32_t* y, float* r,
                      const StatsState* stats, hipStream_t s);
// Captured iterations (of a reconstruction or a batch) are replayed
// kGraphIterations at a time, in runs of at least kGraphMin: a graph of one
// iteration (two kernels) costs 5-15 us more per iteration than launching them
// (its launch waits for the one before: pet 425 against 408 us, the 38,496-element
// matrix 21.9 against 13.8), one of 16 iterations 1.3 us less, and building it takes
// about 100 us.
constexpr int kGraphIterations = 16, kGraphMin = 96;
// Backprojection by atomic scatter over the CSR: u += A^T r (u pre-zeroed).
void launch_scatter(const DevMatrix& m, const float* r, float* u, hipStream_t s);
// One row block of a streamed matrix (kernels.hip).
void launch_fwd_block(const uint32_t* rowptr, const uint2* csr, uint32_t rows, int lanes,
                      bool exact, const float* x, const int32_t* y, float* out, bool ratio,
                      const StatsState* st, int cus, hipStream_t s);
void launch_bwd_block_add(const uint32_t* colptr, const uint2* csc, uint32_t cols, int lanes,
                          bool exact, const float* r, float* u, int cus, hipStream_t s);
// u += (block rows)^T r by atomic scatter over one row block's CSR.
void launch_scatter_block(const uint32_t* rowptr, const uint2* csr, uint32_t rows, int lanes,
                          const float* r, float* u, int cus, hipStream_t s);
// Streamed matrices (stream.cpp): build the blocks from a row index (END
// offsets) and an element source; the projections over every block.
using ElementFetch = std::function<void(void* dst, uint64_t first, uint64_t count)>;
StreamedMatrix* build_streamed(uint32_t rows, uint32_t cols, uint64_t nnz,
                               const uint64_t* rowidx, const ElementFetch& fetch,
                               uint64_t block_bytes, uint64_t resident_bytes, hipStream_t s);
void stream_fwd(const DevMatrix& m, int mode, const float* x, const int32_t* y, float* out,
                bool ratio, const StatsState* st, hipStream_t s);
void stream_bwd(const DevMatrix& m, int mode, const float* r, const float* norm, float* out,
                bool update, hipStream_t s);
void stream_bwd_add(const DevMatrix& m, bool exact, const float* r, float* u, hipStream_t s);
// One pass over the CSR blocks: per block the forward projection with the
// fused ratio into r, then u += (block rows)^T r by atomic scatter while the
// block is on the device (ATOMIC mode: each block crosses PCIe once per
// iteration instead of twice).
void stream_fwd_scatter(const DevMatrix& m, const float* x, const int32_t* y, float* r, float* u,
                        const StatsState* st, hipStream_t s);
// One FAST / EXACT reconstruction iteration over a streamed matrix: per block
// the forward projection with the fused ratio into r, then (with csc_dev) the
// block's CSC built on the device and its backprojection added to u, so each
// CSR part crosses PCIe once; without csc_dev the two passes of stream_fwd and
// stream_bwd. Then x *= (n != 0) ? u/n : u.
void stream_iteration(const DevMatrix& m, int mode, float* x, const int32_t* y, float* r,
                      const StatsState* st, hipStream_t s);
// CSC of one row block (block-local row pointers, global columns) built on the
// device: a stable sort by column keeps the block-local rows ascending inside
// every column. block_csc_scratch gives the scratch bytes it needs.
size_t block_csc_scratch(uint64_t nnz, uint32_t cols);
void build_block_csc(const uint32_t* rowptr, const uint2* csr, uint32_t rows, uint32_t cols,
                     uint64_t nnz, void* scratch, size_t scratch_bytes, uint32_t* colptr,
                     uint2* csc, hipStream_t s);
// Elements of a packed block: heads, steps table and chunks as they arrived.
void launch_unpack(const PackHead* heads, uint64_t nnz, uint2* el, hipStream_t s);
// x *= (n != 0) ? u/n : u; optionally u = 0 afterwards.
void launch_update(uint32_t cols, const float* u, const float* norm, float* x,
                   bool zero_u, hipStream_t s);
// r = (f != 0) ? y/f : 0.
void launch_correl(uint32_t rows, const float* f, const int32_t* y, float* r,
                   hipStream_t s);
// norm from the CSC, sequential per column in ascending row order.
void launch_colsums_csc(const DevMatrix& m, float* norm, hipStream_t s);
// norm by atomic scatter (matrices opened without a CSC).
void launch_colsums_atomic(const DevMatrix& m, float* norm, hipStream_t s);
// Reduced precision: row scales (file row order) and in-place quantization
// of the file-order CSR values to fp16 / bf16 (kept as exact fp32 words).
void launch_quantize(DevMatrix& m, int vk, float* rscale, hipStream_t s);
// norm_j = (float) sum_i (double) s_i q_ij from the CSC, ascending row order.
void launch_colsums_scaled(const DevMatrix& m, float* norm, hipStream_t s);
// r_i *= s_i in device row order (no-op for fp32 values).
void launch_scale_rows(const DevMatrix& m, float* r, hipStream_t s);
// ---- products with W right-hand sides through the tiling (panel.hip) ------
// Build (once per matrix, on the host from the device CSR) and return the
// tiling; free_panels releases it.
const PanelFormat& ensure_panels(DevMatrix& m);
void free_panels(DevMatrix& m);
// part[s * W + f] = dot product of piece s with X (panel order, [cols][W]); a
// row's pieces are rowpiece[rowslot[r]] .. rowpiece[rowslot[r + 1] - 1].
// Slots are numbered box by box in chunks of rows, so that neighbouring rows'
// slots lie together. U[c * W + f] = (A^T R)_c for every panel-order column c,
// R [rows][W] in device row order. One workgroup per box.
template <int W>
void launch_panel_fwd(const PanelFormat& P, const float* X, float* part, hipStream_t s);
template <int W>
void launch_panel_bwd(const PanelFormat& P, const float* R, float* U, hipStream_t s);
// ---- load-time layout (layout.hip) ----------------------------------------
// Renumber rows (sinogram order) and voxels (4x4x2 bricks) when the grid is
// known, build the CSC (file row order inside every column) and the
// device-order CSR. Requires validated column indices.
void build_layout(DevMatrix& m, bool reorder_rows, bool reorder_cols, bool want_csc,
                  hipStream_t s);
// File-order <-> device-order vectors (device buffers, distinct pointers).
void to_device_cols(const DevMatrix& m, const float* file_order, float* dev, hipStream_t s);
void to_file_cols(const DevMatrix& m, const float* dev, float* file_order, hipStream_t s);
template <class T>
void rows_to_device(const DevMatrix& m, const T* file_order, T* dev, hipStream_t s);
template <class T>
void rows_to_file(const DevMatrix& m, const T* dev, T* file_order, hipStream_t s);
// Sums of int32 counts: sum and sum of magnitudes. While the latter stays
// below 2^53, every partial sum of the reference's running double sum
// (seqcsr4mlem.cpp:57-58) is an integer that a double holds exactly, so the
// integer sum in any order equals it; otherwise the host adds in order.
struct CountSum {
  long long sum;
  unsigned long long magnitude;
  bool exact() const { return magnitude < (1ull << 53); }
};
inline double host_count_sum(const int32_t* y, uint32_t rows) {
  double s = 0.0;
  for (uint32_t i = 0; i < rows; ++i) s += y[i];
  return s;
}
// Below this many counts the host's running sum (0.8 ns a count) costs less
// than the kernel and the read-back of its result (about 25 us).
constexpr uint32_t kHostSumRows = 32768;
// out[f] += the sums of y[f*rows .. (f+1)*rows) (out zeroed before).
void launch_count_sums(const int32_t* y, uint32_t rows, uint32_t frames, CountSum* out,
                       hipStream_t s);
// Count column indices >= cols in the CSR (validation).
void launch_check_columns(const DevMatrix& m, unsigned* bad, hipStream_t s);
// Build rowptr (u32) from the csr4 END-offset row index already on device.
void launch_rowptr_from_rowidx(const uint64_t* rowidx, uint32_t rows,
                               uint32_t* rowptr, hipStream_t s);
// Fill a float buffer.
void launch_fill(float* p, float v, size_t n, hipStream_t s);
// Streaming copy kernel (byte-counter calibration).
void launch_copy(const uint4* src, uint4* dst, size_t n16, hipStream_t s);

}  // namespace mlem

// The C-ABI matrix handle (include/mlem.h): the device matrix plus load
// timings. Defined here so every source of the library can reach it.
struct mlem_matrix {
  mlem::DevMatrix m;
  double norm_seconds = 0.0;  // layout, CSC build and column sums at open
  double load_seconds = 0.0;  // file/host -> HBM
  ~mlem_matrix();
};
