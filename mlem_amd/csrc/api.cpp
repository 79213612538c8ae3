// api.cpp — C ABI of libmlem.so: matrix loading into HBM, step functions,
// reconstruction driver, checkpoint/restart, timing.
//
// Reference counterparts: Csr4Matrix (helper_files_common/csr4matrix.cpp),
// mlem() and its step functions (mlem_seq/seqcsr4mlem.cpp:37-189), and the
// checkpoint/restart logic of mlem_mpi/mpicsr4mlem.cpp:95-154,536-553 with
// the interval meaning of mlem_cuda/helper_files/hybCalcFunc.cu:852-853.
#include <hip/hip_runtime.h>
#include <sys/stat.h>
#include <unistd.h>

#include <algorithm>
#include <chrono>
#include <cmath>
#include <cstdlib>
#include <cstring>
#include <iostream>
#include <memory>
#include <new>
#include <string>
#include <vector>

#include "csr4.hpp"
#include "internal.hpp"
#include "mlem.h"
#include "symmetry.hpp"
#include "transfer.hpp"

using namespace mlem;

namespace mlem {

[[noreturn]] void raise(int code, const std::string& msg) { throw ApiError{code, msg}; }

void hip_check(hipError_t e, const char* what) {
  if (e == hipSuccess) return;
  const int code = (e == hipErrorOutOfMemory || e == hipErrorMemoryAllocation) ? MLEM_ENOMEM
                                                                                : MLEM_EDEVICE;
  raise(code, std::string(what) + " failed: " + hipGetErrorString(e));
}

}  // namespace mlem

namespace {
thread_local std::string g_error;
}  // namespace

namespace mlem {
void set_error(const std::string& msg) { g_error = msg; }
void clear_error() { g_error.clear(); }
}  // namespace mlem

namespace {

int env_int(const char* name, int dflt) {
  const char* v = std::getenv(name);
  if (!v || !*v) return dflt;
  return std::atoi(v);
}

double seconds_since(std::chrono::steady_clock::time_point t0) {
  return std::chrono::duration<double>(std::chrono::steady_clock::now() - t0).count();
}

// Pick the lanes-per-row group from the average segment length: about four
// elements per lane per pass, clamped to 4..64.
int lanes_for(double avg) {
  int g = 4;
  while (g < 64 && g * 4 < avg) g *= 2;
  return g;
}

void select_device(int* dev, int* cus) {
  int n = 0;
  hipError_t e = hipGetDeviceCount(&n);
  if (e != hipSuccess || n <= 0)
    raise(MLEM_EDEVICE, "no GPU is visible to the HIP runtime (libmlem needs an MI355X, gfx950)");
  MLEM_HIP(hipGetDevice(dev));
  hipDeviceProp_t p;
  MLEM_HIP(hipGetDeviceProperties(&p, *dev));
  if (std::strncmp(p.gcnArchName, "gfx950", 6) != 0)
    raise(MLEM_EDEVICE, std::string("libmlem is built for gfx950; device is ") + p.gcnArchName);
  *cus = p.multiProcessorCount > 0 ? p.multiProcessorCount : 256;
}

template <class T>
void dfree(T*& p) {
  if (p) (void)hipFree(p);
  p = nullptr;
}

}  // namespace

// --------------------------------------------------------------- handles --
mlem_matrix::~mlem_matrix() {
  {
    dfree(m.rowptr);
    dfree(m.csr);
    dfree(m.colptr);
    dfree(m.csc);
    dfree(m.norm);
    dfree(m.sx);
    dfree(m.su);
    dfree(m.sf);
    dfree(m.sr);
    dfree(m.sy);
    dfree(m.tx);
    dfree(m.tf);
    dfree(m.colmap);
    dfree(m.rowold);
    dfree(m.rowpos);
    dfree(m.rscale);
    dfree(m.tiles_fwd);
    dfree(m.tiles_bwd);
    free_dict(m.dfwd);
    free_dict(m.dbwd);
    delete m.streamed;
    m.streamed = nullptr;
    free_panels(m);
    if (m.stream) (void)hipStreamDestroy(m.stream);
  }
}

struct mlem_recon {
  mlem_matrix* mat = nullptr;
  int mode = MLEM_MODE_FAST;
  int done = 0;
  bool use_graph = false;
  bool want_stats = false;
  char* buf = nullptr;  // one allocation for the vectors and the statistics ring
  int32_t* y = nullptr;
  float* x = nullptr;
  float* r = nullptr;
  float* u = nullptr;   // ATOMIC mode accumulator
  float* xs = nullptr;  // file-order image staging
  StatsState st;        // counter and results in buf, partials their own
  std::vector<double> loglik, fwdtot;  // per completed iteration
  hipGraph_t graph = nullptr;
  hipGraphExec_t exec = nullptr;
  uint64_t graph_gen = 0;  // matrix launch generation the graph was captured at
  std::vector<hipEvent_t> events;
  ~mlem_recon() {
    if (exec) (void)hipGraphExecDestroy(exec);
    if (graph) (void)hipGraphDestroy(graph);
    for (hipEvent_t e : events) (void)hipEventDestroy(e);
    dfree(buf);
    dfree(st.partials);
  }
};

namespace {

void check_dims(const mlem_matrix* h, uint32_t rows, uint32_t cols) {
  if (!h) raise(MLEM_EINVAL, "null matrix handle");
  if (rows != h->m.rows || cols != h->m.cols)
    raise(MLEM_EINVAL, "vector sizes (" + std::to_string(rows) + " rows, " + std::to_string(cols) +
                           " columns) do not match the matrix (" + std::to_string(h->m.rows) +
                           " x " + std::to_string(h->m.cols) + ")");
}

// Time one kernel variant (median of a few launches) with HIP events.
template <class Launch>
float time_variant(hipStream_t s, Launch&& launch, int reps) {
  hipEvent_t a, b;
  MLEM_HIP(hipEventCreate(&a));
  MLEM_HIP(hipEventCreate(&b));
  std::vector<float> t;
  launch();  // warm
  for (int i = 0; i < reps; ++i) {
    MLEM_HIP(hipEventRecord(a, s));
    launch();
    MLEM_HIP(hipEventRecord(b, s));
    MLEM_HIP(hipEventSynchronize(b));
    float ms = 0.f;
    MLEM_HIP(hipEventElapsedTime(&ms, a, b));
    t.push_back(ms);
  }
  (void)hipEventDestroy(a);
  (void)hipEventDestroy(b);
  std::sort(t.begin(), t.end());
  return t[t.size() / 2];
}

// Launch configuration of a kernel family and its parameter (validated).
GroupLaunch make_launch(int kind, int param) {
  GroupLaunch g;
  g.kind = kind;
  if (kind == kTiles) {
    if (param != 4 && param != 8 && param != 16)
      raise(MLEM_EINVAL, "tile elements per lane must be 4, 8 or 16");
    g.ept = param;
  } else if (kind == kDict) {
    if (param != 8 && param != 16 && param != 24 && param != 32 && param != 48 && param != 64)
      raise(MLEM_EINVAL, "dictionary tile elements per lane must be 8, 16, 24, 32, 48 or 64");
    g.ept = param;
  } else if (kind == kDictWide) {
    if (param != 16 && param != 24 && param != 32)
      raise(MLEM_EINVAL, "wide dictionary tile elements per lane must be 16, 24 or 32");
    g.ept = param;
  } else if (kind == kGroups) {
    if (param != 4 && param != 8 && param != 16 && param != 32 && param != 64)
      raise(MLEM_EINVAL, "lanes per row must be 4, 8, 16, 32 or 64");
    g.lanes = param;
  } else {
    raise(MLEM_EINVAL, "unknown kernel family");
  }
  return g;
}

// The launch that a kernel family and its parameter stand for on a matrix that
// was opened with `open` for this projection: that launch itself where they name
// it (mlem_get_launch gives a family and a parameter alone, and its tiles may be
// nested), so that what mlem_get_launch returned can be set again with the same
// tiles and the same FAST sums.
GroupLaunch named_launch(int kind, int param, const GroupLaunch& open) {
  const GroupLaunch g = make_launch(kind, param);
  return is_dict(kind) && open.kind == kind && open.ept == param ? open : g;
}

// Dictionary tiles of a projection whose segments end at ptr. 16384-element
// tiles run by 512-lane blocks, two per CU (LDS- and register-bound), are the
// fastest once every CU gets several: pet (168.4M elements) forward / backward
// 224 / 218 us against 250 / 246 with 8192. A small matrix is bound by the
// latency of one tile and by its last wave of tiles (us of one FAST product, launch
// included, 16384 / 8192 / 2048 elements):
//   lines of response  9.2M elements  23.6 / 22.0 / 22.0 forward, 21.6 / 20.8 / 22.8 backward
//                      4.9M           17.5 / 14.9 / 15.0,         15.9 / 14.2 / 14.1
//                      2.4M           12.8 / 11.2 / 10.2,         12.0 / 11.0 / 10.2
//                      0.4M           11.0 /  9.0 /  7.5,         11.0 /  8.3 /  6.6
// but gathers more lines in all, as a line is gathered once per tile that needs
// it: about 9 us per million lines, which is what it gains at a quarter of a million
//   lines of response 15.2M, 0.3M lines more  31.1 / 33.4 (8192), 28.9 / 30.2
//   random           18.0M, 3.5M              64.8 / 80.0,        62.0 / 76.0
//   random           12.0M, 1.4M              29.7 / 37.5,        28.3 / 36.8
//   random            2.2M, 0.8M              13.3 / 14.1 (2048), 13.3 / 13.6
// And a tile of few segments keeps few lanes busy; where tiles wait for a place
// as well, smaller ones that hold one long segment take longer: 11x12x12 voxels,
// 6.6M elements, backward 44.6 / 57.8 FAST and 99.7 / 136.6 EXACT (8192); 5000
// columns of 400 elements 16.4 / 20.1 EXACT (2048). A segment longer than a tile is
// summed with direct gathers (EXACT: by one lane), so tiles hold the longest
// segment where the largest ones can.
// mlem_autotune measures the alternatives on the real matrix.
constexpr uint64_t kSmallNnz = 2500000, kMidNnz = 20000000, kMoreLines = 250000;
GroupLaunch default_launch(uint64_t nnz, const std::vector<uint32_t>& ptr,
                           const std::array<double, 3>& lines) {
  GroupLaunch g = make_launch(kDictWide, 32);  // the same FAST sums with every tile size
  if (nnz > kMidNnz || nnz == 0) return g;
  uint32_t longest = 0;
  uint64_t squares = 0;
  for (size_t i = 0; i + 1 < ptr.size(); ++i) {
    const uint32_t n = ptr[i + 1] - ptr[i];
    longest = std::max(longest, n);
    squares += (uint64_t)n * n;
  }
  const double length = (double)squares / (double)nnz;  // of an element's segment, on average
  if (longest + 3 > 512 * 16 || (nnz > kSmallNnz && length > 512 * 16 / 5) ||
      lines[1] - lines[0] > (double)kMoreLines)
    return g;
  g = make_launch(kDictWide, 16);
  if (nnz <= kSmallNnz && longest + 3 <= 256 * 8 && length <= 256 * 8 / 5 &&
      lines[2] - lines[1] <= (double)kMoreLines)
    g = make_launch(kDict, 8);
  g.nested = true;
  return g;
}

// Candidate FAST-mode configurations of one projection.
std::vector<GroupLaunch> launch_candidates(const GroupLaunch& open) {
  std::vector<GroupLaunch> c;
  for (int e : {16, 24, 32}) c.push_back(named_launch(kDictWide, e, open));
  for (int e : {8, 16, 24, 32, 48, 64}) c.push_back(named_launch(kDict, e, open));
  for (int e : {4, 8, 16}) c.push_back(named_launch(kTiles, e, open));
  for (int g : {8, 16, 32, 64}) c.push_back(named_launch(kGroups, g, open));
  return c;
}

// Time every forward and backward configuration on this matrix with HIP
// events (median of 3 launches on real-sized vectors) and keep the fastest.
void autotune(DevMatrix& m) {
  if (m.nnz == 0) return;
  float *x = nullptr, *r = nullptr, *xx = nullptr;
  int32_t* y = nullptr;
  struct F {
    void** p[4];
    ~F() {
      for (void** q : p)
        if (*q) (void)hipFree(*q);
    }
  } f{{(void**)&x, (void**)&r, (void**)&y, (void**)&xx}};
  MLEM_HIP(hipMalloc(&x, 4ull * std::max<uint32_t>(m.cols, 1)));
  MLEM_HIP(hipMalloc(&xx, 4ull * std::max<uint32_t>(m.cols, 1)));
  MLEM_HIP(hipMalloc(&r, 4ull * std::max<uint32_t>(m.rows, 1)));
  MLEM_HIP(hipMalloc(&y, 4ull * std::max<uint32_t>(m.rows, 1)));
  launch_fill(x, 1.f, m.cols, m.stream);
  launch_fill(r, 1.f, m.rows, m.stream);
  launch_fill(reinterpret_cast<float*>(y), 0.f, m.rows, m.stream);
  float best = 1e30f;
  GroupLaunch bestF = m.fwd, bestB = m.bwd;
  for (const GroupLaunch& g : launch_candidates(m.fwd_open)) {
    m.fwd = g;
    prepare_tiles(m, m.stream);
    const float t = time_variant(
        m.stream, [&] { launch_fwd(m, MLEM_MODE_FAST, x, y, r, true, nullptr, m.stream); }, 3);
    if (t < best) {
      best = t;
      bestF = g;
    }
  }
  m.fwd = bestF;
  if (m.csc) {
    best = 1e30f;
    for (const GroupLaunch& g : launch_candidates(m.bwd_open)) {
      m.bwd = g;
      prepare_tiles(m, m.stream);
      const float t = time_variant(
          m.stream, [&] { launch_bwd(m, MLEM_MODE_FAST, r, m.norm, xx, false, m.stream); }, 3);
      if (t < best) {
        best = t;
        bestB = g;
      }
    }
    m.bwd = bestB;
  }
  prepare_tiles(m, m.stream);
  MLEM_HIP(hipStreamSynchronize(m.stream));
}

void ensure_scratch(DevMatrix& m);

// Shared tail of mlem_open / mlem_open_host once rowptr and csr are on the
// device: validate columns, build the CSC, column sums, launch tuning.
void finish_open(mlem_matrix* h, unsigned flags) {
  DevMatrix& m = h->m;
  auto t0 = std::chrono::steady_clock::now();
  if ((flags & MLEM_OPEN_FP16) && (flags & MLEM_OPEN_BF16))
    raise(MLEM_EINVAL, "MLEM_OPEN_FP16 and MLEM_OPEN_BF16 are exclusive");
  if ((flags & (MLEM_OPEN_FP16 | MLEM_OPEN_BF16)) && (flags & MLEM_OPEN_NO_CSC))
    raise(MLEM_EINVAL, "16-bit values need the CSC (MLEM_OPEN_NO_CSC not allowed)");
  if (m.nnz > 0) {
    unsigned* bad = nullptr;
    MLEM_HIP(hipMalloc(&bad, sizeof(unsigned)));
    unsigned hbad = 0;
    hipError_t e = hipMemsetAsync(bad, 0, sizeof(unsigned), m.stream);
    if (e == hipSuccess) {
      launch_check_columns(m, bad, m.stream);
      e = hipMemcpyAsync(&hbad, bad, sizeof(unsigned), hipMemcpyDeviceToHost, m.stream);
    }
    if (e == hipSuccess) e = hipStreamSynchronize(m.stream);
    (void)hipFree(bad);
    MLEM_HIP(e);
    if (hbad)
      raise(MLEM_EFORMAT, std::to_string(hbad) + " matrix elements have a column index >= " +
                              std::to_string(m.cols));
  }
  const int vk = (flags & MLEM_OPEN_FP16) ? kF16 : (flags & MLEM_OPEN_BF16) ? kBF16 : kF32;
  struct Scratch {
    float* p = nullptr;
    ~Scratch() {
      if (p) (void)hipFree(p);
    }
  } rscale_file;
  if (vk != kF32) {
    // Row scales and 16-bit values are fixed before the layout is built, so
    // the CSC and both dictionary formats inherit the quantized values.
    MLEM_HIP(hipMalloc(&m.rscale, 4ull * std::max<uint32_t>(m.rows, 1)));
    MLEM_HIP(hipMalloc(&rscale_file.p, 4ull * std::max<uint32_t>(m.rows, 1)));
    launch_quantize(m, vk, rscale_file.p, m.stream);
  }
  const bool reorder = !(flags & MLEM_OPEN_KEEP_ORDER);
  build_layout(m, reorder, reorder, !(flags & MLEM_OPEN_NO_CSC), m.stream);
  MLEM_HIP(hipMalloc(&m.norm, 4ull * std::max<uint32_t>(m.cols, 1)));
  if (vk != kF32) {
    if (m.rows) rows_to_device(m, (const float*)rscale_file.p, m.rscale, m.stream);
    MLEM_HIP(hipStreamSynchronize(m.stream));
    m.vk = vk;
    launch_colsums_scaled(m, m.norm, m.stream);
  } else if (m.csc) {
    launch_colsums_csc(m, m.norm, m.stream);
  } else {
    launch_colsums_atomic(m, m.norm, m.stream);
  }
  ensure_scratch(m);
  to_file_cols(m, m.norm, m.tx, m.stream);
  std::vector<float> norm(m.cols);
  if (m.cols)
    MLEM_HIP(hipMemcpyAsync(norm.data(), m.tx, 4ull * m.cols, hipMemcpyDeviceToHost, m.stream));
  MLEM_HIP(hipStreamSynchronize(m.stream));
  // initImage's sum of the norm: double, file index order (seqcsr4mlem.cpp:55-56).
  double sn = 0.0;
  for (uint32_t j = 0; j < m.cols; ++j) sn += norm[j];
  m.sumnorm = sn;
  h->norm_seconds = seconds_since(t0);

  const double avgRow = m.rows ? (double)m.nnz / m.rows : 1.0;
  download_pointers(m, m.stream);
  GatherSide f{&m.h_rowptr, m.csr, m.cols}, b{&m.h_colptr, m.csc, m.rows};
  if (m.nnz > kMoreLines && m.nnz <= kMidNnz) {  // (no tiles touch more lines than elements)
    if (m.csc)
      tile_lines({&f, &b}, m.stream);
    else
      tile_lines({&f}, m.stream);
  }
  m.fwd = m.fwd_open = default_launch(m.nnz, m.h_rowptr, f.lines);
  m.bwd = m.bwd_open = default_launch(m.nnz, m.h_colptr, b.lines);
  m.scatter = make_launch(kGroups, lanes_for(avgRow));
  prepare_tiles(m, m.stream);
  if (env_int("MLEM_AUTOTUNE", 0) > 0) autotune(m);
}

mlem_matrix* new_matrix(uint32_t rows, uint32_t cols, uint64_t nnz) {
  // u32 element offsets on the device, with headroom for the kernels'
  // unrolled index arithmetic (k + 4*64).
  if (nnz > (1ull << 32) - 1024)
    raise(MLEM_EINVAL, "matrices with 2^32-1024 or more elements are not supported (nnz=" +
                           std::to_string(nnz) + ")");
  if (rows == 0xFFFFFFFFu || cols == 0xFFFFFFFFu) raise(MLEM_EINVAL, "dimension too large");
  std::unique_ptr<mlem_matrix> h(new mlem_matrix());
  DevMatrix& m = h->m;
  m.rows = rows;
  m.cols = cols;
  m.nnz = nnz;
  select_device(&m.device, &m.cus);
  MLEM_HIP(hipStreamCreateWithFlags(&m.stream, hipStreamNonBlocking));
  MLEM_HIP(hipMalloc(&m.rowptr, 4ull * ((uint64_t)rows + 1)));
  MLEM_HIP(hipMalloc(&m.csr, 8ull * std::max<uint64_t>(nnz, 1)));
  return h.release();
}

void upload_rowidx(DevMatrix& m, const uint64_t* rowidx) {
  if (m.rows == 0) {
    MLEM_HIP(hipMemsetAsync(m.rowptr, 0, 4, m.stream));
    return;
  }
  uint64_t* d = nullptr;
  MLEM_HIP(hipMalloc(&d, 8ull * m.rows));
  hipError_t e = hipMemcpyAsync(d, rowidx, 8ull * m.rows, hipMemcpyHostToDevice, m.stream);
  if (e == hipSuccess) {
    launch_rowptr_from_rowidx(d, m.rows, m.rowptr, m.stream);
    e = hipStreamSynchronize(m.stream);
  }
  (void)hipFree(d);
  MLEM_HIP(e);
}

void ensure_scratch(DevMatrix& m) {
  if (!m.sx) MLEM_HIP(hipMalloc(&m.sx, 4ull * std::max<uint32_t>(m.cols, 1)));
  if (!m.su) MLEM_HIP(hipMalloc(&m.su, 4ull * std::max<uint32_t>(m.cols, 1)));
  if (!m.sf) MLEM_HIP(hipMalloc(&m.sf, 4ull * std::max<uint32_t>(m.rows, 1)));
  if (!m.sr) MLEM_HIP(hipMalloc(&m.sr, 4ull * std::max<uint32_t>(m.rows, 1)));
  if (!m.sy) MLEM_HIP(hipMalloc(&m.sy, 4ull * std::max<uint32_t>(m.rows, 1)));
  if (!m.tx) MLEM_HIP(hipMalloc(&m.tx, 4ull * std::max<uint32_t>(m.cols, 1)));
  if (!m.tf) MLEM_HIP(hipMalloc(&m.tf, 4ull * std::max<uint32_t>(m.rows, 1)));
}

void h2d(void* d, const void* h, size_t n, hipStream_t s) {
  if (n) MLEM_HIP(hipMemcpyAsync(d, h, n, hipMemcpyHostToDevice, s));
}
void d2h(void* h, const void* d, size_t n, hipStream_t s) {
  if (n) MLEM_HIP(hipMemcpyAsync(h, d, n, hipMemcpyDeviceToHost, s));
}

constexpr unsigned kStatsRing = 4096;

// Forward launches per projection: one, or one per block of a streamed matrix.
unsigned fwd_launches(const DevMatrix& m) {
  return m.streamed ? (unsigned)std::max<size_t>(m.streamed->blocks.size(), 1) : 1u;
}

void enqueue_iteration(mlem_recon* R) {
  DevMatrix& m = R->mat->m;
  const StatsState* st = R->want_stats ? &R->st : nullptr;
  if (R->mode == MLEM_MODE_ATOMIC) {
    if (m.streamed) {
      stream_fwd_scatter(m, R->x, R->y, R->r, R->u, st, m.stream);
    } else {
      launch_fwd(m, MLEM_MODE_FAST, R->x, R->y, R->r, true, st, m.stream);
      launch_scatter(m, R->r, R->u, m.stream);
    }
    launch_update(m.cols, R->u, m.norm, R->x, true, m.stream);
  } else if (m.streamed) {
    stream_iteration(m, R->mode, R->x, R->y, R->r, st, m.stream);
  } else {
    launch_iteration(m, R->mode, R->x, R->y, R->r, st, m.stream);
  }
}

// Iteration k's statistics: the per-launch results of its forward launches
// (one, or one per streamed block), summed in launch order.
void collect_stats(mlem_recon* R, int first, int count) {
  if (!R->want_stats || count <= 0) return;
  const unsigned per = fwd_launches(R->mat->m);
  std::vector<double2> res(kStatsRing);
  // the ring slots of these iterations (all of them when they wrap around)
  uint64_t lo = (uint64_t)first * per % kStatsRing, n = (uint64_t)count * per;
  if (lo + n > kStatsRing) {
    lo = 0;
    n = kStatsRing;
  }
  d2h(res.data() + lo, R->st.results + lo, sizeof(double2) * n, R->mat->m.stream);
  MLEM_HIP(hipStreamSynchronize(R->mat->m.stream));
  for (int k = 0; k < count; ++k) {
    double ll = 0.0, tot = 0.0;
    for (unsigned b = 0; b < per; ++b) {
      const double2 v = res[((uint64_t)(first + k) * per + b) % kStatsRing];
      ll += v.x;
      tot += v.y;
    }
    R->loglik.push_back(ll);
    R->fwdtot.push_back(tot);
  }
}

void drop_graph(mlem_recon* R) {
  if (R->exec) (void)hipGraphExecDestroy(R->exec);
  if (R->graph) (void)hipGraphDestroy(R->graph);
  R->exec = nullptr;
  R->graph = nullptr;
}

void run_iterations(mlem_recon* R, int iterations) {
  DevMatrix& m = R->mat->m;
  if (R->want_stats && stats_max_blocks(m) > R->st.max_blocks) {
    // a launch change since creation needs more workgroup partials; the
    // captured graph holds the old buffer
    drop_graph(R);
    MLEM_HIP(hipStreamSynchronize(m.stream));
    dfree(R->st.partials);
    R->st.max_blocks = stats_max_blocks(m);
    MLEM_HIP(hipMalloc(&R->st.partials, sizeof(double2) * R->st.max_blocks));
  }
  int left = iterations;
  while (left > 0) {
    const int n =
        R->want_stats ? std::min<int>(left, (int)(kStatsRing / fwd_launches(m))) : left;
    int i = 0;
    if (R->use_graph) {
      if (R->exec && R->graph_gen != m.launch_gen) drop_graph(R);  // kernels or buffers changed
      if (!R->exec && n >= kGraphMin) {
        R->graph_gen = m.launch_gen;
        MLEM_HIP(hipStreamBeginCapture(m.stream, hipStreamCaptureModeThreadLocal));
        try {
          for (int k = 0; k < kGraphIterations; ++k) enqueue_iteration(R);
        } catch (...) {
          hipGraph_t g = nullptr;
          (void)hipStreamEndCapture(m.stream, &g);
          if (g) (void)hipGraphDestroy(g);
          throw;
        }
        MLEM_HIP(hipStreamEndCapture(m.stream, &R->graph));
        MLEM_HIP(hipGraphInstantiate(&R->exec, R->graph, nullptr, nullptr, 0));
      }
      for (; R->exec && i + kGraphIterations <= n; i += kGraphIterations)
        MLEM_HIP(hipGraphLaunch(R->exec, m.stream));
    }
    for (; i < n; ++i) enqueue_iteration(R);
    MLEM_HIP(hipStreamSynchronize(m.stream));
    collect_stats(R, R->done, n);
    R->done += n;
    left -= n;
  }
}

mlem_recon* create_recon(mlem_matrix* h, const int32_t* y, uint32_t rows, const float* x0,
                         uint32_t cols, const mlem_options* o, float* initial_out,
                         double* sumin_out) {
  check_dims(h, rows, cols);
  if (!y) raise(MLEM_EINVAL, "null sinogram");
  mlem_options dflt;
  mlem_options_default(&dflt);
  if (!o) o = &dflt;
  if (o->mode < MLEM_MODE_FAST || o->mode > MLEM_MODE_ATOMIC) raise(MLEM_EINVAL, "unknown mode");
  if (o->init == MLEM_INIT_GIVEN && !x0) raise(MLEM_EINVAL, "MLEM_INIT_GIVEN needs an image");
  if (o->mode != MLEM_MODE_ATOMIC && !h->m.csc && !h->m.streamed)
    raise(MLEM_ESTATE, "matrix was opened without a CSC; only MLEM_MODE_ATOMIC is available");
  DevMatrix& m = h->m;
  std::unique_ptr<mlem_recon> R(new mlem_recon());
  R->mat = h;
  R->mode = o->mode;
  // a streamed iteration spans two streams and host copies: run it directly
  R->use_graph = o->use_graph != 0 && !m.streamed;
  R->want_stats = (o->loglik != nullptr) || (o->fwd_total != nullptr);
  if (R->want_stats && fwd_launches(m) > kStatsRing)
    raise(MLEM_EINVAL, "statistics need at most " + std::to_string(kStatsRing) +
                           " streamed blocks");
  // y, x, r, xs (and u), the counter and the sums of y (4 words), the ring
  const bool atomic = R->mode == MLEM_MODE_ATOMIC;
  size_t off = 0;
  auto take = [&off](size_t bytes) {
    const size_t at = off;
    off = (at + bytes + 255) & ~(size_t)255;
    return at;
  };
  const size_t oy = take(4ull * rows), ox = take(4ull * cols), orr = take(4ull * rows);
  const size_t os = take(4ull * cols), ou = take(atomic ? 4ull * cols : 0);
  const size_t oc = take(8 * sizeof(unsigned));
  const size_t ores = take(R->want_stats ? sizeof(double2) * kStatsRing : 0);
  MLEM_HIP(hipMalloc(&R->buf, off));
  R->y = reinterpret_cast<int32_t*>(R->buf + oy);
  R->x = reinterpret_cast<float*>(R->buf + ox);
  R->r = reinterpret_cast<float*>(R->buf + orr);
  R->xs = reinterpret_cast<float*>(R->buf + os);
  unsigned* words = reinterpret_cast<unsigned*>(R->buf + oc);  // counter[2], pad, sums
  if (atomic) {
    R->u = reinterpret_cast<float*>(R->buf + ou);
    launch_fill(R->u, 0.f, cols, m.stream);
  }
  if (R->want_stats) {
    R->st.ring = kStatsRing;
    R->st.max_blocks = stats_max_blocks(m);
    MLEM_HIP(hipMalloc(&R->st.partials, sizeof(double2) * R->st.max_blocks));
    R->st.counter = words;
    R->st.results = reinterpret_cast<double2*>(R->buf + ores);
  }
  launch_fill(reinterpret_cast<float*>(words), 0.f, 8, m.stream);
  // sinogram into device row order (r is free until the first iteration)
  int32_t* ystage = reinterpret_cast<int32_t*>(R->r);
  h2d(ystage, y, 4ull * rows, m.stream);
  rows_to_device(m, (const int32_t*)ystage, R->y, m.stream);
  // initImage (seqcsr4mlem.cpp:52-66); the norm's double sum was taken in
  // index order at open.
  double sumin = 0.0;
  if (rows < kHostSumRows) {
    sumin = host_count_sum(y, rows);
  } else {
    CountSum cs;
    CountSum* dsum = reinterpret_cast<CountSum*>(words + 4);
    launch_count_sums(ystage, rows, 1, dsum, m.stream);
    d2h(&cs, dsum, sizeof(cs), m.stream);
    MLEM_HIP(hipStreamSynchronize(m.stream));
    sumin = cs.exact() ? (double)cs.sum : host_count_sum(y, rows);
  }
  if (sumin_out) *sumin_out = sumin;
  if (o->init == MLEM_INIT_GIVEN) {
    h2d(R->xs, x0, 4ull * cols, m.stream);
    to_device_cols(m, R->xs, R->x, m.stream);
  } else {
    const float initial = (float)(sumin / m.sumnorm);
    if (initial_out) *initial_out = initial;
    launch_fill(R->x, initial, cols, m.stream);
  }
  MLEM_HIP(hipStreamSynchronize(m.stream));
  return R.release();
}

// Current image in file voxel order into host memory (enqueued, not synced).
void read_image(mlem_recon* R, float* host) {
  DevMatrix& m = R->mat->m;
  to_file_cols(m, R->x, R->xs, m.stream);
  d2h(host, R->xs, 4ull * m.cols, m.stream);
}

bool file_exists(const std::string& p) {
  struct stat st;
  return stat(p.c_str(), &st) == 0;
}

}  // namespace

// ----------------------------------------------------------------- C ABI --
extern "C" {

const char* mlem_last_error(void) { return g_error.c_str(); }

const char* mlem_version(void) { return "mlem-amd 0.1 gfx950"; }

int mlem_open(const char* path, unsigned flags, mlem_matrix** out) {
  return guarded([&] {
    if (!path || !out) raise(MLEM_EINVAL, "null argument");
    *out = nullptr;
    Csr4Header hd;
    std::vector<uint64_t> rowidx;
    int fd = -1;
    csr4_read_header(path, hd, rowidx, &fd);
    struct FdClose {
      int fd;
      ~FdClose() {
        if (fd >= 0) close(fd);
      }
    } fdc{fd};
    auto t0 = std::chrono::steady_clock::now();
    const std::string fn(path);
    auto read_at = [&](void* dst, uint64_t off, uint64_t n) {
      char* p = static_cast<char*>(dst);
      uint64_t done = 0;
      while (done < n) {
        ssize_t got = pread(fd, p + done, n - done, (off_t)(hd.dataOffset + off + done));
        if (got <= 0) raise(MLEM_EIO, "Cannot read matrix elements from " + fn);
        done += (uint64_t)got;
      }
    };
    std::unique_ptr<mlem_matrix> h;
    if ((flags & MLEM_OPEN_EXPAND_SYMMETRY) && (hd.flags & 7u)) {
      // regenerate the omitted elements on the host, then upload the full matrix
      std::vector<Csr4Element> el(hd.nnz);
      if (hd.nnz) read_at(el.data(), 0, 8ull * hd.nnz);
      std::vector<uint64_t> xrow;
      std::vector<Csr4Element> xel;
      expand_symmetry(hd.scanner, hd.flags & 7u, hd.nRows, hd.nColumns, rowidx, el.data(), xrow,
                      xel);
      el.clear();
      el.shrink_to_fit();
      h.reset(new_matrix(hd.nRows, hd.nColumns, xel.size()));
      upload_rowidx(h->m, xrow.data());
      const char* src = reinterpret_cast<const char*>(xel.data());
      stream_to_device(h->m.csr, 8ull * xel.size(), h->m.device, h->m.stream,
                       [&](void* dst, uint64_t off, uint64_t n) { std::memcpy(dst, src + off, n); });
      h->m.symflags = 0;  // the matrix in HBM is complete
    } else {
      h.reset(new_matrix(hd.nRows, hd.nColumns, hd.nnz));
      upload_rowidx(h->m, rowidx.data());
      stream_to_device(h->m.csr, 8ull * hd.nnz, h->m.device, h->m.stream, read_at);
      h->m.symflags = hd.flags & 7u;
    }
    h->m.grid[0] = hd.scanner.grid[0];
    h->m.grid[1] = hd.scanner.grid[1];
    h->m.grid[2] = hd.scanner.grid[2];
    h->load_seconds = seconds_since(t0);
    finish_open(h.get(), flags);
    *out = h.release();
  });
}

int mlem_probe(const char* path, uint32_t* rows, uint32_t* cols, uint64_t* nnz, uint32_t grid[3],
               uint32_t* symflags) {
  return guarded([&] {
    if (!path) raise(MLEM_EINVAL, "null argument");
    Csr4Header hd;
    std::vector<uint64_t> rowidx;
    csr4_read_header(path, hd, rowidx, nullptr);
    if (rows) *rows = hd.nRows;
    if (cols) *cols = hd.nColumns;
    if (nnz) *nnz = hd.nnz;
    if (grid)
      for (int k = 0; k < 3; ++k) grid[k] = hd.scanner.grid[k];
    if (symflags) *symflags = hd.flags & 7u;
  });
}

int mlem_expand_symmetry_file(const char* in_path, const char* out_path) {
  return guarded([&] {
    if (!in_path || !out_path) raise(MLEM_EINVAL, "null argument");
    Csr4Header hd;
    std::vector<uint64_t> rowidx;
    int fd = -1;
    csr4_read_header(in_path, hd, rowidx, &fd);
    struct FdClose {
      int fd;
      ~FdClose() {
        if (fd >= 0) close(fd);
      }
    } fdc{fd};
    std::vector<Csr4Element> el(hd.nnz);
    const uint64_t bytes = 8ull * hd.nnz;
    char* p = reinterpret_cast<char*>(el.data());
    for (uint64_t done = 0; done < bytes;) {
      ssize_t got = pread(fd, p + done, bytes - done, (off_t)(hd.dataOffset + done));
      if (got <= 0) raise(MLEM_EIO, std::string("Cannot read matrix elements from ") + in_path);
      done += (uint64_t)got;
    }
    if (!(hd.flags & 7u)) {
      csr4_write(out_path, hd.flags, hd.nRows, hd.nColumns, hd.nnz, hd.scanner, rowidx.data(),
                 el.data());
      return;
    }
    std::vector<uint64_t> xrow;
    std::vector<Csr4Element> xel;
    expand_symmetry(hd.scanner, hd.flags & 7u, hd.nRows, hd.nColumns, rowidx, el.data(), xrow,
                    xel);
    csr4_write(out_path, (uint8_t)(hd.flags & ~7u), hd.nRows, hd.nColumns, xel.size(),
               hd.scanner, xrow.data(), xel.data());
  });
}

int mlem_open_host(uint32_t rows, uint32_t cols, uint64_t nnz, const uint64_t* rowidx,
                   const void* elements, const uint32_t grid[3], unsigned flags,
                   mlem_matrix** out) {
  return guarded([&] {
    if (!out || (rows && !rowidx) || (nnz && !elements)) raise(MLEM_EINVAL, "null argument");
    *out = nullptr;
    csr4_check_rowidx(rowidx, rows, nnz);
    auto t0 = std::chrono::steady_clock::now();
    std::unique_ptr<mlem_matrix> h(new_matrix(rows, cols, nnz));
    if (grid)
      for (int k = 0; k < 3; ++k) h->m.grid[k] = grid[k];
    upload_rowidx(h->m, rowidx);
    const char* src = static_cast<const char*>(elements);
    stream_to_device(h->m.csr, 8ull * nnz, h->m.device, h->m.stream,
                     [&](void* dst, uint64_t off, uint64_t n) { std::memcpy(dst, src + off, n); });
    h->load_seconds = seconds_since(t0);
    finish_open(h.get(), flags);
    *out = h.release();
  });
}

namespace {

// Handle of a streamed matrix: no device CSR/CSC, the row blocks in pinned
// host memory; column sums by a streamed EXACT backprojection of ones, which
// adds every column's values in ascending row order (calcColumnSums,
// seqcsr4mlem.cpp:37-49).
mlem_matrix* open_streamed(uint32_t rows, uint32_t cols, uint64_t nnz, const uint64_t* rowidx,
                           const ElementFetch& fetch, const uint32_t grid[3], unsigned flags,
                           uint64_t block_bytes, uint64_t resident_bytes) {
  if (flags & (MLEM_OPEN_FP16 | MLEM_OPEN_BF16))
    raise(MLEM_EINVAL, "streamed matrices hold fp32 values");
  if (rows == 0xFFFFFFFFu || cols == 0xFFFFFFFFu) raise(MLEM_EINVAL, "dimension too large");
  std::unique_ptr<mlem_matrix> h(new mlem_matrix());
  DevMatrix& m = h->m;
  m.rows = rows;
  m.cols = cols;
  m.nnz = nnz;
  if (grid)
    for (int k = 0; k < 3; ++k) m.grid[k] = grid[k];
  select_device(&m.device, &m.cus);
  MLEM_HIP(hipStreamCreateWithFlags(&m.stream, hipStreamNonBlocking));
  auto t0 = std::chrono::steady_clock::now();
  m.streamed =
      build_streamed(rows, cols, nnz, rowidx, fetch, block_bytes, resident_bytes, m.stream);
  h->load_seconds = seconds_since(t0);
  t0 = std::chrono::steady_clock::now();
  MLEM_HIP(hipMalloc(&m.norm, 4ull * std::max<uint32_t>(cols, 1)));
  ensure_scratch(m);
  launch_fill(m.norm, 0.f, cols, m.stream);
  launch_fill(m.sr, 1.f, rows, m.stream);
  stream_bwd_add(m, true, m.sr, m.norm, m.stream);
  std::vector<float> norm(cols);
  d2h(norm.data(), m.norm, 4ull * cols, m.stream);
  MLEM_HIP(hipStreamSynchronize(m.stream));
  double sn = 0.0;  // initImage's double sum, index order (seqcsr4mlem.cpp:55-56)
  for (uint32_t j = 0; j < cols; ++j) sn += norm[j];
  m.sumnorm = sn;
  h->norm_seconds = seconds_since(t0);
  m.fwd = make_launch(kGroups, m.streamed->lanes_fwd);
  m.bwd = make_launch(kGroups, m.streamed->lanes_bwd);
  m.scatter = m.bwd;
  return h.release();
}

}  // namespace

int mlem_open_streamed(const char* path, unsigned flags, uint64_t block_bytes,
                       uint64_t resident_bytes, mlem_matrix** out) {
  return guarded([&] {
    if (!path || !out) raise(MLEM_EINVAL, "null argument");
    *out = nullptr;
    Csr4Header hd;
    std::vector<uint64_t> rowidx;
    int fd = -1;
    csr4_read_header(path, hd, rowidx, &fd);
    struct FdClose {
      int fd;
      ~FdClose() {
        if (fd >= 0) close(fd);
      }
    } fdc{fd};
    const std::string fn(path);
    std::unique_ptr<mlem_matrix> h;
    if ((flags & MLEM_OPEN_EXPAND_SYMMETRY) && (hd.flags & 7u)) {
      std::vector<Csr4Element> el(hd.nnz);
      char* p = reinterpret_cast<char*>(el.data());
      for (uint64_t done = 0, n = 8ull * hd.nnz; done < n;) {
        ssize_t got = pread(fd, p + done, n - done, (off_t)(hd.dataOffset + done));
        if (got <= 0) raise(MLEM_EIO, "Cannot read matrix elements from " + fn);
        done += (uint64_t)got;
      }
      std::vector<uint64_t> xrow;
      std::vector<Csr4Element> xel;
      expand_symmetry(hd.scanner, hd.flags & 7u, hd.nRows, hd.nColumns, rowidx, el.data(), xrow,
                      xel);
      el.clear();
      el.shrink_to_fit();
      const char* src = reinterpret_cast<const char*>(xel.data());
      h.reset(open_streamed(
          hd.nRows, hd.nColumns, xel.size(), xrow.data(),
          [&](void* dst, uint64_t first, uint64_t count) {
            std::memcpy(dst, src + 8 * first, 8 * count);
          },
          hd.scanner.grid, flags, block_bytes, resident_bytes));
    } else {
      h.reset(open_streamed(
          hd.nRows, hd.nColumns, hd.nnz, rowidx.data(),
          [&](void* dst, uint64_t first, uint64_t count) {
            char* p = static_cast<char*>(dst);
            const uint64_t n = 8 * count;
            for (uint64_t done = 0; done < n;) {
              ssize_t got = pread(fd, p + done, n - done,
                                  (off_t)(hd.dataOffset + 8 * first + done));
              if (got <= 0) raise(MLEM_EIO, "Cannot read matrix elements from " + fn);
              done += (uint64_t)got;
            }
          },
          hd.scanner.grid, flags, block_bytes, resident_bytes));
      h->m.symflags = hd.flags & 7u;
    }
    *out = h.release();
  });
}

int mlem_open_host_streamed(uint32_t rows, uint32_t cols, uint64_t nnz, const uint64_t* rowidx,
                            const void* elements, const uint32_t grid[3], unsigned flags,
                            uint64_t block_bytes, uint64_t resident_bytes, mlem_matrix** out) {
  return guarded([&] {
    if (!out || (rows && !rowidx) || (nnz && !elements)) raise(MLEM_EINVAL, "null argument");
    *out = nullptr;
    csr4_check_rowidx(rowidx, rows, nnz);
    const char* src = static_cast<const char*>(elements);
    *out = open_streamed(
        rows, cols, nnz, rowidx,
        [&](void* dst, uint64_t first, uint64_t count) {
          std::memcpy(dst, src + 8 * first, 8 * count);
        },
        grid, flags, block_bytes, resident_bytes);
  });
}

int mlem_stream_passes(const mlem_matrix* h, int* passes) {
  return guarded([&] {
    if (!h || !passes) raise(MLEM_EINVAL, "null argument");
    const StreamedMatrix* S = h->m.streamed;
    *passes = !S ? 0 : S->csc_dev ? 1 : 2;
  });
}

int mlem_stream_blocks(const mlem_matrix* h, uint32_t* blocks, uint32_t* resident) {
  return guarded([&] {
    if (!h || !blocks) raise(MLEM_EINVAL, "null argument");
    const StreamedMatrix* S = h->m.streamed;
    *blocks = S ? (uint32_t)S->blocks.size() : 0u;
    if (resident) {
      *resident = 0;
      if (S)
        for (const StreamBlock& B : S->blocks) *resident += B.resident ? 1u : 0u;
    }
  });
}

void mlem_close(mlem_matrix* m) {
  if (!m) return;
  if (m->m.stream) (void)hipStreamSynchronize(m->m.stream);
  delete m;
}

int mlem_dims(const mlem_matrix* h, uint32_t* rows, uint32_t* cols, uint64_t* nnz) {
  return guarded([&] {
    if (!h) raise(MLEM_EINVAL, "null matrix handle");
    if (rows) *rows = h->m.rows;
    if (cols) *cols = h->m.cols;
    if (nnz) *nnz = h->m.nnz;
  });
}

int mlem_geometry(const mlem_matrix* h, uint32_t grid[3], uint32_t* symflags) {
  return guarded([&] {
    if (!h) raise(MLEM_EINVAL, "null matrix handle");
    if (grid)
      for (int k = 0; k < 3; ++k) grid[k] = h->m.grid[k];
    if (symflags) *symflags = h->m.symflags;
  });
}

void* mlem_stream(mlem_matrix* h) { return h ? (void*)h->m.stream : nullptr; }

int mlem_column_sums(mlem_matrix* h, float* norm, uint32_t cols) {
  return guarded([&] {
    check_dims(h, h ? h->m.rows : 0, cols);
    if (!norm && cols) raise(MLEM_EINVAL, "null output");
    ensure_scratch(h->m);
    to_file_cols(h->m, h->m.norm, h->m.tx, h->m.stream);
    d2h(norm, h->m.tx, 4ull * cols, h->m.stream);
    MLEM_HIP(hipStreamSynchronize(h->m.stream));
  });
}

int mlem_init_image(mlem_matrix* h, const float* norm, uint32_t cols, const int32_t* y,
                    uint32_t rows, float* x, float* initial) {
  return guarded([&] {
    check_dims(h, rows, cols);
    if ((cols && (!norm || !x)) || (rows && !y)) raise(MLEM_EINVAL, "null argument");
    // initImage is two sequential double sums and one division on the host,
    // exactly as seqcsr4mlem.cpp:52-66; the broadcast runs on the device.
    double sumnorm = 0.0, sumin = 0.0;
    for (uint32_t j = 0; j < cols; ++j) sumnorm += norm[j];
    for (uint32_t i = 0; i < rows; ++i) sumin += y[i];
    const float v = (float)(sumin / sumnorm);
    if (initial) *initial = v;
    DevMatrix& m = h->m;
    ensure_scratch(m);
    launch_fill(m.sx, v, cols, m.stream);
    d2h(x, m.sx, 4ull * cols, m.stream);
    MLEM_HIP(hipStreamSynchronize(m.stream));
  });
}

int mlem_fwproj(mlem_matrix* h, const float* x, uint32_t cols, float* f, uint32_t rows, int mode) {
  return guarded([&] {
    check_dims(h, rows, cols);
    if ((cols && !x) || (rows && !f)) raise(MLEM_EINVAL, "null argument");
    DevMatrix& m = h->m;
    ensure_scratch(m);
    h2d(m.tx, x, 4ull * cols, m.stream);
    to_device_cols(m, m.tx, m.sx, m.stream);
    launch_fwd(m, mode == MLEM_MODE_EXACT ? MLEM_MODE_EXACT : MLEM_MODE_FAST, m.sx, nullptr, m.sf,
               false, nullptr, m.stream);
    rows_to_file(m, (const float*)m.sf, m.tf, m.stream);
    d2h(f, m.tf, 4ull * rows, m.stream);
    MLEM_HIP(hipStreamSynchronize(m.stream));
  });
}

int mlem_correl(mlem_matrix* h, const float* f, const int32_t* y, float* r, uint32_t rows) {
  return guarded([&] {
    check_dims(h, rows, h ? h->m.cols : 0);
    if (rows && (!f || !y || !r)) raise(MLEM_EINVAL, "null argument");
    DevMatrix& m = h->m;
    ensure_scratch(m);
    h2d(m.sf, f, 4ull * rows, m.stream);
    h2d(m.sy, y, 4ull * rows, m.stream);
    launch_correl(rows, m.sf, m.sy, m.sr, m.stream);
    d2h(r, m.sr, 4ull * rows, m.stream);
    MLEM_HIP(hipStreamSynchronize(m.stream));
  });
}

int mlem_bkproj(mlem_matrix* h, const float* r, uint32_t rows, float* u, uint32_t cols, int mode) {
  return guarded([&] {
    check_dims(h, rows, cols);
    if ((rows && !r) || (cols && !u)) raise(MLEM_EINVAL, "null argument");
    DevMatrix& m = h->m;
    ensure_scratch(m);
    h2d(m.tf, r, 4ull * rows, m.stream);
    rows_to_device(m, (const float*)m.tf, m.sr, m.stream);
    launch_scale_rows(m, m.sr, m.stream);  // 16-bit values: A^T r = Q^T (s r)
    if (mode == MLEM_MODE_ATOMIC) {
      launch_fill(m.su, 0.f, cols, m.stream);
      launch_scatter(m, m.sr, m.su, m.stream);
    } else {
      launch_bwd(m, mode, m.sr, m.norm, m.su, false, m.stream);
    }
    to_file_cols(m, m.su, m.tx, m.stream);
    d2h(u, m.tx, 4ull * cols, m.stream);
    MLEM_HIP(hipStreamSynchronize(m.stream));
  });
}

int mlem_update(mlem_matrix* h, const float* u, const float* norm, float* x, uint32_t cols) {
  return guarded([&] {
    check_dims(h, h ? h->m.rows : 0, cols);
    if (cols && (!u || !norm || !x)) raise(MLEM_EINVAL, "null argument");
    DevMatrix& m = h->m;
    ensure_scratch(m);
    float* dn = m.tx;  // elementwise: file order throughout
    h2d(m.su, u, 4ull * cols, m.stream);
    h2d(dn, norm, 4ull * cols, m.stream);
    h2d(m.sx, x, 4ull * cols, m.stream);
    launch_update(cols, m.su, dn, m.sx, false, m.stream);
    d2h(x, m.sx, 4ull * cols, m.stream);
    MLEM_HIP(hipStreamSynchronize(m.stream));
  });
}

void mlem_options_default(mlem_options* o) {
  if (!o) return;
  std::memset(o, 0, sizeof(*o));
  o->mode = MLEM_MODE_FAST;
  o->init = MLEM_INIT_REFERENCE;
  o->use_graph = 1;
}

int mlem_recon_create(mlem_matrix* h, const int32_t* y, uint32_t rows, const float* x0,
                      uint32_t cols, const mlem_options* opts, mlem_recon** out) {
  return guarded([&] {
    if (!out) raise(MLEM_EINVAL, "null argument");
    *out = create_recon(h, y, rows, x0, cols, opts, nullptr, nullptr);
  });
}

void mlem_recon_destroy(mlem_recon* r) {
  if (!r) return;
  if (r->mat && r->mat->m.stream) (void)hipStreamSynchronize(r->mat->m.stream);
  delete r;
}

int mlem_recon_run(mlem_recon* R, int iterations) {
  return guarded([&] {
    if (!R || iterations < 0) raise(MLEM_EINVAL, "bad argument");
    run_iterations(R, iterations);
  });
}

int mlem_recon_run_timed(mlem_recon* R, int iterations, float* kf, float* kb, float* span) {
  return guarded([&] {
    if (!R || iterations < 0) raise(MLEM_EINVAL, "bad argument");
    if (R->want_stats) raise(MLEM_ESTATE, "timed runs do not record statistics");
    DevMatrix& m = R->mat->m;
    const size_t need = 2 * (size_t)iterations + 1;
    while (R->events.size() < need) {
      hipEvent_t e;
      MLEM_HIP(hipEventCreate(&e));
      R->events.push_back(e);
    }
    hipEvent_t* ev = R->events.data();
    MLEM_HIP(hipEventRecord(ev[0], m.stream));
    for (int i = 0; i < iterations; ++i) {
      if (R->mode == MLEM_MODE_ATOMIC) {
        if (m.streamed) {  // one fused pass: its time counts as the forward's
          stream_fwd_scatter(m, R->x, R->y, R->r, R->u, nullptr, m.stream);
          MLEM_HIP(hipEventRecord(ev[2 * i + 1], m.stream));
        } else {
          launch_fwd(m, MLEM_MODE_FAST, R->x, R->y, R->r, true, nullptr, m.stream);
          MLEM_HIP(hipEventRecord(ev[2 * i + 1], m.stream));
          launch_scatter(m, R->r, R->u, m.stream);
        }
        launch_update(m.cols, R->u, m.norm, R->x, true, m.stream);
      } else {
        launch_fwd(m, R->mode, R->x, R->y, R->r, true, nullptr, m.stream);
        MLEM_HIP(hipEventRecord(ev[2 * i + 1], m.stream));
        launch_bwd(m, R->mode, R->r, m.norm, R->x, true, m.stream);
      }
      MLEM_HIP(hipEventRecord(ev[2 * i + 2], m.stream));
    }
    MLEM_HIP(hipEventSynchronize(ev[2 * iterations]));
    for (int i = 0; i < iterations; ++i) {
      float a = 0.f, b = 0.f;
      MLEM_HIP(hipEventElapsedTime(&a, ev[2 * i], ev[2 * i + 1]));
      MLEM_HIP(hipEventElapsedTime(&b, ev[2 * i + 1], ev[2 * i + 2]));
      if (kf) kf[i] = a;
      if (kb) kb[i] = b;
    }
    if (span) MLEM_HIP(hipEventElapsedTime(span, ev[0], ev[2 * iterations]));
    R->done += iterations;
  });
}

int mlem_recon_image(mlem_recon* R, float* x, uint32_t cols) {
  return guarded([&] {
    if (!R) raise(MLEM_EINVAL, "null handle");
    check_dims(R->mat, R->mat->m.rows, cols);
    if (cols && !x) raise(MLEM_EINVAL, "null output");
    read_image(R, x);
    MLEM_HIP(hipStreamSynchronize(R->mat->m.stream));
  });
}

int mlem_recon_iterations(const mlem_recon* R) { return R ? R->done : -1; }

int mlem_reconstruct(mlem_matrix* h, const int32_t* y, uint32_t rows, float* x, uint32_t cols,
                     int iterations, const mlem_options* opts) {
  return guarded([&] {
    check_dims(h, rows, cols);
    if (iterations < 0) raise(MLEM_EINVAL, "negative iteration count");
    if (cols && !x) raise(MLEM_EINVAL, "null image");
    mlem_options o;
    if (opts)
      o = *opts;
    else
      mlem_options_default(&o);
    const bool verbose = o.verbose != 0;
    const std::string dir = o.checkpoint_dir && *o.checkpoint_dir ? o.checkpoint_dir : ".";
    const std::string imgChk = dir + "/img.chkpt", iterChk = dir + "/iter.chkpt";
    if (verbose)
      std::cout << "Calculated norm, elapsed time: " << h->norm_seconds << "s\n";

    if (o.checkpoint_interval < MLEM_CHECKPOINT_RESTORE_ONLY)
      raise(MLEM_EINVAL, "invalid checkpoint interval " + std::to_string(o.checkpoint_interval));
    // Restart from a complete checkpoint whenever both files exist, whatever
    // the interval (mpicsr4mlem.cpp:536-553); an interval of 0 is the
    // sequential driver, which has no checkpoints.
    int start = 0;
    std::vector<float> restored;
    if (o.checkpoint_interval != 0) {
      const bool hi = file_exists(imgChk), ht = file_exists(iterChk);
      if (hi && ht) {
        restored = read_raw_f32(imgChk);
        if (restored.size() != cols) raise(MLEM_EIO, "Mismatch element number " + imgChk);
        std::vector<int32_t> it = read_raw_i32(iterChk);
        if (it.size() < 1) raise(MLEM_EIO, "Cannot open file " + iterChk);
        start = it[0];
        if (start < 0) raise(MLEM_EIO, "invalid iteration in " + iterChk);
        if (verbose) std::cout << "I got Checkpoint at iteration " << start << "\n";
      } else if (hi || ht) {
        if (verbose) std::cout << "omitted incomplete checkpoint\n";
      }
    }
    mlem_options co = o;
    const float* x0 = x;
    if (!restored.empty()) {
      co.init = MLEM_INIT_GIVEN;
      x0 = restored.data();
    }
    float initial = 0.f;
    double sumin = 0.0;
    std::unique_ptr<mlem_recon> R(create_recon(h, y, rows, x0, cols, &co, &initial, &sumin));
    if (verbose && co.init == MLEM_INIT_REFERENCE)
      std::cout << "INIT: sumnorm=" << h->m.sumnorm << ", sumin=" << sumin
                << ", initial value=" << initial << std::endl;
    if (verbose) std::cout << "Starting " << iterations - std::min(start, iterations) << " MLEM iterations" << std::endl;

    const bool per_iter = verbose || o.checkpoint_interval > 0;
    std::vector<float> img(per_iter ? cols : 0);
    auto t0 = std::chrono::steady_clock::now();
    if (!per_iter) {
      run_iterations(R.get(), std::max(0, iterations - start));
    } else {
      for (int iter = start; iter < iterations; ++iter) {
        run_iterations(R.get(), 1);
        const double el = seconds_since(t0);
        read_image(R.get(), img.data());
        MLEM_HIP(hipStreamSynchronize(h->m.stream));
        if (verbose) {
          // per-iteration statistics of seqcsr4mlem.cpp:172-185
          int cz = 0, cs = 0;
          float s = 0.0f;
          for (uint32_t j = 0; j < cols; ++j) {
            s += img[j];
            const int c = std::fpclassify(img[j]);
            if (c == FP_ZERO) ++cz;
            if (c == FP_SUBNORMAL) ++cs;
          }
          std::cout << "Finished iteration " << iter + 1 << ", ";
          std::cout << " image sum: " << s << ", ";
          std::cout << "elapsed time: " << el << "s\n";
          std::cout << "Zeros: " << cz << " (" << (float)cz / cols * 100.0 << " %), "
                    << " subnormals: " << cs << " (" << (float)cs / cols * 100.0 << " %)\n";
        }
        if (o.checkpoint_interval > 0 && (iter + 1) % o.checkpoint_interval == 0) {
          write_raw(imgChk, img.data(), 4ull * cols, true);
          const int32_t next = iter + 1;
          write_raw(iterChk, &next, sizeof(next), true);
        }
        t0 = std::chrono::steady_clock::now();
      }
    }
    read_image(R.get(), x);
    MLEM_HIP(hipStreamSynchronize(h->m.stream));
    const int ran = (int)R->loglik.size();
    for (int k = 0; k < ran; ++k) {
      if (o.loglik) o.loglik[start + k] = R->loglik[k];
      if (o.fwd_total) o.fwd_total[start + k] = R->fwdtot[k];
    }
    if (o.checkpoint_interval > 0) {  // clean exit (mpicsr4mlem.cpp:656-660)
      std::remove(imgChk.c_str());
      std::remove(iterChk.c_str());
    }
  });
}

int mlem_get_launch(const mlem_matrix* h, int* fk, int* fp, int* bk, int* bp) {
  return guarded([&] {
    if (!h) raise(MLEM_EINVAL, "null matrix handle");
    const GroupLaunch &f = h->m.fwd, &b = h->m.bwd;
    if (fk) *fk = f.kind;
    if (fp) *fp = f.kind == kGroups ? f.lanes : f.ept;
    if (bk) *bk = b.kind;
    if (bp) *bp = b.kind == kGroups ? b.lanes : b.ept;
  });
}

int mlem_set_launch(mlem_matrix* h, int fk, int fp, int bk, int bp) {
  return guarded([&] {
    if (!h) raise(MLEM_EINVAL, "null matrix handle");
    if (h->m.streamed) raise(MLEM_EINVAL, "streamed matrices have a fixed launch configuration");
    const GroupLaunch f = named_launch(fk, fp, h->m.fwd_open),
                      b = named_launch(bk, bp, h->m.bwd_open);
    ++h->m.launch_gen;
    h->m.fwd = f;
    h->m.bwd = b;
    prepare_tiles(h->m, h->m.stream);
  });
}

int mlem_autotune(mlem_matrix* h) {
  return guarded([&] {
    if (!h) raise(MLEM_EINVAL, "null matrix handle");
    if (h->m.streamed) raise(MLEM_EINVAL, "streamed matrices have a fixed launch configuration");
    ++h->m.launch_gen;
    autotune(h->m);
  });
}

int mlem_calibration_copy(size_t bytes, int repeats, float* ms) {
  return guarded([&] {
    if (bytes == 0 || bytes % 16 != 0 || repeats <= 0) raise(MLEM_EINVAL, "bad size");
    int dev = 0, cus = 0;
    select_device(&dev, &cus);
    void *a = nullptr, *b = nullptr;
    hipStream_t s = nullptr;
    struct C {
      void** a;
      void** b;
      hipStream_t* s;
      ~C() {
        if (*a) (void)hipFree(*a);
        if (*b) (void)hipFree(*b);
        if (*s) (void)hipStreamDestroy(*s);
      }
    } c{&a, &b, &s};
    MLEM_HIP(hipStreamCreateWithFlags(&s, hipStreamNonBlocking));
    MLEM_HIP(hipMalloc(&a, bytes));
    MLEM_HIP(hipMalloc(&b, bytes));
    MLEM_HIP(hipMemsetAsync(a, 1, bytes, s));
    float t = time_variant(s, [&] { launch_copy((const uint4*)a, (uint4*)b, bytes / 16, s); }, repeats);
    if (ms) *ms = t;
  });
}

int mlem_device_sync(void) {
  return guarded([&] { MLEM_HIP(hipDeviceSynchronize()); });
}

}  // extern "C"
