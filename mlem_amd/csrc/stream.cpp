// stream.cpp — out-of-core matrices: row blocks in pinned host memory, each
// projection streaming its part of every block over PCIe.
//
// Reference counterpart: mlem_cuda/versions/version_7.cu:205-260 (the matrix
// split into row parts that are copied to the device in turn before each
// projection) with the splitting of mlem_cuda/helper_files/helper_v_7_8.cu:4-72
// (parts sized by the free device memory, balanced by elements). Here every
// block also carries the CSC of its rows, so the backprojection gathers per
// column like the in-core path instead of scattering; a column's sum continues
// from block to block in ascending row order, which keeps EXACT mode equal to
// the sequential sums of seqcsr4mlem.cpp:37-49,108-120.
#include <algorithm>
#include <atomic>
#include <cstring>
#include <string>
#include <thread>
#include <vector>

#include "internal.hpp"
#include "mlem.h"

namespace mlem {

namespace {

uint64_t align16(uint64_t n) { return (n + 15) & ~15ull; }

// Largest element count of one block: the kernels address a block's elements
// with 32-bit offsets.
constexpr uint64_t kMaxBlockNnz = (1ull << 32) - 1024;

uint64_t pack_chunks(uint64_t nnz) { return (nnz + kPackChunk - 1) / kPackChunk; }
// Bytes between a packed part's row pointers and its first chunk.
uint64_t pack_front(uint64_t nnz) { return sizeof(PackHead) * pack_chunks(nnz) + 4 * kPackTable; }

// The steps between neighbouring elements' columns that get a code: the most
// frequent of a sample of 16 chunks.
void pack_table(const uint2* el, uint64_t nnz, uint32_t* table) {
  std::vector<uint32_t> d;
  const uint64_t n = pack_chunks(nnz), every = std::max<uint64_t>(1, n / 16);
  for (uint64_t c = 0; c < n; c += every) {
    const uint64_t e = std::min(nnz, (c + 1) * kPackChunk);
    for (uint64_t k = c * kPackChunk + 1; k < e; ++k) d.push_back(el[k].x - el[k - 1].x);
  }
  std::sort(d.begin(), d.end());
  std::vector<std::pair<uint32_t, uint32_t>> runs;  // {times, step}
  for (size_t i = 0; i < d.size();) {
    size_t j = i;
    while (j < d.size() && d[j] == d[i]) ++j;
    runs.emplace_back((uint32_t)(j - i), d[i]);
    i = j;
  }
  std::sort(runs.begin(), runs.end(), [](const auto& a, const auto& b) {
    return a.first != b.first ? a.first > b.first : a.second < b.second;
  });
  const size_t k = std::min<size_t>(runs.size(), kPackEscape);
  for (size_t i = 0; i < kPackTable; ++i) table[i] = k ? runs[std::min(i, k - 1)].second : 0;
}

// Packs the nnz elements at front + pack_front(nnz) in place (a chunk never grows,
// so its packed form ends before the next chunk's elements). Returns the end of
// the packed part.
char* pack_block(char* front, uint64_t nnz) {
  PackHead* heads = reinterpret_cast<PackHead*>(front);
  uint32_t* table = reinterpret_cast<uint32_t*>(heads + pack_chunks(nnz));
  char* const first = front + pack_front(nnz);
  const uint2* el = reinterpret_cast<const uint2*>(first);
  pack_table(el, nnz, table);
  constexpr uint32_t kSlots = 1024;  // open addressing: step -> code
  std::vector<uint32_t> key(kSlots), code(kSlots, kPackEscape);
  auto slot = [](uint32_t d) { return (d * 2654435761u) >> 22; };
  for (uint32_t c = 0; c < kPackEscape; ++c) {
    uint32_t h = slot(table[c]);
    while (code[h] != kPackEscape && key[h] != table[c]) h = (h + 1) % kSlots;
    if (code[h] != kPackEscape) continue;  // the table's filling
    key[h] = table[c];
    code[h] = c;
  }
  std::vector<uint2> raw(kPackChunk);
  std::vector<uint8_t> codes(kPackChunk);
  std::vector<uint32_t> steps(kPackChunk);
  char* out = first;
  for (uint64_t c = 0; c < pack_chunks(nnz); ++c) {
    const uint32_t m = (uint32_t)std::min<uint64_t>(kPackChunk, nnz - c * kPackChunk);
    std::copy(el + c * kPackChunk, el + c * kPackChunk + m, raw.begin());
    uint32_t prev = 0, ns = 0;
    for (uint32_t k = 0; k < m; ++k) {
      const uint32_t d = raw[k].x - prev;
      prev = raw[k].x;
      uint32_t h = slot(d);
      while (code[h] != kPackEscape && key[h] != d) h = (h + 1) % kSlots;
      codes[k] = (uint8_t)code[h];
      steps[ns] = d;
      ns += code[h] == kPackEscape;
    }
    std::fill(codes.begin() + m, codes.end(), (uint8_t)0);
    const uint64_t vb = align16(4ull * m), cb = align16(m), bytes = vb + cb + align16(4ull * ns);
    const bool keep = bytes >= 8ull * m;
    heads[c] = PackHead{(uint32_t)((out - first) / 16), m, keep ? kPackRaw : ns, 0};
    if (keep) {
      std::memcpy(out, raw.data(), 8ull * m);
      out += align16(8ull * m);
      continue;
    }
    uint32_t* v = reinterpret_cast<uint32_t*>(out);
    for (uint32_t k = 0; k < m; ++k) v[k] = raw[k].y;
    std::memcpy(out + vb, codes.data(), cb);
    std::memcpy(out + vb + cb, steps.data(), 4ull * ns);
    out += bytes;
  }
  return out;
}

}  // namespace

StreamedMatrix::~StreamedMatrix() {
  for (StreamBlock& b : blocks)
    if (b.resident) (void)hipFree(b.resident);
  for (int i = 0; i < 2; ++i) {
    if (copied[i]) (void)hipEventDestroy(copied[i]);
    if (freed[i]) (void)hipEventDestroy(freed[i]);
    if (dev[i]) (void)hipFree(dev[i]);
  }
  if (u) (void)hipFree(u);
  if (csc_dev) (void)hipFree(csc_dev);
  if (expand) (void)hipFree(expand);
  if (copy) (void)hipStreamDestroy(copy);
  if (host) (void)hipHostFree(host);
}

StreamedMatrix* build_streamed(uint32_t rows, uint32_t cols, uint64_t nnz,
                               const uint64_t* rowidx, const ElementFetch& fetch,
                               uint64_t block_bytes, uint64_t resident_bytes, hipStream_t s) {
  const uint64_t colpart = align16(4ull * ((uint64_t)cols + 1));
  if (block_bytes == 0) {
    // an eighth of the free device memory per part, as the reference sizes
    // its parts by cudaMemGetInfo (helper_v_7_8.cu:6-30): the two part
    // buffers and one block's device CSC with its sort scratch (about four
    // parts) then fit
    size_t freeb = 0, total = 0;
    MLEM_HIP(hipMemGetInfo(&freeb, &total));
    block_bytes = freeb / 8;
  }
  auto row_len = [&](uint32_t r) { return rowidx[r] - (r ? rowidx[r - 1] : 0); };

  // Greedy row blocks: both parts of a block fit `block_bytes`.
  std::unique_ptr<StreamedMatrix> S(new StreamedMatrix());
  uint64_t off = 0;
  for (uint32_t r0 = 0; r0 < rows || (rows == 0 && S->blocks.empty());) {
    StreamBlock B;
    B.row0 = r0;
    uint64_t n = 0;
    uint32_t r = r0;
    while (r < rows) {
      const uint64_t n2 = n + row_len(r);
      const uint64_t csr = align16(4ull * ((uint64_t)(r - r0) + 2)) + 8 * n2;
      const uint64_t csc = colpart + 8 * n2;
      if (r > r0 && (csr > block_bytes || csc > block_bytes || n2 > kMaxBlockNnz)) break;
      if (r == r0 && (csr > block_bytes || csc > block_bytes || n2 > kMaxBlockNnz))
        raise(MLEM_EINVAL, "block_bytes (" + std::to_string(block_bytes) + ") cannot hold row " +
                               std::to_string(r) + " and the column pointers of a block");
      n = n2;
      ++r;
    }
    B.rows = r - r0;
    B.nnz = n;
    B.csr_off = off;
    B.csr_bytes = align16(4ull * ((uint64_t)B.rows + 1)) + 8 * n;
    off += align16(B.csr_bytes + pack_front(n));
    B.csc_off = off;
    B.csc_bytes = colpart + 8 * n;
    off += align16(B.csc_bytes);
    S->blocks.push_back(B);
    if (rows == 0) break;
    r0 = r;
  }
  S->host_bytes = std::max<uint64_t>(off, 16);
  MLEM_HIP(hipHostMalloc((void**)&S->host, S->host_bytes, hipHostMallocDefault));

  // Blocks kept in device memory: the first ones whose two parts fit the
  // resident budget; only the others are streamed.
  uint64_t kept = 0, streamed_part = 0;
  for (StreamBlock& B : S->blocks) {
    const uint64_t both = align16(B.csr_bytes) + B.csc_bytes;
    if (kept + both <= resident_bytes && streamed_part == 0) {
      MLEM_HIP(hipMalloc((void**)&B.resident, both));
      kept += both;
    } else {
      const uint64_t packed = B.csr_bytes + pack_front(B.nnz) + 16;
      streamed_part = std::max(streamed_part, std::max(packed, B.csc_bytes));
      S->max_stream_nnz = std::max(S->max_stream_nnz, B.nnz);
    }
  }
  S->part_bytes = streamed_part;
  for (int i = 0; i < 2; ++i) {
    MLEM_HIP(hipMalloc((void**)&S->dev[i], std::max<uint64_t>(S->part_bytes, 16)));
    MLEM_HIP(hipEventCreateWithFlags(&S->copied[i], hipEventDisableTiming));
    MLEM_HIP(hipEventCreateWithFlags(&S->freed[i], hipEventDisableTiming));
    MLEM_HIP(hipEventRecord(S->freed[i], s));
  }
  MLEM_HIP(hipStreamCreateWithFlags(&S->copy, hipStreamNonBlocking));
  MLEM_HIP(hipMalloc((void**)&S->u, 4ull * std::max<uint32_t>(cols, 1)));
  MLEM_HIP(hipMemsetAsync(S->u, 0, 4ull * std::max<uint32_t>(cols, 1), s));
  if (S->max_stream_nnz > 0) {
    // device CSC of one streamed block; if it does not fit, iterations keep
    // streaming the host-built CSC parts
    S->csc_scratch_bytes = block_csc_scratch(S->max_stream_nnz, cols);
    const uint64_t bytes = colpart + align16(8 * S->max_stream_nnz) + S->csc_scratch_bytes;
    if (hipMalloc((void**)&S->csc_dev, bytes) != hipSuccess) {
      (void)hipGetLastError();
      S->csc_dev = nullptr;
    }
    // one block's elements unpacked, if they leave as much memory free as they
    // take (what the caller allocates next still fits); else no block is packed
    size_t freeb = 0, total = 0;
    MLEM_HIP(hipMemGetInfo(&freeb, &total));
    if (S->max_stream_nnz >= kPackMin && freeb / 16 >= S->max_stream_nnz &&
        hipMalloc((void**)&S->expand, 8 * S->max_stream_nnz) != hipSuccess) {
      (void)hipGetLastError();
      S->expand = nullptr;
    }
  }

  // Fill the blocks in parallel: CSR part from the source, CSC part by a
  // counting sort over the block's columns (rows ascending in every column).
  const unsigned nthreads = (unsigned)std::max<size_t>(
      1, std::min<size_t>({S->blocks.size(), 16, std::max(1u, std::thread::hardware_concurrency())}));
  std::atomic<uint64_t> bad{0};
  std::vector<std::string> errors(nthreads);
  auto work = [&](unsigned tid) {
    try {
      std::vector<uint32_t> next(cols);
      for (size_t b = tid; b < S->blocks.size(); b += nthreads) {
        StreamBlock& B = S->blocks[b];
        const bool pack = S->expand && !B.resident && B.nnz >= kPackMin;
        char* csr = S->host + B.csr_off;
        char* csc = S->host + B.csc_off;
        uint32_t* rp = reinterpret_cast<uint32_t*>(csr);
        const uint64_t base = B.row0 ? rowidx[B.row0 - 1] : 0;
        rp[0] = 0;
        for (uint32_t k = 0; k < B.rows; ++k) rp[k + 1] = (uint32_t)(rowidx[B.row0 + k] - base);
        char* front = csr + align16(4ull * ((uint64_t)B.rows + 1));
        uint2* el = reinterpret_cast<uint2*>(front + (pack ? pack_front(B.nnz) : 0));
        if (B.nnz) fetch(el, base, B.nnz);
        uint32_t* cp = reinterpret_cast<uint32_t*>(csc);
        std::fill(cp, cp + (uint64_t)cols + 1, 0u);
        uint64_t nbad = 0;
        for (uint64_t k = 0; k < B.nnz; ++k) {
          if (el[k].x >= cols)
            ++nbad;
          else
            ++cp[el[k].x + 1];
        }
        if (nbad) {
          bad += nbad;
          continue;
        }
        for (uint32_t j = 0; j < cols; ++j) cp[j + 1] += cp[j];
        std::copy(cp, cp + cols, next.begin());
        uint2* ce = reinterpret_cast<uint2*>(csc + colpart);
        for (uint32_t k = 0; k < B.rows; ++k)
          for (uint32_t e = rp[k]; e < rp[k + 1]; ++e)
            ce[next[el[e].x]++] = make_uint2(B.row0 + k, el[e].y);
        if (pack) B.packed_bytes = (uint64_t)(pack_block(front, B.nnz) - csr);
      }
    } catch (const ApiError& e) {
      errors[tid] = e.msg;
    } catch (const std::exception& e) {
      errors[tid] = e.what();
    }
  };
  std::vector<std::thread> pool;
  for (unsigned t = 1; t < nthreads; ++t) pool.emplace_back(work, t);
  work(0);
  for (auto& t : pool) t.join();
  for (const std::string& e : errors)
    if (!e.empty()) raise(MLEM_EIO, e);
  if (bad)
    raise(MLEM_EFORMAT, std::to_string(bad.load()) + " matrix elements have a column index >= " +
                            std::to_string(cols));

  for (StreamBlock& B : S->blocks)
    if (B.resident) {
      MLEM_HIP(hipMemcpyAsync(B.resident, S->host + B.csr_off, B.csr_bytes,
                              hipMemcpyHostToDevice, s));
      MLEM_HIP(hipMemcpyAsync(B.resident + align16(B.csr_bytes), S->host + B.csc_off,
                              B.csc_bytes, hipMemcpyHostToDevice, s));
    }
  // lane groups of about four elements per lane (4..64), as the in-core
  // lane-group kernels choose them
  auto lanes_for = [](double avg) {
    int g = 4;
    while (g < 64 && g * 4 < avg) g *= 2;
    return g;
  };
  const uint64_t nb = S->blocks.size();
  S->lanes_fwd = lanes_for(rows ? (double)nnz / rows : 1.0);
  S->lanes_bwd = lanes_for(cols && nb ? (double)nnz / ((double)cols * (double)nb) : 1.0);
  MLEM_HIP(hipStreamSynchronize(s));
  return S.release();
}

namespace {

// Run `kernel(block, pointers, elements)` for every block on stream s, the copy
// of each block's part (CSR or CSC) on the copy stream: block b waits for its
// copy, the copy into a buffer waits for the kernels of the block before. A
// packed part is unpacked first, after the kernels of the block before (on
// whatever stream they ran).
//
// What bounds it: the host link (52 GB/s). A packed part has 5.1 instead of 8
// bytes per element where rows are lines of response in file order (2.4 % of the
// codes are escapes); 67.4M elements a pass: 10.3 -> 6.9 ms.
template <class K>
void stream_pass(const DevMatrix& m, bool csc, K&& kernel, hipStream_t s) {
  StreamedMatrix& S = *m.streamed;
  const uint64_t colpart = align16(4ull * ((uint64_t)m.cols + 1));
  size_t n_streamed = 0;
  for (size_t b = 0; b < S.blocks.size(); ++b) {
    const StreamBlock& B = S.blocks[b];
    const uint64_t pointers = csc ? colpart : align16(4ull * ((uint64_t)B.rows + 1));
    if (B.resident) {  // in device memory: no copy
      const char* d = csc ? B.resident + align16(B.csr_bytes) : B.resident;
      kernel(B, reinterpret_cast<const uint32_t*>(d), reinterpret_cast<const uint2*>(d + pointers));
      continue;
    }
    const int i = (int)(n_streamed++ & 1);
    const bool packed = !csc && B.packed_bytes;
    const uint64_t off = csc ? B.csc_off : B.csr_off;
    const uint64_t n = csc ? B.csc_bytes : packed ? B.packed_bytes : B.csr_bytes;
    MLEM_HIP(hipStreamWaitEvent(S.copy, S.freed[i], 0));
    MLEM_HIP(hipMemcpyAsync(S.dev[i], S.host + off, n, hipMemcpyHostToDevice, S.copy));
    MLEM_HIP(hipEventRecord(S.copied[i], S.copy));
    MLEM_HIP(hipStreamWaitEvent(s, S.copied[i], 0));
    const uint2* el = reinterpret_cast<const uint2*>(S.dev[i] + pointers);
    if (packed) {
      MLEM_HIP(hipStreamWaitEvent(s, S.freed[i ^ 1], 0));
      launch_unpack(reinterpret_cast<const PackHead*>(S.dev[i] + pointers), B.nnz, S.expand, s);
      el = S.expand;
    }
    kernel(B, reinterpret_cast<const uint32_t*>(S.dev[i]), el);
    MLEM_HIP(hipEventRecord(S.freed[i], s));
  }
}

}  // namespace

void stream_fwd(const DevMatrix& m, int mode, const float* x, const int32_t* y, float* out,
                bool ratio, const StatsState* st, hipStream_t s) {
  const StreamedMatrix& S = *m.streamed;
  const bool exact = mode == MLEM_MODE_EXACT;
  stream_pass(
      m, false,
      [&](const StreamBlock& B, const uint32_t* rp, const uint2* el) {
        // every block launches (also an empty one): statistics expect one
        // result per block
        launch_fwd_block(rp, el, B.rows, S.lanes_fwd, exact, x, y ? y + B.row0 : nullptr,
                         out + B.row0, ratio, st, m.cus, s);
      },
      s);
}

void stream_bwd_add(const DevMatrix& m, bool exact, const float* r, float* u, hipStream_t s) {
  const StreamedMatrix& S = *m.streamed;
  if (m.cols == 0) return;
  stream_pass(
      m, true,
      [&](const StreamBlock&, const uint32_t* cp, const uint2* el) {
        launch_bwd_block_add(cp, el, m.cols, S.lanes_bwd, exact, r, u, m.cus, s);
      },
      s);
}

void stream_fwd_scatter(const DevMatrix& m, const float* x, const int32_t* y, float* r, float* u,
                        const StatsState* st, hipStream_t s) {
  const StreamedMatrix& S = *m.streamed;
  stream_pass(
      m, false,
      [&](const StreamBlock& B, const uint32_t* rp, const uint2* el) {
        launch_fwd_block(rp, el, B.rows, S.lanes_fwd, false, x, y + B.row0, r + B.row0, true, st,
                         m.cus, s);
        if (B.rows) launch_scatter_block(rp, el, B.rows, S.lanes_fwd, r + B.row0, u, m.cus, s);
      },
      s);
}

void stream_iteration(const DevMatrix& m, int mode, float* x, const int32_t* y, float* r,
                      const StatsState* st, hipStream_t s) {
  const StreamedMatrix& S = *m.streamed;
  if (!S.csc_dev) {
    stream_fwd(m, mode, x, y, r, true, st, s);
    stream_bwd(m, mode, r, m.norm, x, true, s);
    return;
  }
  const bool exact = mode == MLEM_MODE_EXACT;
  const uint64_t colpart = align16(4ull * ((uint64_t)m.cols + 1));
  uint32_t* colptr = reinterpret_cast<uint32_t*>(S.csc_dev);
  uint2* csc = reinterpret_cast<uint2*>(S.csc_dev + colpart);
  void* scratch = S.csc_dev + colpart + align16(8 * S.max_stream_nnz);
  launch_fill(S.u, 0.f, m.cols, s);
  stream_pass(
      m, false,
      [&](const StreamBlock& B, const uint32_t* rp, const uint2* el) {
        launch_fwd_block(rp, el, B.rows, S.lanes_fwd, exact, x, y + B.row0, r + B.row0, true, st,
                         m.cus, s);
        if (B.resident) {  // its CSC part is in device memory already (global rows)
          const char* c = B.resident + align16(B.csr_bytes);
          launch_bwd_block_add(reinterpret_cast<const uint32_t*>(c),
                               reinterpret_cast<const uint2*>(c + colpart), m.cols, S.lanes_bwd,
                               exact, r, S.u, m.cus, s);
        } else {  // block-local rows
          build_block_csc(rp, el, B.rows, m.cols, B.nnz, scratch, S.csc_scratch_bytes, colptr, csc,
                          s);
          launch_bwd_block_add(colptr, csc, m.cols, S.lanes_bwd, exact, r + B.row0, S.u, m.cus, s);
        }
      },
      s);
  launch_update(m.cols, S.u, m.norm, x, false, s);
}

void stream_bwd(const DevMatrix& m, int mode, const float* r, const float* norm, float* out,
                bool update, hipStream_t s) {
  float* acc = update ? m.streamed->u : out;
  launch_fill(acc, 0.f, m.cols, s);
  stream_bwd_add(m, mode == MLEM_MODE_EXACT, r, acc, s);
  if (update) launch_update(m.cols, acc, norm, out, false, s);
}

}  // namespace mlem
