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

uint64_t pack_chunks_of(uint64_t nnz) { return (nnz + kPackChunk - 1) / kPackChunk; }
// Bytes between a packed part's row pointers and its first chunk.
uint64_t pack_front(uint64_t nnz) { return sizeof(PackHead) * pack_chunks_of(nnz) + 4 * kPackTable; }

uint32_t step_hash(uint32_t d) { return d * 2654435761u; }

// The steps between neighbouring elements' columns that get a code: the most
// frequent of a sample of 16 chunks, counted in a hash table. pays: whether a block
// packed with them is expected to be at least a tenth smaller (7.25 of 8 bytes an
// element): else the copies would gain less than the packing costs at open.
struct PackSteps {
  uint32_t step[kPackTable];
  bool pays = false;
};
PackSteps pack_steps(const ElementFetch& fetch, uint64_t base, uint64_t nnz) {
  constexpr uint64_t kRuns = 16;
  constexpr uint32_t kBits = 17;  // twice the steps of the sample
  PackSteps t;
  std::vector<uint2> el(kPackChunk + 1), count(1u << kBits, make_uint2(0, 0));  // {step, times}
  uint64_t total = 0;
  for (uint64_t i = 0; i < kRuns; ++i) {
    const uint64_t at = nnz * i / kRuns, n = std::min<uint64_t>(el.size(), nnz - at);
    fetch(el.data(), base + at, n);
    for (uint64_t k = 1; k < n; ++k) {
      const uint32_t d = el[k].x - el[k - 1].x;
      uint32_t h = step_hash(d) >> (32 - kBits);
      while (count[h].y && count[h].x != d) h = (h + 1) & ((1u << kBits) - 1);
      count[h].x = d;
      ++count[h].y;
      ++total;
    }
  }
  std::vector<std::pair<uint32_t, uint32_t>> runs;  // {times, step}
  for (const uint2& c : count)
    if (c.y) runs.emplace_back(c.y, c.x);
  const size_t k = std::min<size_t>(runs.size(), kPackEscape);
  std::partial_sort(runs.begin(), runs.begin() + (std::ptrdiff_t)k, runs.end(),
                    [](const auto& a, const auto& b) {
                      return a.first != b.first ? a.first > b.first : a.second < b.second;
                    });
  uint64_t coded = 0;
  for (size_t i = 0; i < k; ++i) coded += runs[i].first;
  t.pays = total && 4.0 + 1.0 + 4.0 * (double)(total - coded) / (double)total <= 7.25;
  for (size_t i = 0; i < kPackTable; ++i) t.step[i] = k ? runs[std::min(i, k - 1)].second : 0;
  return t;
}

// Packs chunks c0 .. c1-1 of the nnz elements at front + pack_front(nnz) in place,
// from the place of chunk c0's elements on (a chunk never grows, so its packed
// form ends before the next chunk's elements). Returns the end of the packed chunks.
char* pack_chunks(char* front, uint64_t nnz, uint64_t c0, uint64_t c1, const PackSteps& t) {
  PackHead* heads = reinterpret_cast<PackHead*>(front);
  char* const first = front + pack_front(nnz);
  const uint2* el = reinterpret_cast<const uint2*>(first);
  constexpr uint32_t kSlots = 1024;  // open addressing: step -> code
  struct Slot {
    uint32_t step = 0, code = kPackEscape;
  };
  std::vector<Slot> slots(kSlots);
  auto find = [&](uint32_t d) {
    uint32_t h = step_hash(d) >> 22;
    while (slots[h].code != kPackEscape && slots[h].step != d) h = (h + 1) % kSlots;
    return h;
  };
  for (uint32_t c = 0; c < kPackEscape; ++c) {
    Slot& e = slots[find(t.step[c])];
    if (e.code == kPackEscape) e = Slot{t.step[c], c};  // (else the table's filling)
  }
  std::vector<uint8_t> codes(kPackChunk);
  std::vector<uint32_t> steps(kPackChunk);
  char* out = first + 8ull * kPackChunk * c0;
  for (uint64_t c = c0; c < c1; ++c) {
    const uint32_t m = (uint32_t)std::min<uint64_t>(kPackChunk, nnz - c * kPackChunk);
    const uint2* raw = el + c * kPackChunk;  // at `out` or beyond
    uint32_t prev = 0, ns = 0;
    for (uint32_t k = 0; k < m; ++k) {
      const uint32_t d = raw[k].x - prev;
      prev = raw[k].x;
      const uint32_t code = slots[find(d)].code;
      codes[k] = (uint8_t)code;
      steps[ns] = d;
      ns += code == kPackEscape;
    }
    std::fill(codes.begin() + m, codes.end(), (uint8_t)0);
    const uint64_t vb = align16(4ull * m), cb = align16(m), bytes = vb + cb + align16(4ull * ns);
    const bool keep = bytes >= 8ull * m;
    heads[c] = PackHead{(uint32_t)((out - first) / 16), m, keep ? kPackRaw : ns, 0};
    if (keep) {
      std::memmove(out, raw, 8ull * m);
      out += align16(8ull * m);
      continue;
    }
    uint32_t* v = reinterpret_cast<uint32_t*>(out);
    for (uint32_t k = 0; k < m; ++k) v[k] = raw[k].y;  // (reads run ahead of the writes)
    std::memcpy(out + vb, codes.data(), cb);
    std::memcpy(out + vb + cb, steps.data(), 4ull * ns);
    out += bytes;
  }
  return out;
}

// work(0) .. work(n - 1) on threads of their own, as far as there are any.
template <class Work>
void on_threads(unsigned n, Work&& work) {
  std::vector<std::thread> pool;
  unsigned t = 1;
  try {
    for (; t < n; ++t) pool.emplace_back(work, t);
  } catch (const std::exception&) {  // no more threads: this one does the rest
  }
  work(0);
  for (; t < n; ++t) work(t);
  for (auto& th : pool) th.join();
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
    B.csr_bytes = align16(4ull * ((uint64_t)B.rows + 1)) + 8 * n;
    B.csc_bytes = colpart + 8 * n;
    S->blocks.push_back(B);
    if (rows == 0) break;
    r0 = r;
  }

  // Blocks kept in device memory: the first ones whose two parts fit the
  // resident budget; only the others are streamed. Of these, the larger ones may
  // be packed and get room for the chunks' heads and the table of steps.
  uint64_t kept = 0, streamed_part = 0;
  std::vector<char> keep(S->blocks.size(), 0), room(S->blocks.size(), 0);
  for (size_t b = 0; b < S->blocks.size(); ++b) {
    StreamBlock& B = S->blocks[b];
    const uint64_t both = align16(B.csr_bytes) + B.csc_bytes;
    keep[b] = kept + both <= resident_bytes && streamed_part == 0;
    room[b] = !keep[b] && B.nnz >= kPackMin;
    const uint64_t csr = room[b] ? B.csr_bytes + pack_front(B.nnz) + 16 : B.csr_bytes;
    if (keep[b]) {
      kept += both;
    } else {
      streamed_part = std::max(streamed_part, std::max(csr, B.csc_bytes));
      S->max_stream_nnz = std::max(S->max_stream_nnz, B.nnz);
    }
    B.csr_off = off;
    off += align16(csr);
    B.csc_off = off;
    off += align16(B.csc_bytes);
  }
  S->host_bytes = std::max<uint64_t>(off, 16);
  MLEM_HIP(hipHostMalloc((void**)&S->host, S->host_bytes, hipHostMallocDefault));

  for (size_t b = 0; b < S->blocks.size(); ++b)
    if (keep[b]) {
      StreamBlock& B = S->blocks[b];
      MLEM_HIP(hipMalloc((void**)&B.resident, align16(B.csr_bytes) + B.csc_bytes));
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
  const unsigned hw = std::min(16u, std::max(1u, std::thread::hardware_concurrency()));
  const unsigned nthreads = (unsigned)std::max<size_t>(1, std::min<size_t>(S->blocks.size(), hw));
  std::atomic<uint64_t> bad{0};
  std::vector<std::string> errors(hw);
  std::vector<PackSteps> steps(S->blocks.size());
  auto work = [&](unsigned tid) {
    try {
      std::vector<uint32_t> next(cols);
      for (size_t b = tid; b < S->blocks.size(); b += nthreads) {
        StreamBlock& B = S->blocks[b];
        char* csr = S->host + B.csr_off;
        char* csc = S->host + B.csc_off;
        uint32_t* rp = reinterpret_cast<uint32_t*>(csr);
        const uint64_t base = B.row0 ? rowidx[B.row0 - 1] : 0;
        rp[0] = 0;
        for (uint32_t k = 0; k < B.rows; ++k) rp[k + 1] = (uint32_t)(rowidx[B.row0 + k] - base);
        char* front = csr + align16(4ull * ((uint64_t)B.rows + 1));
        if (S->expand && room[b]) steps[b] = pack_steps(fetch, base, B.nnz);
        uint2* el = reinterpret_cast<uint2*>(front + (steps[b].pays ? pack_front(B.nnz) : 0));
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
      }
    } catch (const ApiError& e) {
      errors[tid] = e.msg;
    } catch (const std::exception& e) {
      errors[tid] = e.what();
    }
  };
  auto check = [&] {
    for (const std::string& e : errors)
      if (!e.empty()) raise(MLEM_EIO, e);
    if (bad)
      raise(MLEM_EFORMAT, std::to_string(bad.load()) + " matrix elements have a column index >= " +
                              std::to_string(cols));
  };
  on_threads(nthreads, work);
  check();

  // Pack: a matrix of few blocks has each cut into groups of chunks, so that every
  // thread has some (about 1 ns an element on one thread: 67M elements in one block
  // 75 ms, opened in 690); then the groups of a block are moved together, so that it
  // crosses the link in one copy (each further one costs about 9 us a pass).
  struct Group {
    size_t block;
    uint64_t c0, c1;
    char *begin, *end;
  };
  std::vector<Group> groups;
  std::vector<size_t> first_group;  // of each packed block, and the end
  auto front_of = [&](const StreamBlock& B) {
    return S->host + B.csr_off + align16(4ull * ((uint64_t)B.rows + 1));
  };
  for (size_t b = 0; b < S->blocks.size(); ++b) {
    const StreamBlock& B = S->blocks[b];
    if (!steps[b].pays) continue;
    const uint64_t n = pack_chunks_of(B.nnz);
    const uint64_t g = std::max<uint64_t>(
        1, std::min<uint64_t>(hw / S->blocks.size(), B.nnz / kPackMin));
    std::memcpy(front_of(B) + sizeof(PackHead) * n, steps[b].step, sizeof(steps[b].step));
    first_group.push_back(groups.size());
    for (uint64_t i = 0; i < g; ++i)
      groups.push_back(Group{b, n * i / g, n * (i + 1) / g, nullptr, nullptr});
  }
  first_group.push_back(groups.size());
  const size_t npacked = first_group.size() - 1;
  std::atomic<size_t> next_group{0}, next_block{0};
  auto pack = [&](unsigned tid) {
    try {
      for (size_t i; (i = next_group++) < groups.size();) {
        Group& G = groups[i];
        const StreamBlock& B = S->blocks[G.block];
        G.begin = front_of(B) + pack_front(B.nnz) + 8ull * kPackChunk * G.c0;
        G.end = pack_chunks(front_of(B), B.nnz, G.c0, G.c1, steps[G.block]);
      }
    } catch (const std::exception& e) {
      errors[tid] = e.what();
    }
  };
  auto join = [&](unsigned) {
    for (size_t k; (k = next_block++) < npacked;) {
      StreamBlock& B = S->blocks[groups[first_group[k]].block];
      PackHead* heads = reinterpret_cast<PackHead*>(front_of(B));
      char* end = groups[first_group[k]].end;
      for (size_t i = first_group[k] + 1; i < first_group[k + 1]; ++i) {
        const Group& G = groups[i];
        for (uint64_t c = G.c0; c < G.c1; ++c) heads[c].at -= (uint32_t)((G.begin - end) / 16);
        std::memmove(end, G.begin, (size_t)(G.end - G.begin));
        end += G.end - G.begin;
      }
      B.packed_bytes = (uint64_t)(end - (S->host + B.csr_off));
    }
  };
  if (npacked) {
    on_threads((unsigned)std::min<size_t>(groups.size(), hw), pack);
    check();
    on_threads((unsigned)std::min<size_t>(npacked, hw), join);
  } else if (S->expand) {  // nothing to unpack
    MLEM_HIP(hipFree(S->expand));
    S->expand = nullptr;
  }

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
// bytes per element where rows are lines of response in file order (3 % of the
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
