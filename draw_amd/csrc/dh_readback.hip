// dh_readback.hip -- canvas buffers into a caller's pageable arrays.
//
// A kernel writes the buffers into pinned staging in 64 KB chunks and raises a
// flag in host memory for each; the calling thread and a few helpers copy a
// chunk out as soon as its flag is up, while the device writes the next ones.
// A runtime copy to pageable memory stages through pinned memory as well, but
// one thread copies out, at 18 GB/s: that bounded it (1280x720 frame and depth,
// 7.4 MB: 436 -> 203 us; 640x480 170 -> 102; 4K 3850 -> 1580; PCIe alone some 140,
// 46 and 1250).
#if !defined(__HIP_DEVICE_COMPILE__)
#include <immintrin.h>
#endif

#include <algorithm>
#include <atomic>
#include <condition_variable>
#include <cstring>
#include <mutex>
#include <new>
#include <thread>
#include <vector>

#include "dh_common.hpp"
#include "dh_internal.hpp"

namespace dh {

namespace {
constexpr uint32_t kChunkWords = 4096;  // 16-byte words: 64 KB, a workgroup's
constexpr uint32_t kPartChunks = 15;    // chunks of a part, which one piece of staging holds
constexpr uint32_t kPartWords = kChunkWords * kPartChunks;
constexpr size_t kPieceBytes = 16ull * kPartWords + 4096;  // and its chunks' flags
constexpr uint32_t kPieces = 4;
constexpr int kHelpers = 3;
constexpr int kMaxSegs = 3;

struct ReadSegs {
  const uint32_t* src[kMaxSegs];
  uint32_t n_seg, n_words4;  // 4-byte words of a segment
  uint32_t n_words16;        // ...in 16-byte words, rounded up
};

// Words [w0, w0 + n) of the segments laid end to end (each padded to 16 bytes)
// into the staging of one part or two, a chunk per block, and then the chunk's
// flag, the part's ticket.  PCIe bounds it.
struct ReadParts {
  uint4* stage[2];
  uint32_t* flags[2];
  uint32_t ticket;  // the first part's; the second's follows
};
__global__ __launch_bounds__(256) void k_read_out(ReadSegs g, uint64_t w0, uint32_t n, ReadParts parts) {
  const uint32_t k = blockIdx.x < kPartChunks ? 0u : 1u, c = blockIdx.x - k * kPartChunks;
  uint4* const stage = parts.stage[k];
  w0 += k * kPartWords;
  n -= k * kPartWords;
  const uint32_t b0 = c * kChunkWords, b1 = min(b0 + kChunkWords, n);
  for (uint32_t i = b0 + threadIdx.x; i < b1; i += 256u) {
    const uint64_t w = w0 + i;
    const uint64_t w1 = g.n_words16, w2 = 2ull * g.n_words16;
    const uint32_t* src = w < w1 ? g.src[0] : w < w2 ? g.src[1] : g.src[2];
    const uint64_t e = 4ull * (w - (w < w1 ? 0ull : w < w2 ? w1 : w2));
    uint4 v = make_uint4(0u, 0u, 0u, 0u);
    if (e + 4u <= g.n_words4) {
      v = *reinterpret_cast<const uint4*>(src + e);
    } else {
      v.x = src[e];
      if (e + 1u < g.n_words4) v.y = src[e + 1u];
      if (e + 2u < g.n_words4) v.z = src[e + 2u];
    }
    stage[i] = v;
  }
  __threadfence_system();
  __syncthreads();
  if (threadIdx.x == 0)
    __hip_atomic_store(&parts.flags[k][c], parts.ticket + k, __ATOMIC_RELEASE, __HIP_MEMORY_SCOPE_SYSTEM);
}
}  // namespace

// A context's staging and its helper threads, which sleep between reads.  The
// staging is a ring of pieces, allocated as the reads come (pinned pieces of up
// to 1 MB take some 40 us each, one of 2 or 4 MB 110 to 740): one before the
// first read starts, a second behind its first part, two more during the next
// read.  With all four a launch writes two parts (a launch costs some 5 us of
// PCIe time, a part takes 19).
struct ReadStage {
  struct Piece {
    uint4* stage = nullptr;  // [kPartWords], pinned and coherent, then the chunks' flags: the ticket last written
    uint4* dev = nullptr;
    uint32_t* flags() const { return reinterpret_cast<uint32_t*>(stage + kPartWords); }
    uint32_t* flags_dev() const { return reinterpret_cast<uint32_t*>(dev + kPartWords); }
  };
  Piece piece[kPieces];
  uint32_t n_piece = 0;
  uint32_t ticket = 0, next_ticket = 1;  // part p of a read has ticket + p

  // the read under way
  ReadSegs segs{};
  uint8_t* dst[kMaxSegs] = {};
  uint64_t words = 0;
  uint32_t ring = 0;  // pieces it uses: part p is in piece p % ring
  uint32_t chunks = 0, parts = 0, launched = 0;
  std::atomic<uint32_t> next{0}, done{0}, done_of[kPieces];  // chunks handed out; copied: in all, of the part in each piece
  std::atomic<bool> stop{false};

  std::mutex mu;
  std::condition_variable wake, left;
  uint64_t reads = 0;
  int inside = 0;  // helpers in the read
  bool open = false, quit = false;
  std::vector<std::thread> helpers;

  const Piece& piece_of(uint32_t p) const { return piece[p % ring]; }
  uint32_t chunks_of(uint32_t p) const { return std::min(kPartChunks, chunks - p * kPartChunks); }
  bool add_piece() {
    Piece& h = piece[n_piece];
    hipError_t e = hipSuccess;
    if (!h.stage) e = hipHostMalloc(reinterpret_cast<void**>(&h.stage), kPieceBytes, hipHostMallocCoherent);
    if (e == hipSuccess) e = hipHostGetDevicePointer(reinterpret_cast<void**>(&h.dev), h.stage, 0);
    if (e != hipSuccess) {
      (void)hipGetLastError();
      return false;
    }
    memset(h.flags(), 0, 4u * kPartChunks);
    n_piece++;
    return true;
  }
  void copy_chunk(uint32_t c) {
    const uint64_t a = (uint64_t)c * kChunkWords, b = std::min<uint64_t>(a + kChunkWords, words);
    const uint8_t* from = reinterpret_cast<const uint8_t*>(piece_of(c / kPartChunks).stage + a % kPartWords);
    for (uint64_t w = a; w < b;) {
      const uint64_t s = w / segs.n_words16, r = w - s * segs.n_words16;
      const uint64_t e = std::min<uint64_t>(b - w, segs.n_words16 - r);
      memcpy(dst[s] + 16 * r, from + 16 * (w - a), std::min<uint64_t>(16 * e, 4ull * segs.n_words4 - 16 * r));
      w += e;
    }
  }
  // Takes chunks until none is left.  While chunk c's flag is down, waiting(c,
  // spin) is called; the read ends for all threads when one returns false.
  bool flag_up(uint32_t c) const {
    const uint32_t p = c / kPartChunks;
    return __atomic_load_n(piece_of(p).flags() + c % kPartChunks, __ATOMIC_ACQUIRE) == ticket + p;
  }
  template <class Waiting>
  void work(Waiting waiting) {
    for (uint32_t c; !stop.load() && (c = next.fetch_add(1)) < chunks;) {
      for (uint32_t spin = 1; !flag_up(c); spin++) {
        if (stop.load() || !waiting(c, spin)) {
          stop.store(true);
          return;
        }
        _mm_pause();
      }
      copy_chunk(c);
      done_of[c / kPartChunks % ring].fetch_add(1);
      done.fetch_add(1);
    }
  }
  void helper() {
    uint64_t seen = 0;
    std::unique_lock<std::mutex> lk(mu);
    for (;;) {
      wake.wait(lk, [&] { return quit || (open && seen != reads); });
      if (quit) return;
      seen = reads;
      inside++;
      lk.unlock();
      work([](uint32_t, uint32_t) { return true; });
      lk.lock();
      if (--inside == 0) left.notify_all();
    }
  }
  // Launches the next part, or two, if their staging is free.
  hipError_t launch_next(hipStream_t s) {
    const uint32_t p = launched, k = std::min(ring == kPieces ? 2u : 1u, parts - p);
    if (k == 0u) return hipSuccess;
    for (uint32_t j = p; j < p + k; j++)
      if (j >= ring && done_of[j % ring].load() != chunks_of(j - ring)) return hipSuccess;
    ReadParts rp;
    rp.ticket = ticket + p;
    uint32_t blocks = 0;
    for (uint32_t j = 0; j < 2u; j++) {
      const Piece& h = piece_of(p + (j < k ? j : 0u));
      rp.stage[j] = h.dev;
      rp.flags[j] = h.flags_dev();
      if (j >= k) continue;
      done_of[(p + j) % ring].store(0);
      blocks += chunks_of(p + j);
    }
    const uint64_t w0 = (uint64_t)p * kPartWords;
    const uint32_t n = (uint32_t)std::min<uint64_t>((uint64_t)k * kPartWords, words - w0);
    hipLaunchKernelGGL(k_read_out, dim3(blocks), dim3(256), 0, s, segs, w0, n, rp);
    launched += k;
    return hipGetLastError();
  }
};

void read_stage_destroy(ReadStage* st) {
  if (!st) return;
  {
    std::lock_guard<std::mutex> lk(st->mu);
    st->quit = true;
  }
  st->wake.notify_all();
  for (auto& t : st->helpers) t.join();
  for (auto& h : st->piece)
    if (h.stage) (void)hipHostFree(h.stage);
  delete st;
}

ReadStage* read_stage_create() {
  ReadStage* st = new (std::nothrow) ReadStage;
  if (st && !st->add_piece()) {
    read_stage_destroy(st);
    return nullptr;
  }
  return st;
}

hipError_t read_stage_read(ReadStage* st, const void* const* src, void* const* dst, uint32_t n_seg, uint32_t n_words,
                           hipStream_t s) {
  for (uint32_t k = 0; k < n_seg; k++) {
    st->segs.src[k] = static_cast<const uint32_t*>(src[k]);
    st->dst[k] = static_cast<uint8_t*>(dst[k]);
  }
  st->segs.n_words4 = n_words;
  st->segs.n_words16 = n_words / 4u + (n_words % 4u ? 1u : 0u);
  st->words = (uint64_t)n_seg * st->segs.n_words16;
  st->chunks = (uint32_t)((st->words + kChunkWords - 1u) / kChunkWords);
  st->parts = (st->chunks + kPartChunks - 1u) / kPartChunks;
  st->ticket = st->next_ticket;
  st->next_ticket += st->parts;
  st->launched = 0;
  st->next.store(0);
  st->done.store(0);
  for (auto& d : st->done_of) d.store(0);
  st->stop.store(false);
  st->ring = st->n_piece;
  hipError_t e = st->launch_next(s);
  if (e != hipSuccess) return e;
  // behind the first part's writing: a second piece, the threads (without either
  // the read takes longer)
  if (st->n_piece == 1u && st->parts > 1u && st->add_piece()) st->ring = 2u;
  e = st->launch_next(s);
  try {
    while (st->helpers.size() < (size_t)kHelpers) st->helpers.emplace_back([st] { st->helper(); });
  } catch (...) {
  }
  {
    std::lock_guard<std::mutex> lk(st->mu);
    st->reads++;
    st->open = true;
  }
  st->wake.notify_all();
  // more staging for the reads to come
  for (; st->reads > 1u && st->ring < kPieces && st->n_piece < kPieces && st->parts > st->ring;)
    if (!st->add_piece()) break;
  // Launches what can be; now and then asks whether the device has failed, or
  // has run all it was given and chunk c of it has no flag.
  bool idle = false;  // every part has been written
  auto waiting = [&](uint32_t c, uint32_t spin) {
    if (e == hipSuccess) e = st->launch_next(s);
    if (e != hipSuccess || spin % 4096u) return e == hipSuccess;
    const hipError_t q = hipStreamQuery(s);
    if (q == hipErrorNotReady) {
      (void)hipGetLastError();
      std::this_thread::yield();
      return true;
    }
    idle = st->launched == st->parts;
    if (q != hipSuccess) e = q;
    else if (c / kPartChunks < st->launched && !st->flag_up(c)) e = hipErrorUnknown;
    return e == hipSuccess;
  };
  st->work(waiting);
  // The other chunks are the helpers', however long they take: once their flags
  // are all up there is nothing left to do for them here.
  for (uint32_t spin = 1; st->done.load() < st->chunks && !st->stop.load() && !idle; spin++) {
    if (!waiting(~0u, spin)) st->stop.store(true);
    _mm_pause();
  }
  {
    std::unique_lock<std::mutex> lk(st->mu);
    st->open = false;
    st->left.wait(lk, [&] { return st->inside == 0; });
  }
  const hipError_t done = hipStreamSynchronize(s);
  return e != hipSuccess ? e : done;
}

}  // namespace dh
