// dh_readback.hip -- canvas buffers into a caller's pageable arrays.
//
// One kernel writes the buffers into pinned staging in 256 KB chunks and raises
// a flag in host memory for each; the calling thread and a few helpers copy a
// chunk out as soon as its flag is up, while the kernel writes the next ones.
// A runtime copy to pageable memory stages through pinned memory as well, but
// one thread copies out, at 18 GB/s: that bounded it (1280x720 frame and depth,
// 7.4 MB: 445 -> 190 us; 640x480 160 -> 90; 4K 3845 -> 1538; PCIe alone some 140,
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
constexpr uint32_t kChunkWords = 16384;              // 16-byte words: 256 KB
constexpr uint32_t kBlockWords = 4096;               // four blocks a chunk
constexpr uint32_t kHalfChunks = 8;                  // chunks of a staging half (2 MB)
constexpr uint32_t kHalfWords = kChunkWords * kHalfChunks;
constexpr int kHelpers = 3;
constexpr int kMaxSegs = 3;

struct ReadSegs {
  const uint32_t* src[kMaxSegs];
  uint32_t n_seg, n_words4;  // 4-byte words of a segment
  uint32_t n_words16;        // ...in 16-byte words, rounded up
};

// Words [w0, w0 + n) of the segments laid end to end (each padded to 16 bytes)
// into stage; per finished chunk its flag, by the chunk's last block.  PCIe
// bounds it.
__global__ __launch_bounds__(256) void k_read_out(ReadSegs g, uint64_t w0, uint32_t n, uint4* __restrict__ stage,
                                                  uint32_t* __restrict__ counters, uint32_t* flags, uint32_t ticket) {
  const uint32_t b0 = blockIdx.x * kBlockWords, b1 = min(b0 + kBlockWords, n);
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
  if (threadIdx.x == 0) {
    const uint32_t c = b0 / kChunkWords;
    const uint32_t blocks = (min(kChunkWords, n - c * kChunkWords) + kBlockWords - 1u) / kBlockWords;
    if (atomicAdd(&counters[c], 1u) + 1u == blocks) {
      counters[c] = 0u;  // for the next launch
      __threadfence_system();
      __hip_atomic_store(&flags[c], ticket, __ATOMIC_RELEASE, __HIP_MEMORY_SCOPE_SYSTEM);
    }
  }
}
}  // namespace

// A context's staging, a ring of two parts of kHalfChunks chunks, and its helper
// threads, which sleep between reads.
struct ReadStage {
  uint4* stage = nullptr;        // [2 * kHalfWords], pinned
  uint4* stage_dev = nullptr;
  uint32_t* flags = nullptr;     // [2 * kHalfChunks], pinned and coherent: the ticket of the part last written
  uint32_t* flags_dev = nullptr;
  uint32_t* counters = nullptr;  // [2 * kHalfChunks], device, zero between launches
  uint32_t ticket = 0, next_ticket = 1;  // part p of a read has ticket + p

  // the read under way
  ReadSegs segs{};
  uint8_t* dst[kMaxSegs] = {};
  uint64_t words = 0;
  uint32_t chunks = 0, parts = 0, launched = 0;
  std::atomic<uint32_t> next{0}, done{0}, done_of[2];  // chunks handed out; copied: in all, of the part in each half
  std::atomic<bool> stop{false};

  std::mutex mu;
  std::condition_variable wake, left;
  uint64_t reads = 0;
  int inside = 0;  // helpers in the read
  bool open = false, quit = false;
  std::vector<std::thread> helpers;

  uint32_t chunks_of(uint32_t p) const { return std::min(kHalfChunks, chunks - p * kHalfChunks); }

  void copy_chunk(uint32_t c) {
    const uint64_t a = (uint64_t)c * kChunkWords, b = std::min<uint64_t>(a + kChunkWords, words);
    const uint8_t* from = reinterpret_cast<const uint8_t*>(stage + a % (2ull * kHalfWords));
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
    return __atomic_load_n(flags + c % (2u * kHalfChunks), __ATOMIC_ACQUIRE) == ticket + c / kHalfChunks;
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
      done_of[c / kHalfChunks & 1u].fetch_add(1);
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
  // Launches the next part if its half of the staging is free.
  hipError_t launch_next(hipStream_t s) {
    if (launched == parts) return hipSuccess;
    const uint32_t p = launched, h = p & 1u;
    if (p >= 2u && done_of[h].load() != chunks_of(p - 2u)) return hipSuccess;
    done_of[h].store(0);
    const uint64_t w0 = (uint64_t)p * kHalfWords;
    const uint32_t n = (uint32_t)std::min<uint64_t>(kHalfWords, words - w0);
    hipLaunchKernelGGL(k_read_out, dim3((n + kBlockWords - 1u) / kBlockWords), dim3(256), 0, s, segs, w0, n,
                       stage_dev + (size_t)h * kHalfWords, counters + h * kHalfChunks, flags_dev + h * kHalfChunks,
                       ticket + p);
    launched++;
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
  if (st->stage) (void)hipHostFree(st->stage);
  if (st->flags) (void)hipHostFree(st->flags);
  if (st->counters) (void)hipFree(st->counters);
  delete st;
}

ReadStage* read_stage_create(hipStream_t s) {
  ReadStage* st = new (std::nothrow) ReadStage;
  if (!st) return nullptr;
  const size_t fb = 2u * kHalfChunks * sizeof(uint32_t);
  hipError_t e = hipHostMalloc(reinterpret_cast<void**>(&st->stage), 2ull * kHalfWords * 16u, hipHostMallocCoherent);
  if (e == hipSuccess) e = hipHostGetDevicePointer(reinterpret_cast<void**>(&st->stage_dev), st->stage, 0);
  if (e == hipSuccess) e = hipHostMalloc(reinterpret_cast<void**>(&st->flags), fb, hipHostMallocCoherent);
  if (e == hipSuccess) e = hipHostGetDevicePointer(reinterpret_cast<void**>(&st->flags_dev), st->flags, 0);
  if (e == hipSuccess) e = hipMalloc(reinterpret_cast<void**>(&st->counters), fb);
  if (e == hipSuccess) e = hipMemsetAsync(st->counters, 0, fb, s);
  if (e == hipSuccess) memset(st->flags, 0, fb);
  try {
    for (int k = 0; e == hipSuccess && k < kHelpers; k++) st->helpers.emplace_back([st] { st->helper(); });
  } catch (...) {
    e = hipErrorOutOfMemory;  // no thread: the caller reads the runtime's way
  }
  if (e != hipSuccess) {
    (void)hipGetLastError();
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
  st->parts = (st->chunks + kHalfChunks - 1u) / kHalfChunks;
  st->ticket = st->next_ticket;
  st->next_ticket += st->parts;
  st->launched = 0;
  st->next.store(0);
  st->done.store(0);
  st->done_of[0].store(0);
  st->done_of[1].store(0);
  st->stop.store(false);
  hipError_t e = st->launch_next(s);
  if (e != hipSuccess) return e;
  {
    std::lock_guard<std::mutex> lk(st->mu);
    st->reads++;
    st->open = true;
  }
  st->wake.notify_all();
  e = st->launch_next(s);
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
    else if (c / kHalfChunks < st->launched && !st->flag_up(c)) e = hipErrorUnknown;
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
