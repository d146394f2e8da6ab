// Field and rod downloads.
//
// A copy into a caller's pageable memory makes the runtime pin that memory or
// stage it by itself: 21 us for a few KB (25 to 50 us strided), 10.7 GB/s for
// fresh memory of tens of MB, whose pages the one copying thread faults in as
// it goes (one MI355X host).  Here
//   - what is below kRingFrom goes to pinned memory of the batch in one copy, a
//     rod's lines packed by a kernel that writes it directly, and from there
//     to the caller: 12 us for a few KB, strided or not, 25 us for 350 KB (26
//     or 156 before, by where the caller's memory lies);
//   - beyond, a ring of pinned chunks fills from the batch's two streams while
//     two threads, from 2 MB on four, copy the full ones out, so that page
//     faults and host copies run side by side: 24 MB 1.41 -> 0.59 ms, 72 MB of
//     fresh memory 7.0 -> 2.5 ms.  Six and eight threads were not faster.  A
//     copy costs 14 us beside its bytes, whatever its size, which the other
//     stream's copy hides (0.66 ms on one stream); chunks of 2 MB against 1 MB:
//     0.65 and 0.80 ms on one stream;
//   - longer strided lines, and whatever finds no pinned memory, are copied as
//     before.
#include <sys/mman.h>
#include <unistd.h>

#include <algorithm>
#include <atomic>
#include <cstring>
#include <thread>
#include <utility>
#include <vector>

#include "erod_common.hpp"

namespace erod {

  namespace {
    constexpr size_t kStageBytes = size_t(256) << 10;
    constexpr size_t kRingFrom = size_t(1) << 20, kChunk = size_t(2) << 20;
    constexpr int kRing = 4;  // chunks in the ring
    constexpr int kThreadsMost = 4;

    // lines of cnt values, `pitch` apart, one after another into pinned memory
    __global__ void k_pack_lines(const double* __restrict__ src, uint64_t pitch, uint64_t cnt, int nc,
                                 double* __restrict__ out) {
      const uint64_t n = cnt * uint64_t(nc);
      for (uint64_t i = blockIdx.x * (uint64_t)blockDim.x + threadIdx.x; i < n; i += (uint64_t)gridDim.x * blockDim.x) {
        const uint64_t c = i / cnt;
        out[i] = src[c * pitch + (i - c * cnt)];
      }
    }

    // pinned memory of the batch, allocated on first use; null if there is none
    void* pinned(const erod_batch* b, void*& p, size_t bytes) {
      if (p) return p;
      const OnDevice here(b->device);
      if (hipHostMalloc(&p, bytes, hipHostMallocDefault) != hipSuccess) {
        p = nullptr;
        (void)hipGetLastError();
      }
      return p;
    }

    int ring_events(erod_batch* b) {
      if (b->ring_ev[kRing - 1]) return EROD_OK;
      const OnDevice here(b->device);
      for (int i = 0; i < kRing; ++i)
        if (!b->ring_ev[i]) EROD_HIP(hipEventCreateWithFlags(&b->ring_ev[i], hipEventDisableTiming));
      return EROD_OK;
    }

    // The caller's pages in [p, p + n) that are about to be written, made
    // present in one call if some are not: faulted in one by one by the copy
    // they halve its rate (1.6 MB of fresh memory by one thread 0.32 ms, 0.16
    // with this; a pass that keeps eight fields of 1.6 to 4.8 MB 2.5 -> 2.1 ms).
    // Asking costs nothing that can be measured, and what the system refuses
    // the copy does by itself.  Not for four threads: they fault beside each
    // other, and eight fields of 6 to 18 MB took 5.4 ms with it, 5.0 without.
    // So a download of 2 MB and more still takes about twice as long into memory
    // that is not present (fresh from the allocator) as into memory that is.
    void make_present(char* p, size_t n) {
#if defined(MADV_POPULATE_WRITE)
      static const size_t page = size_t(sysconf(_SC_PAGESIZE));
      const uintptr_t lo = (reinterpret_cast<uintptr_t>(p) + page - 1) / page * page;
      const uintptr_t hi = (reinterpret_cast<uintptr_t>(p) + n) / page * page;
      unsigned char in[512];
      if (hi <= lo || (hi - lo) / page < 16 || (hi - lo) / page > sizeof(in)) return;
      void* const at = reinterpret_cast<void*>(lo);
      if (mincore(at, hi - lo, in) != 0) return;
      for (size_t i = 0; i < (hi - lo) / page; ++i)
        if (!(in[i] & 1)) {
          (void)madvise(at, hi - lo, MADV_POPULATE_WRITE);
          return;
        }
#endif
    }

    // `bytes` from device memory into the caller's through the ring.  The
    // calling thread makes every HIP call: it queues a chunk's copy once the
    // slot's last content has been copied out, waits for copies in order and
    // publishes how many have landed; every thread (it among them) copies its
    // share of each landed chunk.  Chunks go alternately to the batch's two
    // streams, so that one is in flight while the other's copy starts or ends.
    int download_ring(erod_batch* b, const char* src, char* host, size_t bytes) {
      const size_t mb = size_t(1) << 20, want = bytes < 2 * mb ? 2 : kThreadsMost;
      const size_t chunk = bytes < 6 * mb ? kChunk / 2 : kChunk;
      const size_t chunks = (bytes + chunk - 1) / chunk;
      char* ring = static_cast<char*>(b->ring);
      auto size_of = [&](size_t i) { return i + 1 < chunks ? chunk : bytes - i * chunk; };
      auto queue = [&](size_t i) -> int {
        hipStream_t st = (i & 1) ? b->stream2 : b->stream;
        EROD_HIP(hipMemcpyAsync(ring + (i % kRing) * chunk, src + i * chunk, size_of(i), hipMemcpyDeviceToHost, st));
        EROD_HIP(hipEventRecord(b->ring_ev[i % kRing], st));
        return EROD_OK;
      };
      // the second stream starts after the work already queued on the first
      EROD_HIP(hipEventRecord(b->ev_fork, b->stream));
      EROD_HIP(hipStreamWaitEvent(b->stream2, b->ev_fork, 0));
      std::atomic<size_t> landed{0};
      std::atomic<bool> stop{false};
      std::atomic<size_t> out[kThreadsMost];  // chunks each thread has copied its share of
      for (auto& o : out) o.store(0);
      std::vector<std::thread> helpers;
      std::atomic<size_t> n_threads{0};  // known once the helpers are up
      // thread k's share of chunk i: [first, first + second)
      auto share = [&](size_t i, size_t k, size_t n) {
        const size_t size = size_of(i), part = ((size + n - 1) / n + 63) / 64 * 64, lo = std::min(size, k * part);
        return std::pair<size_t, size_t>(lo, std::min(size, lo + part) - lo);
      };
      auto ready = [&](size_t i, size_t k, size_t n) {
        if (n > 2) return;
        const auto [lo, len] = share(i, k, n);
        make_present(host + i * chunk + lo, len);
      };
      auto copy_out = [&](size_t i, size_t k, size_t n) {
        const auto [lo, len] = share(i, k, n);
        std::memcpy(host + i * chunk + lo, ring + (i % kRing) * chunk + lo, len);
        out[k].store(i + 1, std::memory_order_release);
      };
      auto help = [&](size_t k) {
        size_t n;
        while ((n = n_threads.load(std::memory_order_acquire)) == 0) std::this_thread::yield();
        for (size_t i = 0; i < chunks; ++i) {
          ready(i, k, n);
          while (landed.load(std::memory_order_acquire) <= i) {
            if (stop.load(std::memory_order_acquire)) return;
            std::this_thread::yield();
          }
          copy_out(i, k, n);
        }
      };
      size_t queued = 0;
      int rc = EROD_OK;
      for (; queued < chunks && queued < size_t(kRing) && rc == EROD_OK; ++queued) rc = queue(queued);
      try {
        helpers.reserve(want);
        for (size_t k = 1; k < want && rc == EROD_OK; ++k) helpers.emplace_back(help, k);
      } catch (...) {
        // fewer threads: those that are up share the chunks
      }
      const size_t n = helpers.size() + 1;
      n_threads.store(n, std::memory_order_release);
      // whether every thread is done with chunk i
      auto copied = [&](size_t i) {
        for (size_t k = 0; k < n; ++k)
          if (out[k].load(std::memory_order_acquire) <= i) return false;
        return true;
      };
      for (size_t i = 0; i < chunks && rc == EROD_OK; ++i) {
        ready(i, 0, n);
        rc = hip_check(hipEventSynchronize(b->ring_ev[i % kRing]), "download");
        if (rc) break;
        landed.store(i + 1, std::memory_order_release);
        copy_out(i, 0, n);
        // a slot is free again when its chunk is out
        while (queued < chunks && rc == EROD_OK) {
          const size_t old = queued - kRing;
          if (old > i || !copied(old)) {
            if (queued > i + 1) break;  // others are still in flight: look again after the next one lands
            std::this_thread::yield();
            continue;
          }
          rc = queue(queued);
          ++queued;
        }
      }
      if (rc) stop.store(true, std::memory_order_release);
      for (std::thread& t : helpers) t.join();
      if (rc) {
        (void)hipStreamSynchronize(b->stream2);
        (void)hipStreamSynchronize(b->stream);
      }
      return rc;
    }
  }  // namespace

  int download_lines(erod_batch* b, int field, uint64_t slot, uint64_t cnt, double* host) {
    const int nc = field_info(field).ncomp;
    const uint64_t slots = b->field_slots(field);
    const double* src = b->d_field[field] + slot;
    const size_t line = cnt * sizeof(double), bytes = line * nc;
    const bool whole = cnt == slots || nc == 1;
    void* stage = bytes <= kStageBytes ? pinned(b, b->stage, kStageBytes) : pinned(b, b->ring, kRing * kChunk);
    if (stage && bytes < kRingFrom) {
      if (whole) {
        EROD_HIP(hipMemcpyAsync(stage, src, bytes, hipMemcpyDeviceToHost, b->stream));
      } else {
        hipLaunchKernelGGL(k_pack_lines, dim3(static_cast<unsigned>((cnt * nc + kThreads - 1) / kThreads)), dim3(kThreads), 0,
                           b->stream, src, slots, cnt, nc, static_cast<double*>(stage));
        EROD_HIP(hipGetLastError());
      }
      make_present(reinterpret_cast<char*>(host), bytes);  // (while the copy is under way)
      EROD_HIP(hipStreamSynchronize(b->stream));
      std::memcpy(host, stage, bytes);
      return EROD_OK;
    }
    if (stage && whole) {
      if (int rc = ring_events(b)) return rc;
      return download_ring(b, reinterpret_cast<const char*>(src), reinterpret_cast<char*>(host), bytes);
    }
    if (whole) EROD_HIP(hipMemcpyAsync(host, src, bytes, hipMemcpyDeviceToHost, b->stream));
    else
      EROD_HIP(hipMemcpy2DAsync(host, line, src, slots * sizeof(double), line, nc, hipMemcpyDeviceToHost, b->stream));
    EROD_HIP(hipStreamSynchronize(b->stream));
    return EROD_OK;
  }

  void free_transfer_buffers(erod_batch* b) {
    if (b->stage) (void)hipHostFree(b->stage);
    if (b->ring) (void)hipHostFree(b->ring);
    for (hipEvent_t e : b->ring_ev)
      if (e) (void)hipEventDestroy(e);
  }

}  // namespace erod
