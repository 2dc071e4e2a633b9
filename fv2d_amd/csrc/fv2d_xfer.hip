// fv2d_xfer.hip -- copies between pageable host arrays and the device through pinned buffers.
//
// A copy between pageable memory and the device by the runtime alone ran at 10.5 GB/s towards the
// host (into fresh pages) and 29 GB/s towards the device; the link does 57 GB/s with pinned memory.
// Through the lanes below 536 MB go at 42 and 44 GB/s (52 and 19 ms before, 12.8 and 12.3 now), 33 MB
// to the host in 2.9 ms (3.6 before).
// Copies therefore go through lanes of two pinned chunks: while one chunk is on the link, a host
// thread copies the other from or to the caller's array (for a fresh array that is also where its
// pages are first touched, which one thread does at 20 GB/s); large copies are split over several
// threads with a lane each.
// All chunks go through the caller's stream, so stream order holds as for one copy.
#include "fv2d_xfer.h"

#include <string.h>

#include <mutex>
#include <thread>
#include <vector>

namespace fv2d {

namespace {

constexpr size_t MB = 1u << 20;
constexpr size_t CHUNK = 4 * MB;  // a lane has two of these
// Copies from this size on run on several threads, one for each PER_THREAD. Below it the threads cost
// more than they give in a process that keeps its own cores busy (after each of these copies a
// 16-thread conversion whose idle threads spin): a 33 MB copy per pass, 8 threads 12.2 ms per pass,
// one 9.7, the runtime's own copy 11.5; a 96 MB one up and two down: 7.8 (6 threads), 17.7, 22.1.
constexpr size_t SHARED = 64 * MB;
constexpr size_t PER_THREAD = 16 * MB;
constexpr int MAX_THREADS = 8;  // 12 and 14 are no faster
// Copies up to these sizes go to the runtime as they are: to the host 2.1 MB take 0.14 ms either way
// (2.9 MB 0.19 and 0.16); to the device one thread is no faster at any size.
constexpr size_t SMALL_TO_HOST = 2 * MB;
constexpr size_t SMALL_TO_DEVICE = SHARED - 1;
constexpr int MAX_CACHED = MAX_THREADS;  // idle lanes kept per device (64 MB at most)
constexpr int MAX_DEVICES = 64;

struct Lane {
  char *buf[2] = {nullptr, nullptr};
  hipEvent_t ev[2] = {nullptr, nullptr};
};

struct Pool {
  std::mutex lock;
  std::vector<Lane> idle;
  int users = 0;
};
Pool g_pool[MAX_DEVICES];

void lane_free(Lane &l) {
  for (int k = 0; k < 2; ++k) {
    if (l.buf[k]) (void)hipHostFree(l.buf[k]);
    if (l.ev[k]) (void)hipEventDestroy(l.ev[k]);
  }
  l = Lane();
}

// A lane of the current device `dev`: an idle one or a new one.
hipError_t lane_get(int dev, Lane &l) {
  Pool &p = g_pool[dev];
  {
    std::lock_guard<std::mutex> g(p.lock);
    if (!p.idle.empty()) {
      l = p.idle.back();
      p.idle.pop_back();
      return hipSuccess;
    }
  }
  for (int k = 0; k < 2; ++k) {
    hipError_t e = hipHostMalloc((void **)&l.buf[k], CHUNK, hipHostMallocDefault);
    if (e == hipSuccess) e = hipEventCreateWithFlags(&l.ev[k], hipEventDisableTiming);
    if (e != hipSuccess) {
      lane_free(l);
      return e;
    }
  }
  return hipSuccess;
}

void lane_put(int dev, Lane &l) {
  Pool &p = g_pool[dev];
  {
    std::lock_guard<std::mutex> g(p.lock);
    if (p.users > 0 && p.idle.size() < (size_t)MAX_CACHED) {
      p.idle.push_back(l);  // within the capacity reserved by copy_retain
      return;
    }
  }
  lane_free(l);
}

// One thread's share of a copy. Every chunk that was queued is waited for before the lane goes
// back, also after an error.
hipError_t run_lane(bool to_host, char *host, char *devp, size_t bytes, size_t piece, int dev, hipStream_t st) {
  hipError_t e = hipSetDevice(dev);
  if (e != hipSuccess) return e;
  Lane l;
  if ((e = lane_get(dev, l)) != hipSuccess) return e;
  const size_t n = (bytes + piece - 1) / piece;
  auto len = [&](size_t c) { return c + 1 < n ? piece : bytes - c * piece; };
  bool queued[2] = {false, false};
  auto wait = [&](int k) {
    if (!queued[k]) return hipSuccess;
    queued[k] = false;
    return hipEventSynchronize(l.ev[k]);
  };
  for (size_t c = 0; c < n + 1 && e == hipSuccess; ++c) {
    const int k = (int)(c & 1);
    if (c < n) {
      if (!to_host) {
        if ((e = wait(k)) != hipSuccess) break;  // chunk c - 2 has left the buffer
        memcpy(l.buf[k], host + c * piece, len(c));
      }
      e = to_host ? hipMemcpyAsync(l.buf[k], devp + c * piece, len(c), hipMemcpyDeviceToHost, st)
                  : hipMemcpyAsync(devp + c * piece, l.buf[k], len(c), hipMemcpyHostToDevice, st);
      if (e == hipSuccess) {
        queued[k] = true;
        e = hipEventRecord(l.ev[k], st);
      }
    }
    if (to_host && c > 0 && e == hipSuccess && (e = wait(k ^ 1)) == hipSuccess)
      memcpy(host + (c - 1) * piece, l.buf[k ^ 1], len(c - 1));
  }
  if (e != hipSuccess && (queued[0] || queued[1])) (void)hipStreamSynchronize(st);
  for (int k = 0; k < 2; ++k) {
    const hipError_t w = wait(k);
    if (e == hipSuccess) e = w;
  }
  lane_put(dev, l);
  return e;
}

hipError_t copy(bool to_host, char *host, char *devp, size_t bytes, int dev, hipStream_t st) {
  if (bytes <= (to_host ? SMALL_TO_HOST : SMALL_TO_DEVICE) || dev < 0 || dev >= MAX_DEVICES) {
    const hipError_t e = to_host ? hipMemcpyAsync(host, devp, bytes, hipMemcpyDeviceToHost, st)
                                 : hipMemcpyAsync(devp, host, bytes, hipMemcpyHostToDevice, st);
    return e != hipSuccess ? e : hipStreamSynchronize(st);
  }
  int nt = 1;
  if (bytes >= SHARED) nt = (int)(bytes / PER_THREAD < (size_t)MAX_THREADS ? bytes / PER_THREAD : MAX_THREADS);
  // pieces: each costs the link some 15 us besides its bytes (536 MB to the host in pieces of 1, 2
  // and 4 MB: 18.0, 14.3, 12.8 ms), but short copies need several per thread to overlap
  const size_t piece = bytes >= SHARED ? CHUNK : bytes >= 8 * MB ? 2 * MB : MB;
  const size_t share = (bytes / nt / piece + 1) * piece;
  hipError_t err[MAX_THREADS];
  std::thread th[MAX_THREADS];
  for (int i = 0; i < nt; ++i) err[i] = hipSuccess;
  auto part = [&](int i) {
    const size_t off = share * i;
    if (off < bytes)
      err[i] = run_lane(to_host, host + off, devp + off, off + share < bytes ? share : bytes - off, piece, dev, st);
  };
  for (int i = 1; i < nt; ++i) {
    try {
      th[i] = std::thread(part, i);
    } catch (...) {  // no thread to be had: this one does the share
      part(i);
    }
  }
  part(0);
  for (int i = 1; i < nt; ++i)
    if (th[i].joinable()) th[i].join();
  for (int i = 0; i < nt; ++i)
    if (err[i] != hipSuccess) return err[i];
  return hipSuccess;
}

}  // namespace

hipError_t copy_to_host(void *dst, const void *dev_src, size_t bytes, int dev, hipStream_t st) {
  return copy(true, (char *)dst, (char *)const_cast<void *>(dev_src), bytes, dev, st);
}

hipError_t copy_to_device(void *dev_dst, const void *src, size_t bytes, int dev, hipStream_t st) {
  return copy(false, (char *)const_cast<void *>(src), (char *)dev_dst, bytes, dev, st);
}

void copy_retain(int dev) {
  if (dev < 0 || dev >= MAX_DEVICES) return;
  Pool &p = g_pool[dev];
  std::lock_guard<std::mutex> g(p.lock);
  try {
    p.idle.reserve(MAX_CACHED);
  } catch (...) {
    return;  // nothing is kept then
  }
  p.users += 1;
}

void copy_release(int dev) {
  if (dev < 0 || dev >= MAX_DEVICES) return;
  Pool &p = g_pool[dev];
  std::vector<Lane> gone;
  {
    std::lock_guard<std::mutex> g(p.lock);
    if (p.users == 0 || --p.users > 0) return;
    gone.swap(p.idle);
  }
  for (Lane &l : gone) lane_free(l);
}

}  // namespace fv2d
