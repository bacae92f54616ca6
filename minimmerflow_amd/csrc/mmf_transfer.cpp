// mmf_transfer.cpp -- device-to-host copies through pinned chunks.
//
// A copy into pageable memory runs at the rate one host thread moves bytes out
// of the runtime's staging buffer, page faults included: 18 GB/s into touched
// pages, 8-10 into fresh huge pages, 4 into fresh small ones, of the link's 57.
// Four threads moving 1 MB chunks out of a pinned ring take a 20 MB copy from
// 1.9 to 0.75 ms (fresh huge pages), 10 MB from 1.28 to 0.48; eight add
// nothing, and below 2 MB starting the threads costs more than they save.
#include "mmf_transfer.hpp"

#include <algorithm>
#include <atomic>
#include <cstring>
#include <mutex>
#include <exception>
#include <thread>
#include <vector>

#include "mmf_internal.hpp"

namespace mmf {

namespace {

constexpr size_t CHUNK = (size_t)1 << 20;
constexpr size_t RING = 12;
constexpr int WORKERS = 4;
constexpr size_t TRANSFER_MIN = (size_t)2 << 20;

std::mutex users_lock;  // users
int users = 0;
std::mutex ring_lock;  // the ring and its events, held for a whole copy
char *ring = nullptr;
hipEvent_t arrived[RING] = {};

void release_ring() {
  for (hipEvent_t &e : arrived) {
    if (e) (void)hipEventDestroy(e);
    e = nullptr;
  }
  if (ring) (void)hipHostFree(ring);
  ring = nullptr;
}

bool ensure_ring() {
  if (ring) return true;
  if (hipHostMalloc(&ring, RING * CHUNK, hipHostMallocPortable) != hipSuccess) {
    (void)hipGetLastError();
    ring = nullptr;
    return false;
  }
  return true;
}

struct Copy {
  char *dst;
  size_t bytes, chunks;
  std::atomic<size_t> ready{0}, next{0};  // chunks in the ring; chunks taken by a worker
  std::atomic<size_t> moved[RING];        // per slot, chunks moved out of it
  std::atomic<bool> stop{false};
  Copy(char *d, size_t n) : dst(d), bytes(n), chunks((n + CHUNK - 1) / CHUNK) {
    for (auto &m : moved) m.store(0, std::memory_order_relaxed);
  }
  size_t size(size_t i) const { return std::min(CHUNK, bytes - i * CHUNK); }
  void move(size_t i) {
    std::memcpy(dst + i * CHUNK, ring + (i % RING) * CHUNK, size(i));
    moved[i % RING].fetch_add(1, std::memory_order_release);
  }
  void work() {
    for (;;) {
      const size_t i = next.fetch_add(1);
      if (i >= chunks) return;
      while (ready.load(std::memory_order_acquire) <= i) {
        if (stop.load(std::memory_order_acquire)) return;
        std::this_thread::yield();
      }
      move(i);
    }
  }
  // chunk i's slot is free again
  bool free_slot(size_t i) const { return moved[i % RING].load(std::memory_order_acquire) == i / RING; }
};

}  // namespace

hipError_t copy_to_host(void *dst, const void *src, size_t bytes, hipStream_t s) {
  std::unique_lock<std::mutex> hold(ring_lock, std::defer_lock);
  if (bytes < TRANSFER_MIN || !hold.try_lock() || !ensure_ring()) {
    const hipError_t e = hipStreamSynchronize(s);
    return e != hipSuccess ? e : hipMemcpy(dst, src, bytes, hipMemcpyDeviceToHost);
  }
  // events belong to the device they are made on: made for this copy
  hipError_t err = hipSuccess;
  for (hipEvent_t &e : arrived)
    if (err == hipSuccess) err = hipEventCreateWithFlags(&e, hipEventDisableTiming);
  Copy c((char *)dst, bytes);
  std::thread workers[WORKERS];
  int started = 0;
  if (err == hipSuccess) {
    try {
      for (; started < WORKERS; ++started) workers[started] = std::thread([&c] { c.work(); });
    } catch (const std::exception &) {  // fewer of them, or this thread alone
    }
  }
  size_t issued = 0;
  for (size_t i = 0; i < c.chunks && err == hipSuccess; ++i) {
    while (err == hipSuccess && issued < c.chunks && (issued <= i || issued < i + RING)) {
      if (!c.free_slot(issued)) {
        if (issued > i) break;
        std::this_thread::yield();
        continue;
      }
      err = hipMemcpyAsync(ring + (issued % RING) * CHUNK, (const char *)src + issued * CHUNK, c.size(issued),
                           hipMemcpyDeviceToHost, s);
      if (err == hipSuccess) err = hipEventRecord(arrived[issued % RING], s);
      ++issued;
    }
    if (err == hipSuccess) err = hipEventSynchronize(arrived[i % RING]);
    if (err != hipSuccess) break;
    if (started) c.ready.store(i + 1, std::memory_order_release);
    else c.move(i);
  }
  if (err != hipSuccess) {
    c.stop.store(true, std::memory_order_release);
    (void)hipStreamSynchronize(s);  // no copy into the ring is left in flight
  }
  for (int t = 0; t < started; ++t) workers[t].join();
  for (hipEvent_t &e : arrived) {
    if (e) (void)hipEventDestroy(e);
    e = nullptr;
  }
  return err;
}

// Cells below which the host forms the rows, and the planes (us per read-back of
// one batch case / face list, host and device rows: 1024 cells 26 / 37, 4096 19 /
// 28, 10,000 32 / 37, 15,000 47 / 46, 40,000 131 / 97; per upload 448 cells 20 / 24,
// 2512 26 / 27, 7168 40 / 32).
constexpr int64_t HOST_ROWS_MAX = 12 << 10, HOST_PLANES_MAX = 5 << 10;

hipError_t planes_to_rows(double *rows, const double *soa, int64_t N, int64_t fs, double *scratch, hipStream_t s) {
  if (N >= HOST_ROWS_MAX) {
    const hipError_t e = launch_soa_to_aos(soa, nullptr, N, fs, scratch, s);
    return e != hipSuccess ? e : copy_to_host(rows, scratch, sizeof(double) * 5 * (size_t)N, s);
  }
  std::vector<double> planes((size_t)(5 * fs));
  hipError_t e = hipStreamSynchronize(s);
  if (e == hipSuccess) e = hipMemcpy(planes.data(), soa, sizeof(double) * planes.size(), hipMemcpyDeviceToHost);
  if (e != hipSuccess) return e;
  for (int64_t i = 0; i < N; ++i)
    for (int k = 0; k < 5; ++k) rows[5 * i + k] = planes[(size_t)(k * fs + i)];
  return hipSuccess;
}

hipError_t rows_to_planes(const double *rows, double *soa, double *copy, int64_t N, int64_t fs, double *scratch,
                          hipStream_t s) {
  const size_t bytes = sizeof(double) * 5 * (size_t)fs;
  hipError_t e = hipStreamSynchronize(s);
  if (e != hipSuccess) return e;
  if (N >= HOST_PLANES_MAX) {
    e = hipMemcpy(scratch, rows, sizeof(double) * 5 * (size_t)N, hipMemcpyHostToDevice);
    if (e == hipSuccess) e = launch_aos_to_soa(scratch, nullptr, N, fs, soa, s);
    return (e != hipSuccess || !copy) ? e : hipMemcpyAsync(copy, soa, bytes, hipMemcpyDeviceToDevice, s);
  }
  std::vector<double> planes((size_t)(5 * fs), 0.0);
  for (int64_t i = 0; i < N; ++i)
    for (int k = 0; k < 5; ++k) planes[(size_t)(k * fs + i)] = rows[5 * i + k];
  e = hipMemcpy(soa, planes.data(), bytes, hipMemcpyHostToDevice);
  return (e != hipSuccess || !copy) ? e : hipMemcpy(copy, planes.data(), bytes, hipMemcpyHostToDevice);
}

void transfer_attach() {
  std::lock_guard<std::mutex> g(users_lock);
  ++users;
}

void transfer_detach() {
  std::lock_guard<std::mutex> g(users_lock);
  if (--users > 0) return;
  std::lock_guard<std::mutex> hold(ring_lock);
  release_ring();
}

}  // namespace mmf
