// Transfers between the caller's pageable arrays and the device.
//
// The runtime's own pageable copies run at 28 GB/s up and 18 GB/s down on one
// host thread, one direction at a time, against 57 GB/s each way from pinned
// memory.  Large transfers here go through four pinned slots, one per thread: a
// thread copies between its slot and the caller's array while the other slots'
// DMA runs, in both directions at once where a batch is computed chunk by chunk.
// Measured: a computeFlux batch of 500,001 faces 7.9 -> 4.0 ms (smaller batches go
// through the context's own pinned staging, fvm_gpu.hip); 20 steps of 128^3 cells
// with their 168 MB of U read back 47.6 -> 39.0 ms.
//
// The slots belong to the process (20 MB, allocated on first use, freed with the
// last context).  While they are in use, by one context at a time, other fields
// take the runtime's copies and other flux batches go in pieces through their
// context's staging.
#include <hip/hip_runtime.h>

#include <atomic>
#include <cstring>
#include <mutex>
#include <thread>

#include "../../include/fvm_gpu.h"
#include "fvm_internal.h"

namespace {

struct Staging {
  std::mutex users_mu, use_mu;
  int users = 0;
  char *slot[fvm::kXferThreads] = {};
} g_staging;

bool slots_ready() {  // use_mu held
  for (char *&p : g_staging.slot)
    if (!p && hipHostMalloc((void **)&p, fvm::kXferSlot, hipHostMallocPortable) != hipSuccess) {
      p = nullptr;
      (void)hipGetLastError();
      return false;
    }
  return true;
}

}  // namespace

void fvm_xfer_ref() {
  std::lock_guard<std::mutex> lk(g_staging.users_mu);
  g_staging.users++;
}
void fvm_xfer_unref(fvm_ctx *c) {
  for (hipStream_t &s : c->xstream)
    if (s) {
      (void)hipStreamDestroy(s);
      s = nullptr;
    }
  std::lock_guard<std::mutex> lk(g_staging.users_mu);
  if (--g_staging.users > 0) return;
  std::lock_guard<std::mutex> lu(g_staging.use_mu);
  for (char *&p : g_staging.slot) {
    if (p) (void)hipHostFree(p);
    p = nullptr;
  }
}

// Whether the runtime would have to copy p through memory of its own.  The DMA
// reaches pinned arrays directly, faster than through the slots: 18 MB down 366 us
// against 544, a computeFlux batch of 500,001 faces 2.8 ms against 3.3.
bool fvm_pageable(const void *p) {
  hipPointerAttribute_t a;
  if (hipPointerGetAttributes(&a, p) == hipSuccess) return a.type == hipMemoryTypeUnregistered;
  (void)hipGetLastError();
  return true;
}

// chunk(arg, k, slot, stream) for k = 0 .. n - 1 on up to kXferThreads threads, the
// caller among them; false: the slots are in use or could not be had, nothing
// was done.  *err receives the first failure.
bool fvm_xfer_run(fvm_ctx *c, int n, hipError_t (*chunk)(void *, int, char *, hipStream_t), void *arg, hipError_t *err) {
  std::unique_lock<std::mutex> lk(g_staging.use_mu, std::try_to_lock);
  if (!lk.owns_lock() || !slots_ready()) return false;
  const int nt = n < fvm::kXferThreads ? n : fvm::kXferThreads;
  for (int w = 1; w < nt; w++)
    if (!c->xstream[w - 1] && hipStreamCreateWithFlags(&c->xstream[w - 1], hipStreamNonBlocking) != hipSuccess) {
      c->xstream[w - 1] = nullptr;
      (void)hipGetLastError();
      return false;
    }
  std::atomic<int> next{0}, first_err{(int)hipSuccess};
  auto work = [&](int w) {
    hipError_t e = hipSetDevice(c->device);
    hipStream_t st = w == 0 ? c->stream : c->xstream[w - 1];
    for (int k = next.fetch_add(1); e == hipSuccess && k < n && first_err.load() == (int)hipSuccess; k = next.fetch_add(1))
      e = chunk(arg, k, g_staging.slot[w], st);
    if (e != hipSuccess) {
      int ok = (int)hipSuccess;
      first_err.compare_exchange_strong(ok, (int)e);
      (void)hipStreamSynchronize(st);  // nothing of the failed chunk still uses the slot
    }
  };
  std::thread t[fvm::kXferThreads];
  for (int w = 1; w < nt; w++) {
    try {
      t[w] = std::thread(work, w);
    } catch (...) {
      break;  // fewer threads share the chunks
    }
  }
  work(0);
  for (int w = 1; w < nt; w++)
    if (t[w].joinable()) t[w].join();
  *err = (hipError_t)first_err.load();
  return true;
}

// bytes between the caller's array and device memory, after the work on the
// context's stream that produces or uses the device memory.  Down: returns when
// done.  Up: copied or in the stream, which the caller waits for when it has
// enqueued what follows (a wait here as well cost 3 us a field: the 26 fields of
// a 32^3 state 3.91 -> 3.99 ms).
static int copy_host(fvm_ctx *c, void *dst, const void *src, size_t bytes, bool down) {
  hipError_t err = hipSuccess;
  if (bytes >= fvm::kXferMin && fvm_pageable(down ? dst : src)) {
    FVM_HIPCHK(c, hipStreamSynchronize(c->stream));
    const int n = (int)((bytes + fvm::kXferSlot - 1) / fvm::kXferSlot);
    const bool done = fvm_xfer_chunks(c, n, [&](int k, char *slot, hipStream_t st) {
      const size_t o = (size_t)k * fvm::kXferSlot, len = std::min(bytes - o, fvm::kXferSlot);
      if (!down) std::memcpy(slot, (const char *)src + o, len);
      hipError_t e = hipMemcpyAsync(down ? (void *)slot : (void *)((char *)dst + o), down ? (const char *)src + o : slot, len,
                                    down ? hipMemcpyDeviceToHost : hipMemcpyHostToDevice, st);
      if (e == hipSuccess) e = hipStreamSynchronize(st);
      if (e == hipSuccess && down) std::memcpy((char *)dst + o, slot, len);
      return e;
    }, &err);
    if (done) {
      FVM_HIPCHK(c, err);
      return FVM_OK;
    }
  }
  FVM_HIPCHK(c, hipMemcpyAsync(dst, src, bytes, down ? hipMemcpyDeviceToHost : hipMemcpyHostToDevice, c->stream));
  if (down) FVM_HIPCHK(c, hipStreamSynchronize(c->stream));
  return FVM_OK;
}
int fvm_to_device(fvm_ctx *c, void *dst, const void *src, size_t bytes) { return copy_host(c, dst, src, bytes, false); }
int fvm_to_host(fvm_ctx *c, void *dst, const void *src, size_t bytes) { return copy_host(c, dst, src, bytes, true); }
