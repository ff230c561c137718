// mge_xfer.h -- host <-> device transfers of whole fields through a pinned
// ring, and a case's pinned result word.
//
// A copy between device memory and the caller's ordinary (pageable) memory
// goes through the runtime's own staging one piece at a time, about 10 GB/s,
// and an FP32 case's field was then converted by one thread: reading back the
// 0.7 GB state of a 256^3 level took 70 ms, three multigrid cycles' time.
// Here the copy engine fills a ring of pinned pieces while several threads
// empty (or fill) them, converting on the way; the caller's memory is first
// touched by those threads too.  A ring is one transfer's at a time; a transfer
// that finds all of them taken, or no pinned memory, goes the runtime's way by
// itself, so that cases never wait for each other.
#pragma once
#include <hip/hip_runtime.h>

#include <atomic>
#include <cstring>
#include <memory>
#include <mutex>
#include <system_error>
#include <thread>
#include <vector>

namespace mge {

constexpr size_t kPiece = 2u << 20;   // bytes of one piece
constexpr int kPieces = 8;            // pieces of a ring
constexpr int kRings = 4;             // rings of the process
constexpr int kXferThreads = 8;       // threads of one transfer, the caller's among them

// The process's rings: each allocated by the first transfer that takes it, all
// freed with the last case.  A transfer holds the mutex of a ring that it gets
// at once, after waiting for its case's stream without it.
struct XferRing {
  std::mutex mu;
  char *buf = nullptr;   // kPieces * kPiece bytes
};
struct XferPool {
  std::mutex mu;
  int users = 0;         // live cases
  XferRing ring[kRings];
};
inline XferPool &xfer_pool() {
  static XferPool p;
  return p;
}
inline void xfer_user(int delta) {
  XferPool &P = xfer_pool();
  std::lock_guard<std::mutex> lk(P.mu);
  P.users += delta;
  if (P.users > 0) return;
  for (XferRing &r : P.ring) {
    std::lock_guard<std::mutex> lr(r.mu);
    if (r.buf) hipHostFree(r.buf);
    r.buf = nullptr;
  }
}

// The case's device as the thread's current one for a scope: an event records
// only on streams of the device it was made on, and a caller's current device
// may be another.
struct DeviceScope {
  int prev = 0;
  hipError_t rc;
  explicit DeviceScope(int dev) : rc(hipGetDevice(&prev)) {
    if (rc == hipSuccess && prev != dev) rc = hipSetDevice(dev);
  }
  ~DeviceScope() { if (rc == hipSuccess) hipSetDevice(prev); }
  DeviceScope(const DeviceScope &) = delete;
  DeviceScope &operator=(const DeviceScope &) = delete;
};

// A transfer without the ring: the whole field straight from or to the caller's
// memory if it crosses as it is (host), else in pieces of ordinary memory.
template <class Move>
hipError_t xfer_plain(hipStream_t stream, char *dptr, size_t bytes, bool up, Move move, char *host) {
  std::unique_ptr<char[]> buf;
  const size_t step = host ? bytes : (bytes < kPiece ? bytes : kPiece);
  if (!host) {
    buf.reset(new (std::nothrow) char[step]);
    if (!buf) return hipErrorOutOfMemory;
  }
  for (size_t o = 0; o < bytes; o += step) {
    const size_t len = bytes - o < step ? bytes - o : step;
    char *t = host ? host : buf.get();
    if (up && !host) move(o, t, len);
    hipError_t e = up ? hipMemcpyAsync(dptr + o, t, len, hipMemcpyHostToDevice, stream)
                      : hipMemcpyAsync(t, dptr + o, len, hipMemcpyDeviceToHost, stream);
    const hipError_t f = hipStreamSynchronize(stream);
    if (e == hipSuccess) e = f;
    if (e != hipSuccess) return e;
    if (!up && !host) move(o, t, len);
  }
  return hipSuccess;
}

// One transfer of `bytes` bytes: up = false, device -> host: move(piece
// offset, pinned piece, length) empties a piece the copy engine has filled;
// up = true: it fills a piece, which is then copied to the device; host: the
// caller's memory where move only copies (else null).  Returns the first error.
// On return the transfer is complete.
template <class Move>
hipError_t xfer(int dev, hipStream_t stream, void *dptr, size_t bytes, bool up, Move move, void *host = nullptr) {
  if (bytes == 0) return hipSuccess;
  const DeviceScope on(dev);
  if (on.rc != hipSuccess) return on.rc;
  hipError_t e = hipStreamSynchronize(stream);
  if (e != hipSuccess) return e;
  std::unique_lock<std::mutex> lk;
  XferRing *R = nullptr;
  for (XferRing &r : xfer_pool().ring) {
    lk = std::unique_lock<std::mutex>(r.mu, std::try_to_lock);
    if (!lk) continue;
    R = &r;
    break;
  }
  if (R && !R->buf && hipHostMalloc((void **)&R->buf, kPieces * kPiece, hipHostMallocPortable) != hipSuccess)
    R->buf = nullptr;
  if (!R || !R->buf) return xfer_plain(stream, (char *)dptr, bytes, up, move, (char *)host);
  const long np = (long)((bytes + kPiece - 1) / kPiece);
  auto off = [&](long c) { return (size_t)c * kPiece; };
  auto len = [&](long c) { return bytes - off(c) < kPiece ? bytes - off(c) : kPiece; };
  auto slot = [&](long c) { return R->buf + (size_t)(c % kPieces) * kPiece; };
  auto dev_at = [&](long c) { return (char *)dptr + off(c); };
  if (np <= 2) {  // small: the caller's thread alone, one wait
    if (up)
      for (long c = 0; c < np; c++) move(off(c), slot(c), len(c));
    for (long c = 0; c < np && e == hipSuccess; c++)
      e = up ? hipMemcpyAsync(dev_at(c), slot(c), len(c), hipMemcpyHostToDevice, stream)
             : hipMemcpyAsync(slot(c), dev_at(c), len(c), hipMemcpyDeviceToHost, stream);
    hipError_t f = hipStreamSynchronize(stream);
    if (e == hipSuccess) e = f;
    if (!up && e == hipSuccess)
      for (long c = 0; c < np; c++) move(off(c), slot(c), len(c));
    return e;
  }
  hipEvent_t ev[kPieces] = {};
  for (int s = 0; s < kPieces && e == hipSuccess; s++) e = hipEventCreateWithFlags(&ev[s], hipEventDisableTiming);
  std::atomic<long> next{0}, ready{0};   // next piece to move; down: pieces whose copy is on the stream
  std::atomic<int> failed{(int)e};
  std::unique_ptr<std::atomic<char>[]> done(new (std::nothrow) std::atomic<char>[np]);
  std::vector<std::thread> pool;
  if (!done) failed = (int)hipErrorOutOfMemory;
  else
    for (long c = 0; c < np; c++) done[c] = 0;
  auto fail = [&](hipError_t f) {
    int z = (int)hipSuccess;
    failed.compare_exchange_strong(z, (int)f);
  };
  // moves one piece if one may be moved now; down: its copy is on the stream;
  // up: the ring's place is free (the piece before it there was sent)
  auto step = [&]() {
    long c = next.load();
    if (c >= np) return false;
    const bool may = up ? (c < kPieces || done[c - kPieces].load()) : c < ready.load();
    if (!may || !next.compare_exchange_strong(c, c + 1)) return false;
    hipError_t f = hipSuccess;
    if (!up || c >= kPieces) f = hipEventSynchronize(ev[c % kPieces]);
    if (f == hipSuccess) {
      move(off(c), slot(c), len(c));
      if (up) {
        f = hipMemcpyAsync(dev_at(c), slot(c), len(c), hipMemcpyHostToDevice, stream);
        if (f == hipSuccess) f = hipEventRecord(ev[c % kPieces], stream);
      }
    }
    if (f != hipSuccess) fail(f);
    done[c] = 1;
    return true;
  };
  auto work = [&]() {
    if (hipSetDevice(dev) != hipSuccess) return;
    while (!failed && next.load() < np)
      if (!step()) std::this_thread::yield();
  };
  if (!failed) {
    const int nt = (int)std::min<long>(kXferThreads, np / 2) - 1;
    for (int t = 0; t < nt; t++) {
      try {
        pool.emplace_back(work);
      } catch (const std::exception &) {
        break;   // fewer threads
      }
    }
    long put = 0;
    while (!failed && (next.load() < np || put < np)) {
      while (!up && put < np && (put < kPieces || done[put - kPieces].load())) {
        e = hipMemcpyAsync(slot(put), dev_at(put), len(put), hipMemcpyDeviceToHost, stream);
        if (e == hipSuccess) e = hipEventRecord(ev[put % kPieces], stream);
        if (e != hipSuccess) {
          fail(e);
          break;
        }
        ready = ++put;
      }
      if (up) put = np;
      if (!failed && !step()) std::this_thread::yield();
    }
  }
  for (auto &t : pool) t.join();
  e = hipStreamSynchronize(stream);
  for (int s = 0; s < kPieces; s++)
    if (ev[s]) hipEventDestroy(ev[s]);
  return failed ? (hipError_t)failed.load() : e;
}

// What the host reads after a cycle or a call: the residual and the error
// flag, written by k_publish into pinned memory of the case (two copies into
// ordinary memory cost some 40 us each with their waits)
struct HostWord {
  double r;
  int err;
};
__global__ void k_publish(const double *r, const int *err, HostWord *out) {
  if (threadIdx.x != 0) return;
  out->r = r ? *r : 0.0;
  out->err = *err;
}

}  // namespace mge
