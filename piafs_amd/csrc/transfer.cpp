#include "transfer.hpp"

#include <algorithm>
#include <atomic>
#include <cstring>
#include <map>

namespace piafs {

std::shared_ptr<Staging> Staging::of(int device) {
  static std::mutex mu;
  static std::map<int, std::weak_ptr<Staging>> known;
  std::lock_guard<std::mutex> g(mu);
  std::shared_ptr<Staging> s = known[device].lock();
  if (!s) known[device] = s = std::make_shared<Staging>(device);
  return s;
}

Staging::Set::~Set() {
  {
    std::lock_guard<std::mutex> g(m);
    stop = true;
  }
  wake.notify_all();
  for (std::thread &t : pool) t.join();
  hipSetDevice(device);
  release();
}

void Staging::Set::release() {
  for (Slot &s : slots) {
    if (s.ev && s.pending) hipEventSynchronize(s.ev);
    if (s.ev) hipEventDestroy(s.ev);
    if (s.buf) hipHostFree(s.buf);
  }
  for (int k = 0; k < nold; k++) hipHostFree(old[k]);
}

// Chunk size and buffers of a state: an eighth of it, within kMinChunk (below,
// a chunk's fixed cost of a launch and an event exceeds its copy) and
// kSlotBytes (above, the first chunk's copy delays the link).
void Staging::shape(size_t bytes, size_t &chunk, int &n) {
  chunk = std::min(std::max((bytes + kSlots - 1) / kSlots, kMinChunk), kSlotBytes);
  n = (int)std::min<size_t>(kSlots, std::max<size_t>(1, (bytes + chunk - 1) / chunk));
}

bool Staging::Set::grow(size_t bytes) {
  size_t chunk;
  int n;
  shape(bytes, chunk, n);
  if (chunk > cap || n > nslots) {
    size_t c = kMinChunk;  // doubled, so that buffers are replaced four times at most
    while (c < chunk) c *= 2;
    c = std::max(c, cap);
    const int want = std::max(n, nslots);
    int have = 0;
    for (; have < want; have++) {
      Slot &s = slots[have];
      if (!s.ev && hipEventCreateWithFlags(&s.ev, hipEventDisableTiming) != hipSuccess) {
        s.ev = nullptr;
        break;
      }
      if (s.buf && c == cap) continue;
      void *p = nullptr;
      if (hipHostMalloc(&p, c, hipHostMallocDefault) != hipSuccess) break;
      if (s.buf) old[nold++] = s.buf;
      s.buf = (double *)p;
      s.pending = false;
    }
    hipGetLastError();  // a shortage of pinned memory leaves fewer buffers, or the smaller ones
    if (have > 0) {
      for (int k = have; k < nslots; k++) {
        old[nold++] = slots[k].buf;
        slots[k].buf = nullptr;
        slots[k].pending = false;
      }
      nslots = have;
      cap = c;
    }
  }
  while ((int)pool.size() < nslots - 1) {
    const int id = (int)pool.size() + 1;
    try {
      pool.emplace_back([this, id] { worker(id); });
    } catch (...) {
      break;  // fewer threads
    }
  }
  return nslots > 0;
}

bool Staging::Set::settled(hipStream_t st) {
  for (Slot &s : slots)
    if (s.pending && !(st && s.on == st)) {
      const hipError_t e = hipEventQuery(s.ev);
      hipGetLastError();  // "not ready" is no error of the caller's
      if (e != hipSuccess) return false;
      s.pending = false;
    }
  return true;
}

bool Staging::reserve(size_t bytes) {
  hipSetDevice(ahead.device);
  std::unique_lock<std::mutex> g(ahead.use, std::try_to_lock);
  const bool first = g.owns_lock() && ahead.settled(nullptr);
  if (!first) g = std::unique_lock<std::mutex>(after.use);
  Set &s = first ? ahead : after;
  try {
    return s.grow(bytes);
  } catch (...) {
    return s.nslots > 0;
  }
}

void Staging::Set::worker(int id) {
  hipSetDevice(device);
  uint64_t seen = 0;
  std::unique_lock<std::mutex> g(m);
  for (;;) {
    wake.wait(g, [&] { return stop || (round != seen && id <= helpers); });
    if (stop) return;
    seen = round;
    const std::function<void(int)> *f = job;
    g.unlock();
    (*f)(id);
    g.lock();
    if (--busy == 0) idle.notify_one();
  }
}

int Staging::Set::threads(long nchunks) const {
  return (int)std::max(1L, std::min<long>({(long)nslots, (long)pool.size() + 1, nchunks}));
}

// body(chunk, slot) for every chunk, on the calling thread (slot 0) and the
// helpers, each with its own slot.  The first chunk of the thread with slot k is
// chunk k; a thread takes the next chunk when it is done with one.
hipError_t Staging::Set::each(long nchunks, const std::function<hipError_t(long, Slot &)> &body) {
  const int n = threads(nchunks) - 1;
  std::atomic<long> next{n + 1};
  std::atomic<int> err{(int)hipSuccess};
  const std::function<void(int)> run = [&](int s) {
    for (long c = s; c < nchunks && err == (int)hipSuccess; c = next++) {
      const hipError_t e = body(c, slots[s]);
      if (e != hipSuccess) err = (int)e;
    }
  };
  if (n > 0) {
    {
      std::lock_guard<std::mutex> g(m);
      job = &run;
      helpers = busy = n;
      round++;
    }
    wake.notify_all();
  }
  run(0);
  if (n > 0) {
    std::unique_lock<std::mutex> g(m);
    idle.wait(g, [&] { return busy == 0; });
    helpers = 0;
    job = nullptr;
  }
  return (hipError_t)err.load();
}

// waits until no kernel is using the slot's buffer
hipError_t Staging::Set::settle(Slot &s) {
  if (!s.pending) return hipSuccess;
  const hipError_t e = hipEventSynchronize(s.ev);
  if (e == hipSuccess) s.pending = false;
  return e;
}

// A chunk's device side.  Launch errors are kept by thread, so the thread that
// launches reports them (kernel's result).
hipError_t Staging::Set::enqueue(long q0, long np, Slot &s, hipStream_t st, const Kern &kernel) {
  hipError_t e = kernel(q0, np, s.buf);
  if (e != hipSuccess) return e;
  s.on = st;
  e = hipEventRecord(s.ev, st);
  if (e == hipSuccess) s.pending = true;
  else hipStreamSynchronize(st);  // no event to wait for: the buffer is given back idle
  return e;
}

hipError_t Staging::Set::upload(const double *src, long npts, int nv, hipStream_t st, const Kern &kernel) {
  const size_t bytes = (size_t)npts * nv * sizeof(double);
  if (!grow(bytes)) return hipErrorOutOfMemory;
  size_t chunk;
  int n;
  shape(bytes, chunk, n);
  const long per = std::max<long>(1, (long)(std::min(chunk, cap) / (nv * sizeof(double))));
  return each((npts + per - 1) / per, [&](long c, Slot &s) {
    const long q0 = c * per, np = std::min(per, npts - q0);
    const hipError_t e = settle(s);
    if (e != hipSuccess) return e;
    memcpy(s.buf, src + q0 * nv, (size_t)np * nv * sizeof(double));
    return enqueue(q0, np, s, st, kernel);
  });
}

hipError_t Staging::Set::download(double *dst, long npts, int nv, hipStream_t st, const Kern &kernel) {
  const size_t bytes = (size_t)npts * nv * sizeof(double);
  if (!grow(bytes)) return hipErrorOutOfMemory;
  size_t chunk;
  int n;
  shape(bytes, chunk, n);
  const long per = std::max<long>(1, (long)(std::min(chunk, cap) / (nv * sizeof(double)))), nchunks = (npts + per - 1) / per;
  auto fetch = [&](long c, Slot &s) {
    const long q0 = c * per, np = std::min(per, npts - q0);
    const hipError_t e = settle(s);
    if (e != hipSuccess) return e;
    return enqueue(q0, np, s, st, kernel);
  };
  // the first chunk of every thread is asked for from here, and the threads wake
  // when the first is there: until then one thread waits for the stream's work
  const int ahead = threads(nchunks);
  hipError_t e = hipSuccess;
  for (int c = 0; c < ahead && e == hipSuccess; c++) e = fetch(c, slots[c]);
  if (e == hipSuccess) e = settle(slots[0]);
  if (e != hipSuccess) return e;
  return each(nchunks, [&](long c, Slot &s) {
    const long q0 = c * per, np = std::min(per, npts - q0);
    hipError_t e = c < ahead ? hipSuccess : fetch(c, s);
    if (e == hipSuccess) e = settle(s);
    if (e == hipSuccess) memcpy(dst + q0 * nv, s.buf, (size_t)np * nv * sizeof(double));
    return e;
  });
}

// move(set) with a set that this transfer has
template <class F>
hipError_t Staging::on_a_set(hipStream_t st, F move) {
  const hipError_t set = hipSetDevice(ahead.device);  // launches, and events that may be made, are the stream's device's
  if (set != hipSuccess) return set;
  {
    std::unique_lock<std::mutex> g(ahead.use, std::try_to_lock);
    if (g.owns_lock() && ahead.settled(st)) return move(ahead);
  }
  const hipError_t e = hipStreamSynchronize(st);
  if (e != hipSuccess) return e;
  std::lock_guard<std::mutex> g(after.use);
  return move(after);
}

hipError_t Staging::upload(const double *src, long npts, int nv, hipStream_t st, const Kern &kernel) {
  return on_a_set(st, [&](Set &s) { return s.upload(src, npts, nv, st, kernel); });
}

hipError_t Staging::download(double *dst, long npts, int nv, hipStream_t st, const Kern &kernel) {
  return on_a_set(st, [&](Set &s) { return s.download(dst, npts, nv, st, kernel); });
}

}  // namespace piafs
