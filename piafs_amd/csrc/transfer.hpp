// Host <-> device passage of solution states through pinned host memory.
//
// A state crosses in chunks.  Each chunk has a pinned buffer of its own; a
// host thread copies between the caller's array and the buffer, and a kernel
// (k_pack / k_unpack) moves the chunk between the buffer, over the host link,
// and the planar device layout, so the change of layout costs no pass over
// memory.  Several threads work on chunks at the same time, since one thread's
// memory copy is several times slower than the link.  Bound by the link and the
// page faults of a fresh output array: 92 MB (1024 x 1024, 11 variables) go in
// in 2.0 ms and out in 2.4 ms, against 26 and 30 ms for a layout change on one
// host thread and a copy from pageable memory; 1.1 MB 0.107 and 0.127 ms
// against 0.134 and 0.163.
#pragma once

#include <hip/hip_runtime.h>

#include <condition_variable>
#include <cstdint>
#include <functional>
#include <memory>
#include <mutex>
#include <thread>
#include <vector>

namespace piafs {

// The pinned buffers and copy threads of one device, shared by all its cases and
// given back with the last of them.  Two sets of at most 2 * kSlots * kSlotBytes of
// pinned memory each (a state of the largest size, and the buffers it outgrew).  A transfer takes the first if nobody has it, and queues its
// chunks behind whatever its stream holds.  Since that may be a long computation,
// during which the set is taken, any other transfer then waits for its own stream
// alone and takes the second set, which is never held, nor its buffers in use, for
// longer than chunks take to move.  So handles never wait for each other's steps.
// (With one set, held only after a wait for the stream, every transfer pays for the
// wait, the launches and the threads' waking one after the other: a pass of 25 steps
// at 128 x 97 takes 3.65 ms where it takes 3.57, a right-hand side at 512 x 385 1.17
// where it takes 1.11.)
class Staging {
 public:
  static constexpr int kSlots = 8;
  static constexpr size_t kSlotBytes = (size_t)2 << 20, kMinChunk = (size_t)128 << 10;

  // the device's staging (created at the first call, while a holder lives)
  static std::shared_ptr<Staging> of(int device);
  explicit Staging(int dev) : ahead(dev), after(dev) {}
  // pinned buffers for states of `bytes`, so that transfers allocate nothing
  bool reserve(size_t bytes);
  // n doubles from `src` (host) / to `dst` (host) in chunks of whole points of
  // nv doubles: kernel(first point, points, buffer) enqueues the device side of
  // a chunk on st and says whether that failed.  upload returns when src is no longer needed (the kernels
  // may still run), download when dst is complete.
  typedef std::function<hipError_t(long q0, long np, double *buf)> Kern;
  hipError_t upload(const double *src, long npts, int nv, hipStream_t st, const Kern &kernel);
  hipError_t download(double *dst, long npts, int nv, hipStream_t st, const Kern &kernel);

 private:
  struct Slot {
    double *buf = nullptr;
    hipEvent_t ev = nullptr;
    bool pending = false;  // a kernel may still be using buf (ev recorded after it, on `on`)
    hipStream_t on = nullptr;
  };
  // a set of buffers with its threads; whoever holds `use` has it
  struct Set {
    explicit Set(int dev) : device(dev) {}
    ~Set();
    const int device;
    std::mutex use;
    Slot slots[kSlots];
    int nslots = 0;
    size_t cap = 0;  // bytes of every slot's buffer
    // outgrown buffers, kept: freeing pinned memory waits for all work on the device
    void *old[4 * kSlots];
    int nold = 0;

    std::vector<std::thread> pool;
    std::mutex m;
    std::condition_variable wake, idle;
    const std::function<void(int)> *job = nullptr;
    uint64_t round = 0;
    int helpers = 0, busy = 0;
    bool stop = false;

    bool settled(hipStream_t st);  // no kernel is using a buffer, other than on st
    bool grow(size_t bytes);
    void release();
    void worker(int id);
    int threads(long nchunks) const;  // that move nchunks chunks
    hipError_t settle(Slot &s);
    hipError_t enqueue(long q0, long np, Slot &s, hipStream_t st, const Kern &kernel);
    hipError_t each(long nchunks, const std::function<hipError_t(long, Slot &)> &body);
    hipError_t upload(const double *src, long npts, int nv, hipStream_t st, const Kern &kernel);
    hipError_t download(double *dst, long npts, int nv, hipStream_t st, const Kern &kernel);
  };
  Set ahead, after;

  static void shape(size_t bytes, size_t &chunk, int &n);
  template <class F>
  hipError_t on_a_set(hipStream_t st, F move);
};

}  // namespace piafs
