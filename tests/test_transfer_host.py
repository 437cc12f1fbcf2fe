"""The host side of the state transfers (piafs_amd/csrc/transfer.cpp) on the CPU:
compiled against a small model of the HIP runtime in which a stream is a queue
that a thread works off, so that a long computation is a gate the test holds."""
import os
import shutil
import subprocess

import pytest

from conftest import ROOT

CSRC = os.path.join(ROOT, "piafs_amd", "csrc")

RUNTIME = r"""
#pragma once
#include <atomic>
#include <condition_variable>
#include <cstddef>
#include <cstdlib>
#include <deque>
#include <functional>
#include <mutex>
#include <thread>
#include <vector>
enum hipError_t { hipSuccess = 0, hipErrorOutOfMemory = 2, hipErrorNotReady = 600, hipErrorInvalidHandle = 400, hipErrorLaunchFailure = 719 };
struct Stream {  // works in order; done counts what it has finished
  int device = 0;
  std::mutex m;
  std::condition_variable cv;
  std::deque<std::function<void()>> q;
  long queued = 0, done = 0;
  bool stop = false;
  std::thread th{[this] { loop(); }};
  void loop() {
    std::unique_lock<std::mutex> g(m);
    for (;;) {
      cv.wait(g, [&] { return stop || !q.empty(); });
      if (q.empty()) return;
      std::function<void()> f = q.front();
      q.pop_front();
      g.unlock();
      f();
      g.lock();
      done++;
      cv.notify_all();
    }
  }
  void push(std::function<void()> f) {
    std::lock_guard<std::mutex> g(m);
    q.push_back(f);
    queued++;
    cv.notify_all();
  }
  void wait(long n) {
    std::unique_lock<std::mutex> g(m);
    cv.wait(g, [&] { return done >= n; });
  }
  ~Stream() {
    {
      std::lock_guard<std::mutex> g(m);
      stop = true;
      cv.notify_all();
    }
    th.join();
  }
};
inline std::vector<Stream *> streams;  // every one a test has, for what waits for the device
struct Event {
  int device = 0;
  Stream *s = nullptr;
  long n = 0;
};
typedef Stream *hipStream_t;
typedef Event *hipEvent_t;
enum { hipHostMallocDefault = 0, hipEventDisableTiming = 2 };
inline thread_local hipError_t last_error = hipSuccess;
inline hipError_t hipGetLastError() {
  const hipError_t e = last_error;
  last_error = hipSuccess;
  return e;
}
inline thread_local int current_device = 0;
inline hipError_t hipSetDevice(int d) {
  current_device = d;
  return hipSuccess;
}
inline hipError_t hipHostMalloc(void **p, size_t n, int) {
  *p = calloc(n, 1);
  return *p ? hipSuccess : hipErrorOutOfMemory;
}
inline hipError_t hipEventCreateWithFlags(hipEvent_t *e, int) {
  *e = new Event;
  (*e)->device = current_device;
  return hipSuccess;
}
inline hipError_t hipEventDestroy(hipEvent_t e) {
  delete e;
  return hipSuccess;
}
inline hipError_t hipEventRecord(hipEvent_t e, hipStream_t s) {
  if (e->device != s->device) return hipErrorInvalidHandle;
  std::lock_guard<std::mutex> g(s->m);
  e->s = s;
  e->n = s->queued;
  return hipSuccess;
}
inline std::atomic<int> waiting{0}, waiting_most{0};  // threads in hipEventSynchronize
inline hipError_t hipEventSynchronize(hipEvent_t e) {
  const int n = ++waiting;
  for (int m = waiting_most; n > m && !waiting_most.compare_exchange_weak(m, n);) {
  }
  if (e->s) e->s->wait(e->n);
  --waiting;
  return hipSuccess;
}
inline hipError_t hipEventQuery(hipEvent_t e) {
  if (!e->s) return hipSuccess;
  std::lock_guard<std::mutex> g(e->s->m);
  return e->s->done >= e->n ? hipSuccess : (last_error = hipErrorNotReady);
}
inline hipError_t hipStreamSynchronize(hipStream_t s) {
  long n;
  {
    std::lock_guard<std::mutex> g(s->m);
    n = s->queued;
  }
  s->wait(n);
  return hipSuccess;
}
inline hipError_t hipHostFree(void *p) {  // waits for the device's work
  for (Stream *s : streams) hipStreamSynchronize(s);
  free(p);
  return hipSuccess;
}
"""

COMMON = r"""
#include "transfer.hpp"

#include <atomic>
#include <chrono>
#include <cstdio>
#include <cstring>
#include <vector>
using namespace piafs;
typedef std::vector<double> Vec;
static const int NV = 11;
static const long NP = 40000;  // 3.5 MB: several chunks
static Vec state(double x) {
  Vec v(NP * NV);
  for (size_t i = 0; i < v.size(); i++) v[i] = x + i;
  return v;
}
static hipError_t to_device(Staging &s, const Vec &h, Vec &d, Stream &st) {
  return s.upload(h.data(), NP, NV, &st, [&](long q0, long np, double *buf) {
    st.push([=, &d] { memcpy(&d[q0 * NV], buf, np * NV * sizeof(double)); });
    return hipGetLastError();
  });
}
static hipError_t to_host(Staging &s, Vec &h, const Vec &d, Stream &st) {
  return s.download(h.data(), NP, NV, &st, [&](long q0, long np, double *buf) {
    st.push([=, &d] { memcpy(buf, &d[q0 * NV], np * NV * sizeof(double)); });
    return hipGetLastError();
  });
}
struct Gate {
  std::mutex m;
  std::condition_variable cv;
  bool open = false;
  void wait() {
    std::unique_lock<std::mutex> g(m);
    cv.wait(g, [&] { return open; });
  }
  void release() {
    std::lock_guard<std::mutex> g(m);
    open = true;
    cv.notify_all();
  }
};
"""

INDEPENDENT = r"""
// One handle moves its state (argv[1]: up or down) behind a computation that
// runs until the gate opens; another handle's round trip has to end before.
int main(int, char **argv) {
  const bool up = !strcmp(argv[1], "up");
  Staging s(0);
  Stream a, b;
  Gate gate;
  Vec da = state(1.0), ha(NP * NV), src = state(2.0), db(NP * NV), hb(NP * NV), hs = state(3.0);
  a.push([&] { gate.wait(); });
  std::atomic<int> other{0};
  hipError_t ea = hipSuccess;
  std::thread ta([&] { ea = up ? to_device(s, src, da, a) : to_host(s, ha, da, a); });
  std::this_thread::sleep_for(std::chrono::milliseconds(200));
  std::thread tb([&] {
    if (!s.reserve(NP * NV * sizeof(double))) return;  // a new case's buffers
    if (to_device(s, hs, db, b) != hipSuccess || to_host(s, hb, db, b) != hipSuccess) return;
    other = 1;
  });
  for (int i = 0; i < 100 && !other; i++) std::this_thread::sleep_for(std::chrono::milliseconds(50));
  const bool passed = other == 1;
  gate.release();
  ta.join();
  tb.join();
  hipStreamSynchronize(&a);
  if (ea != hipSuccess || other != 1 || hb != hs || (up ? da != src : ha != da)) return 2;
  return passed ? 0 : 1;
}
"""

WAITERS = r"""
// a download behind a computation keeps one thread waiting for it, not one a chunk
int main() {
  Staging s(0);
  Stream a;
  Gate gate;
  Vec da = state(1.0), ha(NP * NV);
  a.push([&] { gate.wait(); });
  hipError_t e = hipSuccess;
  std::thread t([&] { e = to_host(s, ha, da, a); });
  std::this_thread::sleep_for(std::chrono::milliseconds(500));
  const int most = waiting_most;
  gate.release();
  t.join();
  if (e != hipSuccess || ha != da) return 2;
  return most == 1 ? 0 : 1;
}
"""

ERRORS = r"""
// the launch of the last chunk fails (an upload's is a helper's), first in an
// upload, then in a download; after that the buffers serve as before
int main() {
  Staging s(0);
  Stream a;
  const Vec h = state(1.0);
  Vec d(NP * NV), back(NP * NV);
  for (int pass = 0; pass < 4; pass++) {
    auto kernel = [&](bool up) {
      return [&, up](long q0, long np, double *buf) {
        if (q0 + np == NP && pass == (up ? 0 : 1)) {
          last_error = hipErrorLaunchFailure;  // of this thread; nothing is queued
        } else {
          a.push([=, &d] {
            if (up) memcpy(&d[q0 * NV], buf, np * NV * sizeof(double));
            else memcpy(buf, &d[q0 * NV], np * NV * sizeof(double));
          });
        }
        return hipGetLastError();
      };
    };
    const hipError_t eu = s.upload(h.data(), NP, NV, &a, kernel(true));
    const hipError_t ed = s.download(back.data(), NP, NV, &a, kernel(false));
    if (eu != (pass == 0 ? hipErrorLaunchFailure : hipSuccess)) return 1;
    if (ed != (pass == 1 ? hipErrorLaunchFailure : hipSuccess)) return 2;
    if (pass > 1 && back != h) return 3;
  }
  return 0;
}
"""

DEVICES = r"""
// a thread whose current device is another one moves a case's state
int main() {
  Staging s(1);
  Stream a;
  a.device = 1;
  const Vec h = state(1.0);
  Vec d(NP * NV), back(NP * NV);
  auto kernel = [&](bool up) {
    return [&, up](long q0, long np, double *buf) {
      if (current_device != a.device) return hipErrorLaunchFailure;
      a.push([=, &d] {
        if (up) memcpy(&d[q0 * NV], buf, np * NV * sizeof(double));
        else memcpy(buf, &d[q0 * NV], np * NV * sizeof(double));
      });
      return hipSuccess;
    };
  };
  for (int k = 0; k < 2; k++) {
    hipSetDevice(0);
    if (s.upload(h.data(), NP, NV, &a, kernel(true)) != hipSuccess) return 1;
    hipSetDevice(0);
    if (s.download(back.data(), NP, NV, &a, kernel(false)) != hipSuccess || back != h) return 2;
  }
  return 0;
}
"""

GROWTH = r"""
// larger buffers, for a new case beside one whose computation runs, do not wait
// for that computation, and hold what is moved through them
int main() {
  Staging s(0);
  Stream a, b;
  streams = {&a, &b};
  Gate gate;
  const long few = 1000;  // one small chunk
  Vec da(few * NV), ha = state(1.0), hs = state(3.0), db(NP * NV), hb(NP * NV);
  if (s.upload(ha.data(), few, NV, &a, [&](long q0, long np, double *buf) {
        a.push([=, &da] { memcpy(&da[q0 * NV], buf, np * NV * sizeof(double)); });
        return hipGetLastError();
      }) != hipSuccess)
    return 2;
  hipStreamSynchronize(&a);
  a.push([&] { gate.wait(); });
  std::atomic<int> other{0};
  std::thread tb([&] {
    if (!s.reserve(NP * NV * sizeof(double))) return;
    if (to_device(s, hs, db, b) != hipSuccess || to_host(s, hb, db, b) != hipSuccess) return;
    other = 1;
  });
  for (int i = 0; i < 100 && !other; i++) std::this_thread::sleep_for(std::chrono::milliseconds(50));
  const bool passed = other == 1;
  gate.release();
  tb.join();
  hipStreamSynchronize(&a);
  if (other != 1 || hb != hs || memcmp(da.data(), ha.data(), few * NV * sizeof(double))) return 3;
  return passed ? 0 : 1;
}
"""


def _build(tmp_path, main):
    gxx = shutil.which("g++")
    if gxx is None:
        pytest.skip("no g++")
    inc = tmp_path / "hip"
    inc.mkdir()
    (inc / "hip_runtime.h").write_text(RUNTIME)
    (tmp_path / "main.cpp").write_text(COMMON + main)
    exe = str(tmp_path / "t")
    subprocess.run([gxx, "-std=c++17", "-O1", "-Wall", "-pthread", "-I", str(tmp_path), "-I", CSRC,
                    str(tmp_path / "main.cpp"), os.path.join(CSRC, "transfer.cpp"), "-o", exe], check=True)
    return exe


@pytest.mark.parametrize("direction", ["up", "down"])
def test_a_transfer_does_not_wait_for_other_handles_work(tmp_path, direction):
    exe = _build(tmp_path, INDEPENDENT)
    assert subprocess.run([exe, direction], timeout=60).returncode == 0


def test_one_thread_waits_for_queued_work(tmp_path):
    assert subprocess.run([_build(tmp_path, WAITERS)], timeout=60).returncode == 0


def test_failed_launches_are_reported(tmp_path):
    assert subprocess.run([_build(tmp_path, ERRORS)], timeout=60).returncode == 0


def test_the_callers_current_device_does_not_matter(tmp_path):
    assert subprocess.run([_build(tmp_path, DEVICES)], timeout=60).returncode == 0


def test_larger_buffers_do_not_wait_for_the_device(tmp_path):
    assert subprocess.run([_build(tmp_path, GROWTH)], timeout=60).returncode == 0
