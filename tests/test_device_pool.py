"""The pool of device memory between owners (csrc/device_pool.h) on a pretended
device: which blocks it hands out again, its bound, its way out of a full device and
of host memory running out, its cost with many kept blocks, and several threads."""
import os
import subprocess

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

_SOURCE = r"""
#include "device_pool.h"
#include <atomic>
#include <chrono>
#include <cstdio>
#include <cstdlib>
#include <new>
#include <set>
#include <thread>
#include <vector>

static std::atomic<bool> no_host{false};
void* operator new(size_t n) {
  if (no_host) throw std::bad_alloc();
  if (void* p = std::malloc(n)) return p;
  throw std::bad_alloc();
}
void operator delete(void* p) noexcept { std::free(p); }
void operator delete(void* p, size_t) noexcept { std::free(p); }

struct Device {  // addresses only; room in bytes
  static constexpr int kNoMemory = 2;
  static std::mutex m;
  static long room, live, allocs;
  static int dev;
  static std::map<void*, size_t>* size;
  static int device(int* d) { return *d = dev, 0; }
  static int alloc(void** p, size_t n) {
    std::lock_guard<std::mutex> lock(m);
    if ((long)n > room) return kNoMemory;
    const bool off = no_host.exchange(false);  // the device's own bookkeeping is not what is tested
    *p = std::malloc(1);
    (*size)[*p] = n;
    no_host = off;
    room -= n, ++live, ++allocs;
    return 0;
  }
  static void release(void* p) {
    std::lock_guard<std::mutex> lock(m);
    room += size->at(p), --live;
    size->erase(p);
    std::free(p);
  }
};
std::mutex Device::m;
long Device::room = 1 << 30, Device::live = 0, Device::allocs = 0;
int Device::dev = 0;
std::map<void*, size_t>* Device::size = new std::map<void*, size_t>;

#define CHECK(x) do { if (!(x)) { std::printf("line %d: %s\n", __LINE__, #x); return 1; } } while (0)
using Pool = dg::DevicePool<Device>;

int main() {
  void *a, *b, *c;
  {  // handed out again: the smallest that fits, at most an eighth larger, of the same device
    Pool p(1 << 20);
    CHECK(!p.take(&a, 8000) && !p.take(&b, 9000) && a != b);
    p.give(a), p.give(b);
    CHECK(!p.take(&c, 7900) && c == a && !p.take(&a, 8192) && a == b);
    p.give(a), p.give(c);
    CHECK(!p.take(&b, 4096) && b != a && b != c);
    Device::dev = 1;
    CHECK(!p.take(&a, 8000) && a != c);
    Device::dev = 0;
    p.give(a), p.give(b), p.give(nullptr), p.give(&p);
    CHECK(p.release_kept() && !p.release_kept() && Device::live == 0);
  }
  {  // the bound: the longest kept leave first, a larger block goes straight back
    Pool p(16 * 1024);
    void* q[5];
    for (int i = 0; i < 5; ++i) CHECK(!p.take(&q[i], 4096));
    for (int i = 0; i < 5; ++i) p.give(q[i]);
    CHECK(Device::live == 4);
    CHECK(!p.take(&a, 17 * 1024));
    p.give(a);
    CHECK(Device::live == 4 && !p.take(&b, 4096) && b == q[1]);
    p.give(b), p.release_kept();
  }
  {  // a full device: what is kept goes back first, for raw blocks too
    Pool p(1 << 20);
    Device::room = 10000;
    CHECK(!p.take(&a, 4096));
    p.give(a);
    CHECK(!p.take(&b, 8192) && Device::live == 1);
    p.give(b);
    CHECK(!p.raw(&c, 9000) && Device::live == 1);
    CHECK(p.take(&a, 4096) == Device::kNoMemory && !a && p.raw(&a, 4096) == Device::kNoMemory && !a);
    Device::release(c);
    Device::room = 1 << 30;
  }
  {  // no host memory: errors, nothing thrown, nothing lost
    Pool p(1 << 20);
    CHECK(!p.take(&a, 512) && !p.take(&b, 512));
    p.give(a);
    no_host = true;
    CHECK(p.take(&c, 4096) == Device::kNoMemory && !c && Device::live == 2);
    CHECK(!p.take(&c, 512) && c == a);  // a block that is known needs none
    p.give(b), p.give(c), p.give(c);
    no_host = false;
    CHECK(Device::live == 2 && p.release_kept());
    CHECK(Device::live == 0);
  }
  {  // many kept blocks: 1e5 takes beside 1e5 others, in well under the time of 1e10 steps
    Pool p(1 << 28);
    std::vector<void*> q(100000);
    for (size_t i = 0; i < q.size(); ++i) CHECK(!p.take(&q[i], 512 + 512 * (i % 4)));
    for (void* x : q) p.give(x);
    const auto t0 = std::chrono::steady_clock::now();
    for (int i = 0; i < 100000; ++i) {
      CHECK(!p.take(&a, 512 + 512 * (i % 4)));
      p.give(a);
    }
    const double s = std::chrono::duration<double>(std::chrono::steady_clock::now() - t0).count();
    std::printf("100000 takes: %.3f s\n", s);
    CHECK(s < 3.0);
    p.release_kept();
  }
  {  // threads: a block in use has one owner
    Pool p(64 * 1024);
    std::mutex m;
    std::set<void*> used;
    std::atomic<int> wrong{0};
    std::vector<std::thread> ts;
    for (int t = 0; t < 6; ++t)
      ts.emplace_back([&, t] {
        for (int i = 0; i < 4000; ++i) {
          void* x;
          if (p.take(&x, 512 * (1 + (i * 7 + t) % 9))) ++wrong;
          { std::lock_guard<std::mutex> l(m); wrong += !used.insert(x).second; }
          { std::lock_guard<std::mutex> l(m); used.erase(x); }
          p.give(x);
        }
      });
    for (auto& t : ts) t.join();
    p.release_kept();
    CHECK(!wrong && Device::live == 0);
  }
  std::puts("pool ok");
  return 0;
}
"""


def test_pool(tmp_path):
    src, exe = tmp_path / "pool.cpp", tmp_path / "pool"
    src.write_text(_SOURCE)
    subprocess.run(["g++", "-std=c++17", "-O1", "-Wall", "-Werror", "-pthread", "-I",
                    os.path.join(ROOT, "dftcxx_amd", "csrc"), str(src), "-o", str(exe)], check=True)
    r = subprocess.run([str(exe)], capture_output=True, text=True, timeout=100)
    print(r.stdout)
    assert r.returncode == 0 and "pool ok" in r.stdout
