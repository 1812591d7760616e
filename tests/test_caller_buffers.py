"""Callers' device buffers (cuhc_amd/csrc/caller_buffers.hpp).

The pool's rules are checked on the CPU: the header is compiled with g++ into a
driver over a stand-in runtime that records what is allocated, freed and waited
for (skipped when g++ is absent). The GPU test goes through the C ABI.
"""

import ctypes
import shutil
import subprocess
from pathlib import Path

import numpy as np
import pytest

CSRC = Path(__file__).resolve().parent.parent / "cuhc_amd" / "csrc"
INVALID_VALUE, OUT_OF_MEMORY = 1, 2

DRIVER = r"""
#include "caller_buffers.hpp"
#include <atomic>
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <set>
#include <thread>
struct World { // the runtime's state
  std::mutex mutex;
  std::map<void *, size_t> live;
  int device = 0, waited = -1, waitStatus = 0, others = 0;
  size_t room = (size_t)1 << 40, limit = 1000;
} world;
struct Fake {
  int current(int *d) { *d = world.device; return 0; }
  int allocate(void **p, size_t bytes) {
    std::lock_guard<std::mutex> lock(world.mutex);
    size_t used = 0;
    for (auto &e : world.live)
      used += e.second;
    if (bytes > world.room || used > world.room - bytes)
      return cuhc::kStatusOutOfMemory;
    *p = std::malloc(1);
    world.live[*p] = bytes;
    return 0;
  }
  int release(void *p) {
    std::lock_guard<std::mutex> lock(world.mutex);
    return world.live.erase(p) ? 0 : cuhc::kStatusInvalidValue; // addresses are not used again
  }
  int wait(int d) { world.waited = d; return world.waitStatus; }
  bool covers(void *p, size_t bytes) {
    std::lock_guard<std::mutex> lock(world.mutex);
    const auto it = world.live.find(p);
    return it != world.live.end() && it->second >= bytes;
  }
  void releaseOther() { ++world.others; }
  size_t keepLimit() { return world.limit; }
};
#define CHECK(x) do { if (!(x)) { std::printf("line %d: %s\n", __LINE__, #x); return 1; } } while (0)
int main(int argc, char **argv) {
  cuhc::CallerBuffers<Fake> pool;
  void *a = nullptr, *b = nullptr, *c = nullptr;
  const char *test = argv[1];
  if (!std::strcmp(test, "second_free")) {
    CHECK(pool.alloc(&a, 100) == 0 && a);
    CHECK(pool.free(a) == 0 && pool.keptBytes() == 100);
    CHECK(pool.free(a) == cuhc::kStatusInvalidValue);
    CHECK(world.live.count(a) == 1 && pool.keptBytes() == 100); // still an allocation
    CHECK(pool.alloc(&b, 100) == 0 && b == a);                  // used again, once
    CHECK(pool.alloc(&c, 100) == 0 && c != a);
    CHECK(pool.free(b) == 0 && pool.free(b) == cuhc::kStatusInvalidValue);
    CHECK(pool.free(c) == 0 && pool.free(nullptr) == 0);
  } else if (!std::strcmp(test, "foreign")) { // not the pool's: the runtime decides
    Fake f;
    CHECK(f.allocate(&a, 8) == 0 && pool.free(a) == 0 && world.live.empty());
    CHECK(pool.free(a) == cuhc::kStatusInvalidValue);
    CHECK(pool.alloc(&b, 8) == 0 && f.release(b) == 0); // freed past the pool
    CHECK(pool.free(b) == cuhc::kStatusInvalidValue && pool.keptBytes() == 0);
  } else if (!std::strcmp(test, "devices")) { // a buffer stays with its device
    world.device = 1;
    CHECK(pool.alloc(&a, 100) == 0);
    world.device = 0;
    CHECK(pool.free(a) == 0 && world.waited == 1);
    CHECK(pool.alloc(&b, 100) == 0 && b != a);
    world.device = 1;
    CHECK(pool.alloc(&c, 100) == 0 && c == a);
  } else if (!std::strcmp(test, "bounds")) {
    CHECK(pool.alloc(&a, 600) == 0 && pool.alloc(&b, 600) == 0 && pool.alloc(&c, 1001) == 0);
    CHECK(pool.free(a) == 0 && pool.free(b) == 0 && pool.free(c) == 0); // the latest is kept
    CHECK(pool.keptBytes() == 600 && world.live.size() == 1 && world.live.count(b) == 1);
    world.room = 700; // the kept buffer makes way
    void *kept = b;
    CHECK(pool.alloc(&b, 650) == 0 && world.others == 1 && world.live.count(kept) == 0);
    CHECK(pool.alloc(&c, 650) == cuhc::kStatusOutOfMemory && c == nullptr);
    CHECK(pool.alloc(&c, ~(size_t)0) == cuhc::kStatusOutOfMemory && c == nullptr);
    CHECK(pool.free(b) == 0);
    pool.releaseKept();
    CHECK(pool.keptBytes() == 0 && world.live.empty());
    CHECK(pool.free(b) == cuhc::kStatusInvalidValue);
  } else if (!std::strcmp(test, "oldest")) { // many sizes: those of the latest calls are kept
    cuhc::KeptBlocks<size_t> blocks;
    std::vector<int> gone;
    auto release = [&](void *p) { gone.push_back((int)(size_t)p); };
    for (size_t i = 1; i <= 12; ++i) // keys 1 2 3 1 2 3 ..., 100 bytes each
      CHECK(blocks.put((i - 1) % 3 + 1, (void *)i, 100, 1000, release));
    CHECK((gone == std::vector<int>{1, 2}) && blocks.bytes() == 1000);
    CHECK((size_t)blocks.take(1) == 10 && (size_t)blocks.take(1) == 7 && (size_t)blocks.take(1) == 4);
    CHECK(!blocks.take(1) && !blocks.take(9) && blocks.bytes() == 700);
    CHECK(blocks.put(7, (void *)20, 650, 1000, release) && blocks.bytes() == 950);
    CHECK((gone == std::vector<int>{1, 2, 3, 5, 6, 8}));
    CHECK(!blocks.put(7, (void *)21, 1001, 1000, release) && gone.size() == 6);
    blocks.clear(release);
    CHECK((gone == std::vector<int>{1, 2, 3, 5, 6, 8, 9, 11, 12, 20}) && blocks.bytes() == 0);
    CHECK(!blocks.take(7));
  } else if (!std::strcmp(test, "failed_wait")) { // perhaps still in use: not kept
    CHECK(pool.alloc(&a, 100) == 0);
    world.waitStatus = 719;
    CHECK(pool.free(a) == 719 && pool.keptBytes() == 0 && world.live.empty());
  } else { // threads: no buffer in two hands
    std::atomic<int> bad{0};
    std::mutex m;
    std::set<void *> inUse;
    std::vector<std::thread> threads;
    for (int t = 0; t < 8; ++t)
      threads.emplace_back([&, t] {
        for (int i = 0; i < 2000; ++i) {
          void *p = nullptr;
          bad += pool.alloc(&p, 50 + 50 * ((i + t) % 3)) != 0;
          {
            std::lock_guard<std::mutex> lock(m);
            bad += !inUse.insert(p).second;
          }
          {
            std::lock_guard<std::mutex> lock(m);
            inUse.erase(p);
          }
          bad += pool.free(p) != 0;
        }
      });
    for (auto &t : threads)
      t.join();
    CHECK(bad == 0 && pool.keptBytes() <= world.limit);
    pool.releaseKept();
    CHECK(world.live.empty());
  }
  return 0;
}
"""


@pytest.fixture(scope="module")
def driver(tmp_path_factory):
    gxx = shutil.which("g++")
    if gxx is None:
        pytest.skip("g++ not available")
    d = tmp_path_factory.mktemp("caller_buffers")
    (d / "driver.cpp").write_text(DRIVER)
    exe = d / "driver"
    subprocess.run([gxx, "-O1", "-std=c++17", "-pthread", "-I", str(CSRC), str(d / "driver.cpp"),
                    "-o", str(exe)], check=True, capture_output=True, text=True)
    return exe


@pytest.mark.parametrize("rule", ["second_free", "foreign", "devices", "bounds", "oldest",
                                  "failed_wait", "threads"])
def test_rules(driver, rule):
    run = subprocess.run([str(driver), rule], capture_output=True, text=True)
    assert run.returncode == 0, run.stdout


@pytest.mark.gpu
def test_buffers_through_the_abi():
    from cuhc_amd import _lib
    lib = _lib.lib

    def alloc(nbytes):
        p = ctypes.c_void_p()
        _lib.check(lib.cuhc_device_alloc(nbytes, ctypes.byref(p)))
        return p

    nbytes = 12_345 * 4
    a = alloc(nbytes)
    assert lib.cuhc_device_free(a) == 0
    assert lib.cuhc_device_free(a) == INVALID_VALUE
    b, c = alloc(nbytes), alloc(nbytes)  # a's memory again, and another
    assert b.value == a.value and c.value != a.value
    src = np.arange(12_345, dtype=np.int32)
    out = np.zeros((2, 12_345), np.int32)
    for p, x, row in [(b, src, out[0]), (c, -src, out[1])]:
        _lib.check(lib.cuhc_copy_to_device(p, x.ctypes.data_as(ctypes.c_void_p), nbytes))
    for p, row in [(b, out[0]), (c, out[1])]:
        _lib.check(lib.cuhc_copy_to_host(row.ctypes.data_as(ctypes.c_void_p), p, nbytes))
    np.testing.assert_array_equal(out, [src, -src])
    assert lib.cuhc_device_free(b) == 0 and lib.cuhc_device_free(c) == 0
    lib.cuhc_release()
    assert lib.cuhc_device_free(b) != 0  # given back: no buffer any more
    p = ctypes.c_void_p(1)
    assert lib.cuhc_device_alloc(2**64 - 1, ctypes.byref(p)) != 0 and not p.value
