"""csrc/ps_transfer.h on a device made of host memory: transfers of strided rows through blocks of every size
that scarce memory leaves, down to none; no transfer waits for another's stream; the kept blocks are
bounded and given back; an error waits for the stream before the block is used again."""
import os
import shutil
import subprocess

import pytest

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "parallelstencil.jl_amd", "csrc")

SOURCE = r"""
#include <atomic>
#include <condition_variable>
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <functional>
#include <map>
#include <thread>
#include "ps_transfer.h"

#define CHECK(x) do { if (!(x)) { std::printf("line %d: %s\n", __LINE__, #x); std::exit(1); } } while (0)

static std::mutex dmu;
static std::map<char*, size_t> live;
static size_t room = SIZE_MAX, largest = 0, allocs = 0;

struct Dev {
  char* field;
  bool to_field;
  int64_t ny, pitch, plane;
  size_t w;
  int fail_at = -1, calls = 0, pending = 0, syncs = 0;
  std::function<void()> waiting;

  static char* alloc(size_t n) {
    std::lock_guard<std::mutex> lk(dmu);
    size_t used = 0;
    for (auto& b : live) used += b.second;
    if (n > room || used > room - n) return nullptr;
    char* p = (char*)std::malloc(n);
    live[p] = n, largest = std::max(largest, n), ++allocs;
    return p;
  }
  static void free(char* p) {
    std::lock_guard<std::mutex> lk(dmu);
    CHECK(live.erase(p) == 1);
    std::free(p);
  }
  int step() { ++pending; return calls++ == fail_at ? -7 : 0; }
  int copy(char* d, char* h, size_t n) {
    if (int e = step()) return e;
    std::memcpy(to_field ? d : h, to_field ? h : d, n);
    return 0;
  }
  char* row(int64_t r) const { return field + (r % ny) * pitch + (r / ny) * plane; }
  int rows(char* b, int64_t r, int64_t n) {
    if (int e = step()) return e;
    {
      std::lock_guard<std::mutex> lk(dmu);
      CHECK(live.count(b) && live[b] >= w * (size_t)n);
    }
    for (int64_t i = 0; i < n; ++i) std::memcpy(to_field ? row(r + i) : b + i * w, to_field ? b + i * w : row(r + i), w);
    return 0;
  }
  int sync() {
    if (waiting) waiting();
    pending = 0, ++syncs;
    return 0;
  }
};

using Pool = ps::BlockPool<Dev>;

static void round_trip(Pool& pool, size_t w, int64_t ny, int64_t nz) {
  const int64_t pitch = (int64_t)w + 5, plane = pitch * ny + 3, rows = ny * nz;
  std::string a((size_t)(plane * nz), 'x'), h((size_t)rows * w, 0), back(h.size(), 0);
  for (size_t i = 0; i < h.size(); ++i) h[i] = (char)(i * 7 + i / 251);
  Dev up{&a[0], true, ny, pitch, plane, w}, down{&a[0], false, ny, pitch, plane, w};
  CHECK(ps::transfer_rows(up, pool, true, w, rows, &h[0]) == 0 && up.pending == 0);
  CHECK(ps::transfer_rows(down, pool, false, w, rows, &back[0]) == 0 && down.pending == 0);
  CHECK(back == h);
  for (int64_t r = 0; r < rows; ++r)  // nothing beside the rows is written
    for (int64_t i = (int64_t)w; i < pitch; ++i) CHECK(up.row(r)[i] == 'x');
}

int main() {
  Pool pool;
  pool.field_made();
  for (size_t r : {(size_t)SIZE_MAX, (size_t)100000, (size_t)5000, (size_t)999, (size_t)100, (size_t)97, (size_t)96, (size_t)0}) {
    room = r;
    round_trip(pool, 97, 13, 11);
    round_trip(pool, 1, 7, 1);
    round_trip(pool, 1000, 1, 3);
    pool.field_freed(), pool.field_made();  // the kept blocks go with the last field
    CHECK(live.empty());
  }
  room = SIZE_MAX;
  round_trip(pool, 3000001, 7, 3);  // 63 MB in blocks of whole rows
  CHECK(largest <= ps::kBlockMax);
  const size_t before = allocs;
  round_trip(pool, ps::kBlockMax + 1, 2, 1);  // rows wider than a block: one by one
  CHECK(allocs == before);
  round_trip(pool, 3000001, 7, 3);
  CHECK(allocs == before);  // a kept block serves again

  {  // a transfer whose stream is busy holds up no other: the first waits until the second has finished
    std::mutex m;
    std::condition_variable cv;
    bool first_waits = false, second_done = false;
    std::string f1(4000, 0), f2(4000, 0), h1(2000, 1), h2(2000, 2);
    std::thread t([&] {
      Dev d{&f1[0], true, 10, 300, 3000, 200};
      d.waiting = [&] {
        std::unique_lock<std::mutex> lk(m);
        first_waits = true;
        cv.notify_all();
        CHECK(cv.wait_for(lk, std::chrono::seconds(20), [&] { return second_done; }));
      };
      CHECK(ps::transfer_rows(d, pool, true, 200, 10, &h1[0]) == 0);
    });
    {
      std::unique_lock<std::mutex> lk(m);
      CHECK(cv.wait_for(lk, std::chrono::seconds(20), [&] { return first_waits; }));
    }
    Dev d{&f2[0], true, 10, 300, 3000, 200};
    CHECK(ps::transfer_rows(d, pool, true, 200, 10, &h2[0]) == 0);
    {
      std::lock_guard<std::mutex> lk(m);
      second_done = true;
    }
    cv.notify_all();
    t.join();
  }
  {  // many at once: a block each, a few kept
    std::atomic<int> waiting{0};
    std::vector<std::thread> ts;
    for (int i = 0; i < 12; ++i)
      ts.emplace_back([&] {
        std::string f(4000, 0), h(2000, 3);
        Dev d{&f[0], true, 10, 300, 3000, 200};
        d.waiting = [&] {
          ++waiting;
          for (int k = 0; k < 2000 && waiting < 12; ++k) std::this_thread::sleep_for(std::chrono::milliseconds(10));
        };
        CHECK(ps::transfer_rows(d, pool, true, 200, 10, &h[0]) == 0 && waiting == 12);
      });
    for (auto& t : ts) t.join();
    CHECK(live.size() <= ps::kKept);
  }
  for (bool up : {true, false})  // an error at any step: reported, the stream waited for, the block given back
    for (int at = 0; at < 4; ++at) {
      std::string f(4000, 0), h(2000, 4);
      Dev d{&f[0], up, 10, 300, 3000, 200};
      d.fail_at = at;
      room = 1000;
      pool.field_freed(), pool.field_made();
      const int rc = ps::transfer_rows(d, pool, up, 200, 10, &h[0]);
      CHECK(rc == -7 && d.pending == 0 && d.syncs == 1 && live.size() == 1);
    }
  pool.field_freed();
  CHECK(live.empty());
  round_trip(pool, 97, 13, 11);  // with no field alive nothing is kept
  CHECK(live.empty());
  std::puts("ok");
}
"""


@pytest.mark.skipif(shutil.which("g++") is None, reason="no host compiler")
def test_transfers_through_blocks(tmp_path):
    src, exe = tmp_path / "transfer.cpp", tmp_path / "transfer"
    src.write_text(SOURCE)
    subprocess.run(["g++", "-std=c++17", "-O1", "-g", "-pthread", "-D_GLIBCXX_ASSERTIONS", "-I", CSRC, str(src), "-o", str(exe)], check=True)
    out = subprocess.run([str(exe)], capture_output=True, text=True, timeout=120)
    assert out.returncode == 0 and out.stdout == "ok\n", out.stdout + out.stderr
