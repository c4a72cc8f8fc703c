// Transfers between host memory and fields whose rows are not dense, through a dense block on the device
// that a kernel packs or unpacks: a strided copy moves its rows one by one, about 9 us each (64^3 FP64
// 37 ms, 256^3 604 to the device; through a block 0.08 and 4.7). Host code only, on a device given as a
// template argument (ps_runtime.hip: HIP).
//
// Every transfer under way has a block of its own, so transfers on different streams and threads do not
// wait for each other. Up to kKept blocks are kept between transfers, and none once the last field is
// freed. Where memory for a whole block (the field, at most kBlockMax) cannot be had, half of it serves,
// and so on down to one row; where that cannot be had either, the rows are copied one by one.
#pragma once
#include <algorithm>
#include <cstddef>
#include <cstdint>
#include <mutex>
#include <vector>

namespace ps {

constexpr size_t kBlockMax = 32u << 20;
constexpr size_t kKept = 4;

template <class Dev>
class BlockPool {
 public:
  struct Block {
    char* p = nullptr;
    size_t cap = 0;
  };

  // A block of `want` bytes, or of at least `least` where memory is scarce; p is null if there is none.
  Block take(size_t want, size_t least) {
    Block b = kept_of(want);
    if (b.p) return b;
    if ((b.p = Dev::alloc(want))) b.cap = want;
    else b = kept_of(least);
    for (size_t n = want / 2; !b.p && n >= least; n /= 2)
      if ((b.p = Dev::alloc(n))) b.cap = n;
    if (!b.p && want > least && (b.p = Dev::alloc(least))) b.cap = least;
    return b;
  }

  // After the last use of the block on the device has finished.
  void give(Block b) {
    if (!b.p) return;
    {
      std::lock_guard<std::mutex> lk(mu);
      if (fields > 0) {
        kept.push_back(b);
        b = Block{};
        if (kept.size() > kKept) {
          auto least = std::min_element(kept.begin(), kept.end(), [](const Block& x, const Block& y) { return x.cap < y.cap; });
          b = *least;
          kept.erase(least);
        }
      }
    }
    if (b.p) Dev::free(b.p);
  }

  void field_made() {
    std::lock_guard<std::mutex> lk(mu);
    ++fields;
  }
  void field_freed() {
    std::vector<Block> drop;
    {
      std::lock_guard<std::mutex> lk(mu);
      if (--fields > 0) return;
      drop.swap(kept);
    }
    for (auto& b : drop) Dev::free(b.p);
  }

 private:
  // the smallest kept block of at least n bytes
  Block kept_of(size_t n) {
    std::lock_guard<std::mutex> lk(mu);
    auto best = kept.end();
    for (auto it = kept.begin(); it != kept.end(); ++it)
      if (it->cap >= n && (best == kept.end() || it->cap < best->cap)) best = it;
    if (best == kept.end()) return Block{};
    const Block b = *best;
    kept.erase(best);
    return b;
  }

  std::mutex mu;
  std::vector<Block> kept;
  int64_t fields = 0;  // live allocations of fields
};

// `rows` rows of w bytes between the field and `host` (dense). dev.copy(d, h, n) copies between device and
// host and dev.rows(block, r, n) between a block and rows r..r+n-1 of the field, both ordered on the
// transfer's stream, in the direction of the transfer; dev.row(r) is row r's address, dev.sync() waits for
// the stream. Each returns 0 or an error, which ends the transfer.
template <class Dev>
int transfer_rows(Dev& dev, BlockPool<Dev>& pool, bool to_field, size_t w, int64_t rows, char* host) {
  typename BlockPool<Dev>::Block b;
  if (w <= kBlockMax) b = pool.take(std::min<size_t>(w * (size_t)rows, kBlockMax / w * w), w);  // wider rows are worth a copy each
  int rc = 0;
  if (!b.p) {
    for (int64_t r = 0; r < rows && !rc; ++r) rc = dev.copy(dev.row(r), host + (size_t)r * w, w);
    const int e = dev.sync();
    return rc ? rc : e;
  }
  const int64_t per = (int64_t)(b.cap / w);
  for (int64_t r = 0; r < rows && !rc; r += per) {
    const int64_t n = std::min(per, rows - r);
    char* const h = host + (size_t)r * w;
    if (to_field) rc = dev.copy(b.p, h, w * (size_t)n);
    if (!rc) rc = dev.rows(b.p, r, n);
    if (!rc && !to_field) rc = dev.copy(b.p, h, w * (size_t)n);
  }
  const int e = dev.sync();  // also after an error: the block and the host memory may still be in use
  pool.give(b);
  return rc ? rc : e;
}

}  // namespace ps
