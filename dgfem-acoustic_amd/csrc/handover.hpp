// Hand-over of data between the caller's host memory and the device.
//
// The caller's arrays are pageable and often freshly allocated. Here data come through page-locked
// slabs: large results in pieces whose transfer overlaps the copies into the caller's array (126 MB out
// 12.3 -> 9.5 ms), small ones read and written by the kernels in the slab itself, without copy commands.
#pragma once
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cstdint>
#include <cstring>
#include <exception>
#include <mutex>
#include <vector>

namespace dgk {

// Page-locked slabs of kSlabBytes, shared by all contexts and threads of the process: a call takes one
// for itself and gives it back. At most kSlabsKept wait for the next call, and kSlabsIdle when the last
// user has left: a program with one context at a time (a loop that creates, runs and destroys) would
// page-lock anew for each, and page-locking takes 0.2 ms a MB. The size: what the first large download of
// a process pays, against what a smaller slab costs each later one. get_state into fresh memory, one
// context a call, ms (first call of the process / later ones): 34.6 MB, two slabs of 16 MB freed with the
// context 8.7 / 2.5 or 7.3 (as the runtime kept the memory or not), one of 16 MB 6.1 / 2.4, 8 MB 3.3 / 2.4,
// 4 MB 2.5 / 2.4; 159.7 MB, 16 MB 11.3 / 10.4, 8 MB 11.2 / 10.5, 4 MB 11.5 / 10.8. Plain copies: 34.6 MB
// 3.5, 159.7 MB 15.3.
class Slabs {
 public:
  static constexpr size_t kSlabBytes = (size_t)8 << 20;
  static constexpr size_t kSlabsKept = 4, kSlabsIdle = 1;
  static Slabs& get() {
    static Slabs* s = new Slabs();  // never destroyed: contexts may outlive static destruction
    return *s;
  }
  void enter() {
    std::lock_guard<std::mutex> lk(mu_);
    ++users_;
  }
  void leave() {
    void* drop[kSlabsKept];
    size_t n = 0;
    {
      std::lock_guard<std::mutex> lk(mu_);
      if (--users_ == 0)
        while (nfree_ > kSlabsIdle) drop[n++] = free_[--nfree_];
    }
    while (n) (void)hipHostFree(drop[--n]);
  }
  void* take() {
    {
      std::lock_guard<std::mutex> lk(mu_);
      if (nfree_) return free_[--nfree_];
    }
    void* p = nullptr;
    if (hipHostMalloc(&p, kSlabBytes, hipHostMallocPortable) != hipSuccess) {
      (void)hipGetLastError();
      return nullptr;  // the caller falls back to the runtime's own copies
    }
    return p;
  }
  void give(void* p) {
    {
      std::lock_guard<std::mutex> lk(mu_);
      if (nfree_ < (users_ > 0 ? kSlabsKept : kSlabsIdle)) {
        free_[nfree_++] = p;
        return;
      }
    }
    (void)hipHostFree(p);
  }

 private:
  std::mutex mu_;
  void* free_[kSlabsKept];
  size_t nfree_ = 0;
  int64_t users_ = 0;
};

// Membership of a context in the pool's lifetime.
struct SlabUser {
  SlabUser() { Slabs::get().enter(); }
  ~SlabUser() { Slabs::get().leave(); }
  SlabUser(const SlabUser&) = delete;
  SlabUser& operator=(const SlabUser&) = delete;
};

// At most one slab for the length of a call, taken where data() is first asked for (null when none is to
// be had): a call that needs none takes none. Work on stream s that uses it is over when the call ends in
// the ordinary way; when an exception ends it, it is waited for here.
class Slab {
 public:
  explicit Slab(hipStream_t s) : s_(s), unwinding_(std::uncaught_exceptions()) {}
  ~Slab() {
    if (!p_) return;
    if (std::uncaught_exceptions() > unwinding_) (void)hipStreamSynchronize(s_);
    Slabs::get().give(p_);
  }
  Slab(const Slab&) = delete;
  Slab& operator=(const Slab&) = delete;
  char* data() {
    if (!asked_) p_ = (char*)Slabs::get().take();
    asked_ = true;
    return p_;
  }

 private:
  hipStream_t s_;
  int unwinding_;
  bool asked_ = false;
  char* p_ = nullptr;
};

// A piece of a transfer: `bytes` from device memory to host memory.
struct Piece {
  const char* dev;
  char* host;
  size_t bytes;
};

// Copies device pieces to host memory through the call's slab in slots of 2 MB: while slots are in transfer,
// this thread copies out the one that has landed. (Slots of 1 MB: an uneven ensemble's 16 states, 180 MB,
// take 0.5-1 ms more beside spinning threads.) Blocks until everything is in place. What the slab held is
// overwritten, in the order of stream s. The thread polls: one that sleeps gets its core back only at the
// end of a time slice when the caller's other threads (an OpenMP pool after a loop) spin on all of them, 4 ms
// a call; for the same reason the copying has no helper threads, which took 3 of 126 MB's 9.5 ms off on a
// quiet machine and cost 3 ms a call beside spinning ones.
inline hipError_t download(const std::vector<Piece>& pieces, hipStream_t s, Slab& slab) {
  constexpr size_t kSlot = (size_t)2 << 20, kSlots = Slabs::kSlabBytes / kSlot;
  std::vector<Piece> part;
  for (auto& q : pieces)
    for (size_t o = 0; o < q.bytes; o += kSlot)
      part.push_back({q.dev + o, q.host + o, std::min(kSlot, q.bytes - o)});
  const size_t n = part.size();
  char* const buf = n < 2 ? nullptr : slab.data();
  if (!buf) {
    hipError_t e = hipSuccess;
    for (size_t i = 0; i < pieces.size() && e == hipSuccess; ++i)
      e = hipMemcpyAsync(pieces[i].host, pieces[i].dev, pieces[i].bytes, hipMemcpyDeviceToHost, s);
    const hipError_t w = hipStreamSynchronize(s);  // also after an error: the host memory is the caller's
    return e != hipSuccess ? e : w;
  }
  hipEvent_t ev[kSlots];
  size_t nev = 0;
  hipError_t err = hipSuccess;
  for (; nev < std::min(n, kSlots); ++nev)
    if ((err = hipEventCreateWithFlags(&ev[nev], hipEventDisableTiming)) != hipSuccess) break;
  auto start = [&](size_t k) {
    hipError_t e = hipMemcpyAsync(buf + (k % kSlots) * kSlot, part[k].dev, part[k].bytes, hipMemcpyDeviceToHost, s);
    return e == hipSuccess ? hipEventRecord(ev[k % kSlots], s) : e;
  };
  for (size_t k = 0; k < std::min(n, kSlots) && err == hipSuccess; ++k) err = start(k);
  for (size_t k = 0; k < n && err == hipSuccess; ++k) {
    while ((err = hipEventQuery(ev[k % kSlots])) == hipErrorNotReady) {
    }
    if (err != hipSuccess) break;
    memcpy(part[k].host, buf + (k % kSlots) * kSlot, part[k].bytes);
    if (k + kSlots < n) err = start(k + kSlots);
  }
  if (err != hipSuccess) (void)hipStreamSynchronize(s);  // no transfer may outlive the slab's loan
  for (size_t i = 0; i < nev; ++i) (void)hipEventDestroy(ev[i]);
  return err;
}

}  // namespace dgk
