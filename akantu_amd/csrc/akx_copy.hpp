// akx_copy.hpp -- copies between a caller's pageable host arrays and the
// device for the calls that return or take host data.
//
// The runtime's own pageable copies reach 18 GB/s to the host and 30 GB/s to
// the device on a card whose link carries 57: it stages the pages or pins them
// on the calling thread, in turn with the transfer, and a caller's fresh array
// is mapped page by page on the way.  Pages that it has pinned also make later
// calls slow that map or free memory near them: with uploads of 1 to 24 MB
// taken straight from the caller's arrays a process of many operators paid 1.47
// ms for a gradient of 9 MB that takes 0.38 through slots.  Here the data pass
// through small page-locked slots, two per helper thread: a slot travels while
// the other is copied, and large copies use several threads, since one thread
// alone fills fresh pages at 13 GB/s (41 MB into a fresh array: 4.2 ms by
// hipMemcpy).
#pragma once

#include <hip/hip_runtime.h>

#include <atomic>
#include <cstring>
#include <system_error>
#include <thread>
#include <vector>

namespace akx {

class HostCopier {
 public:
  ~HostCopier() { release(); }

  void release() {
    for (auto& lane : lanes_)
      for (auto& s : lane) {
        (void)idle(s);
        if (s.done) (void)hipEventDestroy(s.done);
        if (s.mem) (void)hipHostFree(s.mem);
        s = Slot();
      }
  }

  // Copies that are complete when the call returns, after the work queued on
  // the stream.
  hipError_t to_host(int device, hipStream_t s, void* host, const void* dev, size_t bytes) {
    if (bytes == 0) return hipSuccess;
    hipError_t e;
    if (bytes > SLOT) {
      e = run(device, bytes, [=](int lane, int lanes, size_t chunks) -> hipError_t {
        return fetch(lane, lanes, chunks, s, static_cast<char*>(host),
                     static_cast<const char*>(dev), bytes);
      });
    } else {
      Slot& slot = lanes_[0][0];
      e = fillable(slot, s);
      // An event tells the end, but for small transfers by DMA, where it costs
      // 8 us (17 KB 12 us with the stream's wait).  Up to BY_KERNEL the stream's
      // wait is the slower one behind many launches (12: 72 us, 50 by event),
      // and above SMALL the calls that follow it were (operators on 26,970
      // hexahedra 3.85 ms, 3.79 by events).
      const bool event = bytes <= BY_KERNEL || bytes > SMALL;
      if (e == hipSuccess && event) e = with_event(slot);
      if (e == hipSuccess && bytes > SMALL) e = hipEventSynchronize(slot.done);  // see run
      if (e == hipSuccess) e = hipMemcpyAsync(slot.mem, dev, bytes, hipMemcpyDeviceToHost, s);
      if (e == hipSuccess && event) e = hipEventRecord(slot.done, s);
      if (e == hipSuccess) e = event ? hipEventSynchronize(slot.done) : hipStreamSynchronize(s);
      if (e == hipSuccess) {
        std::memcpy(host, slot.mem, bytes);
        for (auto& up : lanes_[0])
          if (up.upload == s) up.upload = nullptr;
      }
    }
    return e == hipErrorOutOfMemory ? plain(s, host, dev, bytes, hipMemcpyDeviceToHost) : e;
  }
  // Returns when the host array has been read; the device copy is ordered
  // before later work on the stream.
  hipError_t to_device(int device, hipStream_t s, void* dev, const void* host, size_t bytes) {
    if (bytes == 0) return hipSuccess;
    hipError_t e;
    if (bytes > SLOT)
      e = run(device, bytes, [=](int lane, int lanes, size_t chunks) -> hipError_t {
        return send(lane, lanes, chunks, s, static_cast<char*>(dev),
                    static_cast<const char*>(host), bytes);
      });
    else  // an event costs 5 us, as much as the transfer of a small array
      e = send_slot(lanes_[0][turn_ ^= 1], s, dev, host, bytes, bytes > SMALL);
    return e == hipErrorOutOfMemory ? plain(s, dev, host, bytes, hipMemcpyHostToDevice) : e;
  }

 private:
  static constexpr size_t SLOT = size_t(1) << 20;
  static constexpr size_t SMALL = size_t(128) << 10;
  // up to here the runtime fills page-locked memory by a kernel, above by DMA
  static constexpr size_t BY_KERNEL = size_t(16) << 10;
  static constexpr int LANES = 4;
  struct Slot {
    void* mem = nullptr;
    hipEvent_t done = nullptr;     // the last transfer of a longer copy
    hipStream_t upload = nullptr;  // a small upload may be reading the slot
  };
  Slot lanes_[LANES][2];
  int turn_ = 0;  // slot of the last upload

  // One lane up to 8 MB: inference of 200,003 points (5.6 MB each way) takes
  // 0.66 ms with one or two, and starting threads costs a first call 0.4 ms.
  // Above, four: the FEEngine operators on 27,000 hexahedra (results of up to
  // 41 MB) take 5.9 ms with one lane, 4.7 with two, 3.8 with four or eight.
  static int lanes_for(size_t bytes) { return bytes <= (size_t(8) << 20) ? 1 : LANES; }

  // waits until nothing reads or fills the slot
  static hipError_t idle(Slot& s) {
    hipError_t e = hipSuccess;
    if (s.upload) e = hipStreamSynchronize(s.upload);
    s.upload = nullptr;
    if (s.done && e == hipSuccess) e = hipEventSynchronize(s.done);
    return e;
  }
  static hipError_t allocated(Slot& s) {
    if (s.mem || hipHostMalloc(&s.mem, SLOT, hipHostMallocDefault) == hipSuccess)
      return hipSuccess;
    s.mem = nullptr;
    (void)hipGetLastError();
    return hipErrorOutOfMemory;
  }
  // the runtime's own copy, where there is no page-locked memory to be had
  static hipError_t plain(hipStream_t s, void* to, const void* from, size_t bytes,
                          hipMemcpyKind kind) {
    const hipError_t e = hipMemcpyAsync(to, from, bytes, kind, s);
    return e == hipSuccess ? hipStreamSynchronize(s) : e;
  }
  static hipError_t with_event(Slot& s) {
    if (s.done) return hipSuccess;
    const hipError_t e = hipEventCreateWithFlags(&s.done, hipEventDisableTiming);
    if (e != hipSuccess) s.done = nullptr;
    return e;
  }
  // the slot takes a transfer on stream s, which follows an upload on s
  static hipError_t fillable(Slot& slot, hipStream_t s) {
    if (slot.upload && slot.upload != s)
      if (hipError_t e = idle(slot)) return e;
    return allocated(slot);
  }

  template <typename F>
  hipError_t run(int device, size_t bytes, F&& lane_copy) {
    const size_t chunks = (bytes + SLOT - 1) / SLOT;
    const int lanes = lanes_for(bytes);
    std::atomic<int> first{int(hipSuccess)};
    auto work = [&](int lane) {
      hipError_t e = hipSuccess;
      // uploads of the same call first: queued behind them and the kernels that
      // read them, the transfers start up to 30 us late (gradient of 8,000
      // hexahedra, 4.4 MB: 219 us, 243 without the wait)
      if (lane == 0)
        for (auto& up : lanes_[0]) e = e == hipSuccess ? idle(up) : e;
      else
        (void)hipSetDevice(device);
      if (e == hipSuccess) e = lane_copy(lane, lanes, chunks);
      if (e != hipSuccess) {
        int none = int(hipSuccess);
        first.compare_exchange_strong(none, int(e));
      }
    };
    std::thread helpers[LANES];
    int started = 1;
    try {
      for (; started < lanes; ++started) helpers[started] = std::thread(work, started);
    } catch (const std::system_error&) {
      // no more threads: this one takes the remaining lanes in turn
    }
    work(0);
    for (int k = started; k < lanes; ++k) work(k);
    for (int k = 1; k < started; ++k) helpers[k].join();
    return hipError_t(first.load());
  }

  // Chunks lane, lane + lanes, ... of a transfer to the host: two in flight.
  hipError_t fetch(int lane, int lanes, size_t chunks, hipStream_t s, char* host,
                   const char* dev, size_t bytes) {
    auto size = [&](size_t k) { return k + 1 < chunks ? SLOT : bytes - k * SLOT; };
    auto start = [&](size_t k, Slot& slot) -> hipError_t {
      hipError_t e = fillable(slot, s);
      if (e == hipSuccess) e = with_event(slot);
      if (e == hipSuccess)
        e = hipMemcpyAsync(slot.mem, dev + k * SLOT, size(k), hipMemcpyDeviceToHost, s);
      return e == hipSuccess ? hipEventRecord(slot.done, s) : e;
    };
    Slot* slots = lanes_[lane];
    size_t next = size_t(lane);
    for (int j = 0; j < 2 && next < chunks; ++j, next += size_t(lanes))
      if (hipError_t e = start(next, slots[j])) return e;
    int j = 0;
    for (size_t k = size_t(lane); k < chunks; k += size_t(lanes), j ^= 1) {
      if (hipError_t e = hipEventSynchronize(slots[j].done)) return e;
      std::memcpy(host + k * SLOT, slots[j].mem, size(k));
      if (next < chunks) {
        if (hipError_t e = start(next, slots[j])) return e;
        next += size_t(lanes);
      }
    }
    return hipSuccess;
  }

  // from the host array through a slot; without an event the stream tells
  static hipError_t send_slot(Slot& slot, hipStream_t s, void* dev, const void* host,
                              size_t bytes, bool event) {
    hipError_t e = idle(slot);
    if (e == hipSuccess) e = allocated(slot);
    if (e == hipSuccess && event) e = with_event(slot);
    if (e != hipSuccess) return e;
    std::memcpy(slot.mem, host, bytes);
    if ((e = hipMemcpyAsync(dev, slot.mem, bytes, hipMemcpyHostToDevice, s))) return e;
    slot.upload = s;
    if (event && (e = hipEventRecord(slot.done, s)) == hipSuccess) slot.upload = nullptr;
    return e;
  }
  hipError_t send(int lane, int lanes, size_t chunks, hipStream_t s, char* dev, const char* host,
                  size_t bytes) {
    int j = 0;
    for (size_t k = size_t(lane); k < chunks; k += size_t(lanes), j ^= 1) {
      const size_t n = k + 1 < chunks ? SLOT : bytes - k * SLOT;
      if (hipError_t e = send_slot(lanes_[lane][j], s, dev + k * SLOT, host + k * SLOT, n, true))
        return e;
    }
    if (lane == 0) turn_ = j ^ 1;  // the next upload takes the slot used before the last
    return hipSuccess;
  }
};

// Device buffers that the operator calls of one context reuse, taken in order
// by a call and returned at its end (the calls are synchronous).  Between calls
// a buffer of up to KEEP bytes stays allocated while their sum is at most
// KEEP_ALL, which holds the operand and the result of a call; the others are
// given back (freeing and allocating 77 + 206 MB costs B^T D 0.95 ms of 11).
class ScratchPool {
 public:
  static constexpr size_t KEEP = size_t(256) << 20, KEEP_ALL = 2 * KEEP;
  ~ScratchPool() { release(); }
  void release() {
    for (auto& b : bufs_)
      if (b.p) (void)hipFree(b.p);
    bufs_.clear();
  }
  size_t kept() const {  // bytes held now
    size_t sum = 0;
    for (const auto& b : bufs_) sum += b.cap;
    return sum;
  }
  class Use {
   public:
    explicit Use(ScratchPool& p) : pool_(p) { pool_.next_ = 0; }
    ~Use() {
      size_t sum = 0;
      for (auto& b : pool_.bufs_)
        if (b.cap > KEEP || b.cap > KEEP_ALL - sum) {
          (void)hipFree(b.p);
          b = Buf();
        } else {
          sum += b.cap;
        }
      pool_.next_ = 0;
    }

   private:
    ScratchPool& pool_;
  };
  hipError_t take(size_t bytes, void** out) {
    *out = nullptr;
    if (next_ == bufs_.size()) bufs_.emplace_back();
    Buf& b = bufs_[next_];
    if (b.cap < bytes || !b.p) {
      if (b.p) (void)hipFree(b.p);
      b = Buf();
      const size_t cap = bytes < 256 ? 256 : bytes;
      hipError_t e = hipMalloc(&b.p, cap);
      if (e != hipSuccess) {
        b.p = nullptr;
        return e;
      }
      b.cap = cap;
    }
    ++next_;
    *out = b.p;
    return hipSuccess;
  }

 private:
  struct Buf {
    void* p = nullptr;
    size_t cap = 0;
  };
  std::vector<Buf> bufs_;
  size_t next_ = 0;
};

}  // namespace akx
