// Device memory of the library: the pool behind pm_malloc / pm_free.
//
// Freed blocks are kept for the next allocation of the same size.  Every density or potential on device
// arrays allocates its result: hipMalloc + hipFree of a 384^3 grid cost 0.3 ms a call, and the driver
// clears freed memory at about 35 GB/s, so a loop that allocates faster than that ends up waiting for it
// (6.4 ms per 384^3 density, 0.5 ms of which are kernels).
// A block is put back only when its device is idle, as hipFree would have waited too, so no stream can
// still use it when it is handed out again, and only to callers whose current device is its own (the
// freeing thread's current device may be another).  The pool holds at most kPoolBytes (the oldest blocks go
// first), and everything is given back before an allocation fails and before free memory is reported.
//
// A scratch buffer that calls of the library take in turns is kept the same way: grown to the largest
// request, up to kScratchBytes between calls, and given back with the rest while no call uses it.
//
// Api is the device runtime (a CPU stand-in in tests): Error and its values Api::ok, Api::out_of_memory
// and Api::invalid, and the calls used below.
#pragma once
#include <cstddef>
#include <cstdint>
#include <mutex>

namespace pm {

constexpr size_t kPoolBytes = (size_t)4 << 30;
constexpr size_t kPoolGrain = (size_t)64 << 10;  // blocks are whole multiples of this
constexpr int kPoolBlocks = 64;
constexpr size_t kScratchBytes = (size_t)1 << 30;

template <class Api> class DevicePool {
 public:
  using Error = typename Api::Error;

  // Api::malloc that gives back what the pool keeps before it fails (every allocation of the library)
  Error plain_alloc(void** ptr, size_t bytes) {
    Error e = Api::malloc(ptr, bytes);
    if (e == Api::out_of_memory) {
      Api::clear_error();
      give_back();
      e = Api::malloc(ptr, bytes);
      if (e != Api::ok) Api::clear_error();  // reported here, not by the next launch's check
    }
    return e;
  }

  Error alloc(void** ptr, size_t bytes) {
    if (bytes > kPoolBytes) return plain_alloc(ptr, bytes);  // never kept: no rounding, which could overflow
    bytes = (bytes > kPoolGrain ? (bytes + kPoolGrain - 1) / kPoolGrain : 1) * kPoolGrain;
    const int device = Api::current_device();
    {
      std::lock_guard<std::mutex> lk(mu_);
      for (int i = n_ - 1; i >= 0; --i)  // the one freed last
        if (blocks_[i].bytes == bytes && blocks_[i].device == device) {
          *ptr = take(i);
          return Api::ok;
        }
    }
    return plain_alloc(ptr, bytes);
  }

  Error free(void* ptr) {
    void* base = nullptr;
    size_t bytes = 0;
    int device = 0;
    // pointers that do not start an allocation go to Api::free, which names the error
    if (Api::range(&base, &bytes, ptr) != Api::ok || base != ptr || bytes % kPoolGrain || bytes > kPoolBytes ||
        Api::device_of(&device, ptr) != Api::ok || synchronize(device) != Api::ok) {
      Api::clear_error();
      return Api::free(ptr);
    }
    std::lock_guard<std::mutex> lk(mu_);
    for (int i = 0; i < n_; ++i)
      if (blocks_[i].ptr == ptr) return Api::invalid;  // freed twice
    while (n_ == kPoolBlocks || bytes_ + bytes > kPoolBytes) (void)Api::free(take(0));
    blocks_[n_++] = {ptr, bytes, device};
    bytes_ += bytes;
    return Api::ok;
  }

  // The scratch buffer with room for `bytes` (null: no memory); the caller's until scratch_done().  One
  // caller at a time.
  void* scratch(size_t bytes) {
    {
      std::lock_guard<std::mutex> lk(mu_);
      scratch_busy_ = true;
    }
    if (bytes > scratch_bytes_) {
      drop_scratch();
      if (plain_alloc(&scratch_, bytes) == Api::ok) scratch_bytes_ = bytes;
      else scratch_ = nullptr;
    }
    return scratch_;
  }
  // no work uses the scratch buffer any more
  void scratch_done() {
    std::lock_guard<std::mutex> lk(mu_);
    if (scratch_bytes_ > kScratchBytes) drop_scratch();
    scratch_busy_ = false;
  }

  void give_back() {
    std::lock_guard<std::mutex> lk(mu_);
    while (n_) (void)Api::free(take(0));
    if (!scratch_busy_) drop_scratch();
  }

 private:
  struct Block {
    void* ptr;
    size_t bytes;
    int device;
  };

  // waits for everything on `device`, whichever device the thread has current
  static Error synchronize(int device) {
    const int current = Api::current_device();
    if (device == current) return Api::synchronize();
    Error e = Api::set_device(device);
    if (e == Api::ok) e = Api::synchronize();
    const Error back = Api::set_device(current);
    return e != Api::ok ? e : back;
  }

  // (callers hold mu_)
  void* take(int i) {
    void* p = blocks_[i].ptr;
    bytes_ -= blocks_[i].bytes;
    --n_;
    for (; i < n_; ++i) blocks_[i] = blocks_[i + 1];
    return p;
  }

  // (by the scratch buffer's user, or with mu_ held while it has none)
  void drop_scratch() {
    if (scratch_) (void)Api::free(scratch_);
    scratch_ = nullptr;
    scratch_bytes_ = 0;
  }

  std::mutex mu_;
  Block blocks_[kPoolBlocks];  // free blocks, oldest first
  int n_ = 0;
  size_t bytes_ = 0;  // their bytes
  void* scratch_ = nullptr;
  size_t scratch_bytes_ = 0;
  bool scratch_busy_ = false;
};

}  // namespace pm
