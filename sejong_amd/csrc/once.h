// One-time setup per device, for entry points that several host threads may
// call at once.  No HIP here: a caller passes the device's number.
#pragma once
#include <atomic>
#include <mutex>

namespace sj {

// once(device, f): f's status, f run once per device.  A caller that arrives
// while another thread is in f waits for it, so nobody goes on before the
// setup is complete.  Devices past the table run f on every call.
class OncePerDevice {
 public:
  template <class F>
  int operator()(int device, F f) {
    if (device < 0 || device >= DEVICES) return f();
    Slot& s = slots_[device];
    if (!s.done.load(std::memory_order_acquire)) {
      std::lock_guard<std::mutex> lock(mutex_);
      if (!s.done.load(std::memory_order_relaxed)) {
        s.status = f();
        s.done.store(true, std::memory_order_release);
      }
    }
    return s.status;
  }

 private:
  static constexpr int DEVICES = 64;
  struct Slot {
    std::atomic<bool> done{false};
    int status = 0;
  };
  Slot slots_[DEVICES];
  std::mutex mutex_;
};

}  // namespace sj
