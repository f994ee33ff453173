// rf_store.h -- host side of the operator's near store (rf_operator.hip): its
// device memory, and whether what it holds is a system.
//
// The products take their loop bounds and addresses from the store, so nothing
// may read it before an assembly has filled it, nor after one that failed
// part way.  It grows inside a step, which a thread may drive while another GPU
// is its current one: the memory belongs to the simulation's GPU, and the
// thread's current one stays.  Runtime is the device memory's interface: HIP's
// in the library, a model of it in the CPU test.
#pragma once

#include <cstdint>

namespace rf {

template <class Runtime>
class NearMemory {
 public:
  ~NearMemory() { release(); }

  void set_device(int device) { device_ = device; }

  // An assembly begins: there is no system until complete().
  void begin() { complete_ = false; }
  void complete() { complete_ = true; }
  bool holds_system() const { return complete_; }

  // Room for `floats` in place of what there is (which nothing in flight may
  // use, and which is gone either way); false if there is none.
  bool reserve(int64_t floats) {
    release();
    const int caller = Runtime::current_device();
    if (caller != device_ && !Runtime::make_current(device_)) return false;
    data_ = static_cast<float*>(Runtime::allocate(floats * static_cast<int64_t>(sizeof(float))));
    if (caller != device_) (void)Runtime::make_current(caller);
    if (data_ == nullptr) return false;
    capacity_ = floats;
    return true;
  }
  void release() {
    complete_ = false;
    if (data_ != nullptr) Runtime::release(data_);
    data_ = nullptr;
    capacity_ = 0;
  }

  float* data() const { return data_; }
  int64_t capacity() const { return capacity_; }  // floats
  int64_t bytes() const { return capacity_ * static_cast<int64_t>(sizeof(float)); }

 private:
  int device_ = 0;
  float* data_ = nullptr;
  int64_t capacity_ = 0;
  bool complete_ = false;
};

}  // namespace rf
