// What a launch asks the runtime about a kernel, remembered per (kernel, device): whether its dynamic LDS limit
// has been raised and how many of its workgroups can be resident at once.  Both depend on the code object and
// the device alone, so a launch looks them up instead of asking again (the occupancy query and the attribute
// call cost about 2 us of the 4.6 us that a single-pass entry point takes on the host).
#pragma once
#include <hip/hip_runtime.h>

#include <atomic>
#include <cstdint>

namespace launch_facts {

// A fixed open-addressing table without locks.  A slot is claimed by its kernel's address and then holds one
// value per device; a full table or a device past the last only means that the runtime is asked every time.
constexpr int kSlots = 256, kDevices = 16;
struct Slot {
  std::atomic<const void*> kernel{nullptr};
  std::atomic<int> smem[kDevices];      // bytes of dynamic LDS the kernel may use (0: the default)
  std::atomic<int> resident[kDevices];  // resident workgroups (0: not asked yet)
};
inline Slot* slot_of(const void* kernel) {
  static Slot table[kSlots];
  const uintptr_t key = reinterpret_cast<uintptr_t>(kernel) >> 4;
  for (int i = 0; i < kSlots; ++i) {
    Slot& s = table[(key + i) % kSlots];
    const void* seen = s.kernel.load(std::memory_order_acquire);
    if (seen == kernel) return &s;
    if (!seen) {
      if (s.kernel.compare_exchange_strong(seen, kernel, std::memory_order_acq_rel) || seen == kernel) return &s;
    }
  }
  return nullptr;
}
inline int current_device() {
  int dev = -1;
  return hipGetDevice(&dev) == hipSuccess ? dev : -1;
}

// Raises the kernel's dynamic LDS limit on the current device to at least `bytes`.
inline bool smem(const void* kernel, int bytes) {
  const int dev = current_device();
  Slot* s = dev >= 0 && dev < kDevices ? slot_of(kernel) : nullptr;
  if (s && s->smem[dev].load(std::memory_order_acquire) >= bytes) return true;
  if (hipFuncSetAttribute(kernel, hipFuncAttributeMaxDynamicSharedMemorySize, bytes) != hipSuccess) return false;
  if (s) s->smem[dev].store(bytes, std::memory_order_release);
  return true;
}

// Workgroups of the kernel that can be resident at once on the current device, at most max_per_cu on each
// compute unit.  A kernel is always asked about with the same threads, LDS and cap.
inline int resident(const void* kernel, int threads, int lds, int max_per_cu) {
  const int dev = current_device();
  if (dev < 0) return 256;
  Slot* s = dev < kDevices ? slot_of(kernel) : nullptr;
  if (s) {
    const int known = s->resident[dev].load(std::memory_order_acquire);
    if (known > 0) return known;
  }
  int ncu = 0, per_cu = 0;
  bool answered = true;
  if (hipDeviceGetAttribute(&ncu, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess) ncu = 256, answered = false;
  if (hipOccupancyMaxActiveBlocksPerMultiprocessor(&per_cu, kernel, threads, lds) != hipSuccess || per_cu < 1)
    per_cu = 1, answered = false;
  if (per_cu > max_per_cu) per_cu = max_per_cu;
  if (s && answered) s->resident[dev].store(ncu * per_cu, std::memory_order_release);
  return ncu * per_cu;
}

}  // namespace launch_facts
