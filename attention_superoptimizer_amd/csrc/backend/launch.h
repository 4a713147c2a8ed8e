// Kernel launches that can be recorded instead of made.  Everything a customized operator enqueues
// goes through launch_kernel(); while a recorder is installed on the calling thread the launch is
// noted there -- function, grid, LDS, a copy of the arguments -- and nothing is enqueued.  The list
// is what mi355_prepared_run and the timed loop of mi355_customized_profile repeat: plan matching,
// the choice of a kernel and the parameter block cost the host 2.4 - 3.9 us a launch, repeating
// a recorded launch costs the launch call.
#pragma once

#include <hip/hip_runtime.h>

#include <cstring>
#include <memory>
#include <vector>

namespace mi355 {

struct RecordedLaunch {
  void const *fn;
  dim3 grid, block;
  unsigned lds;
  std::unique_ptr<unsigned char[]> bytes;  // the arguments, each 16-byte aligned
  std::vector<void *> args;
};
struct LaunchList {
  std::vector<RecordedLaunch> launches;
};
inline LaunchList *&launch_recorder() {
  static thread_local LaunchList *recorder = nullptr;
  return recorder;
}

inline void record_launch(LaunchList &list, void const *fn, dim3 grid, dim3 block, unsigned lds, void *const *args,
                          size_t const *sizes, int n) {
  RecordedLaunch r{fn, grid, block, lds, nullptr, {}};
  size_t total = 0;
  for (int i = 0; i < n; i++) {
    total += (sizes[i] + 15) / 16 * 16;
  }
  r.bytes.reset(new unsigned char[total + 16]);
  unsigned char *p = r.bytes.get();
  p += (16 - reinterpret_cast<uintptr_t>(p) % 16) % 16;
  for (int i = 0; i < n; i++) {
    std::memcpy(p, args[i], sizes[i]);
    r.args.push_back(p);
    p += (sizes[i] + 15) / 16 * 16;
  }
  list.launches.push_back(std::move(r));
}

template <typename T>
struct LaunchArg {
  using type = T;
};
template <typename... P>
hipError_t launch_kernel(void (*fn)(P...), dim3 grid, dim3 block, unsigned lds, hipStream_t stream,
                         typename LaunchArg<P>::type... args) {
  void *pointers[] = {const_cast<void *>(static_cast<void const *>(&args))...};
  if (LaunchList *list = launch_recorder()) {
    size_t const sizes[] = {sizeof(P)...};
    record_launch(*list, reinterpret_cast<void const *>(fn), grid, block, lds, pointers, sizes, (int)sizeof...(P));
    return hipSuccess;
  }
  return hipLaunchKernel(reinterpret_cast<void const *>(fn), grid, block, pointers, lds, stream);
}

}  // namespace mi355
