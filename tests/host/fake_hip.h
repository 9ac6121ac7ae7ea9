// A HIP runtime for host-only tests: device memory is host memory, streams do
// nothing, and a kernel launch calls a hook with the kernel's name, its grid and its
// arguments instead of running anything.  A test program that links fake_hip.cpp and the
// library runs the library's host code (schedules, arguments, allocations) without a GPU.
#pragma once
#include <cstddef>
#include <functional>
#include <string>

namespace fake {
struct Launch {
  std::string kernel;   // demangled, without "void " and the parameter list
  unsigned grid = 0, block = 0;
  void** args = nullptr;
};
extern std::function<void(const Launch&)> on_launch;
extern long mallocs_left;        // device allocations that still succeed (negative: all)
extern long pinned_left;         // pinned ones
extern long instantiates_left;   // graph instantiations
extern long capture_us, replay_us;   // what a capture, and a graph launch, takes
extern long mallocs, captures;   // calls so far
size_t live();                    // allocations not freed
size_t bytes_at(const void* p);   // bytes from p to the end of its allocation (0: not in one)
}  // namespace fake
