// Device buffers that grow to the largest size asked for.  Host code without
// HIP, so that a program with an allocator of its own can run it.
#pragma once
#include <cstddef>

struct Work {
  void* p = nullptr;
  size_t bytes = 0;
};

// w with at least `bytes`.  When it has to grow: moving() (0, or the code to
// give up with) while the old buffer still stands, release(old), then
// alloc(&p, bytes) (0 or an error code).  The old one goes first, as both may
// not fit.  A failed allocation leaves w empty: no later call takes the freed
// address for a large enough buffer or frees it again.
template <class Moving, class Alloc, class Release>
int work_grow(Work& w, size_t bytes, Moving&& moving, Alloc&& alloc, Release&& release)
{
  if (w.bytes >= bytes) return 0;
  if (const int r = moving()) return r;
  void* old = w.p;
  w = Work{};
  if (old) release(old);
  void* p = nullptr;
  if (const int r = alloc(&p, bytes)) return r;
  w.p = p;
  w.bytes = bytes;
  return 0;
}
