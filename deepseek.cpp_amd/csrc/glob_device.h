// glob_device.h -- what the compiler cannot know of a pointer.
#pragma once
// A pointer that a kernel reads out of memory (a descriptor's) has no address space, and what it points at is then accessed by flat instructions: they
// count for the LDS waits as well as for the memory waits, out of order, so that every wait behind one is a wait for everything on its way.
// The value as an integer, taken as a pointer to global memory, tells the compiler what it is.
template <typename T>
__device__ __forceinline__ T* glob(T* p) {
  typedef __attribute__((address_space(1))) T* global;
  return (T*)(global)(unsigned long long)p;
}
