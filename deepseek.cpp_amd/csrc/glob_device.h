// glob_device.h -- what the compiler cannot know of a pointer.
#pragma once
// A pointer that a kernel reads out of memory (a descriptor's) has no address space, and what it points at is then accessed by flat instructions: they
// count for the LDS waits as well as for the memory waits, out of order, so that every wait behind one is a wait for everything on its way.
// The value as an integer, taken as a pointer to global memory, tells the compiler what it is.  Both in turn on one card, us a token: 27 small layers
// 2084 -> 2064, V3's shapes (5 blocks) 494.6 -> 491.6, with a latent cache 606.5 -> 603.8; V2-Lite's, Q2_K 1434 -> 1431, F8E5M2 1582 -> 1589.
template <typename T>
__device__ __forceinline__ T* glob(T* p) {
  typedef __attribute__((address_space(1))) T* global;
  return (T*)(global)(unsigned long long)p;
}
