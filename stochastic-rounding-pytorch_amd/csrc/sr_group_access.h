// sr_group_access.h -- global loads and stores of elements and element groups.
//
// Used by the kernels, and plain C++ otherwise (for clang, whose vector types
// and non-temporal builtins it needs), so the accesses can be run on a host.
//
// Table entries are plain integers, so pointers are cast to the global
// address space explicitly; otherwise every access would be a flat access.
#pragma once

#include <cstdint>

#if defined(__HIPCC__)
#define SR_DEVICE_INLINE __device__ __forceinline__
#else
#define SR_DEVICE_INLINE inline
#endif
#if defined(__HIP_DEVICE_COMPILE__)
#define SR_GLOBAL __attribute__((address_space(1)))
#else
#define SR_GLOBAL
#endif

namespace sr {

template <class T>
SR_DEVICE_INLINE const SR_GLOBAL T* gptr(const void* p) {
  return (const SR_GLOBAL T*)(p);
}
template <class T>
SR_DEVICE_INLINE SR_GLOBAL T* gptr_mut(void* p) {
  return (SR_GLOBAL T*)(p);
}

// Streaming accesses.  Every operand is read once and written at most once
// per launch, so every global load and store carries the non-temporal hint.
// Measured on MI355X: north star 5.64 -> 6.13 TB/s, SGDM 5.87 -> 6.41 TB/s;
// the hint on loads alone is slower (5.51) and on stores alone neutral.
// For element types only: T's natural alignment is assumed, since a type that
// passes through a template argument loses its `aligned` attribute.
template <class T>
SR_DEVICE_INLINE T stream_load(const void* p) {
  return __builtin_nontemporal_load(gptr<T>(p));
}
template <class T>
SR_DEVICE_INLINE void stream_store(void* p, T v) {
  __builtin_nontemporal_store(v, gptr_mut<T>(p));
}

// The words of one group of four elements, moved as one access.  The types
// promise the alignment of one element only, so groups of views that start
// anywhere move the same way: gfx950's global accesses take any alignment,
// and an access that is aligned costs what a declared alignment would.  Each
// access below names its type directly, never as a template argument, which
// would give it the vector's own alignment back.
typedef uint32_t group16 __attribute__((ext_vector_type(4), aligned(4)));
typedef uint32_t group8 __attribute__((ext_vector_type(2), aligned(2)));
typedef uint32_t group4 __attribute__((aligned(1)));

// kCached keeps the load under the normal cache policy (the small casts'
// input).
template <int BYTES, bool kCached = false>
SR_DEVICE_INLINE void load_words(const char* ptr, uint32_t* w) {
  if constexpr (BYTES == 16) {
    const SR_GLOBAL group16* p = (const SR_GLOBAL group16*)(ptr);
    const group16 a = kCached ? *p : __builtin_nontemporal_load(p);
    __builtin_memcpy(w, &a, BYTES);
  } else if constexpr (BYTES == 8) {
    const SR_GLOBAL group8* p = (const SR_GLOBAL group8*)(ptr);
    const group8 a = kCached ? *p : __builtin_nontemporal_load(p);
    __builtin_memcpy(w, &a, BYTES);
  } else {
    static_assert(BYTES == 4, "a group is 4, 8 or 16 bytes");
    const SR_GLOBAL group4* p = (const SR_GLOBAL group4*)(ptr);
    const group4 a = kCached ? *p : __builtin_nontemporal_load(p);
    __builtin_memcpy(w, &a, BYTES);
  }
}

template <int BYTES>
SR_DEVICE_INLINE void store_words(char* ptr, const uint32_t* w) {
  if constexpr (BYTES == 16) {
    group16 a;
    __builtin_memcpy(&a, w, BYTES);
    __builtin_nontemporal_store(a, (SR_GLOBAL group16*)(ptr));
  } else if constexpr (BYTES == 8) {
    group8 a;
    __builtin_memcpy(&a, w, BYTES);
    __builtin_nontemporal_store(a, (SR_GLOBAL group8*)(ptr));
  } else {
    static_assert(BYTES == 4, "a group is 4, 8 or 16 bytes");
    group4 a;
    __builtin_memcpy(&a, w, BYTES);
    __builtin_nontemporal_store(a, (SR_GLOBAL group4*)(ptr));
  }
}

}  // namespace sr
