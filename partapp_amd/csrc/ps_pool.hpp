// Device memory kept between calls.
//
// The reference-shaped calls plan, run and forget: one message, one image, one
// set of local maxima.  Allocating and freeing their memory took longer than
// their kernels (a 24 x 41 x 57 message: 30 of 80 us; a 48 x 300 x 300 image,
// 258 MB of scratch: 0.5 of 3.8 ms), so freed blocks stay with the library, up
// to kPoolBytes and kPoolBlocks per device, and are handed out again where they fit;
// beyond the bound the longest unused go back to the device, and all of them
// when an allocation fails or ps_release_memory is called.
//
// A block returned here must have no work pending on it: the callers have
// waited for their stream (the synchronous calls) or the device (plans).
#pragma once

#include <hip/hip_runtime.h>

#include <cstddef>

namespace ps {

constexpr size_t kPoolBytes = 1ull << 30;  // 0.35 % of a 288 GB device
constexpr size_t kPoolBlocks = 64;

// at least `bytes` on the current device, 256-byte aligned; contents undefined
hipError_t pool_get(void **p, size_t bytes);
template <class T>
hipError_t pool_get(T **p, size_t bytes) {
  return pool_get(reinterpret_cast<void **>(p), bytes);
}
// give a block back (null: nothing); idle: no work on it is pending, else it
// is freed, which waits for the device
void pool_put(void *p, bool idle);
// A word of pinned host memory that kernels write and the caller reads once its
// stream has ended (a word copied back costs a call some 10 us, one allocated for
// it far more); at most kPoolWords are kept.
constexpr size_t kPoolWords = 16;
hipError_t pool_get_host(unsigned **p);
void pool_put_host(unsigned *p, bool idle);
// free the cached blocks of the current device, and the words
hipError_t pool_trim();

}  // namespace ps
