// dev_cache.hpp -- device memory kept between runs.
//
// A run takes tens of gigabytes (eigensystems and work space of a chunk) and
// gives them back at its end.  Freed device memory has to be cleared before it
// is handed out again, at about 35 GB/s once the cleared memory is used up:
// the 29 GB of a 330-frame run of N = 2048 then took 590 ms beside 265 ms of
// work.  Blocks given back are therefore kept for the next run:
//   - at most an eighth of the device's memory, the oldest block freed first,
//     and only while a quarter of it is free for others;
//   - for at most kCacheIdleSeconds without use, after which a thread frees
//     them; all at once when an allocation of a context does not fit, whichever
//     way it is made (DevBuf), at both ends of cir_run_many, whose jobs take
//     pooled memory instead, and by cir_release_memory();
//   - a block is given back only after the stream that used it is through, so
//     any thread and stream may take it.
#pragma once

#include <cstddef>

namespace cir {

constexpr int kCacheIdleSeconds = 30;

// n bytes on the current device (its index in *dev), from a kept block of at
// most a quarter more (its size in *cap) or a new one.  A HIP error code.
int dev_cache_alloc(void** p, size_t n, size_t* cap, int* dev);
// Keeps the block, which no queued work uses any more, or frees it.
void dev_cache_free(void* p, size_t cap, int dev);
// Frees what is kept on the current device.
void dev_cache_release();
// Kept bytes on the current device (free memory that hipMemGetInfo counts as used).
size_t dev_cache_bytes();

}  // namespace cir
