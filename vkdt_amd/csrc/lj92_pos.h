// lj92_pos.h -- bit positions of the many-lanes lossless-JPEG decode
// (k_lj92.hip), apart so that they can be tested on the CPU.
#pragma once
#include <stdint.h>

#if defined(__HIP__)
#define LJ92_HD __host__ __device__
#else
#define LJ92_HD
#endif

// the position after a symbol of n bits at pos, in a stream of B bits.  A scan
// continues past its data on zeros, with no end but its last sample: every
// position there reads alike, so it stays there and does not wrap round into
// the data after 2^32 bits
LJ92_HD static inline uint32_t lj92_next(uint32_t pos, uint32_t n, uint32_t B)
{
  const uint32_t p = pos + n, end = B + 64;
  return p < end ? p : end;
}
