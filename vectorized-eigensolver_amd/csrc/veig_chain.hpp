// The wavefront of a workgroup that runs the bulge chain (veig_stream.hpp), from
// what the wavefronts have noted of their places: plain functions, for the
// kernels and for a host build.
#pragma once

#if defined(__HIPCC__)
#include <hip/hip_runtime.h>
#define VEIG_CHAIN_HD __host__ __device__ __forceinline__
#else
#define VEIG_CHAIN_HD inline
#endif

namespace veig {

// What wavefront `wave` notes: its SIMD, and, the first one alone, the
// workgroup's place in the CU's LDS.  hw_id, lds_alloc: its hardware registers.
// They say where the wavefront is while it reads them, not where the workgroup
// is for good: after a preemption it may be restored elsewhere.  So each value
// that the choice depends on is read by one wavefront and shared.
VEIG_CHAIN_HD int chain_note(int wave, unsigned hw_id, unsigned lds_alloc) {
  const unsigned base = lds_alloc & 0xfffu, size = (lds_alloc >> 12) & 0xfffu;
  return (int)((hw_id >> 4) & 3u) | (wave == 0 && size ? (int)(base / size) << 2 : 0);
}

// Of the workgroups that share a CU each should have its chain on another SIMD:
// two chains on one SIMD take nearly twice as long.  Four workgroups of three
// wavefronts, three to a SIMD, leave each SIMD out once, and a workgroup that
// takes an ended one's place takes its SIMDs: the SIMD after the one left out is
// another one in each.  Wider workgroups have a wavefront on every SIMD: there
// the workgroup's place in the CU's LDS numbers it among its neighbours.
// notes: one per wavefront, the same ones for every caller.
VEIG_CHAIN_HD int chain_pick(const int *notes, int waves) {
  unsigned there = 0;
  for (int w = 0; w < waves; ++w) there |= 1u << (notes[w] & 3);
  unsigned want = (unsigned)notes[0] >> 2;
  if (there != 15u) {
    want = 1;  // after the lowest SIMD left out
    while (there & 1u) {
      there >>= 1;
      ++want;
    }
  }
  for (unsigned d = 0; d < 4; ++d)
    for (int w = 0; w < waves; ++w)
      if (((unsigned)notes[w] & 3u) == ((want + d) & 3u)) return w;
  return 0;
}

}  // namespace veig
