// The order in which workgroups of decode attention take sequences.
#pragma once

#include "common.h"

constexpr int ORDERED = 256;      // sequences that are put in order, at most
constexpr int MOST = 65535;       // that a grid's last side takes

// The sequence that is r-th by length, longest first, lengths counted in 256ths of
// the keys that a table has room for; equal ones as they come. For all lanes of a
// wave; bsz sequences, at most ORDERED, 0 <= r < bsz. Bit by bit: those that have
// it are the longer ones of what is left.
DEV_INLINE int sequence_at(const int* lens, int bsz, int room, int r) {
  constexpr int PER = ORDERED / WAVE;
  const int lane = threadIdx.x % WAVE;
  const int shift = max(24 - __clz(max(room, 1)), 0);
  int key[PER];
  unsigned long long left[PER];
  #pragma unroll
  for (int i = 0; i < PER; ++i) {
    key[i] = 0;
    left[i] = 0;
    if (i * WAVE < bsz) {
      key[i] = min(lens[min(i * WAVE + lane, bsz - 1)] >> shift, 255);
      left[i] = __ballot(i * WAVE + lane < bsz);
    }
  }
  #pragma unroll
  for (int bit = 7; bit >= 0; --bit) {
    unsigned long long with[PER];
    int many = 0;
    #pragma unroll
    for (int i = 0; i < PER; ++i) {
      with[i] = 0;
      if (i * WAVE < bsz) {
        with[i] = left[i] & __ballot(key[i] >> bit & 1);
        many += __popcll(with[i]);
      }
    }
    const bool longer = r < many;
    if (!longer) r -= many;
    #pragma unroll
    for (int i = 0; i < PER; ++i)
      left[i] = longer ? with[i] : left[i] & ~with[i];
  }
  int at = 0;
  #pragma unroll
  for (int i = 0; i < PER; ++i) {
    const int many = __popcll(left[i]);
    if (r >= 0 && r < many) {
      const int before = __builtin_amdgcn_mbcnt_hi(
          (unsigned)(left[i] >> 32),
          __builtin_amdgcn_mbcnt_lo((unsigned)left[i], 0));
      at = i * WAVE - 1 + __ffsll(__ballot((left[i] >> lane & 1) &&
                                           before == r));
    }
    r -= many;
  }
  return __builtin_amdgcn_readfirstlane(at);
}

// Whether they are put in order: where not all workgroups fit the chip at once, so
// that those of long sequences may be the last ones, and take long. Finding its
// sequence costs a workgroup half a microsecond, a share of a thousand keys ten.
inline bool orders_sequences(int bsz, int max_blocks, int nsplit,
                             long workgroups, int per_cu) {
  return bsz > 1 && bsz <= ORDERED && max_blocks >= 60L * nsplit &&
         workgroups > 256L * per_cu;
}
