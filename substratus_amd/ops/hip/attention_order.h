// The order in which workgroups of decode attention take sequences.
#pragma once

#include "common.h"

constexpr int ORDERED = WAVE;     // sequences that are put in order, at most
constexpr int MOST = 65535;       // that a grid's second side takes
constexpr int LONG = 960;         // keys from which their order matters

// A lane's sequence's length, of bsz sequences, at most ORDERED (the last one's in
// lanes past it).
DEV_INLINE int length_at_lane(const int* lens, int bsz) {
  return lens[min((int)threadIdx.x % WAVE, bsz - 1)];
}

// Lengths in 256ths of the keys that a table has room for.
DEV_INLINE int coarse(int n, int room) {
  return min(n >> max(24 - __clz(max(room, 1)), 0), 255);
}

// Whether putting sequences of these lengths in order pays: some are unlike others,
// and the longest is long. (Finding a sequence takes half a microsecond, a thousand
// keys ten.)
DEV_INLINE bool unlike_lengths(int n, int room) {
  const int key = coarse(n, room);
  return __ballot(n > LONG) &&
         __ballot(key != __builtin_amdgcn_readfirstlane(key));
}

// The sequence that is r-th by length, longest first, 0 <= r < bsz; equal ones as
// they come. For all lanes of a wave. Bit by bit: those that have it are the longer
// ones of what is left.
DEV_INLINE int sequence_at(int n, int bsz, int room, int r) {
  const int lane = threadIdx.x % WAVE, key = coarse(n, room);
  unsigned long long left = __ballot(lane < bsz);
  #pragma unroll
  for (int bit = 7; bit >= 0; --bit) {
    const unsigned long long with = left & __ballot(key >> bit & 1);
    const int many = __popcll(with);
    left = r < many ? with : left & ~with;
    if (r >= many) r -= many;
  }
  const int before = __builtin_amdgcn_mbcnt_hi(
      (unsigned)(left >> 32),
      __builtin_amdgcn_mbcnt_lo((unsigned)left, 0));
  return __ffsll(__ballot((left >> lane & 1) && before == r)) - 1;
}

// What a workgroup has where a sequence's heads come first, then its shares, then
// other sequences.
struct Turn {
  int head, sequence, split;
};
DEV_INLINE Turn turn_of(int heads, int nsplit) {
  const int id = blockIdx.x + gridDim.x * (blockIdx.y + gridDim.y * blockIdx.z);
  return {id % heads, id / (heads * nsplit), id / heads % nsplit};
}

// Whether workgroups look at the lengths: where not all of them fit the chip at once,
// so that those of long sequences may be the last ones, and take long. Of up to 64
// sequences a look is one load, of 256 four and their wait: at 100 keys in a table
// of 4096, 256 x 12 x 64, 12.4 us without, 16.9 with (20.2 where they are put in
// order whatever their lengths).
inline bool orders_sequences(int bsz, int max_blocks, int nsplit,
                             long workgroups, int per_cu) {
  return bsz > 1 && bsz <= ORDERED && max_blocks >= 60L * nsplit &&
         workgroups > 256L * per_cu;
}
