// transfer_way.hpp -- how a state moves between the caller's array of doubles
// and the device.  Host arithmetic only.
#pragma once
#include <cstddef>

namespace bats {

enum TransferWay {
  ONE_COPY,   // every variable in one copy
  EACH_COPY,  // a blocking copy per variable
  SLOTS       // through pinned slots, one per host thread
};

// in: to the device; written: the host array was just written by the calling
// thread (a state of the caller's order turned into the library's).
//
// Small states want few calls.  Large ones go through pinned slots: one thread
// moves 10 to 17 GB/s of pageable memory, eight reach 40 to 50, the link's own
// rate (57); a 1000-block 16^3 state takes 9.0 -> 6.7 ms up and 24 -> 7 ms
// down, in FP32 (262 MB on the host) 11 -> 3.6 and 24 -> 4.8.  Below 8 MiB (FP32
// down, where half the bytes cross the link, and arrays just written: 16)
// starting the threads costs more than they save, and out of the writing
// thread's caches FP64 is ahead without them (256 blocks 19.3 ms, 20.3 with
// slots).  Below that one copy is best on the way up (16 blocks 134 us, 202 in
// eight), and on the way down, where the pages of fresh memory are made while
// it runs, up to 2 MiB (6 blocks 112 us, 153 in eight; 24 blocks 454 and 380).
inline TransferWay transfer_way(size_t nReal, int elemSize, bool in,
                                bool written) {
  const size_t host = 8 * nReal, dev = elemSize * nReal;
  const size_t MiB = (size_t)1 << 20;
  const bool half = elemSize == 4;
  if (!(in && written && !half) &&
      host >= ((in ? written : half) ? 16 * MiB : 8 * MiB))
    return SLOTS;
  if (in ? host < 8 * MiB : dev <= 2 * MiB) return ONE_COPY;
  return EACH_COPY;
}

}  // namespace bats
