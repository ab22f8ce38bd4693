// result_ring.h -- the result entry of each request in flight on a server's
// slot (host code).
//
// A slot has kDepth entries, and a request's epilogue writes the request's
// serial into the entry serial % kDepth.  At most kDepth requests are in flight
// on a slot, in serial order, so while their serials are consecutive no two
// share an entry.  A request that failed before it got to the slot must take
// none: the serials on either side of it would share one, and the later
// epilogue would hide the earlier one's.
#pragma once

#include <cstdint>

namespace lbvh {

template <uint32_t kDepth>
class ResultRing {
 public:
  static int entry(uint32_t serial) { return (int)(serial % kDepth); }

  // Admits a request: prepare() returns 0, and then it takes the next serial,
  // or a status that is returned, and it takes none.
  template <class Prepare>
  int admit(uint32_t *serial, Prepare prepare) {
    const int st = prepare();
    if (st == 0) *serial = next_++;
    return st;
  }

 private:
  uint32_t next_ = 1;  // 0 is in an entry that nothing has written
};

}  // namespace lbvh
