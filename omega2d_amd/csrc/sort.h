// sort.h - stable orders of 32-bit keys made on the device (sort.hip).
#pragma once

#include "o2d_runtime.h"

namespace o2d {

enum KeyKind { kMorton32, kMorton16, kNode };

// where the keys come from: points x, y on their own box (bbox) or on the box given by x0, y0
// and inv (Morton), or panel ends idx with the indices clamped to nnodes - 1 (kNode)
struct KeyGen {
  int kind;
  bool bbox;
  const double* x;
  const double* y;
  double x0, y0, inv;
  const uint32_t* idx;
  uint32_t nnodes;
};

// order_out (n entries) = 0..n-1 in the stable order of the keys' low `bits` bits (no higher bit
// is set); keys_out (n entries of scratch) holds the sorted keys when want_keys. The temporaries
// are the kKeysA, kOrderA, kBBox, kSortTab and kSortTemp slots, or pieces of *ws.
int sort_order(Device* d, hipStream_t s, Workspace* ws, int64_t n, const KeyGen& g, int bits,
               uint32_t* keys_out, uint32_t* order_out, bool want_keys);

}  // namespace o2d
