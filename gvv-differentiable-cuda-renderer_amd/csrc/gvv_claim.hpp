// gvv_claim.hpp -- which corners of a tile's faces are summed into which, in the backward's slot flush.
// Host- and device-callable so that it can be checked on the CPU.
//
// Every corner c (3 slot + corner of the face) stores its own number into its vertex's entry of a
// claim table; after a barrier a corner whose entry holds another corner of the same vertex adds its
// terms to that one.  Corners of one vertex, and of vertices that share an entry, store to one address
// at once, so the entry is a single 32-bit word: whichever corner's store stays, the word is that
// corner's number, and its vertex is looked up in `vid`.  (An entry of two words, vertex and corner,
// would rely on both words staying from one lane, which nothing promises.)  The corner in an entry is
// in the entry of its own vertex, so it adds to no other and its `vid` is never cleared.
#pragma once
#include "gvv_math.hpp"

namespace gvv {

typedef int ClaimEntry;

GVV_HD ClaimEntry claim_entry(int corner) { return corner; }

// The corner that takes the terms of corner c: c itself if no other corner of its vertex holds the entry.
GVV_HD int claim_target(ClaimEntry e, const int* vid, int c) { return vid[e] == vid[c] ? e : c; }

}  // namespace gvv
