// -----------------------------------------------------------------------------
// An element's place in its block, carried along a stride (plain C++: the host
// tests compile it too).
// -----------------------------------------------------------------------------
#ifndef SUNAMD_BLOCK_PLACE_H
#define SUNAMD_BLOCK_PLACE_H

// The place `by` further in blocks of mm elements; at < mm, by < mm.  at + by is
// formed only where it stays below mm, so U need only hold mm itself: for
// mm close to U's range (m = 65280 .. 65535 in 32 bits) at + by would wrap.
template <typename U>
constexpr U block_place_after(U at, U by, U mm)
{
  return (at >= mm - by) ? at - (mm - by) : at + by;
}

#endif
