// Index rules of the persistent sweep's exchange, shared by the kernel and
// the host (no device code: a host compiler checks them too).
#pragma once

namespace iff {

// The array row that the strip loads of tile row j (a tile reaches past the
// domain on every side) address in a field of ny rows.  Lanes that take
// nothing are dropped by the buffer's bounds check, which compares their
// offset with the records left behind the row's start: the row has to lie in
// the field for that difference to be one.
constexpr int strip_row(int j, int ny) { return j < 0 ? 0 : j < ny ? j : ny - 1; }

}  // namespace iff
