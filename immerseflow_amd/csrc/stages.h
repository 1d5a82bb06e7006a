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

// The strip buffer of stage g.  Stages are counted over launches in 32 bits,
// and 2^32 is no multiple of 3: behind a wrap two stages in a row would share a
// buffer, so the counters are zeroed before one (StageCount).
constexpr int kStripBufs = 3;
constexpr unsigned strip_of(unsigned g) { return g % (unsigned)kStripBufs; }

// Stages that the tiles' counters can have counted since they were zeroed.
struct StageCount {
    unsigned long long used = 0;
    // before launches of at most `most` stages: do the counters have to be
    // zeroed (with the strips) so that they do not wrap?
    bool wraps(unsigned long long most)
    {
        const bool w = used + most > 0xffffffffull;
        used = (w ? 0 : used) + most;
        return w;
    }
};

}  // namespace iff
