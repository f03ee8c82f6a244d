// Where a row of a result lies, as the scalar offset of a buffer access whose lanes have their column in the vector offset.
#pragma once

#if defined(__HIPCC__)
#define ONHIP_BOTH __host__ __device__
#else
#define ONHIP_BOTH
#endif

namespace onhip {

constexpr unsigned OOB = 0x80000000u;       // vector offset outside every buffer: loads give 0, stores vanish
constexpr unsigned RSRC_RANGE = 0x80000000u; // num_records of the data buffers (all offsets stay below 2 GiB)

// `rows` rows reach less than 2 GiB; a tile's rows past the last may reach more.  Their lanes are masked (OOB), but the range check adds the scalar
// offset to OOB, and from 2 GiB on that sum is no longer outside by itself: 20 channels of 4700 x 4700 are 1.8 GB, and channel 27 would be at
// 2.4 GB.  So a masked row is asked for where the last row is: OOB and anything below 2 GiB stay at 2 GiB or more, and below 4.
ONHIP_BOTH constexpr unsigned row_offset(int row, int rows, unsigned row_bytes) {
    return (unsigned) (row < rows ? row : rows - 1) * row_bytes;
}

// The same for a patch's row `ih` of channel c, which may lie above or below an image of h rows (its lanes are masked then, and the padding may be of any
// height): the nearest row of the channel, below the image's size.  (3 x 10 x 30000 with 20000 rows of padding below: row 17900 was asked for at 2 GiB and
// 500 KB, which is byte 500000 of the image if the sum with OOB wraps; so was a row above an image of nearly 2 GiB.)
ONHIP_BOTH constexpr unsigned patch_row_offset(int c, int ih, int h, unsigned row_bytes) {
    return (unsigned) (c * h + (ih < 0 ? 0 : ih < h ? ih : h - 1)) * row_bytes;
}

}  // namespace onhip
