// Rows of a result whose place is the scalar offset of a buffer access, the lanes having their column in the vector offset.
#pragma once

#if defined(__HIPCC__)
#define ONHIP_BOTH __host__ __device__
#else
#define ONHIP_BOTH
#endif

namespace onhip {

constexpr unsigned OOB = 0x80000000u;       // vector offset outside every buffer: loads give 0, stores vanish
constexpr unsigned RSRC_RANGE = 0x80000000u; // num_records of the data buffers (all offsets stay below 2 GiB)

// `rows` rows reach less than 2 GiB; a tile's rows past the last may reach more.  A masked lane (OOB) of one of those would ask for OOB plus that, and
// from 2 GiB on the sum is no longer outside by itself: 20 channels of 4700 x 4700 are 1.8 GB, and channel 27 would be at 2.4 GB.  So nothing
// is asked for a row that no lane has; OOB and the place of a row that is there stay at 2 GiB or more, and below 4.  EDGE: the variant for tiles with rows
// past the last, the others have none.  (A branch a row in the last row tile, which also saves it those rows' accesses; the W8A32 store with a residual operand has the row in the vector offset there.  The place bounded
// by the last row's instead was a minimum and a product a row, for which the compiler kept scalars in vector registers: fp32 64 x 64 tiles
// with a residual operand 3-5 % slower.)
template <bool EDGE> ONHIP_BOTH constexpr bool row_there(int row, int rows) { return !EDGE || row < rows; }

// The other way, for the first-layer kernel's variant for large planes and the sum of slices inside a launch: a row past the last where the last is,
ONHIP_BOTH constexpr unsigned row_offset(int row, int rows, unsigned row_bytes) {
    return (unsigned) (row < rows ? row : rows - 1) * row_bytes;
}
// and a patch's row `ih` of channel c, which may lie above or below an image of h rows (its lanes are masked then), at the nearest row of the channel.
ONHIP_BOTH constexpr unsigned patch_row_offset(int c, int ih, int h, unsigned row_bytes) {
    return (unsigned) (c * h + (ih < 0 ? 0 : ih < h ? ih : h - 1)) * row_bytes;
}
// A first-layer convolution that needs it: three channels of h x w, patch rows from -pad_t to last_ih (the padding may be of any height: with 20000 rows of it
// under 10 rows of 30000 pixels, row 17900 is 2 GiB and 500 KB away), a tile of `rows` output channels of `plane` pixels.  Otherwise OOB plus a masked row's
// place, and OOB less that of a row above the image, are outside by themselves.
ONHIP_BOTH constexpr bool far_rows(long long h, long long w, long long pad_t, long long last_ih, long long rows, long long plane) {
    return (3 * h + pad_t) * w * 4 > 1LL << 31 || (2 * h + last_ih) * w * 4 >= 1LL << 31 || rows * plane * 4 >= 1LL << 31;
}

}  // namespace onhip
