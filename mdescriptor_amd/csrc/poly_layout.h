// Where the radial functions of the polynomial basis stand in a run's scratch:
// a slice of consecutive centres, the same number of doubles for each, in one
// of two forms.  Shared by the reservation (run_soap), the kernel that writes
// them (k_poly_radial) and the two that read them; plain C++, so that the
// extents can be checked on the host.
#pragma once

#include <cstdint>

#ifdef __HIPCC__
#define MDX_LAYOUT __host__ __device__
#else
#define MDX_LAYOUT
#endif

namespace mdx {

struct PolyLayout {
    // step groups of a centre as the register-coefficient kernel reads them:
    // every species' rows padded to whole groups of poly_group_slots slots,
    // 64 values per degree and group; 0: by row, L n values per pair row
    int64_t groups = 0;
    int64_t centre = 0; // doubles a centre
};

// slots of a step group (radial_groups: 1 or 2)
MDX_LAYOUT constexpr int poly_group_slots(int radial_groups) { return radial_groups == 2 ? 8 : 16; }

// row_bound: no centre has more rows.  It is the graph's bound and not the
// stride of its row slots, which is wider once the rows have been counted.
inline PolyLayout poly_layout(int64_t row_bound, int species, int degrees, int channels, bool step_groups) {
    const int64_t rows = row_bound > 1 ? row_bound : 1;
    PolyLayout layout;
    if (step_groups) {
        // (a species' last group may be short: one more each)
        layout.groups = rows / poly_group_slots((channels + 3) / 4) + species;
        layout.centre = layout.groups * degrees * 64;
    } else {
        layout.centre = rows * degrees * channels;
    }
    return layout;
}

// first value of a by-row pair row (the row's index among its centre's) of
// the slice that starts at centre `first`
MDX_LAYOUT inline int64_t poly_row(int64_t centre_doubles, int64_t centre, int64_t first, int64_t row, int row_values) {
    return (centre - first) * centre_doubles + row * row_values;
}

// first value of a step group of the slice that starts at centre `first`;
// group_values: 64 per degree
MDX_LAYOUT inline int64_t poly_group(int64_t groups, int64_t centre, int64_t first, int64_t group, int group_values) {
    return ((centre - first) * groups + group) * group_values;
}

} // namespace mdx
