// Which kernel a SOAP run takes and how it is decomposed: a rule on the plan's
// shape and options, the batch's sizes and the graph's row bound.  Plain C++,
// so that the rule can be run on the host by itself.
#pragma once

#include <algorithm>
#include <cstddef>
#include <cstdint>
#include <limits>

#include "poly_layout.h"

namespace mdx {

constexpr int kItemCentres = 32; // centres of an averaged structure per run, at most
// folded partial rows (k_fold_partials)
constexpr int kFoldItems = 16;  // rows per split, at least
constexpr int kFoldSplits = 32; // splits per structure, at most
// rows of a centre that the 4x4 kernels' slot codes can hold
constexpr int64_t kSlotCodeRows = int64_t(1) << 27;
constexpr int64_t kFirstSlots = 512; // rows a centre's slots hold at first (kMinSlotCap)
// largest row (features x 8 bytes) the register-coefficient kernel's outer
// averages accumulate in LDS
constexpr int64_t kBlockOuterLdsBytes = 48 * 1024;
// atoms of a structure whose pairs that kernel streams species-major
constexpr int kBlockSmallAtoms = 64;
// pairs of a structure past which a batch of fewer structures than compute
// units sums runs of its centres instead of whole structures
constexpr int64_t kBlockSpreadPairs = 4096;
// polynomial basis: bytes of radial functions a slice of centres holds, at
// most (what the last-level cache keeps between the two kernels of a slice)
constexpr int64_t kPolySliceBytes = int64_t(256) << 20;
// ... and the fewest centres of a slice: with less room the 16x16 kernel forms
// the functions itself (as fast as slices of 128 centres on the register-
// coefficient kernel: 3,000 atoms, n 6 l 5, 1,255 us, in slices of 128, 256
// and 1,024 centres 1,221, 840 and 507; n 3 l 2, 639 and 756, 522, 325).  By
// row as many as give the device 2,048 wavefronts, one per centre and tile
// (n 4 l 1, a tile: 662 us, in slices of 512, 1,024 and 3,000 centres 1,071,
// 691 and 524; n 3 l 10, eight tiles: 5,751 us, of 256 centres 1,331)
constexpr int64_t kPolyLeastCentres = 256, kPolyLeastWaves = 2048;
constexpr size_t kPolySlack = 4096; // alignment of the scratch's parts

struct ChoiceInput {
    // the plan
    int average = 0;      // 0 off, 1 inner, 2 outer
    int radial_basis = 0; // 0 GTO, 1 polynomial
    int compression = 0;  // 0 off, 1 mu2, 2 mu1nu1, 3 crossover
    int weighted = 0;
    int S = 1, Sc = 1, n = 1, L = 1, l_max = 0; // Sc: species of the coefficients
    int64_t features = 0;
    bool use_mfma = true; // the plan fits the tile kernels
    int tiles = 1;        // 16x16 tiles of its contraction
    int quad_waves = 0;   // 0: not the 4x4-block kernel's
    int block_waves = 0, block_kg = 0, block_ncr = 0; // 0 wavefronts: not the register-coefficient kernel's
    bool block_forced = false, block_float32 = false, block_every_form = false;
    size_t block_width = 0, quad_width = 0, tile_width = 0; // doubles of an inner average's partial row
    // the batch and its graph
    int64_t structures = 0, atoms = 0, largest_structure = 0, most_images = 0, row_bound = 0;
    int64_t units = 256;  // compute units
    int64_t budget = 0;   // bytes its partial rows may take
};

// Rows a centre the rule counts with: the first slots' width while the rows
// have not been counted, and after (both entry points then decide alike).
inline int64_t planned_rows(const ChoiceInput& in) {
    return std::max(in.row_bound, std::min(kFirstSlots, (in.most_images + 15) / 16 * 16));
}

// Centres per run of an averaged structure: kItemCentres where the batch then
// still has a few runs for every compute unit, shorter for smaller batches
// (8,192 atoms at 32 are 256 runs, one workgroup a compute unit) as far as
// their partial rows (width doubles each, and the folded ones) fit the budget.
// About three runs of kItemCentres a compute unit are enough: more of them only
// add rows (200 structures of 100-160 atoms, four species n 8 l 6, 388 us with
// runs of 32, 409 with runs of 12; 500 of 70-100 419 and 472; 60 of 100-160,
// 300 runs of 32, 250 and 183 with runs of 3).
inline int64_t run_centres(const ChoiceInput& in, size_t width) {
    if ((in.atoms + in.structures * (kItemCentres / 2)) / kItemCentres >= 3 * in.units) return kItemCentres;
    const int64_t fill = 8 * in.units;
    int64_t length = std::max<int64_t>(1, std::min<int64_t>(kItemCentres, in.atoms / fill));
    auto bytes = [&](int64_t len) {
        return static_cast<double>(in.atoms / len + 33 * in.structures) * static_cast<double>(width) * sizeof(double);
    };
    while (length < kItemCentres && bytes(length) > static_cast<double>(in.budget)) length *= 2;
    return std::min<int64_t>(length, kItemCentres);
}

// The same on the tile kernels, whose finalize walks a structure's rows one
// after another: up to 2 kFoldItems as they are, else their folded splits
// (k_fold_partials).  A centre of a workgroup's run costs 25-51 us there and a
// row of the walk 11-23 (four species n 4 l 10 to three n 9 l 10 mu1nu1): the
// length whose rounds of workgroups and walk are the shortest by a tenth (more
// rows are also more traffic).  waves: of a workgroup, 8 at a time on a
// compute unit.  One structure, expansion + finalize in us, runs of 32, runs
// as short as run_centres takes them, these: three species n 8 l 10 of 1,000
// atoms 786 + 483, 135 + 529, 207 + 153, of 6,000 820 + 212, 638 + 520, 808 +
// 212; four n 4 l 10 of 12,000 901 + 252, 1,043 + 334, 897 + 248.
inline int64_t tile_run_centres(const ChoiceInput& in, size_t width, int waves) {
    // (as many structures as compute units: splitting them adds rows, 3,000
    // molecules of 2-8 atoms mu2 l 0 40 us whole and 47 in fours)
    if (in.structures >= in.units) return kItemCentres;
    const int64_t slots = in.units * std::max(1, 8 / std::max(1, waves));
    int64_t best = kItemCentres;
    double least = 0.0;
    for (int64_t length = kItemCentres; length >= 1; length /= 2) {
        // (no run is longer than the largest structure)
        const int64_t centres = std::min(length, in.largest_structure);
        const int64_t items =
            length >= in.largest_structure ? in.structures : (in.atoms + in.structures * (length - 1)) / length;
        const double bytes = static_cast<double>(items + 32 * in.structures) * static_cast<double>(width) * sizeof(double);
        if (length < kItemCentres && bytes > static_cast<double>(in.budget)) break;
        const int64_t rows = std::max<int64_t>(1, items / in.structures);
        const int64_t walk = rows <= 2 * kFoldItems ? rows : std::min<int64_t>((rows + kFoldItems - 1) / kFoldItems, kFoldSplits);
        const double cost = static_cast<double>((items + slots - 1) / slots * centres) + 0.6 * static_cast<double>(walk);
        if (length == kItemCentres || cost < 0.9 * least) {
            best = length;
            least = cost;
        }
    }
    return best;
}

// The kernel and the decomposition of a run.
struct Choice {
    bool block = false;           // the register-coefficient kernel
    bool block_inner = false;     // ... a workgroup per structure
    bool block_small = false;     // ... ... its pairs streamed species-major
    bool block_runs = false;      // ... runs of a structure's centres into partial coefficient rows
    bool block_outer = false;     // ... a float64 partial row per centre
    bool block_outer_lds = false; // ... a workgroup per structure, power spectra summed in LDS
    bool f32_exps = false;        // ... with float32 exps
    bool quad = false;            // the 4x4-block kernel
    bool poly_inside = false;     // polynomial basis: radial functions in the 16x16 kernel, without scratch
    int64_t run = kItemCentres;   // centres per run
    size_t partial_width = 0;     // doubles of a partial row
    bool partials() const { return !block_inner && !block_outer_lds; } // (of an average)
};

// Scratch a run may save: kFastest, no more of it than runs of kItemCentres
// take, none for the register-coefficient kernel's partial rows, none beside
// the other kernels' partial rows (no row weights, no radial functions).
constexpr int kFastest = 0, kLongRuns = 1, kShortRows = 2, kLeast = 3;
inline Choice choose(const ChoiceInput& in, int saving) {
    Choice c;
    const double F = static_cast<double>(in.features);
    // The register-coefficient kernel where the plan chose it and every
    // centre's rows fit their slot codes.  It forms a structure's average in
    // one workgroup when the structures are small (a wavefront of atoms) or
    // many enough to fill the device (four per compute unit); the inner
    // averages of a few large structures (16 cells of 4,096 atoms: 16
    // workgroups, 50 ms) sum runs of centres into partial coefficient rows
    // instead, reduced per structure (1.1 ms).
    const bool whole = in.largest_structure <= kBlockSmallAtoms || in.block_forced || in.structures >= 4 * in.units;
    // Outer averages with a workgroup per structure add each centre's power
    // spectrum into the structure's float64 row in LDS and write the mean
    // once, with no partial rows in HBM.  Large structures, and rows past the
    // LDS, take every centre's row as a float64 partial row (at most 4 GiB of
    // them), folded per structure, then the mean (k_finalize_outer); so do
    // fewer structures than two per compute unit, which spread over the
    // device better, where the scratch allows.
    const double centre_rows = static_cast<double>(in.atoms + 5 * in.structures) * F * 8.0;
    const bool few = in.structures < 2 * in.units && centre_rows <= static_cast<double>(in.budget);
    const bool outer_lds = in.average == 2 && whole && in.radial_basis == 0 && F * sizeof(double) <= static_cast<double>(kBlockOuterLdsBytes) &&
                           (!few || saving > kFastest);
    const bool outer_rows = static_cast<double>(in.atoms) * F * 8.0 <= 4294967296.0;
    // The power spectrum's Gram tiles are register pairs of 16 channels here,
    // padded to whole radial groups, and pairs of 16 packed channels in the
    // tile kernels; centres of few neighbours do not repay the padding.
    // 1,000 molecules of 9-29 atoms, tile kernels and here (us):
    //   three radial groups, n 10 l 7 (which also spill registers): rows of
    //     five species 835 and 996 (three: 502 and 425; condensed cells of five
    //     833 and 655), outer averages of three 694 and 826, of five 1,325 and
    //     1,439
    //   one group in two registers where one tile holds the channels (two
    //     from l 8), default options: rows of five species n 2 l 6 146 and 192,
    //     of eight n 1 l 9 0.64 of the rate (with 75-85 atoms 0.87, 115-125
    //     0.96); of eight n 4 l 6 1.19
    //   outer averages, at least twice the tile pairs, default options: five
    //     species n 5 l 9 0.63 of the rate, l 6 493 and 580, l 2 1.27 of it (of
    //     40-60 atoms 0.85; 75-85 1.5); shapes compiled in every form stay
    //   mu1nu1 outer averages past l 8 of three registers: 850 and 1,047
    const int64_t channels = static_cast<int64_t>(in.Sc) * in.n, packed = (channels + 15) / 16;
    const bool twice = in.block_ncr * (in.block_ncr + 1) >= 2 * packed * (packed + 1);
    const bool defaults = in.quad_waves > 0; // (else the tile kernel is the 16x16 one)
    const bool padded =
        in.use_mfma && !in.block_forced && in.average != 1 && in.most_images <= kBlockSmallAtoms &&
        (in.block_kg == 3 ? in.block_ncr >= (in.average == 2 ? 3 : 5)
         : defaults && in.block_kg == 1 && in.block_ncr == 2 && channels <= (in.l_max >= 8 ? 18 : 16) ? true
         : in.average == 2 && !in.block_every_form && defaults ? twice
         : in.average == 2 && in.radial_basis == 0 && in.compression == 2 ? in.l_max > 8 && in.block_ncr >= 3
                                                                       : false);
    // Rows in LDS of too few structures to fill the device, where their centre
    // rows do not fit: the tile kernels' runs of centres fill it (150
    // structures of 40-60 atoms, n 12 l 7 of two species, 475 us and 705; 30,
    // n 8 l 9 of four, 458 and 549; 300, n 12 l 7, 761 and 825)
    const bool underfilled = outer_lds && saving == kFastest && in.use_mfma && !in.block_forced && !in.block_every_form &&
                             in.structures < (in.block_kg == 3 ? 2 : 1) * in.units;
    const bool scratch_rows = in.weighted != 0 || in.radial_basis == 1;
    c.block = in.block_waves > 0 && (in.average != 2 || outer_rows || outer_lds) && !padded && !underfilled && in.row_bound < kSlotCodeRows &&
              !(saving == kLeast && scratch_rows && in.use_mfma && !in.block_forced);
    // By row the radial functions come a species at a time, padded to tiles of
    // 16 rows; the 16x16 kernel forms those of 32 rows at once.  It is the
    // faster of the two for up to eight degrees and channels (past them it
    // meets a barrier every four grid points: from memory 2.6-6 times as
    // fast) with more than six species, or three to six that do not fill two
    // tiles each.  l 1, n 4, from memory and inside: 4,000 condensed atoms of
    // two, four, six, ten species 604 and 830 us, 674 and 825, 822 and 870, 953
    // and 922; 2,000 molecules of 9-29 atoms of two, three, six species 753 and
    // 958, 1,313 and 1,067, 1,709 and 1,384; l 2 n 6, 4,000 atoms of nine 1,276
    // and 1,024.
    const bool short_tiles = in.S > 6 || (in.S > 2 && std::min(in.most_images, planned_rows(in)) < 32 * in.S);
    c.poly_inside = in.radial_basis == 1 && !c.block && (saving == kLeast || (in.L <= 8 && in.n <= 8 && short_tiles));
    const size_t block_width = c.block ? in.block_width : 0;
    // A few small periodic structures hold thousands of pairs each (a
    // workgroup takes about a microsecond per 32 of them): runs too.
    const bool spread = saving == kFastest && !in.block_forced && in.structures < in.units &&
                        in.largest_structure * std::min(in.most_images, planned_rows(in)) > kBlockSpreadPairs &&
                        static_cast<double>(in.atoms + 5 * in.structures) * static_cast<double>(block_width) * 8.0 <=
                            static_cast<double>(in.budget);
    // Centres of the polynomial basis that a slice of radial functions holds.
    // A structure formed in one workgroup needs all of its centres at once: one
    // past that (12,000 atoms among 1,024 molecules: 1.2 GB at l 2) sums runs,
    // and no run is longer.
    const PolyLayout poly = poly_layout(planned_rows(in), in.S, in.L, in.n, c.block);
    const int64_t slice_centres =
        in.radial_basis != 1 || c.poly_inside
            ? std::numeric_limits<int64_t>::max()
            : std::max<int64_t>(1, kPolySliceBytes / (poly.centre * static_cast<int64_t>(sizeof(double))));
    c.block_inner = c.block && in.average == 1 && whole && !spread && in.largest_structure <= slice_centres;
    c.block_small = c.block_inner && in.largest_structure <= kBlockSmallAtoms && in.radial_basis == 0;
    c.block_outer_lds = c.block && outer_lds;
    c.block_runs = c.block && in.average == 1 && !c.block_inner;
    c.block_outer = c.block && in.average == 2 && !outer_lds;
    if (saving >= kShortRows && (c.block_runs || c.block_outer) && !in.block_forced) {
        c.block = c.block_runs = c.block_outer = false;
    }
    // (weighted inner averages: those of few large structures only, whose
    // former kernel had them)
    c.f32_exps = c.block && in.block_float32 && !(in.average == 1 && in.weighted != 0 && whole);
    // else the 4x4-block kernel where the plan chose it (its coefficient rows
    // are its own), the 16x16 kernel, the generic one
    c.quad = !c.block && in.use_mfma && in.quad_waves > 0 && in.row_bound < kSlotCodeRows;
    c.partial_width = c.block_runs      ? block_width
                      : in.average != 1 ? static_cast<size_t>(in.features)
                      : c.quad          ? in.quad_width
                                        : in.tile_width;
    if (in.average != 0 && c.partials() && !c.block_outer) {
        const int64_t run = saving != kFastest ? kItemCentres
                            : c.block          ? run_centres(in, c.partial_width)
                            : tile_run_centres(in, c.partial_width, c.quad ? in.quad_waves : in.use_mfma ? in.tiles : 4);
        // by row, a slice of radial functions holds enough runs to fill the
        // device (kPolyLeastWaves; 500 structures of 70-100 atoms, n 8 l 1 of
        // three species, three slices of 585 runs of one wavefront each:
        // 7.6 ms, in the kernel itself 5.8)
        const int64_t fill = c.block || saving != kFastest || slice_centres >= in.atoms
                                 ? slice_centres
                                 : std::max<int64_t>(1, slice_centres * in.tiles / kPolyLeastWaves);
        c.run = std::min<int64_t>(fill, run);
    }
    return c;
}

// The polynomial basis' radial functions of a run.
inline PolyLayout poly_layout_of(const ChoiceInput& in, const Choice& c) {
    if (in.radial_basis != 1 || c.poly_inside) return {};
    return poly_layout(in.row_bound, in.S, in.L, in.n, c.block);
}

// The least scratch for them: a slice's centres, at least an item's.
inline size_t poly_least_bytes(const ChoiceInput& in, const Choice& c) {
    const PolyLayout layout = poly_layout_of(in, c);
    if (layout.centre == 0) return 0;
    const int64_t item = c.block_inner ? in.largest_structure : in.average != 0 && !c.block_outer ? c.run : 1;
    const int64_t slice = c.block ? kPolyLeastCentres : std::max(kPolyLeastCentres, kPolyLeastWaves / in.tiles);
    const int64_t centres = std::min(in.atoms, std::max(item, slice));
    return static_cast<size_t>(centres * layout.centre) * sizeof(double) + kPolySlack;
}

} // namespace mdx
