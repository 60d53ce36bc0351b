// Host/device interface of the register-coefficient SOAP kernel
// (soap_block.hip, soap_block_kernel.h): GTO basis, every compression, with
// or without neighbour weights; a row per centre, or a row per structure of
// its centres' averaged coefficients (average "inner") or averaged power
// spectra ("outer").
#pragma once

#include "mdx_internal.h"
#include "soap_choice.h"

namespace mdx {

// Kinds of row the kernel is compiled for.
//   rows         a row per centre
//   inner        a row per structure of its centres' averaged coefficients,
//                from a centre-by-centre stream: a workgroup per structure,
//                or for few large structures two launches (partial_out /
//                partial_in): runs of a structure's centres leave their
//                summed coefficient registers in partial rows, then a row per
//                structure from the sum of its partial rows
//   inner small  the same from a species-major stream over the structure's
//                pairs (structures of at most 64 atoms)
//   outer LDS    outer averages, a workgroup per structure: every centre's
//                power spectrum added into the structure's float64 row in
//                LDS and the mean written once
//   inner runs   the first of the two launches above by itself (shapes compiled
//                in every form: with a row's end in the same kernel 500
//                structures of 70-100 atoms, four species n 5 l 6, took 457 us
//                instead of 403)
// Each takes neighbour weights (row_w) and every compression: mu1nu1
// (summed: each channel against the species-summed channels) as a branch at
// the end of a row, the others through the plan's tables.
constexpr int kBlockRows = 0, kBlockInner = 1, kBlockInnerSmall = 2, kBlockOuterLds = 3, kBlockInnerRuns = 4;
// ... and forms: unweighted, weighted (the weights may be 1), the polynomial
// basis (weighted the same way): the radial functions come from memory
// (launch_poly_radial) instead of exps, rows and inner averages only, up to
// two radial groups (its normalisation fails past eight channels);
// unweighted float32 rows of float64 tables; and weighted rows and inner
// averages of the tables' own type (shapes compiled in every form).
constexpr int kBlockPlain = 0, kBlockWeighted = 1, kBlockPolynomial = 2, kBlockHalf = 3, kBlockWeightedFull = 4;
constexpr int kBlockPolyGroups = 2;

// Launch arguments (one struct, passed by value).
struct BlockArgs {
    const double* positions;    // f64[atoms * 3]
    const int64_t* pair_start;  // first pair row of each centre
    const int32_t* counts;      // rows per (centre, species)
    const uint32_t* pair_bin;   // bin of each pair row
    const double* bx;           // binned image positions
    const double* by;
    const double* bz;
    const double* lane_e1;      // [l][register][64]: -a_lk of the lane's exp row (float32 rows: -a_lk 256/ln2), 0 for pad rows
    const double* lane_beta;    // [l][fold term][64]: beta^T operand of the lane
    const int32_t* ps_offsets;  // [tile pair][value][64]: (byte offset at l = 0) << 9 | feature stride per l
    int S;                      // species
    int table_dtype;            // bytes per value the tables are for: 4 (float32 exps and rows) or 8
    int out_bytes;              // bytes per output value, 4 or 8 (tables for 4: 4)
    int64_t F;                  // features per row
    int64_t item_base, items, per_block; // centres, or structures when struct_offsets is set
    const int64_t* struct_offsets;       // null: a row per centre; else first centre of each structure
                                         // (+ end): a row per structure, its centres' average
    int small_structures;                // averages: every structure has at most 64 atoms
    // neighbour weights (soap_weight): distance function kind (0 none),
    // its parameters, w0 for the centre's own image, species weights
    int weighting;
    int has_w0;
    double w_r0, w_c, w_d, w_m, w_w0;
    const double* species_w;             // null: no weights
    const int32_t* bin_atom;             // atom of each binned image
    const int32_t* bin_image;            // image of each binned image (w0: the exact self pair)
    const int32_t* bin_type;             // species of each binned image
    const ImageDesc* images;             // image table (integer shifts)
    // each pair row's weight, at row_w[row & row_w_mask]: the distance
    // function (or w0) times the species weight (k_block_row_weights), mask
    // -1; without weights one value of 1, mask 0
    const double* row_w;
    int64_t row_w_mask;
    // polynomial basis: radial functions of the slice's pairs, a step group
    // of 64 values per degree and exp register at
    // [(centre - poly_first) * poly_groups + group][l][register][lane]
    int polynomial; // that basis (poly_g set)
    const double* poly_g;
    int64_t poly_first, poly_groups;
    int summed;                          // mu1nu1: spectrum against the species-summed coefficients
    int mu2;                             // mu2: every species' sums into the first species' slots
    // inner averages in two launches: the runs' launch writes partial_out
    // (struct_offsets = first centre of each run, + end), the final launch
    // reads partial_in (items = structures, struct_offsets = the batch's
    // atom offsets, part_items = each structure's partial rows, + end).  A
    // partial row holds every wavefront's coefficient registers, lane-major
    // (block_partial_width doubles).
    double* partial_out;
    const double* partial_in;
    const int64_t* part_items;
    // outer averages in LDS (items = structures, struct_offsets = the
    // batch's atom offsets, table_dtype 8): a row per structure, the mean of
    // its centres' power spectra
    int outer_lds;
    void* out;
    int64_t pitch;              // bytes between output rows
};

// Plan tables of the kernel for one SOAP shape.  beta_scaled is
// pi^1.5 beta with index (l*n + n')*n + k, pref the radial prefactor of
// channel l*n + k, expo the radial exponent a_lk.
struct BlockPlanHost {
    int kg = 0;      // radial groups of 4 channels
    int ncr = 0;     // coefficient registers per (l, column group)
    int waves = 0;   // wavefronts per workgroup
    bool every_form = false; // BlockShape::every_form
    std::vector<double> lane_e1, lane_beta;
    std::vector<int32_t> ps_offsets; // packed feature offsets
};

// One compiled shape (soap_block_shape.hip): l_max, radial groups,
// coefficient registers.  every_form: compiled with float32 and float64 exps
// for rows and inner averages, weighted or not; else float64 exps serve
// every output type.
struct BlockShape {
    int l_max, kg, ncr;
    bool every_form;
    int waves;
    void (*launch)(hipStream_t, const BlockArgs&, int64_t);
};

// Fills out and returns true when a compiled shape holds (S, n, l_max).
// compression: 0 off, 1 mu2 (one coefficient species: the shape of S
// species, the feature layout of one), 2 mu1nu1, 3 crossover (the feature
// layouts of soap.cpp:948-1013).  polynomial: that radial basis (float64
// tables).  table_dtype: the value size the tables are built for.
bool block_plan_tables(int S, int n, int l_max, int table_dtype, int compression, bool polynomial,
                       const std::vector<double>& beta_scaled, const std::vector<double>& pref,
                       const std::vector<double>& expo, BlockPlanHost& out);
// Whether a plan takes float32 exps (relative error 1.4e-13 against 5e-15):
// float32 rows of the shapes compiled in every form, and their uncompressed
// inner averages (weighted ones as runs of centres only, Choice::f32_exps).
// There the beta fold does not lift the difference to the rows' own rounding:
// against float64 rows rounded to float32 (2.0-2.9e-8 of the row), twelve
// channels in 5 A (max |beta| 2.0e5) are 1.0e-10 of the row off, in 4 A
// (6.8e5) 5.5e-10, eight in 2 A (2.0e6) 8e-11.  average: 0 off, 1 inner, 2
// outer (whose rows are float64 sums).
bool block_float32_exps(int S, int n, int l_max, int out_dtype, int average, int compression, bool weighted,
                        bool polynomial);
void launch_block_expand(hipStream_t stream, int l_max, int kg, int ncr, const BlockArgs& a, int64_t count);
// doubles in one partial row of the runs' launch
int64_t block_partial_width(int l_max, int ncr);
// Each pair row's weight for the weighted modes, row_w[row] for the rows
// of centres [0, centres): the distance function of the neighbour's
// distance (w0 for the centre's own image under the zero shift) times its
// species weight (soap_weight, soap.cpp:389-420).  Uses the graph, position,
// weighting and species-weight fields of a.
void launch_block_row_weights(hipStream_t stream, const BlockArgs& a, int64_t centres, double* row_w);
// Zero the rows of the structures without atoms (structure averages; the
// expansion writes only the rows of structures it visits).
void launch_block_zero_rows(hipStream_t stream, const int64_t* struct_offsets, int64_t structures, void* out,
                            int64_t pitch, int64_t row_bytes);

} // namespace mdx
