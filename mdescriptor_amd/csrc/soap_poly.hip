// Radial functions of the polynomial basis, one row of L n values per pair:
//   G[row][l n + k] = sum_q K_l(r_q; d) w_q r_q^2 g_k(r_q),
// K_l the Gaussian-smeared radial kernel of polynomial_flir
// (soap.cpp:450-492), by its upward recurrence from two exponentials, with
// the l = 0 special case at d <= 1e-14.  The expansion (k_soap_block, or
// k_soap_mfma for shapes it lacks where that is the faster way, soap_choice.h)
// reads those of a slice of centres; the arithmetic per (pair, point) is the
// reference's, since its clamped upward recurrence amplifies rounding.
//
// A wavefront takes 16 rows and the whole grid, four points a step.  Lane L
// evaluates K_0..K_{L-1} of row L % 16 at point L / 16 of the step, which is
// the A operand of v_mfma_f64_4x4x4f64 (block b = (L / 4) % 4 holds rows
// 4b..4b+3: A_b lane L = A_b[row L % 4][point L / 16]); the B operand is the
// quadrature-weighted basis of radial group g (B lane L = w_q r_q^2
// g_{4g + L % 4}(r_q), the same for every block), so one MFMA per degree and
// radial group accumulates 16 rows x 4 channels, nothing is padded but the
// last channels, and the sums stay in registers over the grid with no
// barrier.  Result lane L holds row 4b + L / 16, channel 4g + L % 4.
//
// Bound by issue: a step of 64 (row, point) pairs takes about 55 vector
// instructions (two table exps of 14, the prefactor's division as one
// Newton step on tabulated reciprocals, 5, and four per degree past the
// second) and L ceil(n/4) MFMAs, which share the issue slots.  Inside the
// expansion's workgroup (one centre, a barrier per 32 rows, 237 registers)
// the same sums ran at a quarter of that rate.  3,000 atoms, n 6 l 5 float64
// rows: 1,257 us for both there, 405 here and 98 in the expansion; 16,384
// atoms, n 7 l 6: 4,433 us, 2,400 and 632.
#include "soap_mfma.h"

#include <algorithm>
#include <cmath>

namespace mdx {
namespace {

constexpr int kThreads = 256;
constexpr int kWaves = kThreads / kWave;
constexpr int kStagedPoints = 128; // grid points staged in LDS, at most

struct PolyArgs {
    const double* positions;
    const int64_t* pair_start;
    const int32_t* counts;
    const uint32_t* pair_bin;
    const double* bx;
    const double* by;
    const double* bz;
    const double* points;  // [steps * 4] r_q (1 past the grid)
    const double* inverse; // [steps * 4] 1 / r_q
    const double* basis;   // [steps * 4][4 KG] w_q r_q^2 g_k(r_q), 0 past the grid and the channels
    const double* centre;  // [n] sum_q e^{-eta r_q^2} w_q r_q^2 g_k(r_q)
    double eta;
    int S, L, n, steps;
    int64_t first, count; // centres [first, first + count)
    int split;            // workgroups per centre, or
    int share;            // centres per workgroup (1, 2 or kWaves)
    PolyLayout layout; // of out
    double* out;
};

// exp(x), x <= 0, by Tang's table method (ACM TOMS 15(2), 1989) with 64
// entries and a degree-5 polynomial (truncation below 4e-17 relative).
// tab[j] = 2^(j/64) with j << 14 taken off its high word, so one integer add
// of (64k + j) << 14 scales it by 2^k.  Arguments below -700 are clamped
// there (1e-304).  The kernels' recurrence amplifies the difference of the
// two exps' errors, and exps of one entry share its: 256 entries, shorter by
// an instruction, put the features 1.3 to 2 times further off.
__device__ __forceinline__ double exp_table(double x, const int2* tab) {
    constexpr double kInvLn2xT = 92.332482616893658071035179584121; // 64 / ln 2
    constexpr double kLn2OverTHi = 0.010830417275428772;             // ln2/64 with 32 trailing zero bits
    constexpr double kLn2OverTLo = 7.420820373486988e-09;            // ln2/64 - kLn2OverTHi
    constexpr double kShifter = 6755399441055744.0;                  // 1.5 * 2^52
    x = fmax(x, -700.0);
    const double s = fma(x, kInvLn2xT, kShifter);
    const double kf = s - kShifter;
    double r = fma(kf, -kLn2OverTHi, x);
    r = fma(kf, -kLn2OverTLo, r);
    double q = fma(r, 1.0 / 120.0, 1.0 / 24.0);
    q = fma(q, r, 1.0 / 6.0);
    q = fma(q, r, 0.5);
    q = fma(q, r, 1.0);
    const int nj = __double2loint(s);
    const int2 t = *reinterpret_cast<const int2*>(reinterpret_cast<const char*>(tab) + ((nj << 3) & (63 << 3)));
    const double tk = __hiloint2double(t.y + (nj << 14), t.x);
    return fma(tk, r * q, tk);
}

template <int LD, int KG, bool kStaged>
__global__ __launch_bounds__(kThreads) void k_poly_radial(PolyArgs a) {
    __shared__ int2 s_tab[64];
    __shared__ double s_grid[kStaged ? kStagedPoints * (2 + 4 * KG) : 1];
    const int tid = threadIdx.x;
    const int lane = tid % kWave;
    const int wave = __builtin_amdgcn_readfirstlane(tid / kWave);
    // this wavefront's tile: 16 slots of a centre, whole step groups (so a
    // group's 512 bytes a degree are written by one wavefront: tiles of 16
    // rows across groups, halves of whose lines come from two dies, took
    // 610 us against 405 for 834,000 pairs, n 6 l 5)
    const unsigned block = blockIdx.x / static_cast<unsigned>(a.split);
    const int part = static_cast<int>(blockIdx.x - block * static_cast<unsigned>(a.split));
    const int per_centre = kWaves / a.share; // wavefronts of a centre here
    const int64_t offset = static_cast<int64_t>(block) * a.share + wave / per_centre;
    const int64_t c = a.first + min(offset, a.count - 1);
    constexpr int R = KG == 2 ? 2 : 1, GS = poly_group_slots(KG); // slots of a step group
    const int tile = part * kWaves + wave % per_centre;
    int groups = 0; // the centre's step groups: every species' rows in whole ones
    for (int t = 0; t < a.S; ++t) groups += (a.counts[c * a.S + t] + GS - 1) / GS;
    // the whole workgroup is past its centre's groups
    if (a.share == 1 && R * part * kWaves >= groups) return;
    if (tid < 64) {
        const double t = exp2(static_cast<double>(tid) / 64.0);
        s_tab[tid] = int2{__double2loint(t), __double2hiint(t) - (tid << 14)};
    }
    const int points = 4 * a.steps;
    if constexpr (kStaged) {
        for (int i = tid; i < points; i += kThreads) {
            s_grid[i] = a.points[i];
            s_grid[kStagedPoints + i] = a.inverse[i];
        }
        for (int i = tid; i < points * 4 * KG; i += kThreads) s_grid[2 * kStagedPoints + i] = a.basis[i];
    }
    __syncthreads();
    const double eta = a.eta;
    if (offset >= a.count || R * tile >= groups) return;
    const int64_t first_row = a.pair_start[c];
    // the pair row of slot s of the tile, -1 past its species' rows
    auto slot_row = [&](int s) {
        int g = R * tile + s / GS, row = 0, rows = 0;
        bool found = false;
        for (int t = 0; t < a.S; ++t) {
            const int count = a.counts[c * a.S + t], n = (count + GS - 1) / GS;
            if (!found) {
                found = g < n;
                rows = count;
                if (!found) {
                    g -= n;
                    row += count;
                }
            }
        }
        const int in_species = g * GS + s % GS;
        return found && in_species < rows ? row + in_species : -1;
    };
    const double cx = a.positions[3 * c], cy = a.positions[3 * c + 1], cz = a.positions[3 * c + 2];
    const uint32_t bin = a.pair_bin[first_row + max(slot_row(lane % 16), 0)];
    const double dx = a.bx[bin] - cx, dy = a.by[bin] - cy, dz = a.bz[bin] - cz;
    const double distance = sqrt(dx * dx + dy * dy + dz * dz);
    const bool at_centre = distance <= 1e-14;
    const double radius = at_centre ? 1.0 : distance;
    const double scale = eta * radius;
    const double inverse_scale = 1.0 / scale;
    double acc[LD][KG];
#pragma unroll
    for (int l = 0; l < LD; ++l) {
#pragma unroll
        for (int g = 0; g < KG; ++g) acc[l][g] = 0.0;
    }
    for (int step = 0; step < a.steps; ++step) {
        const int q = 4 * step + lane / 16;
        double radial, inverse, b[KG];
        if constexpr (kStaged) {
            radial = s_grid[q];
            inverse = s_grid[kStagedPoints + q];
#pragma unroll
            for (int g = 0; g < KG; ++g) b[g] = s_grid[2 * kStagedPoints + q * 4 * KG + 4 * g + lane % 4];
        } else {
            radial = a.points[q];
            inverse = a.inverse[q];
#pragma unroll
            for (int g = 0; g < KG; ++g) b[g] = a.basis[q * 4 * KG + 4 * g + lane % 4];
        }
        // prefactor = 0.25 / (eta radius radial): the product of the
        // reciprocals, corrected by its remainder (bit for bit the division in
        // 10^8 random cases)
        const double product = scale * radial;
        const double reciprocal = inverse_scale * inverse;
        const double quarter = 0.25 * reciprocal;
        const double prefactor = fma(fma(-product, quarter, 0.25), reciprocal, quarter);
        const double below = radial - radius, above = radial + radius;
        // (past eight degrees or channels the recurrence needs exp's last bit)
        constexpr bool kLibrary = LD > 8 || KG > 2;
        const double x_minus = -eta * below * below, x_plus = -eta * above * above;
        const double minus = kLibrary ? exp(x_minus) : exp_table(x_minus, s_tab);
        const double plus = kLibrary ? exp(x_plus) : exp_table(x_plus, s_tab);
        double before = prefactor * (minus - plus);
        double last = prefactor * (minus + plus - 2.0 * before);
#pragma unroll
        for (int g = 0; g < KG; ++g) acc[0][g] = __builtin_amdgcn_mfma_f64_4x4x4f64(before, b[g], acc[0][g], 0, 0, 0);
#pragma unroll
        for (int l = 1; l < LD; ++l) {
            double value = last;
            if (l >= 2) {
                const double next = before - prefactor * (4.0 * l - 2.0) * last;
                value = next > 0.0 ? next : 0.0;
                before = last;
                last = value;
            }
#pragma unroll
            for (int g = 0; g < KG; ++g) acc[l][g] = __builtin_amdgcn_mfma_f64_4x4x4f64(value, b[g], acc[l][g], 0, 0, 0);
        }
    }
    // the lane's result row, and whether that row's atom is the centre
    const int row = 4 * ((lane / 4) % 4) + lane / 16;
    const bool own = ((__ballot(at_centre) >> row) & 1) != 0;
    const int pair = slot_row(row);
    if (a.layout.groups != 0) {
        // 16 lanes per neighbour of a step, 4 per block of a radial group
        // and step phase, one per channel; zero past the species' rows
        if (R * tile + row / GS >= groups) return;
        const int s = row % GS;
        double* out = a.out + poly_group(a.layout.groups, c, a.first, R * tile + row / GS, a.L * (KG / R) * kWave) +
                      s % 4 * 16 + s / 4 * R * 4 + lane % 4;
#pragma unroll
        for (int l = 0; l < LD; ++l) {
#pragma unroll
            for (int g = 0; g < KG; ++g) {
                const int k = 4 * g + lane % 4;
                const double v = !own ? acc[l][g] : l == 0 && k < a.n ? a.centre[k] : 0.0;
                if (l < a.L) out[(l * (KG / R) + g / R) * kWave + g % R * 4] = pair >= 0 ? v : 0.0;
            }
        }
    } else if (pair >= 0) {
        double* out = a.out + poly_row(a.layout.centre, c, a.first, pair, a.L * a.n);
#pragma unroll
        for (int l = 0; l < LD; ++l) {
#pragma unroll
            for (int g = 0; g < KG; ++g) {
                const int k = 4 * g + lane % 4;
                if (l < a.L && k < a.n) out[l * a.n + k] = !own ? acc[l][g] : l == 0 ? a.centre[k] : 0.0;
            }
        }
    }
}

template <int LD, int KG>
void launch(hipStream_t stream, unsigned grid, const PolyArgs& a) {
    if (4 * a.steps <= kStagedPoints) {
        hipLaunchKernelGGL((k_poly_radial<LD, KG, true>), dim3(grid), dim3(kThreads), 0, stream, a);
    } else {
        hipLaunchKernelGGL((k_poly_radial<LD, KG, false>), dim3(grid), dim3(kThreads), 0, stream, a);
    }
}

template <int KG>
void launch_degrees(hipStream_t stream, unsigned grid, const PolyArgs& a) {
    // (the degrees past L are summed and not stored)
    if (a.L <= 4) launch<4, KG>(stream, grid, a);
    else if (a.L <= 6) launch<6, KG>(stream, grid, a);
    else if (a.L <= 7) launch<7, KG>(stream, grid, a);
    else if (a.L <= 8) launch<8, KG>(stream, grid, a);
    else if (a.L <= 11) launch<11, KG>(stream, grid, a);
    else launch<kMaxLmax + 1, KG>(stream, grid, a);
}

} // namespace

std::vector<double> poly_radial_tables(int grid, int n, double eta, const double* points, const std::vector<double>& bw) {
    const int groups = poly_channel_groups(n);
    const size_t padded = static_cast<size_t>((grid + 3) / 4 * 4);
    std::vector<double> t(padded * (2 + 4 * static_cast<size_t>(groups)) + static_cast<size_t>(n), 0.0);
    double* inverse = t.data() + padded;
    double* basis = inverse + padded;
    double* centre = basis + padded * 4 * static_cast<size_t>(groups);
    for (size_t q = 0; q < padded; ++q) {
        const bool on = q < static_cast<size_t>(grid);
        t[q] = on ? points[q] : 1.0;
        inverse[q] = 1.0 / t[q];
        for (int k = 0; on && k < n; ++k) {
            const double value = bw[q * static_cast<size_t>(n) + static_cast<size_t>(k)];
            basis[q * 4 * static_cast<size_t>(groups) + static_cast<size_t>(k)] = value;
            centre[k] += std::exp(-eta * (points[q] * points[q])) * value;
        }
    }
    return t;
}

void launch_poly_radial(hipStream_t stream, const PreparedBatch& pb, const DeviceGraph& g, const double* tables,
                        const MfmaDims& d, int64_t first, int64_t count, const PolyLayout& layout, double* out,
                        int64_t capacity) {
    if (count <= 0) return;
    if (out == nullptr || count * layout.centre > capacity) {
        throw Error(MDX_INTERNAL, "radial functions of a slice of centres outgrow their scratch");
    }
    const int groups = poly_channel_groups(d.n);
    const int64_t padded = (d.grid + 3) / 4 * 4;
    PolyArgs a{};
    a.positions = pb.d_positions.as<double>();
    a.pair_start = g.pair_start.as<int64_t>();
    a.counts = g.counts.as<int32_t>();
    a.pair_bin = g.pair_bin.as<uint32_t>();
    a.bx = g.bin_x.as<double>();
    a.by = g.bin_y.as<double>();
    a.bz = g.bin_z.as<double>();
    const PolyTables t = poly_tables(tables, d.grid, d.n);
    a.points = t.points;
    a.inverse = t.inverse;
    a.basis = t.basis;
    a.centre = t.centre;
    a.eta = d.eta;
    a.S = d.S;
    a.L = d.L;
    a.n = d.n;
    a.steps = static_cast<int>(padded / 4);
    a.first = first;
    a.count = count;
    a.layout = layout;
    a.out = out;
    // a wavefront per tile, as many as the centres' rows can fill: workgroups
    // past them end at once, and the device balances the others (a workgroup
    // per centre left a second round of workgroups a quarter full: 451 us
    // against 405 for 834,000 pairs, n 6 l 5)
    const int64_t slots = poly_group_slots(groups);
    const int64_t tiles = ((std::max<int64_t>(1, g.row_bound) / slots + d.S) * slots + 15) / 16;
    a.split = static_cast<int>((tiles + kWaves - 1) / kWaves);
    a.share = tiles == 1 ? kWaves : tiles == 2 ? 2 : 1;
    const unsigned grid = static_cast<unsigned>((count + a.share - 1) / a.share * a.split);
    if (groups == 1) launch_degrees<1>(stream, grid, a);
    else if (groups == 2) launch_degrees<2>(stream, grid, a);
    else launch_degrees<4>(stream, grid, a);
    MDX_HIP(hipGetLastError());
}

} // namespace mdx
