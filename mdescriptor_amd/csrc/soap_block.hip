// Host side of the register-coefficient kernel (soap_block_kernel.h): its
// compiled shapes, plan tables and launches, and the two small kernels beside
// it (the per-row neighbour weights, the rows of empty structures).
#include "soap_block_kernel.h"

namespace mdx {

// Shapes by l_max and radial groups, one translation unit each
// (soap_block_shape.hip): the coefficient registers of 1-4 and 5-8 species of
// one radial group; 1-2, 3-4 and 5-6 species of two; 1, 2, 3 and 4-5 of three.
// A plan takes the smallest that holds its species.
#define MDX_BLOCK_SHAPES(X) \
    X(2, 1) X(2, 2) X(2, 3) X(3, 1) X(3, 2) X(3, 3) X(4, 1) X(4, 2) X(4, 3) X(5, 1) X(5, 2) X(5, 3) \
    X(6, 1) X(6, 2) X(6, 3) X(7, 1) X(7, 2) X(7, 3) X(8, 1) X(8, 2) X(8, 3) X(9, 1) X(9, 2) X(9, 3)
#define MDX_DECLARE(LM, KG) std::pair<const BlockShape*, int> block_shapes_##LM##_##KG();
MDX_BLOCK_SHAPES(MDX_DECLARE)
#undef MDX_DECLARE

namespace {

// the compiled shape with the fewest coefficient registers that are enough
const BlockShape* find_shape(int l_max, int kg, int ncr) {
    const BlockShape* best = nullptr;
    auto look = [&](std::pair<const BlockShape*, int> list) {
        for (int i = 0; i < list.second; ++i) {
            const BlockShape& e = list.first[i];
            if (e.l_max == l_max && e.kg == kg && e.ncr >= ncr && (best == nullptr || e.ncr < best->ncr)) best = &e;
        }
    };
#define MDX_LOOK(LM, KG) if (l_max == LM && kg == KG) look(block_shapes_##LM##_##KG());
    MDX_BLOCK_SHAPES(MDX_LOOK)
#undef MDX_LOOK
    return best;
}

int coefficient_registers(int S, int kg) { return kg == 3 ? S : (S * kg + 3) / 4; }

} // namespace

int64_t block_partial_width(int l_max, int ncr) {
    return static_cast<int64_t>(units_total(0xffffffffu, l_max + 1)) * ncr * kWaveThreads;
}

bool block_float32_exps(int S, int n, int l_max, int out_dtype, int average, int compression, bool weighted,
                        bool polynomial) {
    const int kg = (n + 3) / 4;
    const BlockShape* e = find_shape(l_max, kg, coefficient_registers(compression == 1 ? 1 : S, kg));
    if (e == nullptr || !e->every_form || out_dtype != 4 || polynomial) return false;
    return average == 0 ? compression != 2 || !weighted : average == 1 && compression == 0;
}

bool block_plan_tables(int S, int n, int l_max, int table_dtype, int compression, bool polynomial,
                       const std::vector<double>& beta_scaled, const std::vector<double>& pref,
                       const std::vector<double>& expo, BlockPlanHost& out) {
    out = BlockPlanHost{};
    if (compression < 0 || compression > 3) return false;
    // species of the coefficients and the feature layout (mu2: one)
    const int St = compression == 1 ? 1 : S;
    const int kg = (n + 3) / 4;
    if (n < 1 || kg > (polynomial ? kBlockPolyGroups : 3)) return false;
    const BlockShape* e = find_shape(l_max, kg, coefficient_registers(St, kg));
    if (e == nullptr) return false;
    // registers past the species' stay zero, and no feature is stored from them
    const int ncr = e->ncr;
    const int L = l_max + 1;
    {
        const int64_t W = static_cast<int64_t>(St) * n;
        const int64_t F = compression == 2 ? W * n * L : compression == 3 ? W * (n + 1) / 2 * L : W * (W + 1) / 2 * L;
        if (F * table_dtype >= kDroppedBytes || n * n >= (1 << kStrideBits)) return false;
    }
    const int R = kg == 2 ? 2 : 1;
    const int RPL = kg / R;
    const int NT = kg == 1 ? 1 : kg == 2 ? 2 : 4;
    auto beta = [&](int l, int np, int k) -> double {
        if (np >= n || k >= n || np < 0 || k < 0) return 0.0;
        return beta_scaled[static_cast<size_t>((l * n + np) * n + k)] * pref[static_cast<size_t>(l * n + k)];
    };
    out.lane_e1.assign(static_cast<size_t>(L) * RPL * 64, 0.0);
    out.lane_beta.assign(static_cast<size_t>(L) * NT * 64, 0.0);
    for (int l = 0; l < L; ++l) {
        for (int lane = 0; lane < 64; ++lane) {
            const int b = (lane / 4) % 4;
            for (int rr = 0; rr < RPL; ++rr) {
                const int rg = rr * R + b % R;
                const int k = 4 * rg + lane % 4;
                out.lane_e1[static_cast<size_t>((l * RPL + rr) * 64 + lane)] =
                    k < n ? exp_lane_constant(expo[static_cast<size_t>(l * n + k)], table_dtype == 4) : 0.0;
            }
            // beta^T operand: lane = beta^T[k = lane / 16][n' = lane % 4] of the
            // fold term's (radial group in -> radial group out) block
            for (int t = 0; t < NT; ++t) {
                double v = 0.0;
                if (kg == 1) {
                    v = beta(l, lane % 4, lane / 16);
                } else if (kg == 2) {
                    const int rg = b % 2;
                    const int rin = t == 0 ? rg : 1 - rg;
                    v = beta(l, 4 * rg + lane % 4, 4 * rin + lane / 16);
                } else {
                    const int rin = (b + t) % 4;
                    if (b < 3 && rin < 3) v = beta(l, 4 * b + lane % 4, 4 * rin + lane / 16);
                }
                out.lane_beta[static_cast<size_t>((l * NT + t) * 64 + lane)] = v;
            }
        }
    }
    // power-spectrum offsets: tile pair p = (ri <= rj), value r, lane: feature
    // index at l = 0 and its stride per degree for channel i (group 4 ri + r,
    // radial channel 4 rg + lane / 16) and channel j (group 4 rj + (lane % 16) / 4,
    // 4 rg + lane % 4); pairs i > j and pad channels get kDroppedBytes
    auto channel = [&](int ri, int slot, int nl) -> int {
        int t = 0, rg = 0;
        if (kg == 3) {
            t = ri;
            rg = slot;
            if (slot >= 3) return -1;
        } else {
            const int g = 4 * ri + slot;
            t = g / kg;
            rg = g % kg;
        }
        const int np = 4 * rg + nl;
        if (t >= St || np >= n) return -1;
        return t * n + np;
    };
    // feature index of channel pair (i, j), i <= j (soap.cpp:997-1013)
    auto feature = [&](int i, int j, int& stride) -> int {
        const int t1 = i / n, n1 = i % n, t2 = j / n, n2 = j % n;
        int base = 0;
        for (int a1 = 0; a1 < St; ++a1) {
            for (int a2 = a1; a2 < St; ++a2) {
                const int size = a1 == a2 ? n * (n + 1) / 2 : n * n;
                if (a1 == t1 && a2 == t2) {
                    stride = size;
                    return base + (t1 == t2 ? n1 * n - n1 * (n1 - 1) / 2 + (n2 - n1) : n1 * n + n2);
                }
                base += L * size;
            }
        }
        return -1;
    };
    if (compression == 2) {
        // mu1nu1 (soap.cpp:969-981): channel i = (t, n1) of register ri
        // against the species-summed channel n2, feature t L n^2 + l n^2 +
        // n1 n + n2.  The summed register repeats its channels in every
        // species' blocks; its first kg blocks are taken.
        for (int ri = 0; ri < ncr; ++ri) {
            for (int r = 0; r < 4; ++r) {
                for (int lane = 0; lane < 64; ++lane) {
                    const int i = channel(ri, r, lane / 16);
                    const int slot = (lane % 16) / 4;
                    const int j = slot < kg ? 4 * slot + lane % 4 : n;
                    int fb = kDroppedBytes, fs = 0;
                    if (i >= 0 && j < n) {
                        const int t = i / n;
                        fb = (t * L * n * n + (i - t * n) * n + j) * table_dtype;
                        fs = n * n;
                    }
                    out.ps_offsets.push_back((fb << kStrideBits) | fs);
                }
            }
        }
    } else {
        for (int ri = 0; ri < ncr; ++ri) {
            for (int rj = ri; rj < ncr; ++rj) {
                for (int r = 0; r < 4; ++r) {
                    for (int lane = 0; lane < 64; ++lane) {
                        const int i = channel(ri, r, lane / 16);
                        const int j = channel(rj, (lane % 16) / 4, lane % 4);
                        int fb = kDroppedBytes, fs = 0;
                        if (i >= 0 && j >= 0 && i <= j) {
                            if (compression == 3) {
                                // crossover (soap.cpp:983-995): same species only
                                const int t1 = i / n, t2 = j / n, n1 = i % n, n2 = j % n;
                                if (t1 == t2) {
                                    fs = n * (n + 1) / 2;
                                    fb = (t1 * L * fs + n1 * n - n1 * (n1 - 1) / 2 + (n2 - n1)) * table_dtype;
                                }
                            } else {
                                fb = feature(i, j, fs) * table_dtype;
                            }
                        }
                        out.ps_offsets.push_back((fb << kStrideBits) | fs);
                    }
                }
            }
        }
    }
    // the kernel stages exactly this many entries
    if (out.ps_offsets.size() != static_cast<size_t>(ps_tiles(ncr, compression == 2)) * 4 * 64) {
        throw Error(MDX_INTERNAL, "power-spectrum offset table does not match the expansion kernel");
    }
    out.kg = kg;
    out.ncr = ncr;
    out.waves = e->waves;
    out.every_form = e->every_form;
    return true;
}


void launch_block_expand(hipStream_t stream, int l_max, int kg, int ncr, const BlockArgs& a, int64_t count) {
    if (count <= 0) return;
    const BlockShape* e = find_shape(l_max, kg, ncr);
    if (e == nullptr) throw Error(MDX_INTERNAL, "SOAP shape is not compiled for the register-coefficient kernel");
    if (a.outer_lds != 0 && (a.struct_offsets == nullptr || a.table_dtype != 8 ||
                             a.F * static_cast<int64_t>(sizeof(double)) > kBlockOuterLdsBytes)) {
        throw Error(MDX_INTERNAL, "outer average row does not fit the register-coefficient kernel's LDS");
    }
    if (a.out_bytes > a.table_dtype || a.row_w == nullptr || (a.table_dtype == 4 && !e->every_form) ||
        (a.polynomial != 0 && (a.poly_g == nullptr || kg > kBlockPolyGroups || a.table_dtype != 8 || a.small_structures || a.outer_lds != 0))) {
        throw Error(MDX_INTERNAL, "register-coefficient kernel launched with inconsistent arguments");
    }
    e->launch(stream, a, count);
    MDX_HIP(hipGetLastError());
}

namespace {

// a wavefront per centre, kRowsPerLane of its rows per lane at a time: every
// row's loads are issued before any weight is formed, so the gathers of
// the batch of rows are in flight together; the distance as the
// expansion's harmonic staging forms it (image - centre, fma order)
constexpr int kRowsPerLane = 4;
__global__ __launch_bounds__(256) void k_block_row_weights(BlockArgs a, int64_t centres, double* row_w) {
    const int lane = threadIdx.x % kWaveThreads;
    const int64_t waves = static_cast<int64_t>(gridDim.x) * (blockDim.x / kWaveThreads);
    for (int64_t c = static_cast<int64_t>(blockIdx.x) * (blockDim.x / kWaveThreads) + threadIdx.x / kWaveThreads;
         c < centres; c += waves) {
        int total = 0;
        for (int t = 0; t < a.S; ++t) total += a.counts[c * a.S + t];
        const int64_t row0 = a.pair_start[c];
        const double cx = a.positions[3 * c], cy = a.positions[3 * c + 1], cz = a.positions[3 * c + 2];
        for (int base = 0; base < total; base += kRowsPerLane * kWaveThreads) {
            uint32_t bin[kRowsPerLane];
            double px[kRowsPerLane], py[kRowsPerLane], pz[kRowsPerLane];
#pragma unroll
            for (int i = 0; i < kRowsPerLane; ++i) {
                const int r = base + i * kWaveThreads + lane;
                bin[i] = r < total ? a.pair_bin[row0 + r] : a.pair_bin[row0];
            }
#pragma unroll
            for (int i = 0; i < kRowsPerLane; ++i) {
                px[i] = a.bx[bin[i]];
                py[i] = a.by[bin[i]];
                pz[i] = a.bz[bin[i]];
            }
#pragma unroll
            for (int i = 0; i < kRowsPerLane; ++i) {
                const int r = base + i * kWaveThreads + lane;
                if (r >= total) continue;
                const uint32_t b = bin[i];
                const double dx = px[i] - cx, dy = py[i] - cy, dz = pz[i] - cz;
                const double r2 = fma(dz, dz, fma(dx, dx, dy * dy));
                // soap_weight (soap.cpp:389-420); w0 for the exact self pair,
                // the centre's own atom under the zero shift
                // (NeighborView::exact_self, neighbor.cpp:683-689).  Such an
                // image is the position plus a zero vector, so its r2 is 0
                // exactly: only rows at r2 == 0 gather the atom and shift
                double v = weight_function(a.weighting, a.w_r0, a.w_c, a.w_d, a.w_m, sqrt(r2));
                if (a.has_w0 != 0 && r2 == 0.0) {
                    const ImageDesc& image = a.images[a.bin_image[b]];
                    const bool zero = image.n[0] == 0 && image.n[1] == 0 && image.n[2] == 0;
                    if (zero && static_cast<int64_t>(a.bin_atom[b]) == c) v = a.w_w0;
                }
                row_w[row0 + r] = v * a.species_w[a.bin_type[b]];
            }
        }
    }
}

// one workgroup per structure without atoms; its row's bytes zeroed
__global__ void k_block_zero_rows(const int64_t* struct_offsets, int64_t structures, char* out, int64_t pitch,
                                  int64_t row_bytes) {
    for (int64_t s = blockIdx.x; s < structures; s += gridDim.x) {
        if (struct_offsets[s + 1] != struct_offsets[s]) continue;
        char* row = out + s * pitch;
        for (int64_t i = threadIdx.x; i < row_bytes; i += blockDim.x) row[i] = 0;
    }
}

} // namespace

void launch_block_row_weights(hipStream_t stream, const BlockArgs& a, int64_t centres, double* row_w) {
    if (centres <= 0) return;
    const unsigned grid =
        static_cast<unsigned>(std::min<int64_t>((centres + 3) / 4, 32 * static_cast<int64_t>(device_compute_units())));
    hipLaunchKernelGGL(k_block_row_weights, dim3(grid), dim3(256), 0, stream, a, centres, row_w);
    MDX_HIP(hipGetLastError());
}

void launch_block_zero_rows(hipStream_t stream, const int64_t* struct_offsets, int64_t structures, void* out,
                            int64_t pitch, int64_t row_bytes) {
    if (structures <= 0 || row_bytes <= 0) return;
    const unsigned grid = static_cast<unsigned>(std::min<int64_t>(structures, 1 << 16));
    hipLaunchKernelGGL(k_block_zero_rows, dim3(grid), dim3(256), 0, stream, struct_offsets, structures,
                       static_cast<char*>(out), pitch, row_bytes);
    MDX_HIP(hipGetLastError());
}

} // namespace mdx
