// Forward operator in the grid form (km_grid.h): rbf and spectral kernels, any number of rhs
// columns.  A row block of 128 rows is one item, worked on by W wavefronts (large launches: by one, four row
// blocks together, see group_item):
//
//   columns -> grid   the wavefronts take the steps of 32 columns of the block's range in turn; V is
//                     the A operand (16 grid points x 32 columns), rhs (spectral: times cos B and
//                     sin B, as in the phase-split table kernel) the B operand.  Grid tiles out of a
//                     step's reach are skipped.  With W > 1 the sums meet in LDS, added in a fixed order.
//   grid -> rows      every wavefront takes 128 / W rows; V is the A operand again (16 rows x 32 grid
//                     points), the sums, moved between lanes into operand layout, the B operand.
//
// Both factors of both contractions are split into two fp16 terms as in the table kernels.  A row
// block whose window does not fit the accumulators (points sparse against the lengthscale), whose
// range is too short to gain, or whose coordinates are not finite is evaluated entry by entry in the
// same launch: each wavefront its rows, tile against tile, those out of reach left out.  A value of rhs
// that is not finite makes its column's results NaN in every row whose range holds it, as does a NaN
// among the range's column coordinates (spectral: an infinity as well) in all columns.
//
// Measured against the entry-wise kernels (a call, queued): rbf n = 65536, k = 64 43.6 -> 21.6 us; the large
// launches below, at group_item.  The small ones are bound by the latency of one wavefront's steps.
#include "km_batch.h"
#include "km_common.h"
#include "km_fwd.h"
#include "km_entries.h"
#include "km_grid.h"
#include "km_group_plan.h"
#include "km_launch.h"

namespace km {

// Columns in a row block's range from which the grid form is taken.
#define KM_GRID_MIN_WIDTH 160
// Sums are exchanged between wavefronts times 2^-16: those over a grid point's columns can be larger than
// any result.
#define KM_GRID_EXCHANGE 16

__device__ __forceinline__ GridVectors vectors(const FwdArgs& a) {
    return {a.x2_s, a.rhs_s0, a.rhs_s1, a.k};
}

// Rows whose values a wavefront holds, two per lane (the layout of BlockRows).
struct HeldRows {
    float y[2], rest[2], cos[2], sin[2];
};

template <int KT>
__device__ __forceinline__ HeldRows hold_rows(const BlockRows& rows, float x_ref, const KernelConsts& kc) {
    HeldRows h;
#pragma unroll
    for (int i = 0; i < 2; i++) {
        const float x = i == 0 ? rows.xa : rows.xb;
        h.y[i] = x - x_ref;
        h.rest[i] = remainder_of(x, x_ref, h.y[i]);
        const float th = KT == KM_KERNEL_SPECTRAL ? phase_rev(kc.f, x, x_ref) : 0.0f;
        h.cos[i] = __builtin_amdgcn_cosf(th);
        h.sin[i] = __builtin_amdgcn_sinf(th);
    }
    return h;
}

// Grid -> rows: `groups` groups of 16 rows from row0 from the sums of their window, in the accumulators'
// layout.  EXCHANGED: the sums come through LDS, scaled back already; else they are times 2^shift and the scale
// of the evaluated factor.  held: the rows, where the wavefront has all 128.
template <int KT, int G, int MT, bool EXCHANGED, bool HELD>
__device__ __forceinline__ void grid_rows(const FwdArgs& a, const WaveView& w, const HeldRows* held, int row0, int groups,
                                          int kbase, const GridWindow& gw, const KernelConsts& kc, const int (&shift)[G],
                                          float4v (&acc)[MT][G * (KT == KM_KERNEL_SPECTRAL ? 2 : 1)]) {
    constexpr bool PHASE = KT == KM_KERNEL_SPECTRAL;
    constexpr int GE = G * (PHASE ? 2 : 1);
    const int lane = threadIdx.x & 63;
    const int li = lane & 15;
    const int kk = lane >> 4;
    // One power-of-two scale per column over the whole window; the operands of all
    // steps of 32 grid points replace the accumulators, so that a row group needs no more than its
    // own accumulator at a time.
    const float hz = gw.h * gw.s2;
    float b2[8];
#pragma unroll
    for (int t = 0; t < 8; t++) {
        const float b = ((float)t - 3.5f) * hz;
        b2[t] = uniform(b + b);
    }
    float fac[8];
#pragma unroll
    for (int t = 0; t < 8; t++) {
        fac[t] = uniform(__builtin_amdgcn_exp2f(-0.25f * b2[t] * b2[t]));
    }
    const float weight = w.params[KernelTraits<KT>::SIGMA * a.params_s] * (hz * KM_GRID_WEIGHT);
    float down[GE];
    constexpr int KSTEPS = (MT + 1) / 2;
    half8v bhi[KSTEPS][GE], blo[KSTEPS][GE];
#pragma unroll
    for (int g = 0; g < GE; g++) {
        float m = 0.0f;
#pragma unroll
        for (int mt = 0; mt < MT; mt++) {
#pragma unroll
            for (int v = 0; v < 4; v++) {
                m = fmaxf(m, fabsf(acc[mt][g][v]));
            }
        }
        m = column_max(m);
        // (126: the largest power of two that fp32 has both ways.  Sums of tiny values come times 2^-16 through LDS; a
        // limit below 116 would lose bits of their halves that the contraction had.)
        const int e = min(14 - __builtin_amdgcn_frexp_expf(m), 126);
        const float up = __builtin_ldexpf(1.0f, e);
        down[g] = shift[g % G] == KM_GRID_NOT_FINITE
                      ? __builtin_nanf("")
                      : weight * __builtin_ldexpf(1.0f, -e - KM_GRID_KS2 + (EXCHANGED ? KM_GRID_EXCHANGE : -shift[g % G] - KM_GRID_KS1));
#pragma unroll
        for (int ks = 0; ks < KSTEPS; ks++) {
            if (2 * ks < gw.tiles) {
                float gv[8];
                constexpr int LAST = MT - 1;
                const float4v none = {0.0f, 0.0f, 0.0f, 0.0f};
                grid_operand(acc[2 * ks][g], 2 * ks + 1 <= LAST ? acc[2 * ks + 1 <= LAST ? 2 * ks + 1 : LAST][g] : none, gv);
#pragma unroll
                for (int t = 0; t < 8; t++) {
                    gv[t] *= up * fac[t];
                }
                split_f16x8(gv, kc.one, &bhi[ks][g], &blo[ks][g]);
                __builtin_amdgcn_sched_barrier(0);  // one operand at a time (registers)
            }
        }
    }
    const float mid0 = (gw.g_lo + (float)(8 * kk) + 3.5f) * gw.h;
    const float mid_step = 32.0f * gw.h;
#pragma unroll 2
    for (int r = 0; r < groups; r++) {
        const int row = row0 + 16 * r;
        float y, rest, ca[4], sa[4];  // (rest: not zero in a block next to the origin)
        if (HELD) {
            const bool upper = r >= 4;
            const int first = 16 * (r & 3);
            y = __shfl(upper ? held->y[1] : held->y[0], first + li, 64);
            rest = __shfl(upper ? held->rest[1] : held->rest[0], first + li, 64);
            if (PHASE) {
                row_phases(upper ? held->cos[1] : held->cos[0], upper ? held->sin[1] : held->sin[0], first, ca, sa);
            }
        } else {
            const float x = w.x1[(long long)min(row + li, a.m - 1) * a.x1_s];
            y = x - gw.x_ref;
            rest = remainder_of(x, gw.x_ref, y);
            if (PHASE) {
                const float th = phase_rev(kc.f, x, gw.x_ref);
                row_phases(__builtin_amdgcn_cosf(th), __builtin_amdgcn_sinf(th), 0, ca, sa);
            }
        }
        float4v res[GE];
#pragma unroll
        for (int g = 0; g < GE; g++) {
            res[g] = (float4v){0.0f, 0.0f, 0.0f, 0.0f};
        }
#pragma unroll
        for (int ks = 0; ks < KSTEPS; ks++) {
            if (2 * ks >= gw.tiles) {
                break;
            }
            const float av = ((y - __builtin_fmaf((float)ks, mid_step, mid0)) + rest) * gw.s2;
            if (!__any(fabsf(av) - 3.5f * hz < KM_GRID_REACH)) {
                continue;
            }
            half2v h2[4], l2[4];
            const float rb = __builtin_fmaf(-av, av, (float)KM_GRID_KS2);
#pragma unroll
            for (int u = 0; u < 4; u++) {
                separable_pair_f16(av, rb, b2[2 * u], b2[2 * u + 1], kc.one, &h2[u], &l2[u]);
            }
            const half8v ahi = join_half2x4(h2);
            const half8v alo = join_half2x4(l2);
#pragma unroll
            for (int g = 0; g < GE; g++) {
                res[g] = __builtin_amdgcn_mfma_f32_16x16x32_f16(ahi, bhi[ks][g], res[g], 0, 0, 0);
                res[g] = __builtin_amdgcn_mfma_f32_16x16x32_f16(ahi, blo[ks][g], res[g], 0, 0, 0);
                res[g] = __builtin_amdgcn_mfma_f32_16x16x32_f16(alo, bhi[ks][g], res[g], 0, 0, 0);
            }
        }
        grid_store<KT, G>(a, w, ca, sa, res, down, row, kbase);
    }
}

// Operand groups (of 16 columns) of G groups of rhs columns, the grid form's largest window, and the columns tabulated
// at a time.
template <int KT, int G>
struct GridShape {
    static constexpr int PARTS = KT == KM_KERNEL_SPECTRAL ? 2 : 1;
    static constexpr int GE = G * PARTS;
    static_assert(GE <= 4, "what the registers hold");
    static constexpr int MT = GE >= 4 ? 4 : 5;
    static constexpr int CHUNK = G == 1 ? KM_GRID_CHUNK_ONE : KM_GRID_CHUNK;
};

// LDS of one item in floats: the wavefronts' tables, overlaid by the exchange of the sums, and the
// flags of each wavefront.
template <int GE, int MT, int W>
constexpr int grid_lds_floats() {
    return W == 1 ? KM_GRID_TABLE_FLOATS
                  : (W * KM_GRID_TABLE_FLOATS > W * MT * GE * 256 ? W * KM_GRID_TABLE_FLOATS : W * MT * GE * 256) +
                        W * (GE + 1);
}

// Whether the wavefronts of a workgroup share the steps of a range entry by entry as well (entry_item), for all rows each; else each
// has rows of its own and takes all steps (grid_entrywise), as one wavefront alone does.  Rows that are far apart (predictions)
// leave hardly any work but looking at the columns: rbf m = 9973, n = 50000, k = 3, 4 sets 27.1 -> 22.0 us.  With two groups of rhs
// columns the sums of all rows are more than three resident wavefronts' registers hold.
// Short ranges do not pay for the exchange of the sums: spectral n = 50000, k = 8, 2 sets at one point per unit (152 columns a row
// block) with two wavefronts 13.8 -> 14.2, n = 8000, k = 16 with eight 9.3 -> 8.0.
#define KM_SHARED_ENTRIES 1024 /* columns times wavefronts */
template <int G, int W, bool SHARES>
constexpr bool shares_entries() { return W > 1 && (G == 1 || SHARES); }

// The LDS of both forms.
template <int KT, int G, int W, bool SHARES = false>
constexpr int item_lds_floats() {
    using S = GridShape<KT, G>;
    constexpr int grid = grid_lds_floats<S::GE, S::MT, W>();
    constexpr int entries = shares_entries<G, W, SHARES>() ? entry_lds_floats(G, 8, W) : 0;
    return grid > entries ? grid : entries;
}

// One item in the grid form for rhs columns [kbase, kbase + 16 G), by W wavefronts of which this is
// number `wave`.  Returns whether it was done (the same in all W); if not, nothing was stored.
// W > 1: synchronises the workgroup three times.
template <int KT, int G, int MT, int W>
__device__ __forceinline__ bool grid_forward(const FwdArgs& a, float* lds, const WaveView& w, int row0, int kbase,
                                             int wave, const GridWindow& gw, const KernelConsts& kc,
                                             float (&xv)[GridShape<KT, G>::CHUNK / 64]) {
    constexpr int PARTS = KT == KM_KERNEL_SPECTRAL ? 2 : 1;
    constexpr int GE = G * PARTS;
    constexpr int R = 8 / W;  // groups of 16 rows of this wavefront
    const int lane = threadIdx.x & 63;
    const int li = lane & 15;

    int shift[G];
    float4v acc[MT][GE];
    bool fine = grid_columns<true, KT, G, MT, W>(vectors(a), lds + wave * KM_GRID_TABLE_FLOATS, w, kbase, wave, gw, kc, nullptr,
                                                 gw.tiles, xv, shift, acc);

    // The sums of all W wavefronts, added in their order.
    if (W > 1) {
        float4v* part = (float4v*)lds;
        unsigned* flags = (unsigned*)(lds + grid_lds_floats<GE, MT, W>() - W * (GE + 1));
#pragma unroll
        for (int g = 0; g < G; g++) {
            const float up = __builtin_ldexpf(1.0f, -shift[g] - KM_GRID_KS1 - KM_GRID_EXCHANGE);
#pragma unroll
            for (int m = 0; m < MT; m++) {
#pragma unroll
                for (int p = 0; p < PARTS; p++) {
                    acc[m][p * G + g] *= up;
                }
            }
        }
        __syncthreads();  // the exchange lies over the tables
        unsigned mine[G];
#pragma unroll
        for (int g = 0; g < G; g++) {
            mine[g] = (unsigned)__ballot(shift[g] == KM_GRID_NOT_FINITE) & 0xffff;
        }
        if (lane == 0) {
            flags[wave * (G + 1)] = fine ? 1 : 0;
#pragma unroll
            for (int g = 0; g < G; g++) {
                flags[wave * (G + 1) + 1 + g] = mine[g];
            }
        }
#pragma unroll
        for (int m = 0; m < MT; m++) {
            if (m < gw.tiles) {
#pragma unroll
                for (int g = 0; g < GE; g++) {
                    part[((wave * MT + m) * GE + g) * 64 + lane] = acc[m][g];
                }
            }
        }
        __syncthreads();
#pragma unroll
        for (int v = 0; v < W; v++) {
            fine = fine && __builtin_amdgcn_readfirstlane(flags[v * (G + 1)]) != 0;
#pragma unroll
            for (int g = 0; g < G; g++) {
                shift[g] = (flags[v * (G + 1) + 1 + g] >> li & 1) != 0 ? KM_GRID_NOT_FINITE : shift[g];
            }
        }
#pragma unroll
        for (int m = 0; m < MT; m++) {
            if (m < gw.tiles) {
#pragma unroll
                for (int g = 0; g < GE; g++) {
                    float4v sum = part[(m * GE + g) * 64 + lane];
#pragma unroll
                    for (int v = 1; v < W; v++) {
                        sum += part[((v * MT + m) * GE + g) * 64 + lane];
                    }
                    acc[m][g] = sum;
                }
            }
        }
        __syncthreads();  // all reads done: the area may become tables again
    }
    if (!fine) {
        return false;
    }

    grid_rows<KT, G, MT, (W > 1), false>(a, w, nullptr, row0 + 16 * R * wave, R, kbase, gw, kc, shift, acc);
    return true;
}

// The item entry by entry: each of the W wavefronts evaluates its rows, up to 64 at a time, against the
// whole range.  Every time the range is tabulated and its rhs operand formed anew, which is most of the work where
// few tiles are in reach; 128 rows at a time would not leave the registers for the other paths of one wavefront
// (37 spilled with one spectral operand group).  Measured, 32 -> 64 rows at a time, n = 1e5, 8 sets, lengthscale 0.5:
// spectral k = 16 at 1 / 3 / 5 points per unit 70.2 -> 59.8 / 72.4 -> 59.3 / 73.8 -> 63.2 us a call, k = 32 at 10
// 155 -> 136; rbf k = 16 at 3 56.9 -> 47.3, k = 64 at 10 251 -> 221; two wavefronts, spectral n = 1e5, 2 sets, at 2
// 30.4 -> 25.2.  Where one or two wavefronts spill (3 to 30 registers, most of them in front of this path's loops) the
// rows' share of the result is written to and read from scratch memory, a tenth to a quarter of it again: n = 1e6, 8 sets at
// 3 points per unit spectral k = 32 1024 us a call with 22 spilled, 998 with 16; rbf k = 32 741 with 25, 712 with 19.
// W > 1: synchronises the workgroup.  What bounds it then are round trips to memory, one after the other: the range's rhs
// values looked at by each wavefront, and 128 instead of 256 columns tabulated at a time, took rbf 9973 rows with 840
// columns each, k = 3, 4 sets 25.8 us instead of 20.7, n = 50000 at one point per unit, k = 8, 2 sets 13.8 instead of 12.5.
template <int KT, int G, int W>
__device__ __forceinline__ void grid_entrywise(const FwdArgs& a, float* lds, const WaveView& w, int row0, int kbase,
                                               int wave, const GridWindow& gw, const KernelConsts& kc) {
    constexpr int PARTS = KT == KM_KERNEL_SPECTRAL ? 2 : 1;
    constexpr int GE = G * PARTS;
    constexpr int R = W == 1 ? 4 : 8 / W;
    constexpr int PIECES = 8 / (W * R);
    static_assert(W == 1 || PIECES == 1, "one barrier");
    const int li = threadIdx.x & 15;
    GridWindow rows = gw;
    if (!is_finite(rows.x_ref)) {
        // Any row that is: the origin must not hand its value on to the other rows' phases.
        const BlockRows block = block_rows(w.x1, a.x1_s, row0, a.m);
        const unsigned long long in_a = __ballot(is_finite(block.xa)), in_b = __ballot(is_finite(block.xb));
        rows.x_ref = uniform(in_a != 0 ? __shfl(block.xa, __builtin_ctzll(in_a), 64)
                                       : (in_b != 0 ? __shfl(block.xb, __builtin_ctzll(in_b), 64) : 0.0f));
    }
    // The rhs values of the whole range, once for all rows: several wavefronts share its steps out and hand what they
    // find on behind their rows.
    int rhs_shift[G];
    unsigned* const flags = (unsigned*)(lds + grid_lds_floats<GE, GridShape<KT, G>::MT, W>() - W * (GE + 1));
    {
        float rhs_scale[G];
#pragma unroll
        for (int g = 0; g < G; g++) {
            rhs_shift[g] = 0;
            rhs_scale[g] = 0.0f;
        }
        const int width = w.range_end - w.range_start - 32 * wave;
        const int steps = width > 0 ? (width - 1) / (32 * W) + 1 : 0;
        look_at_steps<G>(vectors(a), w, kbase, w.range_start + 32 * wave, 32 * W, {steps < 64 ? (1ull << steps) - 1 : ~0ull, 64, steps},
                         rhs_lane<G>(vectors(a), kbase), rhs_shift, rhs_scale);
        if (W > 1) {
#pragma unroll
            for (int g = 0; g < G; g++) {
                const unsigned found = (unsigned)__ballot(rhs_shift[g] == KM_GRID_NOT_FINITE) & 0xffff;
                if ((threadIdx.x & 63) == 0) {
                    flags[wave * G + g] = found;
                }
            }
        }
    }
#pragma unroll 1
    for (int piece = 0; piece < PIECES; piece++) {
        // (anew for each piece: lanes' offsets formed with its strides in front of the loop would be spilled)
        const FwdArgs& f = PIECES > 1 ? fresh_args() : a;
        const int base = row0 + 16 * R * (wave * PIECES + piece);
        float xr[R];
#pragma unroll
        for (int r = 0; r < R; r++) {
            xr[r] = w.x1[(long long)min(base + 16 * r + li, f.m - 1) * f.x1_s];
        }
        // the columns within reach of these rows
        float lo = xr[0] - rows.x_ref, hi = lo;
        bool finite = true;
#pragma unroll
        for (int r = 0; r < R; r++) {
            const float y = xr[r] - rows.x_ref;
            lo = fminf(lo, y);
            hi = fmaxf(hi, y);
            finite = finite && fabsf(y) < 1e30f;
        }
        wave_min_max(&lo, &hi);
        finite = __all(finite);
        rows.reach = uniform(KM_GRID_REACH / kc.s);
        rows.col_lo = uniform(finite ? lo - rows.reach : -__builtin_inff());
        rows.col_hi = uniform(finite ? hi + rows.reach : __builtin_inff());
        constexpr int CHUNK = G == 1 && W == 1 ? KM_GRID_CHUNK_ONE : KM_GRID_CHUNK;
        float xv[CHUNK / 64];
        if (w.range_start < w.range_end) {
            grid_load(w.x2, f.x2_s, w.range_start, 1, w.range_end, xv);
        }
        int shift[G];
        float4v acc[R][GE];
        const bool fine = grid_columns<false, KT, G, R, 1, false, false, CHUNK>(vectors(f), lds + wave * KM_GRID_TABLE_FLOATS, w, kbase, 0, rows, kc, xr,
                                                           R, xv, shift, acc);
        if (W > 1) {
            __syncthreads();
#pragma unroll
            for (int v = 0; v < W; v++) {
#pragma unroll
                for (int g = 0; g < G; g++) {
                    rhs_shift[g] = (flags[v * G + g] >> li & 1) != 0 ? KM_GRID_NOT_FINITE : rhs_shift[g];
                }
            }
        }
        const float sigma = w.params[KernelTraits<KT>::SIGMA * f.params_s];
        float down[GE];
#pragma unroll
        for (int g = 0; g < GE; g++) {
            down[g] = fine && rhs_shift[g % G] != KM_GRID_NOT_FINITE ? __builtin_ldexpf(sigma, -shift[g % G] - KM_F16_KSCALE_LOG2)
                                                                     : __builtin_nanf("");
        }
#pragma unroll
        for (int r = 0; r < R; r++) {
            float ca[4], sa[4];
            if (PARTS == 2) {
                const float th = phase_rev(kc.f, xr[r], rows.x_ref);
                row_phases(__builtin_amdgcn_cosf(th), __builtin_amdgcn_sinf(th), 0, ca, sa);
            }
            grid_store<KT, G>(f, w, ca, sa, acc[r], down, base + 16 * r, kbase);
        }
    }
}

// One item by W wavefronts (this one is number `wave`) for rhs columns [kbase, kbase + 16 G): the grid form, or
// entry by entry.
template <int KT, int G, int W, bool SHARES = false>
__device__ __forceinline__ void grid_item(const FwdArgs& a, float* lds, const WaveView& w, int kbase, int wave) {
    using S = GridShape<KT, G>;
    const int row0 = w.row_block * KM_BLOCK_SIZE;
    // The rows are requested first, then the first columns (which wait for the range), then the
    // window is computed.
    const BlockRows rows = block_rows(w.x1, a.x1_s, row0, a.m);
    KernelConsts kc = make_consts<KT>(w.params, a.params_s, false);
    kc.s = uniform(kc.s);
    __builtin_amdgcn_sched_barrier(0);
    float xv[S::CHUNK / 64];
    if (32 * wave < w.range_end - w.range_start) {
        grid_load(w.x2, a.x2_s, w.range_start + 32 * wave, W, w.range_end, xv);
    }
    const GridWindow gw = grid_window<S::MT>(rows, kc);
    // (the same in every lane, and said so: the barriers inside depend on it)
    const bool grid = __builtin_amdgcn_readfirstlane(gw.ok && w.range_end - w.range_start >= KM_GRID_MIN_WIDTH) != 0;
    // (always so; without the condition the kernel came out slower, rbf n = 65536, k = 64 21.9 against 21.6 us a call)
    if (kbase < a.k) {
        if (!grid || !grid_forward<KT, G, S::MT, W>(a, lds, w, row0, kbase, wave, gw, kc, xv)) {
            if constexpr (shares_entries<G, W, SHARES>()) {
                if (SHARES || w.range_end - w.range_start >= KM_SHARED_ENTRIES / W) {
                    __syncthreads();  // (its tables lie elsewhere in LDS)
                    entry_item<KT, false, G, 8, W>(a, lds, w, row0, kbase, wave);
                    return;
                }
            }
            if constexpr (!SHARES) {
                grid_entrywise<KT, G, W>(a, lds, w, row0, kbase, wave, gw, kc);
            }
        }
    }
}

template <int KT, int G, int W>
__device__ __forceinline__ void grid_item(const FwdArgs& a, float* lds, long long item, int kbase, int wave) {
    int unused;
    grid_item<KT, G, W>(a, lds, wave_view<true>(a, item, 1, &unused), kbase, wave);
}

// ---------------------------------------------------------------------------------------
// Large launches: a workgroup of KM_GROUP wavefronts takes as many neighbouring row blocks of a batch item,
// whose ranges consist of the same columns for the most part, and contracts every column onto the grid once
// for all of them.
//
// The ends of the ranges cut the columns into cells, each of which lies inside or outside each range as a
// whole; a row block's sums are those of its cells, so the ranges are honoured exactly and nothing is
// subtracted.  The middle cell (the core: what all ranges have in common if they are long) is shared out to
// the wavefronts; of the others each wavefront takes one and half of the first or the last one.  The windows of
// these segments and of the row blocks lie on one grid and begin at multiples of four points, the unit in which
// sums are kept in LDS.
//
// Windows follow from the first and the last coordinate of a cell or row block.  Coordinates beyond these
// (unsorted ones, NaN), windows that are too wide for the accumulators or for LDS, and ranges too short to gain
// send the row blocks through grid_item, each by its wavefront.
//
// Measured (a call, queued), one row block per wavefront -> four per workgroup: spectral n = 1e5, k = 16, 8 sets
// at 10 points per unit 64.5 -> 61 us (entry by entry 103.8), at 40 115 -> 70; 4 sets at 160 182 -> 86; n = 1e6,
// k = 32, 8 sets 850 -> 778; rbf n = 1e5, k = 64, 8 sets 130 -> 114.  A row block of the first takes 3450 VALU
// instructions instead of 4450 and the SIMDs' VALU is busy 56 % of the cycles instead of 66: with two wavefronts
// resident on average, what bounds the narrow ranges is the latency of a workgroup's start, windows and exchange.
// Four: the sums of a group and their tables are then a third of the LDS for two operand groups, so that three
// workgroups of four wavefronts are resident, as many as the registers allow; with three row blocks for three or
// four wavefronts one wavefront waits, or less is shared.
// ---------------------------------------------------------------------------------------
#define KM_GROUP_CHUNK 128

// LDS in floats: a table for each wavefront, the cells' sums, and flags.
template <int KT, int G>
struct GroupShape {
    using S = GridShape<KT, G>;
    static constexpr int QUAD = S::GE * 64;  // four grid points' sums
    static constexpr int MAX_QUADS = 4 * S::MT;  // in a wavefront's accumulators
    static constexpr int QUADS = S::GE >= 4 ? 70 : (S::GE > 1 ? 87 : 100);
    static constexpr int TABLE = grid_table_floats(KM_GROUP_CHUNK);
    static constexpr int SUMS = KM_GROUP * TABLE;
    static constexpr int FLAGS = SUMS + QUADS * QUAD;
    static constexpr int FLOATS = FLAGS + 64;
    static_assert(FLOATS >= item_lds_floats<KT, G, KM_GROUP>() && FLOATS >= KM_GROUP * KM_GRID_TABLE_FLOATS, "grid_item's LDS");
    static_assert(KM_GROUP + (KM_GROUP_SEGMENTS + KM_GROUP) * G <= 64, "flags");
};

__device__ __forceinline__ int lane_value(int v, int lane) { return __builtin_amdgcn_readlane(v, lane); }
__device__ __forceinline__ float lane_value(float v, int lane) {
    return __uint_as_float(__builtin_amdgcn_readlane(__float_as_uint(v), lane));
}

// One segment of columns or one row block per lane.
struct GroupPlan {
    int start, end;         // columns
    int rows;               // row blocks whose range holds the segment, as bits
    float first, last;      // smallest and largest coordinate, relative to the origin
    float row_lo, row_hi;   // of these row blocks
    int quad, quads;        // window: first group of four points and their number
    int place;              // of the sums in LDS, in such groups
    bool cooperative;       // the core is in pieces (same in every lane)
    bool ok;                // the form applies (same in every lane)
};

// The segments: ranges into cells and pieces.  False if no range is long enough to gain.
__device__ __forceinline__ bool group_segments(const FwdArgs& a, const BatchOffsets& o, int row_block, int blocks, GroupPlan* p) {
    static_assert(KM_GROUP == 4, "eight ends of ranges");
    const int lane = threadIdx.x & 63;
    // The row blocks' starts in lanes 0 .. 3, ends in 4 .. 7 (as block_range, empty past the last row block).
    const int block = row_block + min(lane & 3, blocks - 1);
    const bool is_end = (lane & 4) != 0;
    const int mine = (is_end ? a.end + o.end : a.start + o.start)[block * (is_end ? a.end_s : a.start_s)];
    const int other = __shfl_xor(mine, 4, 64);
    const int end = max(min(is_end ? mine : other, a.n), 0);
    const int start = min(max(is_end ? other : mine, 0), end);
    const int length = (lane & 3) < blocks ? end - start : 0;
    if (!__any(lane < 4 && length >= KM_GRID_MIN_WIDTH)) {
        return false;
    }
    // (the ends of an empty range cut nothing)
    const int first_start = __builtin_amdgcn_readfirstlane(start);
    const int value = length > 0 || (lane & 3) == 0 ? (is_end ? start + length : start) : first_start;
    int ends[2 * KM_GROUP], rank = 0;
#pragma unroll
    for (int i = 0; i < 2 * KM_GROUP; i++) {
        ends[i] = lane_value(value, i);
        rank += ends[i] < value || (ends[i] == value && i < lane) ? 1 : 0;
    }
    const int cut = __builtin_amdgcn_ds_permute(4 * (lane < 8 ? rank : lane), value);
    int at[2 * KM_GROUP];
#pragma unroll
    for (int i = 0; i < 2 * KM_GROUP; i++) {
        at[i] = lane_value(cut, i);
    }
    const GroupCut c = group_cut(at);
    p->cooperative = c.shared;
    p->start = c.segment[0];
    p->end = c.segment[0];
#pragma unroll
    for (int i = 0; i < KM_GROUP_SEGMENTS; i++) {
        p->start = lane == i ? c.segment[i] : p->start;
        p->end = lane == i ? c.segment[i + 1] : p->end;
    }
    if (c.shared) {
#pragma unroll
        for (int i = 0; i < KM_GROUP; i++) {
            p->start = lane == KM_GROUP_PIECE + i ? c.piece[i] : p->start;
            p->end = lane == KM_GROUP_PIECE + i ? c.piece[i + 1] : p->end;
        }
    }
    p->rows = group_rows(ends, p->start, p->end);
    // (a gap between the ranges is a cell of none)
    p->end = p->rows != 0 ? p->end : p->start;
    return true;
}

// The windows and their places.
template <int KT, int G>
__device__ __forceinline__ void group_windows(const FwdArgs& a, const WaveView& w, int row0, const GridWindow& gw, GroupPlan* plan) {
    using P = GroupShape<KT, G>;
    const int lane = threadIdx.x & 63;
    GroupPlan& p = *plan;
    // First and last coordinates: of the columns, and of the row blocks.
    const bool is_row = lane >= KM_GROUP_ROW && lane < KM_GROUP_ROW + KM_GROUP;
    const float* ends = is_row ? w.x1 : w.x2;
    const long long stride = is_row ? a.x1_s : a.x2_s;
    int at0 = min(p.start, a.n - 1), at1 = min(max(p.end, 1), a.n) - 1;
    if (is_row) {
        at0 = min(row0 + (lane - KM_GROUP_ROW) * KM_BLOCK_SIZE, a.m - 1);
        at1 = min(at0 + KM_BLOCK_SIZE - 1, a.m - 1);
        p.rows = 1 << (lane - KM_GROUP_ROW);
    }
    const float y0 = ends[at0 * stride] - gw.x_ref;
    const float y1 = ends[at1 * stride] - gw.x_ref;
    p.first = fminf(y0, y1);
    p.last = fmaxf(y0, y1);
    p.row_lo = __builtin_inff();
    p.row_hi = -__builtin_inff();
#pragma unroll
    for (int r = 0; r < KM_GROUP; r++) {
        const float lo = lane_value(p.first, KM_GROUP_ROW + r), hi = lane_value(p.last, KM_GROUP_ROW + r);
        p.row_lo = (p.rows >> r & 1) != 0 ? fminf(p.row_lo, lo) : p.row_lo;
        p.row_hi = (p.rows >> r & 1) != 0 ? fmaxf(p.row_hi, hi) : p.row_hi;
    }
    // Windows: the grid points within reach of both the columns and the row blocks.
    const float per_quad = 0.25f * __builtin_amdgcn_rcpf(gw.h);
    const float lo = floorf((fmaxf(p.first, p.row_lo) - gw.reach) * per_quad);
    const float hi = floorf((fminf(p.last, p.row_hi) + gw.reach) * per_quad + 0.25f) + 1.0f;
    const float count = hi - lo;  // (not positive: out of reach)
    const bool used = is_row || p.start < p.end;
    // (a core in pieces is in nobody's accumulators as a whole)
    const float limit = p.cooperative && lane == KM_GROUP_CORE ? (float)P::QUADS : (float)P::MAX_QUADS;
    const bool bad = !(fabsf(y0) + fabsf(y1) < 1e30f) || !(count <= limit) || (count > 0.0f && !(fabsf(lo) < 1000.0f));
    // (the pieces of a core add to the core's window, which its first and last coordinate make)
    const float core_first = lane_value(p.first, KM_GROUP_CORE), core_last = lane_value(p.last, KM_GROUP_CORE);
    const bool beyond = p.cooperative && lane >= KM_GROUP_PIECE && lane < KM_GROUP_PIECE + KM_GROUP &&
                        (p.first < core_first || p.last > core_last);
    p.ok = gw.h > 1e-30f && gw.h < 1e30f && !__any(used && (bad || beyond));
    const bool reached = p.ok && used && count > 0.0f;
    p.quad = reached ? (int)lo : 0;
    p.quads = reached ? (int)count : 0;
    // Places: the core's, then the edges', where before them the pieces of the core lie.
    p.place = 0;
    const int core = lane_value(p.quads, KM_GROUP_CORE);
    int edges = core, pieces = core;
#pragma unroll
    for (int c = 0; c < KM_GROUP_SEGMENTS; c++) {
        if (c != KM_GROUP_CORE) {
            p.place = lane == c ? edges : p.place;
            edges += lane_value(p.quads, c);
        }
    }
    if (p.cooperative) {
#pragma unroll
        for (int i = 0; i < KM_GROUP; i++) {
            p.place = lane == KM_GROUP_PIECE + i ? pieces : p.place;
            pieces += lane_value(p.quads, KM_GROUP_PIECE + i);
        }
    }
    p.ok = p.ok && max(edges, pieces) <= P::QUADS;
}

// The window of one of the segments or row blocks.
__device__ __forceinline__ GridWindow group_window(const GridWindow& common, const GroupPlan& p, int lane) {
    GridWindow gw = common;
    const float cr = gw.reach * (KM_GRID_COLUMN_REACH / KM_GRID_REACH);
    gw.g_lo = uniform(4.0f * (float)lane_value(p.quad, lane));
    gw.tiles = (lane_value(p.quads, lane) + 3) / 4;
    gw.col_lo = uniform(lane_value(p.row_lo, lane) - cr);
    gw.col_hi = uniform(lane_value(p.row_hi, lane) + cr);
    gw.first = lane_value(p.first, lane);
    gw.last = lane_value(p.last, lane);
    grid_tiles(&gw, lane_value(p.row_lo, lane), lane_value(p.row_hi, lane), KM_GRID_MIDDLE / KM_GRID_REACH * gw.reach);
    return gw;
}

// The sums of a segment of columns onto its window, into LDS; bad[]: the rhs columns of each group with a value
// that is not finite, as bits.
template <int KT, int G>
__device__ __forceinline__ bool group_columns(const FwdArgs& a, const WaveView& w, const GroupPlan& p, int lane_of, int kbase,
                                              const GridWindow& common, const KernelConsts& kc, float* tab, float* sums,
                                              float (&xv)[KM_GROUP_CHUNK / 64], unsigned (&bad)[G]) {
    using S = GridShape<KT, G>;
    constexpr int GE = S::GE, MT = S::MT;
    const int lane = threadIdx.x & 63;
    const int kk = lane >> 4;
    WaveView seg = w;
    seg.range_start = lane_value(p.start, lane_of);
    seg.range_end = lane_value(p.end, lane_of);
    const GridWindow gw = group_window(common, p, lane_of);
    int shift[G];
    float4v acc[MT][GE];
    const bool fine = grid_columns<true, KT, G, MT, 1, false, false, KM_GROUP_CHUNK>(vectors(a), tab, seg, kbase, 0, gw, kc, nullptr,
                                                                                     gw.tiles, xv, shift, acc);
    const int quads = lane_value(p.quads, lane_of);
    float4v* out = (float4v*)(sums + lane_value(p.place, lane_of) * GroupShape<KT, G>::QUAD) + (lane & 15);
#pragma unroll
    for (int g = 0; g < G; g++) {
        bad[g] = (unsigned)__ballot(shift[g] == KM_GRID_NOT_FINITE) & 0xffff;
        const float up = __builtin_ldexpf(1.0f, -shift[g] - KM_GRID_KS1 - KM_GRID_EXCHANGE);
#pragma unroll
        for (int m = 0; m < MT; m++) {
            if (4 * m + kk < quads) {
#pragma unroll
                for (int part = 0; part < GE / G; part++) {
                    out[((4 * m + kk) * GE + part * G + g) * 16] = acc[m][part * G + g] * up;
                }
            }
        }
    }
    return fine;
}

// The first coordinates of a segment.
__device__ __forceinline__ void group_load(const FwdArgs& a, const WaveView& w, const GroupPlan& p, int segment,
                                           float (&xv)[KM_GROUP_CHUNK / 64]) {
    // (an empty one's lie in the matrix too)
    const int start = min(lane_value(p.start, segment), a.n - 1);
    grid_load(w.x2, a.x2_s, start, 1, max(lane_value(p.end, segment), start + 1), xv);
}

// The segments of a wavefront in their order: its piece of a shared core, a cell, half of a core that is
// not shared, half of the first or last cell.  -1: none.
__device__ __forceinline__ int group_segment(int stage, int wave, bool cooperative) {
    static_assert(KM_GROUP == 4, "the lanes of the plan");
    const bool outer = wave == 0 || wave == 3;
    switch (stage) {
        case 0: return cooperative ? KM_GROUP_PIECE + wave : -1;
        case 1: return wave < 2 ? wave + 2 : wave + 4;
        case 2: return outer && !cooperative ? (wave == 0 ? KM_GROUP_CORE : KM_GROUP_CORE + 1) : -1;
        case 3: return wave < 2 ? wave : (wave == 2 ? 8 : 9);
        default: return -1;
    }
}

// The row blocks of a workgroup for rhs columns [kbase, kbase + 16 G), from the coordinates xv of the first
// segment on; false (in all wavefronts) if the form does not suit them.  Synchronises the workgroup.
template <int KT, int G>
__device__ __forceinline__ bool group_forward(const FwdArgs& a, float* lds, const WaveView& w, const BlockRows& rows,
                                              const GroupPlan& p, int row0, int kbase, int wave, const GridWindow& common,
                                              const KernelConsts& kc, int first_stage, float (&xv)[KM_GROUP_CHUNK / 64]) {
    using P = GroupShape<KT, G>;
    using S = GridShape<KT, G>;
    constexpr int GE = S::GE, MT = S::MT;
    const int lane = threadIdx.x & 63;
    const int li = lane & 15;
    const int kk = lane >> 4;
    float* const tab = lds + wave * P::TABLE;
    float* const sums = lds + P::SUMS;
    unsigned* const flags = (unsigned*)(lds + P::FLAGS);
    unsigned* const bad_segments = flags + KM_GROUP;
    bool fine = true;
    const int my_row0 = row0 + wave * KM_BLOCK_SIZE;
    if (my_row0 < a.m) {
        const float first = lane_value(p.first, KM_GROUP_ROW + wave), last = lane_value(p.last, KM_GROUP_ROW + wave);
        const float ya = rows.xa - common.x_ref, yb = rows.xb - common.x_ref;
        fine = __all(ya >= first && ya <= last && yb >= first && yb <= last);
    }
#pragma unroll 1
    for (int stage = 0; stage < 4; stage++) {
        if (stage == 1 && p.cooperative) {
            __syncthreads();
            // The pieces' sums, added in their order.
            const int quads = lane_value(p.quads, KM_GROUP_CORE);
            for (int q = 4 * wave + kk; q < quads; q += 4 * KM_GROUP) {
                float4v sum[GE];
#pragma unroll
                for (int g = 0; g < GE; g++) {
                    sum[g] = (float4v){0.0f, 0.0f, 0.0f, 0.0f};
                }
#pragma unroll
                for (int i = 0; i < KM_GROUP; i++) {
                    const int at = q + lane_value(p.quad, KM_GROUP_CORE) - lane_value(p.quad, KM_GROUP_PIECE + i);
                    if (at >= 0 && at < lane_value(p.quads, KM_GROUP_PIECE + i)) {
                        const float4v* part = (const float4v*)(sums + lane_value(p.place, KM_GROUP_PIECE + i) * P::QUAD) + li;
#pragma unroll
                        for (int g = 0; g < GE; g++) {
                            sum[g] += part[(at * GE + g) * 16];
                        }
                    }
                }
#pragma unroll
                for (int g = 0; g < GE; g++) {
                    ((float4v*)sums)[(q * GE + g) * 16 + li] = sum[g];
                }
            }
            __syncthreads();
        }
        const int segment = group_segment(stage, wave, p.cooperative);
        if (segment < 0) {
            continue;
        }
        unsigned bad[G];
#pragma unroll
        for (int g = 0; g < G; g++) {
            bad[g] = 0;
        }
        if (lane_value(p.start, segment) < lane_value(p.end, segment)) {
            if (stage != first_stage) {
                group_load(a, w, p, segment, xv);
            }
            fine = group_columns<KT, G>(a, w, p, segment, kbase, common, kc, tab, sums, xv, bad) && fine;
        }
        if (lane == 0) {
            unsigned* to = bad_segments + segment * G;
#pragma unroll
            for (int g = 0; g < G; g++) {
                to[g] = bad[g];
            }
        }
    }
    if (lane == 0) {
        flags[wave] = fine ? 1 : 0;
    }
    __syncthreads();
#pragma unroll
    for (int v = 0; v < KM_GROUP; v++) {
        fine = fine && __builtin_amdgcn_readfirstlane(flags[v]) != 0;
    }
    if (!fine || my_row0 >= a.m) {
        return fine;
    }
    const GridWindow gw = group_window(common, p, KM_GROUP_ROW + wave);
    const int quad = lane_value(p.quad, KM_GROUP_ROW + wave) + kk;
    float4v acc[MT][GE];
    unsigned bad[G];
#pragma unroll
    for (int m = 0; m < MT; m++) {
#pragma unroll
        for (int g = 0; g < GE; g++) {
            acc[m][g] = (float4v){0.0f, 0.0f, 0.0f, 0.0f};
        }
    }
#pragma unroll
    for (int g = 0; g < G; g++) {
        bad[g] = 0;
    }
#pragma unroll 1
    for (int c = 0; c < KM_GROUP_SEGMENTS; c++) {
        if ((lane_value(p.rows, c) >> wave & 1) == 0) {
            continue;
        }
        const int quads = lane_value(p.quads, c);
        const int offset = quad - lane_value(p.quad, c);
        const float4v* part = (const float4v*)(sums + lane_value(p.place, c) * P::QUAD) + li;
        // (kept as register quadruples, see grid_columns)
#pragma unroll
        for (int m = 0; m < MT; m++) {
#pragma unroll
            for (int g = 0; g < GE; g++) {
                asm volatile("" : "+v"(acc[m][g]));
            }
        }
#pragma unroll
        for (int m = 0; m < MT; m++) {
            if (m >= gw.tiles) {
                break;
            }
            const int at = offset + 4 * m;
            if (at >= 0 && at < quads) {
#pragma unroll
                for (int g = 0; g < GE; g++) {
                    acc[m][g] += part[(at * GE + g) * 16];
                }
            }
        }
#pragma unroll
        for (int g = 0; g < G; g++) {
            if (c == KM_GROUP_CORE && p.cooperative) {
#pragma unroll
                for (int v = 0; v < KM_GROUP; v++) {
                    bad[g] |= bad_segments[(KM_GROUP_PIECE + v) * G + g];
                }
            } else {
                bad[g] |= bad_segments[c * G + g];
            }
        }
    }
    int shift[G];
#pragma unroll
    for (int g = 0; g < G; g++) {
        shift[g] = (bad[g] >> li & 1) != 0 ? KM_GRID_NOT_FINITE : 0;
    }
    const HeldRows held = hold_rows<KT>(rows, common.x_ref, kc);
    grid_rows<KT, G, MT, true, true>(a, w, &held, my_row0, KM_BLOCK_SIZE / 16, kbase, gw, kc, shift, acc);
    return true;
}

template <int KT, int G>
__device__ __forceinline__ void group_item(const FwdArgs& a, float* lds, unsigned item, int kbase, int wave) {
    WaveView w;
    const unsigned batches = (unsigned)a.num_batches;
    const unsigned group = item / batches;
    w.b = spread_batch(item - group * batches, group, batches);
    w.row_block = (int)group * KM_GROUP;
    const int row0 = w.row_block * KM_BLOCK_SIZE;
    const BatchOffsets o = batch_offsets(a, w.b);
    w.x1 = a.x1 + o.x1;
    w.x2 = a.x2 + o.x2;
    w.rhs = a.rhs + o.rhs;
    w.params = a.params + o.params;
    w.range_start = 0;
    w.range_end = 0;
    const int blocks = (a.m - 1) / KM_BLOCK_SIZE + 1 - w.row_block;  // in this group, if fewer than KM_GROUP
    // (rows past the last one repeat it)
    const BlockRows rows = block_rows(w.x1, a.x1_s, row0 + wave * KM_BLOCK_SIZE, a.m);
    GridWindow gw;
    gw.ok = true;
    gw.x_ref = w.x1[(long long)min(row0 + KM_GROUP * KM_BLOCK_SIZE / 2, a.m - 1) * a.x1_s];
    KernelConsts kc = make_consts<KT>(w.params, a.params_s, false);
    GroupPlan p;
    bool grouped = group_segments(a, o, w.row_block, blocks, &p);
    if (grouped) {
        // The first columns are requested together with the ends of all segments, which the windows need.
        float xv[KM_GROUP_CHUNK / 64];
        const int first = p.cooperative ? 0 : 1;
        group_load(a, w, p, group_segment(first, wave, p.cooperative), xv);
        kc.s = uniform(kc.s);
        gw.x_ref = uniform(gw.x_ref);
        gw.s2 = uniform(kc.s * 1.41421356237309504880f);
        const float inv = __builtin_amdgcn_rcpf(gw.s2);
        gw.h = uniform(__uint_as_float(__float_as_uint(KM_GRID_STEP * inv) & 0xfffff000u));
        gw.reach = uniform(KM_GRID_REACH * inv);
        group_windows<KT, G>(a, w, row0, gw, &p);
        grouped = __builtin_amdgcn_readfirstlane(p.ok) != 0 &&
                  group_forward<KT, G>(a, lds, w, rows, p, row0, kbase, wave, gw, kc, first, xv);
        if (!grouped) {
            __syncthreads();  // (tables of the row blocks below lie over the flags' and sums' place)
        }
    }
    if (!grouped && wave < blocks) {
        grid_item<KT, G, 1>(fresh_args(), lds + wave * KM_GRID_TABLE_FLOATS, (long long)(w.row_block + wave) * a.num_batches + w.b, kbase, 0);
    }
}

// The rhs columns of a launch's workgroup.  64 spectral columns are more than the registers hold: two workgroups
// take half each.  An XCD takes the two halves in turn, RUN workgroups at a time (half of what it holds): both write to
// a row of the result before its place leaves the caches, but those that run together read the same half of rhs.
// Measured, two passes of one workgroup (50 to 140 registers spilled) -> two workgroups, a call, cutoff of 6 lengthscales:
// n = 1e5, k = 64, 2 sets at 10 / 40 points per unit 95.3 -> 63.0 / 157 -> 72.7 us, 8 sets 215 -> 188 / 239 -> 216; k = 40
// 2 sets 94.5 -> 61.3; n = 20000, one set 30.5 -> 15.3; k = 64, 8 sets, at 10 points per unit / at 3, all row blocks entry by
// entry: n = 3e5 583 -> 547 / 756 -> 652, 1e6 1719 -> 1638 / 2563 -> 2118.  Neighbours in turn (RUN 1): 532 / 780 and 1585 /
// 2544; all first halves before all second ones 575 / 724 and 1721 / 2370; RUN 8 550 / 783, 64 549 / 645.
template <int KT, int G>
struct GridColumns {
    static constexpr int HALVES = KT == KM_KERNEL_SPECTRAL && G == 4 ? 2 : 1;
    static constexpr int GROUPS = G / HALVES;  // of a workgroup
    static constexpr unsigned RUN = 32;
    using Shape = GridShape<KT, GROUPS>;
    static constexpr int RESIDENT = Shape::GE >= 4 ? 2 : (Shape::GE > 1 ? 3 : 4);
    unsigned block;  // number of the workgroup among those of its half
    int kbase;
    bool beyond;     // no columns, or no work left for the XCD
    // per_xcd: workgroups of an XCD, of one half
    __device__ __forceinline__ GridColumns(const FwdArgs& a, long long per_xcd) {
        if constexpr (HALVES == 1) {
            block = blockIdx.x;
            kbase = blockIdx.y * G * 16;
            beyond = false;
        } else {
            const unsigned slot = blockIdx.x / KM_NUM_XCD;
            const unsigned own = slot / (HALVES * RUN) * RUN + slot % RUN;
            block = blockIdx.x % KM_NUM_XCD + own * KM_NUM_XCD;
            kbase = ((int)blockIdx.y * HALVES + (int)(slot / RUN % HALVES)) * GROUPS * 16;
            beyond = kbase >= a.k || own >= per_xcd;
        }
    }
    static unsigned workgroups(long long per_xcd) {
        return (unsigned)((HALVES == 1 ? per_xcd : (per_xcd + RUN - 1) / RUN * RUN * HALVES) * KM_NUM_XCD);
    }
};

// W: wavefronts per row block, or 1: fewer than one, the workgroup for several row blocks.  (Eight of one are launched where
// there is a workgroup per compute unit at most.)
template <int KT, int G, int W>
__global__ void __launch_bounds__(64 * (W == 1 ? KM_GROUP : W), (W == 8 ? 2 : GridColumns<KT, G>::RESIDENT)) fwd_grid(const FwdArgs a) {
    extern __shared__ float lds[];
    using C = GridColumns<KT, G>;
    const C c(a, a.items_per_xcd);
    const long long item = xcd_item(c.block, a.items_per_xcd);
    if (item >= a.total_items || c.beyond) {
        return;
    }
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    if constexpr (W == 1) {
        group_item<KT, C::GROUPS>(a, lds, (unsigned)item, c.kbase, wave);
    } else {
        grid_item<KT, C::GROUPS, W>(a, lds, item, c.kbase, wave);
    }
}

// The grouped form with a tail: the last `tail_items` groups of every XCD come last and with a workgroup for
// each of their row blocks, so that short pieces fill the SIMDs that would otherwise idle while others finish a
// last group.
template <int KT, int G>
__global__ void __launch_bounds__(64 * KM_GROUP, (GridColumns<KT, G>::RESIDENT)) fwd_grid_grouped(const FwdArgs a) {
    extern __shared__ float lds[];
    using C = GridColumns<KT, G>;
    const C c(a, a.items_per_xcd + (KM_GROUP - 1) * a.tail_items);
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const unsigned xcd = c.block % KM_NUM_XCD;
    const unsigned slot = c.block / KM_NUM_XCD;
    const unsigned first = xcd * (unsigned)a.items_per_xcd;
    const unsigned main_groups = (unsigned)a.items_per_xcd - (unsigned)a.tail_items;
    if (c.beyond) {
        return;
    }
    if (slot < main_groups) {
        if (first + slot < (unsigned)a.total_items) {
            group_item<KT, C::GROUPS>(a, lds, first + slot, c.kbase, wave);
        }
        return;
    }
    const unsigned item = first + main_groups + (slot - main_groups) / KM_GROUP;
    const unsigned batches = (unsigned)a.num_batches;
    const unsigned group = item / batches;
    const unsigned row_block = group * KM_GROUP + (slot - main_groups) % KM_GROUP;
    if (item < (unsigned)a.total_items && (long long)row_block * KM_BLOCK_SIZE < a.m) {
        const unsigned b = spread_batch(item - group * batches, group, batches);
        grid_item<KT, C::GROUPS, KM_GROUP>(fresh_args(), lds, (long long)row_block * batches + b, c.kbase, wave);
    }
}

// Few row blocks: their ranges in shares (launch_sum_shares adds up).
template <int KT, int G>
__global__ void __launch_bounds__(512, (G > 1 ? 2 : GridColumns<KT, G>::RESIDENT)) fwd_grid_shares(const FwdArgs a) {
    extern __shared__ float lds[];
    FwdArgs f = a;
    WaveView w;
    if (!share_view(a, &w, &f.out)) {
        return;
    }
    grid_item<KT, G, 8, true>(f, lds, w, blockIdx.y * G * 16, __builtin_amdgcn_readfirstlane(threadIdx.x >> 6));
}

template <int KT, int G>
static hipError_t launch_grid_shares(FwdArgs& a, const MatmulPlan& plan, unsigned grid_y, hipStream_t stream) {
    a.stream_out = 0;  // (read again)
    a.chunks_per_block = plan.shares;
    a.total_items = ((long long)a.m + KM_BLOCK_SIZE - 1) / KM_BLOCK_SIZE * a.num_batches;
    hipLaunchKernelGGL((fwd_grid_shares<KT, G>), dim3((unsigned)(a.total_items * plan.shares), grid_y, 1), dim3(512, 1, 1),
                       (sizeof(float) * item_lds_floats<KT, G, 8, true>()), stream, a);
    const hipError_t err = hipGetLastError();
    return err == hipSuccess ? launch_sum_shares(a, stream) : err;
}

template <int KT, int G, int W>
static hipError_t launch_grid_as(const FwdArgs& a, dim3 grid, hipStream_t stream) {
    hipLaunchKernelGGL((fwd_grid<KT, G, W>), grid, dim3(64 * W, 1, 1),
                       (sizeof(float) * item_lds_floats<KT, GridColumns<KT, G>::GROUPS, W>()), stream, a);
    return hipGetLastError();
}

template <int KT, int G>
static hipError_t launch_grid_w(FwdArgs& a, const MatmulPlan& plan, unsigned grid_y, hipStream_t stream) {
    using C = GridColumns<KT, G>;
    const long long row_blocks = ((long long)a.m + KM_BLOCK_SIZE - 1) / KM_BLOCK_SIZE;
    if (plan.col_splits == 1) {
        const long long groups = (row_blocks + KM_GROUP - 1) / KM_GROUP;
        a.total_items = groups * a.num_batches;
        a.items_per_xcd = (a.total_items + KM_NUM_XCD - 1) / KM_NUM_XCD;
        if (plan.group_tail <= 0) {
            hipLaunchKernelGGL((fwd_grid<KT, G, 1>), dim3(C::workgroups(a.items_per_xcd), grid_y, 1),
                               dim3(64 * KM_GROUP, 1, 1), (sizeof(float) * GroupShape<KT, C::GROUPS>::FLOATS), stream, a);
            return hipGetLastError();
        }
        const long long tail = (plan.group_tail + KM_GROUP - 1) / KM_GROUP;
        a.tail_items = (int)(tail < a.items_per_xcd ? tail : a.items_per_xcd);
        const dim3 grid(C::workgroups(a.items_per_xcd + (KM_GROUP - 1) * a.tail_items), grid_y, 1);
        hipLaunchKernelGGL((fwd_grid_grouped<KT, G>), grid, dim3(64 * KM_GROUP, 1, 1),
                           (sizeof(float) * GroupShape<KT, C::GROUPS>::FLOATS), stream, a);
        return hipGetLastError();
    }
    a.total_items = row_blocks * a.num_batches;
    a.items_per_xcd = (a.total_items + KM_NUM_XCD - 1) / KM_NUM_XCD;
    const dim3 grid(C::workgroups(a.items_per_xcd), grid_y, 1);
    switch (plan.col_splits) {
        case 2: return launch_grid_as<KT, G, 2>(a, grid, stream);
        case 4: return launch_grid_as<KT, G, 4>(a, grid, stream);
        default: return launch_grid_as<KT, G, 8>(a, grid, stream);
    }
}

template <int KT>
static hipError_t launch_grid_g(FwdArgs& a, const MatmulPlan& plan, unsigned grid_y, hipStream_t stream) {
    switch (plan.k_chunk / 16) {
        case 1: return launch_grid_w<KT, 1>(a, plan, grid_y, stream);
        case 2: return launch_grid_w<KT, 2>(a, plan, grid_y, stream);
        default: return launch_grid_w<KT, 4>(a, plan, grid_y, stream);
    }
}

hipError_t launch_matmul_grid(const MatmulProblem& p, const MatmulPlan& plan, hipStream_t stream) {
    FwdArgs a;
    fill_fwd_args(p, &a);
    a.chunks_per_block = 1;
    const unsigned grid_y = (unsigned)((p.k + plan.k_chunk - 1) / plan.k_chunk);
    if (plan.shares > 1) {
        if (p.kernel_type == KM_KERNEL_SPECTRAL) {
            return plan.k_chunk == 16 ? launch_grid_shares<KM_KERNEL_SPECTRAL, 1>(a, plan, grid_y, stream)
                                      : launch_grid_shares<KM_KERNEL_SPECTRAL, 2>(a, plan, grid_y, stream);
        }
        return plan.k_chunk == 16 ? launch_grid_shares<KM_KERNEL_RBF, 1>(a, plan, grid_y, stream)
                                  : launch_grid_shares<KM_KERNEL_RBF, 2>(a, plan, grid_y, stream);
    }
    if (p.kernel_type == KM_KERNEL_SPECTRAL) {
        return launch_grid_g<KM_KERNEL_SPECTRAL>(a, plan, grid_y, stream);
    }
    return launch_grid_g<KM_KERNEL_RBF>(a, plan, grid_y, stream);
}

}  // namespace km
