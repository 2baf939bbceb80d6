// Forward operator in the grid form (km_grid.h): rbf and spectral kernels, any number of rhs
// columns.  A row block of 128 rows is one item, worked on by W wavefronts:
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
// Measured against the entry-wise kernels (a call, queued): spectral n = 1e5, k = 16, 8 sets 103.8 -> 64.8 us,
// n = 1e6, k = 32 1085 -> 891, rbf n = 65536, k = 64 43.6 -> 21.8.  The large ones are bound by VALU issue (66
// and 70 % of the cycles; exponentials, fma and fp16 roundings are a third of it, the rest rhs scaling,
// maxima, tables, moves and offsets), the small ones by the latency of one wavefront's steps.
#include "km_batch.h"
#include "km_common.h"
#include "km_fwd.h"
#include "km_grid.h"
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

// A group of 16 rows from its accumulators (scaled back by down[]): the two parts of the
// phase-split form combined, and the masked store.
template <int KT, int G>
__device__ __forceinline__ void grid_store(const FwdArgs& a, const WaveView& w, const KernelConsts& kc, float x,
                                           float x_ref, const float4v* res, const float* down, int row, int kbase) {
    constexpr bool PHASE = KT == KM_KERNEL_SPECTRAL;
    const int lane = threadIdx.x & 63;
    const int li = lane & 15;
    const int kk = lane >> 4;
    float ca[4], sa[4];
    if (PHASE) {
        // cos A / sin A of the row this lane holds, fetched into the accumulator layout.
        const float th = phase_rev(kc.f, x, x_ref);
        const float ca_own = __builtin_amdgcn_cosf(th);
        const float sa_own = __builtin_amdgcn_sinf(th);
#pragma unroll
        for (int v = 0; v < 4; v++) {
            ca[v] = __shfl(ca_own, 4 * kk + v, 64);
            sa[v] = __shfl(sa_own, 4 * kk + v, 64);
        }
    }
    float* __restrict__ out = a.out + w.b * (long long)a.m * a.k;
#pragma unroll
    for (int g = 0; g < G; g++) {
        const int c = kbase + 16 * g + li;
#pragma unroll
        for (int v = 0; v < 4; v++) {
            const float value = PHASE ? ca[v] * (res[g][v] * down[g]) + sa[v] * (res[G + g][v] * down[G + g])
                                      : res[g][v] * down[g];
            const int r = row + 4 * kk + v;
            if (r < a.m && c < a.k) {
                out[(long long)r * a.k + c] = value;
            }
        }
    }
}

// LDS of one item in floats: the wavefronts' tables, overlaid by the exchange of the sums, and the
// flags of each wavefront.
template <int GE, int MT, int W>
constexpr int grid_lds_floats() {
    return W == 1 ? KM_GRID_TABLE_FLOATS
                  : (W * KM_GRID_TABLE_FLOATS > W * MT * GE * 256 ? W * KM_GRID_TABLE_FLOATS : W * MT * GE * 256) +
                        W * (GE + 1);
}

// One item in the grid form for rhs columns [kbase, kbase + 16 G), by W wavefronts of which this is
// number `wave`.  Returns whether it was done (the same in all W); if not, nothing was stored.
// W > 1: synchronises the workgroup three times.
template <int KT, int G, int MT, int W>
__device__ __forceinline__ bool grid_forward(const FwdArgs& a, float* lds, const WaveView& w, int row0, int kbase,
                                             int wave, const GridWindow& gw, const KernelConsts& kc,
                                             float (&xv)[KM_GRID_CHUNK / 64]) {
    constexpr int PARTS = KT == KM_KERNEL_SPECTRAL ? 2 : 1;
    constexpr int GE = G * PARTS;
    constexpr int R = 8 / W;  // groups of 16 rows of this wavefront
    const int lane = threadIdx.x & 63;
    const int li = lane & 15;
    const int kk = lane >> 4;

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

    // Grid -> rows.  One power-of-two scale per column over the whole window; the operands of all
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
        const int e = min(14 - __builtin_amdgcn_frexp_expf(m), 100);
        const float up = __builtin_ldexpf(1.0f, e);
        down[g] = shift[g % G] == KM_GRID_NOT_FINITE
                      ? __builtin_nanf("")
                      : weight * __builtin_ldexpf(1.0f, -e - KM_GRID_KS2 + (W > 1 ? KM_GRID_EXCHANGE : -shift[g % G] - KM_GRID_KS1));
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
    for (int r = 0; r < R; r++) {
        const int row = row0 + 16 * (wave * R + r);
        const float x = w.x1[(long long)min(row + li, a.m - 1) * a.x1_s];
        const float y = x - gw.x_ref;
        const float rest = remainder_of(x, gw.x_ref, y);  // (not zero in a block next to the origin)
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
        grid_store<KT, G>(a, w, kc, x, gw.x_ref, res, down, row, kbase);
    }
    return true;
}

// The item entry by entry: each of the W wavefronts evaluates its rows, 32 at a time, against the
// whole range.
template <int KT, int G, int W>
__device__ __forceinline__ void grid_entrywise(const FwdArgs& a, float* lds, const WaveView& w, int row0, int kbase,
                                               int wave, const GridWindow& gw, const KernelConsts& kc) {
    constexpr int PARTS = KT == KM_KERNEL_SPECTRAL ? 2 : 1;
    constexpr int GE = G * PARTS;
    constexpr int R = W == 8 ? 1 : 2;
    constexpr int PIECES = 8 / (W * R);
    const int li = threadIdx.x & 15;
    GridWindow rows = gw;
    if (!is_finite(rows.x_ref)) {
        // Any row that is: the origin must not hand its value on to the other rows' phases.
        const BlockRows block = block_rows(w.x1, a.x1_s, row0, a.m);
        const unsigned long long in_a = __ballot(is_finite(block.xa)), in_b = __ballot(is_finite(block.xb));
        rows.x_ref = uniform(in_a != 0 ? __shfl(block.xa, __builtin_ctzll(in_a), 64)
                                       : (in_b != 0 ? __shfl(block.xb, __builtin_ctzll(in_b), 64) : 0.0f));
    }
    // The rhs values of the whole range, once for all rows.
    int rhs_shift[G];
    {
        float rhs_scale[G];
#pragma unroll
        for (int g = 0; g < G; g++) {
            rhs_shift[g] = 0;
            rhs_scale[g] = 0.0f;
        }
        const int width = w.range_end - w.range_start;
        const int steps = width > 0 ? (width - 1) / 32 + 1 : 0;
        look_at_steps<G>(vectors(a), w, kbase, w.range_start, 32, {steps < 64 ? (1ull << steps) - 1 : ~0ull, 64, steps},
                         rhs_lane<G>(vectors(a), kbase), rhs_shift, rhs_scale);
    }
#pragma unroll 1
    for (int piece = 0; piece < PIECES; piece++) {
        const int base = row0 + 16 * R * (wave * PIECES + piece);
        float xr[R];
#pragma unroll
        for (int r = 0; r < R; r++) {
            xr[r] = w.x1[(long long)min(base + 16 * r + li, a.m - 1) * a.x1_s];
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
        float xv[KM_GRID_CHUNK / 64];
        if (w.range_start < w.range_end) {
            grid_load(w.x2, a.x2_s, w.range_start, 1, w.range_end, xv);
        }
        int shift[G];
        float4v acc[R][GE];
        const bool fine = grid_columns<false, KT, G, R, 1>(vectors(a), lds + wave * KM_GRID_TABLE_FLOATS, w, kbase, 0, rows, kc, xr,
                                                           R, xv, shift, acc);
        const float sigma = w.params[KernelTraits<KT>::SIGMA * a.params_s];
        float down[GE];
#pragma unroll
        for (int g = 0; g < GE; g++) {
            down[g] = fine && rhs_shift[g % G] != KM_GRID_NOT_FINITE ? __builtin_ldexpf(sigma, -shift[g % G] - KM_F16_KSCALE_LOG2)
                                                                     : __builtin_nanf("");
        }
#pragma unroll
        for (int r = 0; r < R; r++) {
            grid_store<KT, G>(a, w, kc, xr[r], rows.x_ref, acc[r], down, base + 16 * r, kbase);
        }
    }
}

// rhs column groups (of 16) that one pass takes, and the grid form's largest window.
template <int KT, int G>
struct GridShape {
    static constexpr int PARTS = KT == KM_KERNEL_SPECTRAL ? 2 : 1;
    static constexpr int GP = G * PARTS > 4 ? 4 / PARTS : G;
    static constexpr int GE = GP * PARTS;
    static constexpr int MT = GE >= 4 ? 4 : 5;
};

// One item by W wavefronts (this one is number `wave`): the grid form, or entry by entry.
template <int KT, int G, int W>
__device__ __forceinline__ void grid_item(const FwdArgs& a, float* lds, long long item, int wave) {
    using S = GridShape<KT, G>;
    int unused;
    const WaveView w = wave_view<true>(a, item, 1, &unused);
    const int row0 = w.row_block * KM_BLOCK_SIZE;
    // The rows are requested first, then the first columns (which wait for the range), then the
    // window is computed.
    const BlockRows rows = block_rows(w.x1, a.x1_s, row0, a.m);
    KernelConsts kc = make_consts<KT>(w.params, a.params_s, false);
    kc.s = uniform(kc.s);
    __builtin_amdgcn_sched_barrier(0);
    float xv[KM_GRID_CHUNK / 64];
    if (32 * wave < w.range_end - w.range_start) {
        grid_load(w.x2, a.x2_s, w.range_start + 32 * wave, W, w.range_end, xv);
    }
    const GridWindow gw = grid_window<S::MT>(rows, kc);
    // (the same in every lane, and said so: the barriers inside depend on it)
    bool grid = __builtin_amdgcn_readfirstlane(gw.ok && w.range_end - w.range_start >= KM_GRID_MIN_WIDTH) != 0;
#pragma unroll 1
    for (int pass = 0; pass < G / S::GP; pass++) {
        const int kbase = (blockIdx.y * G + pass * S::GP) * 16;
        if (kbase < a.k) {
            if (pass > 0 && 32 * wave < w.range_end - w.range_start) {
                grid_load(w.x2, a.x2_s, w.range_start + 32 * wave, W, w.range_end, xv);
            }
            grid = grid && grid_forward<KT, S::GP, S::MT, W>(a, lds, w, row0, kbase, wave, gw, kc, xv);
            if (!grid) {
                grid_entrywise<KT, S::GP, W>(a, lds, w, row0, kbase, wave, gw, kc);
            }
        }
    }
}

template <int KT, int G, int W>
__global__ void __launch_bounds__(64 * W, (GridShape<KT, G>::GE >= 4 ? 2 : (GridShape<KT, G>::GE > 1 ? 3 : 4))) fwd_grid(const FwdArgs a) {
    extern __shared__ float lds[];
    const long long item = xcd_item(blockIdx.x, a.items_per_xcd);
    if (item >= a.total_items) {
        return;
    }
    grid_item<KT, G, W>(a, lds, item, W == 1 ? 0 : __builtin_amdgcn_readfirstlane(threadIdx.x >> 6));
}

// Large launches: workgroups of four wavefronts.  The first items of every XCD go one per wavefront;
// its last `tail_items` are dispatched last, one per workgroup, so that these quarter-length pieces
// fill the SIMDs that would otherwise idle while others finish a last full item.
template <int KT, int G>
__global__ void __launch_bounds__(256, (GridShape<KT, G>::GE >= 4 ? 2 : (GridShape<KT, G>::GE > 1 ? 3 : 4))) fwd_grid_grouped(const FwdArgs a) {
    extern __shared__ float lds[];
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const unsigned xcd = blockIdx.x % KM_NUM_XCD;
    const long long slot = blockIdx.x / KM_NUM_XCD;
    const long long main_items = a.items_per_xcd - a.tail_items;
    const long long main_groups = (main_items + 3) / 4;
    const bool split = slot >= main_groups;
    const long long local = split ? main_items + (slot - main_groups) : slot * 4 + wave;
    const long long item = (long long)xcd * a.items_per_xcd + local;
    if ((!split && local >= main_items) || item >= a.total_items) {
        return;  // (uniform for the workgroup of a split item)
    }
    if (split) {
        grid_item<KT, G, 4>(a, lds, item, wave);
    } else {
        grid_item<KT, G, 1>(a, lds + wave * KM_GRID_TABLE_FLOATS, item, 0);
    }
}

template <int KT, int G, int W>
static hipError_t launch_grid_as(const FwdArgs& a, dim3 grid, hipStream_t stream) {
    using S = GridShape<KT, G>;
    hipLaunchKernelGGL((fwd_grid<KT, G, W>), grid, dim3(64 * W, 1, 1),
                       (sizeof(float) * grid_lds_floats<S::GE, S::MT, W>()), stream, a);
    return hipGetLastError();
}

template <int KT, int G>
static hipError_t launch_grid_w(const FwdArgs& a, int waves, dim3 grid, hipStream_t stream) {
    if (a.tail_items > 0) {
        using S = GridShape<KT, G>;
        const long long main_groups = (a.items_per_xcd - a.tail_items + 3) / 4;
        grid.x = (unsigned)((main_groups + a.tail_items) * KM_NUM_XCD);
        hipLaunchKernelGGL((fwd_grid_grouped<KT, G>), grid, dim3(256, 1, 1),
                           (sizeof(float) * grid_lds_floats<S::GE, S::MT, 4>()), stream, a);
        return hipGetLastError();
    }
    switch (waves) {
        case 1: return launch_grid_as<KT, G, 1>(a, grid, stream);
        case 2: return launch_grid_as<KT, G, 2>(a, grid, stream);
        case 4: return launch_grid_as<KT, G, 4>(a, grid, stream);
        default: return launch_grid_as<KT, G, 8>(a, grid, stream);
    }
}

template <int KT>
static hipError_t launch_grid_g(const FwdArgs& a, int G, int waves, dim3 grid, hipStream_t stream) {
    switch (G) {
        case 1: return launch_grid_w<KT, 1>(a, waves, grid, stream);
        case 2: return launch_grid_w<KT, 2>(a, waves, grid, stream);
        default: return launch_grid_w<KT, 4>(a, waves, grid, stream);
    }
}

hipError_t launch_matmul_grid(const MatmulProblem& p, const MatmulPlan& plan, hipStream_t stream) {
    FwdArgs a;
    fill_fwd_args(p, &a);
    const long long row_blocks = (p.m + KM_BLOCK_SIZE - 1) / KM_BLOCK_SIZE;
    a.chunks_per_block = 1;
    a.total_items = row_blocks * p.num_batches;
    a.items_per_xcd = (a.total_items + KM_NUM_XCD - 1) / KM_NUM_XCD;
    a.tail_items = (int)(plan.group_tail < 0 ? 0 : (plan.group_tail < a.items_per_xcd ? plan.group_tail : a.items_per_xcd));
    const dim3 grid((unsigned)(a.items_per_xcd * KM_NUM_XCD), (unsigned)((p.k + plan.k_chunk - 1) / plan.k_chunk), 1);
    if (p.kernel_type == KM_KERNEL_SPECTRAL) {
        return launch_grid_g<KM_KERNEL_SPECTRAL>(a, plan.k_chunk / 16, plan.col_splits, grid, stream);
    }
    return launch_grid_g<KM_KERNEL_RBF>(a, plan.k_chunk / 16, plan.col_splits, grid, stream);
}

}  // namespace km
