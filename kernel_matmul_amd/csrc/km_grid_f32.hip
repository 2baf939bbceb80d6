// Forward operator with every product of the contraction in fp32 (v_mfma_f32_16x16x4_f32): rbf and spectral kernels through
// the equidistant grid of km_grid.h, locally periodic ones and row blocks that the grid does not suit entry by entry
// (km_entries.h).
//
// A row block of 128 rows is one item, worked on by W wavefronts.  They take the steps of 32 columns of its range in turn and
// contract them onto the grid (MFMA t of a step contracts the columns 8 kk + t, so a lane evaluates eight neighbouring
// ones); with W > 1 the sums meet in LDS, added in a fixed order.  Each then takes 128 / W rows, for which the sums are B
// operands as they lie: MFMA v of a tile of 16 grid points contracts the points 4 kk + v.
//
// Nothing that fp32 holds is left out: the factors reach as far as their values are normal numbers.  What keeps the windows
// small is that an entry's sum over the grid is concentrated about the middle of its row and column (a term u scaled units
// from there counts 2^(-2 u^2)): a step needs the points about the middles of its columns and the rows, a row those about the
// middles of it and the columns.  Sums that leave fp32's range, values that are not finite and coordinates out of order
// send the row block entry by entry.
//
// Measured against the column tables and direct kernels of km_matmul.hip (a call, 10 points per unit, cutoff of 6
// lengthscales, k = 16): spectral n = 1e5, 8 sets 177 -> 117 us, n = 50021, 8 sets 118 -> 67, n = 20000, 2 sets 20.1 -> 17.2; rbf
// n = 1e5, 8 sets 146 -> 80, n = 65536, k = 64, 24 points per unit 104 -> 35; locally periodic n = 1e5, 8 sets 246 -> 169.
// Error against 64 bits (2-norm, 0.3 to 300 points per unit): rbf 6e-8 to 1.1e-6 -> 6e-8 to 5.5e-7, spectral 1.1e-7 to 1.1e-6 ->
// 7e-8 to 5.5e-7 (phases by phase_cos_sin: with the hardware's cosines 1.9e-7 at 2 points per unit, 1.5e-7 before),
// locally periodic 1.2e-7 to 1.1e-6 -> 1.2e-7 to 8e-7.
//
// Bound by the matrix instruction, which keeps the SIMD's VALU from issuing for its 32 clk: 8 of them per operand group for
// 16 points by 32 columns, 4 per 16 rows by 16 points.
#include "km_batch.h"
#include "km_common.h"
#include "km_entries.h"
#include "km_fwd.h"
#include "km_grid.h"
#include "km_launch.h"

namespace km {

// V = 2^-z^2 down to 2^-125; K / sigma, at z apart in the coordinates of V 2^(-z^2 / 2), down to 2^-126.
#define KM_GRID_F32_REACH 11.18f
#define KM_GRID_F32_COLUMN_REACH 15.88f
// Columns in a row block's range from which the grid is taken: three steps, of which the entries take eight tiles each and the grid as
// many and two for every 16 rows.  Measured with ranges of 128 to 256 columns (n = 50000, 8 sets), those below 160 by
// entries / by the grid: spectral 55.2 / 53.8 us a call, rbf 37.7 / 35.2.
#define KM_GRID_F32_MIN_WIDTH 96
// Magnitude of the sums over a grid point from which their products might leave fp32's range.
#define KM_GRID_F32_LARGEST 1e30f

template <int KT, int G>
struct GridF32Shape {
    static constexpr int PARTS = KT == KM_KERNEL_SPECTRAL ? 2 : 1;
    static constexpr int GE = G * PARTS;
    static constexpr int MT = GE > 2 ? 5 : 6;
    static constexpr int CHUNK = KM_GRID_CHUNK_ONE;
    static constexpr int TABLE = grid_table_floats(CHUNK);
};

template <int KT, int G, int W>
constexpr int grid_f32_exchange_floats() {
    using S = GridF32Shape<KT, G>;
    return W * S::TABLE > (W > 1 ? W * S::MT * S::GE * 256 : 0) ? W * S::TABLE : W * S::MT * S::GE * 256;
}

// The window; ok only if the columns of the range lie between its first and last one's coordinates, which the table checks.
template <int MT>
__device__ __forceinline__ GridWindow grid_f32_window(const BlockRows& rows, const KernelConsts& kc, float x_first, float x_last) {
    GridWindow gw;
    gw.x_ref = uniform(rows.middle);
    const float ya = rows.xa - gw.x_ref, yb = rows.xb - gw.x_ref;
    float row_lo = fminf(ya, yb), row_hi = fmaxf(ya, yb);
    gw.first = uniform(x_first - gw.x_ref);
    gw.last = uniform(x_last - gw.x_ref);
    const bool finite = __all(fabsf(ya) + fabsf(yb) < 1e30f) && fabsf(gw.first) + fabsf(gw.last) < 1e30f && gw.first <= gw.last;
    wave_min_max(&row_lo, &row_hi);
    gw.s2 = uniform(kc.s * 1.41421356237309504880f);
    const float inv = __builtin_amdgcn_rcpf(gw.s2);
    gw.h = uniform(__uint_as_float(__float_as_uint(KM_GRID_STEP * inv) & 0xfffff000u));
    const float inv_h = __builtin_amdgcn_rcpf(gw.h);
    gw.reach = uniform(KM_GRID_F32_REACH * inv);
    const float middle = KM_GRID_MIDDLE * inv;
    const float lo = fmaxf(row_lo - gw.reach, 0.5f * (row_lo + gw.first) - middle);
    const float hi = fminf(row_hi + gw.reach, 0.5f * (row_hi + gw.last) + middle);
    gw.g_lo = uniform(floorf(lo * inv_h));
    const float count = ceilf(hi * inv_h) - gw.g_lo;
    gw.ok = finite && gw.h > 1e-30f && gw.h < 1e30f && count >= 0.0f && count < (float)(16 * MT) && fabsf(gw.g_lo) < 16000.0f;
    gw.tiles = __builtin_amdgcn_readfirstlane(gw.ok ? ((int)count + 16) / 16 : 0);
    const float cr = KM_GRID_F32_COLUMN_REACH * inv;
    gw.col_lo = uniform(row_lo - cr);
    gw.col_hi = uniform(row_hi + cr);
    grid_tiles(&gw, row_lo, row_hi, middle);
    return gw;
}

// One step of 32 columns onto the grid.
template <int KT, int G, int MT, int CH>
__device__ __forceinline__ void grid_f32_step(const float* __restrict__ tab, int off, const float (&raw)[G][8], const GridWindow& gw,
                                              float t0, unsigned reached, bool wide,
                                              float4v (&acc)[MT][GridF32Shape<KT, G>::GE]) {
    constexpr int PARTS = GridF32Shape<KT, G>::PARTS;
    constexpr int GE = GridF32Shape<KT, G>::GE;
    float xv[8], bv[GE][8];
#pragma unroll
    for (int t = 0; t < 8; t += 4) {
        const float4v vx = *(const float4v*)(tab + off + t);
        const float4v vc = *(const float4v*)(tab + CH + off + t);
        const float4v vs = PARTS == 2 ? *(const float4v*)(tab + 2 * CH + off + t) : vc;
#pragma unroll
        for (int u = 0; u < 4; u++) {
            xv[t + u] = vx[u];
#pragma unroll
            for (int g = 0; g < G; g++) {
                bv[g][t + u] = raw[g][t + u] * vc[u];
                if (PARTS == 2) {
                    bv[GE - G + g][t + u] = raw[g][t + u] * vs[u];
                }
            }
        }
    }
    const float middle = tab[3 * CH + (off >> 3)];
#pragma unroll
    for (int mt = 0; mt < MT; mt++) {
        if ((reached >> mt & 1) == 0) {
            continue;
        }
        const float t = __builtin_fmaf((float)(16 * mt), gw.h, t0);
        float v[8];
        if (!wide) {
            const float av = __builtin_fmaf(t, gw.s2, -middle);
            const float rb = -av * av;
#pragma unroll
            for (int u = 0; u < 8; u++) {
                v[u] = __builtin_amdgcn_exp2f(__builtin_fmaf(av, xv[u], rb));
            }
        } else {
            const float4v r0 = *(const float4v*)(tab + grid_table_rest(CH) + off);
            const float4v r1 = *(const float4v*)(tab + grid_table_rest(CH) + off + 4);
#pragma unroll
            for (int u = 0; u < 8; u++) {
                const float z = ((t - xv[u]) - (u < 4 ? r0[u & 3] : r1[u & 3])) * gw.s2;
                v[u] = __builtin_amdgcn_exp2f(-z * z);
            }
        }
#pragma unroll
        for (int u = 0; u < 8; u++) {
#pragma unroll
            for (int g = 0; g < GE; g++) {
                acc[mt][g] = __builtin_amdgcn_mfma_f32_16x16x4f32(v[u], bv[g][u], acc[mt][g], 0, 0, 0);
            }
        }
        __builtin_amdgcn_sched_barrier(0);
    }
}

// The columns of the range onto the grid, every W-th step of 32 from step `wave` on; false if a value was met that
// the form does not take.
template <int KT, int G, int W>
__device__ __forceinline__ bool grid_f32_columns(const FwdArgs& a, float* __restrict__ tab, const WaveView& w, int kbase, int wave,
                                                 const GridWindow& gw, const KernelConsts& kc,
                                                 float (&xv)[GridF32Shape<KT, G>::CHUNK / 64],
                                                 float4v (&acc)[GridF32Shape<KT, G>::MT][GridF32Shape<KT, G>::GE]) {
    using S = GridF32Shape<KT, G>;
    constexpr int CH = S::CHUNK, STEPS = CH / 32;
    const int li = threadIdx.x & 15;
    const int kk = (threadIdx.x & 63) >> 4;
    const GridVectors vec = {a.x2_s, a.rhs_s0, a.rhs_s1, a.k};
    const float* __restrict__ rhs = w.rhs + (long long)kbase * a.rhs_s1;
    const RhsLane<G> rl = rhs_lane<G>(vec, kbase);
#pragma unroll
    for (int m = 0; m < S::MT; m++) {
#pragma unroll
        for (int g = 0; g < S::GE; g++) {
            acc[m][g] = (float4v){0.0f, 0.0f, 0.0f, 0.0f};
        }
    }
    const float t0 = (gw.g_lo + (float)li) * gw.h;
    bool fine = true;
    float largest = 0.0f;
    int shift[G];
    float scale[G];
#pragma unroll
    for (int g = 0; g < G; g++) {
        shift[g] = 0;
        scale[g] = 0.0f;
    }
    // (unsigned: the next first column may lie past the largest int)
    for (unsigned next_first = w.range_start + 32u * wave; next_first < (unsigned)w.range_end; next_first += CH * W) {
        const int first = (int)next_first;
        float next[G][8];
        grid_rhs<G>(vec, rhs, first, w.range_end, kk, rl, next);
        unsigned long long reached = 0;
        const unsigned steps = grid_table<true, S::PARTS == 2, CH / 64, true>(xv, first, W, w.range_end, gw, kc, tab, &fine, &reached);
        if (next_first + CH * W < (unsigned)w.range_end) {
            grid_load(w.x2, a.x2_s, first + CH * W, W, w.range_end, xv);
        }
        unsigned need = steps & 0xffff;
        const int present = min((w.range_end - 1 - first) / (32 * W) + 1, STEPS);
        look_at_steps<G>(vec, w, kbase, first, 32 * W, {~need & ((1u << present) - 1), 0, 0}, rl, shift, scale);
        if (need == 0) {
            continue;
        }
        int j = __builtin_ctz(need);
        if (j != 0) {
            grid_rhs<G>(vec, rhs, first + 32 * j * W, w.range_end, kk, rl, next);
        }
#pragma nounroll
        do {
            float raw[G][8];
#pragma unroll
            for (int g = 0; g < G; g++) {
#pragma unroll
                for (int t = 0; t < 8; t++) {
                    raw[g][t] = next[g][t];
                }
                largest = __builtin_elementwise_maximum(largest, magnitude(raw[g]));
            }
            const int off = 32 * j + 8 * kk;
            const bool wide = (steps >> (16 + j) & 1) != 0;
            const unsigned points = (unsigned)(reached >> (8 * j)) & 0xff;
            need &= need - 1;
            if (need != 0) {
                j = __builtin_ctz(need);
                grid_rhs<G>(vec, rhs, first + 32 * j * W, w.range_end, kk, rl, next);
            }
            // (kept as register quadruples, see grid_columns)
#pragma unroll
            for (int m = 0; m < S::MT; m++) {
#pragma unroll
                for (int g = 0; g < S::GE; g++) {
                    asm volatile("" : "+v"(acc[m][g]));
                }
            }
            grid_f32_step<KT, G, S::MT, CH>(tab, off, raw, gw, t0, points, wide, acc);
        } while (need != 0);
        // All reads of the table are done before the next chunk overwrites it.
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
        __builtin_amdgcn_wave_barrier();
    }
    fine = fine && __all(is_finite(largest));
#pragma unroll
    for (int g = 0; g < G; g++) {
        fine = fine && !__any(shift[g] == KM_GRID_NOT_FINITE);
    }
    return fine;
}

// Grid -> rows: `groups` groups of 16 rows from row0 from the sums of their window.
template <int KT, int G>
__device__ __forceinline__ void grid_f32_rows(const FwdArgs& a, const WaveView& w, int row0, int groups, int kbase, const GridWindow& gw, const KernelConsts& kc,
                                              const float4v (&acc)[GridF32Shape<KT, G>::MT][GridF32Shape<KT, G>::GE]) {
    using S = GridF32Shape<KT, G>;
    constexpr bool PHASE = S::PARTS == 2;
    const int lane = threadIdx.x & 63;
    const int li = lane & 15;
    const int kk = lane >> 4;
    // a lane's points 4 kk + v of a tile, v - 1.5 spacings from their middle
    const float hz = gw.h * gw.s2;
    float b2[4], own[4];
#pragma unroll
    for (int v = 0; v < 4; v++) {
        const float b = ((float)v - 1.5f) * hz;
        b2[v] = uniform(b + b);
        own[v] = uniform(-b * b);
    }
    float down[S::GE];
    const float weight = w.params[KernelTraits<KT>::SIGMA * a.params_s] * (hz * KM_GRID_WEIGHT);
#pragma unroll
    for (int g = 0; g < S::GE; g++) {
        down[g] = weight;
    }
    const float mid0 = (gw.g_lo + (float)(4 * kk) + 1.5f) * gw.h;
    const float half = 1.5f * gw.h;
    const float middle = uniform(KM_GRID_MIDDLE / KM_GRID_F32_REACH * gw.reach);
#pragma unroll 1
    for (int r = 0; r < groups; r++) {
        const int row = row0 + 16 * r;
        const float x = w.x1[(long long)min(row + li, a.m - 1) * a.x1_s];
        const float y = x - gw.x_ref;
        const float rest = remainder_of(x, gw.x_ref, y);
        float ca[4], sa[4];
        if (PHASE) {
            float cosine, sine;
            phase_cos_sin(kc.f, x, gw.x_ref, &cosine, &sine);
            row_phases(cosine, sine, 0, ca, sa);
        }
        const float t_lo = fmaxf(y - gw.reach, 0.5f * (y + gw.first) - middle) - half;
        const float t_hi = fminf(y + gw.reach, 0.5f * (y + gw.last) + middle) + half;
        float4v res[S::GE];
#pragma unroll
        for (int g = 0; g < S::GE; g++) {
            res[g] = (float4v){0.0f, 0.0f, 0.0f, 0.0f};
        }
#pragma unroll
        for (int mt = 0; mt < S::MT; mt++) {
            if (mt >= gw.tiles) {
                break;
            }
            const float mid = __builtin_fmaf((float)(16 * mt), gw.h, mid0);
            if (!__any(!(mid < t_lo || mid > t_hi))) {
                continue;
            }
            const float av = ((y - mid) + rest) * gw.s2;
            const float rb = -av * av;
#pragma unroll
            for (int v = 0; v < 4; v++) {
                const float value = __builtin_amdgcn_exp2f(__builtin_fmaf(av, b2[v], rb + own[v]));
#pragma unroll
                for (int g = 0; g < S::GE; g++) {
                    res[g] = __builtin_amdgcn_mfma_f32_16x16x4f32(value, acc[mt][g][v], res[g], 0, 0, 0);
                }
            }
        }
        grid_store<KT, G>(a, w, ca, sa, res, down, row, kbase);
    }
}

// The item through the grid; false (in all wavefronts) if the form does not suit it, and nothing is stored then.
template <int KT, int G, int W>
__device__ __forceinline__ bool grid_f32_item(const FwdArgs& a, float* lds, const WaveView& w, int row0, int kbase, int wave) {
    using S = GridF32Shape<KT, G>;
    constexpr int R = 8 / W;
    const int lane = threadIdx.x & 63;
    if (w.range_end - w.range_start < KM_GRID_F32_MIN_WIDTH) {
        return false;
    }
    const BlockRows rows = block_rows(w.x1, a.x1_s, row0, a.m);
    const float x_first = w.x2[(long long)w.range_start * a.x2_s], x_last = w.x2[(long long)(w.range_end - 1) * a.x2_s];
    KernelConsts kc = make_consts<KT>(w.params, a.params_s, false);
    kc.s = uniform(kc.s);
    __builtin_amdgcn_sched_barrier(0);
    float xv[S::CHUNK / 64];
    if (32 * wave < w.range_end - w.range_start) {
        grid_load(w.x2, a.x2_s, w.range_start + 32 * wave, W, w.range_end, xv);
    }
    const GridWindow gw = grid_f32_window<S::MT>(rows, kc, x_first, x_last);
    if (__builtin_amdgcn_readfirstlane(gw.ok) == 0) {
        return false;
    }
    float4v acc[S::MT][S::GE];
    bool fine = grid_f32_columns<KT, G, W>(a, lds + wave * S::TABLE, w, kbase, wave, gw, kc, xv, acc);
    if constexpr (W > 1) {
        float4v* const part = (float4v*)lds;
        unsigned* const words = (unsigned*)(lds + grid_f32_exchange_floats<KT, G, W>());
        __syncthreads();  // the exchange lies over the tables
        if (lane == 0) {
            words[wave] = fine ? 1 : 0;
        }
#pragma unroll
        for (int m = 0; m < S::MT; m++) {
            if (m < gw.tiles) {
#pragma unroll
                for (int g = 0; g < S::GE; g++) {
                    part[((wave * S::MT + m) * S::GE + g) * 64 + lane] = acc[m][g];
                }
            }
        }
        __syncthreads();
#pragma unroll
        for (int v = 0; v < W; v++) {
            fine = fine && __builtin_amdgcn_readfirstlane(words[v]) != 0;
        }
#pragma unroll
        for (int m = 0; m < S::MT; m++) {
            if (m < gw.tiles) {
#pragma unroll
                for (int g = 0; g < S::GE; g++) {
                    float4v sum = part[(m * S::GE + g) * 64 + lane];
#pragma unroll
                    for (int v = 1; v < W; v++) {
                        sum += part[((v * S::MT + m) * S::GE + g) * 64 + lane];
                    }
                    acc[m][g] = sum;
                }
            }
        }
    }
    float largest = 0.0f;
#pragma unroll
    for (int m = 0; m < S::MT; m++) {
#pragma unroll
        for (int g = 0; g < S::GE; g++) {
#pragma unroll
            for (int v = 0; v < 4; v++) {
                largest = __builtin_elementwise_maximum(largest, m < gw.tiles ? fabsf(acc[m][g][v]) : 0.0f);
            }
        }
    }
    fine = fine && __all(largest < KM_GRID_F32_LARGEST && is_finite(largest));
    if constexpr (W > 1) {
        __syncthreads();  // all reads done: the area may become tables again
    }
    // (the same in all wavefronts, which have the same sums)
    if (__builtin_amdgcn_readfirstlane(fine) == 0) {
        return false;
    }
    grid_f32_rows<KT, G>(a, w, row0 + 16 * R * wave, R, kbase, gw, kc, acc);
    return true;
}

template <int KT, int G, int W>
constexpr int fwd_grid_f32_floats() {
    constexpr int entries = entry_lds_floats(G, 8, W);
    if constexpr (KT == KM_KERNEL_LOCALLY_PERIODIC) {
        return entries;
    } else {
        constexpr int grid = grid_f32_exchange_floats<KT, G, W>() + W;
        return grid > entries ? grid : entries;
    }
}

template <int KT, int G, int W>
__global__ void __launch_bounds__(64 * W, G == 1 ? 3 : 2) fwd_grid_f32(const FwdArgs a) {
    extern __shared__ float lds[];
    const long long slot = xcd_item(blockIdx.x, a.items_per_xcd);
    if (slot >= a.total_items) {
        return;
    }
    // (what is left out differs between the batch items, and with it their work)
    const unsigned batches = (unsigned)a.num_batches;
    const unsigned block = (unsigned)slot / batches;
    const long long item = (long long)block * batches + spread_batch((unsigned)slot - block * batches, block, batches);
    int unused;
    const WaveView w = wave_view<true>(a, item, 1, &unused);
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int row0 = w.row_block * KM_BLOCK_SIZE, kbase = (int)blockIdx.y * G * 16;
    if constexpr (KT != KM_KERNEL_LOCALLY_PERIODIC) {
        if (grid_f32_item<KT, G, W>(a, lds, w, row0, kbase, wave)) {
            return;
        }
    }
    entry_item<KT, true, G, 8, W>(a, lds, w, row0, kbase, wave);
}

template <int KT, int G, int W>
static hipError_t launch_grid_f32_as(const FwdArgs& a, dim3 grid, hipStream_t stream) {
    hipLaunchKernelGGL((fwd_grid_f32<KT, G, W>), grid, dim3(64 * W, 1, 1), (sizeof(float) * fwd_grid_f32_floats<KT, G, W>()), stream, a);
    return hipGetLastError();
}

template <int KT, int G>
static hipError_t launch_grid_f32_w(FwdArgs& a, const MatmulPlan& plan, unsigned grid_y, hipStream_t stream) {
    a.total_items = ((long long)a.m + KM_BLOCK_SIZE - 1) / KM_BLOCK_SIZE * a.num_batches;
    a.items_per_xcd = (a.total_items + KM_NUM_XCD - 1) / KM_NUM_XCD;
    const dim3 grid((unsigned)(a.items_per_xcd * KM_NUM_XCD), grid_y, 1);
    switch (plan.col_splits) {
        case 1:
            if constexpr (KT == KM_KERNEL_LOCALLY_PERIODIC) {
                return hipErrorInvalidValue;
            } else {
                return launch_grid_f32_as<KT, G, 1>(a, grid, stream);
            }
        case 2: return launch_grid_f32_as<KT, G, 2>(a, grid, stream);
        case 4: return launch_grid_f32_as<KT, G, 4>(a, grid, stream);
        default:
            // (the exchange of eight wavefronts' sums would not fit into LDS for four operand groups)
            if constexpr (KT == KM_KERNEL_SPECTRAL && G == 2) {
                return hipErrorInvalidValue;
            } else {
                return launch_grid_f32_as<KT, G, 8>(a, grid, stream);
            }
    }
}

template <int KT>
static hipError_t launch_grid_f32_g(FwdArgs& a, const MatmulPlan& plan, unsigned grid_y, hipStream_t stream) {
    return plan.k_chunk == 16 ? launch_grid_f32_w<KT, 1>(a, plan, grid_y, stream) : launch_grid_f32_w<KT, 2>(a, plan, grid_y, stream);
}

hipError_t launch_matmul_grid_f32(const MatmulProblem& p, const MatmulPlan& plan, hipStream_t stream) {
    FwdArgs a;
    fill_fwd_args(p, &a);
    a.chunks_per_block = 1;
    const unsigned grid_y = (unsigned)((p.k + plan.k_chunk - 1) / plan.k_chunk);
    switch (p.kernel_type) {
        case KM_KERNEL_RBF: return launch_grid_f32_g<KM_KERNEL_RBF>(a, plan, grid_y, stream);
        case KM_KERNEL_SPECTRAL: return launch_grid_f32_g<KM_KERNEL_SPECTRAL>(a, plan, grid_y, stream);
        default: return launch_grid_f32_g<KM_KERNEL_LOCALLY_PERIODIC>(a, plan, grid_y, stream);
    }
}

}  // namespace km
