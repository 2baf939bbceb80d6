// Grid form of the Gaussian factor, shared by the forward and the gradient kernels.
//
// A Gaussian is the convolution of two narrower ones, and the trapezoid rule turns that integral
// into a sum over an equidistant grid t_g = g h with an error that falls off like
// exp(-pi^2 l^2 / (2 h^2)):
//     exp(-(x - y)^2 / (2 l^2)) = C sum_g V(x, t_g) V(y, t_g),   V(x, t) = exp(-(x - t)^2 / l^2),
//     C = (h / l) sqrt(2 / pi).
// Every term is positive, so nothing cancels: the relative error of every entry is that of the
// rule (6e-8 at h = 0.53 l, half an fp32 ulp) plus the rounding of the two factors.  A row block's
// product with a vector is then two short contractions instead of one long one:
//     G_g = sum_j V(y_j, t_g) rhs_j        (columns -> grid, "moments")
//     out_i = C sum_g V(x_i, t_g) G_g      (grid -> rows)
// and the work per column and per row is one grid window (span of the row block plus twice the
// reach of V, 20 to 80 points, 96 at most) instead of one entry per row and column of the pattern.  The column
// ranges [start, end) are honoured exactly: each row block sums the columns of its own range.
//
// Coordinates are taken relative to the row block's middle row (exact for neighbouring points; rows
// and columns carry the rounding of that difference as a second term) and h is rounded to 12
// significant bits, so that all g h are exact.  Scaled coordinates z = x s2 (s2 = sqrt(log2 e) / l)
// make V(x, t) = 2^-(z_x - z_t)^2.
#pragma once

#include <type_traits>

#include "km_common.h"
#include "km_fwd.h"

namespace km {

#define KM_GRID_STEP 0.64f          /* h s2: trapezoid error 2 exp(-7.119 / 0.64^2) = 5.7e-8 */
#define KM_GRID_REACH 6.083f        /* V (and K / sigma) < 2^-37 beyond: the floor of the split-fp16 contraction */
#define KM_GRID_COLUMN_REACH 8.603f /* the same for K / sigma in the coordinates of V: sqrt(2) times as far */
#define KM_GRID_WEIGHT_F64 0.66428247026735920 /* C / (h s2) = sqrt(2 ln 2 / pi) */
#define KM_GRID_WEIGHT ((float)KM_GRID_WEIGHT_F64)
#define KM_GRID_CHUNK 256           /* columns tabulated at a time, per wavefront ... */
#define KM_GRID_CHUNK_ONE 128       /* ... with one group of rhs columns (grid_columns) */
#define KM_GRID_KS1 11              /* V is evaluated times 2^11 (columns: reference within 2) ... */
#define KM_GRID_SPAN 2.0f
#define KM_GRID_KS2 10              /* ... and 2^10 (rows: reference within 3.5 h s2 = 2.24) */
#define KM_GRID_NOT_FINITE 1000     /* in place of a rhs column's shift: it holds a value that is not finite */
// Table of a chunk: coordinate, the two column factors, for each 8 columns what is halfway between their ends (entry by entry:
// the smallest and largest coordinate), and the remainder of the coordinate.
constexpr int grid_table_rest(int chunk) { return 3 * chunk + 2 * chunk / 8; }
constexpr int grid_table_floats(int chunk) { return grid_table_rest(chunk) + chunk; }
#define KM_GRID_TABLE_FLOATS (grid_table_floats(KM_GRID_CHUNK))

// A value that is the same in every lane, as a scalar register.
__device__ __forceinline__ float uniform(float v) {
    return __uint_as_float(__builtin_amdgcn_readfirstlane(__float_as_uint(v)));
}

// Grid window of one row block (the same in every lane).
struct GridWindow {
    bool ok;           // the form applies: finite coordinates, window within the accumulators
    float x_ref;       // origin of the relative coordinates
    float s2, h;       // scale of z and grid spacing
    float g_lo;        // first grid index (t = g h relative to x_ref)
    float col_lo, col_hi;  // relative coordinates beyond which columns contribute nothing
    float reach;       // distance beyond which the evaluated factor counts as zero
    int tiles;         // groups of 16 grid points
    float first, last; // relative coordinates that no column lies beyond (where that is not known: the
                       // largest that the form takes)
    float per_tile, from, from_middle, to, to_middle;  // the tiles of a step (grid_tiles)
};

// An entry's sum over the grid is concentrated about the middle of its row and column: a term u scaled units from there
// counts 2^(-2 u^2), beyond this 2^-28.9 of the entry.
#define KM_GRID_MIDDLE 3.8f

// What a step's groups of 16 grid points follow from: those with a point within reach of its columns and, beyond that
// (middle, in units of length; infinite: not taken), about the middles of its columns and the rows.  In tiles from the window's
// first point; a 64th of a spacing is for rounding.
__device__ __forceinline__ void grid_tiles(GridWindow* gw, float row_lo, float row_hi, float middle) {
    const float per_tile = uniform(0.0625f * __builtin_amdgcn_rcpf(gw->h));
    const float base = gw->g_lo * gw->h;
    gw->per_tile = per_tile;
    gw->from = uniform((-gw->reach - base) * per_tile + 0.0625f * (63.0f / 64.0f));
    gw->from_middle = uniform((0.5f * row_lo - middle - base) * per_tile + 0.0625f * (63.0f / 64.0f));
    gw->to = uniform((gw->reach - base) * per_tile + (1.0f + 1.0f / 1024.0f));
    gw->to_middle = uniform((0.5f * row_hi + middle - base) * per_tile + (1.0f + 1.0f / 1024.0f));
}

// The rows of a block, two per lane, and its middle row.
struct BlockRows {
    float xa, xb, middle;
};

__device__ __forceinline__ BlockRows block_rows(const float* __restrict__ x1, long long x1_s, int row0, int m) {
    const int lane = threadIdx.x & 63;
    BlockRows r;
    // (unsigned: the rows of a group's last wavefronts may lie past the largest int)
    const unsigned row = (unsigned)row0, last = (unsigned)m - 1;
    r.xa = x1[(long long)min(row + lane, last) * x1_s];
    r.xb = x1[(long long)min(row + 64 + lane, last) * x1_s];
    r.middle = x1[(long long)min(row + 64, last) * x1_s];
    return r;
}

// step: grid spacing in units of 1 / s2; middle: as grid_tiles, in the same units.
template <int MT>
__device__ __forceinline__ GridWindow grid_window(const BlockRows& rows, const KernelConsts& kc,
                                                  float step = KM_GRID_STEP, float middle = KM_GRID_MIDDLE) {
    GridWindow gw;
    gw.x_ref = uniform(rows.middle);
    const float xa = rows.xa, xb = rows.xb;
    float lo = fminf(xa - gw.x_ref, xb - gw.x_ref);
    float hi = fmaxf(xa - gw.x_ref, xb - gw.x_ref);
    const bool finite = __all(fabsf(xa - gw.x_ref) + fabsf(xb - gw.x_ref) < 1e30f);
    wave_min_max(&lo, &hi);
    gw.s2 = uniform(kc.s * 1.41421356237309504880f);
    // (none of these has to be exact, only h has to be short)
    const float inv = __builtin_amdgcn_rcpf(gw.s2);
    gw.h = uniform(__uint_as_float(__float_as_uint(step * inv) & 0xfffff000u));
    const float inv_h = __builtin_amdgcn_rcpf(gw.h);
    gw.reach = uniform(KM_GRID_REACH * inv);
    gw.g_lo = uniform(floorf((lo - gw.reach) * inv_h));
    const float g_hi = ceilf((hi + gw.reach) * inv_h);
    // (false for a spacing of zero, infinity or NaN as well)
    gw.ok = finite && gw.h > 1e-30f && gw.h < 1e30f && g_hi - gw.g_lo < (float)(16 * MT);
    gw.tiles = gw.ok ? ((int)(g_hi - gw.g_lo) + 16) / 16 : 0;
    gw.tiles = __builtin_amdgcn_readfirstlane(gw.tiles);
    const float cr = KM_GRID_COLUMN_REACH * inv;
    gw.col_lo = uniform(finite ? lo - cr : -__builtin_inff());
    gw.col_hi = uniform(finite ? hi + cr : __builtin_inff());
    gw.first = -1e30f;
    gw.last = 1e30f;
    grid_tiles(&gw, lo, hi, middle * inv);
    return gw;
}

// What the subtraction d = x - origin rounded off.
__device__ __forceinline__ float remainder_of(float x, float origin, float d) {
    const float bb = d - x;
    return (x - (d - bb)) - (origin + bb);
}

// Coordinates of this wavefront's next CH / 32 steps of 32 columns, in the order grid_table takes them.
template <int N>
__device__ __forceinline__ void grid_load(const float* __restrict__ x2, long long x2_s, int first, int stride, int end,
                                          float (&xv)[N]) {
    const int lane = threadIdx.x & 63;
    const float* xc = x2 + (long long)first * x2_s;
    const int last = end - 1 - first;
#pragma unroll
    for (int i = 0; i < N; i++) {
        const int rel = 32 * ((lane >> 5) + 2 * i) * stride + (lane & 31);
        xv[i] = xc[(unsigned long long)(unsigned)min(rel, last) * (unsigned)x2_s];
    }
}

// Tabulates this wavefront's next 2 N steps of 32 columns (the steps first / 32 + j * stride of the
// range, j = 0 .. 2 N - 1: several wavefronts that share a range take its steps in turn).  Returns the
// steps that reach the rows as a bit mask.
//   GRID: coordinates as 2 b, b = y s2 - r with r halfway between the ends of each group of 8 (times s2; in the table), the
//         column factors times 2^(-b^2).  *tiles: eight bits for each step, its groups of 16 grid points (made here, once
//         for a group of 8 columns, with what bounds them about the middles: looked at tile by tile in grid_step, within reach
//         alone, likelihood gradient n = 1e5, 16 sets 105.7 us instead of 104.1, forward n = 1e6, k = 32 781 instead of 776, fp32
//         n = 1e5 119.0 instead of 118.0; other sizes 0 to 0.3 %; rbf gradients of one column at one point per unit, which
//         reach one or two groups a step, the other way, n = 1e5, 8 sets 52.4 and 53.8).  Steps of which a group spreads further than KM_GRID_SPAN
//         (a gap in the data) come back in the upper half of the mask: their factors lack 2^(-b^2)
//         (it would leave the fp16 range) and their coordinates are y and its remainder, relative to
//         the row block's origin: a reference in the middle of the gap would round them to a fraction
//         of the gap.  *fine is cleared when a coordinate lies beyond gw.first or gw.last or is NaN.
//   else: the coordinates themselves (entry-wise evaluation).  *fine is cleared when a coordinate makes
//         every entry of its column NaN: a NaN, or an infinity under an oscillating factor.
//   EXACT_PHASE: cosines and sines to fp32's rounding (phase_cos_sin) instead of the hardware's.
template <bool GRID, bool PHASE, int N, bool EXACT_PHASE = false>
__device__ __forceinline__ unsigned grid_table(const float (&xv)[N], int first, int stride, int end,
                                               const GridWindow& gw, const KernelConsts& kc, float* __restrict__ tab,
                                               bool* fine, unsigned long long* tiles = nullptr) {
    constexpr int CH = 64 * N;
    static_assert(!GRID || N <= 4, "eight bits for each step");
    const int lane = threadIdx.x & 63;
    const int last = end - 1 - first;
    float lo[N], hi[N];
    bool wide[N];
    unsigned need = 0;
    bool ok = true;
    // the bits of steps 2 i and 2 i + 1 from the lanes that hold their columns
    auto bits = [](bool lanes, int i) {
        const unsigned long long any = __ballot(lanes);
        return (unsigned)((any & 0xffffffffull) != 0) << (2 * i) | (unsigned)((any >> 32) != 0) << (2 * i + 1);
    };
#pragma unroll
    for (int i = 0; i < N; i++) {
        const int rel = 32 * ((lane >> 5) + 2 * i) * stride + (lane & 31);
        const float y = xv[i] - gw.x_ref;
        // (true for NaN, which the entry-wise evaluation hands on)
        need |= bits(rel <= last && !(y < gw.col_lo || y > gw.col_hi), i);
        group8_min_max(GRID ? y : xv[i], &lo[i], &hi[i]);
        if (GRID) {
            const unsigned w = bits(0.5f * (hi[i] - lo[i]) * gw.s2 > KM_GRID_SPAN, i);
            wide[i] = (w >> (2 * i + (lane >> 5)) & 1) != 0;
            need |= w << 16;
            ok = ok && y >= gw.first && y <= gw.last;
        } else {
            ok = ok && (PHASE ? is_finite(xv[i]) : xv[i] == xv[i]);
        }
    }
    need = __builtin_amdgcn_readfirstlane(need);
    *fine = *fine && __all(ok);
    if ((need & 0xffff) == 0) {
        return 0;
    }
    unsigned long long reached = 0;
#pragma unroll
    for (int i = 0; i < N; i++) {
        if ((need >> (2 * i) & 3) == 0) {
            continue;
        }
        const int q = lane + 64 * i;
        float wgt = 1.0f;
        if (GRID) {
            const float y = xv[i] - gw.x_ref;
            const float rest = remainder_of(xv[i], gw.x_ref, y);
            const float middle = 0.5f * (lo[i] + hi[i]) * gw.s2;
            const float b = __builtin_fmaf(rest, gw.s2, __builtin_fmaf(y, gw.s2, -middle));
            tab[q] = b + b;
            if (wide[i]) {
                tab[q] = y;
                tab[grid_table_rest(CH) + q] = rest;
            } else {
                wgt = __builtin_amdgcn_exp2f(-b * b);
            }
            if ((lane & 7) == 0) {
                tab[3 * CH + (q >> 3)] = middle;
            }
            const float first_tile = fmaxf(__builtin_fmaf(lo[i], gw.per_tile, gw.from), __builtin_fmaf(lo[i], 0.5f * gw.per_tile, gw.from_middle));
            const float end_tile = fminf(__builtin_fmaf(hi[i], gw.per_tile, gw.to), __builtin_fmaf(hi[i], 0.5f * gw.per_tile, gw.to_middle));
            const int from = min(max((int)__builtin_floorf(first_tile), 0), gw.tiles);
            const int to = min(max((int)__builtin_floorf(end_tile), from), gw.tiles);
            int mask = (1 << to) - (1 << from);
            mask |= __builtin_amdgcn_update_dpp(0, mask, 0x128, 0xf, 0xf, false);  // row_ror:8
            const unsigned even = __builtin_amdgcn_readlane(mask, 0) | __builtin_amdgcn_readlane(mask, 16);
            const unsigned odd = __builtin_amdgcn_readlane(mask, 32) | __builtin_amdgcn_readlane(mask, 48);
            reached |= (unsigned long long)(even | odd << 8) << (16 * i);
        } else {
            tab[q] = xv[i];
        }
        // (zero past the end of the range, where rhs values are those of the last row again)
        const bool inside = 32 * ((lane >> 5) + 2 * i) * stride + (lane & 31) <= last;
        if (PHASE) {
            float cosine, sine;
            if constexpr (EXACT_PHASE) {
                phase_cos_sin(kc.f, xv[i], gw.x_ref, &cosine, &sine);
            } else {
                const float th = phase_rev(kc.f, xv[i], gw.x_ref);
                cosine = __builtin_amdgcn_cosf(th);
                sine = __builtin_amdgcn_sinf(th);
            }
            tab[CH + q] = inside ? wgt * cosine : 0.0f;
            tab[2 * CH + q] = inside ? wgt * sine : 0.0f;
        } else {
            tab[CH + q] = inside ? wgt : 0.0f;
        }
        if (!GRID && (lane & 7) == 0) {
            tab[3 * CH + (q >> 3)] = lo[i];
            tab[3 * CH + CH / 8 + (q >> 3)] = hi[i];
        }
    }
    if (GRID) {
        *tiles = reached;
    }
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
    return need;
}

// Accumulators of two neighbouring groups of 16 grid points (lane (li, kk): points 4 kk + v of
// column li) rearranged into the layout of a contraction over their 32 points (lane (li, kk):
// points 8 kk .. 8 kk + 7 of column li).
__device__ __forceinline__ void grid_operand(const float4v& a, const float4v& b, float (&g)[8]) {
#pragma unroll
    for (int v = 0; v < 4; v++) {
        const auto halves = __builtin_amdgcn_permlane32_swap(__float_as_uint(a[v]), __float_as_uint(b[v]), false, false);
        const auto rows = __builtin_amdgcn_permlane16_swap(halves[0], halves[1], false, false);
        g[v] = __uint_as_float(rows[0]);
        g[4 + v] = __uint_as_float(rows[1]);
    }
}

// Strides and width of the vectors that are contracted onto the grid.
struct GridVectors {
    long long x2_s, rhs_s0, rhs_s1;
    int k;
};

// This lane's part of a step's rhs operand: byte offsets of its 8 columns' first row (8 kk) and of its
// rhs column in each group.  Inner strides are at most 2^22 elements (the entry point checks), so a
// step spans less than 2^32 bytes and its row offsets come from 24-bit multiplications.
template <int G>
struct RhsLane {
    unsigned row;
    unsigned col[G];
    bool used[G];
};

template <int G, bool PACK = false>
__device__ __forceinline__ RhsLane<G> rhs_lane(const GridVectors& a, int kbase) {
    const int li = threadIdx.x & (PACK ? 7 : 15);
    const unsigned kk = (threadIdx.x & 63) >> 4;
    RhsLane<G> rl;
    rl.row = 4u * __umul24(8u * kk, (unsigned)a.rhs_s0);
#pragma unroll
    for (int g = 0; g < G; g++) {
        const int c = kbase + 16 * g + li;
        rl.col[g] = 4u * __umul24((unsigned)(min(c, a.k - 1) - kbase), (unsigned)a.rhs_s1);
        rl.used[g] = c < a.k;
    }
    return rl;
}

// rhs values of a step (columns c0 + 8 kk + t).  Past the end of the range the last row's are repeated: the table's
// factors of these columns are zero (grid_table).  Nothing here depends on a loaded value, so that all of a step's loads
// are in flight together.
template <int G>
__device__ __forceinline__ void grid_rhs(const GridVectors& a, const float* __restrict__ rhs, int c0, int col_end,
                                         int kk, const RhsLane<G>& lane, float (&raw)[G][8]) {
    const buffer_rsrc ru = uniform_buffer(rhs + (long long)c0 * a.rhs_s0);
    const unsigned s0 = (unsigned)a.rhs_s0;
    if (c0 + 32 <= col_end) {
#pragma unroll
        for (int t = 0; t < 8; t++) {
#pragma unroll
            for (int g = 0; g < G; g++) {
                raw[g][t] = buffer_at(ru, lane.row + lane.col[g], 4u * (unsigned)t * s0);
            }
        }
    } else {
        const int last = col_end - 1 - c0;
#pragma unroll
        for (int t = 0; t < 8; t++) {
            const unsigned row = 4u * __umul24((unsigned)min(8 * kk + t, last), s0);
#pragma unroll
            for (int g = 0; g < G; g++) {
                raw[g][t] = buffer_at(ru, row + lane.col[g], 0u);
            }
        }
    }
}

// The Gaussian factor of a row against two neighbouring columns, split into fp16 halves, times
// 2^KM_F16_KSCALE_LOG2.  (The power of two is applied to the rounded halves, exactly, and in the
// residual: inside the exponent it would cost it four bits.)
__device__ __forceinline__ void entry_pair_f16(float x, float ya, float yb, float scale, half2v* hi, half2v* lo) {
    constexpr float S = (float)(1 << KM_F16_KSCALE_LOG2);
    const float ua = (x - ya) * scale, ub = (x - yb) * scale;
    const float ea = __builtin_amdgcn_exp2f(-ua * ua);
    const float eb = __builtin_amdgcn_exp2f(-ub * ub);
    const float2v kv = {ea, eb};
    const half2v h = __builtin_convertvector(kv, half2v) * (half2v){(_Float16)S, (_Float16)S};
    *hi = h;
    *lo = residual_f16x2(ea, S, eb, S, h);
}

// Two powers of two split into fp16 halves.
__device__ __forceinline__ void exp2_pair_f16(float a, float b, float one, half2v* hi, half2v* lo) {
    const float2v kv = {__builtin_amdgcn_exp2f(a), __builtin_amdgcn_exp2f(b)};
    const half2v h = __builtin_convertvector(kv, half2v);
    *hi = h;
    *lo = residual_f16x2(kv[0], one, kv[1], one, h);
}

// Largest magnitude of 8 values, or NaN if one of them is.
__device__ __forceinline__ float magnitude(const float (&v)[8]) {
    float m = 0.0f;
#pragma unroll
    for (int t = 0; t < 8; t++) {
        m = __builtin_elementwise_maximum(m, fabsf(v[t]));
    }
    return m;
}

// column_max of values of which a NaN is the largest.
__device__ __forceinline__ float column_maximum(float m) {
    const unsigned bits = __float_as_uint(m);
    const auto rows = __builtin_amdgcn_permlane16_swap(bits, bits, false, false);
    m = __builtin_elementwise_maximum(__uint_as_float(rows[0]), __uint_as_float(rows[1]));
    const unsigned bits2 = __float_as_uint(m);
    const auto halves = __builtin_amdgcn_permlane32_swap(bits2, bits2, false, false);
    return __builtin_elementwise_maximum(__uint_as_float(halves[0]), __uint_as_float(halves[1]));
}

// Steps of a wavefront's range that were out of reach: the first 64 as bits, of longer ranges all from
// there on.
struct BeyondSteps {
    unsigned long long bits;
    int rest, total;
    __device__ __forceinline__ bool any() const { return bits != 0 || rest < total; }
    // The next one; the one before again if there is none left.
    __device__ __forceinline__ int next(int before) {
        if (bits != 0) {
            before = __builtin_ctzll(bits);
            bits &= bits - 1;
        } else if (rest < total) {
            before = rest++;
        }
        return before;
    }
};

// Whether rhs can be read in quadruples across its rows or along its columns: dense (k = 1: whatever the stride
// of its one column), and with at least one quadruple up to the range's end.
__device__ __forceinline__ bool dense_rows(const GridVectors& a, int range_end) {
    return (a.rhs_s1 == 1 || a.k == 1) && a.rhs_s0 == a.k && a.k <= 64 && (long long)range_end * a.k >= 4;
}
__device__ __forceinline__ bool dense_columns(const GridVectors& a, int range_end) {
    return a.rhs_s0 == 1 && a.k <= 64 && range_end >= 4;
}

// LOADS quadruples a lane of rhs[., k] in the columns [c0, min(c0 + 32, end)), from the quadruple `base` on:
// one run of all rows (ROWS), or eight quadruples of each rhs column.  Quadruples are whole and at any
// multiple of four bytes: where the run is shorter, up to three values before it are among it.
template <int LOADS, bool ROWS>
__device__ __forceinline__ void step_quads(const GridVectors& a, const float* __restrict__ rhs, int c0, int end, int base,
                                           float4v* __restrict__ v) {
    const int lane = threadIdx.x & 63;
    const int per_column = ROWS ? a.k : 1;
    const int last = min(32, end - c0) * per_column - 4;
    const char* p = (const char*)(rhs + ((long long)c0 * per_column + min(last, 0)));
#pragma unroll
    for (int q = 0; q < LOADS; q++) {
        const int i = base + 64 * q + lane;
        unsigned bytes = 4u * (unsigned)min(4 * (ROWS ? i : i & 7), max(last, 0));
        if (!ROWS) {
            bytes += 4u * __umul24((unsigned)min(i >> 3, a.k - 1), (unsigned)a.rhs_s1);
        }
        __builtin_memcpy(&v[q], p + bytes, sizeof(float4v));
    }
}

template <int N>
__device__ __forceinline__ float quads_magnitude(const float4v (&v)[N], float m) {
#pragma unroll
    for (int i = 0; i < N; i++) {
#pragma unroll
        for (int t = 0; t < 4; t++) {
            m = __builtin_elementwise_maximum(m, fabsf(v[i][t]));
        }
    }
    return m;
}

// Whether the rhs values of the given steps (columns first + j stride on) are all finite.  A step of 16 rhs
// columns is two loads and four operations a lane, where a step within reach costs some 250; the loads of
// several steps are in flight together, as nothing else hides them.
template <int G, bool ROWS>
__device__ __forceinline__ bool columns_finite(const GridVectors& a, const float* __restrict__ rhs, int first, int stride,
                                               int end, BeyondSteps steps) {
    constexpr int LOADS = G < 4 ? 2 * G : 8;  // of 64 quadruples each, at a time and step
    constexpr int STEPS = G < 4 ? 2 / G : 1;  // at a time
    float m = 0.0f;
#pragma unroll 1
    while (steps.any()) {
        int c0[STEPS], j = 0;
#pragma unroll
        for (int i = 0; i < STEPS; i++) {
            j = steps.next(j);
            c0[i] = first + j * stride;
        }
#pragma unroll 1
        for (int base = 0; base < 8 * a.k; base += 64 * LOADS) {
            float4v v[STEPS * LOADS];
#pragma unroll
            for (int i = 0; i < STEPS; i++) {
                step_quads<LOADS, ROWS>(a, rhs, c0[i], end, base, v + i * LOADS);
            }
            m = quads_magnitude(v, m);
        }
    }
    return __all(is_finite(m));
}

// Looks at the rhs values of the given steps: the shift of a column with one that is not finite becomes
// KM_GRID_NOT_FINITE and its scale zero.
template <int G>
__device__ __forceinline__ void look_at_steps(const GridVectors& a, const WaveView& w, int kbase, int first, int stride,
                                              BeyondSteps steps, const RhsLane<G>& rl, int (&shift)[G], float (&scale)[G]) {
    if (!steps.any()) {
        return;
    }
    bool finite = false;
    if (dense_rows(a, w.range_end)) {
        finite = columns_finite<G, true>(a, w.rhs, first, stride, w.range_end, steps);
    } else if (G == 1 && dense_columns(a, w.range_end)) {
        // (with more groups its mere presence costs the others registers: 2 to 3 % at k = 32 and 64)
        finite = columns_finite<G, false>(a, w.rhs, first, stride, w.range_end, steps);
    }
    if (finite) {
        return;
    }
    const float* rhs = w.rhs + (long long)kbase * a.rhs_s1;
#pragma unroll 1
    do {
        float raw[G][8];
        grid_rhs<G>(a, rhs, first + stride * steps.next(0), w.range_end, (threadIdx.x & 63) >> 4, rl, raw);
#pragma unroll
        for (int g = 0; g < G; g++) {
            const float m = column_maximum(magnitude(raw[g]));
            const bool bad = rl.used[g] && !is_finite(m);
            shift[g] = bad ? KM_GRID_NOT_FINITE : shift[g];
            scale[g] = bad ? 0.0f : scale[g];
        }
    } while (steps.any());
}

// The running power-of-two scale of an rhs column, lowered when a magnitude of its values (own: of those that this lane
// holds) would exceed 2^15 (NaN and infinities hand themselves on).  The four lanes of a column compare theirs only then.  first: no step has added to the sums yet (a scale that is still the largest
// does not say so: steps of values below 2^-85 leave it as it is).
template <int G, int PARTS, int MT>
__device__ __forceinline__ void lower_scale(int g, float own, bool used, bool first, int (&shift)[G], float (&scale)[G],
                                            float4v (&acc)[MT][G * PARTS]) {
    if (__any(used && !(own * scale[g] < 32768.0f))) {
        const float m = column_maximum(own);
        const bool grow = used && !(m * scale[g] < 32768.0f);
        if (grow && !is_finite(m)) {
            shift[g] = KM_GRID_NOT_FINITE;
            scale[g] = 0.0f;
        } else if (grow) {
            const int e = __builtin_amdgcn_frexp_expf(m);
            const int new_shift = min(14 - e, 100);
            if (!first) {
                const float factor = __builtin_ldexpf(1.0f, new_shift - shift[g]);
#pragma unroll
                for (int mt = 0; mt < MT; mt++) {
#pragma unroll
                    for (int part = 0; part < PARTS; part++) {
                        acc[mt][part * G + g] *= factor;
                    }
                }
            }
            shift[g] = new_shift;
            scale[g] = __builtin_ldexpf(1.0f, new_shift);
        }
    }
}

// One step of 32 columns: split the scaled rhs operand, then for every tile of 16 points in reach evaluate, split
// and contract.  GRID: the points are the grid's, t0 + 16 mt h, tiles as bits in `reached`; else the rows xr[].
// weights: which of the table's column factors this lane's rhs column takes (PARTS == 1; with two parts
// the cosines for the first and the sines for the second).  EXACT: the product of the low halves as well
// (the gradient: hidden behind the VALU work there, and it halves the error of its long sums).
// WIDE: the step may be one of those whose factors lack 2^(-b^2); `wide` says whether it is.
template <bool GRID, int G, int PARTS, int MT, bool EXACT, int CH, bool WIDE>
__device__ __forceinline__ void grid_step(const float* __restrict__ tab, int off, const float (&raw)[G][8],
                                          const GridWindow& gw, float t0, const float* xr, const KernelConsts& kc,
                                          int tiles, unsigned reached, bool wide, int weights, const float (&scale)[G],
                                          float4v (&acc)[MT][G * PARTS]) {
    constexpr int GE = G * PARTS;
    float xv[8], cb[8], sb[8];
#pragma unroll
    for (int t = 0; t < 8; t += 4) {
        const float4v vx = *(const float4v*)(tab + off + t);
        const float4v vc = *(const float4v*)(tab + weights + off + t);
#pragma unroll
        for (int u = 0; u < 4; u++) {
            xv[t + u] = vx[u];
            cb[t + u] = vc[u];
        }
        if (PARTS == 2) {
            const float4v vs = *(const float4v*)(tab + 2 * CH + off + t);
#pragma unroll
            for (int u = 0; u < 4; u++) {
                sb[t + u] = vs[u];
            }
        }
    }
    const float lo = tab[3 * CH + (off >> 3)];  // (GRID: the group's middle)
    const float hi = GRID ? 0.0f : tab[3 * CH + CH / 8 + (off >> 3)];

    half8v bhi[GE], blo[GE];
#pragma unroll
    for (int g = 0; g < G; g++) {
        float vc[8];
#pragma unroll
        for (int t = 0; t < 8; t++) {
            vc[t] = raw[g][t] * scale[g];
        }
        if (PARTS == 2) {
            float vs[8];
#pragma unroll
            for (int t = 0; t < 8; t++) {
                vs[t] = vc[t] * sb[t];
            }
            split_f16x8(vs, kc.one, &bhi[G + g], &blo[G + g]);
        }
        if (PARTS == 2 || GRID) {
#pragma unroll
            for (int t = 0; t < 8; t++) {
                vc[t] *= cb[t];
            }
        }
        split_f16x8(vc, kc.one, &bhi[g], &blo[g]);
    }

#pragma unroll
    for (int mt = 0; mt < MT; mt++) {
        if (!GRID && mt >= tiles) {
            break;
        }
        const float t = GRID ? __builtin_fmaf((float)(16 * mt), gw.h, t0) : xr[mt];
        if (GRID ? (reached >> mt & 1) == 0 : !__any(!(fmaxf(lo - t, t - hi) > gw.reach))) {
            continue;
        }
        half2v h2[4], l2[4];
        float arg[8];
        if (GRID) {
            if (!WIDE || !wide) {
                const float av = __builtin_fmaf(t, gw.s2, -lo);
                const float rb = __builtin_fmaf(-av, av, (float)KM_GRID_KS1);
#pragma unroll
                for (int u = 0; u < 8; u++) {
                    arg[u] = __builtin_fmaf(av, xv[u], rb);
                }
            } else {
                const float4v r0 = *(const float4v*)(tab + grid_table_rest(CH) + off);
                const float4v r1 = *(const float4v*)(tab + grid_table_rest(CH) + off + 4);
#pragma unroll
                for (int u = 0; u < 8; u++) {
                    const float z = ((t - xv[u]) - (u < 4 ? r0[u & 3] : r1[u & 3])) * gw.s2;
                    arg[u] = __builtin_fmaf(-z, z, (float)KM_GRID_KS1);
                }
            }
        }
#pragma unroll
        for (int u = 0; u < 4; u++) {
            if (GRID) {
                exp2_pair_f16(arg[2 * u], arg[2 * u + 1], kc.one, &h2[u], &l2[u]);
            } else {
                entry_pair_f16(t, xv[2 * u], xv[2 * u + 1], kc.s, &h2[u], &l2[u]);
            }
        }
        const half8v ahi = join_half2x4(h2);
        const half8v alo = join_half2x4(l2);
#pragma unroll
        for (int g = 0; g < GE; g++) {
            acc[mt][g] = __builtin_amdgcn_mfma_f32_16x16x32_f16(ahi, bhi[g], acc[mt][g], 0, 0, 0);
            acc[mt][g] = __builtin_amdgcn_mfma_f32_16x16x32_f16(ahi, blo[g], acc[mt][g], 0, 0, 0);
            acc[mt][g] = __builtin_amdgcn_mfma_f32_16x16x32_f16(alo, bhi[g], acc[mt][g], 0, 0, 0);
            if (EXACT) {
                acc[mt][g] = __builtin_amdgcn_mfma_f32_16x16x32_f16(alo, blo[g], acc[mt][g], 0, 0, 0);
            }
        }
        __builtin_amdgcn_sched_barrier(0);
    }
}

// The columns of [w.range_start, w.range_end) against `tiles` groups of 16 points (GRID: of the
// grid window; else the rows xr[]): acc in the D layout times 2^shift (per rhs column) and the scale
// of the evaluated factor.  The wavefront takes every W-th step of 32 columns from step `wave` on.
// Returns false if a coordinate was met that the form cannot take (see grid_table).  A value of rhs that
// is not finite makes its column's results NaN whatever its distance to the rows (zero times it is NaN):
// the column's shift is then KM_GRID_NOT_FINITE, and the rhs values of steps out of reach are looked at
// as well (by the caller if not GRID).
// A step's rhs values are requested a step ahead (a step is short: two or three tiles), a chunk's
// coordinates a chunk ahead (the first chunk's, in xv, by the caller).
// PACK (spectral, at most 8 rhs columns): lanes 0 .. 7 of a group hold the columns' cosine parts, lanes
// 8 .. 15 their sine parts.
template <bool GRID, int KT, int G, int MT, int W, bool PACK = false, bool EXACT = false, int CH = GRID && G == 1 ? KM_GRID_CHUNK_ONE : KM_GRID_CHUNK>
__device__ __forceinline__ bool grid_columns(const GridVectors& a, float* __restrict__ tab, const WaveView& w, int kbase,
                                             int wave, const GridWindow& gw, const KernelConsts& kc, const float* xr,
                                             int tiles, float (&xv)[CH / 64], int (&shift)[G],
                                             float4v (&acc)[MT][G * (KT == KM_KERNEL_SPECTRAL && !PACK ? 2 : 1)]) {
    constexpr bool PHASE = KT == KM_KERNEL_SPECTRAL;
    constexpr int PARTS = PHASE && !PACK ? 2 : 1;
    static_assert(!PACK || (PHASE && G == 1 && GRID), "packed: eight rhs columns, cosine and sine part in one group");
    const int lane = threadIdx.x & 63;
    const int li = lane & 15;
    const int kk = lane >> 4;
    const float* __restrict__ rhs = w.rhs + (long long)kbase * a.rhs_s1;
    const RhsLane<G> rl = rhs_lane<G, PACK>(a, kbase);
    const int weights = PACK && li >= 8 ? 2 * CH : CH;
    float scale[G];
#pragma unroll
    for (int g = 0; g < G; g++) {
        shift[g] = 100;
        scale[g] = rl.used[g] ? __builtin_ldexpf(1.0f, 100) : 0.0f;
    }
#pragma unroll
    for (int m = 0; m < MT; m++) {
#pragma unroll
        for (int g = 0; g < G * PARTS; g++) {
            acc[m][g] = (float4v){0.0f, 0.0f, 0.0f, 0.0f};
        }
    }
    const float t0 = (gw.g_lo + (float)li) * gw.h;
    bool fine = true;
    // Looked at after each chunk for one group of rhs columns, behind all of them for more (n = 1e5, k = 16:
    // 63.4 against 65.3 us; n = 1e6, k = 32: 876 against 859 us; rbf n = 65536, k = 64: 25.7 against 22.7 us).
    constexpr bool EACH_CHUNK = G == 1;
    BeyondSteps beyond = {0, 64, 0};
    int chunk = 0;
    bool first_step = true;
    constexpr int STEPS = CH / 32;  // of a chunk
    static_assert(64 % STEPS == 0, "whole chunks' bits");
    // (unsigned: the next first column may lie past the largest int)
    for (unsigned next_first = w.range_start + 32u * wave; next_first < (unsigned)w.range_end; next_first += CH * W) {
        const int first = (int)next_first;
        // (the first step's values, mostly needed, are on their way while the table is made)
        float next[G][8];
        grid_rhs<G>(a, rhs, first, w.range_end, kk, rl, next);
        unsigned long long reached = 0;
        const unsigned steps = grid_table<GRID, PHASE>(xv, first, W, w.range_end, gw, kc, tab, &fine, &reached);
        if (next_first + CH * W < (unsigned)w.range_end) {
            grid_load(w.x2, a.x2_s, first + CH * W, W, w.range_end, xv);
        }
        unsigned need = steps & 0xffff;
        if (!GRID) {
            // (the caller has looked at all steps)
        } else if (EACH_CHUNK) {
            const int present = min((w.range_end - 1 - first) / (32 * W) + 1, STEPS);
            look_at_steps<G>(a, w, kbase, first, 32 * W, {~need & ((1u << present) - 1), 0, 0}, rl, shift, scale);
        } else if (chunk < 64 / STEPS) {
            beyond.bits |= (unsigned long long)(~need & ((1u << STEPS) - 1)) << (STEPS * chunk);
        }
        chunk++;
        if (need == 0) {
            continue;
        }
        int j = __builtin_ctz(need);
        if (j != 0) {
            grid_rhs<G>(a, rhs, first + 32 * j * W, w.range_end, kk, rl, next);
        }
        // (the first step is no code of its own: that was a fifth more instructions and 5 % of the time of rbf n = 1e5,
        // k = 64, 2 sets entry by entry)
#pragma nounroll
        do {
            float raw[G][8];
#pragma unroll
            for (int g = 0; g < G; g++) {
#pragma unroll
                for (int t = 0; t < 8; t++) {
                    raw[g][t] = next[g][t];
                }
            }
            if (!GRID && PARTS == 1 && first + 32 * (j * W + 1) > w.range_end) {  // (no column factors to do it)
                const int last = w.range_end - 1 - first - 32 * j * W;
#pragma unroll
                for (int g = 0; g < G; g++) {
#pragma unroll
                    for (int t = 0; t < 8; t++) {
                        raw[g][t] = 8 * kk + t <= last ? raw[g][t] : 0.0f;
                    }
                }
            }
            const int off = 32 * j + 8 * kk;
            const bool wide = (steps >> (16 + j) & 1) != 0;
            const unsigned points = (unsigned)(reached >> (8 * j)) & 0xff;
            need &= need - 1;
            if (need != 0) {
                j = __builtin_ctz(need);
                grid_rhs<G>(a, rhs, first + 32 * j * W, w.range_end, kk, rl, next);
            }
            // (kept as register quadruples: read element by element below, the accumulators are split
            // up and put together again in every step otherwise)
#pragma unroll
            for (int m = 0; m < MT; m++) {
#pragma unroll
                for (int g = 0; g < G * PARTS; g++) {
                    asm volatile("" : "+v"(acc[m][g]));
                }
            }
#pragma unroll
            for (int g = 0; g < G; g++) {
                lower_scale<G, PARTS, MT>(g, magnitude(raw[g]), rl.used[g], first_step, shift, scale, acc);
            }
            first_step = false;
            grid_step<GRID, G, PARTS, MT, EXACT, CH, GRID>(tab, off, raw, gw, t0, xr, kc, tiles, points, wide, weights, scale, acc);
        } while (need != 0);
        // All reads of the table are done before the next chunk overwrites it.
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
        __builtin_amdgcn_wave_barrier();
    }

    const int columns = w.range_end - w.range_start - 32 * wave;
    if (GRID && !EACH_CHUNK && columns > 0) {
        beyond.total = (columns - 1) / (32 * W) + 1;
        if (beyond.total < 64) {
            beyond.bits &= (1ull << beyond.total) - 1;
        }
        look_at_steps<G>(a, w, kbase, w.range_start + 32 * wave, 32 * W, beyond, rl, shift, scale);
    }
    return fine;
}

// A group of 16 rows from its accumulators (scaled back by down[]): the two parts of the phase-split form
// combined (with the cosines and sines of the rows' phases), and the masked store.
template <int KT, int G>
__device__ __forceinline__ void grid_store(const FwdArgs& a, const WaveView& w, const float (&ca)[4], const float (&sa)[4],
                                           const float4v* res, const float* down, int row, int kbase) {
    constexpr bool PHASE = KT == KM_KERNEL_SPECTRAL;
    const int lane = threadIdx.x & 63;
    const int li = lane & 15;
    const int kk = lane >> 4;
    float* __restrict__ out = a.out + (w.b * (long long)a.m + row) * a.k + kbase;
    auto value = [&](int g, int v) {
        return PHASE ? ca[v] * (res[g][v] * down[g]) + sa[v] * (res[G + g][v] * down[G + g]) : res[g][v] * down[g];
    };
    // Whole groups of rows of moderate width: a scalar base and row offset (no address arithmetic per value).
    if (row + 16 <= a.m && a.k <= (1 << 22)) {
        const buffer_rsrc to = uniform_buffer(out);
        const unsigned lane_bytes = 4u * (__umul24(4u * (unsigned)kk, (unsigned)a.k) + (unsigned)li);
        float result[G][4];
#pragma unroll
        for (int g = 0; g < G; g++) {
#pragma unroll
            for (int v = 0; v < 4; v++) {
                result[g][v] = value(g, v);
            }
        }
        auto store = [&](auto streamed) {
#pragma unroll
            for (int g = 0; g < G; g++) {
                if (kbase + 16 * g + li < a.k) {
#pragma unroll
                    for (int v = 0; v < 4; v++) {
                        __builtin_amdgcn_raw_buffer_store_b32(__float_as_uint(result[g][v]), to, (int)(lane_bytes + 64u * g),
                                                              (int)(4u * (unsigned)v * (unsigned)a.k), streamed ? 2 : 0);
                    }
                }
            }
        };
        if (a.stream_out != 0) {
            store(std::true_type{});
        } else {
            store(std::false_type{});
        }
        return;
    }
#pragma unroll
    for (int g = 0; g < G; g++) {
        const int c = 16 * g + li;
#pragma unroll
        for (int v = 0; v < 4; v++) {
            if (row + 4 * kk + v < a.m && kbase + c < a.k) {
                out[(long long)(4 * kk + v) * a.k + c] = value(g, v);
            }
        }
    }
}

// cos A / sin A of the rows, one held by each lane, in the accumulator layout.
__device__ __forceinline__ void row_phases(float own_cos, float own_sin, int first, float (&ca)[4], float (&sa)[4]) {
    const int kk = (threadIdx.x & 63) >> 4;
#pragma unroll
    for (int v = 0; v < 4; v++) {
        ca[v] = __shfl(own_cos, first + 4 * kk + v, 64);
        sa[v] = __shfl(own_sin, first + 4 * kk + v, 64);
    }
}

}  // namespace km
