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
// reach of V, 20 to 60 points) instead of one entry per row and column of the pattern.  The column
// ranges [start, end) are honoured exactly: each row block sums the columns of its own range.
//
// Coordinates are taken relative to the row block's middle row (exact for neighbouring points; the
// column side carries the rounding of that difference as a second term) and h is rounded to 12
// significant bits, so that all g h are exact.  Scaled coordinates z = x s2 (s2 = sqrt(log2 e) / l)
// make V(x, t) = 2^-(z_x - z_t)^2.
#pragma once

#include "km_common.h"
#include "km_fwd.h"

namespace km {

#define KM_GRID_STEP 0.64f          /* h s2: trapezoid error 2 exp(-7.119 / 0.64^2) = 5.7e-8 */
#define KM_GRID_REACH 6.083f        /* V (and K / sigma) < 2^-37 beyond: the floor of the split-fp16 contraction */
#define KM_GRID_COLUMN_REACH 8.603f /* the same for K / sigma in the coordinates of V: sqrt(2) times as far */
#define KM_GRID_WEIGHT 0.66428247026796f /* C / (h s2) = sqrt(2 ln 2 / pi) */
#define KM_GRID_CHUNK 256           /* columns tabulated at a time, per wavefront */
#define KM_GRID_KS1 11              /* V is evaluated times 2^11 (columns: reference within 2) ... */
#define KM_GRID_SPAN 2.0f
#define KM_GRID_KS2 10              /* ... and 2^10 (rows: reference within 3.5 h s2 = 2.24) */
// Table of a chunk: coordinate, the two column factors, and per 8 columns the reference and its span.
#define KM_GRID_TABLE_FLOATS (3 * KM_GRID_CHUNK + 2 * KM_GRID_CHUNK / 8)

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
    int tiles;         // groups of 16 grid points
};

// The rows of a block, two per lane, and its middle row.
struct BlockRows {
    float xa, xb, middle;
};

__device__ __forceinline__ BlockRows block_rows(const float* __restrict__ x1, long long x1_s, int row0, int m) {
    const int lane = threadIdx.x & 63;
    BlockRows r;
    r.xa = x1[(long long)min(row0 + lane, m - 1) * x1_s];
    r.xb = x1[(long long)min(row0 + 64 + lane, m - 1) * x1_s];
    r.middle = x1[(long long)min(row0 + 64, m - 1) * x1_s];
    return r;
}

template <int MT>
__device__ __forceinline__ GridWindow grid_window(const BlockRows& rows, const KernelConsts& kc) {
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
    gw.h = uniform(__uint_as_float(__float_as_uint(KM_GRID_STEP * inv) & 0xfffff000u));
    const float inv_h = __builtin_amdgcn_rcpf(gw.h);
    const float reach = KM_GRID_REACH * inv;
    gw.g_lo = uniform(floorf((lo - reach) * inv_h));
    const float g_hi = ceilf((hi + reach) * inv_h);
    // (false for a spacing of zero, infinity or NaN as well)
    gw.ok = finite && gw.h > 1e-30f && gw.h < 1e30f && g_hi - gw.g_lo < (float)(16 * MT);
    gw.tiles = gw.ok ? ((int)(g_hi - gw.g_lo) + 16) / 16 : 0;
    gw.tiles = __builtin_amdgcn_readfirstlane(gw.tiles);
    const float cr = KM_GRID_COLUMN_REACH * inv;
    gw.col_lo = uniform(finite ? lo - cr : -__builtin_inff());
    gw.col_hi = uniform(finite ? hi + cr : __builtin_inff());
    return gw;
}

// Smallest and largest value within groups of 8 lanes.
__device__ __forceinline__ void group8_min_max(float v, float* lo, float* hi) {
    float a = v, b = v;
#define KM_DPP_STEP(ctrl)                                                                              \
    a = fminf(a, __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(__builtin_bit_cast(int, a),     \
                                                                       __builtin_bit_cast(int, a), ctrl, 0xf, 0xf, false))); \
    b = fmaxf(b, __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(__builtin_bit_cast(int, b),     \
                                                                       __builtin_bit_cast(int, b), ctrl, 0xf, 0xf, false)))
    KM_DPP_STEP(0xb1);   // quad_perm [1, 0, 3, 2]
    KM_DPP_STEP(0x4e);   // quad_perm [2, 3, 0, 1]
    KM_DPP_STEP(0x141);  // row_half_mirror
#undef KM_DPP_STEP
    *lo = a;
    *hi = b;
}

// Coordinates of this wavefront's next 8 steps of 32 columns, in the order grid_table takes them.
__device__ __forceinline__ void grid_load(const float* __restrict__ x2, long long x2_s, int first, int stride, int end,
                                          float (&xv)[KM_GRID_CHUNK / 64]) {
    const int lane = threadIdx.x & 63;
    const float* xc = x2 + (long long)first * x2_s;
    const int last = end - 1 - first;
#pragma unroll
    for (int i = 0; i < KM_GRID_CHUNK / 64; i++) {
        const int rel = 32 * ((lane >> 5) + 2 * i) * stride + (lane & 31);
        xv[i] = xc[(unsigned long long)(unsigned)min(rel, last) * (unsigned)x2_s];
    }
}

// Tabulates this wavefront's next 8 steps of 32 columns (the steps first / 32 + j * stride of the
// range, j = 0 .. 7: several wavefronts that share a range take its steps in turn).  Returns the
// steps that reach the rows as a bit mask.
//   GRID: coordinates as 2 b, b = (y - r) s2 with r in the middle of each group of 8 columns, the
//         column factors times 2^(-b^2).  Steps of which a group spreads further than KM_GRID_SPAN
//         (a gap in the data) come back in the upper half of the mask; their factors lack 2^(-b^2)
//         (it would leave the fp16 range).  *fine is cleared when a coordinate is not finite.
//   else: the coordinates themselves, spans in units of 1 / s (entry-wise evaluation).
template <bool GRID, bool PHASE>
__device__ __forceinline__ unsigned grid_table(const float (&xv)[KM_GRID_CHUNK / 64], int first, int stride, int end,
                                               const GridWindow& gw, const KernelConsts& kc, float* __restrict__ tab,
                                               bool* fine) {
    constexpr int CH = KM_GRID_CHUNK;
    constexpr int N = CH / 64;
    const int lane = threadIdx.x & 63;
    const int last = end - 1 - first;
    float b[N], ref[N], span[N];
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
        float lo, hi;
        group8_min_max(GRID ? y : xv[i], &lo, &hi);
        ref[i] = 0.5f * (lo + hi);
        if (GRID) {
            // the difference to the origin as a sum of two terms: what the subtraction rounded off
            const float bb = y - xv[i];
            const float rest = (xv[i] - (y - bb)) - (gw.x_ref + bb);
            b[i] = ((y - ref[i]) + rest) * gw.s2;
            span[i] = 0.5f * (hi - lo) * gw.s2;
            const unsigned w = bits(span[i] > KM_GRID_SPAN, i);
            wide[i] = (w >> (2 * i + (lane >> 5)) & 1) != 0;
            need |= w << 16;
            ok = ok && fabsf(y) < 1e30f;
        } else {
            span[i] = 0.5f * (hi - lo) * kc.s;
        }
    }
    need = __builtin_amdgcn_readfirstlane(need);
    if (GRID) {
        *fine = *fine && __all(ok);
    }
    if ((need & 0xffff) == 0) {
        return 0;
    }
#pragma unroll
    for (int i = 0; i < N; i++) {
        if ((need >> (2 * i) & 3) == 0) {
            continue;
        }
        const int q = lane + 64 * i;
        const float wgt = GRID && !wide[i] ? __builtin_amdgcn_exp2f(-b[i] * b[i]) : 1.0f;
        tab[q] = GRID ? b[i] + b[i] : xv[i];
        if (PHASE) {
            const float th = phase_rev(kc.f, xv[i], gw.x_ref);
            tab[CH + q] = wgt * __builtin_amdgcn_cosf(th);
            tab[2 * CH + q] = wgt * __builtin_amdgcn_sinf(th);
        } else {
            tab[CH + q] = wgt;
        }
        if ((lane & 7) == 0) {
            tab[3 * CH + (q >> 3)] = ref[i];
            tab[3 * CH + CH / 8 + (q >> 3)] = span[i];
        }
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

}  // namespace km
