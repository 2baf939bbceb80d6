// Forward operator for locally periodic kernels with the periodic factor from tabulated phases.  With A and B the
// phases of a row and a column about the row block's middle row (in turns of the period),
//     K / sigma = 2^(-u^2 - cl / 2 + (cl / 2) cos(A - B)),   cos(A - B) = cos A cos B + sin A sin B,
// and, with r halfway between the ends of each group of 8 columns, a = (x1 - r) s and b = (x2 - r) s,
//     -u^2 = -a^2 + 2 a b - b^2:
// an entry is three fused multiply-adds onto -a^2 - cl / 2 and one exponential; 2^(-b^2) goes into the rhs operand.
// Where cl / 2 times the rounding of a cosine would be more than the exponent's own (cl > 8, second lengthscales below
// 0.36) it is the square of sqrt(cl) sin((A - B) / 2) from the halved phases, one multiplication more.  Evaluated
// directly (fwd_mfma_f16) an entry takes six multiplications and additions and two transcendentals.
//
// A row block of 128 rows is one item, whose steps of 32 columns W wavefronts take in turn; each wavefront keeps the
// sums of all its rows (R groups of 16), and with W > 1 they meet in LDS, added in a fixed order.  Both factors of the
// contraction are split into two fp16 terms as in the other split-fp16 kernels, tiles of 16 rows by 32 columns whose
// entries all round to zero are left out (km_fwd.h), and a value that is not finite reaches what it reaches in a dense
// product.
//
// Steps that take an entry's difference directly: those of which a group of 8 columns spreads further than
// KM_PERIODIC_SPAN (a gap in the data), and all of them where cl is negative or a parameter not finite.
//
// Bound by VALU issue.  Measured against the direct evaluation (a call, k = 16, cutoff of 6 lengthscales, at 10 points per
// unit): n = 50021, 8 sets 73.4 -> 50.2 us, n = 1e6 922 -> 614, n = 20000, 4 sets 35.7 -> 18.8; error against 64 bits (2-norm,
// 2 to 300 points per unit) 2.2e-7 to 5.3e-7 -> 1.2e-7 to 3.5e-7: the power of two that the fp16 halves need is no part of
// the exponent.  Every wavefront prepares its own rhs operand; where four row blocks shared one (km_matmul_block.hip) the
// barriers cost more than that saved.
#include "km_batch.h"
#include "km_common.h"
#include "km_fwd.h"
#include "km_grid.h"
#include "km_launch.h"

namespace km {

#define KM_PERIODIC_CHUNK 128
#define KM_PERIODIC_CL 8.0f      /* up to here the cosine itself */
#define KM_PERIODIC_SPAN 1.375f /* |b|: entries without 2^(-b^2), times 2^14, stay below fp16's largest value */
// A wavefront's table: per column 2 b (or its coordinate), factor, cosine and sine of its phase (or the coordinate's
// remainder), and the smallest and largest coordinate of each 8.
#define KM_PERIODIC_FACTOR KM_PERIODIC_CHUNK
#define KM_PERIODIC_COS (2 * KM_PERIODIC_CHUNK)
#define KM_PERIODIC_SIN (3 * KM_PERIODIC_CHUNK)
#define KM_PERIODIC_ENDS (4 * KM_PERIODIC_CHUNK)
#define KM_PERIODIC_TABLE (4 * KM_PERIODIC_CHUNK + 2 * KM_PERIODIC_CHUNK / 8)

// The rows of a wavefront, as A operand rows: lane % 16 of each group.
template <int R>
struct PeriodicRows {
    float y[R], rest[R];      // relative to the origin, and what that rounded off
    float cos[R], sin[R];     // of the phase, times cl / 2; steep: of half the phase, times sqrt(cl)
    float origin, lo, hi;     // (the same in every lane)
    bool finite, exact;       // coordinates; all remainders zero
};

// How the entries are formed.
struct PeriodicForm {
    float turns;     // of the tabulated phases, per unit
    float constant;  // of the exponent
    bool steep, direct;
};

template <int R>
__device__ __forceinline__ PeriodicRows<R> periodic_rows(const FwdArgs& a, const WaveView& w, int row0, const KernelConsts& kc,
                                                        const PeriodicForm& form) {
    const int li = threadIdx.x & 15;
    PeriodicRows<R> p;
    float x[R];
#pragma unroll
    for (int r = 0; r < R; r++) {
        // (unsigned: rows of a last block may lie past the largest int)
        x[r] = w.x1[(long long)min((unsigned)row0 + 16 * r + li, (unsigned)a.m - 1) * a.x1_s];
    }
    p.origin = uniform(x[R / 2]);
    if (!is_finite(p.origin)) {
        // Any row that is: the origin must not hand its value on to the other rows.
        p.origin = 0.0f;
#pragma unroll
        for (int r = 0; r < R; r++) {
            const unsigned long long in = __ballot(is_finite(x[r]));
            p.origin = in != 0 ? uniform(__shfl(x[r], in != 0 ? __builtin_ctzll(in) : 0, 64)) : p.origin;
        }
    }
    bool finite = true, exact = true;
    p.lo = __builtin_inff();
    p.hi = -__builtin_inff();
    const float factor = form.steep ? __builtin_sqrtf(kc.cl) : 0.5f * kc.cl;
#pragma unroll
    for (int r = 0; r < R; r++) {
        p.y[r] = x[r] - p.origin;
        p.rest[r] = remainder_of(x[r], p.origin, p.y[r]);
        const float th = phase_rev(form.turns, x[r], p.origin);
        p.cos[r] = factor * __builtin_amdgcn_cosf(th);
        p.sin[r] = factor * __builtin_amdgcn_sinf(th);
        p.lo = fminf(p.lo, p.y[r]);
        p.hi = fmaxf(p.hi, p.y[r]);
        finite = finite && fabsf(p.y[r]) < 1e30f;
        exact = exact && p.rest[r] == 0.0f;
    }
    wave_min_max(&p.lo, &p.hi);
    p.finite = __all(finite);
    p.exact = __all(exact);
    return p;
}

// Tabulates this wavefront's next steps of 32 columns (first / 32 + j * stride of the range); returns the ones within
// reach [col_lo, col_hi] as bits, in the upper half those whose entries are evaluated directly, and as the highest bit
// whether a remainder is not zero.  *fine is cleared when a coordinate makes every entry of its column NaN.
__device__ __forceinline__ unsigned periodic_table(const float (&xv)[KM_PERIODIC_CHUNK / 64], int first, int stride, int end,
                                                   float origin, float col_lo, float col_hi, const PeriodicForm& form, const KernelConsts& kc,
                                                   float* __restrict__ tab, bool* fine) {
    constexpr int N = KM_PERIODIC_CHUNK / 64;
    const int lane = threadIdx.x & 63;
    const int last = end - 1 - first;
    float lo[N], hi[N];
    unsigned need = 0;
    bool ok = true, exact = true;
    static_assert(2 * N < 15, "the highest bit is free");
    auto bits = [](bool lanes, int i) {
        const unsigned long long any = __ballot(lanes);
        return (unsigned)((any & 0xffffffffull) != 0) << (2 * i) | (unsigned)((any >> 32) != 0) << (2 * i + 1);
    };
#pragma unroll
    for (int i = 0; i < N; i++) {
        const int rel = 32 * ((lane >> 5) + 2 * i) * stride + (lane & 31);
        const float y = xv[i] - origin;
        need |= bits(rel <= last && !(y < col_lo || y > col_hi), i);
        group8_min_max(y, &lo[i], &hi[i]);
        need |= (form.direct ? 3u << (2 * i) : bits(0.5f * (hi[i] - lo[i]) * kc.s > KM_PERIODIC_SPAN, i)) << 16;
        ok = ok && is_finite(xv[i]);
    }
    need = __builtin_amdgcn_readfirstlane(need);
    *fine = *fine && __all(ok);
#pragma unroll
    for (int i = 0; i < N; i++) {
        if ((need >> (2 * i) & 3) == 0) {
            continue;
        }
        const int q = lane + 64 * i;
        const bool plain = (need >> (16 + 2 * i + (lane >> 5)) & 1) != 0;
        const bool inside = 32 * ((lane >> 5) + 2 * i) * stride + (lane & 31) <= last;
        const float y = xv[i] - origin;
        const float rest = remainder_of(xv[i], origin, y);
        exact = exact && rest == 0.0f;
        // (factors zero past the end of the range, where rhs values are those of the last row again)
        if ((need >> (16 + 2 * i) & 3) == 3) {
            tab[q] = y;
            tab[KM_PERIODIC_FACTOR + q] = inside ? 1.0f : 0.0f;
            tab[KM_PERIODIC_COS + q] = rest;
        } else {
            const float b = ((y - 0.5f * (lo[i] + hi[i])) + rest) * kc.s;
            const float th = phase_rev(form.turns, xv[i], origin);
            tab[q] = plain ? y : b + b;
            tab[KM_PERIODIC_FACTOR + q] = !inside ? 0.0f : (plain ? 1.0f : __builtin_amdgcn_exp2f(-b * b));
            tab[KM_PERIODIC_COS + q] = plain ? rest : __builtin_amdgcn_cosf(th);
            tab[KM_PERIODIC_SIN + q] = __builtin_amdgcn_sinf(th);
        }
        if ((lane & 7) == 0) {
            tab[KM_PERIODIC_ENDS + (q >> 3)] = lo[i];
            tab[KM_PERIODIC_ENDS + KM_PERIODIC_CHUNK / 8 + (q >> 3)] = hi[i];
        }
    }
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
    return need | (__all(exact) ? 0u : 1u << 31);
}

// Two entries from their exponents, split into fp16 halves, times 2^KM_F16_KSCALE_LOG2 (as entry_pair_f16).
__device__ __forceinline__ void periodic_pair_f16(float a0, float a1, half2v* hi, half2v* lo) {
    constexpr float S = (float)(1 << KM_F16_KSCALE_LOG2);
    const float2v kv = {__builtin_amdgcn_exp2f(a0), __builtin_amdgcn_exp2f(a1)};
    const half2v h = __builtin_convertvector(kv, half2v) * (half2v){(_Float16)S, (_Float16)S};
    *hi = h;
    *lo = residual_f16x2(kv[0], S, kv[1], S, h);
}

// One step of 32 columns against the row groups within reach.
template <int G, int R>
__device__ __forceinline__ void periodic_step(const float* __restrict__ tab, int off, const float (&raw)[G][8],
                                              const PeriodicRows<R>& rows, float reach, bool plain, bool exact,
                                              const PeriodicForm& form, const KernelConsts& kc,
                                              const float (&scale)[G], float4v (&acc)[R][G]) {
    float xv[8], cb[8], sb[8];
    half8v bhi[G], blo[G];
    {
        float wgt[8];
#pragma unroll
        for (int t = 0; t < 8; t += 4) {
            const float4v vw = *(const float4v*)(tab + KM_PERIODIC_FACTOR + off + t);
            const float4v vx = *(const float4v*)(tab + off + t);
            const float4v vc = *(const float4v*)(tab + KM_PERIODIC_COS + off + t);
            const float4v vs = *(const float4v*)(tab + KM_PERIODIC_SIN + off + t);
#pragma unroll
            for (int u = 0; u < 4; u++) {
                wgt[t + u] = vw[u];
                xv[t + u] = vx[u];
                cb[t + u] = vc[u];
                sb[t + u] = vs[u];
            }
        }
#pragma unroll
        for (int g = 0; g < G; g++) {
            float v[8];
#pragma unroll
            for (int t = 0; t < 8; t++) {
                v[t] = raw[g][t] * scale[g] * wgt[t];
            }
            split_f16x8(v, kc.one, &bhi[g], &blo[g]);
        }
    }
    const float lo = tab[KM_PERIODIC_ENDS + (off >> 3)];
    const float hi = tab[KM_PERIODIC_ENDS + KM_PERIODIC_CHUNK / 8 + (off >> 3)];
    const float middle = 0.5f * (lo + hi);
#pragma unroll
    for (int r = 0; r < R; r++) {
        if (!__any(!(fmaxf(lo - rows.y[r], rows.y[r] - hi) > reach))) {
            continue;
        }
        float arg[8];
        if (!plain) {
            const float av = ((rows.y[r] - middle) + rows.rest[r]) * kc.s;
            const float rb = __builtin_fmaf(-av, av, form.constant);
#pragma unroll
            for (int t = 0; t < 8; t++) {
                arg[t] = __builtin_fmaf(av, xv[t], rb);
            }
            if (!form.steep) {
#pragma unroll
                for (int t = 0; t < 8; t++) {
                    arg[t] = __builtin_fmaf(rows.sin[r], sb[t], __builtin_fmaf(rows.cos[r], cb[t], arg[t]));
                }
            } else {
#pragma unroll
                for (int t = 0; t < 8; t++) {
                    const float sn = __builtin_fmaf(rows.sin[r], cb[t], -rows.cos[r] * sb[t]);
                    arg[t] = __builtin_fmaf(-sn, sn, arg[t]);
                }
            }
        } else {
            float d[8];
#pragma unroll
            for (int t = 0; t < 8; t++) {
                d[t] = rows.y[r] - xv[t];
            }
            if (!exact) {
#pragma unroll
                for (int t = 0; t < 8; t++) {
                    d[t] += rows.rest[r] - cb[t];
                }
            }
#pragma unroll
            for (int t = 0; t < 8; t++) {
                const float u = d[t] * kc.s;
                const float sn = __builtin_amdgcn_sinf(d[t] * kc.f);
                arg[t] = __builtin_fmaf(-(sn * kc.cl), sn, -u * u);
            }
        }
        half2v h2[4], l2[4];
#pragma unroll
        for (int u = 0; u < 4; u++) {
            periodic_pair_f16(arg[2 * u], arg[2 * u + 1], &h2[u], &l2[u]);
        }
        const half8v ahi = join_half2x4(h2);
        const half8v alo = join_half2x4(l2);
#pragma unroll
        for (int g = 0; g < G; g++) {
            acc[r][g] = __builtin_amdgcn_mfma_f32_16x16x32_f16(ahi, bhi[g], acc[r][g], 0, 0, 0);
            acc[r][g] = __builtin_amdgcn_mfma_f32_16x16x32_f16(ahi, blo[g], acc[r][g], 0, 0, 0);
            acc[r][g] = __builtin_amdgcn_mfma_f32_16x16x32_f16(alo, bhi[g], acc[r][g], 0, 0, 0);
        }
        __builtin_amdgcn_sched_barrier(0);
    }
}

// One item: rows [row0, row0 + 16 R) by W wavefronts, this one number `wave`.
template <int G, int R, int W>
__device__ __forceinline__ void periodic_item(const FwdArgs& a, float* lds, const WaveView& w, int row0, int kbase, int wave) {
    constexpr int CH = KM_PERIODIC_CHUNK;
    constexpr int STEPS = CH / 32;
    const int lane = threadIdx.x & 63;
    const int li = lane & 15;
    const int kk = lane >> 4;
    float* const tab = lds + wave * KM_PERIODIC_TABLE;
    const GridVectors vec = {a.x2_s, a.rhs_s0, a.rhs_s1, a.k};
    const KernelConsts kc = make_consts<KM_KERNEL_LOCALLY_PERIODIC>(w.params, a.params_s, false);
    float xv[CH / 64];
    const bool any = 32 * wave < w.range_end - w.range_start;
    if (any) {
        grid_load(w.x2, a.x2_s, w.range_start + 32 * wave, W, w.range_end, xv);
    }
    PeriodicForm form;
    form.direct = __builtin_amdgcn_readfirstlane(!(kc.cl >= 0.0f && is_finite(kc.cl) && is_finite(kc.f))) != 0;
    form.steep = __builtin_amdgcn_readfirstlane(kc.cl > KM_PERIODIC_CL) != 0;
    form.turns = form.steep ? kc.f : 2.0f * kc.f;
    form.constant = form.steep ? 0.0f : -0.5f * kc.cl;
    const PeriodicRows<R> rows = periodic_rows<R>(a, w, row0, kc, form);
    const float reach = uniform(rows.finite ? periodic_reach(kc) : __builtin_inff());
    const float col_lo = uniform(rows.lo - reach), col_hi = uniform(rows.hi + reach);

    const float* __restrict__ rhs = w.rhs + (long long)kbase * a.rhs_s1;
    const RhsLane<G> rl = rhs_lane<G>(vec, kbase);
    int shift[G];
    float scale[G];
#pragma unroll
    for (int g = 0; g < G; g++) {
        shift[g] = 100;
        scale[g] = rl.used[g] ? __builtin_ldexpf(1.0f, 100) : 0.0f;
    }
    float4v acc[R][G];
#pragma unroll
    for (int r = 0; r < R; r++) {
#pragma unroll
        for (int g = 0; g < G; g++) {
            acc[r][g] = (float4v){0.0f, 0.0f, 0.0f, 0.0f};
        }
    }
    bool fine = true, first_step = true;
    // (unsigned: the next first column may lie past the largest int)
    for (unsigned next_first = w.range_start + 32u * wave; any && next_first < (unsigned)w.range_end; next_first += CH * W) {
        const int first = (int)next_first;
        float next[G][8];
        grid_rhs<G>(vec, rhs, first, w.range_end, kk, rl, next);
        const unsigned steps = periodic_table(xv, first, W, w.range_end, rows.origin, col_lo, col_hi, form, kc, tab, &fine);
        if (next_first + CH * W < (unsigned)w.range_end) {
            grid_load(w.x2, a.x2_s, first + CH * W, W, w.range_end, xv);
        }
        const bool exact = rows.exact && (steps >> 31) == 0;
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
            }
            const int off = 32 * j + 8 * kk;
            const bool plain = (steps >> (16 + j) & 1) != 0;
            need &= need - 1;
            if (need != 0) {
                j = __builtin_ctz(need);
                grid_rhs<G>(vec, rhs, first + 32 * j * W, w.range_end, kk, rl, next);
            }
            // (kept as register quadruples, see grid_columns)
#pragma unroll
            for (int r = 0; r < R; r++) {
#pragma unroll
                for (int g = 0; g < G; g++) {
                    asm volatile("" : "+v"(acc[r][g]));
                }
            }
#pragma unroll
            for (int g = 0; g < G; g++) {
                lower_scale<G, 1, R>(g, magnitude(raw[g]), rl.used[g], first_step, shift, scale, acc);
            }
            first_step = false;
            periodic_step<G, R>(tab, off, raw, rows, reach, plain, exact, form, kc, scale, acc);
        } while (need != 0);
        // All reads of the table are done before the next chunk overwrites it.
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
        __builtin_amdgcn_wave_barrier();
    }

    const float sigma = w.params[KernelTraits<KM_KERNEL_LOCALLY_PERIODIC>::SIGMA * a.params_s];
    float down[G];
#pragma unroll
    for (int g = 0; g < G; g++) {
        down[g] = fine && shift[g] != KM_GRID_NOT_FINITE ? __builtin_ldexpf(sigma, -shift[g] - KM_F16_KSCALE_LOG2) : __builtin_nanf("");
    }
    float* __restrict__ out = a.out + w.b * (long long)a.m * a.k + kbase;
    auto store = [&](int r, int g, const float4v& value) {
        const long long row = (long long)row0 + 16 * r + 4 * kk;
        const int c = 16 * g + li;
        if (kbase + c < a.k) {
#pragma unroll
            for (int v = 0; v < 4; v++) {
                if (row + v < a.m) {
                    out[(row + v) * a.k + c] = value[v];
                }
            }
        }
    };
    if constexpr (W == 1) {
#pragma unroll
        for (int r = 0; r < R; r++) {
#pragma unroll
            for (int g = 0; g < G; g++) {
                store(r, g, acc[r][g] * down[g]);
            }
        }
    } else {
        float4v* part = (float4v*)lds;
        __syncthreads();  // the exchange lies over the tables
#pragma unroll
        for (int r = 0; r < R; r++) {
#pragma unroll
            for (int g = 0; g < G; g++) {
                part[((wave * R + r) * G + g) * 64 + lane] = acc[r][g] * down[g];
            }
        }
        __syncthreads();
        for (int i = wave; i < R * G; i += W) {
            float4v sum = part[i * 64 + lane];
#pragma unroll
            for (int v = 1; v < W; v++) {
                sum += part[(v * R * G + i) * 64 + lane];
            }
            store(i / G, i % G, sum);
        }
    }
}

template <int KT, int G, int R, int W>
__global__ void __launch_bounds__(64 * W, G == 1 ? 3 : 2) fwd_block(const FwdArgs a) {
    extern __shared__ float lds[];
    const long long slot = xcd_item(blockIdx.x, a.items_per_xcd);
    if (slot >= a.total_items) {
        return;
    }
    // (tiles out of reach are left out, so the batch items differ in their work)
    const unsigned batches = (unsigned)a.num_batches;
    const unsigned chunk = (unsigned)slot / batches;
    const long long item = (long long)chunk * batches + spread_batch((unsigned)slot - chunk * batches, chunk, batches);
    int chunk_in_block;
    const WaveView w = wave_view<true>(a, item, a.chunks_per_block, &chunk_in_block);
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    periodic_item<G, R, W>(a, lds, w, w.row_block * KM_BLOCK_SIZE + chunk_in_block * (16 * R), blockIdx.y * G * 16, wave);
}

template <int G, int R, int W>
static hipError_t launch_periodic_as(FwdArgs& a, unsigned grid_y, hipStream_t stream) {
    a.chunks_per_block = KM_BLOCK_SIZE / (16 * R);
    a.total_items = ((long long)a.m + KM_BLOCK_SIZE - 1) / KM_BLOCK_SIZE * a.chunks_per_block * a.num_batches;
    a.items_per_xcd = (a.total_items + KM_NUM_XCD - 1) / KM_NUM_XCD;
    constexpr int EXCHANGE = W == 1 ? 0 : W * R * G * 256;
    constexpr int FLOATS = W * KM_PERIODIC_TABLE > EXCHANGE ? W * KM_PERIODIC_TABLE : EXCHANGE;
    hipLaunchKernelGGL((fwd_block<KM_KERNEL_LOCALLY_PERIODIC, G, R, W>), dim3((unsigned)(a.items_per_xcd * KM_NUM_XCD), grid_y, 1), dim3(64 * W, 1, 1),
                       (sizeof(float) * FLOATS), stream, a);
    return hipGetLastError();
}

template <int G, int R>
static hipError_t launch_periodic_w(FwdArgs& a, const MatmulPlan& plan, unsigned grid_y, hipStream_t stream) {
    if (plan.row_groups < R) {
        return launch_periodic_as<G, R / 2, 8>(a, grid_y, stream);
    }
    switch (plan.col_splits) {
        case 1: return launch_periodic_as<G, R, 1>(a, grid_y, stream);
        case 2: return launch_periodic_as<G, R, 2>(a, grid_y, stream);
        case 4: return launch_periodic_as<G, R, 4>(a, grid_y, stream);
        default: return launch_periodic_as<G, R, 8>(a, grid_y, stream);
    }
}

hipError_t launch_matmul_periodic(const MatmulProblem& p, const MatmulPlan& plan, hipStream_t stream) {
    FwdArgs a;
    fill_fwd_args(p, &a);
    const unsigned grid_y = (unsigned)((p.k + plan.k_chunk - 1) / plan.k_chunk);
    switch (plan.k_chunk / 16) {
        case 1: return plan.row_groups == 2 ? launch_periodic_as<1, 2, 8>(a, grid_y, stream) : launch_periodic_w<1, 8>(a, plan, grid_y, stream);
        case 2: return launch_periodic_w<2, 8>(a, plan, grid_y, stream);
        default: return launch_periodic_w<4, 4>(a, plan, grid_y, stream);
    }
}

}  // namespace km
