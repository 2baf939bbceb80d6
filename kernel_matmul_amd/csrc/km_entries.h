// Forward operator entry by entry from column tables, shared by the kernels of km_periodic.hip, km_grid_f32.hip and km_grid.hip.
#pragma once

#include "km_common.h"
#include "km_fwd.h"
#include "km_grid.h"

namespace km {

#define KM_ENTRY_CHUNK 128
#define KM_ENTRY_CL 8.0f      /* up to here the cosine itself */
#define KM_ENTRY_SPAN 1.375f /* |b|: entries without 2^(-b^2), times 2^14, stay below fp16's largest value */
#define KM_ENTRY_REACH_SQUARED_F32 150.0f /* fp32 entries are zero from there on, denormal ones too */
// A wavefront's table: per column 2 b (or its coordinate), factor, cosine and sine of its phase (or the coordinate's
// remainder), and the smallest and largest coordinate of each 8.
#define KM_ENTRY_FACTOR KM_ENTRY_CHUNK
#define KM_ENTRY_COS (2 * KM_ENTRY_CHUNK)
#define KM_ENTRY_SIN (3 * KM_ENTRY_CHUNK)
#define KM_ENTRY_ENDS (4 * KM_ENTRY_CHUNK)
#define KM_ENTRY_TABLE (4 * KM_ENTRY_CHUNK + 2 * KM_ENTRY_CHUNK / 8)

// The rows of a wavefront, as A operand rows: lane % 16 of each group.
template <int R>
struct EntryRows {
    float y[R], rest[R];      // relative to the origin, and what that rounded off
    float cos[R], sin[R];     // locally periodic: of the phase, times cl / 2; steep: of half the phase, times sqrt(cl)
    float origin, lo, hi;     // (the same in every lane)
    bool finite, exact;       // coordinates; all remainders zero
};

// How the entries are formed.  (rbf and spectral ones always directly: they come here where a row block spreads so far
// that tables do not pay, and the error against 64 bits of a cosine made of two tabulated phases would be the larger, 1.9e-7
// against 1.3e-7 in the 2-norm at 2 points per unit.)
struct EntryForm {
    float turns;     // of the tabulated phases, per unit
    float constant;  // of the exponent
    bool steep, direct;
};

template <int KT>
__device__ __forceinline__ EntryForm entry_form(const KernelConsts& kc) {
    EntryForm form;
    form.direct = KT != KM_KERNEL_LOCALLY_PERIODIC ||
                  __builtin_amdgcn_readfirstlane(!(is_finite(kc.s) && is_finite(kc.f) && kc.cl >= 0.0f && is_finite(kc.cl))) != 0;
    form.steep = __builtin_amdgcn_readfirstlane(kc.cl > KM_ENTRY_CL) != 0;
    form.turns = form.steep ? kc.f : 2.0f * kc.f;
    form.constant = form.steep ? 0.0f : -0.5f * kc.cl;
    return form;
}

// What the subtraction of the origin rounded off (none of it where the difference is infinite).
template <bool F32>
__device__ __forceinline__ float entry_rest(float x, float origin, float y) {
    const float rest = remainder_of(x, origin, y);
    return !F32 || is_finite(y) ? rest : 0.0f;
}

template <int KT, bool F32, int R>
__device__ __forceinline__ EntryRows<R> entry_rows(const FwdArgs& a, const WaveView& w, int row0, const KernelConsts& kc,
                                                        const EntryForm& form) {
    const int li = threadIdx.x & 15;
    EntryRows<R> p;
    float x[R];
#pragma unroll
    for (int r = 0; r < R; r++) {
        // (unsigned: rows of a last block may lie past the largest int)
        x[r] = w.x1[(long long)min((unsigned)row0 + 16 * r + li, (unsigned)a.m - 1) * a.x1_s];
    }
    // (rbf and spectral entries take the difference of the coordinates themselves)
    p.origin = KT == KM_KERNEL_LOCALLY_PERIODIC ? uniform(x[R / 2]) : 0.0f;
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
        p.rest[r] = KT == KM_KERNEL_LOCALLY_PERIODIC ? entry_rest<F32>(x[r], p.origin, p.y[r]) : 0.0f;
        if (KT == KM_KERNEL_LOCALLY_PERIODIC) {
            const float th = phase_rev(form.turns, x[r], p.origin);
            p.cos[r] = factor * __builtin_amdgcn_cosf(th);
            p.sin[r] = factor * __builtin_amdgcn_sinf(th);
        }
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
template <int KT, bool F32>
__device__ __forceinline__ unsigned entry_table(const float (&xv)[KM_ENTRY_CHUNK / 64], int first, int stride, int end,
                                                   float origin, float col_lo, float col_hi, const EntryForm& form, const KernelConsts& kc,
                                                   float* __restrict__ tab, bool* fine) {
    constexpr int N = KM_ENTRY_CHUNK / 64;
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
        need |= (form.direct ? 3u << (2 * i) : bits(0.5f * (hi[i] - lo[i]) * kc.s > KM_ENTRY_SPAN, i)) << 16;
        ok = ok && (!F32 && KT == KM_KERNEL_RBF ? xv[i] == xv[i] : is_finite(xv[i]));
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
        const float rest = KT == KM_KERNEL_LOCALLY_PERIODIC ? entry_rest<F32>(xv[i], origin, y) : 0.0f;
        exact = exact && rest == 0.0f;
        // (factors zero past the end of the range, where rhs values are those of the last row again)
        if ((need >> (16 + 2 * i) & 3) == 3) {
            tab[q] = y;
            tab[KM_ENTRY_FACTOR + q] = inside ? 1.0f : 0.0f;
            tab[KM_ENTRY_COS + q] = rest;
        } else {
            const float b = ((y - 0.5f * (lo[i] + hi[i])) + rest) * kc.s;
            const float th = phase_rev(form.turns, xv[i], origin);
            tab[q] = plain ? y : b + b;
            tab[KM_ENTRY_FACTOR + q] = !inside ? 0.0f : (plain ? 1.0f : __builtin_amdgcn_exp2f(-b * b));
            tab[KM_ENTRY_COS + q] = plain ? rest : __builtin_amdgcn_cosf(th);
            tab[KM_ENTRY_SIN + q] = __builtin_amdgcn_sinf(th);
        }
        if ((lane & 7) == 0) {
            tab[KM_ENTRY_ENDS + (q >> 3)] = lo[i];
            tab[KM_ENTRY_ENDS + KM_ENTRY_CHUNK / 8 + (q >> 3)] = hi[i];
        }
    }
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
    return need | (__all(exact) ? 0u : 1u << 31);
}

// Two entries split into fp16 halves, times 2^KM_F16_KSCALE_LOG2 (as entry_pair_f16).
__device__ __forceinline__ void entry_values_f16(float v0, float v1, half2v* hi, half2v* lo) {
    constexpr float S = (float)(1 << KM_F16_KSCALE_LOG2);
    const half2v h = __builtin_convertvector((float2v){v0, v1}, half2v) * (half2v){(_Float16)S, (_Float16)S};
    *hi = h;
    *lo = residual_f16x2(v0, S, v1, S, h);
}

// One step of 32 columns against the row groups within reach.  F32: the products are fp32 MFMAs, of which number t
// contracts the columns 8 kk + t, so that a lane evaluates the same 8 columns; valid: how many columns of the step there are.
template <int KT, bool F32, int G, int R>
__device__ __forceinline__ void entry_step(const float* __restrict__ tab, int off, const float (&raw)[G][8],
                                           const EntryRows<R>& rows, float reach, bool plain, bool exact, int valid,
                                           const EntryForm& form, const KernelConsts& kc,
                                           const float (&scale)[G], float4v (&acc)[R][G]) {
    constexpr bool SPECTRAL = KT == KM_KERNEL_SPECTRAL, PERIODIC = KT == KM_KERNEL_LOCALLY_PERIODIC;
    float xv[8], cb[8], sb[8];
    half8v bhi[F32 ? 1 : G], blo[F32 ? 1 : G];
    float bv[F32 ? G : 1][8];
    {
        float wgt[8];
#pragma unroll
        for (int t = 0; t < 8; t += 4) {
            const float4v vw = *(const float4v*)(tab + KM_ENTRY_FACTOR + off + t);
            const float4v vx = *(const float4v*)(tab + off + t);
            const float4v vc = *(const float4v*)(tab + KM_ENTRY_COS + off + t);
            const float4v vs = PERIODIC ? *(const float4v*)(tab + KM_ENTRY_SIN + off + t) : vc;
#pragma unroll
            for (int u = 0; u < 4; u++) {
                wgt[t + u] = vw[u];
                xv[t + u] = vx[u];
                cb[t + u] = vc[u];
                sb[t + u] = vs[u];
            }
        }
        if constexpr (F32) {
            const int kk = (threadIdx.x & 63) >> 4;
#pragma unroll
            for (int g = 0; g < G; g++) {
#pragma unroll
                for (int t = 0; t < 8; t++) {
                    bv[g][t] = raw[g][t] * wgt[t];
                }
                if (valid < 32) {  // (zero times a value that is not finite is not zero)
#pragma unroll
                    for (int t = 0; t < 8; t++) {
                        bv[g][t] = 8 * kk + t < valid ? bv[g][t] : 0.0f;
                    }
                }
            }
        } else {
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
    }
    const float lo = tab[KM_ENTRY_ENDS + (off >> 3)];
    const float hi = tab[KM_ENTRY_ENDS + KM_ENTRY_CHUNK / 8 + (off >> 3)];
    const float middle = 0.5f * (lo + hi);
#pragma unroll
    for (int r = 0; r < R; r++) {
        if (!__any(!(fmaxf(lo - rows.y[r], rows.y[r] - hi) > reach))) {
            continue;
        }
        float arg[8], cosine[SPECTRAL ? 8 : 1];
        if (PERIODIC && !plain) {
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
            if (PERIODIC && !exact) {
#pragma unroll
                for (int t = 0; t < 8; t++) {
                    d[t] += rows.rest[r] - cb[t];
                }
            }
#pragma unroll
            for (int t = 0; t < 8; t++) {
                const float u = d[t] * kc.s;
                arg[t] = -u * u;
                // (the phase rounded as what is left of it beyond whole turns)
                if constexpr (SPECTRAL) {
                    cosine[t] = __builtin_amdgcn_cosf(__builtin_fmaf(d[t], kc.f, -__builtin_rintf(d[t] * kc.f)));
                } else if constexpr (PERIODIC) {
                    const float sn = __builtin_amdgcn_sinf(F32 ? __builtin_fmaf(d[t], kc.f, -__builtin_rintf(d[t] * kc.f)) : d[t] * kc.f);
                    arg[t] = __builtin_fmaf(-(sn * kc.cl), sn, arg[t]);
                }
            }
        }
        if constexpr (F32) {
#pragma unroll
            for (int t = 0; t < 8; t++) {
                const float e = __builtin_amdgcn_exp2f(arg[t]);
                arg[t] = SPECTRAL ? e * cosine[SPECTRAL ? t : 0] : e;
            }
#pragma unroll
            for (int t = 0; t < 8; t++) {
#pragma unroll
                for (int g = 0; g < G; g++) {
                    acc[r][g] = __builtin_amdgcn_mfma_f32_16x16x4f32(arg[t], bv[g][t], acc[r][g], 0, 0, 0);
                }
            }
        } else {
            half2v h2[4], l2[4];
#pragma unroll
            for (int u = 0; u < 4; u++) {
                float v0 = __builtin_amdgcn_exp2f(arg[2 * u]), v1 = __builtin_amdgcn_exp2f(arg[2 * u + 1]);
                if (SPECTRAL) {
                    v0 *= cosine[SPECTRAL ? 2 * u : 0];
                    v1 *= cosine[SPECTRAL ? 2 * u + 1 : 0];
                }
                entry_values_f16(v0, v1, &h2[u], &l2[u]);
            }
            const half8v ahi = join_half2x4(h2);
            const half8v alo = join_half2x4(l2);
#pragma unroll
            for (int g = 0; g < G; g++) {
                acc[r][g] = __builtin_amdgcn_mfma_f32_16x16x32_f16(ahi, bhi[g], acc[r][g], 0, 0, 0);
                acc[r][g] = __builtin_amdgcn_mfma_f32_16x16x32_f16(ahi, blo[g], acc[r][g], 0, 0, 0);
                acc[r][g] = __builtin_amdgcn_mfma_f32_16x16x32_f16(alo, bhi[g], acc[r][g], 0, 0, 0);
            }
        }
        __builtin_amdgcn_sched_barrier(0);
    }
}

// LDS in floats: the wavefronts' tables, overlaid by the exchange of their sums, and a word of each.
constexpr int entry_exchange_floats(int G, int R, int W) {
    return W == 1 ? KM_ENTRY_TABLE : (W * KM_ENTRY_TABLE > W * R * G * 256 ? W * KM_ENTRY_TABLE : W * R * G * 256);
}
constexpr int entry_lds_floats(int G, int R, int W) { return entry_exchange_floats(G, R, W) + W; }

// One item: rows [row0, row0 + 16 R) by W wavefronts, this one number `wave`.
template <int KT, bool F32, int G, int R, int W>
__device__ __forceinline__ void entry_item(const FwdArgs& a, float* lds, const WaveView& w, int row0, int kbase, int wave) {
    constexpr int CH = KM_ENTRY_CHUNK;
    constexpr int STEPS = CH / 32;
    const int lane = threadIdx.x & 63;
    const int li = lane & 15;
    const int kk = lane >> 4;
    float* const tab = lds + wave * KM_ENTRY_TABLE;
    const GridVectors vec = {a.x2_s, a.rhs_s0, a.rhs_s1, a.k};
    const KernelConsts kc = make_consts<KT>(w.params, a.params_s, false);
    float xv[CH / 64];
    const bool any = 32 * wave < w.range_end - w.range_start;
    if (any) {
        grid_load(w.x2, a.x2_s, w.range_start + 32 * wave, W, w.range_end, xv);
    }
    EntryForm form = entry_form<KT>(kc);
    const EntryRows<R> rows = entry_rows<KT, F32, R>(a, w, row0, kc, form);
    form.direct = form.direct || (F32 && !rows.finite);
    float reach = __builtin_inff();
    if (rows.finite) {
        if constexpr (!F32) {
            reach = periodic_reach(kc);
        } else if (is_finite(kc.f) && is_finite(kc.cl)) {
            reach = __builtin_sqrtf(KM_ENTRY_REACH_SQUARED_F32 + fmaxf(0.0f, -kc.cl)) / kc.s;
        }
    }
    reach = uniform(reach);

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
    bool fine = true, first_step = true;
    float largest = 0.0f;
    // F32: once more without anything left out if a value is not finite.
#pragma unroll 1
    for (;;) {
        const float col_lo = uniform(rows.lo - reach), col_hi = uniform(rows.hi + reach);
#pragma unroll
        for (int r = 0; r < R; r++) {
#pragma unroll
            for (int g = 0; g < G; g++) {
                acc[r][g] = (float4v){0.0f, 0.0f, 0.0f, 0.0f};
            }
        }
        // (unsigned: the next first column may lie past the largest int)
        for (unsigned next_first = w.range_start + 32u * wave; any && next_first < (unsigned)w.range_end; next_first += CH * W) {
            const int first = (int)next_first;
            float next[G][8];
            grid_rhs<G>(vec, rhs, first, w.range_end, kk, rl, next);
            const unsigned steps = entry_table<KT, F32>(xv, first, W, w.range_end, rows.origin, col_lo, col_hi, form, kc, tab, &fine);
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
                const int valid = w.range_end - first - 32 * j * W;
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
                    if constexpr (F32) {
                        largest = __builtin_elementwise_maximum(largest, magnitude(raw[g]));
                    } else {
                        lower_scale<G, 1, R>(g, magnitude(raw[g]), rl.used[g], first_step, shift, scale, acc);
                    }
                }
                first_step = false;
                entry_step<KT, F32, G, R>(tab, off, raw, rows, reach, plain, exact, valid, form, kc, scale, acc);
            } while (need != 0);
            // All reads of the table are done before the next chunk overwrites it.
            __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
            __builtin_amdgcn_wave_barrier();
        }
        if constexpr (F32) {
            bool bad = !fine || !__all(is_finite(largest));
#pragma unroll
            for (int g = 0; g < G; g++) {
                bad = bad || __any(shift[g] == KM_GRID_NOT_FINITE);
            }
            if constexpr (W > 1) {
                unsigned* const words = (unsigned*)(lds + entry_exchange_floats(G, R, W));
                if (lane == 0) {
                    words[wave] = bad ? 1 : 0;
                }
                __syncthreads();
#pragma unroll
                for (int v = 0; v < W; v++) {
                    bad = bad || __builtin_amdgcn_readfirstlane(words[v]) != 0;
                }
            }
            if (bad && !(reach == __builtin_inff() && form.direct)) {  // (the same in all wavefronts)
                reach = __builtin_inff();
                form.direct = true;
                if constexpr (W > 1) {
                    __syncthreads();  // (the words are written anew)
                }
                if (any) {
                    grid_load(w.x2, a.x2_s, w.range_start + 32 * wave, W, w.range_end, xv);
                }
                continue;
            }
        }
        break;
    }

    const float sigma = w.params[KernelTraits<KT>::SIGMA * a.params_s];
    float down[G];
#pragma unroll
    for (int g = 0; g < G; g++) {
        down[g] = F32 ? sigma : fine && shift[g] != KM_GRID_NOT_FINITE ? __builtin_ldexpf(sigma, -shift[g] - KM_F16_KSCALE_LOG2) : __builtin_nanf("");
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

}  // namespace km
