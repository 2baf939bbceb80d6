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
// KM_ENTRY_SPAN (a gap in the data), and all of them where cl is negative or a parameter not finite.
//
// Bound by VALU issue.  Measured against the direct evaluation (a call, k = 16, cutoff of 6 lengthscales, at 10 points per
// unit): n = 50021, 8 sets 73.4 -> 50.2 us, n = 1e6 922 -> 614, n = 20000, 4 sets 35.7 -> 18.8; error against 64 bits (2-norm,
// 2 to 300 points per unit) 2.2e-7 to 5.3e-7 -> 1.2e-7 to 3.5e-7: the power of two that the fp16 halves need is no part of
// the exponent.  Every wavefront prepares its own rhs operand; where four row blocks shared one (km_matmul_block.hip) the
// barriers cost more than that saved.
#include "km_batch.h"
#include "km_common.h"
#include "km_fwd.h"
#include "km_entries.h"
#include "km_launch.h"

namespace km {

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
    entry_item<KT, false, G, R, W>(a, lds, w, w.row_block * KM_BLOCK_SIZE + chunk_in_block * (16 * R), blockIdx.y * G * 16, wave);
}

// Few row blocks: their ranges in shares (launch_sum_shares adds up).
template <int KT, int G>
__global__ void __launch_bounds__(512, G == 1 ? 3 : 2) fwd_block_shares(const FwdArgs a) {
    extern __shared__ float lds[];
    FwdArgs f = a;
    WaveView w;
    if (!share_view(a, &w, &f.out)) {
        return;
    }
    entry_item<KT, false, G, 8, 8>(f, lds, w, w.row_block * KM_BLOCK_SIZE, blockIdx.y * G * 16, __builtin_amdgcn_readfirstlane(threadIdx.x >> 6));
}

template <int G>
static hipError_t launch_periodic_shares(FwdArgs& a, const MatmulPlan& plan, unsigned grid_y, hipStream_t stream) {
    a.chunks_per_block = plan.shares;
    a.total_items = ((long long)a.m + KM_BLOCK_SIZE - 1) / KM_BLOCK_SIZE * a.num_batches;
    hipLaunchKernelGGL((fwd_block_shares<KM_KERNEL_LOCALLY_PERIODIC, G>), dim3((unsigned)(a.total_items * plan.shares), grid_y, 1), dim3(512, 1, 1), (sizeof(float) * entry_lds_floats(G, 8, 8)), stream, a);
    const hipError_t err = hipGetLastError();
    return err == hipSuccess ? launch_sum_shares(a, stream) : err;
}

template <int G, int R, int W>
static hipError_t launch_periodic_as(FwdArgs& a, unsigned grid_y, hipStream_t stream) {
    a.chunks_per_block = KM_BLOCK_SIZE / (16 * R);
    a.total_items = ((long long)a.m + KM_BLOCK_SIZE - 1) / KM_BLOCK_SIZE * a.chunks_per_block * a.num_batches;
    a.items_per_xcd = (a.total_items + KM_NUM_XCD - 1) / KM_NUM_XCD;
    hipLaunchKernelGGL((fwd_block<KM_KERNEL_LOCALLY_PERIODIC, G, R, W>), dim3((unsigned)(a.items_per_xcd * KM_NUM_XCD), grid_y, 1), dim3(64 * W, 1, 1),
                       (sizeof(float) * entry_lds_floats(G, R, W)), stream, a);
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
        default:
            // (up to 16 columns take eight wavefronts with fewer rows only: periodic_plan)
            if constexpr (G == 1) {
                return hipErrorInvalidValue;
            } else {
                return launch_periodic_as<G, R, 8>(a, grid_y, stream);
            }
    }
}

hipError_t launch_matmul_periodic(const MatmulProblem& p, const MatmulPlan& plan, hipStream_t stream) {
    FwdArgs a;
    fill_fwd_args(p, &a);
    const unsigned grid_y = (unsigned)((p.k + plan.k_chunk - 1) / plan.k_chunk);
    if (plan.shares > 1) {
        return plan.k_chunk == 16 ? launch_periodic_shares<1>(a, plan, grid_y, stream) : launch_periodic_shares<2>(a, plan, grid_y, stream);
    }
    switch (plan.k_chunk / 16) {
        case 1: return plan.row_groups == 2 ? launch_periodic_as<1, 2, 8>(a, grid_y, stream) : launch_periodic_w<1, 8>(a, plan, grid_y, stream);
        case 2: return launch_periodic_w<2, 8>(a, plan, grid_y, stream);
        default: return launch_periodic_w<4, 4>(a, plan, grid_y, stream);
    }
}

}  // namespace km
