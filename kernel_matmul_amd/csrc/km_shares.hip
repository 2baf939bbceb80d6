// Sums of the shares that several workgroups took of each row block's range (take_share of km_fwd.h), in their order.
#include "km_common.h"
#include "km_launch.h"

namespace km {

__global__ void __launch_bounds__(256) sum_shares(const float* __restrict__ partials, float* __restrict__ out, long long count, int shares) {
    const long long i = (long long)blockIdx.x * 256 + threadIdx.x;
    if (i >= count) {
        return;
    }
    float sum = 0.0f;
#pragma unroll 8
    for (int s = 0; s < shares; s++) {
        sum += partials[s * count + i];
    }
    out[i] = sum;
}

hipError_t launch_sum_shares(const MatmulProblem& p, const MatmulPlan& plan, hipStream_t stream) {
    const long long count = p.num_batches * p.m * p.k;
    hipLaunchKernelGGL(sum_shares, dim3((unsigned)((count + 255) / 256), 1, 1), dim3(256, 1, 1), 0, stream, p.partials, p.out, count, plan.shares);
    return hipGetLastError();
}

}  // namespace km
