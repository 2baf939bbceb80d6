// Sums of the shares that several workgroups took of a row block's range (share_view of km_fwd.h), in their order.  A thread for
// each value, which has its shares' loads in flight eight at a time; row blocks of one share have their result already.
// Bound by latency: 1.3 us of a trace where all have, 1.9 to 3.8 with up to 126 shares.
#include "km_batch.h"
#include "km_common.h"
#include "km_fwd.h"
#include "km_launch.h"

namespace km {

__global__ void __launch_bounds__(256) sum_shares(const FwdArgs a) {
    int unused;
    const WaveView w = wave_view<true>(a, blockIdx.x, 1, &unused);
    const ShareOf s = shares_of(max(w.range_end - w.range_start, 0), a.chunks_per_block);
    const int row0 = w.row_block * KM_BLOCK_SIZE;
    const long long i = (long long)blockIdx.y * 256 + threadIdx.x;
    if (s.present == 1 || i >= (long long)min(KM_BLOCK_SIZE, a.m - row0) * a.k) {
        return;
    }
    const long long stride = a.num_batches * a.m * a.k, at = (w.b * a.m + row0) * a.k + i;
    float sum = 0.0f;
#pragma unroll 8
    for (int p = 0; p < s.present; p++) {
        sum += a.partials[p * stride + at];
    }
    a.out[at] = sum;
}

hipError_t launch_sum_shares(const FwdArgs& a, hipStream_t stream) {
    hipLaunchKernelGGL(sum_shares, dim3((unsigned)a.total_items, (unsigned)((KM_BLOCK_SIZE * (long long)a.k + 255) / 256), 1), dim3(256, 1, 1), 0, stream, a);
    return hipGetLastError();
}

}  // namespace km
