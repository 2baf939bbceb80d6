// Dense materialisation of the masked kernel matrix and the hyper-parameter gradient of a
// weighted sum of its entries.
//   dense     : out[b,i,j] = K[b,i,j] inside the row block's [start, end), 0 outside
//               (native/dense/dense.cu:12-98 of the reference; here the zeros are written by
//               the same kernel, so the output needs no prior clearing).
//   dense_bwd : grad[b,p] = d/d params[b,p] sum_{(i,j) in mask} out_grad[b,i,j] K[b,i,j]
//               (native/dense_bwd/dense_bwd.cu:12-116).
// Both stream an m x n fp32 matrix through HBM (4 B per entry): they are bandwidth bound.
#include "km_batch.h"
#include "km_common.h"
#include "km_launch.h"

namespace km {

struct DenseArgs {
    BatchShape batch;
    long long num_batches;
    long long total_items;  // row blocks * col splits * batches
    long long first_item, launch_items;  // of these, the ones of a launch (dense_bwd)
    long long items_per_xcd;
    int m, n;
    int col_splits;
    int cols_per_split;    // dense: columns per share, a multiple of 64
    const float* x1;
    const float* x2;
    const float* params;
    const int* start;
    const int* end;
    float* out;            // dense: [num_batches][m][n]
    const float* weights;  // dense_bwd: out_grad, batch/inner strides below
    float* partials;       // dense_bwd: [num_batches][row_blocks * col_splits][KM_MAX_PARAMS]
    BatchStrides x1_bs, x2_bs, params_bs, start_bs, end_bs, weights_bs;
    long long x1_s, x2_s, params_s, start_s, end_s, weights_s0, weights_s1;
};

struct DenseView {
    long long b;
    long long rest;
    const float* x1;
    const float* x2;
    const float* params;
    const float* weights;
    int range_start, range_end;
};

__device__ __forceinline__ DenseView dense_view(const DenseArgs& a, long long item, int divisor,
                                                int* row_block, int* split) {
    DenseView v;
    v.b = item % a.num_batches;
    v.rest = item / a.num_batches;
    *split = (int)(v.rest % divisor);
    *row_block = (int)(v.rest / divisor);
    int bidx[KM_MAX_BATCH_RANK];
    batch_multi_index(a.batch, v.b, bidx);
    v.x1 = a.x1 + batch_offset(a.batch, a.x1_bs, bidx);
    v.x2 = a.x2 + batch_offset(a.batch, a.x2_bs, bidx);
    v.params = a.params + batch_offset(a.batch, a.params_bs, bidx);
    v.weights = a.weights ? a.weights + batch_offset(a.batch, a.weights_bs, bidx) : nullptr;
    v.range_start = max(a.start[batch_offset(a.batch, a.start_bs, bidx) + *row_block * a.start_s], 0);
    v.range_end = min(a.end[batch_offset(a.batch, a.end_bs, bidx) + *row_block * a.end_s], a.n);
    return v;
}

// One workgroup of 256 threads per (row block, column share, batch item): each wavefront writes 32 of the block's rows
// over the share's columns, lanes run along the columns, V of them each, so that stores are 256 V contiguous bytes
// (V = 4: rows begin at multiples of 16 bytes).  The column shares only exist to fill the device when row blocks x
// batch items are few.  A wavefront keeps its 32 row coordinates one per lane and broadcasts them with v_readlane (no
// load inside the row loop).  Bound by the writes; V = 1 -> 4, spectral n = 7200 35.9 -> 31.6 us (6.5 TB/s), n = 20000 334 -> 312.
template <int KT, int V>
__global__ void __launch_bounds__(256) dense_kernel(const DenseArgs a) {
    typedef float Vec __attribute__((ext_vector_type(V)));
    const long long item = xcd_item(blockIdx.x, a.items_per_xcd);
    if (item >= a.total_items) {
        return;
    }
    int row_block, split;
    const DenseView v = dense_view(a, item, a.col_splits, &row_block, &split);
    const int col_lo = split * a.cols_per_split;
    const int col_hi = col_lo + min(a.n - col_lo, a.cols_per_split);
    const int lane = threadIdx.x & 63;
    const int wave = threadIdx.x >> 6;
    const int row_begin = row_block * KM_BLOCK_SIZE + wave * 32;
    const int rows = min(32, a.m - row_begin);
    if (rows <= 0 || col_lo >= col_hi) {
        return;
    }
    const KernelConsts kc = make_consts<KT>(v.params, a.params_s, true);
    float* __restrict__ out = a.out + v.b * (long long)a.m * a.n + (long long)row_begin * a.n;
    const int x1_bits = __float_as_int(v.x1[(long long)(row_begin + min(lane, rows - 1)) * a.x1_s]);
    // (compared by differences: what follows the last columns may lie past the largest int)
    for (int col0 = col_lo;; col0 += 64 * V) {
        const bool in_matrix = V * lane < col_hi - col0;  // (with all V: their number divides that of the columns)
        const int col = in_matrix ? col0 + V * lane : col0;
        float* __restrict__ o = out + col;
        // Wave-uniform choice: column tiles fully outside the range are only cleared.
        if (col0 < v.range_end && v.range_start - col0 < 64 * V) {
            float x2v[V];
            bool in_range[V];
#pragma unroll
            for (int t = 0; t < V; t++) {
                in_range[t] = in_matrix && col + t >= v.range_start && col + t < v.range_end;
                x2v[t] = in_range[t] ? v.x2[(long long)(col + t) * a.x2_s] : 0.0f;
            }
            for (int r = 0; r < rows; r++) {
                const float x1v = __int_as_float(__builtin_amdgcn_readlane(x1_bits, r));
                Vec kv;
#pragma unroll
                for (int t = 0; t < V; t++) {
                    const float k = kernel_value<KT>(x1v, x2v[t], kc) * kc.sgn;
                    kv[t] = in_range[t] ? k : 0.0f;
                }
                if (in_matrix) {
                    *(Vec*)(o + (long long)r * a.n) = kv;
                }
            }
        } else if (in_matrix) {
            for (int r = 0; r < rows; r++) {
                *(Vec*)(o + (long long)r * a.n) = (Vec)(0.0f);
            }
        }
        if (col_hi - col0 <= 64 * V) {
            return;
        }
    }
}

// One workgroup per (row block, column split, batch item), whose wavefronts take 16 rows each: lanes run along the
// columns, weights are read 256 B contiguous, all 16 rows' together: narrow ranges are bound by that latency, wide ones by
// memory.  Against one wavefront for all 128 rows, eight at a time (spectral, a call with its reduction): n = 7200, 290 /
// 2500 columns a row block 17.0 -> 12.6 / 43.9 -> 24.3 us; n = 20000, all columns 385 -> 311 (5.2 TB/s).
#define KM_DENSE_BWD_ROWS 16
#define KM_DENSE_BWD_WAVES (KM_BLOCK_SIZE / KM_DENSE_BWD_ROWS)
#define KM_DENSE_BWD_LAUNCH (1ll << 22) /* workgroups at a time: 2^31 threads */
template <int KT>
__global__ void __launch_bounds__(64 * KM_DENSE_BWD_WAVES) dense_bwd_partial(const DenseArgs a) {
    __shared__ float sums[KM_DENSE_BWD_WAVES][KM_MAX_PARAMS];
    const long long item = xcd_item(blockIdx.x, a.items_per_xcd);
    if (item >= a.launch_items) {
        return;
    }
    int row_block, split;
    const DenseView v = dense_view(a, a.first_item + item, a.col_splits, &row_block, &split);
    const KernelConsts kc = make_consts<KT>(v.params, a.params_s, false);
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);

    const int width = max(v.range_end - v.range_start, 0);
    const int per_split = ((width + a.col_splits - 1) / a.col_splits + 63) & ~63;
    // (shares past the last column are empty, and may begin past the largest int)
    const int range_end = max(v.range_end, v.range_start);
    const int col_begin = (int)min(v.range_start + (long long)split * per_split, (long long)range_end);
    const int col_end = col_begin + min(per_split, range_end - col_begin);
    const int row_begin = row_block * KM_BLOCK_SIZE + wave * KM_DENSE_BWD_ROWS;
    const int rows = min(KM_DENSE_BWD_ROWS, a.m - row_begin);

    const long long partial_rows = a.total_items / a.num_batches;
    float* __restrict__ partial = a.partials + (v.b * partial_rows + v.rest) * KM_MAX_PARAMS;
    if (col_begin >= col_end) {  // (the same in all wavefronts)
        if (threadIdx.x < KM_MAX_PARAMS) {
            partial[threadIdx.x] = 0.0f;
        }
        return;
    }
    float acc[KM_MAX_PARAMS] = {0.0f, 0.0f, 0.0f, 0.0f};
    if (rows > 0) {
        // The row coordinates one per lane, to be read from there (rows past the matrix repeat the last one; their
        // weights are zero).
        const int x1_bits = __float_as_int(v.x1[(long long)(row_begin + min(lane, rows - 1)) * a.x1_s]);
        for (int col0 = col_begin; col0 < col_end; col0 += 64) {
            const int col = col0 + lane;
            const bool ok = col < col_end;
            const int colc = min(col, col_end - 1);
            const float x2v = v.x2[(long long)colc * a.x2_s];
            const float* __restrict__ w = v.weights + (long long)row_begin * a.weights_s0 + (long long)colc * a.weights_s1;
            float wv[KM_DENSE_BWD_ROWS];
#pragma unroll
            for (int t = 0; t < KM_DENSE_BWD_ROWS; t++) {
                wv[t] = w[(long long)min(t, rows - 1) * a.weights_s0];
            }
#pragma unroll
            for (int t = 0; t < KM_DENSE_BWD_ROWS; t++) {
                const float x1v = __int_as_float(__builtin_amdgcn_readlane(x1_bits, t));
                accumulate_pair<KT>(x1v, x2v, ok && t < rows ? wv[t] : 0.0f, kc, acc);
            }
        }
    }
#pragma unroll
    for (int p = 0; p < KM_MAX_PARAMS; p++) {
        const float total = wave_sum(acc[p]);
        if (lane == 0) {
            sums[wave][p] = total;
        }
    }
    __syncthreads();
    if (threadIdx.x < KM_MAX_PARAMS) {
        float total = sums[0][threadIdx.x];
#pragma unroll
        for (int i = 1; i < KM_DENSE_BWD_WAVES; i++) {
            total += sums[i][threadIdx.x];
        }
        partial[threadIdx.x] = total;
    }
}

static void fill_common(DenseArgs& a, const DenseProblem& p) {
    a.num_batches = p.num_batches;
    a.m = (int)p.m;
    a.n = (int)p.n;
    a.x1 = p.x1;
    a.x2 = p.x2;
    a.params = p.params;
    a.start = p.start;
    a.end = p.end;
    a.out = p.out;
    a.weights = p.weights;
    a.partials = (float*)p.workspace;
    const int r = p.batch_rank;
    a.x1_s = p.x1_strides[r];
    a.x2_s = p.x2_strides[r];
    a.params_s = p.params_strides[r];
    a.start_s = p.start_strides[r];
    a.end_s = p.end_strides[r];
    a.weights_s0 = p.weights ? p.weights_strides[r] : 0;
    a.weights_s1 = p.weights ? p.weights_strides[r + 1] : 0;
}

template <int V>
static void launch_dense_as(int kernel_type, const DenseArgs& a, hipStream_t stream) {
    const unsigned grid = (unsigned)(a.items_per_xcd * KM_NUM_XCD);
    switch (kernel_type) {
        case KM_KERNEL_RBF:
            hipLaunchKernelGGL((dense_kernel<KM_KERNEL_RBF, V>), dim3(grid), dim3(256), 0, stream, a);
            break;
        case KM_KERNEL_SPECTRAL:
            hipLaunchKernelGGL((dense_kernel<KM_KERNEL_SPECTRAL, V>), dim3(grid), dim3(256), 0, stream, a);
            break;
        default:
            hipLaunchKernelGGL((dense_kernel<KM_KERNEL_LOCALLY_PERIODIC, V>), dim3(grid), dim3(256), 0, stream, a);
            break;
    }
}

hipError_t launch_dense(const DenseProblem& p, hipStream_t stream) {
    DenseArgs a;
    const int64_t* const strides[5] = {p.x1_strides, p.x2_strides, p.params_strides,
                                       p.start_strides, p.end_strides};
    BatchStrides* outs[5] = {&a.x1_bs, &a.x2_bs, &a.params_bs, &a.start_bs, &a.end_bs};
    collapse_batch<5>(p.batch_rank, p.batch_sizes, strides, &a.batch, outs);
    fill_common(a, p);
    a.weights = nullptr;
    const long long row_blocks = (p.m + KM_BLOCK_SIZE - 1) / KM_BLOCK_SIZE;
    // Column shares of at least 256 columns until there are 2048 workgroups (8 per CU).
    const long long base = row_blocks * p.num_batches;
    long long splits = base > 0 ? (2048 + base - 1) / base : 1;
    const long long most = (p.n + 255) / 256;
    if (splits > most) splits = most;
    if (splits < 1) splits = 1;
    a.cols_per_split = (int)((((p.n + splits - 1) / splits) + 63) / 64 * 64);
    if (a.cols_per_split < 64) a.cols_per_split = 64;
    a.col_splits = (int)((p.n + a.cols_per_split - 1) / a.cols_per_split);
    if (a.col_splits < 1) a.col_splits = 1;
    a.total_items = row_blocks * a.col_splits * p.num_batches;
    a.items_per_xcd = (a.total_items + KM_NUM_XCD - 1) / KM_NUM_XCD;
    if (p.n % 4 == 0 && (uintptr_t)p.out % 16 == 0) {
        launch_dense_as<4>(p.kernel_type, a, stream);
    } else {
        launch_dense_as<1>(p.kernel_type, a, stream);
    }
    return hipGetLastError();
}

hipError_t launch_dense_bwd(const DenseProblem& p, hipStream_t stream) {
    DenseArgs a;
    const int64_t* const strides[6] = {p.x1_strides, p.x2_strides, p.params_strides,
                                       p.start_strides, p.end_strides, p.weights_strides};
    BatchStrides* outs[6] = {&a.x1_bs, &a.x2_bs, &a.params_bs, &a.start_bs, &a.end_bs, &a.weights_bs};
    collapse_batch<6>(p.batch_rank, p.batch_sizes, strides, &a.batch, outs);
    fill_common(a, p);
    const long long row_blocks = (p.m + KM_BLOCK_SIZE - 1) / KM_BLOCK_SIZE;
    a.col_splits = (int)(param_grad_partials_per_batch(p.m, p.num_batches) / (row_blocks > 0 ? row_blocks : 1));
    // (a share has eight wavefronts here: four workgroups a CU, no more, of which narrow ranges leave most without columns.
    // n = 12000, 230 columns a row block, 2 sets: 24 us with sixteen shares, 20 with six)
    const long long shares = row_blocks * p.num_batches > 0 ? (1024 + row_blocks * p.num_batches - 1) / (row_blocks * p.num_batches) : 1;
    if (a.col_splits > shares) a.col_splits = (int)shares;
    if (a.col_splits < 1) a.col_splits = 1;
    a.total_items = row_blocks * a.col_splits * p.num_batches;
    // (a launch may have 2^32 - 1 threads)
    for (a.first_item = 0; a.first_item < a.total_items; a.first_item += KM_DENSE_BWD_LAUNCH) {
        a.launch_items = a.total_items - a.first_item < KM_DENSE_BWD_LAUNCH ? a.total_items - a.first_item : KM_DENSE_BWD_LAUNCH;
        a.items_per_xcd = (a.launch_items + KM_NUM_XCD - 1) / KM_NUM_XCD;
        const unsigned grid = (unsigned)(a.items_per_xcd * KM_NUM_XCD);
        switch (p.kernel_type) {
            case KM_KERNEL_RBF:
                hipLaunchKernelGGL((dense_bwd_partial<KM_KERNEL_RBF>), dim3(grid), dim3(64 * KM_DENSE_BWD_WAVES), 0, stream, a);
                break;
            case KM_KERNEL_SPECTRAL:
                hipLaunchKernelGGL((dense_bwd_partial<KM_KERNEL_SPECTRAL>), dim3(grid), dim3(64 * KM_DENSE_BWD_WAVES), 0, stream, a);
                break;
            default:
                hipLaunchKernelGGL((dense_bwd_partial<KM_KERNEL_LOCALLY_PERIODIC>), dim3(grid), dim3(64 * KM_DENSE_BWD_WAVES), 0, stream, a);
                break;
        }
        hipError_t err = hipGetLastError();
        if (err != hipSuccess) {
            return err;
        }
    }
    return launch_param_grad_reduce(p.kernel_type, a.batch, p.num_batches, row_blocks * a.col_splits,
                                    a.partials, p.params, a.params_bs, a.params_s, p.grad, stream);
}

}  // namespace km
