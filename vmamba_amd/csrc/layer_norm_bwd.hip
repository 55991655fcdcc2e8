// Backward of the LayerNorm over rows of C contiguous channels in single precision (torch.nn.functional.layer_norm of a block in training,
// classification/models/vmamba.py:1225-1229, :641-646), and column sums, which bias gradients are:
//     g = dy w,  dx = rstd (g - mean(g) - xhat mean(g xhat)),  dw = sum over rows of dy xhat,  db = sum over rows of dy.
// The library's backward is three kernels that read x and dy twice, 52 us for 12 544 rows of 384 where a pass over x, dy and dx (58 MB) takes 11.
// Here a row lives in the registers of a group of 16, 32 or 64 lanes, four channels to a load, and its statistics are computed again
// from it (centred variance, as the forward does) instead of being kept; a workgroup walks its share of the rows with the next
// row's loads in flight and keeps dw and db of its lanes' channels in registers.  The workgroups' sums are added by a second kernel
// in a fixed order: no atomics, the same bits every time.
// 12 544 x 384: 52 -> 16 + 6 us (3.6 TB/s in the first, which has a row in flight per wavefront and eight wavefronts per CU); 100 352 x 384 270 -> 102.  Column
// sums of 12 544 x 1536 30 -> 19, in a graph.
#include "ss2d_common.h"

namespace ss2d {

typedef float nf4_t __attribute__((ext_vector_type(4)));

constexpr int kNbThreads = 512, kNbShares = 256;                     // a workgroup per CU
constexpr int kNbMaxVec = 4;                                         // C <= 1024: 64 lanes x 4 loads x 4 channels

struct NormBwdArgs {
    const float *x, *dy, *w;
    float *dx, *partial;                                             // partial [shares][dw | db][C]
    int64_t rows, share;                                             // rows per workgroup, a multiple of what it has in hand at once
    int32_t C;
    float eps;
};

// Sum over a power-of-two group of lanes, the same value in every lane of it
template <int kLanes> __device__ __forceinline__ float lanes_sum(float v) {
#pragma unroll
    for (int m = kLanes / 2; m >= 1; m /= 2) v += __shfl_xor(v, m);
    return v;
}

// kLanes lanes to a row, kVec loads to a lane.
template <int kLanes, int kVec>
__global__ __launch_bounds__(kNbThreads) void layer_norm_bwd_kernel(const NormBwdArgs p) {
    constexpr int kSlots = kNbThreads / kLanes;                      // rows in hand
    __shared__ nf4_t sums[kNbThreads];
    const int lane = threadIdx.x % kLanes, slot = threadIdx.x / kLanes;
    const int64_t begin = (int64_t)blockIdx.x * p.share, end = begin + p.share < p.rows ? begin + p.share : p.rows;
    const float inv_c = 1.0f / (float)p.C;
    const nf4_t zero = {0, 0, 0, 0};
    nf4_t w[kVec], dw[kVec], db[kVec], x[kVec], dy[kVec];
    bool in[kVec];
#pragma unroll
    for (int i = 0; i < kVec; ++i) {
        const int c = 4 * (lane + kLanes * i);
        in[i] = c < p.C;                                             // (C is a multiple of 4)
        w[i] = !in[i] ? zero : p.w ? *reinterpret_cast<const nf4_t *>(p.w + c) : nf4_t{1, 1, 1, 1};
        dw[i] = db[i] = zero;
    }
    auto load = [&](int64_t row) {
        const int64_t at = (row < p.rows ? row : p.rows - 1) * p.C;
#pragma unroll
        for (int i = 0; i < kVec; ++i) {
            const int64_t o = at + (in[i] ? 4 * (lane + kLanes * i) : 0);
            x[i] = *reinterpret_cast<const nf4_t *>(p.x + o);
            dy[i] = *reinterpret_cast<const nf4_t *>(p.dy + o);
        }
    };
    load(begin + slot);
    for (int64_t row = begin + slot; row - slot < end; row += kSlots) {
        nf4_t v[kVec], d[kVec];
        float s = 0.0f;
#pragma unroll
        for (int i = 0; i < kVec; ++i) {
            v[i] = in[i] ? x[i] : zero;
            d[i] = in[i] && row < end ? dy[i] : zero;
            s += (v[i][0] + v[i][1]) + (v[i][2] + v[i][3]);
        }
        load(row + kSlots);                                          // the next row, under this one's arithmetic
        const float mean = lanes_sum<kLanes>(s) * inv_c;
        float q = 0.0f;
#pragma unroll
        for (int i = 0; i < kVec; ++i) {
            v[i] = in[i] ? v[i] - mean : zero;
#pragma unroll
            for (int t = 0; t < 4; ++t) q = fmaf(v[i][t], v[i][t], q);
        }
        const float rstd = rsqrtf(lanes_sum<kLanes>(q) * inv_c + p.eps);
        float c1 = 0.0f, c2 = 0.0f;
#pragma unroll
        for (int i = 0; i < kVec; ++i) {
            v[i] *= rstd;
            dw[i] += d[i] * v[i];
            db[i] += d[i];
            d[i] *= w[i];
#pragma unroll
            for (int t = 0; t < 4; ++t) { c1 += d[i][t]; c2 = fmaf(d[i][t], v[i][t], c2); }
        }
        c1 = lanes_sum<kLanes>(c1) * inv_c;
        c2 = lanes_sum<kLanes>(c2) * inv_c;
        if (p.dx && row < end) {
#pragma unroll
            for (int i = 0; i < kVec; ++i)
                if (in[i]) *reinterpret_cast<nf4_t *>(p.dx + row * p.C + 4 * (lane + kLanes * i)) = (d[i] - c1 - v[i] * c2) * rstd;
        }
    }
    if (!p.partial) return;
    // the slots' sums, in their order
    float *out = p.partial + (int64_t)blockIdx.x * 2 * p.C;
#pragma unroll
    for (int which = 0; which < 2; ++which)
#pragma unroll
        for (int i = 0; i < kVec; ++i) {
            __syncthreads();
            sums[threadIdx.x] = which ? db[i] : dw[i];
            __syncthreads();
            if (slot == 0 && in[i]) {
                nf4_t t = sums[lane];
                for (int k = 1; k < kSlots; ++k) t += sums[k * kLanes + lane];
                *reinterpret_cast<nf4_t *>(out + which * p.C + 4 * (lane + kLanes * i)) = t;
            }
        }
}

// Shares of the rows' column sums: a workgroup takes 256 columns of its share
__global__ __launch_bounds__(kNbThreads) void column_sums_kernel(const float *x, float *partial, int64_t rows, int64_t share, int N) {
    __shared__ nf4_t sums[kNbThreads];
    const int col = 4 * ((int)blockIdx.y * kWave + (int)threadIdx.x % kWave), slot = threadIdx.x / kWave;
    constexpr int kSlots = kNbThreads / kWave, kFly = 4;
    const int64_t begin = (int64_t)blockIdx.x * share, end = begin + share < rows ? begin + share : rows;
    const int at = min(col, N - 4);
    nf4_t t = {0, 0, 0, 0};
    for (int64_t row = begin + slot; row < end; row += kFly * kSlots) {
        nf4_t v[kFly];
#pragma unroll
        for (int q = 0; q < kFly; ++q) v[q] = *reinterpret_cast<const nf4_t *>(x + (row + q * kSlots < end ? row + q * kSlots : row) * N + at);
#pragma unroll
        for (int q = 0; q < kFly; ++q)
            if (row + q * kSlots < end) t += v[q];
    }
    sums[threadIdx.x] = t;
    __syncthreads();
    if (slot == 0 && col < N) {
        for (int k = 1; k < kSlots; ++k) t += sums[k * kWave + threadIdx.x];
        *reinterpret_cast<nf4_t *>(partial + (int64_t)blockIdx.x * N + col) = t;
    }
}

// out[c] = sum over the shares of partial[share][c]: 16 lanes of four columns, 16 groups of shares
__global__ __launch_bounds__(kBlock) void shares_sum_kernel(const float *partial, float *first, float *second, int shares, int width, int split) {
    __shared__ nf4_t sums[kBlock];
    const int lane = threadIdx.x & 15, group = threadIdx.x >> 4, col = 4 * ((int)blockIdx.x * 16 + lane), at = min(col, width - 4);
    nf4_t t = {0, 0, 0, 0};
    for (int s = group; s < shares; s += 16) t += *reinterpret_cast<const nf4_t *>(partial + (int64_t)s * width + at);
    sums[threadIdx.x] = t;
    __syncthreads();
    if (group == 0 && col < width) {
        for (int k = 1; k < 16; ++k) t += sums[k * 16 + lane];
        float *out = col < split ? first + col : second + (col - split);
        if (col < split ? first != nullptr : second != nullptr) *reinterpret_cast<nf4_t *>(out) = t;
    }
}

static int64_t nb_share(int64_t rows, int64_t unit) {                // rows per workgroup, whole turns of them
    const int64_t per = (rows + kNbShares - 1) / kNbShares;
    return (per + unit - 1) / unit * unit;
}

template <int kLanes, int kVec> static int64_t launch_norm_bwd(NormBwdArgs &a, hipStream_t s) {
    a.share = nb_share(a.rows, kNbThreads / kLanes);
    const int64_t shares = (a.rows + a.share - 1) / a.share;
    hipLaunchKernelGGL((layer_norm_bwd_kernel<kLanes, kVec>), dim3((uint32_t)shares), dim3(kNbThreads), 0, s, a);
    return shares;
}

}  // namespace ss2d

extern "C" int64_t ss2d_layer_norm_bwd_f32_workspace_bytes(int C) { return C > 0 ? (int64_t)ss2d::kNbShares * 2 * C * 4 : SS2D_EINVAL; }

extern "C" int ss2d_layer_norm_bwd_f32(const float *x, const float *dy, const float *weight, float eps, float *dx, float *dweight, float *dbias, int64_t rows,
                                       int C, void *workspace, int64_t workspace_bytes, void *stream) {
    using namespace ss2d;
    if (rows < 0 || C <= 0) return SS2D_EINVAL;
    if (C % 4 != 0 || C > 4 * kWave * kNbMaxVec) return SS2D_ENOTSUP;
    if (rows == 0) return SS2D_ENOTSUP;
    const bool sums = dweight || dbias;
    if (!x || !dy || (!dx && !sums) || (sums && !workspace)) return SS2D_EINVAL;
    if (sums && workspace_bytes < ss2d_layer_norm_bwd_f32_workspace_bytes(C)) return SS2D_ENOMEM;
    const void *ptrs[] = {x, dy, weight, dx, dweight, dbias, workspace};
    for (const void *q : ptrs)
        if (reinterpret_cast<uintptr_t>(q) % 16 != 0) return SS2D_ENOTSUP;
    NormBwdArgs a = {x, dy, weight, dx, sums ? (float *)workspace : nullptr, rows, 0, C, eps};
    hipStream_t s = (hipStream_t)stream;
    const int quads = C / 4;
    const int64_t shares = quads <= 16 ? launch_norm_bwd<16, 1>(a, s) : quads <= 32 ? launch_norm_bwd<32, 1>(a, s) : quads <= 64 ? launch_norm_bwd<64, 1>(a, s)
                         : quads <= 128 ? launch_norm_bwd<64, 2>(a, s) : quads <= 192 ? launch_norm_bwd<64, 3>(a, s) : launch_norm_bwd<64, 4>(a, s);
    if (sums)
        hipLaunchKernelGGL(shares_sum_kernel, dim3((uint32_t)((2 * C + 63) / 64)), dim3(kBlock), 0, s, a.partial, dweight, dbias, (int)shares, 2 * C, C);
    return launch_status();
}

extern "C" int64_t ss2d_column_sums_f32_workspace_bytes(int N) { return N > 0 ? (int64_t)ss2d::kNbShares * N * 4 : SS2D_EINVAL; }

extern "C" int ss2d_column_sums_f32(const float *x, float *out, int64_t rows, int N, void *workspace, int64_t workspace_bytes, void *stream) {
    using namespace ss2d;
    if (rows < 0 || N <= 0) return SS2D_EINVAL;
    if (rows == 0 || N % 4 != 0) return SS2D_ENOTSUP;
    if (!x || !out || !workspace) return SS2D_EINVAL;
    if (workspace_bytes < ss2d_column_sums_f32_workspace_bytes(N)) return SS2D_ENOMEM;
    if ((reinterpret_cast<uintptr_t>(x) | reinterpret_cast<uintptr_t>(out) | reinterpret_cast<uintptr_t>(workspace)) % 16 != 0) return SS2D_ENOTSUP;
    hipStream_t s = (hipStream_t)stream;
    const int64_t share = nb_share(rows, kNbThreads / kWave), shares = (rows + share - 1) / share;
    hipLaunchKernelGGL(column_sums_kernel, dim3((uint32_t)shares, (uint32_t)((N + 255) / 256)), dim3(kNbThreads), 0, s, x, (float *)workspace, rows, share, N);
    hipLaunchKernelGGL(shares_sum_kernel, dim3((uint32_t)((N + 63) / 64)), dim3(kBlock), 0, s, (const float *)workspace, out, nullptr, (int)shares, N, N);
    return launch_status();
}
