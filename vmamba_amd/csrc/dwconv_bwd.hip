// Backward of the depthwise 3 x 3 convolution + SiLU in front of the SS2D core (classification/models/vmamba.py:654-658):
//     z = conv(x) + bias,  y = silu(z);   ds = dy * silu'(z),  dx = ds correlated with the mirrored weights,
//     dw[k] = sum over images and positions of ds * (x shifted by tap k),  dbias = sum of ds.
// The library spent 540 us on the three convolution passes of 64 x 384 maps of 14 x 14 in fp32 (the weights' gradient alone
// 450, a general grouped convolution), more than on any other part of that block's training step; what they move is 58 MB.
// (Now 27 us forward, 45 backward; the step 3.01 -> 2.36 ms with the two layout changes on this package's transpose.)
// Forward and backward through autograd against the library, channel-last, batch 64, us: 96 x 56 x 56 fp32 2296 -> 269, bf16
// 1848 -> 187, fp16 2504 -> 186; 768 x 7 x 7 433 -> 150, 561 -> 149, 342 -> 150; one image of 384 x 14 x 14 183 -> 146, 174 -> 150,
// 165 -> 146 (the host's share); two of 96 x 256 x 256 1301 -> 269, 1807 -> 203, 1341 -> 205: it serves every map that fits.
// Here one kernel reads x and dy once and writes dx once: a workgroup owns one channel of several images -- its nine weights'
// gradients stay in registers over all of them -- and holds their planes in LDS (whole planes where they fit, rows of them
// with a halo where not), zero-padded so that no tap has a bound to test.  z is recomputed from the same x the weights'
// gradient needs anyway, so nothing but x is saved for it.  Every workgroup leaves its ten sums in a workspace and a second
// kernel adds them up in a fixed order: no atomics, the same bits every time.  In single precision the nine products of z and
// of dx are summed in 64 bits, as the library does (relative error of dx 6e-8; 8e-8 with fp32 sums); the weights' gradient is
// off by 1.2e-7 where the library's transform is by 1.1e-6.
#include "ss2d_common.h"

namespace ss2d {

constexpr int kDwbCells = 2048;      // positions of dx a workgroup works on between two barriers

struct DwBwdArgs {
    const void *x, *w, *bias, *dy;
    void *dx;
    float *partial;                  // [n_parts][D][10]
    int32_t B, D, H, W, Th, tiles_h, planes, images;     // planes: per round, images: per workgroup
    FastDiv by_x, by_x_row, by_ds, by_ds_row;            // cells per plane and per row of the x / ds rounds
};

// sums of nine products: 64 bits for fp32 operands, 32 for 16-bit ones
template <typename T> struct TapSum { using type = float; };
template <> struct TapSum<float> { using type = double; };

// kForward: y = silu(z) into dx, nothing else
template <typename T, bool kForward>
__global__ __launch_bounds__(kBlock) void dwconv_bwd_kernel(const DwBwdArgs p) {
    extern __shared__ float dwb_smem[];
    const int xw = p.W + 2, dw_ = p.W + 2;                           // one column of zeros on either side
    const int x_cells = (p.Th + 4) * xw, d_cells = (p.Th + 2) * dw_;
    float *xs = dwb_smem, *ds = dwb_smem + p.planes * x_cells;
    const int d = (int)(blockIdx.x % (uint32_t)p.D);
    const uint32_t part = blockIdx.x / (uint32_t)p.D;
    const int h0 = (int)(part % (uint32_t)p.tiles_h) * p.Th, b0 = (int)(part / (uint32_t)p.tiles_h) * p.images;
    const int b1 = min(p.B, b0 + p.images), rows = min(p.Th, p.H - h0);
    const T *x = reinterpret_cast<const T *>(p.x), *dy = reinterpret_cast<const T *>(p.dy);
    T *dx = reinterpret_cast<T *>(p.dx);
    const int64_t HW = (int64_t)p.H * p.W;
    using S = typename TapSum<T>::type;
    float w[9], acc[10];
#pragma unroll
    for (int k = 0; k < 9; ++k) w[k] = to_f32(reinterpret_cast<const T *>(p.w)[d * 9 + k]);
    const float bias = p.bias ? to_f32(reinterpret_cast<const T *>(p.bias)[d]) : 0.0f;
#pragma unroll
    for (int k = 0; k < 10; ++k) acc[k] = 0.0f;
    for (int b = b0; b < b1; b += p.planes) {
        const int n = min(p.planes, b1 - b);
        // x: rows h0 - 2 .. h0 + Th + 1 of every plane
        for (int i = threadIdx.x; i < n * x_cells; i += kBlock) {
            uint32_t q, r, row, col;
            divmod((uint32_t)i, p.by_x, q, r);
            divmod(r, p.by_x_row, row, col);
            const int h = h0 - 2 + (int)row, c = (int)col - 1;
            xs[i] = h >= 0 && h < p.H && c >= 0 && c < p.W
                        ? to_f32(x[((int64_t)(b + (int)q) * p.D + d) * HW + (int64_t)h * p.W + c]) : 0.0f;
        }
        __syncthreads();
        // ds: rows h0 - 1 .. h0 + Th; the sums over rows h0 .. only, so that every position counts once
        for (int i = threadIdx.x; i < n * d_cells; i += kBlock) {
            uint32_t q, r, row, col;
            divmod((uint32_t)i, p.by_ds, q, r);
            divmod(r, p.by_ds_row, row, col);
            const int h = h0 - 1 + (int)row, c = (int)col - 1;
            float s = 0.0f;
            if constexpr (kForward) {
                if (h < h0 || h >= h0 + rows || c < 0 || c >= p.W) continue;
                const float *at = xs + q * x_cells + (row + 1) * xw + col;
                S z = 0;
#pragma unroll
                for (int k = 0; k < 9; ++k) z = fma((S)w[k], (S)at[(k / 3 - 1) * xw + k % 3 - 1], z);
                const float zf = (float)(z + (S)bias);
                dx[((int64_t)(b + (int)q) * p.D + d) * HW + (int64_t)h * p.W + c] = from_f32<T>(zf / (1.0f + expf(-zf)));
                continue;
            }
            if (h >= 0 && h < p.H && c >= 0 && c < p.W) {
                const float g = to_f32(dy[((int64_t)(b + (int)q) * p.D + d) * HW + (int64_t)h * p.W + c]);
                const float *at = xs + q * x_cells + (row + 1) * xw + col;       // x at (h, c)
                float v[9];
                S zs = 0;
#pragma unroll
                for (int k = 0; k < 9; ++k) {
                    v[k] = at[(k / 3 - 1) * xw + k % 3 - 1];
                    zs = fma((S)w[k], (S)v[k], zs);
                }
                const float z = (float)(zs + (S)bias);
                const float sig = 1.0f / (1.0f + expf(-z));
                s = g * (sig * fmaf(z, 1.0f - sig, 1.0f));
                if (h >= h0 && h < h0 + rows) {
#pragma unroll
                    for (int k = 0; k < 9; ++k) acc[k] = fmaf(s, v[k], acc[k]);
                    acc[9] += s;
                }
            }
            ds[i] = s;
        }
        __syncthreads();
        if constexpr (kForward) continue;                            // (xs is free again)
        for (int i = threadIdx.x; i < n * d_cells; i += kBlock) {
            uint32_t q, r, row, col;
            divmod((uint32_t)i, p.by_ds, q, r);
            divmod(r, p.by_ds_row, row, col);
            const int h = h0 - 1 + (int)row, c = (int)col - 1;
            if (h < h0 || h >= h0 + rows || c < 0 || c >= p.W) continue;
            S o = 0;
#pragma unroll
            for (int k = 0; k < 9; ++k) o = fma((S)w[k], (S)ds[i - (k / 3 - 1) * dw_ - (k % 3 - 1)], o);
            dx[((int64_t)(b + (int)q) * p.D + d) * HW + (int64_t)h * p.W + c] = from_f32<T>((float)o);
        }
        // (the next round writes xs, which nobody reads after the second barrier, and a barrier before it writes ds)
    }
    if constexpr (kForward) return;
    __shared__ float sums[kBlock / kWave][10];
#pragma unroll
    for (int k = 0; k < 10; ++k) {
        for (int m = kWave / 2; m >= 1; m /= 2) acc[k] += __shfl_xor(acc[k], m);
        if ((threadIdx.x & (kWave - 1)) == 0) sums[threadIdx.x / kWave][k] = acc[k];
    }
    __syncthreads();
    if (threadIdx.x < 10) {
        float t = 0.0f;
        for (int v = 0; v < kBlock / kWave; ++v) t += sums[v][threadIdx.x];
        p.partial[((int64_t)part * p.D + d) * 10 + threadIdx.x] = t;
    }
}

// partial [n_parts][D][10] -> dw [D][9] and dbias [D], a wavefront per channel and tap
template <typename T>
__global__ __launch_bounds__(kWave) void dwconv_bwd_sum_kernel(const float *partial, T *dw, T *db, int n_parts, int D) {
    const int d = blockIdx.x / 10, k = blockIdx.x % 10;
    float t = 0.0f;
    for (int i = threadIdx.x; i < n_parts; i += kWave) t += partial[((int64_t)i * D + d) * 10 + k];
    for (int m = kWave / 2; m >= 1; m /= 2) t += __shfl_xor(t, m);
    if (threadIdx.x != 0) return;
    if (k < 9) dw[d * 9 + k] = from_f32<T>(t);
    else if (db) db[d] = from_f32<T>(t);
}

// how a shape is cut: false where not even two rows of a plane fit
static bool dwconv_bwd_plan(int B, int D, int H, int W, DwBwdArgs &a, int64_t &parts, size_t &smem) {
    const int64_t most = 64 * 1024 / 4 - 64;                         // floats of LDS
    auto floats = [&](int64_t th) { return ((th + 4) + (th + 2)) * ((int64_t)W + 2); };
    int64_t th = H;
    if (floats(th) > most) {
        th = (most / ((int64_t)W + 2) - 6) / 2;
        if (th < 2) return false;
        const int64_t n = (H + th - 1) / th;                         // evened out
        th = (H + n - 1) / n;
    }
    a.B = B; a.D = D; a.H = H; a.W = W;
    a.Th = (int)th;
    a.tiles_h = (int)((H + th - 1) / th);
    // several small planes a round, so that its barriers are worth it, in at most 32 KB
    int64_t planes = kDwbCells / (th * W);
    while (planes > 1 && planes * floats(th) > most / 2) --planes;
    planes = planes < 1 ? 1 : planes > B ? B : planes;
    a.planes = (int)planes;
    // rounds per workgroup: the weights' sums cost a reduction per workgroup, but 2048 of them keep the chip full
    int64_t images = planes;
    while (images < B && (int64_t)D * a.tiles_h * ((B + 2 * images - 1) / (2 * images)) >= 2048) images *= 2;
    a.images = (int)(images > B ? B : images);
    parts = (int64_t)a.tiles_h * ((B + a.images - 1) / a.images);
    smem = (size_t)(planes * floats(th)) * 4;
    a.by_x = make_fastdiv((uint32_t)((th + 4) * (W + 2))); a.by_x_row = make_fastdiv((uint32_t)(W + 2));
    a.by_ds = make_fastdiv((uint32_t)((th + 2) * (W + 2))); a.by_ds_row = make_fastdiv((uint32_t)(W + 2));
    return parts * D <= 0x7fffffff && (int64_t)D * 10 <= 0x7fffffff;
}

template <typename T>
static int launch_dwconv_bwd(const DwBwdArgs &a, int64_t parts, size_t smem, void *dw, void *db, hipStream_t s) {
    hipLaunchKernelGGL((dwconv_bwd_kernel<T, false>), dim3((uint32_t)(parts * a.D)), dim3(kBlock), smem, s, a);
    hipLaunchKernelGGL(dwconv_bwd_sum_kernel<T>, dim3((uint32_t)(a.D * 10)), dim3(kWave), 0, s, a.partial,
                       reinterpret_cast<T *>(dw), reinterpret_cast<T *>(db), (int)parts, a.D);
    return launch_status();
}

}  // namespace ss2d

extern "C" int ss2d_dwconv3x3_silu_f32(const float *x, const float *weight, const float *bias, float *y, int B, int D, int H, int W,
                                       void *stream) {
    using namespace ss2d;
    if (B < 0 || D < 0 || H < 0 || W < 0) return SS2D_EINVAL;
    if (B == 0 || D == 0 || H == 0 || W == 0) return SS2D_OK;
    if (!x || !weight || !y) return SS2D_EINVAL;
    DwBwdArgs a;
    int64_t parts;
    size_t smem;
    if (!dwconv_bwd_plan(B, D, H, W, a, parts, smem)) return SS2D_ENOTSUP;
    a.x = x; a.w = weight; a.bias = bias; a.dy = nullptr; a.dx = y; a.partial = nullptr;
    smem = (size_t)a.planes * (a.Th + 4) * (W + 2) * 4;              // no ds
    hipLaunchKernelGGL((dwconv_bwd_kernel<float, true>), dim3((uint32_t)(parts * D)), dim3(kBlock), smem, (hipStream_t)stream, a);
    return launch_status();
}

extern "C" int64_t ss2d_dwconv3x3_silu_bwd_workspace_bytes(int B, int D, int H, int W) {
    using namespace ss2d;
    if (B < 0 || D < 0 || H < 0 || W < 0) return SS2D_EINVAL;
    if (B == 0 || D == 0 || H == 0 || W == 0) return 0;
    DwBwdArgs a;
    int64_t parts;
    size_t smem;
    if (!dwconv_bwd_plan(B, D, H, W, a, parts, smem)) return SS2D_ENOTSUP;
    return parts * D * 10 * 4;
}

extern "C" int ss2d_dwconv3x3_silu_bwd(const void *x, const void *weight, const void *bias, const void *dy, void *dx, void *dweight,
                                       void *dbias, int B, int D, int H, int W, int dtype, void *workspace,
                                       int64_t workspace_bytes, void *stream) {
    using namespace ss2d;
    if (B < 0 || D < 0 || H < 0 || W < 0) return SS2D_EINVAL;
    if (dtype != SS2D_F32 && dtype != SS2D_BF16 && dtype != SS2D_F16) return SS2D_EINVAL;
    if (B == 0 || D == 0 || H == 0 || W == 0) return SS2D_EINVAL;    // no gradient to write: the caller's zeros
    if (!x || !weight || !dy || !dx || !dweight || !workspace) return SS2D_EINVAL;
    DwBwdArgs a;
    int64_t parts;
    size_t smem;
    if (!dwconv_bwd_plan(B, D, H, W, a, parts, smem)) return SS2D_ENOTSUP;
    if (workspace_bytes < parts * D * 10 * 4) return SS2D_ENOMEM;
    a.x = x; a.w = weight; a.bias = bias; a.dy = dy; a.dx = dx;
    a.partial = reinterpret_cast<float *>(workspace);
    hipStream_t s = (hipStream_t)stream;
    switch (dtype) {
        case SS2D_F32: return launch_dwconv_bwd<float>(a, parts, smem, dweight, dbias, s);
        case SS2D_BF16: return launch_dwconv_bwd<bf16_t>(a, parts, smem, dweight, dbias, s);
        default: return launch_dwconv_bwd<f16_t>(a, parts, smem, dweight, dbias, s);
    }
}
