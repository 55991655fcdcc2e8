// Channel-last projection of few positions with its neighbours folded in:
//     out = [GELU]([LayerNorm](x) W^T + bias) + residual          x (M, K), W (N, K), 16-bit tensors
// -- in_proj behind the block's first LayerNorm, out_proj with the residual add, and the MLP's two layers with the second
// LayerNorm, the GELU and the add (classification/models/vmamba.py:1225-1229, :648-650, :662, :1116-1131), where a batch has so
// few positions that every one of these is a launch bound by latency: seven launches of a block become four.
//   * a workgroup owns 32 positions x 32 outputs and its wavefronts split the contraction: a wavefront's whole share of x and W
//     (kPer steps of 16) is loaded straight into matrix-core fragments, all loads in flight together, so that a call costs one
//     trip to the L2 and no loop.  784 x 192 x 192 has 150 workgroups this way, 49 x 768 x 768 48 of 8 wavefronts;
//   * the LayerNorm runs on those fragments: a position's channels lie in two lanes of every wavefront, the sums meet in LDS
//     (fp32, centred variance), the normalised values are rounded to T and multiplied;
//   * the wavefronts' partial sums meet in LDS in fp32, in their order; what is stored is 64 bytes per position.
// Rounding follows the separate operators: LayerNorm output, projection output (+ bias) and GELU are each rounded to T; the
// residual is added before the rounding where no GELU lies between, as the library's addmm does it.
#include "gelu.h"

namespace ss2d {

struct RowsArgs {
    const void *x, *ln_w, *ln_b, *w, *bias, *residual;
    void *out;
    int64_t M;
    int K, N, n_tiles;
    float eps;
};

constexpr int kRowsTile = 32;
constexpr int kRowsMaxLnWaves = 8;

// kFull: every wavefront has kPer steps.
template <typename T, int kPer, int kMaxThreads, bool kLN, bool kGelu, bool kFull>
__global__ __launch_bounds__(kMaxThreads) void linear_rows_kernel(const RowsArgs p) {
    extern __shared__ __align__(16) float4 rows_red[];               // [waves][4][64]: accumulators 4g .. 4g+3 of each lane
    const int lane = threadIdx.x & (kWave - 1);
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave);
    const int waves = blockDim.x / kWave;
    const int j = lane & 31, kh = lane >> 5;
    // outputs fastest: with a multiple of 8 tiles the workgroups that share W's rows meet in one XCD's L2
    const int n0 = (int)(blockIdx.x % (uint32_t)p.n_tiles) * kRowsTile;
    const int64_t m0 = (int64_t)(blockIdx.x / (uint32_t)p.n_tiles) * kRowsTile;
    const int64_t pos = m0 + j < p.M ? m0 + j : p.M - 1;             // rows past the end: any valid row, never stored
    const int n_row = n0 + j < p.N ? n0 + j : p.N - 1;
    const int steps = p.K / 16;
    const int s0 = wave * kPer;
    const int mine = kFull ? kPer : min(kPer, steps - s0);           // this wavefront's steps of 16 (the last one may have fewer)
    const T *xr = reinterpret_cast<const T *>(p.x) + pos * p.K + 16 * s0 + 8 * kh;
    const T *wr = reinterpret_cast<const T *>(p.w) + (int64_t)n_row * p.K + 16 * s0 + 8 * kh;

    u32x4_t xf[kPer], wf[kPer];
#pragma unroll
    for (int s = 0; s < kPer; ++s) {
        const int at = 16 * (kFull ? s : min(s, mine - 1));          // (past the share: loaded again, not used)
        xf[s] = *reinterpret_cast<const u32x4_t *>(xr + at);
        wf[s] = *reinterpret_cast<const u32x4_t *>(wr + at);
    }
    __builtin_amdgcn_sched_barrier(0);                               // all of them in flight before the first is waited for
    if constexpr (kLN) {
        __shared__ float part[2][kRowsMaxLnWaves][kRowsTile];
        float sum = 0.0f;
#pragma unroll
        for (int s = 0; s < kPer; ++s)
            if (kFull || s < mine) {
#pragma unroll
                for (int e = 0; e < 4; ++e) sum += unpack_lo<T>(xf[s][e]) + unpack_hi<T>(xf[s][e]);
            }
        sum += __shfl_xor(sum, 32);
        if (kh == 0) part[0][wave][j] = sum;
        __syncthreads();
        float total = 0.0f;
        for (int v = 0; v < waves; ++v) total += part[0][v][j];
        const float inv_k = 1.0f / (float)p.K, mean = total * inv_k;
        float sq = 0.0f;
#pragma unroll
        for (int s = 0; s < kPer; ++s)
            if (kFull || s < mine) {
#pragma unroll
                for (int e = 0; e < 4; ++e) {
                    const float a = unpack_lo<T>(xf[s][e]) - mean, b = unpack_hi<T>(xf[s][e]) - mean;
                    sq = fmaf(a, a, fmaf(b, b, sq));
                }
            }
        sq += __shfl_xor(sq, 32);
        if (kh == 0) part[1][wave][j] = sq;
        __syncthreads();
        float sq_total = 0.0f;
        for (int v = 0; v < waves; ++v) sq_total += part[1][v][j];
        const float rstd = __builtin_amdgcn_rsqf(sq_total * inv_k + p.eps);
        const T *gr = reinterpret_cast<const T *>(p.ln_w) + 16 * s0 + 8 * kh;
        const T *br = reinterpret_cast<const T *>(p.ln_b) + 16 * s0 + 8 * kh;
#pragma unroll
        for (int s = 0; s < kPer; ++s)
            if (kFull || s < mine) {
                const u32x4_t gw = *reinterpret_cast<const u32x4_t *>(gr + 16 * s);
                u32x4_t bw = {0u, 0u, 0u, 0u};
                if (p.ln_b) bw = *reinterpret_cast<const u32x4_t *>(br + 16 * s);
#pragma unroll
                for (int e = 0; e < 4; ++e)
                    xf[s][e] = pack2_from_f32<T>(fmaf((unpack_lo<T>(xf[s][e]) - mean) * rstd, unpack_lo<T>(gw[e]), unpack_lo<T>(bw[e])),
                                                 fmaf((unpack_hi<T>(xf[s][e]) - mean) * rstd, unpack_hi<T>(gw[e]), unpack_hi<T>(bw[e])));
            }
    }
    floatx16_t acc;
#pragma unroll
    for (int v = 0; v < 16; ++v) acc[v] = 0.0f;
#pragma unroll
    for (int s = 0; s < kPer; ++s)
        if (kFull || s < mine) acc = mfma_32x32x16(T{}, wf[s], xf[s], acc);   // lane (position j): outputs 8g + 4kh + t in accumulator 4g + t
#pragma unroll
    for (int g = 0; g < 4; ++g) rows_red[(wave * 4 + g) * kWave + lane] = make_float4(acc[4 * g], acc[4 * g + 1], acc[4 * g + 2], acc[4 * g + 3]);
    __syncthreads();

    // 32 positions x 8 runs of four outputs, one per thread
    for (int q = threadIdx.x; q < 8 * kRowsTile; q += blockDim.x) {
        const int row = q >> 3, run = q & 7;
        const int src = (run >> 1) * kWave + row + 32 * (run & 1);
        float4 t = rows_red[src];
        for (int v = 1; v < waves; ++v) {
            const float4 o = rows_red[v * 4 * kWave + src];
            t.x += o.x; t.y += o.y; t.z += o.z; t.w += o.w;
        }
        const int64_t at = m0 + row;
        const int n = n0 + 4 * run;
        if (at >= p.M || n >= p.N) continue;
        if (p.bias) {
            const uint2 b = *reinterpret_cast<const uint2 *>(reinterpret_cast<const T *>(p.bias) + n);
            t.x += unpack_lo<T>(b.x); t.y += unpack_hi<T>(b.x); t.z += unpack_lo<T>(b.y); t.w += unpack_hi<T>(b.y);
        }
        uint2 o;
        if constexpr (kGelu) {
            const float *tbl = reinterpret_cast<const float *>(kGeluHalfErfBits);
            o = make_uint2(gelu_pair(T{}, pack2_from_f32<T>(t.x, t.y), tbl), gelu_pair(T{}, pack2_from_f32<T>(t.z, t.w), tbl));
            if (p.residual) { t.x = unpack_lo<T>(o.x); t.y = unpack_hi<T>(o.x); t.z = unpack_lo<T>(o.y); t.w = unpack_hi<T>(o.y); }
        }
        if (p.residual) {
            const uint2 r = *reinterpret_cast<const uint2 *>(reinterpret_cast<const T *>(p.residual) + at * p.N + n);
            t.x += unpack_lo<T>(r.x); t.y += unpack_hi<T>(r.x); t.z += unpack_lo<T>(r.y); t.w += unpack_hi<T>(r.y);
        }
        if (!kGelu || p.residual) o = make_uint2(pack2_from_f32<T>(t.x, t.y), pack2_from_f32<T>(t.z, t.w));
        *reinterpret_cast<uint2 *>(reinterpret_cast<T *>(p.out) + at * p.N + n) = o;
    }
}

template <typename T, int kPer, int kMaxThreads, bool kLN, bool kFull>
static void launch_rows_ln(const RowsArgs &a, bool gelu, uint32_t n_wg, hipStream_t stream) {
    const int waves = (a.K / 16 + kPer - 1) / kPer;
    const dim3 grid(n_wg), block(waves * kWave);
    const size_t smem = (size_t)waves * 16 * kWave * sizeof(float);
    if (gelu) hipLaunchKernelGGL((linear_rows_kernel<T, kPer, kMaxThreads, kLN, true, kFull>), grid, block, smem, stream, a);
    else hipLaunchKernelGGL((linear_rows_kernel<T, kPer, kMaxThreads, kLN, false, kFull>), grid, block, smem, stream, a);
}

template <typename T, int kPer, int kMaxThreads, bool kMayLN>
static void launch_rows(const RowsArgs &a, bool gelu, uint32_t n_wg, hipStream_t stream) {
    const bool full = a.K / 16 % kPer == 0;
    if constexpr (kMayLN)
        if (a.ln_w)
            return full ? launch_rows_ln<T, kPer, kMaxThreads, true, true>(a, gelu, n_wg, stream)
                        : launch_rows_ln<T, kPer, kMaxThreads, true, false>(a, gelu, n_wg, stream);
    return full ? launch_rows_ln<T, kPer, kMaxThreads, false, true>(a, gelu, n_wg, stream)
                : launch_rows_ln<T, kPer, kMaxThreads, false, false>(a, gelu, n_wg, stream);
}

static int64_t rows_grid(int64_t M, int N) { return (M + kRowsTile - 1) / kRowsTile * ((N + kRowsTile - 1) / kRowsTile); }

template <typename T>
static int launch_rows_for(const RowsArgs &a, bool gelu, hipStream_t stream) {
    const int64_t n_wg = rows_grid(a.M, a.N);
    const int steps = a.K / 16;
    // up to 4 wavefronts of 3 steps, 8 or 16 of 6, 16 of 12: the shares a wavefront holds in registers at once
    if (steps <= 12) launch_rows<T, 3, 256, true>(a, gelu, (uint32_t)n_wg, stream);
    else if (steps <= 6 * kRowsMaxLnWaves) launch_rows<T, 6, 512, true>(a, gelu, (uint32_t)n_wg, stream);
    else if (steps <= 96) launch_rows<T, 6, 1024, false>(a, gelu, (uint32_t)n_wg, stream);
    else launch_rows<T, 12, 1024, false>(a, gelu, (uint32_t)n_wg, stream);
    return launch_status();
}

bool linear_rows_takes(int64_t M, int K, int N, bool layer_norm, int dtype) {
    return dtype != SS2D_F32 && K % 16 == 0 && K <= 3072 && N % 8 == 0 && (!layer_norm || K <= 16 * 6 * kRowsMaxLnWaves) &&
           rows_grid(M, N) <= 0x7fffffff;
}

}  // namespace ss2d

extern "C" int ss2d_linear_rows(const void *x, const void *ln_weight, const void *ln_bias, float eps, const void *weight, const void *bias,
                                const void *residual, void *out, int64_t M, int K, int N, int gelu, int dtype, void *stream) {
    using namespace ss2d;
    if (M < 0 || K <= 0 || N <= 0) return SS2D_EINVAL;
    if (dtype != SS2D_F32 && dtype != SS2D_BF16 && dtype != SS2D_F16) return SS2D_EINVAL;
    if (M == 0) return SS2D_OK;
    if (!x || !weight || !out || (ln_bias && !ln_weight)) return SS2D_EINVAL;
    if (!linear_rows_takes(M, K, N, ln_weight != nullptr, dtype)) return SS2D_ENOTSUP;
    const void *ptrs[] = {x, ln_weight, ln_bias, weight, bias, residual, out};
    for (const void *q : ptrs)
        if (q && (reinterpret_cast<uintptr_t>(q) & 15u) != 0) return SS2D_ENOTSUP;
    const RowsArgs a = {x, ln_weight, ln_bias, weight, bias, residual, out, M, K, N, (N + kRowsTile - 1) / kRowsTile, eps};
    if (dtype == SS2D_BF16) return launch_rows_for<bf16_t>(a, gelu != 0, (hipStream_t)stream);
    return launch_rows_for<f16_t>(a, gelu != 0, (hipStream_t)stream);
}
