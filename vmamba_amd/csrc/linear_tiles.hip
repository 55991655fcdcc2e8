// Products of many positions with 16-bit activations and what stands behind them, for the blocks' projections and MLP and for the 3 x 3
// convolutions of stride 2 between the stages (classification/models/vmamba.py:648-662, :1116-1131, :1430-1437):
//     out[m][n] = [GELU](sum_k x[m][k] w[n][k] + bias[n]) + residual[m][n]
// and, for a convolution, x[m][k] = the input pixel and channel that term k = (kh, kw, c) of output pixel m meets, 0 outside the image.
//   * a workgroup of four wavefronts owns kBM x kBN outputs, a wavefront a quarter of them in tiles of 32 x 32; 32 terms a step.  Operands
//     go from memory straight into LDS (global_load_lds, 16 bytes a lane), two steps ahead in a ring of three buffers -- one barrier a
//     step, and a wait that leaves the newer step's loads in flight --, or one step ahead in a ring of two (kTlThreePerCu);
//   * a row of a step is 64 bytes of LDS, its four 16-byte pieces in an order that differs from row to row, so that lanes with a row each read
//     all banks once; the order is made by the addresses the lanes load from, the LDS side being linear;
//   * a lane's accumulators are runs of four outputs of one position, where a residual is added, 8 bytes a lane.  They go through LDS into rows,
//     which leave 16 bytes a lane.
// Rounding follows the separate operators: the product with its bias is rounded to T, GELU of that once more; a residual is added before the
// rounding, as the library's addmm does it.
#include "gelu.h"

namespace ss2d {

struct TilesArgs {
    const void *x, *w, *bias, *residual;
    void *out;
    int64_t M;
    int32_t K, N, tiles_n;
    uint32_t total;
    // a convolution of (B, H, W, C) into (B, Ho, Wo, N)
    int32_t H, W, C;
    FastDiv div_image, div_wo;                                       // Ho * Wo, Wo
};

constexpr int kTlDepth = 32;

template <typename T, int kBM, int kBN, bool kGelu, int kStages> struct TilesLayout {
    static constexpr int kStage = (kBM + kBN) * kTlDepth;            // elements
    static constexpr int kPitch = kBN + 8;                           // of the outputs' rows
    static constexpr bool kTable = kGelu && ElemTraits<T>::dtype == SS2D_BF16;
    static constexpr int kElems = kStages * kStage > 64 * kPitch ? kStages * kStage : 64 * kPitch;
    static constexpr size_t kBytes = (size_t)kElems * 2 + (kTable ? kGeluEntries * sizeof(float) : 0);
};

// LDS offset of terms 8 g .. 8 g + 7 of a row
__device__ __forceinline__ int tl_at(int row, int g) { return row * kTlDepth + 8 * (g ^ (row >> 2 & 3)); }

template <int kNewer> __device__ __forceinline__ void tl_wait_and_meet() {
    // this wavefront's loads but the kNewer youngest are in LDS, and its reads of the buffer that is filled next are done
    asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)\n\ts_barrier" : : "n"(kNewer) : "memory");
}

__device__ const uint4 kTlZeros = {0u, 0u, 0u, 0u};                     // what a pixel outside the image is loaded from

template <typename T, int kBM, int kBN, bool kGelu, bool kConv, int kStages>
__global__ __launch_bounds__(kBlock, kStages == 2 ? 3 : 2) void linear_tiles_kernel(const TilesArgs p) {
    using Lay = TilesLayout<T, kBM, kBN, kGelu, kStages>;
    constexpr int kI = kBM / 64, kE = kBN / 64;                       // a wavefront's 32 x 32 tiles along positions and outputs
    constexpr int kLoadsA = kBM / 64, kLoadsB = kBN / 64;             // of a wavefront a step: 16 rows each
    extern __shared__ __align__(16) uint16_t tl_smem[];
    float *tbl = reinterpret_cast<float *>(tl_smem + Lay::kElems);
    const int lane = threadIdx.x & (kWave - 1), j = lane & 31, kh = lane >> 5;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave);
    const uint32_t id = xcd_contiguous_id(blockIdx.x, p.total);       // neighbours share positions, in one L2
    const int64_t m0 = (int64_t)(id / (uint32_t)p.tiles_n) * kBM;
    const int n0 = (int)(id % (uint32_t)p.tiles_n) * kBN;
    const int steps = p.K / kTlDepth;

    // ---- where a lane loads from: row 16 (wave + 4 i) + lane / 4 of the tile, the piece that belongs into place lane % 4 of it
    const int in_row = lane >> 2;
    const T *xa[kLoadsA], *wb[kLoadsB];
    uint32_t inside[kLoadsA];                                         // convolution: bit 3 kh + kw set where that pixel is in the image
#pragma unroll
    for (int i = 0; i < kLoadsA; ++i) {
        const int row = 16 * (wave + 4 * i) + in_row, piece = (lane & 3) ^ (row >> 2 & 3);
        const int64_t m = m0 + row < p.M ? m0 + row : p.M - 1;        // rows past the end: any valid row, never stored
        if constexpr (kConv) {
            uint32_t b, r, oh, ow;
            divmod((uint32_t)m, p.div_image, b, r);
            divmod(r, p.div_wo, oh, ow);
            const int ih = 2 * (int)oh - 1, iw = 2 * (int)ow - 1;
            uint32_t rows = 0, cols = 0;
#pragma unroll
            for (int q = 0; q < 3; ++q) {
                rows |= ih + q >= 0 && ih + q < p.H ? 7u << (3 * q) : 0u;
                cols |= iw + q >= 0 && iw + q < p.W ? 0x49u << q : 0u;
            }
            inside[i] = rows & cols;
            xa[i] = reinterpret_cast<const T *>(p.x) + (((int64_t)b * p.H + ih) * p.W + iw) * p.C + 8 * piece;
        } else {
            inside[i] = 0;
            xa[i] = reinterpret_cast<const T *>(p.x) + m * p.K + 8 * piece;
        }
    }
#pragma unroll
    for (int i = 0; i < kLoadsB; ++i) {
        const int row = 16 * (wave + 4 * i) + in_row, piece = (lane & 3) ^ (row >> 2 & 3);
        const int n = n0 + row < p.N ? n0 + row : p.N - 1;
        wb[i] = reinterpret_cast<const T *>(p.w) + (int64_t)n * p.K + 8 * piece;
    }
    int tap = 0, c0 = 0;                                              // convolution: the next step's place
    auto fetch = [&](int step, int buffer) {
        uint16_t *a = tl_smem + buffer * Lay::kStage + wave * 16 * kTlDepth, *b = a + kBM * kTlDepth;
        if constexpr (kConv) {
            const int64_t off = ((int64_t)(tap / 3) * p.W + tap % 3) * p.C + c0;
#pragma unroll
            for (int i = 0; i < kLoadsA; ++i) {
                const void *src = inside[i] >> tap & 1u ? (const void *)(xa[i] + off) : (const void *)&kTlZeros;
                load_to_lds_16(src, a + i * 64 * kTlDepth);
            }
            c0 += kTlDepth;
            if (c0 == p.C) { c0 = 0; ++tap; }
        } else {
#pragma unroll
            for (int i = 0; i < kLoadsA; ++i) load_to_lds_16(xa[i] + step * kTlDepth, a + i * 64 * kTlDepth);
        }
#pragma unroll
        for (int i = 0; i < kLoadsB; ++i) load_to_lds_16(wb[i] + step * kTlDepth, b + i * 64 * kTlDepth);
    };

    floatx16_t acc[kI][kE];
#pragma unroll
    for (int i = 0; i < kI; ++i)
#pragma unroll
        for (int e = 0; e < kE; ++e)
#pragma unroll
            for (int v = 0; v < 16; ++v) acc[i][e][v] = 0.0f;
    if constexpr (Lay::kTable)
        for (int i = threadIdx.x; i < kGeluEntries / 4; i += kBlock)
            reinterpret_cast<uint4 *>(tbl)[i] = reinterpret_cast<const uint4 *>(kGeluHalfErfBits)[i];
    const int wm = (wave & 1) * (kBM / 2), wn = (wave >> 1) * (kBN / 2);
    fetch(0, 0);
    if (kStages > 2 && steps > 1) fetch(1, 1);
    int buffer = 0;
    for (int step = 0; step < steps; ++step) {
        if (kStages > 2 && step + 1 < steps) tl_wait_and_meet<kLoadsA + kLoadsB>();
        else tl_wait_and_meet<0>();
        // (the buffer filled here was read in the step before this one, which every wavefront has left)
        if (step + kStages - 1 < steps) fetch(step + kStages - 1, buffer == 0 ? kStages - 1 : buffer - 1);
        const uint16_t *sa = tl_smem + buffer * Lay::kStage, *sb = sa + kBM * kTlDepth;
#pragma unroll
        for (int s = 0; s < 2; ++s) {
            u32x4_t fa[kI], fb[kE];
#pragma unroll
            for (int i = 0; i < kI; ++i) fa[i] = *reinterpret_cast<const u32x4_t *>(sa + tl_at(wm + 32 * i + j, 2 * s + kh));
#pragma unroll
            for (int e = 0; e < kE; ++e) fb[e] = *reinterpret_cast<const u32x4_t *>(sb + tl_at(wn + 32 * e + j, 2 * s + kh));
#pragma unroll
            for (int i = 0; i < kI; ++i)
#pragma unroll
                for (int e = 0; e < kE; ++e) acc[i][e] = mfma_32x32x16(T{}, fb[e], fa[i], acc[i][e]);
        }
        buffer = buffer == kStages - 1 ? 0 : buffer + 1;
    }
    // ---- out, 64 positions at a time through the ring's room: a lane holds, of position wm + 32 i + j, outputs wn + 32 e + 8 g + 4 kh + t
    // in accumulator 4 g + t
    const bool add = p.residual != nullptr;
#pragma unroll
    for (int i = 0; i < kI; ++i) {
        tl_wait_and_meet<0>();
        const int row = wm + 32 * i + j, slot = (wave & 1) * 32 + j;
#pragma unroll
        for (int e = 0; e < kE; ++e)
#pragma unroll
            for (int g = 0; g < 4; ++g) {
                const int n = wn + 32 * e + 8 * g + 4 * kh;
                float v[4];
#pragma unroll
                for (int t = 0; t < 4; ++t) v[t] = acc[i][e][4 * g + t];
                if (p.bias) {
                    const uint2 b = *reinterpret_cast<const uint2 *>(reinterpret_cast<const T *>(p.bias) + min(n0 + n, p.N - 4));
                    v[0] += unpack_lo<T>(b.x); v[1] += unpack_hi<T>(b.x); v[2] += unpack_lo<T>(b.y); v[3] += unpack_hi<T>(b.y);
                }
                uint2 o;
                if constexpr (kGelu) {
                    o = make_uint2(gelu_pair(T{}, pack2_from_f32<T>(v[0], v[1]), tbl), gelu_pair(T{}, pack2_from_f32<T>(v[2], v[3]), tbl));
                } else {
                    if (add && m0 + row < p.M && n0 + n < p.N) {
                        const uint2 r = *reinterpret_cast<const uint2 *>(reinterpret_cast<const T *>(p.residual) + (m0 + row) * p.N + n0 + n);
                        v[0] += unpack_lo<T>(r.x); v[1] += unpack_hi<T>(r.x); v[2] += unpack_lo<T>(r.y); v[3] += unpack_hi<T>(r.y);
                    }
                    o = make_uint2(pack2_from_f32<T>(v[0], v[1]), pack2_from_f32<T>(v[2], v[3]));
                }
                *reinterpret_cast<uint2 *>(tl_smem + slot * Lay::kPitch + n) = o;
            }
        __syncthreads();
        constexpr int kPieces = kBN / 8;
        for (int at = threadIdx.x; at < 64 * kPieces; at += kBlock) {
            const int from = at / kPieces, q = at % kPieces;
            const int64_t m = m0 + (from >> 5) * (kBM / 2) + 32 * i + (from & 31);
            if (m >= p.M || n0 + 8 * q >= p.N) continue;              // (N is a multiple of 8)
            *reinterpret_cast<uint4 *>(reinterpret_cast<T *>(p.out) + m * p.N + n0 + 8 * q) =
                *reinterpret_cast<const uint4 *>(tl_smem + from * Lay::kPitch + 8 * q);
        }
    }
}

template <typename T, int kBM, int kBN, bool kGelu, bool kConv, int kStages>
static int launch_tiles(TilesArgs a, hipStream_t s) {
    a.tiles_n = (a.N + kBN - 1) / kBN;
    const int64_t total = (a.M + kBM - 1) / kBM * a.tiles_n;
    if (total > 0x7fffffff) return SS2D_ENOTSUP;
    a.total = (uint32_t)total;
    auto kern = linear_tiles_kernel<T, kBM, kBN, kGelu, kConv, kStages>;
    constexpr size_t smem = TilesLayout<T, kBM, kBN, kGelu, kStages>::kBytes;
    if (smem > 64 * 1024 && hipFuncSetAttribute(reinterpret_cast<const void *>(kern), hipFuncAttributeMaxDynamicSharedMemorySize, (int)smem) != hipSuccess)
        return SS2D_ELAUNCH;
    hipLaunchKernelGGL(kern, dim3(a.total), dim3(kBlock), smem, s, a);
    return launch_status();
}

// With the GELU a workgroup's time is two parts, the product and what stands behind it (a gather of the table and a pass through LDS), that only
// other workgroups of the CU overlap.  A ring of two buffers leaves room for three of them (50 KB of LDS; the loads one step ahead, which the other
// two cover) where a ring of three leaves two.  us, three buffers / two, bf16 and fp16: 384 -> 1536 at 25 088 positions (1568 workgroups)
// 65 / 61 and 74 / 67, at 50 176 115 / 104 and 130 / 117, at 100 352 261 / 229 and 285 / 259; 512 -> 2048 at 12 544 (1078) 55 / 48 and 60 / 56.
// About as many workgroups as places, or fewer, gain nothing: 384 -> 1536 at 12 544 (784) 38 / 39 and 43 / 42, 256 -> 1024 at 17 000 (798) 31.5 / 32.3 and 38 / 36.
constexpr int64_t kTlThreePerCu = 1024;

template <typename T> static int launch_linear_tiles(const TilesArgs &a, bool gelu, hipStream_t s) {
    const int64_t total = (a.M + 127) / 128 * ((a.N + 191) / 192);
    if (gelu && total > kTlThreePerCu) return launch_tiles<T, 128, 192, true, false, 2>(a, s);
    if (gelu) return launch_tiles<T, 128, 192, true, false, 3>(a, s);
    return launch_tiles<T, 128, 192, false, false, 3>(a, s);
}

}  // namespace ss2d

extern "C" int ss2d_linear_tiles(const void *x, const void *weight, const void *bias, const void *residual, void *out, int64_t M, int K, int N, int gelu,
                                 int dtype, void *stream) {
    using namespace ss2d;
    if (M < 0 || K <= 0 || N <= 0 || (gelu && residual)) return SS2D_EINVAL;
    if (dtype != SS2D_F32 && dtype != SS2D_BF16 && dtype != SS2D_F16) return SS2D_EINVAL;
    if (M == 0) return SS2D_OK;
    if (!x || !weight || !out) return SS2D_EINVAL;
    if (dtype == SS2D_F32 || K % kTlDepth != 0 || N % 8 != 0) return SS2D_ENOTSUP;
    const void *ptrs[] = {x, weight, bias, residual, out};
    for (const void *q : ptrs)
        if (reinterpret_cast<uintptr_t>(q) % 16 != 0) return SS2D_ENOTSUP;
    TilesArgs a = {};
    a.x = x; a.w = weight; a.bias = bias; a.residual = residual; a.out = out; a.M = M; a.K = K; a.N = N;
    if (dtype == SS2D_BF16) return launch_linear_tiles<bf16_t>(a, gelu != 0, (hipStream_t)stream);
    return launch_linear_tiles<f16_t>(a, gelu != 0, (hipStream_t)stream);
}

extern "C" int ss2d_conv3x3s2_cl(const void *x, const void *weight, const void *bias, void *out, int B, int H, int W, int C, int N, int dtype, void *stream) {
    using namespace ss2d;
    if (B < 0 || H < 0 || W < 0 || C <= 0 || N <= 0) return SS2D_EINVAL;
    if (dtype != SS2D_F32 && dtype != SS2D_BF16 && dtype != SS2D_F16) return SS2D_EINVAL;
    if (B == 0 || H == 0 || W == 0) return SS2D_OK;
    if (!x || !weight || !out) return SS2D_EINVAL;
    const int64_t Ho = (H + 1) / 2, Wo = (W + 1) / 2, M = B * Ho * Wo;
    if (dtype == SS2D_F32 || C % kTlDepth != 0 || N % 8 != 0 || M > 0x7fffffff || C > 0x7fffffff / 9) return SS2D_ENOTSUP;
    const void *ptrs[] = {x, weight, bias, out};
    for (const void *q : ptrs)
        if (reinterpret_cast<uintptr_t>(q) % 16 != 0) return SS2D_ENOTSUP;
    TilesArgs a = {};
    a.x = x; a.w = weight; a.bias = bias; a.out = out; a.M = M; a.K = 9 * C; a.N = N; a.H = H; a.W = W; a.C = C;
    a.div_image = make_fastdiv((uint32_t)(Ho * Wo)); a.div_wo = make_fastdiv((uint32_t)Wo);
    if (dtype == SS2D_BF16) return launch_tiles<bf16_t, 128, 192, false, true, 3>(a, (hipStream_t)stream);
    return launch_tiles<f16_t, 128, 192, false, true, 3>(a, (hipStream_t)stream);
}
