// Weight gradient of a projection in single precision: dw[n][k] = sum_m dy[m][n] x[m][k], m the batch's positions (the in_proj /
// out_proj of a block in training, classification/models/vmamba.py:648-662).  Few outputs and a long sum: the library's GEMM
// gives 384 x 384 outputs to 48 workgroups and walks all 12 544 positions in each, on a chip of 256 CUs.
// Here the positions are split: a workgroup owns 64 x 64 outputs over one share of them, its four wavefronts a quarter of the
// share each, and meet in LDS; a second kernel adds the shares in a fixed order (no atomics, the same bits every time).
// v_mfma_f32_16x16x4 (fp32 operands, fp32 accumulate), its operands straight from memory: a lane loads 16 bytes of a row of dy
// and of x, four positions to an instruction, which are the rows (columns) of four MFMA tiles, every fourth one in each --
// 16 products from two loads, so that a wavefront asks for 16 bytes per clock and CU at most.  Tiles of one share are
// neighbours on one XCD and read its rows from that L2.
// 12 544 positions, 384 x 384 outputs: 77 -> 54 us with the sum (69 TFLOP/s of the 154 that a large fp32 product reaches; the
// loads' latency and the shares' sum bound it); 192 x 192 over 50 176: 131 -> 74; 96 x 96 over 200 704: 443 -> 141.  With 768
// workgroups rounded up instead of 1024 rounded down: 62 us, for the few of the last wave.  Relative error against 64 bits:
// 2.2e-7, the library's 2.0e-6.  Training step of a block, 64 x 384 maps of 14 x 14: 2350 -> 2290 us.
#include "ss2d_common.h"

namespace ss2d {

typedef float dwf4_t __attribute__((ext_vector_type(4)));

constexpr int kDwTile = 64;          // outputs per side of a workgroup's tile
constexpr int kDwDepth = 4;          // steps of 4 positions loaded ahead

struct LinearDwArgs {
    const float *x, *dy;
    float *out;                      // [shares][N][K]
    int32_t N, K, tiles_k, tiles;
    int64_t M, share;                // positions, and how many a workgroup sums (a multiple of 16)
    uint32_t total;
};

__global__ __launch_bounds__(kBlock, 2) void linear_dw_kernel(const LinearDwArgs p) {
    __shared__ __align__(16) float sums[2][kDwTile][kDwTile];
    const int lane = threadIdx.x & (kWave - 1), col = lane & 15, g = lane >> 4;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave);
    const uint32_t id = xcd_contiguous_id(blockIdx.x, p.total);
    const uint32_t share = id / (uint32_t)p.tiles, tile = id - share * (uint32_t)p.tiles;
    const int n0 = (int)(tile / (uint32_t)p.tiles_k) * kDwTile, k0 = (int)(tile % (uint32_t)p.tiles_k) * kDwTile;
    const int64_t begin = (int64_t)share * p.share + wave * (p.share / 4);
    const int64_t end = begin + p.share / 4 < p.M ? begin + p.share / 4 : p.M;
    // (columns past the last repeat it, nobody stores what comes of them; N and K are multiples of 4)
    const float *dy = p.dy + min(n0 + 4 * col, p.N - 4), *x = p.x + min(k0 + 4 * col, p.K - 4);
    dwf4_t acc[4][4];
#pragma unroll
    for (int i = 0; i < 4; ++i)
#pragma unroll
        for (int j = 0; j < 4; ++j) acc[i][j] = dwf4_t{0, 0, 0, 0};
    struct Step { dwf4_t a, b; };
    auto load = [&](int64_t m, Step &s) {                            // positions m .. m + 3, lane group g the g-th of them
        const int64_t at = m + g, safe = at < p.M ? at : p.M - 1;
        s.a = *reinterpret_cast<const dwf4_t *>(dy + safe * p.N);
        s.b = *reinterpret_cast<const dwf4_t *>(x + safe * p.K);
    };
    if (begin < end) {
        Step ring[kDwDepth];
#pragma unroll
        for (int q = 0; q < kDwDepth; ++q) load(begin + 4 * q, ring[q]);
        for (int64_t m = begin; m < end; m += 4 * kDwDepth) {
#pragma unroll
            for (int q = 0; q < kDwDepth; ++q) {
                Step s = ring[q];
                load(m + 4 * (q + kDwDepth), ring[q]);
                if (m + 4 * q + g >= end) { s.a = dwf4_t{0, 0, 0, 0}; s.b = dwf4_t{0, 0, 0, 0}; }
#pragma unroll
                for (int i = 0; i < 4; ++i)
#pragma unroll
                    for (int j = 0; j < 4; ++j) acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x4f32(s.a[i], s.b[j], acc[i][j], 0, 0, 0);
            }
        }
    }
    // acc[i][j][v] is output (n0 + 16 g + 4 v + i, k0 + 4 col + j); wavefronts 2 and 3 go to 0 and 1, then 1 to 0
    auto put = [&](int slot) {
#pragma unroll
        for (int i = 0; i < 4; ++i)
#pragma unroll
            for (int v = 0; v < 4; ++v)
                *reinterpret_cast<dwf4_t *>(&sums[slot][16 * g + 4 * v + i][4 * col]) =
                    dwf4_t{acc[i][0][v], acc[i][1][v], acc[i][2][v], acc[i][3][v]};
    };
    auto add = [&](int slot) {
#pragma unroll
        for (int i = 0; i < 4; ++i)
#pragma unroll
            for (int v = 0; v < 4; ++v) {
                const dwf4_t o = *reinterpret_cast<const dwf4_t *>(&sums[slot][16 * g + 4 * v + i][4 * col]);
#pragma unroll
                for (int j = 0; j < 4; ++j) acc[i][j][v] += o[j];
            }
    };
    if (wave >= 2) put(wave - 2);
    __syncthreads();
    if (wave < 2) { add(wave); put(wave); }                          // (each its own slot)
    __syncthreads();
    float *out = p.out + (int64_t)share * p.N * p.K;
    for (int i = threadIdx.x; i < kDwTile * kDwTile / 4; i += kBlock) {
        const int n = i / (kDwTile / 4), k = i % (kDwTile / 4) * 4;
        if (n0 + n >= p.N || k0 + k >= p.K) continue;
        *reinterpret_cast<dwf4_t *>(out + (int64_t)(n0 + n) * p.K + k0 + k) =
            *reinterpret_cast<const dwf4_t *>(&sums[0][n][k]) + *reinterpret_cast<const dwf4_t *>(&sums[1][n][k]);
    }
}

__global__ __launch_bounds__(kBlock) void linear_dw_sum_kernel(const float *partial, float *dw, int shares, int64_t quads) {
    const int64_t i = (int64_t)blockIdx.x * kBlock + threadIdx.x;
    if (i >= quads) return;
    dwf4_t t = {0, 0, 0, 0};
    for (int s = 0; s < shares; ++s) t += reinterpret_cast<const dwf4_t *>(partial)[s * quads + i];
    reinterpret_cast<dwf4_t *>(dw)[i] = t;
}

// Shares of the positions: as many workgroups as are resident at once (four per CU) and no more -- a fifth on a few CUs would
// have the others wait for it --, and at least 32 positions to a wavefront.
static bool linear_dw_plan(int64_t M, int N, int K, LinearDwArgs &a, int64_t &shares) {
    if (M <= 0 || N <= 0 || K <= 0 || N % 4 != 0 || K % 4 != 0) return false;
    const int64_t tiles_k = (K + kDwTile - 1) / kDwTile, tiles = ((N + kDwTile - 1) / kDwTile) * tiles_k;
    if (tiles > 0x7fffff || (int64_t)N * K > 0x7fffffff) return false;
    shares = tiles < 1024 ? 1024 / tiles : 1;
    if (shares > (M + 127) / 128) shares = (M + 127) / 128;
    a.share = ((M + shares - 1) / shares + 15) / 16 * 16;
    shares = (M + a.share - 1) / a.share;
    a.N = N; a.K = K; a.M = M; a.tiles_k = (int)tiles_k; a.tiles = (int)tiles;
    a.total = (uint32_t)(tiles * shares);
    return true;
}

}  // namespace ss2d

extern "C" int64_t ss2d_linear_dw_f32_workspace_bytes(int64_t M, int N, int K) {
    ss2d::LinearDwArgs a;
    int64_t shares;
    if (M < 0 || N < 0 || K < 0) return SS2D_EINVAL;
    if (!ss2d::linear_dw_plan(M, N, K, a, shares)) return SS2D_ENOTSUP;
    return shares * N * K * 4;
}

extern "C" int ss2d_linear_dw_f32(const float *x, const float *dy, float *dw, int64_t M, int N, int K, void *workspace,
                                  int64_t workspace_bytes, void *stream) {
    using namespace ss2d;
    if (M < 0 || N < 0 || K < 0) return SS2D_EINVAL;
    LinearDwArgs a;
    int64_t shares;
    if (!linear_dw_plan(M, N, K, a, shares)) return SS2D_ENOTSUP;
    if (!x || !dy || !dw || !workspace) return SS2D_EINVAL;
    if ((reinterpret_cast<uintptr_t>(x) | reinterpret_cast<uintptr_t>(dy) | reinterpret_cast<uintptr_t>(dw) |
         reinterpret_cast<uintptr_t>(workspace)) % 16 != 0) return SS2D_ENOTSUP;
    if (workspace_bytes < shares * N * K * 4) return SS2D_ENOMEM;
    a.x = x; a.dy = dy; a.out = reinterpret_cast<float *>(workspace);
    hipStream_t s = (hipStream_t)stream;
    hipLaunchKernelGGL(linear_dw_kernel, dim3(a.total), dim3(kBlock), 0, s, a);
    const int64_t quads = (int64_t)N * K / 4;
    hipLaunchKernelGGL(linear_dw_sum_kernel, dim3((uint32_t)((quads + kBlock - 1) / kBlock)), dim3(kBlock), 0, s, a.out, dw, (int)shares, quads);
    return launch_status();
}
