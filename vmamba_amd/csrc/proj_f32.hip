// x_proj and dt_proj of the SS2D core in single precision (classification/models/vmamba.py:605-615): the reference's own
// throughput harness runs fp32.  Both contractions are far too narrow for the library's GEMM tiles -- on 192 x 28 x 28 maps,
// batch 32, dt_proj (12 ranks) took 42 us for 77 MB of result, x_proj (4 x 14 rows) and the CrossScan behind it 22.  Here:
// v_mfma_f32_16x16x4 (fp32 operands, fp32 accumulate: the arithmetic of the library's product), operands straight from
// memory in the lane order the instruction wants, 64 positions to a wavefront.  (The same kernels on the vector units, the
// weights through scalar loads: 25 + 22 us there and 46 for 24 ranks on 384 x 14 x 14, waiting for the scalar loads.)
//   x_proj: 192 x 28 x 28, batch 32: 22 -> 14.5 us; 96 x 56 x 56, batch 32: 50 -> 20.5; 384 x 14 x 14, batch 64: 60 -> 23.4;
//     one map of 768 x 7 x 7: 47 -> 28
//   dt_proj: 42 -> 16.6 us (4.6 TB/s), 104 -> 27 (5.7 TB/s), 39 -> 26.5
#include "ss2d_common.h"

namespace ss2d {

// v_mfma_f32_16x16x4: D (16 x 16) += A (16 x 4) * B (4 x 16).  Lane l supplies A[l % 16][l / 16] and B[l / 16][l % 16] and
// holds D[4 * (l / 16) + v][l % 16] in accumulator v.
typedef float f32x4_t __attribute__((ext_vector_type(4)));
__device__ __forceinline__ f32x4_t mfma_16x16x4(float a, float b, f32x4_t c) {
    return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0);
}

// ---- x_proj + one-by-one CrossScan --------------------------------------------------------------------------------
// A workgroup owns 64 positions (of any images: maps need not fill wavefronts) and up to 64 of the 4 C output rows, so that
// the map is read once where 4 C <= 64.  Its wavefronts split the channels -- 25 088 positions are only 392 wavefronts -- and
// meet in LDS.  A lane loads 4 consecutive positions of a channel: the columns of four MFMA tiles, every fourth position in
// each.  Every row is then stored at its direction's place; the transposing directions write single floats H apart, into a
// result small enough for L2 to assemble.
struct XProjF32Args {
    const float *x, *W;
    float *out;
    int32_t D, C, H, Wd, n_chunks;
    int64_t ks, cs, bs, n_pos;
    uint32_t total;
    bool w_vec;                          // weight rows in 16-byte pieces
    FastDiv by_map, by_row, by_rows;
};

// kVec: a lane's four positions are 16 aligned bytes of one map (H * W a multiple of 4, x on 16 bytes)
template <int kMt, bool kVec>
__global__ __launch_bounds__(kBlock, kMt == 4 ? 2 : 3) void x_proj_f32_kernel(const XProjF32Args p) {
    constexpr int kWaves = kBlock / kWave, kRows = 16 * kMt, kPitch = kWave + 4;
    __shared__ __align__(16) float sums[2][kRows][kPitch];
    const int lane = threadIdx.x & (kWave - 1), col = lane & 15, g = lane >> 4;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave);
    const uint32_t id = xcd_contiguous_id(blockIdx.x, p.total);      // the row chunks of one set of positions share an L2
    const uint32_t tile = id / p.n_chunks, chunk = id - tile * p.n_chunks;
    const int row0 = (int)chunk * kRows, n_rows = min(kRows, 4 * p.C - row0);
    const int64_t HW = (int64_t)p.H * p.Wd, first = (int64_t)tile * kWave;
    const float *xp[kVec ? 1 : 4];
#pragma unroll
    for (int i = 0; i < (kVec ? 1 : 4); ++i) {
        const int64_t at = first + 4 * col + i;
        uint32_t b, pos;
        divmod((uint32_t)(at < p.n_pos ? at : 0), p.by_map, b, pos); // (positions past the last repeat the first: not stored)
        xp[i] = p.x + (int64_t)b * p.D * HW + pos;
    }
    const float *w_row[kMt];
#pragma unroll
    for (int m = 0; m < kMt; ++m) w_row[m] = p.W + (int64_t)(row0 + min(16 * m + col, n_rows - 1)) * p.D;
    f32x4_t acc[kMt][4];
#pragma unroll
    for (int m = 0; m < kMt; ++m)
#pragma unroll
        for (int t = 0; t < 4; ++t) acc[m][t] = f32x4_t{0, 0, 0, 0};
    // 16 channels a step, 4 to a lane group; product s of a step takes channel 4 g + s of every group
    for (int d0 = wave * 16; d0 < p.D; d0 += kWaves * 16) {
        const int d = d0 + 4 * g;
        f32x4_t a[kMt], v[4];
        if (d + 4 <= p.D) {
#pragma unroll
            for (int s = 0; s < 4; ++s) {
                if constexpr (kVec) v[s] = *reinterpret_cast<const f32x4_t *>(xp[0] + (d + s) * HW);
                else v[s] = f32x4_t{xp[0][(d + s) * HW], xp[1][(d + s) * HW], xp[2][(d + s) * HW], xp[3][(d + s) * HW]};
            }
#pragma unroll
            for (int m = 0; m < kMt; ++m) {
                if (p.w_vec) a[m] = *reinterpret_cast<const f32x4_t *>(w_row[m] + d);
                else a[m] = f32x4_t{w_row[m][d], w_row[m][d + 1], w_row[m][d + 2], w_row[m][d + 3]};
            }
        } else {                                                     // channels past the last count as 0
#pragma unroll
            for (int s = 0; s < 4; ++s) {
                const bool in = d + s < p.D;
                const int64_t off = (in ? d + s : 0) * HW;
                if constexpr (kVec) v[s] = *reinterpret_cast<const f32x4_t *>(xp[0] + off);
                else v[s] = f32x4_t{xp[0][off], xp[1][off], xp[2][off], xp[3][off]};
                if (!in) v[s] = f32x4_t{0, 0, 0, 0};
#pragma unroll
                for (int m = 0; m < kMt; ++m) a[m][s] = in ? w_row[m][d + s] : 0.0f;
            }
        }
#pragma unroll
        for (int s = 0; s < 4; ++s)
#pragma unroll
            for (int m = 0; m < kMt; ++m)
#pragma unroll
                for (int t = 0; t < 4; ++t) acc[m][t] = mfma_16x16x4(a[m][s], v[s][t], acc[m][t]);
    }
    // the four wavefronts' sums, pairwise: 2 and 3 to 0 and 1, then 1 to 0.  Accumulator (m, t)[i] is row 16 m + 4 g + i of
    // position 4 col + t.
    auto put = [&](int slot) {
#pragma unroll
        for (int m = 0; m < kMt; ++m)
#pragma unroll
            for (int i = 0; i < 4; ++i)
                *reinterpret_cast<f32x4_t *>(&sums[slot][16 * m + 4 * g + i][4 * col]) =
                    f32x4_t{acc[m][0][i], acc[m][1][i], acc[m][2][i], acc[m][3][i]};
    };
    auto add = [&](int slot) {
#pragma unroll
        for (int m = 0; m < kMt; ++m)
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                const f32x4_t o = *reinterpret_cast<const f32x4_t *>(&sums[slot][16 * m + 4 * g + i][4 * col]);
#pragma unroll
                for (int t = 0; t < 4; ++t) acc[m][t][i] += o[t];
            }
    };
    if (wave >= 2) put(wave - 2);
    __syncthreads();
    if (wave < 2) add(wave);
    __syncthreads();
    if (wave == 1) put(1);
    __syncthreads();
    if (wave == 0) { add(1); put(0); }
    __syncthreads();
    const int64_t at = first + lane;
    if (at >= p.n_pos) return;
    uint32_t b, pos, h, w;
    divmod((uint32_t)at, p.by_map, b, pos);
    divmod(pos, p.by_row, h, w);
    const int64_t turned = (int64_t)w * p.H + h;
    float *out = p.out + (int64_t)b * p.bs;
    for (int r = wave; r < n_rows; r += kWaves) {
        uint32_t k, c;
        divmod((uint32_t)(row0 + r), p.by_rows, k, c);
        const int64_t j = k & 1 ? turned : (int64_t)pos;
        out[k * p.ks + c * p.cs + (k >= 2 ? HW - 1 - j : j)] = sums[0][r][lane];
    }
}

template <bool kVec>
static void launch_x_f32(const XProjF32Args &a, int tiles, hipStream_t s) {
    if (tiles == 1) hipLaunchKernelGGL((x_proj_f32_kernel<1, kVec>), dim3(a.total), dim3(kBlock), 0, s, a);
    else if (tiles == 2) hipLaunchKernelGGL((x_proj_f32_kernel<2, kVec>), dim3(a.total), dim3(kBlock), 0, s, a);
    else hipLaunchKernelGGL((x_proj_f32_kernel<4, kVec>), dim3(a.total), dim3(kBlock), 0, s, a);
}

// ---- dt_proj --------------------------------------------------------------------------------------------------------
// delta[k, d, n] = sum_r W[k, d, r] * x[k, r, n]: bound by the write of delta.  A wavefront keeps the ranks of 64 positions
// (16 bytes of four ranks per product) and walks channels, 16 to a tile; a lane's accumulators are 4 channels of 4 consecutive
// positions, so a store instruction writes 4 rows of 256 bytes.
struct DtF32Args {
    const float *x, *W;
    float *out;
    int32_t K, D, R, d_tiles, n_chunks;  // d_tiles: channel tiles per wavefront
    int64_t N, ks, rs, n_blocks, n_waves;
    bool streaming;
};

template <int kSteps, bool kVec>
__global__ __launch_bounds__(kBlock) void dt_proj_f32_kernel(const DtF32Args p) {
    const int lane = threadIdx.x & (kWave - 1), col = lane & 15, g = lane >> 4;
    int64_t id = (int64_t)blockIdx.x * (kBlock / kWave) + __builtin_amdgcn_readfirstlane(threadIdx.x / kWave);
    if (id >= p.n_waves) return;
    const int chunk = (int)(id % p.n_chunks);
    id /= p.n_chunks;
    const int64_t block = id % p.n_blocks, k = id / p.n_blocks;
    const int64_t n = block * kWave + 4 * col;
    const float *x = p.x + k * p.ks;
    f32x4_t v[kSteps];
#pragma unroll
    for (int s = 0; s < kSteps; ++s) {
        const int r = 4 * s + g;
        const float *row = x + (int64_t)min(r, p.R - 1) * p.rs;
        if constexpr (kVec) v[s] = *reinterpret_cast<const f32x4_t *>(row + (n < p.N ? n : 0));
        else
#pragma unroll
            for (int t = 0; t < 4; ++t) v[s][t] = row[n + t < p.N ? n + t : 0];
        if (r >= p.R) v[s] = f32x4_t{0, 0, 0, 0};
    }
    const int tile0 = chunk * p.d_tiles, tile1 = min((p.D + 15) / 16, tile0 + p.d_tiles);
    const float *W = p.W + k * (int64_t)p.D * p.R;
    auto weights = [&](int tile, float (&a)[kSteps]) {
        const float *row = W + (int64_t)min(tile * 16 + col, p.D - 1) * p.R;
#pragma unroll
        for (int s = 0; s < kSteps; ++s) a[s] = row[min(4 * s + g, p.R - 1)];
    };
    float a[kSteps], next[kSteps];
    weights(tile0, a);
    for (int tile = tile0; tile < tile1; ++tile) {
        weights(min(tile + 1, tile1 - 1), next);                     // in flight during this tile's products
        f32x4_t acc[4];
#pragma unroll
        for (int t = 0; t < 4; ++t) acc[t] = f32x4_t{0, 0, 0, 0};
#pragma unroll
        for (int s = 0; s < kSteps; ++s) {
            const float as = 4 * s + g < p.R ? a[s] : 0.0f;
#pragma unroll
            for (int t = 0; t < 4; ++t) acc[t] = mfma_16x16x4(as, v[s][t], acc[t]);
        }
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const int d = tile * 16 + 4 * g + i;
            if (d >= p.D) continue;
            float *out = p.out + (k * p.D + d) * p.N + n;
            const f32x4_t o = {acc[0][i], acc[1][i], acc[2][i], acc[3][i]};
            if constexpr (kVec) {
                if (n < p.N) {
                    if (p.streaming) __builtin_nontemporal_store(o, reinterpret_cast<f32x4_t *>(out));
                    else *reinterpret_cast<f32x4_t *>(out) = o;
                }
            } else {
#pragma unroll
                for (int t = 0; t < 4; ++t)
                    if (n + t < p.N) out[t] = o[t];
            }
        }
#pragma unroll
        for (int s = 0; s < kSteps; ++s) a[s] = next[s];
    }
}

template <int kSteps>
static void launch_dt_f32(const DtF32Args &a, bool vec, hipStream_t s) {
    const uint32_t grid = (uint32_t)((a.n_waves + kBlock / kWave - 1) / (kBlock / kWave));
    if (vec) hipLaunchKernelGGL((dt_proj_f32_kernel<kSteps, true>), dim3(grid), dim3(kBlock), 0, s, a);
    else hipLaunchKernelGGL((dt_proj_f32_kernel<kSteps, false>), dim3(grid), dim3(kBlock), 0, s, a);
}

// beyond 24 ranks the library's GEMM is level with it (768 x 28 x 28, batch 4, 48 ranks: 29 us either way) or ahead (one
// map of 7 x 7: 5 us against 9)
bool dt_proj_f32_takes(int R) { return R > 0 && R <= 24; }

}  // namespace ss2d

extern "C" int ss2d_x_proj_f32(const float *x, const float *weight, float *out, int B, int D, int C, int H, int W,
                               int64_t out_dir_stride, int64_t out_chan_stride, int64_t out_batch_stride, void *stream) {
    using namespace ss2d;
    if (B < 0 || D < 0 || C < 0 || H < 0 || W < 0) return SS2D_EINVAL;
    if (out_dir_stride < 0 || out_chan_stride < 0 || out_batch_stride < 0) return SS2D_EINVAL;
    if (B == 0 || C == 0 || H == 0 || W == 0) return SS2D_OK;
    if (!x || !weight || !out) return SS2D_EINVAL;
    const int64_t HW = (int64_t)H * W;
    XProjF32Args a;
    a.x = x; a.W = weight; a.out = out;
    a.D = D; a.C = C; a.H = H; a.Wd = W;
    a.ks = out_dir_stride; a.cs = out_chan_stride; a.bs = out_batch_stride;
    a.n_pos = B * HW;
    const int tiles = C <= 4 ? 1 : C <= 8 ? 2 : 4;               // of 16 rows
    a.n_chunks = (4 * C + 16 * tiles - 1) / (16 * tiles);
    const int64_t total = (a.n_pos + kWave - 1) / kWave * a.n_chunks;
    if (D == 0 || a.n_pos > 0x7fffffff || total > 0x7fffffff) return SS2D_ENOTSUP;
    a.total = (uint32_t)total;
    a.by_map = make_fastdiv((uint32_t)HW);
    a.by_row = make_fastdiv((uint32_t)W);
    a.by_rows = make_fastdiv((uint32_t)C);
    a.w_vec = D % 4 == 0 && reinterpret_cast<uintptr_t>(weight) % 16 == 0;
    hipStream_t s = (hipStream_t)stream;
    if (HW % 4 == 0 && reinterpret_cast<uintptr_t>(x) % 16 == 0) launch_x_f32<true>(a, tiles, s);
    else launch_x_f32<false>(a, tiles, s);
    return launch_status();
}

extern "C" int ss2d_dt_proj_f32(const float *x, const float *weight, float *delta, int K, int D, int R, int64_t N,
                                int64_t x_dir_stride, int64_t x_rank_stride, void *stream) {
    using namespace ss2d;
    if (K < 0 || D < 0 || R < 0 || N < 0 || x_dir_stride < 0 || x_rank_stride < 0) return SS2D_EINVAL;
    if (K == 0 || D == 0 || N == 0) return SS2D_OK;
    if (!x || !weight || !delta) return SS2D_EINVAL;
    if (!dt_proj_f32_takes(R)) return SS2D_ENOTSUP;
    DtF32Args a;
    a.x = x; a.W = weight; a.out = delta;
    a.K = K; a.D = D; a.R = R; a.N = N; a.ks = x_dir_stride; a.rs = x_rank_stride;
    a.n_blocks = (N + kWave - 1) / kWave;
    // a wavefront reads its positions' ranks once per chunk of channels: long chunks, shorter ones where the chip would idle
    const int tiles = (D + 15) / 16;
    a.d_tiles = 8;
    while (a.d_tiles > 1 && K * a.n_blocks * ((tiles + a.d_tiles - 1) / a.d_tiles) < 4096) a.d_tiles /= 2;
    a.n_chunks = (tiles + a.d_tiles - 1) / a.d_tiles;
    a.n_waves = K * a.n_blocks * a.n_chunks;
    if (a.n_waves > 0x7fffffff) return SS2D_ENOTSUP;
    // as for the 16-bit kernel: what the last-level cache cannot hold until the core reads it goes past it
    a.streaming = (int64_t)K * D * N * 4 > ((int64_t)256 << 20);
    const bool vec = N % 4 == 0 && x_dir_stride % 4 == 0 && x_rank_stride % 4 == 0 &&
                     reinterpret_cast<uintptr_t>(x) % 16 == 0 && reinterpret_cast<uintptr_t>(delta) % 16 == 0;
    hipStream_t s = (hipStream_t)stream;
    if (R <= 4) launch_dt_f32<1>(a, vec, s);
    else if (R <= 8) launch_dt_f32<2>(a, vec, s);
    else if (R <= 12) launch_dt_f32<3>(a, vec, s);
    else launch_dt_f32<6>(a, vec, s);
    return launch_status();
}
