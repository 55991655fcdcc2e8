// Second layer of the patch embedding in one kernel (classification/models/vmamba.py:1412-1416, patch-embed v2):
//     y = LayerNorm(conv2d(x, w, b; kernel 3, stride 2, padding 1)),  x (B, H, W, 48), y (B, Ho, Wo, 96), 16-bit, channel-last.
// The library's implicit GEMM took 455 us for 128 images of 112 x 112 (33 GFLOP on 231 MB, a tile of 32 columns out of 96), and
// the LayerNorm behind it another pass over the activation.  All 96 x 432 weights fit the LDS of one CU (81 KB), so
//   * one workgroup of 8 wavefronts per CU brings them in once, in the order the matrix cores read them, and after that no
//     wavefront waits for another: each walks its own 64 positions at a time, 9 taps of 3 steps of v_mfma_f32_32x32x16 with the
//     weights as the A operand (rows = output channels) and the positions as columns;
//   * a lane's B operand is 8 channels of one input position, 16 bytes as they lie in memory: loaded straight to registers, one
//     tap ahead, through a buffer descriptor whose range check gives the zeros of the padding;
//   * a lane ends up with half of the channels of its position, so the LayerNorm is a sum over the lane and one exchange; the
//     result leaves through a wavefront-private LDS tile as runs of 1 KB.
// 128 images of 112 x 112: 455 us and the LayerNorm's 35 -> 94 us (2.5 TB/s, 0.35 PFLOP/s: the taps' 16-byte pieces lie 192
// bytes apart, and it is their cache lines through L1 that bound it); one image: 21 + 4 + two layout copies -> 28.
// Rounded to 16 bits where the separate operators are: the convolution (with its bias) and the LayerNorm's result.
#include "ss2d_common.h"

namespace ss2d {

constexpr int kS2Cin = 48, kS2Cout = 96, kS2Waves = 8;
constexpr int kS2Chunks = kS2Cin / 16, kS2Steps = 9 * kS2Chunks, kS2Mt = kS2Cout / 32;
constexpr int kS2Unit = 64;              // positions per wavefront and turn: two MFMA column tiles
constexpr int kS2Pitch = kS2Cout + 8;    // output tile: rows of 208 bytes, 16-byte pieces that meet in few banks
constexpr size_t kS2WeightBytes = (size_t)kS2Steps * kS2Mt * kWave * 16;
constexpr size_t kS2Smem = kS2WeightBytes + 3 * kS2Cout * sizeof(float) + (size_t)kS2Waves * 32 * kS2Pitch * 2;

struct Stem2Args {
    const void *x, *w, *b, *gamma, *beta;
    void *y;
    int32_t H, W, n_pos, n_units, units_per_wg, x_bytes;
    int64_t ws_o, ws_c, ws_h, ws_w;      // weight strides (elements)
    float eps;
    FastDiv by_map, by_row;              // output positions per image, per row
};

template <typename T>
__global__ __launch_bounds__(kS2Waves * kWave, 2) void stem_conv2_ln_kernel(const Stem2Args p) {
    extern __shared__ __align__(16) unsigned char s2_smem[];
    u32x4_t *wl = reinterpret_cast<u32x4_t *>(s2_smem);                      // [step][cout tile][lane]
    float *prm = reinterpret_cast<float *>(s2_smem + kS2WeightBytes);        // bias, gamma, beta
    const int lane = threadIdx.x & (kWave - 1), j = lane & 31, kh = lane >> 5;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave);
    uint16_t *out_tile = reinterpret_cast<uint16_t *>(prm + 3 * kS2Cout) + wave * 32 * kS2Pitch;

    {   // piece (step, tile, lane): 8 channels 16 (step % 3) + 8 (lane / 32) .. of tap step / 3, output channel 32 tile + lane % 32
        const uint16_t *w = reinterpret_cast<const uint16_t *>(p.w);
        for (int i = threadIdx.x; i < kS2Steps * kS2Mt * kWave; i += kS2Waves * kWave) {
            const int l = i % kWave, mt = i / kWave % kS2Mt, step = i / (kWave * kS2Mt);
            const int tap = step / kS2Chunks, c = step % kS2Chunks * 16 + 8 * (l / 32);
            const uint16_t *src = w + (mt * 32 + l % 32) * p.ws_o + c * p.ws_c + tap / 3 * p.ws_h + tap % 3 * p.ws_w;
            uint32_t e[8];
#pragma unroll
            for (int q = 0; q < 8; ++q) e[q] = src[q * p.ws_c];
            wl[i] = u32x4_t{e[0] | e[1] << 16, e[2] | e[3] << 16, e[4] | e[5] << 16, e[6] | e[7] << 16};
        }
        for (int i = threadIdx.x; i < kS2Cout; i += kS2Waves * kWave) {
            prm[i] = p.b ? to_f32(reinterpret_cast<const T *>(p.b)[i]) : 0.0f;
            prm[kS2Cout + i] = p.gamma ? to_f32(reinterpret_cast<const T *>(p.gamma)[i]) : 1.0f;
            prm[2 * kS2Cout + i] = p.beta ? to_f32(reinterpret_cast<const T *>(p.beta)[i]) : 0.0f;
        }
    }
    __syncthreads();

    const __amdgpu_buffer_rsrc_t x = __builtin_amdgcn_make_buffer_rsrc(const_cast<void *>(p.x), 0, p.x_bytes, 0x00020000);
    T *y = reinterpret_cast<T *>(p.y);
    // a workgroup's units are consecutive (they share input rows), and so are the workgroups of one XCD
    const int first = (int)xcd_contiguous_id(blockIdx.x, gridDim.x) * p.units_per_wg, last = min(p.n_units, first + p.units_per_wg);
    for (int unit = first + wave; unit < last; unit += kS2Waves) {
        int off[2], ih0[2], iw0[2];
#pragma unroll
        for (int q = 0; q < 2; ++q) {
            uint32_t b, r, oh, ow;
            divmod((uint32_t)min(unit * kS2Unit + 32 * q + j, p.n_pos - 1), p.by_map, b, r);     // (the last is repeated, not stored)
            divmod(r, p.by_row, oh, ow);
            ih0[q] = 2 * (int)oh - 1; iw0[q] = 2 * (int)ow - 1;
            off[q] = (((int)b * p.H + ih0[q]) * p.W + iw0[q]) * (2 * kS2Cin) + 16 * kh;
        }
        auto load = [&](int tap, u32x4_t (&v)[2][kS2Chunks]) {
            const int th = tap / 3, tw = tap % 3;
#pragma unroll
            for (int q = 0; q < 2; ++q) {
                const bool in = (uint32_t)(ih0[q] + th) < (uint32_t)p.H && (uint32_t)(iw0[q] + tw) < (uint32_t)p.W;
                const int at = in ? off[q] + (th * p.W + tw) * (2 * kS2Cin) : (int)0x80000000;       // out of the buffer: zeros
#pragma unroll
                for (int s = 0; s < kS2Chunks; ++s)
                    v[q][s] = __builtin_bit_cast(u32x4_t, __builtin_amdgcn_raw_buffer_load_b128(x, at, 32 * s, 0));
            }
        };
        floatx16_t acc[kS2Mt][2];
#pragma unroll
        for (int mt = 0; mt < kS2Mt; ++mt)
#pragma unroll
            for (int g = 0; g < 4; ++g) {
                const float4 bv = *reinterpret_cast<const float4 *>(prm + 32 * mt + 8 * g + 4 * kh);
                const float t[4] = {bv.x, bv.y, bv.z, bv.w};
#pragma unroll
                for (int e = 0; e < 4; ++e) acc[mt][0][4 * g + e] = acc[mt][1][4 * g + e] = t[e];
            }
        u32x4_t ring[2][2][kS2Chunks];
        load(0, ring[0]);
#pragma unroll
        for (int tap = 0; tap < 9; ++tap) {
            if (tap + 1 < 9) load(tap + 1, ring[(tap + 1) & 1]);
            __builtin_amdgcn_sched_barrier(0);
#pragma unroll
            for (int s = 0; s < kS2Chunks; ++s)
#pragma unroll
                for (int mt = 0; mt < kS2Mt; ++mt) {
                    const u32x4_t a = wl[((tap * kS2Chunks + s) * kS2Mt + mt) * kWave + lane];
#pragma unroll
                    for (int q = 0; q < 2; ++q) acc[mt][q] = mfma_32x32x16(T{}, a, ring[tap & 1][q][s], acc[mt][q]);
                }
            __builtin_amdgcn_sched_barrier(0);
        }
#pragma unroll
        for (int q = 0; q < 2; ++q) {
            // channel of value (mt, i): 32 mt + 8 (i / 4) + 4 kh + i % 4
            float sum = 0.0f;
#pragma unroll
            for (int mt = 0; mt < kS2Mt; ++mt)
#pragma unroll
                for (int i = 0; i < 16; i += 2) {
                    const uint32_t w2 = pack2_from_f32<T>(acc[mt][q][i], acc[mt][q][i + 1]);
                    acc[mt][q][i] = unpack_lo<T>(w2); acc[mt][q][i + 1] = unpack_hi<T>(w2);
                    sum += acc[mt][q][i] + acc[mt][q][i + 1];
                }
            sum += __shfl_xor(sum, 32);
            const float mean = sum * (1.0f / kS2Cout);
            float sq = 0.0f;
#pragma unroll
            for (int mt = 0; mt < kS2Mt; ++mt)
#pragma unroll
                for (int i = 0; i < 16; ++i) { const float d = acc[mt][q][i] - mean; sq = fmaf(d, d, sq); }
            sq += __shfl_xor(sq, 32);
            const float rstd = __builtin_amdgcn_rsqf(sq * (1.0f / kS2Cout) + p.eps);
#pragma unroll
            for (int mt = 0; mt < kS2Mt; ++mt)
#pragma unroll
                for (int g = 0; g < 4; ++g) {
                    const int ch = 32 * mt + 8 * g + 4 * kh;
                    const float4 gm = *reinterpret_cast<const float4 *>(prm + kS2Cout + ch);
                    const float4 bt = *reinterpret_cast<const float4 *>(prm + 2 * kS2Cout + ch);
                    const floatx16_t &v = acc[mt][q];
                    *reinterpret_cast<uint2 *>(out_tile + j * kS2Pitch + ch) = make_uint2(
                        pack2_from_f32<T>(fmaf((v[4 * g] - mean) * rstd, gm.x, bt.x), fmaf((v[4 * g + 1] - mean) * rstd, gm.y, bt.y)),
                        pack2_from_f32<T>(fmaf((v[4 * g + 2] - mean) * rstd, gm.z, bt.z), fmaf((v[4 * g + 3] - mean) * rstd, gm.w, bt.w)));
                }
            wave_lds_sync();
            const int pos0 = unit * kS2Unit + 32 * q;
#pragma unroll
            for (int i = 0; i < 32 * kS2Cout / 8 / kWave; ++i) {
                const int idx = i * kWave + lane, pos = idx / (kS2Cout / 8), c = idx % (kS2Cout / 8) * 8;
                if (pos0 + pos < p.n_pos)
                    *reinterpret_cast<uint4 *>(y + (size_t)(pos0 + pos) * kS2Cout + c) =
                        *reinterpret_cast<const uint4 *>(out_tile + pos * kS2Pitch + c);
            }
            wave_lds_sync();
        }
    }
}

template <typename T>
static int launch_stem2(Stem2Args a, hipStream_t stream) {
    const void *fn = reinterpret_cast<const void *>(&stem_conv2_ln_kernel<T>);
    if (hipFuncSetAttribute(fn, hipFuncAttributeMaxDynamicSharedMemorySize, (int)kS2Smem) != hipSuccess) {
        (void)hipGetLastError();
        return SS2D_ENOTSUP;
    }
    // a workgroup per CU (the weights leave no room for a second); few positions: a unit per workgroup, whatever its seven
    // other wavefronts do
    const int n_wg = a.n_units < 256 ? a.n_units : 256;
    a.units_per_wg = (a.n_units + n_wg - 1) / n_wg;
    hipLaunchKernelGGL(stem_conv2_ln_kernel<T>, dim3((uint32_t)((a.n_units + a.units_per_wg - 1) / a.units_per_wg)),
                       dim3(kS2Waves * kWave), kS2Smem, stream, a);
    return launch_status();
}

}  // namespace ss2d

extern "C" int ss2d_stem_conv2_ln(const void *x, const void *weight, const int64_t *weight_strides, const void *bias,
                                  const void *ln_weight, const void *ln_bias, float eps, void *y, int B, int H, int W, int Cin,
                                  int Cout, int dtype, void *stream) {
    using namespace ss2d;
    if (B < 0 || H < 0 || W < 0 || Cin <= 0 || Cout <= 0) return SS2D_EINVAL;
    if (dtype != SS2D_F32 && dtype != SS2D_BF16 && dtype != SS2D_F16) return SS2D_EINVAL;
    if (B == 0 || H == 0 || W == 0) return SS2D_OK;
    if (!x || !weight || !weight_strides || !y) return SS2D_EINVAL;
    if (dtype == SS2D_F32 || Cin != kS2Cin || Cout != kS2Cout) return SS2D_ENOTSUP;          // other shapes: the library operators
    const int Ho = (H - 1) / 2 + 1, Wo = (W - 1) / 2 + 1;
    const int64_t bytes = (int64_t)B * H * W * Cin * 2;
    // (offsets into the input are 31 bits; a row before the first one is the most they go below it)
    if (bytes > 0x7fff0000ll || (int64_t)2 * (W + 1) * Cin * 2 > 0x7fff0000ll - bytes) return SS2D_ENOTSUP;
    if ((reinterpret_cast<uintptr_t>(x) | reinterpret_cast<uintptr_t>(y)) & 15u) return SS2D_ENOTSUP;
    Stem2Args a;
    a.x = x; a.w = weight; a.b = bias; a.gamma = ln_weight; a.beta = ln_bias; a.y = y;
    a.H = H; a.W = W;
    a.n_pos = B * Ho * Wo;
    a.n_units = (a.n_pos + kS2Unit - 1) / kS2Unit;
    a.units_per_wg = 1;
    a.x_bytes = (int32_t)bytes;
    a.ws_o = weight_strides[0]; a.ws_c = weight_strides[1]; a.ws_h = weight_strides[2]; a.ws_w = weight_strides[3];
    a.eps = eps;
    a.by_map = make_fastdiv((uint32_t)(Ho * Wo));
    a.by_row = make_fastdiv((uint32_t)Wo);
    hipStream_t s = (hipStream_t)stream;
    return dtype == SS2D_BF16 ? launch_stem2<bf16_t>(a, s) : launch_stem2<f16_t>(a, s);
}
