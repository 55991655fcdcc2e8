// Products in single precision on the bf16 matrix cores, with what stands around them in a block's training step
// (classification/models/vmamba.py:1116-1131 the MLP, :648-650 and :662 the projections):
//     out[m][n] = sum_k A(m, k) B(n, k)       with a bias and a residual, or GELU, or GELU's derivative behind it.
// A is stored [M][K], or [K][M] ("by columns"), B [N][K] or [K][N]: x W^T, dy W and dy^T x without a transposed copy of anything.
//   * an fp32 value is the sum of three bf16 ones, each the rounded remainder of those before: 8 + 8 + 8 bits and two signs for 24.
//     A product is six of theirs -- h h, h m, m h, m m, h l, l h --, summed in the matrix cores' fp32 accumulators; what is left out is
//     below 2^-25 of each term, less than its rounding in fp32.  Six products at 16 times the fp32 rate: the ceiling is 2.5 times the
//     fp32 matrix cores'.
//   * h h and the other five have accumulators of their own, added at the end: the matrix cores drop what lies below the accumulator's last
//     bit, always downwards, and the five small ones would lose 2e-8 of the result to that at 384 terms -- nothing beside the rounding
//     of one output, but the sum of 12 544 of them (a bias gradient behind this one) came out 6e-6 off, 20 times the library's.
//   * a workgroup owns 128 x 128 or 128 x 64 outputs, its four wavefronts a quarter each, 32 terms a step: the next step's floats are on their way
//     while this one's are multiplied; they are split on the way into LDS, [row][term] in three planes whichever way they were
//     stored, the 16-byte pieces of a row in an order of its own, so that neither side of LDS meets itself in a bank.
//   * few outputs and a long sum (a weight gradient) are cut into shares of the terms, added by a second kernel in a fixed order.
//   * a third part of a value v lies down to 2^-24 v, and bf16 ends at 2^-126: values are multiplied by 2^24 on the way into their parts and the sums
//     by 2^-48 behind the last term, exactly, so that every fp32 value, the subnormal ones too, is the sum of its parts, and products of them do
//     not vanish that count in fp32.  (Without it a value of 2^-116 is off by 3e-6 of itself; 1 to 3 % of the time.)
//   * infinities and NaN, and values that round beyond bf16's largest or sums beyond fp32's (from 2^104 and 2^80 on), leave a NaN or an infinity in the
//     sums: a wavefront that finds one computes its outputs again on the fp32 matrix cores, from memory.
// 12 544 x 1536 x 384: 146 us as the library's product (101 TFLOP/s), 104 here (142); 384 x 1536 outputs over 12 544 positions, both by columns,
// 142 -> 91.  What bounds it is the matrix cores' rate under load, 1.2 PFLOP/s in bf16 on this card, a sixth of it here: 200; then the
// split's instructions between them.  One accumulator for all six, three workgroups per CU: 93 where two took 108, and the bias above.  Against 64 bits the error
// is 1.1e-7 (library 3.5e-7), of the gradient 1.6e-7 (2.0e-6).  Two fp16 parts and three products would be twice as fast and hold less
// than fp32's range.
#include "normal_cdf.h"

namespace ss2d {

typedef float pf4_t __attribute__((ext_vector_type(4)));

constexpr int kPfTile = 128, kPfDepth = 32;                          // rows of A (and of B: or 64) per workgroup, terms per step

struct ProductArgs {
    const float *a, *b, *bias, *other;                               // other: residual, or the pre-activation of kPfGeluGrad
    float *out, *out2;                                               // out2: GELU of out (kPfGelu)
    int64_t M, K, share;                                             // share: terms per workgroup, a multiple of kPfDepth
    int32_t N, tiles_n, tile_n;
    uint32_t tiles, total;
};

enum { kPfPlain = 0, kPfGelu = 1, kPfGeluGrad = 2 };

constexpr float kPfScale = 0x1p24f, kPfUnscale = 0x1p-48f;           // of a value, of a sum of products

// Two floats times kPfScale as three packed bf16 pairs: rounded, the rounded remainder, the remainder of both (exact for what 24 bits hold)
__device__ __forceinline__ void split3(float a, float b, uint32_t &h, uint32_t &m, uint32_t &l) {
    a *= kPfScale; b *= kPfScale;
    h = pack2_from_f32<bf16_t>(a, b);
    a -= unpack_lo<bf16_t>(h); b -= unpack_hi<bf16_t>(h);
    m = pack2_from_f32<bf16_t>(a, b);
    l = pack2_from_f32<bf16_t>(a - unpack_lo<bf16_t>(m), b - unpack_hi<bf16_t>(m));
}

// LDS offset of terms 8 g .. 8 g + 7 of a row: 64 bytes a row, the four 16-byte pieces in an order that differs from row to row, so that
// eight lanes with a row each read all banks once.  A tile that arrives by columns is written four rows apart by lanes side by side: its rows
// are transposed in blocks of 4 x 4, so that those are neighbours.
template <bool kByCols> __device__ __forceinline__ int pf_at(int row, int g) {
    if constexpr (kByCols) {
        const int at = (row & ~15) | (row & 3) << 2 | (row >> 2 & 3);
        return at * kPfDepth + 8 * (g ^ (((at >> 2) + (at >> 4)) & 3));
    } else {
        return row * kPfDepth + 8 * (g ^ (row >> 2 & 3));
    }
}

// One operand's kRows x 32 terms: where a thread loads its kLoads x 4 floats, and where it leaves them.
template <bool kByCols, int kRows> struct PfTile {
    static constexpr int kLoads = kRows / 32, kPlane = kRows * kPfDepth;
    static constexpr int kQuads = kRows / 4;                         // by columns: threads side by side, kLoads terms each
    const float *src;                                                // of step 0
    int64_t ld, rows;                                                // by columns: distance of the terms
    int t;
    int64_t row_off[kLoads];
    __device__ __forceinline__ void init(const float *base, int64_t first, int64_t n_rows, int64_t terms, int thread) {
        t = thread; rows = n_rows;
        if constexpr (kByCols) {
            ld = n_rows;
            const int64_t c = first + 4 * (t % kQuads);
            src = base + (c + 4 <= n_rows ? c : n_rows - 4);         // (columns past the last repeat it, nobody stores what comes of them)
        } else {
            ld = terms;
            src = base + 4 * (t & 7);
#pragma unroll
            for (int i = 0; i < kLoads; ++i) {
                const int64_t r = first + (t >> 3) + 32 * i;
                row_off[i] = (r < n_rows ? r : n_rows - 1) * terms;
            }
        }
    }
    // terms from k on, end the last one's successor (k < end; both multiples of 4 from the start of a row); 0 past it
    __device__ __forceinline__ void load(pf4_t (&v)[kLoads], int64_t k, int64_t end) const {
        if constexpr (kByCols) {
            const int64_t at = k + kLoads * (t / kQuads);
#pragma unroll
            for (int i = 0; i < kLoads; ++i) v[i] = *reinterpret_cast<const pf4_t *>(src + (at + i < end ? at + i : end - 1) * ld);
            if (k + kPfDepth > end) {                                // uniform
#pragma unroll
                for (int i = 0; i < kLoads; ++i)
                    if (at + i >= end) v[i] = pf4_t{0, 0, 0, 0};
            }
        } else {
            const bool in = k + 4 * (t & 7) < end;
            const int64_t at = in ? k : -4 * (t & 7);
#pragma unroll
            for (int i = 0; i < kLoads; ++i) v[i] = *reinterpret_cast<const pf4_t *>(src + row_off[i] + at);
            if (k + kPfDepth > end) {
#pragma unroll
                for (int i = 0; i < kLoads; ++i)
                    if (!in) v[i] = pf4_t{0, 0, 0, 0};
            }
        }
    }
    __device__ __forceinline__ void park(const pf4_t (&v)[kLoads], uint16_t *planes) const {
        if constexpr (kByCols) {                                     // kLoads terms of row 4 (t % kQuads) + i
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                const int term = kLoads * (t / kQuads);
                uint32_t h[kLoads / 2], m[kLoads / 2], l[kLoads / 2];
#pragma unroll
                for (int q = 0; q < kLoads / 2; ++q) split3(v[2 * q][i], v[2 * q + 1][i], h[q], m[q], l[q]);
                store<kLoads / 2>(planes + pf_at<true>(4 * (t % kQuads) + i, term / 8) + term % 8, h, m, l);
            }
        } else {                                                     // four terms of row t / 8 + 32 i
#pragma unroll
            for (int i = 0; i < kLoads; ++i) {
                uint32_t h[2], m[2], l[2];
                split3(v[i][0], v[i][1], h[0], m[0], l[0]);
                split3(v[i][2], v[i][3], h[1], m[1], l[1]);
                store<2>(planes + pf_at<false>((t >> 3) + 32 * i, t >> 1 & 3) + 4 * (t & 1), h, m, l);
            }
        }
    }
    template <int kDwords>
    static __device__ __forceinline__ void store(uint16_t *at, const uint32_t (&h)[kDwords], const uint32_t (&m)[kDwords], const uint32_t (&l)[kDwords]) {
        if constexpr (kDwords == 2) {
            *reinterpret_cast<uint2 *>(at) = make_uint2(h[0], h[1]);
            *reinterpret_cast<uint2 *>(at + kPlane) = make_uint2(m[0], m[1]);
            *reinterpret_cast<uint2 *>(at + 2 * kPlane) = make_uint2(l[0], l[1]);
        } else {
            *reinterpret_cast<uint32_t *>(at) = h[0];
            *reinterpret_cast<uint32_t *>(at + kPlane) = m[0];
            *reinterpret_cast<uint32_t *>(at + 2 * kPlane) = l[0];
        }
    }
};

// 12 544 x 1536 x 384, us: 129 with GELU and 124 with its derivative, 103 without and without their second tensor of 77 MB.  One fit of degree 9 took 125 and
// 120 and lost accuracy (normal_cdf.h); erff, two branches of some thirty instructions each, ten more than that.
__device__ __forceinline__ float gelu_f32(float x) {
    float e;
    return x * normal_cdf(x, e);
}
__device__ __forceinline__ float gelu_grad_f32(float x) {
    float e;
    const float cdf = normal_cdf(x, e);
    return fmaf(x * 0.39894228040143268f, e, cdf);
}

// What stands behind the sum: outputs n .. n + 3 of a row, at `at`
template <int kMode>
__device__ __forceinline__ void finish(const ProductArgs &p, float *out, pf4_t v, int64_t at, int n) {
    if (p.bias) v += *reinterpret_cast<const pf4_t *>(p.bias + n);
    if constexpr (kMode == kPfGeluGrad) {
        const pf4_t x = *reinterpret_cast<const pf4_t *>(p.other + at);
#pragma unroll
        for (int t = 0; t < 4; ++t) v[t] *= gelu_grad_f32(x[t]);
    } else if (p.other) {
        v += *reinterpret_cast<const pf4_t *>(p.other + at);
    }
    *reinterpret_cast<pf4_t *>(out + at) = v;
    if constexpr (kMode == kPfGelu) {
#pragma unroll
        for (int t = 0; t < 4; ++t) v[t] = gelu_f32(v[t]);
        *reinterpret_cast<pf4_t *>(p.out2 + at) = v;
    }
}

// kTileN: rows of B per workgroup, 128 or 64
template <bool kACols, bool kBCols, int kTileN, int kMode>
__global__ __launch_bounds__(kBlock, kTileN == 128 ? 2 : 3) void product_f32_kernel(const ProductArgs p) {
    using TileA = PfTile<kACols, kPfTile>;
    using TileB = PfTile<kBCols, kTileN>;
    constexpr int kE = kTileN / 64;                                   // 32 x 32 tiles of a wavefront along B
    __shared__ __align__(16) uint16_t lds[3 * (TileA::kPlane + TileB::kPlane)];
    uint16_t *const sa = lds, *const sb = lds + 3 * TileA::kPlane;
    const int lane = threadIdx.x & (kWave - 1), j = lane & 31, kh = lane >> 5;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave);
    const uint32_t id = xcd_contiguous_id(blockIdx.x, p.total);       // neighbours share rows of A, in one L2
    const uint32_t share = id / p.tiles, tile = id - share * p.tiles;
    const int64_t m0 = (int64_t)(tile / (uint32_t)p.tiles_n) * kPfTile;
    const int n0 = (int)(tile % (uint32_t)p.tiles_n) * kTileN;
    const int64_t k0 = share * p.share, k1 = k0 + p.share < p.K ? k0 + p.share : p.K;
    TileA ta;
    TileB tb;
    ta.init(p.a, m0, p.M, p.K, threadIdx.x);
    tb.init(p.b, n0, p.N, p.K, threadIdx.x);
    const int wm = (wave & 1) * 64, wn = (wave >> 1) * (kTileN / 2);

    floatx16_t acc[2][kE], low[2][kE];                                            // [rows of A][rows of B]
#pragma unroll
    for (int i = 0; i < 2; ++i)
#pragma unroll
        for (int q = 0; q < kE; ++q)
#pragma unroll
            for (int v = 0; v < 16; ++v) acc[i][q][v] = low[i][q][v] = 0.0f;
    pf4_t va[TileA::kLoads], vb[TileB::kLoads];
    ta.load(va, k0, k1);
    tb.load(vb, k0, k1);
    for (int64_t k = k0; k < k1; k += kPfDepth) {
        ta.park(va, sa);
        tb.park(vb, sb);
        __syncthreads();
        if (k + kPfDepth < k1) {
            ta.load(va, k + kPfDepth, k1);
            tb.load(vb, k + kPfDepth, k1);
        }
#pragma unroll
        for (int s = 0; s < 2; ++s) {
            u32x4_t fa[2][3], fb[kE][3];
#pragma unroll
            for (int q = 0; q < 3; ++q) {
#pragma unroll
                for (int i = 0; i < 2; ++i) fa[i][q] = *reinterpret_cast<const u32x4_t *>(sa + q * TileA::kPlane + pf_at<kACols>(wm + 32 * i + j, 2 * s + kh));
#pragma unroll
                for (int e = 0; e < kE; ++e) fb[e][q] = *reinterpret_cast<const u32x4_t *>(sb + q * TileB::kPlane + pf_at<kBCols>(wn + 32 * e + j, 2 * s + kh));
            }
            // (consecutive products go to different accumulators)
            constexpr int kPa[5] = {0, 2, 1, 0, 1}, kPb[5] = {2, 0, 1, 1, 0};
#pragma unroll
            for (int q = 0; q < 6; ++q)
#pragma unroll
                for (int i = 0; i < 2; ++i)
#pragma unroll
                    for (int e = 0; e < kE; ++e) {
                        if (q < 5) low[i][e] = mfma_32x32x16(bf16_t{}, fb[e][kPb[q]], fa[i][kPa[q]], low[i][e]);
                        else acc[i][e] = mfma_32x32x16(bf16_t{}, fb[e][0], fa[i][0], acc[i][e]);
                    }
        }
        __syncthreads();
    }

    // a lane holds, of row m = m0 + wm + 32 i + j, outputs n0 + wn + 32 e + 8 g + 4 kh + t in accumulator 4 g + t
    bool odd = false;
#pragma unroll
    for (int i = 0; i < 2; ++i)
#pragma unroll
        for (int e = 0; e < kE; ++e)
#pragma unroll
            for (int v = 0; v < 16; ++v) {
                acc[i][e][v] += low[i][e][v];
                odd |= !(fabsf(acc[i][e][v]) <= 3.4028235e38f);
                acc[i][e][v] *= kPfUnscale;
            }
    if (__any(odd)) {
        int64_t ra[2], rb[kE];
#pragma unroll
        for (int i = 0; i < 2; ++i) {
            ra[i] = min(m0 + wm + 32 * i + j, p.M - 1);
#pragma unroll
            for (int e = 0; e < kE; ++e)
#pragma unroll
                for (int v = 0; v < 16; ++v) acc[i][e][v] = 0.0f;
        }
#pragma unroll
        for (int e = 0; e < kE; ++e) rb[e] = min(n0 + wn + 32 * e + j, p.N - 1);
        for (int64_t k = k0; k < k1; k += 2) {
            const bool in = k + kh < k1;
            const int64_t at = in ? k + kh : k;
            float xa[2], xb[kE];
#pragma unroll
            for (int i = 0; i < 2; ++i) xa[i] = in ? p.a[kACols ? at * p.M + ra[i] : ra[i] * p.K + at] : 0.0f;
#pragma unroll
            for (int e = 0; e < kE; ++e) xb[e] = in ? p.b[kBCols ? at * p.N + rb[e] : rb[e] * p.K + at] : 0.0f;
#pragma unroll
            for (int i = 0; i < 2; ++i)
#pragma unroll
                for (int e = 0; e < kE; ++e) acc[i][e] = __builtin_amdgcn_mfma_f32_32x32x2f32(xb[e], xa[i], acc[i][e], 0, 0, 0);
        }
    }

    float *const out = p.out + (int64_t)share * p.M * p.N;
#pragma unroll
    for (int i = 0; i < 2; ++i) {
        const int64_t m = m0 + wm + 32 * i + j;
        if (m >= p.M) continue;
#pragma unroll
        for (int e = 0; e < kE; ++e)
#pragma unroll
            for (int g = 0; g < 4; ++g) {
                const int n = n0 + wn + 32 * e + 8 * g + 4 * kh;
                if (n >= p.N) continue;                              // (N is a multiple of 4)
                pf4_t v = {acc[i][e][4 * g], acc[i][e][4 * g + 1], acc[i][e][4 * g + 2], acc[i][e][4 * g + 3]};
                finish<kMode>(p, out, v, m * p.N + n, n);
            }
    }
}

template <int kMode>
__global__ __launch_bounds__(kBlock) void product_f32_sum_kernel(const ProductArgs p, const float *partial, int shares) {
    const int64_t at = 4 * ((int64_t)blockIdx.x * kBlock + threadIdx.x);
    if (at >= p.M * p.N) return;
    pf4_t t = *reinterpret_cast<const pf4_t *>(partial + at);
    for (int s = 1; s < shares; ++s) t += *reinterpret_cast<const pf4_t *>(partial + s * p.M * p.N + at);
    finish<kMode>(p, p.out, t, at, (int)(at % p.N));
}

// How a product is cut.  Tiles of 128 x 128, two workgroups per CU, where there are several rounds of them and for gradients, whose long sum
// is cut into shares until they fill the chip; else 128 x 64, three per CU.  us, 128 x 128 / 128 x 64, over 12 544 positions: 1536 x 384
// 104 / 110, 384 x 1536 (two shares of the larger tiles) 126 / 113, 384 x 384 37 / 33; gradients: 1536 x 384 91 / 109; up to 384 x 384 outputs the smaller tiles
// are ahead, 384 x 384 43 / 42, 256 x 256 35 / 32, 96 x 96 over 200 704 158 / 137 (a block's own of that size are ss2d_linear_dw_f32's).  Shares of
// eight steps at least: fewer terms and the second kernel costs more than the workgroups give.
static int product_plan(int64_t M, int N, int64_t K, bool a_cols, bool b_cols, ProductArgs &a, int64_t &shares) {
    if (M <= 0 || N <= 0 || K <= 0 || N % 4 != 0 || (a_cols ? M % 4 != 0 : K % 4 != 0) || (!b_cols && K % 4 != 0)) return SS2D_ENOTSUP;
    const int64_t tiles_m = (M + kPfTile - 1) / kPfTile, most = K / (8 * kPfDepth);
    a.tile_n = N > 64 && ((a_cols && b_cols) || tiles_m * ((N + 127) / 128) >= 768) ? 128 : 64;
    const int64_t tiles_n = (N + a.tile_n - 1) / a.tile_n, tiles = tiles_m * tiles_n;
    if (tiles > 0x3fffffff) return SS2D_ENOTSUP;
    shares = (a.tile_n == 128 ? 2 : 3) * 256 / tiles;
    if (shares > most) shares = most;
    if (shares < 1) shares = 1;
    a.share = ((K + shares - 1) / shares + kPfDepth - 1) / kPfDepth * kPfDepth;
    shares = (K + a.share - 1) / a.share;
    a.M = M; a.N = N; a.K = K; a.tiles_n = (int)tiles_n; a.tiles = (uint32_t)tiles; a.total = (uint32_t)(tiles * shares);
    return SS2D_OK;
}

template <bool kACols, bool kBCols, int kTileN>
static void launch_product_tiles(const ProductArgs &a, int mode, hipStream_t s) {
    const dim3 grid(a.total), block(kBlock);
    if (mode == kPfGelu) hipLaunchKernelGGL((product_f32_kernel<kACols, kBCols, kTileN, kPfGelu>), grid, block, 0, s, a);
    else if (mode == kPfGeluGrad) hipLaunchKernelGGL((product_f32_kernel<kACols, kBCols, kTileN, kPfGeluGrad>), grid, block, 0, s, a);
    else hipLaunchKernelGGL((product_f32_kernel<kACols, kBCols, kTileN, kPfPlain>), grid, block, 0, s, a);
}

template <bool kACols, bool kBCols> static void launch_product(const ProductArgs &a, int mode, hipStream_t s) {
    if (a.tile_n == 128) launch_product_tiles<kACols, kBCols, 128>(a, mode, s);
    else launch_product_tiles<kACols, kBCols, 64>(a, mode, s);
}

}  // namespace ss2d

extern "C" int64_t ss2d_product_f32_workspace_bytes(int64_t M, int N, int64_t K, int a_by_columns, int b_by_columns) {
    using namespace ss2d;
    ProductArgs a;
    int64_t shares;
    if (M < 0 || N < 0 || K < 0) return SS2D_EINVAL;
    const int rc = product_plan(M, N, K, a_by_columns != 0, b_by_columns != 0, a, shares);
    return rc != SS2D_OK ? rc : shares > 1 ? shares * M * N * 4 : 0;
}

extern "C" int ss2d_product_f32(const float *a_, const float *b, const float *bias, const float *other, float *out, float *out2, int64_t M, int N,
                                int64_t K, int a_by_columns, int b_by_columns, int mode, void *workspace, int64_t workspace_bytes, void *stream) {
    using namespace ss2d;
    if (M < 0 || N < 0 || K < 0 || mode < kPfPlain || mode > kPfGeluGrad) return SS2D_EINVAL;
    ProductArgs a;
    int64_t shares;
    const int rc = product_plan(M, N, K, a_by_columns != 0, b_by_columns != 0, a, shares);
    if (rc != SS2D_OK) return rc;
    if (!a_ || !b || !out || (mode == kPfGelu) != (out2 != nullptr) || (mode == kPfGeluGrad && !other) || (mode == kPfGelu && other)) return SS2D_EINVAL;
    const void *ptrs[] = {a_, b, bias, other, out, out2, workspace};
    for (const void *q : ptrs)
        if (reinterpret_cast<uintptr_t>(q) % 16 != 0) return SS2D_ENOTSUP;
    if (shares > 1 && !workspace) return SS2D_EINVAL;
    if (shares > 1 && workspace_bytes < shares * M * N * 4) return SS2D_ENOMEM;
    a.a = a_; a.b = b;
    hipStream_t s = (hipStream_t)stream;
    const bool split = shares > 1;
    a.bias = split ? nullptr : bias; a.other = split ? nullptr : other; a.out = split ? (float *)workspace : out; a.out2 = split ? nullptr : out2;
    const int first = split ? kPfPlain : mode;
    if (a_by_columns) b_by_columns ? launch_product<true, true>(a, first, s) : launch_product<true, false>(a, first, s);
    else b_by_columns ? launch_product<false, true>(a, first, s) : launch_product<false, false>(a, first, s);
    if (split) {
        a.bias = bias; a.other = other; a.out = out; a.out2 = out2;
        const dim3 grid((uint32_t)((M * N / 4 + kBlock - 1) / kBlock)), block(kBlock);
        const float *partial = (const float *)workspace;
        if (mode == kPfGelu) hipLaunchKernelGGL((product_f32_sum_kernel<kPfGelu>), grid, block, 0, s, a, partial, (int)shares);
        else if (mode == kPfGeluGrad) hipLaunchKernelGGL((product_f32_sum_kernel<kPfGeluGrad>), grid, block, 0, s, a, partial, (int)shares);
        else hipLaunchKernelGGL((product_f32_sum_kernel<kPfPlain>), grid, block, 0, s, a, partial, (int)shares);
    }
    return launch_status();
}
