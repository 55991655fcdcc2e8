// x_proj and the core of a few short maps, one state per channel: forward_core (classification/models/vmamba.py:603-646) where a
// call is the latency of its launches.  One image of 768 x 7 x 7 took 31 us in a graph for 75 KB of input, as x_proj 10, dt_proj 9,
// the core 5 and out_norm 7: grids of 4 to 192 workgroups, each a chain of memory round trips.  Here
//   * x_proj (ss2d_x_proj_few) gives a workgroup 16 output rows of 64 positions and its eight wavefronts an eighth of the channels
//     each, whose loads are all in flight together; the partial sums meet in LDS in the wavefronts' order.  The result is left
//     position-major and in the map's own order, (B, L, 4, few_row(R)) -- a direction's ranks side by side, then B and C --, so that
//     nothing is put into scan order on the way out;
//   * the core (ss2d_core_few) takes dt_proj in: a wavefront owns one channel (two on maps of up to 64 positions) and its groups of 16
//     (8) lanes are that channel's four directions, each lane walking up to 17 consecutive scan positions, whose rank rows it reads from
//     the LDS copy all eight wavefronts share.  The step is the fp32 sum over the ranks, two to an instruction, never rounded to 16
//     bits and never in memory.  Outputs meet in LDS planes, one per direction, and leave as (y0 + y2) + (y1 + y3) + (D0 + .. + D3) x.
// What bounds such a call is a trip to memory per launch and the instructions, which every launch fetches anew (see core_few_kernel):
// the three launches of one image of 768 x 7 x 7 now take 6.1, 6.7 and 6.5 us (17.9 in a graph).  Whole calls: few_pays.
#include "scan_common.h"

namespace ss2d {

constexpr int kFewWaves = 8;                 // wavefronts of an x_proj workgroup: shares of the channels
constexpr int kFewRing = 3;                  // steps of 32 channels a wavefront has in flight
constexpr int kFewThreads = 512;              // of a core workgroup: 8 channels, or 16 on maps of up to 64 positions
constexpr int kFewMaxL = 256, kFewMaxRank = 48;
constexpr int kFewMaxLds = 157 * 1024;      // (beside the 2 KB of the states that enter the lanes)

// Elements of a rank row.  16-bit: the ranks' dwords, a zero in the last one's high half if they are odd in number, then the dword of B
// and C; fp32: the ranks, B, C.  A multiple of 8, so that rows start on 16 bytes.
template <typename T> struct FewRow;
template <> struct FewRow<float> {
    static __host__ __device__ constexpr int b_at(int R) { return R; }
};
template <> struct FewRow<bf16_t> {
    static __host__ __device__ constexpr int b_at(int R) { return (R + 1) & ~1; }
};
template <> struct FewRow<f16_t> : FewRow<bf16_t> {};
// (of a position: 16 bytes more than its four rows, so that consecutive positions start in other LDS banks)
static __host__ __device__ constexpr int few_row(int R, bool f32) { return ((f32 ? R : (R + 1) & ~1) + 2 + 7) & ~7; }

static int few_pitch(int R, bool f32) { return 4 * few_row(R, f32) + (f32 ? 4 : 8); }

struct FewProjArgs {
    const void *x, *W;
    void *out;
    int32_t B, D, R, L, row, pitch, m_tiles, groups;
};

typedef float f32x4_t __attribute__((ext_vector_type(4)));

template <typename T> struct FewStep {       // 8 channels of four positions, and of one weight row
    uint2 x[8];
    u32x4_t w;
};
template <> struct FewStep<float> {
    f32x4_t x[8];
    f32x4_t w[2];
};

template <typename T>
__global__ __launch_bounds__(kFewWaves * kWave) void x_proj_few_kernel(const FewProjArgs p) {
    __shared__ __align__(16) f32x4_t part[kFewWaves][4][kWave];
    constexpr bool kF32 = sizeof(T) == 4;
    const int lane = threadIdx.x & (kWave - 1), col = lane & 15, kg = lane >> 4;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave);
    // tiles of one image side by side: they share its map, and W's rows come back image after image
    const int tile = (int)(blockIdx.x % (uint32_t)p.m_tiles);
    const int group = (int)(blockIdx.x / (uint32_t)p.m_tiles % (uint32_t)p.groups);
    const int64_t b = blockIdx.x / (uint32_t)(p.m_tiles * p.groups);
    // the lane's weight row: output row `slot` of direction slot / row; the rows between (odd ranks, the end) repeat one, and are cleared below
    const int slot = tile * 16 + col, dir = slot / p.row, in_row = slot % p.row, b_at = FewRow<T>::b_at(p.R);
    const int w_row = dir * (p.R + 2) + (in_row < p.R ? in_row : in_row >= b_at && in_row < b_at + 2 ? p.R + in_row - b_at : 0);
    const T *W = reinterpret_cast<const T *>(p.W) + (int64_t)w_row * p.D + 8 * kg;
    // four positions per lane; past the end the map's last four (their sums are those of the lanes that own them)
    const int at = min(group * kWave + 4 * col, p.L - 4);
    const T *x = reinterpret_cast<const T *>(p.x) + (b * p.D + 8 * kg) * p.L + at;
    const int steps = (p.D + 31) / 32, per = (steps + kFewWaves - 1) / kFewWaves, s0 = wave * per, s1 = min(steps, s0 + per);

    f32x4_t acc[4];
#pragma unroll
    for (int s = 0; s < 4; ++s) acc[s] = f32x4_t{0, 0, 0, 0};
    for (int first = s0; first < s1; first += kFewRing) {
        FewStep<T> ring[kFewRing];
#pragma unroll
        for (int q = 0; q < kFewRing; ++q) {
            // past the share the last step again, past D (a multiple of 8) the first channels: read, not used
            const int step = min(first + q, s1 - 1), off = step * 32 + 8 * kg < p.D ? step * 32 : -8 * kg;
#pragma unroll
            for (int i = 0; i < 8; ++i) __builtin_memcpy(&ring[q].x[i], x + (int64_t)(off + i) * p.L, 4 * sizeof(T));     // any element boundary
            if constexpr (kF32) {
                ring[q].w[0] = *reinterpret_cast<const f32x4_t *>(W + off);
                ring[q].w[1] = *reinterpret_cast<const f32x4_t *>(W + off + 4);
            } else {
                ring[q].w = *reinterpret_cast<const u32x4_t *>(W + off);
            }
        }
        __builtin_amdgcn_sched_barrier(0);                           // all of them in flight before the first is waited for
#pragma unroll
        for (int q = 0; q < kFewRing; ++q) {
            if (first + q >= s1) break;                              // uniform
            FewStep<T> &r = ring[q];
            const bool in = (first + q) * 32 + 8 * kg < p.D;
            if constexpr (kF32) {
                if (!in) {
#pragma unroll
                    for (int i = 0; i < 8; ++i) r.x[i] = f32x4_t{0, 0, 0, 0};
                    r.w[0] = r.w[1] = f32x4_t{0, 0, 0, 0};
                }
#pragma unroll
                for (int i = 0; i < 8; ++i)
#pragma unroll
                    for (int s = 0; s < 4; ++s) acc[s] = __builtin_amdgcn_mfma_f32_16x16x4f32(r.w[i / 4][i % 4], r.x[i][s], acc[s], 0, 0, 0);
            } else {
                if (!in) {
#pragma unroll
                    for (int i = 0; i < 8; ++i) r.x[i] = make_uint2(0u, 0u);
                    r.w = u32x4_t{0u, 0u, 0u, 0u};
                }
#pragma unroll
                for (int s = 0; s < 4; ++s) {
                    u32x4_t bf;
#pragma unroll
                    for (int m = 0; m < 4; ++m)
                        bf[m] = __builtin_amdgcn_perm(s < 2 ? r.x[2 * m + 1].x : r.x[2 * m + 1].y, s < 2 ? r.x[2 * m].x : r.x[2 * m].y,
                                                      s % 2 ? 0x07060302u : 0x05040100u);
                    acc[s] = mfma_16x16x32(T{}, r.w, bf, acc[s]);
                }
            }
        }
    }
#pragma unroll
    for (int s = 0; s < 4; ++s) part[wave][s][lane] = acc[s];
    __syncthreads();
    // rows 4 kg .. +3 of position at + s, summed by one lane each
    if (wave >= 4) return;
    f32x4_t sum = part[0][wave][lane];
#pragma unroll
    for (int v = 1; v < kFewWaves; ++v) sum += part[v][wave][lane];
    if (group * kWave + 4 * col >= p.L) return;
    const int out_slot = tile * 16 + 4 * kg, out_in = out_slot % p.row;
#pragma unroll
    for (int e = 0; e < 4; ++e) {
        const int r = out_in + e;
        if (r >= p.R && (r < b_at || r >= b_at + 2)) sum[e] = 0.0f;
    }
    T *dst = reinterpret_cast<T *>(p.out) + (b * p.L + at + wave) * p.pitch + out_slot;
    if constexpr (kF32) *reinterpret_cast<f32x4_t *>(dst) = sum;
    else *reinterpret_cast<uint2 *>(dst) = make_uint2(pack2_from_f32<T>(sum[0], sum[1]), pack2_from_f32<T>(sum[2], sum[3]));
}

struct FewCoreArgs {
    const void *x, *rows, *W;
    const float *A, *Dv, *bias;
    float *y;
    int32_t B, D, H, Wd, L, R, row, pitch, rows_bytes, chan_sets;    // pitch: elements of a position's rank rows; rows_bytes: of an image's
    int32_t per_lane;                                                // scan positions of a lane
    uint32_t per_inv;                                                // t / per_lane = t * per_inv >> 16 for t < 256
    FastDiv div_h, div_w;
};

// ranks 2 r and 2 r + 1 (16-bit), or rank r
__device__ __forceinline__ float few_dot(bf16_t, uint32_t a, uint32_t b, float sum) {
    typedef __bf16 bf16x2_t __attribute__((ext_vector_type(2)));
    return __builtin_amdgcn_fdot2_f32_bf16(__builtin_bit_cast(bf16x2_t, a), __builtin_bit_cast(bf16x2_t, b), sum, false);
}
__device__ __forceinline__ float few_dot(f16_t, uint32_t a, uint32_t b, float sum) {
    typedef _Float16 halfx2_t __attribute__((ext_vector_type(2)));
    return __builtin_amdgcn_fdot2(__builtin_bit_cast(halfx2_t, a), __builtin_bit_cast(halfx2_t, b), sum, false);
}
__device__ __forceinline__ float few_dot(float, uint32_t a, uint32_t b, float sum) { return fmaf(bits_to_f32(a), bits_to_f32(b), sum); }

// kG lanes per direction (8 or 16), kQ 16-byte pieces of ranks.  What such a call waits for is its instructions, fetched from memory by
// every launch anew: the same kernel with its items unrolled was 10 KB and 12.5 us for one image of 768 x 7 x 7 (384 x 14 x 14: 13.4), in
// loops it is 2 KB.
template <typename T, int kG, int kQ>
__global__ __launch_bounds__(kFewThreads) void core_few_kernel(const FewCoreArgs p) {
    extern __shared__ __align__(16) uint8_t few_smem[];
    constexpr bool kF32 = sizeof(T) == 4;
    constexpr int kPerDword = kF32 ? 1 : 2, kPiece = 16 / (int)sizeof(T);
    constexpr int kCh = kWave / (4 * kG), kChans = kCh * (kFewThreads / kWave);  // channels per wavefront and workgroup
    const int lane = threadIdx.x & (kWave - 1);
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave);
    const int L = p.L, per = p.per_lane;
    float2 *s_y = reinterpret_cast<float2 *>(few_smem);                         // [kChans][4][L], in scan order
    T *s_rows = reinterpret_cast<T *>(s_y + (size_t)kChans * 4 * L);            // [L][pitch]
    T *s_x = reinterpret_cast<T *>(reinterpret_cast<uint8_t *>(s_rows) + p.rows_bytes);      // [kChans][L]
    const int64_t b = blockIdx.x / (uint32_t)p.chan_sets;
    const int d0 = (int)(blockIdx.x % (uint32_t)p.chan_sets) * kChans;

    // ---- all of a workgroup's loads, one after the other before the first is waited for: the image's rank rows straight into LDS, its
    // channels of the map, the weights of the lane's direction
    const uint8_t *rows = reinterpret_cast<const uint8_t *>(p.rows) + b * p.rows_bytes;
    for (int at = wave * (16 * kWave); at < p.rows_bytes; at += 16 * kFewThreads)
        if (at + 16 * lane < p.rows_bytes) load_to_lds_16(rows + at + 16 * lane, reinterpret_cast<uint8_t *>(s_rows) + at);
    const int i = lane % kG, dir = lane / kG % 4, chan = wave * kCh + lane / (4 * kG);
    const int kd = dir * p.D + min(d0 + chan, p.D - 1);
    const int nd = (p.R + kPerDword - 1) / kPerDword;                           // dwords of ranks
    uint32_t w[4 * kQ];
    {
        const T *Wr = reinterpret_cast<const T *>(p.W) + (int64_t)kd * p.R;
#pragma unroll
        for (int q = 0; q + 1 < kQ; ++q) __builtin_memcpy(&w[4 * q], Wr + q * kPiece, 16);      // any element boundary
#pragma unroll
        for (int r = 4 * kQ - 4; r < 4 * kQ; ++r) {
            w[r] = 0u;
            if (kPerDword * (r + 1) <= p.R) __builtin_memcpy(&w[r], Wr + kPerDword * r, 4);      // uniform
            else if (kPerDword * r < p.R) w[r] = reinterpret_cast<const uint16_t *>(Wr)[kPerDword * r];
        }
    }
    const float A = p.A[kd] * kLog2e, bias = p.bias ? p.bias[kd] : 0.0f, skip = p.Dv ? p.Dv[kd] : 0.0f;
    const int n_x = min(kChans, p.D - d0) * L;
    const T *map = reinterpret_cast<const T *>(p.x) + (b * p.D + d0) * L;
    constexpr int kFly = 4;
    for (int first = threadIdx.x; first < n_x; first += kFly * kFewThreads) {
        T v[kFly];
#pragma unroll
        for (int q = 0; q < kFly; ++q) v[q] = map[min(first + q * kFewThreads, n_x - 1)];
#pragma unroll
        for (int q = 0; q < kFly; ++q)
            if (first + q * kFewThreads < n_x) s_x[first + q * kFewThreads] = v[q];
    }
    wait_loads_to_lds();
    __syncthreads();

    // ---- the lane's scan positions t = t0 .. t1 - 1, as positions of the map; a lane without any is the pair (1, 0)
    const bool by_cols = dir & 1, mirrored = dir >= 2;
    const int t0 = min(i * per, L), t1 = min(t0 + per, L);
    int pos, left, step, wrap;
    {
        const int tau = mirrored ? max(L - 1 - t0, 0) : min(t0, L - 1);
        uint32_t q, h;
        divmod((uint32_t)tau, p.div_h, q, h);
        pos = by_cols ? (int)h * p.Wd + (int)q : tau;
        left = by_cols ? (mirrored ? (int)h : p.H - 1 - (int)h) : 0x7fffffff;   // steps to the end of the column
        step = (by_cols ? p.Wd : 1) * (mirrored ? -1 : 1);
        wrap = ((p.H - 1) * p.Wd - 1) * (mirrored ? 1 : -1);                    // from there to the start of the next one
    }
    const T *my_rows = s_rows + dir * p.row, *my_x = s_x + chan * L;
    float2 *my_y = s_y + (chan * 4 + dir) * L;
    float prod = t0 == 0 ? 0.0f : 1.0f, h = 0.0f;                                // (nothing enters a scan's first position)
    for (int t = t0; t < t1; ++t) {
        const T *r = my_rows + pos * p.pitch;
        float z[2] = {bias, 0.0f};
#pragma unroll
        for (int q = 0; q < kQ; ++q) {
            const uint4 v = *reinterpret_cast<const uint4 *>(r + q * kPiece);
            const uint32_t e[4] = {v.x, v.y, v.z, v.w};
#pragma unroll
            for (int k = 0; k < 4; ++k)                                         // (behind the ranks: B and C)
                z[k & 1] = few_dot(T{}, q + 1 < kQ || 4 * q + k < nd ? e[k] : 0u, w[4 * q + k], z[k & 1]);
        }
        float Bv, Cv;
        if constexpr (kF32) {
            Bv = r[p.R]; Cv = r[p.R + 1];
        } else {
            const uint32_t bc = reinterpret_cast<const uint32_t *>(r)[nd];
            Bv = unpack_lo<T>(bc); Cv = unpack_hi<T>(bc);
        }
        const float dl = softplus_log2((z[0] + z[1]) * kLog2e);
        const float a = __builtin_amdgcn_exp2f(dl * A);
        h = fmaf(a, h, Bv * (dl * to_f32(my_x[pos])));
        prod *= a;
        my_y[t] = make_float2(Cv * h, Cv * prod);
        const bool end = left == 0;
        pos += end ? wrap : step;
        left = end ? p.H - 1 : left - 1;
    }
    const float h_in = kG == 8 ? octet_scan_state_in(prod, h) : row_scan_state_in<false>(prod, h);      // (of the direction's lanes)
    __shared__ float s_in[kFewThreads];
    s_in[threadIdx.x] = h_in;
    wave_lds_sync();

    // ---- merge: the wavefront's channels, its lanes along the positions
#pragma unroll
    for (int c = 0; c < kCh; ++c) {
        const int ch = wave * kCh + c, from = c * 4 * kG;
        if (d0 + ch >= p.D) break;                                              // uniform
        const float skips = (read_lane(skip, from) + read_lane(skip, from + 2 * kG)) + (read_lane(skip, from + kG) + read_lane(skip, from + 3 * kG));
        const float2 *y = s_y + ch * 4 * L;
        const float *in = s_in + wave * kWave + from;
        float *out = p.y + (b * p.D + d0 + ch) * L;
        for (int l = lane; l < L; l += kWave) {
            uint32_t row, col;
            divmod((uint32_t)l, p.div_w, row, col);
            const int tc = (int)col * p.H + (int)row;
            float v[4];
#pragma unroll
            for (int k = 0; k < 4; ++k) {
                const int fwd = k & 1 ? tc : l, t = k & 2 ? L - 1 - fwd : fwd;
                const float2 e = y[k * L + t];
                v[k] = fmaf(e.y, in[k * kG + ((uint32_t)t * p.per_inv >> 16)], e.x);
            }
            out[l] = fmaf(skips, to_f32(s_x[ch * L + l]), (v[0] + v[2]) + (v[1] + v[3]));
        }
    }
}

static size_t few_lds(int L, int R, bool f32) {
    const size_t es = f32 ? 4 : 2, chans = kFewThreads / kWave * (L <= 64 ? 2 : 1);
    return (size_t)L * few_pitch(R, f32) * es + chans * L * (4 * sizeof(float2) + es);
}

// few_takes: what the two kernels can do, from the sizes and types alone.
bool few_takes(int B, int D, int R, int H, int W, int dtype) {
    const int64_t L = (int64_t)H * W;
    if (B < 1 || R < 1 || R > (dtype == SS2D_F32 ? kFewMaxRank / 2 : kFewMaxRank) || L < 4 || L > kFewMaxL || D < 8 || D % 8 != 0) return false;
    const bool f32 = dtype == SS2D_F32;
    const int64_t tiles = (int64_t)few_row(R, f32) / 4 * ((L + kWave - 1) / kWave) * B, wgs = ((int64_t)D + 3) / 4 * B;
    return few_lds((int)L, R, f32) <= (size_t)kFewMaxLds && tiles <= 0x7fffffff && wgs <= 0x7fffffff && (int64_t)D * L <= 0x7fffffff;
}

int64_t few_rows_bytes(int B, int R, int64_t L, int dtype) {
    const bool f32 = dtype == SS2D_F32;
    return B * L * few_pitch(R, f32) * (f32 ? 4 : 2);
}

// Elements of the map up to which the two kernels are the faster ones.  forward_core with out_norm replayed from a graph, us, as four
// kernels and as these, bf16, for 1 / 8 / 16 / 32 images: 768 x 7 x 7 31 -> 18, 34 -> 24, 40 -> 31, 46 / 45; 384 x 14 x 14 27 -> 15, 32 -> 26,
// 36 / 36, 41 / 58; 192 x 14 x 14 24 -> 14, 26 -> 17, 26 / 24, 33 / 34; 384 x 9 x 11 31 -> 14, 32 -> 19, 39 -> 26, 48 -> 37 (64: 57 / 55);
// 192 x 16 x 16 19 -> 15, 24 -> 19, 28 / 27.  fp32: 384 x 14 x 14 31 -> 17, 44 -> 32, 50 / 46, 63 / 78; 192 x 15 x 13 23 -> 14, 44 -> 29, 51 -> 36,
// 58 -> 49 (64: 73 / 76).  Beyond, every workgroup's copy of its image's rank rows costs more than the launch it saves.  Up to 8 ranks
// the other core takes dt_proj in from 2^19 elements on (kFoldFrom of forward_core.hip), and calls from there on keep to
// ss2d_x_proj's ranks: 32 images of 96 x 14 x 14 stay at 26 where these would take 19.
constexpr int64_t kFewMost = 1 << 20, kFewMostF32 = 5 << 18, kFewMostFolded = (1 << 19) - 1;

bool few_pays(int B, int D, int R, int H, int W, int dtype) {
    const int64_t most = dtype == SS2D_F32 ? kFewMostF32 : R <= 8 ? kFewMostFolded : kFewMost;
    return few_takes(B, D, R, H, W, dtype) && (int64_t)B * D * H * W <= most;
}

template <typename T, int kG>
static int launch_core_few(const FewCoreArgs &a, size_t smem, hipStream_t s) {
    constexpr int kPer = 16 / (int)sizeof(T);                        // ranks in a piece
    const dim3 grid((uint32_t)((int64_t)a.B * a.chan_sets)), block(kFewThreads);
#define SS2D_FEW(Q)                                                                                                                              \
    case Q: {                                                                                                                                    \
        auto kern = core_few_kernel<T, kG, Q>;                                                                                                   \
        if (smem > 60 * 1024 &&                                                                                                                  \
            hipFuncSetAttribute(reinterpret_cast<const void *>(kern), hipFuncAttributeMaxDynamicSharedMemorySize, (int)smem) != hipSuccess)      \
            return SS2D_ELAUNCH;                                                                                                                 \
        hipLaunchKernelGGL(kern, grid, block, smem, s, a);                                                                                       \
        return launch_status();                                                                                                                  \
    }
    switch ((a.R + kPer - 1) / kPer) {
        SS2D_FEW(1) SS2D_FEW(2) SS2D_FEW(3) SS2D_FEW(4) SS2D_FEW(5) SS2D_FEW(6)
        default: return SS2D_ENOTSUP;
    }
#undef SS2D_FEW
}

template <typename T>
static int launch_core_few_for(FewCoreArgs &a, hipStream_t s) {
    constexpr bool kF32 = sizeof(T) == 4;
    const bool two = a.L <= 64;
    const int chans = kFewThreads / kWave * (two ? 2 : 1), lanes = two ? 8 : 16;
    a.chan_sets = (a.D + chans - 1) / chans;
    a.row = few_row(a.R, kF32);
    a.pitch = few_pitch(a.R, kF32);
    a.rows_bytes = a.L * a.pitch * (int)sizeof(T);
    a.per_lane = ((a.L + lanes - 1) / lanes) | 1;                    // (odd: lanes side by side meet in few LDS banks; at 256 positions 17 still cover the map)
    a.per_inv = (65536u + a.per_lane - 1) / a.per_lane;
    a.div_h = make_fastdiv((uint32_t)a.H);
    a.div_w = make_fastdiv((uint32_t)a.Wd);
    const size_t smem = few_lds(a.L, a.R, kF32);
    return two ? launch_core_few<T, 8>(a, smem, s) : launch_core_few<T, 16>(a, smem, s);
}

}  // namespace ss2d

extern "C" int64_t ss2d_few_rows_bytes(int B, int D, int R, int H, int W, int dtype) {
    using namespace ss2d;
    if (dtype != SS2D_F32 && dtype != SS2D_BF16 && dtype != SS2D_F16) return SS2D_EINVAL;
    if (B < 0 || D < 0 || R < 0 || H < 0 || W < 0) return SS2D_EINVAL;
    return few_takes(B, D, R, H, W, dtype) ? few_rows_bytes(B, R, (int64_t)H * W, dtype) : SS2D_ENOTSUP;
}

extern "C" int ss2d_few_applies(int B, int D, int R, int H, int W, int dtype) {
    using namespace ss2d;
    const int64_t need = ss2d_few_rows_bytes(B, D, R, H, W, dtype);
    return need < 0 ? (int)need : few_pays(B, D, R, H, W, dtype) ? SS2D_OK : SS2D_ENOTSUP;
}

extern "C" int ss2d_x_proj_few(const void *x, const void *weight, void *rows, int B, int D, int R, int H, int W, int dtype, void *stream) {
    using namespace ss2d;
    const int64_t need = ss2d_few_rows_bytes(B, D, R, H, W, dtype);
    if (need < 0) return (int)need;
    if (!x || !weight || !rows) return SS2D_EINVAL;
    if (reinterpret_cast<uintptr_t>(weight) % 16 != 0 || reinterpret_cast<uintptr_t>(rows) % 16 != 0) return SS2D_ENOTSUP;
    const int L = H * W, row = few_row(R, dtype == SS2D_F32);
    const FewProjArgs a = {x, weight, rows, B, D, R, L, row, few_pitch(R, dtype == SS2D_F32), row / 4, (L + kWave - 1) / kWave};
    const dim3 grid((uint32_t)((int64_t)B * a.m_tiles * a.groups)), block(kFewWaves * kWave);
    hipStream_t s = (hipStream_t)stream;
    if (dtype == SS2D_F32) hipLaunchKernelGGL((x_proj_few_kernel<float>), grid, block, 0, s, a);
    else if (dtype == SS2D_BF16) hipLaunchKernelGGL((x_proj_few_kernel<bf16_t>), grid, block, 0, s, a);
    else hipLaunchKernelGGL((x_proj_few_kernel<f16_t>), grid, block, 0, s, a);
    return launch_status();
}

extern "C" int ss2d_core_few(const void *x, const void *rows, const void *dt_weight, const float *A, const float *D_skip, const float *delta_bias,
                             float *y, int B, int D, int R, int H, int W, int dtype, void *stream) {
    using namespace ss2d;
    const int64_t need = ss2d_few_rows_bytes(B, D, R, H, W, dtype);
    if (need < 0) return (int)need;
    if (!x || !rows || !dt_weight || !A || !y) return SS2D_EINVAL;
    if (reinterpret_cast<uintptr_t>(rows) % 16 != 0) return SS2D_ENOTSUP;
    FewCoreArgs a = {};
    a.x = x; a.rows = rows; a.W = dt_weight; a.A = A; a.Dv = D_skip; a.bias = delta_bias; a.y = y;
    a.B = B; a.D = D; a.H = H; a.Wd = W; a.L = H * W; a.R = R;
    hipStream_t s = (hipStream_t)stream;
    if (dtype == SS2D_F32) return launch_core_few_for<float>(a, s);
    if (dtype == SS2D_BF16) return launch_core_few_for<bf16_t>(a, s);
    return launch_core_few_for<f16_t>(a, s);
}
