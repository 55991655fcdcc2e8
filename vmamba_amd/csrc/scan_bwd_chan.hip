// Selective-scan backward for 4 / 8 / 16 states per channel: a lane is a channel and a quarter of its states, walked serially along
// the sequence (the equations are at the top of selective_scan_bwd.hip).
//
// A wavefront owns 16 channels of one (image, group): lane = 4 channel + set, the four sets sharing out the states, so that the
// recurrences in both directions are serial chains per lane with no scan across lanes and positions past a row's end cost a chunk of
// 8 at most.  What crosses lanes are sums: S_t and T_t over a channel's four sets (through LDS), dB and dC over the 16 channels
// (sum_over_channels: 8 positions of both at once, 2.1 instructions per value) and over the 64 channels of a workgroup's four
// wavefronts, before they reach memory as one atomic per entry.
//
// Rows are cut into segments of at most 72 positions, which run side by side in two passes with one between them:
//   local   what a segment leaves from state 0 (h), what it hands to the positions before it with nothing behind it (a_t g_t of its
//           first position), its sum of dl, its largest dl and its share of dD;
//   carry   what enters every segment from either side; dD of all but the last segment, so that rounding does not add up over segments;
//   grad    a forward sweep that keeps the state entering every chunk of 8 positions in LDS, and the reverse sweep with the gradients.
// The states lie where the segment's du and d delta will be, so there is no workspace.
//
// What bounds it: vector issue.  16 x 192 maps of 28 x 28 as four directions, 16 states, bf16: 51 + 13 + 158 us (local, carry, grad), the last 82 % of its time
// issuing (25 instructions per position and state, three wavefronts per SIMD); positions in lanes took 411.  Sums added to an LDS tile with LDS atomics, as a first
// version did, took 238 of its own: such an addition keeps the LDS busy for about 200 cycles.
#include "scan_common.h"

namespace ss2d {

constexpr int kBcChan = 16;                       // channels per wavefront
constexpr int kBcSets = 4;                        // lanes per channel
constexpr int kBcSub = 8;                         // positions per chunk
constexpr int kBcPitch = kBcSub + 4;              // floats of an LDS row of a chunk; 16-byte pieces, 8 rows over all banks
constexpr int kBcGroup = kBcSets * kBcPitch + 4;  // floats of the sets' rows of B or C for one of a lane's states, and a row of zeros from the last pad on
constexpr int kBcZeros = kBcSets * kBcPitch - 4;
constexpr int kBcChunks = 9;                      // chunks per segment at most
constexpr int kBcSeg = kBcChunks * kBcSub;

struct BwdChanGeom {
    int32_t n_cb, n_segs;                         // blocks of 64 channels per group; segments per row
    int32_t seg_chunks, n_longer;                 // chunks of a segment; the first n_longer segments have one more
    FastDiv div_cb, div_groups, div_segs;
};

__host__ __device__ __forceinline__ int bwd_chan_begin(int seg, int seg_chunks, int n_longer) {
    return (seg * seg_chunks + (seg < n_longer ? seg : n_longer)) * kBcSub;
}

// Two elements from an even `pos` of a row that a plain (not rounded) base and element `row` give.
template <typename T, bool kDwords>
__device__ __forceinline__ void store2_at(__amdgpu_buffer_rsrc_t buf, uint32_t row, int pos, int L, bool ok, bool whole, float v0, float v1) {
    typedef uint32_t words2_t __attribute__((ext_vector_type(2)));
    const uint32_t at = (row + (uint32_t)pos) * (uint32_t)sizeof(T);
    const int off0 = (int)(ok && pos < L ? at : kNowhere), off1 = (int)(ok && pos + 1 < L ? at + (uint32_t)sizeof(T) : kNowhere);
    if constexpr (sizeof(T) == 2) {
        if constexpr (kDwords) {
            __builtin_amdgcn_raw_buffer_store_b32(pack2_from_f32<T>(v0, v1), buf, off0, 0, 0);
        } else {
            __builtin_amdgcn_raw_buffer_store_b16(from_f32<T>(v0).bits, buf, off0, 0, 0);
            __builtin_amdgcn_raw_buffer_store_b16(from_f32<T>(v1).bits, buf, off1, 0, 0);
        }
    } else if (whole) {
        const words2_t w = {f32_to_bits(v0), f32_to_bits(v1)};
        __builtin_amdgcn_raw_buffer_store_b64(w, buf, off0, 0, 0);
    } else {
        __builtin_amdgcn_raw_buffer_store_b32(f32_to_bits(v0), buf, off0, 0, 0);
        __builtin_amdgcn_raw_buffer_store_b32(f32_to_bits(v1), buf, off1, 0, 0);
    }
}

// v[i] summed over the 16 channels (lane / 4) for every i of 16, entry 8 (lane bit 3) + 4 (bit 2) + 2 (bit 5) + (bit 4) left with each
// lane.  Bits 3 and 2 by DPP additions, bits 5 and 4 by swaps.
__device__ __forceinline__ float sum_over_channels(float (&v)[16]) {
    sum_over_quads(v);
    auto halves = [](float a, float b) {
        const auto r = __builtin_amdgcn_permlane32_swap(f32_to_bits(a), f32_to_bits(b), false, false);
        return bits_to_f32(r[0]) + bits_to_f32(r[1]);
    };
    const float a = halves(v[0], v[2]), b = halves(v[1], v[3]);
    const auto r = __builtin_amdgcn_permlane16_swap(f32_to_bits(a), f32_to_bits(b), false, false);
    return bits_to_f32(r[0]) + bits_to_f32(r[1]);
}

// kGrad: the gradients from the states that enter the segment (see the top); otherwise what the segment leaves on either side.
template <typename in_t, typename dy_t, int kSpw, bool kDwords, bool kGrad>
__global__ __launch_bounds__(kBlock, !kGrad ? (kSpw == 4 ? 4 : 5) : kSpw == 4 && (!kDwords || sizeof(in_t) == 4) ? 2 : 3) void scan_bwd_chan_kernel(const ScanBwdArgs p, const BwdChanGeom geo) {
    constexpr int kN = kBcSets * kSpw;
    constexpr int kTile = 3 * kBcChan * kBcPitch + 2 * kSpw * kBcGroup;
    constexpr int kScratch = kTile > kWave * kBcPitch ? kTile : kWave * kBcPitch;       // also S / T of all lanes
    __shared__ __align__(16) float s_all[kWavesPerWg * kScratch];
    constexpr int kChunk = kWave * kSpw + 4;                                            // (+ 4: the last sums' reads across chunks on other banks)
    // per chunk the state that enters it, [lane][state]; once that has been read its dB and dC over 16 channels, [state][lane]
    __shared__ __align__(16) float s_h_all[kGrad ? kWavesPerWg * kBcChunks * kChunk : 1];

    const int lane = threadIdx.x & (kWave - 1);
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave);
    uint32_t wg = xcd_contiguous_id(blockIdx.x, gridDim.x), bg, cb, b, grp, seg;
    divmod(wg, geo.div_segs, wg, seg);
    divmod(wg, geo.div_cb, bg, cb);
    divmod(bg, geo.div_groups, b, grp);
    const int L = p.L, begin = bwd_chan_begin((int)seg, geo.seg_chunks, geo.n_longer);
    const int stop = min(L, bwd_chan_begin((int)seg + 1, geo.seg_chunks, geo.n_longer));
    const int n_chunks = (stop - begin + kBcSub - 1) / kBcSub;
    const int c_first = (int)cb * 64 + wave * kBcChan, n_chan = min(kBcChan, p.dim_per_group - c_first);
    const bool softplus = p.softplus != 0;

    if (n_chan > 0) {                                       // uniform over the wavefront
        float *s_dl = s_all + wave * kScratch, *s_dlu = s_dl + kBcChan * kBcPitch, *s_dy = s_dlu + kBcChan * kBcPitch;
        float *s_bc = s_dy + kBcChan * kBcPitch;            // rows [B, C][state of the lane][set or zeros]
        float *s_h = s_h_all + wave * kBcChunks * kChunk;
        const int ch = lane >> 2, set = lane & 3;
        const bool chan_ok = ch < n_chan;
        const int d_first = (int)grp * p.dim_per_group + c_first, d = d_first + min(ch, n_chan - 1);
        const int dg_first = d_first / p.dim_per_delta, dg = d / p.dim_per_delta;
        uint32_t u_row, dl_row, dy_row, B_row, C_row;       // the element a lane's row starts at
        const auto u_buf = dwords_of<in_t>(p.u, (int64_t)b * p.u_bs + (int64_t)d_first * p.u_ds, n_chan, p.u_ds, L, u_row);
        const auto dl_buf = dwords_of<in_t>(p.delta, (int64_t)b * p.dl_bs + (int64_t)dg_first * p.dl_ds, (d_first + n_chan - 1) / p.dim_per_delta - dg_first + 1, p.dl_ds, L, dl_row);
        const auto dy_buf = dwords_of<dy_t>(p.dout, (int64_t)b * p.do_bs + (int64_t)d_first * p.do_ds, n_chan, p.do_ds, L, dy_row);
        const auto B_buf = dwords_of<in_t>(p.B, (int64_t)b * p.B_bs + (int64_t)grp * p.B_gs, kN, p.B_ns, L, B_row);
        const auto C_buf = dwords_of<in_t>(p.C, (int64_t)b * p.C_bs + (int64_t)grp * p.C_gs, kN, p.C_ns, L, C_row);
        u_row += (uint32_t)((d - d_first) * p.u_ds);
        dl_row += (uint32_t)((dg - dg_first) * p.dl_ds);
        dy_row += (uint32_t)((d - d_first) * p.do_ds);
        // staging: two positions of a channel's rows per lane (no channel: zeros), and four of a row of B and of C each, the lanes behind those of zeros.
        // A lane without a channel reads the zeros for B and C and has a decay of 1, so that it adds nothing to dB and dC: with the last channel's A and bias
        // its decay may overflow where that channel's does not, and B and C may be infinite.
        const int q2 = 2 * set;
        struct Raw {
            RawGroup<in_t, 2, kDwords> u, dl;
            RawGroup<dy_t, 2, kDwords || sizeof(dy_t) == 4> dy;
            RawGroup<in_t, 4, kDwords> B, C;
        };
        const int r2 = lane >> 1, p4 = 4 * (lane & 1);      // rows of B (and of C): r2 < N
        const bool bc_mine = r2 < kN;
        const int n_row = (r2 & 3) * kSpw + min(r2 >> 2, kSpw - 1);
        float *st_bc = s_bc + (bc_mine ? (r2 >> 2) * kBcGroup + (r2 & 3) * kBcPitch : r2 % kSpw * kBcGroup + kBcZeros) + p4;
        B_row += (uint32_t)(n_row * p.B_ns);
        C_row += (uint32_t)(n_row * p.C_ns);
        auto load_rows = [&](int t, bool all, Raw &r) {
            r.u = load_at<in_t, 2, kDwords>(u_buf, u_row, t + q2, L, chan_ok);
            r.dl = load_at<in_t, 2, kDwords>(dl_buf, dl_row, t + q2, L, chan_ok);
            r.B = load_at<in_t, 4, kDwords>(B_buf, B_row, t + p4, L, bc_mine);
            if (all) {
                r.dy = load_at<dy_t, 2, kDwords || sizeof(dy_t) == 4>(dy_buf, dy_row, t + q2, L, chan_ok);
                r.C = load_at<in_t, 4, kDwords>(C_buf, C_row, t + p4, L, bc_mine);
            }
        };
        const float bias = p.bias && chan_ok ? p.bias[dg] : 0.0f, Dv = p.D ? p.D[d] : 0.0f;
        float A[kSpw], A2[kSpw];
#pragma unroll
        for (int j = 0; j < kSpw; ++j) {
            A[j] = chan_ok ? p.A[(int64_t)d * p.A_ds + (int64_t)(set * kSpw + j) * p.A_ns] : 0.0f;
            A2[j] = A[j] * kLog2e;
        }
        // a chunk's dl, dl u (dy), B (C) into LDS; dl, u, dy, raw: this lane's own positions
        auto stage = [&](const Raw &r, int t, bool all, float (&dl)[2], float (&uv)[2], float (&dy)[2], float (&raw)[2]) {
            widen<in_t, 2, kDwords>(r.dl, dl_row, raw);
            widen<in_t, 2, kDwords>(r.u, u_row, uv);
            float Bv[4], Cv[4];
            widen<in_t, 4, kDwords>(r.B, B_row, Bv);
            if (all) {
                widen<dy_t, 2, kDwords || sizeof(dy_t) == 4>(r.dy, dy_row, dy);
                widen<in_t, 4, kDwords>(r.C, C_row, Cv);
            }
#pragma unroll
            for (int i = 0; i < 2; ++i) dl[i] = softplus ? softplus_log2(fmaf(raw[i], kLog2e, bias * kLog2e)) : raw[i] + bias;
            if (t + kBcSub > L) {                           // uniform; past the row's end 0, the identity of the recurrence
#pragma unroll
                for (int i = 0; i < 2; ++i) {
                    const bool in = t + q2 + i < L;
                    dl[i] = in ? dl[i] : 0.0f;
                    uv[i] = in ? uv[i] : 0.0f;
                    if (all) dy[i] = in ? dy[i] : 0.0f;
                }
#pragma unroll
                for (int i = 0; i < 4; ++i) {
                    const bool in = t + p4 + i < L;
                    Bv[i] = in ? Bv[i] : 0.0f;
                    if (all) Cv[i] = in ? Cv[i] : 0.0f;
                }
            }
            const int at = ch * kBcPitch + q2;
            *reinterpret_cast<float2 *>(s_dl + at) = make_float2(dl[0], dl[1]);
            *reinterpret_cast<float2 *>(s_dlu + at) = make_float2(dl[0] * uv[0], dl[1] * uv[1]);
            *reinterpret_cast<float4 *>(st_bc) = make_float4(Bv[0], Bv[1], Bv[2], Bv[3]);
            if (all) {
                *reinterpret_cast<float2 *>(s_dy + at) = make_float2(dy[0], dy[1]);
                *reinterpret_cast<float4 *>(st_bc + kSpw * kBcGroup) = make_float4(Cv[0], Cv[1], Cv[2], Cv[3]);
            }
        };
        auto read8 = [](const float *from, float (&v)[kBcSub]) {
            const float4 lo = *reinterpret_cast<const float4 *>(from), hi = *reinterpret_cast<const float4 *>(from + 4);
            v[0] = lo.x; v[1] = lo.y; v[2] = lo.z; v[3] = lo.w; v[4] = hi.x; v[5] = hi.y; v[6] = hi.z; v[7] = hi.w;
        };
        const float *my_bc = s_bc + (chan_ok ? set * kBcPitch : kBcZeros);
        auto read_B = [&](int j, float (&v)[kBcSub]) { read8(my_bc + j * kBcGroup, v); };
        auto read_C = [&](int j, float (&v)[kBcSub]) { read8(my_bc + (kSpw + j) * kBcGroup, v); };

        // what enters (leaves) the segment, where its du and d delta will be: N states, the sum of dl and the largest; N adjoints and a share of dD
        uint8_t *h_state = reinterpret_cast<uint8_t *>(reinterpret_cast<in_t *>(p.du) + ((int64_t)b * p.dim + d) * L + begin);
        uint8_t *g_state = reinterpret_cast<uint8_t *>(reinterpret_cast<in_t *>(p.ddelta) + ((int64_t)b * p.dim + d) * L + begin);
        float h[kSpw], g[kSpw];                             // g: a_t+1 g_t+1 of the position t that is next
#pragma unroll
        for (int j = 0; j < kSpw; ++j) { h[j] = 0.0f; g[j] = 0.0f; }

        auto over_quad = [](float x) { x += __shfl_xor(x, 1, kWave); return x + __shfl_xor(x, 2, kWave); };
        if constexpr (!kGrad) {
            float dl_sum = 0.0f, dl_max = 0.0f, dD = 0.0f;
            Raw next;
            load_rows(begin, true, next);
            for (int t = begin; t < stop; t += kBcSub) {
                float own_dl[2], own_u[2], own_dy[2], own_raw[2];
                stage(next, t, true, own_dl, own_u, own_dy, own_raw);
                load_rows(t + kBcSub, true, next);
                wave_lds_sync();
                float dl[kBcSub], dlu[kBcSub], dy[kBcSub];
                read8(s_dl + ch * kBcPitch, dl);
                read8(s_dlu + ch * kBcPitch, dlu);
                read8(s_dy + ch * kBcPitch, dy);
#pragma unroll
                for (int j = 0; j < kSpw; ++j) {
                    float Bv[kBcSub], Cv[kBcSub], a[kBcSub], gl = 0.0f;
                    read_B(j, Bv);
                    read_C(j, Cv);
#pragma unroll
                    for (int i = 0; i < kBcSub; ++i) {
                        a[i] = __builtin_amdgcn_exp2f(dl[i] * A2[j]);
                        h[j] = fmaf(a[i], h[j], Bv[i] * dlu[i]);
                    }
#pragma unroll
                    for (int i = kBcSub - 1; i >= 0; --i) gl = fmaf(Cv[i], dy[i], gl) * a[i];
                    g[j] = gl == 0.0f ? g[j] : fmaf(__builtin_amdgcn_exp2f(A2[j] * dl_sum), gl, g[j]);
                }
                dD += fmaf(own_dy[0], own_u[0], own_dy[1] * own_u[1]);
                dl_max = fmaxf(dl_max, fmaxf(own_dl[0], own_dl[1]));
                dl_sum += ((dl[0] + dl[1]) + (dl[2] + dl[3])) + ((dl[4] + dl[5]) + (dl[6] + dl[7]));
                wave_lds_sync();
            }
            // An infinite gl times a product of a that has left fp32's range is NaN, where it would pass every position unless one of their a is 0: walk the
            // positions in their own order then.
            bool walk = false;
#pragma unroll
            for (int j = 0; j < kSpw; ++j) walk = walk || g[j] != g[j];
            if (__any(walk)) {                              // uniform
#pragma unroll
                for (int j = 0; j < kSpw; ++j) g[j] = 0.0f;
                for (int t = begin + (n_chunks - 1) * kBcSub; t >= begin; t -= kBcSub) {
                    float own_dl[2], own_u[2], own_dy[2], own_raw[2];
                    load_rows(t, true, next);
                    stage(next, t, true, own_dl, own_u, own_dy, own_raw);
                    wave_lds_sync();
                    float dl[kBcSub], dy[kBcSub];
                    read8(s_dl + ch * kBcPitch, dl);
                    read8(s_dy + ch * kBcPitch, dy);
#pragma unroll
                    for (int j = 0; j < kSpw; ++j) {
                        float Cv[kBcSub];
                        read_C(j, Cv);
#pragma unroll
                        for (int i = kBcSub - 1; i >= 0; --i) g[j] = fmaf(Cv[i], dy[i], g[j]) * __builtin_amdgcn_exp2f(dl[i] * A2[j]);
                    }
                    wave_lds_sync();
                }
            }
            dD = over_quad(dD);
            dl_max = fmaxf(dl_max, __shfl_xor(dl_max, 1, kWave));
            dl_max = fmaxf(dl_max, __shfl_xor(dl_max, 2, kWave));
            if (chan_ok) {
                __builtin_memcpy(h_state + sizeof(float) * (set * kSpw), h, sizeof(h));
                __builtin_memcpy(g_state + sizeof(float) * (set * kSpw), g, sizeof(g));
                if (set == 0 && (int)seg + 1 < geo.n_segs) {
                    __builtin_memcpy(h_state + sizeof(float) * kN, &dl_sum, sizeof(float));
                    __builtin_memcpy(h_state + sizeof(float) * (kN + 1), &dl_max, sizeof(float));
                    __builtin_memcpy(g_state + sizeof(float) * kN, &dD, sizeof(float));
                }
            }
        } else {
            if (geo.n_segs > 1 && chan_ok) {
                if (seg > 0) __builtin_memcpy(h, h_state + sizeof(float) * (set * kSpw), sizeof(h));
                if ((int)seg + 1 < geo.n_segs) __builtin_memcpy(g, g_state + sizeof(float) * (set * kSpw), sizeof(g));
            }
            auto keep = [&](int c) {
#pragma unroll
                for (int j = 0; j < kSpw; ++j) s_h[c * kChunk + lane * kSpw + j] = h[j];
            };
            // ---- forward: the state entering every chunk -------------------------------------------------------------------
            Raw next;
            load_rows(begin, n_chunks == 1, next);
            keep(0);
            for (int c = 0; c + 1 < n_chunks; ++c) {
                const int t = begin + c * kBcSub;
                float own_dl[2], own_u[2], own_dy[2], own_raw[2];
                stage(next, t, false, own_dl, own_u, own_dy, own_raw);
                load_rows(t + kBcSub, c + 2 == n_chunks, next);
                wave_lds_sync();
                float dl[kBcSub], dlu[kBcSub];
                read8(s_dl + ch * kBcPitch, dl);
                read8(s_dlu + ch * kBcPitch, dlu);
#pragma unroll
                for (int j = 0; j < kSpw; ++j) {
                    float Bv[kBcSub];
                    read_B(j, Bv);
#pragma unroll
                    for (int i = 0; i < kBcSub; ++i) h[j] = fmaf(__builtin_amdgcn_exp2f(dl[i] * A2[j]), h[j], Bv[i] * dlu[i]);
                }
                keep(c + 1);
                wave_lds_sync();
            }
            // ---- reverse: the gradients ------------------------------------------------------------------------------------
            const auto du_buf = rows_of<in_t>(p.du, ((int64_t)b * p.dim + d_first) * L, n_chan, L, L);
            const auto dd_buf = rows_of<in_t>(p.ddelta, ((int64_t)b * p.dim + d_first) * L, n_chan, L, L);
            const uint32_t out_row = (uint32_t)((d - d_first) * L);
            float dA[kSpw], dD = 0.0f, db = 0.0f;
#pragma unroll
            for (int j = 0; j < kSpw; ++j) dA[j] = 0.0f;
            for (int c = n_chunks - 1; c >= 0; --c) {
                const int t = begin + c * kBcSub;
                float own_dl[2], own_u[2], own_dy[2], own_raw[2];
                stage(next, t, true, own_dl, own_u, own_dy, own_raw);
                load_rows(max(t - kBcSub, begin), true, next);      // (before the first chunk: read again, not used)
                wave_lds_sync();
                float dl[kBcSub], dlu[kBcSub], dy[kBcSub], S[kBcSub], T[kBcSub];
                read8(s_dl + ch * kBcPitch, dl);
                read8(s_dlu + ch * kBcPitch, dlu);
                read8(s_dy + ch * kBcPitch, dy);
                float *h_chunk = s_h + c * kChunk;
#pragma unroll
                for (int j = 0; j < kSpw; ++j) h[j] = h_chunk[lane * kSpw + j];
                wave_lds_sync();
#pragma unroll
                for (int i = 0; i < kBcSub; ++i) { S[i] = 0.0f; T[i] = 0.0f; }
#pragma unroll
                for (int j = 0; j < kSpw; ++j) {
                    float Bv[kBcSub], Cv[kBcSub], a[kBcSub], ah[kBcSub], v[2 * kBcSub];
                    read_B(j, Bv);
                    read_C(j, Cv);
                    float hj = h[j], gj = g[j];
#pragma unroll
                    for (int i = 0; i < kBcSub; ++i) {
                        a[i] = __builtin_amdgcn_exp2f(dl[i] * A2[j]);
                        ah[i] = a[i] * hj;                              // a_t h_t-1
                        hj = fmaf(Bv[i], dlu[i], ah[i]);
                        v[kBcSub + i] = dy[i] * hj;                     // dC
                    }
#pragma unroll
                    for (int i = kBcSub - 1; i >= 0; --i) {
                        gj = fmaf(Cv[i], dy[i], gj);
                        const float da_a = gj * ah[i];                  // dL/da_t * a_t
                        dA[j] = fmaf(da_a, dl[i], dA[j]);
                        T[i] = fmaf(da_a, A[j], T[i]);
                        S[i] = fmaf(gj, Bv[i], S[i]);
                        v[i] = gj * dlu[i];                             // dB
                        gj *= a[i];
                    }
                    g[j] = gj;
                    h_chunk[j * kWave + lane] = sum_over_channels(v);
                }
                // S and T over the four sets: two positions for each
                float own_S[2] = {0.0f, 0.0f}, own_T[2] = {0.0f, 0.0f};
                float *mine = s_dl + lane * kBcPitch;
                const float *theirs = s_dl + (lane & ~3) * kBcPitch + q2;
                auto over_sets = [&](const float (&x)[kBcSub], float (&sum)[2]) {
                    wave_lds_sync();
                    *reinterpret_cast<float4 *>(mine) = make_float4(x[0], x[1], x[2], x[3]);
                    *reinterpret_cast<float4 *>(mine + 4) = make_float4(x[4], x[5], x[6], x[7]);
                    wave_lds_sync();
#pragma unroll
                    for (int k = 0; k < kBcSets; ++k) {
                        const float2 part = *reinterpret_cast<const float2 *>(theirs + k * kBcPitch);
                        sum[0] += part.x;
                        sum[1] += part.y;
                    }
                };
                over_sets(S, own_S);
                over_sets(T, own_T);
                wave_lds_sync();
                float du[2], dd[2], db_own[2];
#pragma unroll
                for (int i = 0; i < 2; ++i) {
                    du[i] = fmaf(own_S[i], own_dl[i], own_dy[i] * Dv);
                    dd[i] = fmaf(own_S[i], own_u[i], own_T[i]);
                    if (softplus) dd[i] *= bwd_sigmoid(own_raw[i], bias);
                    db_own[i] = t + q2 + i < L ? dd[i] : 0.0f;
                }
                dD += fmaf(own_dy[0], own_u[0], own_dy[1] * own_u[1]);
                db += db_own[0] + db_own[1];
                const bool whole = t + kBcSub <= L;
                store2_at<in_t, kDwords>(du_buf, out_row, t + q2, L, chan_ok, whole, du[0], du[1]);
                store2_at<in_t, kDwords>(dd_buf, out_row, t + q2, L, chan_ok, whole, dd[0], dd[1]);
            }
            dD = over_quad(dD);
            db = over_quad(db);
            if (chan_ok) {
#pragma unroll
                for (int j = 0; j < kSpw; ++j) unsafeAtomicAdd(p.dA + (int64_t)d * kN + set * kSpw + j, dA[j]);
                if (set == 0 && p.dD && (int)seg + 1 == geo.n_segs) unsafeAtomicAdd(p.dD + d, dD);
                if (set == 1 && p.dbias) unsafeAtomicAdd(p.dbias + d, db);
            }
        }
    }
    if constexpr (kGrad) {
        __syncthreads();
        // entry (array, state, position) of a chunk is with the lane that sum_over_channels left it with
        const int n_pos = stop - begin, n_waves = min(kWavesPerWg, (p.dim_per_group - (int)cb * 64 + kBcChan - 1) / kBcChan);
        for (int row = wave; row < 2 * kN; row += kWavesPerWg) {
            const int n = row % kN, is_C = row / kN;
            float *to = (is_C ? p.dC : p.dB) + (int64_t)b * p.g_bs + (int64_t)grp * p.g_gs + n * p.g_ns + begin;
            for (int i = lane; i < n_pos; i += kWave) {
                const float *from = s_h_all + (i >> 3) * kChunk + (n % kSpw) * kWave + n / kSpw + 8 * is_C + (i & 4) + 16 * (i & 2) + 16 * (i & 1);
                float sum = from[0];
                for (int w = 1; w < n_waves; ++w) sum += from[w * kBcChunks * kChunk];
                unsafeAtomicAdd(to + i, sum);
            }
        }
    }
}

// What enters every segment of a row from either side, in the place of what the segments left: a thread per (row, state) and side.
template <typename in_t>
__global__ __launch_bounds__(kBlock) void scan_bwd_chan_carry_kernel(const ScanBwdArgs p, int seg_chunks, int n_longer, int n_segs, uint32_t n_items, FastDiv div_n, FastDiv div_dim) {
    const uint32_t item = blockIdx.x * kBlock + threadIdx.x;
    if (item >= n_items) return;
    uint32_t row, n, b, d;
    divmod(item, div_n, row, n);
    divmod(row, div_dim, b, d);
    const float A2 = p.A[(int64_t)d * p.A_ds + (int64_t)n * p.A_ns] * kLog2e;
    uint8_t *h_state = reinterpret_cast<uint8_t *>(reinterpret_cast<in_t *>(p.du) + (int64_t)row * p.L) + sizeof(float) * n;
    uint8_t *g_state = reinterpret_cast<uint8_t *>(reinterpret_cast<in_t *>(p.ddelta) + (int64_t)row * p.L) + sizeof(float) * n;
    const uint8_t *sums = reinterpret_cast<const uint8_t *>(reinterpret_cast<const in_t *>(p.du) + (int64_t)row * p.L) + sizeof(float) * p.N;
    auto place = [&](int s) { return (int64_t)bwd_chan_begin(s, seg_chunks, n_longer) * (int)sizeof(in_t); };
    // Carry through a segment: the product of its a in two halves, so that neither leaves fp32's range before the state would; none of a state of 0, and
    // none of an infinite one: it stays infinite unless one of the a is 0 (the one of the largest dl, where A is negative), which leaves NaN.  A carry that is not
    // finite does not become so again, so a group of segments is walked for finite ones first, and once more where that does not hold (infinite ones looked for at
    // every segment 44 of them took 26.7 us, and 23.8 without a look; so, with dD's shares read among the other loads and not one by one in front, 14.6).
    constexpr int kFly = 8;
    const bool back = blockIdx.y != 0, adds_dD = n == 0 && !back && p.dD;
    uint8_t *own = back ? g_state : h_state;
    float carry = 0.0f;
    double dD = 0.0;
    for (int first = 0; first < n_segs; first += kFly) {
        float left[kFly], sum[kFly], half[kFly], part[kFly];
        int64_t at[kFly];
#pragma unroll
        for (int i = 0; i < kFly; ++i) {                    // (past the last segment: that one again, not used)
            const int nth = min(first + i, n_segs - 1), s = back ? n_segs - 1 - nth : nth;
            at[i] = place(s);
            __builtin_memcpy(&left[i], own + at[i], sizeof(float));
            __builtin_memcpy(&sum[i], sums + place(min(s, n_segs - 2)), sizeof(float));         // (nothing goes through the last one)
            part[i] = 0.0f;
            if (adds_dD) __builtin_memcpy(&part[i], g_state + place(min(s, n_segs - 2)) + sizeof(float) * p.N, sizeof(float));
        }
#pragma unroll
        for (int i = 0; i < kFly; ++i) half[i] = __builtin_amdgcn_exp2f(0.5f * A2 * sum[i]);
        const float entered = carry;
#pragma unroll
        for (int i = 0; i < kFly; ++i) {
            if (first + i >= n_segs) break;
            if (first + i + 1 < n_segs) dD += part[i];
            __builtin_memcpy(own + at[i], &carry, sizeof(float));
            carry = carry == 0.0f ? left[i] : fmaf(carry * half[i], half[i], left[i]);
        }
        if (!(fabsf(carry) < __builtin_inff())) {
            carry = entered;
#pragma unroll
            for (int i = 0; i < kFly; ++i) {
                if (first + i >= n_segs) break;
                __builtin_memcpy(own + at[i], &carry, sizeof(float));
                if (fabsf(carry) == __builtin_inff()) {
                    const int nth = first + i, s = back ? n_segs - 1 - nth : nth;
                    float most;
                    __builtin_memcpy(&most, sums + place(min(s, n_segs - 2)) + sizeof(float), sizeof(float));
                    carry = __builtin_amdgcn_exp2f(A2 * most) > 0.0f ? carry + left[i] : __builtin_nanf("");
                } else {
                    carry = carry == 0.0f ? left[i] : fmaf(carry * half[i], half[i], left[i]);
                }
            }
        }
    }
    if (adds_dD) unsafeAtomicAdd(p.dD + d, (float)dD);
}

// A row's segments: as few as hold it, its chunks of 8 dealt out evenly, the longer ones first.  From 10 chunks on (the first row that is cut) that is 5
// chunks at least: 33 positions in the last segment, room for its 16 states in 16 bits, 40 in the others, room for theirs and two sums.
static void bwd_chan_segments(int L, BwdChanGeom &geo) {
    const int n_chunks = (L + kBcSub - 1) / kBcSub;
    geo.n_segs = (n_chunks + kBcChunks - 1) / kBcChunks;
    geo.seg_chunks = n_chunks / geo.n_segs;
    geo.n_longer = n_chunks % geo.n_segs;
}
static_assert(kBcSub * 4 + 1 >= 2 * 16 && kBcSub * 5 >= 2 * (16 + 2), "a segment's place");

// Where a channel per lane is ahead of positions in lanes (scan_bwd_states_kernel).  That one works in passes of 256 positions, and a few
// images of one or two passes are done before two more kernels have been launched here; many of them or longer rows fill the chip either way,
// and this kernel has half the instructions per (position, state).  us, positions / channels in lanes, wavefronts of whole rows in front (bf16: 16 states, 12: 196 positions 20 / 44,
// 400 36 / 46, 576 51 / 46, 3136 202 / 65; 192: 56 31 / 25, 196 44 / 48, 400 74 / 70, 784 140 / 110; 768: 56 76 / 27, 196 109 / 83, 784 422 / 224; 8 states, 1536: 196 99 / 87;
// 512 of two wavefronts per workgroup (32 channels), in fp32: 130 48 / 45, 1225 209 / 227).  8 states on 209 to 256 positions, nearly whole passes over there (225 and 255): bf16, 648 wavefronts 80 / 69,
// 81 / 73, 960 105 / 84, 107 / 89, 1536 105 / 100, 107 / 108, 3072 201 / 179, 205 / 200; fp32, 1536 94 / 111, 96 / 121, 3072 188 / 196, 182 / 217.  Of 4 states a lane has one, and the work per position is as much as that per state (192: 784 73 / 51;
// 768: 56 28 / 17, 196 41 / 46, 784 132 / 133; 1536: 400 114 / 127).
//
// 8 states on more than 256 positions, many wavefronts: the other kernel's time depends on how well its grid (1024 workgroups at a time) and its passes are filled, by up to 1.5
// (fp32, 1024 positions: 1152 wavefronts 433 us, 1536 419).  Full, it is ahead (fp32, 768: 1024 222 / 211, 1369 342 / 399, 2304 503 / 558; 1536: 484 201 / 198, 1024 419 / 463, 1369 634 / 783; 3072: 484 390 / 519;
// bf16, 1536: 484 214 / 198, 961 472 / 488; 3072: 484 393 / 448, 961 894 / 976), and not where a third of it waits (fp32, 1152: 1024 433 / 357, 2304 995 / 830; 1536: 784 412 / 384; 3072: 784 795 / 738).
static bool bwd_chan_pays(const ScanBwdArgs &a, int in_size, bool others_full) {
    const int64_t units = (int64_t)a.batch * (a.dim / a.dim_per_group) * ((a.dim_per_group + kBcChan - 1) / kBcChan);
    if (a.N == 4) return a.L > 256 ? units <= 192 : a.L <= 96 && units >= 512;
    if (a.dim_per_group < 48 && a.L > 96 && (a.L < 512 || units > 192)) return false;
    if (a.N == 8 && a.L > 256 && others_full && (in_size == 4 ? units >= 768 && units * a.L >= 1 << 20 : units >= 2048)) return false;
    if (a.L >= 512) return true;
    return units >= (a.L > 256 ? 192 : a.L > 128 ? 640 : 256) && (a.N == 16 || a.L <= 208 || a.L > 256 || in_size == 2);
}

// False: no grid for it.
static bool bwd_chan_geom(const ScanBwdArgs &a, BwdChanGeom &geo, uint32_t &n_wg) {
    geo = {};
    bwd_chan_segments(a.L, geo);
    const int64_t groups = a.dim / a.dim_per_group;
    geo.n_cb = (a.dim_per_group + 63) / 64;
    const int64_t n = (int64_t)a.batch * groups * geo.n_cb * geo.n_segs;
    if (n > 0x7fffffff) return false;
    geo.div_cb = make_fastdiv((uint32_t)geo.n_cb);
    geo.div_groups = make_fastdiv((uint32_t)groups);
    geo.div_segs = make_fastdiv((uint32_t)geo.n_segs);
    n_wg = (uint32_t)n;
    return true;
}

bool scan_bwd_chan_takes(const ScanBwdArgs &a, int in_size, int dy_size, bool others_full) {
    BwdChanGeom geo;
    uint32_t n_wg;
    if ((a.N != 4 && a.N != 8 && a.N != 16) || a.dim_per_group < kBcChan || !bwd_chan_pays(a, in_size, others_full) || !bwd_chan_geom(a, geo, n_wg)) return false;
    // the gradients' memory holds the segments' states between the passes
    auto apart = [&](const void *x, int64_t elems, int size) {
        const uintptr_t first = reinterpret_cast<uintptr_t>(x), last = first + (uintptr_t)(elems * size);
        for (const void *out : {a.du, a.ddelta}) {
            const uintptr_t from = reinterpret_cast<uintptr_t>(out), to = from + (uintptr_t)((int64_t)a.batch * a.dim * a.L * in_size);
            if (first < to && from < last) return false;
        }
        return true;
    };
    const int64_t groups = a.dim / a.dim_per_group, delta_dim = a.dim / a.dim_per_delta;
    for (int64_t s : {a.u_bs, a.u_ds, a.dl_bs, a.dl_ds, a.do_bs, a.do_ds, a.B_bs, a.B_gs, a.B_ns, a.C_bs, a.C_gs, a.C_ns})
        if (s < 0) return false;
    const int64_t most = kNowhere / 2 / 4;                  // a wavefront's rows within 32-bit byte offsets
    for (int64_t s : {a.u_ds, a.dl_ds, a.do_ds, (int64_t)a.L})
        if ((kBcChan - 1) * s + a.L > most) return false;
    for (int64_t s : {a.B_ns, a.C_ns})
        if ((a.N - 1) * s + a.L > most) return false;
    if ((int64_t)a.batch * a.dim * a.N > 0x7fffffff) return false;
    return apart(a.u, (a.batch - 1) * a.u_bs + (a.dim - 1) * a.u_ds + a.L, in_size) && apart(a.delta, (a.batch - 1) * a.dl_bs + (delta_dim - 1) * a.dl_ds + a.L, in_size) &&
           apart(a.dout, (a.batch - 1) * a.do_bs + (a.dim - 1) * a.do_ds + a.L, dy_size) &&
           apart(a.B, (a.batch - 1) * a.B_bs + (groups - 1) * a.B_gs + (a.N - 1) * a.B_ns + a.L, in_size) &&
           apart(a.C, (a.batch - 1) * a.C_bs + (groups - 1) * a.C_gs + (a.N - 1) * a.C_ns + a.L, in_size);
}

template <typename in_t, typename dy_t, int kSpw, bool kDwords>
static int launch_bwd_chan(const ScanBwdArgs &a, hipStream_t stream) {
    BwdChanGeom geo;
    uint32_t n;
    if (!bwd_chan_geom(a, geo, n)) return SS2D_ENOTSUP;
    if (geo.n_segs > 1) {
        const uint32_t n_items = (uint32_t)((int64_t)a.batch * a.dim * a.N);
        hipLaunchKernelGGL((scan_bwd_chan_kernel<in_t, dy_t, kSpw, kDwords, false>), dim3(n), dim3(kBlock), 0, stream, a, geo);
        hipLaunchKernelGGL((scan_bwd_chan_carry_kernel<in_t>), dim3((n_items + kBlock - 1) / kBlock, 2), dim3(kBlock), 0, stream, a, geo.seg_chunks, geo.n_longer, geo.n_segs, n_items,
                           make_fastdiv((uint32_t)a.N), make_fastdiv((uint32_t)a.dim));
    }
    hipLaunchKernelGGL((scan_bwd_chan_kernel<in_t, dy_t, kSpw, kDwords, true>), dim3(n), dim3(kBlock), 0, stream, a, geo);
    return launch_status();
}

template <typename in_t, typename dy_t, bool kDwords>
static int launch_bwd_chan_typed(const ScanBwdArgs &a, hipStream_t stream) {
    switch (a.N) {
        case 4: return launch_bwd_chan<in_t, dy_t, 1, kDwords>(a, stream);
        case 8: return launch_bwd_chan<in_t, dy_t, 2, kDwords>(a, stream);
        default: return launch_bwd_chan<in_t, dy_t, 4, kDwords>(a, stream);
    }
}

int launch_scan_bwd_chan(const ScanBwdArgs &a, int in_dtype, int dout_dtype, hipStream_t stream) {
    if (in_dtype == SS2D_F32) return launch_bwd_chan_typed<float, float, true>(a, stream);
    bool dwords = a.L % 2 == 0;                             // every row starts on a dword
    for (const void *ptr : {a.u, a.delta, a.B, a.C, (const void *)a.du, (const void *)a.ddelta}) dwords = dwords && reinterpret_cast<uintptr_t>(ptr) % 4 == 0;
    for (int64_t s : {a.u_bs, a.u_ds, a.dl_bs, a.dl_ds, a.B_bs, a.B_gs, a.B_ns, a.C_bs, a.C_gs, a.C_ns}) dwords = dwords && s % 2 == 0;
    if (dout_dtype != SS2D_F32) dwords = dwords && reinterpret_cast<uintptr_t>(a.dout) % 4 == 0 && a.do_bs % 2 == 0 && a.do_ds % 2 == 0;
#define SS2D_BWD_CHAN(T)                                                                                                                   \
    do {                                                                                                                                   \
        if (dout_dtype == SS2D_F32) return dwords ? launch_bwd_chan_typed<T, float, true>(a, stream) : launch_bwd_chan_typed<T, float, false>(a, stream); \
        return dwords ? launch_bwd_chan_typed<T, T, true>(a, stream) : launch_bwd_chan_typed<T, T, false>(a, stream);                       \
    } while (0)
    if (in_dtype == SS2D_BF16) SS2D_BWD_CHAN(bf16_t);
    SS2D_BWD_CHAN(f16_t);
#undef SS2D_BWD_CHAN
}

}  // namespace ss2d
