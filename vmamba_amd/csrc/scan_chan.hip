// Selective-scan forward for several states per channel (d_state 4 / 8 / 16 / 32): one CHANNEL per lane, walked
// serially along the sequence.
//
// With N states the work per position is N recurrences  h_n = a_n h_n + B_n du,  y += C_n h_n.  The wavefront-scan
// kernels (selective_scan.hip) pay a 64-lane DPP scan per (512 positions, state).  Here a lane is one channel of one (image, group)
// and a quarter of its states, and the recurrence is a plain serial chain per lane -- multiply, exp2, multiply, two fused multiply-adds
// per (position, state) -- with no scan and no carry logic.
//
// A wavefront owns 16 channels: lane = channel % 4 + 4 set + 16 (channel / 4), the four sets sharing out the states.  It meets no other
// wavefront: its LDS tiles are its own and there is no workgroup barrier.  Per step of 32 positions:
//   stage    lane (row r = lane / 4, quarter q) loads 2 x 4 positions of u and delta of channel r (requested a step ahead), computes
//            dl = softplus(delta + bias), du = dl u and the skip term D u, and writes dl / du into LDS tiles [channel][position] -- the
//            transposition that lets global accesses run along the sequence while the compute phase reads along channels;
//   compute  twice 16 positions: B and C of all states go to LDS as fp32 (requested 32 positions ahead) and are read back as 16-byte
//            broadcasts; the four sets' sums meet in DPP additions that leave 4 positions with each set (sum_over_sets);
//   output   through the dl tile back to lane (r, q), which adds the skip term and stores.
// What bounds it: vector issue.  64 maps of 192 x 56 x 56 as four directions, 16 states: 624 us, 98 % of it issuing, at 4.8 cycles per vector
// instruction and 1.9 GHz; 6.7 instructions per (position, state) of which the recurrence is 5 with one exp2 at 8 cycles.  A workgroup of 64
// channels whose wavefronts share out the states and meet at four barriers per step, B and C in scalar registers (a fused multiply-add
// with a scalar operand takes twice the cycles): 641; 16 images of 192 x 28 x 28: 90, now 68, as there are four times as many wavefronts
// as blocks of 64 channels and each is done on its own.
//
// Few wavefronts (small batches) leave the chip idle behind that serial chain.  Their rows are cut into segments that run side by side
// in two launches of the same kernel, with one between them that walks the segments (ChanPhase, chan_segments): what a segment leaves
// from state 0, its sum of dl and its largest dl; what enters each, h_in' = exp2(A sum dl) h_in + h; the outputs from there.
#include "scan_common.h"

namespace ss2d {

constexpr int kChanTile = 32;                     // positions staged per step
constexpr int kChanSub = 16;                      // positions per compute / combine round
constexpr int kChanTilePitch = kChanTile + 4;     // floats; + 4 spreads the 16-byte reads of 8 lanes over all banks
constexpr int kChanSubPitch = kChanSub + 4;
constexpr int kChanBlock = 16;                    // channels per wavefront
constexpr int kChanSets = 4;                      // lanes per channel, each with a quarter of the states

// Four elements from byte offset `off` on (a dword's, kDwords), the first n of them where not all lie inside the row.
template <typename out_t, bool kDwords>
__device__ __forceinline__ void store4(__amdgpu_buffer_rsrc_t rsrc, uint32_t off, bool whole, int n, const float (&v)[4]) {
    typedef uint32_t words4_t __attribute__((ext_vector_type(4)));
    typedef uint32_t words2_t __attribute__((ext_vector_type(2)));
    if (whole && (kDwords || sizeof(out_t) == 4)) {
        const int at = (int)(n > 0 ? off : kNowhere);
        if constexpr (sizeof(out_t) == 4) {
            const words4_t w = {f32_to_bits(v[0]), f32_to_bits(v[1]), f32_to_bits(v[2]), f32_to_bits(v[3])};
            __builtin_amdgcn_raw_buffer_store_b128(w, rsrc, at, 0, 0);
        } else {
            const words2_t w = {pack2_from_f32<out_t>(v[0], v[1]), pack2_from_f32<out_t>(v[2], v[3])};
            __builtin_amdgcn_raw_buffer_store_b64(w, rsrc, at, 0, 0);
        }
    } else {
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const int at = (int)(i < n ? off + i * (uint32_t)sizeof(out_t) : kNowhere);
            if constexpr (sizeof(out_t) == 4) __builtin_amdgcn_raw_buffer_store_b32(f32_to_bits(v[i]), rsrc, at, 0, 0);
            else __builtin_amdgcn_raw_buffer_store_b16((uint16_t)(pack2_from_f32<out_t>(v[i & ~1], v[i | 1]) >> (i & 1) * 16), rsrc, at, 0, 0);
        }
    }
}

struct ChanGeom {
    uint32_t n_units;        // wavefronts
    int32_t n_cb;            // channel blocks per group
    FastDiv div_cb, div_groups;
    int32_t seg_len, n_segs;                 // of a row cut into segments (kLocal, kRest)
    FastDiv div_segs;                        // segments of a row that this launch walks
};

// A row as a whole, or cut into segments: what a segment leaves from state 0, then its outputs from the state that enters it.
enum ChanPhase { kWhole, kLocal, kRest };

// Wavefronts per SIMD to leave registers for.  Four with four states, but for the forms that would then keep 12 to 60 bytes a lane in memory (in single precision with
// CrossScan folded in or a state that enters; off the dword grid with chunk-end states as well): us with four / three, fp32, 64 x 96 maps of 56 x 56 folded in 300 / 246,
// 16 x 96 rows of 3136 cut 89 / 84, with chunk-end states 116 / 84.
template <typename in_t, int kSpw, bool kX, bool kMaps, int kPhase, bool kDwords> constexpr int chan_waves() {
    if (kSpw != 1) return kSpw == 8 ? 2 : 3;
    return (kMaps || kPhase == kRest) && (sizeof(in_t) == 4 || (!kDwords && kX)) ? 3 : 4;
}

// kX: the chunk-end states are written as well -- x[row][chunk][2n] = product of a_n since the row's start,
// x[..][2n + 1] = h_n, after every 2048 positions and at the row's end.  h is what the lane holds; the product is
// exp2(A_n log2e * sum dl), and the sum is per CHANNEL, not per state: each of a channel's four lanes adds up a quarter of
// every round's positions (one LDS read, four adds per 16 positions) and the quarters meet when a chunk ends.
//
// kMaps: CrossScan folded in.  u is not the (batch, 4 D, L) tensor of the four scan-ordered copies but the map itself,
// x (batch, D, L), plus its transpose xt (batch, D, L: every H x W map stored as W x H): direction k = the channel's
// group reads x (k = 0, 2) or xt (k = 1, 3), forwards (k < 2) or backwards -- position t of the scan is element t or
// L - 1 - t of that row (cross_scan_fwd, classification/models/csm_triton.py:22-29).  A lane's four positions are then
// the four elements that END at L - 1 - t, taken in reverse; where fewer are left, the row's first four.
//
// kDwords: the rows of 16-bit inputs start on dwords (RawGroup).
template <typename in_t, typename out_t, int kSpw, bool kSoftplus, bool kX, bool kMaps, int kPhase, bool kDwords>
__global__ __launch_bounds__(kBlock, (chan_waves<in_t, kSpw, kX, kMaps, kPhase, kDwords>())) void scan_chan_kernel(const in_t *__restrict__ u_all, const in_t *__restrict__ dl_all,
                                                           const in_t *__restrict__ B_all, const in_t *__restrict__ C_all,
                                                           const float *__restrict__ A_all, out_t *__restrict__ o_all,
                                                           const ScanArgs p, const ChanGeom geo,
                                                           const in_t *__restrict__ ut_all = nullptr) {
    constexpr int kBcRows = 2 * kChanSets * kSpw;                                       // [B, C][state of the lane][set]
    __shared__ __align__(16) float s_dl_all[kWavesPerWg * kChanBlock * kChanTilePitch]; // later: the outputs
    __shared__ __align__(16) float s_du_all[kWavesPerWg * kChanBlock * kChanTilePitch];
    __shared__ __align__(16) float s_bc_all[kWavesPerWg * kBcRows * kChanSubPitch];

    const int lane = threadIdx.x & (kWave - 1);
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave);
    float *s_dl = s_dl_all + wave * kChanBlock * kChanTilePitch, *s_du = s_du_all + wave * kChanBlock * kChanTilePitch;
    float *s_bc = s_bc_all + wave * kBcRows * kChanSubPitch;
    // neighbouring wavefronts are the channel blocks of one (image, group) and read the same B / C rows: keep them
    // on one XCD (one L2)
    uint32_t unit = xcd_contiguous_id(blockIdx.x, gridDim.x) * kWavesPerWg + wave;
    if (unit >= geo.n_units) return;                        // whole wavefronts; no workgroup barrier in this kernel
    uint32_t bg, cb, b, grp, seg = 0;
    if constexpr (kPhase != kWhole) divmod(unit, geo.div_segs, unit, seg);
    divmod(unit, geo.div_cb, bg, cb);
    divmod(bg, geo.div_groups, b, grp);
    const int L = p.L, dpg = p.dim_per_group;
    const int begin = kPhase == kWhole ? 0 : (int)seg * geo.seg_len;           // (a multiple of kChanTile)
    const int stop = kPhase == kWhole || (int)seg + 1 == geo.n_segs ? L : begin + geo.seg_len;

    // ---- staging / output role: row r, quarter q -------------------------------------------------------------------
    const int r = lane >> 2, q = lane & 3;
    const int c_first = (int)cb * kChanBlock, n_chan = min(kChanBlock, dpg - c_first);
    const int d_first = (int)grp * dpg + c_first, ds = d_first + min(r, n_chan - 1);
    const int dg_first = d_first / p.dim_per_delta, dgs = ds / p.dim_per_delta;
    const in_t *u_first = u_all + (int64_t)b * p.u_bs + (int64_t)d_first * p.u_ds;
    bool u_rev = false;                                     // kMaps: uniform over the wavefront (one group = one direction)
    if constexpr (kMaps) {
        const int Dm = p.dim >> 2, k = d_first / Dm;
        u_first = ((k & 1) ? ut_all : u_all) + (int64_t)b * p.u_bs + (int64_t)(d_first - k * Dm) * p.u_ds;
        u_rev = k >= 2;
    }
    uint32_t u_row, dl_row, B_row, C_row;                   // the element a lane's row starts at
    const auto u_buf = dwords_of<in_t>(u_first, 0, n_chan, p.u_ds, L, u_row);
    const auto dl_buf = dwords_of<in_t>(dl_all, (int64_t)b * p.dl_bs + (int64_t)dg_first * p.dl_ds, (d_first + n_chan - 1) / p.dim_per_delta - dg_first + 1, p.dl_ds, L, dl_row);
    const auto o_buf = rows_of<out_t>(o_all, (int64_t)b * p.o_bs + (int64_t)d_first * p.o_ds, n_chan, p.o_ds, L);
    const uint32_t o_row = (uint32_t)((ds - d_first) * p.o_ds);
    u_row += (uint32_t)((ds - d_first) * p.u_ds);
    dl_row += (uint32_t)((dgs - dg_first) * p.dl_ds);
    using Four = RawGroup<in_t, 4, kDwords>;
    // four positions of u from position pos of the scan on, as they lie in memory: backwards these are the four elements
    // that end at L - 1 - pos, and they are put in scan order where they are widened (unpack_u) -- not here, which
    // would make the wavefront wait for a load it has just issued for the NEXT step
    auto first_of = [&](int pos) { return kMaps && u_rev ? max(L - 4 - pos, 0) : pos; };
    auto load_u = [&](int pos) { return load_at<in_t, 4, kDwords>(u_buf, u_row, first_of(pos), L, pos < L); };
    auto load_dl = [&](int pos) { return load_at<in_t, 4, kDwords>(dl_buf, dl_row, pos, L); };
    auto unpack_u = [&](const Four &raw, int pos, float (&v)[4]) {
        float m[4];
        widen<in_t, 4, kDwords>(raw, u_row + (uint32_t)first_of(pos), m);
#pragma unroll
        for (int i = 0; i < 4; ++i) v[i] = m[i];
        if constexpr (kMaps) {
            if (u_rev) {
#pragma unroll
                for (int i = 0; i < 4; ++i) v[i] = m[3 - i];
                if (L % 4 != 0 && pos + 4 > L) {            // the row's first elements, of which fewer are left
                    const int skip = pos + 4 - L;
#pragma unroll
                    for (int i = 0; i < 3; ++i) {
                        float at = v[i];
#pragma unroll
                        for (int k = 1; k < 4 - i; ++k) at = skip == k ? m[3 - i - k] : at;
                        v[i] = at;
                    }
                }
            }
        }
    };
    const float bias_s = p.bias ? p.bias[dgs] : 0.0f;
    const float D_s = p.D ? p.D[ds] : 0.0f;
    float *st_dl = s_dl + r * kChanTilePitch + 4 * q;
    float *st_du = s_du + r * kChanTilePitch + 4 * q;
    // B / C: four positions of a row per lane and piece, rows [B, C][state of the lane][set]
    constexpr int kBcPieces = kSpw > 4 ? kSpw / 4 : 1;      // of each
    const bool bc_mine = kSpw >= 4 || lane < 16 * kSpw;
    const auto B_buf = dwords_of<in_t>(B_all, (int64_t)b * p.B_bs + (int64_t)grp * p.B_gs, kChanSets * kSpw, p.B_ns, L, B_row);
    const auto C_buf = dwords_of<in_t>(C_all, (int64_t)b * p.C_bs + (int64_t)grp * p.C_gs, kChanSets * kSpw, p.C_ns, L, C_row);
    uint32_t B_rows[kBcPieces], C_rows[kBcPieces];
#pragma unroll
    for (int k = 0; k < kBcPieces; ++k) {
        const int n = (r & 3) * kSpw + (r >> 2) + 4 * k;    // row r + 16 k of the array: state r / 4 + 4 k of set r % 4
        B_rows[k] = B_row + (uint32_t)(n * p.B_ns);
        C_rows[k] = C_row + (uint32_t)(n * p.C_ns);
    }
    auto load_bc = [&](int t, Four (&raw)[2 * kBcPieces]) {
#pragma unroll
        for (int k = 0; k < kBcPieces; ++k) {
            raw[k] = load_at<in_t, 4, kDwords>(B_buf, B_rows[k], t + 4 * q, L, bc_mine);
            if constexpr (kPhase != kLocal) raw[kBcPieces + k] = load_at<in_t, 4, kDwords>(C_buf, C_rows[k], t + 4 * q, L, bc_mine);
        }
    };
    float *st_bc = s_bc + r * kChanSubPitch + 4 * q;

    // ---- compute role: a channel, states set * kSpw .. + kSpw ------------------------------------------------
    const int ch = (lane >> 4) * 4 + (lane & 3), set = (lane >> 2) & 3;
    const int dc = d_first + min(ch, n_chan - 1);
    float A2[kSpw], h[kSpw];
#pragma unroll
    for (int j = 0; j < kSpw; ++j) {
        A2[j] = A_all[(int64_t)dc * p.A_ds + (int64_t)(set * kSpw + j) * p.A_ns] * kLog2e;
        h[j] = 0.0f;
    }
    const float *my_bc = s_bc + set * kChanSubPitch;
    float *my_dl = s_dl + ch * kChanTilePitch;
    const float *my_du = s_du + ch * kChanTilePitch;
    float dl_sum = 0.0f;                                    // kX: this lane's quarter of the channel's sum of dl
    float dl_max = 0.0f;                                    // kLocal: its largest
    const bool chan_ok = ch < n_chan;
    float *x_lane = kX ? p.x + ((int64_t)b * p.dim + dc) * p.n_chunks * 2 * p.N + 2 * (set * kSpw) : nullptr;
    auto over_sets = [&](float v) { v += __shfl_xor(v, 4, kWave); return v + __shfl_xor(v, 8, kWave); };

    // a segment's states, its sum of dl, (from the carry kernel) that of all before it and its largest dl, where its outputs will be
    uint8_t *seg_state = reinterpret_cast<uint8_t *>(o_all + (int64_t)b * p.o_bs + (int64_t)dc * p.o_ds + begin);
    if constexpr (kPhase == kRest) {
        if (seg > 0) {
            __builtin_memcpy(h, seg_state + sizeof(float) * (set * kSpw), sizeof(h));
            if (kX && set == 0) __builtin_memcpy(&dl_sum, seg_state + sizeof(float) * (p.N + 1), sizeof(dl_sum));
        }
    }
    Four ru[2], rd[2], rbc[2][2 * kBcPieces];
#pragma unroll
    for (int s = 0; s < 2; ++s) {
        ru[s] = load_u(begin + s * kChanSub + 4 * q);
        rd[s] = load_dl(begin + s * kChanSub + 4 * q);
    }
    // requested in the order in which a step does: what the compiler waits for is then a count of younger requests, not all
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int s = 0; s < 2; ++s) load_bc(begin + s * kChanSub, rbc[s]);
    __builtin_amdgcn_sched_barrier(0);

    for (int t0 = begin; t0 < stop; t0 += kChanTile) {
        // ---- stage: dl, du into LDS; the skip term stays with this lane -----------------------------------------------
        float skip[2][4];
#pragma unroll
        for (int s = 0; s < 2; ++s) {
            float uv[4], raw[4], dl[4], du[4];
            unpack_u(ru[s], t0 + s * kChanSub + 4 * q, uv);
            widen<in_t, 4, kDwords>(rd[s], dl_row, raw);
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                dl[i] = kSoftplus ? softplus_log2(fmaf(raw[i], kLog2e, bias_s * kLog2e)) : raw[i] + bias_s;
            }
            if (t0 + kChanTile > L) {                       // uniform; past the row's end 0, the identity of the recurrence
#pragma unroll
                for (int i = 0; i < 4; ++i) {
                    const bool in_row = t0 + s * kChanSub + 4 * q + i < L;
                    dl[i] = in_row ? dl[i] : 0.0f;
                    uv[i] = in_row ? uv[i] : 0.0f;
                }
            }
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                du[i] = dl[i] * uv[i];
                skip[s][i] = D_s * uv[i];
            }
            *reinterpret_cast<float4 *>(st_dl + s * kChanSub) = make_float4(dl[0], dl[1], dl[2], dl[3]);
            *reinterpret_cast<float4 *>(st_du + s * kChanSub) = make_float4(du[0], du[1], du[2], du[3]);
        }
        // the next step's inputs travel while this step computes (after the last step of a segment: not used)
#pragma unroll
        for (int s = 0; s < 2; ++s) {
            ru[s] = load_u(t0 + kChanTile + s * kChanSub + 4 * q);
            rd[s] = load_dl(t0 + kChanTile + s * kChanSub + 4 * q);
        }
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int s = 0; s < 2; ++s) {
            const int ps = t0 + s * kChanSub;
            // ---- compute: 16 positions of every lane's states -----------------------------------------------------------
#pragma unroll
            for (int k = 0; k < (kPhase == kLocal ? 1 : 2) * kBcPieces; ++k) {
                float v[4];
                widen<in_t, 4, kDwords>(rbc[s][k], k < kBcPieces ? B_rows[k % kBcPieces] : C_rows[k % kBcPieces], v);
                if (L % 4 != 0 && ps + kChanSub > L) {      // uniform; four elements that the row's end divides
#pragma unroll
                    for (int i = 1; i < 4; ++i) v[i] = ps + 4 * q + i < L ? v[i] : 0.0f;
                }
                const int at = (k / kBcPieces) * kChanSets * kSpw + (k % kBcPieces) * 16;
                if (bc_mine) *reinterpret_cast<float4 *>(st_bc + at * kChanSubPitch) = make_float4(v[0], v[1], v[2], v[3]);
            }
            load_bc(ps + kChanTile, rbc[s]);
            __builtin_amdgcn_sched_barrier(0);
            wave_lds_sync();                                // dl / du of this step, B / C of this round are in place
            if (s > 0 && ps >= L) break;                    // uniform; no memory request is behind it
            float dl[kChanSub], du[kChanSub], y[kChanSub];
#pragma unroll
            for (int v = 0; v < kChanSub / 4; ++v) {
                const float4 a4 = *reinterpret_cast<const float4 *>(my_dl + s * kChanSub + 4 * v);
                const float4 b4 = *reinterpret_cast<const float4 *>(my_du + s * kChanSub + 4 * v);
                dl[4 * v] = a4.x; dl[4 * v + 1] = a4.y; dl[4 * v + 2] = a4.z; dl[4 * v + 3] = a4.w;
                du[4 * v] = b4.x; du[4 * v + 1] = b4.y; du[4 * v + 2] = b4.z; du[4 * v + 3] = b4.w;
            }
#pragma unroll
            for (int i = 0; i < kChanSub; ++i) y[i] = 0.0f;
            if constexpr (kX || kPhase == kLocal) {
                const float4 q4 = *reinterpret_cast<const float4 *>(my_dl + s * kChanSub + 4 * set);
                dl_sum += (q4.x + q4.y) + (q4.z + q4.w);      // (dl is 0 past the row's end)
                if constexpr (kPhase == kLocal) dl_max = fmaxf(fmaxf(dl_max, fmaxf(q4.x, q4.y)), fmaxf(q4.z, q4.w));
            }
#pragma unroll
            for (int j = 0; j < kSpw; ++j) {
                float Bv[kChanSub], Cv[kChanSub];
#pragma unroll
                for (int v = 0; v < kChanSub / 4; ++v) {
                    const float4 b4 = *reinterpret_cast<const float4 *>(my_bc + j * kChanSets * kChanSubPitch + 4 * v);
                    const float4 c4 = *reinterpret_cast<const float4 *>(my_bc + (kSpw + j) * kChanSets * kChanSubPitch + 4 * v);
                    Bv[4 * v] = b4.x; Bv[4 * v + 1] = b4.y; Bv[4 * v + 2] = b4.z; Bv[4 * v + 3] = b4.w;
                    Cv[4 * v] = c4.x; Cv[4 * v + 1] = c4.y; Cv[4 * v + 2] = c4.z; Cv[4 * v + 3] = c4.w;
                }
                float hj = h[j];
#pragma unroll
                for (int i = 0; i < kChanSub; ++i) {
                    hj = fmaf(__builtin_amdgcn_exp2f(dl[i] * A2[j]), hj, Bv[i] * du[i]);
                    if constexpr (kPhase != kLocal) y[i] = fmaf(Cv[i], hj, y[i]);
                }
                h[j] = hj;
            }
            wave_lds_sync();                                // dl / du, B / C of this round are read
            if constexpr (kPhase != kLocal) {
                // the four sets' sums: positions 4 set .. + 4 of the lane's channel, into the place of the dl read above
                sum_over_quads(y);
                *reinterpret_cast<float4 *>(my_dl + s * kChanSub + 4 * set) = make_float4(y[0], y[1], y[2], y[3]);
            }
        }
        if constexpr (kPhase != kLocal) {
            // ---- output: 4 positions of row r, twice -----------------------------------------------------------------
            wave_lds_sync();
#pragma unroll
            for (int s = 0; s < 2; ++s) {
                const float4 part = *reinterpret_cast<const float4 *>(st_dl + s * kChanSub);
                const float acc[4] = {skip[s][0] + part.x, skip[s][1] + part.y, skip[s][2] + part.z, skip[s][3] + part.w};
                const int pos = t0 + s * kChanSub + 4 * q;
                store4<out_t, kDwords>(o_buf, (o_row + (uint32_t)pos) * (uint32_t)sizeof(out_t), L % 4 == 0 || t0 + kChanTile <= L, r < n_chan ? L - pos : 0, acc);
            }
            wave_lds_sync();
        }
        if constexpr (kX) {
            const int t_end = t0 + kChanTile;
            if (t_end % SS2D_SCAN_CHUNK == 0 || t_end >= L) {   // uniform; at least 64 steps apart
                const float total = over_sets(dl_sum);
                if (chan_ok) {
                    float *xo = x_lane + (int64_t)((min(t_end, L) - 1) / SS2D_SCAN_CHUNK) * 2 * p.N;
#pragma unroll
                    for (int j = 0; j < kSpw; ++j) {
                        xo[2 * j] = __builtin_amdgcn_exp2f(A2[j] * total);
                        xo[2 * j + 1] = h[j];
                    }
                }
            }
        }
    }
    if constexpr (kPhase == kLocal) {
        const float total = over_sets(dl_sum);
        const float pair = fmaxf(dl_max, __shfl_xor(dl_max, 4, kWave)), most = fmaxf(pair, __shfl_xor(pair, 8, kWave));
        if (!chan_ok) return;
        __builtin_memcpy(seg_state + sizeof(float) * (set * kSpw), h, sizeof(h));
        if (set == 0) {
            __builtin_memcpy(seg_state + sizeof(float) * p.N, &total, sizeof(total));
            __builtin_memcpy(seg_state + sizeof(float) * (p.N + 2), &most, sizeof(most));
        }
    }
}

// What enters every segment but the first, in the place of what the segment left: a thread per (row, state).
template <typename out_t>
__global__ __launch_bounds__(kBlock) void scan_chan_carry_kernel(const float *__restrict__ A_all, out_t *o_all, const ScanArgs p, int seg_len, int n_segs,
                                                                 uint32_t n_items, FastDiv div_n, FastDiv div_dim) {
    const uint32_t item = blockIdx.x * kBlock + threadIdx.x;
    if (item >= n_items) return;
    uint32_t row, n, b, d;
    divmod(item, div_n, row, n);
    divmod(row, div_dim, b, d);
    const float A2 = A_all[(int64_t)d * p.A_ds + (int64_t)n * p.A_ns] * kLog2e;
    uint8_t *state = reinterpret_cast<uint8_t *>(o_all + (int64_t)b * p.o_bs + (int64_t)d * p.o_ds);
    const int64_t pitch = (int64_t)seg_len * sizeof(out_t);
    float carry = 0.0f, before = 0.0f;
    constexpr int kFly = 8;
    for (int first = 0; first < n_segs; first += kFly) {
        float left[kFly], sum[kFly], most[kFly];
#pragma unroll
        for (int i = 0; i < kFly; ++i) {                    // (past the last but one segment: that one again, not used)
            const uint8_t *from = state + min(first + i, n_segs - 2) * pitch;
            __builtin_memcpy(&left[i], from + sizeof(float) * n, sizeof(float));
            __builtin_memcpy(&sum[i], from + sizeof(float) * p.N, sizeof(float));
            __builtin_memcpy(&most[i], from + sizeof(float) * (p.N + 2), sizeof(float));
        }
#pragma unroll
        for (int i = 0; i < kFly; ++i) {
            const int s = first + i;
            if (s >= n_segs) break;
            if (s > 0) {
                __builtin_memcpy(state + s * pitch + sizeof(float) * n, &carry, sizeof(float));
                if (n == 0) __builtin_memcpy(state + s * pitch + sizeof(float) * (p.N + 1), &before, sizeof(float));
            }
            before += sum[i];
            // the product of the segment's a in two halves, so that neither leaves fp32's range before the state would; none of 0, and none of an
            // infinite state: it stays infinite unless one of the a is 0 (the one of the largest dl, where A is negative), which leaves NaN
            const float half = __builtin_amdgcn_exp2f(0.5f * A2 * sum[i]);
            if (fabsf(carry) == __builtin_inff()) carry = __builtin_amdgcn_exp2f(A2 * most[i]) > 0.0f ? carry + left[i] : __builtin_nanf("");
            else carry = carry == 0.0f ? left[i] : fmaf(carry * half, half, left[i]);
        }
    }
}

// Rows of whole 16-byte pieces and 8 positions are this kernel's at any size.  Others were the flat kernel's or element by element (16 states in bf16, 64 x 96 maps of
// 49 positions 93 us, here 12.5; of 225 182, 37; 16 x 192 of 3306 1390, 266).  Of them, what the kernels with positions in lanes are ahead with is left to those: they do a row in
// steps of 256 or 512 positions, each in the same time however few the rows, where a wavefront here walks its row serially.  So few wavefronts on 100 to 1000 positions, the more
// the fewer the states (us, positions / channels in lanes, wavefronts of whole rows in front, bf16: 16 states, 12: 100 positions 12.0 / 12.3, 196 12.1 / 19.9, 324 12.1 / 32.5; 192: 100 17.9 / 12.7,
// 196 18.4 / 20.5, 324 18.4 / 30.8; 384: 196 27.4 / 21.1, 324 27.9 / 31.3; 768: 324 48.2 / 32.6; 4 states, 192: 77 8.1 / 7.3, 196 8.6 / 12.6; 384: 196 11.9 / 13.0, 324 12.1 / 19.2; 768: 324
// 21.0 / 20.1), and longer ones of 8 states (12: 3306 of 4 10.9 / 23.1, 16 states 29.2 / 30.7; 96: 70.5 / 54.1).  Long rows of 4 states only while there is
// no more than one wavefront to a SIMD (or, whole, many), and above two where the last step over there is less than half of one (time here over the time there, bf16, 1152: 625 .83, 961 1.07, 1225 .94, 1681 .96, 2401 1.32; 1536: .66, .85, .75, 1.02,
// 1.13; 2304: .62, 1.21, 1.08, 1.13, 1.23; fp32, 768: 1332 .92, 1764 .97, 3364 1.03; 1152: 1.20, 1.22, 1.22; 3072:
// .97, .96, 2116 .94).
//
// Single precision of an odd number of fours (whole): those kernels read it in whole pieces and are ahead longer, by 1808 measured sizes (time here over the time there; 16 states: 96 wavefronts of
// 68 positions .91, of 100 1.11; 192: 100 .92, 132 1.10; 384: 196 .98; 768: 324 .84; 1152: 484 1.07; 1536: 484 .84; 576: 676 .98, 900 1.12; 768: 900 .88; 8 states, 384: 196 1.17, 576 .85; 4 states, 2304: 324 .85,
// 484 .98, 3072 .77, 1.14; 1152: 1028 .80, 1332 1.20, 3364 1.22).  Beyond 1024 positions on fewer than 768 wavefronts it wins where there are so few of them that rows are cut, and not
// right behind a step of 512 or, from 2048 on, of 2048 (16 states, 24: 1028 1.08, 1332 1.23, 1764 .82, 2116 1.32, 3364 1.30; 32 states: 1.02 at most up to 2048, 1.07, 1.05, 5476 .81).
static bool chan_pays(const ScanArgs &a, bool whole, int in_size, bool maps) {
    if (whole && a.L % 8 == 0) return true;
    const int64_t units = (int64_t)a.batch * (a.dim / a.dim_per_group) * ((a.dim_per_group + kChanBlock - 1) / kChanBlock);
    const int at = a.N == 4 ? 0 : a.N == 8 ? 1 : a.N == 16 ? 2 : 3;
    const int always[4] = {56, 64, whole ? 72 : 104, 104};        // positions up to which a wavefront's walk is as short as a step
    const int per_ten[4] = {36, whole && !maps ? 28 : 27, whole ? 28 : 24, 19};         // wavefronts wanted per 10 positions behind the first ones, up to 512 positions
    constexpr int kFrom[4] = {45, 55, 60, 60};
    const int medium[4] = {1024, 704, whole ? 640 : 576, whole ? 640 : 576};       // wavefronts wanted up to 1024 positions
    if (a.L <= always[at]) return true;
    if (a.N == 4 && !maps && (a.L > 1300 ? units > 1024 && !(whole && units > 2560) : a.L > 512 ? units > 2048 && (a.L - 1) % 512 >= 256 : whole && a.L > 400)) return false;
    if (a.L <= 512) return 10 * units >= (int64_t)per_ten[at] * (a.L - kFrom[at]);
    if (a.L <= 1024) return units >= medium[at];
    if (whole && units < 768) return units <= 48 && (a.N == 16 ? a.L > 1536 && a.L <= 2048 : a.N == 32 && (a.L <= 2048 || a.L > 4096));
    if (a.N == 4) return units >= (in_size == 4 ? 768 : 1024);
    if (a.N == 8) return units >= 576;
    return a.N == 32 || a.L <= 2048 || units >= 64;
}

bool scan_chan_eligible(const ScanArgs &a, bool vec, int in_size, bool maps) {
    // N/4 states per lane; at least two blocks of channels per group; a block's rows within 32-bit byte offsets
    for (int64_t s : {a.u_ds, a.dl_ds, a.o_ds})
        if (s < 0 || (kChanBlock - 1) * s + a.L > kNowhere / 2 / 4) return false;
    for (int64_t s : {a.B_ns, a.C_ns})
        if (s < 0 || (a.N - 1) * s + a.L > kNowhere / 2 / 4) return false;
    // With CrossScan folded in the other kernels' lead on few wavefronts is not worth the four copies and another launch (forward_core of 4 x 128 maps of 19 x 19,
    // 16 states in bf16, 87 us, 106 apart).
    return (a.N == 4 || a.N == 8 || a.N == 16 || a.N == 32) && a.dim_per_group >= 32 && ((maps && a.N >= 16) || chan_pays(a, vec, in_size, maps));
}

// The number of segments of a row (1: not cut) and the length of all but the last, which has at least 72 positions: a segment's N + 3
// floats (the last one's N + 2) lie where its outputs will be.
//
// A wavefront takes 1.3 us per 16 positions of 16 states while it has its SIMD to itself (0.65 of 4 states, 2.1 of 32).  Cut rows run the
// recurrence twice (the first time without C), in three launches, and are ahead while there are not nearly as many wavefronts as SIMDs (1024).
// us, whole / cut, wavefronts of whole rows in front: 16 states in bf16, 16: 3136 positions 249 / 34, 784 65 / 28, 400 35 / 27; 192: 3136 251 / 78,
// 784 66 / 33, 400 35 / 31; 384: 3136 243 / 133, 784 66 / 48, 400 (three segments) 36 / 38; 768: 3136 246 / 245, 784 66 / 72; in fp32, 384: 3136 231 / 139; 4 states,
// 16: 400 18.2 / 17.0; 384: 784 35 / 28, 400 19 / 21; 768: 1568 63 / 68; 32 states in fp16, 384: 784 108 / 74; 768: 784 107 / 115.  More segments than
// kSegPlaces are no faster (384: 3136 positions in 12: 140, in 24: 137), nor are shorter ones than kSegLeast where many run (192: 784 in 6: 33, in 8: 35).
constexpr int64_t kSegPlaces = 4608, kSegUnits = 576, kSegLeast = 128;

static int64_t chan_segments(const ScanArgs &a, int64_t n_units, int32_t &seg_len) {
    if (a.out == a.u || a.out == a.delta || (int64_t)a.batch * a.dim * a.N > 0x7fffffff || n_units > kSegUnits) return 1;
    const int64_t least = n_units <= 64 ? 96 : kSegLeast;
    int64_t n = kSegPlaces / n_units;
    if (n > a.L / least) n = a.L / least;
    if (n < (n_units <= 192 ? 3 : 4)) return 1;
    const int64_t len = ((a.L + n - 1) / n + kChanTile - 1) / kChanTile * kChanTile;
    n = (a.L + len - 1) / len;
    if (a.L - (n - 1) * len < 72) --n;
    seg_len = (int32_t)len;
    return n;
}

template <typename in_t, typename out_t, bool kDwords>
static int launch_chan_typed(const ScanArgs &a, const void *xt, hipStream_t stream) {
    ChanGeom geo = {};
    geo.n_cb = (a.dim_per_group + kChanBlock - 1) / kChanBlock;
    const int groups = a.dim / a.dim_per_group;
    geo.div_cb = make_fastdiv((uint32_t)geo.n_cb);
    geo.div_groups = make_fastdiv((uint32_t)groups);
    const int64_t n_rows = (int64_t)a.batch * groups * geo.n_cb;
    if (n_rows > 0x7fffffff) return SS2D_ENOTSUP;
    geo.n_units = (uint32_t)n_rows;
    auto n_wg = [&] { return dim3((geo.n_units + kWavesPerWg - 1) / kWavesPerWg); };
#define SS2D_LAUNCH_CHAN(SPW, SP, X, M)                                                                                    \
    hipLaunchKernelGGL((scan_chan_kernel<in_t, out_t, SPW, SP, X, M, kWhole, kDwords>), n_wg(), dim3(kBlock), 0, stream,       \
                       (const in_t *)a.u, (const in_t *)a.delta, (const in_t *)a.B, (const in_t *)a.C, a.A, (out_t *)a.out, a, geo, \
                       (const in_t *)xt)
#define SS2D_LAUNCH_CHAN_N(SP, X, M)                            \
    switch (a.N) {                                              \
        case 4: SS2D_LAUNCH_CHAN(1, SP, X, M); break;           \
        case 8: SS2D_LAUNCH_CHAN(2, SP, X, M); break;           \
        case 16: SS2D_LAUNCH_CHAN(4, SP, X, M); break;          \
        default: SS2D_LAUNCH_CHAN(8, SP, X, M); break;          \
    }
#define SS2D_LAUNCH_CHAN_X(SP, M) \
    if (a.x) { SS2D_LAUNCH_CHAN_N(SP, true, M) } else { SS2D_LAUNCH_CHAN_N(SP, false, M) }
#define SS2D_LAUNCH_CHAN_SPLIT(SPW, X, M)                                                                                   \
    do {                                                                                                                   \
        geo.div_segs = make_fastdiv((uint32_t)segs - 1);                                                                    \
        geo.n_units = (uint32_t)(n_rows * (segs - 1));                                                                      \
        hipLaunchKernelGGL((scan_chan_kernel<in_t, out_t, SPW, true, false, M, kLocal, kDwords>), n_wg(), dim3(kBlock), 0, stream, \
                           (const in_t *)a.u, (const in_t *)a.delta, (const in_t *)a.B, (const in_t *)a.C, a.A, (out_t *)a.out, a, geo, (const in_t *)xt); \
        hipLaunchKernelGGL((scan_chan_carry_kernel<out_t>), dim3((n_items + kBlock - 1) / kBlock), dim3(kBlock), 0, stream, a.A, (out_t *)a.out, a, \
                           geo.seg_len, geo.n_segs, n_items, make_fastdiv((uint32_t)a.N), make_fastdiv((uint32_t)a.dim));   \
        geo.div_segs = make_fastdiv((uint32_t)segs);                                                                        \
        geo.n_units = (uint32_t)(n_rows * segs);                                                                            \
        hipLaunchKernelGGL((scan_chan_kernel<in_t, out_t, SPW, true, X, M, kRest, kDwords>), n_wg(), dim3(kBlock), 0, stream, \
                           (const in_t *)a.u, (const in_t *)a.delta, (const in_t *)a.B, (const in_t *)a.C, a.A, (out_t *)a.out, a, geo, (const in_t *)xt); \
    } while (0)
#define SS2D_LAUNCH_CHAN_SPLIT_N(X, M)                          \
    switch (a.N) {                                              \
        case 4: SS2D_LAUNCH_CHAN_SPLIT(1, X, M); break;         \
        case 8: SS2D_LAUNCH_CHAN_SPLIT(2, X, M); break;         \
        case 16: SS2D_LAUNCH_CHAN_SPLIT(4, X, M); break;        \
        default: SS2D_LAUNCH_CHAN_SPLIT(8, X, M); break;        \
    }
    const int64_t segs = a.softplus ? chan_segments(a, n_rows, geo.seg_len) : 1;
    if (segs > 1) {
        geo.n_segs = (int32_t)segs;
        const uint32_t n_items = (uint32_t)((int64_t)a.batch * a.dim * a.N);
        if (a.x) {
            if (xt) { SS2D_LAUNCH_CHAN_SPLIT_N(true, true) } else { SS2D_LAUNCH_CHAN_SPLIT_N(true, false) }
        } else {
            if (xt) { SS2D_LAUNCH_CHAN_SPLIT_N(false, true) } else { SS2D_LAUNCH_CHAN_SPLIT_N(false, false) }
        }
        return launch_status();
    }
    if (xt) {
        if (a.softplus) { SS2D_LAUNCH_CHAN_X(true, true) } else { SS2D_LAUNCH_CHAN_X(false, true) }
    } else {
        if (a.softplus) { SS2D_LAUNCH_CHAN_X(true, false) } else { SS2D_LAUNCH_CHAN_X(false, false) }
    }
#undef SS2D_LAUNCH_CHAN_X
#undef SS2D_LAUNCH_CHAN_SPLIT_N
#undef SS2D_LAUNCH_CHAN_SPLIT
#undef SS2D_LAUNCH_CHAN_N
#undef SS2D_LAUNCH_CHAN
    return launch_status();
}

int launch_scan_chan(const ScanArgs &a, int in_dtype, int out_dtype, hipStream_t stream, const void *xt) {
    if (in_dtype == SS2D_F32) return launch_chan_typed<float, float, true>(a, xt, stream);
    bool dwords = a.L % 2 == 0;                             // every row starts on a dword
    for (const void *ptr : {a.u, a.delta, a.B, a.C, xt}) dwords = dwords && reinterpret_cast<uintptr_t>(ptr) % 4 == 0;
    for (int64_t s : {a.u_bs, a.u_ds, a.dl_bs, a.dl_ds, a.B_bs, a.B_gs, a.B_ns, a.C_bs, a.C_gs, a.C_ns}) dwords = dwords && s % 2 == 0;
    if (out_dtype != SS2D_F32) dwords = dwords && reinterpret_cast<uintptr_t>(a.out) % 4 == 0 && a.o_bs % 2 == 0 && a.o_ds % 2 == 0;
#define SS2D_CHAN(T)                                                                                                                          \
    do {                                                                                                                                      \
        if (out_dtype == SS2D_F32) return dwords ? launch_chan_typed<T, float, true>(a, xt, stream) : launch_chan_typed<T, float, false>(a, xt, stream); \
        return dwords ? launch_chan_typed<T, T, true>(a, xt, stream) : launch_chan_typed<T, T, false>(a, xt, stream);                          \
    } while (0)
    if (in_dtype == SS2D_BF16) SS2D_CHAN(bf16_t);
    SS2D_CHAN(f16_t);
#undef SS2D_CHAN
}

}  // namespace ss2d
