// Selective-scan backward for gfx950: the adjoint of selective_scan.hip's recurrence, one wavefront per
// (batch, channel) row, 512 positions per pass.
//
//   forward     dl_t = softplus(delta_t + bias);  a_t = exp(dl_t A_n);  h_t = a_t h_t-1 + dl_t B_t u_t;
//               y_t = sum_n C_n,t h_n,t + D u_t
//   backward    g_t = C_t dy_t + a_t+1 g_t+1                      (adjoint state, a reverse-time scan)
//               d dl_t = sum_n g_t (h_t-1 a_t A_n + B_t u_t)       d delta_t = d dl_t * sigmoid(delta_t + bias)
//               du_t   = dy_t D + sum_n g_t dl_t B_t               dB_n,t += g_t dl_t u_t     dC_n,t += dy_t h_t
//               dA_n  += sum_t g_t h_t-1 a_t dl_t                  dD += sum_t dy_t u_t       dbias += sum_t d delta_t
//
// A row is swept twice.  The first sweep runs the forward recurrence and keeps only the state entering every pass
// (one float per pass and state, in LDS).  The second sweep walks the passes backwards: it recomputes a and h inside
// the pass from that entering state (so no state per position is ever stored), runs the reverse scan of g with the same
// wavefront-scan machinery on lane-reversed data, and emits the gradients.  With S_t = sum_n g_n,t B_n,t and
// T_t = sum_n A_n g_n,t a_n,t h_n,t-1 the two per-position gradients are du = D dy + dl S and d dl = T + u S.
//
// dB and dC are shared by all channels of a group and dA / dD / dbias by all batches.  What bounds this pass when it is
// done badly is not arithmetic but those sums: one memory atomic per (channel, state, position) took 9.7 ms for 16
// states on 16 x 192 maps of 28 x 28 (bf16); the kernels below take 420 us, about three quarters of it vector-ALU issue.
// One state, 64 x 96 maps of 56 x 56: 250 us for 1.2 GB (497 us with one LDS atomic per entry, wavefront and pass, and no
// loads in flight under the arithmetic).  A wavefront keeps the sums of its
// positions over ALL channels its workgroup walks in registers, and they reach memory once per pass, as runs of
// consecutive floats:
//   * scan_bwd_one_kernel     one state: a wavefront owns channels, the four wavefronts' sums meet in LDS once per pass;
//   * scan_bwd_states_kernel  2 .. 32 states: a wavefront owns four STATES and walks every channel of the workgroup, the
//                             wavefronts' S and T meet in LDS once per channel and pass;
//   * scan_bwd_chan.hip       4, 8 or 16 states and rows enough, or long ones: a lane is a channel and a quarter of its states;
//   * scan_bwd_kernel         more states: a wavefront per row, atomics per channel.
#include <type_traits>

#include "scan_common.h"

namespace ss2d {

__device__ __forceinline__ float lane_reverse(float v, int lane) { return __shfl(v, kWave - 1 - lane, kWave); }

// One (batch, channel) row by one wavefront.  `h_in` is the wavefront's LDS scratch ((n_pass + 2) * N floats).
template <typename in_t, typename dy_t, bool kSoftplus>
__device__ __forceinline__ void scan_bwd_row(const ScanBwdArgs &p, int b, int d, float *h_in) {
    const int lane = threadIdx.x & (kWave - 1);
    const int N = p.N, L = p.L, P = p.n_pass;
    float *g_carry = h_in + (size_t)P * N, *a_next = g_carry + N;
    const int grp = d / p.dim_per_group, dg = d / p.dim_per_delta;
    const in_t *u_row = reinterpret_cast<const in_t *>(p.u) + b * p.u_bs + d * p.u_ds;
    const in_t *dl_row = reinterpret_cast<const in_t *>(p.delta) + b * p.dl_bs + dg * p.dl_ds;
    const in_t *B_row = reinterpret_cast<const in_t *>(p.B) + b * p.B_bs + grp * p.B_gs;
    const in_t *C_row = reinterpret_cast<const in_t *>(p.C) + b * p.C_bs + grp * p.C_gs;
    const dy_t *dy_row = reinterpret_cast<const dy_t *>(p.dout) + b * p.do_bs + d * p.do_ds;
    in_t *du_row = reinterpret_cast<in_t *>(p.du) + ((size_t)b * p.dim + d) * L;
    in_t *dd_row = reinterpret_cast<in_t *>(p.ddelta) + ((size_t)b * p.dim + d) * L;
    float *dB_row = p.dB + b * p.g_bs + grp * p.g_gs, *dC_row = p.dC + b * p.g_bs + grp * p.g_gs;
    const float *A_row = p.A + d * p.A_ds;
    const float Dv = p.D ? p.D[d] : 0.0f;
    const float bias = p.bias ? p.bias[dg] : 0.0f;
    const bool vec = p.vec_ok != 0;

    auto load8 = [&](const auto *rowp, int pos, float (&v)[kItems], float fill) {
        using T = std::remove_cv_t<std::remove_pointer_t<decltype(rowp)>>;
        if (vec) load_items<T, true>(rowp, pos, L, v, fill);
        else load_items<T, false>(rowp, pos, L, v, fill);
    };
    // dl (bias + softplus applied) and u of one pass; positions past the end give dl = 0, u = 0
    auto load_dl_u = [&](int pos, float (&dl)[kItems], float (&uv)[kItems], float (&z)[kItems]) {
        float raw[kItems], bias_items[kItems];
        load8(dl_row, pos, raw, delta_fill<kSoftplus>());
        load8(u_row, pos, uv, 0.0f);
#pragma unroll
        for (int i = 0; i < kItems; ++i) { bias_items[i] = bias; z[i] = raw[i] + bias; }
        delta_transform<kSoftplus>(raw, bias_items, dl);
        if constexpr (!kSoftplus) {
#pragma unroll
            for (int i = 0; i < kItems; ++i) dl[i] = pos + i < L ? dl[i] : 0.0f;
        }
    };

    // ---- sweep 1: the state entering every pass ---------------------------------------------------------------------
    for (int n = lane; n < N; n += kWave) { h_in[n] = 0.0f; g_carry[n] = 0.0f; a_next[n] = 1.0f; }
    for (int pass = 0; pass + 1 < P; ++pass) {
        const int pos = pass * kPass + lane * kItems;
        float dl[kItems], uv[kItems], z[kItems];
        load_dl_u(pos, dl, uv, z);
        for (int n = 0; n < N; ++n) {
            float Bv[kItems];
            load8(B_row + n * p.B_ns, pos, Bv, 0.0f);
            const float A_log2e = A_row[n * p.A_ns] * kLog2e;
            float ac = 1.0f, hh = 0.0f;
#pragma unroll
            for (int i = 0; i < kItems; ++i) {
                const float a = __builtin_amdgcn_exp2f(dl[i] * A_log2e);
                ac *= a;
                hh = fmaf(a, hh, Bv[i] * (dl[i] * uv[i]));
            }
            float a_ex, h_ex, a_tot, h_tot;
            wave_scan_pairs(ac, hh, a_ex, h_ex, a_tot, h_tot);
            const float carry = h_in[pass * N + n];
            if (lane == 0) h_in[(pass + 1) * N + n] = fmaf(a_tot, carry, h_tot);
        }
    }

    // ---- sweep 2: passes in reverse ------------------------------------------------------------------------------------
    float dD_acc = 0.0f, dbias_acc = 0.0f;
    for (int pass = P - 1; pass >= 0; --pass) {
        const int pos = pass * kPass + lane * kItems;
        float dl[kItems], uv[kItems], z[kItems], dy[kItems];
        load_dl_u(pos, dl, uv, z);
        load8(dy_row, pos, dy, 0.0f);
        float d_dl[kItems], du[kItems];
#pragma unroll
        for (int i = 0; i < kItems; ++i) { d_dl[i] = 0.0f; du[i] = dy[i] * Dv; dD_acc = fmaf(dy[i], uv[i], dD_acc); }

        for (int n = 0; n < N; ++n) {
            float Bv[kItems], Cv[kItems];
            load8(B_row + n * p.B_ns, pos, Bv, 0.0f);
            load8(C_row + n * p.C_ns, pos, Cv, 0.0f);
            const float An = A_row[n * p.A_ns];
            const float A_log2e = An * kLog2e;
            // forward inside the pass: a, and h at every position from the state entering the pass
            float a[kItems], ac[kItems], hh[kItems];
#pragma unroll
            for (int i = 0; i < kItems; ++i) {
                a[i] = __builtin_amdgcn_exp2f(dl[i] * A_log2e);
                const float bb = Bv[i] * (dl[i] * uv[i]);
                ac[i] = i == 0 ? a[i] : ac[i - 1] * a[i];
                hh[i] = i == 0 ? bb : fmaf(a[i], hh[i - 1], bb);
            }
            float a_ex, h_ex, a_tot, h_tot;
            wave_scan_pairs(ac[kItems - 1], hh[kItems - 1], a_ex, h_ex, a_tot, h_tot);
            const float s_in = fmaf(a_ex, h_in[pass * N + n], h_ex);       // h just before this lane's first item
            float h[kItems];
#pragma unroll
            for (int i = 0; i < kItems; ++i) h[i] = fmaf(ac[i], s_in, hh[i]);

            // reverse scan: g_t = C_t dy_t + a_t+1 g_t+1.  a_t+1 of a lane's last item is the next lane's first a
            // (for the last lane: the first a of the pass after this one).
            float a_up = dpp_move<kDppWaveShl1>(0.0f, a[0]);
            const float a_after = a_next[n];
            a_up = lane == kWave - 1 ? a_after : a_up;
            float m[kItems], gl[kItems];
#pragma unroll
            for (int i = kItems - 1; i >= 0; --i) {
                const float sh = i == kItems - 1 ? a_up : a[i + 1];
                const float c = Cv[i] * dy[i];
                m[i] = i == kItems - 1 ? sh : sh * m[i + 1];
                gl[i] = i == kItems - 1 ? c : fmaf(sh, gl[i + 1], c);
            }
            // suffix over lanes = prefix over reversed lanes: with G the g just after a lane's last item,
            // g_first(lane) = gl[0] + m[0] * G(lane),  G(lane) = g_first(lane + 1)
            float me, ge, mt, gt;
            wave_scan_pairs(lane_reverse(m[0], lane), lane_reverse(gl[0], lane), me, ge, mt, gt);
            const float gc = g_carry[n];
            const float G = lane_reverse(fmaf(me, gc, ge), lane);
            if (lane == 0) { g_carry[n] = fmaf(mt, gc, gt); a_next[n] = a[0]; }

            float dA_acc = 0.0f;
#pragma unroll
            for (int i = 0; i < kItems; ++i) {
                const float g = fmaf(m[i], G, gl[i]);
                const float h_prev = i == 0 ? s_in : h[i - 1];
                const float da_a = g * h_prev * a[i];                       // dL/da_t * a_t
                d_dl[i] = fmaf(da_a, An, fmaf(g, Bv[i] * uv[i], d_dl[i]));
                dA_acc = fmaf(da_a, dl[i], dA_acc);
                du[i] = fmaf(g, dl[i] * Bv[i], du[i]);
                if (pos + i < L) {
                    unsafeAtomicAdd(dB_row + n * p.g_ns + pos + i, g * dl[i] * uv[i]);
                    unsafeAtomicAdd(dC_row + n * p.g_ns + pos + i, dy[i] * h[i]);
                }
            }
#pragma unroll
            for (int off = 32; off >= 1; off >>= 1) dA_acc += __shfl_xor(dA_acc, off, kWave);
            if (lane == 0) unsafeAtomicAdd(p.dA + d * N + n, dA_acc);
        }

        float dd[kItems];
#pragma unroll
        for (int i = 0; i < kItems; ++i) {
            if constexpr (kSoftplus) {
                // softplus'(z) = sigmoid(z); beyond the threshold the forward is the identity
                const float sg = z[i] > kSoftplusThreshold ? 1.0f : 1.0f / (1.0f + __expf(-z[i]));
                dd[i] = d_dl[i] * sg;
            } else {
                dd[i] = d_dl[i];
            }
            dd[i] = pos + i < L ? dd[i] : 0.0f;
            dbias_acc += dd[i];
        }
        if (vec) { store_items<in_t, true>(du_row, pos, L, du); store_items<in_t, true>(dd_row, pos, L, dd); }
        else { store_items<in_t, false>(du_row, pos, L, du); store_items<in_t, false>(dd_row, pos, L, dd); }
    }
#pragma unroll
    for (int off = 32; off >= 1; off >>= 1) {
        dD_acc += __shfl_xor(dD_acc, off, kWave);
        dbias_acc += __shfl_xor(dbias_acc, off, kWave);
    }
    if (lane == 0) {
        if (p.dD) unsafeAtomicAdd(p.dD + d, dD_acc);
        if (p.dbias) unsafeAtomicAdd(p.dbias + d, dbias_acc);
    }
}

// One wavefront per row, 4 rows per workgroup; dB / dC straight to memory with atomics (any N, any L).
template <typename in_t, typename dy_t, bool kSoftplus>
__global__ __launch_bounds__(kBlock) void scan_bwd_kernel(const ScanBwdArgs p) {
    extern __shared__ __align__(16) float bwd_smem[];      // per wavefront: h_in [n_pass][N], g carry [N], a_next [N]
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave);
    const int row = (int)(blockIdx.x * kWavesPerWg) + wave;
    if (row >= p.rows) return;           // whole wavefront leaves; no workgroup barrier in this kernel
    scan_bwd_row<in_t, dy_t, kSoftplus>(p, row / p.dim, row % p.dim, bwd_smem + (size_t)wave * (p.n_pass + 2) * p.N);
}

// ---- pieces of the two register-summing kernels -------------------------------------------------------------------
// kI consecutive elements of a row seen through a buffer descriptor: a load past the row's end returns 0, a store there
// is dropped, dword by dword.  kVec: rows are whole dwords (single precision always); otherwise
// the descriptor's base is rounded down to a dword, a dword more is loaded, and settle shifts the elements down.
template <typename T, int kI> struct RawN { uint32_t w[gather_words<T, kI>()]; };
template <typename T, int kI, bool kVec> struct LoadN { uint32_t w[gather_words<T, kI>() + (!kVec && sizeof(T) == 2 && kI > 1)]; };

template <typename T, int kI, bool kVec>
__device__ __forceinline__ LoadN<T, kI, kVec> load_group(__amdgpu_buffer_rsrc_t rsrc, int pos) {
    LoadN<T, kI, kVec> r;
    if constexpr (kVec || kI == 1 || sizeof(T) == 4) {
        gather_group_raw<T, kI>(rsrc, (uint32_t)pos, 0, r.w);
    } else if constexpr (kI == 4) {
        const auto v = __builtin_amdgcn_raw_buffer_load_b96(rsrc, pos * 2, 0, 0);
        r.w[0] = v[0]; r.w[1] = v[1]; r.w[2] = v[2];
    } else {
        static_assert(kI == 8, "groups of 1, 4 or 8");
        const auto v = __builtin_amdgcn_raw_buffer_load_b128(rsrc, pos * 2, 0, 0);
        r.w[0] = v[0]; r.w[1] = v[1]; r.w[2] = v[2]; r.w[3] = v[3];
        r.w[4] = __builtin_amdgcn_raw_buffer_load_b32(rsrc, pos * 2 + 16, 0, 0);
    }
    return r;
}

// The elements as they arrived; `shift`: bits before the row's first element in its dword, n_valid: elements inside the row.
template <typename T, int kI, bool kVec>
__device__ __forceinline__ RawN<T, kI> settle(const LoadN<T, kI, kVec> &r, uint32_t shift, int n_valid) {
    RawN<T, kI> o;
    if constexpr (kVec || kI == 1 || sizeof(T) == 4) {
#pragma unroll
        for (int i = 0; i < gather_words<T, kI>(); ++i) o.w[i] = r.w[i];
    } else {
#pragma unroll
        for (int i = 0; i < kI / 2; ++i) o.w[i] = __builtin_amdgcn_alignbit(r.w[i + 1], r.w[i], shift);
        if (n_valid < kI) {                                     // (the dword that the row's end divides holds another row's element)
#pragma unroll
            for (int i = 0; i < kI / 2; ++i) o.w[i] &= (2 * i < n_valid ? 0xffffu : 0u) | (2 * i + 1 < n_valid ? 0xffff0000u : 0u);
        }
    }
    return o;
}

// A row's buffer for load_group, and its shift.
template <typename T, bool kVec>
__device__ __forceinline__ __amdgpu_buffer_rsrc_t load_buffer(const T *row, int L, uint32_t &shift) {
    if constexpr (kVec || sizeof(T) == 4) {
        shift = 0;
        return row_buffer(row, L);
    } else {
        const uintptr_t at = reinterpret_cast<uintptr_t>(row);
        shift = (uint32_t)(at & 2) * 8;
        return __builtin_amdgcn_make_buffer_rsrc(reinterpret_cast<void *>(at & ~(uintptr_t)3), 0, (2 * L + (int)(at & 2) + 3) & ~3, kBufferRsrcWord3);
    }
}

template <typename T, int kI, bool kVec>
__device__ __forceinline__ void store_group(__amdgpu_buffer_rsrc_t rsrc, int pos, const float (&v)[kI]) {
    typedef uint32_t words4_t __attribute__((ext_vector_type(4)));
    typedef uint32_t words2_t __attribute__((ext_vector_type(2)));
    const int off = pos * (int)sizeof(T);
    if constexpr ((!kVec && sizeof(T) == 2) || kI == 1) {
#pragma unroll
        for (int i = 0; i < kI; ++i) {
            if constexpr (sizeof(T) == 2) __builtin_amdgcn_raw_buffer_store_b16(from_f32<T>(v[i]).bits, rsrc, off + 2 * i, 0, 0);
            else __builtin_amdgcn_raw_buffer_store_b32(f32_to_bits(v[i]), rsrc, off + 4 * i, 0, 0);
        }
    } else if constexpr (sizeof(T) == 4) {
#pragma unroll
        for (int k = 0; k < kI / 4; ++k) {
            const words4_t w = {f32_to_bits(v[4 * k]), f32_to_bits(v[4 * k + 1]), f32_to_bits(v[4 * k + 2]), f32_to_bits(v[4 * k + 3])};
            __builtin_amdgcn_raw_buffer_store_b128(w, rsrc, off + 16 * k, 0, 0);
        }
    } else if constexpr (kI == 8) {
        const words4_t w = {pack2_from_f32<T>(v[0], v[1]), pack2_from_f32<T>(v[2], v[3]), pack2_from_f32<T>(v[4], v[5]),
                            pack2_from_f32<T>(v[6], v[7])};
        __builtin_amdgcn_raw_buffer_store_b128(w, rsrc, off, 0, 0);
    } else {
        static_assert(kI == 4, "groups of 1, 4 or 8");
        const words2_t w = {pack2_from_f32<T>(v[0], v[1]), pack2_from_f32<T>(v[2], v[3])};
        __builtin_amdgcn_raw_buffer_store_b64(w, rsrc, off, 0, 0);
    }
}

// wave_scan_pairs for four independent recurrences at once: interleaved, no instruction waits for the one before it.
__device__ __forceinline__ void wave_scan_pairs4(float (&a)[4], float (&h)[4], float (&a_ex)[4], float (&h_ex)[4]) {
    float ax0 = 1.0f, ax1 = 1.0f, ax2 = 1.0f, ax3 = 1.0f, hx0 = 0.0f, hx1 = 0.0f, hx2 = 0.0f, hx3 = 0.0f;
#define SS2D_FMAC(R, A, CTRL) "v_fmac_f32_dpp %" #R ", %" #R ", %" #A " " CTRL " bank_mask:0xf\n\t"
#define SS2D_MUL(A, CTRL) "v_mul_f32_dpp %" #A ", %" #A ", %" #A " " CTRL " bank_mask:0xf\n\t"
#define SS2D_STEP4(CTRL)                                                                                                  \
    SS2D_FMAC(4, 0, CTRL) SS2D_FMAC(5, 1, CTRL) SS2D_FMAC(6, 2, CTRL) SS2D_FMAC(7, 3, CTRL)                               \
    SS2D_MUL(0, CTRL) SS2D_MUL(1, CTRL) SS2D_MUL(2, CTRL) SS2D_MUL(3, CTRL)
#define SS2D_SHIFT(X, R) "v_mov_b32_dpp %" #X ", %" #R " wave_shr:1 row_mask:0xf bank_mask:0xf\n\t"
    asm("s_nop 1\n\t"
        SS2D_STEP4("row_shr:1 row_mask:0xf")
        SS2D_STEP4("row_shr:2 row_mask:0xf")
        SS2D_STEP4("row_shr:4 row_mask:0xf")
        SS2D_STEP4("row_shr:8 row_mask:0xf")
        SS2D_STEP4("row_bcast:15 row_mask:0xa")
        SS2D_STEP4("row_bcast:31 row_mask:0xc")
        SS2D_SHIFT(12, 4) SS2D_SHIFT(13, 5) SS2D_SHIFT(14, 6) SS2D_SHIFT(15, 7)
        SS2D_SHIFT(8, 0) SS2D_SHIFT(9, 1) SS2D_SHIFT(10, 2) SS2D_SHIFT(11, 3)
        "s_nop 1"
        : "+v"(a[0]), "+v"(a[1]), "+v"(a[2]), "+v"(a[3]), "+v"(h[0]), "+v"(h[1]), "+v"(h[2]), "+v"(h[3]), "+v"(ax0), "+v"(ax1),
          "+v"(ax2), "+v"(ax3), "+v"(hx0), "+v"(hx1), "+v"(hx2), "+v"(hx3));
#undef SS2D_FMAC
#undef SS2D_MUL
#undef SS2D_STEP4
#undef SS2D_SHIFT
    a_ex[0] = ax0; a_ex[1] = ax1; a_ex[2] = ax2; a_ex[3] = ax3;
    h_ex[0] = hx0; h_ex[1] = hx1; h_ex[2] = hx2; h_ex[3] = hx3;
}

// Sums over the 64 lanes of four values; the totals come back as wave-uniform values.
__device__ __forceinline__ void wave_sum4(float &v0, float &v1, float &v2, float &v3) {
#define SS2D_ADD(R, CTRL) "v_add_f32_dpp %" #R ", %" #R ", %" #R " " CTRL " bank_mask:0xf\n\t"
#define SS2D_ADD4(CTRL) SS2D_ADD(0, CTRL) SS2D_ADD(1, CTRL) SS2D_ADD(2, CTRL) SS2D_ADD(3, CTRL)
    asm("s_nop 1\n\t"
        SS2D_ADD4("row_shr:1 row_mask:0xf")
        SS2D_ADD4("row_shr:2 row_mask:0xf")
        SS2D_ADD4("row_shr:4 row_mask:0xf")
        SS2D_ADD4("row_shr:8 row_mask:0xf")
        SS2D_ADD4("row_bcast:15 row_mask:0xa")
        SS2D_ADD4("row_bcast:31 row_mask:0xc")
        "s_nop 1"
        : "+v"(v0), "+v"(v1), "+v"(v2), "+v"(v3));
#undef SS2D_ADD
#undef SS2D_ADD4
    v0 = read_lane(v0, kWave - 1);
    v1 = read_lane(v1, kWave - 1);
    v2 = read_lane(v2, kWave - 1);
    v3 = read_lane(v3, kWave - 1);
}

// The step of kI positions from their raw delta: positions past the row's end get 0, the identity of the recurrence.
template <typename in_t, int kI>
__device__ __forceinline__ void bwd_step(const RawN<in_t, kI> &raw, float bias, bool softplus, int n_valid, float (&dl)[kI]) {
    unpack_group<in_t, kI>(raw.w, dl);
    if (softplus) {
        const float bias_log2e = bias * kLog2e;
#pragma unroll
        for (int i = 0; i < kI; ++i) dl[i] = softplus_log2(fmaf(dl[i], kLog2e, bias_log2e));
    } else {
#pragma unroll
        for (int i = 0; i < kI; ++i) dl[i] += bias;
    }
    if (n_valid < kI) {
#pragma unroll
        for (int i = 0; i < kI; ++i) dl[i] = i < n_valid ? dl[i] : 0.0f;
    }
}

// The rows and constants of channel d of image b; kN states from n_first on, of which ns exist.
template <typename in_t, typename dy_t, int kN, bool kVec> struct BwdRows {
    __amdgpu_buffer_rsrc_t u, dl, dy, du, dd;
    uint32_t u_shift, dl_shift, dy_shift;
    float bias, Dv, A[kN];
    __device__ __forceinline__ void set(const ScanBwdArgs &p, int b, int d, int n_first = 0, int ns = kN) {
        const int dg = d / p.dim_per_delta;
        u = load_buffer<in_t, kVec>(reinterpret_cast<const in_t *>(p.u) + b * p.u_bs + d * p.u_ds, p.L, u_shift);
        dl = load_buffer<in_t, kVec>(reinterpret_cast<const in_t *>(p.delta) + b * p.dl_bs + dg * p.dl_ds, p.L, dl_shift);
        dy = load_buffer<dy_t, kVec>(reinterpret_cast<const dy_t *>(p.dout) + b * p.do_bs + d * p.do_ds, p.L, dy_shift);
        du = row_buffer(reinterpret_cast<const in_t *>(p.du) + ((size_t)b * p.dim + d) * p.L, p.L);
        dd = row_buffer(reinterpret_cast<const in_t *>(p.ddelta) + ((size_t)b * p.dim + d) * p.L, p.L);
        bias = p.bias ? p.bias[dg] : 0.0f;
        Dv = p.D ? p.D[d] : 0.0f;
#pragma unroll
        for (int n = 0; n < kN; ++n) A[n] = n < ns ? p.A[d * p.A_ds + (n_first + n) * p.A_ns] : 0.0f;
    }
};

// ---- one state: a wavefront owns channels ---------------------------------------------------------------------------
// Workgroup: `chunk` channels of one (image, group), channel i of a wavefront being chunk_start + wave + 4 i.  A wavefront
// walks its channels inside every pass, the next channel's loads in flight under this one's arithmetic, and sums their
// dB / dC contributions in registers; the four wavefronts' sums meet in LDS at the end of the pass and leave as one atomic
// per position.  Per-channel scalars between passes (the adjoint carry, the next pass's first a, the row sums) live in lane
// i of a register.  kI positions per lane: a pass of 512 positions would leave a row of 196 with a third of its lanes.
// Three wavefronts per SIMD, although 16-bit rows off the dword grid with a fp32 dout then keep 12 bytes a lane in memory at 8 positions (us with two, none in memory /
// three: 64 x 384 rows of 3249 386 / 385, 16 x 384 of 1353 52 / 48, 128 x 384 of 331 78 / 70).
template <typename in_t, typename dy_t, int kI, bool kVec>
__global__ __launch_bounds__(kBlock, 3) void scan_bwd_one_kernel(const ScanBwdArgs p, int chunk, int chunks_per_group, int n_groups) {
    extern __shared__ __align__(16) float bwd_smem[];      // [wave][dB, dC][pass positions], then per wavefront h_in [nc_max][P]
    constexpr int kLen = kWave * kI;
    const int lane = threadIdx.x & (kWave - 1);
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave);
    const int L = p.L, P = (L + kLen - 1) / kLen;
    const int nc_max = (chunk + kWavesPerWg - 1) / kWavesPerWg;
    float *sums = bwd_smem;
    float *h_in = bwd_smem + kWavesPerWg * 2 * kLen + (size_t)wave * nc_max * P;
    uint32_t wg = blockIdx.x;
    const int ck = (int)(wg % chunks_per_group); wg /= chunks_per_group;
    const int grp = (int)(wg % n_groups);
    const int b = (int)(wg / n_groups);
    const int c_first = ck * chunk + wave, c_end = min((ck + 1) * chunk, p.dim_per_group);
    const int nc = c_first < c_end ? (c_end - c_first + kWavesPerWg - 1) / kWavesPerWg : 0;
    const int d_first = grp * p.dim_per_group + c_first;
    const bool softplus = p.softplus != 0;
    uint32_t B_shift, C_shift;
    const auto B_buf = load_buffer<in_t, kVec>(reinterpret_cast<const in_t *>(p.B) + b * p.B_bs + grp * p.B_gs, L, B_shift);
    const auto C_buf = load_buffer<in_t, kVec>(reinterpret_cast<const in_t *>(p.C) + b * p.C_bs + grp * p.C_gs, L, C_shift);
    using Rows = BwdRows<in_t, dy_t, 1, kVec>;

    // ---- sweep 1: the state entering every pass, for every channel of this wavefront ------------------------------
    for (int i = lane; i < nc; i += kWave) h_in[i * P] = 0.0f;
    if (nc > 0 && P > 1) {
        Rows r;
        r.set(p, b, d_first);
        LoadN<in_t, kI, kVec> u_raw = load_group<in_t, kI, kVec>(r.u, lane * kI), dl_raw = load_group<in_t, kI, kVec>(r.dl, lane * kI);
        for (int pass = 0; pass + 1 < P; ++pass) {
            const int pos = pass * kLen + lane * kI;
            const RawN<in_t, kI> B_raw = settle<in_t, kI, kVec>(load_group<in_t, kI, kVec>(B_buf, pos), B_shift, kI);
            float Bv[kI];
            unpack_group<in_t, kI>(B_raw.w, Bv);
            for (int ci = 0; ci < nc; ++ci) {
                const float bias = r.bias, A_log2e = r.A[0] * kLog2e;
                const RawN<in_t, kI> u_now = settle<in_t, kI, kVec>(u_raw, r.u_shift, kI), dl_now = settle<in_t, kI, kVec>(dl_raw, r.dl_shift, kI);
                // the next channel, or the first one of the next pass
                const bool wrap = ci + 1 == nc;
                const int pos_next = wrap ? pos + kLen : pos;
                r.set(p, b, d_first + (wrap ? 0 : ci + 1) * kWavesPerWg);
                u_raw = load_group<in_t, kI, kVec>(r.u, pos_next);
                dl_raw = load_group<in_t, kI, kVec>(r.dl, pos_next);
                float dl[kI], uv[kI];
                bwd_step<in_t, kI>(dl_now, bias, softplus, kI, dl);           // every pass but the last is full
                unpack_group<in_t, kI>(u_now.w, uv);
                float ac = 1.0f, hh = 0.0f;
#pragma unroll
                for (int i = 0; i < kI; ++i) {
                    const float a = __builtin_amdgcn_exp2f(dl[i] * A_log2e);
                    ac *= a;
                    hh = fmaf(a, hh, Bv[i] * (dl[i] * uv[i]));
                }
                float a_ex, h_ex, a_tot, h_tot;
                wave_scan_pairs(ac, hh, a_ex, h_ex, a_tot, h_tot);
                const float carry = h_in[ci * P + pass];
                if (lane == 0) h_in[ci * P + pass + 1] = fmaf(a_tot, carry, h_tot);
            }
        }
    }

    // ---- sweep 2: passes in reverse, channels inside ------------------------------------------------------------------
    float g_carry = 0.0f, a_next = 1.0f, dA_sum = 0.0f, dD_sum = 0.0f, db_sum = 0.0f;      // lane i: channel i
    Rows r;
    LoadN<in_t, kI, kVec> u_raw, dl_raw;
    LoadN<dy_t, kI, kVec> dy_raw;
    if (nc > 0) {
        const int pos = (P - 1) * kLen + lane * kI;
        r.set(p, b, d_first);
        u_raw = load_group<in_t, kI, kVec>(r.u, pos);
        dl_raw = load_group<in_t, kI, kVec>(r.dl, pos);
        dy_raw = load_group<dy_t, kI, kVec>(r.dy, pos);
    }
    for (int pass = P - 1; pass >= 0; --pass) {
        const int pos = pass * kLen + lane * kI;
        const int n_valid = pass + 1 < P ? kI : L - pos;
        float Bv[kI], Cv[kI], sumB[kI], sumC[kI];
        {
            const auto B_in = load_group<in_t, kI, kVec>(B_buf, pos), C_in = load_group<in_t, kI, kVec>(C_buf, pos);
            const RawN<in_t, kI> B_raw = settle<in_t, kI, kVec>(B_in, B_shift, n_valid), C_raw = settle<in_t, kI, kVec>(C_in, C_shift, n_valid);
            unpack_group<in_t, kI>(B_raw.w, Bv);
            unpack_group<in_t, kI>(C_raw.w, Cv);
        }
#pragma unroll
        for (int i = 0; i < kI; ++i) { sumB[i] = 0.0f; sumC[i] = 0.0f; }
        for (int ci = 0; ci < nc; ++ci) {
            const Rows rn = r;
            const RawN<in_t, kI> u_now = settle<in_t, kI, kVec>(u_raw, rn.u_shift, n_valid), dl_now = settle<in_t, kI, kVec>(dl_raw, rn.dl_shift, n_valid);
            const RawN<dy_t, kI> dy_now = settle<dy_t, kI, kVec>(dy_raw, rn.dy_shift, n_valid);
            const bool wrap = ci + 1 == nc;
            const int pos_next = wrap && pass > 0 ? pos - kLen : pos;      // (after the last one: read again, not used)
            r.set(p, b, d_first + (wrap ? 0 : ci + 1) * kWavesPerWg);
            u_raw = load_group<in_t, kI, kVec>(r.u, pos_next);
            dl_raw = load_group<in_t, kI, kVec>(r.dl, pos_next);
            dy_raw = load_group<dy_t, kI, kVec>(r.dy, pos_next);
            const float An = rn.A[0], A_log2e = An * kLog2e;
            float dl[kI], uv[kI], dy[kI], raw[kI];
            bwd_step<in_t, kI>(dl_now, rn.bias, softplus, n_valid, dl);
            unpack_group<in_t, kI>(dl_now.w, raw);
            unpack_group<in_t, kI>(u_now.w, uv);
            unpack_group<dy_t, kI>(dy_now.w, dy);

            // lane totals: forward (a product, h from 0), and backward -- g_t = C_t dy_t + a_t+1 g_t+1, where a_t+1 of a lane's
            // last item is the next lane's first a (for the last lane: the first a of the pass after this one)
            float a[kI], q = 1.0f, hh = 0.0f;
#pragma unroll
            for (int i = 0; i < kI; ++i) {
                a[i] = __builtin_amdgcn_exp2f(dl[i] * A_log2e);
                hh = fmaf(a[i], hh, Bv[i] * (dl[i] * uv[i]));
                if (i > 0) q *= a[i];
            }
            float a_up = dpp_move<kDppWaveShl1>(0.0f, a[0]);
            a_up = lane == kWave - 1 ? read_lane(a_next, ci) : a_up;
            float gg = 0.0f;
#pragma unroll
            for (int i = kI - 1; i >= 0; --i) gg = fmaf(i == kI - 1 ? 0.0f : a[i + 1], gg, Cv[i] * dy[i]);
            float a_ex, h_ex, a_tot, h_tot, me, ge, mt, gt;
            wave_scan_pairs(q * a[0], hh, a_ex, h_ex, a_tot, h_tot);
            // suffix over lanes = prefix over reversed lanes: with G the g just after a lane's last item,
            // g_first(lane) = gg + (q a_up) G(lane),  G(lane) = g_first(lane + 1)
            wave_scan_pairs(lane_reverse(q * a_up, lane), lane_reverse(gg, lane), me, ge, mt, gt);
            const float gc = read_lane(g_carry, ci);
            float h = fmaf(a_ex, h_in[ci * P + pass], h_ex);                    // just before this lane's first item
            float g = a_up * lane_reverse(fmaf(me, gc, ge), lane);              // a_t+1 g_t+1 of this lane's last item
            g_carry = lane == ci ? fmaf(mt, gc, gt) : g_carry;
            a_next = lane == ci ? read_lane(a[0], 0) : a_next;

            float ah[kI];                                                       // a_t h_t-1
#pragma unroll
            for (int i = 0; i < kI; ++i) {
                ah[i] = a[i] * h;
                h = fmaf(Bv[i], dl[i] * uv[i], ah[i]);
                sumC[i] = fmaf(dy[i], h, sumC[i]);
            }
            float dA_acc = 0.0f, dD_acc = 0.0f, db_acc = 0.0f, du[kI], dd[kI];
#pragma unroll
            for (int i = kI - 1; i >= 0; --i) {
                g = fmaf(Cv[i], dy[i], g);
                const float da_a = g * ah[i];                                   // dL/da_t * a_t
                const float gB = g * Bv[i];
                dA_acc = fmaf(da_a, dl[i], dA_acc);
                dD_acc = fmaf(dy[i], uv[i], dD_acc);
                sumB[i] = fmaf(g, dl[i] * uv[i], sumB[i]);
                du[i] = fmaf(gB, dl[i], dy[i] * rn.Dv);
                dd[i] = fmaf(da_a, An, gB * uv[i]);
                g *= a[i];
            }
            if (softplus) {
#pragma unroll
                for (int i = 0; i < kI; ++i) dd[i] *= bwd_sigmoid(raw[i], rn.bias);
            }
#pragma unroll
            for (int i = 0; i < kI; ++i) db_acc += dd[i];
            store_group<in_t, kI, kVec>(rn.du, pos, du);
            store_group<in_t, kI, kVec>(rn.dd, pos, dd);
            float unused = 0.0f;
            wave_sum4(dA_acc, dD_acc, db_acc, unused);
            dA_sum += lane == ci ? dA_acc : 0.0f;
            dD_sum += lane == ci ? dD_acc : 0.0f;
            db_sum += lane == ci ? db_acc : 0.0f;
        }
        __syncthreads();                                    // the sums of the pass before have been read
        {
            float *mine = sums + wave * 2 * kLen + lane * kI;
#pragma unroll
            for (int i = 0; i < kI; ++i) { mine[i] = sumB[i]; mine[kLen + i] = sumC[i]; }
        }
        __syncthreads();
        float *dB_row = p.dB + b * p.g_bs + grp * p.g_gs + pass * kLen, *dC_row = p.dC + b * p.g_bs + grp * p.g_gs + pass * kLen;
        const int n_pos = min(kLen, L - pass * kLen);
        for (int i = threadIdx.x; i < n_pos; i += kBlock) {
            float sb = 0.0f, sc = 0.0f;
#pragma unroll
            for (int w = 0; w < kWavesPerWg; ++w) { sb += sums[w * 2 * kLen + i]; sc += sums[(w * 2 + 1) * kLen + i]; }
            unsafeAtomicAdd(dB_row + i, sb);
            unsafeAtomicAdd(dC_row + i, sc);
        }
    }
    if (lane < nc) {
        const int d = d_first + lane * kWavesPerWg;
        unsafeAtomicAdd(p.dA + d, dA_sum);
        if (p.dD) unsafeAtomicAdd(p.dD + d, dD_sum);
        if (p.dbias) unsafeAtomicAdd(p.dbias + d, db_sum);
    }
}

// ---- 2 .. 32 states: a wavefront owns four states ---------------------------------------------------------------------
// Workgroup: `chunk` channels of one (image, group), ceil(N / 4) wavefronts, wavefront w owning states 4w .. 4w+3 of every
// channel.  Inside a pass it walks the channels with the pass's B / C items and the dB / dC sums of its states in registers
// (kStates * kI * 2 sums), four recurrences interleaved; per channel the wavefronts put their S and T (see the top) into
// one of two LDS buffers, meet at one barrier and share out the pass's positions for du and d delta.
constexpr int kStates = 4;

template <typename in_t, typename dy_t, int kI, bool kVec>
__global__ __launch_bounds__(512, 2) void scan_bwd_states_kernel(const ScanBwdArgs p, int chunk, int chunks_per_group, int n_groups) {
    // [2 buffers][wave][S, T][kQ][64 lanes][kG], per wavefront a tile of kLen floats, per wavefront h_in [chunk][P][4]
    extern __shared__ __align__(16) float bwd_smem[];
    constexpr int kLen = kWave * kI;
    constexpr int kG = kI < 4 ? kI : 4, kQ = kI / kG;            // positions per finishing task, tasks per lane and gradient
    const int lane = threadIdx.x & (kWave - 1);
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave), n_waves = blockDim.x / kWave;
    const int L = p.L, P = (L + kLen - 1) / kLen;
    float *part = bwd_smem;
    float *tile = bwd_smem + (size_t)4 * n_waves * kLen + (size_t)wave * kLen;
    float4 *h_in = reinterpret_cast<float4 *>(bwd_smem + (size_t)5 * n_waves * kLen) + (size_t)wave * chunk * P;
    uint32_t wg = blockIdx.x;
    const int ck = (int)(wg % chunks_per_group); wg /= chunks_per_group;
    const int grp = (int)(wg % n_groups);
    const int b = (int)(wg / n_groups);
    const int c_first = ck * chunk, nc = min(chunk, p.dim_per_group - c_first);
    const int d_first = grp * p.dim_per_group + c_first;
    const int n_first = wave * kStates, ns = min(kStates, p.N - n_first);
    const bool softplus = p.softplus != 0;
    const in_t *B_rows = reinterpret_cast<const in_t *>(p.B) + b * p.B_bs + grp * p.B_gs + n_first * p.B_ns;
    const in_t *C_rows = reinterpret_cast<const in_t *>(p.C) + b * p.C_bs + grp * p.C_gs + n_first * p.C_ns;
    using Rows = BwdRows<in_t, dy_t, kStates, kVec>;
    auto load_states = [&](const in_t *rows, int64_t stride, int pos, int n_valid, RawN<in_t, kI> (&raw)[kStates]) {
#pragma unroll
        for (int s = 0; s < kStates; ++s) {
            uint32_t shift;
            if (s < ns) raw[s] = settle<in_t, kI, kVec>(load_group<in_t, kI, kVec>(load_buffer<in_t, kVec>(rows + s * stride, L, shift), pos), shift, n_valid);
            else raw[s] = RawN<in_t, kI>{};                      // states past N: B = C = 0, they stay 0
        }
    };

    // ---- sweep 1 ----------------------------------------------------------------------------------------------------
    for (int i = lane; i < nc; i += kWave) h_in[i * P] = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
    if (P > 1) {
        Rows r;
        r.set(p, b, d_first, n_first, ns);
        LoadN<in_t, kI, kVec> u_raw = load_group<in_t, kI, kVec>(r.u, lane * kI), dl_raw = load_group<in_t, kI, kVec>(r.dl, lane * kI);
        for (int pass = 0; pass + 1 < P; ++pass) {
            const int pos = pass * kLen + lane * kI;
            RawN<in_t, kI> B_raw[kStates];
            load_states(B_rows, p.B_ns, pos, kI, B_raw);
            for (int ci = 0; ci < nc; ++ci) {
                const Rows rn = r;
                const RawN<in_t, kI> u_now = settle<in_t, kI, kVec>(u_raw, rn.u_shift, kI), dl_now = settle<in_t, kI, kVec>(dl_raw, rn.dl_shift, kI);
                const bool wrap = ci + 1 == nc;
                const int pos_next = wrap ? pos + kLen : pos;
                r.set(p, b, d_first + (wrap ? 0 : ci + 1), n_first, ns);
                u_raw = load_group<in_t, kI, kVec>(r.u, pos_next);
                dl_raw = load_group<in_t, kI, kVec>(r.dl, pos_next);
                float dl[kI], dlu[kI], ac[kStates], hh[kStates], a_ex[kStates], h_ex[kStates];
                bwd_step<in_t, kI>(dl_now, rn.bias, softplus, kI, dl);           // every pass but the last is full
                unpack_group<in_t, kI>(u_now.w, dlu);
#pragma unroll
                for (int i = 0; i < kI; ++i) dlu[i] *= dl[i];
#pragma unroll
                for (int s = 0; s < kStates; ++s) {
                    float Bv[kI];
                    unpack_group<in_t, kI>(B_raw[s].w, Bv);
                    const float A_log2e = rn.A[s] * kLog2e;
                    ac[s] = 1.0f;
                    hh[s] = 0.0f;
#pragma unroll
                    for (int i = 0; i < kI; ++i) {
                        const float a = __builtin_amdgcn_exp2f(dl[i] * A_log2e);
                        ac[s] *= a;
                        hh[s] = fmaf(a, hh[s], Bv[i] * dlu[i]);
                    }
                }
                wave_scan_pairs4(ac, hh, a_ex, h_ex);
                const float4 carry = h_in[ci * P + pass];
                if (lane == kWave - 1)                                          // the lane that holds the totals
                    h_in[ci * P + pass + 1] = make_float4(fmaf(ac[0], carry.x, hh[0]), fmaf(ac[1], carry.y, hh[1]),
                                                          fmaf(ac[2], carry.z, hh[2]), fmaf(ac[3], carry.w, hh[3]));
            }
        }
    }

    // ---- sweep 2 ----------------------------------------------------------------------------------------------------
    float g_carry[kStates], a_next[kStates], dA_sum[kStates], dD_sum = 0.0f, db_sum = 0.0f;      // lane i: channel i
#pragma unroll
    for (int s = 0; s < kStates; ++s) { g_carry[s] = 0.0f; a_next[s] = 1.0f; dA_sum[s] = 0.0f; }
    Rows r;
    r.set(p, b, d_first, n_first, ns);
    int buffer = 0;
    LoadN<in_t, kI, kVec> u_raw, dl_raw;
    LoadN<dy_t, kI, kVec> dy_raw;
    {
        const int pos = (P - 1) * kLen + lane * kI;
        u_raw = load_group<in_t, kI, kVec>(r.u, pos);
        dl_raw = load_group<in_t, kI, kVec>(r.dl, pos);
        dy_raw = load_group<dy_t, kI, kVec>(r.dy, pos);
    }
    for (int pass = P - 1; pass >= 0; --pass) {
        const int pos = pass * kLen + lane * kI;
        const int n_valid = pass + 1 < P ? kI : L - pos;
        RawN<in_t, kI> B_raw[kStates], C_raw[kStates];
        load_states(B_rows, p.B_ns, pos, n_valid, B_raw);
        load_states(C_rows, p.C_ns, pos, n_valid, C_raw);
        float sumB[kStates][kI], sumC[kStates][kI];
#pragma unroll
        for (int s = 0; s < kStates; ++s)
#pragma unroll
            for (int i = 0; i < kI; ++i) { sumB[s][i] = 0.0f; sumC[s][i] = 0.0f; }

        for (int ci = 0; ci < nc; ++ci) {
            const Rows rn = r;
            const RawN<in_t, kI> u_now = settle<in_t, kI, kVec>(u_raw, rn.u_shift, n_valid), dl_now = settle<in_t, kI, kVec>(dl_raw, rn.dl_shift, n_valid);
            const RawN<dy_t, kI> dy_now = settle<dy_t, kI, kVec>(dy_raw, rn.dy_shift, n_valid);
            const bool wrap = ci + 1 == nc;
            const int pos_next = wrap && pass > 0 ? pos - kLen : pos;      // (after the last one: read again, not used)
            r.set(p, b, d_first + (wrap ? 0 : ci + 1), n_first, ns);
            u_raw = load_group<in_t, kI, kVec>(r.u, pos_next);
            dl_raw = load_group<in_t, kI, kVec>(r.dl, pos_next);
            dy_raw = load_group<dy_t, kI, kVec>(r.dy, pos_next);
            const float4 h4 = h_in[ci * P + pass];
            const float h_pass[kStates] = {h4.x, h4.y, h4.z, h4.w};
            float dl[kI], dlu[kI], dy[kI];
            bwd_step<in_t, kI>(dl_now, rn.bias, softplus, n_valid, dl);
            unpack_group<in_t, kI>(u_now.w, dlu);
#pragma unroll
            for (int i = 0; i < kI; ++i) dlu[i] *= dl[i];
            unpack_group<dy_t, kI>(dy_now.w, dy);

            // lane totals of the forward and the reverse recurrence (see scan_bwd_one_kernel)
            float a[kStates][kI], a_up[kStates], ac[kStates], hh[kStates], m[kStates], gg[kStates];
#pragma unroll
            for (int s = 0; s < kStates; ++s) {
                float Bv[kI], Cv[kI], q = 1.0f;
                unpack_group<in_t, kI>(B_raw[s].w, Bv);
                unpack_group<in_t, kI>(C_raw[s].w, Cv);
                const float A_log2e = rn.A[s] * kLog2e;
                hh[s] = 0.0f;
#pragma unroll
                for (int i = 0; i < kI; ++i) {
                    a[s][i] = __builtin_amdgcn_exp2f(dl[i] * A_log2e);
                    hh[s] = fmaf(a[s][i], hh[s], Bv[i] * dlu[i]);
                    if (i > 0) q *= a[s][i];
                }
                const float up = dpp_move<kDppWaveShl1>(0.0f, a[s][0]);
                a_up[s] = lane == kWave - 1 ? read_lane(a_next[s], ci) : up;
                gg[s] = 0.0f;
#pragma unroll
                for (int i = kI - 1; i >= 0; --i) gg[s] = fmaf(i == kI - 1 ? 0.0f : a[s][i + 1], gg[s], Cv[i] * dy[i]);
                ac[s] = q * a[s][0];
                m[s] = lane_reverse(q * a_up[s], lane);
                gg[s] = lane_reverse(gg[s], lane);
            }
            float a_ex[kStates], h_ex[kStates], m_ex[kStates], g_ex[kStates];
            wave_scan_pairs4(ac, hh, a_ex, h_ex);
            wave_scan_pairs4(m, gg, m_ex, g_ex);

            float S[kI], T[kI], dA_acc[kStates];
#pragma unroll
            for (int i = 0; i < kI; ++i) { S[i] = 0.0f; T[i] = 0.0f; }
#pragma unroll
            for (int s = 0; s < kStates; ++s) {
                float Bv[kI], Cv[kI], ah[kI];
                unpack_group<in_t, kI>(B_raw[s].w, Bv);
                unpack_group<in_t, kI>(C_raw[s].w, Cv);
                const float gc = read_lane(g_carry[s], ci);
                float h = fmaf(a_ex[s], h_pass[s], h_ex[s]);                    // just before this lane's first item
                float g = a_up[s] * lane_reverse(fmaf(m_ex[s], gc, g_ex[s]), lane);
                const float g_new = fmaf(read_lane(m[s], kWave - 1), gc, read_lane(gg[s], kWave - 1));
                g_carry[s] = lane == ci ? g_new : g_carry[s];
                a_next[s] = lane == ci ? read_lane(a[s][0], 0) : a_next[s];
#pragma unroll
                for (int i = 0; i < kI; ++i) {
                    ah[i] = a[s][i] * h;
                    h = fmaf(Bv[i], dlu[i], ah[i]);
                    sumC[s][i] = fmaf(dy[i], h, sumC[s][i]);
                }
                dA_acc[s] = 0.0f;
#pragma unroll
                for (int i = kI - 1; i >= 0; --i) {
                    g = fmaf(Cv[i], dy[i], g);
                    const float da_a = g * ah[i];                               // dL/da_t * a_t
                    dA_acc[s] = fmaf(da_a, dl[i], dA_acc[s]);
                    T[i] = fmaf(da_a, rn.A[s], T[i]);
                    S[i] = fmaf(g, Bv[i], S[i]);
                    sumB[s][i] = fmaf(g, dlu[i], sumB[s][i]);
                    g *= a[s][i];
                }
            }
            wave_sum4(dA_acc[0], dA_acc[1], dA_acc[2], dA_acc[3]);
#pragma unroll
            for (int s = 0; s < kStates; ++s) dA_sum[s] += lane == ci ? dA_acc[s] : 0.0f;

            // S and T of all states: task (gradient, q) of the pass is finished by wavefront (gradient * kQ + q) % n_waves
            auto slot = [&](int w, int which, int q) { return part + ((((buffer * n_waves + w) * 2 + which) * kQ + q) * kWave + lane) * kG; };
#pragma unroll
            for (int q = 0; q < kQ; ++q) {
                float *to_S = slot(wave, 0, q), *to_T = slot(wave, 1, q);
#pragma unroll
                for (int j = 0; j < kG; ++j) { to_S[j] = S[q * kG + j]; to_T[j] = T[q * kG + j]; }
            }
            __syncthreads();
            float dD_acc = 0.0f, db_acc = 0.0f;
            float uv[kI], raw[kI];
            unpack_group<in_t, kI>(u_now.w, uv);
            unpack_group<in_t, kI>(dl_now.w, raw);
#pragma unroll
            for (int q = 0; q < kQ; ++q) {
                const bool does_du = q % n_waves == wave, does_dd = (kQ + q) % n_waves == wave;
                if (!does_du && !does_dd) continue;
                float Sq[kG];
#pragma unroll
                for (int j = 0; j < kG; ++j) Sq[j] = 0.0f;
                for (int w = 0; w < n_waves; ++w) {
                    const float *from = slot(w, 0, q);
#pragma unroll
                    for (int j = 0; j < kG; ++j) Sq[j] += from[j];
                }
                if (does_du) {
                    float du[kG];
#pragma unroll
                    for (int j = 0; j < kG; ++j) {
                        du[j] = fmaf(Sq[j], dl[q * kG + j], dy[q * kG + j] * rn.Dv);
                        dD_acc = fmaf(dy[q * kG + j], uv[q * kG + j], dD_acc);
                    }
                    store_group<in_t, kG, kVec>(rn.du, pos + q * kG, du);
                }
                if (does_dd) {
                    float dd[kG];
#pragma unroll
                    for (int j = 0; j < kG; ++j) dd[j] = Sq[j] * uv[q * kG + j];
                    for (int w = 0; w < n_waves; ++w) {
                        const float *from = slot(w, 1, q);
#pragma unroll
                        for (int j = 0; j < kG; ++j) dd[j] += from[j];
                    }
                    if (softplus) {
#pragma unroll
                        for (int j = 0; j < kG; ++j) dd[j] *= bwd_sigmoid(raw[q * kG + j], rn.bias);
                    }
#pragma unroll
                    for (int j = 0; j < kG; ++j) db_acc += dd[j];
                    store_group<in_t, kG, kVec>(rn.dd, pos + q * kG, dd);
                }
            }
            float unused0 = 0.0f, unused1 = 0.0f;
            wave_sum4(dD_acc, db_acc, unused0, unused1);
            dD_sum += lane == ci ? dD_acc : 0.0f;
            db_sum += lane == ci ? db_acc : 0.0f;
            buffer ^= 1;
        }

        // the pass's dB / dC: turned round in a wavefront-private tile so that an atomic instruction covers 64 consecutive floats
        const int n_pos = min(kLen, L - pass * kLen);
#pragma unroll
        for (int s = 0; s < kStates; ++s) {
            if (s >= ns) continue;
            const int64_t row = b * p.g_bs + grp * p.g_gs + (n_first + s) * p.g_ns + pass * kLen;
#pragma unroll
            for (int which = 0; which < 2; ++which) {
                float *to = (which ? p.dC : p.dB) + row;
                wave_lds_sync();
#pragma unroll
                for (int i = 0; i < kI; ++i) tile[lane * kI + i] = which ? sumC[s][i] : sumB[s][i];
                wave_lds_sync();
                for (int i = lane; i < n_pos; i += kWave) unsafeAtomicAdd(to + i, tile[i]);
            }
        }
    }
    if (lane < nc) {
        const int d = d_first + lane;
#pragma unroll
        for (int s = 0; s < kStates; ++s)
            if (s < ns) unsafeAtomicAdd(p.dA + (int64_t)d * p.N + n_first + s, dA_sum[s]);
        if (p.dD && wave < 2 * kQ) unsafeAtomicAdd(p.dD + d, dD_sum);
        if (p.dbias && wave < 2 * kQ) unsafeAtomicAdd(p.dbias + d, db_sum);
    }
}

// How the register-summing kernels walk a problem, and which kernel that is.
struct BwdPlan {
    int32_t kernel;             // SS2D_SCAN_BWD_KERNEL_*
    int32_t items;              // positions per lane
    bool vec;                   // rows of whole dwords
    int32_t n_waves, chunk, cpg;            // wavefronts and channels per workgroup, workgroups per group
    int64_t n_wg;
    size_t smem;
};

// The arguments in the kernels' terms and the kernel for them; a status where none is launched (SS2D_OK: nothing to do).
static int plan_scan_bwd(const ss2d_scan_bwd_params *q, ScanBwdArgs &a, BwdPlan &plan) {
    plan = {};
    if (!q) return SS2D_EINVAL;
    if (q->batch < 0 || q->dim < 0 || q->seqlen < 0) return SS2D_EINVAL;
    if (q->dstate <= 0 || q->dstate > 256 || q->n_groups <= 0 || q->delta_dim <= 0) return SS2D_EINVAL;
    if (q->in_dtype != SS2D_F32 && q->in_dtype != SS2D_BF16 && q->in_dtype != SS2D_F16) return SS2D_EINVAL;
    if (q->dout_dtype != SS2D_F32 && q->dout_dtype != q->in_dtype) return SS2D_EINVAL;
    if (q->dim % q->n_groups != 0 || q->dim % q->delta_dim != 0) return SS2D_EINVAL;
    if (q->batch == 0 || q->dim == 0 || q->seqlen == 0) return SS2D_OK;
    if (!q->u || !q->delta || !q->A || !q->B || !q->C || !q->dout || !q->du || !q->ddelta || !q->dA || !q->dB || !q->dC)
        return SS2D_EINVAL;
    if ((q->D == nullptr) != (q->dD == nullptr)) return SS2D_EINVAL;
    if ((q->delta_bias == nullptr) != (q->ddelta_bias == nullptr)) return SS2D_EINVAL;
    if ((int64_t)q->batch * q->dim > 0x7fffffff - kWavesPerWg) return SS2D_ENOTSUP;

    a.u = q->u; a.delta = q->delta; a.B = q->B; a.C = q->C; a.dout = q->dout;
    a.A = (const float *)q->A; a.D = (const float *)q->D; a.bias = (const float *)q->delta_bias;
    a.du = q->du; a.ddelta = q->ddelta;
    a.dA = (float *)q->dA; a.dB = (float *)q->dB; a.dC = (float *)q->dC; a.dD = (float *)q->dD; a.dbias = (float *)q->ddelta_bias;
    a.batch = q->batch; a.dim = q->dim; a.L = q->seqlen; a.N = q->dstate;
    a.dim_per_group = q->dim / q->n_groups;
    a.dim_per_delta = q->dim / q->delta_dim;
    a.softplus = q->delta_softplus;
    a.rows = q->batch * q->dim;
    a.n_pass = (q->seqlen + kPass - 1) / kPass;
    a.u_bs = q->u_batch_stride; a.u_ds = q->u_d_stride;
    a.dl_bs = q->delta_batch_stride; a.dl_ds = q->delta_d_stride;
    a.A_ds = q->A_d_stride; a.A_ns = q->A_dstate_stride;
    a.B_bs = q->B_batch_stride; a.B_gs = q->B_group_stride; a.B_ns = q->B_dstate_stride;
    a.C_bs = q->C_batch_stride; a.C_gs = q->C_group_stride; a.C_ns = q->C_dstate_stride;
    a.do_bs = q->dout_batch_stride; a.do_ds = q->dout_d_stride;
    a.g_ns = q->seqlen; a.g_gs = (int64_t)q->dstate * q->seqlen; a.g_bs = (int64_t)q->n_groups * a.g_gs;
    const int in_size = q->in_dtype == SS2D_F32 ? 4 : 2, dy_size = q->dout_dtype == SS2D_F32 ? 4 : 2;
    auto dwords_ok = [&](int items) {                            // rows of whole dwords (with one position per lane elements are read)
        if (items == 1) return true;
        auto odd = [](const void *ptr) { return (reinterpret_cast<uintptr_t>(ptr) & 3) != 0; };
        if (in_size == 2) {
            for (const void *ptr : {q->u, q->delta, q->B, q->C, (const void *)q->du, (const void *)q->ddelta})
                if (odd(ptr)) return false;
            for (int64_t st : {a.u_bs, a.u_ds, a.dl_bs, a.dl_ds, a.B_bs, a.B_gs, a.B_ns, a.C_bs, a.C_gs, a.C_ns})
                if (st % 2 != 0) return false;
            if (q->seqlen % 2 != 0) return false;
        }
        return dy_size == 4 || (!odd(q->dout) && a.do_bs % 2 == 0 && a.do_ds % 2 == 0 && q->seqlen % 2 == 0);
    };
    if (a.N <= 8 * kStates && (int64_t)a.L * 4 < 0x7fffffff) {
        const bool one = a.N == 1;
        // Positions per lane (measured with the others, us): 8 where rows are long, as the wavefront scans are paid per pass
        // (192 channels of 28 x 28, batch 64: 120; with 4: 141); 4 up to 256 positions (384 x 14 x 14 in fp32: 77; with 8: 100,
        // with 1: 166) and with several states, whose B, C and sums fill the registers; 1 for rows that fit 64 lanes
        // (768 x 7 x 7: 70; with 4: 144).
        const int items = a.L <= kWave ? 1 : a.L <= 4 * kWave || !one ? 4 : 8;
        const int n_pass = (a.L + kWave * items - 1) / (kWave * items);
        const int n_waves = one ? kWavesPerWg : (a.N + kStates - 1) / kStates;
        // Channels per workgroup: more of them mean fewer atomics on dB / dC (one per entry and workgroup), fewer mean more
        // wavefronts.  The grid is filled first -- one state: 8 wavefronts per SIMD, as three at a time are resident (96 x 56 x 56,
        // batch 64: 250 us; half as many workgroups: 275); several states: the 2 per SIMD the registers allow -- down to 8
        // channels (57 x 58 maps, batch 16: 109 us; with 4: 119) or, on small problems, 4.  At most 24: no gain beyond, and the
        // per-channel scalars sit in the lanes of a register.  Groups of fewer channels leave wavefronts without one and are
        // still ahead of a wavefront per row: one channel per group, backward through autograd, 64 x 384 rows of 196 positions
        // 320 -> 95 us, 64 x 768 of 49 224 -> 123, 16 x 96 of 3306 361 -> 109; three 333 -> 77, 230 -> 77, 361 -> 78.
        const int64_t want_wg = (one ? 8192 : 2048) / n_waves, images = (int64_t)q->batch * q->n_groups;
        const int64_t per_8 = images * ((a.dim_per_group + 7) / 8);
        const int64_t least = one && per_8 >= want_wg / 4 ? 8 : 4;
        int64_t chunk = a.dim_per_group * images / want_wg;
        chunk = chunk > 24 ? 24 : chunk < least ? least : chunk;
        if (chunk > a.dim_per_group) chunk = a.dim_per_group;
        const size_t fixed = (size_t)(one ? 2 : 5) * n_waves * kWave * items * sizeof(float);
        auto smem_of = [&](int64_t c) {
            const size_t per_wave = one ? (size_t)((c + kWavesPerWg - 1) / kWavesPerWg) * n_pass : (size_t)c * n_pass * 4;
            return fixed + n_waves * per_wave * sizeof(float);
        };
        while (chunk > 1 && smem_of(chunk) > 64 * 1024) chunk = (chunk + 1) / 2;
        const int64_t cpg = (a.dim_per_group + chunk - 1) / chunk;
        chunk = (a.dim_per_group + cpg - 1) / cpg;               // even split
        const int64_t n = images * cpg;
        const size_t smem = smem_of(chunk);
        // several states and enough channels per group: one channel per lane, unless these workgroups' rounds through the chip are nearly full of positions
        const bool full = 25 * a.dim_per_group * images * a.L >= 22 * ((n + want_wg - 1) / want_wg * want_wg) * chunk * n_pass * kWave * items;
        if (scan_bwd_chan_takes(a, in_size, dy_size, full)) {
            plan.kernel = SS2D_SCAN_BWD_KERNEL_CHAN;
            return SS2D_OK;
        }
        plan.items = items; plan.vec = dwords_ok(items);
        plan.n_waves = n_waves; plan.chunk = (int)chunk; plan.cpg = (int)cpg;
        plan.n_wg = n; plan.smem = smem;
        if (n <= 0x7fffffff && smem <= 160 * 1024) {
            plan.kernel = one ? SS2D_SCAN_BWD_KERNEL_ONE : SS2D_SCAN_BWD_KERNEL_STATES;
            return SS2D_OK;
        }
    }
    plan.smem = (size_t)kWavesPerWg * (a.n_pass + 2) * a.N * sizeof(float);
    if (plan.smem > 48 * 1024) return SS2D_ENOTSUP;        // very long rows x many states: the per-pass states do not fit LDS
    // Rows read and written in groups of 8 elements: 16-byte pieces at most, so a group's alignment is that of its piece.  (The kernels above need dwords
    // only, and single precision nothing.)
    const int64_t in_vec = 16 / in_size, dy_vec = 16 / dy_size;
    auto aligned16 = [](const void *ptr) { return (reinterpret_cast<uintptr_t>(ptr) & 15) == 0; };
    bool vec = q->seqlen % in_vec == 0 && q->seqlen % dy_vec == 0 && a.do_bs % dy_vec == 0 && a.do_ds % dy_vec == 0;
    for (const void *ptr : {q->u, q->delta, q->B, q->C, q->dout, (const void *)q->du, (const void *)q->ddelta}) vec = vec && aligned16(ptr);
    for (int64_t st : {a.u_bs, a.u_ds, a.dl_bs, a.dl_ds, a.B_bs, a.B_gs, a.B_ns, a.C_bs, a.C_gs, a.C_ns}) vec = vec && st % in_vec == 0;
    a.vec_ok = vec ? 1 : 0;
    plan.n_wg = (a.rows + kWavesPerWg - 1) / kWavesPerWg;
    plan.kernel = SS2D_SCAN_BWD_KERNEL_ROWS;
    return SS2D_OK;
}

}  // namespace ss2d

extern "C" int ss2d_selective_scan_bwd_kernel(const ss2d_scan_bwd_params *q) {
    using namespace ss2d;
    ScanBwdArgs a;
    BwdPlan plan;
    const int rc = plan_scan_bwd(q, a, plan);
    return rc != SS2D_OK ? rc : plan.kernel;
}

extern "C" int ss2d_selective_scan_bwd(const ss2d_scan_bwd_params *q, void *stream) {
    using namespace ss2d;
    ScanBwdArgs a;
    BwdPlan plan;
    const int rc = plan_scan_bwd(q, a, plan);
    if (rc != SS2D_OK || plan.kernel == SS2D_SCAN_BWD_KERNEL_NONE) return rc;
    hipStream_t s = (hipStream_t)stream;
    if (plan.kernel == SS2D_SCAN_BWD_KERNEL_CHAN) return launch_scan_bwd_chan(a, q->in_dtype, q->dout_dtype, s);
    const dim3 grid((uint32_t)plan.n_wg);
    if (plan.kernel != SS2D_SCAN_BWD_KERNEL_ROWS) {
        const bool one = plan.kernel == SS2D_SCAN_BWD_KERNEL_ONE;
        const dim3 block(plan.n_waves * kWave);
#define SS2D_BWD_LAUNCH(IN, DY, KI, VEC)                                                                                        \
    do {                                                                                                                        \
        if (KI == 8 || one) hipLaunchKernelGGL((scan_bwd_one_kernel<IN, DY, KI, VEC>), grid, block, plan.smem, s, a, plan.chunk, plan.cpg, q->n_groups); \
        else hipLaunchKernelGGL((scan_bwd_states_kernel<IN, DY, KI == 8 ? 4 : KI, VEC>), grid, block, plan.smem, s, a, plan.chunk, plan.cpg, q->n_groups);  \
    } while (0)
#define SS2D_BWD_ITEMS(IN, DY)                                                                                                  \
    do {                                                                                                                        \
        if (plan.items == 8 && plan.vec) SS2D_BWD_LAUNCH(IN, DY, 8, true);                                                      \
        else if (plan.items == 8) SS2D_BWD_LAUNCH(IN, DY, 8, sizeof(IN) == 4);                                                  \
        else if (plan.items == 1) SS2D_BWD_LAUNCH(IN, DY, 1, true);                                                             \
        else if (plan.vec) SS2D_BWD_LAUNCH(IN, DY, 4, true);                                                                    \
        else SS2D_BWD_LAUNCH(IN, DY, 4, sizeof(IN) == 4);                                                                       \
    } while (0)
        if (q->in_dtype == SS2D_F32) SS2D_BWD_ITEMS(float, float);
        else if (q->in_dtype == SS2D_BF16) { if (q->dout_dtype == SS2D_F32) SS2D_BWD_ITEMS(bf16_t, float); else SS2D_BWD_ITEMS(bf16_t, bf16_t); }
        else { if (q->dout_dtype == SS2D_F32) SS2D_BWD_ITEMS(f16_t, float); else SS2D_BWD_ITEMS(f16_t, f16_t); }
#undef SS2D_BWD_ITEMS
#undef SS2D_BWD_LAUNCH
        return launch_status();
    }
#define SS2D_BWD_LAUNCH(IN, DY)                                                                                         \
    do {                                                                                                                \
        if (a.softplus) hipLaunchKernelGGL((scan_bwd_kernel<IN, DY, true>), grid, dim3(kBlock), plan.smem, s, a);       \
        else hipLaunchKernelGGL((scan_bwd_kernel<IN, DY, false>), grid, dim3(kBlock), plan.smem, s, a);                 \
    } while (0)
    if (q->in_dtype == SS2D_F32) SS2D_BWD_LAUNCH(float, float);
    else if (q->in_dtype == SS2D_BF16) { if (q->dout_dtype == SS2D_F32) SS2D_BWD_LAUNCH(bf16_t, float); else SS2D_BWD_LAUNCH(bf16_t, bf16_t); }
    else { if (q->dout_dtype == SS2D_F32) SS2D_BWD_LAUNCH(f16_t, float); else SS2D_BWD_LAUNCH(f16_t, f16_t); }
#undef SS2D_BWD_LAUNCH
    return launch_status();
}
