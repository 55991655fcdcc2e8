// x_proj of the SS2D core with the one-by-one CrossScan folded in (classification/models/vmamba.py:604-607 and
// csm_triton.py:88-131): a projection is a per-position contraction, so the four directions' weights are applied to the map
// in its natural order and only the small result is put into each direction's scan order,
//     out[k, c, b, j] = sum_d W[k, c, d] * x[b, d, r_k(j)],      c < C = R + 2 N rows per direction, d < D channels.
// The library's batched GEMM plus the CrossScan kernel spent 93 us on 77 MB of map and 26 MB of result (96 x 56 x 56, batch
// 128): the GEMM is far too narrow (4 C = 32 rows) for its tiles, and the result went through memory twice more.
//
// A workgroup owns one, two or all four directions of one tile of a map (whole maps where they fit): its result lives in
// LDS between the two phases, position-major, and leaves in scan order, so the transposing directions cost LDS reads instead
// of a pass over memory.  Workgroups of one tile are neighbours on one XCD and find x in its L2.
//   * contraction: v_mfma_f32_16x16x32, rows = output rows, columns = positions, 32 channels a step.  A lane's B operand is 8
//     channels of one position while x is contiguous along positions, so a lane loads 4 positions (8 bytes) of 8 channels and
//     a byte permute per dword pairs the channels up: four MFMA column tiles of every fourth position from 8 loads and 16
//     permutes, no LDS on the way in.  fp32 accumulation and one rounding to the 16-bit result, as the library does.
//   * maps of one or two MFMA column groups (7 x 7 ... 11 x 11) split the channels over the wavefronts instead of the
//     positions and meet in LDS.
// 96 x 56 x 56, batch 128: 25-28 us (3.9 TB/s of the 103 MB); 192 x 28 x 28: 45 -> 20; 384 x 14 x 14: 31 -> 16.5;
// 768 x 7 x 7: 30 -> 17.5; one image of each, replayed from a graph: 9.3 -> 5.8, 9.9 -> 6.8, 22.1 -> 7.6, 20.0 -> 11.5.
#include <type_traits>

#include "ss2d_common.h"

namespace ss2d {

constexpr int kXpGroup = 64;         // positions per MFMA column group: 16 lanes x 4 positions

struct XProjArgs {
    const void *x, *W;
    void *out;
    int32_t D, C, H, Wd, Hp, Wp;         // map H x Wd, written as Hp x Wp (padded at the bottom / right)
    int32_t mask_row;                    // -1: none
    int32_t rank, planes, pair_mask;     // planes > 0: the first `rank` rows leave in pairs (x_proj_pairs)
    int32_t *flags;
    DtsLayout layout;
    int32_t B, real_h, real_w;           // the map's size before rows and columns were added to it
    int32_t n_dirs, Ce;                  // directions per workgroup (1, 2, 4); C rounded up to even: rows per direction in LDS
    int32_t Th, Tw, tiles_h, tiles_w, pitch, k_steps, k_split, v_row, v_col;
    int64_t ks, cs, bs;
    uint32_t total;
};

// q = x / d, r = x % d for 0 <= x < 2^23, inv = 1 / d
__device__ __forceinline__ void small_divmod(int x, int d, float inv, int &q, int &r) {
    q = (int)((float)x * inv);
    r = x - q * d;
    if (r < 0) { --q; r += d; }
    if (r >= d) { ++q; r -= d; }
}

// kPaired: the ranks of the step leave in pairs (x_proj_pairs).
template <typename T, int kMt, bool kPaired>
__global__ __launch_bounds__(kBlock, kMt == 1 ? 4 : kMt <= 3 ? 3 : 2) void x_proj_kernel(const XProjArgs p) {
    extern __shared__ __align__(16) uint16_t xp_smem[];         // [tile positions][pitch], then the split channels' sums
    const int lane = threadIdx.x & (kWave - 1);
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave);
    uint32_t id = xcd_contiguous_id(blockIdx.x, p.total);
    const uint32_t wg = id;
    const int n_sets = 4 / p.n_dirs, k_first = (int)(id % (uint32_t)n_sets) * p.n_dirs;
    id /= (uint32_t)n_sets;
    const int tw = (int)(id % (uint32_t)p.tiles_w); id /= (uint32_t)p.tiles_w;
    const int th = (int)(id % (uint32_t)p.tiles_h);
    const int64_t b = id / (uint32_t)p.tiles_h;
    const bool last_h = th + 1 == p.tiles_h, last_w = tw + 1 == p.tiles_w;
    const int h0 = th * p.Th, h1 = last_h ? p.H : h0 + p.Th, w0 = tw * p.Tw, w1 = last_w ? p.Wd : w0 + p.Tw;
    const int n_cols = w1 - w0, n_pos = (h1 - h0) * n_cols, HW = p.H * p.Wd;
    const uint16_t *x = reinterpret_cast<const uint16_t *>(p.x) + b * p.D * HW;
    const uint16_t *W = reinterpret_cast<const uint16_t *>(p.W) + (int64_t)k_first * p.C * p.D;

    // ---- contraction ------------------------------------------------------------------------------------------------
    // Wavefront (group, part) takes column groups group, group + g_stride ... and, with the channels split, every k_split-th
    // step of them.  Its steps are one sequence across groups, kRing of them in flight: a step's loads go into the registers
    // the step kRing before has just been multiplied from, unconditionally (past the end the last step is loaded again), so
    // that no wait covers more than the step it is for.
    constexpr int kRing = kMt <= 3 ? 3 : 2;
    constexpr int n_waves = kBlock / kWave;
    const int col = lane & 15, kg = lane >> 4;
    const int part = wave % p.k_split, g_first = wave / p.k_split, g_stride = n_waves / p.k_split;
    const int n_groups = (n_pos + kXpGroup - 1) / kXpGroup;
    const int my_groups = g_first < n_groups ? (n_groups - g_first + g_stride - 1) / g_stride : 0;
    const int my_steps = (p.k_steps - part + p.k_split - 1) / p.k_split;      // (k_split <= k_steps)
    const float inv_cols = 1.0f / (float)n_cols;
    struct Step { uint2 raw[8]; u32x4_t a[kMt]; };
    uint32_t w_row[kMt];                                         // the lane's weight rows: row r is row r % Ce of direction r / Ce
#pragma unroll
    for (int m = 0; m < kMt; ++m) {
        const int r = min(m * 16 + col, p.n_dirs * p.Ce - 1);    // (rows past the last repeat it, nobody reads them)
        const int dir = (r >= p.Ce) + (r >= 2 * p.Ce) + (r >= 3 * p.Ce);
        w_row[m] = (uint32_t)((dir * p.C + min(r - dir * p.Ce, p.C - 1)) * p.D);
    }
    auto offset_of = [&](int group) {                            // of the lane's first position in the map
        const int at = min(group * kXpGroup + 4 * col, n_pos - 1);
        // the four positions are consecutive in memory: the tile spans full rows, or its width is a multiple of 4
        if (n_cols == p.Wd) return h0 * p.Wd + at;
        int r, c;
        small_divmod(at, n_cols, inv_cols, r, c);
        return (h0 + r) * p.Wd + w0 + c;
    };
    auto load = [&](int group, int step, Step &r) {
        const int off = min(offset_of(group), HW - 4);           // inside the map: shifted into place below
        const int d0 = step * 32 + 8 * kg;
        const bool in = d0 < p.D;                                // (D is a multiple of 8)
        const uint32_t at_d = (uint32_t)((in ? d0 : 0) * HW + off);      // (D * HW elements fit 31 bits)
#pragma unroll
        for (int i = 0; i < 8; ++i) __builtin_memcpy(&r.raw[i], x + i * HW + at_d, 8);      // any 2-byte boundary
#pragma unroll
        for (int m = 0; m < kMt; ++m)
            r.a[m] = *reinterpret_cast<const u32x4_t *>(W + w_row[m] + (uint32_t)(in ? d0 : 0));
    };
    floatx4_t acc[kMt][4];
    auto multiply = [&](int group, int step, Step &r) {
        if (step * 32 + 32 > p.D) {                              // uniform: channels past D count as 0
            const uint32_t keep = step * 32 + 8 * kg < p.D ? 0xffffffffu : 0u;
#pragma unroll
            for (int i = 0; i < 8; ++i) { r.raw[i].x &= keep; r.raw[i].y &= keep; }
#pragma unroll
            for (int m = 0; m < kMt; ++m) r.a[m] &= keep;
        }
        // the map's last positions, where the tile does not end on a whole four of them (its size decides that, not the
        // map's: nine rows of an 18 x 18 map end two positions short).  Not the last tile alone: on a map one position wide
        // the tile before it ends inside the map's last four positions as well.  Uniform.
        if (n_pos % 4 != 0 && group == n_groups - 1) {
            const int over = max(0, offset_of(group) - (HW - 4));
#pragma unroll
            for (int i = 0; i < 8; ++i) {
                const uint64_t v = ((uint64_t)r.raw[i].y << 32 | r.raw[i].x) >> (16 * over & 63);
                r.raw[i] = make_uint2((uint32_t)v, (uint32_t)(v >> 32));
            }
        }
#pragma unroll
        for (int s = 0; s < 4; ++s) {
            u32x4_t bf;
#pragma unroll
            for (int m = 0; m < 4; ++m) {
                const uint32_t lo = s < 2 ? r.raw[2 * m].x : r.raw[2 * m].y, hi = s < 2 ? r.raw[2 * m + 1].x : r.raw[2 * m + 1].y;
                bf[m] = __builtin_amdgcn_perm(hi, lo, s % 2 ? 0x07060302u : 0x05040100u);
            }
#pragma unroll
            for (int m = 0; m < kMt; ++m) acc[m][s] = mfma_16x16x32(T{}, r.a[m], bf, acc[m][s]);
        }
    };
    auto clear = [&]() {
#pragma unroll
        for (int m = 0; m < kMt; ++m)
#pragma unroll
            for (int s = 0; s < 4; ++s) acc[m][s] = floatx4_t{0, 0, 0, 0};
    };
    // a lane's accumulators are rows 16 m + 4 kg .. +3 of position pos4 + s of the position-major tile
    auto park = [&](int group) {
#pragma unroll
        for (int s = 0; s < 4; ++s) {
            const int pos = group * kXpGroup + 4 * col + s;
            if (pos < n_pos) {
                uint32_t *row = reinterpret_cast<uint32_t *>(xp_smem + (size_t)pos * p.pitch);
#pragma unroll
                for (int m = 0; m < kMt; ++m) {
                    const int c = m * 16 + 4 * kg;
                    if (c < p.pitch) row[c / 2] = pack2_from_f32<T>(acc[m][s][0], acc[m][s][1]);
                    if (c + 2 < p.pitch) row[c / 2 + 1] = pack2_from_f32<T>(acc[m][s][2], acc[m][s][3]);
                }
            }
        }
    };
    clear();
    if (my_groups > 0) {
        const int n_it = my_groups * my_steps;
        int gl = g_first, sl = part, it_l = 0;                   // the step loaded next
        auto load_next = [&](Step &r) {
            load(gl, sl, r);
            if (it_l + 1 < n_it) {
                ++it_l;
                sl += p.k_split;
                if (sl >= p.k_steps) { sl = part; gl += g_stride; }
            }
        };
        Step ring[kRing];
#pragma unroll
        for (int q = 0; q < kRing; ++q) {
            load_next(ring[q]);
            __builtin_amdgcn_sched_barrier(0);                   // in ring order: the waits count on it
        }
        int group = g_first, step = part;
        for (int it = 0; it < n_it; it += kRing) {
#pragma unroll
            for (int q = 0; q < kRing; ++q) {
                if (it + q < n_it) {                             // uniform
                    multiply(group, step, ring[q]);
                    step += p.k_split;
                    if (step >= p.k_steps) {
                        if (p.k_split == 1) { park(group); clear(); }
                        step = part;
                        group += g_stride;
                    }
                }
                load_next(ring[q]);
            }
        }
    }
    if (p.k_split > 1) {
        // every group has one turn (the host sees to it): the parts of a group are summed pairwise through LDS
        floatx4_t *sums = reinterpret_cast<floatx4_t *>(xp_smem + (((size_t)p.Th * p.Tw * p.pitch + 7) & ~(size_t)7));
        const int group = g_first;
        for (int half = p.k_split / 2; half >= 1; half /= 2) {
            floatx4_t *slot = sums + (size_t)(group * half + part % half) * kMt * 4 * kWave + lane;
            if (part >= half && part < 2 * half) {
#pragma unroll
                for (int m = 0; m < kMt; ++m)
#pragma unroll
                    for (int s = 0; s < 4; ++s) slot[(m * 4 + s) * kWave] = acc[m][s];
            }
            __syncthreads();
            if (part < half) {
#pragma unroll
                for (int m = 0; m < kMt; ++m)
#pragma unroll
                    for (int s = 0; s < 4; ++s) acc[m][s] += slot[(m * 4 + s) * kWave];
            }
            __syncthreads();
        }
        if (part == 0 && group * kXpGroup < n_pos) park(group);
    }
    __syncthreads();

    // ---- out, in scan order -------------------------------------------------------------------------------------------
    const int rows_p = (last_h ? p.Hp : h1) - h0, cols_p = (last_w ? p.Wp : w1) - w0;
    const int n_out = rows_p * cols_p, rows_in = h1 - h0;
    const int64_t L = (int64_t)p.Hp * p.Wp;
    if constexpr (kPaired) {
        // x_proj_pairs: the position-major tile holds rows 2 c and 2 c + 1 in one dword already; kV positions of a plane per lane,
        // and in the place of one more plane the rows B and C
        uint32_t exponents = 0;                                      // bits 15 and 31: an exponent of all ones was among the ranks
        auto emit_pairs = [&](int dir, auto v_tag) {
            const int k = k_first + dir;
            const bool by_cols = k & 1, mirrored = k >= 2;
            const int run = by_cols ? rows_p : cols_p;
            uint16_t *out = reinterpret_cast<uint16_t *>(p.out) + k * p.ks;
            const uint32_t *tile = reinterpret_cast<const uint32_t *>(xp_smem + dir * p.Ce);
            constexpr int kV = decltype(v_tag)::value;
            constexpr int kC = 4;
            const int n_groups = n_out / kV, units = p.planes + 1;
            const float inv_run = 1.0f / (float)run, inv_block = 1.0f / (float)(n_groups * kC);
            const uint32_t one = from_f32<T>(1.0f).bits, per_lane_log2 = p.layout.per_lane == 16 ? 4 : 3;
            const int64_t stream = (b - b % p.layout.images) * L;    // of this image: its first position, its length, the image's place in it
            const uint32_t stream_len = (uint32_t)min((int64_t)p.layout.images * L, p.B * L - stream), in_stream = (uint32_t)(b % p.layout.images * L);
            const int n_items = (units + kC - 1) / kC * n_groups * kC;
            for (int item = threadIdx.x; item < n_items; item += kBlock) {
                int block, idx, line, i;
                small_divmod(item, n_groups * kC, inv_block, block, idx);
                const int unit = block * kC + idx % kC;
                if (unit >= units) continue;
                small_divmod(idx / kC * kV, run, inv_run, line, i);
                const int64_t j = by_cols ? (int64_t)(w0 + line) * p.Hp + h0 + i : (int64_t)(h0 + line) * p.Wp + w0 + i;
                const int64_t at = mirrored ? L - kV - j : j;
                const bool bc = unit == p.planes;
                const int c = bc ? p.rank : 2 * unit;                // row in the low half (bc: B)
                const uint32_t keep = bc ? 0xffffffffu : (c < p.rank ? 0xffffu : 0u) | (c + 1 < p.rank ? 0xffff0000u : 0u);
                const uint32_t added = bc || !p.pair_mask ? 0u : c == p.rank ? one : c + 1 == p.rank ? one << 16 : 0u;
                uint32_t e[kV];
#pragma unroll
                for (int q = 0; q < kV; ++q) {
                    const int h = by_cols ? i : line, w = by_cols ? line : i;
                    e[q] = added;
                    if (h0 + h < p.real_h && w0 + w < p.real_w) {
                        const uint32_t *at_pos = tile + (h * n_cols + w) * (p.pitch / 2) + c / 2;
                        e[q] = bc && c % 2 ? at_pos[0] >> 16 | at_pos[1] << 16 : at_pos[0] & keep;
                    }
                    if (++i == run) { i = 0; ++line; }
                }
                if (!bc) {
                    constexpr uint32_t kExp = std::is_same<T, bf16_t>::value ? 0x7f80u : 0x7c00u, kUlp = kExp & ~(kExp << 1);
#pragma unroll
                    for (int q = 0; q < kV; ++q) exponents |= (e[q] & (kExp | kExp << 16)) + (kUlp | kUlp << 16);
                    // the place of the stream's position s: DtsLayout
                    const uint32_t s = in_stream + (uint32_t)at, pass_len = kWave << per_lane_log2;
                    const uint32_t first = s & ~(pass_len - 1), lane_of = (s - first) >> per_lane_log2, g = (s & ((1u << per_lane_log2) - 1)) / 4;
                    const uint32_t lanes = min(pass_len, stream_len - first) >> per_lane_log2;
                    uint32_t *dst = reinterpret_cast<uint32_t *>(out + 2 * unit * p.cs) + stream + first;
                    if constexpr (kV == 1) {
                        dst[(g * lanes + lane_of) * 4 + s % 4] = e[0];
                    } else {
#pragma unroll
                        for (int q = 0; q < kV / 4; ++q)
                            reinterpret_cast<uint4 *>(dst)[(g + q) * lanes + lane_of] = mirrored ? make_uint4(e[kV - 1 - 4 * q], e[kV - 2 - 4 * q], e[kV - 3 - 4 * q], e[kV - 4 - 4 * q])
                                                                         : make_uint4(e[4 * q], e[4 * q + 1], e[4 * q + 2], e[4 * q + 3]);
                    }
                    continue;
                }
#pragma unroll
                for (int row = 0; row < 2; ++row) {
                    uint16_t *dst = out + (2 * p.planes + row) * p.cs + b * L + at;
                    if constexpr (kV == 1) {
                        *dst = (uint16_t)(row ? e[0] >> 16 : e[0]);
                    } else {
                        uint32_t wds[kV / 2];
#pragma unroll
                        for (int q = 0; q < kV / 2; ++q) {
                            const uint32_t lo = mirrored ? e[kV - 1 - 2 * q] : e[2 * q], hi = mirrored ? e[kV - 2 - 2 * q] : e[2 * q + 1];
                            wds[q] = __builtin_amdgcn_perm(hi, lo, row ? 0x07060302u : 0x05040100u);
                        }
                        if constexpr (kV == 8) *reinterpret_cast<uint4 *>(dst) = make_uint4(wds[0], wds[1], wds[2], wds[3]);
                        else *reinterpret_cast<uint2 *>(dst) = make_uint2(wds[0], wds[1]);
                    }
                }
            }
        };
        for (int dir = 0; dir < p.n_dirs; ++dir) {
            const int v = (k_first + dir) & 1 ? p.v_col : p.v_row;
            if (v == 8) emit_pairs(dir, std::integral_constant<int, 8>{});
            else if (v == 4) emit_pairs(dir, std::integral_constant<int, 4>{});
            else emit_pairs(dir, std::integral_constant<int, 1>{});
        }
        const int found = __syncthreads_or((int)(exponents & 0x80008000u));
        if (threadIdx.x == 0) p.flags[wg] = found;
    } else {
        // kV consecutive scan positions of rows 2 c2 and 2 c2 + 1 per lane (one dword per position: the tile's pitch is an odd
        // number of dwords, so that lanes 8 positions apart meet in few banks), kC row pairs side by side in a wavefront
        auto emit = [&](int dir, auto v_tag) {
            const int k = k_first + dir;
            const bool by_cols = k & 1, mirrored = k >= 2;
            const int run = by_cols ? rows_p : cols_p;               // positions per line of the scan inside the tile
            uint16_t *out = reinterpret_cast<uint16_t *>(p.out) + k * p.ks + b * p.bs;
            const uint32_t *tile = reinterpret_cast<const uint32_t *>(xp_smem + dir * p.Ce);
            constexpr int kV = decltype(v_tag)::value;
            constexpr int kC = kV > 1 ? 4 : 1;
            const int n_groups = n_out / kV, pairs = (p.C + 1) / 2;
            const float inv_run = 1.0f / (float)run, inv_block = 1.0f / (float)(n_groups * kC);
            auto store = [&](int row, int64_t j, const uint32_t (&e)[kV]) {       // e: 16 bits each
                uint16_t *dst = out + row * p.cs + (mirrored ? L - kV - j : j);
                if constexpr (kV == 1) {
                    *dst = (uint16_t)e[0];
                } else {
                    uint32_t wds[kV / 2];
#pragma unroll
                    for (int q = 0; q < kV / 2; ++q)
                        wds[q] = mirrored ? e[kV - 1 - 2 * q] | e[kV - 2 - 2 * q] << 16 : e[2 * q] | e[2 * q + 1] << 16;
                    if constexpr (kV == 8) *reinterpret_cast<uint4 *>(dst) = make_uint4(wds[0], wds[1], wds[2], wds[3]);
                    else *reinterpret_cast<uint2 *>(dst) = make_uint2(wds[0], wds[1]);
                }
            };
            auto scan_index = [&](int line, int i) {
                return by_cols ? (int64_t)(w0 + line) * p.Hp + h0 + i : (int64_t)(h0 + line) * p.Wp + w0 + i;
            };
            const int n_items = (pairs + kC - 1) / kC * n_groups * kC;
            for (int item = threadIdx.x; item < n_items; item += kBlock) {
                int block, idx, line, i;
                small_divmod(item, n_groups * kC, inv_block, block, idx);
                const int c2 = block * kC + idx % kC;
                if (c2 >= pairs) continue;
                small_divmod(idx / kC * kV, run, inv_run, line, i);
                const int64_t j = scan_index(line, i);
                uint32_t e[kV];
#pragma unroll
                for (int q = 0; q < kV; ++q) {
                    const int h = by_cols ? i : line, w = by_cols ? line : i;
                    e[q] = h < rows_in && w < n_cols ? tile[(h * n_cols + w) * (p.pitch / 2) + c2] : 0u;
                    if (++i == run) { i = 0; ++line; }
                }
                uint32_t half[kV];
                const int c = 2 * c2, shift = p.mask_row >= 0 ? p.mask_row : p.C;      // rows from the mask row on move up by one
#pragma unroll
                for (int q = 0; q < kV; ++q) half[q] = e[q] & 0xffffu;
                store(c + (c >= shift), j, half);
                if (c + 1 < p.C) {
#pragma unroll
                    for (int q = 0; q < kV; ++q) half[q] = e[q] >> 16;
                    store(c + 1 + (c + 1 >= shift), j, half);
                }
            }
            if (p.mask_row < 0) return;
            for (int idx = threadIdx.x; idx < n_groups; idx += kBlock) {
                int line, i;
                small_divmod(idx * kV, run, inv_run, line, i);
                const int64_t j = scan_index(line, i);
                uint32_t e[kV];
#pragma unroll
                for (int q = 0; q < kV; ++q) {
                    const int h = by_cols ? i : line, w = by_cols ? line : i;
                    e[q] = h < rows_in && w < n_cols ? 0u : from_f32<T>(1.0f).bits;
                    if (++i == run) { i = 0; ++line; }
                }
                store(p.mask_row, j, e);
            }
        };
        for (int dir = 0; dir < p.n_dirs; ++dir) {
            const int v = (k_first + dir) & 1 ? p.v_col : p.v_row;
            if (v == 8) emit(dir, std::integral_constant<int, 8>{});
            else if (v == 4) emit(dir, std::integral_constant<int, 4>{});
            else emit(dir, std::integral_constant<int, 1>{});
        }
    }
}

template <typename T>
static int launch_x_proj(const XProjArgs &a, size_t smem, int m_tiles, hipStream_t s) {
#define SS2D_XP_LAUNCH(M) \
    do {                                                                                                            \
        if (a.planes > 0) hipLaunchKernelGGL((x_proj_kernel<T, M, true>), dim3(a.total), dim3(kBlock), smem, s, a);    \
        else hipLaunchKernelGGL((x_proj_kernel<T, M, false>), dim3(a.total), dim3(kBlock), smem, s, a);                \
    } while (0)
    if (m_tiles == 1) SS2D_XP_LAUNCH(1);
    else if (m_tiles == 2) SS2D_XP_LAUNCH(2);
    else if (m_tiles == 3) SS2D_XP_LAUNCH(3);
    else if (m_tiles == 4) SS2D_XP_LAUNCH(4);
    else SS2D_XP_LAUNCH(6);
#undef SS2D_XP_LAUNCH
    return launch_status();
}

static int64_t xp_gcd(int64_t a, int64_t b) { while (b) { const int64_t t = a % b; a = b; b = t; } return a < 0 ? -a : a; }

// How a problem is cut: everything but the pointers, the output's strides and the stores' width.  SS2D_ENOTSUP: no variant.
static int x_proj_plan(int B, int D, int C, int H, int W, int Hp, int Wp, int dtype, XProjArgs &a, int &m_tiles, size_t &smem) {
    const int64_t HW = (int64_t)H * W, L = (int64_t)Hp * Wp;
    // 8 channels of a weight row are one 16-byte load; at most 96 output rows (six accumulator tiles)
    if (dtype == SS2D_F32 || D == 0 || D % 8 != 0 || C > 96 || HW < 8 || L > 0x0fffffff || (int64_t)D * HW > 0x7fffffff) return SS2D_ENOTSUP;
    a.D = D; a.C = C; a.H = H; a.Wd = W; a.Hp = Hp; a.Wp = Wp;
    a.Ce = (C + 1) & ~1;
    // Directions per workgroup: each set reads the map again, from L2, and that re-reading is what bounds the kernel (loads
    // alone, one direction per workgroup: 30 of 37 us at 96 x 56 x 56, batch 128).  As many as four accumulator tiles hold,
    // halved while the grid would leave compute units idle: all four 25-28 us against 37 with one (192 x 28 x 28: 20 against
    // 24; two at 384 x 14 x 14: 16.5 against 18.4), but one image of 28 x 28 10.5 us against 8.7 with one.
    a.n_dirs = 4 * a.Ce <= 64 ? 4 : 2 * a.Ce <= 64 ? 2 : 1;
    a.k_steps = (D + 31) / 32;
    // Tiles: up to 96 columns whole rows, else pieces of about 64 (a multiple of 8); as many rows as 32 KB of LDS hold (five
    // workgroups per CU; 24 to 64 KB measured the same within 10 %) -- the transposing directions write runs of that many
    // elements --, fewer while the grid has less than two workgroups per CU.
    a.tiles_w = W <= 96 || W % 4 != 0 ? 1 : (W + 63) / 64;
    a.Tw = a.tiles_w == 1 ? W : ((W + a.tiles_w - 1) / a.tiles_w + 7) & ~7;
    a.tiles_w = (W + a.Tw - 1) / a.Tw;
    const int unit = H % 8 == 0 ? 8 : H % 4 == 0 ? 4 : 1;         // rows per tile a multiple of this keep the wide stores
    auto even = [&](int64_t t) {                                   // the same number of tiles, evened out
        const int64_t n = (H + t - 1) / t;
        t = ((H + n - 1) / n + unit - 1) / unit * unit;
        return t > H ? (int64_t)H : t;
    };
    constexpr int64_t kMostLds = 128 * 1024;
    int64_t Th = 1, row_bytes = 0, total = 0;
    for (;; a.n_dirs /= 2) {
        const int rows = a.n_dirs * a.Ce;
        a.pitch = rows + (rows / 2 % 2 == 0 ? 2 : 0);             // an odd number of dwords per position
        row_bytes = (int64_t)a.Tw * a.pitch * 2;
        const int64_t small = 32 * 1024 / row_bytes, large = 64 * 1024 / row_bytes;
        Th = small >= unit ? small : large < unit ? large : unit;
        Th = Th < 1 ? 1 : Th > H ? H : Th;
        if (Th >= unit) Th = even(Th < H ? Th / unit * unit : Th);
        auto grid = [&](int64_t t) { return (int64_t)B * (4 / a.n_dirs) * a.tiles_w * ((H + t - 1) / t); };
        while (Th > 16 && grid(Th) < 512) Th = even((Th + 1) / 2);
        total = grid(Th);
        if (a.n_dirs == 1 || (total >= 256 && row_bytes * Th <= kMostLds)) break;
    }
    // Few workgroups walk all channels of a large tile one step after the other while most of the chip idles: tiles of half
    // the rows -- multiples of 4 where they were, for the wide stores -- double the grid, and from two column groups down the
    // wavefronts share the channels as well (k_split below).  One image, bf16: 768 x 56 x 56, C = 50 34.5 -> 12.9 us, 336 x 45 x 45,
    // C = 23 25.2 -> 8.2, 192 x 28 x 28, C = 14 9.3 -> 6.8.  From 160 workgroups on it costs more than it gives (at 192: 48 images
    // of 384 x 14 x 14, C = 32 11.9 -> 15.3).
    const bool few = total < 160;
    while (total < 160 && Th > 1 && Th * a.Tw > kXpGroup) {
        int64_t t = (Th + 1) / 2;
        if (unit > 1 && t > 2) t = (t + 3) / 4 * 4;
        if (t >= Th) break;
        Th = t;
        total = (int64_t)B * (4 / a.n_dirs) * a.tiles_w * ((H + Th - 1) / Th);
    }
    // A few hundred workgroups pass through the 256 compute units in two or three rounds, and a plan that fills the last of them is worth more than one that shares
    // more of x: a workgroup's time is that of its steps of 32 channels, a turn of four column groups at a time, of the results it puts into order, and a part it has in
    // any case; up to four rounds count whole.  The constants order 1700 measured plans of 60 sizes; a plan is left only for one that this
    // puts a tenth ahead, and not where the channels are few or shared out (k_split), or the rows no multiple of 4, which it knows nothing of.  us, before / so: 20 x 208 maps of 96 x 96 38.9 / 28.6, 125 x 528 of 20 x 20 41.7 / 31.2, 2 x 480 of 84 x 112
    // 22.4 / 18.7, 15 x 496 of 64 x 64 37.1 / 31.4; 90 other sizes 1.02 in the mean, the worst 52.7 / 53.6.
    auto cost = [&](int dirs, int64_t t) {
        const int64_t wgs = (int64_t)B * (4 / dirs) * a.tiles_w * ((H + t - 1) / t), pos = t * a.Tw, out_rows = dirs * a.Ce;
        const double own = (double)((pos + 4 * kXpGroup - 1) / (4 * kXpGroup)) * a.k_steps + 0.003 * pos * out_rows + 2.0;
        return own * (wgs <= 256 ? 1.1 : wgs <= 1024 ? (double)((wgs + 255) / 256) : wgs / 256.0 + 0.5);
    };
    if (!few && D >= 128 && H % 4 == 0 && Th * a.Tw > 2 * kXpGroup) {
        double least = 0.9 * cost(a.n_dirs, Th);
        for (int dirs = 4; dirs >= 1; dirs /= 2) {
            const int out_rows = dirs * a.Ce, pitch = out_rows + (out_rows / 2 % 2 == 0 ? 2 : 0);
            for (int64_t t = 4; out_rows <= 96 && t <= H && t * a.Tw * pitch * 2 <= 64 * 1024; t += 4) {
                if (t * a.Tw <= 2 * kXpGroup || cost(dirs, t) >= least) continue;
                least = cost(dirs, t);
                a.n_dirs = dirs; a.pitch = pitch;
                Th = t;
            }
        }
        row_bytes = (int64_t)a.Tw * a.pitch * 2;
        total = (int64_t)B * (4 / a.n_dirs) * a.tiles_w * ((H + Th - 1) / Th);
    }
    // a row of a width that is no multiple of 4 is not cut: there is a widest one
    if (total > 0x7fffffff || row_bytes * Th > kMostLds || Th * a.Tw * a.pitch > (1 << 22)) return SS2D_ENOTSUP;
    a.total = (uint32_t)total;
    a.Th = (int)Th;
    a.tiles_h = (int)((H + Th - 1) / Th);
    // small_divmod's range: the largest tile on the way out, with the added rows and columns that the last one carries
    const int64_t tail_h = Hp - (int64_t)(a.tiles_h - 1) * Th, tail_w = Wp - (int64_t)(a.tiles_w - 1) * a.Tw;
    if ((tail_h > Th ? tail_h : Th) * (tail_w > a.Tw ? tail_w : a.Tw) * ((a.Ce / 2 + 3) & ~3) >= 1 << 23) return SS2D_ENOTSUP;
    const int64_t n_groups = (Th * a.Tw + kXpGroup - 1) / kXpGroup;
    // maps of one or two column groups: the wavefronts split the channels
    const int n_waves = kBlock / kWave;
    a.k_split = 1;
    while (a.k_split * 2 * n_groups <= n_waves && a.k_split * 2 <= a.k_steps) a.k_split *= 2;
    const int rows = a.n_dirs * a.Ce;
    m_tiles = rows <= 16 ? 1 : rows <= 32 ? 2 : rows <= 48 ? 3 : rows <= 64 ? 4 : 6;
    smem = ((size_t)row_bytes * Th + 15) & ~(size_t)15;
    if (a.k_split > 1) smem += (size_t)(n_waves / 2) * m_tiles * 4 * kWave * sizeof(floatx4_t);
    return SS2D_OK;
}

// The pointers, the output's strides and the stores' width, and the launch.
static int x_proj_run(XProjArgs &a, const void *x, const void *weight, void *out, int Hp, int Wp, int64_t ks, int64_t cs, int64_t bs,
                      size_t smem, int m_tiles, int dtype, hipStream_t s) {
    if (reinterpret_cast<uintptr_t>(weight) % 16 != 0) return SS2D_ENOTSUP;
    a.x = x; a.W = weight; a.out = out;
    a.ks = ks; a.cs = cs; a.bs = bs;
    // elements per store: what divides every row base, the scan's length and the starts of the tiles' lines
    const int64_t L = (int64_t)Hp * Wp;
    int64_t g = xp_gcd(xp_gcd(8, a.ks), xp_gcd(a.cs, a.bs));
    g = xp_gcd(g, xp_gcd(L, (int64_t)(reinterpret_cast<uintptr_t>(out) % 16 / 2)));
    if (reinterpret_cast<uintptr_t>(out) % 2 != 0) return SS2D_EINVAL;
    const int64_t row_start = a.tiles_w == 1 ? (int64_t)a.Th * Wp : xp_gcd(Wp, a.Tw), col_start = a.tiles_h == 1 ? (int64_t)a.Tw * Hp : xp_gcd(Hp, a.Th);
    const int64_t vr = xp_gcd(g, row_start), vc = xp_gcd(g, col_start);
    a.v_row = (int)(vr == 2 ? 1 : vr);
    a.v_col = (int)(vc == 2 ? 1 : vc);
    return dtype == SS2D_BF16 ? launch_x_proj<bf16_t>(a, smem, m_tiles, s) : launch_x_proj<f16_t>(a, smem, m_tiles, s);
}

int x_proj_pairs_workgroups(int B, int D, int R, int H, int W, int dtype) {
    XProjArgs a;
    int m_tiles;
    size_t smem;
    if (R < 1 || B < 1 || x_proj_plan(B, D, R + 2, H, W, H, W, dtype, a, m_tiles, smem) != SS2D_OK) return 0;
    return (int)(a.total / (uint32_t)B);
}

int x_proj_pairs(const void *x, const void *weight, void *out, int32_t *flags, int B, int D, int R, int H, int W, int real_h, int real_w, int64_t dir_stride,
                 int64_t row_stride, const DtsLayout &layout, int dtype, void *stream) {
    XProjArgs a;
    int m_tiles;
    size_t smem;
    const int rc = x_proj_plan(B, D, R + 2, H, W, H, W, dtype, a, m_tiles, smem);
    if (rc != SS2D_OK) return rc;
    const int64_t L = (int64_t)H * W;
    if (reinterpret_cast<uintptr_t>(out) % 16 != 0 || (dir_stride | row_stride) % 8 != 0 || (layout.per_lane != 8 && layout.per_lane != 16) ||
        L % layout.per_lane != 0 || layout.images < 1 || layout.images * L > 0x7fffffff) return SS2D_EINVAL;
    a.layout = layout; a.B = B;
    a.mask_row = -1;
    a.real_h = real_h; a.real_w = real_w;
    a.flags = flags; a.rank = R; a.pair_mask = real_h != H || real_w != W; a.planes = dts_planes(R, a.pair_mask);
    return x_proj_run(a, x, weight, out, H, W, dir_stride, row_stride, L, smem, m_tiles, dtype, (hipStream_t)stream);
}

}  // namespace ss2d

extern "C" int ss2d_x_proj_applies(int B, int D, int C, int H, int W, int dtype) {
    using namespace ss2d;
    if (B < 0 || D < 0 || C < 0 || H < 0 || W < 0 || (dtype != SS2D_F32 && dtype != SS2D_BF16 && dtype != SS2D_F16)) return SS2D_EINVAL;
    if (B == 0 || C == 0 || H == 0 || W == 0) return SS2D_OK;
    XProjArgs a;
    int m_tiles;
    size_t smem;
    return x_proj_plan(B, D, C, H, W, H, W, dtype, a, m_tiles, smem);
}

extern "C" int ss2d_x_proj(const void *x, const void *weight, void *out, int B, int D, int C, int H, int W, int Hp, int Wp,
                           int mask_row, int64_t out_dir_stride, int64_t out_chan_stride, int64_t out_batch_stride, int dtype,
                           void *stream) {
    using namespace ss2d;
    if (B < 0 || D < 0 || C < 0 || H < 0 || W < 0 || Hp < H || Wp < W || mask_row > C) return SS2D_EINVAL;
    if (dtype != SS2D_F32 && dtype != SS2D_BF16 && dtype != SS2D_F16) return SS2D_EINVAL;
    if (out_dir_stride < 0 || out_chan_stride < 0 || out_batch_stride < 0) return SS2D_EINVAL;
    if (B == 0 || C == 0 || H == 0 || W == 0) return SS2D_OK;
    if (!x || !weight || !out) return SS2D_EINVAL;
    XProjArgs a;
    int m_tiles;
    size_t smem;
    const int rc = x_proj_plan(B, D, C, H, W, Hp, Wp, dtype, a, m_tiles, smem);
    if (rc != SS2D_OK) return rc;
    a.mask_row = mask_row < 0 ? -1 : mask_row;
    a.rank = a.planes = a.pair_mask = 0;
    a.flags = nullptr;
    a.layout = {8, 1}; a.B = B; a.real_h = H; a.real_w = W;
    return x_proj_run(a, x, weight, out, Hp, Wp, out_dir_stride, out_chan_stride, out_batch_stride, smem, m_tiles, dtype, (hipStream_t)stream);
}
