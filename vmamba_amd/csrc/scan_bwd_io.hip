// What stands around the selective-scan backward kernel (selective_scan_oflex.cpp:310-352): its accumulators cleared, and the
// fp32 dB / dC rounded to the type of B / C.  As one fill per tensor and one conversion each these were seven launches of about
// 5 us on a few MB at most, bound by launch and drain; here one launch each for all of them (forward and backward of the three
// operators: 594 -> 585 us on 64 x 96 maps of 56 x 56, 553 -> 547 on 16 x 192 of 28 x 28 with 16 states).
#include "ss2d_common.h"

namespace ss2d {

constexpr int kClearMax = SS2D_CLEAR_MAX;
constexpr int kClearBlockBytes = 4 * kBlock * 16;        // four 16-byte stores per thread

struct ClearArgs {
    void *ptr[kClearMax];
    int64_t bytes[kClearMax];
    uint32_t first[kClearMax + 1];       // a tensor's first workgroup
    int32_t n;
};

__global__ __launch_bounds__(kBlock) void clear_kernel(const ClearArgs p) {
    int t = 0;
    while (t + 1 < p.n && blockIdx.x >= p.first[t + 1]) ++t;         // uniform
    char *dst = reinterpret_cast<char *>(p.ptr[t]);
    const int64_t bytes = p.bytes[t], base = (int64_t)(blockIdx.x - p.first[t]) * kClearBlockBytes;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        const int64_t at = base + (i * kBlock + (int)threadIdx.x) * 16;
        if (at + 16 <= bytes) *reinterpret_cast<uint4 *>(dst + at) = make_uint4(0, 0, 0, 0);
        else for (int64_t q = at; q < bytes; q += 4) *reinterpret_cast<uint32_t *>(dst + q) = 0;
    }
}

struct RoundArgs {
    const float *src[2];
    void *dst[2];
    int64_t n[2];
    uint32_t first;                      // the second tensor's first workgroup
};

template <typename T>
__global__ __launch_bounds__(kBlock) void round_pair_kernel(const RoundArgs p) {
    const int t = blockIdx.x >= p.first;
    const float *src = p.src[t];
    T *dst = reinterpret_cast<T *>(p.dst[t]);
    const int64_t i = ((int64_t)(blockIdx.x - (t ? p.first : 0)) * kBlock + threadIdx.x) * 8;
    if (i + 8 <= p.n[t]) {
        const float4 a = *reinterpret_cast<const float4 *>(src + i), b = *reinterpret_cast<const float4 *>(src + i + 4);
        *reinterpret_cast<uint4 *>(dst + i) = make_uint4(pack2_from_f32<T>(a.x, a.y), pack2_from_f32<T>(a.z, a.w),
                                                         pack2_from_f32<T>(b.x, b.y), pack2_from_f32<T>(b.z, b.w));
    } else {
        for (int64_t q = i; q < p.n[t]; ++q) dst[q] = from_f32<T>(src[q]);
    }
}

}  // namespace ss2d

extern "C" int ss2d_clear(void *const *ptrs, const int64_t *bytes, int n, void *stream) {
    using namespace ss2d;
    if (n < 0 || n > kClearMax || (n > 0 && (!ptrs || !bytes))) return SS2D_EINVAL;
    ClearArgs a;
    a.n = 0;
    int64_t wgs = 0;
    for (int i = 0; i < n; ++i) {
        if (bytes[i] < 0 || bytes[i] % 4 != 0) return SS2D_EINVAL;
        if (bytes[i] == 0) continue;
        if (!ptrs[i] || reinterpret_cast<uintptr_t>(ptrs[i]) % 16 != 0) return SS2D_EINVAL;
        a.ptr[a.n] = ptrs[i]; a.bytes[a.n] = bytes[i]; a.first[a.n] = (uint32_t)wgs;
        ++a.n;
        wgs += (bytes[i] + kClearBlockBytes - 1) / kClearBlockBytes;
        if (wgs > 0x7fffffff) return SS2D_ENOTSUP;
    }
    if (a.n == 0) return SS2D_OK;
    a.first[a.n] = (uint32_t)wgs;
    hipLaunchKernelGGL(clear_kernel, dim3((uint32_t)wgs), dim3(kBlock), 0, (hipStream_t)stream, a);
    return launch_status();
}

extern "C" int ss2d_round_pair(const float *src0, void *dst0, int64_t n0, const float *src1, void *dst1, int64_t n1, int dtype,
                               void *stream) {
    using namespace ss2d;
    if (n0 < 0 || n1 < 0 || (dtype != SS2D_BF16 && dtype != SS2D_F16)) return SS2D_EINVAL;
    if (n0 + n1 == 0) return SS2D_OK;
    if ((n0 && (!src0 || !dst0)) || (n1 && (!src1 || !dst1))) return SS2D_EINVAL;
    const uintptr_t all = reinterpret_cast<uintptr_t>(src0) | reinterpret_cast<uintptr_t>(dst0) | reinterpret_cast<uintptr_t>(src1) |
                          reinterpret_cast<uintptr_t>(dst1);
    if (all % 16 != 0) return SS2D_EINVAL;
    const int64_t w0 = (n0 + 8 * kBlock - 1) / (8 * kBlock), w1 = (n1 + 8 * kBlock - 1) / (8 * kBlock);
    if (w0 + w1 > 0x7fffffff) return SS2D_ENOTSUP;
    RoundArgs a;
    a.src[0] = src0; a.src[1] = src1; a.dst[0] = dst0; a.dst[1] = dst1; a.n[0] = n0; a.n[1] = n1;
    a.first = (uint32_t)w0;
    hipStream_t s = (hipStream_t)stream;
    if (dtype == SS2D_BF16) hipLaunchKernelGGL(round_pair_kernel<bf16_t>, dim3((uint32_t)(w0 + w1)), dim3(kBlock), 0, s, a);
    else hipLaunchKernelGGL(round_pair_kernel<f16_t>, dim3((uint32_t)(w0 + w1)), dim3(kBlock), 0, s, a);
    return launch_status();
}
