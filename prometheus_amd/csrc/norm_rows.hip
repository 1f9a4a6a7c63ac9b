// norm_rows.hip — K11: the row normalisation of the model's linear attention
// (model/__init__.py:203-205, x / max(||x||, 1e-6)) and its reverse, each one pass over q
// and k, for the backward (the forward normalises inside its kernels).
//
// Memory-bound: a lane holds eight consecutive elements of a row (16 or 32 bytes), D / 8
// adjacent lanes a row, summed by DPP, so every row is read once and written once in
// coalesced 16-byte accesses.  As elementwise tensor operations these took about twenty
// passes (650 of a 1,042 us training step at B4 T2048 H16 D128, bf16); here 2 x 134 and 268 MB
// are moved once.  Rows whose length is not a multiple of 8, or misaligned ones, take one wave
// a row with element accesses.

#include "pm_common.h"
#include "pm_internal.h"
#include "pm_rec.h"

// (multiply-adds are fused only where written so)
#pragma clang fp contract(off)

namespace pm {
namespace {

constexpr float kEps = 1e-6f;
__device__ __forceinline__ float floored(float n) { return n < kEps ? kEps : n; }  // (NaN stays)

template <typename T>
__device__ __forceinline__ void load8(const T* p, float (&x)[8]);
template <>
__device__ __forceinline__ void load8<float>(const float* p, float (&x)[8]) {
    const float4 a = reinterpret_cast<const float4*>(p)[0], b = reinterpret_cast<const float4*>(p)[1];
    x[0] = a.x, x[1] = a.y, x[2] = a.z, x[3] = a.w, x[4] = b.x, x[5] = b.y, x[6] = b.z, x[7] = b.w;
}
template <>
__device__ __forceinline__ void load8<uint16_t>(const uint16_t* p, float (&x)[8]) {
    const uint4 a = *reinterpret_cast<const uint4*>(p);
    const uint32_t w[4] = {a.x, a.y, a.z, a.w};
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        x[2 * i] = __uint_as_float(w[i] << 16);
        x[2 * i + 1] = __uint_as_float(w[i] & 0xffff0000u);
    }
}
template <typename T>
__device__ __forceinline__ void store8(T* p, const float (&x)[8]);
template <>
__device__ __forceinline__ void store8<float>(float* p, const float (&x)[8]) {
    reinterpret_cast<float4*>(p)[0] = make_float4(x[0], x[1], x[2], x[3]);
    reinterpret_cast<float4*>(p)[1] = make_float4(x[4], x[5], x[6], x[7]);
}
template <>
__device__ __forceinline__ void store8<uint16_t>(uint16_t* p, const float (&x)[8]) {
    uint32_t w[4];
#pragma unroll
    for (int i = 0; i < 4; ++i)
        w[i] = static_cast<uint32_t>(f32_to_bf16(x[2 * i])) | (static_cast<uint32_t>(f32_to_bf16(x[2 * i + 1])) << 16);
    *reinterpret_cast<uint4*>(p) = make_uint4(w[0], w[1], w[2], w[3]);
}

// Sum over a row of the eight values of each of its LPR = D / 8 lanes, in the order of the
// elementwise tensor operations that these kernels stand for: pairs of neighbours throughout at
// D = 64, four consecutive values in sequence and then pairs of neighbours from D = 128 on.  The
// bf16 gradients follow the rounding of the normalised rows to bf16, which another order of
// their norm's sum moves by one unit here and there (1e-3 of the gradients).
template <int LPR>
__device__ __forceinline__ float row_sum8(const float (&y)[8]) {
    float s;
    if constexpr (LPR == 8) s = ((y[0] + y[1]) + (y[2] + y[3])) + ((y[4] + y[5]) + (y[6] + y[7]));
    else s = (((y[0] + y[1]) + y[2]) + y[3]) + (((y[4] + y[5]) + y[6]) + y[7]);
    return lane_sum<LPR>(s);
}
// ... and over a row of any D <= 256 by one wave: f(acc, d) adds element d's value to acc.
// Below 128 elements lane l takes elements l and l + n in two sums, n the power of two at most D
// (and 64); from there on it takes the four elements from 4 l on and from 4 (l + n) on in four,
// n the power of two at most D / 4.  (From 128 on with a remainder of D / 4 those operations' order
// follows each row's alignment; this is the one of aligned rows.)
template <typename F>
__device__ __forceinline__ float row_sum_any(int D, int lane, F f) {
    const int n = 1 << min(6, 31 - __clz(D < 128 ? D : D / 4));
    float a[4] = {0.f, 0.f, 0.f, 0.f};
    if (lane < n) {
        if (D < 128) {
            a[0] = f(0.f, lane);
            if (lane + n < D) a[1] = f(0.f, lane + n);
        } else {
            for (int v = lane; v < D / 4; v += n)
#pragma unroll
                for (int e = 0; e < 4; ++e) a[e] = f(a[e], 4 * v + e);
            if (lane < D % 4) a[0] = f(a[0], D - D % 4 + lane);
        }
    }
    return lane_sum<64>(((a[0] + a[1]) + a[2]) + a[3]);
}

// One element of the gradient of y = x / m, m = max(n, eps), n = ||x||, given g = dL/dy and dot
// = sum -g (x / m) / m = dL/dm: the norm's part only where the norm counts (live: at and above
// the bound; a row with a NaN gives NaNs through m).  norm_dot is one element of dot.
__device__ __forceinline__ float norm_dot(float g, float x, float m) { return -g * ((x / m) / m); }
__device__ __forceinline__ float norm_grad(float g, float x, float m, float dot, bool live) {
    return g / m + (live ? dot : 0.f) * (x / m);
}

// LPR = D / 8 lanes per row; 2 * rows rows in all, q's then k's
template <typename T, int LPR>
__global__ __launch_bounds__(256) void norm_rows_kernel(const T* __restrict__ q, const T* __restrict__ k,
                                                        T* __restrict__ qn, T* __restrict__ kn,
                                                        float* __restrict__ ones, size_t n_ones, long rows) {
    const long t = static_cast<long>(blockIdx.x) * 256 + threadIdx.x;
    const long step = static_cast<long>(gridDim.x) * 256, n = 2 * rows * LPR;
    for (long i = t; i < n; i += step) {
        const bool second = i >= rows * LPR;
        const long o = (second ? i - rows * LPR : i) * 8;
        float x[8], y[8];
        load8<T>((second ? k : q) + o, x);
#pragma unroll
        for (int e = 0; e < 8; ++e) y[e] = x[e] * x[e];
        const float m = floored(sqrtf(row_sum8<LPR>(y)));  // (a row's lanes are adjacent and all in range together)
#pragma unroll
        for (int e = 0; e < 8; ++e) x[e] = x[e] / m;
        store8<T>((second ? kn : qn) + o, x);
    }
    for (size_t i = t; i < n_ones; i += step) ones[i] = 1.f;
}

template <typename T, int LPR>
__global__ __launch_bounds__(256) void norm_rows_bwd_kernel(const T* __restrict__ q, const T* __restrict__ k,
                                                            const float* __restrict__ gqn,
                                                            const float* __restrict__ gkn, T* __restrict__ gq,
                                                            T* __restrict__ gk, long rows) {
    const long step = static_cast<long>(gridDim.x) * 256, n = 2 * rows * LPR;
    for (long i = static_cast<long>(blockIdx.x) * 256 + threadIdx.x; i < n; i += step) {
        const bool second = i >= rows * LPR;
        const long o = (second ? i - rows * LPR : i) * 8;
        float x[8], g[8], y[8];
        load8<T>((second ? k : q) + o, x);
        load8<float>((second ? gkn : gqn) + o, g);
#pragma unroll
        for (int e = 0; e < 8; ++e) y[e] = x[e] * x[e];
        const float nrm = sqrtf(row_sum8<LPR>(y)), m = floored(nrm);
#pragma unroll
        for (int e = 0; e < 8; ++e) y[e] = norm_dot(g[e], x[e], m);
        const float dot = row_sum8<LPR>(y);
#pragma unroll
        for (int e = 0; e < 8; ++e) g[e] = norm_grad(g[e], x[e], m, dot, nrm >= kEps);
        store8<T>((second ? gk : gq) + o, g);
    }
}

// any D: one wave per row, element accesses
template <typename T, bool BWD>
__global__ __launch_bounds__(256) void norm_rows_any_kernel(const T* __restrict__ q, const T* __restrict__ k,
                                                            const float* __restrict__ gqn,
                                                            const float* __restrict__ gkn, T* __restrict__ oq,
                                                            T* __restrict__ ok, float* __restrict__ ones,
                                                            size_t n_ones, long rows, int D) {
    const int lane = threadIdx.x & 63;
    const long wave = static_cast<long>(blockIdx.x) * 4 + (threadIdx.x >> 6), waves = static_cast<long>(gridDim.x) * 4;
    for (long i = wave; i < 2 * rows; i += waves) {
        const bool second = i >= rows;
        const long o = (second ? i - rows : i) * D;
        const T* x = (second ? k : q) + o;
        const float* g = BWD ? (second ? gkn : gqn) + o : nullptr;
        const float nrm = sqrtf(row_sum_any(D, lane, [=](float acc, int d) {
            const float a = to_f32<T>(x[d]);
            return fmaf(a, a, acc);
        }));
        const float m = floored(nrm);
        float dot = 0.f;
        if constexpr (BWD)
            dot = row_sum_any(D, lane, [=](float acc, int d) { return acc + norm_dot(g[d], to_f32<T>(x[d]), m); });
        T* y = (second ? ok : oq) + o;
        for (int d = lane; d < D; d += 64) {
            const float a = to_f32<T>(x[d]);
            y[d] = from_f32<T>(BWD ? norm_grad(g[d], a, m, dot, nrm >= kEps) : a / m);
        }
    }
    if (!BWD)
        for (size_t i = static_cast<size_t>(blockIdx.x) * 256 + threadIdx.x; i < n_ones;
             i += static_cast<size_t>(gridDim.x) * 256)
            ones[i] = 1.f;
}

__global__ void cast_bf16_kernel(const float* __restrict__ s, uint16_t* __restrict__ d, size_t n) {
    const size_t step = static_cast<size_t>(gridDim.x) * blockDim.x;
    for (size_t i = static_cast<size_t>(blockIdx.x) * blockDim.x + threadIdx.x; i < n; i += step) d[i] = f32_to_bf16(s[i]);
}

unsigned blocks_for(long n) {
    const long b = (n + 255) / 256;
    return static_cast<unsigned>(b < 1 ? 1 : b > 16384 ? 16384 : b);
}
bool al16(const void* p) { return reinterpret_cast<uintptr_t>(p) % 16 == 0; }
int lanes_per_row(int D) { return D == 64 ? 8 : D == 128 ? 16 : D == 256 ? 32 : 0; }

template <typename T>
hipError_t norm_t(const T* q, const T* k, T* qn, T* kn, float* ones, size_t n_ones, long rows, int D, hipStream_t st) {
    const int lpr = al16(q) && al16(k) && al16(qn) && al16(kn) ? lanes_per_row(D) : 0;
    const dim3 grid(blocks_for(lpr ? 2 * rows * lpr : 2 * rows * 64)), blk(256);
    if (lpr == 8) hipLaunchKernelGGL((norm_rows_kernel<T, 8>), grid, blk, 0, st, q, k, qn, kn, ones, n_ones, rows);
    else if (lpr == 16) hipLaunchKernelGGL((norm_rows_kernel<T, 16>), grid, blk, 0, st, q, k, qn, kn, ones, n_ones, rows);
    else if (lpr == 32) hipLaunchKernelGGL((norm_rows_kernel<T, 32>), grid, blk, 0, st, q, k, qn, kn, ones, n_ones, rows);
    else hipLaunchKernelGGL((norm_rows_any_kernel<T, false>), grid, blk, 0, st, q, k, nullptr, nullptr, qn, kn, ones, n_ones, rows, D);
    return hipGetLastError();
}
template <typename T>
hipError_t norm_bwd_t(const T* q, const T* k, const float* gqn, const float* gkn, T* gq, T* gk, long rows, int D,
                      hipStream_t st) {
    const int lpr = al16(q) && al16(k) && al16(gqn) && al16(gkn) && al16(gq) && al16(gk) ? lanes_per_row(D) : 0;
    const dim3 grid(blocks_for(lpr ? 2 * rows * lpr : 2 * rows * 64)), blk(256);
    if (lpr == 8) hipLaunchKernelGGL((norm_rows_bwd_kernel<T, 8>), grid, blk, 0, st, q, k, gqn, gkn, gq, gk, rows);
    else if (lpr == 16) hipLaunchKernelGGL((norm_rows_bwd_kernel<T, 16>), grid, blk, 0, st, q, k, gqn, gkn, gq, gk, rows);
    else if (lpr == 32) hipLaunchKernelGGL((norm_rows_bwd_kernel<T, 32>), grid, blk, 0, st, q, k, gqn, gkn, gq, gk, rows);
    else hipLaunchKernelGGL((norm_rows_any_kernel<T, true>), grid, blk, 0, st, q, k, gqn, gkn, gq, gk, nullptr, 0, rows, D);
    return hipGetLastError();
}

}  // namespace

hipError_t launch_norm_rows(const void* q, const void* k, void* qn, void* kn, float* ones, size_t n_ones, long rows,
                            int D, bool bf16, hipStream_t st) {
    if (rows <= 0) return hipSuccess;
    return bf16 ? norm_t(static_cast<const uint16_t*>(q), static_cast<const uint16_t*>(k), static_cast<uint16_t*>(qn),
                         static_cast<uint16_t*>(kn), ones, n_ones, rows, D, st)
                : norm_t(static_cast<const float*>(q), static_cast<const float*>(k), static_cast<float*>(qn),
                         static_cast<float*>(kn), ones, n_ones, rows, D, st);
}
hipError_t launch_norm_rows_bwd(const void* q, const void* k, const float* gqn, const float* gkn, void* gq, void* gk,
                                long rows, int D, bool bf16, hipStream_t st) {
    if (rows <= 0) return hipSuccess;
    return bf16 ? norm_bwd_t(static_cast<const uint16_t*>(q), static_cast<const uint16_t*>(k), gqn, gkn,
                             static_cast<uint16_t*>(gq), static_cast<uint16_t*>(gk), rows, D, st)
                : norm_bwd_t(static_cast<const float*>(q), static_cast<const float*>(k), gqn, gkn,
                             static_cast<float*>(gq), static_cast<float*>(gk), rows, D, st);
}
hipError_t launch_cast_bf16(const float* src, uint16_t* dst, size_t n, hipStream_t st) {
    if (n == 0) return hipSuccess;
    hipLaunchKernelGGL(cast_bf16_kernel, dim3(blocks_for(static_cast<long>(n))), dim3(256), 0, st, src, dst, n);
    return hipGetLastError();
}

}  // namespace pm
