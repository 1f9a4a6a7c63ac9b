// pm_f32mfma.h — fp32 MFMA (v_mfma_f32_16x16x4f32) building blocks shared by the fp32
// chunked forward and backward: the product wrappers and the swizzled LDS tile of 16
// fp32 token rows.  Internal to the translation unit that includes it (after
// pm_cdna4.h).
//
// Layout (lane l = 16 g + r): A operand A[r][g], B operand B[g][r], accumulator register
// v = D[4 g + v][r].  The accumulator registers of a 16x16 matrix M therefore serve as
//   * the B operand of a product contracting over M's rows (step v takes row 4 g + v), and
//   * the A operand of a product with M^T on the left, contracting over the same index,
// and a product contracting over M's columns needs the registers of M^T instead.
#pragma once

#include <atomic>
#include <type_traits>

namespace pm {
namespace {

constexpr int kC16 = 16;  // tokens per chunk

constexpr f32x4_t kZero4 = {0.f, 0.f, 0.f, 0.f};
__device__ __forceinline__ f32x4_t ld4(const unsigned char* p) { return *reinterpret_cast<const f32x4_t*>(p); }
__device__ __forceinline__ void st4(unsigned char* p, f32x4_t x) { *reinterpret_cast<f32x4_t*>(p) = x; }
__device__ __forceinline__ void fence() { __builtin_amdgcn_sched_barrier(0); }

// The dynamic-LDS limit is a per-device function attribute, set once per device for each
// kernel (KERN: one static flag array per kernel, not per signature).
template <auto KERN>
hipError_t set_lds(int bytes) {
    int dev = 0;
    hipError_t e = hipGetDevice(&dev);
    if (e != hipSuccess) return e;
    static std::atomic<bool> done[64] = {};
    if (dev >= 0 && dev < 64 && done[dev].load(std::memory_order_relaxed)) return hipSuccess;
    e = hipFuncSetAttribute(reinterpret_cast<const void*>(KERN), hipFuncAttributeMaxDynamicSharedMemorySize, bytes);
    if (e == hipSuccess && dev >= 0 && dev < 64) done[dev].store(true, std::memory_order_relaxed);
    return e;
}

__device__ __forceinline__ f32x4_t mfma4(float a, float b, f32x4_t c) {
    return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0);
}
// Left * Right over a 16-token contraction, given the accumulators of Left^T and Right
// (plus c), in two accumulators.
__device__ __forceinline__ f32x4_t mm16(f32x4_t lt, f32x4_t r, f32x4_t c = kZero4) {
    f32x4_t a0 = mfma4(lt[0], r[0], c), a1 = mfma4(lt[1], r[1], kZero4);
    a0 = mfma4(lt[2], r[2], a0);
    a1 = mfma4(lt[3], r[3], a1);
    return a0 + a1;
}

// Entry (i, j) of a 16x16 matrix is strictly lower and the highest bit in which i and j differ
// is HB: the lower left block of a 2h x 2h diagonal block, h = 2^HB.
template <int HB>
__device__ __forceinline__ bool in_level(int i, int j) {
    return ((i ^ j) >> HB) == 1 && i > j;
}
// T = (I - N)^-1 of a strictly lower N and T^T, from the accumulators of N and N^T: T starts as
// the inverse of I - N's diagonal 2x2 blocks, and T + T N_h T, N_h the lower left blocks at h,
// is that of its 2h x 2h blocks.  Only true inverses of blocks are multiplied: where the keys of
// a chunk are alike T's entries stay of the size of N's, while the powers of N, of which (I + N)
// (I + N^2)(I + N^4)(I + N^8) is made in as many products, grow as binomials (3,432 at N = -1)
// and cancel (O of a gated rule with keys of mutual cosine 0.9 was 2e-5 off at beta 1 and 8e-3
// at 1.95, now 3e-7 and 9e-7).  TOO false: T^T alone.
template <bool TOO>
__device__ __forceinline__ void inv_lower16(f32x4_t N, f32x4_t Nt, int r, int g, f32x4_t& T, f32x4_t& Tt) {
#pragma unroll
    for (int v = 0; v < 4; ++v) {
        const int i = 4 * g + v;
        const float eye = i == r ? 1.f : 0.f;
        T[v] = in_level<0>(i, r) ? N[v] : eye;
        Tt[v] = in_level<0>(r, i) ? Nt[v] : eye;
    }
    auto level = [&](auto HB, auto BOTH) __attribute__((always_inline)) {
        f32x4_t nt;  // N_h^T
#pragma unroll
        for (int v = 0; v < 4; ++v) nt[v] = in_level<decltype(HB)::value>(r, 4 * g + v) ? Nt[v] : 0.f;
        const f32x4_t y = mm16(nt, T);  // N_h T
        const f32x4_t t = Tt;
        Tt = mm16(y, t, t);  // (N_h T)^T T^T + T^T
        if constexpr (decltype(BOTH)::value) T = mm16(t, y, T);
    };
    using B = std::true_type;
    level(std::integral_constant<int, 1>{}, B{});
    level(std::integral_constant<int, 2>{}, B{});
    level(std::integral_constant<int, 3>{}, std::integral_constant<bool, TOO>{});
}

// LDS tile of 16 fp32 token rows of D values: the 16-byte chunk p of row t is stored at
// chunk t * (D / 4) + (p ^ t).  With it the float4 operand reads (lane (g, r): row r,
// chunk 4 m + g) and the column reads of K^T (lane (g, r): row 4 g + v, element 16 m + r)
// fall in distinct banks across each quarter wave.
template <int D>
__device__ __forceinline__ int f32_chunk(int t, int p) {
    return t * (D / 4) + (p ^ t);
}

// Lane (g, r)'s operand reads of a swizzled tile of 16 fp32 rows (f32_chunk): row(b, i) =
// X[r][16 i + 4 g ..] and col(b, e, i) = X[4 g + e][16 i + r].  The swizzle splits into a
// part that depends on i mod 4 and a constant one: (4 i + x) ^ (4 y + z) = 4 (i ^ y) + (x ^ z)
// for x, z < 4, and y < 4 leaves i's upper bit alone, so 13 registers address every read.
template <int D>
struct TileIdx {
    int rb, rx[4], cb[4], cx[4];  // byte offsets
    __device__ __forceinline__ TileIdx(int r, int g) {
        rb = 16 * (r * (D / 4) + (g ^ (r & 3)));
#pragma unroll
        for (int k = 0; k < 4; ++k) {
            rx[k] = 64 * (k ^ (r >> 2));
            cb[k] = 16 * ((4 * g + k) * (D / 4) + ((r >> 2) ^ k)) + 4 * (r & 3);
            cx[k] = 64 * (k ^ g);
        }
    }
    __device__ __forceinline__ f32x4_t row(const unsigned char* b, int i) const {
        return *reinterpret_cast<const f32x4_t*>(b + rb + rx[i & 3] + 256 * (i >> 2));
    }
    __device__ __forceinline__ float col(const unsigned char* b, int e, int i) const {
        return *reinterpret_cast<const float*>(b + cb[e] + cx[i & 3] + 256 * (i >> 2));
    }
    // Tiles i = hh + 2 j of a wave that holds every other one (TileIdx(r, g, hh)): the same, over j
    int hx[2], hc[2];
    __device__ __forceinline__ TileIdx(int r, int g, int hh) : TileIdx(r, g) {
        hx[0] = hh ? rx[1] : rx[0], hx[1] = hh ? rx[3] : rx[2];
        hc[0] = hh ? cx[1] : cx[0], hc[1] = hh ? cx[3] : cx[2];
    }
    __device__ __forceinline__ f32x4_t row2(const unsigned char* b, int j) const {
        return *reinterpret_cast<const f32x4_t*>(b + rb + hx[j & 1] + 256 * (j >> 1));
    }
    __device__ __forceinline__ float col2(const unsigned char* b, int e, int j) const {
        return *reinterpret_cast<const float*>(b + cb[e] + hc[j & 1] + 256 * (j >> 1));
    }
    // row and col for an i known only at run time
    __device__ __forceinline__ f32x4_t roww(const unsigned char* b, int i, int r) const {
        return *reinterpret_cast<const f32x4_t*>(b + rb + 64 * (i ^ (r >> 2)));
    }
    __device__ __forceinline__ float colw(const unsigned char* b, int e, int i, int g) const {
        return *reinterpret_cast<const float*>(b + cb[e] + 64 * (i ^ g));
    }
};

}  // namespace
}  // namespace pm
