// decay_chunked_f32.hip — K10: the rules with a decay (a log-gate per token and head, or
// one per key channel) in chunked form on fp32 MFMA (v_mfma_f32_16x16x4f32), D in {64, 128},
// fixed-length batches: the reverse mode for fp32 or bf16 q/k/v, the forward for fp32.  Every product is fp32 x fp32
// with fp32 accumulation, as in the per-token kernels (delta_bwd.hip).
//
// Per token, alpha_t = exp(g_t) (a d_k-vector; constant over d_k for the per-head gate):
//   P_t = Diag(alpha_t) S_{t-1},  u_t = v_t - P_t^T k_t,  S_t = P_t + beta_t k_t u_t^T,
//   o_t = q_t S_t.
// Per chunk of C = 16 tokens with start state S, F_t = prod_{j <= t} alpha_j and
// E_s = prod_{j > s} alpha_j inside the chunk, gC = F_{C-1}, and
// D_ts = prod_{s < j <= t} alpha_j (all per channel):
//   K^ = K F,  Q^ = Q F,  K- = K E,
//   A'_ts = sum_d k_t k_s D_ts (s < t),  P_ts = sum_d q_t k_s D_ts (s <= t),
//   T = (I + diag(beta) A')^-1,  T'' = -T diag(beta),  X = K^ S - V,  U = T'' X,
//   S' = Diag(gC) S + K-^T U,  O = Q^ S + P U.
// Reverse, given G = dL/dS' and dO (dP = lower_incl(dO U^T), dA = -strict_lower(W U^T)):
//   W  = T^T (K- G + P^T dO),  dV = diag(beta) W
//   dS = Diag(gC) G + Q^^T dO - K^^T diag(beta) W
//   dQ_t = F_t (dO S^T)_t + sum_s dP_ts k_s D_ts
//   dK_t = -beta_t F_t (W S^T)_t + E_t (U G^T)_t + sum_{s<t} beta_t dA_ts k_s D_ts
//          + sum_{r>t} beta_r dA_rt k_r D_rt + sum_{r>=t} dP_rt q_r D_rt
//   dbeta_t = W_t . V_t - K^_t . (W S^T)_t + sum_s dA_ts A'_ts
//   dg_j = sum_{t>=j} (Q^ dO S^T - K^ beta W S^T)_t + sum_{s<j} (K- U G^T)_s
//          + gC <S, G>_rows + sum_{t>=j, s<j} x_ts,
// x_ts the pair term dP_ts q_t k_s D_ts + beta_t dA_ts k_t k_s D_ts.  Every term of dg_j holds
// alpha_j: none is a difference of larger ones, which a strong decay would leave without a digit
// (as <S', G'> less the chunk's own terms, gC <S, G> was 4e-5 of dg off at g = -8 throughout
// and noise at -20; now 1e-7 to 3e-7 at every strength).
//
// Decays without exponents of differences.  D_ts is never formed as exp(G_t - G_s) (whose
// difference of prefix sums loses what a strong decay elsewhere in the chunk adds to both)
// nor as a quotient.  The strictly lower pairs (t, s) split over four levels h = 1, 2, 4, 8
// by the highest bit in which t and s differ: at level h, t lies in the upper and s in the
// lower half of one aligned block of 2h tokens, and
//   D_ts = F^h_t E^h_s,
// F^h the inclusive prefix product of alpha inside the aligned block of h tokens and E^h
// the exclusive suffix product.  Both are products of at most 8 alphas, at most 1 for
// g <= 0 and exact to rounding for any g, and each level is one masked matrix product:
// A' = sum_h mask_h((K F^h) (K E^h)^T).  The last level's F and E are the chunk's own.
//
// Launches:
//   K10p (prep, one wave per (b, h, chunk)): K^, K-, Q^, T'', T, P, A', gC, beta.
//   K10s (one workgroup per (b, h, 16 or 32 columns of d_v)): the state recurrence
//     forwards (U per token, S at every span start) beside the G recurrence backwards (W
//     and dV per token, G at every span end, dS0).
//   K10c (one workgroup of D/16 waves per (b, h, span of 2 to 8 chunks)): the span forwards from
//     its start state (dQ, dbeta, dK and dg but for what depends on G), then backwards from
//     its end gradient (the rest).  S cannot be walked back as the ungated backward does
//     (that divides by gC), hence the two walks; <S, G> needs S at every chunk's start again, which
//     the way forwards keeps (the last one in registers, the middle one in LDS, the others in the
//     workspace: 64 KiB a chunk at D = 128, 4% of the training pass).

// Why chunks: the per-token kernels walk T tokens in sequence at about 500 (forward) and
// 1,270 cycles (reverse) a token, bound by VALU issue; here a chunk of 16 tokens takes about
// 2,800 to 4,100 cycles of the one sequential launch, and the rest is parallel over chunks.
// Measured (backward alone), B4 T4096 H16 D128, bf16 q/k/v, per-head gate: 6.0 -> 1.53 ms (K10p
// 122, K10s 515, K10c 870 us); B2, per-channel gate: 5.9 -> 0.93 ms (97, 344, 480); B3 T1000 H6
// D64 fp32: 1.11 -> 0.11 ms (11, 57, 39).  Against 64 bits the gradients of training inputs are at
// 1.6e-7 to 2.5e-7 (the per-token kernels: 1.3e-7 to 1.9e-7).  What bounds it, by counters: K10s
// the products of its recurrence waves (MFMA pipes busy 59% of the time at 64 pairs and 47% at 32,
// where each chain wave has a SIMD to itself; the rest is the two exchanges and barriers of a
// chunk), K10c the two together of the fp32 MFMA pipe (busy 46%, 41% per channel; its two waves
// per SIMD wait to issue half of their time and at barriers a quarter) and of its workspace (3.2
// GB in 870 us, 3.7 TB/s, where a copy reaches 4.7; 1.3 GB of it the states of the chunks).

#include <type_traits>

#include "pm_cdna4.h"
#include "pm_f32mfma.h"
#include "pm_internal.h"

namespace pm {
namespace {

constexpr int kSpan = 8;  // chunks per span (128 tokens) at most
// Chunks of a span whose start states K10c leaves in the workspace: not the first, the middle
// and the last one's
__host__ __device__ constexpr int kept_starts(int span_len) { return span_len > 2 ? span_len - 3 : 0; }

__device__ __forceinline__ f32x4_t fma4(f32x4_t a, f32x4_t b, f32x4_t c) {
    const f32x4_t r = {fmaf(a[0], b[0], c[0]), fmaf(a[1], b[1], c[1]), fmaf(a[2], b[2], c[2]), fmaf(a[3], b[3], c[3])};
    return r;
}

// Infinities and NaN keep to the tokens that they reach in the recurrence.  A product over the
// chunk's tokens would carry one to all of them, through the exact zeros of T'', T^T and P: where
// an operand of such a product holds one (looked for once a chunk, behind the product) the rows
// that it does not reach are formed again without it.
__device__ __forceinline__ bool any_bad(f32x4_t x) {
    const float z = fmaf(x[0], 0.f, fmaf(x[1], 0.f, fmaf(x[2], 0.f, x[3] * 0.f)));  // 0, or NaN
    return __any(z != 0.f);
}
__device__ __forceinline__ bool bad(float x) { return !__builtin_isfinite(x); }
// First (16: none) and last (-1: none) row of this lane's column that holds one
__device__ __forceinline__ int first_bad(f32x4_t x, int g) {
    int b = 16;
#pragma unroll
    for (int e = 3; e >= 0; --e) b = bad(x[e]) ? 4 * g + e : b;
    b = min(b, __shfl_xor(b, 16));
    return min(b, __shfl_xor(b, 32));
}
__device__ __forceinline__ int last_bad(f32x4_t x, int g) {
    int b = -1;
#pragma unroll
    for (int e = 0; e < 4; ++e) b = bad(x[e]) ? 4 * g + e : b;
    b = max(b, __shfl_xor(b, 16));
    return max(b, __shfl_xor(b, 32));
}
// x where this lane's rows 4 g + e are before row b, else y
__device__ __forceinline__ f32x4_t before(int b, int g, f32x4_t x, f32x4_t y) {
    f32x4_t z;
#pragma unroll
    for (int e = 0; e < 4; ++e) z[e] = 4 * g + e < b ? x[e] : y[e];
    return z;
}

// One chunk's record (floats): T''^T, T, P, A'^T as accumulator registers, then gC (D) and
// beta (16), padded to a multiple of 64 (copied 256 bytes an instruction).
template <int D>
struct DecRec {
    static constexpr int T2 = 0, TA = 256, PA = 512, AT = 768, GB = 1024, GBN = D + 64;
    static constexpr int FLOATS = GB + GBN;
    // the forward's: T''^T, P^T, gC
    static constexpr int FPT = 256, FGB = 512, FFLOATS = FGB + D;
};

// One element, and four consecutive ones, of a row through a range-checked buffer (byte
// offsets off; zeros past the range)
template <typename InT>
__device__ __forceinline__ float buf_el(__amdgpu_buffer_rsrc_t rs, unsigned elem) {
    if constexpr (sizeof(InT) == 2)
        return __uint_as_float(static_cast<unsigned>(__builtin_amdgcn_raw_buffer_load_b16(rs, elem * 2, 0, 0)) << 16);
    else
        return __uint_as_float(__builtin_amdgcn_raw_buffer_load_b32(rs, elem * 4, 0, 0));
}
template <typename InT>
__device__ __forceinline__ f32x4_t buf_el4(__amdgpu_buffer_rsrc_t rs, unsigned elem) {
    if constexpr (sizeof(InT) == 2)
        return widen4(__builtin_bit_cast(u32x2_t, __builtin_amdgcn_raw_buffer_load_b64(rs, elem * 2, 0, 0)));
    else
        return __builtin_bit_cast(f32x4_t, __builtin_amdgcn_raw_buffer_load_b128(rs, elem * 4, 0, 0));
}
// One gradient element of GE bytes (rows past the range dropped)
template <int GE>
__device__ __forceinline__ void put(float x, __amdgpu_buffer_rsrc_t rs, unsigned elem) {
    if constexpr (GE == 2)
        __builtin_amdgcn_raw_buffer_store_b16(f32_to_bf16(x), rs, elem * 2, 0, 0);
    else
        __builtin_amdgcn_raw_buffer_store_b32(__float_as_uint(x), rs, elem * 4, 0, 0);
}
template <int CTRL>
__device__ __forceinline__ float dpp_mov(float x) {
    return __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(x), CTRL, 0xF, 0xF, false));
}
// 4 bytes per lane buffer -> LDS (lane L's at lds_dst + 4 L), as dma16_asm
__device__ __forceinline__ void dma4_asm(__amdgpu_buffer_rsrc_t rs, const void* lds_dst, unsigned voffset) {
    const unsigned m0 = uniform(lds_addr(lds_dst));
    __asm__ volatile("buffer_load_dword %0, %1, 0 offen lds" ::"v"(voffset), "s"(rs), "{m0}"(m0) : "memory");
}
// Ordering of this wave's own LDS accesses for the compiler (the hardware keeps a wave's
// LDS operations in order)
__device__ __forceinline__ void wave_lds_fence() { __asm__ volatile("" ::: "memory"); }

// ---------------------------------------------------------------- K10p
// Lane (r, g) = (lane & 15, lane >> 4) holds token r at d = 16 j + 4 g + v: the A and the B
// operand of products contracting over d.  MFMA-bound: 4 levels x 2 products of 16 x 16 x D
// (256 MFMAs at D = 128; a per-head gate needs the two Gram products only once, since its
// D_ts does not depend on d).
// FWD: what the forward needs alone: Q^ as rows, T''^T, P^T and gC.
template <int D, typename InT, bool CHAN, bool FWD>
__global__ __launch_bounds__(256) void dec_prep_kernel(
    const InT* __restrict__ q, const InT* __restrict__ k, const float* __restrict__ beta,
    const float* __restrict__ gate, int T, int H, int n_ch, long n_items, float* __restrict__ kh_ws,
    float* __restrict__ kb_ws, float* __restrict__ qh_ws, float* __restrict__ rec_ws) {
    // a per-channel gate takes 64 channels at a time (five values per channel and token live
    // in registers); a per-head one needs all of them before its levels
    constexpr int NH = CHAN ? D / 64 : 1, NJ = D / 16 / NH, NF = CHAN ? NJ : 1, NV = CHAN ? 4 : 1;
    using R = DecRec<D>;
    constexpr int TILE = kC16 * D * 4, TR = 16 * 17 * 4;
    __shared__ __attribute__((aligned(16))) unsigned char smem[4 * (TILE + TR)];
    const int lane = threadIdx.x & 63;
    const int w = static_cast<int>(uniform(threadIdx.x >> 6));
    const long item = static_cast<long>(blockIdx.x) * 4 + w;
    if (item >= n_items) return;  // (waves are independent: no barrier below)
    unsigned char* tile = smem + w * (TILE + TR);
    float* tr = reinterpret_cast<float*>(tile + TILE);
    const int pair = static_cast<int>(item / n_ch), c = static_cast<int>(item % n_ch);
    const int seq = pair / H, h = pair % H;
    const int base = c * kC16, clen = min(kC16, T - base);
    const size_t tok0 = static_cast<size_t>(seq) * T + base;
    const int r = lane & 15, g = lane >> 4;
    const size_t tstride = static_cast<size_t>(H) * D;
    const size_t row0 = tok0 * tstride + static_cast<size_t>(h) * D;
    const unsigned n_el = static_cast<unsigned>((clen - 1) * tstride + D), n_hd = static_cast<unsigned>((clen - 1) * H + 1);
    float* const kh = kh_ws + static_cast<size_t>(item) * kC16 * D;
    float* const kb = kb_ws + static_cast<size_t>(item) * kC16 * D;
    float* const qh = qh_ws + static_cast<size_t>(item) * kC16 * D;
    constexpr int kGB = FWD ? R::FGB : R::GB;
    float* const rec = rec_ws + static_cast<size_t>(item) * (FWD ? R::FFLOATS : R::FLOATS);

    const __amdgpu_buffer_rsrc_t rb = make_rsrc(beta + tok0 * H + h, n_hd * 4);
    const float bc = buf_el<float>(rb, static_cast<unsigned>(r * H));
    f32x4_t bt;
#pragma unroll
    for (int v = 0; v < 4; ++v) bt[v] = buf_el<float>(rb, static_cast<unsigned>((4 * g + v) * H));

    f32x4_t A = kZero4, P = kZero4;
    float qk = 0.f;  // q_r . k_r, P's diagonal
#pragma unroll
    for (int hf = 0; hf < NH; ++hf) {
        f32x4_t kf[NJ], qf[NJ];
        float al[NF][NV];  // alpha of token r (rows past the end read g = 0: alpha = 1)
        {
            const __amdgpu_buffer_rsrc_t rk = make_rsrc(k + row0, n_el * sizeof(InT));
            const __amdgpu_buffer_rsrc_t rq = make_rsrc(q + row0, n_el * sizeof(InT));
#pragma unroll
            for (int j = 0; j < NJ; ++j) {
                const unsigned el = static_cast<unsigned>(r * tstride + 16 * (hf * NJ + j) + 4 * g);
                kf[j] = buf_el4<InT>(rk, el);
                qf[j] = buf_el4<InT>(rq, el);
            }
            if constexpr (CHAN) {
                const __amdgpu_buffer_rsrc_t rg = make_rsrc(gate + row0, n_el * 4);
#pragma unroll
                for (int j = 0; j < NJ; ++j) {
                    const f32x4_t x = buf_el4<float>(rg, static_cast<unsigned>(r * tstride + 16 * (hf * NJ + j) + 4 * g));
#pragma unroll
                    for (int v = 0; v < 4; ++v) al[j][v] = expf(x[v]);
                }
            } else {
                al[0][0] = expf(buf_el<float>(make_rsrc(gate + tok0 * H + h, n_hd * 4), static_cast<unsigned>(r * H)));
            }
        }
        // the levels: F, E and the block's product tot, of aligned blocks of h = 1, 2, 4, 8 tokens
        float F[NF][NV], E[NF][NV], tot[NF][NV];
#pragma unroll
        for (int j = 0; j < NF; ++j)
#pragma unroll
            for (int v = 0; v < NV; ++v) F[j][v] = tot[j][v] = al[j][v], E[j][v] = 1.f;
        auto fac = [](const float (&x)[NF][NV], int j, int v) { return CHAN ? x[CHAN ? j : 0][CHAN ? v : 0] : x[0][0]; };
        f32x4_t gk = kZero4, gq = kZero4;  // per-head gate: K K^T and Q K^T
        if constexpr (!CHAN) {
            f32x4_t aa[4] = {kZero4, kZero4, kZero4, kZero4}, pa[4] = {kZero4, kZero4, kZero4, kZero4};
#pragma unroll
            for (int j = 0; j < NJ; ++j)
#pragma unroll
                for (int v = 0; v < 4; ++v) {
                    aa[v] = mfma4(kf[j][v], kf[j][v], aa[v]);
                    pa[v] = mfma4(qf[j][v], kf[j][v], pa[v]);
                }
            gk = (aa[0] + aa[1]) + (aa[2] + aa[3]);
            gq = (pa[0] + pa[1]) + (pa[2] + pa[3]);
        }
        auto level = [&](auto HB) __attribute__((always_inline)) {
            constexpr int hb = decltype(HB)::value, hh = 1 << hb;
            f32x4_t a4 = gk, p4 = gq;
            if constexpr (CHAN) {
                f32x4_t aa[4] = {kZero4, kZero4, kZero4, kZero4}, pa[4] = {kZero4, kZero4, kZero4, kZero4};
#pragma unroll
                for (int j = 0; j < NJ; ++j)
#pragma unroll
                    for (int v = 0; v < 4; ++v) {
                        const float rr = kf[j][v] * E[j][v];
                        aa[v] = mfma4(kf[j][v] * F[j][v], rr, aa[v]);
                        pa[v] = mfma4(qf[j][v] * F[j][v], rr, pa[v]);
                    }
                a4 = (aa[0] + aa[1]) + (aa[2] + aa[3]);
                p4 = (pa[0] + pa[1]) + (pa[2] + pa[3]);
            }
            // entry (t, s) = (4 g + v, r) belongs to this level: t > s, highest differing bit hb
#pragma unroll
            for (int v = 0; v < 4; ++v) {
                const int t = 4 * g + v;
                const bool in = in_level<hb>(t, r);
                float d = 1.f;
                if constexpr (!CHAN) d = __shfl(F[0][0], t) * E[0][0];
                A[v] += in ? d * a4[v] : 0.f;
                P[v] += in ? d * p4[v] : 0.f;
            }
            constexpr int CTRL = hb == 0 ? 0xB1 : hb == 1 ? 0x4E : hb == 2 ? 0x141 : 0x140;
            const bool up = (r & hh) != 0;
#pragma unroll
            for (int j = 0; j < NF; ++j)
#pragma unroll
                for (int v = 0; v < NV; ++v) {
                    const float sib = dpp_mov<CTRL>(tot[j][v]);  // the other half's product
                    F[j][v] *= up ? sib : 1.f;
                    E[j][v] *= up ? 1.f : sib;
                    tot[j][v] *= sib;
                }
        };
        level(std::integral_constant<int, 0>{});
        level(std::integral_constant<int, 1>{});
        level(std::integral_constant<int, 2>{});
        level(std::integral_constant<int, 3>{});
        // K^, K- as swizzled row tiles; Q^ in operand order (below); gC
#pragma unroll
        for (int j = 0; j < NJ; ++j) {
            f32x4_t x, y, z, gc;
#pragma unroll
            for (int v = 0; v < 4; ++v) {
                qk = fmaf(qf[j][v], kf[j][v], qk);
                x[v] = kf[j][v] * fac(F, j, v);
                y[v] = kf[j][v] * fac(E, j, v);
                z[v] = qf[j][v] * fac(F, j, v);
                gc[v] = fac(tot, j, v);
            }
            const int o = 4 * f32_chunk<D>(r, 4 * (hf * NJ + j) + g);
            *reinterpret_cast<f32x4_t*>(kh + o) = x;
            *reinterpret_cast<f32x4_t*>(kb + o) = y;
            if constexpr (FWD) *reinterpret_cast<f32x4_t*>(qh + o) = z;
            else st4(tile + 4 * o, z);
            if (r == 0) *reinterpret_cast<f32x4_t*>(rec + kGB + 16 * (hf * NJ + j) + 4 * g) = gc;
        }
    }
    qk += __shfl_xor(qk, 16);
    qk += __shfl_xor(qk, 32);
#pragma unroll
    for (int v = 0; v < 4; ++v) P[v] = (4 * g + v == r) ? qk : P[v];
    if (!FWD && g == 0) rec[R::GB + D + r] = bc;
    // A'^T (FWD: and P^T) through LDS
#pragma unroll
    for (int v = 0; v < 4; ++v) tr[(4 * g + v) * 17 + r] = A[v];
    wave_lds_fence();
    f32x4_t At;  // A'[r][4 g + v]
#pragma unroll
    for (int v = 0; v < 4; ++v) At[v] = tr[r * 17 + 4 * g + v];
    f32x4_t Pt = kZero4;  // P[r][4 g + v]
    if constexpr (FWD) {
        wave_lds_fence();
#pragma unroll
        for (int v = 0; v < 4; ++v) tr[(4 * g + v) * 17 + r] = P[v];
        wave_lds_fence();
#pragma unroll
        for (int v = 0; v < 4; ++v) Pt[v] = tr[r * 17 + 4 * g + v];
    } else {
    // Q^ as the A operand of Q^^T dO: [m][lane][e] = Q^[4 g + e][16 m + r]
    const TileIdx<D> ix(r, g);
#pragma unroll
    for (int m = 0; m < D / 16; ++m) {
        f32x4_t x;
#pragma unroll
        for (int e = 0; e < 4; ++e) x[e] = ix.col(tile, e, m);
        *reinterpret_cast<f32x4_t*>(qh + 4 * (64 * m + lane)) = x;
    }
    }

    // T = (I + diag(beta) A')^-1 = (I - N)^-1, N = -diag(beta) A'
    f32x4_t N, Nt, Ta, Tt;
#pragma unroll
    for (int v = 0; v < 4; ++v) {
        N[v] = 4 * g + v > r ? -bt[v] * A[v] : 0.f;
        Nt[v] = r > 4 * g + v ? -bc * At[v] : 0.f;
    }
    // (an infinity or NaN counts where it stands: its row of U and the columns of W before it)
    f32x4_t Nf, Ntf;
#pragma unroll
    for (int v = 0; v < 4; ++v) {
        Nf[v] = bad(N[v]) ? 0.f : N[v];
        Ntf[v] = bad(Nt[v]) ? 0.f : Nt[v];
    }
    inv_lower16<!FWD>(Nf, Ntf, r, g, Ta, Tt);
#pragma unroll
    for (int v = 0; v < 4; ++v) {
        Ta[v] = bad(N[v]) ? N[v] : Ta[v];
        Tt[v] = bad(Nt[v]) ? Nt[v] : Tt[v];
    }
    f32x4_t tw;
#pragma unroll
    for (int v = 0; v < 4; ++v) tw[v] = 4 * g + v <= r ? -bt[v] * Tt[v] : 0.f;
    *reinterpret_cast<f32x4_t*>(rec + R::T2 + 4 * lane) = tw;
    if constexpr (FWD) {
        *reinterpret_cast<f32x4_t*>(rec + R::FPT + 4 * lane) = Pt;
    } else {
        *reinterpret_cast<f32x4_t*>(rec + R::TA + 4 * lane) = Ta;
        *reinterpret_cast<f32x4_t*>(rec + R::PA + 4 * lane) = P;
        *reinterpret_cast<f32x4_t*>(rec + R::AT + 4 * lane) = At;
    }
}

// ---------------------------------------------------------------- K10f
// The forward (fp32 q/k/v): one workgroup per (b, h, DV columns of d_v).  Per 16 columns two
// chain waves as K10s's state chain and an output wave (Y = Q^ S one chunk behind, O = Y + P U
// two behind, stores), which the chains hand S and U through LDS.  The last wave copies every
// chunk two ahead through four buffers; one barrier per chunk, at which the halves of X are
// exchanged.
// The chain bounds it: one wave per 16 columns (68 products in sequence at D = 128) took 108 us
// at 32 pairs of T 1024, D = 128, per-head gate, and 63 at 2 pairs of D = 64; now 78 and 51.  At
// many pairs of D = 64 the shared pipes cost a little (128 pairs 104, now 108).
template <int D, int DV>
struct DfGeo {
    static constexpr int NCW = DV / 16, NT = D / 16, NI = kC16 * D * 4 / 1024, TILE = kC16 * D * 4, NB = 4;
    static constexpr int WAVES = 3 * NCW + 1;
    static constexpr int B_KH = 0, B_KB = TILE, B_QH = 2 * TILE, B_T = 3 * TILE, B_P = B_T + 1024, B_V = B_P + 1024;
    static constexpr int B_G = B_V + NCW * 1024, BUF = B_G + D * 4;
    static constexpr int OFF_S = NB * BUF;                    // 2 slots x NCW: S of a chunk's start
    static constexpr int OFF_U = OFF_S + 2 * NCW * NT * 1024; // 2 slots x NCW: U
    static constexpr int OFF_X = OFF_U + 2 * NCW * 1024;      // 2 slots x NCW x 2 halves of X
    static constexpr int BYTES = OFF_X + 4096 * NCW;
    static constexpr int NCP = 3 * NI + 2 + NCW + D / 64;     // copies per chunk
    static_assert(BYTES <= 160 * 1024 && NCP <= 63, "LDS / vmcnt");
};

template <int D, int DV, bool OUT_BF16>
__global__ __launch_bounds__((DfGeo<D, DV>::WAVES * 64)) void dec_fwd_kernel(
    const float* __restrict__ v, const float* __restrict__ s0, void* __restrict__ o_out, float* __restrict__ s_out,
    const float* __restrict__ kh, const float* __restrict__ kb, const float* __restrict__ qh,
    const float* __restrict__ rec, int n_pairs, int T, int H, int n_ch) {
    using G = DfGeo<D, DV>;
    using R = DecRec<D>;
    constexpr int NCW = G::NCW, NT = G::NT, n_tiles = D / DV;
    extern __shared__ __attribute__((aligned(16))) unsigned char smem[];
    // XCD-aware placement: the n_tiles workgroups of a pair share bid % 8
    const int bid = blockIdx.x, xcd = bid & 7, bslot = bid >> 3;
    const int tile = bslot % n_tiles, pair = (bslot / n_tiles) * 8 + xcd;
    if (pair >= n_pairs || n_ch <= 0) return;
    const int seq = pair / H, h = pair % H;
    const size_t tok0 = static_cast<size_t>(seq) * T;
    const int col0 = tile * DV;
    const int w = static_cast<int>(uniform(threadIdx.x >> 6)), lane = threadIdx.x & 63;
    const int r = lane & 15, g = lane >> 4;
    const size_t tstride = static_cast<size_t>(H) * D;
    const size_t sbase = static_cast<size_t>(pair) * D * D;
    const size_t item0 = static_cast<size_t>(pair) * n_ch;
    auto buf = [=](int c) { return smem + (c % G::NB) * G::BUF; };
    auto sslot = [=](int c, int which) { return smem + G::OFF_S + ((c & 1) * NCW + which) * NT * 1024; };
    auto uslot = [=](int c, int which) { return smem + G::OFF_U + ((c & 1) * NCW + which) * 1024; };
    auto row0_of = [=](int c, int col) { return (tok0 + c * kC16) * tstride + static_cast<size_t>(h) * D + col; };
    auto els_of = [=](int c, int cols) {
        return static_cast<unsigned>((min(kC16, T - c * kC16) - 1) * tstride + cols);
    };

    if (w < 2 * NCW) {
        // ============ chain wave hh of two: S columns col0 + 16 cw + [0, 16), tiles m = hh + 2 j ============
        // Phase p (up to barrier M_p) finishes chunk p - 1 (the other wave's half of X, U, S's own
        // rows) and forms this wave's half of X of chunk p.
        constexpr int NH = NT / 2;
        const int cw = w >> 1, hh = w & 1, ecol = col0 + 16 * cw + r;
        const TileIdx<D> ix(r, g, hh);
        f32x4_t S[NH];
#pragma unroll
        for (int j = 0; j < NH; ++j)
#pragma unroll
            for (int e = 0; e < 4; ++e)
                S[j][e] = s0 ? s0[sbase + static_cast<size_t>(16 * (hh + 2 * j) + 4 * g + e) * D + ecol] : 0.f;
        __builtin_amdgcn_s_waitcnt(0x0F70);  // vmcnt(0), seen by the compiler: no wait for these in the loop
        __builtin_amdgcn_s_setprio(3);
        lds_barrier();  // B0
        unsigned char* const xs = smem + G::OFF_X + 2048 * cw + 16 * lane;
        float kt[4][NH] = {};  // K-^T operand of the last chunk
        f32x4_t kf[NH], gc[NH] = {}, half = kZero4, tt = kZero4;
        for (int p = 0; p <= n_ch; ++p) {
            const bool run = p < n_ch;
            const unsigned char* b = buf(run ? p : n_ch - 1);  // (past the end: read, unused)
            const f32x4_t other = ld4(xs + ((p & 1) ^ 1) * 2048 * NCW + (hh ^ 1) * 1024);
            f32x4_t tn, vr;
#pragma unroll
            for (int j = 0; j < NH; ++j) kf[j] = ix.row2(b + G::B_KH, j);
#pragma unroll
            for (int e = 0; e < 4; ++e)
                vr[e] = reinterpret_cast<const float*>(b + G::B_V + 1024 * cw)[(4 * g + e) * 16 + r];
            tn = ld4(b + G::B_T + 16 * lane);
            fence();
            if (p > 0) {
                const f32x4_t X = half + other;
                f32x4_t u0 = mfma4(tt[0], X[0], kZero4), u1 = mfma4(tt[1], X[1], kZero4);
                __asm__ volatile("" : "+v"(u0), "+v"(u1));  // (issued here, with what follows in their shadow)
#pragma unroll
                for (int j = 0; j < NH; ++j) {
                    S[j] = gc[j] * S[j];
                    __asm__ volatile("" : "+v"(S[j]));
                }
                const bool xbad = any_bad(X);
                u0 = mfma4(tt[2], X[2], u0), u1 = mfma4(tt[3], X[3], u1);
                f32x4_t U = u0 + u1;
                if (__builtin_expect(xbad, 0)) {
                    const int b = first_bad(X, g);
                    U = before(b, g, mm16(tt, before(b, g, X, kZero4)), U);
                }
                if (hh == 0) st4(uslot(p - 1, cw) + 16 * lane, U);
#pragma unroll
                for (int e = 0; e < 4; ++e)
#pragma unroll
                    for (int j = 0; j < NH; ++j) S[j] = mfma4(kt[e][j], U[e], S[j]);
            }
            fence();
            if (run) {
                tt = tn;
                f32x4_t xa[4] = {kZero4, kZero4, kZero4, kZero4};
                if (hh == 0) xa[0] = -vr;
                unsigned char* ss = sslot(p, cw) + 16 * lane;
#pragma unroll
                for (int j = 0; j < NH; ++j)
#pragma unroll
                    for (int e = 0; e < 4; ++e) {
                        xa[e] = mfma4(kf[j][e], S[j][e], xa[e]);
                        kt[e][j] = ix.col2(b + G::B_KB, e, j);
                        if (e == 1) gc[j] = ld4(b + G::B_G + 4 * (16 * (hh + 2 * j) + 4 * g));
                        if (e == 3) st4(ss + 1024 * (hh + 2 * j), S[j]);
                        fence();
                    }
                half = (xa[0] + xa[1]) + (xa[2] + xa[3]);
                st4(xs + (p & 1) * 2048 * NCW + hh * 1024, half);
            }
            __builtin_amdgcn_s_waitcnt(0xC07F);  // lgkmcnt(0), seen by the compiler
            lds_barrier();                       // M_p
        }
#pragma unroll
        for (int j = 0; j < NH; ++j)
#pragma unroll
            for (int e = 0; e < 4; ++e)
                s_out[sbase + static_cast<size_t>(16 * (hh + 2 * j) + 4 * g + e) * D + ecol] = S[j][e];
    } else if (w < 3 * NCW) {
        // ============ output wave: phase p finishes O of chunk p - 2 and forms Y of chunk p - 1 ============
        const int cw = w - 2 * NCW;
        constexpr int ES = OUT_BF16 ? 2 : 4;
        const TileIdx<D> ix(r, g);
        f32x4_t y = kZero4, pt = kZero4;
        lds_barrier();  // B0
        for (int p = 0; p <= n_ch + 1; ++p) {
            if (p >= 2) {
                const int c = p - 2;
                const f32x4_t U = ld4(uslot(c, cw) + 16 * lane);
                f32x4_t O = mm16(pt, U, y);
                if (__builtin_expect(any_bad(U), 0)) {
                    const int b = first_bad(U, g);
                    O = before(b, g, mm16(pt, before(b, g, U, kZero4), y), O);
                }
                // lane (g, r) holds O[4 g + e][16 cw + r]; rows past the end are dropped
                const __amdgpu_buffer_rsrc_t ro = make_rsrc(
                    static_cast<unsigned char*>(o_out) + row0_of(c, col0 + 16 * cw) * ES, els_of(c, 16) * ES);
#pragma unroll
                for (int e = 0; e < 4; ++e) put<ES>(O[e], ro, static_cast<unsigned>((4 * g + e) * tstride + r));
            }
            if (p > n_ch) break;
            if (p >= 1) {
                const unsigned char* b = buf(p - 1);
                const unsigned char* ss = sslot(p - 1, cw) + 16 * lane;
                f32x4_t ya[4] = {kZero4, kZero4, kZero4, kZero4}, qy[NT], sc[NT];
                auto rd = [&](int m) __attribute__((always_inline)) {
                    qy[m] = ix.row(b + G::B_QH, m);
                    sc[m] = ld4(ss + 1024 * m);
                };
                rd(0);
                rd(1);
                pt = ld4(b + G::B_P + 16 * lane);
                fence();
#pragma unroll
                for (int m = 0; m < NT; ++m) {
                    if (m + 2 < NT) rd(m + 2);
#pragma unroll
                    for (int e = 0; e < 4; ++e) ya[e] = mfma4(qy[m][e], sc[m][e], ya[e]);
                    fence();
                }
                y = (ya[0] + ya[1]) + (ya[2] + ya[3]);
            }
            lds_barrier();
        }
    } else {
        // ============ copy wave: phase p issues chunk p + 2's copies ============
        auto copies = [=](int c) __attribute__((always_inline)) {
            unsigned char* b = buf(c);
            const float* rc = rec + (item0 + c) * R::FFLOATS;
            const float* src[3] = {kh, kb, qh};
#pragma unroll
            for (int x = 0; x < 3; ++x) {
                const __amdgpu_buffer_rsrc_t rs = make_rsrc(src[x] + (item0 + c) * kC16 * D, G::TILE);
                unsigned char* d0 = uniform_ptr(b + x * G::TILE);
#pragma unroll
                for (int i = 0; i < G::NI; ++i) dma16_asm(rs, d0 + 1024 * i, static_cast<unsigned>(1024 * i + 16 * lane));
            }
            dma16_asm(make_rsrc(rc + R::T2, 1024), uniform_ptr(b + G::B_T), static_cast<unsigned>(16 * lane));
            dma16_asm(make_rsrc(rc + R::FPT, 1024), uniform_ptr(b + G::B_P), static_cast<unsigned>(16 * lane));
#pragma unroll
            for (int j = 0; j < NCW; ++j)
                dma16_asm(make_rsrc(v + row0_of(c, col0 + 16 * j), els_of(c, 16) * 4), uniform_ptr(b + G::B_V + 1024 * j),
                          static_cast<unsigned>((lane >> 2) * tstride * 4 + 16 * (lane & 3)));
            const __amdgpu_buffer_rsrc_t rg = make_rsrc(rc + R::FGB, D * 4);
#pragma unroll
            for (int j = 0; j < D / 64; ++j)
                dma4_asm(rg, uniform_ptr(b + G::B_G + 256 * j), static_cast<unsigned>(256 * j + 4 * lane));
        };
        copies(0);
        if (n_ch > 1) {
            copies(1);
            wait_vm_n<G::NCP>();
        } else {
            wait_vm_n<0>();
        }
        lds_barrier();  // B0
        for (int p = 0; p <= n_ch; ++p) {
            // chunk p + 1 has landed; the copies of the one after may be in flight
            if (p + 2 < n_ch) {
                copies(p + 2);
                wait_vm_n<G::NCP>();
            } else {
                wait_vm_n<0>();
            }
            lds_barrier();
        }
    }
}

// ---------------------------------------------------------------- K10s
// The two recurrences, over S forwards and over G backwards, in one workgroup per (b, h, DV
// columns of d_v).  They bound the launch: their chunks run in sequence, and a chain of one
// wave per 16 columns needs 72 products of 32 cycles a chunk.  So two waves share 16 columns,
// each holding every other tile of 16 rows of d (and half of every product over or onto d):
// the products that contract over d (X = K^ S, Y = K- G) come in two halves, exchanged through
// LDS at a barrier in mid-chunk and added by both, and each wave updates its own rows.  Per
// chunk and wave 40 products (S) and 54 (G, its Q^^T dO among them) instead of 72 and 104;
// one wave per 16 columns, with Q^^T dO in helper waves, took 510 us at 32 pairs of T 4096
// (now 340) and 535 at 64 (now 505).
// Waves: 2 DV/16 for S, as many for G (a SIMD holds one of each at DV = 32, one of either at
// 16), one that copies for S (and Q^), one that copies for G and stores W and dV.  Each
// recurrence keeps three chunk buffers: a chain holds its chunk's operands in registers and
// reads the next chunk's, each behind a product (fenced: a product holds the MFMA pipe for 32
// cycles, in which its wave issues a read for free, while a group of reads between products
// holds the products up), so the copies run three chunks ahead into the buffer of the chunk
// in registers.  (With the end-of-chunk barrier left out and the exchange slots doubled the
// chains alone gain 4%, but the copies then come in one burst and the whole is 8% slower.)
template <int D, int DV>
struct DsGeo {
    static constexpr int NC = DV / 16, NT = D / 16, NH = NT / 2, NI = kC16 * D * 4 / 1024, TILE = kC16 * D * 4;
    static constexpr int NB = 3, WAVES = 4 * NC + 2;
    // state half: K^, K- rows, T''^T, V columns, gC
    static constexpr int H_KH = 0, H_KB = TILE, H_T = 2 * TILE, H_V = H_T + 1024, H_G = H_V + NC * 1024;
    static constexpr int HBUF = H_G + D * 4;
    static constexpr int H_NCP = 3 * NI + 1 + NC + D / 64;
    // gradient half: K^, K- rows, Q^ in operand order, dO columns, T, P, gC and beta
    static constexpr int S_KH = 0, S_KB = TILE, S_QH = 2 * TILE, S_O = 3 * TILE, S_T = S_O + NC * 1024, S_P = S_T + 1024, S_G = S_P + 1024;
    static constexpr int SBUF = S_G + DecRec<D>::GBN * 4;
    static constexpr int S_NCP = 2 * NI + 2 + NC + DecRec<D>::GBN / 64;
    static constexpr int S_NST = 2 * NC;  // W and dV stores per chunk
    static constexpr int OFF_S = NB * HBUF;
    static constexpr int OFF_X = OFF_S + NB * SBUF;     // half products: S, G x NC x 2 halves
    static constexpr int OFF_W = OFF_X + 4 * NC * 1024; // 2 slots x NC: W, beta
    static constexpr int WSLOT = 1024 + 64;
    static constexpr int BYTES = OFF_W + 2 * NC * WSLOT;
    static_assert(BYTES <= 160 * 1024 && S_NCP + S_NST <= 63 && H_NCP <= 63, "LDS / vmcnt");
    static_assert(HBUF % 16 == 0 && SBUF % 16 == 0, "alignment");
};

// GE: bytes per element of dQ, dK and dV (4: fp32; 2: bf16, rounded to nearest even)
template <int D, int DV, typename InT, int GE>
__global__ __launch_bounds__((DsGeo<D, DV>::WAVES * 64)) void dec_sweep_kernel(
    const InT* __restrict__ v, const float* __restrict__ s0, const float* __restrict__ go,
    const float* __restrict__ gs, void* __restrict__ gv, float* __restrict__ gs0, const float* __restrict__ kh,
    const float* __restrict__ kb, const float* __restrict__ qh, const float* __restrict__ rec,
    float* __restrict__ w_out, float* __restrict__ u_out, float* __restrict__ s_hist, float* __restrict__ g_hist,
    int n_pairs, int T, int H, int n_ch, int n_span, int span_len) {
    using G = DsGeo<D, DV>;
    using R = DecRec<D>;
    constexpr int NC = G::NC, NT = G::NT, NH = G::NH, NI = G::NI, NB = G::NB, n_tiles = D / DV;
    extern __shared__ __attribute__((aligned(16))) unsigned char smem[];
    // XCD-aware placement: the n_tiles workgroups of a pair share bid % 8
    const int bid = blockIdx.x, xcd = bid & 7, bslot = bid >> 3;
    const int tile = bslot % n_tiles, pair = (bslot / n_tiles) * 8 + xcd;
    if (pair >= n_pairs || n_ch <= 0) return;
    const int seq = pair / H, h = pair % H;
    const size_t tok0 = static_cast<size_t>(seq) * T;
    const int col0 = tile * DV;
    const int w = static_cast<int>(uniform(threadIdx.x >> 6)), lane = threadIdx.x & 63;
    const int r = lane & 15, g = lane >> 4;
    const size_t tstride = static_cast<size_t>(H) * D;
    const size_t sbase = static_cast<size_t>(pair) * D * D;
    const size_t item0 = static_cast<size_t>(pair) * n_ch;

    auto hbuf = [=](int c) { return smem + (c % NB) * G::HBUF; };
    auto sbuf = [=](int c) { return smem + G::OFF_S + (c % NB) * G::SBUF; };
    auto wslot = [=](int c, int which) { return smem + G::OFF_W + ((c & 1) * NC + which) * G::WSLOT; };
    auto row0_of = [=](int c, int col) { return (tok0 + c * kC16) * tstride + static_cast<size_t>(h) * D + col; };
    auto els_of = [=](int c, int cols) {  // elements from a column block's first row to its last row's end
        return static_cast<unsigned>((min(kC16, T - c * kC16) - 1) * tstride + cols);
    };
    auto copy_tile = [=](const float* ws, int c, unsigned char* dst) __attribute__((always_inline)) {
        const __amdgpu_buffer_rsrc_t rs = make_rsrc(ws + (item0 + c) * kC16 * D, G::TILE);
        unsigned char* d0 = uniform_ptr(dst);
#pragma unroll
        for (int i = 0; i < NI; ++i) dma16_asm(rs, d0 + 1024 * i, static_cast<unsigned>(1024 * i + 16 * lane));
    };

    if (w < 4 * NC) {
        // ============ chain waves: columns col0 + 16 cw + [0, 16), tiles m = hh + 2 j of 16 rows ============
        const bool state = w < 2 * NC;
        const int cw = (w >> 1) % NC, hh = w & 1;
        const int ecol = col0 + 16 * cw + r;
        const TileIdx<D> ix(r, g, hh);
        unsigned char* const xs = smem + G::OFF_X + ((state ? 0 : NC) + cw) * 2048 + 16 * lane;
        f32x4_t M[NH];  // this wave's rows of S or G
        {
            const float* m0 = state ? s0 : gs;
#pragma unroll
            for (int j = 0; j < NH; ++j)
#pragma unroll
                for (int e = 0; e < 4; ++e)
                    M[j][e] = m0 ? m0[sbase + static_cast<size_t>(16 * (hh + 2 * j) + 4 * g + e) * D + ecol] : 0.f;
        }
        __builtin_amdgcn_s_waitcnt(0x0F70);  // vmcnt(0), seen by the compiler: no wait for these in the loop
        __builtin_amdgcn_s_setprio(3);
        lds_barrier();  // B0
        // this wave's operand over d (rows) and onto d (columns), and the decay of its rows
        f32x4_t kf[NH], gc[NH];
        float kt[4][NH];
        auto rd_kt = [&](const unsigned char* b, int e, int j) __attribute__((always_inline)) { kt[e][j] = ix.col2(b, e, j); };
        // a product over d from this wave's half and, after the barrier, the other's
        auto total = [&](f32x4_t p) __attribute__((always_inline)) {
            return p + ld4(xs + 1024 * (hh ^ 1));
        };
        if (state) {
            f32x4_t vr, tt;
            auto rd_v = [&](const unsigned char* b, int e) __attribute__((always_inline)) {
                vr[e] = to_f32<InT>(reinterpret_cast<const InT*>(b + G::H_V + 1024 * cw)[(4 * g + e) * 16 + r]);
            };
            auto rd_gc = [&](const unsigned char* b, int j) __attribute__((always_inline)) {
                gc[j] = ld4(b + G::H_G + 4 * (16 * (hh + 2 * j) + 4 * g));
            };
            {
                const unsigned char* b = hbuf(0);
#pragma unroll
                for (int j = 0; j < NH; ++j) {
                    kf[j] = ix.row2(b + G::H_KH, j);
                    rd_gc(b, j);
                }
#pragma unroll
                for (int e = 0; e < 4; ++e) {
                    rd_v(b, e);
#pragma unroll
                    for (int j = 0; j < NH; ++j) rd_kt(b + G::H_KB, e, j);
                }
                tt = ld4(b + G::H_T + 16 * lane);
                __builtin_amdgcn_s_waitcnt(0xC07F);
                lds_barrier();  // B1: chunk 0's buffer may be refilled
            }
            for (int i = 0; i < n_ch; ++i) {
                const unsigned char* bn = hbuf(min(i + 1, n_ch - 1));  // (the last chunk reads itself again, unused)
                // X = K^ S - V, this wave's half
                f32x4_t xa[4] = {kZero4, kZero4, kZero4, kZero4};
                if (hh == 0) xa[0] = -vr;
                fence();
#pragma unroll
                for (int j = 0; j < NH; ++j)
#pragma unroll
                    for (int e = 0; e < 4; ++e) {
                        xa[e] = mfma4(kf[j][e], M[j][e], xa[e]);
                        if (e == 1 && j > 0) kf[j - 1] = ix.row2(bn + G::H_KH, j - 1);
                        if (j < 2 && (e == 2 || e == 3)) rd_v(bn, 2 * j + e - 2);
                        fence();
                    }
                kf[NH - 1] = ix.row2(bn + G::H_KH, NH - 1);
                const f32x4_t p = (xa[0] + xa[1]) + (xa[2] + xa[3]);
                st4(xs + 1024 * hh, p);
                if ((i & (span_len - 1)) == 0) {
                    float* hp = s_hist + ((static_cast<size_t>(pair) * n_span + i / span_len) * NT + col0 / 16 + cw) * NT * 256;
#pragma unroll
                    for (int j = 0; j < NH; ++j) *reinterpret_cast<f32x4_t*>(hp + (hh + 2 * j) * 256 + 4 * lane) = M[j];
                }
                lds_barrier();  // mid-chunk: the halves are in LDS
                const f32x4_t X = total(p);
                const f32x4_t tn = ld4(bn + G::H_T + 16 * lane);
                f32x4_t u0 = mfma4(tt[0], X[0], kZero4), u1 = mfma4(tt[1], X[1], kZero4);
                __asm__ volatile("" : "+v"(u0), "+v"(u1));  // (issued here, with what follows in their shadow)
#pragma unroll
                for (int j = 0; j < NH; ++j) {
                    M[j] = gc[j] * M[j];
                    __asm__ volatile("" : "+v"(M[j]));
                    rd_gc(bn, j);
                }
                const bool xbad = any_bad(X);
                u0 = mfma4(tt[2], X[2], u0), u1 = mfma4(tt[3], X[3], u1);
                f32x4_t U = u0 + u1;
                if (__builtin_expect(xbad, 0)) {
                    const int b = first_bad(X, g);
                    U = before(b, g, mm16(tt, before(b, g, X, kZero4)), U);
                }
                // S = Diag(gC) S + K-^T U
                fence();
#pragma unroll
                for (int e = 0; e < 4; ++e)
#pragma unroll
                    for (int j = 0; j < NH; ++j) {
                        M[j] = mfma4(kt[e][j], U[e], M[j]);
                        if (e > 0) rd_kt(bn + G::H_KB, e - 1, j);
                        if (e == 3) rd_kt(bn + G::H_KB, 3, j);
                        fence();
                    }
                // U's rows (U^T = X^T T''^T): lane (g, r) holds U[r][col0 + 16 cw + 4 g ..]
                if (hh == 0) {
                    f32x4_t Ur = mm16(X, tt);
                    if (__builtin_expect(xbad, 0)) {
                        const int b = first_bad(X, g);
                        const f32x4_t clean = mm16(before(b, g, X, kZero4), tt);
#pragma unroll
                        for (int e = 0; e < 4; ++e) Ur[e] = r < __shfl(b, 4 * g + e) ? clean[e] : Ur[e];
                    }
                    *reinterpret_cast<f32x4_t*>(u_out + (item0 + i) * kC16 * D +
                                                4 * f32_chunk<D>(r, (col0 + 16 * cw) / 4 + g)) = Ur;
                }
                tt = tn;
                __builtin_amdgcn_s_waitcnt(0xC07F);  // lgkmcnt(0), seen by the compiler
                lds_barrier();                       // end of the chunk
            }
        } else {
            f32x4_t dOc, ta, b4, qc[NH];
            bool obad;  // any_bad(dOc)
            f32x2_t pp;  // P^T's operand for tokens e = 2 hh, 2 hh + 1: each half adds its part of P^T dO
            auto rd_do = [&](const unsigned char* b, int e) __attribute__((always_inline)) {
                return reinterpret_cast<const float*>(b + G::S_O + 1024 * cw)[(4 * g + e) * 16 + r];
            };
            auto rd_gc = [&](const unsigned char* b, int j) __attribute__((always_inline)) {
                gc[j] = ld4(b + G::S_G + 4 * (16 * (hh + 2 * j) + 4 * g));
            };
            auto rd_q = [&](const unsigned char* b, int j) __attribute__((always_inline)) {
                qc[j] = ld4(b + G::S_QH + 1024 * (hh + 2 * j) + 16 * lane);
            };
            {
                const unsigned char* b = sbuf(n_ch - 1);
#pragma unroll
                for (int j = 0; j < NH; ++j) {
                    kf[j] = ix.row2(b + G::S_KB, j);
                    rd_q(b, j);
                    rd_gc(b, j);
                }
#pragma unroll
                for (int e = 0; e < 4; ++e) {
                    dOc[e] = rd_do(b, e);
#pragma unroll
                    for (int j = 0; j < NH; ++j) rd_kt(b + G::S_KH, e, j);
                }
                ta = ld4(b + G::S_T + 16 * lane);
                pp = *reinterpret_cast<const f32x2_t*>(b + G::S_P + 16 * lane + 8 * hh);
                b4 = ld4(b + G::S_G + 4 * D + 16 * g);
                __builtin_amdgcn_s_waitcnt(0xC07F);
                obad = any_bad(dOc);
                lds_barrier();  // B1
            }
            for (int c = n_ch - 1; c >= 0; --c) {
                const unsigned char* bn = sbuf(max(c - 1, 0));
                f32x4_t dOn, tn, bn4;
                f32x2_t pn;
                if (c == n_ch - 1 || ((c + 1) & (span_len - 1)) == 0) {
                    float* hp = g_hist + ((static_cast<size_t>(pair) * n_span + c / span_len) * NT + col0 / 16 + cw) * NT * 256;
#pragma unroll
                    for (int j = 0; j < NH; ++j) *reinterpret_cast<f32x4_t*>(hp + (hh + 2 * j) * 256 + 4 * lane) = M[j];
                }
                // dU = K- G + P^T dO, this wave's half; a tile's decay behind its last product
                f32x4_t ya[4] = {kZero4, kZero4, kZero4, kZero4};
                float do0 = hh ? dOc[2] : dOc[0], do1 = hh ? dOc[3] : dOc[1];
                if (__builtin_expect(obad, 0)) {
                    do0 = bad(do0) ? 0.f : do0;
                    do1 = bad(do1) ? 0.f : do1;
                }
                ya[0] = mfma4(pp[0], do0, kZero4);
                ya[1] = mfma4(pp[1], do1, kZero4);
                fence();
#pragma unroll
                for (int j = 0; j < NH; ++j)
#pragma unroll
                    for (int e = 0; e < 4; ++e) {
                        ya[e] = mfma4(kf[j][e], M[j][e], ya[e]);
                        if (e == 1 && j > 0) kf[j - 1] = ix.row2(bn + G::S_KB, j - 1);
                        if (j < 2 && (e == 2 || e == 3)) dOn[2 * j + e - 2] = rd_do(bn, 2 * j + e - 2);
                        if (e == 0 && j > 0) M[j - 1] = gc[j - 1] * M[j - 1];
                        fence();
                    }
                kf[NH - 1] = ix.row2(bn + G::S_KB, NH - 1);
                M[NH - 1] = gc[NH - 1] * M[NH - 1];
                fence();
                // G = Diag(gC) G + Q^^T dO: half of it ahead of the exchange, the rest in its latency
                auto q_prod = [&](int e, int j) __attribute__((always_inline)) { M[j] = mfma4(qc[j][e], dOc[e], M[j]); };
#pragma unroll
                for (int j = 0; j < NH; ++j) {
                    q_prod(0, j);
                    rd_gc(bn, j);
                    fence();
                }
                const f32x4_t p = (ya[0] + ya[1]) + (ya[2] + ya[3]);
                st4(xs + 1024 * hh, p);
                fence();
#pragma unroll
                for (int j = 0; j < NH; ++j) {
                    q_prod(1, j);
                    if (j == 0) tn = ld4(bn + G::S_T + 16 * lane);
                    if (j == 1) pn = *reinterpret_cast<const f32x2_t*>(bn + G::S_P + 16 * lane + 8 * hh);
                    fence();
                }
                lds_barrier();  // mid-chunk
                const f32x4_t po = ld4(xs + 1024 * (hh ^ 1));
                fence();
#pragma unroll
                for (int j = 0; j < NH; ++j) {
                    q_prod(2, j);
                    fence();
                }
                // W = T^T dU
                const f32x4_t dU = p + po;
                f32x4_t w0 = mfma4(ta[0], dU[0], kZero4), w1 = mfma4(ta[1], dU[1], kZero4);
                __asm__ volatile("" : "+v"(w0), "+v"(w1));  // (issued here, not where the sum needs them)
                fence();
                q_prod(3, 0);
                rd_q(bn, 0);
                fence();
                w0 = mfma4(ta[2], dU[2], w0), w1 = mfma4(ta[3], dU[3], w1);
                __asm__ volatile("" : "+v"(w0), "+v"(w1));
                const bool wbad = static_cast<int>(obad) | static_cast<int>(any_bad(dU));
                fence();
#pragma unroll
                for (int j = 1; j < NH; ++j) {
                    q_prod(3, j);
                    rd_q(bn, j);
                    if (j == 1) bn4 = ld4(bn + G::S_G + 4 * D + 16 * g);
                    fence();
                }
                f32x4_t W = w0 + w1;
                if (__builtin_expect(wbad, 0)) {
                    const int b = max(last_bad(dOc, g), last_bad(dU, g)) + 1;
                    W = before(b, g, kZero4 + __builtin_nanf(""), mm16(ta, before(b, g, kZero4, dU)));
                }
                const f32x4_t nbW = -(W * b4);
                // G -= K^^T diag(beta) W
                fence();
#pragma unroll
                for (int e = 0; e < 4; ++e)
#pragma unroll
                    for (int j = 0; j < NH; ++j) {
                        M[j] = mfma4(kt[e][j], nbW[e], M[j]);
                        if (e > 0) rd_kt(bn + G::S_KH, e - 1, j);
                        if (e == 3) rd_kt(bn + G::S_KH, 3, j);
                        if (e == 0 && j == 0 && hh == 0) st4(wslot(c, cw) + 16 * lane, W);
                        if (e == 0 && j == 1 && hh == 0 && r == 0) st4(wslot(c, cw) + 1024 + 16 * g, b4);
                        if (e == 2 && j == 0) obad = any_bad(dOn);
                        fence();
                    }
                dOc = dOn, ta = tn, pp = pn, b4 = bn4;
                __builtin_amdgcn_s_waitcnt(0xC07F);
                lds_barrier();  // end of the chunk
            }
#pragma unroll
            for (int j = 0; j < NH; ++j)
#pragma unroll
                for (int e = 0; e < 4; ++e)
                    gs0[sbase + static_cast<size_t>(16 * (hh + 2 * j) + 4 * g + e) * D + ecol] = M[j][e];
        }
    } else if (w == 4 * NC) {
        // ============ the state half's copies, three chunks ahead ============
        // (each half of a chunk issues half of the copies: 28 in one go hold the barrier up)
        auto copies_a = [=](int c) __attribute__((always_inline)) {
            unsigned char* b = hbuf(c);
            copy_tile(kh, c, b + G::H_KH);
            copy_tile(kb, c, b + G::H_KB);
        };
        auto copies_b = [=](int c) __attribute__((always_inline)) {
            unsigned char* b = hbuf(c);
            const float* rc = rec + (item0 + c) * R::FLOATS;
            copy_tile(qh, n_ch - 1 - c, sbuf(n_ch - 1 - c) + G::S_QH);  // (a share of the gradient half's)
            dma16_asm(make_rsrc(rc + R::T2, 1024), uniform_ptr(b + G::H_T), static_cast<unsigned>(16 * lane));
            constexpr int LPR = 16 * sizeof(InT) / 16;  // lanes per row of 16 columns
#pragma unroll
            for (int j = 0; j < NC; ++j)  // (bf16: lanes 32 .. 63 address rows past the chunk and read zeros)
                dma16_asm(make_rsrc(v + row0_of(c, col0 + 16 * j), els_of(c, 16) * sizeof(InT)),
                          uniform_ptr(b + G::H_V + 1024 * j),
                          static_cast<unsigned>((lane / LPR) * tstride * sizeof(InT) + 16 * (lane % LPR)));
            const __amdgpu_buffer_rsrc_t rg = make_rsrc(rc + R::GB, D * 4);
#pragma unroll
            for (int j = 0; j < D / 64; ++j)
                dma4_asm(rg, uniform_ptr(b + G::H_G + 256 * j), static_cast<unsigned>(256 * j + 4 * lane));
        };
        auto copies = [=](int c) __attribute__((always_inline)) {
            copies_a(c);
            copies_b(c);
        };
        copies(0);
        if (n_ch > 1) copies(1);
        if (n_ch > 2) {
            copies(2);
            wait_vm_n<G::H_NCP>();
        } else {
            wait_vm_n<0>();
        }
        lds_barrier();  // B0: chunks 0 and 1 landed
        lds_barrier();  // B1
        for (int i = 0; i < n_ch; ++i) {
            // chunk i's buffer is free (its operands were read before this iteration); chunk i + 2
            // has landed at the end
            if (i + 3 < n_ch) copies_a(i + 3);
            lds_barrier();  // mid-chunk
            if (i + 3 < n_ch) {
                copies_b(i + 3);
                wait_vm_n<G::H_NCP>();
            } else {
                wait_vm_n<0>();
            }
            lds_barrier();
        }
    } else {
        // ============ the gradient half's copies, and its stores one chunk behind ============
        auto copies_a = [=](int c) __attribute__((always_inline)) {
            unsigned char* b = sbuf(c);
            copy_tile(kh, c, b + G::S_KH);
            copy_tile(kb, c, b + G::S_KB);
        };
        auto copies_b = [=](int c) __attribute__((always_inline)) {
            unsigned char* b = sbuf(c);
            const float* rc = rec + (item0 + c) * R::FLOATS;
#pragma unroll
            for (int j = 0; j < NC; ++j)  // a null dO reads zeros (a zero-length range)
                dma16_asm(make_rsrc(go ? go + row0_of(c, col0 + 16 * j) : go, go ? els_of(c, 16) * 4 : 0u),
                          uniform_ptr(b + G::S_O + 1024 * j),
                          static_cast<unsigned>((lane >> 2) * tstride * 4 + 16 * (lane & 3)));
            dma16_asm(make_rsrc(rc + R::TA, 1024), uniform_ptr(b + G::S_T), static_cast<unsigned>(16 * lane));
            dma16_asm(make_rsrc(rc + R::PA, 1024), uniform_ptr(b + G::S_P), static_cast<unsigned>(16 * lane));
            const __amdgpu_buffer_rsrc_t rg = make_rsrc(rc + R::GB, R::GBN * 4);
#pragma unroll
            for (int j = 0; j < R::GBN / 64; ++j)
                dma4_asm(rg, uniform_ptr(b + G::S_G + 256 * j), static_cast<unsigned>(256 * j + 4 * lane));
        };
        auto store = [=](int cs) __attribute__((always_inline)) {
            const int t = lane >> 2, p = lane & 3;
#pragma unroll
            for (int j = 0; j < NC; ++j) {
                const float* ws = reinterpret_cast<const float*>(wslot(cs, j));
                const float bt = ws[256 + t];
                f32x4_t x;
#pragma unroll
                for (int e = 0; e < 4; ++e) x[e] = ws[4 * (16 * (t >> 2) + 4 * p + e) + (t & 3)];
                *reinterpret_cast<f32x4_t*>(w_out + (item0 + cs) * kC16 * D +
                                            4 * f32_chunk<D>(t, (col0 + 16 * j) / 4 + p)) = x;
                const __amdgpu_buffer_rsrc_t rv = make_rsrc(
                    static_cast<unsigned char*>(gv) + row0_of(cs, col0 + 16 * j) * GE, els_of(cs, 16) * GE);
                const unsigned off = static_cast<unsigned>((t * tstride + 4 * p) * GE);
                if constexpr (GE == 2)
                    __builtin_amdgcn_raw_buffer_store_b64(cvt4(x * bt), rv, off, 0, 0);
                else
                    __builtin_amdgcn_raw_buffer_store_b128(__builtin_bit_cast(u32x4_t, x * bt), rv, off, 0, 0);
            }
        };
        auto copies = [=](int c) __attribute__((always_inline)) {
            copies_a(c);
            copies_b(c);
        };
        const int last = n_ch - 1;
        copies(last);
        if (n_ch > 1) copies(last - 1);
        if (n_ch > 2) {
            copies(last - 2);
            wait_vm_n<G::S_NCP>();
        } else {
            wait_vm_n<0>();
        }
        lds_barrier();  // B0
        lds_barrier();  // B1
        for (int c = last; c >= 0; --c) {
            const bool cp = c >= 3, st = c < last;
            // chunk c's buffer is free; chunk c - 2 has landed at the end (the newest copies and
            // this iteration's stores may be in flight)
            if (cp) copies_a(c - 3);
            lds_barrier();  // mid-chunk
            if (cp) copies_b(c - 3);
            if (st) store(c + 1);  // what the chains handed over in the last chunk
            if (cp && st) wait_vm_n<G::S_NCP + G::S_NST>();
            else if (cp) wait_vm_n<G::S_NCP>();
            else wait_vm_n<0>();
            lds_barrier();
        }
        store(0);
    }
}

// ---------------------------------------------------------------- K10c
// Wave w owns rows 16 w + [0, 16) of d: lane (g, r) holds S^T and G^T [16 i + 4 g + e][16 w + r]
// in tile i, and of each chunk's tokens 4 g + e the values at d = 16 w + r (k, q, v, alpha
// from global memory, one chunk ahead), from which it forms its decay factors: its own four
// alphas give F^4 and E^4, two lane exchanges the levels 8 and 16.  The pairs (t, s) of
// levels 8 and 4 are masked matrix products over the chunk's tokens, those inside a lane's
// four tokens plain arithmetic.
template <int D>
struct DcGeo {
    static constexpr int NW = D / 16, NT = D / 16, NI = kC16 * D * 4 / 1024, TILE = kC16 * D * 4;
    static constexpr int B_O = 0, B_W = TILE, B_U = 2 * TILE, BUF = 3 * TILE;  // dO, W, U rows
    static constexpr int NC = 3 * NI;                        // copies per chunk
    static constexpr int OFF_PP = 2 * BUF;                   // per wave: dO U^T, W U^T parts [t][s]
    static constexpr int OFF_TR = OFF_PP + NW * 2048;        // totals dP, diag(beta) dA as rows [t][s]
    static constexpr int OFF_TC = OFF_TR + 2048;             // ... as columns [s][t], stride 20
    static constexpr int OFF_DB = OFF_TC + 2 * 16 * 20 * 4;  // dbeta parts: 2 slots x NW x 16
    static constexpr int OFF_GG = OFF_DB + 2 * NW * 64;      // per-head gate: dg parts, chunk x wave x 16
    static constexpr int OFF_MID = OFF_GG + kSpan * NW * 64;  // S^T in mid-span
    static constexpr int BYTES = OFF_MID + NW * NT * 1024;
    static_assert(BYTES <= 160 * 1024, "LDS");
};

template <int D, typename InT, bool CHAN, int GE>
__global__ __launch_bounds__(D * 4) void dec_span_kernel(
    const InT* __restrict__ q, const InT* __restrict__ k, const InT* __restrict__ v, const float* __restrict__ gate,
    const float* __restrict__ go, const float* __restrict__ rec, const float* __restrict__ s_hist,
    const float* __restrict__ g_hist, const float* __restrict__ w_in, const float* __restrict__ u_in,
    void* __restrict__ gq, void* __restrict__ gk, float* __restrict__ gbeta, float* __restrict__ gg,
    float* __restrict__ pk_ws, float* __restrict__ pg_ws, float* __restrict__ s_ch, int T, int H, int n_ch, int n_span, int span_len) {
    // multiply-adds are fused only where written so (fmaf): every build of this kernel gives the
    // same bits, and bf16 gradients are the fp32 ones rounded
#pragma clang fp contract(off)
    using G = DcGeo<D>;
    using R = DecRec<D>;
    constexpr int NW = G::NW, NT = G::NT;
    extern __shared__ __attribute__((aligned(16))) unsigned char smem[];
    const int pair = blockIdx.x / n_span, span = blockIdx.x % n_span;
    const int seq = pair / H, h = pair % H;
    const int c0 = span * span_len, nm = min(span_len, n_ch - c0);  // chunks of this span
    const size_t tok0 = static_cast<size_t>(seq) * T + static_cast<size_t>(c0) * kC16;
    const int tid = threadIdx.x, lane = tid & 63;
    const int w = static_cast<int>(uniform(static_cast<unsigned>(tid >> 6)));
    const int r = lane & 15, g = lane >> 4;
    const size_t tstride = static_cast<size_t>(H) * D;
    const size_t item0 = static_cast<size_t>(pair) * n_ch + c0;
    const TileIdx<D> ix(r, g);

    auto buf = [=](int m) { return smem + (m & 1) * G::BUF; };
    auto clen_of = [=](int m) { return min(kC16, T - (c0 + m) * kC16); };
    auto row0_of = [=](int m, int col) { return (tok0 + m * kC16) * tstride + static_cast<size_t>(h) * D + col; };
    // copy number x of chunk m (one branch per source); wave w issues x = w, w + NW, ...
    auto issue = [=](int m) __attribute__((always_inline)) {
        unsigned char* b = buf(m);
#pragma unroll
        for (int n = 0; n < G::NC / NW; ++n) {
            const int x = w + n * NW, which = x / G::NI, i = x % G::NI;
            if (which == 0) {
                // dO rows, swizzled here; a null dO reads zeros (a zero-length range)
                const int ch = 64 * i + lane, t = ch / (D / 4), p = (ch % (D / 4)) ^ t;
                const unsigned nb = static_cast<unsigned>(((clen_of(m) - 1) * tstride + D) * 4);
                dma16_asm(make_rsrc(go ? go + row0_of(m, 0) : go, go ? nb : 0u), uniform_ptr(b + G::B_O + 1024 * i),
                          static_cast<unsigned>(t * tstride * 4 + 16 * p));
            } else if (which == 1) {
                dma16_asm(make_rsrc(w_in + (item0 + m) * kC16 * D, G::TILE), uniform_ptr(b + G::B_W + 1024 * i),
                          static_cast<unsigned>(1024 * i + 16 * lane));
            } else {
                dma16_asm(make_rsrc(u_in + (item0 + m) * kC16 * D, G::TILE), uniform_ptr(b + G::B_U + 1024 * i),
                          static_cast<unsigned>(1024 * i + 16 * lane));
            }
        }
    };
    constexpr int kMine = G::NC / NW;  // copies each wave issues per chunk
    static_assert(G::NC % NW == 0, "copies divide over the waves");

    // this lane's four values of a chunk in the scratch that the way forwards leaves the
    // gradients of k and of a per-channel gate in for the way back (fp32, one 16-byte store)
    auto part_of = [=](int m) { return (item0 + m) * kC16 * D + 256 * w + 4 * lane; };
    // this lane's tokens of a chunk, as loaded (tokens past the end read zeros)
    struct Own {
        f32x4_t k, q, x, lg, b4;  // x: v (forwards) or the gradient so far of k (backwards)
        f32x4_t y;                // forwards: A'[r][4 g ..]; backwards: the gradient so far of the gate
        float br;
    };
    auto load_own = [=](int m, bool fwd) __attribute__((always_inline)) {
        Own o;
        const int clen = clen_of(m);
        const unsigned nel = static_cast<unsigned>((clen - 1) * tstride + 16);
        const size_t r0 = row0_of(m, 16 * w);
        const __amdgpu_buffer_rsrc_t rk = make_rsrc(k + r0, nel * sizeof(InT)), rq = make_rsrc(q + r0, nel * sizeof(InT));
        const __amdgpu_buffer_rsrc_t rv = make_rsrc(v + r0, nel * sizeof(InT));
        const __amdgpu_buffer_rsrc_t rg = CHAN ? make_rsrc(gate + r0, nel * 4)
                                               : make_rsrc(gate + (tok0 + m * kC16) * H + h,
                                                           static_cast<unsigned>(((clen - 1) * H + 1) * 4));
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            const unsigned el = static_cast<unsigned>((4 * g + e) * tstride + r);
            o.k[e] = buf_el<InT>(rk, el);
            o.q[e] = buf_el<InT>(rq, el);
            o.lg[e] = buf_el<float>(rg, CHAN ? el : static_cast<unsigned>((4 * g + e) * H));
            if (fwd) o.x[e] = buf_el<InT>(rv, el);
        }
        if (!fwd) {
            o.x = *reinterpret_cast<const f32x4_t*>(pk_ws + part_of(m));
            o.y = CHAN ? *reinterpret_cast<const f32x4_t*>(pg_ws + part_of(m)) : kZero4;
        }
        const float* rc = rec + (item0 + m) * R::FLOATS;
        if (fwd) o.y = *reinterpret_cast<const f32x4_t*>(rc + R::AT + 4 * lane);
        o.b4 = *reinterpret_cast<const f32x4_t*>(rc + R::GB + D + 4 * g);
        o.br = rc[R::GB + D + r];
        return o;
    };
    // decay factors of this lane's four tokens at d = 16 w + r
    struct Dec {
        f32x4_t al, F4, E4, F8, E8, F, E;
        float gc;
    };
    auto decays = [=](f32x4_t lg) __attribute__((always_inline)) {
        Dec x;
#pragma unroll
        for (int e = 0; e < 4; ++e) x.al[e] = expf(lg[e]);
        x.F4[0] = x.al[0];
#pragma unroll
        for (int e = 1; e < 4; ++e) x.F4[e] = x.F4[e - 1] * x.al[e];
        x.E4[3] = 1.f;
        x.E4[2] = x.al[3];
        x.E4[1] = x.al[2] * x.E4[2];
        x.E4[0] = x.al[1] * x.E4[1];
        const float s4 = __shfl_xor(x.F4[3], 16);  // the sibling block's product
        x.F8 = (g & 1) ? x.F4 * s4 : x.F4;
        x.E8 = (g & 1) ? x.E4 : x.E4 * s4;
        const float t8 = x.F4[3] * s4, s8 = __shfl_xor(t8, 32);
        x.F = (g & 2) ? x.F8 * s8 : x.F8;
        x.E = (g & 2) ? x.E8 : x.E8 * s8;
        x.gc = t8 * s8;
        return x;
    };
    // sums over the 16 tokens of a lane's column (4 own, 4 lane groups), all groups equal
    auto col_total = [=](f32x4_t x) __attribute__((always_inline)) {
        float s = (x[0] + x[1]) + (x[2] + x[3]);
        s += __shfl_xor(s, 16);
        s += __shfl_xor(s, 32);
        return s;
    };

    // tile i of S^T or G^T at the span's start or end, by rows of d, gathered from the column-block
    // layout: S[16 w + r][16 i + 4 g + e] is in column block i, tile w, lane 16 (r >> 2) + 4 g + e,
    // register r & 3
    auto gather = [=](const float* hist, int i) __attribute__((always_inline)) {
        const __amdgpu_buffer_rsrc_t rs = make_rsrc(hist + (static_cast<size_t>(pair) * n_span + span) * D * D, D * D * 4);
        const unsigned off = static_cast<unsigned>(4 * (4 * (16 * (r >> 2) + 4 * g) + (r & 3)));
        f32x4_t x;
#pragma unroll
        for (int e = 0; e < 4; ++e)
            x[e] = __uint_as_float(__builtin_amdgcn_raw_buffer_load_b32(rs, off + 16 * e, (i * NT + w) * 1024, 0));
        return x;
    };
    // this wave's S^T at the start of chunk m, left for the way back; m = 0 is in s_hist, m =
    // span_len / 2 in LDS, and the last chunk's stays in registers
    auto start_of = [=](int m) __attribute__((always_inline)) {
        const size_t slot = (static_cast<size_t>(pair) * n_span + span) * kept_starts(span_len) + m - (m < span_len / 2 ? 1 : 2);
        return make_rsrc(s_ch + slot * D * D + w * NT * 256, NT * 1024);
    };
    f32x4_t St[NT];
#pragma unroll
    for (int i = 0; i < NT; ++i) St[i] = gather(s_hist, i);
    issue(0);
    if (nm > 1) issue(1);
    Own own = load_own(0, true);
    wait_vm_n<0>();
    lds_barrier();

    // ================ forwards ================
    // S^T in mid-span, kept for the way back (this wave's own)
    unsigned char* const mid = smem + G::OFF_MID + w * NT * 1024 + 16 * lane;
    for (int m = 0; m < nm; ++m) {
        const unsigned char* b = buf(m);
        Own next = own;  // the next chunk's values, loaded a whole chunk ahead
        if (m + 1 < nm) next = load_own(m + 1, true);
        // dO S^T, W S^T, and this wave's parts of dO U^T and W U^T.  (Operand reads go two
        // tiles ahead of their products, fenced: left to itself the compiler reads each right
        // before its use and waits out the LDS latency.)
        f32x4_t qa[2] = {kZero4, kZero4}, wa[2] = {kZero4, kZero4}, pp = kZero4, pa = kZero4;
        {
            f32x4_t dor[NT], wrw[NT];
            const f32x4_t uw = ix.roww(b + G::B_U, w, r), dw = ix.roww(b + G::B_O, w, r), ww = ix.roww(b + G::B_W, w, r);
            auto rd = [&](int i) __attribute__((always_inline)) {
                dor[i] = ix.row(b + G::B_O, i);
                wrw[i] = ix.row(b + G::B_W, i);
            };
            rd(0);
            fence();
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                pp = mfma4(uw[e], dw[e], pp);  // (U dO^T)[4 g + v][r] = (dO U^T)[r][4 g + v]
                pa = mfma4(uw[e], ww[e], pa);
            }
            rd(1);
            fence();
#pragma unroll
            for (int i = 0; i < NT; ++i) {
                if (i + 2 < NT) rd(i + 2);
#pragma unroll
                for (int e = 0; e < 4; ++e) {
                    qa[e & 1] = mfma4(dor[i][e], St[i][e], qa[e & 1]);
                    wa[e & 1] = mfma4(wrw[i][e], St[i][e], wa[e & 1]);
                }
                fence();
            }
        }
        unsigned char* part = smem + G::OFF_PP + w * 2048;
        st4(part + 16 * (4 * r + g), pp);
        st4(part + 1024 + 16 * (4 * r + g), pa);
        const f32x4_t kk = own.k, qq = own.q, b4 = own.b4, at = own.y;
        const float br = own.br;
        const Dec x = decays(own.lg);
        const f32x4_t khat = kk * x.F, kbar = kk * x.E;
        const f32x4_t dQh = qa[0] + qa[1];          // dO S^T [4 g + v][16 w + r]
        const f32x4_t WS = wa[0] + wa[1];           // W S^T
        const f32x4_t kdk = -(b4 * WS);             // dL/dK^
        const bool last = m + 1 == nm;
        if (m == span_len / 2 && !last) {
#pragma unroll
            for (int i = 0; i < NT; ++i) st4(mid + 1024 * i, St[i]);
        } else if (m != 0 && !last) {
            const __amdgpu_buffer_rsrc_t rs = start_of(m);
#pragma unroll
            for (int i = 0; i < NT; ++i)
                __builtin_amdgcn_raw_buffer_store_b128(__builtin_bit_cast(u32x4_t, St[i]), rs, 16 * lane, 1024 * i, 0);
        }
        lds_barrier();  // Y: the parts are in LDS
        // the totals' operands, read here and summed behind the state update
        constexpr int NZ = 512 / (NW * 64);  // entries of [dP, dA][t][s] per thread
        float tv[NZ][NW];
#pragma unroll
        for (int n = 0; n < NZ; ++n)
#pragma unroll
            for (int u = 0; u < NW; ++u)
                tv[n][u] = reinterpret_cast<const float*>(smem + G::OFF_PP + u * 2048)[tid + n * NW * 64];
        f32x4_t wj;  // W at this lane's columns 16 w + r of d_v
#pragma unroll
        for (int e = 0; e < 4; ++e) wj[e] = ix.colw(b + G::B_W, e, w, g);
        // S^T = gC S^T + U^T K-, tiles i and i + 4 together (their reads pair up); nothing reads the
        // span's end state
        if (!last) {
            constexpr int NP = NT > 4 ? 2 : 1;
            float uc[2][NP][4];
            auto rd = [&](int i) __attribute__((always_inline)) {
#pragma unroll
                for (int e = 0; e < 4; ++e)
#pragma unroll
                    for (int p = 0; p < NP; ++p) uc[i & 1][p][e] = ix.col(b + G::B_U, e, i + 4 * p);
            };
            rd(0);
#pragma unroll
            for (int i = 0; i < NT; ++i) St[i] = St[i] * x.gc;
            fence();
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                if (i + 1 < 4) rd(i + 1);
#pragma unroll
                for (int e = 0; e < 4; ++e)
#pragma unroll
                    for (int p = 0; p < NP; ++p) St[i + 4 * p] = mfma4(uc[i & 1][p][e], kbar[e], St[i + 4 * p]);
                fence();
            }
        }
#pragma unroll
        for (int n = 0; n < NZ; ++n) {
            float sum = tv[n][0];
#pragma unroll
            for (int u = 1; u < NW; ++u) sum += tv[n][u];
            const int z = tid + n * NW * 64, mat = z >> 8, t = (z >> 4) & 15, s = z & 15;
            const float val = mat == 0 ? (s <= t ? sum : 0.f) : (s < t ? -sum : 0.f);
            reinterpret_cast<float*>(smem + G::OFF_TR + mat * 1024)[16 * t + s] = val;
            reinterpret_cast<float*>(smem + G::OFF_TC + mat * 1280)[20 * s + t] = val;
        }
        {
            // this wave's part of W.V - K^ . W S^T per token 4 g + v
            f32x4_t s = fma4(wj, own.x, -(khat * WS));
#pragma unroll
            for (int e = 0; e < 4; ++e) s[e] = row16_sum(s[e]);
            if (r == 0) st4(smem + G::OFF_DB + ((m & 1) * NW + w) * 64 + 16 * g, s);
        }
        // chunk m + 1's copies have landed (they are older than chunk m - 1's five stores, and those
        // of S^T above are the newest)
        if (m != 0 && m != span_len / 2 && !last) wait_vm_n<4 + NT>();
        else wait_vm_n<4>();
        lds_barrier();  // Z: totals in LDS, chunk m + 1 in its buffer, every wave done with chunk m's
        if (m + 2 < nm) issue(m + 2);
        const f32x4_t dpr = ld4(smem + G::OFF_TR + 16 * (4 * r + g));            // dP[r][4 g ..]
        const f32x4_t dar = ld4(smem + G::OFF_TR + 1024 + 16 * (4 * r + g));     // dA[r][4 g ..]
        const f32x4_t dpc = ld4(smem + G::OFF_TC + 4 * (20 * r + 4 * g));        // dP[4 g ..][r]
        const f32x4_t dac = ld4(smem + G::OFF_TC + 1280 + 4 * (20 * r + 4 * g)); // dA[4 g ..][r]
        // pairs between blocks of four tokens: rows (t = r, s = 4 g + e) and columns (s = r,
        // t = 4 g + e) of each level's mask; dA' = diag(beta) dA
        const int rb = r >> 2;
        const bool r8 = r >= 8 && g < 2, c8 = r < 8 && g >= 2;
        const bool r4 = (rb & 1) && g == rb - 1, c4 = !(rb & 1) && g == rb + 1;
        f32x4_t ke8 = kk * x.E8, kf8 = kk * x.F8, qf8 = qq * x.F8;
        f32x4_t ke4 = kk * x.E4, kf4 = kk * x.F4, qf4 = qq * x.F4;
        {
            // (as above: a token's infinity or NaN in k, q or the decays stays with its own pairs, in
            // which dP, dA or the decay by which a sum is scaled carries it too)
            const f32x4_t z = kk * kZero4 + qq * kZero4;
            if (__builtin_expect(any_bad(f32x4_t{z[0] + z[1], z[2] + z[3], x.gc, 0.f}), 0)) {
#pragma unroll
                for (int e = 0; e < 4; ++e)
                    for (f32x4_t* y : {&ke8, &kf8, &qf8, &ke4, &kf4, &qf4}) (*y)[e] = bad((*y)[e]) ? 0.f : (*y)[e];
            }
        }
        f32x4_t zq8 = kZero4, zk8 = kZero4, zc8 = kZero4, zq4 = kZero4, zk4 = kZero4, zc4 = kZero4;
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            const float a = dpr[e], bb = br * dar[e], cc = dpc[e], dd = dac[e] * b4[e];
            zq8 = mfma4(r8 ? a : 0.f, ke8[e], zq8);
            zk8 = mfma4(r8 ? bb : 0.f, ke8[e], zk8);
            zc8 = mfma4(c8 ? cc : 0.f, qf8[e], zc8);
            zq4 = mfma4(r4 ? a : 0.f, ke4[e], zq4);
            zk4 = mfma4(r4 ? bb : 0.f, ke4[e], zk4);
            zc4 = mfma4(c4 ? cc : 0.f, qf4[e], zc4);
            zc8 = mfma4(c8 ? dd : 0.f, kf8[e], zc8);
            zc4 = mfma4(c4 ? dd : 0.f, kf4[e], zc4);
        }
        f32x4_t pq = fma4(x.F8, zq8, x.F4 * zq4), pk = fma4(x.F8, zk8, x.F4 * zk4), pc = fma4(x.E8, zc8, x.E4 * zc4);
        // the gate's pair terms, t >= j > s: of a level, for j in the upper half of a block the rows
        // t from j on, for j in the lower half the columns s before j
        const bool up8 = g >= 2, up4 = g & 1;
        const f32x4_t x8 = (up8 ? x.F8 : x.E8) * (up8 ? fma4(qq, zq8, kk * zk8) : kk * zc8);
        const f32x4_t x4 = (up4 ? x.F4 : x.E4) * (up4 ? fma4(qq, zq4, kk * zk4) : kk * zc4);
        f32x4_t pg;
        {
            const float t8 = __shfl_xor((x8[0] + x8[1]) + (x8[2] + x8[3]), 16);  // the half's other four tokens
            const f32x4_t a = up8 ? x8 : f32x4_t{x8[2], x8[1], x8[0], 0.f};
            const f32x4_t b = up4 ? x4 : f32x4_t{x4[2], x4[1], x4[0], 0.f};
            const float a2 = a[3] + a[2], a1 = a2 + a[1], b2 = b[3] + b[2], b1 = b2 + b[1];
            const f32x4_t sa = {a1 + a[0], a1, a2, a[3]}, sb = {b1 + b[0], b1, b2, b[3]};  // from each on
            pg = (up8 ? sa : f32x4_t{0.f, sa[2], sa[1], sa[0]}) + (up4 ? sb : f32x4_t{0.f, sb[2], sb[1], sb[0]}) +
                 ((g == 1 || g == 2) ? t8 : 0.f);
        }
        // pairs inside this lane's four tokens
        f32x4_t dg;
#pragma unroll
        for (int a = 0; a < 4; ++a) {
            const f32x4_t dp = ld4(smem + G::OFF_TR + 16 * (4 * (4 * g + a) + g));         // dP[4 g + a][4 g ..]
            const f32x4_t da = ld4(smem + G::OFF_TR + 1024 + 16 * (4 * (4 * g + a) + g));  // dA[4 g + a][4 g ..]
            dg[a] = dp[a];
            float f = 1.f;  // D of (a, s)
#pragma unroll
            for (int s = a - 1; s >= 0; --s) {
                f *= x.al[s + 1];
                const float ws = kk[s] * f, ab = b4[a] * da[s], both = fmaf(dp[s], qq[a], ab * kk[a]);
                pq[a] = fmaf(dp[s], ws, pq[a]);
                pk[a] = fmaf(ab, ws, pk[a]);
                pc[s] = fmaf(both, f, pc[s]);
#pragma unroll
                for (int j = s + 1; j <= a; ++j) pg[j] = fmaf(both, ws, pg[j]);
            }
        }
        // the gate: own terms, summed over the tokens at and after each, and the pair terms.  (Rows
        // less columns of all pairs, summed over the tokens at and after, is the same sum but
        // leaves a strongly decaying token's to the rounding of its neighbours'.)
        const f32x4_t own_t = fma4(qq, x.F * dQh, khat * kdk);
        f32x4_t suf = own_t;
        suf[2] += suf[3];
        suf[1] += suf[2];
        suf[0] += suf[1];
        {
            const float t4 = suf[0], s4 = __shfl_xor(t4, 16);  // the sibling block's sum
            const float t8 = t4 + s4, s8 = __shfl_xor(t8, 32);
            suf += ((g & 1) ? 0.f : s4) + ((g & 2) ? 0.f : s8);
        }
        suf += pg;
        const f32x4_t dQ = fma4(x.F, dQh, fma4(dg, kk, pq));
        const f32x4_t dK = fma4(x.F, kdk, fma4(dg, qq, pk + pc));
        {
            const unsigned nb = static_cast<unsigned>(((clen_of(m) - 1) * tstride + 16) * GE);
            const size_t r0 = row0_of(m, 16 * w);
            const __amdgpu_buffer_rsrc_t rq = make_rsrc(static_cast<unsigned char*>(gq) + r0 * GE, nb);
#pragma unroll
            for (int e = 0; e < 4; ++e) put<GE>(dQ[e], rq, static_cast<unsigned>((4 * g + e) * tstride + r));
            *reinterpret_cast<f32x4_t*>(pk_ws + part_of(m)) = dK;
            if constexpr (CHAN) *reinterpret_cast<f32x4_t*>(pg_ws + part_of(m)) = suf;
        }
        if constexpr (!CHAN) {
#pragma unroll
            for (int e = 0; e < 4; ++e) suf[e] = row16_sum(suf[e]);
            if (r == 0) st4(smem + G::OFF_GG + (m * NW + w) * 64 + 16 * g, suf);
        }
        if (w == 0) {
            // dbeta_t = W_t . V_t - K^_t . (W S^T)_t + sum_s dA_ts A'_ts, t = r
            float s = fmaf(dar[0], at[0], fmaf(dar[1], at[1], fmaf(dar[2], at[2], dar[3] * at[3])));
            s += __shfl_xor(s, 16);
            s += __shfl_xor(s, 32);
            float wx = 0.f;
#pragma unroll
            for (int ww = 0; ww < NW; ++ww)
                wx += reinterpret_cast<const float*>(smem + G::OFF_DB + ((m & 1) * NW + ww) * 64)[r];
            if (g == 0 && r < clen_of(m)) gbeta[(tok0 + m * kC16 + r) * H + h] = wx + s;
        }
        own = next;
    }

    // ================ backwards ================
    // (the last two chunks are still in their buffers; this wave's own stores of the scratch
    // are read back below, after the wait)
    f32x4_t Gt[NT];
#pragma unroll
    for (int i = 0; i < NT; ++i) Gt[i] = gather(g_hist, i);
    wait_vm_n<0>();
    own = load_own(nm - 1, false);
    for (int m = nm - 1; m >= 0; --m) {
        const unsigned char* b = buf(m);
        Own next = own;
        if (m > 0) next = load_own(m - 1, false);
        // S^T at the chunk's start
        if (m + 1 == nm) {
        } else if (m == 0) {
#pragma unroll
            for (int i = 0; i < NT; ++i) St[i] = gather(s_hist, i);
        } else if (m == span_len / 2) {
#pragma unroll
            for (int i = 0; i < NT; ++i) St[i] = ld4(mid + 1024 * i);
        } else {
            const __amdgpu_buffer_rsrc_t rs = start_of(m);
#pragma unroll
            for (int i = 0; i < NT; ++i)
                St[i] = __builtin_bit_cast(f32x4_t, __builtin_amdgcn_raw_buffer_load_b128(rs, 16 * lane, 1024 * i, 0));
        }
        // U G^T
        f32x4_t ka[2] = {kZero4, kZero4};
        {
            f32x4_t ur[NT];
            ur[0] = ix.row(b + G::B_U, 0);
            ur[1] = ix.row(b + G::B_U, 1);
            fence();
#pragma unroll
            for (int i = 0; i < NT; ++i) {
                if (i + 2 < NT) ur[i + 2] = ix.row(b + G::B_U, i + 2);
#pragma unroll
                for (int e = 0; e < 4; ++e) ka[e & 1] = mfma4(ur[i][e], Gt[i][e], ka[e & 1]);
                fence();
            }
        }
        const Dec x = decays(own.lg);
        const f32x4_t khat = own.k * x.F, qhat = own.q * x.F;
        f32x4_t sg = kZero4;  // <S, G> of row 16 w + r, S from the chunk's start and G from its end
        // G^T = gC G^T + dO^T Q^ - W^T diag(beta) K^
        {
            constexpr int NP = NT > 4 ? 2 : 1;
            const f32x4_t nk = -(own.b4 * khat);
            float dc[2][NP][4], wc[2][NP][4];
            auto rd = [&](int i) __attribute__((always_inline)) {
#pragma unroll
                for (int e = 0; e < 4; ++e)
#pragma unroll
                    for (int p = 0; p < NP; ++p) {
                        dc[i & 1][p][e] = ix.col(b + G::B_O, e, i + 4 * p);
                        wc[i & 1][p][e] = ix.col(b + G::B_W, e, i + 4 * p);
                    }
            };
            rd(0);
#pragma unroll
            for (int i = 0; i < NT; ++i) {
                sg = fma4(St[i], Gt[i], sg);
                Gt[i] = Gt[i] * x.gc;
            }
            fence();
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                if (i + 1 < 4) rd(i + 1);
#pragma unroll
                for (int e = 0; e < 4; ++e)
#pragma unroll
                    for (int p = 0; p < NP; ++p) {
                        Gt[i + 4 * p] = mfma4(dc[i & 1][p][e], qhat[e], Gt[i + 4 * p]);
                        Gt[i + 4 * p] = mfma4(wc[i & 1][p][e], nk[e], Gt[i + 4 * p]);
                    }
                fence();
            }
        }
        const f32x4_t dKb = x.E * (ka[0] + ka[1]);  // dL/dK- scaled: dK's part
        const f32x4_t ct = own.k * dKb;             // K- . dL/dK- per token
        const f32x4_t dK = own.x + dKb;
        // dg: gC <S, G> plus the sums over the tokens before each
        f32x4_t pre;
        pre[0] = 0.f;
        pre[1] = ct[0];
        pre[2] = pre[1] + ct[1];
        pre[3] = pre[2] + ct[2];
        {
            const float t4 = pre[3] + ct[3], s4 = __shfl_xor(t4, 16);
            const float t8 = t4 + s4, s8 = __shfl_xor(t8, 32);
            pre += x.gc * col_total(sg) + (((g & 1) ? s4 : 0.f) + ((g & 2) ? s8 : 0.f));
        }
        {
            const unsigned nel = static_cast<unsigned>((clen_of(m) - 1) * tstride + 16);
            const size_t r0 = row0_of(m, 16 * w);
            const __amdgpu_buffer_rsrc_t rk = make_rsrc(static_cast<unsigned char*>(gk) + r0 * GE, nel * GE);
            const __amdgpu_buffer_rsrc_t rgg = make_rsrc(CHAN ? gg + r0 : gg, CHAN ? nel * 4 : 0u);
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                const unsigned el = static_cast<unsigned>((4 * g + e) * tstride + r);
                put<GE>(dK[e], rk, el);
                if constexpr (CHAN) put<4>(own.y[e] + pre[e], rgg, el);
            }
        }
        if constexpr (!CHAN) {
#pragma unroll
            for (int e = 0; e < 4; ++e) pre[e] = row16_sum(pre[e]);
            unsigned char* p = smem + G::OFF_GG + (m * NW + w) * 64 + 16 * g;
            if (r == 0) st4(p, ld4(p) + pre);
        }
        // chunk m - 1's copies have landed (they are older than this chunk's four gk stores)
        if (m >= 1) {
            wait_vm_n<4>();
            lds_barrier();
            if (m >= 2) issue(m - 2);
            own = next;
        }
    }
    if constexpr (!CHAN) {
        lds_barrier();
        for (int z = tid; z < nm * kC16; z += NW * 64) {
            const int m = z >> 4, t = z & 15;
            float s = 0.f;
#pragma unroll
            for (int ww = 0; ww < NW; ++ww)
                s += reinterpret_cast<const float*>(smem + G::OFF_GG + (m * NW + ww) * 64)[t];
            if (t < clen_of(m)) gg[(tok0 + z) * H + h] = s;
        }
    }
}

// Chunks per span: a power of two up to kSpan, halved while the span kernel would leave CUs
// without a workgroup (a span is one workgroup's sequence of 2 x span_len chunk steps; the
// histories it reads grow as it shrinks, a quarter of the other traffic at 2).
int span_len_for(long n_pairs, int T) {
    const long n_ch = (T + kC16 - 1) / kC16;
    int s = kSpan;
    while (s > 2 && n_pairs * ((n_ch + s - 1) / s) < 256) s /= 2;
    return s;
}

struct DecBwdWs {
    size_t kh, kb, qh, rec, s_hist, g_hist, w, u, s_ch, bytes;
};
DecBwdWs dec_bwd_ws(long n_pairs, int T, int D) {
    const size_t n_ch = static_cast<size_t>((T + kC16 - 1) / kC16), sl = span_len_for(n_pairs, T);
    const size_t n_span = (n_ch + sl - 1) / sl;
    const size_t np = static_cast<size_t>(n_pairs), tile = np * n_ch * kC16 * D * 4;
    const size_t rec = np * n_ch * (D == 128 ? DecRec<128>::FLOATS : DecRec<64>::FLOATS) * 4;
    auto al = [](size_t x) { return (x + 255) & ~static_cast<size_t>(255); };
    DecBwdWs w;
    w.kh = 0;
    w.kb = al(w.kh + tile);
    w.qh = al(w.kb + tile);
    w.rec = al(w.qh + tile);
    w.s_hist = al(w.rec + rec);
    w.g_hist = al(w.s_hist + np * n_span * D * D * 4);
    w.w = al(w.g_hist + np * n_span * D * D * 4);
    w.u = al(w.w + tile);
    w.s_ch = al(w.u + tile);
    w.bytes = w.s_ch + np * n_span * kept_starts(static_cast<int>(sl)) * D * D * 4;
    return w;
}

// forward workspace: K^, K-, Q^ tiles and the records
struct DecFwdWs {
    size_t kh, kb, qh, rec, bytes;
};
DecFwdWs dec_fwd_ws(long n_pairs, int T, int D) {
    const size_t n = static_cast<size_t>(n_pairs) * ((T + kC16 - 1) / kC16), tile = n * kC16 * D * 4;
    DecFwdWs w;
    w.kh = 0;
    w.kb = w.kh + tile;
    w.qh = w.kb + tile;
    w.rec = w.qh + tile;
    w.bytes = w.rec + n * (D == 128 ? DecRec<128>::FFLOATS : DecRec<64>::FFLOATS) * 4;
    return w;
}

template <int D, int DV, bool OB>
hipError_t launch_fwd_t(const DecayFwdArgs& a, hipStream_t st) {
    const int n_ch = (a.T + kC16 - 1) / kC16, n_pairs = a.B * a.H;
    const DecFwdWs o = dec_fwd_ws(n_pairs, a.T, D);
    unsigned char* base = static_cast<unsigned char*>(a.workspace);
    auto at = [&](size_t off) { return reinterpret_cast<float*>(base + off); };
    const long n_items = static_cast<long>(n_pairs) * n_ch;
    const dim3 pg(static_cast<unsigned>((n_items + 3) / 4));
    if (a.per_channel)
        hipLaunchKernelGGL((dec_prep_kernel<D, float, true, true>), pg, dim3(256), 0, st, a.q, a.k, a.beta, a.g, a.T, a.H,
                           n_ch, n_items, at(o.kh), at(o.kb), at(o.qh), at(o.rec));
    else
        hipLaunchKernelGGL((dec_prep_kernel<D, float, false, true>), pg, dim3(256), 0, st, a.q, a.k, a.beta, a.g, a.T, a.H,
                           n_ch, n_items, at(o.kh), at(o.kb), at(o.qh), at(o.rec));
    hipError_t e = hipGetLastError();
    if (e != hipSuccess) return e;
    using G = DfGeo<D, DV>;
    if ((e = set_lds<dec_fwd_kernel<D, DV, OB>>(G::BYTES)) != hipSuccess) return e;
    const int slots = (n_pairs + 7) / 8;
    hipLaunchKernelGGL((dec_fwd_kernel<D, DV, OB>), dim3(static_cast<unsigned>(slots * (D / DV) * 8)), dim3(G::WAVES * 64),
                       G::BYTES, st, a.v, a.s0, a.o, a.s_out, at(o.kh), at(o.kb), at(o.qh), at(o.rec), n_pairs, a.T, a.H,
                       n_ch);
    return hipGetLastError();
}

template <int D, typename InT, bool CHAN, int GE>
hipError_t launch_t(const BwdArgs& a, hipStream_t st) {
    const int n_ch = (a.T + kC16 - 1) / kC16, sl = span_len_for(a.n_pairs, a.T), n_span = (n_ch + sl - 1) / sl;
    const DecBwdWs o = dec_bwd_ws(a.n_pairs, a.T, D);
    unsigned char* base = reinterpret_cast<unsigned char*>(a.workspace);
    auto at = [&](size_t off) { return reinterpret_cast<float*>(base + off); };
    const InT *q = static_cast<const InT*>(a.q), *k = static_cast<const InT*>(a.k), *v = static_cast<const InT*>(a.v);
    hipError_t e;
    if ((e = set_lds<dec_span_kernel<D, InT, CHAN, GE>>(DcGeo<D>::BYTES)) != hipSuccess) return e;
    const long n_items = static_cast<long>(a.n_pairs) * n_ch;
    hipLaunchKernelGGL((dec_prep_kernel<D, InT, CHAN, false>), dim3(static_cast<unsigned>((n_items + 3) / 4)), dim3(256), 0, st,
                       q, k, a.beta, a.g, a.T, a.H, n_ch, n_items, at(o.kh), at(o.kb), at(o.qh), at(o.rec));
    if ((e = hipGetLastError()) != hipSuccess) return e;
    // 16 columns a workgroup while that leaves at most one per CU: a chain wave then has its
    // SIMD to itself (T 4096, D 128: 367 us against 489 at 32 pairs, 668 against 512 at 48)
    const long slots = (a.n_pairs + 7) / 8;
    auto sweep = [&](auto VV) {
        constexpr int DV = decltype(VV)::value;
        using G = DsGeo<D, DV>;
        const hipError_t err = set_lds<dec_sweep_kernel<D, DV, InT, GE>>(G::BYTES);
        if (err != hipSuccess) return err;
        hipLaunchKernelGGL((dec_sweep_kernel<D, DV, InT, GE>), dim3(static_cast<unsigned>(slots * (D / DV) * 8)),
                           dim3(G::WAVES * 64), G::BYTES, st, v, a.s0, a.go, a.gs, a.gv, a.gs0, at(o.kh), at(o.kb),
                           at(o.qh), at(o.rec), at(o.w), at(o.u), at(o.s_hist), at(o.g_hist), a.n_pairs, a.T, a.H, n_ch,
                           n_span, sl);
        return hipGetLastError();
    };
    e = a.n_pairs * (D / 16) <= 256 ? sweep(std::integral_constant<int, 16>{}) : sweep(std::integral_constant<int, 32>{});
    if (e != hipSuccess) return e;
    hipLaunchKernelGGL((dec_span_kernel<D, InT, CHAN, GE>), dim3(static_cast<unsigned>(a.n_pairs * n_span)), dim3(D * 4),
                       DcGeo<D>::BYTES, st, q, k, v, a.g, a.go, at(o.rec), at(o.s_hist), at(o.g_hist), at(o.w), at(o.u),
                       a.gq, a.gk, a.gbeta, a.gg, at(o.kh), at(o.kb), at(o.s_ch), a.T, a.H, n_ch, n_span, sl);
    return hipGetLastError();
}

}  // namespace

size_t decay_bwd_ws_bytes(long n_pairs, int T, int D) { return dec_bwd_ws(n_pairs, T, D).bytes; }
size_t decay_fwd_ws_bytes(long n_pairs, int T, int D) { return dec_fwd_ws(n_pairs, T, D).bytes; }

hipError_t launch_decay_fwd(const DecayFwdArgs& a, hipStream_t st) {
    const long n_pairs = static_cast<long>(a.B) * a.H;
    if (n_pairs == 0 || a.T == 0) return hipSuccess;
    if (!f32_bwd_supported(a.D, a.H)) return hipErrorInvalidValue;
    const int dv = chunked_f32_pick_tile(a.D, n_pairs, a.dv_tile);
    auto go = [&](auto DD, auto VV) {
        constexpr int D = decltype(DD)::value, DV = decltype(VV)::value;
        return a.out_bf16 ? launch_fwd_t<D, DV, true>(a, st) : launch_fwd_t<D, DV, false>(a, st);
    };
    using I = std::integral_constant<int, 128>;
    using J = std::integral_constant<int, 64>;
    using W = std::integral_constant<int, 32>;
    using N = std::integral_constant<int, 16>;
    if (a.D == 128) return dv == 16 ? go(I{}, N{}) : go(I{}, W{});
    return dv == 16 ? go(J{}, N{}) : go(J{}, W{});
}

hipError_t launch_decay_bwd(const BwdArgs& a, hipStream_t st) {
    if (a.n_pairs == 0 || a.T == 0) return hipSuccess;
    if (!f32_bwd_supported(a.D, a.H)) return hipErrorInvalidValue;
    if (a.gqk_bf16 != a.gv_bf16 || (a.gv_bf16 && !a.in_bf16)) return hipErrorInvalidValue;
    auto go = [&](auto DD) {
        constexpr int D = decltype(DD)::value;
        if (a.gv_bf16)
            return a.per_channel ? launch_t<D, uint16_t, true, 2>(a, st) : launch_t<D, uint16_t, false, 2>(a, st);
        if (a.per_channel)
            return a.in_bf16 ? launch_t<D, uint16_t, true, 4>(a, st) : launch_t<D, float, true, 4>(a, st);
        return a.in_bf16 ? launch_t<D, uint16_t, false, 4>(a, st) : launch_t<D, float, false, 4>(a, st);
    };
    return a.D == 128 ? go(std::integral_constant<int, 128>{}) : go(std::integral_constant<int, 64>{});
}

}  // namespace pm
