// delta_chunked_f32_bwd.hip — K9: the chunked backward for fp32 q/k/v on fp32 MFMA
// (v_mfma_f32_16x16x4f32), D in {64, 128}, fixed-length batches.  Every product is
// fp32 x fp32 with fp32 accumulation.
//
// The reference's VJP (kernels/__init__.py:460-527, :529-588) in the WY/UT chunk form,
// chunks of C = 16 tokens.  Per chunk with start state S, T = (I + A)^-1,
// A = strict_lower(diag(beta) K K^T), T'' = -T diag(beta), X' = K S - V, U = T'' X',
// P = lower_incl(Q K^T), the forward is O = Q S + P U, S' = S + K^T U.  Given
// G = dL/dS' and dO:
//   W  = T^T (K G + P^T dO)                      (= dL/d(diag(beta)(V - K S)))
//   G <- G + Q^T dO - K^T diag(beta) W           (dL/dS)
//   dV = diag(beta) W
//   dP = lower_incl(dO U^T),  dA = -strict_lower(W U^T)
//   dQ = dO S^T + dP K
//   dK = U G^T + dP^T Q - diag(beta) W S^T + diag(beta) dA K + dA^T diag(beta) K
//   dbeta_t = -W_t . X'_t + sum_s dA_ts (k_t . k_s)
// Only G travels backwards from chunk to chunk, only S forwards.
//
// Launches (on the caller's stream):
//   K9p (delta_chunked_f32.hip): (T'')^T, T, K K^T, beta and P per chunk.
//   K9a + K9b (one launch, one workgroup per (b, h, 16 or 32 columns of d_v)): the S
//     recurrence forwards, storing U per token and S at the start of every span of kF32Span
//     chunks and at the end of the sequence; beside it the G recurrence backwards over all
//     chunks, storing W and dV per token, G at the end of every span, dS0.
//   K9c (span, one workgroup per (b, h, span)): backwards from the span's end state and end
//     gradient: S reconstructed as S - K^T U (no growth: U is the stored forward value),
//     G as in K9b, and dQ, dK, dbeta.
// Column ownership differs by phase: the recurrences over S and G keep their columns
// independent (a wave owns 16 columns of d_v), while the products contracting over d_v
// (dO S^T, U G^T, ...) need all of them: K9c keeps S^T and G^T by rows of d (a wave owns 16
// of them), and the two small products that contract over d_v inside a chunk (dO U^T,
// W U^T) are summed over the waves in LDS, in a fixed order.

#include <type_traits>

#include "pm_cdna4.h"
#include "pm_f32mfma.h"
#include "pm_internal.h"

namespace pm {
namespace {

// ---------------------------------------------------------------- K9a + K9b
// The two recurrences, over S forwards and over G backwards, in one workgroup per (b, h, DV
// columns of d_v).  They bound the launch: their chunks run in sequence.  Two waves share 16
// columns of a recurrence, each holding every other tile of 16 rows of d: the products that
// contract over d (X = K S, Y = K G) come in two halves, exchanged through LDS at a barrier in
// mid-chunk and added by both, and each wave updates its own rows.  Per chunk and wave 40
// products (S) and 54 (G, its Q^T dO among them) of 32 cycles; one wave per 16 columns needs
// 72, with Q^T dO's 32 in helper waves: 16 pairs of 2,003 tokens, D 128, 230 us, now 144 (2,400
// cycles a chunk, 1,728 of them the G chain's products).
// Waves: 2 DV/16 for S, as many for G (a SIMD holds one of each at DV = 32, one of either at
// 16), one that copies for S (and Q), one that copies for G and stores W and dV.  Each
// recurrence keeps three chunk buffers: a chain holds its chunk's operands in registers and
// reads the next chunk's, each behind a product (fenced: a product holds the MFMA pipe for 32
// cycles, in which its wave issues a read for free), so the copies run three chunks ahead into
// the buffer of the chunk in registers.
template <int D, int DV>
struct SwGeo {
    static constexpr int NC = DV / 16, NT = D / 16, NH = NT / 2, NI = kC16 * D * 4 / 1024, TILE = kC16 * D * 4;
    static constexpr int NB = 3, WAVES = 4 * NC + 2;
    // state half: K rows, T''^T, V columns
    static constexpr int H_K = 0, H_T = TILE, H_V = H_T + 1024, HBUF = H_V + NC * 1024;
    // gradient half: K and Q rows, dO columns, T, P, beta (64 bytes; the copy fills 1 KiB)
    static constexpr int S_K = 0, S_Q = TILE, S_O = 2 * TILE, S_T = S_O + NC * 1024, S_P = S_T + 1024, S_B = S_P + 1024;
    static constexpr int SBUF = S_B + 1024;
    static constexpr int H_NCP = 2 * NI + 1 + NC, S_NCP = NI + 3 + NC;  // copies per chunk
    static constexpr int S_NST = 2 * NC;                                // W and dV stores per chunk
    static constexpr int OFF_S = NB * HBUF;
    static constexpr int OFF_X = OFF_S + NB * SBUF;      // half products: S, G x NC x 2 halves
    static constexpr int OFF_W = OFF_X + 4 * NC * 1024;  // 2 slots x NC: W, beta
    static constexpr int WSLOT = 1024 + 64;
    static constexpr int BYTES = OFF_W + 2 * NC * WSLOT;
    static_assert(BYTES <= 160 * 1024 && S_NCP + S_NST <= 63 && H_NCP <= 63, "LDS / vmcnt");
};

template <int D, int DV>
__global__ __launch_bounds__((SwGeo<D, DV>::WAVES * 64)) void f32_sweep_kernel(
    const float* __restrict__ q, const float* __restrict__ k, const float* __restrict__ v,
    const float* __restrict__ s0, const float* __restrict__ go, const float* __restrict__ gs, float* __restrict__ gv,
    float* __restrict__ gs0, const float* __restrict__ t2, const float* __restrict__ rec, float* __restrict__ w_out,
    float* __restrict__ s_hist, float* __restrict__ g_hist, float* __restrict__ u_out, int n_pairs, int T, int H,
    int n_ch, int n_span) {
    using G = SwGeo<D, DV>;
    constexpr int NC = G::NC, NT = G::NT, NH = G::NH, NI = G::NI, NB = G::NB, n_tiles = D / DV;
    extern __shared__ __attribute__((aligned(16))) unsigned char smem[];
    // XCD-aware placement: the n_tiles workgroups of a pair share bid % 8
    const int bid = blockIdx.x, xcd = bid & 7, bslot = bid >> 3;
    const int tile = bslot % n_tiles, pair = (bslot / n_tiles) * 8 + xcd;
    if (pair >= n_pairs) return;
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
    auto bytes_of = [=](int c, int cols) {  // from a column block's first row to its last row's end
        return static_cast<unsigned>(((min(kC16, T - c * kC16) - 1) * tstride + cols) * 4);
    };
    // 16 token rows of a tensor as a swizzled tile (zeros past the end)
    auto copy_tile = [=](const float* base, int c, unsigned char* dst) __attribute__((always_inline)) {
        const __amdgpu_buffer_rsrc_t rs = make_rsrc(base + row0_of(c, 0), bytes_of(c, D));
        unsigned char* d0 = uniform_ptr(dst);
#pragma unroll
        for (int i = 0; i < NI; ++i) {
            const int qc = 64 * i + lane, t = qc / (D / 4), p = (qc % (D / 4)) ^ t;
            dma16_asm(rs, d0 + 1024 * i, static_cast<unsigned>(t * tstride * 4 + 16 * p));
        }
    };
    // 16 columns of 16 token rows, as [16][16] (a null tensor reads zeros: a zero-length range)
    auto copy_cols = [=](const float* base, int c, int j, unsigned char* dst) __attribute__((always_inline)) {
        dma16_asm(make_rsrc(base ? base + row0_of(c, col0 + 16 * j) : base, base ? bytes_of(c, 16) : 0u),
                  uniform_ptr(dst + 1024 * j), static_cast<unsigned>((lane >> 2) * tstride * 4 + 16 * (lane & 3)));
    };
    auto copy_1k = [=](const float* src, unsigned bytes, unsigned char* dst) __attribute__((always_inline)) {
        dma16_asm(make_rsrc(src, bytes), uniform_ptr(dst), static_cast<unsigned>(16 * lane));
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
        // S or G (its rows of this wave), lane order, where a span starts or ends
        auto keep = [&](float* hist, int per_pair, int index) __attribute__((always_inline)) {
            float* hp = hist + ((static_cast<size_t>(pair) * per_pair + index) * NT + col0 / 16 + cw) * NT * 256;
#pragma unroll
            for (int j = 0; j < NH; ++j) *reinterpret_cast<f32x4_t*>(hp + (hh + 2 * j) * 256 + 4 * lane) = M[j];
        };
        // this wave's operand over d (rows) and onto d (columns)
        f32x4_t kf[NH];
        float kt[4][NH];
        auto rd_kt = [&](const unsigned char* b, int e, int j) __attribute__((always_inline)) { kt[e][j] = ix.col2(b, e, j); };
        if (n_ch > 0) lds_barrier();  // B0
        if (state) {
            f32x4_t vr, tt;
            auto rd_v = [&](const unsigned char* b, int e) __attribute__((always_inline)) {
                vr[e] = reinterpret_cast<const float*>(b + G::H_V + 1024 * cw)[(4 * g + e) * 16 + r];
            };
            if (n_ch > 0) {
                const unsigned char* b = hbuf(0);
#pragma unroll
                for (int j = 0; j < NH; ++j) kf[j] = ix.row2(b + G::H_K, j);
#pragma unroll
                for (int e = 0; e < 4; ++e) {
                    rd_v(b, e);
#pragma unroll
                    for (int j = 0; j < NH; ++j) rd_kt(b + G::H_K, e, j);
                }
                tt = ld4(b + G::H_T + 16 * lane);
                __builtin_amdgcn_s_waitcnt(0xC07F);
                lds_barrier();  // B1: chunk 0's buffer may be refilled
            }
            for (int i = 0; i < n_ch; ++i) {
                const unsigned char* bn = hbuf(min(i + 1, n_ch - 1));  // (the last chunk reads itself again, unused)
                if (i % kF32Span == 0) keep(s_hist, n_span + 1, i / kF32Span);
                // X = K S - V, this wave's half
                f32x4_t xa[4] = {kZero4, kZero4, kZero4, kZero4};
                if (hh == 0) xa[0] = -vr;
                fence();
#pragma unroll
                for (int j = 0; j < NH; ++j)
#pragma unroll
                    for (int e = 0; e < 4; ++e) {
                        xa[e] = mfma4(kf[j][e], M[j][e], xa[e]);
                        if (e == 1 && j > 0) kf[j - 1] = ix.row2(bn + G::H_K, j - 1);
                        if (j < 2 && (e == 2 || e == 3)) rd_v(bn, 2 * j + e - 2);
                        fence();
                    }
                kf[NH - 1] = ix.row2(bn + G::H_K, NH - 1);
                const f32x4_t p = (xa[0] + xa[1]) + (xa[2] + xa[3]);
                st4(xs + 1024 * hh, p);
                lds_barrier();  // mid-chunk: the halves are in LDS
                const f32x4_t X = p + ld4(xs + 1024 * (hh ^ 1));
                const f32x4_t tn = ld4(bn + G::H_T + 16 * lane);
                const f32x4_t U = mm16(tt, X);
                // S += K^T U
                fence();
#pragma unroll
                for (int e = 0; e < 4; ++e)
#pragma unroll
                    for (int j = 0; j < NH; ++j) {
                        M[j] = mfma4(kt[e][j], U[e], M[j]);
                        if (e > 0) rd_kt(bn + G::H_K, e - 1, j);
                        if (e == 3) rd_kt(bn + G::H_K, 3, j);
                        fence();
                    }
                // U's rows (U^T = X^T T''^T): lane (g, r) holds U[r][col0 + 16 cw + 4 g ..] (rows past
                // the end dropped by the range)
                if (hh == 0)
                    __builtin_amdgcn_raw_buffer_store_b128(
                        __builtin_bit_cast(u32x4_t, mm16(X, tt)),
                        make_rsrc(u_out + row0_of(i, col0 + 16 * cw), bytes_of(i, 16)),
                        static_cast<unsigned>((r * tstride + 4 * g) * 4), 0, 0);
                tt = tn;
                __builtin_amdgcn_s_waitcnt(0xC07F);  // lgkmcnt(0), seen by the compiler
                lds_barrier();                       // end of the chunk
            }
            keep(s_hist, n_span + 1, n_span);  // the state at the end closes the last span
        } else {
            f32x4_t dOc, ta, b4;
            float qt[4][NH];  // Q^T operand
            f32x2_t pp;       // P^T's operand for tokens e = 2 hh, 2 hh + 1: each half adds its part of P^T dO
            auto rd_do = [&](const unsigned char* b, int e) __attribute__((always_inline)) {
                return reinterpret_cast<const float*>(b + G::S_O + 1024 * cw)[(4 * g + e) * 16 + r];
            };
            auto rd_q = [&](const unsigned char* b, int e, int j) __attribute__((always_inline)) {
                qt[e][j] = ix.col2(b + G::S_Q, e, j);
            };
            auto rd_p = [&](const unsigned char* b) __attribute__((always_inline)) {
                return *reinterpret_cast<const f32x2_t*>(b + G::S_P + 16 * lane + 8 * hh);
            };
            if (n_ch > 0) {
                const unsigned char* b = sbuf(n_ch - 1);
#pragma unroll
                for (int j = 0; j < NH; ++j) kf[j] = ix.row2(b + G::S_K, j);
#pragma unroll
                for (int e = 0; e < 4; ++e) {
                    dOc[e] = rd_do(b, e);
#pragma unroll
                    for (int j = 0; j < NH; ++j) {
                        rd_kt(b + G::S_K, e, j);
                        rd_q(b, e, j);
                    }
                }
                ta = ld4(b + G::S_T + 16 * lane);
                pp = rd_p(b);
                b4 = ld4(b + G::S_B + 16 * g);
                __builtin_amdgcn_s_waitcnt(0xC07F);
                lds_barrier();  // B1
            }
            for (int c = n_ch - 1; c >= 0; --c) {
                const unsigned char* bn = sbuf(max(c - 1, 0));
                f32x4_t dOn, tn, bn4;
                f32x2_t pn;
                if (c == n_ch - 1 || c % kF32Span == kF32Span - 1) keep(g_hist, n_span, c / kF32Span);
                // dU = K G + P^T dO, this wave's half
                f32x4_t ya[4] = {kZero4, kZero4, kZero4, kZero4};
                ya[0] = mfma4(pp[0], hh ? dOc[2] : dOc[0], kZero4);
                ya[1] = mfma4(pp[1], hh ? dOc[3] : dOc[1], kZero4);
                fence();
#pragma unroll
                for (int j = 0; j < NH; ++j)
#pragma unroll
                    for (int e = 0; e < 4; ++e) {
                        ya[e] = mfma4(kf[j][e], M[j][e], ya[e]);
                        if (e == 1 && j > 0) kf[j - 1] = ix.row2(bn + G::S_K, j - 1);
                        if (j < 2 && (e == 2 || e == 3)) dOn[2 * j + e - 2] = rd_do(bn, 2 * j + e - 2);
                        fence();
                    }
                kf[NH - 1] = ix.row2(bn + G::S_K, NH - 1);
                fence();
                // G += Q^T dO: half of it ahead of the exchange, the rest in its latency
                auto q_prod = [&](int e, int j) __attribute__((always_inline)) {
                    M[j] = mfma4(qt[e][j], dOc[e], M[j]);
                    fence();
                };
#pragma unroll
                for (int j = 0; j < NH; ++j) {
                    q_prod(0, j);
                    if (j == 0) tn = ld4(bn + G::S_T + 16 * lane);
                    if (j == 1) pn = rd_p(bn);
                }
                const f32x4_t p = (ya[0] + ya[1]) + (ya[2] + ya[3]);
                st4(xs + 1024 * hh, p);
                fence();
#pragma unroll
                for (int j = 0; j < NH; ++j) {
                    q_prod(1, j);
                    rd_q(bn, 0, j);
                }
                lds_barrier();  // mid-chunk
                const f32x4_t po = ld4(xs + 1024 * (hh ^ 1));
                fence();
#pragma unroll
                for (int j = 0; j < NH; ++j) {
                    q_prod(2, j);
                    rd_q(bn, 1, j);
                }
                // W = T^T dU
                const f32x4_t dU = p + po;
                f32x4_t w0 = mfma4(ta[0], dU[0], kZero4), w1 = mfma4(ta[1], dU[1], kZero4);
                __asm__ volatile("" : "+v"(w0), "+v"(w1));  // (issued here, not where the sum needs them)
                fence();
                q_prod(3, 0);
                w0 = mfma4(ta[2], dU[2], w0), w1 = mfma4(ta[3], dU[3], w1);
                __asm__ volatile("" : "+v"(w0), "+v"(w1));
                fence();
#pragma unroll
                for (int j = 1; j < NH; ++j) {
                    q_prod(3, j);
                    rd_q(bn, 2, j - 1);
                    if (j == 1) bn4 = ld4(bn + G::S_B + 16 * g);
                }
                rd_q(bn, 2, NH - 1);
                const f32x4_t W = w0 + w1;
                const f32x4_t nbW = -(W * b4);
                // G -= K^T diag(beta) W
                fence();
#pragma unroll
                for (int e = 0; e < 4; ++e)
#pragma unroll
                    for (int j = 0; j < NH; ++j) {
                        M[j] = mfma4(kt[e][j], nbW[e], M[j]);
                        if (e == 0) rd_q(bn, 3, j);
                        if (e > 0) rd_kt(bn + G::S_K, e - 1, j);
                        if (e == 3) rd_kt(bn + G::S_K, 3, j);
                        if (e == 0 && j == 0 && hh == 0) st4(wslot(c, cw) + 16 * lane, W);
                        if (e == 0 && j == 1 && hh == 0 && r == 0) st4(wslot(c, cw) + 1024 + 16 * g, b4);
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
    } else if (n_ch == 0) {
        return;
    } else if (w == 4 * NC) {
        // ============ the state half's copies (and Q), three chunks ahead, half of them in each half of a chunk ============
        auto copies_a = [=](int c) __attribute__((always_inline)) { copy_tile(k, c, hbuf(c) + G::H_K); };
        auto copies_b = [=](int c) __attribute__((always_inline)) {
            unsigned char* b = hbuf(c);
            copy_tile(q, n_ch - 1 - c, sbuf(n_ch - 1 - c) + G::S_Q);
            copy_1k(t2 + (item0 + c) * 256, 1024, b + G::H_T);
#pragma unroll
            for (int j = 0; j < NC; ++j) copy_cols(v, c, j, b + G::H_V);
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
        auto copies_a = [=](int c) __attribute__((always_inline)) { copy_tile(k, c, sbuf(c) + G::S_K); };
        auto copies_b = [=](int c) __attribute__((always_inline)) {
            unsigned char* b = sbuf(c);
            const float* rc = rec + (item0 + c) * kF32BwdRec;
#pragma unroll
            for (int j = 0; j < NC; ++j) copy_cols(go, c, j, b + G::S_O);
            copy_1k(rc, 1024, b + G::S_T);
            copy_1k(rc + 528, 1024, b + G::S_P);
            copy_1k(rc + 512, 64, b + G::S_B);
        };
        auto copies = [=](int c) __attribute__((always_inline)) {
            copies_a(c);
            copies_b(c);
        };
        auto store = [=](int cs) __attribute__((always_inline)) {
            const int t = lane >> 2, p = lane & 3;
            const unsigned off = static_cast<unsigned>((t * tstride + 4 * p) * 4);
#pragma unroll
            for (int j = 0; j < NC; ++j) {
                const float* ws = reinterpret_cast<const float*>(wslot(cs, j));
                const float bt = ws[256 + t];
                f32x4_t x;
#pragma unroll
                for (int e = 0; e < 4; ++e) x[e] = ws[4 * (16 * (t >> 2) + 4 * p + e) + (t & 3)];
                const size_t row0 = row0_of(cs, col0 + 16 * j);
                const unsigned nb = bytes_of(cs, 16);
                __builtin_amdgcn_raw_buffer_store_b128(__builtin_bit_cast(u32x4_t, x), make_rsrc(w_out + row0, nb), off,
                                                       0, 0);
                __builtin_amdgcn_raw_buffer_store_b128(__builtin_bit_cast(u32x4_t, x * bt), make_rsrc(gv + row0, nb), off,
                                                       0, 0);
            }
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

// ---------------------------------------------------------------- K9c
template <int D>
struct SpGeo {
    static constexpr int NW = D / 16;              // waves; wave w owns rows 16 w .. of d
    static constexpr int NT = D / 16;
    static constexpr int NI = kC16 * D * 4 / 1024; // 1 KiB copies per row tile
    static constexpr int TILE = kC16 * D * 4;
    static constexpr int B_K = 0;                  // row tiles (f32_chunk): K, Q, dO, W, U, V
    static constexpr int B_Q = B_K + TILE;
    static constexpr int B_O = B_Q + TILE;
    static constexpr int B_W = B_O + TILE;
    static constexpr int B_U = B_W + TILE;
    static constexpr int B_V = B_U + TILE;
    static constexpr int B_G = B_V + TILE;         // K K^T, accumulator registers
    static constexpr int B_B = B_G + 1024;         // beta (64 bytes; the copy fills 1 KiB)
    static constexpr int BUF = B_B + 1024;
    static constexpr int OFF_DB = 2 * BUF;                     // dbeta parts: 2 slots x NW x 16
    static constexpr int OFF_PP = OFF_DB + 2 * NW * 64;        // per wave: dO U^T, W U^T parts [t][s]
    static constexpr int OFF_TR = OFF_PP + NW * 2048;          // totals dP, dA as rows [t][s]
    static constexpr int OFF_TC = OFF_TR + 2048;               // totals dP, dA as columns [s][t], stride 20
    static constexpr int BYTES = OFF_TC + 2 * 16 * 20 * 4;
    static constexpr int NC = 6 * NI + 2;                      // copies per chunk
    static_assert(BYTES <= 160 * 1024, "LDS");
};

// s_waitcnt vmcnt(n) for a wave-uniform n in [0, 20] (more waits for 20)
__device__ __forceinline__ void wait_vm_upto(int n) {
    switch (n) {
        case 0: wait_vm_n<0>(); break;
        case 1: wait_vm_n<1>(); break;
        case 2: wait_vm_n<2>(); break;
        case 3: wait_vm_n<3>(); break;
        case 4: wait_vm_n<4>(); break;
        case 5: wait_vm_n<5>(); break;
        case 6: wait_vm_n<6>(); break;
        case 7: wait_vm_n<7>(); break;
        case 8: wait_vm_n<8>(); break;
        case 9: wait_vm_n<9>(); break;
        case 10: wait_vm_n<10>(); break;
        case 11: wait_vm_n<11>(); break;
        case 12: wait_vm_n<12>(); break;
        case 13: wait_vm_n<13>(); break;
        case 14: wait_vm_n<14>(); break;
        case 15: wait_vm_n<15>(); break;
        case 16: wait_vm_n<16>(); break;
        case 17: wait_vm_n<17>(); break;
        case 18: wait_vm_n<18>(); break;
        case 19: wait_vm_n<19>(); break;
        default: wait_vm_n<20>(); break;
    }
}

// One workgroup of NW waves per (b, h, span of kF32Span chunks), the span's chunks
// backwards from its end state and end gradient (S^T and G^T by rows of d: wave w holds
// S^T[16 i + 4 g + v][16 w + r] in tile i, G^T likewise, gathered from the histories).
// Per chunk, from the chunk's K, Q, dO, W, U (the forward's, stored by the history pass)
// and V rows:
//   S^T -= U^T K (S^T at the chunk's start: U is the forward's own value, so the
//   subtraction does not amplify error); dQ = dO S^T; WS = W S^T; dK = U G^T -
//   diag(beta) WS; G^T += dO^T Q - (diag(beta) W)^T K; this wave's parts of dO U^T and
//   W U^T, and of -W.X' = -sum_d K WS + W.V (X' = K S - V);
// a barrier; each wave sums 1/NW of the parts' entries (in a fixed order) and masks them
// into dP and dA; a barrier; dQ += dP K, dK += dP^T Q + diag(beta) dA K + dA^T diag(beta)
// K; wave 0 forms dbeta.  Staging: two chunk buffers; chunk m - 2's copies are issued
// once every wave has read chunk m (after the first barrier) and waited for before the
// second barrier of chunk m - 1.
template <int D>
__global__ __launch_bounds__(D * 4) void f32_bwd_span_kernel(
    const float* __restrict__ q, const float* __restrict__ k, const float* __restrict__ v,
    const float* __restrict__ go, const float* __restrict__ rec, const float* __restrict__ s_hist,
    const float* __restrict__ g_hist, const float* __restrict__ w_in, const float* __restrict__ u_in,
    float* __restrict__ gq, float* __restrict__ gk, float* __restrict__ gbeta, int T, int H, int n_ch, int n_span) {
    using G = SpGeo<D>;
    constexpr int NW = G::NW, NT = G::NT;
    extern __shared__ __attribute__((aligned(16))) unsigned char smem[];

    const int pair = blockIdx.x / n_span, span = blockIdx.x % n_span;
    const int seq = pair / H, h = pair % H;
    const long tok0 = static_cast<long>(seq) * T;
    const int c0 = span * kF32Span;
    const int nm = min(kF32Span, n_ch - c0);  // chunks in this span
    const int tid = threadIdx.x, lane = tid & 63;
    const int w = static_cast<int>(uniform(static_cast<unsigned>(tid >> 6)));
    const int r = lane & 15, g = lane >> 4;
    const size_t tstride = static_cast<size_t>(H) * D;
    const f32x4_t zero = {0.f, 0.f, 0.f, 0.f};

    auto buf = [=](int m) { return smem + (m & 1) * G::BUF; };
    auto col_read = [=](const unsigned char* tileb, int t, int d) {  // X[t][d] of a row tile
        return reinterpret_cast<const float*>(tileb)[4 * f32_chunk<D>(t, d >> 2) + (d & 3)];
    };
    auto row_read = [=](const unsigned char* tileb, int i) {  // X[r][16 i + 4 g ..]
        return ld4(tileb + 16 * f32_chunk<D>(r, 4 * i + g));
    };
    auto row0_of = [=](int m, int col) {
        return static_cast<size_t>(tok0 + (c0 + m) * kC16) * tstride + static_cast<size_t>(h) * D + col;
    };
    auto bytes_of = [=](int m, int row_floats) {
        const int clen = min(kC16, T - (c0 + m) * kC16);
        return static_cast<unsigned>(((clen - 1) * tstride + row_floats) * 4);
    };
    // copy number x of chunk m (one branch per source: a selected pointer would become a
    // table in scratch); wave w issues x = w, w + NW, ...
    auto copy_one = [=](int m, int x, unsigned char* b) __attribute__((always_inline)) {
        const size_t cslot = static_cast<size_t>(pair) * n_ch + c0 + m;
        if (x < 6 * G::NI) {
            const int which = x / G::NI, i = x % G::NI;
            const int qc = 64 * i + lane, t = qc / (D / 4), p = (qc % (D / 4)) ^ t;
            const unsigned vo = static_cast<unsigned>(t * tstride * 4 + 16 * p);
            const size_t r0 = row0_of(m, 0);
            const unsigned nb = bytes_of(m, D);
            if (which == 0) {
                dma16_asm(make_rsrc(k + r0, nb), uniform_ptr(b + G::B_K + 1024 * i), vo);
            } else if (which == 1) {
                dma16_asm(make_rsrc(q + r0, nb), uniform_ptr(b + G::B_Q + 1024 * i), vo);
            } else if (which == 2) {
                // a null dO reads zeros (a zero-length range)
                dma16_asm(make_rsrc(go ? go + r0 : go, go ? nb : 0u), uniform_ptr(b + G::B_O + 1024 * i), vo);
            } else if (which == 3) {
                dma16_asm(make_rsrc(w_in + r0, nb), uniform_ptr(b + G::B_W + 1024 * i), vo);
            } else if (which == 4) {
                dma16_asm(make_rsrc(u_in + r0, nb), uniform_ptr(b + G::B_U + 1024 * i), vo);
            } else {
                dma16_asm(make_rsrc(v + r0, nb), uniform_ptr(b + G::B_V + 1024 * i), vo);
            }
        } else if (x == 6 * G::NI) {
            dma16_asm(make_rsrc(rec + cslot * kF32BwdRec + 256, 1024), uniform_ptr(b + G::B_G),
                      static_cast<unsigned>(16 * lane));
        } else {
            dma16_asm(make_rsrc(rec + cslot * kF32BwdRec + 512, 64), uniform_ptr(b + G::B_B),
                      static_cast<unsigned>(16 * lane));
        }
    };
    auto issue = [=](int m) __attribute__((always_inline)) {
        if (m < 0) return;
        unsigned char* b = buf(m);
        for (int x = w; x < G::NC; x += NW) copy_one(m, x, b);
    };
    const int n_mine = (G::NC - w + NW - 1) / NW;  // copies this wave issues per chunk

    // ---- the span's end state and end gradient, by rows of d, gathered from the column-
    // block layout of the histories: S^T[16 i + 4 g + e][16 w + r] = S[16 w + r][16 i + 4 g + e]
    // is in column block i, tile w, lane 16 (r >> 2) + 4 g + e, register r & 3 ----
    f32x4_t St[NT], Gt[NT];
    {
        const float* sp = s_hist + (static_cast<size_t>(pair) * (n_span + 1) + span + 1) * D * D;
        const float* gp = g_hist + (static_cast<size_t>(pair) * n_span + span) * D * D;
#pragma unroll
        for (int i = 0; i < NT; ++i)
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                const size_t o = (static_cast<size_t>(i) * NT + w) * 256 + 4 * (16 * (r >> 2) + 4 * g + e) + (r & 3);
                St[i][e] = sp[o];
                Gt[i][e] = gp[o];
            }
    }
    issue(nm - 1);
    issue(nm - 2);
    wait_vm_n<0>();
    lds_barrier();

    for (int m = nm - 1; m >= 0; --m) {
        const unsigned char* b = buf(m);
        const int dbs = m & 1;  // the dbeta parts' slot
        // B operands for this wave's rows 16 w + r of d; beta; K K^T
        f32x4_t kc, qc, wj, vj;
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            kc[e] = col_read(b + G::B_K, 4 * g + e, 16 * w + r);
            qc[e] = col_read(b + G::B_Q, 4 * g + e, 16 * w + r);
            wj[e] = col_read(b + G::B_W, 4 * g + e, 16 * w + r);  // W, V at columns 16 w + r of d_v
            vj[e] = col_read(b + G::B_V, 4 * g + e, 16 * w + r);
        }
        const f32x4_t b4 = ld4(b + G::B_B + 16 * g);
        const float br = reinterpret_cast<const float*>(b + G::B_B)[r];
        const f32x4_t gram = ld4(b + G::B_G + 16 * lane);  // K K^T[4 g + v][r] = K K^T[r][4 g + v]
        fence();
        // S^T -= U^T K: S^T at the chunk's start
#pragma unroll
        for (int i = 0; i < NT; ++i) {
            float uc[4];
#pragma unroll
            for (int e = 0; e < 4; ++e) uc[e] = col_read(b + G::B_U, 4 * g + e, 16 * i + r);
#pragma unroll
            for (int e = 0; e < 4; ++e) St[i] = mfma4(uc[e], -kc[e], St[i]);
        }
        // dQ = dO S^T, WS = W S^T, U G^T, and this wave's parts of dO U^T, W U^T
        f32x4_t qa[2] = {zero, zero}, wa[2] = {zero, zero}, ka[2] = {zero, zero};
        f32x4_t pp = zero, pa = zero;
#pragma unroll
        for (int i = 0; i < NT; ++i) {
            const f32x4_t dor = row_read(b + G::B_O, i);
            const f32x4_t wrw = row_read(b + G::B_W, i);
            const f32x4_t ur = row_read(b + G::B_U, i);
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                qa[e & 1] = mfma4(dor[e], St[i][e], qa[e & 1]);
                wa[e & 1] = mfma4(wrw[e], St[i][e], wa[e & 1]);
                ka[e & 1] = mfma4(ur[e], Gt[i][e], ka[e & 1]);
            }
            if (i == w) {
#pragma unroll
                for (int e = 0; e < 4; ++e) {
                    pp = mfma4(ur[e], dor[e], pp);  // (U dO^T)[4 g + v][r] = (dO U^T)[r][4 g + v]
                    pa = mfma4(ur[e], wrw[e], pa);
                }
            }
        }
        const f32x4_t WS = wa[0] + wa[1];  // W S^T[4 g + v][16 w + r]
        f32x4_t dK = ka[0] + ka[1] - b4 * WS;
        // this wave's part of -W.X' per token 4 g + v: -sum over its d of K WS, plus W.V over
        // its 16 columns of d_v
        {
            f32x4_t x = wj * vj - kc * WS;
#pragma unroll
            for (int sh = 1; sh < 16; sh <<= 1)
#pragma unroll
                for (int e = 0; e < 4; ++e) x[e] += __shfl_xor(x[e], sh);
            if (r == 0) st4(smem + G::OFF_DB + (dbs * NW + w) * 64 + 16 * g, x);
        }
        unsigned char* part = smem + G::OFF_PP + w * 2048;
        // row t = r, entries s = 4 g .. 4 g + 3 of each [t][s] part (16 bytes)
        st4(part + 16 * (4 * r + g), pp);
        st4(part + 1024 + 16 * (4 * r + g), pa);
        // G^T += dO^T Q - (diag(beta) W)^T K (after its use above)
#pragma unroll
        for (int i = 0; i < NT; ++i) {
            float dc[4], wc[4];
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                dc[e] = col_read(b + G::B_O, 4 * g + e, 16 * i + r);
                wc[e] = -b4[e] * col_read(b + G::B_W, 4 * g + e, 16 * i + r);
            }
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                Gt[i] = mfma4(dc[e], qc[e], Gt[i]);
                Gt[i] = mfma4(wc[e], kc[e], Gt[i]);
            }
        }
        lds_barrier();  // Y: the parts are in LDS; every wave is done reading chunk m
        issue(m - 2);   // into chunk m's buffer
        for (int x = tid; x < 512; x += NW * 64) {
            const int mat = x >> 8, t = (x >> 4) & 15, s = x & 15;
            float sum = 0.f;
#pragma unroll
            for (int ww = 0; ww < NW; ++ww)
                sum += reinterpret_cast<const float*>(smem + G::OFF_PP + ww * 2048 + mat * 1024)[16 * t + s];
            const float val = mat == 0 ? (s <= t ? sum : 0.f) : (s < t ? -sum : 0.f);
            reinterpret_cast<float*>(smem + G::OFF_TR + mat * 1024)[16 * t + s] = val;
            reinterpret_cast<float*>(smem + G::OFF_TC + mat * 1280)[20 * s + t] = val;
        }
        // chunk m - 1's copies have landed (issued after the previous chunk's first barrier);
        // still in flight may be the previous chunk's stores and chunk m - 2's copies
        if (m >= 1) wait_vm_upto((m + 1 < nm ? 8 + (w == 0 ? 1 : 0) : 0) + (m >= 2 ? n_mine : 0));
        lds_barrier();  // Z: totals in LDS, chunk m - 1 in its buffer
        // dQ += dP K; dK += dP^T Q + diag(beta) dA K + dA^T diag(beta) K
        const f32x4_t dpr = ld4(smem + G::OFF_TR + 16 * (4 * r + g));            // dP[r][4 g ..]
        const f32x4_t dar = ld4(smem + G::OFF_TR + 1024 + 16 * (4 * r + g));     // dA[r][4 g ..]
        const f32x4_t dpc = ld4(smem + G::OFF_TC + 4 * (20 * r + 4 * g));        // dP[4 g ..][r]
        const f32x4_t dac = ld4(smem + G::OFF_TC + 1280 + 4 * (20 * r + 4 * g)); // dA[4 g ..][r]
        f32x4_t dQ = qa[0] + qa[1];
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            dQ = mfma4(dpr[e], kc[e], dQ);
            dK = mfma4(dpc[e], qc[e], dK);
            dK = mfma4(br * dar[e], kc[e], dK);
            dK = mfma4(dac[e] * b4[e], kc[e], dK);
        }
        // rows 4 g + v of dQ and dK, columns 16 w + r
        {
            const size_t row0 = row0_of(m, 16 * w);
            const unsigned nb = bytes_of(m, 16);
            const __amdgpu_buffer_rsrc_t rq = make_rsrc(gq + row0, nb), rk = make_rsrc(gk + row0, nb);
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                const unsigned off = static_cast<unsigned>(((4 * g + e) * tstride + r) * 4);
                __builtin_amdgcn_raw_buffer_store_b32(__float_as_uint(dQ[e]), rq, off, 0, 0);
                __builtin_amdgcn_raw_buffer_store_b32(__float_as_uint(dK[e]), rk, off, 0, 0);
            }
        }
        if (w == 0) {
            // dbeta_t = -W_t . X'_t + sum_s dA_ts (k_t . k_s), t = r
            float sdg = dar[0] * gram[0] + dar[1] * gram[1] + dar[2] * gram[2] + dar[3] * gram[3];
            sdg += __shfl_xor(sdg, 16);
            sdg += __shfl_xor(sdg, 32);
            float wx = 0.f;
#pragma unroll
            for (int ww = 0; ww < NW; ++ww)
                wx += reinterpret_cast<const float*>(smem + G::OFF_DB + (dbs * NW + ww) * 64)[r];
            const int clen = min(kC16, T - (c0 + m) * kC16);
            const __amdgpu_buffer_rsrc_t rb = make_rsrc(gbeta + (tok0 + (c0 + m) * kC16) * H + h,
                                                        static_cast<unsigned>(((clen - 1) * H + 1) * 4));
            // every lane stores (lanes r of each group write the same value), one store per wave
            __builtin_amdgcn_raw_buffer_store_b32(__float_as_uint(wx + sdg), rb, static_cast<unsigned>(r * H * 4), 0,
                                                  0);
        }
    }
}

template <int D>
hipError_t launch_d(const BwdArgs& a, hipStream_t st) {
    const int n_ch = (a.T + kC16 - 1) / kC16;
    const int n_span = (n_ch + kF32Span - 1) / kF32Span;
    const F32BwdWs ws = f32_bwd_ws(a.n_pairs, a.T, D);
    unsigned char* base = reinterpret_cast<unsigned char*>(a.workspace);
    float* t2 = reinterpret_cast<float*>(base + ws.t2);
    float* rec = reinterpret_cast<float*>(base + ws.rec);
    float* s_hist = reinterpret_cast<float*>(base + ws.s_hist);
    float* g_hist = reinterpret_cast<float*>(base + ws.g_hist);
    float* w_ws = reinterpret_cast<float*>(base + ws.w);
    float* u_ws = reinterpret_cast<float*>(base + ws.u);
    const float* q = static_cast<const float*>(a.q);
    const float* k = static_cast<const float*>(a.k);
    const float* v = static_cast<const float*>(a.v);
    hipError_t e;
    if ((e = set_lds<f32_bwd_span_kernel<D>>(SpGeo<D>::BYTES)) != hipSuccess) return e;
    if (n_ch > 0 && (e = launch_f32_bwd_prep(q, k, a.beta, a.n_pairs, a.T, a.H, D, t2, rec, st)) != hipSuccess) return e;
    // 16 columns a workgroup while that leaves at most one per CU: a chain wave then has its SIMD
    // to itself (the decayed rules' same sweep: 367 us against 489 at 32 pairs, 668 against 512 at 48)
    const long slots = (a.n_pairs + 7) / 8;
    auto sweep = [&](auto VV) {
        constexpr int DV = decltype(VV)::value;
        using G = SwGeo<D, DV>;
        const hipError_t err = set_lds<f32_sweep_kernel<D, DV>>(G::BYTES);
        if (err != hipSuccess) return err;
        hipLaunchKernelGGL((f32_sweep_kernel<D, DV>), dim3(static_cast<unsigned>(slots * (D / DV) * 8)),
                           dim3(G::WAVES * 64), G::BYTES, st, q, k, v, a.s0, a.go, a.gs, a.gv, a.gs0, t2, rec, w_ws,
                           s_hist, g_hist, u_ws, a.n_pairs, a.T, a.H, n_ch, n_span);
        return hipGetLastError();
    };
    e = a.n_pairs * (D / 16) <= 256 ? sweep(std::integral_constant<int, 16>{}) : sweep(std::integral_constant<int, 32>{});
    if (e != hipSuccess) return e;
    if (n_ch == 0) return hipSuccess;
    hipLaunchKernelGGL(f32_bwd_span_kernel<D>, dim3(static_cast<unsigned>(a.n_pairs * n_span)), dim3(D * 4),
                       SpGeo<D>::BYTES, st, q, k, v, a.go, rec, s_hist, g_hist, w_ws, u_ws, a.gq, a.gk, a.gbeta, a.T,
                       a.H, n_ch, n_span);
    return hipGetLastError();
}

}  // namespace

F32BwdWs f32_bwd_ws(long n_pairs, int T, int D) {
    const size_t n_ch = static_cast<size_t>((T + kC16 - 1) / kC16);
    const size_t n_span = (n_ch + kF32Span - 1) / kF32Span;
    const size_t np = static_cast<size_t>(n_pairs);
    auto al = [](size_t x) { return (x + 255) & ~static_cast<size_t>(255); };
    F32BwdWs w;
    w.t2 = 0;
    w.rec = al(w.t2 + np * n_ch * 256 * 4);
    w.s_hist = al(w.rec + np * n_ch * kF32BwdRec * 4);
    w.g_hist = al(w.s_hist + np * (n_span + 1) * D * D * 4);
    w.w = al(w.g_hist + np * n_span * D * D * 4);
    w.u = al(w.w + np * static_cast<size_t>(T) * D * 4);
    w.bytes = al(w.u + np * static_cast<size_t>(T) * D * 4);
    return w;
}

// 32-bit buffer offsets: a chunk of fp32 rows spans 16 token rows of H*D values.
bool f32_bwd_supported(int D, int H) { return (D == 64 || D == 128) && static_cast<long>(H) * D <= (1L << 24); }

hipError_t launch_bwd_chunked_f32(const BwdArgs& a, hipStream_t st) {
    if (a.n_pairs == 0) return hipSuccess;
    if (a.in_bf16 || !f32_bwd_supported(a.D, a.H)) return hipErrorInvalidValue;
    return a.D == 128 ? launch_d<128>(a, st) : launch_d<64>(a, st);
}

}  // namespace pm
