// delta_chunked_f32.hip — K7: the chunked forward for fp32 q/k/v on fp32 MFMA
// (v_mfma_f32_16x16x4f32), D in {64, 128}, in chunks of C = 16 tokens.
//
// The reference's recurrence (kernels/__init__.py:357-376 per token, :421-458 over
// the sequence) in the WY/UT chunk form, per chunk with start state S:
//   A = strict_lower(diag(beta) K K^T)     T = (I + A)^-1     T'' = -T diag(beta)
//   X = K S - V     U = T'' X  (= T diag(beta) (V - K S))
//   O = Q S + lower_incl_diag(Q K^T) U     S <- S + K^T U
// every product on fp32 MFMA with fp32 accumulation: fp32 arithmetic throughout.
//
// MFMA layout (lane l = 16 g + r): A operand A[r][g], B operand B[g][r], accumulator
// register v = D[4 g + v][r].  Each product's contraction index is mapped so that an
// operand which is itself a product comes straight from accumulator registers:
//   * over d (X = K S, Y = Q S): step (m, v) covers d = 16 m + 4 g + v, so register v
//     of S's accumulator tile m (rows 16 m ..) is the B operand, and lane (g, r) reads
//     K[r][16 m + 4 g .. + 3] as one float4 for the four steps of tile m;
//   * over tokens (U = T'' X, S += K^T U, O += P U): step v covers token 4 g + v, so
//     register v of X's or U's accumulator is the B operand, and the A operand M[r][4 g
//     + v] is register v of the accumulator of M^T.
//
// K7p (prep, one wave per (sequence, head, chunk), all chunks at once): G = K K^T from K
// rows read straight into operand registers, N = -A and N^T from G (which is symmetric),
// and T = (I - N)^-1 from the inverses of its diagonal blocks of 2, 4 and 8 (inv_lower16), as
// products of accumulators with transposed accumulators.  It writes (T'')^T as
// accumulator registers, 1 KiB per chunk: the A operand of U = T'' X, lane-linear.
//
// K7 (recurrence): one workgroup per (sequence, head, d_v tile of DV columns).  Per 16 columns,
// two chain waves hold every other 16-row tile of S each (and half of every product over or
// onto d: X = K S in two halves, exchanged through LDS and added by both, S += K^T U on the
// own rows), 36 products a chunk at D = 128; an output wave forms Y = Q S one chunk behind and
// O = Y + P U two behind.  One wave builds P^T = K Q^T for all and issues every HBM -> LDS
// copy (buffer_load ... lds) two chunks ahead.  One LDS-only barrier per chunk.
// The chain bounds it: with one wave per 16 columns (68 products, the output wave as many with
// P^T) 32 pairs of T 1024 took 113 us at D = 128 and 76 at D = 64, now 72 and 51; 128 pairs of
// D = 128, where the MFMA pipes of every CU are shared, 208, now 195.  At D = 64 and 32 columns
// (128 pairs on) one wave holds 16 columns alone: its 36 products are few enough, and the
// exchange and two waves more cost what the halves save (128 pairs 73 us, with two chain waves
// 75; 200 pairs 113 and 116).  There the output waves share P^T and the copies.
#include <type_traits>

#include "pm_cdna4.h"
#include "pm_f32mfma.h"
#include "pm_internal.h"

namespace pm {
namespace {

constexpr int kBwdRec = kF32BwdRec;  // floats per chunk of the backward's record: T, K K^T, beta, P
// workspace floats per chunk: (T'')^T, then (normalised mode) the 16 keys' 1 / max(||k||, 1e-6)
template <bool NORM>
constexpr int ws_floats() { return NORM ? 256 + 16 : 256; }


// Workspace slots (16-token chunks), as the split form's: fixed length, row = pair, slot
// = c; varlen, row = h and slot = floor(tok0 / 16) + seq + c (consecutive sequences never
// share a slot).
__host__ __device__ inline int f32_n_slot(bool varlen, int T, int n_seq) {
    return varlen ? (T + kC16 - 1) / kC16 + n_seq : (T + kC16 - 1) / kC16;
}


// ---------------------------------------------------------------- K7p
template <int D, bool NORM, bool BWD = false>
__global__ __launch_bounds__(256) void delta_f32_prep_kernel(const float* __restrict__ k,
                                                             const float* __restrict__ beta,
                                                             const int32_t* __restrict__ cu_seqlens,
                                                             int n_seq, int T, int H, int n_slot, long n_items,
                                                             float* __restrict__ ws, float* __restrict__ ws_b = nullptr,
                                                             const float* __restrict__ q = nullptr) {
    constexpr int NJ = D / 16;
    const int lane = threadIdx.x & 63;
    const long item = static_cast<long>(blockIdx.x) * 4 + (threadIdx.x >> 6);
    if (item >= n_items) return;
    const int row = static_cast<int>(item / n_slot), slot = static_cast<int>(item % n_slot);
    int seq, h, c, len;
    long tok0;
    if (cu_seqlens) {
        h = row;
        // the sequence whose slot range starts at or before `slot`: the largest s with
        // floor(cu[s] / 16) + s <= slot (non-decreasing in s)
        int lo = 0, hi = n_seq - 1;
        while (lo < hi) {
            const int mid = (lo + hi + 1) >> 1;
            const int a = min(max(cu_seqlens[mid], 0), T);
            if (a / kC16 + mid <= slot) lo = mid; else hi = mid - 1;
        }
        seq = lo;
        const int a = min(max(cu_seqlens[seq], 0), T);
        const int z = min(max(cu_seqlens[seq + 1], a), T);
        tok0 = a;
        len = z - a;
        c = slot - (a / kC16 + seq);
        if (c < 0 || c * kC16 >= len) return;
    } else {
        seq = row / H;
        h = row % H;
        tok0 = static_cast<long>(seq) * T;
        len = T;
        c = slot;
    }
    const int r = lane & 15, g = lane >> 4;
    const int base = c * kC16, clen = min(kC16, len - base);
    const size_t tstride = static_cast<size_t>(H) * D;
    const size_t row0 = static_cast<size_t>(tok0 + base) * tstride + static_cast<size_t>(h) * D;
    const unsigned nb = static_cast<unsigned>(((clen - 1) * tstride + D) * 4);
    const __amdgpu_buffer_rsrc_t rk = make_rsrc(k + row0, nb);
    f32x4_t kf[NJ];
#pragma unroll
    for (int j = 0; j < NJ; ++j) {
        const unsigned vo = static_cast<unsigned>((r * tstride + 16 * j + 4 * g) * 4);
        kf[j] = __builtin_bit_cast(f32x4_t, __builtin_amdgcn_raw_buffer_load_b128(rk, vo, 0, 0));
    }
    // beta of this lane's column token r (bc) and of its accumulator rows 4 g + v (bt); in the
    // normalised mode beta = 1 and sk / s4 are the keys' 1 / max(||k||, 1e-6) instead
    float bc = 1.f, sk = 1.f;
    f32x4_t bt = {1.f, 1.f, 1.f, 1.f}, s4 = {1.f, 1.f, 1.f, 1.f};
    if constexpr (NORM) {
        float ss = 0.f;
#pragma unroll
        for (int j = 0; j < NJ; ++j)
#pragma unroll
            for (int v = 0; v < 4; ++v) ss = fmaf(kf[j][v], kf[j][v], ss);
        ss += __shfl_xor(ss, 16);  // row r's four slices (every lane of the row gets equal bits)
        ss += __shfl_xor(ss, 32);
        sk = 1.f / fmaxf(sqrtf(ss), 1e-6f);
#pragma unroll
        for (int v = 0; v < 4; ++v) s4[v] = __shfl(sk, 4 * g + v);
    } else {
        const __amdgpu_buffer_rsrc_t rb =
            make_rsrc(beta + (tok0 + base) * H + h, static_cast<unsigned>(((clen - 1) * H + 1) * 4));
        bc = __uint_as_float(__builtin_amdgcn_raw_buffer_load_b32(rb, static_cast<unsigned>(r * H * 4), 0, 0));
#pragma unroll
        for (int v = 0; v < 4; ++v)
            bt[v] = __uint_as_float(
                __builtin_amdgcn_raw_buffer_load_b32(rb, static_cast<unsigned>((4 * g + v) * H * 4), 0, 0));
    }

    // G = K K^T (one accumulator per step of a tile, summed at the end)
    f32x4_t ga[4] = {kZero4, kZero4, kZero4, kZero4};
#pragma unroll
    for (int j = 0; j < NJ; ++j)
#pragma unroll
        for (int v = 0; v < 4; ++v) ga[v] = mfma4(kf[j][v], kf[j][v], ga[v]);
    f32x4_t G = (ga[0] + ga[1]) + (ga[2] + ga[3]);
    if constexpr (NORM) G = G * s4 * sk;  // Gram matrix of the normalised keys
    // N[i][j] = -beta_i G[i][j] (i > j), N^T[i][j] = -beta_j G[i][j] (j > i); i = 4 g + v, j = r
    f32x4_t N, Nt, Tacc, Tt;
#pragma unroll
    for (int v = 0; v < 4; ++v) {
        const int i = 4 * g + v;
        N[v] = i > r ? -bt[v] * G[v] : 0.f;
        Nt[v] = r > i ? -bc * G[v] : 0.f;
    }
    inv_lower16<BWD>(N, Nt, r, g, Tacc, Tt);
    f32x4_t tw;
#pragma unroll
    for (int v = 0; v < 4; ++v) tw[v] = -bt[v] * Tt[v];  // (T'')^T[i][j] = -beta_i T[j][i]
    float* out = ws + (static_cast<size_t>(row) * n_slot + slot) * ws_floats<NORM>();
    *reinterpret_cast<f32x4_t*>(out + lane * 4) = tw;
    if constexpr (BWD) {
        // the backward's record: T (accumulator registers: T[4 g + v][r]), the Gram matrix
        // K K^T (symmetric, so its registers are also those of its transpose), beta and P
        float* ob = ws_b + (static_cast<size_t>(row) * n_slot + slot) * kBwdRec;
        *reinterpret_cast<f32x4_t*>(ob + lane * 4) = Tacc;
        *reinterpret_cast<f32x4_t*>(ob + 256 + lane * 4) = G;
        if (g == 0) ob[512 + r] = bc;
        // P = lower_incl(Q K^T): P[4 g + v][r] = q_{4 g + v} . k_r, kept for r <= 4 g + v
        const __amdgpu_buffer_rsrc_t rq = make_rsrc(q + row0, nb);
        f32x4_t pa[4] = {kZero4, kZero4, kZero4, kZero4};
#pragma unroll
        for (int j = 0; j < NJ; ++j) {
            const unsigned vo = static_cast<unsigned>((r * tstride + 16 * j + 4 * g) * 4);
            const f32x4_t qf = __builtin_bit_cast(f32x4_t, __builtin_amdgcn_raw_buffer_load_b128(rq, vo, 0, 0));
#pragma unroll
            for (int v = 0; v < 4; ++v) pa[v] = mfma4(qf[v], kf[j][v], pa[v]);
        }
        f32x4_t P = (pa[0] + pa[1]) + (pa[2] + pa[3]);
#pragma unroll
        for (int v = 0; v < 4; ++v) P[v] = (r <= 4 * g + v) ? P[v] : 0.f;
        *reinterpret_cast<f32x4_t*>(ob + 528 + lane * 4) = P;
    }
    if constexpr (NORM) {
        if (g == 0) out[256 + r] = sk;
    }
}

// ---------------------------------------------------------------- K7
template <int D, int DV, bool NORM>
struct F32Geo {
    static constexpr int NCW = DV / 16;            // 16-column blocks: CW chain waves and an output wave each
    static constexpr int CW = D == 64 && DV == 32 ? 1 : 2;
    // chain 0 .., output CW NCW .., and at CW 2 a last one for P^T and the copies, which the two
    // output waves share at CW 1
    static constexpr int WAVES = (CW + 1) * NCW + CW - 1;
    static constexpr int NT = D / 16;              // S accumulator tiles per block
    static constexpr int NI = kC16 * D * 4 / 1024; // 1 KiB copies per K or Q tile
    static constexpr int NB = 4;        // rotating chunk buffers
    // one chunk buffer: K rows, Q rows, (T'')^T, V columns of each chain wave
    static constexpr int B_K = 0;
    static constexpr int B_Q = B_K + kC16 * D * 4;
    static constexpr int B_T = B_Q + kC16 * D * 4;
    static constexpr int B_V = B_T + (NORM ? 2048 : 1024);  // (T'')^T, then the keys' scales
    static constexpr int BUF = B_V + NCW * 1024;
    static constexpr int OFF_S = NB * BUF;                                  // 2 slots x NCW x NT KiB: S_i
    static constexpr int OFF_U = OFF_S + 2 * NCW * NT * 1024;  // 2 slots x NCW KiB: U_i
    static constexpr int PSLOT = NORM ? 1024 + 64 : 1024;                   // P^T, then the queries' scales
    static constexpr int OFF_P = OFF_U + 2 * NCW * 1024;       // 2 slots: P^T of a chunk
    static constexpr int OFF_X = OFF_P + 2 * PSLOT;            // 2 slots x NCW x 2 halves of X
    static constexpr int BYTES = OFF_X + 4096 * NCW;
    // the last wave issues every copy of a chunk: K and Q rows,
    // (T'')^T and the V columns of each chain wave
    static constexpr int NCP = 2 * NI + 1 + NCW + (NORM ? 1 : 0);
    static_assert(D == 64 || D == 128, "D");
    static_assert(DV == 16 || DV == 32, "DV");
    static_assert(BYTES <= 160 * 1024 && NCP <= 63, "LDS / vmcnt");
};

template <int D, int DV, bool OUT_BF16, bool NORM>
__global__ __launch_bounds__((F32Geo<D, DV, NORM>::WAVES * 64)) void delta_f32_kernel(
    const float* __restrict__ q, const float* __restrict__ k, const float* __restrict__ v,
    const float* __restrict__ s0, void* __restrict__ o_out, float* __restrict__ s_out,
    const int32_t* __restrict__ cu_seqlens, const float* __restrict__ ws, int n_pairs, int T, int H,
    int n_tiles, int n_slot) {
    extern __shared__ __attribute__((aligned(16))) unsigned char smem[];
    using G = F32Geo<D, DV, NORM>;
    constexpr int NCW = G::NCW, NT = G::NT;
    constexpr int NCP = G::NCP;  // copies per chunk
    constexpr int WSF = ws_floats<NORM>();
    const int w = static_cast<int>(uniform(static_cast<unsigned>(threadIdx.x >> 6)));

    // XCD-aware placement: the n_tiles workgroups of a pair share bid % 8
    const int bid = blockIdx.x;
    const int xcd = bid & 7, bslot = bid >> 3;
    const int tile = bslot % n_tiles;
    const int pair = (bslot / n_tiles) * 8 + xcd;
    if (pair >= n_pairs) return;
    const int seq = pair / H, h = pair % H;
    long tok0;
    int len;
    if (cu_seqlens) {
        const int a = min(max(cu_seqlens[seq], 0), T);
        const int z = min(max(cu_seqlens[seq + 1], a), T);
        tok0 = a;
        len = z - a;
    } else {
        tok0 = static_cast<long>(seq) * T;
        len = T;
    }
    const int col0 = tile * DV;
    const int n_chunks = (len + kC16 - 1) / kC16;
    const int ws_row = cu_seqlens ? h : pair;
    const int ws_slot0 = cu_seqlens ? static_cast<int>(tok0 / kC16) + seq : 0;

    const int lane = threadIdx.x & 63;
    const int r = lane & 15, g = lane >> 4;
    constexpr int CW = G::CW;
    const bool chain = w < CW * NCW, copy_wave = w == G::WAVES - 1;
    const int cw = chain ? w / CW : w - CW * NCW;  // the 16 columns this wave works on
    const size_t tstride = static_cast<size_t>(H) * D;
    const size_t sbase = static_cast<size_t>(pair) * D * D;

    auto buf = [&](int c) { return smem + (c % G::NB) * G::BUF; };
    auto sslot = [&](int c, int which) { return smem + G::OFF_S + ((c & 1) * NCW + which) * NT * 1024; };
    auto uslot = [&](int c, int which) { return smem + G::OFF_U + ((c & 1) * NCW + which) * 1024; };
    auto pslot = [&](int c) { return smem + G::OFF_P + (c & 1) * G::PSLOT; };

    // ---- HBM -> LDS copies of chunk c (c < n_chunks) ----
    auto chunk_rsrc = [&](const float* base, int c, int row_floats, int col) {
        const int clen = min(kC16, len - c * kC16);
        const size_t row0 = static_cast<size_t>(tok0 + c * kC16) * tstride + static_cast<size_t>(h) * D + col;
        return make_rsrc(base + row0, static_cast<unsigned>(((clen - 1) * tstride + row_floats) * 4));
    };
    auto copy_tile = [&](const float* base, int c, unsigned char* dst) __attribute__((always_inline)) {
        const __amdgpu_buffer_rsrc_t rs = chunk_rsrc(base, c, D, 0);
        unsigned char* d0 = uniform_ptr(dst);
#pragma unroll
        for (int i = 0; i < G::NI; ++i) {
            const int qc = 64 * i + lane;  // LDS chunk
            const int t = qc / (D / 4), p = (qc % (D / 4)) ^ t;
            dma16_asm(rs, d0 + 1024 * i, static_cast<unsigned>(t * tstride * 4 + 16 * p));
        }
    };
    auto copy_ws = [&](int c, unsigned char* dst) __attribute__((always_inline)) {
        const float* src = ws + (static_cast<size_t>(ws_row) * n_slot + ws_slot0 + c) * WSF;
        dma16_asm(make_rsrc(src, 1024), uniform_ptr(dst), static_cast<unsigned>(16 * lane));
        // the keys' scales: 64 bytes (lanes past them read zeros)
        if constexpr (NORM) dma16_asm(make_rsrc(src + 256, 64), uniform_ptr(dst + 1024), static_cast<unsigned>(16 * lane));
    };
    auto copy_v = [&](int c, int j, unsigned char* dst) __attribute__((always_inline)) {
        const __amdgpu_buffer_rsrc_t rs = chunk_rsrc(v, c, 16, col0 + 16 * j);
        const int t = lane >> 2, p = lane & 3;
        dma16_asm(rs, uniform_ptr(dst), static_cast<unsigned>(t * tstride * 4 + 16 * p));
    };
    // the copy wave's copies of chunk c
    auto copies = [&](int c) __attribute__((always_inline)) {
        unsigned char* b = buf(c);
        copy_tile(k, c, b + G::B_K);
        copy_tile(q, c, b + G::B_Q);
        copy_ws(c, b + G::B_T);
#pragma unroll
        for (int j = 0; j < NCW; ++j) copy_v(c, j, b + G::B_V + 1024 * j);
    };
    // P^T of chunk c (registers: q_r . k_{4 g + e}) into its slot, kept for i <= j (lower_incl P);
    // normalised mode: the queries' scales 1 / max(||q||, 1e-6) beside it (qss: this lane's
    // part of ||q_r||^2; a row's four slices are lanes r, r + 16, r + 32, r + 48)
    auto store_p = [&](int c, f32x4_t pq, float qss) __attribute__((always_inline)) {
        f32x4_t pt;
#pragma unroll
        for (int e = 0; e < 4; ++e) pt[e] = (4 * g + e <= r) ? pq[e] : 0.f;
        st4(pslot(c) + 16 * lane, pt);
        if constexpr (NORM) {
            float ss = qss;
            ss += __shfl_xor(ss, 16);
            ss += __shfl_xor(ss, 32);
            if (g == 0) reinterpret_cast<float*>(pslot(c) + 1024)[r] = 1.f / fmaxf(sqrtf(ss), 1e-6f);
        }
    };
    // O = Y + P U of chunk c, stored: lane (g, r) holds O[4 g + e][16 cw + r]; rows past the end
    // are dropped by the range-checked stores
    auto store_o = [&](int c, f32x4_t y) __attribute__((always_inline)) {
        constexpr int ES = OUT_BF16 ? 2 : 4;
        const f32x4_t pt = ld4(pslot(c) + 16 * lane);
        const f32x4_t u = ld4(uslot(c, cw) + 16 * lane);
        f32x4_t O = mm16(pt, u, y);
        if constexpr (NORM) O = O * ld4(pslot(c) + 1024 + 16 * g);  // rows scaled by the queries' scales
        const int clen = min(kC16, len - c * kC16);
        const size_t rowe = static_cast<size_t>(tok0 + c * kC16) * tstride + static_cast<size_t>(h) * D + col0 + 16 * cw;
        const __amdgpu_buffer_rsrc_t ro = make_rsrc(static_cast<unsigned char*>(o_out) + rowe * ES,
                                                    static_cast<unsigned>(((clen - 1) * tstride + 16) * ES));
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            const unsigned off = static_cast<unsigned>(((4 * g + e) * tstride + r) * ES);
            if constexpr (OUT_BF16)
                __builtin_amdgcn_raw_buffer_store_b16(f32_to_bf16(O[e]), ro, off, 0, 0);
            else
                __builtin_amdgcn_raw_buffer_store_b32(__float_as_uint(O[e]), ro, off, 0, 0);
        }
    };

    // Y = Q S of chunk c (returned) and P^T of it (stored), either or both: a tile's operands are
    // read two tiles ahead of its products, accumulator e takes the steps (m, e)
    auto products = [&](int c, auto DO_Y, auto DO_P) __attribute__((always_inline)) {
        constexpr bool doy = decltype(DO_Y)::value, dop = decltype(DO_P)::value;
        const unsigned char* b = buf(c);
        const unsigned char* ss = sslot(c, doy ? cw : 0);
        f32x4_t ya[4] = {kZero4, kZero4, kZero4, kZero4}, pa[4] = {kZero4, kZero4, kZero4, kZero4}, qv[NT], kp[NT], sc[NT];
        float qss = 0.f;  // normalised mode: this lane's part of ||q_r||^2
        auto rd = [&](int m) __attribute__((always_inline)) {
            qv[m] = ld4(b + G::B_Q + 16 * f32_chunk<D>(r, 4 * m + g));
            if constexpr (doy) sc[m] = ld4(ss + 1024 * m + 16 * lane);
            if constexpr (dop) kp[m] = ld4(b + G::B_K + 16 * f32_chunk<D>(r, 4 * m + g));
        };
        rd(0);
        rd(1);
        fence();
#pragma unroll
        for (int m = 0; m < NT; ++m) {
            if (m + 2 < NT) rd(m + 2);
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                if constexpr (doy) ya[e] = mfma4(qv[m][e], sc[m][e], ya[e]);
                if constexpr (dop) pa[e] = mfma4(kp[m][e], qv[m][e], pa[e]);
                if constexpr (dop && NORM) qss = fmaf(qv[m][e], qv[m][e], qss);
            }
            fence();
        }
        if constexpr (dop) store_p(c, (pa[0] + pa[1]) + (pa[2] + pa[3]), qss);
        return (ya[0] + ya[1]) + (ya[2] + ya[3]);
    };
    using Yes = std::true_type;
    using No = std::false_type;

    if (n_chunks > 0) {
        if (copy_wave) {
            copies(0);
            if (n_chunks > 1) copies(1);
            if (n_chunks > 1) wait_vm_n<NCP>();
            else wait_vm_n<0>();
        }
        lds_barrier();  // B0
    }

    if (chain) {
        // ============ chain wave hh of CW: S columns col0 + 16 cw + [0, 16), tiles m = hh + CW j ============
        // Phase p (up to barrier M_p) finishes chunk p - 1 (the other wave's half of X, U, S +=
        // K^T U) and forms this wave's half of X of chunk p: one barrier a chunk.  Every LDS
        // read is issued ahead of the products or behind one of them.  A wave alone forms U
        // right behind X and leaves the LDS accesses to the end, in U's latency (spread over the
        // products as the halves' they hold its one sequence up: 75 us for 73 at 128 pairs).
        constexpr int NH = NT / CW;
        const int hh = CW == 2 ? w & 1 : 0, ecol = col0 + 16 * cw + r;
        const TileIdx<D> ix(r, g, hh);
        f32x4_t S[NH];
#pragma unroll
        for (int j = 0; j < NH; ++j)
#pragma unroll
            for (int e = 0; e < 4; ++e)
                S[j][e] = s0 ? s0[sbase + static_cast<size_t>(16 * (hh + CW * j) + 4 * g + e) * D + ecol] : 0.f;
        __builtin_amdgcn_s_waitcnt(0x0F70);  // vmcnt(0), seen by the compiler: no wait for these in the loop
        __builtin_amdgcn_s_setprio(3);
        unsigned char* const xs = smem + G::OFF_X + 2048 * cw + 16 * lane;
        float kt[4][NH] = {};
        f32x4_t kf[NH], half = kZero4, tt = kZero4, vr = kZero4, skc = kZero4, U = kZero4;
        auto form_u = [&](f32x4_t X) __attribute__((always_inline)) {
            if constexpr (NORM) X = X * skc - vr;
            f32x4_t u = mm16(tt, X);
            if constexpr (NORM) u = u * skc;
            return u;
        };
        if (n_chunks > 0) {
            for (int p = 0; p <= n_chunks; ++p) {
                const bool run = p < n_chunks;
                const unsigned char* b = buf(run ? p : n_chunks - 1);  // (past the end: read, unused)
                f32x4_t other = kZero4;
                if constexpr (CW == 2) other = ld4(xs + ((p & 1) ^ 1) * 2048 * NCW + (hh ^ 1) * 1024);
                f32x4_t tn, vn, sn = kZero4;
#pragma unroll
                for (int j = 0; j < NH; ++j) kf[j] = CW == 2 ? ix.row2(b + G::B_K, j) : ix.row(b + G::B_K, j);
#pragma unroll
                for (int e = 0; e < 4; ++e)
                    vn[e] = reinterpret_cast<const float*>(b + G::B_V + 1024 * cw)[(4 * g + e) * 16 + r];
                tn = ld4(b + G::B_T + 16 * lane);
                if constexpr (NORM) sn = ld4(b + G::B_T + 1024 + 16 * g);
                fence();
                if (p > 0) {
                    if constexpr (CW == 2) U = form_u(half + other);
                    if (hh == 0) st4(uslot(p - 1, cw) + 16 * lane, U);
#pragma unroll
                    for (int e = 0; e < 4; ++e)
#pragma unroll
                        for (int j = 0; j < NH; ++j) S[j] = mfma4(kt[e][j], U[e], S[j]);
                }
                fence();
                if (run) {
                    tt = tn, vr = vn, skc = sn;
                    // (a wave alone sums its even and odd tiles apart: the bits of the two halves)
                    f32x4_t xa[4] = {kZero4, kZero4, kZero4, kZero4}, xb[4] = {kZero4, kZero4, kZero4, kZero4};
                    if constexpr (!NORM) {
                        if (hh == 0) xa[0] = -vr;
                    }
                    unsigned char* ss = sslot(p, cw) + 16 * lane;
#pragma unroll
                    for (int j = 0; j < NH; ++j)
#pragma unroll
                        for (int e = 0; e < 4; ++e) {
                            f32x4_t& x = CW == 1 && (j & 1) ? xb[e] : xa[e];
                            x = mfma4(kf[j][e], S[j][e], x);
                            if constexpr (CW == 2) {
                                kt[e][j] = ix.col2(b + G::B_K, e, j);
                                if (e == 3) st4(ss + 1024 * (hh + CW * j), S[j]);
                                fence();
                            }
                        }
                    half = (xa[0] + xa[1]) + (xa[2] + xa[3]);
                    if constexpr (CW == 2) st4(xs + (p & 1) * 2048 * NCW + hh * 1024, half);
                    else {
                        U = form_u(half + ((xb[0] + xb[1]) + (xb[2] + xb[3])));
#pragma unroll
                        for (int j = 0; j < NH; ++j) st4(ss + 1024 * j, S[j]);
#pragma unroll
                        for (int e = 0; e < 4; ++e)
#pragma unroll
                            for (int j = 0; j < NH; ++j) kt[e][j] = ix.col(b + G::B_K, e, j);
                    }
                }
                __builtin_amdgcn_s_waitcnt(0xC07F);  // lgkmcnt(0), seen by the compiler
                lds_barrier();                       // M_p
            }
        }
#pragma unroll
        for (int j = 0; j < NH; ++j)
#pragma unroll
            for (int e = 0; e < 4; ++e)
                s_out[sbase + static_cast<size_t>(16 * (hh + CW * j) + 4 * g + e) * D + ecol] = S[j][e];
    } else if (CW == 2 && n_chunks > 0 && copy_wave) {
        // ============ P and copy wave: phase p builds P^T of chunk p - 1, copies chunk p + 2 ============
        for (int p = 0; p <= n_chunks; ++p) {
            const bool cp = p + 2 < n_chunks;
            if (cp) copies(p + 2);
            if (p >= 1) products(p - 1, No{}, Yes{});
            // chunk p + 1 has landed; the copies of the one after may be in flight
            if (cp) wait_vm_n<NCP>();
            else wait_vm_n<0>();
            lds_barrier();
        }
    } else if (n_chunks > 0) {
        // ============ output wave: phase p finishes O of chunk p - 2 and forms Y = Q S of chunk p - 1 ============
        // (CW 1: the first one builds P^T of chunk p - 1 too, the last one issues the copies of p + 2)
        f32x4_t y = kZero4;
        for (int p = 0; p <= n_chunks + 1; ++p) {
            const bool cp = CW == 1 && copy_wave && p + 2 < n_chunks;
            if (cp) copies(p + 2);
            if (p >= 2) store_o(p - 2, y);
            if (p > n_chunks) break;
            if (p >= 1) y = CW == 1 && cw == 0 ? products(p - 1, Yes{}, Yes{}) : products(p - 1, Yes{}, No{});
            if (CW == 1 && copy_wave) {
                // as above, with the four stores of this phase behind this phase's copies
                if (cp && p >= 2) wait_vm_n<NCP + 4>();
                else if (cp) wait_vm_n<NCP>();
                else wait_vm_n<0>();
            }
            lds_barrier();
        }
    }
}

template <int D, int DV, bool OB, bool NORM>
hipError_t launch_f32_t(const ChunkedF32Args& a, float* ws, hipStream_t st) {
    using G = F32Geo<D, DV, NORM>;
    const bool varlen = a.cu_seqlens != nullptr;
    const int n_pairs = a.n_seq * a.H;
    const int n_slot = f32_n_slot(varlen, a.T, a.n_seq);
    const long n_items = static_cast<long>(varlen ? a.H : n_pairs) * n_slot;
    const float *q = a.q, *k = a.k, *v = a.v;
    if (n_items > 0) {
        hipLaunchKernelGGL((delta_f32_prep_kernel<D, NORM>), dim3(static_cast<unsigned>((n_items + 3) / 4)), dim3(256), 0,
                           st, k, a.beta, a.cu_seqlens, a.n_seq, a.T, a.H, n_slot, n_items, ws, nullptr, nullptr);
        hipError_t e = hipGetLastError();
        if (e != hipSuccess) return e;
    }
    auto kern = delta_f32_kernel<D, DV, OB, NORM>;
    hipError_t e = set_lds<delta_f32_kernel<D, DV, OB, NORM>>(G::BYTES);
    if (e != hipSuccess) return e;
    const int n_tiles = D / DV;
    const int slots = (n_pairs + 7) / 8;
    hipLaunchKernelGGL(kern, dim3(static_cast<unsigned>(slots * n_tiles * 8)), dim3(G::WAVES * 64), G::BYTES, st, q, k,
                       v, a.s0, a.o, a.s_out, a.cu_seqlens, ws, n_pairs, a.T, a.H, n_tiles, n_slot);
    return hipGetLastError();
}

template <int D, int DV, bool NORM>
hipError_t launch_f32_n(const ChunkedF32Args& a, float* ws, hipStream_t st) {
    return a.out_bf16 ? launch_f32_t<D, DV, true, NORM>(a, ws, st) : launch_f32_t<D, DV, false, NORM>(a, ws, st);
}
template <int D, int DV>
hipError_t launch_f32_dv(const ChunkedF32Args& a, float* ws, hipStream_t st) {
    return a.norm ? launch_f32_n<D, DV, true>(a, ws, st) : launch_f32_n<D, DV, false>(a, ws, st);
}

}  // namespace

size_t chunked_f32_ws_bytes(bool varlen, int n_seq, int T, int H, bool norm) {
    const long rows = varlen ? H : static_cast<long>(n_seq) * H;
    return static_cast<size_t>(rows) * f32_n_slot(varlen, T, n_seq) * (norm ? ws_floats<true>() : ws_floats<false>()) * 4;
}

// D = 128: 16 columns a workgroup while that leaves at most one per CU (LDS holds one), so that
// a chain wave has its SIMD to itself; a second round costs more than the wider form (T 1024:
// 32 pairs 72 against 95 us, 33 pairs 126 against 97, 63 pairs 128 against 100).  D = 64: two
// fit a CU, and the two forms are level from 65 to 128 pairs (71 us at 96, 74 against 73 at 128)
// before the narrow one needs a second round (200 pairs 135 against 113).
int chunked_f32_pick_tile(int D, long n_pairs, int requested) {
    if (requested == 16 || requested == 32) return requested;
    if (requested == 64) return 32;
    return n_pairs > (D == 128 ? 32 : 127) ? 32 : 16;
}

hipError_t launch_f32_bwd_prep(const float* q, const float* k, const float* beta, int n_pairs, int T, int H, int D,
                               float* ws_t2, float* ws_rec, hipStream_t st) {
    if (n_pairs == 0 || T == 0) return hipSuccess;
    const int n_slot = f32_n_slot(false, T, 0);
    const long n_items = static_cast<long>(n_pairs) * n_slot;
    const dim3 grid(static_cast<unsigned>((n_items + 3) / 4));
    if (D == 128)
        hipLaunchKernelGGL((delta_f32_prep_kernel<128, false, true>), grid, dim3(256), 0, st, k, beta, nullptr,
                           n_pairs / H, T, H, n_slot, n_items, ws_t2, ws_rec, q);
    else
        hipLaunchKernelGGL((delta_f32_prep_kernel<64, false, true>), grid, dim3(256), 0, st, k, beta, nullptr,
                           n_pairs / H, T, H, n_slot, n_items, ws_t2, ws_rec, q);
    return hipGetLastError();
}

hipError_t launch_chunked_f32(const ChunkedF32Args& a, void* ws, hipStream_t st) {
    if (a.n_seq == 0 || a.H == 0) return hipSuccess;
    float* w = static_cast<float*>(ws);
    const int dv = chunked_f32_pick_tile(a.D, static_cast<long>(a.n_seq) * a.H, a.dv_tile);
    if (a.D == 128) return dv == 16 ? launch_f32_dv<128, 16>(a, w, st) : launch_f32_dv<128, 32>(a, w, st);
    return dv == 16 ? launch_f32_dv<64, 16>(a, w, st) : launch_f32_dv<64, 32>(a, w, st);
}

}  // namespace pm
