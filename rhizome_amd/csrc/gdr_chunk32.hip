// gdr_chunk32.hip -- fp32-input gated delta-rule prefill for gfx950 in chunks
// of 16 positions on fp32 MFMA, fp32 throughout.
//
// Per 16-token chunk with entering state S0 (rows of d_k key columns),
// D_rs = prod_{s < u <= r} alpha_u and gamma_r = prod_{u <= r} alpha_u:
//
//   A_rs = beta_r D_rs k_r.k_s  (s < r),   T = (I + A)^-1
//   P_rs = D_rs q_r.k_s         (s <= r)
//   R    = diag(beta) (V - diag(gamma) K S0^T),   U = T R
//   O    = diag(gamma) Q S0^T + P U
//   S'   = gamma_15 S0 + sum_r D_15,r u_r k_r^T
//
// which is the recurrence of crates/ops/src/delta.rs:94-127 applied to 16
// positions (u_r = beta_r (v_r - alpha_r S_{r-1} k_r)).  The decays are
// products of the alphas themselves, never differences of summed logarithms,
// so alpha = 0 forgets the past exactly and every factor is as accurate as
// the recurrence's.
//
// What bounds it: fp32 MFMA (64 flop per cycle and SIMD, 16x16x4 in 32
// cycles).  A chunk of c tokens costs a 32-row tile c/4 (c/16) ... per token:
// at c = 16 (K K^T, Q K^T: 64 MFMAs; K S0^T, Q S0^T, S': 64 each; T R, P U:
// 8 each) 272 MFMAs per 16 tokens, at c = 32 316 and at c = 64 412 for the
// same tokens, so the shortest MFMA-shaped chunk does least.  The 272 are
// split evenly over the four SIMDs of a CU (68 each, 2176 cycles per chunk):
// the state-dependent chain (K S0^T, T R, S') of 16 rows on one SIMD, their
// outputs (Q S0^T, P U) one chunk later on another, beside the chunk's K K^T
// (or Q K^T) one chunk earlier.
//
// One workgroup of 8 waves per (sequence, head, 32 rows of S), in lockstep:
// one barrier per chunk, every wave at its own stage of the pipeline:
//   period p: waves 4, 5 stage chunk p into LDS (and load chunk p + 2),
//             wave 6 forms T and wave 7 P of chunk p - 1,
//             waves 0, 1 run the state through chunk p - 2,
//             waves 2, 3 form the outputs of chunk p - 3.
//
// No operand is converted, transposed or shuffled on the way: the key
// columns that MFMA step j contracts, and the order in which a block's rows
// stand for key columns, are chosen so that every operand is either an
// accumulator as it stands or 16 consecutive bytes of an LDS row.
//
// Inputs outside the op's domain (delta.rs:17-20) -- alpha outside [0, 1],
// beta |k|^2 outside [0, 2], or values that are not finite, where a product
// with a masked zero would spread a NaN to earlier positions -- are noticed
// as they pass, and the workgroup then recomputes its rows with the
// token-sequential recurrence (staged_rows) in the same launch.

#include "gdr_device.hpp"
#include "gdr_internal.hpp"
#include "gdr_solve.hpp"
#include "gdr_staged.hpp"

namespace rhz {
namespace {

constexpr int kC = 16;    // tokens per chunk
constexpr int kRows = 32; // rows of S per workgroup (two scan waves of 16)
constexpr int kLdV = 36;  // fp32 row stride of the V tile (4 rows apart: 16 banks apart)
constexpr int kQSlots = 5;  // chunks of Q (and gamma) held: staged at period c, last read at c + 4
constexpr int kLdA = 20;  // fp32 row stride of A and D
constexpr float kKeyBetaMax = 2.0f;  // largest beta |k|^2 (the step is non-expansive up to 2)

struct Chunk32Params {
    SeqParams sp;
    int units, n_tiles;
};

// Key columns of the operands.  Lane (m, g) = (lane & 15, lane >> 4).
// Accumulator block (h, v), v < VW, of the state holds the rows of S in its
// columns, and its row 4 g + r stands for key column 16 VW h + VW (4 g + r) + v,
// so that lane (n, g) of the NB = NH VW blocks holds, of row n and for every h,
// the 4 VW consecutive key columns from 16 VW h + 4 VW g on: the slots of an
// operand read as VW 16-byte pieces of a K or Q row.
template <int DK>
struct Shape32 {
    static constexpr int VW = DK >= 64 ? 4 : 2;
    static constexpr int NH = DK / (16 * VW);
    static constexpr int NB = DK / 16;     // state blocks, and 16-byte pieces of an operand row per lane
    static constexpr int NL = DK / 32;     // 16-byte pieces of K (and Q) per loader thread and chunk
};

// K and Q tiles: 16 rows of DK floats; the 16-byte pieces of a row are
// permuted by an XOR with the row, so that the 16 rows of one piece, and the
// 16 pieces of one row, fall into different banks.
template <int DK>
__device__ __forceinline__ int kq_off(int row, int piece) {
    const int f = DK >= 64 ? row : row >> 1;
    return row * DK + ((piece ^ f) << 2);
}

template <int DK>
struct Smem32 {
    float k[4][kC * DK];  // [chunk & 3]
    float q[kQSlots][kC * DK];  // [chunk % kQSlots]
    float v[4][kC * kLdV];
    float gam[kQSlots][kC];  // gamma_r
    float beta[4][kC];
    float gdl[4][kC];        // D_15,r
    float bgl[4][kC];        // beta_r D_15,r
    float d[2][kC * kLdA];   // D, [chunk & 1]
    float a[kC * kLdA];      // A, wave 6 only
    float t[2][kC * kC];     // T below the diagonal, column s times beta_s
    float p[4][kC * kC];     // P
    float s0[2][2][Shape32<DK>::NB * 256];  // entering state of scan wave w: [chunk & 1][w]
    float u[2][2][256];                     // U of scan wave w
    int rerun;  // an input left the domain
};

template <int DK>
union KernelSmem32 {
    Smem32<DK> chunk;
    StageSmem<16, 8, 8> rerun;  // 128 key columns, 32 rows
};
static_assert(StageSmem<16, 8, 8>::RPB == kRows && StageShape<16, 8, 8>::THREADS == 512, "the rerun covers the tile");

__device__ __forceinline__ f32x4 lds4(const float* p) { return *reinterpret_cast<const f32x4*>(p); }
__device__ __forceinline__ void st4(float* p, f32x4 x) { *reinterpret_cast<f32x4*>(p) = x; }
__device__ __forceinline__ f32x4 mfma4(float a, float b, f32x4 c) {
    return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0);
}

// The end of a period: this wave's LDS accesses are done, then every wave's.
// Global loads and stores stay in flight across it.
__device__ __forceinline__ void period_end() {
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
}

// The operand pieces of lane (m, g): row m of a K or Q tile.
template <int DK>
__device__ __forceinline__ void load_operand(const float* tile, int m, int g, f32x4 (&x)[Shape32<DK>::NB]) {
    constexpr int VW = Shape32<DK>::VW;
#pragma unroll
    for (int h = 0; h < Shape32<DK>::NH; ++h)
#pragma unroll
        for (int i = 0; i < VW; ++i) x[h * VW + i] = lds4(&tile[kq_off<DK>(m, 4 * VW * h + VW * g + i)]);
}

// Sum over the key columns of X_m Y_n for operands x, y of load_operand's
// layout, in NA accumulators added pairwise at the end.  fp32 MFMA
// rounds after every product, so the error grows with the length of an
// accumulator's chain: Q K^T and Q S0^T, whose sums go into o as they are, take
// DK / 8 (chains of 8 products, as the recurrence's lanes), the others 4.
template <int DK, int NA>
struct Dots {
    f32x4 acc[NA];
    __device__ __forceinline__ void mma(const f32x4 (&x)[Shape32<DK>::NB], const f32x4 (&y)[Shape32<DK>::NB]) {
#pragma unroll
        for (int i = 0; i < NA; ++i) acc[i] = (f32x4){0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int i = 0; i < Shape32<DK>::NB; ++i)
#pragma unroll
            for (int e = 0; e < 4; ++e) acc[(4 * i + e) % NA] = mfma4(x[i][e], y[i][e], acc[(4 * i + e) % NA]);
    }
    __device__ __forceinline__ f32x4 sum() const {
        f32x4 s[NA];
#pragma unroll
        for (int i = 0; i < NA; ++i) s[i] = acc[i];
#pragma unroll
        for (int w = NA / 2; w >= 1; w /= 2)
#pragma unroll
            for (int i = 0; i < w; ++i) s[i] += s[i + w];
        return s[0];
    }
};

// The state's accumulators as operand pieces: piece VW h + i, element e is key
// column 16 VW h + 4 VW g + 4 i + e, i.e. block (h, v), row r with
// VW r + v = 4 i + e.
template <int DK>
__device__ __forceinline__ void state_operand(const f32x4 (&S)[Shape32<DK>::NB], f32x4 (&y)[Shape32<DK>::NB]) {
    constexpr int VW = Shape32<DK>::VW;
#pragma unroll
    for (int h = 0; h < Shape32<DK>::NH; ++h)
#pragma unroll
        for (int i = 0; i < VW; ++i)
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                const int j = 4 * i + e;
                y[h * VW + i][e] = S[h * VW + j % VW][j / VW];
            }
}

// Keeps NaN once x was infinite or NaN.
__device__ __forceinline__ void watch(float& w, float x) { w = fmaf(x, 0.f, w); }

template <int DK>
__device__ __forceinline__ void flag32(Smem32<DK>& sm, bool bad) {
    if (__builtin_amdgcn_ballot_w64(bad) != 0 && (threadIdx.x & 63) == 0) sm.rerun = 1;
}

struct Unit32 {
    int seq, h, i0, tb, te, nch;
};

// ------------------------------------------------------------ loader waves
template <int DK>
struct In32 {
    f32x4 k[Shape32<DK>::NL], q[Shape32<DK>::NL], v;
    float g, b;
};

// Chunk min(c, nch - 1) into registers (thread j of 128); rows past the
// sequence's end and columns past the row's repeat the last ones and are
// zeroed as they are staged.
template <int DK>
__device__ __forceinline__ void load32(const SeqParams& p, const Unit32& u, int c, int j, In32<DK>& r) {
    constexpr int PPR = DK / 4;
    c = min(c, u.nch - 1);
    const int t0 = u.tb + c * kC, last = u.te - t0 - 1;
    const size_t th = size_t(t0) * p.heads + u.h;
    const char* kb = reinterpret_cast<const char*>(static_cast<const float*>(p.k) + th * p.d_k);
    const char* qb = reinterpret_cast<const char*>(static_cast<const float*>(p.q) + th * p.d_k);
    const char* vb = reinterpret_cast<const char*>(static_cast<const float*>(p.v) + th * p.d_v + u.i0);
    const uint32_t H = p.heads;
#pragma unroll
    for (int i = 0; i < Shape32<DK>::NL; ++i) {
        const int f = j + 128 * i, row = min(f / PPR, last), col = min(4 * (f % PPR), p.d_k - 4);
        const uint32_t off = (uint32_t(row) * H * p.d_k + col) * 4u;
        r.k[i] = *reinterpret_cast<const f32x4*>(kb + off);
        r.q[i] = *reinterpret_cast<const f32x4*>(qb + off);
    }
    const int vcol = min(4 * (j & 7), p.d_v - 4 - u.i0);
    r.v = *reinterpret_cast<const f32x4*>(vb + (uint32_t(min(j >> 3, last)) * H * p.d_v + vcol) * 4u);
    const size_t gi = th + size_t(min(j & 15, last)) * H;
    r.g = p.gate[gi];
    r.b = p.beta[gi];
}

// A product carried as an unevaluated sum hi + lo.
struct TwoFloat {
    float hi = 1.f, lo = 0.f;
    __device__ __forceinline__ void mul(float x) {
        const float p = hi * x;
        lo = fmaf(lo, x, fmaf(hi, x, -p));
        hi = p;
    }
    __device__ __forceinline__ float value() const { return hi + lo; }
};

// Chunk c from registers into its LDS slot; wave 4's lanes 0..15 (GATES) also
// form the decays, lane r holding row r of D.
template <int DK, bool GATES>
__device__ __forceinline__ void stage32(const SeqParams& p, const Unit32& u, Smem32<DK>& sm, int c, int j,
                                        const In32<DK>& r, bool& bad) {
    constexpr int PPR = DK / 4;
    const int len = u.te - (u.tb + c * kC);
    const int slot = c & 3;
    const f32x4 z = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int i = 0; i < Shape32<DK>::NL; ++i) {
        const int f = j + 128 * i, row = f / PPR, piece = f % PPR;
        const bool ok = row < len && 4 * piece < p.d_k;
        st4(&sm.k[slot][kq_off<DK>(row, piece)], ok ? r.k[i] : z);
        st4(&sm.q[c % kQSlots][kq_off<DK>(row, piece)], ok ? r.q[i] : z);
    }
    const int vrow = j >> 3, vcol = 4 * (j & 7);
    st4(&sm.v[slot][vrow * kLdV + vcol], vrow < len && u.i0 + vcol < p.d_v ? r.v : z);
    if constexpr (GATES) {
        const int n = j & 15;
        const float alpha = n < len ? decay_factor(r.g, p.gate_is_alpha) : 1.f;
        bad |= !(alpha >= 0.f && alpha <= 1.f);
        // D_{n, s-1} = D_{n, s} alpha_s for s <= n, from the right (1 for s > n),
        // and D_15,n: products carried as two floats and rounded once (a chain
        // of 15 fp32 roundings would cost slowly decaying states more than
        // all their other roundings do; f64 multiplies take three times as long)
        const float beta = n < len ? r.b : 0.f;
        TwoFloat d, e;
        float row[kC];
        row[kC - 1] = 1.f;
#define RHZ_DECAY_STEP(s)                                  \
    {                                                      \
        const float as = dpp_mov<0x150 + s>(alpha);        \
        d.mul(s <= n ? as : 1.f);                          \
        e.mul(s > n ? as : 1.f);                           \
        row[s - 1] = d.value();                            \
    }
        RHZ_DECAY_STEP(15) RHZ_DECAY_STEP(14) RHZ_DECAY_STEP(13) RHZ_DECAY_STEP(12) RHZ_DECAY_STEP(11)
        RHZ_DECAY_STEP(10) RHZ_DECAY_STEP(9) RHZ_DECAY_STEP(8) RHZ_DECAY_STEP(7) RHZ_DECAY_STEP(6)
        RHZ_DECAY_STEP(5) RHZ_DECAY_STEP(4) RHZ_DECAY_STEP(3) RHZ_DECAY_STEP(2) RHZ_DECAY_STEP(1)
#undef RHZ_DECAY_STEP
        d.mul(dpp_mov<0x150>(alpha));
        if (j < kC) {
#pragma unroll
            for (int i = 0; i < 4; ++i)
                st4(&sm.d[c & 1][n * kLdA + 4 * i], (f32x4){row[4 * i], row[4 * i + 1], row[4 * i + 2], row[4 * i + 3]});
            sm.gam[c % kQSlots][n] = d.value();
            sm.gdl[slot][n] = e.value();
            e.mul(beta);
            sm.bgl[slot][n] = e.value();
            sm.beta[slot][n] = beta;
        }
    }
}

template <int DK, bool GATES>
__device__ __forceinline__ void loader32(const SeqParams& p, const Unit32& u, Smem32<DK>& sm, int j) {
    bool bad = false;
    if (u.nch > 0) {
        In32<DK> r0, r1;
        load32<DK>(p, u, 0, j, r0);
        load32<DK>(p, u, 1, j, r1);
        for (int c = 0; c < u.nch; c += 2) {
            stage32<DK, GATES>(p, u, sm, c, j, r0, bad);
            load32<DK>(p, u, c + 2, j, r0);
            period_end();
            if (c + 1 >= u.nch) break;
            stage32<DK, GATES>(p, u, sm, c + 1, j, r1, bad);
            load32<DK>(p, u, c + 3, j, r1);
            period_end();
        }
    }
    if constexpr (GATES) flag32(sm, bad);
    for (int i = 0; i < 5; ++i) period_end();
}

// ------------------------------------------------------------ T and P
// Wave 6: K K^T of chunk c on MFMA in period c + 1, beside the substitution
// of chunk c - 1 (a chain of VALU and LDS latencies).
template <int DK>
__device__ __forceinline__ void t_wave32(const Unit32& u, Smem32<DK>& sm, int l) {
    const int n = l & 15, g = l >> 4;
    bool bad = false;
    Dots<DK, 4> kk;  // of the previous chunk, with its beta and decays
    float b = 0.f;
    f32x4 d = {0.f, 0.f, 0.f, 0.f};
    period_end();
    for (int c = 0; c <= u.nch; ++c) {
        f32x4 x[Shape32<DK>::NB];
        const float bprev = b;
        const f32x4 dprev = d;
        if (c < u.nch) {
            load_operand<DK>(sm.k[c & 3], n, g, x);
            b = sm.beta[c & 3][n];
            d = lds4(&sm.d[c & 1][n * kLdA + 4 * g]);
        }
        if (c > 0) {
            const f32x4 y = kk.sum();  // K K^T is symmetric: lane (n, g) holds [n][4 g + e]
            f32x4 a;
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                const int s = 4 * g + e;
                const float bk = bprev * y[e];
                if (s == n) bad |= !(bk >= 0.f && bk <= kKeyBetaMax);
                a[e] = s < n ? bk * dprev[e] : 0.f;
            }
            st4(&sm.a[n * kLdA + 4 * g], a);
            asm volatile("" ::: "memory");  // one wave's LDS accesses are performed in order
            float row[kC], t[kC];
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                const f32x4 z = lds4(&sm.a[n * kLdA + 4 * i]);
#pragma unroll
                for (int e = 0; e < 4; ++e) row[4 * i + e] = z[e];
            }
#pragma unroll
            for (int r = 0; r < kC; ++r) t[r] = r == n ? 1.f : 0.f;
            t_diag_solve(t, row, n, std::make_integer_sequence<int, 15>{});
            // t[r] = T[r][n] in all four lane groups; group g writes rows 4 g + e
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                const float te = g == 0 ? t[e] : g == 1 ? t[4 + e] : g == 2 ? t[8 + e] : t[12 + e];
                sm.t[(c - 1) & 1][(4 * g + e) * kC + n] = 4 * g + e == n ? 0.f : te * bprev;
            }
        }
        if (c < u.nch)
            kk.mma(x, x);
        else
            flag32(sm, bad);
        period_end();
    }
    for (int i = 0; i < 3; ++i) period_end();
}

// Wave 7: operands of chunk c in period c + 1, P of chunk c in period c + 2.
template <int DK>
__device__ __forceinline__ void p_wave32(const Unit32& u, Smem32<DK>& sm, int l) {
    constexpr int NB = Shape32<DK>::NB;
    const int n = l & 15, g = l >> 4;
    f32x4 x[NB], y[NB], d;
    auto load = [&](int c) {
        load_operand<DK>(sm.k[c & 3], n, g, x);
        load_operand<DK>(sm.q[c % kQSlots], n, g, y);
        d = lds4(&sm.d[c & 1][n * kLdA + 4 * g]);
    };
    period_end();
    if (u.nch > 0) load(0);
    period_end();
    for (int c = 0; c < u.nch; ++c) {
        Dots<DK, DK / 8> kq;
        kq.mma(x, y);  // lane (n, g): k_{4g+e}.q_n
        // q_n.k_n again in f64: it weighs most in o_n, and its fp32 rounding
        // alone would exceed everything else's
        double s0 = 0.0, s1 = 0.0;
#pragma unroll
        for (int i = 0; i < NB; ++i) {
            s0 = fma(double(x[i][0]), double(y[i][0]), s0);
            s1 = fma(double(x[i][1]), double(y[i][1]), s1);
            s0 = fma(double(x[i][2]), double(y[i][2]), s0);
            s1 = fma(double(x[i][3]), double(y[i][3]), s1);
        }
        s0 += s1;
        s0 += __shfl_xor(s0, 16, kWave);
        s0 += __shfl_xor(s0, 32, kWave);
        const f32x4 dc = d;
        load(min(c + 1, u.nch - 1));
        const f32x4 z = kq.sum();
        f32x4 w;
#pragma unroll
        for (int e = 0; e < 4; ++e) w[e] = 4 * g + e < n ? z[e] * dc[e] : 4 * g + e == n ? float(s0) : 0.f;
        st4(&sm.p[c & 3][n * kC + 4 * g], w);
        period_end();
    }
    for (int i = 0; i < 3; ++i) period_end();
}

// ------------------------------------------------------------ scan waves
template <int DK>
__device__ __forceinline__ void scan32(const SeqParams& p, const Unit32& u, Smem32<DK>& sm, int w, int l) {
    using Sh = Shape32<DK>;
    constexpr int VW = Sh::VW, NH = Sh::NH, NB = Sh::NB;
    const int n = l & 15, g = l >> 4;
    const int i = u.i0 + 16 * w + n;  // this lane's row of S
    const size_t srow = ((size_t(u.seq) * p.heads + u.h) * p.d_v + i) * p.d_k;
    f32x4 S[NB];
    {
        f32x4 y[NB];
#pragma unroll
        for (int h = 0; h < NH; ++h)
#pragma unroll
            for (int e = 0; e < VW; ++e) {
                const int col = 16 * VW * h + 4 * VW * g + 4 * e;
                y[h * VW + e] = (f32x4){0.f, 0.f, 0.f, 0.f};
                if (p.init && i < p.d_v && col < p.d_k) y[h * VW + e] = *reinterpret_cast<const f32x4*>(p.init + srow + col);
            }
#pragma unroll
        for (int h = 0; h < NH; ++h)
#pragma unroll
            for (int v = 0; v < VW; ++v)
#pragma unroll
                for (int r = 0; r < 4; ++r) {
                    const int j = VW * r + v;
                    S[h * VW + v][r] = y[h * VW + j / 4][j % 4];
                }
    }
    float finite = 0.f;
    f32x4 kx[NB];
    period_end();
    period_end();
    if (u.nch > 0) load_operand<DK>(sm.k[0], n, g, kx);
    period_end();
    for (int c = 0; c < u.nch; ++c) {
        const int slot = c & 3, B = c & 1;
        f32x4 y[NB];
        state_operand<DK>(S, y);
#pragma unroll
        for (int b = 0; b < NB; ++b) st4(&sm.s0[B][w][(b * 64 + l) * 4], y[b]);
        Dots<DK, 4> xk;
        xk.mma(kx, y);
        // K's rows 4 g + e as the transposed operand: VW key columns per block set
        float kt[4][NH][VW];
#pragma unroll
        for (int e = 0; e < 4; ++e)
#pragma unroll
            for (int h = 0; h < NH; ++h) {
                if constexpr (VW == 4) {
                    const f32x4 z = lds4(&sm.k[slot][kq_off<DK>(4 * g + e, 16 * h + n)]);
#pragma unroll
                    for (int v = 0; v < 4; ++v) kt[e][h][v] = z[v];
                } else {
                    const float2 z = *reinterpret_cast<const float2*>(&sm.k[slot][kq_off<DK>(4 * g + e, n >> 1) + 2 * (n & 1)]);
                    kt[e][h][0] = z.x, kt[e][h][1] = z.y;
                }
            }
        const f32x4 be = lds4(&sm.beta[slot][4 * g]), gd = lds4(&sm.gdl[slot][4 * g]), bg = lds4(&sm.bgl[slot][4 * g]);
        const f32x4 ga = lds4(&sm.gam[c % kQSlots][4 * g]), tr = lds4(&sm.t[B][n * kC + 4 * g]);
        const float gl = sm.gam[c % kQSlots][kC - 1];
        const f32x4 X = xk.sum();  // lane (n, g): (K S0^T)[4g+e][n]
        // With W = V - gamma X and M = (T - I) diag(beta) W: U = beta W + M,
        // and U times its decay to the chunk's end, each rounded once
        f32x4 W;
#pragma unroll
        for (int e = 0; e < 4; ++e) W[e] = fmaf(-ga[e], X[e], sm.v[slot][(4 * g + e) * kLdV + 16 * w + n]);
        const f32x4 z = {0.f, 0.f, 0.f, 0.f};
        f32x4 M = mfma4(tr[0], W[0], z), M1 = mfma4(tr[2], W[2], z);
        M = mfma4(tr[1], W[1], M);
        M1 = mfma4(tr[3], W[3], M1);
        M += M1;
        f32x4 U, Uh;
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            U[e] = fmaf(be[e], W[e], M[e]);
            Uh[e] = fmaf(bg[e], W[e], gd[e] * M[e]);
        }
        st4(&sm.u[B][w][4 * l], U);
#pragma unroll
        for (int e = 0; e < 4; ++e) watch(finite, U[e]);
#pragma unroll
        for (int b = 0; b < NB; ++b) S[b] *= gl;
#pragma unroll
        for (int e = 0; e < 4; ++e)
#pragma unroll
            for (int b = 0; b < NB; ++b) S[b] = mfma4(kt[e][b / VW][b % VW], Uh[e], S[b]);
        load_operand<DK>(sm.k[min(c + 1, u.nch - 1) & 3], n, g, kx);
        period_end();
    }
#pragma unroll
    for (int b = 0; b < NB; ++b)
#pragma unroll
        for (int e = 0; e < 4; ++e) watch(finite, S[b][e]);
    flag32(sm, !(finite == 0.f));
    period_end();
    period_end();
    // after the last barrier: every wave has set its flag; a tile that will be
    // recomputed leaves the final state alone (it may be the initial state's
    // own buffer)
    if (sm.rerun == 0 && p.fin && i < p.d_v) {
        f32x4 y[NB];
        state_operand<DK>(S, y);
#pragma unroll
        for (int h = 0; h < NH; ++h)
#pragma unroll
            for (int e = 0; e < VW; ++e) {
                const int col = 16 * VW * h + 4 * VW * g + 4 * e;
                if (col < p.d_k) *reinterpret_cast<f32x4*>(p.fin + srow + col) = y[h * VW + e];
            }
    }
}

// ------------------------------------------------------------ output waves
// Operands of chunk c in period c + 4, its outputs in period c + 5.
template <int DK>
__device__ __forceinline__ void out32(const SeqParams& p, const Unit32& u, Smem32<DK>& sm, int w, int l) {
    constexpr int NB = Shape32<DK>::NB;
    const int n = l & 15, g = l >> 4;
    const int i = u.i0 + 16 * w + 4 * g;  // first of this lane's 4 output rows
    float finite = 0.f;
    f32x4 x[NB], y[NB], pt, ut;
    float ga = 0.f;
    auto load = [&](int c) {
        load_operand<DK>(sm.q[c % kQSlots], n, g, x);
#pragma unroll
        for (int b = 0; b < NB; ++b) y[b] = lds4(&sm.s0[c & 1][w][(b * 64 + l) * 4]);
        pt = lds4(&sm.p[c & 3][n * kC + 4 * g]);
        ut = lds4(&sm.u[c & 1][w][4 * l]);
        ga = sm.gam[c % kQSlots][n];
    };
    for (int k = 0; k < 4; ++k) period_end();
    if (u.nch > 0) load(0);
    period_end();
    for (int c = 0; c < u.nch; ++c) {
        const int t0 = u.tb + c * kC;
        Dots<DK, DK / 8> qs;
        qs.mma(y, x);  // O^T: lane (n, g) holds rows 4 g + e of token n
        const f32x4 pc = pt, uc = ut;
        const float gc = ga;
        load(min(c + 1, u.nch - 1));
        f32x4 O = qs.sum() * gc;
#pragma unroll
        for (int e = 0; e < 4; ++e) O = mfma4(uc[e], pc[e], O);
#pragma unroll
        for (int e = 0; e < 4; ++e) watch(finite, O[e]);
        if (t0 + n < u.te && i < p.d_v)
            *reinterpret_cast<f32x4*>(static_cast<float*>(p.o) + ((size_t(t0) + n) * p.heads + u.h) * p.d_v + i) = O;
        if (c + 1 == u.nch) flag32(sm, !(finite == 0.f));
        period_end();
    }
}

template <int DK>
__global__ __launch_bounds__(512, DK == 128 ? 2 : 4) void gdr_chunk32_kernel(Chunk32Params cp) {
    __shared__ __align__(16) KernelSmem32<DK> smu;
    Smem32<DK>& sm = smu.chunk;
    const SeqParams& p = cp.sp;
    int unit, tile;
    map_block(blockIdx.x, cp.units, cp.n_tiles, unit, tile);
    Unit32 u;
    u.seq = unit / p.heads;
    u.h = unit - u.seq * p.heads;
    u.i0 = tile * kRows;
    seq_bounds(p.cu_seqlens, u.seq, p.seq_len, u.tb, u.te);
    u.nch = (u.te - u.tb + kC - 1) / kC;
    const int l = threadIdx.x & 63;
    const int w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    if (threadIdx.x == 0) sm.rerun = 0;
    period_end();

    // every role passes nch + 5 period ends
    if (w < 2)
        scan32<DK>(p, u, sm, w, l);
    else if (w < 4)
        out32<DK>(p, u, sm, w - 2, l);
    else if (w == 4)
        loader32<DK, true>(p, u, sm, l);
    else if (w == 5)
        loader32<DK, false>(p, u, sm, 64 + l);
    else if (w == 6)
        t_wave32<DK>(u, sm, l);
    else
        p_wave32<DK>(u, sm, l);

    const int rerun = sm.rerun;
    if (rerun != 0) {  // uniform: set before the last barrier
        __syncthreads();  // every wave has read the flag: the LDS is free
        staged_rows<16, float, 8, 8>(p, smu.rerun, u.seq, u.h, u.i0, threadIdx.x);
    }
}

}  // namespace

bool chunk32_supported(const rhz_gdr_prefill_args& a) {
    const auto al16 = [](const void* p) { return (reinterpret_cast<uintptr_t>(p) & 15u) == 0; };
    // 16-byte accesses throughout, and 32-bit byte offsets within a chunk
    return a.dtype == RHZ_F32 && a.d_k % 4 == 0 && a.d_k <= 128 && a.d_v % 4 == 0 && al16(a.q) && al16(a.k) &&
           al16(a.v) && al16(a.o) && al16(a.initial_state) && al16(a.final_state) &&
           (int64_t)a.heads * (a.d_k > a.d_v ? a.d_k : a.d_v) * 4 * kC <= INT32_MAX;
}

hipError_t launch_chunk32(const rhz_gdr_prefill_args& a, hipStream_t st) {
    Chunk32Params cp{{a.q, a.k, a.v, a.gate, a.beta, a.cu_seqlens, a.initial_state, a.final_state, a.o, a.seq_len,
                      a.heads, a.d_k, a.d_v, a.gate_kind == RHZ_GATE_ALPHA},
                     a.batch * a.heads, (a.d_v + kRows - 1) / kRows};
    const dim3 grid(cp.units * cp.n_tiles);
    if (a.d_k <= 32)
        hipLaunchKernelGGL(gdr_chunk32_kernel<32>, grid, dim3(512), 0, st, cp);
    else if (a.d_k <= 64)
        hipLaunchKernelGGL(gdr_chunk32_kernel<64>, grid, dim3(512), 0, st, cp);
    else
        hipLaunchKernelGGL(gdr_chunk32_kernel<128>, grid, dim3(512), 0, st, cp);
    return hipGetLastError();
}

}  // namespace rhz
