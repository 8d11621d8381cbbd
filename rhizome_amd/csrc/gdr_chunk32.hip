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
// What bounds it: the SIMDs' issue of fp32 MFMA and VALU together.  On gfx950
// a 16x16x4 fp32 MFMA takes 32 cycles during which its SIMD issues no VALU
// instruction of any wave (measured; 16-bit MFMA leaves half of its cycles),
// so a SIMD's time is the sum of both.  Per 16 tokens a tile of 32 rows needs
// 272 MFMAs at c = 16 (K K^T and Q K^T 32 each, K S0^T, Q S0^T and S' 64 each,
// T R and P U 8 each); the same tokens would take 316 at c = 32 and 412 at
// c = 64.  They are spread evenly over the four SIMDs, 68 each = 2176 cycles
// per chunk: the state-dependent chain (K S0^T, T R, S') of 16 rows on each of
// SIMDs 0 and 1, their outputs (Q S0^T, P U) on SIMDs 2 and 3 two chunks later,
// beside K K^T and Q K^T.  The VALU work that does not follow from the state --
// the decays and T -- is done for four chunks at once, one chunk to each row
// of 16 lanes.
//
// Measured, B = 4 H = 16 T = 4096 d = 128: 429 us (85 TFLOP/s of fp32 MFMA, 55 %
// of what a large fp32 matrix product reaches) against 1066 us for the
// token-by-token kernel; a period takes about 3880 cycles, 2176 of them MFMA.
//
// One workgroup of 8 waves per (sequence, head, 32 rows of S), in lockstep:
// one barrier per chunk, every wave at its own stage of the pipeline:
//   period p: waves 4, 5 stage chunk p into LDS,
//             wave 7 reads chunk p - 1 and forms P of chunk p - 2,
//             waves 0, 1 run the state through chunk p - 2,
//             waves 2, 3 read chunk p - 3 and form the outputs of chunk p - 4;
//   wave 6 forms the decays and T of the four chunks from 4 s + 4 on in
//             periods 4 s + 1 .. 4 s + 4, with K from its own loads.
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
// token-sequential recurrence (staged_rows) in the same launch: at once where a
// key, gate or beta of the first 64 tokens is outside, else at the sequence's
// end.

#include "gdr_device.hpp"
#include "gdr_internal.hpp"
#include "gdr_solve.hpp"
#include "gdr_staged.hpp"

namespace rhz {
namespace {

constexpr int kC = 16;    // tokens per chunk
constexpr int kRows = 32; // rows of S per workgroup (two scan waves of 16)
constexpr int kLdV = 36;  // fp32 row stride of the V tile (4 rows apart: 16 banks apart)
constexpr int kLdA = 20;  // fp32 row stride of A and D
constexpr float kKeyBetaMax = 2.0f;  // largest beta |k|^2 (the step is non-expansive up to 2)

// Sequences of up to short_len tokens are run by the recurrence.  A sequence's
// arithmetic must not depend on its batch, so the line follows from its length
// and d_k alone, while the times cross at lengths that depend on how often the
// launch fills the CUs.  H = 16, recurrence against this kernel, us:
//   d_k = d_v = 128: B=16 52/68 at 65 tokens, 74/75 at 96, 100/86 at 128
//                    B=1  19/17 at 65, 26/19 at 96
//   d_k 64, d_v 256: B=64 155/380 at 65, 221/421 at 96, 437/636 at 192
//                    B=16 47/97 at 65, 64/106 at 96, 406/425 at 640
//                    B=1  22/13 at 65, 30/14 at 96, 55/21 at 192, 175/54 at 640
//   d_k 32, d_v 128: B=64 50/92 at 65, 66/101 at 96, 126/157 at 192
//                    B=1  20/10 at 65, 28/11 at 96, 54/16 at 192
// At d_k > 64 the line is where full launches cross.  Below, where a CU takes
// three of the recurrence's workgroups of 64 or 128 rows, it is where what full
// launches lose and what the others gain are about the same factor.
__host__ __device__ constexpr int short_len(int d_k) { return d_k > 32 ? 96 : 64; }
// the roles take it that a sequence has five chunks or more, two superblocks
static_assert(short_len(32) >= 4 * kC && short_len(128) >= 4 * kC, "every sequence here has a second superblock");

struct Chunk32Params {
    SeqParams sp;
    int batch, units, n_tiles;
    int long_only;  // units count the sequences of more than short_len tokens (the recurrence kernel runs the others)
    int first;      // the launch's first workgroup
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
    static constexpr int NA = DK == 32 ? 8 : 16;  // accumulators of the sums that go into o
    static constexpr int NL = DK / 32;     // 16-byte pieces of K (and Q) per loader thread and chunk
};

// Token of a chunk that MFMA row 4 g + e stands for, 4 e + g (and the position
// at which per-token values are kept in LDS): register e of lane group g then
// holds token 4 e + g, and MFMA e of a sum over the chunk's tokens adds tokens
// 4 e .. 4 e + 3, in the recurrence's order.  The order matters where decays
// make the last terms the largest: fp32 MFMA rounds after every product, and
// with tokens 4 g + e in its place the state's error was 1.2 to 1.3 times this.
__host__ __device__ constexpr int sig(int m) { return (m & 3) << 2 | m >> 2; }

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
    // [chunk & 3]: K read until period c + 2, Q until c + 3
    float k[4][kC * DK];
    float q[4][kC * DK];
    float v[4][kC * kLdV];
    float p[4][kC * kC];     // P, the columns of token s at sig(s)
    // [superblock & 1][chunk & 3], written by wave 6
    // (the values of token r at position sig(r))
    float d[8][kC * kLdA];   // D, the columns of token s at sig(s)
    float t[8][kC * kC];     // T below the diagonal, column s times beta_s
    float gam[8][kC];        // gamma_r
    float beta[8][kC];
    float gdl[8][kC];        // D_15,r
    float bgl[8][kC];        // beta_r D_15,r, and what its rounding left out
    float bge[8][kC];
    float kk[4][kC * kLdA];  // K K^T of a superblock's chunks, wave 6 only
    float kn[4][kC];         // |k_r|^2
    // [chunk & 1][scan wave]
    float s0[2][2][Shape32<DK>::NB * 256];  // entering state
    float u[2][2][256];                     // U
    int rerun;  // an input left the domain
};

// The recurrence in this kernel (short sequences and reruns), in the lanes per
// row and columns per lane that the recurrence's own kernel has for these d_k:
// equal to it bit for bit.  The tile's rows take one, two or eight of the
// workgroup's waves; all of them stage.
template <int DK>
struct Recurrence32 {
    static constexpr int LPR = DK == 128 ? 16 : DK / 16;
    static constexpr int VPL = DK / LPR;
    static constexpr int NW = kRows * LPR / kWave;
    using Smem = StageSmem<LPR, VPL, NW>;
    static_assert(Smem::RPB == kRows && Smem::DKP == DK, "the recurrence covers the tile");
};

template <int DK>
union KernelSmem32 {
    Smem32<DK> chunk;
    typename Recurrence32<DK>::Smem rec;
};

template <int DK>
__device__ __forceinline__ void recurrence32(const SeqParams& p, KernelSmem32<DK>& smu, int seq, int h, int i0) {
    using R = Recurrence32<DK>;
    staged_rows<R::LPR, float, R::VPL, R::NW, 8>(p, smu.rec, seq, h, i0, threadIdx.x);
}

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

// The end of period 1.  True where wave 6 found an input of the first superblock
// outside the domain in period 0: every wave then leaves the pipeline.  (No
// flag is set in period 1, so all waves read the same.  A check at every
// superblock cost sequences inside the domain 1 to 2 %.)
template <int DK>
__device__ __forceinline__ bool period1_leaves(Smem32<DK>& sm) {
    const int rerun = sm.rerun;
    period_end();
    return __builtin_amdgcn_readfirstlane(rerun) != 0;
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
// layout, in NA accumulators added pairwise at the end.  fp32 MFMA rounds
// after every product, so the error grows with the length of an accumulator's
// chain: Q K^T and Q S0^T, whose sums go into o as they are, take as many as
// give chains of 4 or 8 products (the recurrence's lanes sum 8), the others 4.
template <int DK, int NA>
struct Dots {
    f32x4 acc[NA];
    __device__ __forceinline__ void zero() {
#pragma unroll
        for (int i = 0; i < NA; ++i) acc[i] = (f32x4){0.f, 0.f, 0.f, 0.f};
    }
    // pieces [I0, I1)
    template <int I0 = 0, int I1 = Shape32<DK>::NB>
    __device__ __forceinline__ void mma(const f32x4 (&x)[Shape32<DK>::NB], const f32x4 (&y)[Shape32<DK>::NB]) {
#pragma unroll
        for (int i = I0; i < I1; ++i)
#pragma unroll
            for (int e = 0; e < 4; ++e) acc[(4 * i + e) % NA] = mfma4(x[i][e], y[i][e], acc[(4 * i + e) % NA]);
    }
    // x in load_operand's layout, S the state's accumulators: element j of lane
    // (., g) is key column 16 VW h + 4 VW g + j, i.e. row j / VW of block
    // (h, j % VW).  FIRST: the state is the MFMA's first operand.
    template <bool FIRST>
    __device__ __forceinline__ void mma_state(const f32x4 (&x)[Shape32<DK>::NB], const f32x4 (&S)[Shape32<DK>::NB]) {
        constexpr int VW = Shape32<DK>::VW;
#pragma unroll
        for (int h = 0; h < Shape32<DK>::NH; ++h)
#pragma unroll
            for (int j = 0; j < 4 * VW; ++j) {
                const float a = x[h * VW + j / 4][j % 4], s = S[h * VW + j % VW][j / VW];
                f32x4& c = acc[(4 * VW * h + j) % NA];
                c = FIRST ? mfma4(s, a, c) : mfma4(a, s, c);
            }
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
};

// Byte offsets of a loader thread's pieces from its chunk's first token; rows
// past `last` and columns past the row's end repeat the last ones (they are
// zeroed as they are staged).
template <int DK>
struct Off32 {
    uint32_t kq[Shape32<DK>::NL], v;
    __device__ __forceinline__ void set(const SeqParams& p, int i0, int j, int last) {
        constexpr int PPR = DK / 4;
        const uint32_t H = p.heads;
#pragma unroll
        for (int i = 0; i < Shape32<DK>::NL; ++i) {
            const int f = j + 128 * i;
            kq[i] = (uint32_t(min(f / PPR, last)) * H * p.d_k + min(4 * (f % PPR), p.d_k - 4)) * 4u;
        }
        v = (uint32_t(min(j >> 3, last)) * H * p.d_v + min(4 * (j & 7), p.d_v - 4 - i0)) * 4u;
    }
};

// Chunk min(c, nch - 1) into registers (thread j of 128).  The offsets become
// the last chunk's once it is reached; no other follows.
template <int DK>
__device__ __forceinline__ void load32(const SeqParams& p, const Unit32& u, int c, int j, Off32<DK>& o, In32<DK>& r) {
    c = min(c, u.nch - 1);
    const int t0 = u.tb + c * kC;
    if (c == u.nch - 1) o.set(p, u.i0, j, min(u.te - t0, kC) - 1);
    const size_t th = size_t(t0) * p.heads + u.h;
    const char* kb = reinterpret_cast<const char*>(static_cast<const float*>(p.k) + th * p.d_k);
    const char* qb = reinterpret_cast<const char*>(static_cast<const float*>(p.q) + th * p.d_k);
    const char* vb = reinterpret_cast<const char*>(static_cast<const float*>(p.v) + th * p.d_v + u.i0);
#pragma unroll
    for (int i = 0; i < Shape32<DK>::NL; ++i) {
        r.k[i] = *reinterpret_cast<const f32x4*>(kb + o.kq[i]);
        r.q[i] = *reinterpret_cast<const f32x4*>(qb + o.kq[i]);
    }
    r.v = *reinterpret_cast<const f32x4*>(vb + o.v);
}

// Chunk c from registers into its LDS slot.
template <int DK>
__device__ __forceinline__ void stage32(const SeqParams& p, const Unit32& u, Smem32<DK>& sm, int c, int j,
                                        const In32<DK>& r) {
    constexpr int PPR = DK / 4;
    const int len = u.te - (u.tb + c * kC), slot = c & 3;
    const int vrow = j >> 3, vcol = 4 * (j & 7);
    if (len >= kC && p.d_k == DK && u.i0 + kRows <= p.d_v) {  // uniform
#pragma unroll
        for (int i = 0; i < Shape32<DK>::NL; ++i) {
            const int f = j + 128 * i;
            st4(&sm.k[slot][kq_off<DK>(f / PPR, f % PPR)], r.k[i]);
            st4(&sm.q[slot][kq_off<DK>(f / PPR, f % PPR)], r.q[i]);
        }
        st4(&sm.v[slot][vrow * kLdV + vcol], r.v);
        return;
    }
    const f32x4 z = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int i = 0; i < Shape32<DK>::NL; ++i) {
        const int f = j + 128 * i, row = f / PPR, piece = f % PPR;
        const bool ok = row < len && 4 * piece < p.d_k;
        st4(&sm.k[slot][kq_off<DK>(row, piece)], ok ? r.k[i] : z);
        st4(&sm.q[slot][kq_off<DK>(row, piece)], ok ? r.q[i] : z);
    }
    st4(&sm.v[slot][vrow * kLdV + vcol], vrow < len && u.i0 + vcol < p.d_v ? r.v : z);
}

template <int DK>
__device__ __forceinline__ void loader32(const SeqParams& p, const Unit32& u, Smem32<DK>& sm, int j) {
    In32<DK> r0, r1;
    Off32<DK> o;
    o.set(p, u.i0, j, kC - 1);
    load32<DK>(p, u, 0, j, o, r0);
    load32<DK>(p, u, 1, j, o, r1);
    for (int c = 0; c < u.nch; c += 2) {
        stage32<DK>(p, u, sm, c, j, r0);
        load32<DK>(p, u, c + 2, j, o, r0);
        period_end();
        if (c + 1 >= u.nch) break;
        stage32<DK>(p, u, sm, c + 1, j, r1);
        load32<DK>(p, u, c + 3, j, o, r1);
        if (c > 0)
            period_end();
        else if (period1_leaves(sm))
            return;
    }
    for (int i = 0; i < 4; ++i) period_end();
}

// ------------------------------------------------------------ decays and T
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

// Wave 6: decays and T of superblocks of four chunks, lane l = token l of the
// superblock wherever a lane stands for a token.
template <int DK>
struct TWave {
    static constexpr int NB = Shape32<DK>::NB;
    const SeqParams& p;
    const Unit32& u;
    Smem32<DK>& sm;
    const int l;
    float graw, braw;   // gate and beta as loaded
    float beta;         // of this lane's token
    float row[kC];      // this lane's row of D
    float gam, gdl, bgl, bge;
    f32x4 x0[NB], x1[NB];  // K operands of even and odd chunks: row l & 15, pieces 4 j + l / 16
    Dots<DK, 4> acc;
    bool bad = false;

    __device__ __forceinline__ int token(int t) const { return min(u.tb + t, u.te - 1); }
    __device__ __forceinline__ void load_gates(int sb) {
        const size_t i = size_t(token(64 * sb + l)) * p.heads + u.h;
        graw = p.gate[i];
        braw = p.beta[i];
    }
    __device__ __forceinline__ void load_k(int c, f32x4 (&x)[NB]) {
        const int g = l >> 4;
        const float* kr = static_cast<const float*>(p.k) + (size_t(token(16 * c + (l & 15))) * p.heads + u.h) * p.d_k;
#pragma unroll
        for (int j = 0; j < NB; ++j) x[j] = *reinterpret_cast<const f32x4*>(kr + min(16 * j + 4 * g, p.d_k - 4));
        if (p.d_k != DK) {  // uniform
#pragma unroll
            for (int j = 0; j < NB; ++j)
                if (16 * j + 4 * g >= p.d_k) x[j] = (f32x4){0.f, 0.f, 0.f, 0.f};
        }
    }
    // D_{n, s-1} = D_{n, s} alpha_s for s <= n, from the right (1 for s > n),
    // and D_15,n: products carried as two floats and rounded once (a chain of
    // 15 fp32 roundings would cost slowly decaying states more than all their
    // other roundings do).
    __device__ __forceinline__ void decays(int sb) {
        int n = l & 15;
        asm volatile("" : "+v"(n));  // the comparisons with n are made here: kept, they would spill
        const bool ok = u.tb + 64 * sb + l < u.te;
        const float alpha = ok ? decay_factor(graw, p.gate_is_alpha) : 1.f;
        beta = ok ? braw : 0.f;
        bad |= !(alpha >= 0.f && alpha <= 1.f) || !(beta >= 0.f);
        TwoFloat d, e;
        row[kC - 1] = 1.f;
#define RHZ_DECAY_STEP(s)                           \
    {                                               \
        const float as = dpp_mov<0x150 + s>(alpha); \
        d.mul(s <= n ? as : 1.f);                   \
        e.mul(s > n ? as : 1.f);                    \
        row[s - 1] = d.value();                     \
    }
        RHZ_DECAY_STEP(15) RHZ_DECAY_STEP(14) RHZ_DECAY_STEP(13) RHZ_DECAY_STEP(12) RHZ_DECAY_STEP(11)
        RHZ_DECAY_STEP(10) RHZ_DECAY_STEP(9) RHZ_DECAY_STEP(8) RHZ_DECAY_STEP(7) RHZ_DECAY_STEP(6)
        RHZ_DECAY_STEP(5) RHZ_DECAY_STEP(4) RHZ_DECAY_STEP(3) RHZ_DECAY_STEP(2) RHZ_DECAY_STEP(1)
#undef RHZ_DECAY_STEP
        d.mul(dpp_mov<0x150>(alpha));
        gam = d.value();
        gdl = e.value();
        e.mul(beta);
        bgl = e.value();
        bge = e.lo - (bgl - e.hi);
    }
    // the decays to LDS, for the other waves
    __device__ __forceinline__ void publish(int sb) {
        const int ch = 4 * (sb & 1) + (l >> 4), n = l & 15;
#pragma unroll
        for (int i = 0; i < 4; ++i)
            st4(&sm.d[ch][n * kLdA + 4 * i], (f32x4){row[i], row[4 + i], row[8 + i], row[12 + i]});
        const int at = sig(n);
        sm.gam[ch][at] = gam;
        sm.beta[ch][at] = beta;
        sm.gdl[ch][at] = gdl;
        sm.bgl[ch][at] = bgl;
        sm.bge[ch][at] = bge;
    }
    // K K^T of chunk c of the superblock, once its MFMAs are issued (it is
    // symmetric: lane (n, g) holds [n][4 g + e])
    __device__ __forceinline__ void keep_kk(int c) {
        const int n = l & 15, g = l >> 4;
        const f32x4 y = acc.sum();
        st4(&sm.kk[c][n * kLdA + 4 * g], y);
        const int e = n & 3;
        if (g == n >> 2) sm.kn[c][n] = e == 0 ? y[0] : e == 1 ? y[1] : e == 2 ? y[2] : y[3];
    }
    // T of the superblock's four chunks by forward substitution: lane (blk, n)
    // holds row n of chunk blk's A and solves column n of its T
    __device__ __forceinline__ void solve(int sb) {
        int n = l & 15;
        const int blk = l >> 4;
        asm volatile("" : "+v"(n));
        asm volatile("" ::: "memory");  // one wave's LDS accesses are performed in order
        const float bk = beta * sm.kn[blk][n];
        bad |= !(bk <= kKeyBetaMax);
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            f32x4 a = lds4(&sm.kk[blk][n * kLdA + 4 * i]);
#pragma unroll
            for (int e = 0; e < 4; ++e) a[e] = 4 * i + e < n ? (beta * a[e]) * row[4 * i + e] : 0.f;
            st4(&sm.kk[blk][n * kLdA + 4 * i], a);
        }
        asm volatile("" ::: "memory");
        float a[kC], t[kC];
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const f32x4 z = lds4(&sm.kk[blk][n * kLdA + 4 * i]);
#pragma unroll
            for (int e = 0; e < 4; ++e) a[4 * i + e] = z[e];
        }
#pragma unroll
        for (int r = 0; r < kC; ++r) t[r] = r == n ? 1.f : 0.f;
        t_diag_solve(t, a, n, std::make_integer_sequence<int, 15>{});
        float* tt = sm.t[4 * (sb & 1) + blk];
#pragma unroll
        for (int r = 0; r < kC; ++r) tt[sig(r) * kC + sig(n)] = r == n ? 0.f : t[r] * beta;
    }
    // K K^T of chunk c of the superblock from x, then x becomes chunk `next`'s
    __device__ __forceinline__ void product(f32x4 (&x)[NB], int c, int next) {
        acc.zero();
        acc.mma(x, x);
        load_k(next, x);
        keep_kk(c);
    }
    __device__ __forceinline__ void run() {
        constexpr int HB = NB / 2;
        const int nsb = (u.nch + 3) / 4;
        // superblock 0, in period 0
        load_gates(0);
        load_k(0, x0);
        load_k(1, x1);
        decays(0);
        publish(0);
        product(x0, 0, 2);
        product(x1, 1, 3);
        product(x0, 2, 4);
        product(x1, 3, 5);
        solve(0);
        const bool leave = __builtin_amdgcn_ballot_w64(bad) != 0;  // as period1_leaves
        flag32(sm, bad);
        load_gates(1);
        period_end();
        const int last = u.nch + 4;  // periods in all
        for (int q = 1, sb = 1; q < last; q += 4, ++sb) {
            const bool on = sb < nsb;
            if (on) {
                decays(sb);
                load_gates(sb + 1);
                acc.zero();
                acc.template mma<0, HB>(x0, x0);
            }
            period_end();
            if (q + 1 >= last || (q == 1 && leave)) break;
            if (on) {
                acc.template mma<HB, NB>(x0, x0);
                load_k(4 * sb + 2, x0);
                keep_kk(0);
                product(x1, 1, 4 * sb + 3);
            }
            period_end();
            if (q + 2 >= last) break;
            if (on) {
                publish(sb);
                product(x0, 2, 4 * sb + 4);
                acc.zero();
                acc.template mma<0, HB>(x1, x1);
            }
            period_end();
            if (q + 3 >= last) break;
            if (on) {
                acc.template mma<HB, NB>(x1, x1);
                load_k(4 * sb + 5, x1);
                keep_kk(3);
                solve(sb);
                if (sb + 1 == nsb) flag32(sm, bad);
            }
            period_end();
        }
    }
};

// ------------------------------------------------------------ P
// Wave 7: operands of chunk c in period c + 1, P of chunk c in period c + 2.
template <int DK>
__device__ __forceinline__ void p_wave32(const Unit32& u, Smem32<DK>& sm, int l) {
    constexpr int NB = Shape32<DK>::NB;
    const int g = l >> 4, n = sig(l & 15);  // this lane's token of K's and Q's rows
    struct In {
        f32x4 x[NB], y[NB], d;
    };
    auto load = [&](int c, In& in) {
        load_operand<DK>(sm.k[c & 3], n, g, in.x);
        load_operand<DK>(sm.q[c & 3], n, g, in.y);
        in.d = lds4(&sm.d[c & 7][n * kLdA + 4 * g]);
    };
    auto step = [&](int c, const In& in, In& next) {
        Dots<DK, Shape32<DK>::NA> kq;
        kq.zero();
        kq.mma(in.x, in.y);  // lane (., g): k_{4e+g}.q_n
        load(min(c + 1, u.nch - 1), next);
        // q_n.k_n again, summed in f64 (over pairs of products for the longest
        // rows): it weighs most in o_n,
        // and an fp32 chain's rounding alone would exceed all other errors
        double s0 = 0.0;
#pragma unroll
        for (int i = 0; i < NB; ++i) {
            if constexpr (DK == 128) {
                s0 += double(fmaf(in.x[i][1], in.y[i][1], in.x[i][0] * in.y[i][0]));
                s0 += double(fmaf(in.x[i][3], in.y[i][3], in.x[i][2] * in.y[i][2]));
            } else {
#pragma unroll
                for (int e = 0; e < 4; ++e) s0 = fma(double(in.x[i][e]), double(in.y[i][e]), s0);
            }
        }
        s0 += __shfl_xor(s0, 16, kWave);
        s0 += __shfl_xor(s0, 32, kWave);
        const f32x4 z = kq.sum();
        f32x4 w;
#pragma unroll
        for (int e = 0; e < 4; ++e) w[e] = 4 * e + g < n ? z[e] * in.d[e] : 4 * e + g == n ? float(s0) : 0.f;
        st4(&sm.p[c & 3][n * kC + 4 * g], w);
        period_end();
    };
    In a, b;
    period_end();
    load(0, a);
    if (period1_leaves(sm)) return;
    for (int c = 0; c < u.nch; c += 2) {  // by two, so that the operands need no copies
        step(c, a, b);
        if (c + 1 < u.nch) step(c + 1, b, a);
    }
    for (int i = 0; i < 2; ++i) period_end();
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
    load_operand<DK>(sm.k[0], sig(n), g, kx);
    if (period1_leaves(sm)) return;
    for (int c = 0; c < u.nch; ++c) {
        const int slot = c & 3, sb = c & 7, B = c & 1;
#pragma unroll
        for (int b = 0; b < NB; ++b) st4(&sm.s0[B][w][(b * 64 + l) * 4], S[b]);
        Dots<DK, 4> xk;
        xk.zero();
        xk.template mma_state<false>(kx, S);
        // K's rows 4 e + g as the transposed operand: VW key columns per block set
        float kt[4][NH][VW];
#pragma unroll
        for (int e = 0; e < 4; ++e)
#pragma unroll
            for (int h = 0; h < NH; ++h) {
                if constexpr (VW == 4) {
                    const f32x4 z = lds4(&sm.k[slot][kq_off<DK>(4 * e + g, 16 * h + n)]);
#pragma unroll
                    for (int v = 0; v < 4; ++v) kt[e][h][v] = z[v];
                } else {
                    const float2 z = *reinterpret_cast<const float2*>(&sm.k[slot][kq_off<DK>(4 * e + g, n >> 1) + 2 * (n & 1)]);
                    kt[e][h][0] = z.x, kt[e][h][1] = z.y;
                }
            }
        const f32x4 be = lds4(&sm.beta[sb][4 * g]), gd = lds4(&sm.gdl[sb][4 * g]), bg = lds4(&sm.bgl[sb][4 * g]);
        const f32x4 bz = lds4(&sm.bge[sb][4 * g]);
        const f32x4 ga = lds4(&sm.gam[sb][4 * g]), tr = lds4(&sm.t[sb][n * kC + 4 * g]);
        const float gl = sm.gam[sb][kC - 1];
        const f32x4 X = xk.sum();  // lane (n, g): (K S0^T)[4e+g][n]
        // With W = V - gamma X and M = (T - I) diag(beta) W: U = beta W + M,
        // and U times its decay to the chunk's end, each rounded once
        f32x4 W;
#pragma unroll
        for (int e = 0; e < 4; ++e) W[e] = fmaf(-ga[e], X[e], sm.v[slot][(4 * e + g) * kLdV + 16 * w + n]);
        const f32x4 z = {0.f, 0.f, 0.f, 0.f};
        f32x4 M = mfma4(tr[0], W[0], z), M1 = mfma4(tr[2], W[2], z);
        M = mfma4(tr[1], W[1], M);
        M1 = mfma4(tr[3], W[3], M1);
        M += M1;
        f32x4 U, Uh;
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            U[e] = fmaf(be[e], W[e], M[e]);
            Uh[e] = fmaf(bg[e], W[e], fmaf(bz[e], W[e], gd[e] * M[e]));
        }
        st4(&sm.u[B][w][4 * l], U);
#pragma unroll
        for (int e = 0; e < 4; ++e) watch(finite, U[e]);
        // the chunk's first eight tokens are summed apart and join the scaled
        // state in one rounding, so that a slowly decaying state is rounded
        // 9 times per chunk, not 17
        f32x4 first[NB];
#pragma unroll
        for (int b = 0; b < NB; ++b) first[b] = mfma4(kt[0][b / VW][b % VW], Uh[0], z);
#pragma unroll
        for (int b = 0; b < NB; ++b) first[b] = mfma4(kt[1][b / VW][b % VW], Uh[1], first[b]);
#pragma unroll
        for (int b = 0; b < NB; ++b) {
#pragma unroll
            for (int e = 0; e < 4; ++e) S[b][e] = fmaf(S[b][e], gl, first[b][e]);
            S[b] = mfma4(kt[2][b / VW][b % VW], Uh[2], S[b]);
        }
#pragma unroll
        for (int b = 0; b < NB; ++b) S[b] = mfma4(kt[3][b / VW][b % VW], Uh[3], S[b]);
        load_operand<DK>(sm.k[min(c + 1, u.nch - 1) & 3], sig(n), g, kx);
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
#pragma unroll
        for (int h = 0; h < NH; ++h)
#pragma unroll
            for (int i4 = 0; i4 < VW; ++i4) {
                const int col = 16 * VW * h + 4 * VW * g + 4 * i4;
                f32x4 y;
#pragma unroll
                for (int e = 0; e < 4; ++e) y[e] = S[h * VW + (4 * i4 + e) % VW][(4 * i4 + e) / VW];
                if (col < p.d_k) *reinterpret_cast<f32x4*>(p.fin + srow + col) = y;
            }
    }
}

// ------------------------------------------------------------ output waves
// Operands of chunk c in period c + 3, its outputs in period c + 4.
template <int DK>
__device__ __forceinline__ void out32(const SeqParams& p, const Unit32& u, Smem32<DK>& sm, int w, int l) {
    constexpr int NB = Shape32<DK>::NB;
    const int n = l & 15, g = l >> 4;
    const int i = u.i0 + 16 * w + 4 * g;  // first of this lane's 4 output rows
    float finite = 0.f;
    struct In {
        f32x4 x[NB], S[NB], p, u;
        float gam;
    };
    auto load = [&](int c, In& in) {
        load_operand<DK>(sm.q[c & 3], n, g, in.x);
#pragma unroll
        for (int b = 0; b < NB; ++b) in.S[b] = lds4(&sm.s0[c & 1][w][(b * 64 + l) * 4]);
        in.p = lds4(&sm.p[c & 3][n * kC + 4 * g]);
        in.u = lds4(&sm.u[c & 1][w][4 * l]);
        in.gam = sm.gam[c & 7][sig(n)];
    };
    float* orow = static_cast<float*>(p.o) + ((size_t(u.tb) + n) * p.heads + u.h) * p.d_v + i;
    const size_t ostride = size_t(kC) * p.heads * p.d_v;
    auto step = [&](int c, const In& in, In& next) {
        Dots<DK, Shape32<DK>::NA> qs;
        qs.zero();
        qs.template mma_state<true>(in.x, in.S);  // O^T: lane (n, g) holds rows 4 g + e of token n
        load(min(c + 1, u.nch - 1), next);
        // P U's first eight tokens apart, as in the state's sum
        const f32x4 z = {0.f, 0.f, 0.f, 0.f};
        f32x4 O = mfma4(in.u[1], in.p[1], mfma4(in.u[0], in.p[0], z));
        const f32x4 so = qs.sum();
#pragma unroll
        for (int e = 0; e < 4; ++e) O[e] = fmaf(so[e], in.gam, O[e]);
        O = mfma4(in.u[3], in.p[3], mfma4(in.u[2], in.p[2], O));
#pragma unroll
        for (int e = 0; e < 4; ++e) watch(finite, O[e]);
        if (u.tb + c * kC + n < u.te && i < p.d_v) *reinterpret_cast<f32x4*>(orow) = O;
        orow += ostride;
        if (c + 1 == u.nch) flag32(sm, !(finite == 0.f));
        period_end();
    };
    In a, b;
    period_end();
    if (period1_leaves(sm)) return;
    period_end();
    load(0, a);
    period_end();
    for (int c = 0; c < u.nch; c += 2) {
        step(c, a, b);
        if (c + 1 < u.nch) step(c + 1, b, a);
    }
}

// The r-th sequence of a pack (from 0) among those of more than short_len
// tokens, or -1.  Called by the whole workgroup; `scratch`, nine ints of LDS,
// is free after the caller's next barrier.
__device__ __forceinline__ int nth_long(const SeqParams& p, int batch, int r, int* scratch) {
    const int l = threadIdx.x & 63, w = threadIdx.x >> 6;
    for (int base = 0; base < batch; base += 512) {
        const int s = base + threadIdx.x;
        bool is_long = false;
        if (s < batch) {
            int t0, t1;
            seq_bounds(p.cu_seqlens, s, p.seq_len, t0, t1);
            is_long = t1 - t0 > short_len(p.d_k);
        }
        const uint64_t m = __builtin_amdgcn_ballot_w64(is_long);
        if (l == 0) scratch[w] = __popcll(m);
        __syncthreads();
        int before = __popcll(m & ((uint64_t(1) << l) - 1)), all = 0;
        for (int i = 0; i < 8; ++i) {
            before += i < w ? scratch[i] : 0;
            all += scratch[i];
        }
        if (is_long && before == r) scratch[8] = s;
        __syncthreads();
        if (r < all) return scratch[8];  // uniform
        r -= all;
    }
    return -1;
}

template <int DK>
__global__ __launch_bounds__(512, 2) void gdr_chunk32_kernel(Chunk32Params cp) {
    __shared__ __align__(16) KernelSmem32<DK> smu;
    Smem32<DK>& sm = smu.chunk;
    const SeqParams& p = cp.sp;
    int unit, tile;
    map_block(cp.first + int(blockIdx.x), cp.units, cp.n_tiles, unit, tile);
    Unit32 u;
    u.seq = unit / p.heads;
    u.h = unit - u.seq * p.heads;
    u.i0 = tile * kRows;
    if (cp.long_only) {
        u.seq = nth_long(p, cp.batch, u.seq, reinterpret_cast<int*>(&smu));
        if (u.seq < 0) return;  // uniform
    }
    seq_bounds(p.cu_seqlens, u.seq, p.seq_len, u.tb, u.te);
    u.nch = (u.te - u.tb + kC - 1) / kC;
    if (u.te - u.tb <= short_len(DK)) {  // uniform
        recurrence32<DK>(p, smu, u.seq, u.h, u.i0);
        return;
    }
    const int l = threadIdx.x & 63;
    const int w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    if (threadIdx.x == 0) sm.rerun = 0;
    period_end();

    // every role passes nch + 4 period ends, or leaves after the second
    if (w < 2)
        scan32<DK>(p, u, sm, w, l);
    else if (w < 4)
        out32<DK>(p, u, sm, w - 2, l);
    else if (w == 4)
        loader32<DK>(p, u, sm, l);
    else if (w == 5)
        loader32<DK>(p, u, sm, 64 + l);
    else if (w == 6)
        TWave<DK>{p, u, sm, l}.run();
    else
        p_wave32<DK>(u, sm, l);

    const int rerun = sm.rerun;
    if (rerun != 0) {  // uniform: set before the last barrier
        __syncthreads();  // every wave has read the flag: the LDS is free
        recurrence32<DK>(p, smu, u.seq, u.h, u.i0);
    }
}

}  // namespace

bool chunk32_supported(const rhz_gdr_prefill_args& a) {
    const auto al16 = [](const void* p) { return (reinterpret_cast<uintptr_t>(p) & 15u) == 0; };
    if (!a.cu_seqlens && a.seq_len <= short_len(a.d_k)) return false;
    // 16-byte accesses throughout, and 32-bit byte offsets within a chunk
    return a.dtype == RHZ_F32 && a.d_k % 4 == 0 && a.d_k <= 128 && a.d_v % 4 == 0 && al16(a.q) && al16(a.k) &&
           al16(a.v) && al16(a.o) && al16(a.initial_state) && al16(a.final_state) &&
           (int64_t)a.heads * (a.d_k > a.d_v ? a.d_k : a.d_v) * 4 * kC <= INT32_MAX;
}

hipError_t launch_chunk32(const rhz_gdr_prefill_args& a, hipStream_t st) {
    Chunk32Params cp{{a.q, a.k, a.v, a.gate, a.beta, a.cu_seqlens, a.initial_state, a.final_state, a.o, a.seq_len,
                      a.heads, a.d_k, a.d_v, a.gate_kind == RHZ_GATE_ALPHA},
                     a.batch, a.batch * a.heads, (a.d_v + kRows - 1) / kRows, 0, 0};
    // A pack of mostly short sequences that more than fills the chip's 256 CUs:
    // the short ones run in the recurrence's own kernel, two or three of whose
    // workgroups share a CU where this kernel's LDS leaves room for one, and the
    // rest here, in as many workgroups as its tokens could need (each finds its
    // sequence by counting; workgroups for every sequence, most of them with
    // nothing to do, took 0.55 us per 256).  H=16 d=64: 1024 sequences of one
    // token 227 us in one launch, 154 with empty workgroups, 87 so; 16 of 64
    // tokens, 512 workgroups, 39 and 26 us in one and two launches, with one of
    // 97 to 99 tokens among them 43 and 45.  A sequence's arithmetic follows from
    // its own length in either case.
    const int len = short_len(a.d_k);
    if (a.cu_seqlens && a.seq_len / a.batch <= len && (int64_t)cp.units * cp.n_tiles > 256) {
        const hipError_t e = launch_staged_short(cp.sp, cp.units, len, st);
        const int most = a.seq_len / (len + 1);
        if (e != hipSuccess || most == 0) return e;
        cp.units = (most < a.batch ? most : a.batch) * a.heads;
        cp.long_only = 1;
    }
    // A grid holds less than 2^32 work-items (the runtime truncates a larger one
    // without an error): whole rounds over the XCDs of as many as fit.
    constexpr int kMost = int(UINT32_MAX / 512) & ~7;
    const int blocks = cp.units * cp.n_tiles;
    hipError_t e = hipSuccess;
    for (int64_t first = 0; first < blocks && e == hipSuccess; first += kMost) {
        cp.first = int(first);
        const dim3 grid(blocks - first > kMost ? kMost : int(blocks - first));
        if (a.d_k <= 32)
            hipLaunchKernelGGL(gdr_chunk32_kernel<32>, grid, dim3(512), 0, st, cp);
        else if (a.d_k <= 64)
            hipLaunchKernelGGL(gdr_chunk32_kernel<64>, grid, dim3(512), 0, st, cp);
        else
            hipLaunchKernelGGL(gdr_chunk32_kernel<128>, grid, dim3(512), 0, st, cp);
        e = hipGetLastError();
    }
    return e;
}

}  // namespace rhz
