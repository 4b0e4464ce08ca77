// Split-precision FP64 GEMM by the Chinese remainder theorem (the integer modular scheme of
// H. Ozaki, Y. Uchino, T. Imamura, "Ozaki Scheme II: A GEMM-oriented emulation of
// floating-point matrix multiplication using an integer modular technique", 2024),
// on the int8 MFMA of gfx950:
//
//   1. Scaling: A'(i,p) = rint(A(i,p) 2^(kb - e_i)) with max_p |A(i,p)| < 2^e_i, and
//      B'(p,j) = rint(B(p,j) 2^(kb - f_j)) per column; |A'|, |B'| <= 2^kb are integers held
//      exactly in FP64 (kb <= 53).
//   2. Residues: for each of the L pairwise coprime moduli m_l <= 256, a_l = A' mod m_l and
//      b_l = B' mod m_l as symmetric representatives, which fit int8.
//   3. One int8 GEMM per modulus, exact in int32 (|a_l b_l| <= 2^14 over at most 65536
//      contraction steps per launch; longer contractions add the residues of several
//      launches): R_l = (a_l b_l) mod m_l in [0, m_l), stored as bytes.
//   4. Reconstruction: S = sum_l R_l W_l with W_l the CRT basis of M = prod m_l, and
//      C' = S - M rint(S / M), the representative in (-M/2, M/2). kb is the largest value
//      with 4 K 2^(2 kb) <= M, so |A'B'| <= M/4 and C' = A'B' exactly. W_l and M are kept in
//      limbs of 40 bits (three, up to 15 moduli) or 32 bits (four, 16 moduli), so every limb
//      sum of S and every limb of S - qM is an exact FP64 integer; the limbs of C' are then
//      added as a double-double (error-free two-sums), which rounds C' once even where its
//      limbs cancel.
//      C = alpha C' 2^(e_i + f_j - 2 kb) + beta C.
//
// Every product of A' and B' is formed exactly, so the only error is the rounding of A
// and B to kb bits relative to their row (column) maximum. The number of moduli sets kb:
// 13 moduli give kb = 44 at K = 2304 and 42 at K = 65536.
//
// Against the 21 products of six int8 slices, L moduli take L int8 GEMMs, each with one
// int32 accumulator per output, where six slices leave room for 128 x 64 tiles only.
//
// The residue planes are stored as the GEMM stages them: blocks of 16 rows by 64 steps, 1024
// consecutive bytes (blocks of a row group along k), so that every DMA instruction reads eight
// whole cache lines. Row-major planes gave it sixteen halves, and at the same bytes twice the
// requests (4096^3, 12 moduli: 1378 -> 1259 us from this alone).
#include <algorithm>
#include <cmath>
#include <string>

#include "ozaki.hpp"
#include "tile_engine.hpp"

namespace ein {

namespace {

constexpr int CRT_MAX_MODS = 16;
// pairwise coprime, descending from 256; the first L are used
constexpr int32_t CRT_MODS[CRT_MAX_MODS] = {256, 255, 253, 251, 247, 241, 239, 233,
                                            229, 227, 223, 211, 199, 197, 193, 191};
constexpr int CRT_FOLD_STAGES = 1024; // stages of one launch, 65536 contraction steps: |int32 sum| <= 2^30

typedef int v4i __attribute__((ext_vector_type(4)));

struct CrtMods {
    int32_t nmod;
    int32_t kbits;
    int32_t mod[CRT_MAX_MODS];
    int32_t c15[CRT_MAX_MODS];    // 2^15 mod m, symmetric
    float finv[CRT_MAX_MODS];     // 1 / m
    double rinv[CRT_MAX_MODS];    // 1 / m
};

// Limbs of M and of the CRT basis: three of 40 bits up to 15 moduli (M < 2^120: a sum of 15
// products of a residue byte and a limb stays below 2^52, an exact FP64 integer), four of 32
// for 16.
constexpr int crt_limbs(int nmod) { return nmod < 16 ? 3 : 4; }
constexpr int crt_limb_bits(int limbs) { return limbs == 3 ? 40 : 32; }

struct CrtBasis {
    int32_t nmod;
    int32_t shift;             // 2 kb
    double w[CRT_MAX_MODS][4]; // W_l in limbs, lowest first
    double mlimb[4];           // M in the same limbs
    double inv_m;              // 1 / M (rounded)
};

// ------------------------------------------------------------------ residues
// 64 x 64 tiles of X staged through LDS so that the read follows X's unit-stride axis. Each
// thread takes four consecutive p of four rows and writes one 32-bit word (four residues) per
// row and modulus into the blocked plane.
// FAST (kb <= 50): with q = rint(x/m) in the low bits of x rinv + 1.5 2^52, the residue's byte
// is the low byte of x - q m = x + q (256 - m) mod 256: one FP64 and one 24-bit operation. The
// product with the rounded 1/m is off by less than 2^(50 - 7.6 - 53) = 2^-10.6, and x/m is at
// least 1/(2m) >= 2^-9 from a tie (m odd; for m = 256 either tie is the same byte), so q is the
// nearest integer. Above 50 bits the quotient may be one off and is corrected. 134 MB of
// operand to 12 moduli: 143 -> 85 us.
template <bool ROWS_FAST, bool FAST>
__global__ __launch_bounds__(256) void crt_residue_kernel(SliceSrc S, int32_t const *__restrict__ e, CrtMods K,
                                                          int8_t *__restrict__ out, int64_t plane) {
    constexpr double ROUND = 0x1.8p52; // x + ROUND: x rounded to an integer, in the low bits
    __shared__ double tile[64][65];
    int64_t const r0 = int64_t(blockIdx.y) * 64;
    int64_t const p0 = int64_t(blockIdx.x) * 64;
    int const t      = threadIdx.x;
    if constexpr (ROWS_FAST) {
        int const lr = t & 63;
#pragma unroll
        for (int q = 0; q < 16; ++q) {
            int lp       = (t >> 6) + 4 * q;
            int64_t r    = r0 + lr, p = p0 + lp;
            tile[lr][lp] = (r < S.rows && p < S.k) ? S.X[r * S.s_row + p * S.s_k] : 0.0;
        }
    } else {
        int const lp = t & 63;
#pragma unroll
        for (int q = 0; q < 16; ++q) {
            int lr       = (t >> 6) + 4 * q;
            int64_t r    = r0 + lr, p = p0 + lp;
            tile[lr][lp] = (r < S.rows && p < S.k) ? S.X[r * S.s_row + p * S.s_k] : 0.0;
        }
    }
    __syncthreads();
    int const p4    = (t & 15) * 4;
    int64_t const p = p0 + p4; // kp is a multiple of 64: p .. p+3 < kp whenever p < kp
    if (p >= S.kp) return;
#pragma unroll 1
    for (int q = 0; q < 4; ++q) {
        int const lr    = (t >> 4) + 16 * q;
        int64_t const r = r0 + lr;
        if (r >= S.rows) continue;
        int const sh = K.kbits - e[r];
        double x[4];
        uint32_t xl[4]; // x mod 2^32
#pragma unroll
        for (int u = 0; u < 4; ++u) {
            x[u]  = rint(ldexp(tile[lr][p4 + u], sh)); // |x| <= 2^kb, exact
            xl[u] = FAST ? uint32_t(__double2loint(x[u] + ROUND)) : 0u;
        }
        int8_t *__restrict__ dst = out + (r >> 4) * 16 * S.kp + (p0 >> 6) * 1024 + (r & 15) * 64 + p4;
        if constexpr (FAST) {
#pragma unroll 4
            for (int l = 0; l < K.nmod; ++l) {
                uint32_t b[4];
#pragma unroll
                for (int u = 0; u < 4; ++u)
                    b[u] = __umul24(uint32_t(__double2loint(fma(x[u], K.rinv[l], ROUND))), uint32_t(256 - K.mod[l])) + xl[u];
                uint32_t const lo = __builtin_amdgcn_perm(b[1], b[0], 0x0c0c0400u), hi = __builtin_amdgcn_perm(b[3], b[2], 0x04000c0cu);
                *reinterpret_cast<uint32_t *>(dst + int64_t(l) * plane) = lo | hi;
            }
        } else {
#pragma unroll 1
            for (int l = 0; l < K.nmod; ++l) {
                double const m  = double(K.mod[l]);
                double const hi = K.mod[l] == 256 ? 127.0 : 0.5 * (m - 1.0);
                double const lo = K.mod[l] == 256 ? -128.0 : -hi;
                uint32_t word   = 0;
#pragma unroll
                for (int u = 0; u < 4; ++u) {
                    double v = fma(-rint(x[u] * K.rinv[l]), m, x[u]); // x - m*q: an exact small integer
                    v        = v > hi ? v - m : v;
                    v        = v < lo ? v + m : v;
                    word |= uint32_t(uint8_t(int8_t(v))) << (8 * u);
                }
                *reinterpret_cast<uint32_t *>(dst + int64_t(l) * plane) = word;
            }
        }
    }
}

// ------------------------------------------------------------- residue GEMM
// R_l(j, i) = (sum_p a_l(i,p) b_l(j,p)) mod m_l for all moduli in one launch, as a byte in
// [0, m_l].
constexpr int CG_TI = 256, CG_TJ = 128, CG_KS = 64, CG_NBUF = 3, CG_WAVES = 4;
constexpr int CG_SA = CG_TI * 4, CG_SB = CG_TJ * 4;   // 16-byte chunks per operand stage
constexpr int CG_DA = CG_SA / 64 / CG_WAVES, CG_DB = CG_SB / 64 / CG_WAVES; // DMA instructions per wave and stage

struct CrtGemm {
    int64_t n, kp;            // rows of b (j, this panel), padded contraction length
    int64_t k0, kc;           // contraction steps [k0, k0 + kc) of this launch (multiples of 64)
    int32_t accumulate;       // add to the stored residues instead of overwriting them
    uint32_t items;           // (modulus, tile) pairs
    int64_t a_plane, b_plane; // elements between the moduli of the residue operands
    int8_t const *A;
    int8_t const *B;
    uint8_t *R; // [l][j][i], i fastest
    int64_t ldr, r_plane;
    uint32_t tiles_m, tiles_n;
    CrtMods K;
};

// 16-byte chunk c of row `row` of an operand sits at slot row*4 + (c ^ f(row)); f puts the 16
// rows of one fragment read (see the kernel) on distinct 16-byte bank groups.
template <bool A>
__device__ __forceinline__ int cg_swz(int row) { return A ? (row >> 5) & 3 : (row >> 2) & 3; }

// Workgroup barrier that no memory access of the code is moved across.
__device__ __forceinline__ void cg_barrier() {
    asm volatile("" ::: "memory");
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
}

// One operand stage: lane l of instruction n = wave + 4x fills slot 64n + l, i.e. chunk l % 4
// (swizzled) of row 16n + l / 4, out of block n of the stage. `tile` is the tile's first block,
// `off` the lane's offset for x = 0; the swizzle of A moves the chunk by two for odd x. Rows
// beyond the operand are whatever follows in the workspace: they only reach outputs that are
// not stored, or lie in the padding of R.
template <bool A, int N>
__device__ __forceinline__ void cg_dma(int8_t const *__restrict__ tile, int64_t kp, int64_t off, int8_t *lds, int wave) {
#pragma unroll
    for (int x = 0; x < N; ++x) {
        int8_t const *src = tile + 64 * x * kp + (A && (x & 1) ? off ^ 32 : off);
        __builtin_amdgcn_global_load_lds(src, EIN_LDS_PTR(lds + (wave + CG_WAVES * x) * 64 * 16), 16, 0, 0);
    }
}

// Persistent: two workgroups per CU, each walking every grid-th (modulus, 256 x 128 tile), four
// waves of 128 x 64, 8 x 4 blocks of the 16 x 16 x 64 int8 MFMA. 64-step operand stages go
// global -> LDS by DMA through a ring of three buffers. While a stage's 32 MFMAs run from
// registers, the next stage's fragments are read and the DMA of the one three ahead is issued
// into the buffer just read; one barrier a stage. The next item's first stages are in flight
// during the epilogue.
// At k = 1024 a tile has 16 stages, about as long as its epilogue (the reduction of 128
// accumulators a lane), so what matters is that the other workgroup's MFMAs run meanwhile: one
// 256 x 256 tile per CU in lockstep took 5214 us for 16384^2 x 1024, 12 moduli (MFMA busy 26%
// of 12.0M cycles at 2.19 GHz), this 4108 (42% of 7.5M cycles at 1.79 GHz: it is now the power
// limit that sets the clock). 4096^3 in all 1339 -> 1057 us, 2304^2 x 65536 9.32 -> 7.53 ms.
//
// Row 16a + r of a wave's A fragment a is row (r/4)*32 + 4a + r%4 of its 128: with that order
// a lane's results of one column are 32 consecutive bytes of R, two 16-byte stores.
// The reduction mod m: x = 2^15 hi + lo -> hi (2^15 mod m) + lo, below 2^23 in magnitude and
// exact in 24-bit integer arithmetic and FP32; then y - m floor(y / m), whose floor is right or,
// at a multiple of m, one low, which stores m for 0: the same residue, and m <= 255 (for 256
// the division is exact) still fits the byte.
// The contraction is at most CRT_FOLD_STAGES stages (|int32 sum| <= 2^30); longer ones run
// as several launches with `accumulate` set, each adding its residues to the stored ones.
__global__ __launch_bounds__(64 * CG_WAVES, 2) void crt_gemm_kernel(CrtGemm P) {
    __shared__ __attribute__((aligned(16))) int8_t lds[CG_NBUF * (CG_SA + CG_SB) * 16];

    int const tid  = threadIdx.x;
    int const lane = tid & 63;
    int const wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    int const wm   = wave & 1;
    int const wn   = wave >> 1;
    int const r    = lane & 15;
    int const q    = lane >> 4;
    // fragment slots of this lane: A row (r/4)*32 + 4a + r%4 of the wave's 128, B row 16b + r
    int const a_row = wm * 128 + (r >> 2) * 32 + (r & 3);
    int const a_sl  = a_row * 4 + (q ^ cg_swz<true>(a_row)); // + 16 a: the swizzle depends on r/4 only
    int const b_row = wn * 64 + r;
    int const b_sl  = CG_SA + b_row * 4 + (q ^ cg_swz<false>(b_row)); // + 64 b

    uint32_t const ntiles = P.tiles_m * P.tiles_n;
    int64_t const nst     = P.kc / CG_KS;
    auto buf = [&](int z) { return lds + z * ((CG_SA + CG_SB) * 16); };
    struct Item {
        int8_t const *A, *B;
        int64_t i0, j0;
        uint32_t l;
    };
    auto item_of = [&](uint32_t it) {
        Item x;
        x.l                 = it / ntiles;
        uint32_t const tile = it - x.l * ntiles;
        uint32_t tm, tn;
        tile_coords(tile, P.tiles_m, P.tiles_n, tm, tn);
        x.i0 = int64_t(tm) * CG_TI;
        x.j0 = int64_t(tn) * CG_TJ;
        x.A  = P.A + int64_t(x.l) * P.a_plane + P.k0 * 16 + x.i0 * P.kp;
        x.B  = P.B + int64_t(x.l) * P.b_plane + P.k0 * 16 + x.j0 * P.kp;
        return x;
    };
    int const d_row     = wave * 16 + (lane >> 2);
    int64_t const a_off = wave * 16 * P.kp + (lane >> 2) * 64 + 16 * ((lane & 3) ^ cg_swz<true>(d_row));
    int64_t const b_off = wave * 16 * P.kp + (lane >> 2) * 64 + 16 * ((lane & 3) ^ cg_swz<false>(d_row));
    auto dma = [&](Item const &x, int64_t s, int z) {
        int8_t *dst = buf(z);
        cg_dma<true, CG_DA>(x.A + s * 1024, P.kp, a_off, dst, wave);
        cg_dma<false, CG_DB>(x.B + s * 1024, P.kp, b_off, dst + CG_SA * 16, wave);
    };
    uint32_t it = xcd_remap(blockIdx.x, gridDim.x);
    if (it >= P.items) return;
    Item cur = item_of(it);
    for (int s = 0; s < CG_NBUF && s < nst; ++s) dma(cur, s, s);

    for (;;) {
        v4i acc[8][4];
#pragma unroll
        for (int a = 0; a < 8; ++a)
#pragma unroll
            for (int b = 0; b < 4; ++b) acc[a][b] = v4i{0, 0, 0, 0};
        v4i fa[2][8], fb[2][4];
        auto frags = [&](int8_t const *__restrict__ st, v4i (&xa)[8], v4i (&xb)[4]) {
            v4i const *p = reinterpret_cast<v4i const *>(st);
#pragma unroll
            for (int a = 0; a < 8; ++a) xa[a] = p[a_sl + 16 * a];
#pragma unroll
            for (int b = 0; b < 4; ++b) xb[b] = p[b_sl + 64 * b];
        };
        // the first stage (and the last item's stores)
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
        cg_barrier();
        frags(buf(0), fa[0], fb[0]);
        int z = 0; // buffer of stage s
        auto stage = [&](int64_t s, v4i (&xa)[8], v4i (&xb)[4], v4i (&ya)[8], v4i (&yb)[4]) {
            int const z1 = z == CG_NBUF - 1 ? 0 : z + 1;
            if (s + 1 < nst) {
                // stage s+2 may stay in flight (the item's first three were waited for)
                static_assert(CG_DA + CG_DB == 6 && CG_NBUF == 3, "the vmcnt below");
                if (s + 2 < nst && s > 0)
                    asm volatile("s_waitcnt vmcnt(6) lgkmcnt(0)" ::: "memory");
                else
                    asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)" ::: "memory");
                cg_barrier(); // stage s+1 is there, and every wave has read stage s
                if (s + 3 < nst) dma(cur, s + 3, z);
                frags(buf(z1), ya, yb);
            }
            z = z1;
#pragma unroll
            for (int a = 0; a < 8; ++a)
#pragma unroll
                for (int b = 0; b < 4; ++b) acc[a][b] = __builtin_amdgcn_mfma_i32_16x16x64_i8(xa[a], xb[b], acc[a][b], 0, 0, 0);
        };
        for (int64_t s = 0; s < nst; s += 2) {
            stage(s, fa[0], fb[0], fa[1], fb[1]);
            if (s + 1 < nst) stage(s + 1, fa[1], fb[1], fa[0], fb[0]);
        }
        // every wave has read its last fragments: the ring is free for the next item
        uint32_t const nx = it + gridDim.x;
        Item next         = cur;
        asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
        cg_barrier();
        if (nx < P.items) {
            next = item_of(nx);
            for (int s = 0; s < CG_NBUF && s < nst; ++s) dma(next, s, s);
        }
        // D[4q+v][r] of block (a, b): i = wm*128 + 32q + 4a + v, j = wn*128 + 16b + r: a lane's
        // 32 consecutive bytes of column j
        float const m    = float(P.K.mod[cur.l]);
        float const inv  = P.K.finv[cur.l];
        int const c15    = P.K.c15[cur.l];
        uint8_t *__restrict__ Rl = P.R + int64_t(cur.l) * P.r_plane + cur.i0 + wm * 128 + q * 32;
#pragma unroll
        for (int b = 0; b < 4; ++b) {
            int64_t const j = cur.j0 + wn * 64 + b * 16 + r;
            if (j >= P.n) continue;
            v4i *dst = reinterpret_cast<v4i *>(Rl + j * P.ldr);
            v4i out[2];
#pragma unroll
            for (int a = 0; a < 8; ++a) {
                uint32_t word = 0;
#pragma unroll
                for (int v = 0; v < 4; ++v) {
                    int const x = acc[a][b][v];
                    float const y = float(__mul24(x >> 15, c15) + (x & 0x7fff)); // exact: below 2^23
                    float const t = fmaf(-floorf(y * inv), m, y);                // in [0, m]
                    word = __builtin_amdgcn_cvt_pk_u8_f32(t, v, word);
                }
                out[a >> 2][a & 3] = int(word);
            }
            if (P.accumulate) {
#pragma unroll
                for (int h = 0; h < 2; ++h) {
                    v4i const old = dst[h];
#pragma unroll
                    for (int w = 0; w < 4; ++w) {
                        uint32_t const o = uint32_t(old[w]), n = uint32_t(out[h][w]);
                        uint32_t word = 0;
#pragma unroll
                        for (int v = 0; v < 4; ++v) {
                            uint32_t x = ((o >> (8 * v)) & 0xffu) + ((n >> (8 * v)) & 0xffu);
                            x = x >= uint32_t(P.K.mod[cur.l]) ? x - uint32_t(P.K.mod[cur.l]) : x;
                            x = x >= uint32_t(P.K.mod[cur.l]) ? x - uint32_t(P.K.mod[cur.l]) : x;
                            word |= x << (8 * v);
                        }
                        out[h][w] = int(word);
                    }
                }
            }
            dst[0] = out[0];
            dst[1] = out[1];
        }
        if (nx >= P.items) break;
        it  = nx;
        cur = next;
    }
}

// ------------------------------------------------------------ reconstruction
// C(i,j) = alpha 2^(e_i + f_j - 2kb) C'(i,j) + beta C(i,j) for the panel's columns; each
// thread takes four consecutive i of one column (one 32-bit word of every residue plane).
struct CrtRec {
    int64_t m, n;                     // rows, panel columns
    uint8_t const *R;                 // [l][j][i]
    int64_t ldr, r_plane;
    int32_t const *ea, *eb;           // eb already offset to the panel
    double *C;                        // offset to the panel
    int64_t c_sm, c_sn;
    double alpha, beta;
    CrtBasis W;
};

// a + b = s + e exactly (Knuth's two-sum)
__device__ __forceinline__ double two_sum(double a, double b, double &e) {
    double const s  = a + b;
    double const bb = s - a;
    e               = (a - (s - bb)) + (b - bb);
    return s;
}

// Bytes 0..3 of a word as doubles: the byte under the exponent of 2^52, minus 2^52 (two
// full-rate operations, against a quarter-rate conversion).
__device__ __forceinline__ double byte_to_double(uint32_t word, int v) {
    return __hiloint2double(0x43300000, int((word >> (8 * v)) & 0xffu)) - 0x1p52;
}

// HBM-bound: L bytes of residues and 8 or 16 of C per element. All residue words and C are
// requested before the arithmetic, C moves as 16-byte vectors where it can, three 40-bit limbs
// take a quarter fewer products than four of 32 bits. 16384^2, 12 moduli, beta = 1 (7.5 GB):
// 1935 -> 1468 us (5.1 TB/s).
template <int NL, bool VEC>
__global__ __launch_bounds__(256) void crt_reconstruct_kernel(CrtRec P) {
    constexpr double B1 = NL == 3 ? 0x1p40 : 0x1p32, B2 = B1 * B1, B3 = B2 * B1;
    int64_t const words = P.ldr / 4;
    int64_t const g     = int64_t(blockIdx.x) * 256 + threadIdx.x;
    int64_t const j     = g / words;
    int64_t const i     = (g - j * words) * 4;
    if (j >= P.n || i >= P.m) return;
    uint8_t const *__restrict__ src = P.R + j * P.ldr + i;
    double *const c                 = P.C + i * P.c_sm + j * P.c_sn;
    // all reads first
    uint32_t word[CRT_MAX_MODS];
#pragma unroll
    for (int l = 0; l < CRT_MAX_MODS; ++l)
        if (l < P.W.nmod) word[l] = *reinterpret_cast<uint32_t const *>(src + int64_t(l) * P.r_plane);
    double old[4] = {0.0, 0.0, 0.0, 0.0};
    bool const whole = i + 4 <= P.m;
    if (P.beta != 0.0) {
        if (VEC && whole) {
#pragma unroll
            for (int h = 0; h < 2; ++h) {
                double2 const t = *reinterpret_cast<double2 const *>(c + 2 * h);
                old[2 * h]      = t.x;
                old[2 * h + 1]  = t.y;
            }
        } else {
#pragma unroll
            for (int v = 0; v < 4; ++v)
                if (i + v < P.m) old[v] = c[v * P.c_sm];
        }
    }
    double s[4][NL];
#pragma unroll
    for (int v = 0; v < 4; ++v)
#pragma unroll
        for (int t = 0; t < NL; ++t) s[v][t] = 0.0;
#pragma unroll
    for (int l = 0; l < CRT_MAX_MODS; ++l)
        if (l < P.W.nmod) {
#pragma unroll
            for (int v = 0; v < 4; ++v) {
                double const rv = byte_to_double(word[l], v);
#pragma unroll
                for (int t = 0; t < NL; ++t) s[v][t] = fma(rv, P.W.w[l][t], s[v][t]); // exact
            }
        }
    int const eb = P.eb[j];
    double val[4];
#pragma unroll
    for (int v = 0; v < 4; ++v) {
        double approx = fma(s[v][2], B2, fma(s[v][1], B1, s[v][0]));
        if constexpr (NL == 4) approx = fma(s[v][NL - 1], B3, approx);
        double const qm = rint(approx * P.W.inv_m); // S / M rounded: |C'| <= M/4 leaves margin
        double lim[NL];
#pragma unroll
        for (int t = 0; t < NL; ++t) lim[t] = fma(-qm, P.W.mlimb[t], s[v][t]); // exact limbs of S - qM
        double e0, e1, e2 = 0.0;
        double h = two_sum(lim[1] * B1, lim[0], e0);
        h        = two_sum(lim[2] * B2, h, e1);
        if constexpr (NL == 4) h = two_sum(lim[NL - 1] * B3, h, e2);
        double const cp = h + ((e0 + e1) + e2);
        int const e     = i + v < P.m ? P.ea[i + v] : 0;
        val[v]          = P.alpha * ldexp(cp, e + eb - P.W.shift);
        if (P.beta != 0.0) val[v] = fma(P.beta, old[v], val[v]);
    }
    if (VEC && whole) {
#pragma unroll
        for (int h = 0; h < 2; ++h) *reinterpret_cast<double2 *>(c + 2 * h) = double2{val[2 * h], val[2 * h + 1]};
    } else {
#pragma unroll
        for (int v = 0; v < 4; ++v)
            if (i + v < P.m) c[v * P.c_sm] = val[v];
    }
}

// ------------------------------------------------------------------- host
typedef unsigned __int128 u128;

int crt_kbits(int nmod, int64_t k) {
    u128 M = 1;
    for (int l = 0; l < nmod; ++l) M *= u128(CRT_MODS[l]);
    int kb = 0;
    // largest kb with 4 k 2^(2 kb) <= M, at most 53 (A' must stay an exact FP64 integer)
    while (kb < 53) {
        int const sh = 2 * (kb + 1) + 2;
        u128 const need = u128(uint64_t(k)) << sh;
        if (sh >= 126 || (need >> sh) != u128(uint64_t(k)) || need > M) break;
        ++kb;
    }
    return kb;
}

void crt_constants(int nmod, int kbits, CrtMods &K, CrtBasis &W) {
    K       = CrtMods{};
    W       = CrtBasis{};
    K.nmod  = nmod;
    K.kbits = kbits;
    W.nmod  = nmod;
    W.shift = 2 * kbits;
    u128 M  = 1;
    for (int l = 0; l < nmod; ++l) M *= u128(CRT_MODS[l]);
    int const nl = crt_limbs(nmod), bits = crt_limb_bits(nl);
    auto limbs = [&](u128 x, double *out) {
        for (int t = 0; t < nl; ++t) out[t] = double(uint64_t(x >> (bits * t)) & ((uint64_t(1) << bits) - 1));
    };
    for (int l = 0; l < nmod; ++l) {
        uint32_t const m = uint32_t(CRT_MODS[l]);
        K.mod[l]         = int32_t(m);
        int32_t const c  = int32_t((1u << 15) % m);
        K.c15[l]         = 2 * c > int32_t(m) ? c - int32_t(m) : c;
        K.finv[l]        = 1.0f / float(m);
        K.rinv[l]        = 1.0 / double(m);
        u128 const Mi    = M / m;
        // inverse of Mi mod m by search (m <= 256)
        uint32_t const mi = uint32_t(Mi % m);
        uint32_t inv      = 0;
        for (uint32_t x = 1; x < m; ++x)
            if ((mi * x) % m == 1) {
                inv = x;
                break;
            }
        limbs(Mi * inv % M, W.w[l]); // W_l = Mi * (Mi^-1 mod m) < M
    }
    limbs(M, W.mlimb);
    W.inv_m = 1.0 / (double(uint64_t(M >> 64)) * 0x1p64 + double(uint64_t(M)));
}

int crt_residues(SliceSrc const &S, CrtMods const &K, int32_t *e, int8_t *out, int64_t plane, double *scratch,
                 hipStream_t stream) {
    bool const rows_fast = S.s_row == 1 || (S.s_k != 1 && std::llabs(S.s_row) < std::llabs(S.s_k));
    EIN_TRY(row_exponents(S, e, false, scratch, stream));
    dim3 grid{uint32_t(ceil_div(S.kp, 64)), uint32_t(ceil_div(S.rows, 64))};
    if (grid.y > 65535) return fail(EIN_ERROR_UNSUPPORTED, "split gemm: more than 4M rows");
    bool const fast   = K.kbits <= 50;
    auto const kernel = rows_fast ? (fast ? crt_residue_kernel<true, true> : crt_residue_kernel<true, false>)
                                  : (fast ? crt_residue_kernel<false, true> : crt_residue_kernel<false, false>);
    kernel<<<grid, 256, 0, stream>>>(S, e, K, out, plane);
    EIN_LAUNCH_CHECK();
    return EIN_SUCCESS;
}

} // namespace

// Residue planes are written for column panels of at most this many bytes, each reconstructed
// before the next is formed. On a side stream, beside the next panel's residue GEMM, the
// reconstruction takes CUs from workgroups that each own a fixed share of the panel:
// 65536^2 x 2304 (12 moduli) 174.8 ms, in order 142.3; 49152^2 93.7 and 79.2; panels of 8 GiB
// 142.5 and 79.9.
constexpr size_t CRT_PANEL_BYTES = size_t(4) << 30;

int gemm_split_crt(GemmProblem<double> P, int nmod, hipStream_t stream) {
    if (nmod < CRT_MIN_MODULI || nmod > CRT_MAX_MODS)
        return fail(EIN_ERROR_VALUE, "split gemm: the CRT scheme takes " + std::to_string(CRT_MIN_MODULI) + ".." +
                                         std::to_string(CRT_MAX_MODS) + " moduli");
    int64_t const kp     = ceil_div(P.k, CG_KS) * CG_KS;
    int const kbits      = crt_kbits(nmod, P.k);
    if (kbits < 8) return fail(EIN_ERROR_UNSUPPORTED, "split gemm: contraction too long for the CRT scheme");
    CrtMods K;
    CrtBasis W;
    crt_constants(nmod, kbits, K, W);

    uint32_t const tiles_m = uint32_t(ceil_div(P.m, CG_TI));
    int64_t const ldr      = int64_t(tiles_m) * CG_TI;
    // column panels of whole 256-column tiles whose residue planes take at most CRT_PANEL_BYTES
    int64_t pn = int64_t(CRT_PANEL_BYTES / (size_t(nmod) * size_t(ldr))) / CG_TI * CG_TI;
    pn         = std::max<int64_t>(CG_TI, std::min<int64_t>(pn, ceil_div(P.n, CG_TI) * CG_TI));

    int64_t const a_plane = ceil_div(P.m, 16) * 16 * kp, b_plane = ceil_div(P.n, 16) * 16 * kp;
    size_t const a_bytes = size_t(nmod) * size_t(a_plane);
    size_t const b_bytes = size_t(nmod) * size_t(b_plane);
    size_t const r_bytes = size_t(nmod) * size_t(pn) * size_t(ldr);
    auto up              = [](size_t x) { return (x + 255) / 256 * 256; };
    size_t const b_off   = up(a_bytes);
    size_t const r_off   = b_off + up(b_bytes);
    size_t const ea_off  = r_off + up(r_bytes);
    size_t const eb_off  = ea_off + up(size_t(P.m) * 4);
    size_t const x_off   = eb_off + up(size_t(P.n) * 4);
    // the GEMM's tiles read up to CG_TI rows past the last plane of an operand
    size_t const total   = std::max(x_off + row_exp_scratch(std::max(P.m, P.n)) * sizeof(double),
                                    r_off + size_t(CG_TI) * size_t(kp));
    void *ws             = nullptr;
    EIN_TRY(workspace(stream, total, &ws));
    char *base      = static_cast<char *>(ws);
    int8_t *As      = reinterpret_cast<int8_t *>(base);
    int8_t *Bs      = reinterpret_cast<int8_t *>(base + b_off);
    uint8_t *R      = reinterpret_cast<uint8_t *>(base + r_off);
    int32_t *ea     = reinterpret_cast<int32_t *>(base + ea_off);
    int32_t *eb     = reinterpret_cast<int32_t *>(base + eb_off);
    double *scratch = reinterpret_cast<double *>(base + x_off);

    SliceSrc SA{P.m, P.k, kp, P.A, P.a_sm, P.a_sk};
    SliceSrc SB{P.n, P.k, kp, P.B, P.b_sn, P.b_sk};
    EIN_TRY(crt_residues(SA, K, ea, As, a_plane, scratch, stream));
    EIN_TRY(crt_residues(SB, K, eb, Bs, b_plane, scratch, stream));

    for (int64_t j0 = 0; j0 < P.n; j0 += pn) {
        int64_t const nj = std::min(pn, P.n - j0);
        CrtGemm G{};
        G.n       = nj;
        G.kp      = kp;
        G.a_plane = a_plane;
        G.b_plane = b_plane;
        G.A       = As;
        G.B       = Bs + j0 * kp;
        G.R       = R;
        G.ldr     = ldr;
        G.r_plane = nj * ldr;
        G.tiles_m = tiles_m;
        G.tiles_n = uint32_t(ceil_div(nj, CG_TJ));
        G.K       = K;
        uint64_t const grid = uint64_t(G.tiles_m) * G.tiles_n * uint64_t(nmod);
        if (grid > 0x7fffffffu) return fail(EIN_ERROR_UNSUPPORTED, "split gemm: tile grid too large");
        for (int64_t k0 = 0; k0 < kp; k0 += int64_t(CRT_FOLD_STAGES) * CG_KS) {
            G.k0         = k0;
            G.kc         = std::min<int64_t>(int64_t(CRT_FOLD_STAGES) * CG_KS, kp - k0);
            G.accumulate = k0 > 0;
            G.items      = uint32_t(grid);
            crt_gemm_kernel<<<uint32_t(std::min<uint64_t>(grid, 2 * uint64_t(num_cus()))), 64 * CG_WAVES, 0, stream>>>(
                G);
            EIN_LAUNCH_CHECK();
        }

        CrtRec Q{};
        Q.m       = P.m;
        Q.n       = nj;
        Q.R       = R;
        Q.ldr     = ldr;
        Q.r_plane = nj * ldr;
        Q.ea      = ea;
        Q.eb      = eb + j0;
        Q.C       = P.C + j0 * P.c_sn;
        Q.c_sm    = P.c_sm;
        Q.c_sn    = P.c_sn;
        Q.alpha   = P.alpha;
        Q.beta    = P.beta;
        Q.W       = W;
        int64_t const threads = nj * (ldr / 4);
        if (ceil_div(threads, 256) > 0x7fffffff) return fail(EIN_ERROR_UNSUPPORTED, "split gemm: panel too large");
        bool const vec = Q.c_sm == 1 && Q.c_sn % 2 == 0 && reinterpret_cast<uintptr_t>(Q.C) % 16 == 0;
        auto const rec = crt_limbs(nmod) == 3 ? (vec ? crt_reconstruct_kernel<3, true> : crt_reconstruct_kernel<3, false>)
                                              : (vec ? crt_reconstruct_kernel<4, true> : crt_reconstruct_kernel<4, false>);
        rec<<<uint32_t(ceil_div(threads, 256)), 256, 0, stream>>>(Q);
        EIN_LAUNCH_CHECK();
    }
    return EIN_SUCCESS;
}

int crt_bits(int nmod, int64_t k) {
    if (nmod < CRT_MIN_MODULI || nmod > CRT_MAX_MODS || k < 0) return -1;
    return crt_kbits(nmod, std::max<int64_t>(k, 1));
}

int crt_auto_moduli(int64_t k) {
    for (int L = CRT_MIN_MODULI; L < CRT_MAX_MODS; ++L)
        if (crt_kbits(L, std::max<int64_t>(k, 1)) >= CRT_AUTO_BITS) return L;
    return CRT_MAX_MODS;
}

} // namespace ein

extern "C" {

int ein_split_crt_bits(int32_t nmoduli, int64_t k) {
    if (nmoduli == 0 && k >= 0) nmoduli = ein::crt_auto_moduli(k);
    return ein::crt_bits(nmoduli, k);
}

int ein_split_crt_moduli(int64_t k) { return k < 0 ? -1 : ein::crt_auto_moduli(k); }

} // extern "C"
