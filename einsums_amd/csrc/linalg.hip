// Dense symmetric eigensolver and LU solve for the small matrices of the SCF loop around the
// einsum path (Fock matrices of nbf x nbf, DIIS systems of a few dozen unknowns), so that a
// whole SCF iteration stays on the device and can be captured in a graph. Both run on one
// 1024-thread workgroup and report LAPACK's `info` in device memory instead of returning it,
// which keeps the calls asynchronous.
//
// Reference interfaces (paths relative to the Einsums source tree):
//   syev: blas::syev(job, uplo, n, a, lda, w, work, lwork)  libs/Einsums/BLAS/include/Einsums/BLAS.hpp:306
//         linear_algebra::syev(&A, &W)                      libs/Einsums/LinearAlgebra/include/Einsums/LinearAlgebra.hpp:362
//   gesv: blas::gesv(n, nrhs, a, lda, ipiv, b, ldb)         libs/Einsums/BLAS/include/Einsums/BLAS.hpp:529
//         linear_algebra::gesv(&A, &B)                      libs/Einsums/LinearAlgebra/include/Einsums/LinearAlgebra.hpp:495
// used by the reference HF/DIIS test, libs/Einsums/TensorAlgebra/tests/unit/QChemTests.cpp:157,266,312.
//
// syev: cyclic two-sided Jacobi (Golub & Van Loan, Matrix Computations, 4th ed., 8.5: the
// symmetric Schur decomposition of each 2x2 block, Algorithm 8.5.1) with the round-robin
// ordering of Brent and Luk, so every step rotates n/2 disjoint planes at once. A sweep is
// n-1 steps; the loop stops once the off-diagonal Frobenius norm is below n*eps times that of
// A (converged), or after 60 sweeps (info = 1). Eigenvalues come out ascending, eigenvectors
// as the columns of A, as from LAPACK dsyev.
// gesv: right-looking LU with partial pivoting (the first largest magnitude in the column, as
// LAPACK's idamax picks), then unit-lower and upper triangular solves of B; ipiv is 1-based.
#include <cmath>
#include <type_traits>

#include "ein_common.hpp"

namespace ein {

namespace {

constexpr int LA_THREADS = 1024;
constexpr int LA_WAVES   = LA_THREADS / 64;
constexpr int SYEV_MAX_N = 1024; // n/2 rotation pairs held in LDS
constexpr int GESV_MAX_N = 4096;
constexpr int SYEV_MAX_SWEEPS = 60;

// LDS for the matrices of a solve above n = 64: M, or M and V.
constexpr int SYEV_LDS_BYTES = 160000;
template <typename T>
constexpr int SYEV_LDS_ELEMS = SYEV_LDS_BYTES / int(sizeof(T));

// 1/sqrt(x) for x in (0, 4]: the hardware estimate and one third-order step,
// y + y (e/2 + 3 e^2/8) with e = 1 - x y^2, which leaves rounding only (the estimates are
// good to 2^-22 and better). A divide and a square root by the library's sequences take
// about four times as long, and the rotations are on the solver's critical path.
__device__ __forceinline__ double rsqrt_step(double x) {
    double const y = __builtin_amdgcn_rsq(x);
    double const e = fma(-x * y, y, 1.0);
    return fma(y * e, fma(0.375, e, 0.5), y);
}
__device__ __forceinline__ float rsqrt_step(float x) {
    float const y = __builtin_amdgcn_rsqf(x);
    float const e = fmaf(-x * y, y, 1.0f);
    return fmaf(y * e, fmaf(0.375f, e, 0.5f), y);
}

// Jacobi rotation (c, s) that diagonalises [[app, apq], [apq, aqq]], t = s/c the smaller root
// of t^2 + (aqq - app)/apq t - 1 = 0, from the double angle: with h = 2 apq, d = aqq - app,
// cos 2a = |d| / sqrt(d^2 + h^2) and sin 2a = sign(d) h / sqrt(d^2 + h^2) give
// c = sqrt((1 + cos 2a) / 2), s = sin 2a / (2 c). A common power-of-two scaling first, so
// that the squares neither overflow nor vanish.
template <typename T>
__device__ __forceinline__ void jacobi_rotation(T app, T aqq, T apq, T &c, T &s, T &t) {
    c = T(1);
    s = t = T(0);
    if (apq == T(0)) return;
    T d = aqq - app, h = T(2) * apq;
    int e;
    (void)frexp(fmax(fabs(d), fabs(h)), &e);
    d            = ldexp(d, -e);
    h            = ldexp(h, -e);
    T const inv  = rsqrt_step(fma(d, d, h * h)); // the sum is in [1/4, 2)
    T const cc   = fma(T(0.5) * fabs(d), inv, T(0.5));
    T const rc   = rsqrt_step(cc);
    T const half = T(0.5) * (d >= T(0) ? h : -h) * inv;
    c            = cc * rc;
    s            = half * rc;
    t            = s * rc;
}

// Upper triangle, packed: element (i, j) of the symmetric matrix.
__host__ __device__ __forceinline__ int tri(int i, int j) {
    int const lo = i < j ? i : j, hi = i < j ? j : i;
    return lo + hi * (hi + 1) / 2;
}

// The convergence norm is a sum of squares, which leaves the range of the type long before the
// entries do (FP32: near 1e19 and 1e-19). Where `fro`, the sum over the packed triangle M of
// order m, or n^2 eps^2 times it would, M is scaled so that its largest entry is in [1/2, 1), and
// `fro` is formed again. Powers of two scale exactly and the rotations do not depend on them;
// returns the exponent by which the eigenvalues are scaled back. With an infinite entry no scale
// helps: `fro` stays infinite.
template <typename T, typename Sum>
__device__ __forceinline__ int bring_into_range(T *M, int m, T *red, Sum const &sum, T &fro) {
    constexpr T LEAST = sizeof(T) == 8 ? T(1e-200) : T(1e-20), MOST = sizeof(T) == 8 ? T(1e300) : T(1e37);
    // the same in every lane; the compiler has to know, or the sweeps' scalar state goes to vectors
    auto uniform = [](bool x) { return __builtin_amdgcn_readfirstlane(int(x)) != 0; };
    if (__builtin_expect(uniform(fro >= LEAST && fro <= MOST), 1)) return 0;
    int const lane = threadIdx.x & 63, wave = threadIdx.x >> 6, waves = blockDim.x >> 6;
    T big = T(0);
    for (int x = threadIdx.x; x < m * (m + 1) / 2; x += blockDim.x) big = fmax(big, fabs(M[x]));
#pragma unroll
    for (int o = 32; o >= 1; o >>= 1) big = fmax(big, __shfl_xor(big, o, 64));
    __syncthreads();
    if (lane == 0) red[wave] = big;
    __syncthreads();
    for (int i = 0; i < waves; ++i) big = fmax(big, red[i]);
    if (uniform(!(big > T(0)) || isinf(big))) return 0;
    int e;
    (void)frexp(big, &e);
    T f = T(0);
    for (int j = wave; j < m; j += waves)
        for (int i = lane; i <= j; i += 64) {
            T const v    = ldexp(M[tri(i, j)], -e);
            M[tri(i, j)] = v;
            f += i == j ? v * v : T(2) * v * v;
        }
    fro = sum(f);
    return __builtin_amdgcn_readfirstlane(e);
}

// Jacobi for n <= 64 with M and V in LDS, on one workgroup. What bounds it is the chain of
// steps (n-1 per sweep), each waiting for the one before, so the work between its barriers is
// what is kept short:
// - M and V are kept in the order of the step's pairs: pair i sits at positions 2i and 2i+1,
//   and a step writes its results to the positions of the next step (M in the other of two
//   buffers, V in place, since it is read before a barrier and written after). Every address
//   is then the same in all steps and is formed once; working out the pairs' indices in each
//   step was most of it.
// - Phase A: n/2 threads form the rotations and the diagonal 2 x 2 blocks, while the other
//   waves read what they will rotate into registers. Phase B: a thread on M owns off-diagonal
//   blocks, rows (2i, 2i+1) by columns (2k, 2k+1), both rotations at once, upper triangle
//   only; a wave on V owns pairs of columns, a lane a row.
// An odd n gets a row and column of zeros, index n, in pair 0, whose rotation is the identity.
// FP64 with M and V in L2, rows, columns and V in phases of their own and three barriers a
// step, against this form (call from Python): n = 16 152 -> 79 us, 32 483 -> 167, 48 1370 -> 287,
// 64 3645 -> 493.
constexpr int SYEV_SMALL_N = 64;
constexpr int SYEV_PAIRS   = SYEV_SMALL_N / 2;
constexpr int SYEV_TRI     = SYEV_SMALL_N * (SYEV_SMALL_N + 1) / 2;
constexpr int SYEV_VPAIRS  = SYEV_PAIRS / 8; // pairs of V's columns per wave: at least eight waves are on V at n = 64

template <typename T>
__global__ __launch_bounds__(LA_THREADS) void syev_lds_kernel(int n, int upper, int vectors, T *__restrict__ A,
                                                              int64_t lda, T *__restrict__ W, FastDiv by_pairs,
                                                              int32_t *__restrict__ info) {
    __shared__ T lds[2 * SYEV_TRI + SYEV_SMALL_N * SYEV_SMALL_N];
    __shared__ T cs[SYEV_PAIRS], sn[SYEV_PAIRS];
    __shared__ T red[LA_WAVES];
    int const m      = n + (n & 1);
    int const npairs = m / 2;
    T *const V       = lds + 2 * SYEV_TRI;
    int const tid    = threadIdx.x;
    int const lane   = tid & 63;
    int const wave   = __builtin_amdgcn_readfirstlane(tid >> 6);
    int const waves  = blockDim.x >> 6;
    // sum over the workgroup in a fixed order (deterministic)
    auto sum = [&](T v) {
        v = wave_reduce_sum(v);
        __syncthreads();
        if (lane == 0) red[wave] = v;
        __syncthreads();
        T s = T(0);
        for (int i = 0; i < waves; ++i) s += red[i];
        return s;
    };
    // Round-robin ordering: pair i of step r holds indices p = r+i and q = r-i (mod m-1), pair
    // 0 the fixed index m-1 and r. Where step 0 puts an index, and what it puts at a position:
    auto position = [&](int x) { return x == m - 1 ? 0 : x == 0 ? 1 : x < npairs ? 2 * x : 2 * (m - 1 - x) + 1; };
    auto index_at = [&](int pos) {
        int const i = pos >> 1;
        return pos & 1 ? (i == 0 ? 0 : m - 1 - i) : (i == 0 ? m - 1 : i);
    };
    // and where a position's index goes in the next step: the p side moves down one pair, the
    // q side up one, p_1 becomes q_0 and the last q the last p
    auto moves_to = [&](int pos) {
        int const i = pos >> 1;
        if (npairs == 1 || pos == 0) return pos;
        if (pos & 1) return i == npairs - 1 ? pos - 1 : pos + 2;
        return i == 1 ? 1 : pos - 2;
    };
    // the referenced triangle
    T fro = T(0);
    for (int j = wave; j < m; j += waves)
        for (int i = lane; i < m; i += 64) {
            if (i <= j) {
                T const v = j >= n ? T(0) : upper ? A[i + int64_t(j) * lda] : A[j + int64_t(i) * lda];
                lds[tri(position(i), position(j))] = v;
                fro += i == j ? v * v : T(2) * v * v;
            }
            if (vectors && i < n) V[i + position(j) * n] = i == j ? T(1) : T(0);
        }
    fro = sum(fro); // also orders the writes above before the reads below
    int const back = bring_into_range(lds, m, red, sum, fro);
    T const eps   = sizeof(T) == 8 ? T(2.220446049250313e-16) : T(1.1920929e-7);
    T const limit = isinf(fro) ? T(0) : T(n) * T(n) * eps * eps * fro;

    // the diagonal block of the thread's rotation: where it is read and written
    int const rot  = tid < npairs ? tid : 0;
    int const a_pp = tri(2 * rot, 2 * rot), a_qq = tri(2 * rot + 1, 2 * rot + 1), a_pq = tri(2 * rot, 2 * rot + 1);
    int const to_p = moves_to(2 * rot), to_q = moves_to(2 * rot + 1);
    int const b_pp = tri(to_p, to_p), b_qq = tri(to_q, to_q), b_pq = tri(to_p, to_q);
    int const nblocks = npairs * (npairs - 1) / 2;
    int const wm      = vectors ? min(max(1, (nblocks + 63) >> 6), waves >> 1) : waves; // waves on M
    int const nv      = waves - wm;                                                     // and on V
    bool const on_m   = wave < wm;
    // the thread's block of M: where its elements are read and written, and its rotations.
    // Every unordered pair {i, k} once: k = i + d (mod npairs), d = 1..npairs/2, the last d
    // only half way round when npairs is even. With eight of 16 waves on M at n = 64 there is
    // one block per thread at every n; without V all waves are on M.
    int const d     = int(fast_div(uint32_t(tid), by_pairs)) + 1;
    bool const has  = on_m && tid < nblocks;
    int const bi    = has ? tid - (d - 1) * npairs : 0;
    int const bk    = !has ? 0 : bi + d >= npairs ? bi + d - npairs : bi + d;
    int src[4], dst[4];
#pragma unroll
    for (int x = 0; x < 4; ++x) {
        int const a = 2 * bi + (x >> 1), b = 2 * bk + (x & 1);
        src[x]      = tri(a, b);
        dst[x]      = tri(moves_to(a), moves_to(b));
    }
    // the wave's pairs of V's columns: v0, v0 + nv, ...
    int const v0   = wave - wm;
    int const mine = !on_m && v0 < npairs ? (npairs - v0 + nv - 1) / nv : 0;
    int vdst[2 * SYEV_VPAIRS];
#pragma unroll
    for (int z = 0; z < 2 * SYEV_VPAIRS; ++z) vdst[z] = moves_to((z >> 1) < mine ? 2 * (v0 + (z >> 1) * nv) + (z & 1) : 0) * n;

    auto step = [&](auto buf) {
        T const *const M = lds + decltype(buf)::value * SYEV_TRI;
        T *const N       = lds + (decltype(buf)::value ^ 1) * SYEV_TRI;
        T x[2 * SYEV_VPAIRS > 4 ? 2 * SYEV_VPAIRS : 4];
        if (tid < npairs) {
            T const app = M[a_pp], aqq = M[a_qq], apq = M[a_pq];
            T c, s, t;
            jacobi_rotation(app, aqq, apq, c, s, t);
            cs[tid] = c;
            sn[tid] = s;
            N[b_pp] = app - t * apq;
            N[b_qq] = aqq + t * apq;
            N[b_pq] = T(0);
        }
        if (has) {
#pragma unroll
            for (int y = 0; y < 4; ++y) x[y] = M[src[y]];
        } else if (!on_m && lane < n) {
#pragma unroll
            for (int z = 0; z < 2 * SYEV_VPAIRS; ++z)
                if ((z >> 1) < mine) x[z] = V[(2 * (v0 + (z >> 1) * nv) + (z & 1)) * n + lane];
        }
        __syncthreads();
        if (has) {
            T const si = sn[bi], sk = sn[bk], ci = cs[bi], ck = cs[bk];
            // rows by rotation i, then columns by rotation k
            T const rpp = ci * x[0] - si * x[2], rqp = si * x[0] + ci * x[2];
            T const rpq = ci * x[1] - si * x[3], rqq = si * x[1] + ci * x[3];
            N[dst[0]] = ck * rpp - sk * rpq;
            N[dst[1]] = sk * rpp + ck * rpq;
            N[dst[2]] = ck * rqp - sk * rqq;
            N[dst[3]] = sk * rqp + ck * rqq;
        } else if (!on_m && lane < n) {
            // all rotations are read before the first write: the compiler cannot know that
            // they do not overlap, and would wait for each in turn
            T c[SYEV_VPAIRS], s[SYEV_VPAIRS];
#pragma unroll
            for (int z = 0; z < SYEV_VPAIRS; ++z)
                if (z < mine) {
                    c[z] = cs[v0 + z * nv];
                    s[z] = sn[v0 + z * nv];
                }
#pragma unroll
            for (int z = 0; z < SYEV_VPAIRS; ++z)
                if (z < mine) {
                    T const u = x[2 * z], v = x[2 * z + 1];
                    V[vdst[2 * z] + lane]     = c[z] * u - s[z] * v;
                    V[vdst[2 * z + 1] + lane] = s[z] * u + c[z] * v;
                }
        }
        __syncthreads();
    };

    int cur   = 0; // the buffer that holds M
    bool conv = false;
    for (int sweep = 0; sweep <= SYEV_MAX_SWEEPS; ++sweep) {
        T off = T(0);
        for (int j = wave; j < m; j += waves)
            for (int i = lane; i < j; i += 64) {
                T const v = lds[cur * SYEV_TRI + tri(i, j)];
                off += T(2) * v * v;
            }
        off = sum(off);
        if (off <= limit) {
            conv = true;
            break;
        }
        if (sweep == SYEV_MAX_SWEEPS) break;
        for (int r = 0; r < m - 1; ++r) {
            if (cur == 0)
                step(std::integral_constant<int, 0>{});
            else
                step(std::integral_constant<int, 1>{});
            cur ^= 1;
        }
    }
    // ascending order, ties by index (stable); the columns of V follow
    T const *const M = lds + cur * SYEV_TRI;
    for (int i = wave; i < n; i += waves) {
        int const at = position(i);
        T const d    = M[tri(at, at)];
        int pos      = 0;
        for (int j = lane; j < n; j += 64) {
            int const o = position(j);
            T const e   = M[tri(o, o)];
            pos += (e < d || (e == d && j < i)) ? 1 : 0;
        }
#pragma unroll
        for (int o = 32; o >= 1; o >>= 1) pos += __shfl_xor(pos, o, 64);
        if (lane == 0) W[pos] = ldexp(d, back);
        if (vectors)
            for (int k = lane; k < n; k += 64) A[k + int64_t(pos) * lda] = V[k + at * n];
    }
    if (tid == 0) *info = conv ? 0 : 1;
}

// One index of the round-robin ordering: 0..m-2 move up by one per step and wrap (last =
// m-1), the fixed index m-1 stays (last = -1).
struct RoundRobin {
    int at, last;
    __device__ __forceinline__ void advance() {
        at += last >= 0 ? 1 : 0;
        at = at == last ? 0 : at;
    }
};

// Jacobi above n = 64. M (the matrix being diagonalised, its upper triangle packed) and V (the
// accumulated rotations, column-major) are in LDS where they fit (M_LDS, V_LDS) and in the
// workspace otherwise. An odd n gets a dummy row of zeros, index n, that never rotates: it is
// always in pair 0.
//
// A step is two phases: (A) the first waves form the n/2 rotations and update the 2 x 2
// diagonal blocks, whose values they hold, while the others apply the previous step's
// rotations to V; (B) the off-diagonal 2 x 2 blocks, rows (p_i, q_i) by columns (p_k, q_k),
// one thread each: rows and columns rotate in one pass without a barrier between them. Up to
// n = 114 (FP64) the LDS traffic of V and the index arithmetic of the blocks bound it, beyond
// that one workgroup's L2 bandwidth. The register-resident form of the small kernel needs
// more than the 128 registers of a 1024-thread workgroup here and spills (n = 100: 2455 us).
// FP64 with M and V in L2, rows, columns and V in phases of their own against now: n = 100
// 12.2 -> 1.86 ms, 130 30.7 -> 8.9, 200 120 -> 55.
template <typename T, bool M_LDS, bool V_LDS>
__global__ __launch_bounds__(LA_THREADS) void syev_jacobi_kernel(int n, int upper, int vectors, T *__restrict__ A,
                                                                 int64_t lda, T *__restrict__ W, T *__restrict__ Mg,
                                                                 T *__restrict__ Vg, FastDiv by_pairs,
                                                                 int32_t *__restrict__ info) {
    constexpr int NP = !M_LDS ? SYEV_MAX_N / 2 : sizeof(T) == 8 ? 99 : 141; // rotation pairs: n <= 198, 282 in LDS
    __shared__ T lds[M_LDS ? SYEV_LDS_ELEMS<T> : 1];
    __shared__ T cs[2][NP], sn[2][NP];
    __shared__ T red[LA_WAVES];
    int const m      = n + (n & 1);
    int const first  = n & 1; // pair 0 holds the dummy index
    int const npairs = m / 2;
    int const ntri   = m * (m + 1) / 2;
    T *const M       = M_LDS ? lds : Mg;
    T *const V       = V_LDS ? lds + ntri : Vg;
    int const tid    = threadIdx.x;
    int const nt     = blockDim.x;
    int const lane   = tid & 63;
    int const wave   = __builtin_amdgcn_readfirstlane(tid >> 6);
    int const waves  = nt >> 6;
    // sum over the workgroup in a fixed order (deterministic)
    auto sum = [&](T v) {
        v = wave_reduce_sum(v);
        __syncthreads();
        if (lane == 0) red[wave] = v;
        __syncthreads();
        T s = T(0);
        for (int i = 0; i < waves; ++i) s += red[i];
        return s;
    };
    // the referenced triangle
    T fro = T(0);
    for (int j = wave; j < m; j += waves)
        for (int i = lane; i < m; i += 64) {
            if (i <= j) {
                T const v    = j >= n ? T(0) : upper ? A[i + int64_t(j) * lda] : A[j + int64_t(i) * lda];
                M[tri(i, j)] = v;
                fro += i == j ? v * v : T(2) * v * v;
            }
            if (vectors && i < n && j < n) V[i + int64_t(j) * n] = i == j ? T(1) : T(0);
        }
    fro = sum(fro); // also orders the writes above before the reads below
    int const back = bring_into_range(M, m, red, sum, fro);
    T const eps   = sizeof(T) == 8 ? T(2.220446049250313e-16) : T(1.1920929e-7);
    T const limit = isinf(fro) ? T(0) : T(n) * T(n) * eps * eps * fro;
    // round-robin pairing (p_i, q_i) of step r: index m-1 fixed in pair 0, the others move by
    // one per step, so a thread keeps the indices of its pairs and advances them; after the
    // m-1 steps of a sweep they are where they began
    auto p_of = [&](int r, int i) {
        int const x = r + i;
        return RoundRobin{i == 0 ? m - 1 : x >= m - 1 ? x - (m - 1) : x, i == 0 ? -1 : m - 1};
    };
    auto q_of = [&](int r, int i) { return RoundRobin{r < i ? r - i + m - 1 : r - i, m - 1}; };
    // every unordered pair {i, k} of rotations once: k = i + d (mod npairs), d = 1..npairs/2,
    // the last d only half way round when npairs is even
    int const nblocks = npairs * (npairs - 1) / 2;
    auto block_of     = [&](int e, int &i, int &k) {
        int const d = int(fast_div(uint32_t(e), by_pairs)) + 1;
        i           = e - (d - 1) * npairs;
        k           = i + d >= npairs ? i + d - npairs : i + d;
    };
    int i_first, k_first; // the thread's first block is the same in every step
    block_of(tid, i_first, k_first);
    RoundRobin bpi = p_of(0, i_first), bqi = q_of(0, i_first), bpk = p_of(0, k_first), bqk = q_of(0, k_first);
    RoundRobin rp = p_of(0, tid), rq = q_of(0, tid); // of the thread's rotation (tid < npairs)
    int const rotators = (npairs + 63) >> 6; // waves that form rotations in phase A
    bool const split   = waves > rotators;   // the other waves apply V meanwhile
    int set            = 0;                  // rotation set of the current step
    bool pending       = false;              // the other set is not yet in V

    // V <- V J for pairs i and j (the same one twice: i alone), their four columns read together
    auto rotate_columns = [&](int which, int i, int j, int p1, int q1, int p2, int q2) {
        T const s1 = sn[which][i], s2 = sn[which][j], c1 = cs[which][i], c2 = cs[which][j];
        T *const vp = V + int64_t(p1) * n, *const vq = V + int64_t(q1) * n;
        T *const wp = V + int64_t(p2) * n, *const wq = V + int64_t(q2) * n;
        for (int k = lane; k < n; k += 64) {
            T const u = vp[k], v = vq[k], x = wp[k], y = wq[k];
            vp[k] = c1 * u - s1 * v;
            vq[k] = s1 * u + c1 * v;
            if (j != i) {
                wp[k] = c2 * x - s2 * y;
                wq[k] = s2 * x + c2 * y;
            }
        }
    };
    // the rotations of the step before the current one, by waves w0, w0 + 1, ... of nw
    int const w0 = split ? wave - rotators : wave, nw = split ? waves - rotators : waves;
    int const vi = first + (w0 < 0 ? 0 : w0), vj = vi + nw < npairs ? vi + nw : vi;
    RoundRobin vp1 = p_of(0, vi), vq1 = q_of(0, vi), vp2 = p_of(0, vj), vq2 = q_of(0, vj);
    int vr         = 0; // the step V takes next
    auto apply_v   = [&](int which) {
        if (w0 < 0) return;
        if (vi < npairs) rotate_columns(which, vi, vj, vp1.at, vq1.at, vp2.at, vq2.at);
        for (int i = vi + 2 * nw; i < npairs; i += 2 * nw) {
            int const j = i + nw < npairs ? i + nw : i;
            rotate_columns(which, i, j, p_of(vr, i).at, q_of(vr, i).at, p_of(vr, j).at, q_of(vr, j).at);
        }
        vp1.advance();
        vq1.advance();
        vp2.advance();
        vq2.advance();
        vr = vr + 1 == m - 1 ? 0 : vr + 1;
    };

    bool conv = false;
    for (int sweep = 0; sweep <= SYEV_MAX_SWEEPS; ++sweep) {
        T off = T(0);
        for (int j = wave; j < n; j += waves)
            for (int i = lane; i < j; i += 64) {
                T const v = M[tri(i, j)];
                off += T(2) * v * v;
            }
        off = sum(off);
        if (__builtin_amdgcn_readfirstlane(int(off <= limit)) != 0) { // the same in every lane
            conv = true;
            break;
        }
        if (sweep == SYEV_MAX_SWEEPS) break;
        for (int r = 0; r < m - 1; ++r) {
            if (tid < npairs) { // npairs <= nt
                int const xp = tri(rp.at, rp.at), xq = tri(rq.at, rq.at), xpq = tri(rp.at, rq.at);
                T const app = M[xp], aqq = M[xq], apq = M[xpq];
                T c, s, t;
                jacobi_rotation(app, aqq, apq, c, s, t);
                cs[set][tid] = c;
                sn[set][tid] = s;
                M[xp]        = app - t * apq;
                M[xq]        = aqq + t * apq;
                M[xpq]       = T(0);
                rp.advance();
                rq.advance();
            }
            if (vectors && pending) apply_v(set ^ 1);
            __syncthreads();
            for (int e = tid; e < nblocks; e += nt) {
                int i = i_first, k = k_first, pi = bpi.at, qi = bqi.at, pk = bpk.at, qk = bqk.at;
                if (e != tid) {
                    block_of(e, i, k);
                    pi = p_of(r, i).at;
                    qi = q_of(r, i).at;
                    pk = p_of(r, k).at;
                    qk = q_of(r, k).at;
                }
                T const si = sn[set][i], sk = sn[set][k], ci = cs[set][i], ck = cs[set][k];
                int const xpp = tri(pi, pk), xpq = tri(pi, qk), xqp = tri(qi, pk), xqq = tri(qi, qk);
                T const vpp = M[xpp], vpq = M[xpq], vqp = M[xqp], vqq = M[xqq];
                // rows by rotation i, then columns by rotation k
                T const rpp = ci * vpp - si * vqp, rqp = si * vpp + ci * vqp;
                T const rpq = ci * vpq - si * vqq, rqq = si * vpq + ci * vqq;
                M[xpp] = ck * rpp - sk * rpq;
                M[xpq] = sk * rpp + ck * rpq;
                M[xqp] = ck * rqp - sk * rqq;
                M[xqq] = sk * rqp + ck * rqq;
            }
            bpi.advance();
            bqi.advance();
            bpk.advance();
            bqk.advance();
            __syncthreads();
            set ^= 1;
            pending = true;
        }
    }
    // the last step's rotations; the waves that formed them have no share of V
    if (vectors && pending) apply_v(set ^ 1);
    // ascending order, ties by index (stable); the columns of V follow
    __syncthreads();
    for (int i = wave; i < n; i += waves) {
        T const d = M[tri(i, i)];
        int pos   = 0;
        for (int j = lane; j < n; j += 64) {
            T const e = M[tri(j, j)];
            pos += (e < d || (e == d && j < i)) ? 1 : 0;
        }
#pragma unroll
        for (int o = 32; o >= 1; o >>= 1) pos += __shfl_xor(pos, o, 64);
        if (lane == 0) W[pos] = ldexp(d, back);
        if (vectors)
            for (int k = lane; k < n; k += 64) A[k + int64_t(pos) * lda] = V[k + int64_t(i) * n];
    }
    if (tid == 0) *info = conv ? 0 : 1;
}

template <typename T>
__global__ __launch_bounds__(LA_THREADS) void gesv_kernel(int n, int nrhs, T *__restrict__ A, int64_t lda,
                                                          int64_t *__restrict__ ipiv, T *__restrict__ B, int64_t ldb,
                                                          int32_t *__restrict__ info) {
    __shared__ T bv[LA_WAVES];
    __shared__ int bi[LA_WAVES];
    int const tid  = threadIdx.x;
    int const lane = tid & 63;
    int const w    = tid >> 6;
    int first_zero = 0; // 1-based column of the first exactly zero pivot
    for (int j = 0; j < n; ++j) {
        // pivot: the first row of largest magnitude in column j at or below the diagonal
        T best  = T(-1);
        int row = n;
        for (int i = j + tid; i < n; i += LA_THREADS) {
            T const v = std::fabs(A[i + int64_t(j) * lda]);
            if (v > best) {
                best = v;
                row  = i;
            }
        }
#pragma unroll
        for (int off = 32; off >= 1; off >>= 1) {
            T const ob  = __shfl_xor(best, off, 64);
            int const o = __shfl_xor(row, off, 64);
            if (ob > best || (ob == best && o < row)) {
                best = ob;
                row  = o;
            }
        }
        if (lane == 0) {
            bv[w] = best;
            bi[w] = row;
        }
        __syncthreads();
        best = bv[0];
        row  = bi[0];
        for (int k = 1; k < LA_WAVES; ++k)
            if (bv[k] > best || (bv[k] == best && bi[k] < row)) {
                best = bv[k];
                row  = bi[k];
            }
        __syncthreads();
        int const p = row < n ? row : j; // a column of NaNs compares false everywhere: keep row j
        if (tid == 0) ipiv[j] = p + 1;
        if (p != j) {
            for (int k = tid; k < n; k += LA_THREADS) {
                T const t               = A[j + int64_t(k) * lda];
                A[j + int64_t(k) * lda] = A[p + int64_t(k) * lda];
                A[p + int64_t(k) * lda] = t;
            }
        }
        __syncthreads();
        T const ujj = A[j + int64_t(j) * lda];
        if (ujj == T(0)) {
            if (first_zero == 0) first_zero = j + 1;
            continue; // LAPACK completes the factorization past an exactly singular pivot
        }
        for (int i = j + 1 + tid; i < n; i += LA_THREADS) A[i + int64_t(j) * lda] /= ujj;
        __syncthreads();
        int const t = n - j - 1;
        for (int64_t e = tid; e < int64_t(t) * t; e += LA_THREADS) {
            int const i = j + 1 + int(e % t), k = j + 1 + int(e / t);
            A[i + int64_t(k) * lda] -= A[i + int64_t(j) * lda] * A[j + int64_t(k) * lda];
        }
        __syncthreads();
    }
    if (first_zero == 0) {
        // P b (the interchanges in order), L y = P b (unit lower), then U x = y; B is left
        // untouched when the factor is singular, as by LAPACK
        for (int j = 0; j < n; ++j) {
            int const p = int(ipiv[j]) - 1;
            if (p != j) {
                for (int r = tid; r < nrhs; r += LA_THREADS) {
                    T const t               = B[j + int64_t(r) * ldb];
                    B[j + int64_t(r) * ldb] = B[p + int64_t(r) * ldb];
                    B[p + int64_t(r) * ldb] = t;
                }
            }
            __syncthreads();
        }
        for (int j = 0; j < n; ++j) {
            int const t = n - j - 1;
            for (int64_t e = tid; e < int64_t(t) * nrhs; e += LA_THREADS) {
                int const i = j + 1 + int(e % t), r = int(e / t);
                B[i + int64_t(r) * ldb] -= A[i + int64_t(j) * lda] * B[j + int64_t(r) * ldb];
            }
            __syncthreads();
        }
        for (int j = n - 1; j >= 0; --j) {
            for (int r = tid; r < nrhs; r += LA_THREADS) B[j + int64_t(r) * ldb] /= A[j + int64_t(j) * lda];
            __syncthreads();
            for (int64_t e = tid; e < int64_t(j) * nrhs; e += LA_THREADS) {
                int const i = int(e % j), r = int(e / j);
                B[i + int64_t(r) * ldb] -= A[i + int64_t(j) * lda] * B[j + int64_t(r) * ldb];
            }
            __syncthreads();
        }
    }
    if (tid == 0) *info = first_zero;
}

// n == 0: only the status (a kernel rather than a memset node, so that it can be captured)
__global__ void clear_info_kernel(int32_t *info) { *info = 0; }

} // namespace

template <typename T>
int syev_impl(char job, char uplo, int64_t n, T *A, int64_t lda, T *W, int32_t *info, hipStream_t stream) {
    bool const vectors = job == 'V' || job == 'v';
    if (!vectors && job != 'N' && job != 'n') return fail(-1, "syev: job must be 'V' or 'N'");
    bool const upper = uplo == 'U' || uplo == 'u';
    if (!upper && uplo != 'L' && uplo != 'l') return fail(-2, "syev: uplo must be 'U' or 'L'");
    if (n < 0) return fail(-3, "syev: n < 0");
    if (n > SYEV_MAX_N) return fail(EIN_ERROR_UNSUPPORTED, "syev: n above 1024 (a one-workgroup solver for small matrices)");
    if (lda < std::max<int64_t>(1, n)) return fail(-5, "syev: lda < max(1, n)");
    if (info == nullptr) return fail(-7, "syev: info must point to device memory");
    if (n == 0) {
        clear_info_kernel<<<1, 1, 0, stream>>>(info);
        EIN_LAUNCH_CHECK();
        return EIN_SUCCESS;
    }
    int const up = upper ? 1 : 0, vec = vectors ? 1 : 0;
    FastDiv const by_pairs = make_fastdiv(uint32_t((n + 1) / 2));
    if (n <= SYEV_SMALL_N) {
        // a small problem has work for a few waves only, and fewer waves meet sooner at a barrier
        int const threads = n <= 16 ? 256 : n <= 32 ? 512 : LA_THREADS;
        syev_lds_kernel<T><<<1, threads, 0, stream>>>(int(n), up, vec, A, lda, W, by_pairs, info);
        EIN_LAUNCH_CHECK();
        return EIN_SUCCESS;
    }
    // M and V in LDS (FP64 n <= 114, FP32 n <= 162), M alone (n <= 198 and 282), or neither
    size_t const nn   = size_t(n) * size_t(n);
    size_t const m    = size_t(n) + size_t(n & 1);
    size_t const ntri = m * (m + 1) / 2;
    bool const m_lds  = ntri * sizeof(T) <= SYEV_LDS_BYTES;
    bool const v_lds  = (ntri + nn) * sizeof(T) <= SYEV_LDS_BYTES;
    size_t const global = (m_lds ? 0 : ntri) + (v_lds || !vectors ? 0 : nn); // less than 2 n^2
    T *Mg = nullptr, *Vg = nullptr;
    if (global > 0) {
        void *ws = nullptr;
        EIN_TRY(workspace(stream, global * sizeof(T), &ws));
        Mg = static_cast<T *>(ws);
        Vg = m_lds ? Mg : Mg + ntri;
    }
    if (v_lds)
        syev_jacobi_kernel<T, true, true><<<1, LA_THREADS, 0, stream>>>(int(n), up, vec, A, lda, W, Mg, Vg, by_pairs, info);
    else if (m_lds)
        syev_jacobi_kernel<T, true, false><<<1, LA_THREADS, 0, stream>>>(int(n), up, vec, A, lda, W, Mg, Vg, by_pairs, info);
    else
        syev_jacobi_kernel<T, false, false><<<1, LA_THREADS, 0, stream>>>(int(n), up, vec, A, lda, W, Mg, Vg, by_pairs, info);
    EIN_LAUNCH_CHECK();
    return EIN_SUCCESS;
}

template <typename T>
int gesv_impl(int64_t n, int64_t nrhs, T *A, int64_t lda, int64_t *ipiv, T *B, int64_t ldb, int32_t *info,
              hipStream_t stream) {
    if (n < 0) return fail(-1, "gesv: n < 0");
    if (nrhs < 0) return fail(-2, "gesv: nrhs < 0");
    if (lda < std::max<int64_t>(1, n)) return fail(-4, "gesv: lda < max(1, n)");
    if (ldb < std::max<int64_t>(1, n)) return fail(-7, "gesv: ldb < max(1, n)");
    if (info == nullptr) return fail(-8, "gesv: info must point to device memory");
    if (n > GESV_MAX_N || nrhs > (int64_t{1} << 30))
        return fail(EIN_ERROR_UNSUPPORTED, "gesv: n above 4096 (a one-workgroup solver for small systems)");
    if (n == 0) {
        clear_info_kernel<<<1, 1, 0, stream>>>(info);
        EIN_LAUNCH_CHECK();
        return EIN_SUCCESS;
    }
    gesv_kernel<T><<<1, LA_THREADS, 0, stream>>>(int(n), int(nrhs), A, lda, ipiv, B, ldb, info);
    EIN_LAUNCH_CHECK();
    return EIN_SUCCESS;
}

} // namespace ein

extern "C" {

int ein_syev_f64(char job, char uplo, int64_t n, double *A, int64_t lda, double *W, int32_t *info,
                 ein_stream_t stream) {
    return ein::syev_impl<double>(job, uplo, n, A, lda, W, info, ein::as_stream(stream));
}
int ein_syev_f32(char job, char uplo, int64_t n, float *A, int64_t lda, float *W, int32_t *info, ein_stream_t stream) {
    return ein::syev_impl<float>(job, uplo, n, A, lda, W, info, ein::as_stream(stream));
}
int ein_gesv_f64(int64_t n, int64_t nrhs, double *A, int64_t lda, int64_t *ipiv, double *B, int64_t ldb, int32_t *info,
                 ein_stream_t stream) {
    return ein::gesv_impl<double>(n, nrhs, A, lda, ipiv, B, ldb, info, ein::as_stream(stream));
}
int ein_gesv_f32(int64_t n, int64_t nrhs, float *A, int64_t lda, int64_t *ipiv, float *B, int64_t ldb, int32_t *info,
                 ein_stream_t stream) {
    return ein::gesv_impl<float>(n, nrhs, A, lda, ipiv, B, ldb, info, ein::as_stream(stream));
}

} // extern "C"
