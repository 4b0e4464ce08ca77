// Coulomb and exchange matrices of a four-index tensor in one pass over it (the Fock build
// of a Hartree-Fock iteration):
//   F = beta*F + alpha_j*J + alpha_k*K,
//   J(a,b) = sum_cd g(a,b,c,d) D(c,d),   K(a,c) = sum_bd g(a,b,c,d) D(b,d),
// with g row-major n^4 and D, F row-major n x n (leading dimensions ldd, ldf).
//
// The reference forms these with two einsum calls that each read all of g:
//   einsum(1, {i,j}, &F,  2, {k,l}, D, {i,j,k,l}, TEI)   J, the GEMV case
//   einsum(1, {i,j}, &F, -1, {k,l}, D, {i,k,j,l}, TEI)   K, the generic case
// (libs/Einsums/TensorAlgebra/tests/unit/QChemTests.cpp:299-304; the J and K builds of
// devtools/profiling/profile_einsums.cpp:23-30). Element g(a,b,c,d) feeds J(a,b) with D(c,d)
// and K(a,c) with D(b,d), so both can be accumulated from one read of g: half the HBM traffic
// of the two calls, which is what bounds them (0.25 flop per byte).
//
// For n <= 64, kernel 1: workgroup (a, four b's) reads the slabs g(a,b,:,:) of its b's. Wave w
// takes the rows c = w, w+4, ...; its lanes run over d. Per lane it keeps
// K partials per row; J(a,b) is complete inside the workgroup and is written directly, K is
// written as one partial row per chunk. Kernel 2 adds the chunks' K partials in chunk order
// and forms F (deterministic: fixed summation trees, no atomics). For even n with 16-byte
// aligned rows, kernel 1 reads two elements per lane (fock_jk16_kernel). For 64 < n <= 128 a
// slab is large enough to fill a CU's loads, and one workgroup per CU streams its share of all
// slabs (fock_jk_stream_kernel). n <= 128.
#include <algorithm>
#include <string>

#include "ein_common.hpp"

namespace ein {

namespace {

constexpr int FOCK_MAX_N = 128;

// n <= 64. MR >= ceil(n / 4) rows c per wave; BC = b's per workgroup. Each lane keeps the
// D(c, d) of its own (c, d) positions in registers (the same for every slab), so no LDS
// staging or barrier precedes the slab loads: all of a workgroup's slab reads are in
// flight at once, and the many resident workgroups keep HBM busy.
template <int MR, int BC>
__global__ __launch_bounds__(256) void fock_jk_kernel(int n, double const *__restrict__ g, double const *__restrict__ D,
                                                      int64_t ldd, double *__restrict__ J, double *__restrict__ Kp) {
    constexpr int WAVES = 4;
    __shared__ double red[WAVES][BC];
    int const a    = int(blockIdx.x);
    int const ch   = int(blockIdx.y);
    int const wave = int(threadIdx.x) >> 6;
    int const lane = int(threadIdx.x) & 63; // d
    int const b0   = ch * BC;
    int const rows = (n - wave + WAVES - 1) / WAVES; // rows c = wave + WAVES*i, i < rows
    int64_t const nn = int64_t(n) * n;

    double x[BC][MR];
#pragma unroll
    for (int q = 0; q < BC; ++q) {
        bool const b_in = b0 + q < n;
        double const *__restrict__ slab = g + (int64_t(a) * n + (b_in ? b0 + q : b0)) * nn;
#pragma unroll
        for (int i = 0; i < MR; ++i) {
            int const c = wave + WAVES * i;
            x[q][i]     = (b_in && i < rows && lane < n) ? slab[int64_t(c) * n + lane] : 0.0;
        }
    }
    double dc[MR], db[BC];
#pragma unroll
    for (int i = 0; i < MR; ++i) {
        int const c = wave + WAVES * i;
        dc[i]       = (i < rows && lane < n) ? D[int64_t(c) * ldd + lane] : 0.0;
    }
#pragma unroll
    for (int q = 0; q < BC; ++q) db[q] = (b0 + q < n && lane < n) ? D[int64_t(b0 + q) * ldd + lane] : 0.0;

    double kacc[MR];
#pragma unroll
    for (int i = 0; i < MR; ++i) kacc[i] = 0.0;
#pragma unroll
    for (int q = 0; q < BC; ++q) {
        double jsum = 0.0;
#pragma unroll
        for (int i = 0; i < MR; ++i) {
            jsum += x[q][i] * dc[i];
            kacc[i] += x[q][i] * db[q];
        }
        // J(a, b): lanes here, the waves after the barrier
        jsum = wave_reduce_sum(jsum);
        if (lane == 0) red[wave][q] = jsum;
    }
    // K partial row of this chunk: Kp[(a * chunks + ch) * n + c]
    double *__restrict__ kp = Kp + (int64_t(a) * gridDim.y + ch) * n;
#pragma unroll
    for (int i = 0; i < MR; ++i) {
        double const s = wave_reduce_sum(kacc[i]);
        if (lane == 0 && i < rows) kp[wave + WAVES * i] = s;
    }
    __syncthreads();
    if (int(threadIdx.x) < BC && b0 + int(threadIdx.x) < n) {
        double s = 0.0;
#pragma unroll
        for (int w = 0; w < WAVES; ++w) s += red[w][threadIdx.x];
        J[int64_t(a) * n + b0 + int(threadIdx.x)] = s;
    }
}

// The same pass with 16-byte loads, for even n <= 64 with 16-byte aligned rows of g and D
// (even ldd): lane l reads d = 2(l%32), 2(l%32)+1 of row c = 2p + l/32 (lanes with
// 2(l%32) >= n idle), so one load covers two adjacent rows of a slab; wave w takes the row
// pairs p = w, w+4, ... (MP >= ceil(n/8) of them). K's row sums reduce within each 32-lane
// half. Measured at n = 48 (HF): 18.0 against 21.1 us cold for the two launches.
template <int MP, int BC>
__global__ __launch_bounds__(256) void fock_jk16_kernel(int n, double const *__restrict__ g, double const *__restrict__ D,
                                                        int64_t ldd, double *__restrict__ J, double *__restrict__ Kp) {
    constexpr int WAVES = 4;
    __shared__ double red[WAVES][BC];
    int const a      = int(blockIdx.x);
    int const ch     = int(blockIdx.y);
    int const wave   = int(threadIdx.x) >> 6;
    int const lane   = int(threadIdx.x) & 63;
    int const h      = lane >> 5;
    int const d0     = 2 * (lane & 31);
    bool const d_in  = d0 < n;
    int const b0     = ch * BC;
    int const np     = (n / 2 - wave + WAVES - 1) / WAVES; // row pairs p = wave + WAVES*i, i < np
    int64_t const nn = int64_t(n) * n;

    double2 x[BC][MP];
#pragma unroll
    for (int q = 0; q < BC; ++q) {
        bool const b_in = b0 + q < n;
        double const *__restrict__ slab = g + (int64_t(a) * n + (b_in ? b0 + q : b0)) * nn;
#pragma unroll
        for (int i = 0; i < MP; ++i) {
            int const c = 2 * (wave + WAVES * i) + h;
            x[q][i]     = (b_in && i < np && d_in) ? *reinterpret_cast<double2 const *>(slab + int64_t(c) * n + d0)
                                                   : double2{0.0, 0.0};
        }
    }
    double2 dc[MP], db[BC];
#pragma unroll
    for (int i = 0; i < MP; ++i) {
        int const c = 2 * (wave + WAVES * i) + h;
        dc[i] = (i < np && d_in) ? *reinterpret_cast<double2 const *>(D + int64_t(c) * ldd + d0) : double2{0.0, 0.0};
    }
#pragma unroll
    for (int q = 0; q < BC; ++q)
        db[q] = (b0 + q < n && d_in) ? *reinterpret_cast<double2 const *>(D + int64_t(b0 + q) * ldd + d0)
                                     : double2{0.0, 0.0};

    double kacc[MP];
#pragma unroll
    for (int i = 0; i < MP; ++i) kacc[i] = 0.0;
#pragma unroll
    for (int q = 0; q < BC; ++q) {
        double jsum = 0.0;
#pragma unroll
        for (int i = 0; i < MP; ++i) {
            jsum += x[q][i].x * dc[i].x + x[q][i].y * dc[i].y;
            kacc[i] += x[q][i].x * db[q].x + x[q][i].y * db[q].y;
        }
        jsum = wave_reduce_sum(jsum);
        if (lane == 0) red[wave][q] = jsum;
    }
    double *__restrict__ kp = Kp + (int64_t(a) * gridDim.y + ch) * n;
#pragma unroll
    for (int i = 0; i < MP; ++i) {
        double s = kacc[i];
#pragma unroll
        for (int o = 16; o > 0; o >>= 1) s += __shfl_xor(s, o, 64); // within the 32-lane half
        if ((lane & 31) == 0 && i < np) kp[2 * (wave + WAVES * i) + h] = s;
    }
    __syncthreads();
    if (int(threadIdx.x) < BC && b0 + int(threadIdx.x) < n) {
        double s = 0.0;
#pragma unroll
        for (int w = 0; w < WAVES; ++w) s += red[w][threadIdx.x];
        J[int64_t(a) * n + b0 + int(threadIdx.x)] = s;
    }
}

// 64 < n <= 128: one workgroup of 16 waves per CU takes `units` consecutive slabs
// s = a*n + b, and holds the next slab's loads in registers while it works on one. HBM-bound:
// one slab (34 to 131 KB) in flight per CU covers the latency, and no workgroup start, D read
// or K reduction comes between two slabs of the same a. MR = ceil(n / 16) rows c = wave + 16 i;
// VEC: a lane reads d = 2l, 2l+1 as 16 bytes (even n, 16-byte aligned rows), otherwise d = l
// and l + 64. All loads are unconditional, from clamped addresses, so that the wait before a
// slab counts exactly the loads behind it; what lies outside is dropped before it is summed.
// J(a,b) sums its waves from LDS at the end; K is written per a as piece 2w (the first a of
// workgroup w) or 2w+1. One workgroup per slab, whose shuffle reductions and start nothing
// overlapped, took 195 + 13.5 us at n = 96 (3.4 TB/s over the call). Now, per call: n = 65 47 us
// (before 77), 96 126 us = 5.4 TB/s (202), 97 146 (314), 112 215 (435), 127 367 (620), 128 361 (621).
constexpr int FOCK_WAVES = 16, FOCK_UNITS = 64; // LDS for the J sums of 64 slabs

template <int MR, bool VEC>
__global__ __launch_bounds__(64 * FOCK_WAVES) void fock_jk_stream_kernel(int n, int units, double const *__restrict__ g,
                                                                         double const *__restrict__ D, int64_t ldd,
                                                                         double *__restrict__ J,
                                                                         double *__restrict__ Kp) {
    // D(c,d) in registers, or in LDS where two slabs of x leave no room for it in the 128 of a
    // 1024-thread workgroup (n = 127 then spilled: 672 us)
    constexpr bool D_LDS = !VEC || MR == 8;
    __shared__ double jred[FOCK_UNITS][FOCK_WAVES];
    __shared__ double dl[D_LDS ? FOCK_MAX_N * FOCK_MAX_N : 1];
    int const wave = __builtin_amdgcn_readfirstlane(int(threadIdx.x) >> 6);
    int const lane = int(threadIdx.x) & 63;
    int const nn   = n * n;
    if constexpr (D_LDS) { // zeros outside
        for (int c = wave; c < FOCK_WAVES * MR; c += FOCK_WAVES)
            for (int d = lane; d < FOCK_MAX_N; d += 64) dl[c * FOCK_MAX_N + d] = c < n && d < n ? D[int64_t(c) * ldd + d] : 0.0;
        __syncthreads();
    }
    int const s0 = int(blockIdx.x) * units, s1 = s0 + units < nn ? s0 + units : nn;
    bool const in0 = !VEC || 2 * lane < n, in1 = VEC || lane + 64 < n; // the lane's two elements
    bool const last_in = wave + FOCK_WAVES * (MR - 1) < n;             // its last row
    int const d0 = VEC ? (in0 ? 2 * lane : n - 2) : lane;
    int const d1 = VEC ? d0 + 1 : (in1 ? lane + 64 : n - 1);
    auto load_row = [&](double const *__restrict__ row, double (&v)[2]) {
        if constexpr (VEC) {
            double2 const t = *reinterpret_cast<double2 const *>(row + d0);
            v[0] = t.x;
            v[1] = t.y;
        } else {
            // byte offsets without a sign, opaque at each load, which then adds them to the row's
            // address by itself: the compiler would keep a 64-bit address per row, and spill
            uint32_t o0 = 8u * uint32_t(d0), o1 = 8u * uint32_t(d1);
            asm volatile("" : "+v"(o0), "+v"(o1));
            v[0] = *reinterpret_cast<double const *>(reinterpret_cast<char const *>(row) + o0);
            v[1] = *reinterpret_cast<double const *>(reinterpret_cast<char const *>(row) + o1);
        }
    };
    int row[MR]; // offset of the wave's rows in a slab
    double dc[D_LDS ? 1 : MR][2];
#pragma unroll
    for (int i = 0; i < MR; ++i) {
        int const c = i < MR - 1 || last_in ? wave + FOCK_WAVES * i : n - 1;
        row[i]      = c * n;
        if constexpr (!D_LDS) load_row(D + int64_t(c) * ldd, dc[i]);
    }
    auto load = [&](int s, int b, double (&x)[MR][2], double (&db)[2]) {
        double const *__restrict__ slab = g + int64_t(s) * nn;
        load_row(D + int64_t(b) * ldd, db);
#pragma unroll
        for (int i = 0; i < MR; ++i) load_row(slab + row[i], x[i]);
    };
    double kacc[MR];
#pragma unroll
    for (int i = 0; i < MR; ++i) kacc[i] = 0.0;
    int const a0 = s0 / n;
    int a = a0, b = s0 - a0 * n;
    auto write_k = [&]() {
        double *__restrict__ kp = Kp + int64_t(2 * int(blockIdx.x) + (a != a0 ? 1 : 0)) * n;
#pragma unroll
        for (int i = 0; i < MR; ++i) {
            double const s = wave_reduce_sum(in0 ? kacc[i] : 0.0);
            if (lane == 0 && (i < MR - 1 || last_in)) kp[wave + FOCK_WAVES * i] = s;
            kacc[i] = 0.0;
        }
    };
    auto work = [&](int s, double (&x)[MR][2], double (&db)[2]) {
        double jsum = 0.0;
        double const dby = in1 ? db[1] : 0.0;
        int e0 = wave * FOCK_MAX_N + d0;
        if constexpr (D_LDS) asm volatile("" : "+v"(e0)); // read each time, not kept in registers
        int const e1 = VEC ? e0 + 1 : e0 + 64;
#pragma unroll
        for (int i = 0; i < MR; ++i) {
            // a lane without a second element has zeros on both sides of its products: what its
            // clamped address holds may be an infinity, in g as in D
            constexpr int ROW = FOCK_WAVES * FOCK_MAX_N;
            double const y    = in1 ? x[i][1] : 0.0;
            double const j    = x[i][0] * (D_LDS ? dl[e0 + i * ROW] : dc[D_LDS ? 0 : i][0]) +
                             y * (D_LDS ? dl[e1 + i * ROW] : dc[D_LDS ? 0 : i][1]);
            jsum += i < MR - 1 || last_in ? j : 0.0;
            kacc[i] += x[i][0] * db[0] + y * dby;
        }
        jsum = wave_reduce_sum(in0 ? jsum : 0.0);
        if (lane == 0) jred[s - s0][wave] = jsum;
        if (++b == n) {
            write_k();
            b = 0;
            ++a;
        }
    };
    double xa[MR][2], xb[MR][2], dba[2], dbb[2];
    auto next_b = [&](int ahead) { return b + ahead < n ? b + ahead : b + ahead - n; };
    load(s0, b, xa, dba);
    int s = s0;
    for (; s + 2 < s1; s += 2) {
        load(s + 1, next_b(1), xb, dbb);
        work(s, xa, dba);
        load(s + 2, next_b(1), xa, dba); // b has moved on
        work(s + 1, xb, dbb);
    }
    if (s + 1 < s1) {
        load(s + 1, next_b(1), xb, dbb);
        work(s, xa, dba);
        work(s + 1, xb, dbb);
    } else {
        work(s, xa, dba);
    }
    if (b != 0) write_k();
    __syncthreads();
    if (int(threadIdx.x) < s1 - s0) {
        double j = 0.0;
#pragma unroll
        for (int w = 0; w < FOCK_WAVES; ++w) j += jred[threadIdx.x][w];
        J[s0 + int(threadIdx.x)] = j;
    }
}

// F(a,c) from J and the K pieces of row a, in workgroup order.
__global__ __launch_bounds__(256) void fock_finish_pieces_kernel(int n, int units, double const *__restrict__ J,
                                                                 double const *__restrict__ Kp, double alpha_j,
                                                                 double alpha_k, double beta, double *__restrict__ F,
                                                                 int64_t ldf) {
    int const e = int(blockIdx.x) * 256 + int(threadIdx.x);
    if (e >= n * n) return;
    int const a = e / n, c = e - a * n;
    double k = 0.0;
    for (int w = a * n / units; w <= (a * n + n - 1) / units; ++w)
        k += Kp[int64_t(2 * w + (w * units / n != a ? 1 : 0)) * n + c];
    double *fp = F + int64_t(a) * ldf + c;
    double v   = alpha_j * J[e] + alpha_k * k;
    if (beta != 0.0) v += beta * *fp;
    *fp = v;
}

template <int MR>
void launch_stream(bool vec, int grid, int n, int units, double const *g, double const *D, int64_t ldd, double *J,
                   double *Kp, hipStream_t stream) {
    if (vec)
        fock_jk_stream_kernel<MR, true><<<grid, 64 * FOCK_WAVES, 0, stream>>>(n, units, g, D, ldd, J, Kp);
    else
        fock_jk_stream_kernel<MR, false><<<grid, 64 * FOCK_WAVES, 0, stream>>>(n, units, g, D, ldd, J, Kp);
}

// F(a,c) = beta*F(a,c) + alpha_j*J(a,c) + alpha_k*sum_chunk Kp(a,chunk,c), chunks in order.
__global__ __launch_bounds__(256) void fock_finish_kernel(int n, int chunks, double const *__restrict__ J,
                                                          double const *__restrict__ Kp, double alpha_j, double alpha_k,
                                                          double beta, double *__restrict__ F, int64_t ldf) {
    int64_t const e = int64_t(blockIdx.x) * 256 + threadIdx.x;
    if (e >= int64_t(n) * n) return;
    int const a = int(e / n), c = int(e % n);
    // four independent partial sums so the chunk loads are in flight together
    double const *__restrict__ kp = Kp + int64_t(a) * chunks * n + c;
    double k4[4] = {0.0, 0.0, 0.0, 0.0};
    int ch = 0;
    for (; ch + 3 < chunks; ch += 4)
#pragma unroll
        for (int u = 0; u < 4; ++u) k4[u] += kp[int64_t(ch + u) * n];
    for (; ch < chunks; ++ch) k4[0] += kp[int64_t(ch) * n];
    double const k = (k4[0] + k4[1]) + (k4[2] + k4[3]);
    double *fp = F + int64_t(a) * ldf + c;
    double v   = alpha_j * J[e] + alpha_k * k;
    if (beta != 0.0) v += beta * *fp;
    *fp = v;
}

} // namespace

int fock_jk_f64(int64_t n, double const *g, double const *D, int64_t ldd, double alpha_j, double alpha_k, double beta,
                double *F, int64_t ldf, hipStream_t stream) {
    if (n < 0) return fail(-1, "fock_jk: n < 0");
    if (ldd < std::max<int64_t>(1, n)) return fail(-4, "fock_jk: ldd < n");
    if (ldf < std::max<int64_t>(1, n)) return fail(-9, "fock_jk: ldf < n");
    if (n > FOCK_MAX_N)
        return fail(EIN_ERROR_UNSUPPORTED, "fock_jk: n = " + std::to_string(n) + " exceeds " + std::to_string(FOCK_MAX_N) +
                                               " (use the two einsum calls)");
    if (n == 0) return EIN_SUCCESS;
    if (g == nullptr || D == nullptr || F == nullptr) return fail(-2, "fock_jk: null pointer");
    bool const wide = n % 2 == 0 && ldd % 2 == 0 && reinterpret_cast<uintptr_t>(g) % 16 == 0 &&
                      reinterpret_cast<uintptr_t>(D) % 16 == 0;
    int const ni    = int(n);
    if (n > 64) {
        // units <= FOCK_UNITS <= n - 1, so a workgroup's slabs meet at most two values of a
        int const units = int(std::min<int64_t>(ceil_div(n * n, num_cus()), FOCK_UNITS));
        int const grid  = int(ceil_div(n * n, units));
        void *ws        = nullptr;
        EIN_TRY(workspace(stream, (size_t(n) * size_t(n) + 2 * size_t(grid) * size_t(n)) * sizeof(double), &ws));
        double *J  = static_cast<double *>(ws);
        double *Kp = J + size_t(n) * size_t(n);
        switch (int(ceil_div(n, FOCK_WAVES))) {
        case 5: launch_stream<5>(wide, grid, ni, units, g, D, ldd, J, Kp, stream); break;
        case 6: launch_stream<6>(wide, grid, ni, units, g, D, ldd, J, Kp, stream); break;
        case 7: launch_stream<7>(wide, grid, ni, units, g, D, ldd, J, Kp, stream); break;
        default: launch_stream<8>(wide, grid, ni, units, g, D, ldd, J, Kp, stream); break;
        }
        EIN_LAUNCH_CHECK();
        fock_finish_pieces_kernel<<<uint32_t(ceil_div(n * n, 256)), 256, 0, stream>>>(ni, units, J, Kp, alpha_j, alpha_k,
                                                                                    beta, F, ldf);
        EIN_LAUNCH_CHECK();
        return EIN_SUCCESS;
    }
    constexpr int bc = 4; // the kernels' BC
    int const chunks = int(ceil_div(n, bc));
    void *ws = nullptr;
    size_t const j_bytes = size_t(n) * size_t(n) * sizeof(double);
    size_t const k_bytes = size_t(n) * size_t(chunks) * size_t(n) * sizeof(double);
    EIN_TRY(workspace(stream, j_bytes + k_bytes, &ws));
    double *J  = static_cast<double *>(ws);
    double *Kp = J + size_t(n) * size_t(n);
    dim3 grid{uint32_t(n), uint32_t(chunks)};
    if (wide && n <= 32)
        fock_jk16_kernel<4, 4><<<grid, 256, 0, stream>>>(ni, g, D, ldd, J, Kp);
    else if (wide && n <= 48)
        fock_jk16_kernel<6, 4><<<grid, 256, 0, stream>>>(ni, g, D, ldd, J, Kp);
    else if (wide)
        fock_jk16_kernel<8, 4><<<grid, 256, 0, stream>>>(ni, g, D, ldd, J, Kp);
    else if (n <= 32)
        fock_jk_kernel<8, 4><<<grid, 256, 0, stream>>>(ni, g, D, ldd, J, Kp);
    else if (n <= 48)
        fock_jk_kernel<12, 4><<<grid, 256, 0, stream>>>(ni, g, D, ldd, J, Kp);
    else
        fock_jk_kernel<16, 4><<<grid, 256, 0, stream>>>(ni, g, D, ldd, J, Kp);
    EIN_LAUNCH_CHECK();
    fock_finish_kernel<<<uint32_t(ceil_div(n * n, 256)), 256, 0, stream>>>(int(n), chunks, J, Kp, alpha_j, alpha_k, beta,
                                                                         F, ldf);
    EIN_LAUNCH_CHECK();
    return EIN_SUCCESS;
}

} // namespace ein

extern "C" {

int ein_fock_jk_f64(int64_t n, const double *g, const double *D, int64_t ldd, double alpha_j, double alpha_k,
                    double beta, double *F, int64_t ldf, ein_stream_t stream) {
    return ein::fock_jk_f64(n, g, D, ldd, alpha_j, alpha_k, beta, F, ldf, ein::as_stream(stream));
}

} // extern "C"
