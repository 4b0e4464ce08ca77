// Out-of-place tensor permutation C = beta*C + alpha*perm(A) for gfx950.
//
// Axis i of C is axis perm[i] of A (the convention of the reference permute_kernel,
// TensorAlgebra/Backends/DevicePermute.hpp:34-73, which writes B[.. idx[perm[i]] ..]).
// After dropping unit axes and merging axes that are contiguous in both tensors:
//   * if C's unit-stride axis is also A's unit-stride axis, an element-wise pass in C
//     order moves contiguous runs (both sides coalesced, 16-byte vectors when aligned);
//   * otherwise a 64x64 tile is staged through LDS (one padded row per tile row) so the
//     A read runs along A's unit-stride axis and the C write along C's, in 16-byte
//     vectors on full tiles of aligned operands;
// alpha == 1 and beta == 0 is a pure copy, so the result is bit-exact.
#include <algorithm>
#include <type_traits>
#include <vector>

#include "blas1.hpp"

namespace ein {

namespace {

constexpr int PMAX = EIN_MAX_RANK;

struct PermAxes {
    int32_t n;
    uint32_t ext[PMAX];
    FastDiv fd[PMAX];
    int64_t ext64[PMAX];
    int64_t sa[PMAX];
    int64_t sc[PMAX];
    int64_t total;
};

template <bool WIDE>
__device__ __forceinline__ void perm_decode(int64_t e, PermAxes const &P, int n, int64_t &oa, int64_t &oc) {
    oa = 0;
    oc = 0;
    if constexpr (WIDE) {
        for (int d = n - 1; d >= 0; --d) {
            int64_t q = e / P.ext64[d];
            int64_t r = e - q * P.ext64[d];
            oa += r * P.sa[d];
            oc += r * P.sc[d];
            e = q;
        }
    } else {
        uint32_t u = uint32_t(e);
        for (int d = n - 1; d >= 0; --d) {
            uint32_t q = fast_div(u, P.fd[d]);
            uint32_t r = u - q * P.ext[d];
            oa += int64_t(r) * P.sa[d];
            oc += int64_t(r) * P.sc[d];
            u = q;
        }
    }
}

template <typename T>
__device__ __forceinline__ T perm_value(T a, T const *cptr, T alpha, T beta, bool copy) {
    if (copy) return a;
    T v = alpha * a;
    if (beta != T(0)) v += beta * *cptr;
    return v;
}

// Element-wise pass in C order; the last axis is C's fastest. VEC consecutive
// elements of the last axis per thread (requires unit strides on that axis in both).
template <typename T, int VEC, bool WIDE>
__global__ __launch_bounds__(256) void permute_elem_kernel(PermAxes P, T alpha, T const *__restrict__ A, T beta,
                                                           T *__restrict__ C, int copy) {
    int64_t const stride = int64_t(gridDim.x) * blockDim.x;
    int64_t const nvec   = P.total / VEC;
    for (int64_t e = int64_t(blockIdx.x) * blockDim.x + threadIdx.x; e < nvec; e += stride) {
        int64_t oa, oc;
        perm_decode<WIDE>(e * VEC, P, P.n, oa, oc);
        if constexpr (VEC == 2) {
            using V  = typename std::conditional<sizeof(T) == 8, double2, float2>::type;
            V a      = *reinterpret_cast<V const *>(A + oa);
            V *cp    = reinterpret_cast<V *>(C + oc);
            if (copy) {
                *cp = a;
            } else {
                V c = beta != T(0) ? *cp : V{};
                V r;
                r.x = alpha * a.x + (beta != T(0) ? beta * c.x : T(0));
                r.y = alpha * a.y + (beta != T(0) ? beta * c.y : T(0));
                *cp = r;
            }
        } else {
            C[oc] = perm_value<T>(A[oa], C + oc, alpha, beta, copy != 0);
        }
    }
}

// TS x TS LDS tile transpose (TS = 64, or 32 where the extents are multiples of 32 but not
// of 64, so no tile is partial: the Wmbej operand pack at v = 96 has a 96-long axis). X = C's
// unit-stride axis (A stride ax), Y = A's unit-stride axis (C stride cy). Remaining axes (P,
// n entries) are decoded from the batch index. Every load of a tile is issued before its LDS
// writes (a load and LDS write under one bounds test per element serialised the loads: 4.3
// against 5.2 TB/s on a 2.4 GB transpose). Full tiles of operands whose strides and base
// addresses allow it (vec) move 16-byte vectors.
template <typename T, bool WIDE, int TS>
__global__ __launch_bounds__(256) void permute_tile_kernel(PermAxes P, int64_t ex, int64_t ax, int64_t ey, int64_t cy,
                                                           int64_t tiles_x, T alpha, T const *__restrict__ A, T beta,
                                                           T *__restrict__ C, int copy, int vec) {
    constexpr int VW  = 16 / int(sizeof(T)); // elements per 16-byte vector
    constexpr int LPR = TS / VW;             // lanes per tile row
    constexpr int RPP = 256 / LPR;           // tile rows per pass of the workgroup
    constexpr int NP  = TS / RPP;            // passes per tile
    constexpr int TPR = 256 / TS;            // thread rows of the element-wise path
    constexpr int NR  = TS / TPR;            // elements per thread of the element-wise path
    static_assert(NP >= 1 && NR >= 1, "tile too small for 256 threads");
    struct alignas(16) Vec {
        T v[VW];
    };
    __shared__ T tile[TS][TS + 1];
    int64_t const ntiles = tiles_x * ((ey + TS - 1) / TS);
    int const t          = threadIdx.x;
    for (int64_t b = blockIdx.y; b < P.total; b += gridDim.y) {
        int64_t oa, oc;
        perm_decode<WIDE>(b, P, P.n, oa, oc);
        for (int64_t tt = blockIdx.x; tt < ntiles; tt += gridDim.x) {
            int64_t const x0 = (tt % tiles_x) * TS;
            int64_t const y0 = (tt / tiles_x) * TS;
            bool const full  = vec != 0 && x0 + TS <= ex && y0 + TS <= ey;
            if (full) {
                int const c  = t % LPR;
                int const r0 = t / LPR;
                T const *src = A + oa + (x0 + r0) * ax + y0 + VW * c;
                Vec v[NP];
#pragma unroll
                for (int p = 0; p < NP; ++p) v[p] = *reinterpret_cast<Vec const *>(src + int64_t(p * RPP) * ax);
#pragma unroll
                for (int p = 0; p < NP; ++p)
#pragma unroll
                    for (int i = 0; i < VW; ++i) tile[r0 + p * RPP][VW * c + i] = v[p].v[i];
            } else {
                int const ly = t % TS;
                int const lx = t / TS;
                T v[NR];
#pragma unroll
                for (int r = 0; r < NR; ++r) {
                    int const x = lx + TPR * r;
                    v[r]        = (x0 + x < ex && y0 + ly < ey) ? A[oa + (x0 + x) * ax + (y0 + ly)] : T(0);
                }
#pragma unroll
                for (int r = 0; r < NR; ++r) tile[lx + TPR * r][ly] = v[r];
            }
            __syncthreads();
            if (full) {
                int const c  = t % LPR;
                int const r0 = t / LPR;
                T *dst       = C + oc + (y0 + r0) * cy + x0 + VW * c;
#pragma unroll
                for (int p = 0; p < NP; ++p) {
                    Vec w;
#pragma unroll
                    for (int i = 0; i < VW; ++i) w.v[i] = tile[VW * c + i][r0 + p * RPP];
                    Vec *cp = reinterpret_cast<Vec *>(dst + int64_t(p * RPP) * cy);
                    if (!copy) {
                        Vec const old = beta != T(0) ? *cp : Vec{};
#pragma unroll
                        for (int i = 0; i < VW; ++i) w.v[i] = alpha * w.v[i] + (beta != T(0) ? beta * old.v[i] : T(0));
                    }
                    *cp = w;
                }
            } else {
                int const lx = t % TS;
                int const ly = t / TS;
#pragma unroll
                for (int r = 0; r < NR; ++r) {
                    int y = ly + TPR * r;
                    if (x0 + lx < ex && y0 + y < ey) {
                        T *cp = C + oc + (y0 + y) * cy + (x0 + lx);
                        *cp   = perm_value<T>(tile[lx][y], cp, alpha, beta, copy != 0);
                    }
                }
            }
            __syncthreads();
        }
    }
}

// ext64 holds the true extents; ext/fd are only used by the 32-bit decode, which is
// selected only when every extent and the index range fit below 2^31.
void fill_divs(PermAxes &P) {
    for (int d = 0; d < P.n; ++d) {
        P.ext[d] = uint32_t(P.ext64[d] < (int64_t{1} << 31) ? P.ext64[d] : 1);
        P.fd[d]  = make_fastdiv(P.ext[d] == 0 ? 1u : P.ext[d]);
    }
}

struct MergedAx {
    int64_t e, sa, sc;
};

// The axes in C order without those of extent 1, those merged that are C-adjacent and contiguous
// in both tensors; `total` is the number of elements (no axes for 0).
std::vector<MergedAx> merged_axes(int32_t rank, int64_t const *dims_A, int32_t const *perm, int64_t const *strides_A,
                                  int64_t const *strides_C, int64_t &total) {
    std::vector<MergedAx> m;
    total = 1;
    for (int i = 0; i < rank; ++i) total *= dims_A[perm[i]];
    if (total == 0) return m;
    for (int i = 0; i < rank; ++i) {
        MergedAx const a{dims_A[perm[i]], strides_A[perm[i]], strides_C[i]};
        if (a.e == 1) continue;
        if (!m.empty() && m.back().sa == a.sa * a.e && m.back().sc == a.sc * a.e) {
            m.back().e *= a.e;
            m.back().sa = a.sa;
            m.back().sc = a.sc;
        } else {
            m.push_back(a);
        }
    }
    if (m.empty()) m.push_back({1, 1, 1});
    return m;
}

// C's and A's fastest axis; whether tiles of the two are transposed through LDS.
bool fastest_axes(std::vector<MergedAx> const &m, int &ic, int &ia) {
    ic = ia = 0;
    for (int i = 0; i < int(m.size()); ++i) {
        if (std::llabs(m[i].sc) < std::llabs(m[ic].sc)) ic = i;
        if (std::llabs(m[i].sa) < std::llabs(m[ia].sa)) ia = i;
    }
    return ic != ia && m[ic].sc == 1 && m[ia].sa == 1 && m[ic].e >= 16 && m[ia].e >= 16;
}

// 32-wide tiles where they leave no partial tile and 64-wide ones would
bool tiles_of_32(int64_t ex, int64_t ey) { return ex % 32 == 0 && ey % 32 == 0 && (ex % 64 != 0 || ey % 64 != 0); }

template <typename T>
int permute_impl(int32_t rank, int64_t const *dims_A, int32_t const *perm, T alpha, T const *A,
                 int64_t const *strides_A, T beta, T *C, int64_t const *strides_C, hipStream_t stream) {
    if (rank < 0 || rank > PMAX) return fail(-1, "permute: rank out of range");
    if (rank > 0 && (dims_A == nullptr || perm == nullptr || strides_A == nullptr || strides_C == nullptr))
        return fail(-2, "permute: null shape array");
    bool seen[PMAX] = {false};
    for (int i = 0; i < rank; ++i) {
        if (perm[i] < 0 || perm[i] >= rank || seen[perm[i]]) return fail(-3, "permute: perm is not a permutation");
        seen[perm[i]] = true;
        if (dims_A[i] < 0) return fail(-2, "permute: negative extent");
    }
    int64_t total            = 1;
    std::vector<MergedAx> const m = merged_axes(rank, dims_A, perm, strides_A, strides_C, total);
    if (total == 0) return EIN_SUCCESS;
    if (int(m.size()) > PMAX) return fail(EIN_ERROR_UNSUPPORTED, "permute: too many axes");
    int const copy = (alpha == T(1) && beta == T(0)) ? 1 : 0;

    int ic, ia;
    if (fastest_axes(m, ic, ia)) {
        PermAxes P{};
        P.n     = 0;
        P.total = 1;
        for (int i = 0; i < int(m.size()); ++i) {
            if (i == ic || i == ia) continue;
            P.ext64[P.n] = m[i].e;
            P.sa[P.n]    = m[i].sa;
            P.sc[P.n]    = m[i].sc;
            P.total *= m[i].e;
            ++P.n;
        }
        fill_divs(P);
        int64_t ex = m[ic].e, axs = m[ic].sa, ey = m[ia].e, cy = m[ia].sc;
        bool const t32   = tiles_of_32(ex, ey);
        int64_t const ts = t32 ? 32 : 64;
        int64_t tiles_x = ceil_div(ex, ts), tiles = tiles_x * ceil_div(ey, ts);
        int64_t gy      = std::min<int64_t>(P.total, 65535);
        // one tile per workgroup (tiles of one batch entry used to share a workgroup and ran
        // one after another)
        int64_t gx = std::min<int64_t>(tiles, 65535);
        bool const wide = P.total >= (int64_t{1} << 31);
        dim3 const grid{uint32_t(gx), uint32_t(gy)};
        // 16-byte vectors along both unit-stride axes: every batch offset, the row strides
        // and both base addresses must keep them aligned
        constexpr int VW = 16 / int(sizeof(T));
        bool vec = axs % VW == 0 && cy % VW == 0 && (reinterpret_cast<uintptr_t>(A) | reinterpret_cast<uintptr_t>(C)) % 16 == 0;
        for (int d = 0; d < P.n; ++d) vec = vec && P.sa[d] % VW == 0 && P.sc[d] % VW == 0;
        int const vf = vec ? 1 : 0;
        if (wide && t32)
            permute_tile_kernel<T, true, 32><<<grid, 256, 0, stream>>>(P, ex, axs, ey, cy, tiles_x, alpha, A, beta, C, copy, vf);
        else if (wide)
            permute_tile_kernel<T, true, 64><<<grid, 256, 0, stream>>>(P, ex, axs, ey, cy, tiles_x, alpha, A, beta, C, copy, vf);
        else if (t32)
            permute_tile_kernel<T, false, 32><<<grid, 256, 0, stream>>>(P, ex, axs, ey, cy, tiles_x, alpha, A, beta, C, copy, vf);
        else
            permute_tile_kernel<T, false, 64><<<grid, 256, 0, stream>>>(P, ex, axs, ey, cy, tiles_x, alpha, A, beta, C, copy, vf);
        EIN_LAUNCH_CHECK();
        return EIN_SUCCESS;
    }

    // element-wise in C order with C's fastest axis last
    PermAxes P{};
    P.n     = 0;
    P.total = total;
    for (int i = 0; i < int(m.size()); ++i) {
        if (i == ic) continue;
        P.ext64[P.n] = m[i].e;
        P.sa[P.n]    = m[i].sa;
        P.sc[P.n]    = m[i].sc;
        ++P.n;
    }
    P.ext64[P.n] = m[ic].e;
    P.sa[P.n]    = m[ic].sa;
    P.sc[P.n]    = m[ic].sc;
    ++P.n;
    fill_divs(P);
    bool const wide = total >= (int64_t{1} << 31);
    bool const vec2 = !wide && P.sa[P.n - 1] == 1 && P.sc[P.n - 1] == 1 && (m[ic].e % 2) == 0 &&
                      (reinterpret_cast<uintptr_t>(A) % (2 * sizeof(T)) == 0) &&
                      (reinterpret_cast<uintptr_t>(C) % (2 * sizeof(T)) == 0) && [&] {
                          for (int d = 0; d < P.n - 1; ++d)
                              if ((P.sa[d] % 2) != 0 || (P.sc[d] % 2) != 0) return false;
                          return true;
                      }();
    int64_t work   = vec2 ? total / 2 : total;
    // one element (vector) per thread: consecutive workgroups stream consecutive memory,
    // which measured 6.2 TB/s on a 2.4 GB copy against 4.5-4.8 TB/s for a grid-stride loop
    // over 2k-16k workgroups (the loop remains for what one grid, fewer than 2^32 threads, leaves)
    uint32_t grid  = uint32_t(std::max<int64_t>(1, std::min<int64_t>(ceil_div(work, 256), int64_t((1 << 24) - 1))));
    if (vec2)
        permute_elem_kernel<T, 2, false><<<grid, 256, 0, stream>>>(P, alpha, A, beta, C, copy);
    else if (wide)
        permute_elem_kernel<T, 1, true><<<grid, 256, 0, stream>>>(P, alpha, A, beta, C, copy);
    else
        permute_elem_kernel<T, 1, false><<<grid, 256, 0, stream>>>(P, alpha, A, beta, C, copy);
    EIN_LAUNCH_CHECK();
    return EIN_SUCCESS;
}

} // namespace

// What a permute reaches depends on its inner axes: tiles lose what their edges cut off, runs
// along one common fastest axis the part of a line that a short or odd run leaves, and where a
// fastest axis is too short for tiles, one side is scattered over lines (1 to 2 TB/s, more where
// the short axis and the other side's are neighbours). Of 260 permutes of 0.2 to 30 million
// elements the tiles and common axes took 0.6 to 1.5 times the estimate, the scattered ones
// 0.5 to 3.5 times, where one rate of 5 TB/s is exceeded up to 10 times.
double permute_time_us(int32_t rank, int64_t const *dims_A, int32_t const *perm, int64_t const *strides_A,
                       int64_t const *strides_C, int elem_bytes) {
    int64_t total;
    std::vector<MergedAx> const m = merged_axes(rank, dims_A, perm, strides_A, strides_C, total);
    if (total == 0) return 0.0;
    int ic, ia;
    bool const tiled = fastest_axes(m, ic, ia);
    bool const f64   = elem_bytes == 8;
    int64_t const ex = m[ic].e, ey = m[ia].e;
    double rate, launch = 2.0; // TB/s, us
    if (tiled) {
        int64_t const ts = tiles_of_32(ex, ey) ? 32 : 64;
        double const use = double(ex) * double(ey) / (double(ceil_div(ex, ts) * ts) * double(ceil_div(ey, ts) * ts));
        rate             = f64 ? 5.4 * std::min(1.0, 0.45 + use) : 4.5 * std::min(1.0, 0.3 + use);
        launch           = 3.5;
    } else if (ic == ia) {
        rate = f64 ? (ex >= 32 ? 5.2 : ex >= 8 ? 4.0 : 2.0) : ex >= 32 ? 3.8 : 2.1;
    } else {
        bool const near = (ex < 16 && m[ia].sc == ex) || (ey < 16 && m[ic].sa == ey);
        rate            = near ? 3.0 : f64 ? 1.8 : 1.5;
    }
    return launch + 2e-6 * elem_bytes * double(total) / rate;
}

template <typename T>
int permute_tensor(int32_t rank, int64_t const *dims_A, int32_t const *perm, T alpha, T const *A,
                   int64_t const *strides_A, T beta, T *C, int64_t const *strides_C, hipStream_t stream) {
    return permute_impl<T>(rank, dims_A, perm, alpha, A, strides_A, beta, C, strides_C, stream);
}
template int permute_tensor<double>(int32_t, int64_t const *, int32_t const *, double, double const *, int64_t const *,
                                    double, double *, int64_t const *, hipStream_t);
template int permute_tensor<float>(int32_t, int64_t const *, int32_t const *, float, float const *, int64_t const *, float,
                                   float *, int64_t const *, hipStream_t);

} // namespace ein

extern "C" {

int ein_permute_f64(int32_t rank, const int64_t *dims_A, const int32_t *perm, double alpha, const double *A,
                    const int64_t *strides_A, double beta, double *C, const int64_t *strides_C, ein_stream_t stream) {
    return ein::permute_impl<double>(rank, dims_A, perm, alpha, A, strides_A, beta, C, strides_C, ein::as_stream(stream));
}

int ein_permute_f32(int32_t rank, const int64_t *dims_A, const int32_t *perm, float alpha, const float *A,
                    const int64_t *strides_A, float beta, float *C, const int64_t *strides_C, ein_stream_t stream) {
    return ein::permute_impl<float>(rank, dims_A, perm, alpha, A, strides_A, beta, C, strides_C, ein::as_stream(stream));
}

} // extern "C"
