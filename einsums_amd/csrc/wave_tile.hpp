// MFMA tiles of one wave each, for contractions too small for LDS tiles: grouped plans,
// small dense GEMMs and small generic contractions share them.
#pragma once

#include <type_traits>

#include "contract.hpp"
#include "gemm_core.hpp"

namespace ein {

// One contraction as the wave kernel sees it: C[i,j] = alpha sum_p A[i,p] B[p,j] + beta C[i,j]
// with element offsets from tables. C's unit stride, if it has one, is along i.
template <typename T>
struct WaveItem {
    T const *A;
    T const *B;
    T *C;
    T alpha, beta;
    int64_t const *rowA, *rowC, *colB, *colC, *kA, *kB;
    int64_t kA_in, kB_in; // stride per contraction step where k_mode says so
    int64_t sA, sC, tB, tC; // strides of a single row digit (i) and column digit (j)
    int32_t m, n, k;
    int32_t k_mode; // 2: p * kA_in; 1: kA[p0] + (p - p0) * kA_in within 16 steps from p0; 0: kA[p]
    int32_t m_lin, n_lin; // offsets of i (j) are i * sA, i * sC (j * tB, j * tC): no table
};

// Offsets of a grouped item: strides where one digit makes them, tables otherwise.
template <typename T>
struct TableOffsets {
    WaveItem<T> const &it;
    __device__ __forceinline__ int64_t rowA(int i) const { return it.m_lin ? i * it.sA : it.rowA[i]; }
    __device__ __forceinline__ int64_t rowC(int i) const { return it.m_lin ? i * it.sC : it.rowC[i]; }
    __device__ __forceinline__ int64_t colB(int j) const { return it.n_lin ? j * it.tB : it.colB[j]; }
    __device__ __forceinline__ int64_t colC(int j) const { return it.n_lin ? j * it.tC : it.colC[j]; }
    __device__ __forceinline__ int64_t kA(int p) const { return it.kA[p]; }
    __device__ __forceinline__ int64_t kB(int p) const { return it.kB[p]; }
};

struct WaveTile {
    int32_t item, tm, tn, pad; // tile (tm, tn) of the item, in units of its wave tile
    int64_t oa, ob, oc;        // batch offsets
};

// Blocks of 16 rows (columns) in a wave tile: as many as the extent fills, up to most.
__host__ __device__ __forceinline__ int wave_blocks(int64_t extent, int most) {
    return extent <= 16 ? 1 : extent <= 32 || most < 4 ? 2 : 4;
}

// One wave's tile of 16*FM x 16*FN of C. The operands go from global memory straight to the
// registers that feed the MFMA, 16 contraction steps at a time, the next 16 in flight during
// the MFMAs: tiles of the small blocks that a grouped plan is made of share little that LDS
// could hold for them, and without it there is no barrier, no padding to a slab layout, and
// any alignment takes whole elements. Rows and columns outside the problem read its last one
// and are not stored; steps beyond k are zeros in both operands. What bounds a plan of many
// small items is the latency of a tile's first loads, so several waves share a SIMD and only
// multi-digit indices go through tables. 1024 FP64 GEMMs with extents 4..512 took 1022 us with
// 64/128 x 64 LDS tiles in a persistent walk, and take 133; 4096 of them 3.24 -> 0.51 ms
// (FP32 1.20 -> 0.32); 2048 of 32 x 32 x 256 619 -> 53 us; 64 of 384^3 823 -> 198 (36 TFLOP/s).
//
// With KS > 1 the block's KS waves share one tile, each takes whole chunks of the contraction,
// and the first adds the others' sums, in order, through LDS (KS * 64 * FM * FN * 4 elements).
template <int FM, int FN, int KS = 1, typename T, typename Offsets>
__device__ __forceinline__ void wave_tile(WaveItem<T> const &it, WaveTile const &e, Offsets const &off, int lane,
                                          int part = 0, T *sums = nullptr) {
    int const r  = lane & 15;
    int const q  = lane >> 4;
    int const i0 = e.tm * 16 * FM, j0 = e.tn * 16 * FN;
    int const per  = KS == 1 ? it.k : 16 * ((it.k + 16 * KS - 1) / (16 * KS));
    int const from = part * per;
    int const k    = KS == 1 || it.k < from + per ? it.k : from + per;
    T const *pa[FM];
    T const *pb[FN];
#pragma unroll
    for (int a = 0; a < FM; ++a) {
        int const i = i0 + a * 16 + r;
        int const ic = i < it.m ? i : it.m - 1;
        pa[a]        = it.A + e.oa + off.rowA(ic);
    }
#pragma unroll
    for (int b = 0; b < FN; ++b) {
        int const j = j0 + b * 16 + r;
        int const jc = j < it.n ? j : it.n - 1;
        pb[b]        = it.B + e.ob + off.colB(jc);
    }
    typename Mfma<T>::acc_t acc[FM][FN];
#pragma unroll
    for (int a = 0; a < FM; ++a)
#pragma unroll
        for (int b = 0; b < FN; ++b)
#pragma unroll
            for (int v = 0; v < 4; ++v) acc[a][b][v] = T(0);

    struct Chunk {
        T a[FM][4], b[FN][4];
    };
    // Which of a chunk's 16 steps lane group q feeds to the s-th MFMA does not matter as long as
    // both operands agree. In a whole chunk it is V consecutive ones, so that an operand
    // contiguous along k is read 16 bytes at a time (from any element: the hardware takes
    // 16-byte loads at 4-byte alignment).
    constexpr int V = 16 / int(sizeof(T));
    typedef T vec_t __attribute__((ext_vector_type(V), aligned(sizeof(T))));
    auto load = [&](int k0, Chunk &x) {
        if (k0 + 16 <= k && it.k_mode != 0) {
            int64_t const ba = it.k_mode == 2 ? k0 * it.kA_in : off.kA(k0);
            int64_t const bb = it.k_mode == 2 ? k0 * it.kB_in : off.kB(k0);
            auto operand = [&](auto const &ptr, int64_t base, int64_t step, auto &out, auto blocks) {
                constexpr int NBK = decltype(blocks)::value;
                if (step == 1) {
#pragma unroll
                    for (int h = 0; h < 4 / V; ++h)
#pragma unroll
                        for (int a = 0; a < NBK; ++a) {
                            vec_t const t = *reinterpret_cast<vec_t const *>(ptr[a] + base + 4 * V * h + V * q);
#pragma unroll
                            for (int v = 0; v < V; ++v) out[a][V * h + v] = t[v];
                        }
                } else {
#pragma unroll
                    for (int s = 0; s < 4; ++s) {
                        int64_t const o = base + (4 * V * (s / V) + V * q + s % V) * step;
#pragma unroll
                        for (int a = 0; a < NBK; ++a) out[a][s] = ptr[a][o];
                    }
                }
            };
            operand(pa, ba, it.kA_in, x.a, std::integral_constant<int, FM>{});
            operand(pb, bb, it.kB_in, x.b, std::integral_constant<int, FN>{});
        } else {
#pragma unroll
            for (int s = 0; s < 4; ++s) {
                if (k0 + 4 * s >= k) break;
                int const p0     = k0 + 4 * s + q;
                bool const in    = p0 < k;
                int const p      = in ? p0 : k - 1;
                int64_t const oa = it.k_mode == 2 ? p * it.kA_in : off.kA(p);
                int64_t const ob = it.k_mode == 2 ? p * it.kB_in : off.kB(p);
#pragma unroll
                for (int a = 0; a < FM; ++a) {
                    T const t  = pa[a][oa];
                    x.a[a][s] = in ? t : T(0);
                }
#pragma unroll
                for (int b = 0; b < FN; ++b) {
                    T const t  = pb[b][ob];
                    x.b[b][s] = in ? t : T(0);
                }
            }
        }
    };
    auto multiply = [&](int k0, Chunk const &x) {
#pragma unroll
        for (int s = 0; s < 4; ++s) {
            if (k0 + 4 * s >= k) break;
#pragma unroll
            for (int a = 0; a < FM; ++a)
#pragma unroll
                for (int b = 0; b < FN; ++b) acc[a][b] = Mfma<T>::mma(x.b[b][s], x.a[a][s], acc[a][b]);
        }
    };
    Chunk x, y;
    if (KS == 1 || from < k) load(from, x);
    for (int k0 = from; k0 < k; k0 += 32) {
        if (k0 + 16 < k) load(k0 + 16, y);
        multiply(k0, x);
        if (k0 + 16 >= k) break;
        if (k0 + 32 < k) load(k0 + 32, x);
        multiply(k0 + 16, y);
    }

    if constexpr (KS > 1) {
#pragma unroll
        for (int a = 0; a < FM; ++a)
#pragma unroll
            for (int b = 0; b < FN; ++b)
#pragma unroll
                for (int v = 0; v < 4; ++v)
                    sums[(((part * FM + a) * FN + b) * 4 + v) * 64 + lane] = acc[a][b][v];
        __syncthreads();
        if (part != 0) return;
#pragma unroll
        for (int w = 1; w < KS; ++w)
#pragma unroll
            for (int a = 0; a < FM; ++a)
#pragma unroll
                for (int b = 0; b < FN; ++b)
#pragma unroll
                    for (int v = 0; v < 4; ++v)
                        acc[a][b][v] += sums[(((w * FM + a) * FN + b) * 4 + v) * 64 + lane];
    }

    T *__restrict__ C = it.C + e.oc;
#pragma unroll
    for (int a = 0; a < FM; ++a) {
        int const i = i0 + a * 16 + r;
        if (i >= it.m) continue;
        T *ci = C + off.rowC(i);
#pragma unroll
        for (int b = 0; b < FN; ++b) {
            int64_t oc[4];
            T old[4];
#pragma unroll
            for (int v = 0; v < 4; ++v) {
                int const j = j0 + b * 16 + Mfma<T>::row(q, v);
                int const jc = j < it.n ? j : it.n - 1;
                oc[v]        = off.colC(jc);
                old[v]      = it.beta != T(0) && j < it.n ? ci[oc[v]] : T(0);
            }
#pragma unroll
            for (int v = 0; v < 4; ++v)
                if (j0 + b * 16 + Mfma<T>::row(q, v) < it.n)
                    ci[oc[v]] = it.beta != T(0) ? it.alpha * acc[a][b][v] + it.beta * old[v] : it.alpha * acc[a][b][v];
        }
    }
}

// A single problem: the offsets come from its index groups, decoded in the kernel (no table, no
// second launch), or for a dense GEMM from strides alone.
template <typename T>
struct WaveLaunch {
    WaveItem<T> it;
    IndexGroup gm, gn, gk, gb; // (A, C), (B, C), (A, B) and (A, B, C) strides
    int64_t a_sb, b_sb, c_sb;  // batch strides of a dense GEMM
    int64_t batch;
    uint32_t tiles_m, tiles_n, ntiles;
    uint32_t first; // tile of the launch's first wave
};

template <typename T>
struct DecodeOffsets {
    WaveLaunch<T> const &P;
    __device__ __forceinline__ int64_t at(IndexGroup const &G, int i, int o) const {
        int64_t x[2];
        group_decode<2>(uint32_t(i), G, x);
        return x[o];
    }
    __device__ __forceinline__ int64_t rowA(int i) const { return P.it.m_lin ? i * P.it.sA : at(P.gm, i, 0); }
    __device__ __forceinline__ int64_t rowC(int i) const { return P.it.m_lin ? i * P.it.sC : at(P.gm, i, 1); }
    __device__ __forceinline__ int64_t colB(int j) const { return P.it.n_lin ? j * P.it.tB : at(P.gn, j, 0); }
    __device__ __forceinline__ int64_t colC(int j) const { return P.it.n_lin ? j * P.it.tC : at(P.gn, j, 1); }
    __device__ __forceinline__ int64_t kA(int p) const { return at(P.gk, p, 0); }
    __device__ __forceinline__ int64_t kB(int p) const { return at(P.gk, p, 1); }
};

template <typename T>
struct DenseOffsets {
    WaveItem<T> const &it;
    __device__ __forceinline__ int64_t rowA(int i) const { return i * it.sA; }
    __device__ __forceinline__ int64_t rowC(int i) const { return i * it.sC; }
    __device__ __forceinline__ int64_t colB(int j) const { return j * it.tB; }
    __device__ __forceinline__ int64_t colC(int j) const { return j * it.tC; }
    __device__ __forceinline__ int64_t kA(int) const { return 0; } // k_mode 2: not asked for
    __device__ __forceinline__ int64_t kB(int) const { return 0; }
};

template <typename T, int FM, int FN, int KS, bool DENSE>
__global__ __launch_bounds__(KS == 1 ? GEMM_THREADS : 64 * KS, KS > 4 ? 1 : 2) void wave_kernel(WaveLaunch<T> P) {
    int const w      = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    uint32_t const t = KS == 1 ? P.first + blockIdx.x * 4 + w : blockIdx.x;
    if (t >= P.ntiles) return;
    __shared__ T sums[KS == 1 ? 1 : KS * FM * FN * 256];
    uint32_t const mn = P.tiles_m * P.tiles_n;
    uint32_t const z  = t / mn, x = t - z * mn;
    WaveTile e{};
    e.tn = int32_t(x / P.tiles_m);
    e.tm = int32_t(x - uint32_t(e.tn) * P.tiles_m);
    int const lane = threadIdx.x & 63;
    if constexpr (DENSE) {
        e.oa = int64_t(z) * P.a_sb;
        e.ob = int64_t(z) * P.b_sb;
        e.oc = int64_t(z) * P.c_sb;
        wave_tile<FM, FN, KS>(P.it, e, DenseOffsets<T>{P.it}, lane, KS == 1 ? 0 : w, sums);
    } else {
        int64_t o[3];
        group_decode<3>(z, P.gb, o);
        e.oa = o[0];
        e.ob = o[1];
        e.oc = o[2];
        wave_tile<FM, FN, KS>(P.it, e, DecodeOffsets<T>{P}, lane, KS == 1 ? 0 : w, sums);
    }
}

// A grid holds fewer than 2^32 threads (beyond, it is cut without an error), so this many tiles
// of a wave each, four to a workgroup, are the most of one launch; longer lists go in parts.
constexpr uint32_t WAVE_TILES_MAX = (1u << 26) - 4;

template <typename F>
int for_wave_parts(uint32_t ntiles, F const &launch) {
    for (uint32_t first = 0; first < ntiles;) {
        uint32_t const count = ntiles - first < WAVE_TILES_MAX ? ntiles - first : WAVE_TILES_MAX;
        EIN_TRY(launch(first, count));
        first += count;
    }
    return EIN_SUCCESS;
}

template <typename T, int FM, int FN, int KS, bool DENSE>
int launch_wave_tiles(WaveLaunch<T> &P, hipStream_t stream) {
    int64_t const tm = ceil_div(P.it.m, 16 * FM), tn = ceil_div(P.it.n, 16 * FN);
    if (tm * tn * P.batch > 0x7fffffff) return fail(EIN_ERROR_UNSUPPORTED, "contraction tile grid too large");
    P.tiles_m = uint32_t(tm);
    P.tiles_n = uint32_t(tn);
    P.ntiles  = uint32_t(tm * tn * P.batch);
    if constexpr (KS > 1) { // few tiles (launch_wave)
        wave_kernel<T, FM, FN, KS, DENSE><<<P.ntiles, 64 * KS, 0, stream>>>(P);
        EIN_LAUNCH_CHECK();
        return EIN_SUCCESS;
    } else {
        return for_wave_parts(P.ntiles, [&](uint32_t first, uint32_t count) {
            P.first = first;
            wave_kernel<T, FM, FN, KS, DENSE><<<uint32_t(ceil_div(count, 4)), GEMM_THREADS, 0, stream>>>(P);
            EIN_LAUNCH_CHECK();
            return EIN_SUCCESS;
        });
    }
}

// Whether a problem is small for tiles staged through LDS: fewer of their 64 x 64 tiles than
// max_tiles, each a serial chain of barriers, leave most of the chip idle, while a wave of
// 16 x 16 to 64 x 32 has up to eight waves for every SIMD. Above 0.4 GFLOP the LDS kernel has
// the operands' reuse that a wave lacks (FP64 640^3 NT 24 us, here 38; 768^3 33, here 67), and
// above 32768 steps its split over the whole chip beats 16 waves to a tile (16 x 16 x 100000
// 352 us, here 519; 64 x 64 x 32768 388, here 175).
inline bool wave_small(int64_t m, int64_t n, int64_t k, int64_t batch, int64_t max_tiles, double max_flops = 4e8) {
    return k <= 32768 && ceil_div(m, 64) * ceil_div(n, 64) <= max_tiles / batch &&
           2.0 * double(m) * double(n) * double(k) * double(batch) <= max_flops;
}

// Whether the wave kernel can index a problem at all.
inline bool wave_fits(int64_t m, int64_t n, int64_t k, int64_t batch) {
    int64_t const most = int64_t{1} << 30;
    auto extent        = [&](int64_t x) { return x > 0 && x < most; };
    return extent(m) && extent(n) && extent(k) && extent(batch) && ceil_div(m, 16) * ceil_div(n, 16) < most / batch;
}

// Launches one problem with the largest tiles that still give every SIMD (four per CU) one, and
// where even 16 x 16 ones do not, with several waves to a tile: the latency of their loads is
// the time, so up to eight waves a SIMD are worth it with 4 to a tile (560^3 FP64 27.1 -> 19.6
// us), up to four with 16, whose sums cost more (300 x 300 x 600 9.0 us with 4, 12.8 with 16).
// FP64 256^3 23 us with LDS tiles, 9.1 with one wave to a tile, 4.8 with 4; 128 x 128 x 4096 304,
// 101 and (16) 26; a 24 x 24 x 13824 product 694, 507 and (16) 77.
template <typename T, bool DENSE>
int launch_wave(WaveLaunch<T> &P, hipStream_t stream) {
    int64_t const simds = 4 * int64_t(num_cus());
    int fm = wave_blocks(P.it.m, 4), fn = wave_blocks(P.it.n, 2);
    auto tiles = [&](int a, int b) { return ceil_div(P.it.m, 16 * a) * ceil_div(P.it.n, 16 * b) * P.batch; };
    while ((fm > 1 || fn > 1) && tiles(fm, fn) < simds) {
        if (fm >= fn)
            fm /= 2;
        else
            fn /= 2;
    }
    if (fm == 4 && fn == 2) return launch_wave_tiles<T, 4, 2, 1, DENSE>(P, stream);
    if (fm == 4) return launch_wave_tiles<T, 4, 1, 1, DENSE>(P, stream);
    if (fm == 2 && fn == 2) return launch_wave_tiles<T, 2, 2, 1, DENSE>(P, stream);
    if (fm == 2) return launch_wave_tiles<T, 2, 1, 1, DENSE>(P, stream);
    if (fn == 2) return launch_wave_tiles<T, 1, 2, 1, DENSE>(P, stream);
    if (P.it.k >= 512 && 16 * tiles(1, 1) <= 4 * simds) return launch_wave_tiles<T, 1, 1, 16, DENSE>(P, stream);
    if (P.it.k >= 64 && 4 * tiles(1, 1) <= 8 * simds) return launch_wave_tiles<T, 1, 1, 4, DENSE>(P, stream);
    return launch_wave_tiles<T, 1, 1, 1, DENSE>(P, stream);
}

} // namespace ein
