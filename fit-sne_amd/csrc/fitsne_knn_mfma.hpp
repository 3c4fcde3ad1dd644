// fitsne_knn_mfma.hpp -- k nearest neighbours on f16 matrix cores, with the exact FP64 result (gfx950).
//
// The FP64 kernel of fitsne_knn.hpp (the VP tree's distance, vptree.h:97-107, rounded the same way)
// costs N^2 D FP64 operations on the vector units.  Here the same neighbours come from a filter and a
// re-rank:
//  1. the data are centred, scaled by a power of two so that the largest coordinate lies in [1, 2), and
//     each coordinate is split into two halves, x = xh + xl (22 bits and more); a dot product is the
//     three products xh.yl + xl.yh + xh.yh on v_mfma_f32_32x32x16_f16, accumulated in FP32;
//  2. six further coordinates carry the norms (each split into three halves, exactly 33 bits, times 1),
//     so that the accumulator comes out as  -|x - y|^2 / 2  plus a constant of the query, and the
//     selection is a comparison with 0 instead of arithmetic on every pair;
//  3. threshold: over a sample of the points (every `stride`-th) a distance that about 33 of them are
//     nearer to each query than, so about 33 strides of all points;
//  4. candidates: the same over all points, those nearer than the threshold go to the query's list
//     with their approximate distance;
//  5. exact: of the list, only the points whose approximate distance can belong to the K nearest (two
//     error bounds beyond the K-th) get their FP64 distance in the reference's order and rounding, are
//     sorted by (distance, index) like the FP64 kernel's, and the first K kept.
// Why it is exact: knn_err below bounds the difference between the accumulator and the true value.  A
// point left out of the list has a true distance of at least the threshold less that bound; if the K-th
// exact distance is below it, no point left out can be among the K nearest.  A query whose list is
// short, overflows or fails that margin is recomputed by the FP64 kernel.
//
// The halves are stored tile by tile as the matrix instruction reads them: 32 points x 16 coordinates are
// 64 lanes x 8 halves (lane l: point l % 32, coordinates 8 (l / 32) ..), 1 KB, first the xh, then the xl,
// so a tile goes to LDS by 16-byte direct loads in order and comes back as 16-byte reads without bank
// conflicts.  A wavefront keeps 64 queries (two tiles) in registers; the workgroup's four wavefronts
// share the staged points.  Result element v of lane l: query 8 (v / 4) + 4 (l / 32) + v % 4, point l % 32.
#pragma once

#include <cfloat>
#include <climits>

#include "fitsne_common.hpp"
#include "fitsne_knn.hpp"

namespace fitsne {

constexpr int kKmWaves = 4;                    // wavefronts per workgroup
constexpr int kKmThreads = kKmWaves * kWave;
constexpr int kKmT = 2;                        // query tiles of 32 per wavefront
constexpr int kKmQ = kKmT * 32;                // queries per wavefront
constexpr int kKmWg = kKmWaves * kKmQ;         // queries per workgroup
constexpr int kKmRank = 26;                    // the threshold: sample points of this many classes are nearer
constexpr int kKmQueue = 2048;                 // candidate pass: queued hits per workgroup
constexpr int kKmAug = 6;                      // the last coordinates of the last chunk: the norms
constexpr int kKmMaxCh = 9;                    // chunks of 16 coordinates: D + 6 <= 144
constexpr int kKmMaxD = 128, kKmMaxK = 256;
constexpr double kKmNever = -60000.0;          // a constant that keeps every accumulator below 0 (they reach 2,048)

typedef _Float16 f16x8 __attribute__((ext_vector_type(8)));
typedef _Float16 f16x4 __attribute__((ext_vector_type(4)));
typedef float f32x16 __attribute__((ext_vector_type(16)));

// Points staged per step: two tiles while two double-buffered stages fit twice in a CU's LDS.
template <int NCH>
constexpr int kKmCt = NCH <= 7 ? 2 : 1;

// The data's scale and the largest centred norm, filled by k_knn_scale.
struct KnnScale {
    double scale;  // power of two: the largest |x_d - mean_d| times it lies in [1, 2)
    double nmax;   // largest scaled squared norm
};

// Bound on |accumulator - true value| for a query of scaled squared norm nq whose constant has magnitude
// c, with u = 2^-23 for one rounding (twice the unit roundoff) and any order of the additions inside an
// instruction:
//   * the small products xh.yl and xl.yh come first, so that their 2 Kp additions round values 2^-10 of
//     the rest: with the dropped xl.yl and the halves' own 2^-22 less than 6 u |x||y|;
//   * the Kp additions of xh.yh round partial sums of at most |x||y| <= (nq + nmax) / 2, those of the
//     last two chunks (the norms) at most nq + nmax + c;
//   * f16's subnormal spacing: 2^-25 per coordinate, by sqrt(D) <= 12 against the norms, and the split
//     constants.
__host__ __device__ __forceinline__ double knn_err(double nq, double nmax, double c, int kp) {
    const double u = 1.0 / 8388608.0;
    return u * ((0.5 * kp + 38.0) * (nq + nmax) + 34.0 * c + 4.0 * (sqrt(nq) + sqrt(nmax)) + 2.0);
}

// Column sums of X[N][D] (D <= kKmMaxD) over blocks of kKmRows rows, then their total: mean[d].  Thread
// (r, d) of a block takes every (256 / W)-th row, W the power of two from D on; the r parts add up in LDS.
constexpr int kKmRows = 256;
__device__ __forceinline__ int knn_width(int D) { return D <= 1 ? 1 : 1 << (32 - __clz(D - 1)); }
__global__ __launch_bounds__(256) void k_knn_colsum(const double *__restrict__ X, int N, int D,
                                                    double *__restrict__ part) {
    __shared__ double sh[256];
    const int W = knn_width(D), d = threadIdx.x % W, r0 = blockIdx.x * kKmRows, r1 = min(N, r0 + kKmRows);
    double s = 0;
    if (d < D) {
#pragma unroll 8
        for (int r = r0 + threadIdx.x / W; r < r1; r += 256 / W) s += X[(long)r * D + d];
    }
    sh[threadIdx.x] = s;
    __syncthreads();
    if (threadIdx.x < D) {
        for (int i = threadIdx.x + W; i < 256; i += W) s += sh[i];
        part[(long)blockIdx.x * D + d] = s;
    }
}
__global__ __launch_bounds__(1024) void k_knn_colmean(const double *__restrict__ part, int nblk, int N, int D,
                                                      double *__restrict__ mean) {
    __shared__ double sh[1024];
    const int W = knn_width(D), d = threadIdx.x % W;
    double s = 0;
    if (d < D) {
#pragma unroll 8
        for (int b = threadIdx.x / W; b < nblk; b += 1024 / W) s += part[(long)b * D + d];
    }
    sh[threadIdx.x] = s;
    __syncthreads();
    if (threadIdx.x < D) {
        for (int i = threadIdx.x + W; i < 1024; i += W) s += sh[i];
        s /= (double)N;
        mean[d] = fabs(s) <= DBL_MAX ? s : 0.0;  // sums of huge coordinates may overflow: leave those uncentred
    }
}

// Per block of 256 points: the largest centred |coordinate| (unscaled).
__global__ __launch_bounds__(256) void k_knn_extent(const double *__restrict__ X, int N, int D,
                                                    const double *__restrict__ mean, double *__restrict__ part) {
    const int lane = threadIdx.x % kWave, wv = threadIdx.x / kWave;
    double m = 0;
    for (int r = blockIdx.x * 256 + wv; r < min(N, (int)(blockIdx.x + 1) * 256); r += 4)
        for (int d = lane; d < D; d += kWave) m = fmax(m, fabs(X[(long)r * D + d] - mean[d]));
    m = wave_max(m);
    __shared__ double sh[4];
    if (lane == 0) sh[wv] = m;
    __syncthreads();
    if (threadIdx.x == 0) part[blockIdx.x] = fmax(fmax(sh[0], sh[1]), fmax(sh[2], sh[3]));
}
// The scale.  0 (every halves zero, so no point passes a threshold and every query goes to the FP64 kernel)
// where the filter's error bound would not hold: coordinates so small or large that FP64 squares under- or
// overflow, or a mean so far off that centring leaves less than f16's two halves resolve.
__global__ __launch_bounds__(1024) void k_knn_scale(const double *__restrict__ part, int nblk,
                                                    const double *__restrict__ mean, int D,
                                                    KnnScale *__restrict__ out) {
    double m = 0, mm = 0;
    for (int b = threadIdx.x; b < nblk; b += 1024) m = fmax(m, part[b]);
    for (int d = threadIdx.x; d < D; d += 1024) mm = fmax(mm, fabs(mean[d]));
    m = wave_max(m);
    mm = wave_max(mm);
    __shared__ double sh[2][1024 / kWave];
    if (threadIdx.x % kWave == 0) {
        sh[0][threadIdx.x / kWave] = m;
        sh[1][threadIdx.x / kWave] = mm;
    }
    __syncthreads();
    if (threadIdx.x == 0) {
        for (int i = 1; i < 1024 / kWave; i++) {
            m = fmax(m, sh[0][i]);
            mm = fmax(mm, sh[1][i]);
        }
        const bool ok = m > ldexp(1.0, -400) && m < ldexp(1.0, 400) && mm < m * ldexp(1.0, 26);
        out->scale = ok ? ldexp(1.0, -ilogb(m)) : 0.0;
        out->nmax = 0;
    }
}
// nmax = max of v[0 .. n) (one workgroup of 1024).
__global__ __launch_bounds__(1024) void k_knn_nmax(const double *__restrict__ v, int n, KnnScale *__restrict__ out) {
    double m = 0;
    for (int b = threadIdx.x; b < n; b += 1024) m = fmax(m, v[b]);
    m = wave_max(m);
    __shared__ double sh[1024 / kWave];
    if (threadIdx.x % kWave == 0) sh[threadIdx.x / kWave] = m;
    __syncthreads();
    if (threadIdx.x == 0) {
        for (int i = 1; i < 1024 / kWave; i++) m = fmax(m, sh[i]);
        out->nmax = m;
    }
}

// v as three halves (exact to 2^-33 of v, or f16's subnormal spacing); |v| < 65504.
__device__ __forceinline__ f16x4 knn_split3(double v) {
    const _Float16 a = (_Float16)(float)v;
    const double r = v - (double)a;
    const _Float16 b = (_Float16)(float)r;
    return f16x4{a, b, (_Float16)(float)(r - (double)b), (_Float16)0.f};
}

// Halves of every point as candidate, its scaled squared norm nrm[n], the block's largest norm, and of
// every stride-th point the same in the sample tiles XS.  A workgroup takes one tile of 32 points through
// LDS: coalesced reads of X, 1 KB contiguous writes per chunk and half.  Tiles past N, up to npad points,
// and the end of the sample's last tile are padding whose accumulator stays far below 0.
__global__ __launch_bounds__(256) void k_knn_prep(const double *__restrict__ X, int N, int D, int nch,
                                                  const double *__restrict__ mean, const KnnScale *__restrict__ sc,
                                                  int stride, int NS, int nspad, f16x8 *__restrict__ XC,
                                                  f16x8 *__restrict__ XS, double *__restrict__ nrm,
                                                  double *__restrict__ part) {
    __shared__ double x[32][kKmMaxD + 1];
    __shared__ double sn[32];
    const int n0 = blockIdx.x * 32, rows = max(0, min(32, N - n0)), t = threadIdx.x;
    const double s = sc->scale;
    for (int e = t; e < rows * D; e += 256) {
        const int r = e / D, d = e - r * D;
        x[r][d] = (X[(long)n0 * D + e] - mean[d]) * s;
    }
    __syncthreads();
    {  // norms: 8 threads per point
        const int r = t / 8;
        double v = 0;
        if (r < rows)
            for (int d = t % 8; d < D; d += 8) v += x[r][d] * x[r][d];
        for (int o = 4; o > 0; o >>= 1) v += __shfl_xor(v, o, 8);
        if (t % 8 == 0) {
            sn[r] = v;
            if (r < rows) nrm[n0 + r] = v;
        }
    }
    __syncthreads();
    if (t == 0) {
        double m = 0;
        for (int r = 0; r < rows; r++) m = fmax(m, sn[r]);
        part[blockIdx.x] = m;
    }
    auto pieces = [&](int r, int c, int g, bool real, f16x8 &h, f16x8 &l) {
        const f16x4 b = knn_split3(real ? -0.5 * sn[r] : kKmNever);
#pragma unroll
        for (int j = 0; j < 8; j++) {
            const int k = 16 * c + 8 * g + j;
            h[j] = (_Float16)0.f;
            l[j] = (_Float16)0.f;
            if (k < D && real) {
                h[j] = (_Float16)(float)x[r][k];
                l[j] = (_Float16)(float)(x[r][k] - (double)h[j]);
            }
        }
        if (c == nch - 1 && g == 1) {
            h[2] = b[0];
            h[3] = b[1];
            h[4] = b[2];
            h[5] = h[6] = h[7] = (_Float16)1.f;
        }
    };
    for (int e = t; e < nch * kWave; e += 256) {
        const int c = e / kWave, lane = e % kWave, r = lane % 32, g = lane / 32, n = n0 + r;
        f16x8 h, l;
        pieces(r, c, g, r < rows, h, l);
        f16x8 *base = XC + ((long)blockIdx.x * nch + c) * 2 * kWave + lane;
        base[0] = h;
        base[kWave] = l;
        if (r < rows && n % stride == 0) {
            const int slot = n / stride;
            base = XS + ((long)(slot / 32) * nch + c) * 2 * kWave + g * 32 + slot % 32;
            base[0] = h;
            base[kWave] = l;
        }
    }
    if (blockIdx.x == 0)  // padding of the sample's last tile
        for (int e = t; e < nch * 2 * (nspad - NS); e += 256) {
            const int slot = NS + e / (nch * 2), c = e % (nch * 2) / 2, g = e % 2;
            f16x8 h, l;
            pieces(0, c, g, false, h, l);
            f16x8 *base = XS + ((long)(slot / 32) * nch + c) * 2 * kWave + g * 32 + slot % 32;
            base[0] = h;
            base[kWave] = l;
        }
}

// The query's constant -|x|^2 / 2 - cut[q] as three halves (cut null: no threshold yet).  Queries past N, and with
// kKmNever as their constant also those that the exact pass must refuse in any case (the threshold lies within the
// error bound of distance zero: many coinciding points, or a scale set by far outliers), never pass.
__global__ __launch_bounds__(256) void k_knn_query(const double *__restrict__ nrm, int N, int npad, int kp,
                                                   const float *__restrict__ cut, const KnnScale *__restrict__ sc,
                                                   f16x4 *__restrict__ QA) {
    const int q = blockIdx.x * 256 + threadIdx.x;
    if (q >= npad) return;
    double c = kKmNever;
    if (q < N) {
        const double k = cut ? (double)cut[q] : 0.0;
        if (!cut || knn_err(nrm[q], sc->nmax, fabs(k), kp) < -k) c = -0.5 * nrm[q] - k;
    }
    QA[q] = knn_split3(c);
}

// The sweep both passes share: the workgroup's queries q0 .. q0 + 255 of XQ (candidate tiles, the norm
// coordinates replaced by 1 and QA) against tiles t0, t0 + TS, .. below t1 of XC.  visit(t, j0, acc) runs per wavefront for
// its query tile t and the 32 points from j0; step(s) by the whole workgroup before each stage.
// Bound: the matrix cores.  A stage of 64 points costs a wavefront 12 NCH instructions of 32 cycles, for
// one barrier and 6 KB NCH of LDS reads (half the LDS rate at eight wavefronts per CU); the next stage is
// loaded straight to LDS meanwhile.
template <int NCH, int TS, typename V, typename S>
__device__ __forceinline__ void knn_sweep(const f16x8 *__restrict__ XQ, const f16x4 *__restrict__ QA, int q0,
                                          const f16x8 *__restrict__ XC, int t0, int t1, f16x8 *stage, V &&visit,
                                          S &&step) {
    constexpr int CT = kKmCt<NCH>, TILE = NCH * 2 * kWave;  // f16x8 per tile
    const int w = threadIdx.x / kWave, l = threadIdx.x % kWave;
    f16x8 a[kKmT][NCH][2];
#pragma unroll
    for (int t = 0; t < kKmT; t++) {
        const int qt = (q0 + w * kKmQ) / 32 + t;
        const f16x4 qa = QA[qt * 32 + l % 32];
#pragma unroll
        for (int c = 0; c < NCH; c++) {
            a[t][c][0] = XQ[(long)qt * TILE + (c * 2 + 0) * kWave + l];
            a[t][c][1] = XQ[(long)qt * TILE + (c * 2 + 1) * kWave + l];
        }
        if (l >= 32) {  // the norm coordinates: 1, 1, 1, and the query's constant
            f16x8 &h = a[t][NCH - 1][0];
            h[2] = h[3] = h[4] = (_Float16)1.f;
            h[5] = qa[0];
            h[6] = qa[1];
            h[7] = qa[2];
        }
    }
    // 1 KB pieces of a stage, dealt over the wavefronts; pieces past the last tile are not read
    auto load = [&](int tile, f16x8 *dst) {
        const int pieces = min(CT, (t1 - tile + TS - 1) / TS) * NCH * 2;
        for (int p = w; p < pieces; p += kKmWaves) {
            const f16x8 *src = XC + (long)(tile + p / (NCH * 2) * TS) * TILE + p % (NCH * 2) * kWave;
            __builtin_amdgcn_global_load_lds((const __attribute__((address_space(1))) void *)(src + l),
                                             (__attribute__((address_space(3))) void *)(dst + p * kWave), 16, 0, 0);
        }
    };
    if (t0 < t1) load(t0, stage);
    int s = 0;
    for (int tile = t0; tile < t1; tile += CT * TS, s++) {
        __builtin_amdgcn_s_waitcnt(0x0f70);  // vmcnt(0): this wavefront's pieces are in LDS
        __syncthreads();
        step(s);
        const f16x8 *b = stage + (s & 1) * CT * TILE;
        if (tile + CT * TS < t1) load(tile + CT * TS, stage + ((s + 1) & 1) * CT * TILE);
#pragma unroll 1
        for (int u = 0; u < CT; u++) {
            if (tile + u * TS < t1) {
                f32x16 acc[kKmT];
#pragma unroll
                for (int t = 0; t < kKmT; t++)
#pragma unroll
                    for (int v = 0; v < 16; v++) acc[t][v] = 0.f;
#pragma unroll
                for (int c = 0; c < NCH; c++) {
                    const f16x8 bh = b[u * TILE + (c * 2 + 0) * kWave + l], bl = b[u * TILE + (c * 2 + 1) * kWave + l];
#pragma unroll
                    for (int t = 0; t < kKmT; t++)
                        acc[t] = __builtin_amdgcn_mfma_f32_32x32x16_f16(a[t][c][0], bl, acc[t], 0, 0, 0);
#pragma unroll
                    for (int t = 0; t < kKmT; t++)
                        acc[t] = __builtin_amdgcn_mfma_f32_32x32x16_f16(a[t][c][1], bh, acc[t], 0, 0, 0);
                }
#pragma unroll
                for (int c = 0; c < NCH; c++) {
                    const f16x8 bh = b[u * TILE + (c * 2 + 0) * kWave + l];
#pragma unroll
                    for (int t = 0; t < kKmT; t++)
                        acc[t] = __builtin_amdgcn_mfma_f32_32x32x16_f16(a[t][c][0], bh, acc[t], 0, 0, 0);
                }
                static_assert(kKmT == 2, "one visit per query tile");
                visit(std::integral_constant<int, 0>{}, (tile + u * TS) * 32, acc[0]);
                visit(std::integral_constant<int, 1>{}, (tile + u * TS) * 32, acc[1]);
            }
        }
    }
}

// Largest of a result's 16 values.
__device__ __forceinline__ float knn_max16(const f32x16 &v) {
    float m = v[0];
#pragma unroll
    for (int i = 1; i < 16; i++) m = fmaxf(m, v[i]);
    return m;
}

// Order-preserving bits of a float (ascending), and back.
__device__ __forceinline__ unsigned knn_bits(float f) {
    const unsigned u = __float_as_uint(f);
    return u & 0x80000000u ? ~u : u | 0x80000000u;
}
__device__ __forceinline__ float knn_unbits(unsigned u) {
    return __uint_as_float(u & 0x80000000u ? u & 0x7fffffffu : ~u);
}

// Threshold pass: cut[q], an accumulator value that about 1.3 kKmRank sample points other than q exceed.
// The sample falls into 64 classes (position mod 64: the lanes' 32 columns, first the tiles of even
// number, then the odd ones), and every lane keeps the largest accumulator of its class for each of its queries: one
// instruction per value, no list.  The kKmRank-th largest of a query's 64 class maxima is its cut, found
// bit by bit with ballots (the upper 20 bits are enough: any cut is valid).  The nearest K points hold
// fewer than K of all points above the cut only if their sample hits kKmRank classes.  (Kept instead as a
// list of the 32 nearest with a running cut, the pass took 64.9 ms at N = 300,000, D = 100 and stride 8; this
// takes 8.4 ms.)
template <int NCH>
__global__ __launch_bounds__(kKmThreads, NCH <= 7 ? 2 : 1) void k_knn_tau(const f16x8 *__restrict__ XC,
                                                           const f16x4 *__restrict__ QA, int N,
                                                           const f16x8 *__restrict__ XS, int NS, int stride,
                                                           float *__restrict__ cut) {
    extern __shared__ f16x8 knn_stage[];
    const int w = threadIdx.x / kWave, l = threadIdx.x % kWave;
    const int q0 = blockIdx.x * kKmWg, qw = q0 + w * kKmQ;
    // best[class half][query tile], as vectors so that they stay in registers
    f32x16 b00, b01, b10, b11;
#pragma unroll
    for (int v = 0; v < 16; v++) b00[v] = b01[v] = b10[v] = b11[v] = -INFINITY;
    auto keep = [&](f32x16 &best, int t, int j0, const f32x16 &acc) {
        const long f0 = (long)j0 * stride;  // the tile's first point
        if (f0 < qw + kKmQ && f0 + 31l * stride >= qw) {  // it may hold one of the queries itself
            const int own = (int)(f0 + (long)(l % 32) * stride - qw) - t * 32 - 4 * (l / 32);
#pragma unroll
            for (int v = 0; v < 16; v++)
                if (own != 8 * (v / 4) + v % 4) best[v] = fmaxf(best[v], acc[v]);
        } else {
#pragma unroll
            for (int v = 0; v < 16; v++) best[v] = fmaxf(best[v], acc[v]);
        }
    };
    const int tiles = (NS + 31) / 32;
    knn_sweep<NCH, 2>(
        XC, QA, q0, XS, 0, tiles, knn_stage,
        [&](auto T, int j0, const f32x16 &acc) { keep(T.value == 0 ? b00 : b01, T.value, j0, acc); }, [](int) {});
    __syncthreads();  // the stage is free
    knn_sweep<NCH, 2>(
        XC, QA, q0, XS, 1, tiles, knn_stage,
        [&](auto T, int j0, const f32x16 &acc) { keep(T.value == 0 ? b10 : b11, T.value, j0, acc); }, [](int) {});
    auto finish = [&](int t, const f32x16 &v0, const f32x16 &v1) {
#pragma unroll
        for (int v = 0; v < 16; v++) {
            // both halves of the wavefront at once, each its own query's 64 values
            const unsigned k0 = knn_bits(v0[v]), k1 = knn_bits(v1[v]);
            unsigned pre = 0;
#pragma unroll 1
            for (int b = 31; b >= 12; b--) {
                const unsigned test = pre | 1u << b;
                const unsigned long long m0 = __ballot(k0 >= test), m1 = __ballot(k1 >= test);
                const int c = l < 32 ? __popc((unsigned)m0) + __popc((unsigned)m1)
                                     : __popc((unsigned)(m0 >> 32)) + __popc((unsigned)(m1 >> 32));
                if (c >= kKmRank) pre = test;
            }
            const int q = qw + t * 32 + 8 * (v / 4) + 4 * (l / 32) + v % 4;
            if (l % 32 == 0 && q < N) cut[q] = knn_unbits(pre);
        }
    };
    finish(0, b00, b10);
    finish(1, b01, b11);
}

// Candidate pass of the queries first .. first + kKmWg qblocks: every point j != q whose accumulator (the constant of QA
// holds the threshold) is above 0 into cand[q - first][0 .. cap) as (~accumulator bits, j): ascending keys are ascending distances; count[q]
// (zeroed by the caller) = how many there were.  Workgroup (query block, part of the points).  Hits are
// queued in LDS and written out when the queue is half full: ranks within the queue by LDS atomics, then
// one global atomic per query; what the queue cannot take goes out by itself, unless the query's list has overflowed
// already (full: a bit each), as where many points lie at one distance just inside the threshold: N hits for every
// query (5,000 points in 30 places: 4.7 ms a call with a global atomic for each, 1.9 so).
template <int NCH>
__global__ __launch_bounds__(kKmThreads, 2) void k_knn_collect(const f16x8 *__restrict__ XC,
                                                            const f16x4 *__restrict__ QA, int N, int first,
                                                            int qblocks, int per, int cap,
                                                            unsigned long long *__restrict__ cand,
                                                            int *__restrict__ count) {
    extern __shared__ f16x8 knn_stage[];
    __shared__ unsigned long long qkey[kKmQueue];
    __shared__ unsigned char qq_[kKmQueue];
    __shared__ int hist[kKmWg];
    __shared__ unsigned full[kKmWg / 32];
    __shared__ int qn, qflag[2];
    static_assert(kKmWg <= 256, "a queued hit's query is one byte");
    const int w = threadIdx.x / kWave, l = threadIdx.x % kWave, tid = threadIdx.x;
    const int q0 = first + (blockIdx.x % qblocks) * kKmWg, part = blockIdx.x / qblocks;
    unsigned long long *mine_at = cand + (long)(q0 - first) * cap;  // the workgroup's lists
    const int tiles = (N + 31) / 32;
    const int t0 = part * per, t1 = min(tiles, t0 + per);
    if (!__syncthreads_or((float)QA[q0 + tid][0] > 0.5f * (float)kKmNever)) return;  // none of the queries can pass
    if (tid == 0) {
        qn = 0;
        qflag[0] = qflag[1] = 0;
    }
    if (tid < kKmWg / 32) full[tid] = 0;
    auto flush = [&]() {  // whole workgroup
        __syncthreads();
        const int n = min(qn, kKmQueue);
        hist[tid] = 0;
        __syncthreads();
        int rank[kKmQueue / kKmThreads];
#pragma unroll
        for (int i = 0; i < kKmQueue / kKmThreads; i++) {
            const int e = i * kKmThreads + tid;
            rank[i] = e < n ? atomicAdd(&hist[qq_[e]], 1) : 0;
        }
        __syncthreads();
        const int mine = hist[tid];
        int base = 0;
        if (mine && q0 + tid < N) base = atomicAdd(&count[q0 + tid], mine);
        if (base + mine > cap) atomicOr(&full[tid / 32], 1u << tid % 32);
        __syncthreads();
        hist[tid] = base;
        __syncthreads();
#pragma unroll
        for (int i = 0; i < kKmQueue / kKmThreads; i++) {
            const int e = i * kKmThreads + tid;
            if (e < n) {
                const int pos = hist[qq_[e]] + rank[i];
                if (pos < cap && q0 + qq_[e] < N) mine_at[qq_[e] * cap + pos] = qkey[e];
            }
        }
        __syncthreads();
        if (tid == 0) qn = 0;
        __syncthreads();
    };
    knn_sweep<NCH, 1>(
        XC, QA, q0, XC, t0, t1, knn_stage,
        [&](auto T, int j0, const f32x16 &acc) {
            constexpr int t = T.value;
            if (!__any(knn_max16(acc) > 0.f)) return;
            int j = j0 + l % 32;
            int qb = w * kKmQ + t * 32 + 4 * (l / 32);
            asm volatile("" : "+v"(j), "+v"(qb));  // nothing of this path is computed ahead of the loop
            const int self = j - q0 - qb;  // the row that is point j itself (padding points never pass)
            int total = 0;
#pragma unroll
            for (int v = 0; v < 16; v++)
                total += __popcll(__ballot(acc[v] > 0.f && self != 8 * (v / 4) + v % 4));
            if (!total) return;
            int at = 0;
            if (l == 0) at = atomicAdd(&qn, total);
            at = __shfl(at, 0, kWave);
#pragma unroll
            for (int v = 0; v < 16; v++) {
                const int qq = qb + 8 * (v / 4) + v % 4;
                const bool hit = acc[v] > 0.f && self != 8 * (v / 4) + v % 4;
                const unsigned long long m = __ballot(hit);
                if (!m) continue;
                if (hit) {
                    const unsigned long long key =
                        (unsigned long long)~__float_as_uint(acc[v]) << 32 | (unsigned)j;
                    const int pos = at + __popcll(m & ((1ull << l) - 1ull));
                    if (pos < kKmQueue) {
                        qkey[pos] = key;
                        qq_[pos] = (unsigned char)qq;
                    } else if (q0 + qq < N && !(*(volatile unsigned *)&full[qq / 32] >> qq % 32 & 1u)) {
                        const int p = atomicAdd(&count[q0 + qq], 1);
                        if (p < cap) mine_at[qq * cap + p] = key;
                        else atomicOr(&full[qq / 32], 1u << qq % 32);
                    }
                }
                at += __popcll(m);
            }
        },
        [&](int s) {
            // the flag of this parity was written before the barrier just passed, the other parity's is
            // written during this stage
            if (qflag[s & 1]) flush();
            if (tid == 0) qflag[(s + 1) & 1] = qn > kKmQueue / 2;
        });
    flush();
}

// Exact pass: one workgroup of one wavefront per query, from `first` on.  Of its candidates, those whose accumulator is
// within two error bounds of the K-th largest (nearest) are evaluated: FP64 squared distances
// (coordinate order, no fused multiply-add, as the FP64 kernel), sorted by (distance, index); the first K
// go to out_idx / out_dist (square root correctly rounded).  A query
// whose list is short or overflowed, or whose K-th distance does not clear the threshold less the error
// bound, is appended to redo[] instead.
constexpr int kKmExact = 512;  // FP64 distances per query
template <int CAPL>
__global__ __launch_bounds__(kWave) void k_knn_rerank(const double *__restrict__ X, int first, int D, int K, int kp,
                                                      const unsigned long long *__restrict__ cand,
                                                      const int *__restrict__ count, const float *__restrict__ cut,
                                                      const double *__restrict__ nrm,
                                                      const KnnScale *__restrict__ sc, int *__restrict__ out_idx,
                                                      double *__restrict__ out_dist, int *__restrict__ redo,
                                                      int *__restrict__ nredo) {
    __shared__ double kk[kKmExact];
    __shared__ int ii[kKmExact];
    constexpr int CAP = CAPL * kWave;
    const int l = threadIdx.x;
    const int q = first + blockIdx.x;
    const int n = count[q];
    auto give_up = [&]() {
        if (l == 0) redo[atomicAdd(nredo, 1)] = q;
    };
    if (n < K || n > CAP) return give_up();
    const double err = knn_err(nrm[q], sc->nmax, fabs((double)cut[q]), kp);
    unsigned hi[CAPL];
    int id[CAPL];
#pragma unroll
    for (int s = 0; s < CAPL; s++) {
        hi[s] = 0xffffffffu;
        id[s] = -1;
        if (s * kWave < n) {
            const int e = s * kWave + l;
            if (e < n) {
                const unsigned long long key = cand[(long)blockIdx.x * CAP + e];
                hi[s] = (unsigned)(key >> 32);
                id[s] = (int)(unsigned)key;
            }
        }
    }
    // K-th smallest hi word: the largest value with fewer than K words below it
    unsigned pre = 0;
    for (int b = 31; b >= 0; b--) {
        const unsigned test = pre | 1u << b;
        int c = 0;
#pragma unroll
        for (int s = 0; s < CAPL; s++)
            if (s * kWave < n) c += __popcll(__ballot(id[s] >= 0 && hi[s] < test));
        if (c < K) pre = test;
    }
    const float low = (float)((double)__uint_as_float(~pre) - 2.0 * err) * 0.9999998f;  // rounded down
    int m = 0;
#pragma unroll
    for (int s = 0; s < CAPL; s++) {
        if (s * kWave < n) {
            const bool take = id[s] >= 0 && __uint_as_float(~hi[s]) >= low;
            const unsigned long long b = __ballot(take);
            const int pos = m + __popcll(b & ((1ull << l) - 1ull));
            if (take && pos < kKmExact) ii[pos] = id[s];
            m += __popcll(b);
        }
    }
    if (m > kKmExact) return give_up();
    __syncthreads();
    int B = 64;
    while (B < m) B <<= 1;
    const double *xq = X + (long)q * D;
    for (int i = l; i < B; i += kWave) {
        if (i < m) {
            const double *xc = X + (long)ii[i] * D;
            double acc = 0.0;
#pragma unroll 4
            for (int d = 0; d < D; d++) {
#pragma clang fp contract(off)
                const double diff = xq[d] - xc[d];
                acc += diff * diff;
            }
            kk[i] = acc;
        } else {
            kk[i] = DBL_MAX;
            ii[i] = INT_MAX;
        }
    }
    __syncthreads();
    knn_sort(kk, ii, B);  // by (distance, index), as the FP64 kernel's buffers
    const double dk = kk[K - 1] * sc->scale * sc->scale * 0.5;
    if (!(dk < -(double)cut[q] - err)) return give_up();
    for (int i = l; i < K; i += kWave) {
        out_idx[(long)q * K + i] = ii[i];
        out_dist[(long)q * K + i] = __dsqrt_rn(kk[i]);
    }
}

}  // namespace fitsne
