// fitsne_seqsum.hpp -- a sum in index order, rounded after every addition, by one workgroup (gfx950, wave64).
#pragma once

namespace fitsne {

// sum_Q = sum of Q[i] in index order (tsne.cpp:612-614), rounded after every addition as a loop would:
// out[0] = sum_Q.  While the running sum s stays in one binade it is an integer S of its ulp u, and adding
// v >= 0 moves it by the integer nearest to v / u: by a fixed amount, or in a tie by one that depends on
// the parity of S.  Such steps compose: a run of them is two numbers, its move from an even and from an odd
// S.  So the workgroup folds runs in parallel (each thread 16 values, the threads in order).  Where the sum
// leaves its binade, about log2(n) times (or a value is negative or not finite), the 16 values of the thread
// concerned are added one by one, and the rest is folded again in the new binade.  A sum without such an ulp
// (zero, below 1e-250, above 1e250, not finite) has the rest of a wavefront's values added one by one.  (One
// thread adding everything from LDS took 0.79 ms at n = 100,000; this takes 0.12 ms.)
struct SeqMove {
    long long d0, d1;  // move from an even / odd S; kSeqStop or more: not composable
};
constexpr long long kSeqStop = 1ll << 60;
__device__ __forceinline__ SeqMove seq_then(SeqMove a, SeqMove b) {  // a, then b
    SeqMove r;
    r.d0 = a.d0 + ((a.d0 & 1) ? b.d1 : b.d0);
    r.d1 = a.d1 + ((a.d1 & 1) ? b.d0 : b.d1);
    if (a.d0 >= kSeqStop || a.d1 >= kSeqStop || b.d0 >= kSeqStop || b.d1 >= kSeqStop) r.d0 = r.d1 = kSeqStop;
    return r;
}
__device__ __forceinline__ SeqMove seq_step(double v, double inv_u) {
    const double x = v * inv_u;  // a power of two: exact
    if (!(v >= 0.0 && x < 4503599627370496.0)) return {kSeqStop, kSeqStop};
    const double f = floor(x), r = x - f;
    const long long k = (long long)f;
    if (r < 0.5) return {k, k};
    if (r > 0.5) return {k + 1, k + 1};
    return {k + (k & 1), k + 1 - (k & 1)};  // ties to even
}
// The moves of lanes 0 .. l, in lane order, as one.
__device__ __forceinline__ SeqMove seq_scan(SeqMove a) {
    const int l = threadIdx.x % kWave;
    for (int o = 1; o < kWave; o <<= 1) {
        const SeqMove b{__shfl_up(a.d0, o, kWave), __shfl_up(a.d1, o, kWave)};
        if (l >= o) a = seq_then(b, a);
    }
    return a;
}
// s (a multiple of 1 / inv_u) after the moves m, if the sum stays in its binade.  No move fits any sum: it is
// what the threads whose values are in s already have.
__device__ __forceinline__ bool seq_apply(double &s, double inv_u, SeqMove m) {
    if (m.d0 == 0 && m.d1 == 0) return true;
    const long long S = (long long)(s * inv_u), d = (S & 1) ? m.d1 : m.d0;
    if (inv_u == 0.0 || d >= kSeqStop || S + d >= (1ll << 53)) return false;
    s = (double)(S + d) / inv_u;
    return true;
}
constexpr int kSeqPer = 16, kSeqChunk = 1024 * kSeqPer;
__global__ __launch_bounds__(1024) void k_seq_sum(const double *__restrict__ v, int n, double *__restrict__ out) {
    constexpr int NW = 1024 / kWave;
    __shared__ SeqMove part[NW];
    __shared__ double ssum;
    __shared__ int sfrom;
    const int t = threadIdx.x, w = t / kWave, l = t % kWave;
    if (t == 0) ssum = 0.0;
    for (int base = 0; base < n; base += kSeqChunk) {
        double x[kSeqPer];
#pragma unroll
        for (int k = 0; k < kSeqPer; k++) {
            const int e = base + t * kSeqPer + k;
            x[k] = e < n ? v[e] : 0.0;
        }
        int from = 0;  // threads below it are done
        do {
            __syncthreads();
            double s = ssum;
            // 1 / ulp(s) for a positive s in a range where it is normal too, else 0
            const double iu = s > 1e-250 && s < 1e250 ? ldexp(1.0, 52 - ilogb(s)) : 0.0;
            SeqMove m{0, 0};
            if (t >= from && iu > 0.0) {
                // without ties every value moves S by rint(v / u)
                double sum = 0.0;
                bool plain = true;
#pragma unroll
                for (int k = 0; k < kSeqPer; k++) {
                    const double q = x[k] * iu, r = rint(q);
                    sum += r;
                    plain &= x[k] >= 0.0 && q < 35184372088832.0 && fabs(q - r) != 0.5;  // 2^45: sums stay exact
                }
                m.d0 = m.d1 = plain ? (long long)sum : 0;
                if (!plain)
#pragma unroll
                    for (int k = 0; k < kSeqPer; k++) m = seq_then(m, seq_step(x[k], iu));
            } else if (t >= from) {
                m.d0 = m.d1 = kSeqStop;
            }
            m = seq_scan(m);
            if (l == kWave - 1) part[w] = m;
            __syncthreads();
            // every wavefront: the sums behind each of the 16, and the first that does not fit
            const SeqMove p = seq_scan(l < NW ? part[l] : SeqMove{0, 0});
            double r = s;
            const int stop = __ffsll((long long)__ballot(!seq_apply(r, iu, p))) - 1;
            if (stop < 0) {
                if (t == NW - 1) {  // all fit: the chunk's total
                    ssum = r;
                    sfrom = 1024;
                }
            } else if (stop == w) {  // here: from the first thread whose values do not fit, one by one
                if (w > 0) s = __shfl(r, w - 1, kWave);
                r = s;
                const bool fits = seq_apply(r, iu, m);
                const int j = __ffsll((long long)__ballot(!fits)) - 1;
                if (j > 0) s = __shfl(r, j - 1, kWave);
                const int end = iu > 0.0 ? j + 1 : kWave;
                for (int i = j; i < end; i++) {
                    double a = s;
#pragma unroll
                    for (int k = 0; k < kSeqPer; k++) a += x[k];
                    s = __shfl(a, i, kWave);
                }
                if (l == 0) {
                    ssum = s;
                    sfrom = w * kWave + end;
                }
            }
            __syncthreads();
            from = sfrom;
        } while (from < 1024 && base + from * kSeqPer < n);
    }
    __syncthreads();
    if (t == 0) {
        out[0] = ssum;
        out[1] = 1.0 / ssum;
    }
}

}  // namespace fitsne
