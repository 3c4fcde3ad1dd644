// fitsne_bh.hpp -- Barnes-Hut t-SNE gradient (nbody_algo = 1) in FP64: the reference's SPTree, its
// traversal and the edge forces on the GPU (gfx950, wave64).
//
// The reference builds an SPTree over Y every iteration (sptree.cpp:57-84, :189-277): a 2^D-ary tree of
// axis-aligned cells, one point per leaf, each node with an online center of mass updated in insertion
// order; exact duplicates stop at the leaf that holds their first copy.  computeNonEdgeForces
// (sptree.cpp:322-354) walks it depth first for every point and summarises a cell when
// max half-width / |y - com| < theta; computeEdgeForces (sptree.cpp:358-376) adds the attractive term
// over the CSR P, and dC = pos_f - neg_f / sum_Q (tsne.cpp:596-640).
//
// The tree's shape does not depend on the insertion order as long as no two points coincide and every
// point lies in a child of each of its cells; the centers of mass do.  So on the GPU:
//   1. the root's center is the mean of Y summed in index order, as the reference sums it.  That chain of N
//      additions runs beside the rest: the shape is built from a mean summed in parallel, and every key is
//      compared with the exact root's before the tree is used;
//   2. every point descends by the reference's cell arithmetic (centers halved down, the reference's
//      bounds test and child order) to a key of kBhLevels child numbers, and the keys are sorted (points
//      whose keys are equal by a second key of as many levels more): a node is a run of keys with a common
//      prefix, an internal one if it holds several points;
//   3. the nodes are laid out in depth-first pre-order (an empty cell needs no node, the walk passes it
//      by): the first child of an internal node is the next slot, skip[] the slot after its subtree;
//   4. from the deepest level up, each node's points in index order are merged from its children's
//      lists, every point finding its rank by binary search in its siblings' lists;
//   5. every node's center of mass is the reference's running update over that list, all nodes at once:
//      a serial chain of a product and a sum per point, whose longest (the root's) starts first and runs
//      beside everything else.
// Coinciding points, points closer than 2 kBhLevels halvings and points that rounding leaves outside every
// child, and keys that the exact root changes, are recognised, and that iteration's tree is built on the
// host by the reference's insertions (BhTree), as it is for few points.  Contraction is off and sqrt / divisions
// are correctly rounded, so the result is the reference's to the bit either way.
#pragma once

#include <cfloat>
#include <vector>

#include <rocprim/device/device_radix_sort.hpp>
#include <rocprim/device/device_scan.hpp>

#include "fitsne_kernels.hpp"
#include "fitsne_seqsum.hpp"

namespace fitsne {

constexpr int kBhMaxDims = 3;

// ---------------------------------------------------------------- host: the tree

// One cell: center and half-width (the reference's Cell corner / width), online center of mass,
// cum_size, at most one stored point, and the first of its 2^D consecutive children.
template <int D>
struct BhNode {
    double c[D], w[D], m[D];
    unsigned cum, pt;
    int first;
    unsigned char size, leaf;
};

template <int D>
struct BhTree {
    static constexpr int NC = 1 << D;
    const double *Y = nullptr;
    std::vector<BhNode<D>> nodes;

    int add(const double *center, const double *hw) {
        BhNode<D> n;
        for (int d = 0; d < D; d++) {
            n.c[d] = center[d];
            n.w[d] = hw[d];
            n.m[d] = 0.0;
        }
        n.cum = 0;
        n.pt = 0;
        n.first = -1;
        n.size = 0;
        n.leaf = 1;
        nodes.push_back(n);
        return (int)nodes.size() - 1;
    }

    // sptree.cpp:235-262: child ch takes the lower half of dimension d when bit d of ch is 1
    void subdivide(int k) {
        double nc[D], nw[D];
        int f = -1;
        for (int ch = 0; ch < NC; ch++) {
            unsigned div = 1;
            const BhNode<D> &p = nodes[k];
            for (int d = 0; d < D; d++) {
                nw[d] = .5 * p.w[d];
                nc[d] = ((unsigned)ch / div) % 2 == 1 ? p.c[d] - .5 * p.w[d] : p.c[d] + .5 * p.w[d];
                div *= 2;
            }
            const int id = add(nc, nw);  // may move nodes[]
            if (ch == 0) f = id;
        }
        nodes[k].first = f;
        if (nodes[k].size == 1) {
            const unsigned q = nodes[k].pt;
            for (int ch = 0; ch < NC; ch++)
                if (insert(f + ch, q)) break;
        }
        nodes[k].size = 0;
        nodes[k].leaf = 0;
    }

    // sptree.cpp:189-232
    bool insert(int k, unsigned i) {
        const double *p = Y + (size_t)i * D;
        {
            BhNode<D> &n = nodes[k];
            for (int d = 0; d < D; d++)
                if (n.c[d] - n.w[d] > p[d] || n.c[d] + n.w[d] < p[d]) return false;
            n.cum++;
            const double mult1 = (double)(n.cum - 1) / (double)n.cum, mult2 = 1.0 / (double)n.cum;
            for (int d = 0; d < D; d++) n.m[d] *= mult1;
            for (int d = 0; d < D; d++) n.m[d] += mult2 * p[d];
            if (n.leaf && n.size < 1) {
                n.pt = i;
                n.size = 1;
                return true;
            }
            if (n.size == 1) {
                bool same = true;
                for (int d = 0; d < D; d++)
                    if (p[d] != Y[(size_t)n.pt * D + d]) {
                        same = false;
                        break;
                    }
                if (same) return true;
            }
        }
        if (nodes[k].leaf) subdivide(k);
        const int f = nodes[k].first;
        for (int ch = 0; ch < NC; ch++)
            if (insert(f + ch, i)) return true;
        return false;
    }

    // sptree.cpp:57-84 and :275-277
    void build(const double *Yin, int N) {
        Y = Yin;
        nodes.clear();
        nodes.reserve((size_t)3 * N + 16);
        double mean[D], mn[D], mx[D], hw[D];
        for (int d = 0; d < D; d++) {
            mean[d] = 0.0;
            mn[d] = DBL_MAX;
            mx[d] = -DBL_MAX;
        }
        for (size_t n = 0; n < (size_t)N; n++)
            for (int d = 0; d < D; d++) {
                const double v = Y[n * D + d];
                mean[d] += v;
                if (v < mn[d]) mn[d] = v;
                if (v > mx[d]) mx[d] = v;
            }
        for (int d = 0; d < D; d++) mean[d] /= (double)N;
        for (int d = 0; d < D; d++) hw[d] = std::fmax(mx[d] - mean[d], mean[d] - mn[d]) + 1e-5;
        add(mean, hw);
        for (unsigned i = 0; i < (unsigned)N; i++) insert(0, i);
    }
};

// A node as the walk reads it, in depth-first pre-order.
template <int D>
struct BhCell {
    double com[D];
    double maxw;   // largest half-width; -1 for a leaf
    unsigned cum;  // points in the cell
    int skip;      // slot after the subtree, -1 at the end of the walk
};

// Lay out host node k's subtree from slot s in pre-order; returns the slot after it (the subtree's skip).
template <int D>
int bh_lay(const BhTree<D> &t, BhCell<D> *cell, int *leafpt, int k, int s) {
    const BhNode<D> &n = t.nodes[k];
    double mw = 0.0;
    for (int d = 0; d < D; d++) {
        cell[s].com[d] = n.m[d];
        mw = mw > n.w[d] ? mw : n.w[d];
    }
    cell[s].maxw = n.leaf ? -1.0 : mw;
    cell[s].cum = n.cum;
    leafpt[s] = (n.leaf && n.size == 1) ? (int)n.pt : -1;
    int next = s + 1;
    if (!n.leaf)
        for (int ch = 0; ch < BhTree<D>::NC; ch++) next = bh_lay(t, cell, leafpt, n.first + ch, next);
    cell[s].skip = next;
    return next;
}

template <int D>
void bh_flatten(const BhTree<D> &t, BhCell<D> *cell, int *leafpt) {
    const int n = bh_lay(t, cell, leafpt, 0, 0);
    for (int s = 0; s < n; s++)
        if (cell[s].skip == n) cell[s].skip = -1;  // the end of the walk
}

// ---------------------------------------------------------------- device: the tree

// Child numbers in a key: D bits each.
template <int D>
constexpr int kBhLevels = D == 1 ? 48 : D == 2 ? 32 : 21;

struct BhRoot {
    double c[kBhMaxDims], w[kBhMaxDims];
};
// What the host reads back before the nodes are written, and the lists of long chains.
struct BhInfo {
    int bad;      // the tree needs the host's insertions
    int deepest;  // depth of the deepest internal node
    int nhuge, nbig;
};
// A node while the tree is built: its points' positions in key order, its parent and depth.
struct BhSpan {
    int start, size, parent, depth;
};
constexpr int kBhSmall = 48;    // longest chain of a single thread
constexpr int kBhHuge = 2048;   // chains from here on start first

// step(load(i)) for i = 0 .. len - 1 in order, len a multiple of 2 G (the callers pad with steps that change
// nothing): groups of G, the next group's loads (LDS; up to G past the end, unused) issued before the
// current group's steps, so that a chain of dependent operations does not wait for them.  A group has at
// most 12 LDS instructions: the wait counter reaches 15, and beyond it the wait for one group takes in the
// next.
template <int G, typename V, typename L, typename S>
__device__ __forceinline__ void bh_ordered(int len, L &&load, S &&step) {
    V va[G], vb[G];
#pragma unroll
    for (int k = 0; k < G; k++) va[k] = load(k);
    for (int i = 0; i < len; i += 2 * G) {
#pragma unroll
        for (int k = 0; k < G; k++) vb[k] = load(i + G + k);
        __builtin_amdgcn_sched_barrier(0);  // the compiler would move the loads next to their steps
#pragma unroll
        for (int k = 0; k < G; k++) step(va[k]);
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int k = 0; k < G; k++) va[k] = load(i + 2 * G + k);
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int k = 0; k < G; k++) step(vb[k]);
        __builtin_amdgcn_sched_barrier(0);
    }
}
constexpr int kBhMeanG = 24, kBhComG = 12;

// Sum, min and max of every coordinate over a block's points, [block][3 D].
constexpr int kBhExtentPer = 8 * kThreads;
template <int D>
__global__ __launch_bounds__(kThreads) void k_bh_extent(const double *__restrict__ Y, int N, double *__restrict__ part) {
    double v[3 * D];
#pragma unroll
    for (int d = 0; d < D; d++) {
        v[3 * d] = 0.0;
        v[3 * d + 1] = DBL_MAX;
        v[3 * d + 2] = -DBL_MAX;
    }
    const int i0 = blockIdx.x * kBhExtentPer, i1 = min(N, i0 + kBhExtentPer);
    for (int i = i0 + threadIdx.x; i < i1; i += kThreads)
#pragma unroll
        for (int d = 0; d < D; d++) {
            const double y = Y[(long)i * D + d];
            v[3 * d] += y;
            v[3 * d + 1] = y < v[3 * d + 1] ? y : v[3 * d + 1];
            v[3 * d + 2] = y > v[3 * d + 2] ? y : v[3 * d + 2];
        }
    __shared__ double sh[3 * D][kThreads / kWave];
#pragma unroll
    for (int d = 0; d < D; d++) {
        const double s = wave_sum(v[3 * d]), mn = wave_min(v[3 * d + 1]), mx = wave_max(v[3 * d + 2]);
        if (threadIdx.x % kWave == 0) {
            sh[3 * d][threadIdx.x / kWave] = s;
            sh[3 * d + 1][threadIdx.x / kWave] = mn;
            sh[3 * d + 2][threadIdx.x / kWave] = mx;
        }
    }
    __syncthreads();
    if (threadIdx.x < 3 * D) {
        double r = sh[threadIdx.x][0];
        for (int i = 1; i < kThreads / kWave; i++) {
            const double x = sh[threadIdx.x][i];
            r = threadIdx.x % 3 == 0 ? r + x : threadIdx.x % 3 == 1 ? (x < r ? x : r) : (x > r ? x : r);
        }
        part[(long)blockIdx.x * 3 * D + threadIdx.x] = r;
    }
}

// The root cell for a given mean: half-widths from the extremes (sptree.cpp:57-84).
__device__ __forceinline__ void bh_set_root(BhRoot *root, int d, double mean, double mn, double mx) {
    root->c[d] = mean;
    root->w[d] = fmax(mx - mean, mean - mn) + 1e-5;
}

// Totals of k_bh_extent's blocks: the root with the mean as the blocks sum it, the extremes into ext[2 D]
// (min, max), and cleared counters.  One wavefront.
template <int D>
__global__ __launch_bounds__(kWave) void k_bh_approx_root(const double *__restrict__ part, int nblk, int N,
                                                          BhRoot *__restrict__ root, double *__restrict__ ext,
                                                          BhInfo *__restrict__ info) {
    const int l = threadIdx.x;
    for (int d = 0; d < D; d++) {
        double s = 0.0, mn = DBL_MAX, mx = -DBL_MAX;
        for (int b = l; b < nblk; b += kWave) {
            const double *p = part + (long)b * 3 * D + 3 * d;
            s += p[0];
            mn = p[1] < mn ? p[1] : mn;
            mx = p[2] > mx ? p[2] : mx;
        }
        s = wave_sum(s);
        mn = wave_min(mn);
        mx = wave_max(mx);
        if (l == 0) {
            bh_set_root(root, d, s / (double)N, mn, mx);
            ext[2 * d] = mn;
            ext[2 * d + 1] = mx;
        }
    }
    if (l == 0) *info = BhInfo{0, -1, 0, 0};
}

// The mean of Y in index order, as the reference sums it, into mean[D].  One workgroup: its first
// wavefront adds chunk after chunk from LDS, a lane per coordinate, while the others stage the next one.
// Bound: the chain of N dependent FP64 additions (2.5 ns each by themselves; 100,000 in 0.44 ms).
constexpr int kBhMeanChunk = 40 * 2 * kBhMeanG;
template <int D>
__global__ __launch_bounds__(256) void k_bh_mean(const double *__restrict__ Y, int N, double *__restrict__ mean) {
    __shared__ double buf[2][(kBhMeanChunk + kBhMeanG) * D];
    const int t = threadIdx.x, w = t / kWave, l = t % kWave;
    const long n = (long)N * D;
    constexpr int C = kBhMeanChunk * D;
    auto stage = [&](long base, double *dst) {
#pragma unroll 8
        for (int i = t - kWave; i < C; i += 256 - kWave) dst[i] = base + i < n ? Y[base + i] : -0.0;  // x + -0.0 is x
    };
    if (w > 0) stage(0, buf[0]);
    __syncthreads();
    double s = 0.0;
    int cur = 0;
    for (long base = 0; base < n; base += C, cur ^= 1) {
        if (w > 0) {
            if (base + C < n) stage(base + C, buf[cur ^ 1]);
        } else if (l < D) {
            constexpr int M = 2 * kBhMeanG;
            const int len = ((int)((n - base < C ? n - base : C) / D) + M - 1) / M * M;
            const double *b = buf[cur] + l;
            bh_ordered<kBhMeanG, double>(len, [&](int i) { return b[i * D]; }, [&](double v) { s += v; });
        }
        __syncthreads();
    }
    if (w == 0 && l < D) mean[l] = s / (double)N;
}

// A point's key: kBhLevels child numbers from the root down, by the reference's descent (sptree.cpp:235-262:
// child bit d is 1 for the lower half; the children are tried upper halves first), with LONG the next
// kBhLevels into key2.  gone: the depth of the cell none of whose children holds the point (255: none).
// False if it lies outside the root.
template <int D, bool LONG>
__device__ __forceinline__ bool bh_descend(const double *__restrict__ Y, int i, const double (&rc)[D],
                                           const double (&rw)[D], uint64_t &key, uint64_t &key2, int &gone) {
#pragma clang fp contract(off)
    double p[D], c[D], w[D];
    bool in = true;
#pragma unroll
    for (int d = 0; d < D; d++) {
        p[d] = Y[(long)i * D + d];
        c[d] = rc[d];
        w[d] = rw[d];
        in = in && c[d] - w[d] <= p[d] && c[d] + w[d] >= p[d];
    }
    key = key2 = 0;
    gone = 255;
    for (int level = 0; level < kBhLevels<D> * (LONG ? 2 : 1); level++) {
        int ch = 0;
#pragma unroll
        for (int d = 0; d < D; d++) {
            const double nw = .5 * w[d];
            const double up = c[d] + .5 * w[d], lo = c[d] - .5 * w[d];
            const bool in_up = !(up - nw > p[d] || up + nw < p[d]);
            const bool in_lo = !(lo - nw > p[d] || lo + nw < p[d]);
            if (!in_up) ch |= 1 << d;
            if (!in_up && !in_lo && gone == 255) gone = level;
            c[d] = in_up ? up : lo;
            w[d] = nw;
        }
        if (LONG && level >= kBhLevels<D>) key2 = key2 << D | (uint64_t)ch;
        else key = key << D | (uint64_t)ch;
    }
    return in;
}

template <int D>
__global__ __launch_bounds__(kThreads) void k_bh_keys(const double *__restrict__ Y, int N,
                                                      const BhRoot *__restrict__ root, uint64_t *__restrict__ key,
                                                      uint32_t *__restrict__ idx, unsigned char *__restrict__ lost,
                                                      BhInfo *__restrict__ info) {
    const int i = blockIdx.x * kThreads + threadIdx.x;
    if (i >= N) return;
    double c[D], w[D];
#pragma unroll
    for (int d = 0; d < D; d++) {
        c[d] = root->c[d];
        w[d] = root->w[d];
    }
    uint64_t k, k2;
    int gone;
    if (!bh_descend<D, false>(Y, i, c, w, k, k2, gone)) info->bad = 1;
    key[i] = k;
    idx[i] = (uint32_t)i;
    lost[i] = (unsigned char)gone;
}

// Levels two keys share.
template <int D>
__device__ __forceinline__ int bh_common(uint64_t a, uint64_t b) {
    const uint64_t x = a ^ b;
    return x ? (__clzll((long long)x) - (64 - D * kBhLevels<D>)) / D : kBhLevels<D>;
}

// Runs of equal keys (pairs of close points, as a rule): the run's first thread sorts its points by their
// second keys, key2[j] for the positions of the run.  A run of more than kBhRun, or second keys that are
// equal too (coinciding points), go to the host.
constexpr int kBhRun = 64;
template <int D>
__global__ __launch_bounds__(kThreads) void k_bh_ties(const double *__restrict__ Y, int N,
                                                      const BhRoot *__restrict__ root, const uint64_t *__restrict__ key,
                                                      uint32_t *__restrict__ idx, uint64_t *__restrict__ key2,
                                                      unsigned char *__restrict__ lost, BhInfo *__restrict__ info) {
    const int j = blockIdx.x * kThreads + threadIdx.x;
    if (j + 1 >= N) return;
    const uint64_t k = key[j];
    if (key[j + 1] != k || (j > 0 && key[j - 1] == k)) return;
    double c[D], w[D];
#pragma unroll
    for (int d = 0; d < D; d++) {
        c[d] = root->c[d];
        w[d] = root->w[d];
    }
    for (int e = j; e < N && key[e] == k; e++) {
        if (e - j >= kBhRun) {
            info->bad = 1;
            return;
        }
        const uint32_t i = idx[e];
        uint64_t k1, k2;
        int gone;
        (void)bh_descend<D, true>(Y, (int)i, c, w, k1, k2, gone);
        lost[i] = (unsigned char)gone;
        int at = e;
        for (; at > j && key2[at - 1] > k2; at--) {
            key2[at] = key2[at - 1];
            idx[at] = idx[at - 1];
        }
        if (at > j && key2[at - 1] == k2) info->bad = 1;
        key2[at] = k2;
        idx[at] = i;
    }
}

// lcp[j] = levels that sorted keys j - 1 and j share (-1 at both ends), cnt[j] = nodes that first occur at
// point j in pre-order: those below the level it shares with its left neighbour, down to its leaf, one
// level below what it shares with either.
template <int D>
__global__ __launch_bounds__(kThreads) void k_bh_count(const uint64_t *__restrict__ key,
                                                       const uint64_t *__restrict__ key2,
                                                       const uint32_t *__restrict__ idx,
                                                       const unsigned char *__restrict__ lost, int N,
                                                       int *__restrict__ lcp, int *__restrict__ cnt,
                                                       BhInfo *__restrict__ info) {
    const int j = blockIdx.x * kThreads + threadIdx.x;
    int deep = -1;
    if (j < N) {
        const uint64_t k = key[j];
        auto common = [&](int a, uint64_t ka, int b, uint64_t kb) {
            return ka != kb ? bh_common<D>(ka, kb) : kBhLevels<D> + bh_common<D>(key2[a], key2[b]);
        };
        const int left = j > 0 ? common(j - 1, key[j - 1], j, k) : -1;
        const int right = j + 1 < N ? common(j, k, j + 1, key[j + 1]) : -1;
        const int leaf = max(left, right) + 1;
        deep = leaf - 1;
        lcp[j] = left;
        cnt[j] = leaf - left;
        if (leaf > 2 * kBhLevels<D> || lost[idx[j]] < leaf) info->bad = 1;
    } else if (j == N) {
        lcp[j] = -1;
        cnt[j] = 0;
    }
    for (int o = kWave / 2; o > 0; o >>= 1) deep = max(deep, __shfl_xor(deep, o, kWave));
    if (threadIdx.x % kWave == 0 && deep > info->deepest) atomicMax(&info->deepest, deep);
}

// The exact root (mean[D], extremes ext[2 D]) into `root`, and whether it changes the path of any point
// (position j in key order) down to its leaf.  differs: cleared by k_bh_clear before.
__global__ void k_bh_clear(int *differs) { *differs = 0; }
template <int D>
__global__ __launch_bounds__(kThreads) void k_bh_check(const double *__restrict__ Y, int N,
                                                       const double *__restrict__ mean, const double *__restrict__ ext,
                                                       const uint64_t *__restrict__ key,
                                                       const uint64_t *__restrict__ key2,
                                                       const uint32_t *__restrict__ idx, const int *__restrict__ lcp,
                                                       BhRoot *__restrict__ root, int *__restrict__ differs) {
    const int j = blockIdx.x * kThreads + threadIdx.x;
    double c[D], w[D];
#pragma unroll
    for (int d = 0; d < D; d++) {
        BhRoot r;
        bh_set_root(&r, d, mean[d], ext[2 * d], ext[2 * d + 1]);
        c[d] = r.c[d];
        w[d] = r.w[d];
    }
    if (j == 0)
#pragma unroll
        for (int d = 0; d < D; d++) {
            root->c[d] = c[d];
            root->w[d] = w[d];
        }
    if (j >= N) return;
    const int leaf = max(lcp[j], lcp[j + 1]) + 1, L = kBhLevels<D>;
    uint64_t k, k2;
    int gone;
    bool same;
    if (leaf <= L) {
        same = bh_descend<D, false>(Y, (int)idx[j], c, w, k, k2, gone);
        const int sh = D * (L - leaf);
        same = same && (sh >= 64 || (k ^ key[j]) >> sh == 0);
    } else {
        same = bh_descend<D, true>(Y, (int)idx[j], c, w, k, k2, gone);
        same = same && k == key[j] && (k2 ^ key2[j]) >> (D * (2 * L - leaf)) == 0;
    }
    if (!same || gone < leaf) *differs = 1;
}

// First position in [lo, hi) whose key has at least (above 0) or more than (above 1) the given prefix of
// `depth` levels (at most kBhLevels).
template <int D>
__device__ __forceinline__ int bh_bound(const uint64_t *__restrict__ key, int lo, int hi, uint64_t k, int depth,
                                        int above) {
    const int sh = D * (kBhLevels<D> - depth);
    const uint64_t p = sh < 64 ? k >> sh : 0;
    while (lo < hi) {
        const int mid = lo + (hi - lo) / 2;
        const uint64_t m = sh < 64 ? key[mid] >> sh : 0;
        if (m < p || (above && m == p)) lo = mid + 1;
        else hi = mid;
    }
    return lo;
}

// The nodes that first occur at point j: spans, cells (the leaves' centers of mass; the internal nodes' and
// their widths follow), leaf points, and the lists of the longer chains; at[j] = the leaf's slot.
template <int D>
__global__ __launch_bounds__(kThreads) void k_bh_nodes(const uint64_t *__restrict__ key,
                                                       const uint32_t *__restrict__ idx, const int *__restrict__ lcp,
                                                       const int *__restrict__ off, const double *__restrict__ Y,
                                                       int N, BhSpan *__restrict__ span,
                                                       BhCell<D> *__restrict__ cell, int *__restrict__ leafpt,
                                                       int *__restrict__ at,
                                                       int *__restrict__ huge, int *__restrict__ big,
                                                       BhInfo *__restrict__ info) {
    const int j = blockIdx.x * kThreads + threadIdx.x;
    if (j >= N) return;
    const uint64_t k = key[j];
    const int left = lcp[j], right = lcp[j + 1], leaf = max(left, right) + 1;
    int slot = off[j], parent = -1, end = N;
    if (left >= 0) {  // the deepest node shared with the left neighbour opened earlier
        int j0 = j;
        if (left <= kBhLevels<D>) j0 = bh_bound<D>(key, 0, j, k, left, 0);
        else  // inside a run of equal keys
            while (lcp[j0] >= left) j0--;
        parent = off[j0] + left - lcp[j0] - 1;
    }
    for (int d = left + 1; d <= leaf; d++, slot++) {
        const bool is_leaf = d == leaf;
        // a subtree's points end where its parent's do or earlier
        if (is_leaf) {
            end = j + 1;
        } else if (d <= kBhLevels<D>) {
            end = bh_bound<D>(key, j + 1, end, k, d, 1);
        } else {
            end = j + 1;
            while (lcp[end] >= d) end++;  // lcp[N] = -1
        }
        const int size = end - j;
        span[slot] = BhSpan{j, size, parent, d};
        BhCell<D> c;
        c.cum = (unsigned)size;
        c.skip = end < N ? off[end] : -1;
        c.maxw = -1.0;
#pragma unroll
        for (int e = 0; e < D; e++) c.com[e] = 0.0 + Y[(long)idx[j] * D + e];
        cell[slot] = c;
        leafpt[slot] = is_leaf ? (int)idx[j] : -1;
        if (!is_leaf && d > 0) {
            if (size > kBhHuge) huge[atomicAdd(&info->nhuge, 1)] = slot;
            else if (size > kBhSmall) big[atomicAdd(&info->nbig, 1)] = slot;
        }
        parent = slot;
    }
    at[j] = slot - 1;
}

// Level d of the lists: every node of depth d gets its points in index order from its children's lists
// (in, out: by position; points whose leaf lies at depth d or above stay).  at[p]: the node of position p
// whose list holds it, moved up to its parent here.
template <int D>
__global__ __launch_bounds__(kThreads) void k_bh_merge(const BhSpan *__restrict__ span,
                                                       const BhCell<D> *__restrict__ cell, int N, int d,
                                                       const uint32_t *__restrict__ in, uint32_t *__restrict__ out,
                                                       int *__restrict__ at) {
    const int p = blockIdx.x * kThreads + threadIdx.x;
    if (p >= N) return;
    const int k = at[p];
    const BhSpan me = span[k];
    const uint32_t v = in[p];
    if (me.depth != d + 1) {
        out[p] = v;
        return;
    }
    const BhSpan up = span[me.parent];
    int rank = p - me.start;
    int s = me.parent + 1;
    for (;;) {
        const BhSpan b = s == k ? me : span[s];
        if (s != k) {
            int lo = b.start, hi = b.start + b.size;
            while (lo < hi) {
                const int mid = lo + (hi - lo) / 2;
                if (in[mid] < v) lo = mid + 1;
                else hi = mid;
            }
            rank += lo - b.start;
        }
        if (b.start + b.size >= up.start + up.size) break;
        s = cell[s].skip;
    }
    out[up.start + rank] = v;
    at[p] = me.parent;
}

// ab[n] = ((n - 1) / n, 1 / n), n = 1 .. N: the factors of the n-th update of a center of mass
// (sptree.cpp:189-232).
__global__ __launch_bounds__(kThreads) void k_bh_factors(double2 *__restrict__ ab, int N) {
    const int n = blockIdx.x * kThreads + threadIdx.x + 1;
    if (n <= N) ab[n] = make_double2((double)(n - 1) / (double)n, 1.0 / (double)n);
}

// Centers of mass of the internal nodes with at most kBhSmall points, a thread each.
// order: the lists by depth, `stride` apart, depth d at (d - 1) stride.
template <int D>
__global__ __launch_bounds__(kThreads) void k_bh_com_small(const BhSpan *__restrict__ span, int nodes,
                                                           const uint32_t *__restrict__ order, long stride,
                                                           const double *__restrict__ Y,
                                                           const double2 *__restrict__ ab, BhCell<D> *__restrict__ cell) {
#pragma clang fp contract(off)
    const int k = blockIdx.x * kThreads + threadIdx.x;
    if (k >= nodes) return;
    const BhSpan s = span[k];
    if (s.size > kBhSmall || s.size < 2 || s.depth == 0) return;
    const uint32_t *o = order + (long)(s.depth - 1) * stride + s.start;
    double m[D];
#pragma unroll
    for (int d = 0; d < D; d++) m[d] = 0.0;
    for (int t0 = 0; t0 < s.size; t0 += 4) {
        double y[4][D];
        double2 f[4];
#pragma unroll
        for (int u = 0; u < 4; u++) {
            const int t = min(t0 + u, s.size - 1);
            const long i = o[t];
            f[u] = ab[t + 1];
#pragma unroll
            for (int d = 0; d < D; d++) y[u][d] = Y[i * D + d];
        }
#pragma unroll
        for (int u = 0; u < 4; u++)
            if (t0 + u < s.size)
#pragma unroll
                for (int d = 0; d < D; d++) {
                    m[d] *= f[u].x;
                    m[d] += f[u].y * y[u][d];
                }
    }
#pragma unroll
    for (int d = 0; d < D; d++) cell[k].com[d] = m[d];
}

// One wavefront's chain over n points (list o, or all points in index order): the center of mass into m
// (lanes below D).  Chunks of kBhChunk points go through LDS: factors and scaled coordinates are computed by
// all lanes, the loads of the next chunk are in flight during the chain.  Bound: the chain, a dependent
// product and sum per point (4.7 ns by themselves; 100,000 points in 0.86 ms, 1.41 before the loads ran
// ahead of the steps).
constexpr int kBhPer = 6, kBhChunk = kWave * kBhPer;
static_assert(kBhChunk % (2 * kBhComG) == 0, "whole groups in a chunk");
template <int D>
struct BhChunk {
    double2 v[2][D][kBhChunk + kBhComG];  // factor of the old center, scaled coordinate
};
template <int D, bool LIST>
__device__ __forceinline__ double bh_chain(const uint32_t *__restrict__ o, int n, const double *__restrict__ Y,
                                           const double2 *__restrict__ ab, BhChunk<D> &lds) {
#pragma clang fp contract(off)
    const int l = threadIdx.x;
    double m = 0.0;
    double2 f[kBhPer];
    double y[kBhPer][D];
    long next[kBhPer];
    auto points = [&](int t0) {
#pragma unroll
        for (int u = 0; u < kBhPer; u++) {
            const int t = min(t0 + u * kWave + l, n - 1);
            next[u] = LIST ? (long)o[t] : (long)t;
        }
    };
    auto fetch = [&](int t0) {
#pragma unroll
        for (int u = 0; u < kBhPer; u++) {
            f[u] = ab[min(t0 + u * kWave + l, n - 1) + 1];
#pragma unroll
            for (int d = 0; d < D; d++) y[u][d] = Y[next[u] * D + d];
        }
    };
    points(0);
    fetch(0);
    points(kBhChunk);
    int cur = 0;
    for (int t0 = 0; t0 < n; t0 += kBhChunk, cur ^= 1) {
#pragma unroll
        for (int u = 0; u < kBhPer; u++)
#pragma unroll
            for (int d = 0; d < D; d++)  // past the end: m * 1 + -0.0 is m
                lds.v[cur][d][u * kWave + l] =
                    t0 + u * kWave + l < n ? make_double2(f[u].x, f[u].y * y[u][d]) : make_double2(1.0, -0.0);
        fetch(t0 + kBhChunk);
        points(t0 + 2 * kBhChunk);
        __syncthreads();
        if (l < D) {
            const double2 *v = lds.v[cur][l];
            constexpr int M = 2 * kBhComG;
            bh_ordered<kBhComG, double2>((min(kBhChunk, n - t0) + M - 1) / M * M, [&](int i) { return v[i]; }, [&](const double2 &x) {
#pragma clang fp contract(off)
                m *= x.x;
                m += x.y;
            });
        }
    }
    return m;
}

// Centers of mass of the listed nodes (huge ones first), a wavefront each.
template <int D>
__global__ __launch_bounds__(kWave) void k_bh_com_long(const int *__restrict__ huge, const int *__restrict__ big,
                                                       const BhInfo *__restrict__ info,
                                                       const BhSpan *__restrict__ span,
                                                       const uint32_t *__restrict__ order, long stride,
                                                       const double *__restrict__ Y, const double2 *__restrict__ ab,
                                                       BhCell<D> *__restrict__ cell) {
    __shared__ BhChunk<D> lds;
    const int nh = info->nhuge, n = nh + info->nbig;
    for (int e = blockIdx.x; e < n; e += gridDim.x) {
        const int k = e < nh ? huge[e] : big[e - nh];
        const BhSpan s = span[k];
        const double m = bh_chain<D, true>(order + (long)(s.depth - 1) * stride + s.start, s.size, Y, ab, lds);
        if ((int)threadIdx.x < D) cell[k].com[threadIdx.x] = m;
        __syncthreads();
    }
}

// The root's, over all points in index order, into out[D]; k_bh_finish puts it in its cell.
template <int D>
__global__ __launch_bounds__(kWave) void k_bh_com_root(const double *__restrict__ Y, int N,
                                                       const double2 *__restrict__ ab, double *__restrict__ out) {
    __shared__ BhChunk<D> lds;
    const double m = bh_chain<D, false>(nullptr, N, Y, ab, lds);
    if ((int)threadIdx.x < D) out[threadIdx.x] = m;
}
// The widths of the internal nodes from the exact root (halved at each level: exact), and the root's center of mass.
template <int D>
__global__ __launch_bounds__(kThreads) void k_bh_finish(const BhSpan *__restrict__ span, int nodes,
                                                        const BhRoot *__restrict__ root, const double *__restrict__ com,
                                                        BhCell<D> *__restrict__ cell) {
    const int k = blockIdx.x * kThreads + threadIdx.x;
    if (k >= nodes) return;
    const BhSpan s = span[k];
    if (s.size < 2) return;
    double mw = root->w[0];
#pragma unroll
    for (int d = 1; d < D; d++) mw = mw > root->w[d] ? mw : root->w[d];
    cell[k].maxw = ldexp(mw, -s.depth);
    if (k == 0)
#pragma unroll
        for (int d = 0; d < D; d++) cell[0].com[d] = com[d];
}

// ---------------------------------------------------------------- device: forces

// maxw / sqrt(dd) < theta, as the reference rounds it.  The squares decide unless they are within 1e-12 of
// each other (or out of the normal range), when the quotient is formed.
__device__ __forceinline__ bool bh_far(double maxw, double dd, double theta) {
    const double a = maxw * maxw, b = theta * theta * dd;
    if (b > 1e-280 && b < 1e280 && a < 1e280) {
        if (a < b * (1.0 - 1e-12)) return true;
        if (a > b * (1.0 + 1e-12)) return false;
    }
    return maxw / __dsqrt_rn(dd) < theta;
}

// computeNonEdgeForces for every point (sptree.cpp:322-354): neg_f[i] (D) and Q[i].  The skip links
// replace the recursion; the order of the summarised cells is the reference's.  With neg_f null only Q.
// order (nullable): the points in key order, so that a wavefront's lanes walk the same part of the tree
// (N = 100,000 in 2D: 0.51 ms in index order with six arrays per node, 0.12 in key order with one record).
template <int D>
__global__ __launch_bounds__(kWave) void k_bh_nonedge(const double *__restrict__ Y, int N,
                                                      const BhCell<D> *__restrict__ cell,
                                                      const int *__restrict__ leafpt,
                                                      const uint32_t *__restrict__ order, double theta,
                                                      double *__restrict__ neg_f, double *__restrict__ Q) {
#pragma clang fp contract(off)
    const int t = blockIdx.x * kWave + threadIdx.x;
    if (t >= N) return;
    const int i = order ? (int)order[t] : t;
    double y[D], nf[D];
#pragma unroll
    for (int d = 0; d < D; d++) {
        y[d] = Y[(long)i * D + d];
        nf[d] = 0.0;
    }
    double q = 0.0;
    int k = 0;
    while (k >= 0) {
        const BhCell<D> c = cell[k];
        const bool leaf = c.maxw < 0.0;
        if (c.cum == 0u || (leaf && leafpt[k] == i)) {
            k = c.skip;
            continue;
        }
        double diff[D], dd = 0.0;
#pragma unroll
        for (int d = 0; d < D; d++) {
            diff[d] = y[d] - c.com[d];
            dd += diff[d] * diff[d];
        }
        if (leaf || bh_far(c.maxw, dd, theta)) {
            dd = 1.0 / (1.0 + dd);
            double mult = (double)c.cum * dd;
            q += mult;
            mult *= dd;
#pragma unroll
            for (int d = 0; d < D; d++) nf[d] += mult * diff[d];
            k = c.skip;
        } else {
            k = k + 1;  // first child
        }
    }
    Q[i] = q;
    if (neg_f) {
#pragma unroll
        for (int d = 0; d < D; d++) neg_f[(long)i * D + d] = nf[d];
    }
}

// computeEdgeForces (sptree.cpp:358-376): one thread per row, its entries in CSR order.
template <int D>
__global__ __launch_bounds__(kThreads) void k_bh_edge(const int64_t *__restrict__ rowP,
                                                      const uint32_t *__restrict__ colP,
                                                      const double *__restrict__ val, const double *__restrict__ Y,
                                                      int N, double *__restrict__ pos_f) {
#pragma clang fp contract(off)
    const int n = blockIdx.x * kThreads + threadIdx.x;
    if (n >= N) return;
    double y[D], pf[D];
#pragma unroll
    for (int d = 0; d < D; d++) {
        y[d] = Y[(long)n * D + d];
        pf[d] = 0.0;
    }
    for (long e = rowP[n]; e < rowP[n + 1]; e++) {
        const long j = colP[e];
        double dd = 1.0;
#pragma unroll
        for (int d = 0; d < D; d++) dd += (y[d] - Y[j * D + d]) * (y[d] - Y[j * D + d]);
        dd = val[e] / dd;
#pragma unroll
        for (int d = 0; d < D; d++) pf[d] += dd * (y[d] - Y[j * D + d]);
    }
#pragma unroll
    for (int d = 0; d < D; d++) pos_f[(long)n * D + d] = pf[d];
}

// dC = pos_f - neg_f / sum_Q (tsne.cpp:626-627).
__global__ __launch_bounds__(kThreads) void k_bh_combine(const double *__restrict__ pos_f,
                                                         const double *__restrict__ neg_f,
                                                         const double *__restrict__ zbuf, long n,
                                                         double *__restrict__ dC) {
    const double Z = zbuf[0];
    for (long e = (long)blockIdx.x * kThreads + threadIdx.x; e < n; e += (long)gridDim.x * kThreads)
        dC[e] = pos_f[e] - (neg_f[e] / Z);
}

}  // namespace fitsne
