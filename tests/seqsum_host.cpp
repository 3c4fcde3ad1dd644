// One workgroup of k_seq_sum on the CPU: its 1024 threads as coroutines, a wavefront's shuffles and ballots
// and the workgroup's barriers as points where they wait for each other.
// Input: n, then n doubles (raw).  Output: the two results as hexadecimal bits.  Exit 3: it does not end (more
// than `limit` barriers, four times what adding every value by itself would take).
#include <ucontext.h>

#include <cmath>
#include <cstdint>
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <vector>

#define __global__
#define __device__
#define __forceinline__ inline
#define __restrict__ __restrict
#define __shared__ static
#define __launch_bounds__(n)

namespace {
constexpr int kLanes = 64, kBlock = 1024;
struct Idx {
    int x;
} threadIdx;

ucontext_t g_main, g_ctx[kBlock];
bool g_done[kBlock];
long g_limit, g_barriers;

void yield() {
    const int me = threadIdx.x;
    swapcontext(&g_ctx[me], &g_main);
    threadIdx.x = me;
}

// Threads that meet: everyone leaves when the last one has come.
struct Meet {
    int came = 0;
    long gen = 0;
    void wait(int count) {
        const long mine = gen;
        if (++came == count) {
            came = 0;
            gen++;
        }
        while (gen == mine) yield();
    }
} g_block, g_wave[kBlock / kLanes];

void __syncthreads() {
    if (threadIdx.x == 0 && ++g_barriers > g_limit) {
        std::printf("no end after %ld barriers\n", g_barriers);
        std::exit(3);
    }
    g_block.wait(kBlock);
}

// v of every lane of the wavefront
template <typename T>
std::vector<T> all_lanes(T v) {
    static T slot[kBlock];
    const int w = threadIdx.x / kLanes;
    slot[threadIdx.x] = v;
    g_wave[w].wait(kLanes);
    std::vector<T> r(slot + w * kLanes, slot + (w + 1) * kLanes);
    g_wave[w].wait(kLanes);
    return r;
}
template <typename T>
T __shfl(T v, int lane, int) {
    return all_lanes(v)[lane & (kLanes - 1)];
}
template <typename T>
T __shfl_up(T v, int by, int) {
    const auto a = all_lanes(v);
    const int l = threadIdx.x % kLanes;
    return l >= by ? a[l - by] : v;
}
unsigned long long __ballot(bool p) {
    const auto a = all_lanes((int)p);
    unsigned long long m = 0;
    for (int l = 0; l < kLanes; l++)
        if (a[l]) m |= 1ull << l;
    return m;
}
int __ffsll(long long v) { return __builtin_ffsll(v); }
}  // namespace

namespace fitsne {
constexpr int kWave = kLanes;
}
#include "../fit-sne_amd/csrc/fitsne_seqsum.hpp"

static std::vector<double> g_v;
static double g_out[2];

static void thread_main() {
    fitsne::k_seq_sum(g_v.data(), (int)g_v.size(), g_out);
    g_done[threadIdx.x] = true;
    for (;;) yield();
}

int main() {
    int64_t n = 0;
    if (std::fread(&n, sizeof n, 1, stdin) != 1 || n < 0 || n > (1 << 24)) return 2;
    g_v.resize((size_t)n);
    if (n && std::fread(g_v.data(), sizeof(double), (size_t)n, stdin) != (size_t)n) return 2;
    g_limit = 2 * (100 + 2 * (n / 1024 + 1));
    std::vector<char> stacks((size_t)kBlock * 65536);
    for (int t = 0; t < kBlock; t++) {
        getcontext(&g_ctx[t]);
        g_ctx[t].uc_stack.ss_sp = stacks.data() + (size_t)t * 65536;
        g_ctx[t].uc_stack.ss_size = 65536;
        makecontext(&g_ctx[t], thread_main, 0);
    }
    for (bool left = true; left;) {
        left = false;
        for (int t = 0; t < kBlock; t++) {
            if (g_done[t]) continue;
            threadIdx.x = t;
            swapcontext(&g_main, &g_ctx[t]);
            left |= !g_done[t];
        }
    }
    for (double r : g_out) {
        uint64_t b;
        std::memcpy(&b, &r, sizeof b);
        std::printf("%016llx\n", (unsigned long long)b);
    }
    return 0;
}
