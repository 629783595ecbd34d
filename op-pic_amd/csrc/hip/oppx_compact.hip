// Particle compaction on gfx950: hole-fill after a move.
//
// Reference semantics (opp_lib/src/core/opp_particle_organize_core.cpp:124-218; identical live range
// in omp opp_lib/src/omp/opp_particle_mover.cpp:153-218 and hip opp_lib/src/hip/opp_particle_sorter.cpp:271-359):
// with N particles, R removed and S = N - R, the k-th hole below S (ascending) receives the k-th
// live record at or above S (descending). No sort of hole indices is needed here: the move pass
// leaves a removal bitmap (one 64-bit ballot word per wave), and
//   #holes below index v        = wp[v/64] + popcount(word & low bits)      (wp = word prefix)
//   rank of live v >= S from top = (N-1-v) - (R - #holes below v)
// so every live tail record finds its destination hole by a binary search over wp and a
// select inside one word. Two launches (one for a small set): the word prefixes inside each block of words and the block counts;
// then the tail copy, whose blocks scan the block counts themselves and one of which writes the counters.

#include <mutex>

#include "oppx_internal.h"

// Scratch of oppx_holefill_noalloc: a file-scope device array, one copy per GPU, held until the process
// ends. In host code this name stands for the array but is no device address: kernels receive the
// address hipGetSymbolAddress returns for the current device (oppx::noalloc_scratch).
static __device__ __align__(256) unsigned char scratch[OPPX_HOLEFILL_NOALLOC_SCRATCH_BYTES];

namespace oppx {
namespace {

constexpr int kB = 256;
constexpr int kMaxDats = 16;
constexpr int kMaxComps = 64;   // components one fill launch moves (more take further launches)
constexpr int kMaxGroups = 4096;  // group prefixes a fill block holds in LDS
constexpr int kSmallThreads = 1024;
constexpr int kSmallWords = 128;  // bitmap words of a set one block fills alone
constexpr int kCopyBatch = 12;  // components loaded before any of them is stored (a FEM-PIC particle has 11)

// The dats as single components: base address of each, and which of them have 8-byte elements.
struct CompTable {
    int n;
    uint64_t wide;
    void* base[kMaxComps];
};

__device__ __forceinline__ int64_t words_of(int64_t n) { return (n + 63) >> 6; }

// live count before compaction, clamped to the host's bound (grids and scratch are sized by it)
__device__ __forceinline__ int64_t live_count(const oppx_move_counters* ctr, int64_t n_max) {
    const int64_t n = ctr->size;
    return n < 0 ? 0 : (n > n_max ? n_max : n);
}

// exclusive block scan of one uint32 per thread (kB threads); returns the prefix, total in *tot
__device__ __forceinline__ uint32_t block_exclusive_scan(uint32_t v, uint32_t* tot) {
    __shared__ uint32_t s_w[kB / kWave];
    const int lane = threadIdx.x & (kWave - 1), w = threadIdx.x / kWave;
    uint32_t inc = v;
#pragma unroll
    for (int d = 1; d < kWave; d <<= 1) {
        const uint32_t t = __shfl_up(inc, d);
        if (lane >= d) inc += t;
    }
    if (lane == kWave - 1) s_w[w] = inc;
    __syncthreads();
    uint32_t off = 0, all = 0;
    for (int q = 0; q < kB / kWave; q++) {
        if (q < w) off += s_w[q];
        all += s_w[q];
    }
    __syncthreads();
    *tot = all;
    return off + inc - v;
}

// Removals of every bitmap word before it in its block of kB words (wp), of every block (bsum), and the
// live count (head[0]): the fill reads the count from here, so that it may write the new one while its
// other blocks still run.
__global__ void __launch_bounds__(kB) hf_count(const uint64_t* __restrict__ bits,
                                               const oppx_move_counters* __restrict__ ctr, uint32_t* __restrict__ bsum,
                                               uint32_t* __restrict__ wp, uint32_t* __restrict__ head, int64_t n_max) {
    const int64_t N = live_count(ctr, n_max), W = words_of(N);
    const int64_t w = (int64_t)blockIdx.x * kB + threadIdx.x;
    const uint32_t c = (w < W) ? (uint32_t)__popcll(bits[w]) : 0u;
    uint32_t tot;
    const uint32_t ex = block_exclusive_scan(c, &tot);
    if (w < W) wp[w] = ex;
    if (threadIdx.x == 0) bsum[blockIdx.x] = tot;
    if (blockIdx.x == 0 && threadIdx.x == 0) head[0] = (uint32_t)N;
}

// Record v to hole h.
template <typename Index>
__device__ __forceinline__ void move_record(const CompTable& T, Index v, Index h) {
    for (int c0 = 0; c0 < T.n; c0 += kCopyBatch) {
        uint64_t x[kCopyBatch];
#pragma unroll
        for (int u = 0; u < kCopyBatch; u++) {
            if (c0 + u >= T.n) continue;
            if ((T.wide >> (c0 + u)) & 1ull) x[u] = reinterpret_cast<const uint64_t*>(T.base[c0 + u])[v];
            else x[u] = reinterpret_cast<const uint32_t*>(T.base[c0 + u])[v];
        }
#pragma unroll
        for (int u = 0; u < kCopyBatch; u++) {
            if (c0 + u >= T.n) continue;
            if ((T.wide >> (c0 + u)) & 1ull) reinterpret_cast<uint64_t*>(T.base[c0 + u])[h] = x[u];
            else reinterpret_cast<uint32_t*>(T.base[c0 + u])[h] = (uint32_t)x[u];
        }
    }
}

// Every block scans the block counts into LDS itself (group e: blocks [e * per, (e + 1) * per)), then its
// threads move the live records of the tail [S, N) to their holes. What bounds this is the chain of
// dependent reads of one record (its hole's search, then the copy): a scan kernel, a word-prefix kernel and a
// finalize kernel beside it cost a launch each, 4.5-5 us after a large kernel. Measured (kernel time, a few
// percent removed), five launches before and these two: 4,000 particles 14.5 and 11.5 us, 1 M 38.9 and 23.7 us,
// 24 M 64 and 48 us; since then a record's components are loaded in one batch, and this kernel alone takes 19 us at 1 M, 45 at
// 24 M.
__global__ void __launch_bounds__(kB) hf_fill(const uint64_t* __restrict__ bits, oppx_move_counters* __restrict__ ctr,
                                              const uint32_t* __restrict__ bsum, const uint32_t* __restrict__ wp,
                                              const uint32_t* __restrict__ head, CompTable T, int64_t nb, int per,
                                              int finish) {
    __shared__ uint32_t s_pre[kMaxGroups];
    const int64_t N = head[0];
    const int ng = (int)((nb + per - 1) / per);
    for (int e = threadIdx.x; e < ng; e += kB) {
        uint32_t c = 0;
        for (int64_t b = (int64_t)e * per; b < (int64_t)(e + 1) * per && b < nb; b++) c += bsum[b];
        s_pre[e] = c;
    }
    __syncthreads();
    const int items = (ng + kB - 1) / kB;  // groups of one thread, consecutive
    const int e0 = (int)threadIdx.x * items, e1 = e0 + items < ng ? e0 + items : ng;
    uint32_t mine = 0, total;
    for (int e = e0; e < e1; e++) mine += s_pre[e];
    uint32_t run = block_exclusive_scan(mine, &total);
    for (int e = e0; e < e1; e++) {
        const uint32_t c = s_pre[e];
        s_pre[e] = run;
        run += c;
    }
    __syncthreads();
    const int64_t R = total, S = N - R, W = words_of(N);
    // removals before word w
    auto before = [&](int64_t w) {
        const int64_t b = w / kB;
        const int e = (int)(b / per);
        int64_t c = (int64_t)s_pre[e] + wp[w];
        for (int64_t q = (int64_t)e * per; q < b; q++) c += bsum[q];
        return c;
    };
    const bool some = R > 0 && R <= N;
    if (finish && blockIdx.x == 0 && threadIdx.x == 0) {
        ctr->removed = (int32_t)R;
        if (some) {
            const int j = (int)(S & 63);
            const uint64_t lowmask = j ? ((1ull << j) - 1ull) : 0ull;
            ctr->holes_low = (int32_t)(before(S >> 6) + __popcll(bits[S >> 6] & lowmask));
            ctr->size = (int32_t)S;
        } else {
            ctr->holes_low = 0;
        }
    }
    if (!some) return;
    for (int64_t v = S + (int64_t)blockIdx.x * kB + threadIdx.x; v < N; v += (int64_t)gridDim.x * kB) {
        const uint64_t word = bits[v >> 6];
        const int j = (int)(v & 63);
        if ((word >> j) & 1ull) continue;  // a hole itself
        const int64_t k = (N - 1 - v) - (R - (before(v >> 6) + __popcll(word & ((1ull << j) - 1ull))));
        // k-th hole: the last group, block and word with at most k removals before it, then the set bit
        int glo = 0, ghi = ng - 1;
        while (glo < ghi) {
            const int mid = (glo + ghi + 1) >> 1;
            if ((int64_t)s_pre[mid] <= k) glo = mid;
            else ghi = mid - 1;
        }
        int64_t b = (int64_t)glo * per, left = k - (int64_t)s_pre[glo];
        while (b + 1 < nb && b + 1 < (int64_t)(glo + 1) * per && (int64_t)bsum[b] <= left) left -= bsum[b++];
        int64_t lo = b * kB, hi = (b + 1) * kB < W ? (b + 1) * kB - 1 : W - 1;
        while (lo < hi) {
            const int64_t mid = (lo + hi + 1) >> 1;
            if ((int64_t)wp[mid] <= left) lo = mid;
            else hi = mid - 1;
        }
        uint64_t hw = bits[lo];
        for (int64_t r = left - (int64_t)wp[lo]; r > 0 && hw; r--) hw &= hw - 1ull;
        if (hw == 0ull) continue;  // inconsistent bitmap: never write outside [0, S)
        const int64_t h = lo * 64 + (__ffsll((long long)hw) - 1);
        if (h < 0 || h >= S) continue;
        move_record<int64_t>(T, v, h);
    }
}

// The whole fill of a small set by one block, one launch instead of two. Each thread puts the places it looks at into two
// lists in LDS, the holes below the new size and the live records past it, in the order in which they belong
// together, so that a record needs no search and the moves are dense however much was removed. us in a graph,
// with 3, 10, 30, 50, 70 and 90% removed, five launches as it once was / the two of hf_count and hf_fill / this: 2,000
// particles 10.3 10.5 11.3 12.0 12.3 13.2 / 8.2 8.0 7.9 8.5 8.7 9.9 / 4.5 4.3 4.5 4.4 4.4 4.2; 4,000 10.6 11.5 11.9 12.7
// 12.5 14.5 / 7.4 8.5 9.0 9.2 9.2 10.8 / 4.8 4.9 5.5 5.8 5.4 4.9; 8,192 11.3 12.2 12.2 12.7 13.0 14.2 / 7.6 8.6 8.7 9.2 9.6
// 11.0 / 5.4 6.9 9.2 9.3 8.7 6.6 (a search for every record of the tail took 40 at the last). Beyond, one block is too few.
__global__ void __launch_bounds__(kSmallThreads) hf_small(const uint64_t* __restrict__ bits,
                                                          oppx_move_counters* __restrict__ ctr, CompTable T, int64_t n_max) {
    __shared__ uint16_t s_hole[32 * kSmallWords], s_live[32 * kSmallWords];  // at most half of the set moves
    __shared__ uint64_t s_bits[kSmallWords];
    __shared__ uint32_t s_pre[kSmallWords], s_wave[kSmallThreads / kWave];
    const int N = (int)live_count(ctr, n_max), W = (int)words_of(N);
    const int w = threadIdx.x, lane = w & (kWave - 1);
    const uint64_t mine = w < W ? bits[w] : 0ull;
    const uint32_t c = (uint32_t)__popcll(mine);
    uint32_t inc = c;
#pragma unroll
    for (int d = 1; d < kWave; d <<= 1) {
        const uint32_t t = __shfl_up(inc, d);
        if (lane >= d) inc += t;
    }
    if (lane == kWave - 1) s_wave[w / kWave] = inc;
    if (w < kSmallWords) s_bits[w] = mine;
    __syncthreads();  // also: every thread has read the live count
    uint32_t off = 0, total = 0;
#pragma unroll
    for (int q = 0; q < kSmallThreads / kWave; q++) {
        off += q < w / kWave ? s_wave[q] : 0u;
        total += s_wave[q];
    }
    if (w < kSmallWords) s_pre[w] = off + inc - c;
    __syncthreads();
    const int R = (int)total, S = N - R;
    const bool some = R > 0 && R <= N;
    // holes below the new size (R > 0 and not past N, so S is a place in the set)
    const int moves = some ? (int)s_pre[S >> 6] + __popcll(s_bits[S >> 6] & ((1ull << (S & 63)) - 1ull)) : 0;
    if (threadIdx.x == 0) {
        ctr->removed = R;
        ctr->holes_low = moves;
        if (some) ctr->size = S;
    }
    if (moves == 0) return;
    for (int v = (int)threadIdx.x; v < N; v += kSmallThreads) {
        const uint64_t word = s_bits[v >> 6];
        const int j = v & 63, below = (int)s_pre[v >> 6] + __popcll(word & ((1ull << j) - 1ull));
        const bool hole = (word >> j) & 1ull;
        if (v < S) {
            if (hole) s_hole[below] = (uint16_t)v;
        } else if (!hole) {
            const int k = (N - 1 - v) - (R - below);  // its place among the live records, from the end
            if (k >= 0) s_live[k] = (uint16_t)v;       // (below 0 only where a bit past N is set)
        }
    }
    __syncthreads();
    for (int k = (int)threadIdx.x; k < moves; k += kSmallThreads) move_record<uint32_t>(T, s_live[k], s_hole[k]);
}

struct Scratch {
    uint32_t* bsum;
    uint32_t* wp;
    uint32_t* head;  // of the 64 spare words
    int64_t nb;
};

// bsum (block counts, padded to 64 words), wp (one prefix per bitmap word) and 64 spare words
constexpr size_t scratch_need(int64_t n_max) {
    const int64_t W = (n_max + 63) / 64;
    const int64_t nb = (W + kB - 1) / kB < 1 ? 1 : (W + kB - 1) / kB;
    return (size_t)(((nb + 63) / 64) * 64 + W + 64) * sizeof(uint32_t);
}
static_assert(scratch_need(OPPX_HOLEFILL_NOALLOC_MAX_PARTICLES) <= OPPX_HOLEFILL_NOALLOC_SCRATCH_BYTES,
              "the static scratch must hold the hole fill of the largest set oppx_holefill_noalloc accepts");

Scratch carve(void* scratch, int64_t n_max) {
    const int64_t W = (n_max + 63) / 64;
    const int64_t nb = (W + kB - 1) / kB;
    Scratch s;
    s.nb = nb > 0 ? nb : 1;
    s.bsum = reinterpret_cast<uint32_t*>(scratch);
    s.wp = s.bsum + ((s.nb + 63) / 64) * 64;
    s.head = s.wp + W;
    return s;
}

int holefill_impl(int64_t n_max, int64_t stride, oppx_move_counters* counters, const uint64_t* hole_bits,
                  const oppx_dat_desc* dats, int n_dats, void* work, hipStream_t s) {
    for (int q = 0; q < n_dats; q++) {
        OPPX_ARG_CHECK(dats[q].base && dats[q].dim > 0, "oppx_holefill: bad dat descriptor");
        OPPX_ARG_CHECK(dats[q].elem_bytes == 4 || dats[q].elem_bytes == 8, "oppx_holefill: elem_bytes 4 or 8");
    }
    int comps = 0;
    for (int q = 0; q < n_dats && comps <= kMaxComps; q++) comps += dats[q].dim;
    const bool small = n_max <= 64 * kSmallWords && comps <= kMaxComps;
    // every scratch word a pass reads was written by an earlier pass of the same call: nothing to clear
    Scratch sc = carve(work, n_max);
    if (!small) {
        hf_count<<<(unsigned)sc.nb, kB, 0, s>>>(hole_bits, counters, sc.bsum, sc.wp, sc.head, n_max);
        OPPX_LAUNCH_CHECK("hf_count");
    }
    const int per = (int)((sc.nb + kMaxGroups - 1) / kMaxGroups);
    // A thread for every particle, so that at most one record is a thread's to move, whatever share was removed; more than
    // 1,024 blocks add nothing. us, with 3, 30, 60 and 90% removed, five launches as it once was / a block for 2,048
    // particles / this: 9,000 particles 11.5 12.6 12.9 14.3 / 8.2 17.5 26.7 40.6 / 7.8 9.0 9.4 10.9, 131,072 14.9 15.5 16.3
    // 16.9 / 9.8 20.5 30.9 52.5 / 9.9 11.1 11.6 12.9, 1 M 18.8 33.1 41.2 50.6 / 12.3 29.8 41.5 60.4 / 12.3 25.8 33.2 37.9,
    // 24 M 332 824 1,060 1,444 / 320 826 722 844 / 321 826 722 842.
    int64_t g = (n_max + kB - 1) / kB;
    g = g < 1 ? 1 : (g > 1024 ? 1024 : g);
    CompTable T{};
    for (int q = 0, d = 0; q < n_dats;) {  // flatten the dats; a full table is launched and started again
        if (dats[q].elem_bytes == 8) T.wide |= 1ull << T.n;
        T.base[T.n++] = reinterpret_cast<char*>(dats[q].base) + (size_t)d * (size_t)stride * (size_t)dats[q].elem_bytes;
        if (++d == dats[q].dim) { d = 0; q++; }
        if (T.n == kMaxComps || q == n_dats) {
            if (small) hf_small<<<1, kSmallThreads, 0, s>>>(hole_bits, counters, T, n_max);
            else hf_fill<<<(unsigned)g, kB, 0, s>>>(hole_bits, counters, sc.bsum, sc.wp, sc.head, T, sc.nb, per, q == n_dats);
            OPPX_LAUNCH_CHECK("hf_fill");
            T = CompTable{};
        }
    }
    return OPPX_OK;
}

constexpr int kMaxDevices = 64;
std::mutex g_scratch_mu;
void* g_scratch_dev[kMaxDevices];  // address of `scratch` on each device, once looked up

}  // namespace

// Device address of the static scratch array on `device`, which must be current: looked up with
// hipGetSymbolAddress on the first call for the device, then kept.
int noalloc_scratch(int device, void** out) {
    OPPX_ARG_CHECK(device >= 0 && device < kMaxDevices, "oppx: device index beyond the static scratch table");
    std::lock_guard<std::mutex> lock(g_scratch_mu);
    if (g_scratch_dev[device] == nullptr) {
        void* p = nullptr;
        OPPX_HIP_TRY(hipGetSymbolAddress(&p, HIP_SYMBOL(scratch)));
        OPPX_ARG_CHECK(p != nullptr, "oppx: hipGetSymbolAddress returned no address for the static scratch");
        g_scratch_dev[device] = p;
    }
    if (out) *out = g_scratch_dev[device];
    return OPPX_OK;
}

}  // namespace oppx

using namespace oppx;

extern "C" {

// a move covers whole tiles: at most ceil(n_max/64) words plus one partial block of the largest tile
int64_t oppx_hole_bits_words(int64_t n_max) { return (n_max > 0 ? (n_max + 63) / 64 : 0) + 32; }

size_t oppx_holefill_scratch_bytes(int64_t n_max) { return n_max < 0 ? 0 : scratch_need(n_max); }

int oppx_holefill(int64_t n_max, int64_t stride, oppx_move_counters* counters, const uint64_t* hole_bits,
                  const oppx_dat_desc* dats, int n_dats, void* work, size_t work_bytes, void* stream) {
    OPPX_ARG_CHECK(counters && hole_bits && work, "oppx_holefill: null pointer");
    OPPX_ARG_CHECK(n_max >= 0 && stride >= n_max, "oppx_holefill: need 0 <= n_max <= stride");
    OPPX_ARG_CHECK(n_dats >= 1 && n_dats <= kMaxDats && dats, "oppx_holefill: 1..16 dats required");
    OPPX_ARG_CHECK(work_bytes >= oppx_holefill_scratch_bytes(n_max), "oppx_holefill: scratch too small");
    return holefill_impl(n_max, stride, counters, hole_bits, dats, n_dats, work, as_stream(stream));
}

int oppx_holefill_noalloc(int64_t n_max, int64_t stride, oppx_move_counters* counters, const uint64_t* hole_bits,
                          const oppx_dat_desc* dats, int n_dats, void* stream) {
    OPPX_ARG_CHECK(counters && hole_bits, "oppx_holefill_noalloc: null pointer");
    OPPX_ARG_CHECK(n_max >= 0 && stride >= n_max, "oppx_holefill_noalloc: need 0 <= n_max <= stride");
    OPPX_ARG_CHECK(n_max <= OPPX_HOLEFILL_NOALLOC_MAX_PARTICLES,
                   "oppx_holefill_noalloc: n_max exceeds OPPX_HOLEFILL_NOALLOC_MAX_PARTICLES (the static scratch "
                   "holds the hole fill of at most 134217728 particles); use oppx_holefill with a workspace");
    OPPX_ARG_CHECK(n_dats >= 1 && n_dats <= kMaxDats && dats, "oppx_holefill_noalloc: 1..16 dats required");
    int dev = 0;
    OPPX_HIP_TRY(hipGetDevice(&dev));
    void* work = nullptr;
    const int rc = noalloc_scratch(dev, &work);  // looked up by oppx_init, or here on a device's first call
    if (rc != OPPX_OK) return rc;
    return holefill_impl(n_max, stride, counters, hole_bits, dats, n_dats, work, as_stream(stream));
}

}  // extern "C"
