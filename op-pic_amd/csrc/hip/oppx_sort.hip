// Particle sort by cell on gfx950: stable LSD radix sort of (cell, index) pairs, then one
// permutation gather per particle dat (the p2c dat itself is written from the sorted keys).
//
// Reference: opp_particle_sort / the Sort_* fill policies (opp_lib/src/core/opp_particle_organize_core.cpp:98-121,
// opp_lib/src/omp/opp_particle_mover.cpp:223-265, hip opp_lib/src/hip/opp_particle_sorter.cpp:188-267) order the
// particles by p2c with removed particles (MAX_CELL_INDEX) last. Their tie order differs between backends
// (std::sort / thrust radix); this build's contract is stable by (p2c, index).
//
// Each pass sorts by one 8-bit digit. A tile is 256 * sort_items consecutive elements (tuning), each
// wave of its block a contiguous part of them; ranks come from wave-level digit matching (8 ballots
// give the lanes holding the same digit) against the wave's own digit counts, so equal digits keep
// their index order and no LDS atomic is contended by nearly sorted keys. A pass is three launches: per-tile
// digit counts (they need no ranks), one block per digit that scans its row of counts across the tiles, and
// the scatter, whose blocks scan the 256 row totals themselves to give every (digit, tile) its output
// offset. Every kernel reads the live count on the device: the histogram and scatter grids (sized by the
// capacity, capped at a few times the resident blocks) stride over the live tiles only, the counts are laid
// out with the live tile count as row stride, and the row scan covers only those. Histogram, scatter and gather
// blocks take their tiles XCD by XCD, a contiguous eighth each (XcdTiles, xcd_block): the runs that neighbouring
// tiles write, and the lines that neighbouring records are gathered from, then meet in one L2. Measured, sort of
// two-steps-old particles: 24 M lazy 587 -> 523 us, their gather 1,880 -> 1,640 us; 1 M gather 81 -> 56 us;
// 3 M 257 -> 219 us. The first row scan leaves
// the live count and the removed count in the scratch; the later launches read them there, so that the last
// one can write the counters while its other blocks still run.

#include "oppx_internal.h"

namespace oppx {
namespace {

constexpr int kB = 256;
constexpr int kItems = 16;           // elements per thread of the row scan
constexpr int kElems = kB * kItems;
constexpr int kMinSortItems = 4;     // smallest radix block (elements per thread) the scratch is sized for
constexpr int kBins = 256;
constexpr int kMaxDats = 16;
constexpr unsigned kGridMult = 4;  // grids that stride over live work: this many times the resident blocks
constexpr unsigned kMaxHistGrid = 8192;  // blocks of a histogram launch at most (one removed count each)

struct GatherTable {
    int n;
    int64_t stride;
    const void* in[kMaxDats];
    void* out[kMaxDats];
    int dim[kMaxDats];
    int eb[kMaxDats];
};

// live count behind `live` (the counters' size, or its copy in the scratch), clamped to the host's bound
__device__ __forceinline__ int64_t live_n(const int32_t* live, int64_t n_max) {
    const int64_t n = *live;
    return n < 0 ? 0 : (n > n_max ? n_max : n);
}

// What a sort does to the counters, by one thread of its last launch. state: live count, removed count.
struct Finish {
    oppx_move_counters* ctr;  // null: not the last launch
    const int32_t* state;
    int drop;
};

__device__ __forceinline__ void finish_sort(const Finish& F) {
    if (!F.ctr || blockIdx.x != 0 || threadIdx.x != 0) return;
    F.ctr->removed = F.state[1];
    F.ctr->holes_low = 0;
    if (F.drop) F.ctr->size = F.state[0] - F.state[1];
}

constexpr uint32_t kFewBatch = 32;  // tile counts of a digit in flight

// A sort of few tiles: its scatters sum the tiles' counts themselves (hist is tile-major, no row scan runs), and the
// first one also leaves the live and removed counts in `state`.
struct Few {
    const uint32_t* rem_block;
    unsigned rem_blocks;
    int32_t* state;
};

// lanes of the wave (among `active`) holding the same 8-bit digit as this lane
__device__ __forceinline__ unsigned long long digit_peers(uint32_t d, unsigned long long active) {
    unsigned long long peers = active;
#pragma unroll
    for (int bit = 0; bit < 8; bit++) {
        const unsigned long long m = __ballot((d >> bit) & 1u);
        peers &= ((d >> bit) & 1u) ? m : ~m;
    }
    return peers;
}

// Key of a particle: its cell, MAX_CELL_INDEX mapped to n_cells (the last bucket). The first digit
// pass reads the keys from p2c and takes the particle index as the value, so no key/value arrays
// are written beforehand; it also counts the removed particles.
__device__ __forceinline__ uint32_t cell_key(int32_t c, uint32_t n_cells) {
    return c == kMaxCell ? n_cells : (uint32_t)c;
}

// Per-block digit counts of one pass. All of a thread's keys are loaded before any is counted
// (independent loads in flight). Counting needs no ranks: a wave whose live lanes share one digit adds
// once (nearly sorted keys), any other wave adds per lane.
template <int ITEMS, bool FIRST, bool FEW>
__global__ void __launch_bounds__(kB) __attribute__((amdgpu_waves_per_eu(8)))
sort_hist(const uint32_t* __restrict__ keys, const int32_t* __restrict__ p2c, uint32_t n_cells,
          const int32_t* __restrict__ live, int64_t n_max, int shift, uint32_t* __restrict__ hist,
          uint32_t* __restrict__ rem_block) {
    __shared__ uint32_t s_h[kBins];
    const int64_t n = live_n(live, n_max);
    const int lane = threadIdx.x & (kWave - 1);
    // the grid strides over the tiles below the live count; tile t's count of digit d goes to
    // hist[d * tiles + t], so the scan covers the live tiles only
    const int64_t tiles = (n + kB * ITEMS - 1) / (kB * ITEMS);
    uint32_t removed = 0;  // of the wave
    const XcdTiles X(tiles);
    for (int64_t t = X.first; t < X.end; t += X.step) {
        s_h[threadIdx.x] = 0;  // each thread clears the word it wrote out last tile
        __syncthreads();
        const int64_t base = t * (kB * ITEMS);
        uint32_t key[ITEMS];
#pragma unroll
        for (int r = 0; r < ITEMS; r++) {
            const int64_t i = base + r * kB + threadIdx.x;
            key[r] = i < n ? (FIRST ? cell_key(p2c[i], n_cells) : keys[i]) : 0u;
        }
#pragma unroll
        for (int r = 0; r < ITEMS; r++) {
            const bool ok = base + r * kB + threadIdx.x < n;
            const uint32_t k = key[r];
            if (FIRST) removed += (uint32_t)__popcll(__ballot(ok && k == n_cells));
            const uint32_t d = (k >> shift) & 0xFFu;
            const unsigned long long act = __ballot(ok);
            if (act == 0ull) continue;  // uniform over the wave
            const int lead = __ffsll((long long)act) - 1;
            const uint32_t d_lead = (uint32_t)__shfl((int)d, lead);
            if (__ballot(ok && d == d_lead) == act) {
                if (lane == lead) atomicAdd(&s_h[d], (uint32_t)__popcll(act));
            } else if (ok) {
                atomicAdd(&s_h[d], 1u);
            }
        }
        __syncthreads();
        // digit-major rows of the live tiles; tile-major where the scatter sums the tiles itself
        hist[FEW ? t * kBins + threadIdx.x : (int64_t)threadIdx.x * tiles + t] = s_h[threadIdx.x];
    }
    // the block's removed particles: a word of its own, which nothing has to clear beforehand
    if (FIRST) {
        __shared__ uint32_t s_rem[kB / kWave];
        if (lane == 0) s_rem[threadIdx.x / kWave] = removed;
        __syncthreads();
        if (threadIdx.x == 0) {
            uint32_t r = 0;
            for (int w = 0; w < kB / kWave; w++) r += s_rem[w];
            rem_block[blockIdx.x] = r;
        }
    }
}

// ---- one digit pass over a tile of 256 * ITEMS consecutive elements ----
// Wave w of the block owns the 64 * ITEMS consecutive elements [w * 64 * ITEMS, (w + 1) * 64 * ITEMS)
// of the tile and takes them 64 at a time (round r: element w * 64 * ITEMS + r * 64 + lane), so an
// element's stable rank among the tile's elements of its digit is: that digit's elements in the
// waves before (summed once, after all rounds), plus the wave's own in earlier rounds (a per-wave
// count in LDS, updated round by round without block barriers), plus the lanes below holding the
// same digit (8 ballots). The tile is then laid out in LDS in digit order and each digit's run is
// written to its global offset with consecutive threads on consecutive addresses, so the global
// writes are whole runs instead of one scattered word per lane.
template <int ITEMS>
struct TileLds {
    uint32_t run[kBins];               // the tile's elements of each digit, then the digit's start in the tile
    uint32_t wave[kB / kWave][kBins];  // per-wave digit counts, then their exclusive prefix over the waves
    uint32_t base[kBins];              // global offset of each digit
    uint32_t dst[kBins];               // global offset of each digit's run of the tile
    uint32_t tot[kB / kWave];          // wave totals of the digit-start scan
    uint32_t key[kB * ITEMS], val[kB * ITEMS];
};

template <int ITEMS>
__device__ __forceinline__ int tile_elem(int tid, int r) {
    return (int)(tid / kWave) * (kWave * ITEMS) + r * kWave + (int)(tid & (kWave - 1));
}

template <int ITEMS, bool FIRST>
__device__ __forceinline__ void tile_load(const uint32_t* __restrict__ kin, const uint32_t* __restrict__ vin,
                                          const int32_t* __restrict__ p2c, uint32_t n_cells, int64_t base, int m, int tid,
                                          uint32_t (&key)[ITEMS], uint32_t (&val)[ITEMS]) {
#pragma unroll
    for (int r = 0; r < ITEMS; r++) {
        const int li = tile_elem<ITEMS>(tid, r);
        const bool ok = li < m;
        if (FIRST) {  // keys straight from p2c, the particle index as the value
            key[r] = ok ? cell_key(p2c[base + li], n_cells) : 0u;
            val[r] = (uint32_t)(base + li);
        } else {
            key[r] = ok ? kin[base + li] : 0u;
            val[r] = ok ? vin[base + li] : 0u;
        }
    }
}

// Ranks of the tile's elements inside their wave's part; leaves the tile's count of every digit in
// L.run and the exclusive prefix over the waves in L.wave. L.wave must be zeroed (and that made
// visible) by the caller.
template <int ITEMS>
__device__ __forceinline__ void tile_rank(TileLds<ITEMS>& L, int tid, const uint32_t (&key)[ITEMS], int m, int shift,
                                          uint32_t (&rank)[ITEMS]) {
    const int w = tid / kWave, lane = tid & (kWave - 1);
    const unsigned long long below = (1ull << lane) - 1ull;
#pragma unroll
    for (int r = 0; r < ITEMS; r++) {
        const bool ok = tile_elem<ITEMS>(tid, r) < m;
        const uint32_t d = (key[r] >> shift) & 0xFFu;
        const unsigned long long peers = digit_peers(d, __ballot(ok));
        // every lane reads the wave's count before the lowest lane of each digit group adds the group
        // (one wave's LDS operations complete in program order)
        const uint32_t before = L.wave[w][d];
        rank[r] = before + (uint32_t)__popcll(peers & below);
        if (ok && lane == __ffsll((long long)peers) - 1) L.wave[w][d] = before + (uint32_t)__popcll(peers);
    }
    __syncthreads();
    uint32_t run = 0;
    for (int q = 0; q < kB / kWave; q++) {
        const uint32_t c = L.wave[q][tid];
        L.wave[q][tid] = run;
        run += c;
    }
    L.run[tid] = run;
    __syncthreads();
}

// Digit starts inside the tile: exclusive scan of L.run (one digit per thread), in place.
template <int ITEMS>
__device__ __forceinline__ void tile_digit_starts(TileLds<ITEMS>& L, int tid) {
    const int w = tid / kWave, lane = tid & (kWave - 1);
    const uint32_t c = L.run[tid];
    uint32_t inc = c;
#pragma unroll
    for (int dd = 1; dd < kWave; dd <<= 1) {
        const uint32_t t = __shfl_up(inc, dd);
        if (lane >= dd) inc += t;
    }
    if (lane == kWave - 1) L.tot[w] = inc;
    __syncthreads();
    uint32_t off = 0;
    for (int q = 0; q < w; q++) off += L.tot[q];
    L.run[tid] = off + inc - c;
    __syncthreads();
}

// Digit-ordered layout in LDS, then the runs to L.dst[d] + (position in the run). Writes at or past
// `limit` are dropped (never taken by a correct sort; a bound on every store). The last pass writes no
// keys, except as sorted p2c into p2c_out (nullable; key n_cells back to MAX_CELL_INDEX).
template <int ITEMS, bool LAST>
__device__ __forceinline__ void tile_write(TileLds<ITEMS>& L, int tid, const uint32_t (&key)[ITEMS], const uint32_t (&val)[ITEMS],
                                           const uint32_t (&rank)[ITEMS], int m, int shift, uint64_t limit,
                                           uint32_t* __restrict__ kout, uint32_t* __restrict__ vout,
                                           int32_t* __restrict__ p2c_out, uint32_t n_cells) {
    const int w = tid / kWave;
#pragma unroll
    for (int r = 0; r < ITEMS; r++) {
        if (tile_elem<ITEMS>(tid, r) < m) {
            const uint32_t d = (key[r] >> shift) & 0xFFu;
            const uint32_t pos = L.run[d] + L.wave[w][d] + rank[r];
            L.key[pos] = key[r];
            L.val[pos] = val[r];
        }
    }
    __syncthreads();
#pragma unroll
    for (int r = 0; r < ITEMS; r++) {
        const int p = r * kB + tid;
        if (p < m) {
            const uint32_t k = L.key[p];
            const uint32_t d = (k >> shift) & 0xFFu;
            const uint64_t dst = (uint64_t)L.dst[d] + (uint32_t)(p - (int)L.run[d]);
            if (dst < limit) {
                if (!LAST) kout[dst] = k;
                else if (p2c_out) p2c_out[dst] = k == n_cells ? kMaxCell : (int32_t)k;
                vout[dst] = L.val[p];
            }
        }
    }
}

__device__ __forceinline__ uint32_t block_scan_excl(uint32_t v, uint32_t* total);

// Scatter of one digit pass: a tile's run of digit d goes to the elements of smaller digits (the scanned row
// totals) plus those of d in earlier tiles (the scanned row). Every block scans the 256 totals itself, which
// costs it one read of 1 KB; before, scanning digits and tiles as one array took three launches a pass.
// Four waves per SIMD: the occupancy the 16-key tile's LDS allows (four 39 KB blocks per CU), reached
// without spilling.
template <int ITEMS, bool LAST, bool FIRST, bool FEW>
__global__ void __launch_bounds__(kB) __attribute__((amdgpu_waves_per_eu(4)))
sort_scatter(const uint32_t* __restrict__ kin, const uint32_t* __restrict__ vin, const int32_t* __restrict__ p2c,
             uint32_t n_cells, const int32_t* __restrict__ live, int64_t n_max, int shift,
             const uint32_t* __restrict__ offs, const uint32_t* __restrict__ row_total, uint32_t* __restrict__ kout,
             uint32_t* __restrict__ vout, int32_t* __restrict__ p2c_out, Finish F, Few W) {
    __shared__ TileLds<ITEMS> L;
    const int64_t n = live_n(live, n_max);
    if constexpr (!FEW) {
        uint32_t all;
        const uint32_t b = block_scan_excl(row_total[threadIdx.x], &all);
        L.base[threadIdx.x] = b;
    } else if (FIRST && blockIdx.x == 0 && threadIdx.x < kWave) {  // what the row scan's last block does otherwise
        uint32_t r = 0;
        for (unsigned q = threadIdx.x; q < W.rem_blocks; q += kWave) r += W.rem_block[q];
        r = (uint32_t)wave_sum_i32((int)r);
        if (threadIdx.x == 0) {
            W.state[0] = (int32_t)n;
            W.state[1] = (int32_t)r;
        }
    }
    finish_sort(F);
    // the grid (at most the blocks that fit the chip at once) strides over the tiles that hold live
    // elements: a tile past the live count is never dispatched, where each such block would still have
    // had to be given its LDS (40 KB) before it could leave
    const int64_t tiles = (n + kB * ITEMS - 1) / (kB * ITEMS);
    const XcdTiles X(tiles);
    for (int64_t t = X.first; t < X.end; t += X.step) {
        const int64_t base = t * (kB * ITEMS);
        const int m = (int)((n - base) < kB * ITEMS ? (n - base) : kB * ITEMS);  // elements of the tile
        // the thread index, opaque to the compiler inside each tile: the per-element indexes and LDS
        // addresses derived from it are recomputed per tile instead of held in registers across the loop
        int tid = (int)threadIdx.x;
        asm volatile("" : "+v"(tid));
        for (int q = 0; q < kB / kWave; q++) L.wave[q][tid] = 0;
        if constexpr (FEW) {
            uint32_t before = 0, all = 0, total;  // of digit tid, in the tiles before and in all
            for (uint32_t q0 = 0; q0 < (uint32_t)tiles; q0 += kFewBatch) {
                uint32_t c[kFewBatch];  // loaded together: the reads' latency is what this costs
#pragma unroll
                for (uint32_t k = 0; k < kFewBatch; k++) {
                    const uint32_t q = q0 + k;
                    c[k] = q < (uint32_t)tiles ? offs[q * kBins + (uint32_t)tid] : 0u;
                }
#pragma unroll
                for (uint32_t k = 0; k < kFewBatch; k++) {
                    before += q0 + k < (uint32_t)t ? c[k] : 0u;
                    all += c[k];
                }
            }
            L.dst[tid] = block_scan_excl(all, &total) + before;
        } else {
            L.dst[tid] = L.base[tid] + offs[(uint32_t)tid * (uint32_t)tiles + (uint32_t)t];  // < 2^31 counts (n below 2^32)
        }
        uint32_t key[ITEMS], val[ITEMS], rank[ITEMS];
        tile_load<ITEMS, FIRST>(kin, vin, p2c, n_cells, base, m, tid, key, val);
        __syncthreads();
        tile_rank<ITEMS>(L, tid, key, m, shift, rank);
        tile_digit_starts<ITEMS>(L, tid);
        tile_write<ITEMS, LAST>(L, tid, key, val, rank, m, shift, (uint64_t)n, kout, vout, p2c_out, n_cells);
        __syncthreads();  // every thread is done with the tile's LDS before the next tile fills it
    }
}

__device__ __forceinline__ uint32_t block_scan_excl(uint32_t v, uint32_t* total) {
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
    *total = all;
    return off + inc - v;
}

// Block d < kBins: exclusive scan of digit d's counts over the live tiles, in place, and the digit's total. A
// chunk of kElems counts at a time passes through LDS so that global loads and stores are coalesced while each
// thread scans kItems consecutive words; word e sits at e + e / kItems (thread t's words from 17 t on: distinct
// banks across the wave). One more block in the first pass (rem_block given): the sum of the histogram blocks'
// removed counts, and the live count, for the later launches.
__global__ void __launch_bounds__(kB) sort_rows(uint32_t* __restrict__ hist, const int32_t* __restrict__ live,
                                                int64_t n_max, int64_t per_tile, uint32_t* __restrict__ row_total,
                                                const uint32_t* __restrict__ rem_block, unsigned rem_blocks,
                                                int32_t* __restrict__ state) {
    __shared__ uint32_t s_a[kElems + kElems / kItems];
    const int64_t n = live_n(live, n_max);
    if (blockIdx.x == kBins) {
        uint32_t r = 0, tot;
        for (unsigned q = threadIdx.x; q < rem_blocks; q += kB) r += rem_block[q];
        block_scan_excl(r, &tot);
        if (threadIdx.x == 0) {
            state[0] = (int32_t)n;
            state[1] = (int32_t)tot;
        }
        return;
    }
    const int64_t tiles = (n + per_tile - 1) / per_tile;
    uint32_t* __restrict__ a = hist + (int64_t)blockIdx.x * tiles;
    uint32_t carry = 0;
    for (int64_t base = 0; base < tiles; base += kElems) {
        for (int r = 0; r < kItems; r++) {
            const int e = r * kB + threadIdx.x;
            s_a[e + e / kItems] = base + e < tiles ? a[base + e] : 0u;
        }
        __syncthreads();
        const int t0 = threadIdx.x * (kItems + 1);
        uint32_t loc[kItems];
        uint32_t sum = 0;
        for (int r = 0; r < kItems; r++) {
            loc[r] = s_a[t0 + r];
            sum += loc[r];
        }
        uint32_t tot;
        uint32_t run = carry + block_scan_excl(sum, &tot);
        for (int r = 0; r < kItems; r++) {
            s_a[t0 + r] = run;
            run += loc[r];
        }
        __syncthreads();
        for (int r = 0; r < kItems; r++) {
            const int e = r * kB + threadIdx.x;
            if (base + e < tiles) a[base + e] = s_a[e + e / kItems];
        }
        carry += tot;
        __syncthreads();  // the chunk is stored before the next one is loaded
    }
    if (threadIdx.x == 0) row_total[blockIdx.x] = carry;
}

constexpr int kGatherRows = 4;   // particles a thread moves of its column
constexpr int kGatherCols = 64;  // most columns side by side in the grid
constexpr int64_t kCacheBytes = 256ll << 20;
constexpr uint32_t kGatherTiles = 512;        // tiles of a chunk
constexpr uint32_t kGatherBlocks = 1u << 18;  // workgroups of a launch

// An XCD's share of the tiles goes column by column in chunks of this many tiles: all of them where the results fit the
// cache (and then at most 2^16 workgroups move them, a 4-byte word or more a lane).
template <bool STREAM>
__host__ __device__ inline uint32_t gather_chunk(uint32_t share) {
    return share < 1 ? 1 : (!STREAM || share < kGatherTiles ? share : kGatherTiles);
}

template <typename T, bool STREAM>
__device__ __forceinline__ void gather_column(const void* in, void* out, int64_t first, const uint32_t (&from)[kGatherRows],
                                              const bool (&ok)[kGatherRows], int64_t j) {
    const T* s = reinterpret_cast<const T*>(in) + first;
    T* d = reinterpret_cast<T*>(out) + first;
    T v[kGatherRows];
#pragma unroll
    for (int r = 0; r < kGatherRows; r++)
        if (ok[r]) v[r] = s[from[r]];
#pragma unroll
    for (int r = 0; r < kGatherRows; r++)
        if (ok[r]) {
            if (STREAM) __builtin_nontemporal_store(v[r], d + j + r * kB);
            else d[j + r * kB] = v[r];
        }
}

// Bound by the lines it reads: cells of neighbouring planes take particles out of the same lines, and moving whole
// particles an XCD's L2 lost a line before its last reader came (3 M particles on 40^3 cubes: 75,000 particles
// between two planes, 6.3 MB of their dats against 4 MB of L2). So an XCD runs through its tiles one column (a
// component of a dat) after the other, where the same window is 0.6 MB, in chunks of 512 tiles, half a million
// particles, whose part of the permutation is still in L2 for the next column. Whole particles before / one column of
// the whole set after the other / chunks, pos, vel, lc and p2c, us: displaced by up to 100,000 places 1 M 118 / 64 /
// 64, 3 M 363 / 244 / 244, 24 M 2,912 / 2,102 / 2,010, 80 M 9,746 / 6,966 / 7,320; in random order 3 M 639 / 540 /
// 541, 24 M 6,355 / 5,090 / 5,090, 80 M 22,960 / 17,490 / 22,870; nearly in place already, where every line is read
// once anyway, 3 M 94 / 98 / 98, 24 M 710 / 865 / 731, 80 M 2,324 / 2,856 / 2,463. Chunks of 16 to 128 tiles lose the
// window (24 M within 3 M places 4,180 at 512, 6,300 at 32). At most 2^18 workgroups: with 16 of 100 M particles live
// the rest are launched for nothing (763 us with all, 512 so), while with 2^16 the blocks of a full set drift apart
// (24 M 2,247).
template <bool STREAM>
__global__ void __launch_bounds__(kB) sort_gather(const uint32_t* __restrict__ perm, const int32_t* __restrict__ live,
                                                  int64_t n_max, GatherTable T, int cols, int side,
                                                  int32_t* __restrict__ perm_out, Finish F) {
    const int64_t n = live_n(live, n_max);
    finish_sort(F);
    // each XCD takes one contiguous eighth of the tiles, a chunk of them at a time, column by column
    const uint32_t tiles = (uint32_t)((n + kB * kGatherRows - 1) / (kB * kGatherRows));
    const uint32_t share = (tiles + kXcds - 1) / kXcds;
    const uint32_t ch = gather_chunk<STREAM>(share), per = ch * (uint32_t)side, steps = (share + ch - 1) / ch * per;
    for (uint32_t k = blockIdx.x / kXcds; k < steps; k += STREAM ? gridDim.x / kXcds : steps) {
        const uint32_t before = STREAM ? k / per : 0u, in = k - before * per, col = in / ch;
        const uint32_t tile = before * ch + in - col * ch;
        if (STREAM && tile >= share) continue;
        const int64_t j = (int64_t)((blockIdx.x % kXcds) * share + tile) * (kB * kGatherRows) + threadIdx.x;
        uint32_t from[kGatherRows];
        bool ok[kGatherRows];
#pragma unroll
        for (int r = 0; r < kGatherRows; r++) {
            const int64_t i = j + r * kB;
            ok[r] = i < n;
            from[r] = ok[r] ? perm[i] : 0u;
            ok[r] = ok[r] && from[r] < T.stride;  // never read outside the dats
        }
        for (int c = (int)col; c < cols; c += side) {
            int q = 0, d = c;
            while (d >= T.dim[q]) d -= T.dim[q++];
            if (T.eb[q] == 8) gather_column<double, STREAM>(T.in[q], T.out[q], d * T.stride, from, ok, j);
            else gather_column<int32_t, STREAM>(T.in[q], T.out[q], d * T.stride, from, ok, j);
        }
        if (perm_out && col == 0) {
#pragma unroll
            for (int r = 0; r < kGatherRows; r++)
                if (ok[r]) perm_out[j + r * kB] = (int32_t)from[r];
        }
    }
}

void launch_gather(const uint32_t* perm, const int32_t* live, int64_t n_max, const GatherTable& T, int32_t* perm_out,
                   const Finish& finish, hipStream_t s) {
    int cols = 0;
    int64_t record = 0;
    for (int q = 0; q < T.n; q++) {
        cols += T.dim[q];
        record += (int64_t)T.dim[q] * T.eb[q];
    }
    const int side = cols < 1 ? 1 : (cols < kGatherCols ? cols : kGatherCols);
    const uint32_t share = (grid_for(n_max, kB * kGatherRows) + kXcds - 1) / kXcds;
    const bool stream = n_max * record > kCacheBytes;
    const uint32_t ch = stream ? gather_chunk<true>(share) : gather_chunk<false>(share);
    uint32_t g = (share + ch - 1) / ch * ch * (uint32_t)side * kXcds;
    if (stream && g > kGatherBlocks) g = kGatherBlocks;
    // Results past the 256 MB cache are stored streaming, which keeps the L2 for the lines being gathered (24 M a lazily
    // sorted step later 2,010 -> 1,940 us); in smaller ones the kernels that follow find their input there (serving
    // steps of 500,000 particles 150 us, 163 with streaming stores).
    if (stream) sort_gather<true><<<g, kB, 0, s>>>(perm, live, n_max, T, cols, side, perm_out, finish);
    else sort_gather<false><<<g, kB, 0, s>>>(perm, live, n_max, T, cols, side, perm_out, finish);
}

__global__ void lower_bound_kernel(const int32_t* __restrict__ p2c, const oppx_move_counters* ctr, int64_t n_max,
                                   const int32_t* __restrict__ keys, int64_t k, int64_t* __restrict__ out) {
    const int64_t j = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (j >= k) return;
    const int64_t n = live_n(&ctr->size, n_max);
    const int32_t key = keys[j];
    int64_t lo = 0, hi = n;  // first index with p2c >= key in [lo, hi]
    while (lo < hi) {
        const int64_t mid = (lo + hi) >> 1;
        if (p2c[mid] < key) lo = mid + 1;
        else hi = mid;
    }
    out[j] = lo;
}

// the counters after a sort of a set that can hold no particle (n_max 0)
__global__ void sort_empty(oppx_move_counters* ctr, int drop) {
    ctr->removed = 0;
    ctr->holes_low = 0;
    if (drop) ctr->size = 0;
}

// Tiles up to which a sort runs without its row scans, one launch less a pass: every scatter block then reads all the
// tiles' counts, 1 KB each. us, two digit passes of a lazy sort in a graph, with the scans and without: 1,000
// particles 21.7 and 16.4, 10,000 23.5 and 18.6, 30,000 24.3 and 19.3, 60,000 (59 tiles) 25.3 and 22.8, 120,000 25.0
// and 28.5 (with 16 counts in flight 15.5 / 17.8 / 20.3 / 24.9, with 64 18.0 / 20.1 / 20.6 / 21.8 at the first four).
// Not where one launch does it all: it would set the live count while its other blocks read it.
constexpr int64_t kFewTiles = 64;
struct SortScratch {
    uint32_t *ka, *va, *kb, *vb, *hist, *row_total, *rem_block;
    int32_t* state;
    int64_t nblocks;
};

// Keys per thread of a sort of at most n_max particles: tuning.sort_items, or fewer where the tiles are then too few for
// the chip's 256 CUs and a pass is one tile's chain of rounds. Measured, lazy sort with 4 / 8 / 16 keys: 20,000
// particles 27.5 / 32 / 42.5 us, 300,000 31 / 34 / 45.5, 1 M 40.5 / 40 / 49, 3 M 99 / 91 / 99.5, 6 M 159 / 139.5 / 151,
// 12 M 309 / 257 / 268, 24 M 745 / 564 / 502 us (longer runs per digit).
int tile_items(int64_t n_max, int most) {
    const int want = n_max < (1 << 20) ? 4 : (n_max < 12'000'000 ? 8 : most);
    return want < most ? want : most;
}

// int32 words of the histogram region: per-block histograms at the smallest radix block
int64_t hist_words(int64_t n_max) {
    const int64_t nb = n_max > 0 ? (n_max + kB * kMinSortItems - 1) / (kB * kMinSortItems) : 1;
    return nb * kBins;
}

size_t align256(size_t b) { return (b + 255) & ~(size_t)255; }

SortScratch carve(void* base, int64_t n_max, int items) {
    SortScratch s;
    const int64_t per_block = (int64_t)kB * items;
    s.nblocks = (n_max + per_block - 1) / per_block;
    if (s.nblocks < 1) s.nblocks = 1;
    char* p = reinterpret_cast<char*>(base);
    const size_t arr = align256((size_t)(n_max > 0 ? n_max : 1) * sizeof(uint32_t));
    s.ka = reinterpret_cast<uint32_t*>(p); p += arr;
    s.va = reinterpret_cast<uint32_t*>(p); p += arr;
    s.kb = reinterpret_cast<uint32_t*>(p); p += arr;
    s.vb = reinterpret_cast<uint32_t*>(p); p += arr;
    s.hist = reinterpret_cast<uint32_t*>(p); p += align256((size_t)hist_words(n_max) * sizeof(uint32_t));
    s.row_total = reinterpret_cast<uint32_t*>(p); p += kBins * sizeof(uint32_t);
    s.state = reinterpret_cast<int32_t*>(p); p += 256;
    s.rem_block = reinterpret_cast<uint32_t*>(p);
    return s;
}

size_t scratch_need(int64_t n_max) {
    return 4 * align256((size_t)(n_max > 0 ? n_max : 1) * 4) + align256((size_t)hist_words(n_max) * 4) +
           kBins * sizeof(uint32_t) + 256 + kMaxHistGrid * sizeof(uint32_t);
}

}  // namespace
}  // namespace oppx

using namespace oppx;

extern "C" {

size_t oppx_sort_scratch_bytes(int64_t n_max) { return n_max < 0 ? 0 : scratch_need(n_max); }

int oppx_sort_by_cell(int64_t n_max, int64_t stride, oppx_move_counters* counters, int64_t n_cells,
                      const int32_t* p2c, const oppx_dat_desc* dats, const oppx_dat_desc* out_dats, int n_dats,
                      int32_t* perm_out, int drop_removed, void* scratch, size_t scratch_bytes, void* stream) {
    OPPX_ARG_CHECK(counters && p2c && scratch, "oppx_sort_by_cell: null pointer");
    OPPX_ARG_CHECK(n_max >= 0 && stride >= n_max, "oppx_sort_by_cell: need 0 <= n_max <= stride");
    OPPX_ARG_CHECK(n_cells > 0 && n_cells < kMaxCell, "oppx_sort_by_cell: n_cells out of range");
    OPPX_ARG_CHECK(n_max < (int64_t)0xFFFFFFFFll, "oppx_sort_by_cell: n_max beyond 32-bit indices");
    OPPX_ARG_CHECK(n_dats >= 0 && n_dats <= kMaxDats && (n_dats == 0 || (dats && out_dats)),
                   "oppx_sort_by_cell: 0..16 dats with output buffers");
    OPPX_ARG_CHECK(scratch_bytes >= scratch_need(n_max), "oppx_sort_by_cell: scratch too small");
    GatherTable T{};
    T.n = 0;
    T.stride = stride;
    int32_t* p2c_out = nullptr;  // the p2c dat itself is written from the keys by the last pass
    for (int q = 0; q < n_dats; q++) {
        OPPX_ARG_CHECK(dats[q].base && out_dats[q].base && dats[q].dim > 0 && dats[q].dim == out_dats[q].dim &&
                           dats[q].elem_bytes == out_dats[q].elem_bytes &&
                           (dats[q].elem_bytes == 4 || dats[q].elem_bytes == 8) && dats[q].base != out_dats[q].base,
                       "oppx_sort_by_cell: bad dat descriptor (dims/sizes must match, output must be a separate buffer)");
        if (dats[q].base == p2c && dats[q].dim == 1 && dats[q].elem_bytes == 4 && !p2c_out) {
            p2c_out = reinterpret_cast<int32_t*>(out_dats[q].base);
            continue;
        }
        T.in[T.n] = dats[q].base;
        T.out[T.n] = out_dats[q].base;
        T.dim[T.n] = dats[q].dim;
        T.eb[T.n] = dats[q].elem_bytes;
        T.n++;
    }
    hipStream_t s = as_stream(stream);
    const int items = tile_items(n_max, g_tuning.sort_items);
    OPPX_ARG_CHECK(items == 4 || items == 8 || items == 16 || items == 32,
                   "oppx_sort_by_cell: tuning.sort_items must be 4, 8, 16 or 32");
    SortScratch sc = carve(scratch, n_max, items);
    int bits = 1;
    while (bits < 32 && ((int64_t)1 << bits) <= n_cells) bits++;  // keys are in [0, n_cells]
    const int passes = (bits + 7) / 8;
    if (n_max == 0) {
        sort_empty<<<1, 1, 0, s>>>(counters, drop_removed);
        OPPX_LAUNCH_CHECK("sort_empty");
    } else {
        uint32_t *kin = sc.ka, *vin = sc.va, *kout = sc.kb, *vout = sc.vb;
        const uint32_t kc = (uint32_t)n_cells;
        // no dat left to gather: the last digit pass writes the permutation straight into perm_out
        const bool direct = T.n == 0 && perm_out != nullptr;
        const bool gather = !direct && (T.n > 0 || perm_out);
        const bool few = items == 4 && sc.nblocks <= kFewTiles && (passes > 1 || gather);
        const Finish no_finish{nullptr, nullptr, 0}, finish{counters, sc.state, drop_removed};
        for (int pass = 0; pass < passes; pass++) {
            const int shift = 8 * pass;
            const bool first = pass == 0;
            const bool last = pass == passes - 1;  // the keys of the last pass are not needed
            uint32_t* vdst = (last && direct) ? reinterpret_cast<uint32_t*>(perm_out) : vout;
            {
                // the first pass's histogram and row scan read the counters, the later launches the scratch copy
                const int32_t* live = first ? &counters->size : sc.state;
                unsigned hist_grid = 1;
#define OPPX_HIST_W(I, F, W)                                                                                         \
    do {                                                                                                             \
        auto kern = sort_hist<I, F, W>;                                                                              \
        hist_grid = stride_grid(reinterpret_cast<const void*>(kern), kB, sc.nblocks, kGridMult);                     \
        hist_grid = xcd_grid(hist_grid < kMaxHistGrid ? hist_grid : kMaxHistGrid);                                   \
        kern<<<hist_grid, kB, 0, s>>>(kin, p2c, kc, live, n_max, shift, sc.hist, sc.rem_block);                      \
    } while (0)
#define OPPX_HIST(I, F) OPPX_HIST_W(I, F, false)
                if (few) { if (first) OPPX_HIST_W(4, true, true); else OPPX_HIST_W(4, false, true); }
                else if (items == 4) { if (first) OPPX_HIST(4, true); else OPPX_HIST(4, false); }
                else if (items == 8) { if (first) OPPX_HIST(8, true); else OPPX_HIST(8, false); }
                else if (items == 16) { if (first) OPPX_HIST(16, true); else OPPX_HIST(16, false); }
                else { if (first) OPPX_HIST(32, true); else OPPX_HIST(32, false); }
#undef OPPX_HIST
#undef OPPX_HIST_W
                OPPX_LAUNCH_CHECK("sort_hist");
                if (!few)
                    sort_rows<<<kBins + (first ? 1 : 0), kB, 0, s>>>(sc.hist, live, n_max, (int64_t)kB * items,
                                                                     sc.row_total, sc.rem_block, hist_grid, sc.state);
                OPPX_LAUNCH_CHECK("sort_rows");
#define OPPX_SCATTER(I, LST, F, FW)                                                                 \
    do {                                                                                              \
        auto kern = sort_scatter<I, LST, F, FW>;                                                     \
        const unsigned res = resident_blocks(reinterpret_cast<const void*>(kern), kB);               \
        const unsigned g = xcd_grid((int64_t)res < sc.nblocks ? res : (unsigned)sc.nblocks);           \
        kern<<<g, kB, 0, s>>>(kin, vin, p2c, kc, FW ? live : sc.state, n_max, shift, sc.hist, sc.row_total, kout, vdst, \
                              p2c_out, last && !gather ? finish : no_finish, Few{sc.rem_block, hist_grid, sc.state}); \
    } while (0)
#define OPPX_SCATTER_LF(I, FW)                                                 \
    do {                                                                       \
        if (last) { if (first) OPPX_SCATTER(I, true, true, FW); else OPPX_SCATTER(I, true, false, FW); } \
        else { if (first) OPPX_SCATTER(I, false, true, FW); else OPPX_SCATTER(I, false, false, FW); }   \
    } while (0)
                if (few) OPPX_SCATTER_LF(4, true);
                else if (items == 4) OPPX_SCATTER_LF(4, false);
                else if (items == 8) OPPX_SCATTER_LF(8, false);
                else if (items == 16) OPPX_SCATTER_LF(16, false);
                else OPPX_SCATTER_LF(32, false);
#undef OPPX_SCATTER_LF
#undef OPPX_SCATTER
                OPPX_LAUNCH_CHECK("sort_scatter");
            }
            uint32_t* t = kin; kin = kout; kout = t;
            t = vin; vin = vout; vout = t;
        }
        if (gather) {
            launch_gather(vin, sc.state, n_max, T, perm_out, finish, s);
            OPPX_LAUNCH_CHECK("sort_gather");
        }
    }
    return OPPX_OK;
}

int oppx_gather_dats(int64_t n_max, int64_t stride, const oppx_move_counters* counters, const int32_t* perm,
                     const oppx_dat_desc* dats, const oppx_dat_desc* out_dats, int n_dats, void* stream) {
    OPPX_ARG_CHECK(counters && perm && n_dats > 0 && n_dats <= kMaxDats && dats && out_dats,
                   "oppx_gather_dats: bad arguments");
    OPPX_ARG_CHECK(n_max >= 0 && stride >= n_max, "oppx_gather_dats: need 0 <= n_max <= stride");
    GatherTable T{};
    T.n = n_dats;
    T.stride = stride;
    for (int q = 0; q < n_dats; q++) {
        OPPX_ARG_CHECK(dats[q].base && out_dats[q].base && dats[q].dim > 0 && dats[q].dim == out_dats[q].dim &&
                           dats[q].elem_bytes == out_dats[q].elem_bytes &&
                           (dats[q].elem_bytes == 4 || dats[q].elem_bytes == 8) && dats[q].base != out_dats[q].base,
                       "oppx_gather_dats: bad dat descriptor");
        T.in[q] = dats[q].base;
        T.out[q] = out_dats[q].base;
        T.dim[q] = dats[q].dim;
        T.eb[q] = dats[q].elem_bytes;
    }
    if (n_max == 0) return OPPX_OK;
    launch_gather(reinterpret_cast<const uint32_t*>(perm), &counters->size, n_max, T, nullptr,
                  Finish{nullptr, nullptr, 0}, as_stream(stream));
    OPPX_LAUNCH_CHECK("gather_dats");
    return OPPX_OK;
}

int oppx_lower_bound(int64_t n_max, const oppx_move_counters* counters, const int32_t* p2c, const int32_t* keys,
                     int64_t k, int64_t* out, void* stream) {
    OPPX_ARG_CHECK(counters && p2c && keys && out && n_max >= 0 && k >= 0, "oppx_lower_bound: bad arguments");
    if (k == 0) return OPPX_OK;
    lower_bound_kernel<<<grid_for(k, kB), kB, 0, as_stream(stream)>>>(p2c, counters, n_max, keys, k, out);
    OPPX_LAUNCH_CHECK("lower_bound");
    return OPPX_OK;
}

}  // extern "C"
