// FEM-PIC particle hot path on gfx950: push, direct-hop relocation, multi-hop barycentric walk,
// FP64 atomic charge deposit, and the fused single-pass step.
//
// Elemental math: apps/app_fempic/kernels.h:93-175. Loop semantics: the generated seq/omp/hip
// loops under apps_codegen/app_fempic_cg/{seq,omp,hip}/. The reference's GCC -O3 build contracts
// the barycentric and push expressions into FMAs; they are written out here with fma() and this
// file is compiled with -ffp-contract=off so cell assignment and hop counts are bit-exact.
//
// One lane per particle; particles are SoA (coalesced), cell records are AoS (one 128 B line of
// c_det + a 32 B aux record per hop). Blocks are remapped so each XCD walks one contiguous
// eighth of the particle range.

#include "oppx_internal.h"

namespace oppx {
namespace {

constexpr int kBlock = 256;
constexpr int kMaxBlock = 1024;  // largest block of the first-hop pass

// Direct-hop overlay as a kernel sees it (one per instance in batched mode).
struct DhView {
    const int32_t* __restrict__ cell;
    int64_t dx, dy, dz;
    double mx, my, mz, inv_gs;
};

struct StepArgs {
    int64_t n_cells;
    int64_t n_nodes;
    const double* __restrict__ det;
    const oppx_tet_aux* __restrict__ aux;
    const int32_t* __restrict__ c2n;
    const double* __restrict__ ef;
    int64_t stride;
    double* __restrict__ pos;
    double* __restrict__ vel;
    double* __restrict__ lc;
    int32_t* __restrict__ p2c;
    DhView dh;
    // gather mode: particle i of the pass reads its state at perm[i] of the src arrays (a pending
    // sort permutation applied on the fly) and writes every field at i of pos/vel/lc/p2c
    const int32_t* __restrict__ perm;
    const double* __restrict__ src_pos;
    const double* __restrict__ src_vel;
    const double* __restrict__ src_lc;
    const int32_t* __restrict__ src_p2c;
    // 48-byte position/velocity records {x, y, z, vx, vy, vz}: src_rec (gather mode) replaces
    // src_pos/src_vel as the input, read at perm[i]; rec_out receives the pass's new position and
    // velocity of particle i at 6i instead of pos/vel (a step before a lazy sort)
    const double* __restrict__ src_rec;
    double* __restrict__ rec_out;
    double k, dt;
    int64_t n_max;
    int tile;        // particles per wave tile (multiple of 64, <= kMaxTile)
    int refill_min;  // free lanes that trigger a refill
    int persistent;  // 1: resident grid taking block tiles from the per-XCD queues
    int n_insts;     // batched mode: instance table size
    const int32_t* __restrict__ cell_inst;       // batched mode: instance of every cell
    const oppx_batch_inst* __restrict__ insts;   // batched mode: per-instance overlay, k, dt
    oppx_move_counters* ctr;
    struct StatSlot* slots;  // nullable: per-block statistics spread over kSlots lines, reduced after the pass
    int reset;               // first pass: clear the per-move counters (the walk pass adds to them)
    uint64_t* __restrict__ hole_bits;
    int32_t* __restrict__ hops;
    double* __restrict__ charge;
};

// findStructuredCellIndex3D (opp_lib/include/opp_direct_hop_core.h:410-426) with the x86
// size_t conversion made explicit: an axis is inside iff -1 < t < dims (t in (-1,0) truncates
// to 0); then the overlay owner (kMaxCell = no owner -> remove, opp_lib/include/opp_omp.h:206-212).
__device__ __forceinline__ int dh_lookup(const DhView& D, double x, double y, double z) {
    const double tx = (x - D.mx) * D.inv_gs;
    const double ty = (y - D.my) * D.inv_gs;
    const double tz = (z - D.mz) * D.inv_gs;
    if (!(tx > -1.0 && tx < (double)D.dx && ty > -1.0 && ty < (double)D.dy && tz > -1.0 && tz < (double)D.dz))
        return kMaxCell;
    const int64_t ix = (int64_t)tx, iy = (int64_t)ty, iz = (int64_t)tz;
    return D.cell[ix + D.dx * (iy + D.dy * iz)];
}

// Particle dats are touched once per pass: non-temporal loads and stores keep them from evicting the
// cell records the walk re-reads from L2.
template <typename T>
__device__ __forceinline__ T ld_stream(const T* p) { return __builtin_nontemporal_load(p); }
template <typename T>
__device__ __forceinline__ void st_stream(T* p, T v) { __builtin_nontemporal_store(v, p); }

typedef double f64x2 __attribute__((ext_vector_type(2)));

// Tile walk: per-block statistics go to one of kSlots slots (blockIdx modulo kSlots) instead of the single
// counters record: thousands of blocks adding to one address serialise in one L2 channel. The
// slots are zeroed before the pass and folded into the counters by slots_reduce_kernel after it.
constexpr int kSlots = 256;
struct StatSlot {
    unsigned long long hops;
    int max_hops, removed, faults, pad[3];
};

// Two-pass move: what a block of the first pass hands to the walk pass. Each block stores its own record, so
// nothing is cleared before the pass and no atomic is needed; the walk pass, which follows anyway, adds the
// records up. Before, clearing and folding the slots were launches of their own, 4.5 us each after a large kernel.
struct BlockStat {
    unsigned long long hops;
    int max_hops, removed, faults;
    int pending;  // worklist entries of the block; kScattered: none, and the walk pass deposits its particles
};
constexpr int kScattered = -1;

// The block's totals, valid in thread 0 (ends with the other threads free to leave).
__device__ __forceinline__ BlockStat block_totals(long long hsum, int hmax, int nrem, int nfault) {
    __shared__ long long s_sum[kMaxBlock / kWave];
    __shared__ int s_max[kMaxBlock / kWave], s_rem[kMaxBlock / kWave], s_flt[kMaxBlock / kWave];
    const int lane = threadIdx.x & (kWave - 1), w = threadIdx.x / kWave;
    const long long hs = wave_sum_i64(hsum);
    const int hm = wave_max_i32(hmax), nr = wave_sum_i32(nrem), nf = wave_sum_i32(nfault);
    if (lane == 0) { s_sum[w] = hs; s_max[w] = hm; s_rem[w] = nr; s_flt[w] = nf; }
    __syncthreads();
    BlockStat t{0ull, 0, 0, 0, 0};
    if (threadIdx.x == 0) {
        for (int q = 0; q < (int)(blockDim.x / kWave); q++) {
            t.hops += (unsigned long long)s_sum[q];
            t.max_hops = t.max_hops > s_max[q] ? t.max_hops : s_max[q];
            t.removed += s_rem[q];
            t.faults += s_flt[q];
        }
    }
    return t;
}

// One thread adds a block's totals to the counters.
__device__ __forceinline__ void add_stats(const StepArgs& P, const BlockStat& t) {
    if (t.hops) atomicAdd((unsigned long long*)&P.ctr->total_hops, t.hops);
    if (t.max_hops) atomicMax(&P.ctr->max_hops, t.max_hops);
    if (t.removed) atomicAdd(&P.ctr->removed, t.removed);
    if (t.faults) atomicAdd(&P.ctr->faults, t.faults);
}

__device__ __forceinline__ void block_stats(const StepArgs& P, long long hsum, int hmax, int nrem, int nfault) {
    const BlockStat t = block_totals(hsum, hmax, nrem, nfault);
    if (threadIdx.x == 0) {
        if (P.slots) {
            StatSlot* sl = P.slots + (blockIdx.x % kSlots);
            if (t.hops) atomicAdd(&sl->hops, t.hops);
            if (t.max_hops) atomicMax(&sl->max_hops, t.max_hops);
            if (t.removed) atomicAdd(&sl->removed, t.removed);
            if (t.faults) atomicAdd(&sl->faults, t.faults);
        } else {
            add_stats(P, t);
        }
    }
}

__device__ __forceinline__ void reset_counters(oppx_move_counters* ctr) {
    ctr->removed = 0;
    ctr->holes_low = 0;
    ctr->max_hops = 0;
    ctr->total_hops = 0;
    for (int x = 0; x < kXcds; x++) ctr->queue[x] = 0;
}

__global__ void slots_reset_kernel(StatSlot* slots) {
    const int t = threadIdx.x;  // kSlots threads
    slots[t].hops = 0ull;
    slots[t].max_hops = 0;
    slots[t].removed = 0;
    slots[t].faults = 0;
}

__global__ void slots_reduce_kernel(const StatSlot* slots, oppx_move_counters* ctr) {
    const int t = threadIdx.x;  // kSlots threads
    const StatSlot sl = slots[t];
    const long long hs = wave_sum_i64((long long)sl.hops);
    const int hm = wave_max_i32(sl.max_hops), nr = wave_sum_i32(sl.removed), nf = wave_sum_i32(sl.faults);
    if ((t & (kWave - 1)) == 0) {
        if (hs) atomicAdd((unsigned long long*)&ctr->total_hops, (unsigned long long)hs);
        if (hm) atomicMax(&ctr->max_hops, hm);
        if (nr) atomicAdd(&ctr->removed, nr);
        if (nf) atomicAdd(&ctr->faults, nf);
    }
}

// Workgroup-level deposit aggregation: (node, value) pairs go into an LDS open-addressing table
// (ds_add_f64), then one device-scope atomic per distinct node leaves the workgroup. Cell-ordered
// particles share most of their nodes, so this removes most of the global atomics. A pair that
// finds no slot within kProbe probes goes straight to global memory.
// What bounds the deposit is the flush: scattered FP64 adds go at some 20 a nanosecond over the whole chip,
// adds of consecutive lanes to consecutive words at 100, because those of one 128-byte line leave together. So the
// table keeps the 16 nodes of a line side by side: a node's line is hashed to one of 64 groups of 16 slots, its place
// in the group is its place in the line, and a probe moves to another group (an odd number of groups on, so that
// all are reached) at the same place. Against hashing every node by itself: 24 M particles, a pass over sorted /
// one- / two-steps-old particles 1,422 / 1,579 / 1,873 -> 1,376 / 1,441 / 1,561 us, the deposit alone (after 1, 2, 3
// unsorted steps) 612 / 887 / 1,298 -> 322 / 291 / 390 us; 1.5 M in x-fastest order 40 / 55 / 72 -> 26 / 26 / 32 us;
// 1 M in no order 229 -> 195 us. Groups of 8 and 4 slots, one group of 1024 (low bits only), and probes to the next
// slot measured between the two.
constexpr int kLine = 16;  // nodes of a 128-byte line
constexpr int kProbe = 16;
constexpr int kProbeStep = 11 * kLine;

template <int GROUP_BITS>
struct DepositTableOf {
    static constexpr int kSlots = (1 << GROUP_BITS) * kLine;
    static constexpr int kGroupBits = GROUP_BITS;
    int key[kSlots];
    double val[kSlots];
};
using DepositTable = DepositTableOf<6>;

template <typename Table>
__device__ __forceinline__ void table_clear(Table& T) {
    for (int q = threadIdx.x; q < Table::kSlots; q += blockDim.x) {
        T.key[q] = -1;
        T.val[q] = 0.0;
    }
}

enum TableAdd { kOldEntry = 0, kNewEntry = 1, kNoEntry = 2 };  // kNoEntry: the value went to global memory

template <typename Table>
__device__ __forceinline__ int table_add(Table& T, double* __restrict__ charge, int node, double v) {
    uint32_t h = ((((uint32_t)node / kLine) * 2654435761u) >> (32 - Table::kGroupBits)) * kLine + (uint32_t)node % kLine;
    for (int p = 0; p < kProbe; p++) {
        const int k = T.key[h];
        if (k == node) {
            atomicAdd(&T.val[h], v);
            return kOldEntry;
        }
        if (k == -1) {
            const int prev = atomicCAS(&T.key[h], -1, node);
            if (prev == -1 || prev == node) {
                atomicAdd(&T.val[h], v);
                return prev == -1 ? kNewEntry : kOldEntry;
            }
        }
        h = (h + kProbeStep) & (Table::kSlots - 1);
    }
    atomicAdd(charge + node, v);
    return kNoEntry;
}

template <typename Table>
__device__ __forceinline__ void table_flush(Table& T, double* __restrict__ charge) {
    for (int q = threadIdx.x; q < Table::kSlots; q += blockDim.x) {
        const int k = T.key[q];
        if (k >= 0) atomicAdd(charge + k, T.val[q]);
    }
}

// The deposit by itself: PARTS particles a lane, their cells, weights and nodes loaded before the first add. It is bound
// by the table's flush, one global add per distinct node of a block, and 512 particles have far fewer than twice the
// nodes of 256 where a cell holds a few; their table has 2048 slots. A deposit after 1, 2, 3 unsorted steps, us, one
// particle a lane and 1024 slots against two and 2048: 24 M particles in 3 M cells 324 / 293 / 382 and 255 / 215 / 237,
// 1.5 M in 197,000 27 / 26 / 32 and 26 / 23 / 28, 1 M in no order in 48,000 190 and 171; but 200,000 in 663,000 10 and
// 13: the clear and the sweep of the larger table.
template <int PARTS, int GROUP_BITS>
__global__ void __launch_bounds__(kBlock) fempic_deposit_kernel(StepArgs P, uint32_t nblocks) {
    int64_t n = P.ctr->size;
    n = n < 0 ? 0 : (n > P.n_max ? P.n_max : n);
    const uint32_t nlive = live_blocks(n, kBlock * PARTS, nblocks);
    if (blockIdx.x >= nlive) return;
    const uint32_t b = xcd_block(blockIdx.x, nlive);
    const int64_t S = P.stride, i0 = (int64_t)b * kBlock * PARTS + threadIdx.x;
    __shared__ DepositTableOf<GROUP_BITS> T;
    int cell[PARTS];
    double l[PARTS][4];
#pragma unroll
    for (int u = 0; u < PARTS; u++) {
        const int64_t i = i0 + u * kBlock;
        cell[u] = i < n ? ld_stream(P.p2c + i) : kMaxCell;
#pragma unroll
        for (int d = 0; d < 4; d++) l[u][d] = i < n ? ld_stream(P.lc + d * S + i) : 0.0;
    }
    table_clear(T);
    int4 m[PARTS];
    int nfault = 0;
#pragma unroll
    for (int u = 0; u < PARTS; u++) {  // particles already removed hold MAX_CELL_INDEX and are skipped
        const bool ok = (unsigned)cell[u] < (unsigned)P.n_cells;
        if (!ok && cell[u] != kMaxCell) nfault++;
        if (!ok) cell[u] = kMaxCell;
        else m[u] = *reinterpret_cast<const int4*>(P.c2n + 4 * (int64_t)cell[u]);
    }
    __syncthreads();
#pragma unroll
    for (int u = 0; u < PARTS; u++) {
        if (cell[u] == kMaxCell) continue;
        table_add(T, P.charge, m[u].x, l[u][0]);
        table_add(T, P.charge, m[u].y, l[u][1]);
        table_add(T, P.charge, m[u].z, l[u][2]);
        table_add(T, P.charge, m[u].w, l[u][3]);
    }
    __syncthreads();
    table_flush(T, P.charge);
    nfault = wave_sum_i32(nfault);
    if ((threadIdx.x & (kWave - 1)) == 0 && nfault) atomicAdd(&P.ctr->faults, nfault);
}

// The push, and with DH the relocation through the overlay (the walk runs in a second pass).
template <bool DH>
__global__ void __launch_bounds__(kBlock) fempic_push_kernel(StepArgs P, uint32_t nblocks) {
    int64_t n = P.ctr->size;
    n = n < 0 ? 0 : (n > P.n_max ? P.n_max : n);  // never beyond the host's bound
    const uint32_t nlive = live_blocks(n, kBlock, nblocks);
    if (blockIdx.x >= nlive) return;  // no block of live particles left for this workgroup
    const uint32_t b = xcd_block(blockIdx.x, nlive);
    const int64_t i = (int64_t)b * kBlock + threadIdx.x;
    const int64_t S = P.stride;

    const int cell = i < n ? P.p2c[i] : kMaxCell;
    // a particle already holding MAX_CELL_INDEX is skipped, as the reference loops do
    // (apps_codegen/app_fempic_cg/seq/move_kernel_loop.hpp:92-94)
    bool fault = cell != kMaxCell && !((unsigned)cell < (unsigned)P.n_cells);
    if (cell != kMaxCell && !fault) {
        // calculate_new_pos_vel_kernel: v = fma(k, E, v); x = fma(v, dt, x)
        double x = P.pos[i], y = P.pos[S + i], z = P.pos[2 * S + i];
        const double* e = P.ef + 3 * (int64_t)cell;
        const double ex = e[0], ey = e[1], ez = e[2];
        double vx = P.vel[i], vy = P.vel[S + i], vz = P.vel[2 * S + i];
        vx = fma(P.k, ex, vx);
        x = fma(vx, P.dt, x);
        vy = fma(P.k, ey, vy);
        y = fma(vy, P.dt, y);
        vz = fma(P.k, ez, vz);
        z = fma(vz, P.dt, z);
        P.vel[i] = vx; P.vel[S + i] = vy; P.vel[2 * S + i] = vz;
        P.pos[i] = x; P.pos[S + i] = y; P.pos[2 * S + i] = z;
        if (DH) {
            const int c = dh_lookup(P.dh, x, y, z);
            P.p2c[i] = c;
            if (c != kMaxCell && !((unsigned)c < (unsigned)P.n_cells)) fault = true;
        }
    }
    block_stats(P, 0, 0, 0, fault ? 1 : 0);
}

// ---------------------------------------------------------------------------------------------
// Two-pass move. The first pass is one lane per particle over the whole set (full occupancy, every
// load independent across lanes): push, overlay lookup and up to `inline_hops` evaluations of the
// elemental move kernel. A particle still moving after that is appended to its block's worklist
// (wave-aggregated append) with its current cell in p2c; the second pass walks only those, on a
// resident grid, to completion, and adds up the first pass's statistics. Per-particle results are those
// of the single walk.

enum HopResult { kHopInside = 0, kHopMove = 1, kHopExit = 2, kHopBad = 3 };

// One evaluation of apps/app_fempic/kernels.h:106-161 at `cell`: inside -> kHopInside; otherwise
// cell becomes the face neighbour of the most negative weight (first index wins ties), or
// kMaxCell when that face is on the boundary. In two steps, the four weights and what follows from them, so
// that the cell's records (its 128 B c_det line and 32 B aux record {c2, c2c[0..1], c2c[2..3], pad}) can come
// from global memory or from LDS.
__device__ __forceinline__ double hop_weight(double c2, double2 ab, double2 gd, double x, double y, double z) {
    return c2 * fma(-gd.y, z, fma(gd.x, y, fma(-ab.y, x, ab.x)));  // alpha, beta ; gamma, delta of one vertex
}

__device__ __forceinline__ int hop_choose(const StepArgs& P, double c2c01, double c2c23, int& cell, double l0, double l1,
                                          double l2, double l3) {
    if ((l0 > -1e-10) && ((l0 - 1.0) < 1e-10) && (l1 > -1e-10) && ((l1 - 1.0) < 1e-10) && (l2 > -1e-10) &&
        ((l2 - 1.0) < 1e-10) && (l3 > -1e-10) && ((l3 - 1.0) < 1e-10))
        return kHopInside;
    const int2 n01 = __builtin_bit_cast(int2, c2c01), n23 = __builtin_bit_cast(int2, c2c23);
    int nb = n01.x;
    double ml = l0;
    if (l1 < ml) { ml = l1; nb = n01.y; }
    if (l2 < ml) { ml = l2; nb = n23.x; }
    if (l3 < ml) { ml = l3; nb = n23.y; }
    if (nb < 0) {
        cell = kMaxCell;
        return kHopExit;
    }
    if (nb >= P.n_cells) return kHopBad;
    cell = nb;
    return kHopMove;
}

__device__ __forceinline__ int hop_eval(const StepArgs& P, double x, double y, double z, int& cell, double& l0,
                                        double& l1, double& l2, double& l3) {
    const double2* __restrict__ d = reinterpret_cast<const double2*>(P.det + 16 * (int64_t)cell);
    const double2 a0 = d[0], a1 = d[1], a2 = d[2], a3 = d[3], a4 = d[4], a5 = d[5], a6 = d[6], a7 = d[7];
    const double4 au = *reinterpret_cast<const double4*>(P.aux + cell);
    l0 = hop_weight(au.x, a0, a1, x, y, z);
    l1 = hop_weight(au.x, a2, a3, x, y, z);
    l2 = hop_weight(au.x, a4, a5, x, y, z);
    l3 = hop_weight(au.x, a6, a7, x, y, z);
    return hop_choose(P, au.y, au.z, cell, l0, l1, l2, l3);
}

// How an evaluation's result ends a walk of the first pass (h evaluations so far): kWalkOn (still moving),
// kWalkIn (inside its cell), kWalkOut (removed), kWalkBad (fault) or kWalkHandOff (to the worklist).
enum WalkState { kWalkOn = 0, kWalkIn = 1, kWalkOut = 2, kWalkBad = 3, kWalkHandOff = 4 };
__device__ __forceinline__ int walk_state(int r, int h, int inline_hops) {
    if (r == kHopInside) return kWalkIn;
    if (r == kHopExit) return kWalkOut;
    if (r == kHopBad || h >= OPPX_MAX_HOPS) return kWalkBad;
    return h >= inline_hops ? kWalkHandOff : kWalkOn;
}

// The first pass's walks, wave by wave: the lanes still moving need 160 bytes of cell records each, and loading
// them lane by lane (ten 16-byte loads at 64 unrelated lines each) kept the vector memory unit's addresser busy
// nine tenths of the pass. Here the wave's lanes fetch the records together, straight into LDS
// (global_load_lds, 16 bytes a lane): eight lanes take one 128-byte c_det line and two lanes one aux record, so one
// instruction brings 8 lines, or 32 aux records, whole, and needs no registers for them. Only as many records as there
// are lanes still moving are fetched, and neighbouring lanes in one cell share one (without an overlay, a sorted
// wave starts in a handful of cells). The buffer holds 32 records: with the 21 KB of a block seven blocks fit a
// CU; a wave with more goes twice. In LDS the 16-byte chunk q of record r sits at q ^ (r & 7), so that lanes
// reading the same chunk of consecutive records meet different banks. The weights are computed one vertex at a time
// and the particle index is recomputed after the push (an opaque copy), which keeps the kernel at 72 registers and
// seven waves per SIMD without spills; five waves (natural, 95 registers) were slower than the lane-wise loads.
// Measured, 24 M particles in 3 M tets (a pass over sorted, one- and two-steps-old particles): 1,551 / 1,771 / 2,063 us
// with lane-wise loads behind a block cache of the first evaluation's cells, 1,433 / 1,575 / 1,859 us so (without
// the deposit 1,346 / 1,491 / 1,608 and 1,190 / 1,283 / 1,388), and 1,868 -> 1,739 us through a sort's permutation;
// 3 M: 195 / 219 / 236 -> 181 / 199 / 218 us. 24 or 16 records at eight waves (64 registers, 4-6 spilled): 1,750 /
// 1,875 / 2,154 us and more.
constexpr int kCoopRecs = 32;
struct CoopBuf {
    double2 det[kCoopRecs * 8];
    double2 aux[kCoopRecs * 2];
    int cell[kCoopRecs];
};

// 16 bytes per lane from `src` (the lane's own) to dst + 16 * lane (dst wave-uniform), asynchronously.
__device__ __forceinline__ void load_to_lds(const void* src, void* dst) {
    __builtin_amdgcn_global_load_lds((const __attribute__((address_space(1))) void*)src,
                                     (__attribute__((address_space(3))) void*)dst, 16, 0, 0);
}

// Walks the wave's moving lanes until each has ended, or has made inline_hops evaluations.
__device__ __forceinline__ void coop_walk(const StepArgs& P, CoopBuf& C, bool moving, int lane, double x, double y, double z,
                                          int& cell, double& l0, double& l1, double& l2, double& l3, int& h, int& walk,
                                          int inline_hops) {
    static_assert(kCoopRecs % 8 == 0 && kCoopRecs <= 32, "an aux load brings 32 records");
    unsigned long long m;
    while ((m = __ballot(moving)) != 0ull) {
        const int prev = __shfl_up(cell, 1);
        const bool lead = moving && (lane == 0 || !((m >> (lane - 1)) & 1ull) || prev != cell);
        const unsigned long long leads = __ballot(lead);
        const int rank = __popcll(leads & ((2ull << lane) - 1ull)) - 1;  // the record of a moving lane
        const int total = __popcll(leads);
        for (int base = 0; base < total; base += kCoopRecs) {
            const int cnt = total - base < kCoopRecs ? total - base : kCoopRecs;
            const int r = rank - base;
            const bool mine = ((m >> lane) & 1ull) && r >= 0 && r < cnt;
            if (mine && lead) C.cell[r] = cell;
            __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
#pragma unroll
            for (int q = 0; q < kCoopRecs / 8; q++) {
                const int rec = q * 8 + (lane >> 3);
                if (rec < cnt)
                    load_to_lds(P.det + 16 * (int64_t)C.cell[rec] + 2 * ((lane & 7) ^ (rec & 7)), &C.det[q * 64]);
            }
            if ((lane >> 1) < cnt)
                load_to_lds(reinterpret_cast<const double*>(P.aux + C.cell[lane >> 1]) + 2 * (lane & 1), C.aux);
            asm volatile("s_waitcnt vmcnt(0)" ::: "memory");  // the records are in LDS
            if (mine) {
                const double2 a0 = C.aux[2 * r];
                const char* row = reinterpret_cast<const char*>(C.det + 8 * r);
                const int sw = (r & 7) << 4;
                double l[4];
#pragma unroll
                for (int v = 0; v < 4; v++) {
                    const double2 ab = *reinterpret_cast<const double2*>(row + ((32 * v) ^ sw));
                    const double2 gd = *reinterpret_cast<const double2*>(row + ((32 * v + 16) ^ sw));
                    l[v] = hop_weight(a0.x, ab, gd, x, y, z);
                    __builtin_amdgcn_sched_barrier(0);  // one vertex's coefficients in registers at a time
                }
                l0 = l[0]; l1 = l[1]; l2 = l[2]; l3 = l[3];
                const int res = hop_choose(P, a0.y, C.aux[2 * r + 1].x, cell, l0, l1, l2, l3);
                h++;
                walk = walk_state(res, h, inline_hops);
                moving = walk == kWalkOn;
            }
            // The next batch may overwrite the buffer: its loads need C.cell, and LDS reads return in order, so those
            // above have returned before any of them is issued.
            __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
        }
    }
}

// LDS of a first-pass block: the record staging, the waves' fetch buffers and the deposit table in turn.
template <int BS, bool COOP>
union FirstLds {
    DepositTable dep;
    double2 stage[3 * BS];
    CoopBuf coop[BS / kWave];
};
template <int BS>
union FirstLds<BS, false> {
    DepositTable dep;
};

// What the first pass leaves for the walk pass: one record per block, and the blocks' worklists, `parts`
// (the particles of a block) entries {particle, hops so far} each.
struct WorkList {
    BlockStat* __restrict__ rec;
    int2* __restrict__ entry;
    int parts;
};

template <int BS, bool PUSH, bool DH, bool DEPOSIT, bool BATCH, bool GATHER, bool DENSE, bool COOP>
__global__ void __launch_bounds__(BS) __attribute__((amdgpu_waves_per_eu(COOP && BS == kBlock ? 7 : 4)))
fempic_first_kernel(StepArgs P, uint32_t nblocks, int inline_hops, WorkList W) {
    int64_t n = P.ctr->size;
    n = n < 0 ? 0 : (n > P.n_max ? P.n_max : n);
    // workgroups past the blocks of live particles (the grid is sized by the host's bound) leave at
    // once; the removal-bitmap words past the live count are never read
    const uint32_t nlive = live_blocks(n, BS, nblocks);
    if (P.reset && blockIdx.x == 0 && threadIdx.x == 0) reset_counters(P.ctr);
    if (blockIdx.x >= nlive) return;
    __shared__ int s_pending;
    __shared__ unsigned s_order;  // deposits << 12 + new first nodes; from kKeep on: the table stays
    constexpr unsigned kKeep = 1u << 28;
    if (threadIdx.x == 0) s_pending = s_order = 0;  // a barrier comes before their first use
    if constexpr (!COOP) __syncthreads();  // here, where no load is waited for yet
    const uint32_t b = xcd_block(blockIdx.x, nlive);
    int64_t i = (int64_t)b * BS + threadIdx.x;
    const bool live = i < n;
    const int64_t S = P.stride;
    const int lane = threadIdx.x & (kWave - 1);
    const double* __restrict__ spos = GATHER ? P.src_pos : P.pos;
    const double* __restrict__ svel = GATHER ? P.src_vel : P.vel;
    const int32_t* __restrict__ sp2c = GATHER ? P.src_p2c : P.p2c;
    // streamed particle loads are non-temporal; loads through a permutation are ordinary cached
    // loads, so the neighbours of a gathered word still find its line in L2
    auto ld = [](const auto* p) { return GATHER ? *p : ld_stream(p); };
    uint32_t from = (uint32_t)i;
    bool fault = false;
    if (GATHER && live) {
        from = (uint32_t)P.perm[i];
        if (!((uint64_t)from < (uint64_t)S)) {  // a corrupt permutation entry: report, touch nothing
            fault = true;
            from = (uint32_t)i;
        }
    }
    int64_t src = from;

    // the sort may have written the sorted p2c into the target already (src_p2c null): read in place
    const bool p2c_in_place = GATHER && P.src_p2c == nullptr;
    int cell = (live && !fault) ? (p2c_in_place ? ld_stream(P.p2c + i) : ld(sp2c + src)) : kMaxCell;
    // a particle already holding MAX_CELL_INDEX is skipped, as the reference loops do
    // (apps_codegen/app_fempic_cg/seq/move_kernel_loop.hpp:92-94)
    const bool skip = live && !fault && cell == kMaxCell;
    fault = fault || (live && !skip && !((unsigned)cell < (unsigned)P.n_cells));
    bool removed = false, pending = false, pushed = false, p2c_done = false, lc_done = false;
    int h = 0;
    double l0 = 0.0, l1 = 0.0, l2 = 0.0, l3 = 0.0;
    __shared__ FirstLds<BS, COOP> s_lds;
    DepositTable& s_table = s_lds.dep;

    // push: the particle's new position and velocity (or, for a particle this pass does not push, the
    // ones it carries over)
    const bool go = live && !skip && !fault;
    double x = 0.0, y = 0.0, z = 0.0, vx = 0.0, vy = 0.0, vz = 0.0;
    DhView D = P.dh;
    if (go) {
        double kk = P.k, dt = P.dt;
        if (BATCH) {  // the instance of the particle's cell supplies k, dt and its overlay
            const int in = P.cell_inst[cell];
            if ((unsigned)in < (unsigned)P.n_insts) {
                const oppx_batch_inst* I = P.insts + in;
                kk = I->k;
                dt = I->dt;
                D.cell = I->dh_cell;
                D.dx = I->dims[0]; D.dy = I->dims[1]; D.dz = I->dims[2];
                D.mx = I->min[0]; D.my = I->min[1]; D.mz = I->min[2];
                D.inv_gs = I->inv_gs;
            } else {
                fault = true;
            }
        }
        if (!fault) {
            if (GATHER && P.src_rec) {  // one 48-byte record instead of six SoA words at permuted addresses
                const double2* r = reinterpret_cast<const double2*>(P.src_rec + 6 * src);
                const double2 r0 = r[0], r1 = r[1], r2 = r[2];
                x = r0.x; y = r0.y; z = r1.x; vx = r1.y; vy = r2.x; vz = r2.y;
            } else {
                x = ld(spos + src); y = ld(spos + S + src); z = ld(spos + 2 * S + src);
                if (PUSH) { vx = ld(svel + src); vy = ld(svel + S + src); vz = ld(svel + 2 * S + src); }
            }
            if (PUSH) {
                // calculate_new_pos_vel_kernel: v = fma(k, E, v); x = fma(v, dt, x)
                const double* e = P.ef + 3 * (int64_t)cell;
                const double ex = e[0], ey = e[1], ez = e[2];
                vx = fma(kk, ex, vx);
                x = fma(vx, dt, x);
                vy = fma(kk, ey, vy);
                y = fma(vy, dt, y);
                vz = fma(kk, ez, vz);
                z = fma(vz, dt, z);
                if (!P.rec_out) {
                    st_stream(P.vel + i, vx); st_stream(P.vel + S + i, vy); st_stream(P.vel + 2 * S + i, vz);
                    st_stream(P.pos + i, x); st_stream(P.pos + S + i, y); st_stream(P.pos + 2 * S + i, z);
                }
                pushed = true;
            }
        }
    }
    if ((GATHER || P.rec_out) && live && !pushed) {
        // every field of the output slot is written: what the pass did not produce is carried over
        double pv[6];
        if (GATHER && P.src_rec) {
            for (int d = 0; d < 6; d++) pv[d] = P.src_rec[6 * src + d];
        } else {
            for (int d = 0; d < 3; d++) {
                pv[d] = spos[d * S + src];
                pv[3 + d] = svel[d * S + src];
            }
        }
        if (P.rec_out) {
            x = pv[0]; y = pv[1]; z = pv[2]; vx = pv[3]; vy = pv[4]; vz = pv[5];
        } else {
            for (int d = 0; d < 3; d++) {
                st_stream(P.pos + d * S + i, pv[d]);
                st_stream(P.vel + d * S + i, pv[3 + d]);
            }
        }
    }
    // records out (block-uniform): every live particle's {x, y, z, vx, vy, vz}. Where there is LDS for it the wave's 64
    // records pass through it so that each of the three 16-byte stores of a lane lands next to its neighbours' (1 KB
    // contiguous per instruction)
    if (P.rec_out) {
        if constexpr (COOP) {
            const int wave = threadIdx.x / kWave;
            f64x2* slice = reinterpret_cast<f64x2*>(s_lds.stage) + wave * (3 * kWave);
            if (live) {
                slice[3 * lane] = f64x2{x, y};
                slice[3 * lane + 1] = f64x2{z, vx};
                slice[3 * lane + 2] = f64x2{vy, vz};
            }
            __syncthreads();
            const int64_t base = (int64_t)b * BS + wave * kWave;  // first particle of the wave
            const int64_t nw = n - base;                          // live particles of the wave
            f64x2* dst = reinterpret_cast<f64x2*>(P.rec_out + 6 * base);
            for (int k = 0; k < 3; k++) {
                const int q = k * kWave + lane;  // pair q of the wave's 192: record q / 3
                if (q / 3 < nw) __builtin_nontemporal_store(slice[q], dst + q);
            }
        } else if (live) {  // ordinary stores: L2 merges a wave's three partial-line writes into whole lines
            f64x2* r = reinterpret_cast<f64x2*>(P.rec_out + 6 * i);
            r[0] = f64x2{x, y};
            r[1] = f64x2{z, vx};
            r[2] = f64x2{vy, vz};
        }
    }
    if constexpr (COOP) __syncthreads();  // the staging's readers are done, and s_pending is set
    {   // the indexes, opaque: addresses formed above are not kept in registers across the walk
        uint32_t at = (uint32_t)i;
        asm volatile("" : "+v"(at));
        i = at;
        if (GATHER) {
            asm volatile("" : "+v"(from));
            src = from;
        }
    }

    // direct hop
    bool moving = false;
    int walk = kWalkOn;
    if (go && !fault) {
        if (DH && (!BATCH || D.cell != nullptr)) {
            cell = dh_lookup(D, x, y, z);
            if (cell == kMaxCell) removed = true;
            else if (!((unsigned)cell < (unsigned)P.n_cells)) fault = true;
        }
        moving = !removed && !fault;
    }
    if constexpr (COOP) {
        coop_walk(P, s_lds.coop[threadIdx.x / kWave], moving, lane, x, y, z, cell, l0, l1, l2, l3, h, walk, inline_hops);
    } else {
        while (moving) {
            const int r = hop_eval(P, x, y, z, cell, l0, l1, l2, l3);
            h++;
            walk = walk_state(r, h, inline_hops);
            moving = walk == kWalkOn;
        }
    }
    removed = removed || walk == kWalkOut;
    fault = fault || walk == kWalkBad;
    pending = walk == kWalkHandOff;
    if (DEPOSIT) {
        __syncthreads();  // every wave is done with its fetch buffer
        table_clear(s_table);
    }
    if (go) {
        if (!fault) {
            if (!pending && !removed && h > 0) {
                st_stream(P.lc + i, l0); st_stream(P.lc + S + i, l1);
                st_stream(P.lc + 2 * S + i, l2); st_stream(P.lc + 3 * S + i, l3);
                lc_done = true;
            }
            st_stream(P.p2c + i, removed ? kMaxCell : cell);  // a pending particle resumes from `cell`
            p2c_done = true;
        }
        if (P.hops) st_stream(P.hops + i, h);
    }
    if (GATHER && live) {
        // (a pending particle's lc is final only after the worklist walk, which overwrites this)
        if (!p2c_done && !p2c_in_place) st_stream(P.p2c + i, sp2c[src]);
        if (!lc_done)
            for (int d = 0; d < 4; d++) st_stream(P.lc + d * S + i, P.src_lc[d * S + src]);
        if (P.hops && !(live && !skip && !fault)) P.hops[i] = h;
    }

    // hand the still-moving particles to the block's worklist
    const unsigned long long pmask = __ballot(pending);
    if (pmask) {
        int base = 0;
        if (lane == 0) base = atomicAdd(&s_pending, __popcll(pmask));
        base = __shfl(base, 0);
        if (pending)
            W.entry[(int64_t)blockIdx.x * BS + base + __popcll(pmask & ((1ull << lane) - 1ull))] = make_int2((int)i, h);
    }
    bool scattered = false;  // of the block
    if (DEPOSIT) {
        const bool give = live && !skip && !fault && !removed && !pending;
        __syncthreads();  // table cleared
        int4 m = make_int4(0, 0, 0, 0);
        if (give) m = *reinterpret_cast<const int4*>(P.c2n + 4 * (int64_t)cell);
        if constexpr (DENSE) {
            // Particles in no order: nearly every one of them brings a first node that no other has. The block then
            // forgets its table and leaves its deposit to the walk pass -- unless something has left the table
            // already, or the walk pass could not tell which particles deposit.
            const int first = give ? table_add(s_table, P.charge, m.x, l0) : kOldEntry;
            const int gives = __popcll(__ballot(give)), news = __popcll(__ballot(first == kNewEntry));
            const bool keep = __ballot(fault || pending || first == kNoEntry) != 0ull;
            if (lane == 0) atomicAdd(&s_order, keep ? kKeep : ((unsigned)gives << 12) + (unsigned)news);
            __syncthreads();
            const unsigned order = s_order, all = order >> 12;
            scattered = order < kKeep && all >= 64 && 4 * (order & 0xFFFu) > 3 * all;
        }
        if (!scattered) {
            if (give) {
                if (!DENSE) table_add(s_table, P.charge, m.x, l0);
                table_add(s_table, P.charge, m.y, l1);
                table_add(s_table, P.charge, m.z, l2);
                table_add(s_table, P.charge, m.w, l3);
            }
            __syncthreads();
            table_flush(s_table, P.charge);
        }
    }
    // removal bitmap: one word per wave, written for every word the grid covers
    const unsigned long long rmask = __ballot(live && removed);
    if (lane == 0) P.hole_bits[i >> 6] = rmask;
    const bool done = live && !skip && !pending;
    BlockStat t = block_totals(done ? h : 0, done ? h : 0, (live && removed) ? 1 : 0, fault ? 1 : 0);
    if (threadIdx.x == 0) {
        t.pending = scattered ? kScattered : s_pending;
        if (W.rec) W.rec[blockIdx.x] = t;
        else add_stats(P, t);
    }
}

// ---------------------------------------------------------------------------------------------
// Quad variant of the first pass: four lanes walk one particle. Lane r of a quad owns vertex r of the
// current tet: it loads that vertex's four plane coefficients (32 B of the tet's 128 B c_det line) and
// one 8 B word of the 32 B aux record, and computes lc_r; the quad combines the inside test and the
// first-minimum neighbour choice through quad DPP moves, so every branch is the same in all four lanes.
// Per hop a lane issues 3 loads instead of the one-lane walk's 10, the four lanes of a quad touch one
// line per load, and a wave's longest walk is the longest of 16 particles instead of 64. The push is
// split the same way (lane d < 3 owns component d), so are the deposit's four node adds and the lc stores.
// Same results as fempic_first_kernel.
constexpr int kQuadBlock = 256;                  // threads per block
constexpr int kQuadParts = kQuadBlock / 4;       // particles per block (one 64-bit removal word)

// Value of lane SRC of the quad (DPP quad_perm broadcast); every lane of the quad must be active.
template <int SRC>
__device__ __forceinline__ int quad_bcast_i32(int v) {
    return __builtin_amdgcn_mov_dpp(v, SRC * 0x55, 0xF, 0xF, false);
}
template <int SRC>
__device__ __forceinline__ double quad_bcast(double v) {
    const int2 h = __builtin_bit_cast(int2, v);
    return __builtin_bit_cast(double, make_int2(quad_bcast_i32<SRC>(h.x), quad_bcast_i32<SRC>(h.y)));
}
// AND over the quad (quad_perm [1,0,3,2] then [2,3,0,1]).
__device__ __forceinline__ int quad_and(int v) {
    v &= __builtin_amdgcn_mov_dpp(v, 0xB1, 0xF, 0xF, false);
    v &= __builtin_amdgcn_mov_dpp(v, 0x4E, 0xF, 0xF, false);
    return v;
}
// Bits 0, 4, 8, ..., 60 of m packed into bits 0..15.
__device__ __forceinline__ uint32_t every_fourth_bit(unsigned long long m) {
    m &= 0x1111111111111111ull;
    m = (m | (m >> 3)) & 0x0303030303030303ull;
    m = (m | (m >> 6)) & 0x000F000F000F000Full;
    m = (m | (m >> 12)) & 0x000000FF000000FFull;
    m = (m | (m >> 24)) & 0xFFFFull;
    return (uint32_t)m;
}

// One evaluation of apps/app_fempic/kernels.h:106-161 by the quad at `cell` (quad-uniform): lane r
// returns lc_r in l; the result code and the new cell are the same in all four lanes.
__device__ __forceinline__ int quad_hop(const StepArgs& P, int r, double x, double y, double z, int& cell, double& l) {
    const double2* __restrict__ d = reinterpret_cast<const double2*>(P.det + 16 * (int64_t)cell + 4 * r);
    const double2 ab = d[0], gd = d[1];  // alpha, beta ; gamma, delta of vertex r
    const double w = reinterpret_cast<const double*>(P.aux + cell)[r];  // c2 | c2c[0..1] | c2c[2..3] | pad
    const double c2 = quad_bcast<0>(w);
    l = c2 * fma(-gd.y, z, fma(gd.x, y, fma(-ab.y, x, ab.x)));
    const int in = (l > -1e-10) && ((l - 1.0) < 1e-10);
    if (quad_and(in)) return kHopInside;
    const double l0 = quad_bcast<0>(l), l1 = quad_bcast<1>(l), l2 = quad_bcast<2>(l), l3 = quad_bcast<3>(l);
    const int2 n01 = __builtin_bit_cast(int2, quad_bcast<1>(w)), n23 = __builtin_bit_cast(int2, quad_bcast<2>(w));
    int nb = n01.x;
    double ml = l0;
    if (l1 < ml) { ml = l1; nb = n01.y; }
    if (l2 < ml) { ml = l2; nb = n23.x; }
    if (l3 < ml) { ml = l3; nb = n23.y; }
    if (nb < 0) {
        cell = kMaxCell;
        return kHopExit;
    }
    if (nb >= P.n_cells) return kHopBad;
    cell = nb;
    return kHopMove;
}

template <bool PUSH, bool DH, bool DEPOSIT, bool BATCH, bool GATHER>
__global__ void __launch_bounds__(kQuadBlock) fempic_quad_kernel(StepArgs P, uint32_t nblocks, int inline_hops, WorkList W) {
    int64_t n = P.ctr->size;
    n = n < 0 ? 0 : (n > P.n_max ? P.n_max : n);
    const uint32_t nlive = live_blocks(n, kQuadParts, nblocks);
    if (P.reset && blockIdx.x == 0 && threadIdx.x == 0) reset_counters(P.ctr);
    if (blockIdx.x >= nlive) return;  // no block of live particles left for this workgroup
    const uint32_t b = xcd_block(blockIdx.x, nlive);
    const int r = threadIdx.x & 3;
    const int64_t i = (int64_t)b * kQuadParts + (threadIdx.x >> 2);
    const bool live = i < n;                     // quad-uniform
    const int64_t S = P.stride;
    const int lane = threadIdx.x & (kWave - 1), wave = threadIdx.x / kWave;
    const double* __restrict__ spos = GATHER ? P.src_pos : P.pos;
    const double* __restrict__ svel = GATHER ? P.src_vel : P.vel;
    const int32_t* __restrict__ sp2c = GATHER ? P.src_p2c : P.p2c;
    auto ld = [](const auto* p) { return GATHER ? *p : ld_stream(p); };
    int64_t src = i;
    bool fault = false;
    if (GATHER && live) {
        src = P.perm[i];
        if (!((uint64_t)src < (uint64_t)S)) {
            fault = true;
            src = i;
        }
    }
    const bool p2c_in_place = GATHER && P.src_p2c == nullptr;
    int cell = (live && !fault) ? (p2c_in_place ? ld_stream(P.p2c + i) : ld(sp2c + src)) : kMaxCell;
    const bool skip = live && !fault && cell == kMaxCell;
    fault = fault || (live && !skip && !((unsigned)cell < (unsigned)P.n_cells));
    bool removed = false, pending = false, pushed = false, p2c_done = false, lc_done = false;
    int h = 0;
    double l = 0.0;
    __shared__ DepositTable s_table;
    __shared__ uint32_t s_bits[kQuadBlock / kWave];
    __shared__ int s_pending;
    if (threadIdx.x == 0) s_pending = 0;
    if (DEPOSIT) table_clear(s_table);
    __syncthreads();

    if (live && !skip && !fault) {
        double kk = P.k, dt = P.dt;
        DhView D = P.dh;
        if (BATCH) {
            const int in = P.cell_inst[cell];
            if ((unsigned)in < (unsigned)P.n_insts) {
                const oppx_batch_inst* I = P.insts + in;
                kk = I->k;
                dt = I->dt;
                D.cell = I->dh_cell;
                D.dx = I->dims[0]; D.dy = I->dims[1]; D.dz = I->dims[2];
                D.mx = I->min[0]; D.my = I->min[1]; D.mz = I->min[2];
                D.inv_gs = I->inv_gs;
            } else {
                fault = true;
            }
        }
        if (!fault) {
            // lane d < 3 owns component d: x_d (and, pushing, v_d = fma(k, E_d, v_d); x_d = fma(v_d, dt, x_d))
            const int d = r < 3 ? r : 2;
            const bool from_rec = GATHER && P.src_rec;
            double xd = from_rec ? P.src_rec[6 * src + d] : ld(spos + d * S + src);
            if (PUSH) {
                const double e = P.ef[3 * (int64_t)cell + d];
                double vd = from_rec ? P.src_rec[6 * src + 3 + d] : ld(svel + d * S + src);
                vd = fma(kk, e, vd);
                xd = fma(vd, dt, xd);
                if (r < 3) {
                    if (P.rec_out) {
                        st_stream(P.rec_out + 6 * i + d, xd);
                        st_stream(P.rec_out + 6 * i + 3 + d, vd);
                    } else {
                        st_stream(P.vel + d * S + i, vd);
                        st_stream(P.pos + d * S + i, xd);
                    }
                }
                pushed = true;
            }
            const double x = quad_bcast<0>(xd), y = quad_bcast<1>(xd), z = quad_bcast<2>(xd);
            if (DH && (!BATCH || D.cell != nullptr)) {
                cell = dh_lookup(D, x, y, z);
                if (cell == kMaxCell) removed = true;
                else if (!((unsigned)cell < (unsigned)P.n_cells)) fault = true;
            }
            while (!removed && !fault) {
                const int res = quad_hop(P, r, x, y, z, cell, l);
                h++;
                if (res == kHopInside) break;
                if (res == kHopExit) { removed = true; break; }
                if (res == kHopBad || h >= OPPX_MAX_HOPS) { fault = true; break; }
                if (h >= inline_hops) { pending = true; break; }
            }
        }
        if (!fault) {
            if (!pending && !removed && h > 0) {
                st_stream(P.lc + r * S + i, l);
                lc_done = true;
            }
            if (r == 0) st_stream(P.p2c + i, removed ? kMaxCell : cell);
            p2c_done = true;
        }
        if (P.hops && r == 0) st_stream(P.hops + i, h);
    }
    if ((GATHER || P.rec_out) && live && !pushed && r < 3) {  // carry over what the pass did not push
        const bool from_rec = GATHER && P.src_rec;
        const double xr = from_rec ? P.src_rec[6 * src + r] : spos[r * S + src];
        const double vr = from_rec ? P.src_rec[6 * src + 3 + r] : svel[r * S + src];
        if (P.rec_out) {
            st_stream(P.rec_out + 6 * i + r, xr);
            st_stream(P.rec_out + 6 * i + 3 + r, vr);
        } else {
            st_stream(P.pos + r * S + i, xr);
            st_stream(P.vel + r * S + i, vr);
        }
    }
    if (GATHER && live) {
        if (!p2c_done && !p2c_in_place && r == 0) st_stream(P.p2c + i, sp2c[src]);
        if (!lc_done) st_stream(P.lc + r * S + i, P.src_lc[r * S + src]);
        if (P.hops && r == 0 && !(live && !skip && !fault)) P.hops[i] = h;
    }

    // still-moving particles go to the worklist (one entry per quad, from its lane 0)
    const bool lead = r == 0;
    const unsigned long long pmask = __ballot(pending && lead);
    if (pmask) {
        int base = 0;
        if (lane == 0) base = atomicAdd(&s_pending, __popcll(pmask));
        base = __shfl(base, 0);
        if (pending && lead)
            W.entry[(int64_t)blockIdx.x * kQuadParts + base + __popcll(pmask & ((1ull << lane) - 1ull))] =
                make_int2((int)i, h);
    }
    if (DEPOSIT) {
        if (live && !skip && !fault && !removed && !pending) {
            const int node = P.c2n[4 * (int64_t)cell + r];
            table_add(s_table, P.charge, node, l);
        }
    }
    // removal bitmap: the block's 64 particles are one word, 16 bits per wave
    const uint32_t bits16 = every_fourth_bit(__ballot(live && removed && lead));
    if (lane == 0) s_bits[wave] = bits16;
    __syncthreads();
    if (DEPOSIT) table_flush(s_table, P.charge);
    if (threadIdx.x == 0) {
        unsigned long long word = 0ull;
        for (int w = 0; w < kQuadBlock / kWave; w++) word |= (unsigned long long)s_bits[w] << (16 * w);
        P.hole_bits[b] = word;
    }
    const bool done = live && !skip && !pending && lead;
    BlockStat t = block_totals(done ? h : 0, done ? h : 0, (live && removed && lead) ? 1 : 0, (fault && lead) ? 1 : 0);
    if (threadIdx.x == 0) {
        t.pending = s_pending;
        if (W.rec) W.rec[blockIdx.x] = t;
        else add_stats(P, t);
    }
}

// The walk pass: its first `adders` blocks add up the first pass's block records, and every block walks worklists of them to
// completion. A block takes `per` first-pass blocks at a time, all of one XCD (first-pass block p ran on XCD p % 8), and
// walks their entries as one dense list.
// DENSE: it also deposits the particles of the first-pass blocks that found theirs scattered. A block then holds the
// whole charge array in LDS, adds to it there, and adds it to the global one at its end, consecutive lanes to
// consecutive nodes. Scattered adds to global memory go at 20 a nanosecond over the chip, such a sweep at 100, and LDS
// takes 16,384 scattered adds a CU in 8 us: 1 M particles in no order on 9,261 nodes,
// a fused pass 236 -> 112 us; 6 M on 15,625: 1,083 -> 627 us. In cell order no block is scattered, and a block that finds
// nothing in its first chunk looks at the records of all the others at once: a pass over 1 M on 2,197 nodes 66 (one chunk after
// the other 66, without the form 64, a pass of before it 68), 6 M on 2,197 295 (299, 292, 295), 20 M on 15,625 943 (975, 950,
// 950). A look ahead of every first chunk cost unordered sets 0.8 us a pass.
template <bool DEPOSIT, bool DENSE>
__global__ void __launch_bounds__(DENSE ? kMaxBlock : kBlock) fempic_walk_kernel(StepArgs P, WorkList W, uint32_t nblocks,
                                                                                 int per, uint32_t adders) {
    constexpr int BT = DENSE ? kMaxBlock : kBlock;
    extern __shared__ double s_dense[];
    int64_t n = P.ctr->size;
    n = n < 0 ? 0 : (n > P.n_max ? P.n_max : n);
    const uint32_t nlive = live_blocks(n, W.parts, nblocks);
    const uint32_t x = blockIdx.x % kXcds, mine = nlive > x ? (nlive - x + kXcds - 1) / kXcds : 0;
    const uint32_t chunks = (mine + per - 1) / per;
    const int64_t S = P.stride;
    __shared__ DepositTable s_table;
    __shared__ int s_off[BT], s_wave[BT / kWave];
    const int lane = threadIdx.x & (kWave - 1), wave = threadIdx.x / kWave;

    long long hsum = 0;
    int hmax = 0, nrem = 0, nfault = 0;
    bool used = false;  // s_dense holds something (uniform over the block)
    bool looked = false;
    auto take = [&](const BlockStat& t) {
        hsum += (long long)t.hops;
        hmax = hmax > t.max_hops ? hmax : t.max_hops;
        nrem += t.removed;
        nfault += t.faults;
    };
    if (blockIdx.x < adders)
        for (uint32_t q = blockIdx.x * BT + threadIdx.x; q < nlive; q += adders * BT) take(W.rec[q]);
    if constexpr (!DENSE) {  // the records of the block's chunks, without a barrier between them
        int any = 0;
#pragma unroll 4
        for (uint32_t c = blockIdx.x / kXcds; c < chunks; c += gridDim.x / kXcds) {
            if ((int)threadIdx.x >= per || c * (uint32_t)per + threadIdx.x >= mine) continue;
            any |= W.rec[x + kXcds * (c * (uint32_t)per + threadIdx.x)].pending;
        }
        if (!__syncthreads_or(any)) {  // the usual case: nothing was handed over
            if (blockIdx.x < adders) block_stats(P, hsum, hmax, nrem, nfault);
            return;
        }
    }
    for (uint32_t c = blockIdx.x / kXcds; c < chunks; c += gridDim.x / kXcds) {
        const uint32_t first = x + kXcds * c * (uint32_t)per;  // first-pass blocks first, first + 8, ...
        BlockStat t{0ull, 0, 0, 0, 0};
        if ((int)threadIdx.x < per && c * (uint32_t)per + threadIdx.x < mine) t = W.rec[first + kXcds * threadIdx.x];
        if (!__syncthreads_or(t.pending)) {
            if (DENSE && !looked) {  // particles in order, most likely: the chunks to come at one look
                looked = true;
                int any = 0;
                for (uint32_t e = threadIdx.x;; e += BT) {
                    const uint32_t k = (c + (1 + e / (uint32_t)per) * (gridDim.x / kXcds)) * (uint32_t)per + e % (uint32_t)per;
                    if (k >= mine) break;  // (k grows with e)
                    any |= W.rec[x + kXcds * k].pending;
                }
                if (!__syncthreads_or(any)) break;
            }
            continue;
        }
        if constexpr (DENSE) {
            s_off[threadIdx.x] = t.pending;
            if (__syncthreads_or(t.pending == kScattered)) {
                if (!used) {
                    for (int64_t q = threadIdx.x; q < P.n_nodes; q += BT) s_dense[q] = 0.0;
                    used = true;
                    __syncthreads();
                }
                for (int e = threadIdx.x; e < per * kBlock; e += BT) {
                    const int k = e / kBlock;  // the chunk's k-th first-pass block
                    if (s_off[k] != kScattered) continue;
                    const int64_t i = (int64_t)xcd_block(first + kXcds * (uint32_t)k, nlive) * kBlock + e % kBlock;
                    if (i >= n) continue;
                    const int cell = ld_stream(P.p2c + i);
                    const double l0 = ld_stream(P.lc + i), l1 = ld_stream(P.lc + S + i),
                                 l2 = ld_stream(P.lc + 2 * S + i), l3 = ld_stream(P.lc + 3 * S + i);
                    if (!((unsigned)cell < (unsigned)P.n_cells)) continue;  // removed
                    const int4 m = *reinterpret_cast<const int4*>(P.c2n + 4 * (int64_t)cell);
                    auto add = [&](int node, double v) {
                        if ((uint64_t)node < (uint64_t)P.n_nodes) atomicAdd(&s_dense[node], v);
                        else atomicAdd(P.charge + node, v);
                    };
                    add(m.x, l0);
                    add(m.y, l1);
                    add(m.z, l2);
                    add(m.w, l3);
                }
            }
            __syncthreads();
            t.pending = t.pending == kScattered ? 0 : t.pending;
        }
        int inc = t.pending;  // exclusive scan of the worklist lengths over the block
#pragma unroll
        for (int d = 1; d < kWave; d <<= 1) {
            const int v = __shfl_up(inc, d);
            if (lane >= d) inc += v;
        }
        if (lane == kWave - 1) s_wave[wave] = inc;
        __syncthreads();
        int off = 0, total = 0;
        for (int q = 0; q < BT / kWave; q++) {
            if (q < wave) off += s_wave[q];
            total += s_wave[q];
        }
        s_off[threadIdx.x] = off + inc - t.pending;
        // block-uniform rounds of BT entries; with the deposit, the LDS table is flushed after every
        // round so that it never fills (a full table sends every further add to a global atomic)
        for (int base = 0; base < total; base += BT) {
            if (DEPOSIT) table_clear(s_table);
            __syncthreads();  // table cleared, offsets written
            const int e = base + (int)threadIdx.x;
            if (e < total) {
                int lo = 0, hi = per - 1;  // the last worklist that begins at or before entry e
                while (lo < hi) {
                    const int mid = (lo + hi + 1) >> 1;
                    if (s_off[mid] <= e) lo = mid;
                    else hi = mid - 1;
                }
                const int2 w = W.entry[(int64_t)(first + kXcds * (uint32_t)lo) * W.parts + (e - s_off[lo])];
                const int64_t i = w.x;
                int h = w.y;
                int cell = P.p2c[i];
                const bool rec = P.rec_out != nullptr;  // the first pass left the pushed position in a record
                const double px = rec ? P.rec_out[6 * i] : P.pos[i];
                const double py = rec ? P.rec_out[6 * i + 1] : P.pos[S + i];
                const double pz = rec ? P.rec_out[6 * i + 2] : P.pos[2 * S + i];
                double l0 = 0.0, l1 = 0.0, l2 = 0.0, l3 = 0.0;
                bool removed = false, fault = !((unsigned)cell < (unsigned)P.n_cells);
                while (!fault) {
                    const int r = hop_eval(P, px, py, pz, cell, l0, l1, l2, l3);
                    h++;
                    if (r == kHopInside) break;
                    if (r == kHopExit) { removed = true; break; }
                    if (r == kHopBad || h >= OPPX_MAX_HOPS) fault = true;
                }
                if (!fault) {
                    P.lc[i] = l0; P.lc[S + i] = l1; P.lc[2 * S + i] = l2; P.lc[3 * S + i] = l3;
                    P.p2c[i] = removed ? kMaxCell : cell;
                    if (removed) {
                        atomicOr((unsigned long long*)&P.hole_bits[i >> 6], 1ull << (i & 63));
                        nrem++;
                    } else if (DEPOSIT) {
                        const int4 m = *reinterpret_cast<const int4*>(P.c2n + 4 * (int64_t)cell);
                        table_add(s_table, P.charge, m.x, l0);
                        table_add(s_table, P.charge, m.y, l1);
                        table_add(s_table, P.charge, m.z, l2);
                        table_add(s_table, P.charge, m.w, l3);
                    }
                } else {
                    nfault++;
                }
                if (P.hops) P.hops[i] = h;
                hsum += h;
                hmax = hmax > h ? hmax : h;
            }
            __syncthreads();  // the round's adds are in the table; its entries' offsets are read
            if (DEPOSIT) {
                table_flush(s_table, P.charge);
                __syncthreads();
            }
        }
    }
    if (DENSE && used) {
        __syncthreads();
        const int64_t from = P.n_nodes * blockIdx.x / gridDim.x;  // blocks start at different nodes
        for (int64_t q = threadIdx.x; q < P.n_nodes; q += BT) {
            const int64_t node = q + from < P.n_nodes ? q + from : q + from - P.n_nodes;
            if (s_dense[node] != 0.0) atomicAdd(P.charge + node, s_dense[node]);
        }
    }
    block_stats(P, hsum, hmax, nrem, nfault);
}

// Zero the per-XCD queue counters before a launch that uses them.
__global__ void reset_queue_kernel(oppx_move_counters* ctr) {
    if (threadIdx.x < kXcds) ctr->queue[threadIdx.x] = 0;
}

// ---------------------------------------------------------------------------------------------
// Wavefront-cooperative walk. Each wave owns a tile of kTile consecutive particles; a lane whose
// particle has finished its walk (or was removed) retires it and, once enough lanes are free,
// the free lanes take the next particles of the tile (ranks from a ballot, no atomics). Lanes
// stay busy while the longest walks of the tile finish, instead of idling until the slowest
// lane of a fixed 64-particle group is done. Removal bits gather in LDS per tile; the deposit
// is aggregated in the workgroup's LDS table.
constexpr int kMaxTile = 512;
constexpr int kMaxTileWords = kMaxTile / kWave;
constexpr int kWavesPerBlock = kBlock / kWave;

template <bool PUSH, bool DH, bool DEPOSIT, bool PRE, bool BATCH>
__global__ void __launch_bounds__(kBlock) fempic_tile_kernel(StepArgs P, uint32_t nblocks) {
    const int wave = threadIdx.x / kWave, lane = threadIdx.x & (kWave - 1);
    int64_t n = P.ctr->size;
    n = n < 0 ? 0 : (n > P.n_max ? P.n_max : n);
    const int tile = P.tile, tile_words = P.tile / kWave;
    const int64_t S = P.stride;

    __shared__ unsigned long long s_holes[kWavesPerBlock][kMaxTileWords];
    __shared__ DepositTable s_table;
    __shared__ uint32_t s_next;

    // Block tiles (kWavesPerBlock consecutive wave tiles) are split into one contiguous range per
    // XCD. A plain launch maps block ids onto those ranges; a persistent launch keeps a resident grid
    // whose blocks take the next block tile of their XCD's range from a queue in the counters.
    // Only the block tiles that hold live particles are split, so every XCD gets 1/8 of them.
    const uint32_t xcd = blockIdx.x % kXcds;
    const uint32_t nlive = live_blocks(n, (int64_t)kWavesPerBlock * tile, nblocks);
    const uint32_t q8 = nlive / kXcds, r8 = nlive % kXcds;
    const uint32_t range0 = xcd * q8 + (xcd < r8 ? xcd : r8), range_n = q8 + (xcd < r8 ? 1u : 0u);

    const unsigned long long below = (1ull << lane) - 1ull;
    long long hsum = 0;
    int hmax = 0, nfault = 0, nrem_total = 0;

    for (uint32_t round = 0;; round++) {
        uint32_t b;
        if (P.persistent) {
            if (threadIdx.x == 0) s_next = (uint32_t)atomicAdd(&P.ctr->queue[xcd], 1);
            __syncthreads();
            const uint32_t t = s_next;
            __syncthreads();
            if (t >= range_n) break;  // uniform over the block: every wave leaves here
            b = range0 + t;
        } else {
            if (round > 0 || blockIdx.x >= nlive) break;
            b = xcd_block(blockIdx.x, nlive);
        }
        // block tiles past the live count hold no particle (and later ones of this range neither)
        if ((int64_t)b * kWavesPerBlock * tile >= n) break;
        const int64_t tile0 = ((int64_t)b * kWavesPerBlock + wave) * tile;
        const int64_t tile_end = (tile0 + tile < n) ? tile0 + tile : n;

        if (lane < tile_words) s_holes[wave][lane] = 0ull;
        if (DEPOSIT) table_clear(s_table);
        __syncthreads();

        int64_t next = tile0 + kWave;  // wave-uniform: first particle no lane has taken yet
        int64_t p = tile0 + lane;
        bool have = false, walking = false, removed = false, fault = false, skip = false;
        int cell = 0, h = 0;
        double x = 0.0, y = 0.0, z = 0.0, l0 = 0.0, l1 = 0.0, l2 = 0.0, l3 = 0.0;

        auto begin = [&](int64_t q) {
            have = true;
            walking = false;
            removed = false;
            fault = false;
            skip = false;
            h = 0;
            cell = P.p2c[q];
            if (cell == kMaxCell) {
                if (PRE) removed = true;  // removed by the relocation pass
                else skip = true;         // already removed: skipped, as the reference loops do
                return;
            }
            if (!((unsigned)cell < (unsigned)P.n_cells)) {
                fault = true;
                return;
            }
            double kk = P.k, dt = P.dt;
            DhView D = P.dh;
            if (BATCH) {  // the instance of the particle's cell supplies k, dt and its overlay
                const int in = P.cell_inst[cell];
                if (!((unsigned)in < (unsigned)P.n_insts)) {
                    fault = true;
                    return;
                }
                const oppx_batch_inst* I = P.insts + in;
                kk = I->k;
                dt = I->dt;
                D.cell = I->dh_cell;
                D.dx = I->dims[0]; D.dy = I->dims[1]; D.dz = I->dims[2];
                D.mx = I->min[0]; D.my = I->min[1]; D.mz = I->min[2];
                D.inv_gs = I->inv_gs;
            }
            x = P.pos[q];
            y = P.pos[S + q];
            z = P.pos[2 * S + q];
            if (PUSH) {
                const double* e = P.ef + 3 * (int64_t)cell;
                const double ex = e[0], ey = e[1], ez = e[2];
                double vx = P.vel[q], vy = P.vel[S + q], vz = P.vel[2 * S + q];
                vx = fma(kk, ex, vx);
                x = fma(vx, dt, x);
                vy = fma(kk, ey, vy);
                y = fma(vy, dt, y);
                vz = fma(kk, ez, vz);
                z = fma(vz, dt, z);
                P.vel[q] = vx; P.vel[S + q] = vy; P.vel[2 * S + q] = vz;
                P.pos[q] = x; P.pos[S + q] = y; P.pos[2 * S + q] = z;
            }
            if (DH && (!BATCH || D.cell != nullptr)) {
                cell = dh_lookup(D, x, y, z);
                if (cell == kMaxCell) {
                    removed = true;
                    return;
                }
                if (!((unsigned)cell < (unsigned)P.n_cells)) {
                    fault = true;
                    return;
                }
            }
            walking = true;
        };

        if (p < tile_end) begin(p);

        for (;;) {
            if (walking) {
                // one evaluation of the elemental move kernel (apps/app_fempic/kernels.h:106-161)
                const double2* __restrict__ d = reinterpret_cast<const double2*>(P.det + 16 * (int64_t)cell);
                const double2 a0 = d[0], a1 = d[1], a2 = d[2], a3 = d[3], a4 = d[4], a5 = d[5], a6 = d[6], a7 = d[7];
                const double4 au = *reinterpret_cast<const double4*>(P.aux + cell);
                const double c2 = au.x;
                l0 = c2 * fma(-a1.y, z, fma(a1.x, y, fma(-a0.y, x, a0.x)));
                l1 = c2 * fma(-a3.y, z, fma(a3.x, y, fma(-a2.y, x, a2.x)));
                l2 = c2 * fma(-a5.y, z, fma(a5.x, y, fma(-a4.y, x, a4.x)));
                l3 = c2 * fma(-a7.y, z, fma(a7.x, y, fma(-a6.y, x, a6.x)));
                h++;
                if ((l0 > -1e-10) && ((l0 - 1.0) < 1e-10) && (l1 > -1e-10) && ((l1 - 1.0) < 1e-10) && (l2 > -1e-10) &&
                    ((l2 - 1.0) < 1e-10) && (l3 > -1e-10) && ((l3 - 1.0) < 1e-10)) {
                    walking = false;
                } else {
                    const int2 n01 = __builtin_bit_cast(int2, au.y), n23 = __builtin_bit_cast(int2, au.z);
                    int nb = n01.x;
                    double ml = l0;
                    if (l1 < ml) { ml = l1; nb = n01.y; }
                    if (l2 < ml) { ml = l2; nb = n23.x; }
                    if (l3 < ml) { ml = l3; nb = n23.y; }
                    if (nb < 0) {
                        removed = true;
                        cell = kMaxCell;
                        walking = false;
                    } else if (nb >= P.n_cells || h >= OPPX_MAX_HOPS) {
                        fault = true;
                        walking = false;
                    } else {
                        cell = nb;
                    }
                }
            }
            if (have && !walking) {  // retire
                if (skip) {
                    // nothing to write: the particle keeps MAX_CELL_INDEX
                } else if (!fault) {
                    if (h > 0) {
                        P.lc[p] = l0; P.lc[S + p] = l1; P.lc[2 * S + p] = l2; P.lc[3 * S + p] = l3;
                    }
                    P.p2c[p] = removed ? kMaxCell : cell;
                    if (removed) {
                        const int64_t r = p - tile0;
                        atomicOr(&s_holes[wave][r >> 6], 1ull << (r & 63));
                    } else if (DEPOSIT) {
                        const int4 m = *reinterpret_cast<const int4*>(P.c2n + 4 * (int64_t)cell);
                        table_add(s_table, P.charge, m.x, l0);
                        table_add(s_table, P.charge, m.y, l1);
                        table_add(s_table, P.charge, m.z, l2);
                        table_add(s_table, P.charge, m.w, l3);
                    }
                } else {
                    nfault++;
                }
                if (P.hops) P.hops[p] = h;
                hsum += h;
                hmax = hmax > h ? hmax : h;
                have = false;
            }
            const unsigned long long free_mask = __ballot(!have);
            const unsigned long long walk_mask = __ballot(walking);
            const int nfree = __popcll(free_mask);
            if (next < tile_end && (nfree >= P.refill_min || walk_mask == 0ull)) {
                if (!have) {
                    const int64_t q = next + __popcll(free_mask & below);
                    if (q < tile_end) {
                        p = q;
                        begin(q);
                    }
                }
                next += nfree;
            } else if (walk_mask == 0ull && __ballot(have) == 0ull) {
                break;
            }
        }

        __syncthreads();
        if (threadIdx.x < kWavesPerBlock * tile_words) {
            const int w = threadIdx.x / tile_words, k = threadIdx.x % tile_words;
            const unsigned long long bits = s_holes[w][k];
            P.hole_bits[((int64_t)b * kWavesPerBlock + w) * tile_words + k] = bits;
            nrem_total += __popcll(bits);
        }
        if (DEPOSIT) table_flush(s_table, P.charge);
        __syncthreads();  // the next round clears the table and the hole words
    }

    block_stats(P, hsum, hmax, nrem_total, nfault);
}

// Per-move reset of the counters (a kernel, not a memset, so the step can be graph-captured).
__global__ void reset_counters_kernel(oppx_move_counters* ctr) { reset_counters(ctr); }

// Start of a fused step: zero the deposit target and the per-step counters in one launch.
__global__ void step_begin_kernel(oppx_move_counters* __restrict__ ctr, double* __restrict__ charge, int64_t n_nodes) {
    const int64_t j = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (j == 0) {
        ctr->removed = 0;
        ctr->holes_low = 0;
        ctr->max_hops = 0;
        ctr->total_hops = 0;
    }
    if (j < kXcds) ctr->queue[j] = 0;
    if (charge)
        for (int64_t q = j; q < n_nodes; q += (int64_t)gridDim.x * blockDim.x) charge[q] = 0.0;
}

// c2c entries are copied as they are: a negative entry is a boundary face (the walk removes the
// particle, as the reference's `opp_c2c[min_i] >= 0` test does, apps/app_fempic/kernels.h:148-159);
// an entry at or past n_cells is a corrupt map, which the walk reports as a fault.
__global__ void tet_aux_kernel(const double* __restrict__ vol, const int32_t* __restrict__ c2c, int64_t n,
                               oppx_tet_aux* __restrict__ aux) {
    const int64_t c = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (c >= n) return;
    oppx_tet_aux a;
    a.c2 = (1.0 / 6.0) / vol[c];  // coefficient2 of apps/app_fempic/kernels.h:110, IEEE division
    for (int q = 0; q < 4; q++) a.c2c[q] = c2c[4 * c + q];
    a.pad[0] = a.pad[1] = 0;
    aux[c] = a;
}

// pos/vel SoA from 48-byte records: slot i takes record perm[i] (perm null: record i)
__global__ void __launch_bounds__(kBlock) gather_records_kernel(int64_t n_max, int64_t stride,
                                                                const oppx_move_counters* __restrict__ ctr,
                                                                const int32_t* __restrict__ perm,
                                                                const double* __restrict__ rec, double* __restrict__ pos,
                                                                double* __restrict__ vel, int32_t* __restrict__ faults) {
    int64_t n = ctr->size;
    n = n < 0 ? 0 : (n > n_max ? n_max : n);
    // A permuted record's lines in one L2: each XCD takes runs of `group` tiles, an eighth of them all in smaller sets, 64
    // tiles (16,384 particles) in larger ones, where eight regions far apart cost more than neighbouring XCDs' shared
    // lines. With 8,192 workgroups a large set's blocks strode over their tiles and drifted apart; with 65,536 most of them
    // take one tile, and they are few enough for a set of which little is left alive (16 of 113 M in order 299 / 286 / 269
    // us, 326 with 2^18). us, single tiles on 8,192 workgroups as it once was / these runs on 8,192 / on 65,536: 3 M
    // displaced by up to 100,000 places 84 / 68 / 58, 8 M 222 / 219 / 200, 24 M 702 / 679 / 615, in order 472 / 458 / 412,
    // 100 M 2,924 / 2,915 / 2,722, in order 1,963 / 1,892 / 1,798; an ensemble of 256 instances and 102 M particles after
    // its first step 3,153 / 3,215 / 2,584, 62 M after the fourth 1,773 / 1,772 / 1,515. Runs of 16 or 256 tiles 2,567 and
    // 2,699 at the last but one, eighths 2,936.
    const uint32_t tiles = (uint32_t)((n + kBlock - 1) / kBlock);
    const uint32_t group = tiles > 65536u ? 64u : (tiles + kXcds - 1) / kXcds;
    const uint32_t slots = group ? (tiles + kXcds * group - 1) / (kXcds * group) * group : 0;  // tiles of an XCD
    for (uint32_t q = blockIdx.x / kXcds; q < slots; q += gridDim.x / kXcds) {
        const int64_t t = (int64_t)(q / group * kXcds + blockIdx.x % kXcds) * group + q % group;
        const int64_t i = t * kBlock + threadIdx.x;
        if (i >= n) continue;
        const int64_t src = perm ? (int64_t)perm[i] : i;
        if (!((uint64_t)src < (uint64_t)stride)) {  // a corrupt permutation entry: report, touch nothing
            atomicAdd(faults, 1);
            continue;
        }
        const f64x2* r = reinterpret_cast<const f64x2*>(rec + 6 * src);
        const f64x2 a = r[0], b = r[1], c = r[2];
        st_stream(pos + i, a.x); st_stream(pos + stride + i, a.y); st_stream(pos + 2 * stride + i, b.x);
        st_stream(vel + i, b.y); st_stream(vel + stride + i, c.x); st_stream(vel + 2 * stride + i, c.y);
    }
}

int fill_args(StepArgs& P, const oppx_fempic_parts* parts, const oppx_tet_mesh* mesh, const oppx_dh_grid* dh,
              oppx_move_counters* ctr) {
    OPPX_ARG_CHECK(parts && mesh && ctr, "fempic: null descriptor");
    OPPX_ARG_CHECK(mesh->n_cells > 0 && mesh->n_cells < kMaxCell, "fempic: n_cells out of range");
    OPPX_ARG_CHECK(parts->stride >= 0, "fempic: negative stride");
    P = StepArgs{};
    P.n_cells = mesh->n_cells;
    P.n_nodes = mesh->n_nodes;
    P.det = mesh->det;
    P.aux = mesh->aux;
    P.c2n = mesh->c2n;
    P.ef = mesh->ef;
    P.stride = parts->stride;
    P.pos = parts->pos;
    P.vel = parts->vel;
    P.lc = parts->lc;
    P.p2c = parts->p2c;
    P.ctr = ctr;
    P.tile = g_tuning.tile;
    P.refill_min = g_tuning.refill_min;
    P.persistent = g_tuning.persistent;
    if (dh) {
        OPPX_ARG_CHECK(dh->inv_gs > 0, "fempic: overlay grid spacing must be positive");
        OPPX_ARG_CHECK(dh->cell && dh->dims[0] > 0 && dh->dims[1] > 0 && dh->dims[2] > 0, "fempic: bad overlay");
        P.dh.cell = dh->cell;
        P.dh.dx = dh->dims[0]; P.dh.dy = dh->dims[1]; P.dh.dz = dh->dims[2];
        P.dh.mx = dh->min[0]; P.dh.my = dh->min[1]; P.dh.mz = dh->min[2];
        P.dh.inv_gs = dh->inv_gs;
    }
    return OPPX_OK;
}

// Grid of a tile-kernel launch: one block per block tile, or (persistent) the resident grid,
// a multiple of the XCD count so every XCD's queue has blocks draining it.
unsigned tile_grid(const void* kernel, unsigned block_tiles, bool persistent) {
    if (!persistent) return block_tiles;
    unsigned g = resident_blocks(kernel, kBlock);
    const unsigned need = ((block_tiles + kXcds - 1) / kXcds) * kXcds;
    if (g > need) g = need;
    g = (g / kXcds) * kXcds;
    return g < (unsigned)kXcds ? (unsigned)kXcds : g;
}

template <bool PUSH, bool DH, bool DEPOSIT, bool PRE, bool BATCH>
void launch_tile(const StepArgs& P, int64_t n_max, hipStream_t s) {
    const int64_t per_block = (int64_t)P.tile * kWavesPerBlock;
    const unsigned nbt = (unsigned)((n_max + per_block - 1) / per_block);
    auto kern = fempic_tile_kernel<PUSH, DH, DEPOSIT, PRE, BATCH>;
    const unsigned g = tile_grid(reinterpret_cast<const void*>(kern), nbt, P.persistent != 0);
    if (P.persistent) reset_queue_kernel<<<1, kWave, 0, s>>>(P.ctr);
    kern<<<g, kBlock, 0, s>>>(P, nbt);
}

constexpr int kDenseNodes = 16384;  // nodes of the largest LDS charge copy (128 KB)

// Work buffer of the move. Tile walk: statistics slots [kSlots]. Two-pass move: one record per block of the
// first pass (64, 256 or 1024 particles), then the blocks' worklists.
constexpr size_t kSlotBytes = kSlots * sizeof(StatSlot);

size_t record_bytes(int64_t n_max) {
    const int64_t blocks = n_max > 0 ? (n_max + kQuadParts - 1) / kQuadParts : 0;
    return ((size_t)blocks * sizeof(BlockStat) + 255) & ~(size_t)255;
}

size_t work_need(int64_t n_max) {
    const size_t two = record_bytes(n_max) + (size_t)(n_max + kMaxBlock) * sizeof(int2);
    return two > kSlotBytes ? two : kSlotBytes;
}

// Point P's statistics at the slots of the work buffer (when it holds them) and zero them.
void attach_slots(StepArgs& P, void* work, size_t work_bytes, hipStream_t s) {
    if (!work || work_bytes < kSlotBytes) return;
    P.slots = reinterpret_cast<StatSlot*>(work);
    slots_reset_kernel<<<1, kSlots, 0, s>>>(P.slots);
}

void fold_slots(const StepArgs& P, hipStream_t s) {
    if (P.slots) slots_reduce_kernel<<<1, kSlots, 0, s>>>(P.slots, P.ctr);
}

constexpr int kLaneBlocks = 768;  // first-pass blocks up to which their lanes load cell records by themselves
constexpr int kFewBlocks = 256;  // first-pass blocks up to which there is no walk pass

// Two-pass move (first-hop pass + worklist walk) when the work buffer is large enough and the
// tuning asks for it; returns false when the caller should use the cooperative tile walk instead.
template <bool PUSH, bool DH, bool DEPOSIT, bool BATCH, bool GATHER = false>
bool launch_two_pass(const StepArgs& P, int64_t n_max, void* work, size_t work_bytes, hipStream_t s) {
    if (!work || g_tuning.inline_hops < 1 || work_bytes < work_need(n_max)) return false;
    WorkList W{reinterpret_cast<BlockStat*>(work),
               reinterpret_cast<int2*>(reinterpret_cast<char*>(work) + record_bytes(n_max)), kBlock};
    // Scattered blocks' deposits through LDS copies of the charge: 256 blocks sweep n_nodes adds each at 100 a
    // nanosecond where the particles' adds would go at 20, so from some 14 particles a node on; 32, to be clear of
    // the second read of lc and p2c. A copy fits a CU's LDS beside the rest up to 16,384 nodes.
    const bool dense = DEPOSIT && g_tuning.lanes == 1 && g_tuning.first_block == kBlock && P.n_nodes > 0 &&
                       P.n_nodes <= kDenseNodes && n_max >= 32 * P.n_nodes && n_max >= (1 << 18);
    // A few blocks walk everything themselves and add their totals to the counters, one after the other in some 10 ns each: no
    // walk pass, whose launch the smallest sets wait for. A fused step, us, with it and without: 1,000 particles 21.4 and
    // 18.4, 4,000 22.8 and 19.3, 16,000 28.9 and 25.6, 32,000 35.3 and 31.8, 65,000 36.4 and 34.4, 130,000 (508 blocks) 41 and
    // 41. Where the pass also clears the counters its blocks' adds would race that, and the walk pass adds up their records.
    const int per_block = g_tuning.lanes == 4 ? kQuadParts : (g_tuning.first_block == kMaxBlock ? kMaxBlock : kBlock);
    const bool far = !dense && g_tuning.inline_hops >= 16;
    const bool few = far && n_max <= (int64_t)kFewBlocks * per_block, alone = few && !P.reset;
    // Up to 768 blocks walk lane by lane: they wait for one evaluation after the other, 0.45 us each, where the cooperative
    // fetch takes 0.95 and pays only once the loads of many waves queue. A pass without an overlay, us, cooperative / lane
    // by lane / as it once was: 80,000 particles, walks of 2.6 evaluations at the mean 21.8 / 16.9 / 23.4, of 5.8 38 / 27 /
    // 33, of 9.6 70 / 49 / 57; 160,000 of 5.8 42 / 35 / 42, of 9.6 78 / 61 / 69; 250,000 of 2.6 28.5 / 26.5 / 31.5, but in no
    // order 75 / 79 / 92; 65,000 of which 0.1% walk 200 evaluations 128 / 84 / 96. (In larger sets such few long walks cost 10
    // to 25% over lane-wise loads, and so do particles in no order on meshes past the L2s, 3 to 11%; blocks of 1024, in
    // place, are the lane-wise form there.)
    const bool lanewise = few || (far && per_block == kBlock && n_max <= (int64_t)kLaneBlocks * kBlock);
    const int inline_hops = lanewise ? OPPX_MAX_HOPS : g_tuning.inline_hops;
    if (alone) W.rec = nullptr;
    unsigned g;
    if (g_tuning.lanes == 4) {
        W.parts = kQuadParts;
        g = grid_for(n_max, kQuadParts);
        fempic_quad_kernel<PUSH, DH, DEPOSIT, BATCH, GATHER><<<g, kQuadBlock, 0, s>>>(P, g, inline_hops, W);
    } else if (g_tuning.first_block == kMaxBlock) {
        // Of the blocks of 1024 those that read through a permutation fetch together. The 16 buffers of such a block take 84
        // KB, so that one fits a CU where two with lane-wise loads do (54 registers). In place that costs more than the
        // fetch gains: 113 M particles of 256 instances, the move of a first / second step 7.14 / 7.07 ms with the fetch, 5.85 /
        // 6.12 without, and 7.16 / 6.33 where it stages records; through a permutation, where the reads of the particles
        // themselves are the longer wait, 8.98 with it and 9.58 without.
        W.parts = kMaxBlock;
        g = grid_for(n_max, kMaxBlock);
        if constexpr (GATHER) {
            if (lanewise) fempic_first_kernel<kMaxBlock, PUSH, DH, DEPOSIT, BATCH, true, false, false>
                              <<<g, kMaxBlock, 0, s>>>(P, g, inline_hops, W);
            else fempic_first_kernel<kMaxBlock, PUSH, DH, DEPOSIT, BATCH, true, false, true>
                     <<<g, kMaxBlock, 0, s>>>(P, g, inline_hops, W);
        } else {
            fempic_first_kernel<kMaxBlock, PUSH, DH, DEPOSIT, BATCH, false, false, false>
                <<<g, kMaxBlock, 0, s>>>(P, g, inline_hops, W);
        }
    } else {
        g = grid_for(n_max, kBlock);
        if (lanewise) {
            fempic_first_kernel<kBlock, PUSH, DH, DEPOSIT, BATCH, GATHER, false, false>
                <<<g, kBlock, 0, s>>>(P, g, inline_hops, W);
        } else {
            auto first = fempic_first_kernel<kBlock, PUSH, DH, DEPOSIT, BATCH, GATHER, false, true>;
            if constexpr (DEPOSIT) {
                if (dense) first = fempic_first_kernel<kBlock, PUSH, DH, true, BATCH, GATHER, true, true>;
            }
            first<<<g, kBlock, 0, s>>>(P, g, inline_hops, W);
        }
    }
    if (alone) return true;
    // The walk pass. Its first `adders` blocks add all the records up (each adds to the one counters record: 94,000 records 9.0
    // us on 64 blocks, 13.4 on 256). The records are also dealt out evenly, for their worklists, over 512 blocks, as many as
    // keep long walks from queueing behind each other (200,000 particles walking 96 evaluations each: 723 us, on 256 blocks
    // 855, with 256 records a block and so 8 blocks 9,860; 1,024 and 2,048 no better), or over the resident grid where the
    // first pass hands over walks of fewer than 16. With dense deposits 8 records, 2048 particles, a block at a time, one block
    // a CU.
    const uint32_t each = (g + kXcds - 1) / kXcds;  // first-pass blocks of an XCD
    const void* plain = reinterpret_cast<const void*>(fempic_walk_kernel<DEPOSIT, false>);
    const unsigned cap = dense ? 256u : (g_tuning.inline_hops >= 16 ? 512u : resident_blocks(plain, kBlock));
    uint32_t per = dense ? 8u : (each * kXcds + cap - 1) / cap;
    if (per > (uint32_t)kBlock) per = kBlock;
    unsigned wg = (each + per - 1) / per * kXcds;  // every chunk of every XCD
    if (wg > cap) wg = cap / kXcds * kXcds;
    const uint32_t most = dense ? 2u * kXcds : 64u, adders = wg < most ? wg : most;
    if constexpr (DEPOSIT) {
        if (dense) {
            const size_t bytes = (size_t)P.n_nodes * sizeof(double);
            (void)hipFuncSetAttribute(reinterpret_cast<const void*>(fempic_walk_kernel<true, true>),
                                      hipFuncAttributeMaxDynamicSharedMemorySize, kDenseNodes * (int)sizeof(double));
            fempic_walk_kernel<true, true><<<wg, kMaxBlock, bytes, s>>>(P, W, g, (int)per, adders);
            return true;
        }
    }
    fempic_walk_kernel<DEPOSIT, false><<<wg, kBlock, 0, s>>>(P, W, g, (int)per, adders);
    return true;
}

// The cooperative tile walk, with or without the overlay lookup.
template <bool PUSH, bool DEPOSIT>
void launch_walk(const StepArgs& P, bool dh, int64_t n_max, hipStream_t s) {
    if (dh) launch_tile<PUSH, true, DEPOSIT, false, false>(P, n_max, s);
    else launch_tile<PUSH, false, DEPOSIT, false, false>(P, n_max, s);
}

template <bool DH, bool BATCH, bool GATHER>
void launch_rec(const StepArgs& P, bool deposit, int64_t n_max, void* work, size_t work_bytes, hipStream_t s) {
    if (deposit) launch_two_pass<true, DH, true, BATCH, GATHER>(P, n_max, work, work_bytes, s);
    else launch_two_pass<true, DH, false, BATCH, GATHER>(P, n_max, work, work_bytes, s);
}

// The fused step with 48-byte position/velocity records on either side (oppx_fempic_step_fused_rec and its
// batched form): argument checks shared by both, then the two-pass move with the gather mode when a pending
// permutation is given. P carries the mesh, particle arrays, push coefficients and (BATCH) instance tables.
template <bool BATCH>
int step_rec(StepArgs& P, const char* who, int64_t n_max, const int32_t* perm, const double* src_rec,
             const double* src_lc, const oppx_fempic_parts* parts, double* rec_out, bool dh, uint64_t* hole_bits,
             void* work, size_t work_bytes, int32_t* hops, double* node_charge, hipStream_t s) {
    const std::string w(who);
    OPPX_ARG_CHECK(perm ? (src_rec && src_lc) : (!src_rec && !src_lc),
                   w + ": src_rec and src_lc go with perm (all three or none)");
    OPPX_ARG_CHECK(perm || rec_out, w + ": neither records in nor records out");
    OPPX_ARG_CHECK(parts->lc && parts->p2c && (rec_out || (parts->pos && parts->vel)) &&
                       (perm || (parts->pos && parts->vel)),
                   w + ": particle arrays missing");
    OPPX_ARG_CHECK(!rec_out || rec_out != src_rec, w + ": rec_out must not be src_rec");
    OPPX_ARG_CHECK(!perm || src_lc != parts->lc, w + ": src_lc and parts->lc must be separate");
    OPPX_ARG_CHECK(n_max >= 0 && n_max <= parts->stride, w + ": n_max beyond capacity");
    OPPX_ARG_CHECK(hole_bits != nullptr, w + ": hole_bits required");
    OPPX_ARG_CHECK(g_tuning.inline_hops >= 1 && work && work_bytes >= work_need(n_max),
                   w + ": needs the two-pass move (tuning.inline_hops >= 1 and its workspace)");
    if (n_max == 0) return OPPX_OK;
    P.n_max = n_max;
    P.hole_bits = hole_bits;
    P.hops = hops;
    P.charge = node_charge;
    P.rec_out = rec_out;
    if (perm) {
        P.perm = perm;
        P.src_rec = src_rec;
        P.src_lc = src_lc;
        P.src_pos = nullptr;  // never read: records replace them
        P.src_vel = nullptr;
        P.src_p2c = nullptr;  // the sort wrote the sorted p2c into parts->p2c: read in place
    }
    // batched: each instance brings its own overlay (the instance table), so the DH form is the one built
    if (BATCH || dh) {
        if (perm) launch_rec<true, BATCH, true>(P, node_charge != nullptr, n_max, work, work_bytes, s);
        else launch_rec<true, BATCH, false>(P, node_charge != nullptr, n_max, work, work_bytes, s);
    } else if constexpr (!BATCH) {
        if (perm) launch_rec<false, false, true>(P, node_charge != nullptr, n_max, work, work_bytes, s);
        else launch_rec<false, false, false>(P, node_charge != nullptr, n_max, work, work_bytes, s);
    }
    OPPX_LAUNCH_CHECK(who);
    return OPPX_OK;
}

}  // namespace
}  // namespace oppx

using namespace oppx;

extern "C" {

int oppx_tet_aux_build(const double* c_vol, const int32_t* c2c, int64_t n_cells, oppx_tet_aux* aux, void* stream) {
    OPPX_ARG_CHECK(c_vol && c2c && aux && n_cells > 0, "oppx_tet_aux_build: bad arguments");
    tet_aux_kernel<<<grid_for(n_cells, 256), 256, 0, as_stream(stream)>>>(c_vol, c2c, n_cells, aux);
    OPPX_LAUNCH_CHECK("tet_aux");
    return OPPX_OK;
}

int oppx_fempic_push(int64_t n_max, const oppx_fempic_parts* parts, const oppx_tet_mesh* mesh, double k,
                     double dt, oppx_move_counters* counters, void* stream) {
    StepArgs P;
    int rc = fill_args(P, parts, mesh, nullptr, counters);
    if (rc) return rc;
    OPPX_ARG_CHECK(n_max >= 0 && n_max <= parts->stride, "oppx_fempic_push: n_max beyond capacity");
    if (n_max == 0) return OPPX_OK;
    P.n_max = n_max;
    P.k = k;
    P.dt = dt;
    const unsigned g = grid_for(n_max, kBlock);
    fempic_push_kernel<false><<<g, kBlock, 0, as_stream(stream)>>>(P, g);
    OPPX_LAUNCH_CHECK("fempic_push");
    return OPPX_OK;
}

int oppx_fempic_move(int64_t n_max, const oppx_fempic_parts* parts, const oppx_tet_mesh* mesh,
                     const oppx_dh_grid* dh, oppx_move_counters* counters, uint64_t* hole_bits, void* work,
                     size_t work_bytes, int32_t* hops, void* stream) {
    StepArgs P;
    int rc = fill_args(P, parts, mesh, dh, counters);
    if (rc) return rc;
    OPPX_ARG_CHECK(n_max >= 0 && n_max <= parts->stride, "oppx_fempic_move: n_max beyond capacity");
    OPPX_ARG_CHECK(hole_bits != nullptr, "oppx_fempic_move: hole_bits required");
    hipStream_t s = as_stream(stream);
    if (n_max == 0) {
        reset_counters_kernel<<<1, 1, 0, s>>>(counters);
        OPPX_LAUNCH_CHECK("reset_counters");
        return OPPX_OK;
    }
    P.n_max = n_max;
    P.hole_bits = hole_bits;
    P.hops = hops;
    P.reset = 1;  // the first pass clears the counters, which only the walk pass adds to
    const bool two = dh ? launch_two_pass<false, true, false, false>(P, n_max, work, work_bytes, s)
                        : launch_two_pass<false, false, false, false>(P, n_max, work, work_bytes, s);
    if (!two) {
        reset_counters_kernel<<<1, 1, 0, s>>>(counters);
        OPPX_LAUNCH_CHECK("reset_counters");
        attach_slots(P, work, work_bytes, s);
        launch_walk<false, false>(P, dh != nullptr, n_max, s);
        fold_slots(P, s);
    }
    OPPX_LAUNCH_CHECK("fempic_move");
    return OPPX_OK;
}

int oppx_fempic_deposit_atomic(int64_t n_max, const oppx_fempic_parts* parts, const oppx_tet_mesh* mesh,
                               double* node_charge, oppx_move_counters* counters, void* stream) {
    StepArgs P;
    int rc = fill_args(P, parts, mesh, nullptr, counters);
    if (rc) return rc;
    OPPX_ARG_CHECK(node_charge && mesh->c2n, "oppx_fempic_deposit_atomic: null node array or c2n");
    OPPX_ARG_CHECK(n_max >= 0 && n_max <= parts->stride, "oppx_fempic_deposit_atomic: n_max beyond capacity");
    if (n_max == 0) return OPPX_OK;
    P.n_max = n_max;
    P.charge = node_charge;
    hipStream_t s = as_stream(stream);
    // two particles a lane where their block's nodes are mostly shared, and where half the blocks still fill the chip
    if (n_max >= 2 * P.n_cells && n_max >= (1 << 18)) {
        const unsigned g = grid_for(n_max, 2 * kBlock);
        fempic_deposit_kernel<2, 7><<<g, kBlock, 0, s>>>(P, g);
    } else {
        const unsigned g = grid_for(n_max, kBlock);
        fempic_deposit_kernel<1, 6><<<g, kBlock, 0, s>>>(P, g);
    }
    OPPX_LAUNCH_CHECK("fempic_deposit");
    return OPPX_OK;
}

int oppx_fempic_step_fused(int64_t n_max, const oppx_fempic_parts* parts, const oppx_tet_mesh* mesh,
                           const oppx_dh_grid* dh, double k, double dt, oppx_move_counters* counters,
                           uint64_t* hole_bits, void* work, size_t work_bytes, int32_t* hops, double* node_charge,
                           void* stream) {
    StepArgs P;
    int rc = fill_args(P, parts, mesh, dh, counters);
    if (rc) return rc;
    OPPX_ARG_CHECK(n_max >= 0 && n_max <= parts->stride, "oppx_fempic_step_fused: n_max beyond capacity");
    OPPX_ARG_CHECK(hole_bits != nullptr, "oppx_fempic_step_fused: hole_bits required");
    hipStream_t s = as_stream(stream);
    if (n_max == 0) return OPPX_OK;
    P.n_max = n_max;
    P.k = k;
    P.dt = dt;
    P.hole_bits = hole_bits;
    P.hops = hops;
    P.charge = node_charge;
    bool two;
    if (dh) two = node_charge ? launch_two_pass<true, true, true, false>(P, n_max, work, work_bytes, s)
                              : launch_two_pass<true, true, false, false>(P, n_max, work, work_bytes, s);
    else two = node_charge ? launch_two_pass<true, false, true, false>(P, n_max, work, work_bytes, s)
                           : launch_two_pass<true, false, false, false>(P, n_max, work, work_bytes, s);
    if (!two) attach_slots(P, work, work_bytes, s);
    if (two) {
    } else if (g_tuning.split == 1 && dh != nullptr) {
        // two passes: coalesced push + overlay relocation, then the cooperative walk (+ deposit)
        fempic_push_kernel<true><<<grid_for(n_max, kBlock), kBlock, 0, s>>>(
            P, grid_for(n_max, kBlock));
        OPPX_LAUNCH_CHECK("fempic_push_relocate");
        if (node_charge) launch_tile<false, false, true, true, false>(P, n_max, s);
        else launch_tile<false, false, false, true, false>(P, n_max, s);
    } else if (node_charge) {
        launch_walk<true, true>(P, dh != nullptr, n_max, s);
    } else {
        launch_walk<true, false>(P, dh != nullptr, n_max, s);
    }
    fold_slots(P, s);
    OPPX_LAUNCH_CHECK("fempic_step_fused");
    return OPPX_OK;
}

int oppx_fempic_step_fused_gather(int64_t n_max, const int32_t* perm, const oppx_fempic_parts* src,
                                  const oppx_fempic_parts* parts, const oppx_tet_mesh* mesh, const oppx_dh_grid* dh,
                                  double k, double dt, oppx_move_counters* counters, uint64_t* hole_bits, void* work,
                                  size_t work_bytes, int32_t* hops, double* node_charge, void* stream) {
    StepArgs P;
    int rc = fill_args(P, parts, mesh, dh, counters);
    if (rc) return rc;
    OPPX_ARG_CHECK(perm && src && src->pos && src->vel && src->lc,
                   "oppx_fempic_step_fused_gather: permutation and source state required");
    OPPX_ARG_CHECK(src->stride == parts->stride, "oppx_fempic_step_fused_gather: source and target strides differ");
    OPPX_ARG_CHECK(src->pos != parts->pos && src->vel != parts->vel && src->lc != parts->lc && src->p2c != parts->p2c,
                   "oppx_fempic_step_fused_gather: source and target must be separate buffers");
    OPPX_ARG_CHECK(n_max >= 0 && n_max <= parts->stride, "oppx_fempic_step_fused_gather: n_max beyond capacity");
    OPPX_ARG_CHECK(hole_bits != nullptr, "oppx_fempic_step_fused_gather: hole_bits required");
    OPPX_ARG_CHECK(g_tuning.inline_hops >= 1 && work && work_bytes >= work_need(n_max),
                   "oppx_fempic_step_fused_gather: needs the two-pass move (tuning.inline_hops >= 1 and its workspace)");
    hipStream_t s = as_stream(stream);
    if (n_max == 0) return OPPX_OK;
    P.n_max = n_max;
    P.k = k;
    P.dt = dt;
    P.hole_bits = hole_bits;
    P.hops = hops;
    P.charge = node_charge;
    P.perm = perm;
    P.src_pos = src->pos;
    P.src_vel = src->vel;
    P.src_lc = src->lc;
    P.src_p2c = src->p2c;
    if (dh) {
        if (node_charge) launch_two_pass<true, true, true, false, true>(P, n_max, work, work_bytes, s);
        else launch_two_pass<true, true, false, false, true>(P, n_max, work, work_bytes, s);
    } else {
        if (node_charge) launch_two_pass<true, false, true, false, true>(P, n_max, work, work_bytes, s);
        else launch_two_pass<true, false, false, false, true>(P, n_max, work, work_bytes, s);
    }
    OPPX_LAUNCH_CHECK("fempic_step_fused_gather");
    return OPPX_OK;
}

int oppx_fempic_step_fused_rec(int64_t n_max, const int32_t* perm, const double* src_rec, const double* src_lc,
                               const oppx_fempic_parts* parts, double* rec_out, const oppx_tet_mesh* mesh,
                               const oppx_dh_grid* dh, double k, double dt, oppx_move_counters* counters,
                               uint64_t* hole_bits, void* work, size_t work_bytes, int32_t* hops, double* node_charge,
                               void* stream) {
    StepArgs P;
    int rc = fill_args(P, parts, mesh, dh, counters);
    if (rc) return rc;
    P.k = k;
    P.dt = dt;
    return step_rec<false>(P, "oppx_fempic_step_fused_rec", n_max, perm, src_rec, src_lc, parts, rec_out, dh != nullptr,
                           hole_bits, work, work_bytes, hops, node_charge, as_stream(stream));
}

int oppx_fempic_batch_step_fused_rec(int64_t n_max, const int32_t* perm, const double* src_rec, const double* src_lc,
                                     const oppx_fempic_parts* parts, double* rec_out, const oppx_tet_mesh* mesh,
                                     const int32_t* cell_inst, const oppx_batch_inst* insts, int32_t n_insts,
                                     oppx_move_counters* counters, uint64_t* hole_bits, void* work, size_t work_bytes,
                                     int32_t* hops, double* node_charge, void* stream) {
    StepArgs P;
    int rc = fill_args(P, parts, mesh, nullptr, counters);
    if (rc) return rc;
    OPPX_ARG_CHECK(cell_inst && insts && n_insts > 0, "oppx_fempic_batch_step_fused_rec: instance tables required");
    P.cell_inst = cell_inst;
    P.insts = insts;
    P.n_insts = n_insts;
    return step_rec<true>(P, "oppx_fempic_batch_step_fused_rec", n_max, perm, src_rec, src_lc, parts, rec_out, true,
                          hole_bits, work, work_bytes, hops, node_charge, as_stream(stream));
}

int oppx_gather_records(int64_t n_max, int64_t stride, oppx_move_counters* counters, const int32_t* perm,
                        const double* rec, double* pos, double* vel, void* stream) {
    OPPX_ARG_CHECK(counters && rec && pos && vel, "oppx_gather_records: null array");
    OPPX_ARG_CHECK(n_max >= 0 && stride >= n_max, "oppx_gather_records: need 0 <= n_max <= stride");
    if (n_max == 0) return OPPX_OK;
    unsigned g = grid_for(n_max, kBlock);
    g = xcd_grid(g > 65536 ? 65536 : g);
    gather_records_kernel<<<g, kBlock, 0, as_stream(stream)>>>(n_max, stride, counters, perm, rec, pos, vel,
                                                              &counters->faults);
    OPPX_LAUNCH_CHECK("gather_records");
    return OPPX_OK;
}

int oppx_fempic_batch_step_fused(int64_t n_max, const oppx_fempic_parts* parts, const oppx_tet_mesh* mesh,
                                 const int32_t* cell_inst, const oppx_batch_inst* insts, int32_t n_insts,
                                 oppx_move_counters* counters, uint64_t* hole_bits, void* work, size_t work_bytes,
                                 int32_t* hops, double* node_charge, void* stream) {
    StepArgs P;
    int rc = fill_args(P, parts, mesh, nullptr, counters);
    if (rc) return rc;
    OPPX_ARG_CHECK(cell_inst && insts && n_insts > 0, "oppx_fempic_batch_step_fused: instance tables required");
    OPPX_ARG_CHECK(n_max >= 0 && n_max <= parts->stride, "oppx_fempic_batch_step_fused: n_max beyond capacity");
    OPPX_ARG_CHECK(hole_bits != nullptr, "oppx_fempic_batch_step_fused: hole_bits required");
    if (n_max == 0) return OPPX_OK;
    P.n_max = n_max;
    P.hole_bits = hole_bits;
    P.hops = hops;
    P.charge = node_charge;
    P.cell_inst = cell_inst;
    P.insts = insts;
    P.n_insts = n_insts;
    hipStream_t s = as_stream(stream);
    const bool two = node_charge ? launch_two_pass<true, true, true, true>(P, n_max, work, work_bytes, s)
                                 : launch_two_pass<true, true, false, true>(P, n_max, work, work_bytes, s);
    if (!two) {
        attach_slots(P, work, work_bytes, s);
        if (node_charge) launch_tile<true, true, true, false, true>(P, n_max, s);
        else launch_tile<true, true, false, false, true>(P, n_max, s);
        fold_slots(P, s);
    }
    OPPX_LAUNCH_CHECK("fempic_batch_step_fused");
    return OPPX_OK;
}

size_t oppx_fempic_work_bytes(int64_t n_max) { return n_max < 0 ? 0 : work_need(n_max); }

int oppx_set_tuning(const oppx_tuning* t) {
    OPPX_ARG_CHECK(t != nullptr, "oppx_set_tuning: null");
    OPPX_ARG_CHECK(t->tile >= kWave && t->tile <= kMaxTile && t->tile % kWave == 0,
                   "oppx_set_tuning: tile must be a multiple of 64 in [64, 512]");
    OPPX_ARG_CHECK(t->refill_min >= 1 && t->refill_min <= kWave, "oppx_set_tuning: refill_min in [1, 64]");
    OPPX_ARG_CHECK((t->split == 0 || t->split == 1) && (t->persistent == 0 || t->persistent == 1),
                   "oppx_set_tuning: split and persistent are 0 or 1");
    OPPX_ARG_CHECK(t->sort_items == 4 || t->sort_items == 8 || t->sort_items == 16 || t->sort_items == 32,
                   "oppx_set_tuning: sort_items must be 4, 8, 16 or 32");
    OPPX_ARG_CHECK(t->inline_hops >= 0 && t->inline_hops <= 64, "oppx_set_tuning: inline_hops in [0, 64]");
    OPPX_ARG_CHECK(t->first_block == kBlock || t->first_block == kMaxBlock, "oppx_set_tuning: first_block 256 or 1024");
    OPPX_ARG_CHECK(t->lanes == 1 || t->lanes == 4, "oppx_set_tuning: lanes (per particle in the first pass) 1 or 4");
    g_tuning = *t;
    return OPPX_OK;
}

int oppx_get_tuning(oppx_tuning* t) {
    OPPX_ARG_CHECK(t != nullptr, "oppx_get_tuning: null");
    *t = g_tuning;
    return OPPX_OK;
}

int oppx_fempic_step_begin(oppx_move_counters* counters, double* node_charge, int64_t n_nodes, void* stream) {
    OPPX_ARG_CHECK(counters != nullptr && n_nodes >= 0, "oppx_fempic_step_begin: bad arguments");
    int64_t g = node_charge ? grid_for(n_nodes, 256) : 1;
    if (g < 1) g = 1;
    if (g > 2048) g = 2048;
    step_begin_kernel<<<(unsigned)g, 256, 0, as_stream(stream)>>>(counters, node_charge, n_nodes);
    OPPX_LAUNCH_CHECK("step_begin");
    return OPPX_OK;
}

}  // extern "C"
