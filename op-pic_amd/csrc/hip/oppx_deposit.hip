// OPP_INC charge deposit in FP32 with compensated (Kahan) sums over cell-sorted particles.
//
// Reference semantics: deposit_charge_on_nodes (apps/app_fempic/kernels.h:164-175) through the
// double-indirect c2n[p2c] map; the reference's segmented-reduction variant sorts (node, value)
// pairs and reduces by key (apps_codegen/app_fempic_cg/hip/deposit_charge_on_nodes_kernel_loop.hpp:98-158,
// opp_lib/include/device_kernels/hip_inline_kernels.h:396-535). Here particles are already ordered
// by cell (oppx_sort_by_cell), so:
//   pass 1: tile by tile of the particle set, p2c and lc (FP32) are read once, coalesced; the places where
//           p2c changes are compacted in LDS, and one lane per run of equal cells that starts in the tile
//           sums lc[0..3] of its run in index order (FP32 Kahan) from LDS -- every lane owns a run instead
//           of one lane in ~(run length) holding it. A run longer than kLongRun particles is listed and
//           summed by a whole wave instead: lane l takes particles head + l, head + l + 64, ... (Kahan),
//           and the 64 lane sums are added in lane order, so a long run no longer holds its wave for its
//           whole length. Either way the order depends only on the run itself (not on where it sits in the
//           particle set);
//   pass 2: one lane per node sums its (cell, vertex) partials in the fixed node->cell order
//           (FP32 Kahan) and stores the result.
// The order of every addition is fixed by the data, so the result does not depend on scheduling
// or on other work sharing the GPU.

#include "oppx_internal.h"

namespace oppx {
namespace {

constexpr int kB = 256;
constexpr unsigned kGridMult = 4;  // grids that stride over live work: this many times the resident blocks

struct Kahan {
    float s = 0.0f, c = 0.0f;
    __device__ __forceinline__ void add(float x) {
        const float y = x - c;
        const float t = s + y;
        c = (t - s) - y;
        s = t;
    }
};

// Zeroes the cells' partials (cells without particles keep them) and the number of listed long runs.
__global__ void __launch_bounds__(kB) zero_partials(float* __restrict__ part, int64_t n, uint32_t* __restrict__ n_long) {
    if (n_long && blockIdx.x == 0 && threadIdx.x == 0) *n_long = 0u;
    for (int64_t i = (int64_t)blockIdx.x * kB + threadIdx.x; i < n; i += (int64_t)gridDim.x * kB) part[i] = 0.0f;
}

constexpr int kRunElems = 2048;  // particles per tile
constexpr int kLongRun = 64;     // runs longer than this are summed by a whole wave

__device__ __forceinline__ int64_t live_of(const oppx_move_counters* ctr, int64_t n_max) {
    const int64_t n = ctr->size;
    return n < 0 ? 0 : (n > n_max ? n_max : n);
}

// lc index of the particle at sorted position q: perm[q] with PERM (lc left in the order before the
// sort), else q. An entry outside [0, stride) gives particle 0 (never outside the dat) and counts in bad.
template <bool PERM>
__device__ __forceinline__ int perm_at(const int32_t* __restrict__ perm, int64_t q, int64_t stride, int& bad) {
    if (!PERM) return (int)q;
    const int32_t p = perm[q];
    if ((uint64_t)(int64_t)p < (uint64_t)stride) return p;
    bad++;
    return 0;
}

// One block per tile of kRunElems particles. The tile and the kLongRun particles after it are staged in LDS with
// coalesced loads: lc in FP32 (with PERM, loaded through the permutation) and the places where p2c differs from
// the entry before (one ballot word per 64 entries, compacted into a list). A run of a valid cell reaches from
// its place to the next one; one lane per run that starts in the tile sums it from LDS in index order (Kahan), and
// a run of at most kLongRun particles ends inside the window. Longer runs are listed for cell_runs_long. The sums
// are those of lane-per-run loops over lc in global memory, bit for bit. lc_f32 (nullable) receives the staged FP32
// values of every live particle in sorted order (16 B each, coalesced), from which cell_runs_long then reads instead
// of gathering through the permutation a second time. The grid strides over the live tiles, a contiguous eighth per
// XCD (the permuted lines of neighbouring tiles meet in one L2). Finding the runs in three launches beforehand
// (count, scan, compaction: two more reads of p2c) measured 20 us of a 63 us deposit of 3 M particles.
// Also checks the precondition: a valid cell right after a larger cell or after an entry that is not a
// valid cell (a removed particle) means p2c is not sorted, and two runs of one cell would overwrite each
// other's partials; every such entry is counted in ctr->faults.
constexpr int kLcThreads = 512;
constexpr int kWindow = kRunElems + kLongRun;
constexpr int kWords = kWindow / kWave;
static_assert(kWindow % kWave == 0 && kWords <= kWave, "one wave scans the words of a window");
struct LcTile {
    float v[4][kWindow];
    unsigned long long change[kWords];
    int pre[kWords + 1];
    uint16_t place[kWindow];
};

template <bool PERM>
__global__ void __launch_bounds__(kLcThreads) cell_runs(const int32_t* __restrict__ p2c, const double* __restrict__ lc,
                                                        const int32_t* __restrict__ perm, int64_t stride,
                                                        oppx_move_counters* ctr, int64_t n_max, int64_t n_cells,
                                                        uint32_t* __restrict__ n_long, int32_t* __restrict__ long_runs,
                                                        float* __restrict__ part, float4* __restrict__ lc_f32) {
    __shared__ LcTile T;
    const int64_t n = live_of(ctr, n_max);
    const int lane = threadIdx.x & (kWave - 1);
    int bad = 0, bad_over = 0;  // bad permutation entries of the tile's own particles / of the overlap
    int unsorted = 0;
    const XcdTiles X((n + kRunElems - 1) / kRunElems);
    for (int64_t t = X.first; t < X.end; t += X.step) {
        const int64_t base = t * kRunElems;
        for (int e = threadIdx.x; e < kWindow; e += kLcThreads) {  // whole waves: kWindow is a multiple of 64
            const int64_t q = base + e;
            float v0 = 0.0f, v1 = 0.0f, v2 = 0.0f, v3 = 0.0f;
            bool change = q == n;  // the live particles end here
            if (q < n) {
                const int64_t p = PERM ? (int64_t)perm_at<PERM>(perm, q, stride, e < kRunElems ? bad : bad_over) : q;
                const int32_t c = p2c[q], prev = q > 0 ? p2c[q - 1] : -1;
                v0 = (float)lc[p];
                v1 = (float)lc[stride + p];
                v2 = (float)lc[2 * stride + p];
                v3 = (float)lc[3 * stride + p];
                change = q == 0 || c != prev;
                if (change && e < kRunElems && q > 0 && (unsigned)c < (unsigned)n_cells &&
                    (!((unsigned)prev < (unsigned)n_cells) || prev > c))
                    unsorted++;
            }
            T.v[0][e] = v0;
            T.v[1][e] = v1;
            T.v[2][e] = v2;
            T.v[3][e] = v3;
            const unsigned long long m = __ballot(change);
            if (lane == 0) T.change[e / kWave] = m;
            if (lc_f32 && e < kRunElems && q < n) lc_f32[q] = make_float4(v0, v1, v2, v3);  // sorted FP32 copy
        }
        __syncthreads();
        if (threadIdx.x < kWave) {  // changes before every word
            const int c = lane < kWords ? (int)__popcll(T.change[lane]) : 0;
            int inc = c;
#pragma unroll
            for (int d = 1; d < kWave; d <<= 1) {
                const int x = __shfl_up(inc, d);
                if (lane >= d) inc += x;
            }
            if (lane < kWords) T.pre[lane] = inc - c;
            if (lane == kWave - 1) T.pre[kWords] = inc;
        }
        __syncthreads();
        for (int e = threadIdx.x; e < kWindow; e += kLcThreads) {
            const unsigned long long m = T.change[e / kWave];
            if ((m >> lane) & 1ull) T.place[T.pre[e / kWave] + __popcll(m & ((1ull << lane) - 1ull))] = (uint16_t)e;
        }
        __syncthreads();
        const int places = T.pre[kWords];
        for (int r = threadIdx.x; r < places; r += kLcThreads) {
            const int j = T.place[r];
            if (j >= kRunElems || base + j >= n) continue;  // the next tile's run, or the end of the live particles
            const int32_t c = p2c[base + j];
            if (!((unsigned)c < (unsigned)n_cells)) continue;
            const int e = r + 1 < places ? T.place[r + 1] : 2 * kWindow;
            if (e - j > kLongRun) {  // summed by cell_runs_long
                long_runs[atomicAdd(n_long, 1u)] = (int32_t)(base + j);
                continue;
            }
            Kahan k0, k1, k2, k3;
            for (int q = j; q < e; q++) {
                k0.add(T.v[0][q]);
                k1.add(T.v[1][q]);
                k2.add(T.v[2][q]);
                k3.add(T.v[3][q]);
            }
            float4 v;
            v.x = k0.s; v.y = k1.s; v.z = k2.s; v.w = k3.s;
            *reinterpret_cast<float4*>(part + 4 * (int64_t)c) = v;
        }
        __syncthreads();  // every lane is done with the tile before the next one is staged
    }
    if (PERM && bad) atomicAdd(&ctr->faults, bad);
    unsorted = wave_sum_i32(unsorted);
    if (lane == 0 && unsorted) atomicAdd(&ctr->faults, unsorted);
}

// One wave per long run (waves stride over the list): lane l sums particles head + l + 64 t in index
// order (Kahan) while they hold the run's cell, four of them loaded at a time, then lane 0 adds the 64 lane
// sums in lane order (Kahan).
template <bool PERM, bool F32>
__global__ void __launch_bounds__(kB) cell_runs_long(const int32_t* __restrict__ p2c, const double* __restrict__ lc,
                                                     const int32_t* __restrict__ perm, const float4* __restrict__ lc_f32,
                                                     int64_t stride, const oppx_move_counters* ctr, int64_t n_max,
                                                     const uint32_t* __restrict__ n_long,
                                                     const int32_t* __restrict__ long_runs, float* __restrict__ part) {
    const int lane = threadIdx.x & (kWave - 1);
    const int64_t wave = ((int64_t)blockIdx.x * kB + threadIdx.x) / kWave;
    const int64_t n_waves = (int64_t)gridDim.x * (kB / kWave);
    const int64_t nl = (int64_t)*n_long;
    const int64_t n = live_of(ctr, n_max);
    int bad = 0;  // counted by cell_runs
    for (int64_t k = wave; k < nl; k += n_waves) {
        const int64_t j = long_runs[k];
        const int32_t c = p2c[j];
        Kahan ks[4];
        bool on = true;
        for (int64_t q = j + lane; on; q += 4 * kWave) {
            bool ok[4];
            float v[4][4];
#pragma unroll
            for (int u = 0; u < 4; u++) {
                const int64_t i = q + u * kWave;
                ok[u] = i < n && p2c[i] == c;
                if (!ok[u]) continue;
                if constexpr (F32) {  // the sorted FP32 copy: the same values, read in the same order
                    const float4 f = lc_f32[i];
                    v[u][0] = f.x; v[u][1] = f.y; v[u][2] = f.z; v[u][3] = f.w;
                } else {
                    const int64_t p = PERM ? (int64_t)perm_at<PERM>(perm, i, stride, bad) : i;
#pragma unroll
                    for (int d = 0; d < 4; d++) v[u][d] = (float)lc[d * stride + p];
                }
            }
#pragma unroll
            for (int u = 0; u < 4; u++) {
                on = on && ok[u];  // the run is contiguous: the first other cell ends it
                if (on)
#pragma unroll
                    for (int d = 0; d < 4; d++) ks[d].add(v[u][d]);
            }
        }
        Kahan t0, t1, t2, t3;
        for (int l = 0; l < kWave; l++) {  // the same on every lane: lane l's sums, in lane order
            t0.add(__shfl(ks[0].s, l));
            t1.add(__shfl(ks[1].s, l));
            t2.add(__shfl(ks[2].s, l));
            t3.add(__shfl(ks[3].s, l));
        }
        if (lane == 0) {
            float4 v;
            v.x = t0.s; v.y = t1.s; v.z = t2.s; v.w = t3.s;
            *reinterpret_cast<float4*>(part + 4 * (int64_t)c) = v;
        }
    }
}

// Scratch: the number of long runs, then their first particles (each holds more than kLongRun of the particles).
size_t run_scratch_need(int64_t n_max) { return 256 + (size_t)((n_max > 0 ? n_max : 0) / kLongRun + 1) * sizeof(int32_t); }

__global__ void __launch_bounds__(kB) node_gather(const int32_t* __restrict__ node_start,
                                                  const int32_t* __restrict__ node_end,
                                                  const int32_t* __restrict__ node_ref, int64_t n_nodes,
                                                  const float* __restrict__ part, double* __restrict__ charge,
                                                  float* __restrict__ charge_f32) {
    const int64_t v = (int64_t)blockIdx.x * kB + threadIdx.x;
    if (v >= n_nodes) return;
    Kahan k;
    const int32_t e1 = node_end ? node_end[v] : node_start[v + 1];
    int32_t e = node_start[v];
    for (; e + 4 <= e1; e += 4) {  // four loads in flight, then the four adds in order
        const int32_t r0 = node_ref[e], r1 = node_ref[e + 1], r2 = node_ref[e + 2], r3 = node_ref[e + 3];
        const float p0 = part[r0], p1 = part[r1], p2 = part[r2], p3 = part[r3];
        k.add(p0);
        k.add(p1);
        k.add(p2);
        k.add(p3);
    }
    for (; e < e1; e++) k.add(part[node_ref[e]]);
    if (charge) charge[v] = (double)k.s;
    if (charge_f32) charge_f32[v] = k.s;
}

// The deposit over cell-sorted p2c, with lc in the same order (perm null) or in the order before the sort
// (perm[q]: the source index of sorted slot q).
int deposit_f32(const char* name, int64_t n_max, int64_t stride, oppx_move_counters* counters, const int32_t* p2c,
                const double* lc, const int32_t* perm, float* lc_f32, int64_t n_cells, const int32_t* node_start,
                const int32_t* node_end, const int32_t* node_ref, int64_t n_nodes, float* cell_partials,
                double* node_charge, float* node_charge_f32, void* scratch, size_t scratch_bytes, void* stream) {
    const std::string fn(name);
    OPPX_ARG_CHECK(counters && p2c && lc && node_start && node_ref && cell_partials && scratch,
                   fn + ": null pointer");
    OPPX_ARG_CHECK(node_charge || node_charge_f32, fn + ": no output");
    OPPX_ARG_CHECK(n_max >= 0 && stride >= n_max && n_cells > 0 && n_cells < kMaxCell && n_nodes > 0,
                   fn + ": bad sizes");
    OPPX_ARG_CHECK(n_max < (int64_t)0x7FFFFFFF, fn + ": n_max beyond 32-bit indices");
    OPPX_ARG_CHECK(scratch_bytes >= run_scratch_need(n_max), fn + ": scratch too small");
    hipStream_t s = as_stream(stream);
    const int64_t np = 4 * n_cells;
    int64_t gz = grid_for(np, kB);
    if (gz > 4096) gz = 4096;
    uint32_t* n_long = reinterpret_cast<uint32_t*>(scratch);
    int32_t* long_runs = reinterpret_cast<int32_t*>(reinterpret_cast<char*>(scratch) + 256);
    zero_partials<<<(unsigned)gz, kB, 0, s>>>(cell_partials, np, n_long);
    OPPX_LAUNCH_CHECK("zero_partials");
    if (n_max > 0) {
        const int64_t nb = (n_max + kRunElems - 1) / kRunElems;
        int64_t gl = grid_for(n_max, kLongRun * (kB / kWave));  // at most one long run per kLongRun particles
        if (gl > 2048) gl = 2048;
        float4* f32 = reinterpret_cast<float4*>(lc_f32);
        if (perm) {
            auto kern = cell_runs<true>;
            kern<<<xcd_grid(stride_grid(reinterpret_cast<const void*>(kern), kLcThreads, nb, kGridMult)), kLcThreads, 0,
                   s>>>(p2c, lc, perm, stride, counters, n_max, n_cells, n_long, long_runs, cell_partials, f32);
            auto lng = f32 ? cell_runs_long<true, true> : cell_runs_long<true, false>;
            lng<<<(unsigned)gl, kB, 0, s>>>(p2c, lc, perm, f32, stride, counters, n_max, n_long, long_runs, cell_partials);
        } else {
            auto kern = cell_runs<false>;
            kern<<<xcd_grid(stride_grid(reinterpret_cast<const void*>(kern), kLcThreads, nb, kGridMult)), kLcThreads, 0,
                   s>>>(p2c, lc, nullptr, stride, counters, n_max, n_cells, n_long, long_runs, cell_partials, nullptr);
            cell_runs_long<false, false><<<(unsigned)gl, kB, 0, s>>>(p2c, lc, nullptr, nullptr, stride, counters, n_max,
                                                                      n_long, long_runs, cell_partials);
        }
        OPPX_LAUNCH_CHECK("cell_runs");
    }
    node_gather<<<grid_for(n_nodes, kB), kB, 0, s>>>(node_start, node_end, node_ref, n_nodes, cell_partials,
                                                     node_charge, node_charge_f32);
    OPPX_LAUNCH_CHECK("node_gather");
    return OPPX_OK;
}

}  // namespace
}  // namespace oppx

using namespace oppx;

extern "C" {

size_t oppx_fempic_deposit_scratch_bytes(int64_t n_max) { return n_max < 0 ? 0 : run_scratch_need(n_max); }

int oppx_fempic_deposit_sorted_f32(int64_t n_max, int64_t stride, oppx_move_counters* counters, const int32_t* p2c,
                                   const double* lc, int64_t n_cells, const int32_t* node_start, const int32_t* node_end,
                                   const int32_t* node_ref, int64_t n_nodes, float* cell_partials, double* node_charge,
                                   float* node_charge_f32, void* scratch, size_t scratch_bytes, void* stream) {
    return deposit_f32("oppx_fempic_deposit_sorted_f32", n_max, stride, counters, p2c, lc, nullptr, nullptr, n_cells,
                       node_start, node_end, node_ref, n_nodes, cell_partials, node_charge, node_charge_f32, scratch,
                       scratch_bytes, stream);
}

int oppx_fempic_deposit_sorted_f32_perm(int64_t n_max, int64_t stride, oppx_move_counters* counters,
                                        const int32_t* p2c, const double* lc, const int32_t* perm, float* lc_f32,
                                        int64_t n_cells, const int32_t* node_start, const int32_t* node_end,
                                        const int32_t* node_ref, int64_t n_nodes, float* cell_partials,
                                        double* node_charge, float* node_charge_f32, void* scratch,
                                        size_t scratch_bytes, void* stream) {
    if (!perm) {
        set_error("oppx_fempic_deposit_sorted_f32_perm: null perm");
        return OPPX_ERR_ARG;
    }
    if (lc_f32 && (reinterpret_cast<uintptr_t>(lc_f32) & 15)) {
        set_error("oppx_fempic_deposit_sorted_f32_perm: lc_f32 not 16-byte aligned");
        return OPPX_ERR_ARG;
    }
    return deposit_f32("oppx_fempic_deposit_sorted_f32_perm", n_max, stride, counters, p2c, lc, perm, lc_f32, n_cells,
                       node_start, node_end, node_ref, n_nodes, cell_partials, node_charge, node_charge_f32, scratch,
                       scratch_bytes, stream);
}

}  // extern "C"
