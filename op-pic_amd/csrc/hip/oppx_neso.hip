// NESO-advection hot path on gfx950: periodic drift + axis-wise multi-hop walk over a 2-D quad
// mesh, one lane per particle.
//
// Elemental math: apps/app_neso_advection/kernels.h:41-113; loops:
// apps_codegen/app_neso_advection_mdir_cg/{seq,hip}/{update_pos,move}_kernel_loop.hpp. The reference's
// GCC build contracts pos += vel*dt, pos + n*extent and FMOD's a - b*trunc(a/b) into FMAs; they
// are explicit fma() here (file built with -ffp-contract=off). OPP_DO_ONCE holds on the first
// hop only.

#include "oppx_internal.h"

namespace oppx {
namespace {

// Threads per block at most. Every block adds to the one counters record at its end, and adds to one address from several
// XCDs take some 10-20 ns each, one after the other: 2,048 blocks of 256 threads spent 20-40 us on that. Blocks of
// 1024 make it 512: 1.5 M particles on the grid 61 -> 31 us, gathered 89 -> 64 us, 0.1 M gathered 18 -> 12.5 us.
constexpr int kBlock = 1024;
constexpr int kVerifyBlock = 256;

struct NesoArgs {
    int64_t n_cells;
    const oppx_quad_cell* __restrict__ cells;
    int64_t stride;
    double* __restrict__ pos;
    const double* __restrict__ vel;
    int32_t* __restrict__ mdir;
    int32_t* __restrict__ p2c;
    double dt, cw, ext_x, ext_y;
    int64_t n_max;
    oppx_move_counters* ctr;
    int32_t* __restrict__ hops;
    int gnx, gny;  // grid mode: the mesh is the nx x ny periodic grid, its records computed in registers
    double inv_gnx;
};

// Record of quad (ix, iy) of the periodic grid, as apps/app_neso_advection/advec_misc.h:115-143 builds
// it: lower-left corner (x * cell_width, y * cell_width), neighbours wrapped on both axes.
__device__ __forceinline__ int grid_wrap(int v, int n) { return v < 0 ? v + n : (v >= n ? v - n : v); }

__device__ __forceinline__ double periodic_update(double p, double v, double dt, double ext) {
    p = fma(v, dt, p);
    const int off = (int)(fabs(p) + 2.0);
    const double t = fma((double)off, ext, p);
    return fma(-ext, trunc(t / ext), t);
}

// The halves of a quad record as one load each; records are 8-byte aligned, no more.
typedef double QuadHalf __attribute__((ext_vector_type(2), aligned(8)));
typedef int QuadNb __attribute__((ext_vector_type(4), aligned(8)));

// Particle state as one grid-stride iteration loads it.
struct NesoPart {
    double x, y, vx, vy;
    int cell;
};

// (The first evaluation sets the directions: the ones the particle comes with are not read.)
__device__ __forceinline__ NesoPart neso_load(const NesoArgs& P, int flags, int64_t i) {
    const int64_t S = P.stride;
    NesoPart q;
    q.x = __builtin_nontemporal_load(P.pos + i);
    q.y = __builtin_nontemporal_load(P.pos + S + i);
    q.vx = q.vy = 0.0;
    if (flags & OPPX_NESO_UPDATE) {
        q.vx = __builtin_nontemporal_load(P.vel + i);
        q.vy = __builtin_nontemporal_load(P.vel + S + i);
    }
    q.cell = (flags & OPPX_NESO_MOVE) ? __builtin_nontemporal_load(P.p2c + i) : kMaxCell;
    return q;
}

// A particle between the evaluations of its walk.
struct NesoWalk {
    double x, y;
    int cell, mx, my, ix, iy, h;
    bool on, fault;
};

// update_pos_kernel for particle i, and where its walk begins (on: it has one).
template <bool GRID>
__device__ __forceinline__ NesoWalk neso_begin(const NesoArgs& P, int flags, int64_t i, const NesoPart& q) {
    NesoWalk w{q.x, q.y, q.cell, 0, 0, 0, 0, 0, false, false};
    if (flags & OPPX_NESO_UPDATE) {
        w.x = periodic_update(w.x, q.vx, P.dt, P.ext_x);
        w.y = periodic_update(w.y, q.vy, P.dt, P.ext_y);
        __builtin_nontemporal_store(w.x, P.pos + i);
        __builtin_nontemporal_store(w.y, P.pos + P.stride + i);
    }
    if (w.cell == kMaxCell) return w;
    w.fault = !((unsigned)w.cell < (unsigned)P.n_cells);
    w.on = !w.fault;
    if (GRID && w.on) {
        // cell = ix + nx * iy: the quotient from one FP64 product, then corrected by one step
        // (the product's error stays below one for cells under 2^31)
        w.iy = (int)((double)w.cell * P.inv_gnx);
        w.ix = w.cell - w.iy * P.gnx;
        if (w.ix < 0) { w.iy--; w.ix += P.gnx; }
        else if (w.ix >= P.gnx) { w.iy++; w.ix -= P.gnx; }
    }
    return w;
}

// One evaluation of move_kernel with the cell's corner (llx, lly) and neighbours nb (not read with GRID).
template <bool GRID>
__device__ __forceinline__ void neso_eval(const NesoArgs& P, NesoWalk& w, double llx, double lly, int4 nb) {
    const double cw = P.cw;
    const double dx = w.x - llx, dy = w.y - lly;
    w.h++;
    if (w.h == 1) {
        const bool xp = ((dx > cw) && (P.ext_x > 2 * dx - cw)) || ((dx < 0) && (P.ext_x < cw - 2 * dx));
        const bool yp = ((dy > cw) && (P.ext_y > 2 * dy - cw)) || ((dy < 0) && (P.ext_y < cw - 2 * dy));
        w.mx = xp ? 1 : -1;
        w.my = yp ? 1 : -1;
    }
    int next = 0;
    bool hop = false;
    if ((dx >= 0.0) && (dx <= cw)) w.mx = 0;
    else if (w.mx > 0) { next = nb.y; hop = true; if (GRID) w.ix = grid_wrap(w.ix + 1, P.gnx); }
    else if (w.mx < 0) { next = nb.x; hop = true; if (GRID) w.ix = grid_wrap(w.ix - 1, P.gnx); }
    if (!hop) {
        if ((dy >= 0.0) && (dy <= cw)) w.my = 0;
        else if (w.my > 0) { next = nb.w; hop = true; if (GRID) w.iy = grid_wrap(w.iy + 1, P.gny); }
        else if (w.my < 0) { next = nb.z; hop = true; if (GRID) w.iy = grid_wrap(w.iy - 1, P.gny); }
    }
    if (!hop) {  // MOVE_DONE
        w.on = false;
        return;
    }
    if (GRID) next = w.ix + P.gnx * w.iy;
    if (!((unsigned)next < (unsigned)P.n_cells) || w.h >= OPPX_MAX_HOPS) {
        w.fault = true;
        w.on = false;
        return;
    }
    w.cell = next;
}

__device__ __forceinline__ void neso_end(const NesoArgs& P, int64_t i, const NesoWalk& w) {
    if (w.h == 0) return;  // no walk: removed, or a cell out of range
    __builtin_nontemporal_store(w.mx, P.mdir + i);
    __builtin_nontemporal_store(w.my, P.mdir + P.stride + i);
    if (!w.fault) __builtin_nontemporal_store(w.cell, P.p2c + i);
}

// Resident grid, grid-stride over the particles, PER particles per lane per iteration, all loaded before any is
// walked, so each lane keeps that many particles' loads in flight. Two where the walk computes its records in blocks of 1024 (50
// VGPRs, two blocks per CU; four take 76 and one block: 32 M particles 549 and 685 us), one where it gathers them:
// there the waves in flight are what hides a walk's chain of dependent reads (16 M particles on 1024 x 1024 cells
// 1,021 us; two walks a lane advancing together 1,149, four 1,379).
template <bool GRID, int BT>
__global__ void __launch_bounds__(BT) neso_step_kernel(NesoArgs P, int flags) {
    constexpr int PER = GRID && BT == kBlock ? 2 : 1;
    int64_t n = P.ctr->size;
    n = n < 0 ? 0 : (n > P.n_max ? P.n_max : n);
    long long hsum = 0;
    int hmax = 0, nfault = 0;
    const int64_t stride = (int64_t)gridDim.x * BT;
    for (int64_t i0 = (int64_t)blockIdx.x * BT + threadIdx.x; i0 < n; i0 += PER * stride) {
        NesoPart part[PER];
#pragma unroll
        for (int u = 0; u < PER; u++) {
            const int64_t i = i0 + u * stride;
            part[u] = i < n ? neso_load(P, flags, i) : NesoPart{};
        }
#pragma unroll
        for (int u = 0; u < PER; u++) {
            const int64_t i = i0 + u * stride;
            if (i >= n) continue;
            NesoWalk w = neso_begin<GRID>(P, flags, i, part[u]);
            while (w.on) {
                if (GRID) {
                    neso_eval<true>(P, w, (double)w.ix * P.cw, (double)w.iy * P.cw, int4{});
                } else {
                    const QuadHalf ll = *reinterpret_cast<const QuadHalf*>(P.cells + w.cell);
                    const QuadNb n4 = *reinterpret_cast<const QuadNb*>(P.cells[w.cell].c2c);
                    int4 nb = make_int4(n4.x, n4.y, n4.z, n4.w);
                    // both halves of the record at once: left to itself the compiler reads the one neighbour it
                    // needs after the corner has arrived, a second trip in the chain (64 -> 76 us above)
                    asm volatile("" : "+v"(nb.x), "+v"(nb.y), "+v"(nb.z), "+v"(nb.w));
                    neso_eval<false>(P, w, ll.x, ll.y, nb);
                }
            }
            neso_end(P, i, w);
            if (P.hops && (flags & OPPX_NESO_MOVE)) P.hops[i] = w.h;
            hsum += w.h;
            hmax = hmax > w.h ? hmax : w.h;
            nfault += w.fault ? 1 : 0;
        }
    }
    __shared__ long long s_sum[BT / kWave];
    __shared__ int s_max[BT / kWave], s_flt[BT / kWave];
    const int lane = threadIdx.x & (kWave - 1), w = threadIdx.x / kWave;
    const long long hs = wave_sum_i64(hsum);
    const int hm = wave_max_i32(hmax), nf = wave_sum_i32(nfault);
    if (lane == 0) { s_sum[w] = hs; s_max[w] = hm; s_flt[w] = nf; }
    __syncthreads();
    if (threadIdx.x == 0) {
        long long t = 0;
        int m = 0, f = 0;
        for (int q = 0; q < BT / kWave; q++) { t += s_sum[q]; m = m > s_max[q] ? m : s_max[q]; f += s_flt[q]; }
        if (t) atomicAdd((unsigned long long*)&P.ctr->total_hops, (unsigned long long)t);
        if (m) atomicMax(&P.ctr->max_hops, m);
        if (f) atomicAdd(&P.ctr->faults, f);
    }
}

// Counts the records that differ, bit for bit, from the nx x ny periodic grid's.
__global__ void quad_grid_check_kernel(const oppx_quad_cell* __restrict__ cells, int64_t n, int nx, int ny, double cw,
                                       int32_t* __restrict__ mismatches) {
    const int64_t c = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    bool bad = false;
    if (c < n) {
        const int ix = (int)(c % nx), iy = (int)(c / nx);
        const oppx_quad_cell q = cells[c];
        bad = __double_as_longlong(q.llx) != __double_as_longlong((double)ix * cw) ||
              __double_as_longlong(q.lly) != __double_as_longlong((double)iy * cw) ||
              q.c2c[0] != grid_wrap(ix - 1, nx) + nx * iy || q.c2c[1] != grid_wrap(ix + 1, nx) + nx * iy ||
              q.c2c[2] != ix + nx * grid_wrap(iy - 1, ny) || q.c2c[3] != ix + nx * grid_wrap(iy + 1, ny);
    }
    const unsigned long long m = __ballot(bad);
    if ((threadIdx.x & (kWave - 1)) == 0 && m) atomicAdd(mismatches, (int)__popcll(m));
}

__global__ void neso_reset_kernel(oppx_move_counters* ctr) {
    ctr->removed = 0;
    ctr->holes_low = 0;
    ctr->max_hops = 0;
    ctr->total_hops = 0;
}

__global__ void quad_cells_kernel(const double* __restrict__ ll, const int32_t* __restrict__ c2c, int64_t n,
                                  oppx_quad_cell* __restrict__ out) {
    const int64_t c = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (c >= n) return;
    oppx_quad_cell q;
    q.llx = ll[2 * c];
    q.lly = ll[2 * c + 1];
    for (int k = 0; k < 4; k++) {
        const int v = c2c[4 * c + k];
        q.c2c[k] = (v >= 0 && v < n) ? v : -2;  // invalid neighbours are rejected by the walk as faults
    }
    out[c] = q;
}

__global__ void zero_i32_kernel(int32_t* p) { *p = 0; }

int neso_step_impl(int64_t n_max, const oppx_neso_parts* parts, const oppx_quad_cell* cells, int64_t n_cells,
                   int gnx, int gny, double dt, double cell_width, double ext_x, double ext_y, int flags,
                   oppx_move_counters* counters, int32_t* hops, void* stream) {
    const bool grid = gnx > 0;
    OPPX_ARG_CHECK(parts && counters, "oppx_neso_step: null pointer");
    OPPX_ARG_CHECK(flags >= 1 && flags <= 3, "oppx_neso_step: flags must be OPPX_NESO_UPDATE and/or OPPX_NESO_MOVE");
    OPPX_ARG_CHECK(!(flags & OPPX_NESO_MOVE) || ((cells || grid) && parts->mdir && parts->p2c),
                   "oppx_neso_step: move needs cells, mdir, p2c");
    OPPX_ARG_CHECK(!(flags & OPPX_NESO_UPDATE) || (parts->pos && parts->vel), "oppx_neso_step: update needs pos, vel");
    OPPX_ARG_CHECK(n_cells > 0 && n_cells < kMaxCell, "oppx_neso_step: n_cells out of range");
    OPPX_ARG_CHECK(n_max >= 0 && n_max <= parts->stride, "oppx_neso_step: n_max beyond capacity");
    OPPX_ARG_CHECK(cell_width > 0 && ext_x > 0 && ext_y > 0, "oppx_neso_step: widths must be positive");
    hipStream_t s = as_stream(stream);
    neso_reset_kernel<<<1, 1, 0, s>>>(counters);
    OPPX_LAUNCH_CHECK("neso_reset");
    if (n_max == 0) return OPPX_OK;
    NesoArgs P{};
    P.n_cells = n_cells;
    P.cells = cells;
    P.stride = parts->stride;
    P.pos = parts->pos;
    P.vel = parts->vel;
    P.mdir = parts->mdir;
    P.p2c = parts->p2c;
    P.dt = dt;
    P.cw = cell_width;
    P.ext_x = ext_x;
    P.ext_y = ext_y;
    P.n_max = n_max;
    P.ctr = counters;
    P.hops = hops;
    P.gnx = gnx;
    P.gny = gny;
    P.inv_gnx = grid ? 1.0 / gnx : 0.0;
    // Smaller sets take smaller blocks, for a block of 1024 with one or two particles a thread leaves the CUs beside it idle.
    // A step, us, blocks of 256 / 512 / 1024, records computed, then gathered from 490,000 cells at 4 cells a step: 1,000
    // particles 8.3 8.5 9.8, 10.0 10.6 13.5; 10,000 8.3 8.7 10.2, 10.2 10.9 14.6; 23,000 9.7 9.2 10.6, 11.4 11.2 15.0; 50,000
    // 12.1 10.3 11.0, 13.8 12.2 15.2; 100,000 17.1 12.7 12.2, 19.0 15.1 16.4. From 6 M particles on the grid is twice the
    // resident blocks, four times where records are gathered, so that the last wave is a smaller share: 8.2 M in half-cell
    // steps, resident / so 109 / 102, gathered 171 / 163, 32 M 391 / 374, 616 / 605; but 3 M 43 / 47, 67 / 74.
    const int bt = n_max < 16'384 ? 256 : (n_max < 65'536 ? 512 : kBlock);
    auto kern = bt == 256 ? (grid ? neso_step_kernel<true, 256> : neso_step_kernel<false, 256>)
                          : bt == 512 ? (grid ? neso_step_kernel<true, 512> : neso_step_kernel<false, 512>)
                                      : (grid ? neso_step_kernel<true, kBlock> : neso_step_kernel<false, kBlock>);
    unsigned g = resident_blocks(reinterpret_cast<const void*>(kern), bt);
    if (n_max >= 6'000'000) g *= grid ? 2 : 4;
    const unsigned need = grid_for(n_max, bt);
    if (g > need) g = need;
    kern<<<g, bt, 0, s>>>(P, flags);
    OPPX_LAUNCH_CHECK("neso_step");
    return OPPX_OK;
}
// verify_kernel (apps/app_neso_advection/kernels.h:115-150) over the counters->size particles: a
// particle counts as incorrect when its cell's global index c_gbl_idx[p2c] splits into a negative
// (ix, iy) = (g mod nx, g div nx), or when a coordinate lies outside [ll, ll + cell_width] with
// ll = ix * cell_width (a product then a sum: the reference build forms them apart, no FMA). Block
// sums of the count are added to *count.
__global__ void __launch_bounds__(kVerifyBlock) neso_verify_kernel(int64_t n_max, int64_t stride, const double* __restrict__ pos,
                                                             const int32_t* __restrict__ p2c,
                                                             const int32_t* __restrict__ c_gbl_idx, int64_t n_cells,
                                                             int nx, double cw, const oppx_move_counters* __restrict__ ctr,
                                                             int32_t* __restrict__ count, int32_t* __restrict__ faults) {
    int64_t n = ctr->size;
    n = n < 0 ? 0 : (n > n_max ? n_max : n);
    int bad = 0, flt = 0;
    for (int64_t i = (int64_t)blockIdx.x * kVerifyBlock + threadIdx.x; i < n; i += (int64_t)gridDim.x * kVerifyBlock) {
        const int c = p2c[i];
        if (!((unsigned)c < (unsigned)n_cells)) {  // the reference would read outside c_idx
            flt++;
            continue;
        }
        const int g = c_gbl_idx[c];
        const int iy = g / nx, ix = g - iy * nx;
        if (ix < 0 || iy < 0) {
            bad++;
            continue;
        }
        const double llx = (double)ix * cw, x = pos[i];
        if (x < llx || x > llx + cw) {
            bad++;
            continue;
        }
        const double lly = (double)iy * cw, y = pos[stride + i];
        if (y < lly || y > lly + cw) bad++;
    }
    __shared__ int s_bad[kVerifyBlock / kWave], s_flt[kVerifyBlock / kWave];
    bad = wave_sum_i32(bad);
    flt = wave_sum_i32(flt);
    const int lane = threadIdx.x & (kWave - 1), w = threadIdx.x / kWave;
    if (lane == 0) { s_bad[w] = bad; s_flt[w] = flt; }
    __syncthreads();
    if (threadIdx.x == 0) {
        int b = 0, f = 0;
        for (int q = 0; q < kVerifyBlock / kWave; q++) { b += s_bad[q]; f += s_flt[q]; }
        if (b) atomicAdd(count, b);
        if (f && faults) atomicAdd(faults, f);
    }
}

}  // namespace
}  // namespace oppx

using namespace oppx;

extern "C" {

int oppx_quad_cells_build(const double* c_pos_ll, const int32_t* c2c, int64_t n_cells, oppx_quad_cell* cells,
                          void* stream) {
    OPPX_ARG_CHECK(c_pos_ll && c2c && cells && n_cells > 0 && n_cells < kMaxCell, "oppx_quad_cells_build: bad args");
    quad_cells_kernel<<<grid_for(n_cells, 256), 256, 0, as_stream(stream)>>>(c_pos_ll, c2c, n_cells, cells);
    OPPX_LAUNCH_CHECK("quad_cells");
    return OPPX_OK;
}

int oppx_quad_grid_check(const oppx_quad_cell* cells, int64_t n_cells, int nx, int ny, double cell_width,
                         int32_t* mismatches, void* stream) {
    OPPX_ARG_CHECK(cells && mismatches && nx > 0 && ny > 0 && (int64_t)nx * ny == n_cells && n_cells < kMaxCell,
                   "oppx_quad_grid_check: bad arguments (n_cells must be nx * ny)");
    hipStream_t s = as_stream(stream);
    zero_i32_kernel<<<1, 1, 0, s>>>(mismatches);
    quad_grid_check_kernel<<<grid_for(n_cells, 256), 256, 0, s>>>(cells, n_cells, nx, ny, cell_width, mismatches);
    OPPX_LAUNCH_CHECK("quad_grid_check");
    return OPPX_OK;
}


int oppx_neso_step(int64_t n_max, const oppx_neso_parts* parts, const oppx_quad_cell* cells, int64_t n_cells,
                   double dt, double cell_width, double ext_x, double ext_y, int flags,
                   oppx_move_counters* counters, int32_t* hops, void* stream) {
    return neso_step_impl(n_max, parts, cells, n_cells, 0, 0, dt, cell_width, ext_x, ext_y, flags, counters, hops,
                          stream);
}

int oppx_neso_step_grid(int64_t n_max, const oppx_neso_parts* parts, int nx, int ny, double dt, double cell_width,
                        double ext_x, double ext_y, int flags, oppx_move_counters* counters, int32_t* hops,
                        void* stream) {
    OPPX_ARG_CHECK(nx > 0 && ny > 0 && (int64_t)nx * ny < kMaxCell, "oppx_neso_step_grid: nx, ny out of range");
    return neso_step_impl(n_max, parts, nullptr, (int64_t)nx * ny, nx, ny, dt, cell_width, ext_x, ext_y, flags,
                          counters, hops, stream);
}

int oppx_neso_verify(int64_t n_max, int64_t stride, const double* pos, const int32_t* p2c, const int32_t* c_gbl_idx,
                     int64_t n_cells, int nx, double cell_width, oppx_move_counters* counters, int32_t* count,
                     void* stream) {
    OPPX_ARG_CHECK(n_max >= 0 && stride >= n_max, "oppx_neso_verify: need 0 <= n_max <= stride");
    OPPX_ARG_CHECK(counters && count, "oppx_neso_verify: null counters or count");
    OPPX_ARG_CHECK(nx > 0 && n_cells > 0 && n_cells < kMaxCell, "oppx_neso_verify: nx or n_cells out of range");
    if (n_max == 0) return OPPX_OK;
    OPPX_ARG_CHECK(pos && p2c && c_gbl_idx, "oppx_neso_verify: null array");
    unsigned g = grid_for(n_max, kVerifyBlock);
    if (g > 4096) g = 4096;
    neso_verify_kernel<<<g, kVerifyBlock, 0, as_stream(stream)>>>(n_max, stride, pos, p2c, c_gbl_idx, n_cells, nx, cell_width,
                                                            counters, count, &counters->faults);
    OPPX_LAUNCH_CHECK("neso_verify");
    return OPPX_OK;
}

}  // extern "C"
