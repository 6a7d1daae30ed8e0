// small_step.hip — the integration, the rebuild decision and the whole sort of
// a small system's MD step in one workgroup.
//
// A step of the fused loop is twelve launches for a system in the brick layout
// (kick, thermostat, seven rebuild stages that mostly leave at once, forces,
// kick, thermostat). At a few thousand atoms each is 1.5-4.5 us of latency
// (dependent loads of the control block, then of the atoms, then a reduction)
// plus a launch gap, and together they were three quarters of the step. One
// 1024-thread workgroup holds up to kSmallMaxAtoms atoms in its registers, so here
// the second half of step k, the first half of step k + 1 and, when the list is
// stale, the counting sort, the permutation and the halo tables are one launch
// whose stages meet at workgroup barriers; the list build and the forces stay
// one workgroup per brick. A step is three launches (500 atoms, FP64: 46 -> 19
// us, 17 with the wide force kernel).
//
// Every value is the multi-block stages' value bit for bit (the batched step
// runs those, and a member equals the same system run alone): the per-atom
// arithmetic is shared (integrate.hpp), kinetic energies are summed over the
// same 256-atom groups in the same order, and the sorted order (cell rank, then
// tag) does not depend on how it is found.

#include "atvh_internal.hpp"
#include "batch.hpp"
#include "brick.hpp"
#include "integrate.hpp"
#include "pair_common.hpp"

#include <algorithm>
#include <type_traits>

using namespace atvh;

namespace {

constexpr int kHeadThreads = 1024;
constexpr int kHeadWaves = kHeadThreads / 64;
constexpr int kHeadItems = 2; // most atoms per thread
constexpr int kSmallMaxAtoms = kHeadThreads * kHeadItems;
constexpr int kMidMaxAtoms = 45000;
constexpr int kMidMaxCells = 13000;
// cells + atoms the sort's LDS tables hold (start of every cell, tag of every slot)
constexpr int kHeadLdsInts = 14000;

struct HeadArgs {
    IntArgs i;
    FinalizeArgs e;   // energy totals of the step that ends here
    int do_energy, do_final, do_initial;
    double* record_ke; // may be null
    int step;          // record index of the step that ends here
    int every, delay, check;
    // sort
    int *tag, *type;
    double* q;
    double *xs, *ys, *zs;
    int with_q, with_type;
    double csx, csy, csz;
    int ncells;
    int* start; // [ncells + 1]
    // halo tables
    BrickGeom g;
    int nbricks;
    const int* halo_cells;
    int* halo_off;
    int* halo_rows;
    int* halo_n;
    int2* brick_range;
};

// OpBin's cell of a position: wrapped, then wrapped once more as bin_atoms
// does, floor(x / cs) clamped, z-fastest reference index.
__device__ __forceinline__ int bin_cell(const IntArgs& i, const BrickGeom& g, double csx, double csy, double csz,
                                        const double (&x)[3]) {
    double w0 = x[0], w1 = x[1], w2 = x[2];
    for (int pass = 0; pass < 2; ++pass) {
        w0 -= i.lx * floor(w0 / i.lx);
        w1 -= i.ly * floor(w1 / i.ly);
        w2 -= i.lz * floor(w2 / i.lz);
    }
    int cx = static_cast<int>(floor((w0 - 0.0) / csx));
    int cy = static_cast<int>(floor((w1 - 0.0) / csy));
    int cz = static_cast<int>(floor((w2 - 0.0) / csz));
    cx = max(0, min(cx, g.nc[0] - 1));
    cy = max(0, min(cy, g.nc[1] - 1));
    cz = max(0, min(cz, g.nc[2] - 1));
    return cx * g.nc[1] * g.nc[2] + cy * g.nc[2] + cz;
}

// Cell counts in LDS to cell starts (start[ncells] = n): each thread a run of
// cells. One barrier inside; the caller separates it from what precedes and
// follows.
__device__ __forceinline__ void exclusive_scan_cells(int* start, int ncells, int n, int* s_wave, int lane, int wid) {
    const int per = (ncells + kHeadThreads - 1) / kHeadThreads;
    const int h0 = min(static_cast<int>(threadIdx.x) * per, ncells), h1 = min(h0 + per, ncells);
    int sum = 0;
    for (int h = h0; h < h1; ++h)
        sum += start[h];
    const int inc = wave_inclusive_sum(sum);
    if (lane == 63)
        s_wave[wid] = inc;
    __syncthreads();
    int run = inc - sum;
    for (int w = 0; w < wid; ++w)
        run += s_wave[w];
    for (int h = h0; h < h1; ++h) {
        const int cnt = start[h];
        start[h] = run;
        run += cnt;
    }
    if (threadIdx.x == 0)
        start[ncells] = n;
}

// Sum of m v^2 over the workgroup in the multi-block order: ws[w] holds the
// wavefront sums of 64-atom runs, four to a 256-atom group, the groups added
// as block_fixed_sums adds at most 64 rows. Valid on thread 0.
__device__ __forceinline__ double group_total(const double* ws, int nb) {
    const int t = threadIdx.x;
    double v = 0.0;
    if (t < nb) {
        double p = 0.0;
        for (int w = 0; w < kBlock / 64; ++w)
            p += ws[t * (kBlock / 64) + w];
        v += p;
    }
    for (int off = 32; off > 0; off >>= 1)
        v += __shfl_down(v, off, 64);
    return v;
}

__device__ __forceinline__ void load_positions(const HeadArgs& a, int i, double (&x)[3], double (&xs)[3]) {
    x[0] = a.i.x[i];
    x[1] = a.i.y[i];
    x[2] = a.i.z[i];
    xs[0] = a.i.xs[i];
    xs[1] = a.i.ys[i];
    xs[2] = a.i.zs[i];
}

template <int ITEMS>
__global__ __launch_bounds__(kHeadThreads) void k_small_head(HeadArgs a) {
    extern __shared__ int dyn[]; // a rebuild: cell starts [ncells + 1], then slot tags [n]
    __shared__ double ws[ITEMS * kHeadWaves];
    __shared__ double s_scale;
    __shared__ int s_moved, s_rebuild;
    __shared__ int s_wave[kHeadWaves];
    const int tid = threadIdx.x, lane = tid & 63, wid = tid >> 6;
    const int n = static_cast<int>(a.i.n);
    DevCtl* c = a.i.ctl;
    const bool typed = a.i.ntypes > 1;
    const double dtfm0 = a.i.dtfm[0], m0 = a.i.mass[0];
    const int nb = (n + kBlock - 1) / kBlock;
    // everything the step reads, issued before the first value is needed
    const int stop = c->overflow | c->halo_overflow;
    double scale = a.i.thermostat ? c->nh_scale : 1.0;
    double xi = c->xi;
    const double Q = c->nh_Q, ndof_kT = c->nh_ndof_kT;
    const int was_moved = c->disp_flag;
    KickAtom k[ITEMS];
    double x[ITEMS][3], xs[ITEMS][3];
#pragma unroll
    for (int j = 0; j < ITEMS; ++j) {
        const int i = j * kHeadThreads + tid;
        if (i < n) {
            k[j] = kick_load(a.i, i, typed);
            if (a.do_initial)
                load_positions(a, i, x[j], xs[j]);
        }
    }
    if (stop) { // halted: nothing of this step is integrated, and no rebuild is decided
        if (tid == 0 && a.do_initial)
            c->rebuild = 0;
        return;
    }
    if (a.do_energy)
        finalize_totals(a.e);
    if (tid == 0)
        s_moved = 0;
    if (a.do_final) {
#pragma unroll
        for (int j = 0; j < ITEMS; ++j) {
            double mv2 = 0.0;
            if (j * kHeadThreads + tid < n)
                mv2 += kick_apply(a.i, k[j], scale, typed, dtfm0, m0);
            mv2 = wave_sum(mv2);
            if (lane == 0)
                ws[j * kHeadWaves + wid] = mv2;
        }
        __syncthreads();
        if (wid == 0) {
            const double mv2 = group_total(ws, nb);
            if (tid == 0) {
                const double ke = 0.5 * mass_v2_to_energy * mv2;
                double s = 1.0;
                if (a.i.thermostat) {
                    s = nh_update(ke, a.i.dt, ndof_kT, Q, xi);
                    c->xi = xi;
                    c->nh_scale = s;
                }
                const double ke_end = ke * s * s; // KineticEnergy at end_of_step (scaled v)
                c->ke = ke_end;
                if (a.record_ke)
                    a.record_ke[a.step] = ke_end;
                c->steps_done += 1;
                s_scale = s;
            }
        }
        __syncthreads();
        if (a.i.thermostat)
            scale = s_scale;
    }
    if (!a.do_initial) {
#pragma unroll
        for (int j = 0; j < ITEMS; ++j) {
            const int i = j * kHeadThreads + tid;
            if (i < n) {
                a.i.vx[i] = k[j].vx;
                a.i.vy[i] = k[j].vy;
                a.i.vz[i] = k[j].vz;
            }
        }
        return;
    }
    if (!a.do_final)
        __syncthreads(); // s_moved is clear
    bool moved = false;
#pragma unroll
    for (int j = 0; j < ITEMS; ++j) {
        const int i = j * kHeadThreads + tid;
        double mv2 = 0.0;
        if (i < n) {
            mv2 += kick_apply(a.i, k[j], scale, typed, dtfm0, m0);
            x[j][0] = x[j][0] + a.i.dt * k[j].vx;
            x[j][1] = x[j][1] + a.i.dt * k[j].vy;
            x[j][2] = x[j][2] + a.i.dt * k[j].vz;
            a.i.x[i] = x[j][0];
            a.i.y[i] = x[j][1];
            a.i.z[i] = x[j][2];
            a.i.vx[i] = k[j].vx;
            a.i.vy[i] = k[j].vy;
            a.i.vz[i] = k[j].vz;
            moved = moved || moved_past_skin(a.i, x[j][0] - xs[j][0], x[j][1] - xs[j][1], x[j][2] - xs[j][2]);
        }
        mv2 = wave_sum(mv2);
        if (lane == 0)
            ws[j * kHeadWaves + wid] = mv2;
    }
    if (__any(moved) && lane == 0)
        s_moved = 1;
    __syncthreads();
    if (wid == 0) {
        const double mv2 = group_total(ws, nb);
        if (tid == 0) {
            const double ke = 0.5 * mass_v2_to_energy * mv2;
            if (a.i.thermostat) {
                c->nh_scale = nh_update(ke, a.i.dt, ndof_kT, Q, xi);
                c->xi = xi;
            }
            c->ke_half = ke;
            s_rebuild = decide_reneighbor(c, a.every, a.delay, a.check, was_moved != 0 || s_moved != 0) ? 1 : 0;
        }
    }
    __syncthreads();
    if (!s_rebuild)
        return;

    // ---- counting sort by (cell rank, tag), permutation and x_save ----
    int* start = dyn;
    int* stag = dyn + a.ncells + 1;
    for (int h = tid; h <= a.ncells; h += kHeadThreads)
        start[h] = 0;
    __syncthreads();
    int key[ITEMS], place[ITEMS], tag[ITEMS], type[ITEMS];
    double q[ITEMS];
#pragma unroll
    for (int j = 0; j < ITEMS; ++j) {
        const int i = j * kHeadThreads + tid;
        if (i < n) {
            tag[j] = a.tag[i];
            type[j] = a.with_type ? a.type[i] : 0;
            q[j] = a.with_q ? a.q[i] : 0.0;
            key[j] = a.g.cell_rank[bin_cell(a.i, a.g, a.csx, a.csy, a.csz, x[j])];
            // wrapped at the rebuild (OpBin)
            x[j][0] -= a.i.lx * floor(x[j][0] / a.i.lx);
            x[j][1] -= a.i.ly * floor(x[j][1] / a.i.ly);
            x[j][2] -= a.i.lz * floor(x[j][2] / a.i.lz);
            place[j] = atomicAdd(&start[key[j]], 1);
        }
    }
    __syncthreads();
    exclusive_scan_cells(start, a.ncells, n, s_wave, lane, wid);
    __syncthreads();
#pragma unroll
    for (int j = 0; j < ITEMS; ++j)
        if (j * kHeadThreads + tid < n)
            stag[start[key[j]] + place[j]] = tag[j];
    for (int h = tid; h <= a.ncells; h += kHeadThreads)
        a.start[h] = start[h];
    __syncthreads();
#pragma unroll
    for (int j = 0; j < ITEMS; ++j)
        if (j * kHeadThreads + tid < n) {
            const int b = start[key[j]], e = start[key[j] + 1];
            int d = b;
            for (int s = b; s < e; ++s)
                d += stag[s] < tag[j] ? 1 : 0;
            a.i.x[d] = x[j][0];
            a.i.y[d] = x[j][1];
            a.i.z[d] = x[j][2];
            a.xs[d] = x[j][0];
            a.ys[d] = x[j][1];
            a.zs[d] = x[j][2];
            a.i.vx[d] = k[j].vx;
            a.i.vy[d] = k[j].vy;
            a.i.vz[d] = k[j].vz;
            a.tag[d] = tag[j];
            if (a.with_type)
                a.type[d] = type[j];
            if (a.with_q)
                a.q[d] = q[j];
        }

    // ---- halo tables, one wavefront per brick (OpHalo's values) ----
    for (int b = wid; b < a.nbricks; b += kHeadWaves) {
        int bx, by, bz;
        brick_coords(a.g, b, bx, by, bz);
        const int o[3] = {bx * a.g.bdim[0], by * a.g.bdim[1], bz * a.g.bdim[2]};
        int ncell = 1;
        for (int d = 0; d < 3; ++d)
            ncell *= min(a.g.bdim[d], a.g.nc[d] - o[d]) + 2 * a.g.R[d];
        const int* __restrict__ tab = a.halo_cells + (int64_t)b * kHaloCellCap;
        int* __restrict__ hoff = a.halo_off + (int64_t)b * (kHaloCellCap + 1);
        int* __restrict__ rows = a.halo_rows + (int64_t)b * kHaloCap;
        int run = 0;
        for (int h0 = 0; h0 < ncell; h0 += 64) {
            const int h = h0 + lane;
            int e = 0, s0 = 0, cnt = 0;
            if (h < ncell) {
                e = tab[h];
                const int r = e & kRowSlotMask;
                s0 = start[r];
                cnt = start[r + 1] - s0;
            }
            const int inc = wave_inclusive_sum(cnt);
            const int at = run + inc - cnt;
            if (h < ncell)
                hoff[h] = at;
            const int image = static_cast<int>(static_cast<unsigned>(e) >> kRowSlotBits) << kRowSlotBits;
            for (int s = 0; s < cnt; ++s)
                if (at + s < kHaloCap) // an overfull halo is reported below and never read
                    rows[at + s] = (s0 + s) | image;
            run += __builtin_amdgcn_readlane(inc, 63);
        }
        if (lane == 0) {
            hoff[ncell] = run;
            const int a0 = start[a.g.brick_cell_base[b]];
            const int nat = start[a.g.brick_cell_base[b + 1]] - a0;
            a.halo_n[b] = run;
            a.brick_range[b] = make_int2(a0, nat);
            if (brick_skipped(run, nat, a.g.max_atoms))
                atomicAdd(&c->halo_overflow, 1);
        }
    }
}

// ---- some tens of thousand atoms ----
//
// Beyond kSmallMaxAtoms the atoms go over blocks again and a step is six
// launches instead of twelve: the final kick leaves its partial sums, and the
// next step's first kernel adds them in every block (a few hundred values)
// instead of a launch of its own; the decision and the sort's counting are one
// workgroup, which needs only the 4-byte cell keys that kernel leaves; the
// placement and the list build follow as two launches (nl_enqueue_place).
// 32,000 atoms mixed 44.0 -> 37.1 us a step, 4,000 FP64 46 -> 31 (33.5 and 26.5
// with the force kernels as they are now).

struct MidArgs {
    IntArgs i;
    int do_final;
    const double* final_partials; // m v^2 of the final kick (256-atom groups)
    int nb;
    double* record_ke; // may be null
    int step;
    BrickGeom g;
    double csx, csy, csz;
    int* key; // cell rank of every slot at its new position (MID)
};

// The NH half of the step that ends (every block finds the same kinetic total
// and scale; block 0 records), then kick, drift, displacement test and, for the
// mid path, the cell of every atom. xi and the scale are written by the next
// launch only: blocks still read them here. A thread's first atom is loaded
// ahead of the reduction.
// MID: a thread per atom, with keys (as one kernel with a loop and a test for
// the keys the mid path's launch took 0.4 us more of 5.3).
template <bool MID>
__global__ __launch_bounds__(kBlock) void k_step_initial(MidArgs a) {
    __shared__ double s_scale;
    DevCtl* c = a.i.ctl;
    const bool typed = a.i.ntypes > 1;
    using Index = std::conditional_t<MID, int, int64_t>;
    Index i = blockIdx.x * static_cast<Index>(kBlock) + threadIdx.x;
    const Index stride = static_cast<Index>(gridDim.x) * kBlock;
    const int stop = c->overflow | c->halo_overflow;
    double scale = a.i.thermostat ? c->nh_scale : 1.0;
    KickAtom k{};
    double x[3] = {0, 0, 0}, xs[3] = {0, 0, 0};
    const auto load = [&]() {
        k = kick_load(a.i, i, typed);
        x[0] = a.i.x[i];
        x[1] = a.i.y[i];
        x[2] = a.i.z[i];
        xs[0] = a.i.xs[i];
        xs[1] = a.i.ys[i];
        xs[2] = a.i.zs[i];
    };
    const bool act = i < static_cast<Index>(a.i.n);
    if (act)
        load();
    if (stop)
        return;
    if (a.do_final) {
        double sum[1];
        block_fixed_sums<1>(a.final_partials, a.nb, 1, sum);
        if (threadIdx.x == 0) {
            const double ke = 0.5 * mass_v2_to_energy * sum[0];
            double s = 1.0, xi = c->xi;
            if (a.i.thermostat)
                s = nh_update(ke, a.i.dt, c->nh_ndof_kT, c->nh_Q, xi);
            s_scale = s;
            if (blockIdx.x == 0) {
                const double ke_end = ke * s * s; // KineticEnergy at end_of_step (scaled v)
                c->xi_mid = xi;
                c->ke = ke_end;
                if (a.record_ke)
                    a.record_ke[a.step] = ke_end;
                c->steps_done += 1;
            }
        }
        __syncthreads();
        if (a.i.thermostat)
            scale = s_scale;
    } else if (blockIdx.x == 0 && threadIdx.x == 0) {
        c->xi_mid = c->xi;
    }
    double mv2 = 0.0;
    bool moved = false;
    const auto step = [&]() {
        mv2 += kick_apply(a.i, k, scale, typed, a.i.dtfm[0], a.i.mass[0]);
        x[0] = x[0] + a.i.dt * k.vx;
        x[1] = x[1] + a.i.dt * k.vy;
        x[2] = x[2] + a.i.dt * k.vz;
        a.i.x[i] = x[0];
        a.i.y[i] = x[1];
        a.i.z[i] = x[2];
        a.i.vx[i] = k.vx;
        a.i.vy[i] = k.vy;
        a.i.vz[i] = k.vz;
        moved |= moved_past_skin(a.i, x[0] - xs[0], x[1] - xs[1], x[2] - xs[2]);
        if (MID)
            a.key[i] = a.g.cell_rank[bin_cell(a.i, a.g, a.csx, a.csy, a.csz, x)];
    };
    if (act)
        step();
    if (!MID)
        for (i += stride; i < a.i.n; i += stride) {
            load();
            step();
        }
    if (__any(moved) && (threadIdx.x & 63) == 0)
        c->disp_flag = 1;
    block_sum_to(mv2, &a.i.ke_partials[blockIdx.x]);
}

struct MidSortArgs {
    StepDecision d;
    FinalizeArgs e;
    int do_energy;
    int n, ncells;
    const int* key;
    int* start; // [ncells + 1]
    int* perm;  // slots cell by cell, in no order within a cell
};

// NH and the decision, then, on a rebuild, the cell starts and the slots of
// every cell: one workgroup counts and places n keys in LDS.
__global__ __launch_bounds__(kHeadThreads) void k_mid_sort(MidSortArgs a) {
    extern __shared__ int start[]; // [ncells + 1]
    __shared__ int s_rebuild;
    __shared__ int s_wave[kHeadWaves];
    const int tid = threadIdx.x, lane = tid & 63, wid = tid >> 6;
    DevCtl* c = a.d.ctl;
    if (halted(c)) {
        if (tid == 0)
            c->rebuild = 0;
        return;
    }
    if (a.do_energy)
        finalize_totals(a.e);
    double sum[1];
    block_fixed_sums<1>(a.d.partials, a.d.nb, 1, sum);
    if (tid == 0) {
        initial_nh(a.d, sum[0]);
        s_rebuild = decide_reneighbor(c, a.d.every, a.d.delay, a.d.check, c->disp_flag != 0) ? 1 : 0;
    }
    __syncthreads();
    if (!s_rebuild)
        return;
    for (int h = tid; h <= a.ncells; h += kHeadThreads)
        start[h] = 0;
    __syncthreads();
    for (int i = tid; i < a.n; i += kHeadThreads)
        atomicAdd(&start[a.key[i]], 1);
    __syncthreads();
    exclusive_scan_cells(start, a.ncells, a.n, s_wave, lane, wid);
    __syncthreads();
    for (int h = tid; h <= a.ncells; h += kHeadThreads)
        a.start[h] = start[h];
    __syncthreads(); // the starts become cursors
    for (int i = tid; i < a.n; i += kHeadThreads)
        a.perm[atomicAdd(&start[a.key[i]], 1)] = i;
}

template <int ITEMS>
void launch_head(const HeadArgs& a, int lds, hipStream_t st) {
    k_small_head<ITEMS><<<1, kHeadThreads, lds, st>>>(a);
}

} // namespace

namespace atvh {

// The line at kSmallMaxAtoms is one CU's memory path: at 4,000 atoms (four a
// thread) this launch takes 20 us and a step 41 us, against 31 us with the
// atoms spread over blocks (mid_enqueue_first_half); at 500 atoms it takes 5
// us and a step 19 us (46 us with the multi-block stages). Cells count too: the
// sort's LDS tables hold kHeadLdsInts of them with the atoms, and a sparse box
// gains little by then (700 atoms in 12,852 cells: a step 35 us, 32-36 us with
// the atoms over blocks, 43 us beyond that form's lines).
bool small_step_fits(const atvh_system* s) {
    return s->brick_mode && s->n <= kSmallMaxAtoms && s->ncells + s->n < kHeadLdsInts;
}

void small_enqueue_head(atvh_system* s, int final_step, bool final_energy, bool initial, ThermoRec rec) {
    ScopedTimer tm(s->ctx, "integrate");
    HeadArgs a{};
    a.i = make_int_args(s);
    a.do_final = final_step >= 0 ? 1 : 0;
    a.do_energy = a.do_final && final_energy ? 1 : 0;
    a.do_initial = initial ? 1 : 0;
    if (a.do_energy)
        a.e = make_finalize_args(s, rec.pe, final_step, true);
    a.record_ke = rec.ke;
    a.step = final_step;
    a.every = s->every;
    a.delay = s->delay;
    a.check = s->check;
    a.tag = s->tag;
    a.type = s->type;
    a.q = s->q;
    a.xs = s->xs;
    a.ys = s->ys;
    a.zs = s->zs;
    a.with_q = s->has_charge ? 1 : 0;
    a.with_type = s->ntypes > 1 ? 1 : 0;
    a.csx = s->cs[0];
    a.csy = s->cs[1];
    a.csz = s->cs[2];
    a.ncells = s->ncells;
    a.start = s->cell_start;
    a.g = brick_geom(s);
    a.nbricks = s->nbricks;
    a.halo_cells = s->halo_cells;
    a.halo_off = s->halo_off;
    a.halo_rows = s->halo_rows;
    a.halo_n = s->halo_n;
    a.brick_range = s->brick_range;
    const int lds = static_cast<int>((s->ncells + 1 + s->n) * sizeof(int));
    hipStream_t st = s->ctx->stream;
    if (s->n <= kHeadThreads)
        launch_head<1>(a, lds, st);
    else
        launch_head<kHeadItems>(a, lds, st);
    ATVH_HIP(hipGetLastError());
}

// One workgroup counts and places all keys, against a launch or two more that
// spread the sort over the chip; us a step here / in large_enqueue_first_half:
//   atoms, at few cells: 36,000 in 5,832 cells 61 / 60 FP64 and 63 / 63 mixed;
//   50,000 in 8,000 82 / 79 and 73 / 70; 65,536 in 10,648 97 / 93 and 87 / 82.
//   At cutoffs that make more cells of the same atoms the even point is higher
//   (50,000 in 12,167 cells 57 / 57 and 48 / 51), so the line is between.
//   cells, at the usual density: 31,500 atoms in 12,167 cells 37 / 41 and 39 / 44;
//   40,000 in 15,625 47 / 51 and 44 / 47; 80,000 in 32,768 63 / 54 and 58 / 51.
//   The table would fit LDS at any of these; the line is on the safe side.
bool mid_step_fits(const atvh_system* s) {
    return s->brick_mode && s->n <= kMidMaxAtoms && s->ncells < kMidMaxCells;
}

// The initial kick's launch (with the NH half of final_step); what the launch
// after it needs to decide.
static StepDecision enqueue_step_initial(atvh_system* s, int final_step, ThermoRec rec, int* key) {
    ScopedTimer tm(s->ctx, "integrate");
    MidArgs a{};
    a.i = make_int_args(s);
    a.final_partials = ke_partials_of(s, 0);
    a.i.ke_partials = ke_partials_of(s, 1);
    a.nb = integ_grid(s);
    a.do_final = final_step >= 0 ? 1 : 0;
    a.record_ke = rec.ke;
    a.step = final_step;
    a.g = brick_geom(s);
    a.csx = s->cs[0];
    a.csy = s->cs[1];
    a.csz = s->cs[2];
    a.key = key;
    if (key) // n <= kMidMaxAtoms: integ_grid's cap is above that
        k_step_initial<true><<<a.nb, kBlock, 0, s->ctx->stream>>>(a);
    else
        k_step_initial<false><<<a.nb, kBlock, 0, s->ctx->stream>>>(a);
    ATVH_HIP(hipGetLastError());
    return StepDecision{s->ctl, a.i.ke_partials, a.nb, s->thermostat, s->dt, s->every, s->delay, s->check};
}

void mid_enqueue_first_half(atvh_system* s, int final_step, bool final_energy, ThermoRec rec) {
    hipStream_t st = s->ctx->stream;
    const StepDecision d = enqueue_step_initial(s, final_step, rec, s->acell_of);
    {
        ScopedTimer tm(s->ctx, "integrate");
        MidSortArgs m{};
        m.d = d;
        m.do_energy = final_step >= 0 && final_energy ? 1 : 0;
        if (m.do_energy)
            m.e = make_finalize_args(s, rec.pe, final_step, true);
        m.n = static_cast<int>(s->n);
        m.ncells = s->ncells;
        m.key = s->acell_of;
        m.start = s->cell_start;
        m.perm = s->perm;
        k_mid_sort<<<1, kHeadThreads, (s->ncells + 1) * sizeof(int), st>>>(m);
        ATVH_HIP(hipGetLastError());
    }
    nl_enqueue_place(s);
}

// Larger systems sort over many blocks: eight launches a step (initial kick,
// bin, scan, scatter, placement, list, forces, final kick) instead of twelve.
// A launch that has nothing to do still takes 1.5-2 us of the stream, and on
// nine steps of ten the rebuild's have nothing. The run's time a step: 499,999
// atoms FP64 151 -> 144 us, 2,048,000 mixed 371 -> 363, melts of 110,592 ions
// FP64 177 -> 170 and of 512,000 mixed 376 -> 366.
bool large_step_fits(const atvh_system* s) { return s->brick_mode && nl_step_sort_fits(s); }

void large_enqueue_first_half(atvh_system* s, int final_step, ThermoRec rec) {
    nl_enqueue_step_sort(s, enqueue_step_initial(s, final_step, rec, nullptr));
    nl_enqueue_placed_lists(s);
}

} // namespace atvh
