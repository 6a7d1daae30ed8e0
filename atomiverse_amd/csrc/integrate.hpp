// integrate.hpp — the per-atom and scalar pieces of one velocity Verlet +
// Nose-Hoover step, shared by the multi-block stages (integrate.hip) and the
// one-workgroup step of small systems (small_step.hip).
#pragma once

#include "atvh_internal.hpp"
#include "pair_common.hpp"

namespace atvh {

struct IntArgs {
    int64_t n;
    double *x, *y, *z, *vx, *vy, *vz;
    const double *fx, *fy, *fz;
    const int* type;
    const double *xs, *ys, *zs;
    double dtfm[kMaxTypes];
    double mass[kMaxTypes];
    int ntypes;
    double dt;
    double lx, ly, lz;
    double skin_sq;
    int thermostat;
    DevCtl* ctl;
    double* ke_partials;
};

// The kicks: one atom per grid-stride step, its loads issued before its
// stores. A one-type frame takes dtfm and mass from scalars (no dependent
// per-atom table loads). (Two atoms per step, both loaded before either is
// stored, needed 142 registers for the initial kick and lost on the batched
// ladder what it gained on the 2.048M-atom fluid.)
struct KickAtom {
    double vx, vy, vz, fx, fy, fz;
    int t;
};

__device__ __forceinline__ KickAtom kick_load(const IntArgs& a, int64_t i, bool typed) {
    KickAtom k;
    k.t = typed ? a.type[i] : 0;
    k.vx = a.vx[i];
    k.vy = a.vy[i];
    k.vz = a.vz[i];
    k.fx = a.fx[i];
    k.fy = a.fy[i];
    k.fz = a.fz[i];
    return k;
}

// v <- (v s) + dtfm f (the reference's order: the pending NH scale, then the
// kick); returns m v^2 of the new velocity
__device__ __forceinline__ double kick_apply(const IntArgs& a, KickAtom& k, double s, bool typed, double dtfm0,
                                             double m0) {
    double dtfm = dtfm0, m = m0;
    if (typed) {
        dtfm = a.dtfm[k.t];
        m = a.mass[k.t];
    }
    if (a.thermostat) {
        k.vx *= s;
        k.vy *= s;
        k.vz *= s;
    }
    k.vx += dtfm * k.fx;
    k.vy += dtfm * k.fy;
    k.vz += dtfm * k.fz;
    return m * (k.vx * k.vx + k.vy * k.vy + k.vz * k.vz);
}

// The displacement half of needs_rebuild (cell_list.cpp:372-391) for one
// atom: 4 |min_image(x - x_save)|^2 > skin^2. Up to half a box length the
// image count nearbyint(d / L) is zero (0.5 ties to 0), so the divisions run
// only in a wavefront that holds an atom past it.
__device__ __forceinline__ bool moved_past_skin(const IntArgs& a, double dx, double dy, double dz) {
    if (!(fabs(dx) <= 0.5 * a.lx && fabs(dy) <= 0.5 * a.ly && fabs(dz) <= 0.5 * a.lz)) {
        dx -= a.lx * nearbyint(dx / a.lx);
        dy -= a.ly * nearbyint(dy / a.ly);
        dz -= a.lz * nearbyint(dz / a.lz);
    }
    const double dsq = dx * dx + dy * dy + dz * dz;
    return dsq * 4.0 > a.skin_sq;
}

// Sum over a kBlock-thread block, the waves added in order.
__device__ __forceinline__ void block_sum_to(double v, double* out) {
    __shared__ double sh[kBlock / 64];
    v = wave_sum(v);
    const int lane = threadIdx.x & 63, wid = threadIdx.x >> 6;
    if (lane == 0)
        sh[wid] = v;
    __syncthreads();
    if (threadIdx.x == 0) {
        double t = 0.0;
        for (int w = 0; w < kBlock / 64; ++w)
            t += sh[w];
        *out = t;
    }
}

// NoseHoover::launch: xi from the kinetic energy; the velocity scale to apply.
__device__ __forceinline__ double nh_update(double ke, double dt, double ndof_kT, double Q, double& xi) {
    xi += (dt * 0.5) * (2.0 * ke - ndof_kT) / Q;
    return exp(-dt * 0.5 * xi);
}

// NeighborList::decide_reneighbor, in the parts its callers order differently:
// whether the list is due `ago` steps after its build, ...
__device__ __forceinline__ bool reneighbor_due(int ago, int every, int delay, int check, bool moved) {
    return ago >= delay && (ago % every) == 0 && (!check || moved);
}
// ... the decision as the rebuild stages read it (one thread) ...
__device__ __forceinline__ void publish_rebuild(DevCtl* c, bool rb) {
    c->rebuild = rb ? 1 : 0;
    if (rb) {
        c->nrebuilds += 1;
        c->nbr_total = 0;
        c->max_nbr = 0;
    }
}
// ... and the state the next decision reads (one thread).
__device__ __forceinline__ void reneighbor_next(DevCtl* c, bool rb, int ago) {
    c->disp_flag = 0;
    c->ago = rb ? 0 : ago;
}

// NeighborList::decide_reneighbor for this step (one thread).
__device__ __forceinline__ bool decide_reneighbor(DevCtl* c, int every, int delay, int check, bool moved) {
    const int ago = c->ago + 1;
    const bool rb = reneighbor_due(ago, every, delay, check, moved);
    publish_rebuild(c, rb);
    reneighbor_next(c, rb, ago);
    return rb;
}

// The NH half after the initial kick and the rebuild decision, for a launch
// that finds both itself (k_step_bin).
struct StepDecision {
    DevCtl* ctl;
    const double* partials; // m v^2 of the initial kick
    int nb;
    int thermostat;
    double dt;
    int every, delay, check;
};

// xi, scale and the half-step kinetic energy from the kick's total (one thread).
__device__ __forceinline__ void initial_nh(const StepDecision& d, double mv2) {
    DevCtl* c = d.ctl;
    const double ke = 0.5 * mass_v2_to_energy * mv2;
    double xi = c->xi_mid;
    if (d.thermostat)
        c->nh_scale = nh_update(ke, d.dt, c->nh_ndof_kT, c->nh_Q, xi);
    c->xi = xi;
    c->ke_half = ke;
}

struct FinalizeArgs {
    DevCtl* ctl;
    const double* partials; // pair style, per workgroup
    int nb;
    const double* kpartials; // k-space influence, per workgroup (kspace only)
    int knb;
    double escale, e_self, e_net;
    double* record_pe;
    int step; // record index; < 0: the device counter ctl->rec_step
};

// Fixed-order totals of the force phase: pair energy and virial, then the
// k-space terms in the reference's order (self first, then reciprocal + net
// charge; pme.cpp:222-246).
__device__ __forceinline__ void finalize_totals(const FinalizeArgs& a) {
    double v[7], k[7];
    block_fixed_sums<7>(a.partials, a.nb, kPartialStride, v);
    block_fixed_sums<7>(a.kpartials, a.knb, kPartialStride, k);
    if (threadIdx.x == 0) {
        double pe = v[0];
        if (a.knb > 0) {
            const double e_recip = k[0] * a.escale;
            pe += a.e_self;
            pe += e_recip + a.e_net;
            for (int c = 0; c < 6; ++c)
                v[c + 1] += k[c + 1] * a.escale;
            a.ctl->e_kspace[0] = e_recip;
            a.ctl->e_kspace[1] = a.e_self;
            a.ctl->e_kspace[2] = a.e_net;
        }
        a.ctl->pe = pe;
        for (int c = 0; c < 6; ++c)
            a.ctl->vir[c] = v[c + 1];
        if (a.record_pe)
            a.record_pe[a.step >= 0 ? a.step : a.ctl->rec_step] = pe;
    }
}

// The multi-block stages the one-launch paths still use (integrate.hip).
void enqueue_final_kick(atvh_system* s, const IntArgs& a);
void enqueue_final_post(atvh_system* s, int step, ThermoRec rec);
double* ke_partials_of(const atvh_system* s, int which); // two sets of integ_grid partials

// Launches of the multi-block steps (small_step.hip): the NH half of
// final_step (< 0: none ends here), the next initial kick and drift, then the
// decision and, on a rebuild, the sort and the lists.
bool large_step_fits(const atvh_system* s);
void large_enqueue_first_half(atvh_system* s, int final_step, ThermoRec rec);
bool nl_step_sort_fits(const atvh_system* s); // neighbor.hip
void nl_enqueue_step_sort(atvh_system* s, const StepDecision& d);
int integ_grid(const atvh_system* s);

IntArgs make_int_args(atvh_system* s);
FinalizeArgs make_finalize_args(atvh_system* s, double* record_pe, int step, bool with_pair);

} // namespace atvh
