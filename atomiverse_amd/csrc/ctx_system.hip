// ctx_system.hip — context, device frame (upload/download), timing, C-ABI glue.
//
// Replaces cuda::Backend::init / materialize / retrieve
// (src/cuda/driver/driver.cu:25-86,177) and cpu::to_cuda / cuda::to_cpu
// (src/cuda/frame/transfer.cu:145-475).

#include "atvh_internal.hpp"

#include <cmath>
#include <cstring>

using namespace atvh;

namespace atvh {

hipEvent_t take_event(atvh_ctx* c) {
    if (!c->event_pool.empty()) {
        hipEvent_t e = c->event_pool.back();
        c->event_pool.pop_back();
        return e;
    }
    hipEvent_t e;
    ATVH_HIP(hipEventCreate(&e));
    return e;
}

bool timing_on(const atvh_ctx* c, const char* nm) {
    return c->timing && (c->timing_only.empty() || c->timing_only == nm);
}

ScopedTimer::ScopedTimer(atvh_ctx* c, const char* nm) : ctx(c), name(nm) {
    if (timing_on(ctx, nm)) {
        start = take_event(ctx);
        ATVH_HIP(hipEventRecord(start, ctx->stream));
    }
}

ScopedTimer::~ScopedTimer() {
    if (!start)
        return;
    hipEvent_t stop = take_event(ctx);
    if (hipEventRecord(stop, ctx->stream) == hipSuccess)
        ctx->timers[name].pending.emplace_back(start, stop);
}

void* ctx_pin(atvh_ctx* c, size_t bytes) {
    if (bytes > kPinMax)
        throw Error(ATVH_E_ARG, "staging request beyond the pinned buffer's bound");
    if (bytes > c->pin_bytes) {
        if (c->pin)
            (void)hipHostFree(c->pin);
        c->pin = nullptr;
        c->pin_bytes = 0;
        const size_t want = bytes <= kPinMin ? kPinMin : kPinMax;
        if (hipHostMalloc(&c->pin, want, hipHostMallocDefault) != hipSuccess) {
            c->pin = nullptr;
            throw Error(ATVH_E_NOMEM, "hipHostMalloc of the staging buffer failed");
        }
        c->pin_bytes = want;
    }
    return c->pin;
}

void read_ctl(atvh_system* s, DevCtl& h) {
    atvh_ctx* c = s->ctx;
    void* p = ctx_pin(c, sizeof(DevCtl));
    ATVH_HIP(hipMemcpyAsync(p, s->ctl, sizeof(DevCtl), hipMemcpyDeviceToHost, c->stream));
    ATVH_HIP(hipStreamSynchronize(c->stream));
    std::memcpy(&h, p, sizeof(DevCtl));
}

void fetch_pieces(atvh_ctx* c, const std::vector<HostPiece>& pieces) {
    // pieces that follow each other on the device (columns of one allocation)
    // leave as one copy; `at` is each piece's place in the pinned buffer
    auto up = [](size_t b) { return (b + 511) & ~size_t(511); };
    struct Run {
        const char* src;
        size_t bytes, at;
    };
    std::vector<Run> runs;
    std::vector<size_t> at;
    size_t total = 0;
    for (const HostPiece& q : pieces) {
        const char* src = static_cast<const char*>(q.src);
        if (!runs.empty() && runs.back().src + up(runs.back().bytes) == src) {
            at.push_back(runs.back().at + (src - runs.back().src));
            runs.back().bytes = (src - runs.back().src) + q.bytes;
        } else {
            if (!runs.empty())
                total = runs.back().at + up(runs.back().bytes);
            runs.push_back(Run{src, q.bytes, total});
            at.push_back(total);
        }
        total = runs.back().at + up(runs.back().bytes);
    }
    if (total > kStageMax) {
        // three pageable copies in flight at most, none queued behind kernels:
        // nine queued at once left the caller's next host threads stalled for
        // 10-40 ms now and then (a 512,000-ion run's snapshots)
        ATVH_HIP(hipStreamSynchronize(c->stream));
        int queued = 0;
        for (const HostPiece& q : pieces) {
            ATVH_HIP(hipMemcpyAsync(q.dst, q.src, q.bytes, hipMemcpyDeviceToHost, c->stream));
            if (++queued % 3 == 0)
                ATVH_HIP(hipStreamSynchronize(c->stream));
        }
        ATVH_HIP(hipStreamSynchronize(c->stream));
        return;
    }
    char* pin = static_cast<char*>(ctx_pin(c, total));
    for (const Run& r : runs)
        ATVH_HIP(hipMemcpyAsync(pin + r.at, r.src, r.bytes, hipMemcpyDeviceToHost, c->stream));
    ATVH_HIP(hipStreamSynchronize(c->stream));
    for (size_t k = 0; k < pieces.size(); ++k)
        std::memcpy(pieces[k].dst, pin + at[k], pieces[k].bytes);
}

static void resolve_timers(atvh_ctx* c) {
    ATVH_HIP(hipStreamSynchronize(c->stream));
    for (auto& kv : c->timers) {
        for (auto& pr : kv.second.pending) {
            float ms = 0.f;
            ATVH_HIP(hipEventElapsedTime(&ms, pr.first, pr.second));
            kv.second.total_ms += ms;
            kv.second.launches += 1;
            c->event_pool.push_back(pr.first);
            c->event_pool.push_back(pr.second);
        }
        kv.second.pending.clear();
    }
}

} // namespace atvh

#define API_TRY try {
#define API_CATCH(C)                                                                    \
    }                                                                                   \
    catch (const atvh::Error& e_) {                                                     \
        if (C)                                                                          \
            (C)->err = e_.what();                                                       \
        return e_.code;                                                                 \
    }                                                                                   \
    catch (const std::exception& e_) {                                                  \
        if (C)                                                                          \
            (C)->err = e_.what();                                                       \
        return ATVH_E_ARG;                                                              \
    }

namespace {

// Frame-order gather for downloads; positions are wrapped into [0, L) here
// (wrap_orthorhombic, pbc.h:37-51), velocities get the pending NH scale. The
// nine state columns are `col` apart from `in` on, their frame-order copies
// from `out` on; groups: bit 0 positions, 1 velocities, 2 forces.
__global__ void k_gather_out(int64_t n, int64_t col, const int* __restrict__ tag, const double* __restrict__ in,
                             double* __restrict__ out, const DevCtl* ctl, int groups, double la, double lb,
                             double lc) {
    const double s = ctl->nh_scale;
    for (int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; i < n;
         i += (int64_t)gridDim.x * blockDim.x) {
        const int t = tag[i];
        if (groups & 1) {
            const double va = in[i], vb = in[col + i], vc = in[2 * col + i];
            out[t] = va - la * floor(va / la);
            out[col + t] = vb - lb * floor(vb / lb);
            out[2 * col + t] = vc - lc * floor(vc / lc);
        }
        if (groups & 2)
            for (int k = 3; k < 6; ++k)
                out[k * col + t] = in[k * col + i] * s;
        if (groups & 4)
            for (int k = 6; k < 9; ++k)
                out[k * col + t] = in[k * col + i];
    }
}

// A fresh frame: slots in frame order, no pending thermostat scale.
__global__ void k_frame_reset(int64_t n, int* __restrict__ tag, DevCtl* ctl) {
    for (int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; i < n;
         i += (int64_t)gridDim.x * blockDim.x)
        tag[i] = static_cast<int>(i);
    if (blockIdx.x == 0 && threadIdx.x == 0) {
        ctl->nh_scale = 1.0;
        ctl->always = 1;
    }
}


void sys_free_all(atvh_system* s) {
    dev_free(s->slab);
    dev_free(s->islab);
    dev_free(s->partials);
    dev_free(s->d_thermo);
    dev_free(s->ctl);
    nl_free(s);
    pair_free(s);
    coul_free(s);
    npt_free(s);
}

} // namespace

extern "C" {

int atvh_ctx_create(int device, atvh_ctx** out) {
    if (!out)
        return ATVH_E_ARG;
    *out = nullptr;
    auto* c = new atvh_ctx();
    c->device = device;
    hipError_t e = hipSetDevice(device);
    if (e == hipSuccess)
        e = hipStreamCreateWithFlags(&c->own_stream, hipStreamNonBlocking);
    if (e != hipSuccess) {
        delete c;
        return ATVH_E_HIP;
    }
    c->stream = c->own_stream;
    try {
        noalloc_bind(device);
        ctx_pin(c, kPinMin);
    } catch (const Error&) {
        (void)hipStreamDestroy(c->own_stream);
        delete c;
        return ATVH_E_HIP;
    }
    *out = c;
    return ATVH_OK;
}

int atvh_ctx_destroy(atvh_ctx* c) {
    if (!c)
        return ATVH_OK;
    if (c->live_systems > 0) {
        c->err = "atvh_ctx_destroy: systems created on this context are still alive";
        return ATVH_E_STATE;
    }
    (void)hipSetDevice(c->device);
    (void)hipStreamSynchronize(c->stream);
    for (auto& kv : c->timers)
        for (auto& pr : kv.second.pending) {
            (void)hipEventDestroy(pr.first);
            (void)hipEventDestroy(pr.second);
        }
    for (auto e : c->event_pool)
        (void)hipEventDestroy(e);
    if (c->own_stream)
        (void)hipStreamDestroy(c->own_stream);
    if (c->pin)
        (void)hipHostFree(c->pin);
    delete c;
    return ATVH_OK;
}

const char* atvh_last_error(const atvh_ctx* c) { return c ? c->err.c_str() : "null context"; }

int atvh_ctx_set_stream(atvh_ctx* c, void* stream) {
    if (!c)
        return ATVH_E_ARG;
    c->stream = stream ? static_cast<hipStream_t>(stream) : c->own_stream;
    return ATVH_OK;
}

void* atvh_ctx_stream(atvh_ctx* c) { return c ? static_cast<void*>(c->stream) : nullptr; }

int atvh_ctx_synchronize(atvh_ctx* c) {
    if (!c)
        return ATVH_E_ARG;
    API_TRY
    ATVH_HIP(hipStreamSynchronize(c->stream));
    return ATVH_OK;
    API_CATCH(c)
}

int atvh_ctx_enable_timing(atvh_ctx* c, int enable) {
    if (!c)
        return ATVH_E_ARG;
    c->timing = enable != 0;
    return ATVH_OK;
}

int atvh_ctx_timing_only(atvh_ctx* c, const char* name) {
    if (!c)
        return ATVH_E_ARG;
    API_TRY
    c->timing_only = name ? name : "";
    return ATVH_OK;
    API_CATCH(c)
}

int atvh_ctx_kernel_time(atvh_ctx* c, const char* name, double* total_ms, int64_t* launches) {
    if (!c || !name)
        return ATVH_E_ARG;
    API_TRY
    resolve_timers(c);
    auto it = c->timers.find(name);
    if (total_ms)
        *total_ms = it == c->timers.end() ? 0.0 : it->second.total_ms;
    if (launches)
        *launches = it == c->timers.end() ? 0 : it->second.launches;
    return ATVH_OK;
    API_CATCH(c)
}

int atvh_ctx_reset_timing(atvh_ctx* c) {
    if (!c)
        return ATVH_E_ARG;
    API_TRY
    resolve_timers(c);
    for (auto& kv : c->timers) {
        kv.second.total_ms = 0;
        kv.second.launches = 0;
    }
    return ATVH_OK;
    API_CATCH(c)
}

int atvh_ctx_mem_info(atvh_ctx* c, int64_t* free_bytes, int64_t* total_bytes) {
    if (!c)
        return ATVH_E_ARG;
    API_TRY
    ATVH_HIP(hipSetDevice(c->device));
    size_t f = 0, t = 0;
    ATVH_HIP(hipMemGetInfo(&f, &t));
    if (free_bytes)
        *free_bytes = static_cast<int64_t>(f);
    if (total_bytes)
        *total_bytes = static_cast<int64_t>(t);
    return ATVH_OK;
    API_CATCH(c)
}

int atvh_system_create(atvh_ctx* c, int64_t n, const double box[3], atvh_system** out) {
    if (!c || !out || !box || n <= 0)
        return ATVH_E_ARG;
    *out = nullptr;
    auto* s = new atvh_system();
    API_TRY
    if (n > (int64_t(1) << 30))
        throw Error(ATVH_E_ARG, "atvh_system_create: n exceeds 2^30 atoms");
    for (int d = 0; d < 3; ++d)
        if (!(box[d] > 0.0) || !std::isfinite(box[d]))
            throw Error(ATVH_E_ARG, "atvh_system_create: box lengths must be positive");
    ATVH_HIP(hipSetDevice(c->device));
    s->ctx = c;
    s->n = n;
    s->npad = (n + 63) / 64 * 64;
    std::memcpy(s->box, box, sizeof(double) * 3);
    double** arrs[] = {&s->x,  &s->y,  &s->z,   &s->vx,  &s->vy,  &s->vz,  &s->fx, &s->fy, &s->fz,
                       &s->q,  &s->ax, &s->ay,  &s->az,  &s->avx, &s->avy, &s->avz, &s->afx,
                       &s->afy, &s->afz, &s->aq, &s->xs, &s->ys, &s->zs};
    s->col = s->npad;
    constexpr int kCols = sizeof(arrs) / sizeof(arrs[0]);
    dev_alloc(&s->slab, size_t(kCols) * s->col);
    for (int k = 0; k < kCols; ++k)
        *arrs[k] = s->slab + k * s->col;
    int** iarrs[] = {&s->type, &s->tag, &s->atype, &s->atag};
    dev_alloc(&s->islab, size_t(4) * s->col);
    for (int k = 0; k < 4; ++k)
        *iarrs[k] = s->islab + k * s->col;
    dev_alloc(&s->ctl, 1);
    s->npartials = kMaxGrid;
    dev_alloc(&s->partials, size_t(2 * s->npartials) * kPartialStride); // pair | kinetic
    DevCtl h{};
    h.nh_scale = 1.0;
    h.always = 1;
    ATVH_HIP(hipMemcpyAsync(s->ctl, &h, sizeof(h), hipMemcpyHostToDevice, c->stream));
    ATVH_HIP(hipMemsetAsync(s->slab, 0, size_t(kCols) * s->col * sizeof(double), c->stream));
    ATVH_HIP(hipMemsetAsync(s->islab, 0, size_t(4) * s->col * sizeof(int), c->stream));
    k_frame_reset<<<grid_capped(n), kBlock, 0, c->stream>>>(n, s->tag, s->ctl);
    ATVH_HIP(hipGetLastError());
    ATVH_HIP(hipStreamSynchronize(c->stream));
    c->live_systems += 1;
    *out = s;
    return ATVH_OK;
    }
    catch (const atvh::Error& e_) {
        c->err = e_.what();
        sys_free_all(s);
        delete s;
        return e_.code;
    }
    catch (const std::exception& e_) {
        c->err = e_.what();
        sys_free_all(s);
        delete s;
        return ATVH_E_ARG;
    }
}

int atvh_system_destroy(atvh_system* s) {
    if (!s)
        return ATVH_OK;
    if (s->ctx) {
        (void)hipSetDevice(s->ctx->device);
        (void)hipStreamSynchronize(s->ctx->stream);
    }
    sys_free_all(s);
    if (s->ctx)
        s->ctx->live_systems -= 1;
    delete s;
    return ATVH_OK;
}

int64_t atvh_system_natoms(const atvh_system* s) { return s ? s->n : 0; }

int atvh_system_memory(const atvh_system* s, int part, int64_t* bytes) {
    if (!s || !bytes)
        return ATVH_E_ARG;
    const int64_t n = s->n;
    switch (part) {
    case ATVH_MEM_FRAME:
        // 23 FP64 per-atom columns (state, staging, x_save), 4 int32 columns,
        // the reduction partials and the control block
        *bytes = n * (23 * 8 + 4 * 4) + int64_t(2) * s->npartials * kPartialStride * 8 + int64_t(sizeof(DevCtl));
        return ATVH_OK;
    case ATVH_MEM_NLIST:
        *bytes = nl_device_bytes(s);
        return ATVH_OK;
    case ATVH_MEM_PAIR:
        *bytes = pair_device_bytes(s);
        return ATVH_OK;
    case ATVH_MEM_PME:
        *bytes = pme_device_bytes(s);
        return ATVH_OK;
    case ATVH_MEM_INTEGRATOR:
        *bytes = int64_t(2) * s->thermo_cap * 8; // the per-step energy record
        return ATVH_OK;
    default:
        return ATVH_E_ARG;
    }
}

int atvh_system_box(const atvh_system* s, double box[3]) {
    if (!s || !box)
        return ATVH_E_ARG;
    std::memcpy(box, s->box, sizeof(double) * 3);
    return ATVH_OK;
}

int atvh_frame_upload(atvh_system* s, const double* x, const double* y, const double* z,
                      const double* vx, const double* vy, const double* vz, const double* fx,
                      const double* fy, const double* fz, const double* mass, const int* type,
                      const double* charge) {
    if (!s || !x || !y || !z || !mass)
        return ATVH_E_ARG;
    atvh_ctx* c = s->ctx;
    API_TRY
    ATVH_HIP(hipSetDevice(c->device));
    const int64_t n = s->n;
    // per-type masses (the integrators read mass by type)
    int ntypes = 1;
    double mt[kMaxTypes];
    bool seen[kMaxTypes] = {false};
    // the common frame (one type, one mass) is recognised in vectorisable
    // chunks, given up at the first one that differs; any other frame takes
    // the checks atom by atom
    const double m0 = mass[0];
    bool uniform = m0 > 0.0;
    for (int64_t i0 = 0; uniform && i0 < n; i0 += 1024) {
        const int64_t i1 = std::min<int64_t>(n, i0 + 1024);
        int differ = 0;
        for (int64_t i = i0; i < i1; ++i)
            differ |= mass[i] != m0;
        if (type)
            for (int64_t i = i0; i < i1; ++i)
                differ |= type[i];
        uniform = differ == 0;
    }
    if (uniform) {
        seen[0] = true;
        mt[0] = mass[0];
    } else {
        for (int64_t i = 0; i < n; ++i) {
            const int t = type ? type[i] : 0;
            if (t < 0 || t >= kMaxTypes)
                throw Error(ATVH_E_ARG, "atvh_frame_upload: type out of range [0,16)");
            if (!(mass[i] > 0.0))
                throw Error(ATVH_E_ARG, "atvh_frame_upload: mass must be positive");
            if (!seen[t]) {
                seen[t] = true;
                mt[t] = mass[i];
            } else if (mt[t] != mass[i]) {
                throw Error(ATVH_E_ARG, "atvh_frame_upload: atoms of one type must share one mass");
            }
            if (t + 1 > ntypes)
                ntypes = t + 1;
        }
    }
    for (int t = 0; t < ntypes; ++t)
        s->mass_t[t] = seen[t] ? mt[t] : 1.0;
    s->ntypes = ntypes;
    hipStream_t st = c->stream;
    // the state columns x .. q are the first ten of the frame's allocation
    const double* cols[] = {x, y, z, vx, vy, vz, fx, fy, fz, charge};
    constexpr int kUp = sizeof(cols) / sizeof(cols[0]);
    const size_t nb = size_t(n) * sizeof(double), cb = size_t(s->col) * sizeof(double);
    const size_t staged = kUp * cb + size_t(n) * sizeof(int);
    if (staged <= kStageMax) {
        char* pin = static_cast<char*>(ctx_pin(c, staged));
        for (int k = 0; k < kUp; ++k) {
            if (cols[k])
                std::memcpy(pin + k * cb, cols[k], nb);
            else
                std::memset(pin + k * cb, 0, nb);
        }
        char* tp = pin + kUp * cb;
        if (type)
            std::memcpy(tp, type, size_t(n) * sizeof(int));
        else
            std::memset(tp, 0, size_t(n) * sizeof(int));
        ATVH_HIP(hipMemcpyAsync(s->slab, pin, kUp * cb, hipMemcpyHostToDevice, st));
        ATVH_HIP(hipMemcpyAsync(s->type, tp, size_t(n) * sizeof(int), hipMemcpyHostToDevice, st));
    } else {
        for (int k = 0; k < kUp; ++k) {
            double* d = s->slab + k * s->col;
            if (cols[k])
                ATVH_HIP(hipMemcpyAsync(d, cols[k], nb, hipMemcpyHostToDevice, st));
            else
                ATVH_HIP(hipMemsetAsync(d, 0, nb, st));
        }
        if (type)
            ATVH_HIP(hipMemcpyAsync(s->type, type, n * sizeof(int), hipMemcpyHostToDevice, st));
        else
            ATVH_HIP(hipMemsetAsync(s->type, 0, n * sizeof(int), st));
    }
    s->has_charge = charge != nullptr;
    // charge sums in ascending atom order (KSpacePME self / net-charge terms,
    // pme.cpp:222-226) and the bound of any spread grid point
    s->q_sum = s->q_sq = s->q_abs = s->q_max = 0.0;
    if (charge)
        for (int64_t i = 0; i < n; ++i) {
            s->q_sq += charge[i] * charge[i];
            s->q_sum += charge[i];
            s->q_abs += std::fabs(charge[i]);
            s->q_max = std::max(s->q_max, std::fabs(charge[i]));
        }
    // a fresh frame: no pending thermostat scale; list must be rebuilt
    k_frame_reset<<<grid_capped(n), kBlock, 0, st>>>(n, s->tag, s->ctl);
    ATVH_HIP(hipGetLastError());
    s->nl_built = false;
    ATVH_HIP(hipStreamSynchronize(st));
    return ATVH_OK;
    API_CATCH(c)
}

int atvh_frame_download(atvh_system* s, double* x, double* y, double* z, double* vx, double* vy,
                        double* vz, double* fx, double* fy, double* fz) {
    if (!s)
        return ATVH_E_ARG;
    atvh_ctx* c = s->ctx;
    API_TRY
    ATVH_HIP(hipSetDevice(c->device));
    const int64_t n = s->n;
    hipStream_t st = c->stream;
    double* host[] = {x, y, z, vx, vy, vz, fx, fy, fz};
    int groups = 0;
    for (int k = 0; k < 9; ++k)
        groups |= host[k] ? 1 << (k / 3) : 0;
    if (!groups)
        return ATVH_OK;
    // the state columns, then their frame-order copies in the permutation
    // scratch (the same order there): one launch, one copy
    k_gather_out<<<grid_capped(n), kBlock, 0, st>>>(n, s->col, s->tag, s->x, s->ax, s->ctl, groups, s->box[0],
                                                    s->box[1], s->box[2]);
    ATVH_HIP(hipGetLastError());
    std::vector<HostPiece> pieces;
    for (int k = 0; k < 9; ++k)
        if (host[k])
            pieces.push_back(HostPiece{host[k], s->ax + k * s->col, size_t(n) * sizeof(double)});
    fetch_pieces(c, pieces);
    return ATVH_OK;
    API_CATCH(c)
}

int atvh_energy(atvh_system* s, double* pe, double* virial6, double* ke) {
    if (!s)
        return ATVH_E_ARG;
    atvh_ctx* c = s->ctx;
    API_TRY
    DevCtl h{};
    read_ctl(s, h);
    if (pe)
        *pe = h.pe;
    if (virial6)
        for (int k = 0; k < 6; ++k)
            virial6[k] = h.vir[k];
    if (ke)
        *ke = h.ke;
    return ATVH_OK;
    API_CATCH(c)
}

int atvh_thermostat_state(atvh_system* s, double* xi_out, const double* xi_in) {
    if (!s)
        return ATVH_E_ARG;
    atvh_ctx* c = s->ctx;
    API_TRY
    DevCtl h{};
    read_ctl(s, h);
    if (xi_out)
        *xi_out = h.xi;
    if (xi_in) {
        h.xi = *xi_in;
        ATVH_HIP(hipMemcpy(s->ctl, &h, sizeof(h), hipMemcpyHostToDevice));
    }
    return ATVH_OK;
    API_CATCH(c)
}

} // extern "C"
