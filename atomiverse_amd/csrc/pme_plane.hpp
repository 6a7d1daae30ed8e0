// pme_plane.hpp — the PME mesh transforms as three launches, for meshes whose
// x-planes fit LDS, any sizes of factors 2, 3, 5 and 7, FP32 and FP64.
//
// The FFT library runs such a mesh (25^3 ... 120^3: a serving segment, a melt
// of a hundred thousand ions) as four to eight launches of 2-12 us, most of
// them latency, beside an unfix and an influence launch. Here a workgroup
// owns an x-plane: it reads the fixed-point mesh (clearing it), transforms the
// z-lines and then the y-lines in LDS and writes the plane's half spectrum
// once; a second launch owns tiles of x-lines (forward transform, influence
// function with its energy and virial sums, inverse transform); the third is
// the first in reverse. The spectrum crosses memory four times instead of
// ten, and ten (six) launches are three. 25^3 in FP32: ten launches of 32 us in
// all -> 6.5 + 6.0 + 6.3 us; 80^3 in FP64: six of 44.6 us -> 15.8 + 9.9 + 14.2.
// What bounds them: the chain of LDS passes, each a read, a butterfly, a write
// and a barrier, with one workgroup on a CU and K0 of the 256 CUs busy; the
// 80^3 mesh's bytes would take 9 us of the 40 at the rate of a large copy.
//
// Threads, measured before the divisions moved to the host: 1,024 a plane
// instead of 512 cost 25^3 1.2 us a launch (wider barriers) and gave 80^3 1 us;
// 512 a tile of x-lines instead of 256 gave 25^3 0.7 us and 80^3 2.2 us.
//
// Real z-lines go two to a complex line (a + i b), which needs no even length.
// Lines are transformed by Stockham's autosort passes between two LDS buffers
// (natural order in and out), radices 2, 3, 4, 5, 7; twiddles come from
// host-built tables (long double sin/cos, rounded once). The reference
// transforms with FFTW r2c / c2r (src/cpu/longrange/pme.cpp:152-253).
#pragma once

#include "atvh_internal.hpp"
#include "pair_common.hpp"
#include "pme_fft.hpp"

namespace atvh {
namespace pmeplane {

using pmefft::cadd;
using pmefft::cconj;
using pmefft::cmul;
using pmefft::Cplx;
using pmefft::csub;

constexpr int kMaxStages = 6;
constexpr int kPlaneThreads = 512;
constexpr int kLineThreads = 512;
constexpr int kTile = 16;                    // x-lines per workgroup: 64 B of FP32 spectrum a row
constexpr int kPlaneAxisMax = 128;           // points of an axis (a tile of x-lines then takes 66 KB in FP64)
constexpr int kPlaneLds = 150 * 1024;        // LDS a plane's workgroup may take (of 160 KB)

// x / d for x, d < 2^16 as a high multiply by ceil(2^32 / d). Made on the host:
// the same constants made in the kernel, an integer division each, cost two
// per pass and 1.1-1.4 us a launch (25^3 7.8 -> 6.5 us).
struct FastDiv {
    unsigned m, d;
    __device__ __forceinline__ int div(int x) const { return d == 1 ? x : static_cast<int>(__umulhi(x, m)); }
};
inline FastDiv fast_div(int d) { return FastDiv{d > 1 ? 0xffffffffu / static_cast<unsigned>(d) + 1 : 0, static_cast<unsigned>(d)}; }

// One Stockham pass over lines of K values: radix R, s the product of the
// radices done, m = n / R of the length n still to be split.
struct Pass {
    int R, m, s, ws; // ws = K / n: stride of the pass's twiddles in the table
    FastDiv per, by_s; // per = K / R butterflies a line
};

// The passes of one axis, odd radices first: the first pass writes with a
// stride of its radix, which odd radices spread over the LDS banks.
struct Axis {
    int K;
    int ns;
    Pass p[kMaxStages];
};

// Whether K has only the factors 2, 3, 5, 7 and at most kMaxStages passes.
inline bool make_axis(int K, Axis& a) {
    a.K = K;
    a.ns = 0;
    int n = K, s = 1;
    for (int r : {7, 5, 3, 4, 2})
        while (n % r == 0) {
            if (a.ns == kMaxStages)
                return false;
            a.p[a.ns++] = Pass{r, n / r, s, K / n, fast_div(K / r), fast_div(s)};
            n /= r;
            s *= r;
        }
    return n == 1 && K > 1;
}

// Line strides in LDS: odd, so the lines' same elements fall in different banks.
__host__ __device__ constexpr int line_stride(int K) { return K | 1; }

struct PlaneArgs {
    Axis a0, a1, a2;
    int Kh;
    FastDiv by2, byh; // by K2 and Kh
    double inv_fix;
    unsigned long long* fix; // [K0][K1][K2]
    void* real;              // [K0][K1][K2]
    void* cplx;              // [K0][K1][Kh]
    const void *tw0, *tw1, *tw2; // exp(-2 pi i k / K), k < K
    const double* H;
    double ic0, ic1, ic2, pi2_a2;
    double* partials;
};

// Complex values of one LDS buffer of a plane's workgroup.
__host__ __device__ inline int plane_values(int K1, int K2, int Kh) {
    const int z = (K1 + 1) / 2 * line_stride(K2), y = Kh * line_stride(K1);
    return z > y ? z : y;
}

// R-point transform of v in place; INV conjugates.
template <class T2, int R, bool INV>
__device__ __forceinline__ void small_dft(T2 (&v)[R]) {
    using T = decltype(T2::x);
    if constexpr (R == 2) {
        const T2 a = v[0], b = v[1];
        v[0] = cadd(a, b);
        v[1] = csub(a, b);
    } else if constexpr (R == 4) {
        const T2 a = cadd(v[0], v[2]), b = csub(v[0], v[2]), c = cadd(v[1], v[3]);
        T2 d = csub(v[1], v[3]); // times -i (forward) or i
        const T t = d.x;
        d.x = INV ? -d.y : d.y;
        d.y = INV ? t : -t;
        v[0] = cadd(a, c);
        v[2] = csub(a, c);
        v[1] = cadd(b, d);
        v[3] = csub(b, d);
    } else {
        // odd R: sums and differences of the pairs (r, R - r);
        // cos and sin of 2 pi j / R, j = 1 .. (R - 1) / 2
        constexpr int P = (R - 1) / 2;
        constexpr double c3[] = {-0.5}, s3[] = {0.86602540378443864676};
        constexpr double c5[] = {0.30901699437494742410, -0.80901699437494742410},
                         s5[] = {0.95105651629515357212, 0.58778525229247312917};
        constexpr double c7[] = {0.62348980185873353053, -0.22252093395631440429, -0.90096886790241912624},
                         s7[] = {0.78183148246802980871, 0.97492791218182360702, 0.43388373911755812048};
        T2 s[P], d[P];
        T2 sum = v[0];
#pragma unroll
        for (int r = 0; r < P; ++r) {
            s[r] = cadd(v[r + 1], v[R - 1 - r]);
            d[r] = csub(v[r + 1], v[R - 1 - r]);
            sum = cadd(sum, s[r]);
        }
        const T2 v0 = v[0];
        v[0] = sum;
#pragma unroll
        for (int k = 1; k <= P; ++k) {
            T2 e = v0, o;
            o.x = T(0);
            o.y = T(0);
#pragma unroll
            for (int r = 1; r <= P; ++r) {
                const int j = (r * k) % R;
                const int jj = j <= P ? j : R - j;
                const double cc = R == 3 ? c3[(jj - 1) % 1] : (R == 5 ? c5[(jj - 1) % 2] : c7[(jj - 1) % 3]);
                const double ss = R == 3 ? s3[(jj - 1) % 1] : (R == 5 ? s5[(jj - 1) % 2] : s7[(jj - 1) % 3]);
                const T c = static_cast<T>(cc), q = static_cast<T>(j <= P ? ss : -ss);
                e.x += c * s[r - 1].x;
                e.y += c * s[r - 1].y;
                o.x += q * d[r - 1].x;
                o.y += q * d[r - 1].y;
            }
            // forward: X_k = e - i o, X_{R-k} = e + i o
            T2 lo, hi;
            lo.x = e.x + o.y;
            lo.y = e.y - o.x;
            hi.x = e.x - o.y;
            hi.y = e.y + o.x;
            v[k] = INV ? hi : lo;
            v[R - k] = INV ? lo : hi;
        }
    }
}

// One pass of radix R over `lines` lines, ls apart.
template <class T2, int R, bool INV>
__device__ __forceinline__ void pass(const T2* x, T2* y, const T2* tw, const Pass& ps, int ls, int lines) {
    const int m = ps.m, s = ps.s, ws = ps.ws, per = ps.per.d, total = lines * per;
    for (int it = threadIdx.x; it < total; it += blockDim.x) {
        const int line = ps.per.div(it), u = it - line * per;
        const int p = ps.by_s.div(u), q = u - p * s;
        const T2* xl = x + line * ls + q + s * p;
        T2 v[R];
#pragma unroll
        for (int r = 0; r < R; ++r)
            v[r] = xl[s * m * r];
        small_dft<T2, R, INV>(v);
        T2* yl = y + line * ls + q + s * R * p;
        yl[0] = v[0];
#pragma unroll
        for (int k = 1; k < R; ++k) {
            T2 w = tw[p * k * ws];
            if (INV)
                w.y = -w.y;
            yl[s * k] = cmul(v[k], w);
        }
    }
    __syncthreads();
}

// All passes of an axis over lines in `cur`; `cur` ends at the buffer that
// holds the result. Barriers follow every pass.
template <class T2, bool INV>
__device__ __forceinline__ void transform(T2*& cur, T2*& other, const T2* tw, const Axis& a, int ls, int lines) {
    for (int st = 0; st < a.ns; ++st) {
        const Pass& ps = a.p[st];
        switch (ps.R) {
        case 2: pass<T2, 2, INV>(cur, other, tw, ps, ls, lines); break;
        case 3: pass<T2, 3, INV>(cur, other, tw, ps, ls, lines); break;
        case 4: pass<T2, 4, INV>(cur, other, tw, ps, ls, lines); break;
        case 5: pass<T2, 5, INV>(cur, other, tw, ps, ls, lines); break;
        default: pass<T2, 7, INV>(cur, other, tw, ps, ls, lines); break;
        }
        T2* t = cur;
        cur = other;
        other = t;
    }
}

// Fixed-point plane -> its half spectrum.
template <class T>
__global__ __launch_bounds__(kPlaneThreads) void k_plane_forward(PlaneArgs a) {
    using T2 = typename Cplx<T>::type;
    extern __shared__ __align__(16) char lds[];
    const int K1 = a.a1.K, K2 = a.a2.K, Kh = a.Kh, L = (K1 + 1) / 2;
    const int ls1 = line_stride(K1), ls2 = line_stride(K2), nv = plane_values(K1, K2, Kh);
    T2* cur = reinterpret_cast<T2*>(lds);
    T2* other = cur + nv;
    T2* tw1 = other + nv;
    T2* tw2 = tw1 + K1;
    for (int k = threadIdx.x; k < K1; k += kPlaneThreads)
        tw1[k] = static_cast<const T2*>(a.tw1)[k];
    for (int k = threadIdx.x; k < K2; k += kPlaneThreads)
        tw2[k] = static_cast<const T2*>(a.tw2)[k];
    unsigned long long* fix = a.fix + (int64_t)blockIdx.x * K1 * K2;
    const FastDiv by2 = a.by2, byh = a.byh;
    for (int e = threadIdx.x; e < L * K2; e += kPlaneThreads) {
        const int l = by2.div(e), k = e - l * K2;
        const int i = 2 * l * K2 + k;
        const bool two = 2 * l + 1 < K1;
        T2 z;
        z.x = static_cast<T>(static_cast<double>(static_cast<long long>(fix[i])) * a.inv_fix);
        z.y = two ? static_cast<T>(static_cast<double>(static_cast<long long>(fix[i + K2])) * a.inv_fix) : T(0);
        fix[i] = 0ull;
        if (two)
            fix[i + K2] = 0ull;
        cur[l * ls2 + k] = z;
    }
    __syncthreads();
    transform<T2, false>(cur, other, tw2, a.a2, ls2, L);
    // the two lines of each packed one: (Z_k + conj Z_-k) / 2, -i (Z_k - conj Z_-k) / 2
    for (int e = threadIdx.x; e < L * Kh; e += kPlaneThreads) {
        const int l = byh.div(e), k = e - l * Kh;
        const T2 zk = cur[l * ls2 + k], zc = cconj(cur[l * ls2 + (k ? K2 - k : 0)]);
        const T2 p = cadd(zk, zc), m = csub(zk, zc);
        T2 va, vb;
        va.x = T(0.5) * p.x;
        va.y = T(0.5) * p.y;
        vb.x = T(0.5) * m.y;
        vb.y = T(-0.5) * m.x;
        other[k * ls1 + 2 * l] = va;
        if (2 * l + 1 < K1)
            other[k * ls1 + 2 * l + 1] = vb;
    }
    __syncthreads();
    T2* c = other;
    T2* o = cur;
    transform<T2, false>(c, o, tw1, a.a1, ls1, Kh);
    T2* out = static_cast<T2*>(a.cplx) + (int64_t)blockIdx.x * K1 * Kh;
    for (int e = threadIdx.x; e < K1 * Kh; e += kPlaneThreads) {
        const int m1 = byh.div(e), m2 = e - m1 * Kh;
        out[e] = c[m2 * ls1 + m1];
    }
}

// Half spectrum of a plane -> its real potential mesh.
template <class T>
__global__ __launch_bounds__(kPlaneThreads) void k_plane_inverse(PlaneArgs a) {
    using T2 = typename Cplx<T>::type;
    extern __shared__ __align__(16) char lds[];
    const int K1 = a.a1.K, K2 = a.a2.K, Kh = a.Kh, L = (K1 + 1) / 2;
    const int ls1 = line_stride(K1), ls2 = line_stride(K2), nv = plane_values(K1, K2, Kh);
    T2* cur = reinterpret_cast<T2*>(lds);
    T2* other = cur + nv;
    T2* tw1 = other + nv;
    T2* tw2 = tw1 + K1;
    for (int k = threadIdx.x; k < K1; k += kPlaneThreads)
        tw1[k] = static_cast<const T2*>(a.tw1)[k];
    for (int k = threadIdx.x; k < K2; k += kPlaneThreads)
        tw2[k] = static_cast<const T2*>(a.tw2)[k];
    const T2* in = static_cast<const T2*>(a.cplx) + (int64_t)blockIdx.x * K1 * Kh;
    const FastDiv by2 = a.by2, byh = a.byh;
    for (int e = threadIdx.x; e < K1 * Kh; e += kPlaneThreads) {
        const int m1 = byh.div(e), m2 = e - m1 * Kh;
        cur[m2 * ls1 + m1] = in[e];
    }
    __syncthreads();
    transform<T2, true>(cur, other, tw1, a.a1, ls1, Kh);
    // packed lines A + i B over the whole period (X_{K-k} = conj X_k)
    for (int e = threadIdx.x; e < L * K2; e += kPlaneThreads) {
        const int l = by2.div(e), k = e - l * K2;
        const bool back = k >= Kh;
        const int kk = back ? K2 - k : k;
        T2 va = cur[kk * ls1 + 2 * l], vb;
        vb.x = T(0);
        vb.y = T(0);
        if (2 * l + 1 < K1)
            vb = cur[kk * ls1 + 2 * l + 1];
        if (back) {
            va = cconj(va);
            vb = cconj(vb);
        }
        T2 z;
        z.x = va.x - vb.y;
        z.y = va.y + vb.x;
        other[l * ls2 + k] = z;
    }
    __syncthreads();
    T2* c = other;
    T2* o = cur;
    transform<T2, true>(c, o, tw2, a.a2, ls2, L);
    T* real = static_cast<T*>(a.real) + (int64_t)blockIdx.x * K1 * K2;
    for (int e = threadIdx.x; e < L * K2; e += kPlaneThreads) {
        const int l = by2.div(e), k = e - l * K2;
        const T2 z = c[l * ls2 + k];
        real[2 * l * K2 + k] = z.x;
        if (2 * l + 1 < K1)
            real[(2 * l + 1) * K2 + k] = z.y;
    }
}

__host__ __device__ inline int line_tiles(int K1, int Kh) { return (K1 * Kh + kTile - 1) / kTile; }

// x-lines of kTile adjacent columns of the spectrum: forward, influence
// function and its sums (pme_apply_influence_tables, pme_influence.h:179-222,
// folded over the Hermitian partners as the separate influence kernel does),
// inverse. EV: 0 none, 1 energy, 2 energy and virial.
template <class T, int EV>
__global__ __launch_bounds__(kLineThreads) void k_lines_influence(PlaneArgs a) {
    using T2 = typename Cplx<T>::type;
    extern __shared__ __align__(16) char lds[];
    const int K0 = a.a0.K, K1 = a.a1.K, K2 = a.a2.K, Kh = a.Kh, C = K1 * Kh;
    const int ls0 = line_stride(K0);
    T2* cur = reinterpret_cast<T2*>(lds);
    T2* other = cur + kTile * ls0;
    T2* tw0 = other + kTile * ls0;
    for (int k = threadIdx.x; k < K0; k += kLineThreads)
        tw0[k] = static_cast<const T2*>(a.tw0)[k];
    const int c0 = blockIdx.x * kTile, ncol = min(kTile, C - c0);
    T2* S = static_cast<T2*>(a.cplx) + c0;
    for (int e = threadIdx.x; e < kTile * K0; e += kLineThreads) {
        const int i = e / kTile, col = e % kTile;
        T2 v;
        v.x = T(0);
        v.y = T(0);
        if (col < ncol)
            v = S[(int64_t)i * C + col];
        cur[col * ls0 + i] = v;
    }
    __syncthreads();
    transform<T2, false>(cur, other, tw0, a.a0, ls0, kTile);
    double acc[7] = {0, 0, 0, 0, 0, 0, 0};
    for (int e = threadIdx.x; e < kTile * K0; e += kLineThreads) {
        const int m0 = e / kTile, col = e % kTile;
        if (col >= ncol)
            continue;
        const double h = a.H[(int64_t)m0 * C + c0 + col];
        T2 v = cur[col * ls0 + m0];
        if (EV && h != 0.0) {
            const int m1 = (c0 + col) / Kh, m2 = (c0 + col) % Kh;
            const double re = static_cast<double>(v.x), im = static_cast<double>(v.y);
            const double ug = h * (re * re + im * im);
            const bool pair = m2 != 0 && 2 * m2 != K2;
            const double w = pair ? 2.0 : 1.0;
            acc[0] += w * ug;
            if (EV == 2) {
                const int h0 = (m0 <= K0 / 2) ? m0 : m0 - K0;
                const int h1 = (m1 <= K1 / 2) ? m1 : m1 - K1;
                const double mx = h0 * a.ic0, my = h1 * a.ic1, mz = m2 * a.ic2;
                const double msq = mx * mx + my * my + mz * mz;
                const double vt = -2.0 * (1.0 / msq + a.pi2_a2);
                const double sx = (2 * m0 == K0) ? 1.0 : -1.0;
                const double sy = (2 * m1 == K1) ? 1.0 : -1.0;
                const double oxy = pair ? 1.0 + sx * sy : 1.0;
                const double oxz = pair ? 1.0 - sx : 1.0;
                const double oyz = pair ? 1.0 - sy : 1.0;
                acc[1] += w * ug * (1.0 + vt * mx * mx);
                acc[2] += w * ug * (1.0 + vt * my * my);
                acc[3] += w * ug * (1.0 + vt * mz * mz);
                acc[4] += oxy * ug * (vt * mx * my);
                acc[5] += oxz * ug * (vt * mx * mz);
                acc[6] += oyz * ug * (vt * my * mz);
            }
        }
        v.x *= static_cast<T>(h);
        v.y *= static_cast<T>(h);
        cur[col * ls0 + m0] = v;
    }
    __syncthreads();
    transform<T2, true>(cur, other, tw0, a.a0, ls0, kTile);
    for (int e = threadIdx.x; e < kTile * K0; e += kLineThreads) {
        const int i = e / kTile, col = e % kTile;
        if (col < ncol)
            S[(int64_t)i * C + col] = cur[col * ls0 + i];
    }
    if (EV)
        block_partials<kLineThreads>(acc, a.partials, blockIdx.x);
}

} // namespace pmeplane
} // namespace atvh
