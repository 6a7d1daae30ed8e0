// pair_common.hpp — pieces shared by the brick pair kernels: wavefront and
// fixed-order block reductions of (energy, virial) partials, and the periodic
// image of a halo row.
#pragma once

#include "atvh_internal.hpp"
#include "brick.hpp"

namespace atvh {

template <class T>
__device__ __forceinline__ T wave_sum(T v) {
    for (int off = 32; off > 0; off >>= 1)
        v += __shfl_down(v, off, 64);
    return v;
}

// Fixed-order block reduction of 7 doubles into partials[slot*8 + k]
// (kThreads-thread blocks: the waves summed in order by thread k); slot is
// the block's index within its system's launch.
template <int kThreads = kBlock>
__device__ __forceinline__ void block_partials(double (&acc)[7], double* partials, int slot) {
    __shared__ double sh[kThreads / 64][7];
    const int lane = threadIdx.x & 63, wid = threadIdx.x >> 6;
#pragma unroll
    for (int k = 0; k < 7; ++k)
        acc[k] = wave_sum(acc[k]);
    if (lane == 0)
#pragma unroll
        for (int k = 0; k < 7; ++k)
            sh[wid][k] = acc[k];
    __syncthreads();
    if (threadIdx.x < 7) {
        double t = 0.0;
        for (int w = 0; w < kThreads / 64; ++w)
            t += sh[w][threadIdx.x];
        partials[slot * kPartialStride + threadIdx.x] = t;
    }
}

// Fixed-order sums of C columns over nb partial rows of `stride` doubles, by
// one kBlock-thread block: thread t adds rows t, t + kBlock, ..., then the
// threads are added in halves (t + 128, t + 64, ..., t + 1); threads past
// kBlock of a larger block only meet the barriers. Valid on thread 0. One pass over the rows for all columns, the halves below a wavefront by
// shuffles, one barrier (a pass and eight barriers per column before: energy
// and virial of 2,048,000 atoms, 8,575 rows, 44 -> 11 us).
template <int C>
__device__ __forceinline__ void block_fixed_sums(const double* __restrict__ p, int nb, int stride, double (&out)[C]) {
    __shared__ double sh[C][kBlock];
    double t[C];
#pragma unroll
    for (int c = 0; c < C; ++c)
        t[c] = 0.0;
    if (threadIdx.x < kBlock)
#pragma unroll 4
        for (int b = threadIdx.x; b < nb; b += kBlock)
#pragma unroll
            for (int c = 0; c < C; ++c)
                t[c] += p[(int64_t)b * stride + c];
    __syncthreads(); // sh may still be read by an earlier call
    if (threadIdx.x < kBlock)
#pragma unroll
        for (int c = 0; c < C; ++c)
            sh[c][threadIdx.x] = t[c];
    __syncthreads();
    if (threadIdx.x >= 64)
        return;
#pragma unroll
    for (int c = 0; c < C; ++c) {
        const double* s = sh[c] + threadIdx.x;
        double v = (s[0] + s[128]) + (s[64] + s[192]);
        for (int off = 32; off > 0; off >>= 1)
            v += __shfl_down(v, off, 64);
        out[c] = v;
    }
}

// Image position of a halo row: the global slot's position plus the periodic
// shift recorded at the build (positions are not re-wrapped between builds).
__device__ __forceinline__ void row_image(const double* __restrict__ x, const double* __restrict__ y,
                                          const double* __restrict__ z, double lx, double ly, double lz,
                                          int row, int& gs, double& xx, double& yy, double& zz) {
    gs = row & kRowSlotMask;
    const int code = static_cast<unsigned>(row) >> kRowSlotBits;
    xx = x[gs] + shift_of(code, 0, lx);
    yy = y[gs] + shift_of(code, 1, ly);
    zz = z[gs] + shift_of(code, 2, lz);
}

// Centre of brick b (FP64), the reference point of the FP32 relative
// coordinates of the mixed kernels.
__device__ __forceinline__ void brick_centre(int b, const int nb[3], const int bdim[3], const int nc[3],
                                             const double cs[3], double& cx, double& cy, double& cz) {
    const int bz = b % nb[2], by = (b / nb[2]) % nb[1], bx = b / (nb[1] * nb[2]);
    const int ox = bx * bdim[0], oy = by * bdim[1], oz = bz * bdim[2];
    cx = (ox + 0.5 * min(bdim[0], nc[0] - ox)) * cs[0];
    cy = (oy + 0.5 * min(bdim[1], nc[1] - oy)) * cs[1];
    cz = (oz + 0.5 * min(bdim[2], nc[2] - oz)) * cs[2];
}

// What a thread of a brick pair kernel loads ahead of the halo barrier. The
// kernels used to find the halo size, then the rows, then the positions, and
// after the barrier the atom's row header, then its list: five dependent trips
// to memory of ~1 us each before the first pair, most of a small system's
// force call. The rows are read without waiting for the halo's size (the table
// always holds kHaloCap entries; those past the halo are not used), and the
// row header and first two list groups while the positions are on their way.
struct AtomRow {
    int li; // the atom, brick-local
    int h;  // which of its threads this is
    int qs; // its own halo row
    int ng; // list groups
};

// Thread t's atom with tpa (1, 2 or 4) threads per atom in adjacent lanes; a
// thread past the brick's atoms takes the last one's row header and uses none
// of it.
__device__ __forceinline__ AtomRow atom_row(const uint16_t* __restrict__ self16, const int* __restrict__ numneigh,
                                            int a0, int nat, int tpa, int t) {
    AtomRow r;
    r.li = t >> (tpa >> 1);
    r.h = t & (tpa - 1);
    r.qs = 0;
    r.ng = 0;
    if (r.li < nat) {
        r.qs = self16[a0 + r.li];
        r.ng = (numneigh[a0 + r.li] + kGroup - 1) / kGroup;
    } else {
        r.li = 0;
    }
    return r;
}

// Index (16-byte groups from the brick's list) of the k-th group of this
// thread, clamped to the atom's last one (to group 0 of an empty row: the
// brick's rows always exist while it has atoms).
__device__ __forceinline__ int group_at(const AtomRow& r, int nat, int k, int tpa) {
    return __umul24(min(r.h + k * tpa, max(r.ng - 1, 0)), nat) + r.li;
}

// Systems of at most this many bricks leave CUs with one workgroup or none, so
// their force call is the latency of one brick: the wide kernels put more
// threads on it. Beyond, workgroups share the CUs, which the narrow ones do
// better, the FP64 LJ + Coulomb kernel first. Launches, narrow / wide:
//   FP64 LJ: 216 bricks 16.4 / 12.6 us, 252 24.7 / 15.9, 343 20.5 / 18.3,
//   448 22.5 / 23.0, 640 37.7 / 37.7;
//   FP64 LJ + Coulomb: 125 bricks 24.6 / 20.8, 288 25.5 / 27.2, 343 30.3 / 34.7,
//   1,134 64 / 76;
//   mixed LJ + Coulomb: 125 bricks 17.5 / 14.0, 288 19.2 / 16.1, 343 20.4 / 19.2,
//   1,134 32.6 / 30.0.
// One line for all, where none of them loses.
constexpr int kWideBricks = 256; // one brick per CU

// Small-grid pair kernels: kSmallLanes consecutive lanes share an atom, lane k
// taking entries k, k + kSmallLanes, ... of its row. Those systems are a few
// hundred atoms (or a thin box), where one thread per atom is a serial chain
// of ~80 neighbours on a handful of wavefronts (216 atoms, FP64 with energy
// and virial: 29.7 us a launch, against 6.3 us with 16 lanes).
constexpr int kSmallLanes = 16;

// Sum over an atom's kSmallLanes lanes, in every one of them.
template <class T>
__device__ __forceinline__ void small_lane_sum(T& v) {
#pragma unroll
    for (int off = kSmallLanes / 2; off > 0; off >>= 1)
        v += __shfl_xor(v, off, 64);
}

// Inclusive prefix sum over the 64 lanes (DPP row shifts, then the row
// broadcasts of lanes 15 and 31).
__device__ __forceinline__ int wave_inclusive_sum(int x) {
    x += __builtin_amdgcn_update_dpp(0, x, 0x111, 0xf, 0xf, true); // row_shr:1
    x += __builtin_amdgcn_update_dpp(0, x, 0x112, 0xf, 0xf, true); // row_shr:2
    x += __builtin_amdgcn_update_dpp(0, x, 0x114, 0xf, 0xf, true); // row_shr:4
    x += __builtin_amdgcn_update_dpp(0, x, 0x118, 0xf, 0xf, true); // row_shr:8
    x += __builtin_amdgcn_update_dpp(0, x, 0x142, 0xa, 0xf, false); // row_bcast:15 -> rows 1, 3
    x += __builtin_amdgcn_update_dpp(0, x, 0x143, 0xc, 0xf, false); // row_bcast:31 -> rows 2, 3
    return x;
}

// Unpack entry u (0..7) of an 8-wide group of 16-bit halo rows.
__device__ __forceinline__ int group_entry(const uint4& g, int u) {
    const unsigned long long lo = g.x | (static_cast<unsigned long long>(g.y) << 32);
    const unsigned long long hi = g.z | (static_cast<unsigned long long>(g.w) << 32);
    return static_cast<int>(((u < 4 ? lo : hi) >> (16 * (u & 3))) & 0xffffu);
}

} // namespace atvh
