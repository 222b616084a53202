// sfh_circ.hpp -- building blocks of the circulant products of the spectral derivatives
//   y_k = sum_j c[(k - j) mod n] v_j
// for a few rows k of one surface per workgroup, samples and a window of the kernel staged in LDS.
//
// A thread takes 4 neighbouring columns of 8 neighbouring rows (32 products per kernel), for which it
// reads 4 samples and 11 kernel entries from LDS: 12 bytes per row and column in
// zphi_circ_kernel, against 36 when each wave had rows of its own and LDS bandwidth bounded it.  The 8
// rows' sums meet by register swaps between halves and rows of 16 lanes (reduce_lanes), a third of the
// instructions of one wave sum each.  zphi_circ_kernel, before and after: N = 2048 10.2 -> 8.0 us (of which 5 are launch, first loads and the last reductions), N = 4096 film
// 27.4 -> 15.1, 64 surfaces of N = 256 38.5 -> 8.7; mu_circ_kernel of the latter 9.8 -> 4.7.
#pragma once
#include "sfh_kernels.hpp"

namespace sfh {

constexpr int kCC = 4;   // columns per thread
constexpr int kCR = 8;   // rows per thread

// TC threads side by side over the columns of a chunk, TR groups of rows.
template <int TC, int TR>
struct CircGeo {
    static constexpr int NT = TC * TR, CHUNK = kCC * TC, ROWS = kCR * TR;
    static constexpr int PER = (CHUNK + NT - 1) / NT;               // staged samples per thread
    static constexpr int WPER = (CHUNK + ROWS - 1 + NT - 1) / NT;   // staged kernel entries per thread
    static constexpr int WIN = (CHUNK + ROWS + 31) / 32 * 32;
    static_assert(TC % 64 == 0 && CHUNK % NT == 0, "whole waves per row group, whole passes");
};

// Position of element i of a staged array.  A thread reads 16-byte pairs at a stride of 32 bytes from its
// neighbour's: every second run of 16 pairs has its even and odd pairs exchanged, so 16 lanes read 16
// different banks.
__device__ inline int circ_at(int i) { return i ^ ((i >> 4) & 2); }
__device__ inline double2 circ_pair(const double* a, int i) { return *reinterpret_cast<const double2*>(a + circ_at(i)); }

// Window entry u of rows k0 .. k0 + ROWS - 1 and the chunk at j0 is c[(k0 + ROWS - 1 - j0 - u) mod n]: row r,
// column c of the chunk read entry ROWS - 1 - r + c.  The kernel indices of the entries u = t + NT e that a
// thread stages (entries beyond the window get valid indices too).
template <class G>
__device__ inline void circ_entries(int k0, int j0, int n, int (&q)[G::WPER]) {
    int r = (k0 + G::ROWS - 1 - j0 - (int)threadIdx.x) % n;
    if (r < 0) r += n;
    const int step = G::NT % n;
#pragma unroll
    for (int e = 0; e < G::WPER; ++e) {
        q[e] = r;
        r -= step;
        if (r < 0) r += n;
    }
}

// 4 samples and 11 (of 12) window entries of this thread.
__device__ inline void circ_samples(const double* a, int c0, double (&v)[kCC]) {
#pragma unroll
    for (int h = 0; h < kCC / 2; ++h) {
        const double2 x = circ_pair(a, c0 + 2 * h);
        v[2 * h] = x.x;
        v[2 * h + 1] = x.y;
    }
}
__device__ inline void circ_kernel(const double* a, int u0, double (&v)[kCC + kCR]) {
#pragma unroll
    for (int h = 0; h < (kCC + kCR) / 2; ++h) {
        const double2 x = circ_pair(a, u0 + 2 * h);
        v[2 * h] = x.x;
        v[2 * h + 1] = x.y;
    }
}
// acc_r += sum_c kernel(r, c) v_c
__device__ inline void circ_fma(const double (&w)[kCC + kCR], const double (&v)[kCC], double (&acc)[kCR], double sign = 1.0) {
#pragma unroll
    for (int c = 0; c < kCC; ++c) {
        const double x = sign * v[c];
#pragma unroll
        for (int r = 0; r < kCR; ++r) acc[r] += w[c + kCR - 1 - r] * x;
    }
}

// Sums of NV values per lane over a wave into out[0..NV) (LDS).  A swap of the upper half of one register
// with the lower half of another turns two sums over 64 lanes into one over 32 of both, and likewise for
// rows of 16 lanes: NV (1/2 + 1/4) swaps and adds, then row sums of NV / 4 values.
__device__ inline double swap_add32(double a, double b) {
    const auto lo = __builtin_amdgcn_permlane32_swap(__double2loint(a), __double2loint(b), false, false);
    const auto hi = __builtin_amdgcn_permlane32_swap(__double2hiint(a), __double2hiint(b), false, false);
    return __hiloint2double(hi[0], lo[0]) + __hiloint2double(hi[1], lo[1]);
}
__device__ inline double swap_add16(double a, double b) {
    const auto lo = __builtin_amdgcn_permlane16_swap(__double2loint(a), __double2loint(b), false, false);
    const auto hi = __builtin_amdgcn_permlane16_swap(__double2hiint(a), __double2hiint(b), false, false);
    return __hiloint2double(hi[0], lo[0]) + __hiloint2double(hi[1], lo[1]);
}
template <int NV>
__device__ inline void reduce_lanes(const double (&v)[NV], double* out) {
    static_assert(NV % 4 == 0, "groups of four values");
    const int lane = threadIdx.x & 63, row = lane >> 4;
#pragma unroll
    for (int q = 0; q < NV / 4; ++q) {
        double s = swap_add16(swap_add32(v[4 * q], v[4 * q + 1]), swap_add32(v[4 * q + 2], v[4 * q + 3]));
        s += dpp_double<0xB1>(s);    // quad_perm [1,0,3,2]
        s += dpp_double<0x4E>(s);    // quad_perm [2,3,0,1]
        s += dpp_double<0x141>(s);   // row_half_mirror
        s += dpp_double<0x140>(s);   // row_mirror
        if ((lane & 15) == 0) out[4 * q + 2 * (row & 1) + (row >> 1)] = s;
    }
}

}  // namespace sfh
