// sfh_pairs.hpp -- cotangent sums of a vector over the nodes of one surface, for a few rows per group of 256 threads:
//   S_k = sum_{j != k} v_j cot((z_k - z_j)/2),   film also   Si_k = sum_{j != k} v_j cot((z_k - conj z_j)/2 + i h).
// The product with the dipole matrix, (M v)_k = M_kk v_k + c Im(Z'_k S_k) - ci Im Si_k, and the surface velocity are local
// combinations of these sums (createM.cuh:43-92, WaterVelocities.cuh:38-107), and the sums are linear in v.
#pragma once
#include "sfh_circ.hpp"
#include "sfh_physics.hpp"

namespace sfh {

constexpr int kSumRows = 4;      // rows of a group
constexpr int kSumCols = 8;      // columns per thread and pass
constexpr int kSumPass = 256 * kSumCols;

// Half-angle table entries of this thread's columns j0 + t + 256 e (clamped), tg = thread in its group of 256.
__device__ __forceinline__ void sum_columns(const NodeTrig* __restrict__ tr, int n, int j0, int tg, NodeTrig (&tj)[kSumCols]) {
#pragma unroll
    for (int e = 0; e < kSumCols; ++e) tj[e] = tr[min(j0 + tg + 256 * e, n - 1)];
}

// acc[a * kSumRows + r] += this thread's columns' terms of sum a (Re S, Im S, Re Si, Im Si) of row k0 + r; value(j) = v_j.
template <int NA, class F>
__device__ __forceinline__ void sum_pass(const NodeTrig (&tk)[kSumRows], const NodeTrig (&tj)[kSumCols], int n, int k0, int j0,
                                         int tg, double eh, double ehi, F&& value, double (&acc)[NA * kSumRows]) {
#pragma unroll
    for (int e = 0; e < kSumCols; ++e) {
        const int j = j0 + tg + 256 * e;
        if (j >= n) break;
        const double v = value(j);
#pragma unroll
        for (int r = 0; r < kSumRows; ++r) {
            if (j == k0 + r) continue;
            const CotParts cp = cot_parts(tk[r], tj[e]);
            const double w = v * cp.id;
            acc[r] += w * cp.p;
            acc[kSumRows + r] -= w * cp.q;
            if constexpr (NA == 4) {
                const CotParts cq = cot_image_parts(tk[r], tj[e], eh, ehi);
                const double wi = v * cq.id;
                acc[2 * kSumRows + r] += wi * cq.p;
                acc[3 * kSumRows + r] -= wi * cq.q;
            }
        }
    }
}

// The transposed product's sum of each row (reverse mode): with w_k = v_k Z'_k,
//   (M^T v)_j = M_jj v_j - c Im sum_{k != j} w_k cot((z_j - z_k)/2) - ci Im sum_{k != j} v_k cot((z_j - conj z_k)/2 + i h),
// the image part being symmetric; acc[r] is minus the sums' contribution.  value(j) = v_j.
template <bool FILM, class F>
__device__ __forceinline__ void transpose_pass(const NodeTrig (&tk)[kSumRows], const NodeTrig (&tj)[kSumCols],
                                               const double2 (&zj)[kSumCols], int n, int k0, int j0, int tg, double c, double ci,
                                               double eh, double ehi, F&& value, double (&acc)[kSumRows]) {
#pragma unroll
    for (int e = 0; e < kSumCols; ++e) {
        const int j = j0 + tg + 256 * e;
        if (j >= n) break;
        const double v = value(j);
        const double wx = c * v * zj[e].x, wy = c * v * zj[e].y, vi = ci * v;
#pragma unroll
        for (int r = 0; r < kSumRows; ++r) {
            if (j == k0 + r) continue;
            const CotParts cp = cot_parts(tk[r], tj[e]);
            acc[r] += cp.id * (wx * cp.q - wy * cp.p);
            if constexpr (FILM) {
                const CotParts cq = cot_image_parts(tk[r], tj[e], eh, ehi);
                acc[r] += vi * (cq.q * cq.id);
            }
        }
    }
}

// The group's sums of its rows, in LDS red (one row of NA * kSumRows values per wave; the caller synchronises after
// sum_store): row r's sum a.
template <int NA>
__device__ inline void sum_store(const double (&acc)[NA * kSumRows], double (*red)[NA * kSumRows]) {
    reduce_lanes(acc, red[threadIdx.x >> 6]);
}
template <int NA>
__device__ inline double sum_total(const double (*red)[NA * kSumRows], int group, int r, int a) {
    double s = 0.0;
#pragma unroll
    for (int w = 0; w < 4; ++w) s += red[4 * group + w][a * kSumRows + r];
    return s;
}

// Constants of the matrix (createM.cuh:52, :78, :87-88).
struct SumConst {
    double c, ci, eh, ehi;
};

template <int NA>
__device__ inline double product_of_sums(const double (&s)[NA], const SumConst& k, double2 zp, double diag, double v) {
    double w = k.c * (zp.x * s[1] + zp.y * s[0]) + diag * v;
    if constexpr (NA == 4) w -= k.ci * s[3];
    return w;
}

}  // namespace sfh
