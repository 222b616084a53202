// sfh_wg.hpp -- building blocks of the per-surface workgroup kernels (the batched stage kernel
// and the adjoint kernel): workgroups of 1024 threads on one surface of N <= 1024 nodes, thread t owns
// node t, the pair loops are those of sfh_sym.hpp.  Everything a surface needs besides its matrix lives
// in LDS (BLds); reductions are workgroup-local.
#pragma once
#include "sfh_kernels.hpp"
#include "sfh_fft.hpp"
#include "sfh_physics.hpp"
#include "sfh_circ.hpp"

namespace sfh {

constexpr int kBT = kBatchThreads;   // threads per workgroup
constexpr int kBW = kBT / 64;         // waves per workgroup
constexpr int kBK = 8;                // Krylov vectors per GMRES cycle
constexpr int kBR = kBK + 2;          // reduction slots: kBK + 1 dots and one norm

struct BLds {
    // three transform fields, one after the other
    double2 fa[kBatchMaxN];
    double2 fb[kBatchMaxN];
    union {
        double2 zp[kBatchMaxN];
        double2 fc[kBatchMaxN];   // wg_derivatives' third field, before Z' is there
    };
    double2 tw[kBatchMaxN];
    NodeTrig tr[kBatchMaxN];
    double diag[kBatchMaxN];
    double vs[kBatchMaxN];
    double part[kBT];
    double red[kBW][kBR];
    double sums[kBR];
    double H[kBK + 1][kBK];
    double cs[kBK], sn[kBK], g[kBK + 1], y[kBK];
    double col[kBK + 2];
    double scal[4];
    double prered[kBW][2 * kPreModes + 1];   // film: wg_precondition's sums and coefficients
    double precoef[2 * kPreModes + 1];
};

// Sums each of the C slots of v over the workgroup into L.sums (all threads take part).
template <int C>
__device__ inline void bsum(const double (&v)[C], BLds& L) {
    const int t = threadIdx.x, lane = t & 63, w = t >> 6;
#pragma unroll
    for (int i = 0; i < C; ++i) {
        const double s = wave_sum(v[i]);
        if (lane == 0) L.red[w][i] = s;
    }
    __syncthreads();
    if (t < C) {
        double acc = 0.0;
#pragma unroll
        for (int q = 0; q < kBW; ++q) acc += L.red[q][t];
        L.sums[t] = acc;
    }
    __syncthreads();
}

__device__ inline double bsum1(double v, BLds& L) {
    const double a[1] = {v};
    bsum(a, L);
    return L.sums[0];
}

// L.sums[i] = sum over the workgroup of V[i] * w for i <= j < kBK, and L.sums[j + 1] = |w|^2 with_norm.  Four values
// share a wave's lane swaps (reduce_lanes), and only the groups that hold something run: with the rotation by one
// rsqrt and the first norms formed together, a solve of one step of N = 128 takes 17 us in place of 23.
__device__ inline void bsum_dots(const double (&V)[kBK + 1], double w, int j, bool with_norm, BLds& L) {
    static_assert(kBK == 8, "two groups of four, and the norm of the last step");
    const int t = threadIdx.x, wv = t >> 6, last = j + (with_norm ? 1 : 0);
    const auto value = [&](int i) { return i <= j ? V[i] * w : (i == last ? w * w : 0.0); };
#pragma unroll
    for (int g = 0; g < 2; ++g) {
        if (4 * g <= last) {
            const double v[4] = {value(4 * g), value(4 * g + 1), value(4 * g + 2), value(4 * g + 3)};
            reduce_lanes(v, &L.red[wv][4 * g]);
        }
    }
    if (last == kBK) {
        const double s = wave_sum(w * w);
        if ((t & 63) == 0) L.red[wv][kBK] = s;
    }
    __syncthreads();
    if (t <= last) {
        double acc = 0.0;
#pragma unroll
        for (int q = 0; q < kBW; ++q) acc += L.red[q][t];
        L.sums[t] = acc;
    }
    __syncthreads();
}

// Register-array element i (runtime i) without dynamic register indexing.
template <int K>
__device__ inline double rget(const double (&V)[K], int i) {
    double r = V[0];
#pragma unroll
    for (int u = 1; u < K; ++u) r = (i == u) ? V[u] : r;
    return r;
}
template <int K>
__device__ inline void rset(double (&V)[K], int i, double x) {
#pragma unroll
    for (int u = 0; u < K; ++u) V[u] = (i == u) ? x : V[u];
}

struct PairConst {
    double c;     // coefficient of Im(Z'_k cot) (createM.cuh:52, :78)
    double ci;    // coefficient of the image term (:87-88)
    double eh, ehi;
    int image;
};

// The film's preconditioner of a surface: modes < 0 when none is used.
struct Precond {
    int modes;
    double height;
};

// P^{-1} v for the flat film's matrix P (film_eigenvalue): 2 v + the first modes' (1/lam_m - 2)
// projections.  Thread t < n holds v_t (the others 0) and gets the result (the others 0); L.tw holds the
// twiddles exp(-2 pi i t / n).
__device__ inline double wg_precondition(double v, int n, const Precond& pre, BLds& L) {
    const int t = threadIdx.x, lane = t & 63, wv = t >> 6;
    const double2 w = L.tw[min(t, n - 1)];
    const double c = w.x, s = -w.y;
    const double s0 = wave_sum(v);
    if (lane == 0) L.prered[wv][0] = s0;
    double c1 = 1.0, s1 = 0.0, cm = c, sm = s;
    for (int m = 1; m <= pre.modes; ++m) {
        const double a = wave_sum(v * cm), b = wave_sum(v * sm);
        if (lane == 0) {
            L.prered[wv][2 * m - 1] = a;
            L.prered[wv][2 * m] = b;
        }
        const double cn = 2.0 * c * cm - c1, sn = 2.0 * c * sm - s1;   // the next mode, by recurrence
        c1 = cm;
        s1 = sm;
        cm = cn;
        sm = sn;
    }
    __syncthreads();
    if (t <= 2 * pre.modes) {
        double a = 0.0;
#pragma unroll
        for (int q = 0; q < kBW; ++q) a += L.prered[q][t];
        const int m = (t + 1) >> 1;
        L.precoef[t] = a * (m == 0 ? 1.0 : 2.0) / n * (1.0 / film_eigenvalue(n, m, pre.height) - 2.0);
    }
    __syncthreads();
    double z = 2.0 * v + L.precoef[0];
    c1 = 1.0;
    s1 = 0.0;
    cm = c;
    sm = s;
    for (int m = 1; m <= pre.modes; ++m) {
        z += L.precoef[2 * m - 1] * cm + L.precoef[2 * m] * sm;
        const double cn = 2.0 * c * cm - c1, sn = 2.0 * c * sm - s1;
        c1 = cm;
        s1 = sm;
        cm = cn;
        sm = sn;
    }
    return t < n ? z : 0.0;
}

// The first residual rhs - A x and its squared norm, when the caller has formed them.
struct FirstResidual {
    bool given;
    double r, rr;
};

// Restarted GMRES on A x = rhs over the workgroup; x (thread t < n holds x_t) is updated in
// place.  With a preconditioner the basis is that of A P^{-1} and x += P^{-1} V y, so residual and
// tolerance are those of A x = rhs as without.  x_zero: x is known to be 0 (the first residual is rhs, no product needed); with a
// given first residual none is needed either.  Returns the number of
// Arnoldi steps; *unconv is set when tol_abs was not reached.
// sums keeps a linear by-product of mv (pair sums that mv forms anyway): keep(j) its value for the product of basis
// vector j, fresh() replaces the value for x by the last product's, add(k, y) adds that of the correction.
struct NoSums {
    __device__ void keep(int) {}
    __device__ void fresh() {}
    __device__ void add(int, const double*) {}
};

template <class MV, class Sums>
__device__ int wg_gmres(MV&& mv, Sums&& sums, int n, double rhs, double& x, bool x_zero, double tol_abs, int cycles,
                        BLds& L, int* unconv, const FirstResidual first = {}, const Precond pre = {-1, 0.0}) {
    const int t = threadIdx.x;
    const bool own = t < n;
    int total = 0;
    for (int cyc = 0; cyc < cycles; ++cyc) {
        double r = own ? rhs : 0.0, rr = first.rr;
        if (cyc == 0 && first.given) {
            r = own ? first.r : 0.0;   // the caller formed rhs - M x already
        } else if (!(x_zero && cyc == 0)) {
            if (own) L.vs[t] = x;
            __syncthreads();
            const double w = mv();
            sums.fresh();
            r = own ? rhs - w : 0.0;
        }
        if (cyc > 0 || !first.given) rr = bsum1(r * r, L);
        const double beta = sqrt(rr);
        if (!(beta > tol_abs)) return total;
        double V[kBK + 1];
#pragma unroll
        for (int i = 0; i <= kBK; ++i) V[i] = 0.0;
        V[0] = r / beta;
        if (t == 0) L.g[0] = beta;
        int k = 0;
        bool conv = false;
        for (int j = 0; j < kBK; ++j) {
            double u = rget(V, j);
            if (pre.modes >= 0) u = wg_precondition(u, n, pre, L);
            if (own) L.vs[t] = u;
            __syncthreads();
            double w = mv();
            sums.keep(j);
            // classical Gram-Schmidt ...
            bsum_dots(V, w, j, false, L);
            if (t == 0)
                for (int i = 0; i <= j; ++i) L.col[i] = L.sums[i];
#pragma unroll
            for (int i = 0; i <= kBK; ++i)
                if (i <= j) w -= L.sums[i] * V[i];
            // ... with one re-orthogonalisation; |w|^2 after it by Pythagoras (the second-pass
            // coefficients are O(eps |w|), so the subtraction does not cancel)
            __syncthreads();
            bsum_dots(V, w, j, true, L);
            double hh = L.sums[j + 1];
#pragma unroll
            for (int i = 0; i <= kBK; ++i) {
                if (i <= j) {
                    const double c2 = L.sums[i];
                    w -= c2 * V[i];
                    hh -= c2 * c2;
                }
            }
            const double hn = sqrt(fmax(hh, 0.0));
            rset(V, j + 1, (own && hn > 0.0) ? w / hn : 0.0);
            if (t == 0) {   // new Hessenberg column, previous rotations, new rotation
                double* col = L.col;
                for (int i = 0; i <= j; ++i) col[i] += L.sums[i];
                col[j + 1] = hn;
                for (int i = 0; i < j; ++i) {
                    const double a0 = L.cs[i] * col[i] + L.sn[i] * col[i + 1];
                    const double a1 = -L.sn[i] * col[i] + L.cs[i] * col[i + 1];
                    col[i] = a0;
                    col[i + 1] = a1;
                }
                // the entries are of the order of |M| or underflow together with the residual: no scaling
                const double sq = col[j] * col[j] + col[j + 1] * col[j + 1], inv = sq > 0.0 ? rsqrt(sq) : 0.0;
                const double cj = sq > 0.0 ? col[j] * inv : 1.0;
                const double sj = col[j + 1] * inv;
                L.cs[j] = cj;
                L.sn[j] = sj;
                col[j] = sq * inv;
                for (int i = 0; i <= j; ++i) L.H[i][j] = col[i];
                L.g[j + 1] = -sj * L.g[j];
                L.g[j] = cj * L.g[j];
                L.scal[0] = fabs(L.g[j + 1]);
                L.scal[1] = hn;
            }
            __syncthreads();
            k = j + 1;
            if (L.scal[0] <= tol_abs || L.scal[1] == 0.0) {
                conv = L.scal[0] <= tol_abs;
                break;
            }
        }
        // x += V_k y with H_k y = g (upper triangular after the rotations)
        if (t == 0) {
            for (int i = k - 1; i >= 0; --i) {
                double s = L.g[i];
                for (int l = i + 1; l < k; ++l) s -= L.H[i][l] * L.y[l];
                L.y[i] = s / L.H[i][i];
            }
        }
        __syncthreads();
        sums.add(k, L.y);
        if (pre.modes >= 0) {
            double u = 0.0;
#pragma unroll
            for (int i = 0; i < kBK; ++i)
                if (i < k) u += L.y[i] * V[i];
            u = wg_precondition(u, n, pre, L);
            if (own) x += u;
        } else if (own) {
#pragma unroll
            for (int i = 0; i < kBK; ++i)
                if (i < k) x += L.y[i] * V[i];
        }
        __syncthreads();
        total += k;
        if (conv) return total;
    }
    if (unconv) *unconv = 1;
    return total;
}

// Node values produced by the derivative phase (valid on threads t < n).
struct NodeVals {
    double2 z, zp, zpp;
    double phi, b;
};

// Spectral derivatives of one surface in LDS (Derivatives.cuh:310-384): Z' and Z'' from ONE
// forward transform of Z - 2 pi j / N, Re Phi' from a second, both at once, then the three inverse ones at once; also fills L.tw (twiddles),
// L.tr (half-angle table) and L.zp.
__device__ inline NodeVals wg_derivatives(const SurfDesc& d, const double2* __restrict__ tw_all,
                                          const double2* __restrict__ Zin, const double* __restrict__ Pin,
                                          const Phys& ph, BLds& L) {
    const int n = d.n, off = d.voff, t = threadIdx.x;
    const bool own = t < n;
    const double twopi_n = 2.0 * kPi / n;
    for (int i = t; i < n; i += kBT) L.tw[i] = tw_all[d.twoff + i];
    const double plin = -(1 + ph.rho) * kPi * ph.U / n;   // Derivatives.cuh:286
    double2* const fc = L.fc;   // Phi, then its derivative
    NodeVals v;
    v.z = make_double2(0.0, 0.0);
    v.phi = 0.0;
    if (own) {
        v.z = Zin[off + t];
        v.phi = Pin[off + t];
        L.tr[t] = node_trig(v.z);
        const int i = lds_index(d, t);
        L.fa[i] = make_double2(v.z.x - twopi_n * (double)t, v.z.y);   // :285,317
        fc[i] = make_double2(v.phi - plin * (double)t, 0.0);
    }
    __syncthreads();
    fft_dit<2>(L.fa, 2 * kBatchMaxN, d, -1, L.tw);   // fa and fc
    __syncthreads();
    for (int i = t; i < n; i += kBT) {
        const double2 c = L.fa[i];
        L.fb[i] = second_mult(c, i, n);
        L.fa[i] = first_mult(c, i, n);
        fc[i] = first_mult(fc[i], i, n);
    }
    __syncthreads();
    fft_dif<3>(L.fa, kBatchMaxN, d, +1, L.tw);   // fa, fb and fc
    __syncthreads();
    v.zp = make_double2(1.0, 0.0);
    v.zpp = make_double2(0.0, 0.0);
    v.b = 0.0;
    if (own) {
        const int i = lds_index(d, t);
        const double2 a = L.fa[i], c = L.fb[i];
        const double sc2 = 4.0 * kPi * kPi / ((double)n * n);
        v.zp = make_double2(a.x * twopi_n + twopi_n, a.y * twopi_n);   // :323, :374
        v.zpp = make_double2(c.x * sc2, c.y * sc2);                    // :321
        v.b = fc[i].x * twopi_n;   // :324, BaseBoundaryIntegrator.cuh:299
        if (ph.U != 0) v.b += plin;                 // :380-383
    }
    __syncthreads();
    if (own) L.zp[t] = v.zp;
    __syncthreads();
    return v;
}

// Pair constants and the diagonal M_kk (createM.cuh:43-92) into L.diag.
__device__ inline PairConst wg_diagonal(const Phys& ph, const NodeVals& v, int n, BLds& L) {
    const bool water = ph.kind == 0;
    PairConst pc;
    pc.c = water ? 0.25 * (1 - ph.rho) / kPi : 0.25 / kPi;
    pc.ci = 0.25 / kPi;
    pc.eh = exp(ph.depth);
    pc.ehi = exp(-ph.depth);
    pc.image = ph.image;
    if ((int)threadIdx.x < n) {
        const double2 r = cdiv(v.zpp, v.zp);
        double dg = (water ? 0.5 * (1 + ph.rho) : 0.5) + pc.c * r.y;
        if (ph.image) dg -= pc.ci * cot64(0.0, v.z.y + ph.depth).y;
        L.diag[threadIdx.x] = dg;
    }
    __syncthreads();
    return pc;
}

// In-LDS spectral first derivative of a field already stored at L.fa[lds_index(j)]; the result is
// left at the same slots (unscaled).  conj_mult applies the adjoint table (every first-derivative
// multiplier is imaginary, so the adjoint is the negated table).
__device__ inline void wg_first_derivative(const SurfDesc& d, BLds& L, bool adjoint) {
    const int n = d.n, t = threadIdx.x;
    __syncthreads();
    fft_dit(L.fa, d, -1, L.tw);
    __syncthreads();
    for (int i = t; i < n; i += kBT) {
        const double2 c = first_mult(L.fa[i], i, n);
        L.fa[i] = adjoint ? make_double2(-c.x, -c.y) : c;
    }
    __syncthreads();
    fft_dif(L.fa, d, +1, L.tw);
    __syncthreads();
}

}  // namespace sfh
