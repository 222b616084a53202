// spectral.hip -- tangential derivatives of the multi-workgroup path as circulant products.
//
// Replaces ZPhiDerivative::exec (CuSuperHelium/Derivatives.cuh:310-384) and the mu' derivative of
// BaseBoundaryIntegrator.cuh:201-203 (FftDerivative::exec, Derivatives.cuh:189-257).  Forward
// DFT, multiplier table (utilities.cuh:119-147 first derivative, :185-199 second), inverse DFT is
// a circulant linear map of the samples:
//   y_k = sum_j c[(k - j) mod n] v_j,   c_q = sum_i m_i exp(+2 pi i i q / n),
// c being the inverse transform of the multipliers (complex for the first derivative, whose table
// is not conjugate-symmetric at n/2 and n/2 + 1; real for the second).  The tables are built once
// per node count in extended precision on the host.
//
// An in-LDS FFT of one field is a chain of dependent LDS passes inside a single workgroup, so at
// n = 2048 it takes ~4 us each way on one CU while the rest of the GPU idles.  As circulant
// products the three derivatives of a right-hand side (Z', Z'', Re Phi') are 7 n^2 multiply-adds
// spread over all CUs, and every row is summed inside one workgroup (no cross-workgroup reduction).
#include "sfh_circ.hpp"
#include "sfh_gmres.hpp"

namespace sfh {

// Z' (field scale 2 pi / n, plus the slope of the linear part), Z'' (4 pi^2 / n^2) and
// b = Re Phi' (2 pi / n, plus the uniform-flow term) for CircGeo::ROWS rows of one surface;
// also the rows' half-angle table, and with GMRES the rows' initial guess and the solve's
// control block.  grid = (ceil(max n / ROWS), surfaces).
template <int TC, int TR>
__global__ __launch_bounds__(TC * TR) void zphi_circ_kernel(const SurfDesc* __restrict__ sd,
                                                        const double* __restrict__ circ,
                                                        const double2* __restrict__ Z,
                                                        const double* __restrict__ phi,
                                                        double2* __restrict__ Zp, double2* __restrict__ Zpp,
                                                        double* __restrict__ b, double* __restrict__ work,
                                                        Phys ph, int* __restrict__ status,
                                                        NodeTrig* __restrict__ trig, GmArgs gm, int gm_on) {
    using G = CircGeo<TC, TR>;
    constexpr int kCircRows = G::ROWS;
    __shared__ struct alignas(16) {
        double zx[G::CHUNK], zy[G::CHUNK];   // samples of the chunk: Z minus its linear part
        double p[G::CHUNK];                  // phi minus its linear part
        double ar[G::WIN], ai[G::WIN];       // first-derivative kernel over the chunk's window of k - j
        double b[G::WIN];                    // second-derivative kernel
        double red[G::NT / 64][5 * kCR];
    } L;
    const SurfDesc d = sd[blockIdx.y];
    const int n = d.n, off = d.voff;
    const int k0 = blockIdx.x * kCircRows;
    if (k0 >= n) return;
    const int t = threadIdx.x;
    // re-arm the surface's interchange flag / GMRES control block for the solve that follows
    if (blockIdx.x == 0 && t == 0) {
        if (status) status[2 * blockIdx.y] = 0;
        if (gm_on) {
            GmCtl* c = reinterpret_cast<GmCtl*>(gm.ctl) + blockIdx.y;
            c->done = 0;
            c->iters = 0;
            c->refine_iters = 0;
            if (gm.stage > 0 && gm.hvalid[gm.stage - 1] < kHistDepth) c->fill_iters = 0;
            if (gm.stage == 1) c->most = 0;
        }
    }
    const double* c1r = circ + d.coff;
    const double* c1i = c1r + n;
    const double* c2 = c1i + n;
    const double xs = 2.0 * kPi / n;                       // Derivatives.cuh:285,317
    const double plin = -(1 + ph.rho) * kPi * ph.U / n;    // Derivatives.cuh:286
    // the own rows' inputs of the half-angle table and of the initial guess (threads t < kCircRows),
    // loaded first, so that the table is formed while the samples arrive
    const int kt = min(k0 + t, n - 1);
    double2 zk = {0.0, 0.0};
    int hv = 0;
    double hk[kHistDepth] = {}, solk = 0.0;
    if (t < kCircRows) {
        zk = Z[off + kt];
        if (gm_on) {
            hv = gm.stage > 0 ? gm.hvalid[gm.stage - 1] : 0;
            if (hv > 0) {
                const double* h0 = gm.hist + (long long)(gm.stage - 1) * kHistDepth * gm.total + off + kt;
#pragma unroll
                for (int l = 0; l < kHistDepth; ++l) hk[l] = l < hv ? h0[(long long)l * gm.total] : 0.0;
            } else {
                solk = gm.sol[off + kt];
            }
        }
    }
    double acc[5][kCR];   // Re Z', Im Z', Re Z'', Im Z'', Re Phi'
#pragma unroll
    for (int i = 0; i < 5; ++i)
#pragma unroll
        for (int r = 0; r < kCR; ++r) acc[i][r] = 0.0;
    double ysum = 0.0;   // film: the mean height, for the preconditioner of the solve
    const int c0 = kCC * (t % TC), u0 = c0 + kCR * (TR - 1 - t / TC);   // first column, first window entry
    for (int j0 = 0; j0 < n; j0 += G::CHUNK) {
        const int jn = min(G::CHUNK, n - j0);
        if (j0 > 0) __syncthreads();   // the previous chunk has been consumed
        {   // every load of the chunk in flight before the first LDS store
            double2 zv[G::PER];
            double pv[G::PER], ar[G::WPER], ai[G::WPER], bv[G::WPER];
#pragma unroll
            for (int e = 0; e < G::PER; ++e) {
                const int j = min(j0 + t + G::NT * e, n - 1);
                zv[e] = Z[off + j];
                pv[e] = phi[off + j];
            }
            int q[G::WPER];
            circ_entries<G>(k0, j0, n, q);
#pragma unroll
            for (int e = 0; e < G::WPER; ++e) {
                ar[e] = c1r[q[e]];
                ai[e] = c1i[q[e]];
                bv[e] = c2[q[e]];
            }
            if (j0 == 0 && t < kCircRows && k0 + t < n) {   // while they arrive
                const int k = k0 + t;
                if (trig) trig[off + k] = node_trig(zk);
                // GMRES initial guess of this RK stage: its mu over the previous steps extrapolated
                // (error O(dt^5) once five are kept), else the last solve's mu
                if (gm_on) gm.x[off + k] = hv > 0 ? extrapolate_values(hk, hv) : solk;
            }
#pragma unroll
            for (int e = 0; e < G::PER; ++e) {
                const int c = t + G::NT * e, j = j0 + c, i = circ_at(c);
                const bool in = c < jn;
                L.zx[i] = in ? zv[e].x - 2 * kPi * (double)j / n : 0.0;
                L.zy[i] = in ? zv[e].y : 0.0;
                L.p[i] = in ? pv[e] - plin * (double)j : 0.0;
                ysum += in ? zv[e].y : 0.0;
            }
#pragma unroll
            for (int e = 0; e < G::WPER; ++e) {
                const int u = t + G::NT * e;
                if (u < G::CHUNK + G::ROWS) {
                    L.ar[circ_at(u)] = ar[e];
                    L.ai[circ_at(u)] = ai[e];
                    L.b[circ_at(u)] = bv[e];
                }
            }
        }
        __syncthreads();
        if (c0 < jn) {
            double x[kCC], y[kCC], p[kCC], w[kCC + kCR];
            circ_samples(L.zx, c0, x);
            circ_samples(L.zy, c0, y);
            circ_samples(L.p, c0, p);
            circ_kernel(L.ar, u0, w);
            circ_fma(w, x, acc[0]);
            circ_fma(w, y, acc[1]);
            circ_fma(w, p, acc[4]);
            circ_kernel(L.ai, u0, w);
            circ_fma(w, y, acc[0], -1.0);
            circ_fma(w, x, acc[1]);
            circ_kernel(L.b, u0, w);
            circ_fma(w, x, acc[2]);
            circ_fma(w, y, acc[3]);
        }
    }
#pragma unroll
    for (int i = 0; i < 5; ++i) reduce_lanes(acc[i], &L.red[t >> 6][kCR * i]);
    __syncthreads();
    if (t < kCircRows && k0 + t < n) {
        const int k = k0 + t;
        double v[5];
#pragma unroll
        for (int i = 0; i < 5; ++i) {
            v[i] = 0.0;
#pragma unroll
            for (int w = 0; w < TC / 64; ++w) v[i] += L.red[t / kCR * (TC / 64) + w][kCR * i + t % kCR];
        }
        Zp[off + k] = make_double2(v[0] * xs + xs, v[1] * xs);                 // :323,374
        const double s2 = 4.0 * kPi * kPi / ((double)n * n);                  // :321
        Zpp[off + k] = make_double2(v[2] * s2, v[3] * s2);
        double r = v[4] * xs;                                                  // :324, :299
        if (ph.U != 0) r += -(1 + ph.rho) * kPi * ph.U / n;                   // :380-383
        b[off + k] = r;
        work[off + k] = r;
    }
    if (gm_on && gm.pre && blockIdx.x == 0) {
        __shared__ double red4[G::NT / 64];
        const double height = block_sum<G::NT / 64>(ysum, red4) / n + ph.depth;
        if (t == 0) {
            GmCtl* c = reinterpret_cast<GmCtl*>(gm.ctl) + blockIdx.y;
            c->height = height;
            c->pre_modes = film_modes(n, height);
        }
    }
}

// mu' = D1 mu * 2 pi / n (BaseBoundaryIntegrator.cuh:201-203), mu real, for CircGeo::ROWS rows of one
// surface.  grid = (ceil(max n / ROWS), surfaces).
template <int TC, int TR>
__global__ __launch_bounds__(TC * TR) void mu_circ_kernel(const SurfDesc* __restrict__ sd,
                                                          const double* __restrict__ circ,
                                                          const double* __restrict__ mu,
                                                          double2* __restrict__ mup) {
    using G = CircGeo<TC, TR>;
    __shared__ struct alignas(16) {
        double m[G::CHUNK];
        double ar[G::WIN], ai[G::WIN];
        double red[G::NT / 64][2 * kCR];
    } L;
    const SurfDesc d = sd[blockIdx.y];
    const int n = d.n, off = d.voff;
    const int k0 = blockIdx.x * G::ROWS;
    if (k0 >= n) return;
    const int t = threadIdx.x;
    const double* c1r = circ + d.coff;
    const double* c1i = c1r + n;
    double re[kCR], im[kCR];
#pragma unroll
    for (int r = 0; r < kCR; ++r) re[r] = im[r] = 0.0;
    const int c0 = kCC * (t % TC), u0 = c0 + kCR * (TR - 1 - t / TC);
    for (int j0 = 0; j0 < n; j0 += G::CHUNK) {
        const int jn = min(G::CHUNK, n - j0);
        if (j0 > 0) __syncthreads();
        {   // every load of the chunk in flight before the first LDS store
            double mv[G::PER], ar[G::WPER], ai[G::WPER];
#pragma unroll
            for (int e = 0; e < G::PER; ++e) mv[e] = mu[off + min(j0 + t + G::NT * e, n - 1)];
            int q[G::WPER];
            circ_entries<G>(k0, j0, n, q);
#pragma unroll
            for (int e = 0; e < G::WPER; ++e) {
                ar[e] = c1r[q[e]];
                ai[e] = c1i[q[e]];
            }
#pragma unroll
            for (int e = 0; e < G::PER; ++e) {
                const int c = t + G::NT * e;
                L.m[circ_at(c)] = c < jn ? mv[e] : 0.0;
            }
#pragma unroll
            for (int e = 0; e < G::WPER; ++e) {
                const int u = t + G::NT * e;
                if (u < G::CHUNK + G::ROWS) {
                    L.ar[circ_at(u)] = ar[e];
                    L.ai[circ_at(u)] = ai[e];
                }
            }
        }
        __syncthreads();
        if (c0 < jn) {
            double x[kCC], w[kCC + kCR];
            circ_samples(L.m, c0, x);
            circ_kernel(L.ar, u0, w);
            circ_fma(w, x, re);
            circ_kernel(L.ai, u0, w);
            circ_fma(w, x, im);
        }
    }
    reduce_lanes(re, &L.red[t >> 6][0]);
    reduce_lanes(im, &L.red[t >> 6][kCR]);
    __syncthreads();
    if (t < G::ROWS && k0 + t < n) {
        const double xs = 2.0 * kPi / n;
        double a = 0.0, c = 0.0;
#pragma unroll
        for (int w = 0; w < TC / 64; ++w) {
            const double* r = L.red[t / kCR * (TC / 64) + w];
            a += r[t % kCR];
            c += r[kCR + t % kCR];
        }
        mup[off + k0 + t] = make_double2(a * xs, c * xs);
    }
}

// (TC, TR) that SFH_WITH_CIRC (solver.hip) chooses
#define SFH_CIRC_INSTANCES(TC, TR)                                                                                 \
    template __global__ void zphi_circ_kernel<TC, TR>(const SurfDesc*, const double*, const double2*, const double*, \
                                                      double2*, double2*, double*, double*, Phys, int*, NodeTrig*,  \
                                                      GmArgs, int);                                                 \
    template __global__ void mu_circ_kernel<TC, TR>(const SurfDesc*, const double*, const double*, double2*);
SFH_CIRC_INSTANCES(64, 4)
SFH_CIRC_INSTANCES(256, 1)
SFH_CIRC_INSTANCES(512, 1)

}  // namespace sfh
