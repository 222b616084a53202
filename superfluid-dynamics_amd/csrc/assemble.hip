// assemble.hip -- dipole matrix M = I/2 + K in FP64, one wave per row.
//
// Replaces createMKernel (CuSuperHelium/createM.cuh:43-63) and createFiniteDepthMKernel
// (:65-92), which run one thread per entry on 16x16 blocks.  Here a workgroup owns kPairRows
// rows: every thread takes the columns j = t (mod 256), loads the node's half-angle table entry
// (NodeTrig) once and forms the entries of all the workgroup's rows with it, so each table entry
// is read once per kPairRows rows, a thread has kPairRows independent entries in flight per
// column, and a wave's stores to one row are 512 contiguous bytes.  cot comes from the table with
// no transcendental call per entry.
//   M_kk = (1+rho)/2 + (1-rho)/(4 pi) Im(Z''_k / Z'_k)                       (water)
//   M_kj = (1-rho)/(4 pi) Im(Z'_k cot((z_k - z_j)/2))
//   helium: rho -> 0 and, with finite depth h, the image terms
//   M_kk -= Im(cot(i (y_k + h)))/(4 pi),  M_kj -= Im(cot((z_k - conj z_j)/2 + i h))/(4 pi)
//
// With the GMRES solver the kernel also starts the solve: while it writes row k it accumulates
// (M x0)_k and stores r0_k = b_k - (M x0)_k as the first (unnormalised) basis vector; the first
// Arnoldi step normalises it.
#include "sfh_circ.hpp"

namespace sfh {

// The rows of M (stored as T: FP64, or FP32 rounded from the FP64 entries; not stored when M is
// null) and, with gm_on, r = b - M x in FP64 for x = the initial guess, or (residual pass) x = the
// solution, whose own rows the pass then copies into the initial guess of the next solve.
template <typename T, int R>
__device__ inline void assemble_rows(const SurfDesc* __restrict__ sd, const NodeTrig* __restrict__ trig,
                                     const double2* __restrict__ Z, const double2* __restrict__ Zp,
                                     const double2* __restrict__ Zpp, T* __restrict__ M, const Phys& ph,
                                     const GmArgs& gm, int gm_on, bool residual) {
    const SurfDesc d = sd[blockIdx.y];
    const int n = d.n;
    const int k0 = blockIdx.x * R;
    if (k0 >= n) return;
    const int t = threadIdx.x;
    if (residual && blockIdx.x == 0 && t == 0) reinterpret_cast<int*>(gm.ctl)[kGmCtlInts * blockIdx.y] = 0;   // done
    const NodeTrig* tr = trig + d.voff;
    const double* x0 = gm_on ? (residual ? gm.sol : gm.x) + d.voff : nullptr;
    const bool water = ph.kind == 0;
    const double c = water ? 0.25 * (1 - ph.rho) / kPi : 0.25 / kPi;
    const double ci = 0.25 / kPi;
    const double h = ph.depth, eh = exp(h), ehi = exp(-h);
    // the rows' constants (the same in every thread)
    NodeTrig tk[R];
    double czx[R], czy[R];   // c Z'_k
    double diag[R];
#pragma unroll
    for (int r = 0; r < R; ++r) {
        const int k = min(k0 + r, n - 1);
        tk[r] = tr[k];
        const double2 zpk = Zp[d.voff + k];
        czx[r] = c * zpk.x;
        czy[r] = c * zpk.y;
        const double2 q = cdiv(Zpp[d.voff + k], zpk);
        diag[r] = (water ? 0.5 * (1 + ph.rho) : 0.5) + c * q.y;
        if (ph.image) diag[r] -= ci * cot64(0.0, Z[d.voff + k].y + h).y;
    }
    // b of the rows whose residual the threads t < R store at the end
    const double bt = (gm_on && t < R) ? gm.b[d.voff + min(k0 + t, n - 1)] : 0.0;
    T* Mk = M ? M + d.moff + (long long)k0 * n : nullptr;
    double acc[R];
#pragma unroll
    for (int r = 0; r < R; ++r) acc[r] = 0.0;
    // columns in passes of 8 per thread: a pass loads the table entries of its 8 columns (all in
    // flight) and then forms their entries of every row.  Each workgroup starts its sweep at its
    // own column offset (a multiple of 64): rows are n * 8 bytes apart, so workgroups sweeping in
    // lockstep from column 0 would all store to the same few memory channels at once.
    const int shift = (int)(((long long)blockIdx.x * 64) % n);
    for (int j0 = 0; j0 < n; j0 += 8 * 256) {
        NodeTrig tj[8];
        double xj[8];
        int jc[8];
#pragma unroll
        for (int e = 0; e < 8; ++e) {   // unconditional (clamped) loads: no branch between them
            int j = min(j0 + t + 256 * e, n - 1) + shift;
            if (j >= n) j -= n;
            jc[e] = j;
            tj[e] = tr[j];
            xj[e] = gm_on ? x0[j] : 0.0;
        }
#pragma unroll
        for (int e = 0; e < 8; ++e) {
            if (j0 + t + 256 * e >= n) break;
            const int j = jc[e];
#pragma unroll
            for (int r = 0; r < R; ++r) {
                const int k = k0 + r;
                if (k >= n) break;
                double v;
                if (j == k) {
                    v = diag[r];
                } else {
                    // c Im(Z'_k cot) = id (c y'_k p - c x'_k q)
                    const CotParts cp = cot_parts(tk[r], tj[e]);
                    v = cp.id * (czy[r] * cp.p - czx[r] * cp.q);
                    if (ph.image) {
                        const CotParts ci2 = cot_image_parts(tk[r], tj[e], eh, ehi);
                        v += ci * (ci2.q * ci2.id);
                    }
                }
                if (Mk) Mk[(long long)r * n + j] = static_cast<T>(v);
                acc[r] += v * xj[e];
            }
        }
    }
    if (!gm_on) return;
    __shared__ double red[(R < 4 ? 4 : R) * 256];
    __shared__ double out[R];
    rows_reduce<R>(acc, red, out);
    if (t < R && k0 + t < n) {
        gm.V[(long long)(gm.m + 1) * d.voff + k0 + t] = bt - out[t];
        if (residual) gm.x[d.voff + k0 + t] = x0[k0 + t];
    }
}

template <int R>
__global__ __launch_bounds__(256) void assemble64_kernel(const SurfDesc* __restrict__ sd,
                                                         const NodeTrig* __restrict__ trig,
                                                         const double2* __restrict__ Z,
                                                         const double2* __restrict__ Zp,
                                                         const double2* __restrict__ Zpp,
                                                         double* __restrict__ M, Phys ph,
                                                         GmArgs gm, int gm_on) {
    assemble_rows<double, R>(sd, trig, Z, Zp, Zpp, M, ph, gm, gm_on, false);
}

// Mixed precision: M stored in FP32, r0 = b - M x0 from the FP64 entries.
template <int R>
__global__ __launch_bounds__(256) void assemble32_kernel(const SurfDesc* __restrict__ sd,
                                                         const NodeTrig* __restrict__ trig,
                                                         const double2* __restrict__ Z,
                                                         const double2* __restrict__ Zp,
                                                         const double2* __restrict__ Zpp,
                                                         float* __restrict__ M, Phys ph, GmArgs gm) {
    assemble_rows<float, R>(sd, trig, Z, Zp, Zpp, M, ph, gm, 1, false);
}

// Mixed precision, refinement: r = b - M mu in FP64, matrix-free (the assembly's entries, not
// stored), into the first basis vector; mu becomes the next solve's initial guess, and the
// control block is re-armed (done = 0) for that solve.
template <int R>
__global__ __launch_bounds__(256) void residual64_kernel(const SurfDesc* __restrict__ sd,
                                                         const NodeTrig* __restrict__ trig,
                                                         const double2* __restrict__ Z,
                                                         const double2* __restrict__ Zp,
                                                         const double2* __restrict__ Zpp, Phys ph, GmArgs gm) {
    assemble_rows<double, R>(sd, trig, Z, Zp, Zpp, static_cast<double*>(nullptr), ph, gm, 1, true);
}

// Surfaces of up to 256 nodes (LU): the derivatives, the half-angle table and the matrix rows in one launch.  A wave has 4
// rows and all their columns, 16 products and 16 entries per lane, and only the rows' own lanes form the diagonal; a
// workgroup's 16 rows share the samples, the table (formed anew by every workgroup) and the windows of the derivatives'
// kernels in LDS.  With 256 threads across the columns a workgroup had 4 entries per thread and was mostly first loads and
// row constants: 64 surfaces of 256 nodes 34 us with assemble64_kernel<4>, 16 with whole rows; that and the
// derivatives' launch 16.8 + 6.5 us, 19.2 together; one surface of 256 4.9 + 4.8, 6.3 together.
__global__ __launch_bounds__(256) void form_small_kernel(const SurfDesc* __restrict__ sd, const double* __restrict__ circ,
                                                         const double2* __restrict__ Z, const double* __restrict__ phi,
                                                         double2* __restrict__ Zp, double2* __restrict__ Zpp,
                                                         double* __restrict__ b, double* __restrict__ work,
                                                         double* __restrict__ M, NodeTrig* __restrict__ trig, Phys ph,
                                                         int* __restrict__ status) {
    constexpr int WIN = kSmallRows + kSmallNodes;   // entry u of a window is c[(kb + kSmallRows - 1 - u) mod n], kb the first row
    __shared__ double zx[kSmallNodes], zy[kSmallNodes], p[kSmallNodes];   // samples minus their linear parts
    __shared__ double ts[kSmallNodes], tc[kSmallNodes], te[kSmallNodes], ti[kSmallNodes];
    __shared__ double cw[3][WIN], red[4][20];
    const SurfDesc d = sd[blockIdx.y];
    const int n = d.n, off = d.voff, t = threadIdx.x, lane = t & 63, w = t >> 6;
    const int kb = blockIdx.x * kSmallRows, k0 = kb + 4 * w;
    if (kb >= n) return;   // the whole workgroup
    if (blockIdx.x == 0 && t == 0) status[2 * blockIdx.y] = 0;   // re-armed for the solve that follows
    const double xs = 2.0 * kPi / n;                       // Derivatives.cuh:285,317
    const double plin = -(1 + ph.rho) * kPi * ph.U / n;    // Derivatives.cuh:286
    const double2 zt = Z[off + min(t, n - 1)];
    const double pt = phi[off + min(t, n - 1)];
    int q = (kb + kSmallRows - 1 - t) % n;
    if (q < 0) q += n;
    const int q2 = (q + n - 256 % n) % n;
    double c[2][3];
#pragma unroll
    for (int i = 0; i < 3; ++i) {
        c[0][i] = circ[d.coff + i * n + q];
        c[1][i] = circ[d.coff + i * n + q2];
    }
    const NodeTrig own = node_trig(zt);
    zx[t] = t < n ? zt.x - 2 * kPi * (double)t / n : 0.0;
    zy[t] = t < n ? zt.y : 0.0;
    p[t] = t < n ? pt - plin * (double)t : 0.0;
    ts[t] = own.s;
    tc[t] = own.c;
    te[t] = own.e;
    ti[t] = own.ei;
#pragma unroll
    for (int i = 0; i < 3; ++i) {
        cw[i][t] = c[0][i];
        if (t < kSmallRows) cw[i][256 + t] = c[1][i];
    }
    __syncthreads();
    double acc[20];   // 4 rows each of Re Z', Im Z', Re Z'', Im Z'', Re Phi'
#pragma unroll
    for (int i = 0; i < 20; ++i) acc[i] = 0.0;
#pragma unroll
    for (int e = 0; e < 4; ++e) {
        const int j = lane + 64 * e;
        if (j >= n) break;
        const double x = zx[j], y = zy[j], f = p[j];
        const int u = kSmallRows - 1 - 4 * w + j;
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            const double wr = cw[0][u - r], wi = cw[1][u - r], w2 = cw[2][u - r];
            acc[r] += wr * x;
            acc[r] -= wi * y;
            acc[4 + r] += wr * y;
            acc[4 + r] += wi * x;
            acc[8 + r] += w2 * x;
            acc[12 + r] += w2 * y;
            acc[16 + r] += wr * f;
        }
    }
    reduce_lanes(acc, red[w]);
    __syncthreads();
    if (k0 >= n) return;
    const double* S = red[w];
    double* Mk = M + d.moff + (long long)k0 * n;
    const double cm = ph.kind == 0 ? 0.25 * (1 - ph.rho) / kPi : 0.25 / kPi, ci = 0.25 / kPi;
    const double h = ph.depth, eh = exp(h), ehi = exp(-h);
    if (lane < 4 && k0 + lane < n) {
        const int k = k0 + lane, g = off + k;
        const double s2 = 4.0 * kPi * kPi / ((double)n * n);                  // Derivatives.cuh:321
        const double2 zp = {S[lane] * xs + xs, S[4 + lane] * xs}, zpp = {S[8 + lane] * s2, S[12 + lane] * s2};
        Zp[g] = zp;                                                           // :323,374
        Zpp[g] = zpp;
        double r = S[16 + lane] * xs;                                         // :324, :299
        if (ph.U != 0) r += -(1 + ph.rho) * kPi * ph.U / n;                   // :380-383
        b[g] = r;
        work[g] = r;
        trig[g] = NodeTrig{ts[k], tc[k], te[k], ti[k]};
        double v = (ph.kind == 0 ? 0.5 * (1 + ph.rho) : 0.5) + cm * cdiv(zpp, zp).y;
        if (ph.image) v -= ci * cot64(0.0, zy[k] + h).y;
        Mk[(long long)lane * n + k] = v;
    }
    NodeTrig tk[4];
    double2 zk[4];
#pragma unroll
    for (int r = 0; r < 4; ++r) {
        const int k = min(k0 + r, n - 1);
        tk[r] = NodeTrig{ts[k], tc[k], te[k], ti[k]};
        zk[r] = {S[r] * xs + xs, S[4 + r] * xs};
    }
#pragma unroll
    for (int e = 0; e < 4; ++e) {
        const int j = lane + 64 * e;
        if (j >= n) break;
        const NodeTrig tj = {ts[j], tc[j], te[j], ti[j]};
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            if (k0 + r >= n) break;
            if (j == k0 + r) continue;
            const CotParts cp = cot_parts(tk[r], tj);
            double v = cp.id * (cm * zk[r].y * cp.p - cm * zk[r].x * cp.q);
            if (ph.image) {
                const CotParts cq = cot_image_parts(tk[r], tj, eh, ehi);
                v += ci * (cq.q * cq.id);
            }
            Mk[(long long)r * n + j] = v;
        }
    }
}

// rows per workgroup the solver may launch with (chosen per surface size by the autotuner)
#define SFH_ASSEMBLE_INSTANCES(R)                                                                             \
    template __global__ void assemble64_kernel<R>(const SurfDesc*, const NodeTrig*, const double2*, const double2*, \
                                                  const double2*, double*, Phys, GmArgs, int);                    \
    template __global__ void assemble32_kernel<R>(const SurfDesc*, const NodeTrig*, const double2*, const double2*, \
                                                  const double2*, float*, Phys, GmArgs);                          \
    template __global__ void residual64_kernel<R>(const SurfDesc*, const NodeTrig*, const double2*, const double2*, \
                                                  const double2*, Phys, GmArgs);
SFH_ASSEMBLE_INSTANCES(1)
SFH_ASSEMBLE_INSTANCES(2)
SFH_ASSEMBLE_INSTANCES(4)

}  // namespace sfh
