// velocity.hip -- surface velocity, Bernoulli right-hand side and RK4 stage update, fused.
//
// Replaces createVelocityMatrices / createHeliumVelocityMatrices (CuSuperHelium/
// WaterVelocities.cuh:38-107), which materialise the N x N complex V1 (64 MB at N = 2048,
// written twice per RHS), the Zgemv pair of VelocityCalculator::calculateVelocities (:205-242),
// conjugate_vector, compute_rhs_phi_expression / compute_rhs_helium_phi_expression
// (createM.cuh:96-117,171-211) and the Zaxpy / add_k_vectors stages of
// AutonomousRungeKuttaStepper::runStep (AutonomousRungeKuttaStepper.cuh:123-361).
//
// A workgroup owns kPairRows nodes k.  Every thread takes the columns j = t (mod 256) (each
// workgroup starting at its own offset), loads the node's half-angle table entry and mu_j once per
// column and adds its terms to the sums of all the workgroup's rows,
//   S_k = sum_j mu_j cot((z_k - z_j)/2)      Si_k = sum_j mu_j cot((z_k - conj z_j)/2 + i h),
// the sums are reduced over the workgroup, and one thread per row finishes
//   w_k = V2_k mu'_k + V1_kk mu_k + i (-1/4pi) S_k [+ i (1/4pi) Si_k]
//   V2_k = i / (2 pi Z'_k),  V1_kk = i (-1/4pi) Z''_k / Z'_k^2 [+ i (1/4pi) cot(i (y_k + h))] +- 1/(2 Z'_k)
//   q_k = conj(w_k),  dphi_k = Bernoulli(q_k, y_k),  then the RK4 stage of node k.
//
// GMRES solves with products from cotangent sums form S_k themselves and finish in gm_close_mu_kernel; this kernel
// is for LU, and for GMRES with the stored matrix.
#include "sfh_circ.hpp"
#include "sfh_physics.hpp"

namespace sfh {

template <int R>
__global__ __launch_bounds__(256) void velocity_stage_kernel(const SurfDesc* __restrict__ sd,
                                                             const NodeTrig* __restrict__ trig,
                                                             const double2* __restrict__ Z,
                                                             const double2* __restrict__ Zp,
                                                             const double2* __restrict__ Zpp,
                                                             const double* __restrict__ mu,
                                                             const double2* __restrict__ mup,
                                                             Phys ph, StageCtl ctl) {
    const SurfDesc d = sd[blockIdx.y];
    const int n = d.n;
    const int k0 = blockIdx.x * R;
    if (k0 >= n) return;
    const int t = threadIdx.x;
    const double2* z = Z + d.voff;
    const double* m = mu + d.voff;
    const NodeTrig* tr = trig + d.voff;
    // createM.cuh:104 reads V1[1].real() (lower velocity of node 1) in the rho * q1.q2 term; with
    // rho != 0 every workgroup also sums node 1 (entry R of the row arrays; each surface its own)
    const bool quirk = ph.kind == 0 && ph.rho_quirk && ph.rho != 0.0 && n > 1;
    const double h = ph.depth, eh = exp(h), ehi = exp(-h);
    const int shift = (int)(((long long)blockIdx.x * 64) % n);
    NodeTrig tk[R + 1];
#pragma unroll
    for (int r = 0; r < R; ++r) tk[r] = tr[min(k0 + r, n - 1)];
    tk[R] = tr[min(1, n - 1)];
    double sx[R + 1], sy[R + 1], ix[R], iy[R];
#pragma unroll
    for (int r = 0; r <= R; ++r) sx[r] = sy[r] = 0.0;
#pragma unroll
    for (int r = 0; r < R; ++r) ix[r] = iy[r] = 0.0;
    // the finishing threads' own inputs (and those of node 1 for the quirk), loaded before the
    // sweep so that their latency overlaps it
    const int kt = min(k0 + min(t, R - 1), n - 1), gt = d.voff + kt;
    double2 zp_t = {0.0, 0.0}, zpp_t = {0.0, 0.0}, mup_t = {0.0, 0.0}, z_t = {0.0, 0.0};
    double m_t = 0.0;
    StageIn st{};
    double2 zp_1 = {0.0, 0.0}, zpp_1 = {0.0, 0.0}, mup_1 = {0.0, 0.0};
    double m_1 = 0.0, y_1 = 0.0;
    if (t < R) {
        zp_t = Zp[gt];
        zpp_t = Zpp[gt];
        z_t = z[kt];
        st = stage_load(ctl, gt);
        mup_t = mup[gt];
        m_t = m[kt];
        if (quirk) {
            const int g1 = d.voff + 1;
            zp_1 = Zp[g1];
            zpp_1 = Zpp[g1];
            mup_1 = mup[g1];
            m_1 = m[1];
            y_1 = z[1].y;
        }
    }
    for (int j0 = 0; j0 < n; j0 += 8 * 256) {
        NodeTrig tj[8];
        double mj[8];
        int jc[8];
#pragma unroll
        for (int e = 0; e < 8; ++e) {   // unconditional (clamped) loads: no branch between them
            int j = min(j0 + t + 256 * e, n - 1) + shift;
            if (j >= n) j -= n;
            jc[e] = j;
            tj[e] = tr[j];
            mj[e] = m[j];
        }
#pragma unroll
        for (int e = 0; e < 8; ++e) {
            const int c = t + 256 * e;
            if (j0 + c >= n) break;
            const int j = jc[e];
#pragma unroll
            for (int r = 0; r < R; ++r) {
                if (k0 + r >= n) break;
                if (j == k0 + r) continue;
                const CotParts cp = cot_parts(tk[r], tj[e]);
                const double w = mj[e] * cp.id;
                sx[r] += w * cp.p;
                sy[r] -= w * cp.q;
                if (ph.image) {
                    const CotParts cq = cot_image_parts(tk[r], tj[e], eh, ehi);
                    const double wi = mj[e] * cq.id;
                    ix[r] += wi * cq.p;
                    iy[r] -= wi * cq.q;
                }
            }
            if (quirk && j != 1) {
                const CotParts cp = cot_parts(tk[R], tj[e]);
                const double w = mj[e] * cp.id;
                sx[R] += w * cp.p;
                sy[R] -= w * cp.q;
            }
        }
    }
    __shared__ double red[2 * R * 256];
    __shared__ double so[2 * R], io[2 * R], qo[2];
    {
        double v[2 * R];
#pragma unroll
        for (int r = 0; r < R; ++r) {
            v[r] = sx[r];
            v[R + r] = sy[r];
        }
        rows_reduce<2 * R>(v, red, so);
    }
    if (ph.image) {
        double v[2 * R];
#pragma unroll
        for (int r = 0; r < R; ++r) {
            v[r] = ix[r];
            v[R + r] = iy[r];
        }
        rows_reduce<2 * R>(v, red, io);
    }
    if (quirk) {
        const double v[2] = {sx[R], sy[R]};
        rows_reduce<2>(v, red, qo);
    }
    if (t >= R || k0 + t >= n) return;
    double2 q1, q2;
    velocity_from_sums(ph, zp_t, zpp_t, mup_t, m_t, z_t.y, so[t], so[R + t], ph.image ? io[t] : 0.0,
                       ph.image ? io[R + t] : 0.0, q1, q2);
    double2 q1q = q1;
    if (quirk && k0 + t != 1) {
        double2 u2;
        velocity_from_sums(ph, zp_1, zpp_1, mup_1, m_1, y_1, qo[0], qo[1], 0.0, 0.0, q1q, u2);
    }
    finish_node(ph, ctl, d.voff + k0 + t, z_t, zp_t, zpp_t, m_t, q1, q2, q1q, st);
}

// Surfaces of up to 256 nodes, not with the rho quirk: a wave has 4 rows and all their columns, 16 pairs per lane, and its
// own sums.  With 256 threads across the columns a workgroup had 4 pairs per thread and was mostly first loads, reductions
// and the rows' end: 64 surfaces of 256 nodes 39 us with velocity_stage_kernel<4>, 16 here.  mu' of the rows is formed
// here too, from a window of the derivative's kernel in LDS that the workgroup's 16 rows share: 15.8 -> 16.2 us there and
// 4.9 -> 5.9 for one surface, for a launch of 4.5 us less.
template <int NA>
__global__ __launch_bounds__(256) void velocity_small_kernel(const SurfDesc* __restrict__ sd, const NodeTrig* __restrict__ trig,
                                                             const double2* __restrict__ Z, const double2* __restrict__ Zp,
                                                             const double2* __restrict__ Zpp, const double* __restrict__ mu,
                                                             const double* __restrict__ circ, Phys ph, StageCtl ctl) {
    constexpr int WIN = kSmallRows + kSmallNodes;   // entry u of the window is c[(k0 + kSmallRows - 1 - u) mod n], k0 the first row
    __shared__ double red[4][4 * NA + 8], c1[2][WIN];
    const SurfDesc d = sd[blockIdx.y];
    const int n = d.n, lane = threadIdx.x & 63, w = threadIdx.x >> 6;
    const int k0 = blockIdx.x * kSmallRows + 4 * w;
    if (blockIdx.x * kSmallRows >= n) return;   // the whole workgroup: the waves meet below
    const NodeTrig* tr = trig + d.voff;
    const double eh = exp(ph.depth), ehi = exp(-ph.depth);
    const double* c1r = circ + d.coff;
    double cw[2][2];
    {
        int q = ((int)blockIdx.x * kSmallRows + kSmallRows - 1 - (int)threadIdx.x) % n;
        if (q < 0) q += n;
        const int q2 = (q + n - 256 % n) % n;
        cw[0][0] = c1r[q];
        cw[0][1] = c1r[n + q];
        cw[1][0] = c1r[q2];
        cw[1][1] = c1r[n + q2];
    }
    NodeTrig tk[4], tj[4];
    double mj[4];
#pragma unroll
    for (int e = 0; e < 4; ++e) {
        const int j = min(lane + 64 * e, n - 1);
        tj[e] = tr[j];
        mj[e] = mu[d.voff + j];
    }
#pragma unroll
    for (int r = 0; r < 4; ++r) tk[r] = tr[min(k0 + r, n - 1)];
    const int k = k0 + lane, g = d.voff + min(k, n - 1);
    const bool own = lane < 4 && k < n;
    double2 zp = {1.0, 0.0}, zpp = {0.0, 0.0}, z = {0.0, 0.0};
    double m = 0.0;
    StageIn st{};
    if (own) {
        zp = Zp[g];
        zpp = Zpp[g];
        z = Z[g];
        st = stage_load(ctl, g);
        m = mu[g];
    }
#pragma unroll
    for (int h = 0; h < 2; ++h) {
        c1[h][threadIdx.x] = cw[0][h];
        if (threadIdx.x < kSmallRows) c1[h][256 + threadIdx.x] = cw[1][h];
    }
    double acc[4 * NA + 8];
#pragma unroll
    for (int q = 0; q < 4 * NA + 8; ++q) acc[q] = 0.0;
#pragma unroll
    for (int e = 0; e < 4; ++e) {
        const int j = lane + 64 * e;
        if (j >= n) break;
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            if (j == k0 + r) continue;
            const CotParts cp = cot_parts(tk[r], tj[e]);
            const double v = mj[e] * cp.id;
            acc[r] += v * cp.p;
            acc[4 + r] -= v * cp.q;
            if constexpr (NA == 4) {
                const CotParts cq = cot_image_parts(tk[r], tj[e], eh, ehi);
                const double vi = mj[e] * cq.id;
                acc[8 + r] += vi * cq.p;
                acc[12 + r] -= vi * cq.q;
            }
        }
    }
    __syncthreads();
#pragma unroll
    for (int e = 0; e < 4; ++e) {
        const int j = lane + 64 * e;
        if (j >= n) break;
        const int u = kSmallRows - 1 - 4 * w + j;
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            acc[4 * NA + r] += c1[0][u - r] * mj[e];
            acc[4 * NA + 4 + r] += c1[1][u - r] * mj[e];
        }
    }
    reduce_lanes(acc, red[w]);
    __syncthreads();
    if (!own) return;
    const double* S = red[w] + lane;
    const double xs = 2.0 * kPi / n;
    const double2 mp = {S[4 * NA] * xs, S[4 * NA + 4] * xs};
    double2 q1, q2;
    velocity_from_sums(ph, zp, zpp, mp, m, z.y, S[0], S[4], NA == 4 ? S[NA == 4 ? 8 : 0] : 0.0, NA == 4 ? S[NA == 4 ? 12 : 0] : 0.0, q1, q2);
    finish_node(ph, ctl, g, z, zp, zpp, m, q1, q2, q1, st);
}
template __global__ void velocity_small_kernel<2>(const SurfDesc*, const NodeTrig*, const double2*, const double2*, const double2*,
                                                  const double*, const double*, Phys, StageCtl);
template __global__ void velocity_small_kernel<4>(const SurfDesc*, const NodeTrig*, const double2*, const double2*, const double2*,
                                                  const double*, const double*, Phys, StageCtl);

// rows per workgroup the solver may launch with (chosen per surface size by the autotuner)
#define SFH_VELOCITY_INSTANCES(R)                                                                                  \
    template __global__ void velocity_stage_kernel<R>(const SurfDesc*, const NodeTrig*, const double2*,                \
                                                      const double2*, const double2*, const double*, const double2*, \
                                                      Phys, StageCtl);
SFH_VELOCITY_INSTANCES(1)
SFH_VELOCITY_INSTANCES(2)
SFH_VELOCITY_INSTANCES(4)

}  // namespace sfh
