// batched.hip -- persistent per-surface stage kernel for ensembles of independent surfaces
// (every N <= 1024): ONE launch per RK4 stage advances all surfaces.
//
// Workgroup b works on surface order[b]; the order is by decreasing N, so the in-order dispatch of
// workgroups schedules the largest surfaces first and the small ones fill the machine behind them.
// With as many surfaces as CUs a surface has one workgroup, which runs its whole right-hand side with no
// inter-workgroup synchronisation; with fewer, the largest surfaces have several, which share the pair sweeps and the
// products (sfh_cluster.hpp; SHARED).  The right-hand side is BaseBoundaryIntegralCalculator::runTimeStep
// (CuSuperHelium/BaseBoundaryIntegrator.cuh:137-314) for one member of the batch:
//   A  spectral derivatives in LDS: Z' and Z'' from ONE forward transform of Z - 2 pi j / N,
//      Phi' from a second (Derivatives.cuh:310-384), plus the per-node half-angle table;
//   B  the dipole matrix M = I/2 + K (createM.cuh:43-92) into HBM, in the order in which the sweeps visit it
//      (sfh_sym.hpp), FP64 or FP32 (FP64 entries rounded), and in the same pair loop M x for the warm start x (the first residual);
//   C  the solve M mu = b, warm-started from the surface's previous mu, with products of the stored matrix or
//      (as B's, without storing) of sums that the velocity needs anyway:
//        FP64  : GMRES on the FP64 matrix (classical Gram-Schmidt with one
//                re-orthogonalisation, restarted cycles of kBK vectors);
//        mixed : FP64 iterative refinement  r = b - M mu  with the residual evaluated
//                matrix-free in FP64 (same pair formula as the assembly), correction solves by
//                GMRES on the FP32 matrix (or on M itself); a correction whose GMRES residual plus
//                ||M - M32||_F |d| (bounded by 2^-24 ||M||_F) is within the tolerance ends the
//                refinement without another FP64 residual pass;
//   D  mu' (one more transform pair);
//   E  the cot-sum velocity, Bernoulli and the RK4 stage update (WaterVelocities.cuh:38-107,
//      createM.cuh:96-117, AutonomousRungeKuttaStepper.cuh:338-375).
//
// Thread t owns node t.  The pair loops (assembly, the matrix-free FP64 product, velocity) visit
// every unordered pair of nodes once in 64 x 64 tiles and give both rows of the pair their
// contribution (sfh_sym.hpp); a wave stores the entries it forms in rows of its own, so every store
// and every load of the stored product is one contiguous 512-byte (FP64) or 256-byte (FP32) row
// per wave, and node data is read from LDS without bank conflicts.
//
// Bounds: N = 1024 mixed water among 512 surfaces, one Arnoldi step, 293 us: derivatives 16, sweep of the warm start 132,
// sweep of the step 130, the rest of the solve 7, mu' 6, stage 2; the sweeps issue FP64 instructions back to back (150
// cycles for 64 pairs).
#include <type_traits>

#include "sfh_sym.hpp"

namespace sfh {

// The cotangent sums of the vector last multiplied, of the solution so far, and (in the matrix's place) of the basis.
template <int NA>
struct CotSums {
    double* basis;   // NA * n for each basis vector
    int n;
    double last[NA], sum[NA];
    __device__ void keep(int j) {
        const int t = threadIdx.x;
        if (t >= n) return;
#pragma unroll
        for (int a = 0; a < NA; ++a) basis[(size_t)(j * NA + a) * n + t] = last[a];
    }
    __device__ void fresh() {
#pragma unroll
        for (int a = 0; a < NA; ++a) sum[a] = last[a];
    }
    __device__ void add(int k, const double* y) {
        const int t = threadIdx.x;
        if (t >= n) return;
        for (int i = 0; i < k; ++i) {
            const double c = y[i];
#pragma unroll
            for (int a = 0; a < NA; ++a) sum[a] += c * basis[(size_t)(i * NA + a) * n + t];
        }
    }
};

template <bool MIXED, bool FILM, bool SHARED>
__global__ __launch_bounds__(1024) void batched_stage_kernel(BatchArgs a, Phys ph, StageCtl ctl) {
    constexpr bool stored = FILM;   // the matrix: see the assembly
    constexpr int NA = FILM ? 4 : 2;
    __shared__ BLds L;
    const int s = a.order[blockIdx.x];
    const SurfDesc d = a.sd[s];
    const int n = d.n, off = d.voff, t = threadIdx.x;
    const bool own = t < n;
    const double twopi_n = 2.0 * kPi / n;
    Cluster cl{1, 1, 0, 1, 0, false, nullptr, nullptr, nullptr};
    int ticket = 0;
    if constexpr (SHARED) cl.parts = a.parts[s];
    if (cl.parts > 1) {
        cl.launched = min(cl.parts, a.max_wgs);
        cl.xb = a.xbuf + a.xoff[s];
        cl.words = a.words + 16 * s;
        cl.failed = a.status + 2 * s + 1;
        if (t == 0) ticket = Cluster::add(cl.words, 1);
    }

    // ---------------------------------------------------------------- A: derivatives
    const NodeVals nv = wg_derivatives(d, a.tw_all, a.Zin, a.Pin, ph, L);
    const double2 zk = nv.z, zpk = nv.zp, zppk = nv.zpp;
    const double bk = nv.b;
    if (cl.parts > 1) {
        __shared__ int joined[2];
        if (t == 0) {
            cl.join(ticket);
            joined[0] = cl.rank;
            joined[1] = cl.members;
            if (cl.members == 0) cl.leave();
        }
        __syncthreads();
        cl.rank = __builtin_amdgcn_readfirstlane(joined[0]);
        cl.members = __builtin_amdgcn_readfirstlane(joined[1]);
        if (cl.members == 0) return;
    }
    const bool lead = cl.rank == 0;   // the one that stores what the others hold as well
    if (own && lead) {
        a.Zp[off + t] = zpk;
        a.Zpp[off + t] = zppk;
        a.b[off + t] = bk;
    }

    // warm start: this stage's mu extrapolated over the previous steps (error O(dt^5) once five
    // are kept), else the previous solve's mu
    double x = own ? a.mu[off + t] : 0.0;
    double* h0 = nullptr;
    int hv = 0;
    if (ctl.stage > 0 && a.hist) {
        hv = a.hvalid[(ctl.stage - 1) * a.nsurf + s];
        h0 = a.hist + (long long)(ctl.stage - 1) * kHistDepth * a.total + off;
        if (own && hv >= 1) x = extrapolate_history(h0 + t, a.total, hv);
    }

    // ---------------------------------------------------------------- B: assembly
    // The solve's products come from a stored matrix or from the cotangent sums S(v), of which (M v)_k and the velocity
    // are local combinations.  With the sums nothing is stored, and as S is linear, the velocity's S(mu) is S of the
    // warm start plus the solve's coefficients times the S of its basis: no sweep of its own.  With k Arnoldi steps that
    // makes 1 + k sweeps in place of an assembly, k products and the velocity's sweep.  Microseconds per stage of
    // N = 1024 water: sweep 130, assembly 181 (149 without its stores), product stored in FP32 155 when every CU loads
    // its own surface's and 65 on an idle GPU: water takes the sums (512 mixed surfaces 450 -> 297 us per stage).  A film's
    // pair has two cotangents (N = 768 FP64: sweep 124, assembly 147, stored product 75) and its cold solves take 6 or 7
    // steps, and the four sums leave the solve too few registers: with sums for the solves of one or two steps 96 films
    // took 11.1 ms, with the stored matrix 9.8.
    const bool water = ph.kind == 0;
    PairConst pc = wg_diagonal(ph, nv, n, L);
    pc.image = FILM;   // known when compiled
    using MT = std::conditional_t<MIXED, float, double>;
    MT* const Mt = reinterpret_cast<MT*>(a.M) + d.moff;
    const int nbk = (n + kTile - 1) / kTile;
    if (t < nbk * kTile) L.vs[t] = own ? x : 0.0;   // the padding entries stay 0 for every product
    __syncthreads();
    double* const psy = reinterpret_cast<double*>(L.fa);   // 2 kBT doubles each
    double* const piy = reinterpret_cast<double*>(L.fb);
    double dsq = 0.0;   // mixed: this thread's share of ||M||_F^2
    double mx0;         // (M x)_t
    CotSums<NA> S{reinterpret_cast<double*>(Mt) + (long long)cl.rank * kBK * NA * n, n, {}, {}};   // each workgroup's own
    const auto sums_of_vs = [&]() {
        if constexpr (FILM) {
            double* const acc[4] = {L.part, psy, psy + kBT, piy};
            cot_sums<4>(n, acc, pc, cl, L, S.last);
        } else {
            double* const acc[2] = {L.part, psy};
            cot_sums<2>(n, acc, pc, cl, L, S.last);
        }
    };
    const auto product = [&]() {
        if constexpr (stored) {
            return mv_pairs(Mt, n, cl, L);
        } else {
            sums_of_vs();
            const double w = own ? product_of_sums<NA>(S.last, pc, zpk, L.diag[t], L.vs[t]) : 0.0;
            __syncthreads();   // the sums and L.vs have been read
            return w;
        }
    };
    if constexpr (!stored) {
        mx0 = product();
        S.fresh();
    } else {
        // One sweep over the unordered pairs (sfh_sym.hpp) writes both entries of each pair into the
        // wave's rows of the matrix (FP64, or FP64 entries rounded to FP32) and forms (M x)_k for the warm start
        // x in FP64 from the unrounded entries: the first residual of the solve.
        const SymGeo sg = sym_geo(n);
        const int kr = sg.I * kTile + sg.l;
        const NodeTrig tk = L.tr[kr];
        const double2 zq = L.zp[kr];
        const double2 czk = make_double2(pc.c * zq.x, pc.c * zq.y);
        const double vk = L.vs[kr];
        MT* const Mi = Mt + (long long)(sg.I * nbk) * kTileElems;   // wave-uniform; the offsets are 32-bit
        const unsigned l = sg.l;
        double* const acc[1] = {L.part};
        double mx[1];
        if (MIXED && own && lead) dsq = L.diag[t] * L.diag[t];
        sym_sums<1>(n, acc, [&](int k, int j, int q, auto mirror, auto full, double (&row)[1], double (&col)[1]) {
            double e = 0.0, em = 0.0;
            if (decltype(full)::value || (k < n && j < n)) {
                entry_pair(tk, L.tr[j], czk, L.zp[j], pc, e, em);
                row[0] += e * L.vs[j];
                if constexpr (MIXED) dsq += e * e;
                if constexpr (decltype(mirror)::value) {
                    col[0] += em * vk;
                    if constexpr (MIXED) dsq += em * em;
                }
            }
            Mi[(unsigned)(2 * q) * kTile + l] = (MT)e;
            Mi[(unsigned)(2 * q + 1) * kTile + l] = decltype(mirror)::value ? (MT)em : (MT)0;
        }, cl, mx);
        mx0 = own ? mx[0] + L.diag[t] * L.vs[t] : 0.0;
    }
    __syncthreads();

    // ---------------------------------------------------------------- C: solve
    const double r0 = own ? bk - mx0 : 0.0;
    const double norms[3] = {own ? bk * bk : 0.0, r0 * r0, own ? zk.y : 0.0};
    bsum(norms, L);
    const double bn = sqrt(L.sums[0]), rr0 = L.sums[1];
    const double tol_abs = a.tol * bn;
    // Film: the image term's few large eigenvalues are divided out (wg_precondition).  A warm solve of N = 768,
    // h = 1 takes 1-2 products of the stored matrix (75 us each from one CU) in place of 4-5.
    Precond pre = {-1, 0.0};
    if constexpr (FILM) {
        pre.height = L.sums[2] / n + ph.depth;
        pre.modes = film_modes(n, pre.height);
    }
    __syncthreads();   // the sums are read before they are formed again
    NoSums none;
    auto& sums = [&]() -> auto& {
        if constexpr (stored)
            return none;
        else
            return S;
    }();
    int unconv = 0, iters = 0, sweeps = 0;
    if constexpr (!MIXED) {
        iters = wg_gmres(product, sums, n, bk, x, false, tol_abs, a.cycles, L, &unconv,
                         {true, r0, rr0}, pre);
    } else {
        // ||M - M32||_F <= 2^-24 ||M||_F (round to nearest, normal range) + N 2^-150 (subnormal range)
        double dM = 0.0;   // products that are not stored are those of M itself
        if constexpr (stored) {
            dsq = bsum1(dsq, L);
            if (cl.parts > 1) dsq = cl.sum_members(n, dsq);
            dM = 0x1p-24 * sqrt(dsq) + n * 0x1p-150;
        }
        bool done = false;
        for (; sweeps < a.max_refine; ++sweeps) {
            double mx = mx0;   // sweep 0: formed by the assembly
            if (sweeps > 0) {
                if (own) L.vs[t] = x;
                __syncthreads();
                if constexpr (stored) {
                    mx = mv_free_sym(n, pc, cl, L);   // every thread: it synchronises
                } else {
                    mx = product();
                    S.fresh();
                }
            }
            const double r = sweeps > 0 ? (own ? bk - mx : 0.0) : r0;
            const double rr = sweeps > 0 ? bsum1(r * r, L) : rr0;
            const double rn = sqrt(rr);
            if (!(rn > tol_abs)) {
                done = true;
                break;
            }
            double dx = 0.0;
            iters += wg_gmres(product, sums, n, r, dx, true,
                              stored ? fmax(1e-7 * rn, 0.25 * tol_abs) : 0.25 * tol_abs, 1, L, nullptr, {true, r, rr},
                              pre);
            x += dx;
            // the FP64 residual of the corrected x, bounded without forming it:
            //   |b - M x| <= |r - M32 dx| + |(M - M32) dx| <= (GMRES residual) + ||M - M32||_F |dx|
            // which at steady state is far below the tolerance (|dx| is the warm start's error)
            const double est = L.scal[0];   // |r - M32 dx|, the last rotated right-hand side entry
            const double dn = stored ? sqrt(bsum1(own ? dx * dx : 0.0, L)) : 0.0;
            if (est + dM * dn <= tol_abs) {
                ++sweeps;
                done = true;
                break;
            }
        }
        if (!done) unconv = 1;
    }
    if (t == 0 && lead) {
        int* st = a.stats + 4 * s;
        st[0] = iters;
        st[1] += unconv;
        st[2] = sweeps;
        if (h0) a.hvalid[(ctl.stage - 1) * a.nsurf + s] = min(hv + 1, kHistDepth);
    }
    if (own && lead && h0) push_history(h0 + t, a.total, x);

    // ---------------------------------------------------------------- D: mu'
    if (own) {
        if (lead) a.mu[off + t] = x;
        L.fa[lds_index(d, t)] = make_double2(x, 0.0);
    }
    wg_first_derivative(d, L, false);
    double2 mupk = make_double2(0.0, 0.0);
    if (own) {
        const double2 v = L.fa[lds_index(d, t)];
        mupk = make_double2(v.x * twopi_n, v.y * twopi_n);   // BaseBoundaryIntegrator.cuh:201-203
        if (lead) a.mup[off + t] = mupk;
        L.vs[t] = x;
    }
    __syncthreads();

    // ---------------------------------------------------------------- E: velocity + stage
    // The cotangent sums of mu (the image sums too for the film): from the solve, or one sweep.
    if constexpr (stored) sums_of_vs();
    double vsum[NA];
#pragma unroll
    for (int i = 0; i < NA; ++i) vsum[i] = stored ? S.last[i] : S.sum[i];
    if (cl.parts > 1) {
        if (t == 0) cl.leave();
        if (!lead) return;
    }
    double2 q1 = make_double2(0.0, 0.0), q2 = make_double2(0.0, 0.0);
    if (own) {
        velocity_from_sums(ph, zpk, zppk, mupk, x, zk.y, vsum[0], vsum[1], FILM ? vsum[FILM ? 2 : 0] : 0.0,
                           FILM ? vsum[FILM ? 3 : 0] : 0.0, q1, q2);
    }
    // createM.cuh:104 reads the lower velocity of node 1 in the rho * q1.q2 term
    double2 q1q = q1;
    if (water && ph.rho_quirk && ph.rho != 0.0 && n > 1) {
        __syncthreads();
        if (t == 1) {
            L.scal[2] = q1.x;
            L.scal[3] = q1.y;
        }
        __syncthreads();
        q1q = make_double2(L.scal[2], L.scal[3]);
    }
    if (!own) return;
    const int gi = off + t;
    if (ctl.mu_keep) ctl.mu_keep[gi] = x;
    if (ctl.qup) ctl.qup[gi] = q2;
    if (!ph.need_upper) q2 = make_double2(0.0, 0.0);
    double dphi = bernoulli(ph, zk.y, q1, q2, q1q, zpk, zppk);
    if (ctl.energy) energy_store(ph, ctl, gi, zk.x, zk.y, ctl.Pin[gi], zpk, q1);
    if (ph.drive) {
        double dD;
        dphi = drive_terms(ph, ctl, gi, zk.x, zk.y, q1, dphi, dD);
        if (ph.augmented) stage_store_delayed(ctl, gi, dD);
    }
    stage_update(ctl, gi, q1, dphi);
}

#define SFH_BATCHED_INSTANCES(SHARED)                                                        \
    template __global__ void batched_stage_kernel<false, false, SHARED>(BatchArgs, Phys, StageCtl); \
    template __global__ void batched_stage_kernel<false, true, SHARED>(BatchArgs, Phys, StageCtl);  \
    template __global__ void batched_stage_kernel<true, false, SHARED>(BatchArgs, Phys, StageCtl);  \
    template __global__ void batched_stage_kernel<true, true, SHARED>(BatchArgs, Phys, StageCtl);
SFH_BATCHED_INSTANCES(false)
SFH_BATCHED_INSTANCES(true)

}  // namespace sfh
