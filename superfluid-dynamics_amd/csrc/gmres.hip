// gmres.hip -- FP64 GMRES for the dipole system M mu = b, all workgroups of the GPU on one or a few
// large surfaces (the iterative alternative to the LU of MatrixSolver::solve,
// CuSuperHelium/MatrixSolver.cuh:113-172).
//
// M = I/2 + K is a second-kind operator: its spectrum clusters at 1/2 (for the helium film one
// outlier sits far to the right), so GMRES converges in a handful of iterations, and the stepper
// warm starts every solve from the previous stage's mu.
//
// A solve is a fixed sequence of L launches; launch i first finishes Arnoldi step i - 1 and then,
// unless the solve is done, runs step i.  No workgroup waits for another: every grid-wide result
// is read by the next launch.  Launches 0 .. L-2 are gm_sums_kernel (products formed from the cotangent sums
// that the velocity needs as well, sfh_pairs.hpp) or gm_iter_kernel (products of the stored matrix); the last one,
// which only finishes a step, is gm_close_mu_kernel, which goes on to form the derivative mu' of the
// solution and, from the sums, the velocity stage (with L = 1 the single launch is gm_iter_kernel).
//   finish step i-1 (i >= 1), in every workgroup: sum the partial dots v_l . w_{i-1} of all
//     workgroups (fixed order, so every workgroup gets the same h_{l,i-1}); rebuild
//     u = w_{i-1} - sum_l h_{l,i-1} v_l over all N entries into LDS (classical Gram-Schmidt, one
//     pass) and its norm h_{i,i-1} = |u|; rotate the Hessenberg column by the stored Givens
//     rotations and form the new one.  Workgroup 0 stores the column, the rotation and the scale.
//     Each workgroup stores its own rows of V[i] = u.
//   converged (or the last launch): y from the rotated Hessenberg system; the last launch stores
//     x0 + V y as the solution, each workgroup its own rows, and pushes them into the warm-start
//     history (a launch that finds convergence earlier only keeps y for it).  The initial guess
//     x0 and the solution are separate arrays.
//   step i: w_i = M v_i for the workgroup's rows, and the partial dots v_l . w_i, l <= i.
//     For the film w_i = M P^{-1} v_i with the preconditioner P of its image term (precondition), and
//     the solution is x0 + P^{-1} V y, P^{-1} V being kept beside V.
// Launch 0 takes v_0 = r0 / |r0|.  gm_start_kernel (or the assembly, while it writes M) forms
// r0 = b - M x0, and every workgroup of launch 0 reduces |r0| and |b| over its own full copies.
// L launches therefore run up to L - 1 Arnoldi steps.  Once the residual estimate reaches
// tol * |b|, the remaining launches return at once.  Partial dots and the rotated right-hand side
// live in per-launch (even/odd or per-index) slots, because a slot must not be overwritten while
// a slower workgroup of the same launch still reads it.
//
// Initial guess of an RK stage: mu of the same stage extrapolated over the previous steps by the
// polynomial through them (extrapolate_history; with five steps kept its error is fifth order in
// dt, against first order for the previous stage's mu), which saves Krylov steps on every solve of
// a time integration.
#include "sfh_pairs.hpp"
#include "sfh_gmres.hpp"

namespace sfh {

// RR rows of the matrix (row r at R + r n) times vs (LDS) by one wave.  The rows stream through two
// register buffers of 1024 / RR columns each, one refilled while the other is multiplied; row_start fills both
// before vs is ready.  The matrix is FP64, or FP32 in the mixed-precision form (entries widened to FP64
// as they are used).  Loads beyond the row's end are clamped to its last entry and meet a zero.
template <typename T, int RR>
struct RowBuf {
    T v[2][RR][16 / RR];
};
template <typename T, int RR>
__device__ inline void row_load(const T* __restrict__ R, int n, int rows, int c0, int lane, T (&v)[RR][16 / RR]) {
#pragma unroll
    for (int u = 0; u < 16 / RR; ++u)
#pragma unroll
        for (int r = 0; r < RR; ++r) v[r][u] = R[(unsigned)min(r, rows - 1) * (unsigned)n + (unsigned)min(c0 + lane + 64 * u, n - 1)];
}
template <typename T, int RR>
__device__ inline void row_start(const T* __restrict__ R, int n, int rows, int lane, RowBuf<T, RR>& b) {
    row_load(R, n, rows, 0, lane, b.v[0]);
    if (n > 1024 / RR) row_load(R, n, rows, 1024 / RR, lane, b.v[1]);
}
template <typename T, int RR>
__device__ inline void row_dots(const T* __restrict__ R, RowBuf<T, RR>& b, const double* vs, int n, int rows, int lane,
                                double (&out)[RR]) {
    constexpr int C = 1024 / RR;
    double acc[RR][2];
#pragma unroll
    for (int r = 0; r < RR; ++r) acc[r][0] = acc[r][1] = 0.0;
    auto use = [&](int c0, T(&v)[RR][16 / RR]) {
#pragma unroll
        for (int u = 0; u < 16 / RR; ++u) {
            const int c = c0 + lane + 64 * u;
            const double x = c < n ? vs[c] : 0.0;
#pragma unroll
            for (int r = 0; r < RR; ++r) acc[r][u & 1] += (double)v[r][u] * x;
        }
    };
    for (int c0 = 0; c0 < n; c0 += 2 * C) {
        use(c0, b.v[0]);
        if (c0 + 2 * C < n) row_load(R, n, rows, c0 + 2 * C, lane, b.v[0]);
        if (c0 + C < n) {
            use(c0 + C, b.v[1]);
            if (c0 + 3 * C < n) row_load(R, n, rows, c0 + 3 * C, lane, b.v[1]);
        }
    }
#pragma unroll
    for (int r = 0; r < RR; ++r) out[r] = wave_sum(acc[r][0] + acc[r][1]);
}

// u = w - sum_{i<j} co[i] V[i] over all n entries into vs (LDS); returns |u|^2 over the workgroup
// of NT threads.  Each thread handles E entries per pass with the basis loads of 4 vectors in
// flight together; pre and v0pre hold the first pass of w and V[0].
template <int NT, int E>
__device__ inline void load_first_pass(const double* __restrict__ w, int n, double (&u)[E]) {
#pragma unroll
    for (int e = 0; e < E; ++e) {
        const int c = threadIdx.x + NT * e;
        u[e] = c < n ? w[c] : 0.0;
    }
}
template <int NT, int E>
__device__ inline double rebuild_vector(const double* __restrict__ w, const double* __restrict__ V, const double* co,
                                        int j, int n, double* vs, double* red, const double (&pre)[E],
                                        const double (&v0pre)[E]) {
    const int t = threadIdx.x;
    double ss = 0.0;
    for (int base = 0; base < n; base += E * NT) {
        double u[E];
#pragma unroll
        for (int e = 0; e < E; ++e) {
            const int c = base + t + NT * e;
            u[e] = base == 0 ? pre[e] : (c < n ? w[c] : 0.0);
        }
        int i = 0;
        for (; i + 4 <= j; i += 4) {
            double vv[4][E];
#pragma unroll
            for (int q = 0; q < 4; ++q)
#pragma unroll
                for (int e = 0; e < E; ++e) {
                    const int c = base + t + NT * e;
                    vv[q][e] = (base == 0 && i + q == 0) ? v0pre[e] : (c < n ? V[(long long)(i + q) * n + c] : 0.0);
                }
#pragma unroll
            for (int q = 0; q < 4; ++q) {
                const double cq = co[i + q];
#pragma unroll
                for (int e = 0; e < E; ++e) u[e] -= cq * vv[q][e];
            }
        }
        for (; i < j; ++i) {
            double vv[E];
#pragma unroll
            for (int e = 0; e < E; ++e) {
                const int c = base + t + NT * e;
                vv[e] = (base == 0 && i == 0) ? v0pre[e] : (c < n ? V[(long long)i * n + c] : 0.0);
            }
            const double ci = co[i];
#pragma unroll
            for (int e = 0; e < E; ++e) u[e] -= ci * vv[e];
        }
#pragma unroll
        for (int e = 0; e < E; ++e) {
            const int c = base + t + NT * e;
            if (c < n) {
                vs[c] = u[e];
                ss += u[e] * u[e];
            }
        }
    }
    return block_sum<NT / 64>(ss, red);
}

// The film's right preconditioner: vs = P^{-1} vs (LDS, all n entries; NT threads).  On a flat film at
// the surface's mean height y the direct kernel vanishes and the image term is circulant, a Poisson
// kernel: its eigenvalue on the Fourier modes +-m of the node index is lam_m = 1/2 + n/(4 pi) exp(-2 m (y + h))
// (createM.cuh:87-88 has no Z'_k factor, so it grows with n).  These few large eigenvalues are what an
// unpreconditioned solve spends its steps on: with P = that matrix a warm-started film solve takes 1-2 steps
// in place of 4-7 (N = 768 .. 4096, h = 1), a cold one 5-9 in place of 10-13: 66.3 -> 34.6 ms per 40 steps of
// the N = 4096 film.  lam_m falls to 1/2 within a few modes, so P^{-1} = 2 + the modes' (1/lam_m - 2)
// projections, m <= modes.  GMRES on M P^{-1} leaves the residual b - M x what it was, and the tolerance on it.
template <int NT>
__device__ inline void precondition(double* vs, int n, const double2* __restrict__ tw, int modes, double height,
                                    double (*red)[2 * kPreModes + 1], double* coef) {
    constexpr int NW = NT / 64;
    const int t = threadIdx.x, lane = t & 63, wv = t >> 6;
    const double2 w0 = tw[min(t, n - 1)], ws = tw[NT % n];   // (cos, -sin) of the first entry's angle, of a step of NT
    double s0 = 0.0, ac[kPreModes], as[kPreModes];
#pragma unroll
    for (int m = 0; m < kPreModes; ++m) ac[m] = as[m] = 0.0;
    double c = w0.x, s = -w0.y;
    for (int j = t; j < n; j += NT) {
        const double u = vs[j];
        s0 += u;
        double c1 = 1.0, s1 = 0.0, cm = c, sm = s;
#pragma unroll
        for (int m = 0; m < kPreModes; ++m) {
            if (m >= modes) break;
            ac[m] += u * cm;
            as[m] += u * sm;
            const double cn = 2.0 * c * cm - c1, sn = 2.0 * c * sm - s1;   // the next mode, by recurrence
            c1 = cm;
            s1 = sm;
            cm = cn;
            sm = sn;
        }
        const double cr = c * ws.x + s * ws.y;   // angle + the step's
        s = s * ws.x - c * ws.y;
        c = cr;
    }
    s0 = wave_sum(s0);
    if (lane == 0) red[wv][0] = s0;
#pragma unroll
    for (int m = 0; m < kPreModes; ++m) {
        if (m >= modes) break;
        const double x = wave_sum(ac[m]), y = wave_sum(as[m]);
        if (lane == 0) {
            red[wv][2 * m + 1] = x;
            red[wv][2 * m + 2] = y;
        }
    }
    __syncthreads();
    if (t <= 2 * modes) {
        double x = 0.0;
#pragma unroll
        for (int w = 0; w < NW; ++w) x += red[w][t];
        const int m = (t + 1) >> 1;
        const double lam = film_eigenvalue(n, m, height);
        coef[t] = x * (m == 0 ? 1.0 : 2.0) / n * (1.0 / lam - 2.0);
    }
    __syncthreads();
    const double a0 = coef[0];
#pragma unroll
    for (int m = 0; m < kPreModes; ++m) {
        if (m >= modes) break;
        ac[m] = coef[2 * m + 1];
        as[m] = coef[2 * m + 2];
    }
    c = w0.x;
    s = -w0.y;
    for (int j = t; j < n; j += NT) {
        double z = 2.0 * vs[j] + a0;
        double c1 = 1.0, s1 = 0.0, cm = c, sm = s;
#pragma unroll
        for (int m = 0; m < kPreModes; ++m) {
            if (m >= modes) break;
            z += ac[m] * cm + as[m] * sm;
            const double cn = 2.0 * c * cm - c1, sn = 2.0 * c * sm - s1;
            c1 = cm;
            s1 = sm;
            cm = cn;
            sm = sn;
        }
        vs[j] = z;
        const double cr = c * ws.x + s * ws.y;
        s = s * ws.x - c * ws.y;
        c = cr;
    }
    __syncthreads();
}

// Rotates column jc of the Hessenberg matrix (entries 0..jc+1 in col, LDS) by the stored rotations
// 0..jc-1 and forms rotation jc; returns it in (c, s).
__device__ inline void givens_column(double* col, const double* cs, const double* sn, int jc, double& c,
                                     double& s) {
    for (int q = 0; q < jc; ++q) {
        const double t0 = cs[q] * col[q] + sn[q] * col[q + 1];
        const double t1 = -sn[q] * col[q] + cs[q] * col[q + 1];
        col[q] = t0;
        col[q + 1] = t1;
    }
    const double den = hypot(col[jc], col[jc + 1]);
    c = den > 0.0 ? col[jc] / den : 1.0;
    s = den > 0.0 ? col[jc + 1] / den : 0.0;
    col[jc] = den;
    col[jc + 1] = 0.0;
}

// y from R y = g over the k rotated columns, into y[0..k): column k - 1 (col, LDS) is this
// launch's, columns before it (H, column l at H[l (m+1)]) and g[0..k-2] come from earlier
// launches.
__device__ inline void back_substitute(const double* g, const double* H, int m, int k, double gk, const double* col,
                                       double* y) {
    for (int q = k - 1; q >= 0; --q) {
        double acc = (q == k - 1) ? gk : g[q];
        for (int l = q + 1; l < k; ++l) {
            const double hql = (l == k - 1) ? col[q] : H[l * (m + 1) + q];
            acc -= hql * y[l];
        }
        const double hqq = (q == k - 1) ? col[q] : H[q * (m + 1) + q];
        y[q] = acc / hqq;
    }
}

// Where a launch's products come from: a policy with W waves and ROWS matrix rows per workgroup.  start() requests what
// the product needs besides the vector; run() forms the rows' products of vs (LDS), w = sj * (M vs), in wl (LDS) and wi
// (the caller synchronises).
//
// The stored matrix, RR rows per wave.
template <typename T, int WAVES, int RR>
struct StoredRows {
    static constexpr int W = WAVES, ROWS = W * RR, MAXN = kGmMaxN;
    static constexpr bool PRE = false;
    const T* R;
    RowBuf<T, RR> rc;
    int n, row, rows, lane, wv;
    __device__ StoredRows(const GmArgs&, const GmView& v, const SurfDesc&, int r0) {
        lane = threadIdx.x & 63;
        wv = threadIdx.x >> 6;
        n = v.n;
        row = r0 + wv * RR;
        rows = max(1, min(RR, n - row));   // this wave's rows (at least one is loaded)
        R = (sizeof(T) == 8 ? reinterpret_cast<const T*>(v.M) : reinterpret_cast<const T*>(v.M32)) + (long long)min(row, n - 1) * n;
    }
    __device__ void start() { row_start(R, n, rows, lane, rc); }
    __device__ void run(const double* vs, double sj, double* wi, double* wl, int) {
        double d[RR];
        row_dots(R, rc, vs, n, rows, lane, d);
        if (lane == 0) {
#pragma unroll
            for (int r = 0; r < RR; ++r) {
                wl[wv * RR + r] = row + r < n ? sj * d[r] : 0.0;
                if (row + r < n) wi[row + r] = sj * d[r];
            }
        }
    }
};

// Cotangent sums (sfh_pairs.hpp), H groups of 256 threads with 4 rows each; the sums are kept for the velocity.  The
// evaluation is bound by FP64 issue (23 instructions per pair for water, 41 for the film): N = 4096 film 40 us per
// launch, of which 22 are issue, N = 2048 water 8 us, of which 3 are issue and 4 the finishing work and first loads.
template <int NA, int H>
struct PairSums {
    static constexpr int W = 4 * H, ROWS = kSumRows * H, MAXN = kGmMaxN;
    static constexpr bool PRE = NA == 4;   // the film's preconditioner
    const NodeTrig* tr;
    double* S;
    NodeTrig tk[kSumRows];
    SumConst kc;
    double2 zp;
    double diag;
    long long stride;
    int n, r0, tg, k0;
    __device__ PairSums(const GmArgs& a, const GmView& v, const SurfDesc& d, int first) {
        n = v.n;
        r0 = first;
        tg = threadIdx.x & 255;
        k0 = r0 + kSumRows * (threadIdx.x >> 8);
        tr = a.trig + d.voff;
        S = a.S + d.voff;
        stride = a.total;
        kc = {a.pc, a.pci, a.eh, a.ehi};
        const int own = d.voff + min(r0 + (int)threadIdx.x, n - 1);
        zp = a.Zp[own];
        diag = a.diag[own];
    }
    __device__ void start() {
#pragma unroll
        for (int r = 0; r < kSumRows; ++r) tk[r] = tr[min(k0 + r, n - 1)];
    }
    __device__ void run(const double* vs, double sj, double* wi, double* wl, int i) {
        __shared__ double red[W][NA * kSumRows];
        double acc[NA * kSumRows];
#pragma unroll
        for (int q = 0; q < NA * kSumRows; ++q) acc[q] = 0.0;
        const auto value = [&](int j) { return vs[j]; };
        for (int j0 = 0; j0 < n; j0 += kSumPass) {
            NodeTrig tj[kSumCols];
            sum_columns(tr, n, j0, tg, tj);
            sum_pass<NA>(tk, tj, n, k0, j0, tg, kc.eh, kc.ehi, value, acc);
        }
        sum_store<NA>(acc, red);
        __syncthreads();
        const int t = threadIdx.x;
        if (t < ROWS) {
            double w = 0.0;
            if (r0 + t < n) {
                double s[NA];
#pragma unroll
                for (int q = 0; q < NA; ++q) {
                    s[q] = sum_total<NA>(red, t / kSumRows, t % kSumRows, q);
                    S[(long long)((1 + i) * NA + q) * stride + r0 + t] = s[q];
                }
                w = sj * product_of_sums<NA>(s, kc, zp, diag, vs[r0 + t]);
                wi[r0 + t] = w;
            }
            wl[t] = w;
        }
    }
};

// The transposed product (reverse mode), one sum per row, nothing kept.  Surfaces of up to N nodes.
template <bool FILM, int N>
struct TransposeSums {
    static constexpr int W = 4, ROWS = kSumRows, MAXN = N;
    static constexpr bool PRE = false;
    const NodeTrig* tr;
    const double2* zp;
    NodeTrig tk[kSumRows];
    SumConst kc;
    double diag;
    int n, r0;
    __device__ TransposeSums(const GmArgs& a, const GmView& v, const SurfDesc& d, int first) {
        n = v.n;
        r0 = first;
        tr = a.trig + d.voff;
        zp = a.Zp + d.voff;
        kc = {a.pc, a.pci, a.eh, a.ehi};
        diag = a.diag[d.voff + min(r0 + (int)threadIdx.x, n - 1)];
    }
    __device__ void start() {
#pragma unroll
        for (int r = 0; r < kSumRows; ++r) tk[r] = tr[min(r0 + r, n - 1)];
    }
    // (M^T v) of row r0 + t on threads t < ROWS, 0 beyond the surface
    template <class F>
    __device__ double product(F&& value) {
        __shared__ double red[W][kSumRows];
        const int t = threadIdx.x;
        double acc[kSumRows] = {};
        for (int j0 = 0; j0 < n; j0 += kSumPass) {
            NodeTrig tj[kSumCols];
            double2 zj[kSumCols];
            sum_columns(tr, n, j0, t, tj);
#pragma unroll
            for (int e = 0; e < kSumCols; ++e) zj[e] = zp[min(j0 + t + 256 * e, n - 1)];
            transpose_pass<FILM>(tk, tj, zj, n, r0, j0, t, kc.c, kc.ci, kc.eh, kc.ehi, value, acc);
        }
        reduce_lanes(acc, red[t >> 6]);
        __syncthreads();
        double w = 0.0;
        if (t < ROWS && r0 + t < n) {
#pragma unroll
            for (int q = 0; q < W; ++q) w += red[q][t];
            w += diag * value(r0 + t);
        }
        return w;
    }
    __device__ void run(const double* vs, double sj, double* wi, double* wl, int) {
        const int t = threadIdx.x;
        const double w = sj * product([&](int j) { return vs[j]; });
        if (t < ROWS) {
            wl[t] = w;
            if (r0 + t < n) wi[r0 + t] = w;
        }
    }
};

// Launch i of a solve's sequence (see the file comment).  Every workgroup repeats the finishing work (the basis, the
// partial sums, the preconditioner), so the rows per workgroup follow the size (Solver::alloc_gmres).
template <class P>
__device__ __forceinline__ void gm_step(const GmArgs& a, const SurfDesc* __restrict__ sd, int i) {
    GmCtl* ctl = reinterpret_cast<GmCtl*>(a.ctl) + blockIdx.z;
    // solves finished by an earlier launch return at once.  A finish stamped by this launch
    // (workgroup 0 can get there before a late workgroup starts) does not count.  Launch 0 needs
    // no check (the derivative kernel re-armed the block), and launch 1 makes it after its row
    // loads have gone out (an earlier finish is the exception there); later launches first.
    if (i >= 2 || (i == 1 && a.check_first)) {
        const int fin = ctl->done;
        if (fin != 0 && fin <= i) return;
    }
    const GmView v = gm_view(a, sd);
    const int m = a.m;
    constexpr int W = P::W, rpw = P::ROWS, NT = 64 * W, E = 8;   // E entries per thread and pass
    if ((int)blockIdx.x * rpw >= v.n) return;
    __shared__ double vs[P::MAXN];
    __shared__ double co[kMaxKrylov + 1];
    __shared__ double col[kMaxKrylov + 2];
    __shared__ double red8[2 * W];
    __shared__ double wl[rpw], vown[rpw];
    __shared__ double pred[P::PRE ? W : 1][2 * kPreModes + 1], pcoef[2 * kPreModes + 1];
    __shared__ double sums[kMaxKrylov + 2];
    __shared__ double ys[kMaxKrylov + 4];   // g[j], gc[j+1], c, s, then y
    const int t = threadIdx.x, lane = t & 63, wv = t >> 6, n = v.n;
    const int r0 = blockIdx.x * rpw;
    P prod(a, v, sd[blockIdx.z], r0);
    const long long pslot = (long long)v.nwg * (m + 1);   // one partial-dot slot per launch parity
    // Loads go out in the order their results are needed, because a wait for one load waits for
    // all loads issued before it: first the vectors and sums of the step being finished (launch
    // 0: r0 and b), then the matrix rows, which the finishing work then overlaps.
    const int j = i - 1;
    const double* wprev = (j & 1) ? v.w1 : v.w0;
    const double* part = v.part + (j & 1) * pslot;
    double pa[E], pb[E];   // first pass: launch 0 r0 and b, later w_{i-1} and V[0]
    DotLoads dl;
    const bool fastdots = i >= 1 && dots_fast(v.nwg, i);
    double sc_t = 0.0, gold = 0.0, bnorm = 0.0;
    if (i == 0) {
        load_first_pass<NT>(v.V, n, pa);
        load_first_pass<NT>(v.b, n, pb);
    } else {
        load_first_pass<NT>(wprev, n, pa);
        load_first_pass<NT>(v.V, n, pb);
        if (fastdots) dots_load<NT>(part, v.nwg, i, dl);
        sc_t = t <= j ? v.sc[t] : 0.0;
        gold = v.gc[j];
        bnorm = ctl->bnorm;
    }
    const int pre_modes = P::PRE ? v.ctl->pre_modes : -1;
    const double height = P::PRE ? v.ctl->height : 0.0;
    // the rows up front, except in a refinement solve, which most often ends at once: there they
    // are fetched when the step is known to run
    const bool early_rows = !a.check_first;
    if (i < m - 1 && early_rows) prod.start();
    if (i == 1 && !a.check_first) {
        const int fin = ctl->done;
        if (fin != 0 && fin <= i) return;
    }
    int k = 0;        // Arnoldi steps completed
    double sj = 0.0;  // scale of v_i = sj * vs
    bool done = false;
    // this workgroup's own rows (threads t < rpw): x, V[0] and the history levels that move
    // down, for the correction at the end of a solve, loaded up front
    double* h0 = history(a, sd, blockIdx.z);
    const int oc = min(r0 + t, n - 1);
    double xo = 0.0, vo0 = 0.0, ho[kHistDepth - 1];
#pragma unroll
    for (int l = 0; l < kHistDepth - 1; ++l) ho[l] = 0.0;
    if (t < rpw) {
        xo = v.x[oc];
        vo0 = v.Z[oc];
        if (h0) {
#pragma unroll
            for (int l = 0; l < kHistDepth - 1; ++l) ho[l] = h0[(long long)l * a.total + oc];
        }
    }
    if (i == 0) {
        // v_0 = r0 / |r0|; beta = |r0| and |b| reduced by every workgroup over its own copies
        double sq = 0.0, bq = 0.0;
        for (int base = 0; base < n; base += NT * E) {
#pragma unroll
            for (int e = 0; e < E; ++e) {
                const int c = base + t + NT * e;
                const double x = base == 0 ? pa[e] : (c < n ? v.V[c] : 0.0);
                const double bc = base == 0 ? pb[e] : (c < n ? v.b[c] : 0.0);
                if (c < n) {
                    vs[c] = x;
                    sq += x * x;
                    bq += bc * bc;
                }
            }
        }
        sq = wave_sum(sq);
        bq = wave_sum(bq);
        if (lane == 0) {
            red8[wv] = sq;
            red8[W + wv] = bq;
        }
        __syncthreads();
        sq = bq = 0.0;
#pragma unroll
        for (int w = 0; w < W; ++w) {
            sq += red8[w];
            bq += red8[W + w];
        }
        const double beta = sqrt(sq), bnorm = sqrt(bq);
        if (blockIdx.x == 0 && t == 0) {
            ctl->bnorm = bnorm;
            ctl->beta = beta;
            ctl->res = beta;
            v.gc[0] = beta;
            v.sc[0] = beta > 0.0 ? 1.0 / beta : 0.0;
        }
        done = beta <= a.tol * bnorm || m < 2;
        if (done && blockIdx.x == 0 && t == 0 && !(beta <= a.tol * bnorm)) ctl->unconverged += 1;
        sj = beta > 0.0 ? 1.0 / beta : 0.0;
    } else {
        // ---- finish step i - 1
        if (fastdots)
            dots_finish<NT>(dl, j + 1, sums);
        else
            reduce_partials<NT>(part, v.nwg, j + 1, sums);
        if (t <= j) co[t] = sums[t] * sc_t;
        __syncthreads();
        const double hn = sqrt(rebuild_vector<NT, E>(wprev, v.V, co, j + 1, n, vs, red8, pa, pb));
        if (t == 0) {
            for (int q = 0; q <= j; ++q) col[q] = sums[q];
            col[j + 1] = hn;
            double c, s;
            givens_column(col, v.cs, v.sn, j, c, s);
            ys[0] = c * gold;          // g[j]
            ys[1] = -s * gold;         // gc[j + 1]
            ys[2] = c;
            ys[3] = s;
        }
        __syncthreads();
        const double gj = ys[0], gnext = ys[1], res = fabs(gnext);
        if (blockIdx.x == 0 && t == 0) {
            double* Hc = v.H + (long long)j * (m + 1);
            for (int q = 0; q <= j + 1; ++q) Hc[q] = col[q];
            v.cs[j] = ys[2];
            v.sn[j] = ys[3];
            v.g[j] = gj;
            v.gc[j + 1] = gnext;
            v.sc[j + 1] = hn > 0.0 ? 1.0 / hn : 0.0;
            ctl->res = res;
            ctl->hnext = hn;
        }
        k = i;
        const bool conv = res <= a.tol * bnorm || hn == 0.0;
        done = conv || i >= m - 1;
        if (done && !conv && blockIdx.x == 0 && t == 0) ctl->unconverged += 1;
        if (!done) {
            // V[i] = u: this workgroup's rows (every workgroup holds all of u in LDS)
            if (t < rpw && r0 + t < n) v.V[(long long)i * n + r0 + t] = vs[r0 + t];
            sj = hn > 0.0 ? 1.0 / hn : 0.0;
        } else if (t == 0) {
            back_substitute(v.g, v.H, m, k, gj, col, ys + 4);   // then scaled by sc
        }
        if (done) {   // y_q sc_q
            __syncthreads();
            if (t <= j) ys[4 + t] *= sc_t;
        }
    }
    if (done && i < m - 1) {
        // converged before the last launch, which stores the solution (gm_close_mu_kernel): keep y
        if (blockIdx.x == 0) {
            if (t < k) v.y[t] = ys[4 + t];   // scaled by this thread above
            if (t == 0) {
                set_iters(ctl, a, k);
                ctl->done = i + 1;
            }
        }
        return;
    }
    if (done) {
        // the single launch of a one-launch sequence: x0 + V y on this workgroup's rows; the
        // stage's history
        __syncthreads();
        if (t < rpw && r0 + t < n) {
            const int c = r0 + t;
            double x = xo;
            if (k > 0) x += ys[4] * vo0;
            for (int q = 1; q < k; ++q) x += ys[4 + q] * v.Z[(long long)q * n + c];
            v.sol[c] = x;
            if (h0) {
#pragma unroll
                for (int l = kHistDepth - 1; l > 0; --l) h0[(long long)l * a.total + c] = ho[l - 1];
                h0[c] = x;
            }
        }
        if (blockIdx.x == 0 && t == 0) {
            set_iters(ctl, a, k);
            ctl->done = i + 1;
            if (h0 && blockIdx.z == 0) count_history(a);
        }
        return;
    }
    // ---- step i: w_i = M P^{-1} v_i (v_i = sj * vs) for this workgroup's rows, partial dots v_l . w_i
    if (t < rpw) vown[t] = vs[min(r0 + t, n - 1)];
    if constexpr (P::PRE) {
        __syncthreads();
        const SurfDesc d = sd[blockIdx.z];
        if (pre_modes >= 0) precondition<NT>(vs, n, a.tw + d.twoff, pre_modes, height, pred, pcoef);
        if (t < rpw && r0 + t < n) v.Z[(long long)i * n + r0 + t] = vs[r0 + t];
    }
    double vrow[rpw];
#pragma unroll
    for (int r = 0; r < rpw; ++r) vrow[r] = (t < i && r0 + r < n) ? v.V[(long long)t * n + r0 + r] : 0.0;
    const double sct = (t < i) ? v.sc[t] : 0.0;
    double* wi = (i & 1) ? v.w1 : v.w0;
    if (!early_rows) prod.start();
    prod.run(vs, sj, wi, wl, i);
    __syncthreads();
    if (t <= i) {
        double s = 0.0;
#pragma unroll
        for (int r = 0; r < rpw; ++r) {
            if (r0 + r < n) {
                const double vi = (t == i) ? sj * vown[r] : sct * vrow[r];
                s += vi * wl[r];
            }
        }
        v.part[(i & 1) * pslot + (long long)t * v.nwg + blockIdx.x] = s;
    }
}

template <typename T, int W, int RR>
__global__ __launch_bounds__(64 * W) void gm_iter_kernel(GmArgs a, const SurfDesc* __restrict__ sd, int i) {
    gm_step<StoredRows<T, W, RR>>(a, sd, i);
}
template <int NA, int H>
__global__ __launch_bounds__(256 * H) void gm_sums_kernel(GmArgs a, const SurfDesc* __restrict__ sd, int i) {
    gm_step<PairSums<NA, H>>(a, sd, i);
}

template <bool FILM, int N>
__global__ __launch_bounds__(256) void gm_tsums_kernel(GmArgs a, const SurfDesc* __restrict__ sd, int i) {
    gm_step<TransposeSums<FILM, N>>(a, sd, i);
}

// The warm start of a transposed solve: r0 = b - M^T x0 as the first basis vector.  grid = (ceil(max n / kSumRows), surfaces).
template <bool FILM>
__global__ __launch_bounds__(256) void gm_tstart_kernel(GmArgs a, const SurfDesc* __restrict__ sd, int reset) {
    const SurfDesc d = sd[blockIdx.y];
    const int r0 = blockIdx.x * kSumRows, t = threadIdx.x;
    if (blockIdx.x == 0 && t == 0) {
        GmCtl* c = reinterpret_cast<GmCtl*>(a.ctl) + blockIdx.y;
        c->done = 0;
        c->refine_iters = 0;
        c->iters = 0;
        if (reset) c->most = 0;
    }
    if (r0 >= d.n) return;
    const GmView v = gm_view(a, sd, blockIdx.y);
    const double* x0 = a.x + d.voff;
    const double b = a.b[d.voff + min(r0 + t, d.n - 1)];
    TransposeSums<FILM, kGmMaxNT> prod(a, v, d, r0);   // the product alone keeps nothing of size N
    prod.start();
    const double w = prod.product([&](int j) { return x0[j]; });
    if (t < kSumRows && r0 + t < d.n) a.V[(long long)(a.m + 1) * d.voff + r0 + t] = b - w;
}
// the vector of up to 4096 nodes leaves room for four workgroups on a CU; larger surfaces, which only LU handles have,
// get an instance of their own
template __global__ void gm_tsums_kernel<false, kGmMaxN>(GmArgs, const SurfDesc*, int);
template __global__ void gm_tsums_kernel<true, kGmMaxN>(GmArgs, const SurfDesc*, int);
template __global__ void gm_tsums_kernel<false, kGmMaxNT>(GmArgs, const SurfDesc*, int);
template __global__ void gm_tsums_kernel<true, kGmMaxNT>(GmArgs, const SurfDesc*, int);
template __global__ void gm_tstart_kernel<false>(GmArgs, const SurfDesc*, int);
template __global__ void gm_tstart_kernel<true>(GmArgs, const SurfDesc*, int);

// The start of a solve with products from cotangent sums: S of the initial guess, M_kk, and r0 = b - M x0 as the first
// (unnormalised) basis vector.  grid = (ceil(max n / kSumRows), surfaces).
template <int NA>
__global__ __launch_bounds__(256) void gm_start_kernel(GmArgs a, const SurfDesc* __restrict__ sd, const double2* __restrict__ Z,
                                                       const double2* __restrict__ Zpp, Phys ph) {
    const SurfDesc d = sd[blockIdx.y];
    const int n = d.n, k0 = blockIdx.x * kSumRows, t = threadIdx.x;
    if (k0 >= n) return;
    __shared__ double red[4][NA * kSumRows];
    const NodeTrig* tr = a.trig + d.voff;
    const double* x0 = a.x + d.voff;
    NodeTrig tk[kSumRows], tj[kSumCols];
    double xj[kSumCols];
    double acc[NA * kSumRows];
#pragma unroll
    for (int r = 0; r < kSumRows; ++r) tk[r] = tr[min(k0 + r, n - 1)];
    sum_columns(tr, n, 0, t, tj);
#pragma unroll
    for (int e = 0; e < kSumCols; ++e) xj[e] = x0[min(t + 256 * e, n - 1)];
    // the own rows' inputs, before the sweep
    const int g = d.voff + min(k0 + t, n - 1);
    double2 zp = {1.0, 0.0}, zpp = {0.0, 0.0};
    double y = 0.0, b = 0.0, x = 0.0;
    if (t < kSumRows) {
        zp = a.Zp[g];
        zpp = Zpp[g];
        y = Z[g].y;
        b = a.b[g];
        x = a.x[g];
    }
#pragma unroll
    for (int q = 0; q < NA * kSumRows; ++q) acc[q] = 0.0;
    for (int j0 = 0; j0 < n; j0 += kSumPass) {
        if (j0 > 0) {
            sum_columns(tr, n, j0, t, tj);
#pragma unroll
            for (int e = 0; e < kSumCols; ++e) xj[e] = x0[min(j0 + t + 256 * e, n - 1)];
        }
        int e = 0;
        sum_pass<NA>(tk, tj, n, k0, j0, t, a.eh, a.ehi, [&](int) { return xj[e++]; }, acc);
    }
    sum_store<NA>(acc, red);
    double dg = 0.0;
    if (t < kSumRows) {
        const double2 q = cdiv(zpp, zp);
        dg = (ph.kind == 0 ? 0.5 * (1 + ph.rho) : 0.5) + a.pc * q.y;
        if constexpr (NA == 4) dg -= a.pci * cot64(0.0, y + ph.depth).y;
    }
    __syncthreads();
    if (t < kSumRows && k0 + t < n) {
        double s[NA];
#pragma unroll
        for (int q = 0; q < NA; ++q) {
            s[q] = sum_total<NA>(red, 0, t, q);
            a.S[(long long)q * a.total + g] = s[q];
        }
        a.diag[g] = dg;
        const SumConst kc = {a.pc, a.pci, a.eh, a.ehi};
        a.V[(long long)(a.m + 1) * d.voff + k0 + t] = b - product_of_sums<NA>(s, kc, zp, dg, x);
    }
}

// The closing launch's circulant product: 256 threads, two runs of 4 columns each, 8 rows.
struct CloseGeo {
    static constexpr int NT = 256, CHUNK = kCircChunk, ROWS = kCircRowsPerWG;
    static constexpr int WPER = (CHUNK + ROWS - 1 + NT - 1) / NT;
    static constexpr int WIN = (CHUNK + ROWS + 31) / 32 * 32;
    static_assert(ROWS == kCR && CHUNK == 2 * kCC * NT, "one group of rows, two runs of columns");
};

// The last launch of a sequence (i = m - 1 >= 1) fused with the derivative of the solution,
// mu' = D1 mu 2 pi / n (mu_circ_kernel's circulant product; BaseBoundaryIntegrator.cuh:201-203).
// Every workgroup finishes Arnoldi step i - 1 as gm_iter_kernel does, forms y and stages
// mu = x0 + V y of all nodes in LDS, kCircChunk at a time.  It stores its own kCircRowsPerWG rows
// of the solution (and pushes them into the stage's history) from the staged values, and
// multiplies the staged mu by the circulant kernel for mu' of the same rows.  A solve that
// converged in an earlier launch left its (scaled) y behind, and this launch stores its solution
// all the same.  Everything the launch reads that does not depend on another of its loads is
// requested at the start: the kernel window of the first chunk, the first 2048 entries of x0,
// V[0], V[1] and w_{i-1}, the partial dots, and the small state (scales, rotations, g, H, y) into
// LDS, so that the finishing work runs on data already at hand.  A workgroup reads the initial
// guess, the basis and earlier launches' results, never the solution entries that other
// workgroups of this launch are storing.  grid = (ceil(max n / kCircRowsPerWG), surfaces).
template <bool PRE, int NA>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(2))) void gm_close_mu_kernel(GmArgs a, const SurfDesc* __restrict__ sd,
                                                          const double* __restrict__ circ,
                                                          double2* __restrict__ mup, int i,
                                                          const double2* __restrict__ Z,
                                                          const double2* __restrict__ Zpp, Phys ph, StageCtl sc) {
    constexpr int NT = 256;
    constexpr int CR = kCircRowsPerWG;
    constexpr int KM = kMaxKrylov;
    static_assert(kCircPer == 8, "the first staged chunk reuses the 8-entry first passes");
    const int s = blockIdx.y;
    const SurfDesc d = sd[s];
    const int n = d.n;
    const int k0 = blockIdx.x * CR;
    if (k0 >= n) return;
    const GmView v = gm_view(a, sd, s);
    GmCtl* ctl = reinterpret_cast<GmCtl*>(a.ctl) + s;
    const int m = a.m;
    const int j = i - 1;
    using G = CloseGeo;
    __shared__ alignas(16) double ms[G::CHUNK];
    __shared__ alignas(16) double c1re[G::WIN], c1im[G::WIN];
    __shared__ double cred[NT / 64][2 * kCR];
    __shared__ double Hs[KM * (KM + 1)];
    __shared__ double cs_s[KM], sn_s[KM], g_s[KM + 1];
    __shared__ double co[KM + 1];
    __shared__ double col[KM + 2];
    __shared__ double red8[8];
    __shared__ double sums[KM + 2];
    __shared__ double ys[KM + 4];   // g[j], gc[j+1], c, s, then y
    const int t = threadIdx.x, wv = t >> 6;
    // with the solve's cotangent sums: the own rows' sums of x0 and of the first two basis vectors, Z', Z'' and Z
    constexpr int F = 3 * NA + 6;
    __shared__ double own[NA ? CR * F : 1];
    double own_v = 0.0;
    if constexpr (NA > 0) {
        if (t < CR * F) {
            const int f = t / CR, g = d.voff + min(k0 + t % CR, n - 1);
            const double2* node[3] = {a.Zp, Zpp, Z};
            const double2* p = f < 3 * NA + 2 ? node[0] : f < 3 * NA + 4 ? node[1] : node[2];
            own_v = f < 3 * NA ? a.S[(long long)f * a.total + g] : reinterpret_cast<const double*>(p + g)[(f - 3 * NA) & 1];
        }
    }
    const double* c1r = circ + d.coff;
    const double* c1i = c1r + n;
    double ar[G::WPER], ai[G::WPER];
    {
        int q[G::WPER];
        circ_entries<G>(k0, 0, n, q);
#pragma unroll
        for (int e = 0; e < G::WPER; ++e) {
            ar[e] = c1r[q[e]];
            ai[e] = c1i[q[e]];
        }
    }
    const double* wprev = (j & 1) ? v.w1 : v.w0;
    double xpre[8], v0pre[8], v1pre[8], wpre[8];
    load_first_pass<NT>(v.x, n, xpre);
    load_first_pass<NT>(v.V, n, v0pre);
    load_first_pass<NT>(j >= 1 ? v.V + n : v.V, n, v1pre);
    load_first_pass<NT>(wprev, n, wpre);
    double z0pre[8], z1pre[8];   // with a preconditioner: Z[0], Z[1]
    if constexpr (PRE) {
        load_first_pass<NT>(v.Z, n, z0pre);
        load_first_pass<NT>(j >= 1 ? v.Z + n : v.Z, n, z1pre);
    }
    const long long pslot = (long long)v.nwg * (m + 1);
    const double* part = v.part + (j & 1) * pslot;
    DotLoads dl;
    const bool fastdots = dots_fast(v.nwg, j + 1);
    if (fastdots) dots_load(part, v.nwg, j + 1, dl);
    const double sc_t = t <= j ? v.sc[t] : 0.0;
    const double y_t = t < m ? v.y[t] : 0.0;
    const double gold = v.gc[j];
    double cs_t = 0.0, sn_t = 0.0, g_t = 0.0, hreg[4];
    if (t < j) {
        cs_t = v.cs[t];
        sn_t = v.sn[t];
        g_t = v.g[t];
    }
    static_assert(4 * 256 >= (KM - 1) * (KM + 1), "H columns 0 .. j-1 in four registers per thread");
#pragma unroll
    for (int r = 0; r < 4; ++r) {
        const int e = t + 256 * r;
        hreg[r] = e < j * (m + 1) ? v.H[e] : 0.0;
    }
    double* h0 = history(a, sd, s);
    double ho[kHistDepth - 1];
#pragma unroll
    for (int l = 0; l < kHistDepth - 1; ++l) ho[l] = 0.0;
    if (h0 && t < CR) {
        const int oc = min(k0 + t, n - 1);
#pragma unroll
        for (int l = 0; l < kHistDepth - 1; ++l) ho[l] = h0[(long long)l * a.total + oc];
    }
    // the control block last: its fields decide branches, so the first use waits for them
    const int fin = ctl->done;
    const int iters_before = a.check_first ? ctl->refine_iters : ctl->iters;
    const double bnorm = ctl->bnorm;
    if constexpr (NA > 0)
        if (t < CR * F) own[t] = own_v;
    // all loads are out; the small state into LDS and the partial dots summed (used when the
    // solve is open)
    if (t < j) {
        cs_s[t] = cs_t;
        sn_s[t] = sn_t;
        g_s[t] = g_t;
    }
#pragma unroll
    for (int r = 0; r < 4; ++r) {
        const int e = t + 256 * r;
        if (e < j * (m + 1)) Hs[e] = hreg[r];
    }
    if (fastdots)
        dots_finish(dl, j + 1, sums);
    else
        reduce_partials(part, v.nwg, j + 1, sums);
    // a finish stamped by this launch (workgroup 0 got there first) leaves the solve open here
    const bool open = !(fin != 0 && fin <= i);
    int k;
    if (!open) {
        // converged in an earlier launch, which kept y (scaled) for this one
        k = iters_before;
        if (t < k) ys[4 + t] = y_t;
        __syncthreads();
    } else {
        // ---- finish step j: h_{l,j} = sums[l] sc_l, |u| with u = w_j - sum_l h_{l,j} v_l
        if (t <= j) co[t] = sums[t] * sc_t;
        __syncthreads();
        double ss = 0.0;
        for (int base = 0; base < n; base += 2048) {
            double u[8];
            if (base == 0) {
#pragma unroll
                for (int e = 0; e < 8; ++e) u[e] = wpre[e] - co[0] * v0pre[e];
                if (j >= 1) {
#pragma unroll
                    for (int e = 0; e < 8; ++e) u[e] -= co[1] * v1pre[e];
                }
                for (int l = 2; l <= j; ++l) {
                    double vv[8];
                    load_first_pass<NT>(v.V + (long long)l * n, n, vv);
#pragma unroll
                    for (int e = 0; e < 8; ++e) u[e] -= co[l] * vv[e];
                }
            } else {
#pragma unroll
                for (int e = 0; e < 8; ++e) {
                    const int c = base + t + 256 * e;
                    u[e] = c < n ? wprev[c] : 0.0;
                }
                for (int l = 0; l <= j; ++l) {
                    double vv[8];
#pragma unroll
                    for (int e = 0; e < 8; ++e) {
                        const int c = base + t + 256 * e;
                        vv[e] = c < n ? v.V[(long long)l * n + c] : 0.0;
                    }
#pragma unroll
                    for (int e = 0; e < 8; ++e) u[e] -= co[l] * vv[e];
                }
            }
#pragma unroll
            for (int e = 0; e < 8; ++e) {
                const int c = base + t + 256 * e;
                if (c < n) ss += u[e] * u[e];
            }
        }
        const double hn = sqrt(block_sum<4>(ss, red8));
        if (t == 0) {
            for (int q = 0; q <= j; ++q) col[q] = sums[q];
            col[j + 1] = hn;
            double c, sn;
            givens_column(col, cs_s, sn_s, j, c, sn);
            ys[0] = c * gold;    // g[j]
            ys[1] = -sn * gold;  // gc[j + 1]
            ys[2] = c;
            ys[3] = sn;
            back_substitute(g_s, Hs, m, j + 1, ys[0], col, ys + 4);
        }
        __syncthreads();
        const double gj = ys[0], gnext = ys[1], res = fabs(gnext);
        k = i;
        if (blockIdx.x == 0 && t == 0) {
            double* Hc = v.H + (long long)j * (m + 1);
            for (int q = 0; q <= j + 1; ++q) Hc[q] = col[q];
            v.cs[j] = ys[2];
            v.sn[j] = ys[3];
            v.g[j] = gj;
            v.gc[j + 1] = gnext;
            v.sc[j + 1] = hn > 0.0 ? 1.0 / hn : 0.0;
            ctl->res = res;
            ctl->hnext = hn;
            if (!(res <= a.tol * bnorm || hn == 0.0)) ctl->unconverged += 1;
            set_iters(ctl, a, k);
            ctl->done = i + 1;
        }
        if (t <= j) ys[4 + t] *= sc_t;   // y_q sc_q
        __syncthreads();
    }
    if (h0 && s == 0 && blockIdx.x == 0 && t == 0) count_history(a);
    // mu = x0 + y_0 Z[0] + y_1 Z[1] (+ the rest when k > 2), without branches in the common case
    double mu_t = 0.0;   // own row, threads t < CR
    StageIn st{};
    if constexpr (NA > 0)
        if (t < CR) st = stage_load(sc, d.voff + min(k0 + t, n - 1));
    const double y0 = k > 0 ? ys[4] : 0.0, y1 = k > 1 ? ys[5] : 0.0;
    double re[kCR], im[kCR];
#pragma unroll
    for (int r = 0; r < kCR; ++r) re[r] = im[r] = 0.0;
    for (int j0 = 0; j0 < n; j0 += kCircChunk) {
        const int jn = min(kCircChunk, n - j0);
        if (j0 > 0) {
            __syncthreads();   // the previous chunk has been consumed
            int q[G::WPER];
            circ_entries<G>(k0, j0, n, q);
#pragma unroll
            for (int e = 0; e < G::WPER; ++e) {
                ar[e] = c1r[q[e]];
                ai[e] = c1i[q[e]];
            }
            load_first_pass<NT>(v.x + j0, n - j0, xpre);
            load_first_pass<NT>(v.Z + j0, n - j0, PRE ? z0pre : v0pre);
            load_first_pass<NT>(v.Z + n + j0, n - j0, PRE ? z1pre : v1pre);
        }
        double mv[kCircPer];
#pragma unroll
        for (int e = 0; e < kCircPer; ++e) mv[e] = xpre[e] + y0 * (PRE ? z0pre[e] : v0pre[e]) + y1 * (PRE ? z1pre[e] : v1pre[e]);
        for (int q = 2; q < k; ++q) {
            double vq[8];
            load_first_pass<NT>(v.Z + (long long)q * n + j0, n - j0, vq);
            const double yq = ys[4 + q];
#pragma unroll
            for (int e = 0; e < kCircPer; ++e) mv[e] += yq * vq[e];
        }
#pragma unroll
        for (int e = 0; e < kCircPer; ++e) {
            const int c = t + 256 * e;
            ms[circ_at(c)] = c < jn ? mv[e] : 0.0;
        }
#pragma unroll
        for (int e = 0; e < G::WPER; ++e) {
            const int u = t + 256 * e;
            if (u < G::CHUNK + G::ROWS) {
                c1re[circ_at(u)] = ar[e];
                c1im[circ_at(u)] = ai[e];
            }
        }
        __syncthreads();
        if (t < CR) {   // the own rows of the solution, as staged
            const int r = k0 + t;
            if (r < n && r >= j0 && r < j0 + jn) {
                const double x = ms[circ_at(r - j0)];
                v.sol[r] = x;
                mu_t = x;
                if (h0) {
#pragma unroll
                    for (int l = kHistDepth - 1; l > 0; --l) h0[(long long)l * a.total + r] = ho[l - 1];
                    h0[r] = x;
                }
            }
        }
#pragma unroll
        for (int h = 0; h < 2; ++h) {
            const int c0 = kCC * (t + NT * h);
            if (c0 < jn) {
                double x[kCC], w[kCC + kCR];
                circ_samples(ms, c0, x);
                circ_kernel(c1re, c0, w);
                circ_fma(w, x, re);
                circ_kernel(c1im, c0, w);
                circ_fma(w, x, im);
            }
        }
    }
    reduce_lanes(re, &cred[wv][0]);
    reduce_lanes(im, &cred[wv][kCR]);
    __syncthreads();
    if (t < CR && k0 + t < n) {
        double x = 0.0, y = 0.0;
#pragma unroll
        for (int w = 0; w < NT / 64; ++w) {
            x += cred[w][t];
            y += cred[w][kCR + t];
        }
        const double xs = 2.0 * kPi / n;
        const double2 mp = make_double2(x * xs, y * xs);
        mup[d.voff + k0 + t] = mp;
        if constexpr (NA > 0) {
            const int g = d.voff + k0 + t;
            double S[NA];
#pragma unroll
            for (int c = 0; c < NA; ++c) S[c] = own[c * CR + t] + y0 * own[(NA + c) * CR + t] + y1 * own[(2 * NA + c) * CR + t];
            for (int q = 2; q < k; ++q)
#pragma unroll
                for (int c = 0; c < NA; ++c) S[c] += ys[4 + q] * a.S[(long long)((1 + q) * NA + c) * a.total + g];
            const double* o = own + 3 * NA * CR + t;
            const double2 zp = make_double2(o[0], o[CR]), zpp = make_double2(o[2 * CR], o[3 * CR]);
            const double2 z = make_double2(o[4 * CR], o[5 * CR]);
            double2 q1, q2;
            velocity_from_sums(ph, zp, zpp, mp, mu_t, z.y, S[0], S[1], NA == 4 ? S[NA == 4 ? 2 : 0] : 0.0,
                               NA == 4 ? S[NA == 4 ? 3 : 0] : 0.0, q1, q2);
            finish_node(ph, sc, g, z, zp, zpp, mu_t, q1, q2, q1, st);
        }
    }
}

#define SFH_GM_INSTANCES(W, RR)                                                     \
    template __global__ void gm_iter_kernel<double, W, RR>(GmArgs, const SurfDesc*, int); \
    template __global__ void gm_iter_kernel<float, W, RR>(GmArgs, const SurfDesc*, int);
SFH_GM_INSTANCES(4, 1)
SFH_GM_INSTANCES(8, 2)
#define SFH_SUMS_INSTANCES(NA)                                                                          \
    template __global__ void gm_start_kernel<NA>(GmArgs, const SurfDesc*, const double2*, const double2*, Phys); \
    template __global__ void gm_sums_kernel<NA, 1>(GmArgs, const SurfDesc*, int);                            \
    template __global__ void gm_sums_kernel<NA, 2>(GmArgs, const SurfDesc*, int);
SFH_SUMS_INSTANCES(2)
SFH_SUMS_INSTANCES(4)
// stored matrix; sums for water; sums for the film, whose solves always have the preconditioner
template __global__ void gm_close_mu_kernel<false, 0>(GmArgs, const SurfDesc*, const double*, double2*, int, const double2*,
                                                      const double2*, Phys, StageCtl);
template __global__ void gm_close_mu_kernel<false, 2>(GmArgs, const SurfDesc*, const double*, double2*, int, const double2*,
                                                      const double2*, Phys, StageCtl);
template __global__ void gm_close_mu_kernel<true, 4>(GmArgs, const SurfDesc*, const double*, double2*, int, const double2*,
                                                     const double2*, Phys, StageCtl);

}  // namespace sfh
