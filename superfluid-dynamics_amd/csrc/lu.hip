// lu.hip -- dense FP64 solve M mu = b for the dipole strengths (one large surface per launch
// grid, uniform batches on gridDim.z).
//
// Replaces MatrixSolver::solve (CuSuperHelium/MatrixSolver.cuh:113-172): cusolverDnDgetrf +
// cusolverDnDgetrs (LU with partial pivoting), or getrfBatched/getrsBatched with a host sync.
//
// Algorithm.  Right-looking blocked LU with 64-wide panels, one launch (lu_step_kernel) per panel
// p (columns k0..k0+kb): every panel workgroup applies panel p-1's update to the diagonal block A11 and
// factors A11 = L11 U11 in LDS, in four steps of 16 columns (wave 0 the pivots of a 16 x 16 tile, the
// matrix cores (v_mfma_f64_16x16x4) the tiles around it); each "row" workgroup forms
// L21_i = A21_i U11^{-1} and b_i -= L21_i y_p and each "column" workgroup U12_j = L11^{-1} A12_j on its
// other four waves, one step behind the factorisation, workgroup 0 stores U11^{-1} and
// y_p = L11^{-1} b_p; the other workgroups of the launch apply panel p-1's update A22 -= L21 U12 to the
// rest of the trailing matrix.
// lu_backsolve_kernel then runs x_p = U_pp^{-1} (y_p - sum_{q>p} U_pq x_q), one workgroup per
// block row, chained through the entries of x themselves.
//
// Row interchanges.  Partial pivoting (getrf: first row of maximal |a| in the current column)
// leaves the rows in place exactly when every multiplier satisfies |l_ij| <= 1.  Both the
// diagonal-block elimination and the L21 blocks check that condition; if it ever fails,
// status[0] is set and gepp_fallback_kernel re-solves the freshly re-assembled system with
// explicit interchanges.  The result is therefore the GEPP solution in every case, with the
// interchange-free path taken for the diagonally dominated second-kind systems of this method.
#include <type_traits>

#include "sfh_kernels.hpp"

namespace sfh {

typedef double v4d __attribute__((ext_vector_type(4)));

constexpr int LD = kNB + 1;   // LDS leading dimension of 64 x 64 FP64 blocks
constexpr int LDB = kNB + 16;  // ... of blocks read as the MFMA's B operand only (4 rows x 16 columns a wave)

__device__ inline v4d mfma_f64(double a, double b, v4d c) {
    return __builtin_amdgcn_mfma_f64_16x16x4f64(a, b, c, 0, 0, 0);
}
// c - a b: the FP64 form takes its last operand field as sign bits (bit 0: A negated)
__device__ inline v4d mfma_f64_sub(double a, double b, v4d c) {
    return __builtin_amdgcn_mfma_f64_16x16x4f64(a, b, c, 0, 0, 1);
}

// The L21 block of the block row at R0 (rows rows) and the panel at kp, from the strips' layout (below)
// into LDS, row-major; by the NW waves from W0 on, one 512-byte row of the layout at a time.
template <int W0, int NW>
__device__ __forceinline__ void load_l21(double* dst, const double* A, int n, int R0, int kp, int rows) {
    constexpr int IT = (kNB + NW - 1) / NW;
    const int lane = threadIdx.x & 63, f0 = (threadIdx.x >> 6) - W0;
    const double* src = A + (long long)R0 * n + kp;
    double v[IT];
#pragma unroll
    for (int it = 0; it < IT; ++it) v[it] = src[(unsigned)min(f0 + NW * it, rows - 1) * (unsigned)n + (unsigned)lane];
#pragma unroll
    for (int it = 0; it < IT; ++it) {
        const int f = f0 + NW * it;
        if (f < kNB) dst[((f & ~15) + (lane & 15)) * LD + 4 * (f & 15) + (lane >> 4)] = v[it];
    }
}

// The rows x cols block at src (leading dimension ld) into LDS (leading dimension LDX), by the same waves.
template <int LDX, int W0, int NW>
__device__ __forceinline__ void load_rows(double* dst, const double* src, int ld, int rows, int cols) {
    constexpr int IT = (kNB + NW - 1) / NW;
    const int lane = threadIdx.x & 63, f0 = (threadIdx.x >> 6) - W0;
    double v[IT];
#pragma unroll
    for (int it = 0; it < IT; ++it)
        v[it] = src[(unsigned)min(f0 + NW * it, rows - 1) * (unsigned)ld + (unsigned)min(lane, cols - 1)];
#pragma unroll
    for (int it = 0; it < IT; ++it) {
        const int f = f0 + NW * it;
        if (f < kNB) dst[f * LDX + lane] = v[it];
    }
}

// ------------------------------------------------------------------ the panel's diagonal block
// The 64 x 64 diagonal block A11 = L11 U11 is factored in LDS in four steps of 16 columns by the waves
// 0 .. 3 of the workgroup, two barriers a step:
//   wave 0 factors the 16 x 16 diagonal tile in registers and leaves both inverses, L_ss^{-1} and
//     U_ss^{-1} (factor_tile), while the waves 1 .. 3 finish the tiles of step s-1;
//   waves 0 .. 2 form U_sj = L_ss^{-1} A_sj and L_js = A_js U_ss^{-1}, one j each, on the matrix cores;
//   the tiles below and right of the step take A_ij -= L_is U_sj: the next diagonal tile by wave 0,
//     which goes straight on to factor it, the others by the waves 1 .. 3 beside it.
// No 64 x 64 inverse is formed: the blocks of the panel's row and column need only the inverses of
// the diagonal tiles (strip_solve).
// What bounds it: the chain of 64 dependent pivots (a reciprocal with its Newton step, a multiply
// and a multiply-add each, about 170 cycles with what is placed between them: 3700 cycles a tile) and
// the matrix products of the three tiles that follow each (FP64 MFMA and FMA issue at the same rate
// here, 64 cycles for 16 x 16 x 4).  A panel launch takes 22 us at N = 2048 (42 us with an elimination on
// 4 x 4 register tiles exchanged through LDS, two barriers every four columns, and explicit 64 x 64
// inverses): about 3 us until the operands are in LDS, 16 us for the four steps, 2 us for the stores.

// Orders this wave's LDS accesses where one lane reads what another wrote.
__device__ inline void wave_lds_fence() {
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// x in the lanes of the mask M, 0 or y elsewhere.
template <unsigned long long M>
__device__ inline double keep_lanes(double x) {
    int lo, hi;
    asm("v_cndmask_b32_e64 %0, 0, %1, %2" : "=v"(lo) : "v"(__double2loint(x)), "s"(M));
    asm("v_cndmask_b32_e64 %0, 0, %1, %2" : "=v"(hi) : "v"(__double2hiint(x)), "s"(M));
    return __hiloint2double(hi, lo);
}
template <unsigned long long M>
__device__ inline double merge_lanes(double y, double x) {
    int lo, hi;
    asm("v_cndmask_b32_e64 %0, %1, %2, %3" : "=v"(lo) : "v"(__double2loint(y)), "v"(__double2loint(x)), "s"(M));
    asm("v_cndmask_b32_e64 %0, %1, %2, %3" : "=v"(hi) : "v"(__double2hiint(y)), "v"(__double2hiint(x)), "s"(M));
    return __hiloint2double(hi, lo);
}

#define ROW_FMAC(x, m, l) "v_fmac_f64_dpp " x ", " x ", " m " row_newbcast:" l " row_mask:0xf bank_mask:0xf\n\t"

// One pivot of factor_tile, rows of 16 lanes.  On entry column P of v is up to date and 15 other
// registers wait for the previous pivot's update x += nl (x of row P - 1), nl its negated multipliers:
// columns P + 1 .. 15 of v and 0 .. P - 1 of e.  A wave issues in order, so they are placed between
// the links of this pivot's chain: the pivot in every row (DPP row broadcast), its reciprocal
// (v_rcp_f64 with inv (1 + t + t^2), t its error: t^3 is left), the multipliers, the update of the
// next pivot's column.  The wait states that a DPP operand needs after a vector write are inside the
// statements, as the compiler does not see the instructions; within a statement a register is
// written at least two instructions before a DPP operand reads it.
template <int P>
__device__ __forceinline__ void factor_pivot(double (&v)[16], double (&e)[16], double& nl, double& ri, double& lmax) {
    auto w = [&](int i) -> double& {   // the waiting registers, the next pivot's column first
        if (i == 0) return P < 15 ? v[P < 15 ? P + 1 : 15] : e[14];
        return i - 1 < (P < 15 ? P : 14) ? e[i - 1] : v[i + 1 > 15 ? 15 : i + 1];
    };
    double d, inv, t, l;
    if constexpr (P == 0) {
        asm("s_nop 1\n\t"
            "v_mov_b64_dpp %0, %3 row_newbcast:0 row_mask:0xf bank_mask:0xf\n\t"
            "s_nop 0\n\t"
            "v_rcp_f64_e32 %1, %0\n\t"
            "s_nop 0\n\t"
            "v_fma_f64 %2, -%0, %1, 1.0\n\t"
            "v_fma_f64 %2, %2, %2, %2"
            : "=&v"(d), "=&v"(inv), "=&v"(t)
            : "v"(v[0]));
        inv = fma(t, inv, inv);
        l = -(v[0] * inv);
    } else {
        asm("s_nop 1\n\t"
            "v_mov_b64_dpp %0, %10 row_newbcast:%12 row_mask:0xf bank_mask:0xf\n\t"
            ROW_FMAC("%3", "%11", "%13") ROW_FMAC("%4", "%11", "%13")
            "v_rcp_f64_e32 %1, %0\n\t"
            ROW_FMAC("%5", "%11", "%13") ROW_FMAC("%6", "%11", "%13") ROW_FMAC("%7", "%11", "%13") ROW_FMAC("%8", "%11", "%13")
            "v_fma_f64 %2, -%0, %1, 1.0\n\t"
            ROW_FMAC("%9", "%11", "%13")
            "v_fma_f64 %2, %2, %2, %2"
            : "=&v"(d), "=&v"(inv), "=&v"(t), "+v"(w(0)), "+v"(w(1)), "+v"(w(2)), "+v"(w(3)), "+v"(w(4)), "+v"(w(5)),
              "+v"(w(6))
            : "v"(v[P]), "v"(nl), "n"(P), "n"(P - 1));
        asm("s_nop 1\n\t"
            ROW_FMAC("%2", "%12", "%13")
            "v_fma_f64 %1, %10, %1, %1\n\t"
            ROW_FMAC("%3", "%12", "%13") ROW_FMAC("%4", "%12", "%13")
            "v_mul_f64 %0, %11, -%1\n\t"
            ROW_FMAC("%5", "%12", "%13") ROW_FMAC("%6", "%12", "%13") ROW_FMAC("%7", "%12", "%13") ROW_FMAC("%8", "%12", "%13")
            ROW_FMAC("%9", "%12", "%13")
            : "=&v"(l), "+v"(inv), "+v"(w(7)), "+v"(w(8)), "+v"(w(9)), "+v"(w(10)), "+v"(w(11)), "+v"(w(12)), "+v"(w(13)),
              "+v"(w(14))
            : "v"(t), "v"(v[P]), "v"(nl), "n"(P - 1));
    }
    // lanes of the rows below the pivot; the others keep what they have (a multiplier of 0)
    constexpr unsigned long long below = ((0xffffull << (P + 1)) & 0xffffull) * 0x0001000100010001ull;
    constexpr unsigned long long here = (1ull << P) * 0x0001000100010001ull;
    nl = keep_lanes<below>(l);
    lmax = fmax(lmax, fabs(nl));
    ri = merge_lanes<here>(ri, inv);
    if constexpr (P < 15)
        asm("s_nop 1\n\t" ROW_FMAC("%0", "%1", "%2") : "+v"(v[P < 15 ? P + 1 : 15]) : "v"(nl), "n"(P));
}

// LU of the 16 x 16 tile T (leading dimension LD) by one wave, without interchanges, multipliers by
// the reciprocal pivot: Li = L^{-1} and Ui = U^{-1} (full tiles with zeros, leading dimension LT).  Lanes
// 0 .. 15 hold the rows of [T | I] and take the row operations of the elimination: what becomes of I
// is L^{-1}.  Lanes 16 .. 31 do the same to [T' | I] (T' the transpose): its unit lower factor is
// (D^{-1} U)' with D the pivots, so that what becomes of I, transposed and its column r divided by
// pivot r, is U^{-1}.  Returns whether a multiplier of L exceeds 1 in magnitude or is NaN.
constexpr int LT = 17;   // leading dimension of the inverse tiles
__device__ __forceinline__ bool factor_tile(const double* T, double* Li, double* Ui, int lane) {
    const int r = lane & 15;
    const bool tr = (lane >> 4) & 1;
    double v[16], e[16];
    const double* in = T + (tr ? r : r * LD);
    const int in_step = tr ? LD : 1;
#pragma unroll
    for (int c = 0; c < 16; ++c) v[c] = in[c * in_step];
#pragma unroll
    for (int c = 0; c < 16; ++c) e[c] = r == c ? 1.0 : 0.0;
    double nl = 0.0, ri = 0.0, lmax = 0.0;
    factor_pivot<0>(v, e, nl, ri, lmax);
    factor_pivot<1>(v, e, nl, ri, lmax);
    factor_pivot<2>(v, e, nl, ri, lmax);
    factor_pivot<3>(v, e, nl, ri, lmax);
    factor_pivot<4>(v, e, nl, ri, lmax);
    factor_pivot<5>(v, e, nl, ri, lmax);
    factor_pivot<6>(v, e, nl, ri, lmax);
    factor_pivot<7>(v, e, nl, ri, lmax);
    factor_pivot<8>(v, e, nl, ri, lmax);
    factor_pivot<9>(v, e, nl, ri, lmax);
    factor_pivot<10>(v, e, nl, ri, lmax);
    factor_pivot<11>(v, e, nl, ri, lmax);
    factor_pivot<12>(v, e, nl, ri, lmax);
    factor_pivot<13>(v, e, nl, ri, lmax);
    factor_pivot<14>(v, e, nl, ri, lmax);
    factor_pivot<15>(v, e, nl, ri, lmax);   // no rows below it: nothing waits
    double* out = tr ? Ui + r : Li + r * LT;
    const int out_step = tr ? LT : 1;
    if (!tr) ri = 1.0;
    if (lane < 32) {
#pragma unroll
        for (int c = 0; c < 16; ++c) out[c * out_step] = e[c] * ri;
    }
    // a NaN multiplier has turned its row's e[0] into a NaN
    return __ballot(lane < 16 && !(lmax <= 1.0 && e[0] == e[0])) != 0;
}

// The 16 x 16 tile of D at C: A -= sum_k L_ik U_kj over K / 4 chunks of the operands A (16 rows) and B
// (16 columns), in LDS with leading dimensions LA and LB, in two accumulation chains.  v_mfma_f64_16x16x4 lane
// layout: A[m = l%16][k = l/16], B[k = l/16][n = l%16], D[m = 4 r + l/16][n = l%16] (register r of lane l).
template <int K, int LA, int LB>
__device__ __forceinline__ void tile_mac(v4d& acc0, v4d& acc1, const double* A, const double* B, int lane) {
    const int l16 = lane & 15, l4 = lane >> 4;
    double a[K / 4], b[K / 4];
#pragma unroll
    for (int q = 0; q < K / 4; ++q) {
        a[q] = A[l16 * LA + 4 * q + l4];
        b[q] = B[(4 * q + l4) * LB + l16];
    }
    __builtin_amdgcn_sched_barrier(0);   // every read is out before the first product
#pragma unroll
    for (int q = 0; q < K / 4; q += 2) {
        acc0 = mfma_f64_sub(a[q], b[q], acc0);
        acc1 = mfma_f64_sub(a[q + 1], b[q + 1], acc1);
    }
}
__device__ inline v4d tile_load(const double* C, int lane) {
    v4d acc;
#pragma unroll
    for (int r = 0; r < 4; ++r) acc[r] = C[(4 * r + (lane >> 4)) * LD + (lane & 15)];
    return acc;
}
__device__ inline void tile_store(double* C, v4d acc, int lane) {
#pragma unroll
    for (int r = 0; r < 4; ++r) C[(4 * r + (lane >> 4)) * LD + (lane & 15)] = acc[r];
}
// Step s's update of tile (i, j) of D.
__device__ __forceinline__ void trail_tile(double* D, int s, int i, int j, int lane) {
    double* C = D + 16 * i * LD + 16 * j;
    v4d acc0 = tile_load(C, lane), acc1 = {0.0, 0.0, 0.0, 0.0};
    tile_mac<16, LD, LD>(acc0, acc1, D + 16 * i * LD + 16 * s, D + 16 * s * LD + 16 * j, lane);
    tile_store(C, acc0 + acc1, lane);
}
// Panel p-1's update (all 64 of its columns) of the diagonal block's tiles but the first, spread over
// the waves 1 .. 7 (beside step 0's factor_tile): two or three each.
__device__ __forceinline__ void update_prev_tiles(double* D, const double* Lp, const double* Up, int w, int lane) {
#pragma unroll 1
    for (int q = w; q < 16; q += 7) {
        double* C = D + 16 * (q >> 2) * LD + 16 * (q & 3);
        v4d acc0 = tile_load(C, lane), acc1 = {0.0, 0.0, 0.0, 0.0};
        tile_mac<64, LD, LDB>(acc0, acc1, Lp + 16 * (q >> 2) * LD, Up + 16 * (q & 3), lane);
        tile_store(C, acc0 + acc1, lane);
    }
}

// ------------------------------------------------------------------ 64 x 16 strips
// A wave holds a strip of 16 columns of a 64 x 64 block as four 16 x 16 accumulator tiles.  The
// accumulator layout of the MFMA (register r of lane l: element (4 r + l/16, l%16)) is also the
// layout of its B operand, so a strip feeds the next product straight from its registers.  Blocks
// of the panel's column are taken transposed (L21^T = U11^{-T} A21^T), so that both kinds read
// the diagonal block through the same code with the strides of its row and column exchanged: COL
// (blocks of the panel's row) or not, a compile-time choice, so that every LDS offset is a constant.
//
// L21 is kept for the next launch only, in the strips' own layout: row R0 + 16 e + q of the block's place
// in A holds register q = 4 i + r of strip e, lane by lane (L21[R0 + 16 e + l%16][4 q + l/16] at column
// l), so that a register is stored and loaded as one contiguous 512 bytes.  (Only the last block row can
// have fewer than 64 rows, a multiple of 16 of them.)
template <bool COL>
__device__ inline constexpr int blk_at(int m, int k) { return COL ? m * LD + k : k * LD + m; }

// acc[I] += P_I b: P the 64 x 64 LDS operand, b the strip (64 x 16, negated by its loads).
template <bool COL, int I>
__device__ __forceinline__ void strip_update(v4d (&acc)[4], const double (&b)[16], const double* P, int lane) {
    const int l16 = lane & 15, l4 = lane >> 4;
    double a[16];
#pragma unroll
    for (int q = 0; q < 16; ++q) a[q] = P[COL ? (16 * I + l16) * LD + 4 * q + l4 : (4 * q + l4) * LDB + 16 * I + l16];
    __builtin_amdgcn_sched_barrier(0);   // every read is out before the first product
    v4d odd = {0.0, 0.0, 0.0, 0.0};
#pragma unroll
    for (int q = 0; q < 16; q += 2) {
        acc[I] = mfma_f64(a[q], b[q], acc[I]);
        odd = mfma_f64(a[q + 1], b[q + 1], odd);
    }
    acc[I] += odd;
}

// acc[I] -= sum_{k < I} G_Ik x_k of the forward substitution with G (lower triangular) and the solved
// tiles acc[k] = -x_k.
template <bool COL, int I>
__device__ __forceinline__ void strip_sum(v4d (&acc)[4], const double* D, int lane) {
    const int l16 = lane & 15, l4 = lane >> 4;
    double a[4 * I];
#pragma unroll
    for (int q = 0; q < 4 * I; ++q) a[q] = D[blk_at<COL>(16 * I + l16, 4 * q + l4)];
    __builtin_amdgcn_sched_barrier(0);
    v4d odd = {0.0, 0.0, 0.0, 0.0};
#pragma unroll
    for (int q = 0; q < 4 * I; q += 2) {
        acc[I] = mfma_f64(a[q], acc[q >> 2][q & 3], acc[I]);
        odd = mfma_f64(a[q + 1], acc[q >> 2][(q & 3) + 1], odd);
    }
    acc[I] += odd;
}

// acc[i] = -x_i = -G_ii^{-1} acc[i], inv the inverse tile: L_ii^{-1} or, for the transposed blocks, U_ii^{-1}.
template <bool COL, int I>
__device__ __forceinline__ void strip_solve(v4d (&acc)[4], const double* inv, int lane) {
    const int l16 = lane & 15, l4 = lane >> 4;
    v4d x = {0.0, 0.0, 0.0, 0.0};
#pragma unroll
    for (int q = 0; q < 4; ++q) {
        const int k = 4 * q + l4;
        x = mfma_f64(COL ? inv[l16 * LT + k] : inv[k * LT + l16], acc[I][q], x);
    }
    acc[I] = -x;
}

// Per-surface views for gridDim.z batches of equal size: surface s uses A + s n^2, vectors + s n,
// uinv + s P 64^2, status + 2 s.
struct LuView {
    double *A, *work, *y, *x, *uinv;
    int* status;
};
__device__ inline LuView view(const LuArgs& a) {
    const int s = blockIdx.z, n = a.n, P = (n + kNB - 1) / kNB;
    LuView v;
    v.A = a.A + (long long)s * n * n;
    v.work = a.work + (long long)s * n;
    v.y = a.y + (long long)s * n;
    v.x = a.x + (long long)s * n;
    v.uinv = a.uinv + (long long)s * P * kNB * kNB;
    v.status = a.status + 2 * s;
    return v;
}

// Panel p-1's update C -= A_i B_j of the trailing 64 x 64 tiles r0 .. r1 - 1 (tile r: block row r % nrb,
// block column r / nrb of the blocks from K0 on), A_i = its L21 block, B_j = its U12 block, staged in LDS
// (As alternating between two buffers, Bs kept while the column stays).  The next tile's loads are in
// flight while the current one is multiplied: one workgroup fits a CU, so nothing else hides them.
// Wave w takes rows 16 (w / 2) .. and columns 32 (w % 2) .. of a tile.
__device__ __forceinline__ void update_tiles(const LuView& v, int n, int kp, int K0, int nrb, int r0, int r1, double* As0,
                                             double* As1, double* Bs) {
    const int t = threadIdx.x, lane = t & 63, w = t >> 6, wr = w >> 1, wc = w & 1;
    const int l16 = lane & 15, l4 = lane >> 4;
    constexpr int IT = kNB * kNB / kLuThreads;
    double a[IT], b[IT];
    v4d c[2];
    auto request = [&](int r, bool col) {   // A, C and with a new column B
        const int R0 = K0 + (r % nrb) * kNB, C0 = K0 + (r / nrb) * kNB;
        const int rb = min(kNB, n - R0), cb = min(kNB, n - C0);
        const double* A = v.A + (long long)R0 * n + kp;
#pragma unroll
        for (int it = 0; it < IT; ++it) a[it] = A[(unsigned)min(w + 8 * it, rb - 1) * (unsigned)n + (unsigned)lane];
        if (col) {
            const double* B = v.A + (long long)kp * n + C0;
#pragma unroll
            for (int it = 0; it < IT; ++it) b[it] = B[(unsigned)(w + 8 * it) * (unsigned)n + (unsigned)min(lane, cb - 1)];
        }
        const double* C = v.A + (long long)R0 * n + C0;
#pragma unroll
        for (int j = 0; j < 2; ++j)
#pragma unroll
            for (int q = 0; q < 4; ++q)
                c[j][q] = C[(unsigned)min(wr * 16 + 4 * q + l4, rb - 1) * (unsigned)n + (unsigned)min(wc * 32 + j * 16 + l16, cb - 1)];
    };
    request(r0, true);
    bool col = true;
    for (int r = r0; r < r1; ++r) {
        const int R0 = K0 + (r % nrb) * kNB, C0 = K0 + (r / nrb) * kNB;
        const int rb = min(kNB, n - R0), cb = min(kNB, n - C0);
        double* As = (r - r0) & 1 ? As1 : As0;
        if (col && r > r0) __syncthreads();   // the previous column has been consumed
#pragma unroll
        for (int it = 0; it < IT; ++it) {
            const int f = w + 8 * it;
            As[((f & ~15) + l16) * LD + 4 * (f & 15) + l4] = a[it];
            if (col) Bs[f * LDB + lane] = b[it];
        }
        v4d acc[2] = {c[0], c[1]};
        __syncthreads();
        col = (r + 1) % nrb == 0;
        if (r + 1 < r1) request(r + 1, col);
#pragma unroll
        for (int q = 0; q < 16; ++q) {
            const double x = As[(wr * 16 + l16) * LD + 4 * q + l4];
#pragma unroll
            for (int j = 0; j < 2; ++j) acc[j] = mfma_f64_sub(x, Bs[(4 * q + l4) * LDB + wc * 32 + j * 16 + l16], acc[j]);
        }
        double* C = v.A + (long long)R0 * n + C0;
#pragma unroll
        for (int j = 0; j < 2; ++j)
#pragma unroll
            for (int q = 0; q < 4; ++q) {
                const int row = wr * 16 + 4 * q + l4, cl = wc * 32 + j * 16 + l16;
                if (row < rb && cl < cb) C[(unsigned)row * (unsigned)n + (unsigned)cl] = acc[j][q];
            }
    }
}

// LDS of lu_step_kernel.
struct LuLds {
    double D[kNB * LD];            // the diagonal block; at the end its off-diagonal tiles hold L and U
    double Lp[kNB * LD], Up[kNB * LDB];   // panel p-1's L21 block of row p and U12 block of column p
    double Li[4][16 * LT], Ui[4][16 * LT];   // inverses of the diagonal tiles' factors
    double yv[kNB];
};

// The waves 4 .. 7 of the panel roles: strip w - 4 of the role's own block (role 0 has none: a copy of the
// diagonal block, not used), one step behind the factorisation, with the barriers of lu_panel.
template <bool COL>
__device__ __forceinline__ void lu_strips(const LuView& v, int n, int k0, int kb, int nrb, int role, int w, int lane,
                                          LuLds& S) {
    double *D = S.D, *Lp = S.Lp, *Up = S.Up, *yv = S.yv;
    const int l16 = lane & 15, l4 = lane >> 4;
    const bool prev = k0 > 0;
    const int kp = k0 - kNB;
    __syncthreads();   // the loads below overlap the first step, not the fill of the LDS
    // strip e of the role's own block (role 0 has none: a copy of the diagonal block, not used);
    // element (m, c) of the block at base + m sm + c sc, transposed for row roles
    const unsigned sm = COL ? n : 1, sc = COL ? 1 : n;
    const int blk = role == 0 ? k0 : k0 + kb + (COL ? role - 1 - nrb : role - 1) * kNB;   // its first column (row)
    const int e = 16 * (w - 4) + l16, width = min(kNB, n - blk);
    const bool mine = e < width;
    // loads are clamped, not predicated, so that no branch parts them; what they bring beyond the block
    // meets only zeros of L and U (identity rows and columns beyond kb), and none of it is stored
    const unsigned ec = min(e, width - 1);
    double* base = COL ? v.A + (long long)k0 * n + blk : v.A + (long long)blk * n + k0;
    v4d acc[4];
    double b[16];   // panel p-1's other factor of the strip, the B operand of its update
#pragma unroll
    for (int i = 0; i < 4; ++i)
#pragma unroll
        for (int r = 0; r < 4; ++r) acc[i][r] = base[(unsigned)min(16 * i + 4 * r + l4, kb - 1) * sm + ec * sc];
    if (prev) {
        const double* pb = COL ? v.A + (long long)kp * n + blk : v.A + (long long)blk * n + kp;
        const unsigned e0 = min(16 * (w - 4), width - 16);
#pragma unroll
        for (int q = 0; q < 16; ++q)
            b[q] = -(COL ? pb[(unsigned)(4 * q + l4) * sm + ec * sc] : pb[(e0 + q) * (unsigned)n + (unsigned)lane]);
    }
    const double* P = COL ? Lp : Up;
    const double(*inv)[16 * LT] = COL ? S.Li : S.Ui;
    if (prev) update_prev_tiles(D, Lp, Up, w, lane);
    __syncthreads();   // the inverses of step 0
    if (prev) strip_update<COL, 0>(acc, b, P, lane);
    __syncthreads();   // L and U tiles of step 0
    strip_solve<COL, 0>(acc, inv[0], lane);
    if (prev) strip_update<COL, 1>(acc, b, P, lane);
    strip_sum<COL, 1>(acc, D, lane);
    __syncthreads();   // the inverses of step 1
    strip_solve<COL, 1>(acc, inv[1], lane);
    __syncthreads();   // L and U tiles of step 1
    if (prev) strip_update<COL, 2>(acc, b, P, lane);
    strip_sum<COL, 2>(acc, D, lane);
    __syncthreads();   // the inverses of step 2
    strip_solve<COL, 2>(acc, inv[2], lane);
    __syncthreads();   // L and U tiles of step 2
    if (prev) strip_update<COL, 3>(acc, b, P, lane);
    strip_sum<COL, 3>(acc, D, lane);
    __syncthreads();   // the inverses of step 3
    strip_solve<COL, 3>(acc, inv[3], lane);
    if (role > 0) {
#pragma unroll
        for (int i = 0; i < 4; ++i)
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                const int m = 16 * i + 4 * r + l4;
                if (COL) {
                    if (mine && m < kb) base[(unsigned)m * sm + ec * sc] = -acc[i][r];
                } else if (16 * (w - 4) < width) {
                    base[(unsigned)(16 * (w - 4) + 4 * i + r) * (unsigned)n + (unsigned)lane] = -acc[i][r];
                }
            }
    }
    __syncthreads();   // y
    if (!COL && role > 0) {
        bool bad = false;
        double sum = 0.0;
#pragma unroll
        for (int i = 0; i < 4; ++i)
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                bad |= !(fabs(acc[i][r]) <= 1.0);   // the multipliers against GEPP's pivot rule
                sum -= acc[i][r] * yv[16 * i + 4 * r + l4];
            }
        if (bad && mine) atomicOr(&v.status[0], 1);
        sum += __shfl_xor(sum, 16, 64);
        sum += __shfl_xor(sum, 32, 64);
        if (mine && l4 == 0) v.work[blk + e] -= sum;   // b_i -= L21_i y_p
    }
}

// The panel roles.
__device__ __forceinline__ void lu_panel(const LuView& v, int n, int k0, int kb, int nrb, int role, LuLds& S) {
    double *D = S.D, *Lp = S.Lp, *Up = S.Up, *yv = S.yv;
    const int t = threadIdx.x, lane = t & 63, w = __builtin_amdgcn_readfirstlane(t >> 6);
    const int l16 = lane & 15, l4 = lane >> 4;
    const bool prev = k0 > 0;
    const int kp = k0 - kNB;
    v4d first;   // wave 0: the first diagonal tile, with panel p-1's update
    if (w == 0) {
        // its operands straight into the MFMA's registers, so that it is ready when the other waves have
        // filled the LDS
        const double* C = v.A + (long long)k0 * n + k0;
#pragma unroll
        for (int r = 0; r < 4; ++r) first[r] = C[(unsigned)min(4 * r + l4, kb - 1) * (unsigned)n + (unsigned)min(l16, kb - 1)];
        if (prev) {
            const double* lp = v.A + (long long)k0 * n + kp;
            const double* up = v.A + (long long)kp * n + k0;
            double a[16], b[16];
#pragma unroll
            for (int q = 0; q < 16; ++q) {
                a[q] = lp[(unsigned)min(q, kb - 1) * (unsigned)n + (unsigned)lane];
                b[q] = up[(unsigned)(4 * q + l4) * (unsigned)n + (unsigned)min(l16, kb - 1)];
            }
            v4d c1 = {0.0, 0.0, 0.0, 0.0};
#pragma unroll
            for (int q = 0; q < 16; q += 2) {
                first = mfma_f64_sub(a[q], b[q], first);
                c1 = mfma_f64_sub(a[q + 1], b[q + 1], c1);
            }
            first += c1;
        }
#pragma unroll
        for (int r = 0; r < 4; ++r)
            if (4 * r + l4 >= kb || l16 >= kb) first[r] = 4 * r + l4 == l16 ? 1.0 : 0.0;
        yv[lane] = v.work[k0 + min(lane, kb - 1)];
        if (lane >= kb) yv[lane] = 0.0;
#pragma unroll
        for (int r = 0; r < 4; ++r) asm volatile("" : "+v"(first[r]));   // formed here, not behind the barrier
    } else {
        load_rows<LD, 1, 7>(D, v.A + (long long)k0 * n + k0, n, kb, kb);
        if (prev) {
            load_l21<1, 7>(Lp, v.A, n, k0, kp, kb);
            load_rows<LDB, 1, 7>(Up, v.A + (long long)kp * n + k0, n, kNB, kb);
        }
        if (kb < kNB) {   // beyond kb: identity rows and columns, and nothing to update them with
#pragma unroll 1
            for (int f = w - 1; f < kNB; f += 7) {   // each wave the rows that it stored
                if (f >= kb || lane >= kb) D[f * LD + lane] = f == lane ? 1.0 : 0.0;
                if (prev && lane >= kb) Up[f * LDB + lane] = 0.0;
                const int r = (f & ~15) + l16;
                if (prev && r >= kb) Lp[r * LD + 4 * (f & 15) + l4] = 0.0;
            }
        }
    }
    // From here the two halves of the workgroup run their own code, with the same barriers.
    if (w >= 4) {
        if (role > nrb)
            lu_strips<true>(v, n, k0, kb, nrb, role, w, lane, S);
        else
            lu_strips<false>(v, n, k0, kb, nrb, role, w, lane, S);
        return;
    }
    __builtin_amdgcn_s_setprio(2);   // the chain's waves before the strips' on a shared SIMD
    bool bad = false;
    __syncthreads();
    if (w == 0) {
        tile_store(D, first, lane);
    } else if (prev) {
        update_prev_tiles(D, Lp, Up, w, lane);
    }
    // `ln` keeps what depends on the lane out of the compiler's hoisting from the loop
#pragma unroll 1
    for (int s = 0; s < 4; ++s) {
        int ln = lane;
        asm volatile("" : "+v"(ln));
        if (w == 0) {
            wave_lds_fence();   // the diagonal tile's last update, by this wave
            bad |= factor_tile(D + 16 * s * (LD + 1), S.Li[s], S.Ui[s], ln);
        }
        __syncthreads();
        const int m16 = ln & 15, m4 = ln >> 4;
        if (w < 3 - s) {   // U_sj = L_ss^{-1} A_sj and L_js^T = U_ss^{-T} A_js^T, j = s + 1 + w
            const int j = s + 1 + w;
            double* Uj = D + 16 * s * LD + 16 * j;
            double* Lj = D + 16 * j * LD + 16 * s;
            v4d u = {0.0, 0.0, 0.0, 0.0}, l = u;
            double ua[4], ub[4], la[4], lb[4];
#pragma unroll
            for (int q = 0; q < 4; ++q) {
                ua[q] = S.Li[s][m16 * LT + 4 * q + m4];
                ub[q] = Uj[(4 * q + m4) * LD + m16];
                la[q] = S.Ui[s][(4 * q + m4) * LT + m16];
                lb[q] = Lj[m16 * LD + 4 * q + m4];
            }
            v4d a0 = tile_load(D + 16 * j * (LD + 1), ln);   // wave 0: the next diagonal tile
            __builtin_amdgcn_sched_barrier(0);
#pragma unroll
            for (int q = 0; q < 4; ++q) {
                u = mfma_f64(ua[q], ub[q], u);
                l = mfma_f64(la[q], lb[q], l);
            }
            if (w == 0) {   // the next diagonal tile, its operands at hand: l is the A operand, u the B operand
                double* C = D + 16 * j * (LD + 1);
                v4d a1 = {0.0, 0.0, 0.0, 0.0};
                a0 = mfma_f64_sub(l[0], u[0], a0);
                a1 = mfma_f64_sub(l[1], u[1], a1);
                a0 = mfma_f64_sub(l[2], u[2], a0);
                a1 = mfma_f64_sub(l[3], u[3], a1);
                tile_store(C, a0 + a1, ln);
            }
            tile_store(Uj, u, ln);
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                Lj[m16 * LD + 4 * r + m4] = l[r];
                bad |= !(fabs(l[r]) <= 1.0);
            }
        }
        if (w == 3) {   // y_s = L_ss^{-1} b_s, row m16, four k per lane
            double ys = 0.0;
#pragma unroll
            for (int q = 0; q < 4; ++q) ys = fma(S.Li[s][m16 * LT + 4 * m4 + q], yv[16 * s + 4 * m4 + q], ys);
            ys += __shfl_xor(ys, 16, 64);
            ys += __shfl_xor(ys, 32, 64);
            wave_lds_fence();   // every lane has read b_s
            if (ln < 16) yv[16 * s + ln] = ys;
        }
        __syncthreads();
        if (w > 0) {   // the other tiles (i, j) > s
            const int m = 3 - s;
            for (int q = w; q < m * m; q += 3)
                trail_tile(D, s, s + 1 + q / m, s + 1 + q % m, ln);
            if (w == 3 && ln >= 16 * (s + 1)) {   // b of the rows below
                double ay = yv[ln];
#pragma unroll
                for (int k = 0; k < 16; ++k) ay = fma(-D[ln * LD + 16 * s + k], yv[16 * s + k], ay);
                yv[ln] = ay;
            }
        }
    }
    if (role == 0) {
        if (bad) atomicOr(&v.status[0], 1);
        if (t < kb) v.y[k0 + t] = yv[t];
        // U11^{-1}, column strip w: X_w = U_ww^{-1}, X_i = -U_ii^{-1} sum_{i < k <= w} U_ik X_k
        v4d X[4];
        double* U = v.uinv + (long long)(k0 / kNB) * kNB * kNB;
#pragma unroll
        for (int i = 3; i >= 0; --i) {
            v4d x4 = {0.0, 0.0, 0.0, 0.0};
            if (i == w) {
#pragma unroll
                for (int r = 0; r < 4; ++r) {
                    const int m = 4 * r + l4;
                    x4[r] = S.Ui[i][m * LT + l16];
                }
            } else if (i < w) {
                v4d sum = {0.0, 0.0, 0.0, 0.0};
#pragma unroll
                for (int k = i + 1; k < 4; ++k)
                    if (k <= w) {
#pragma unroll
                        for (int q = 0; q < 4; ++q)
                            sum = mfma_f64_sub(D[(16 * i + l16) * LD + 16 * k + 4 * q + l4], X[k][q], sum);
                    }
#pragma unroll
                for (int q = 0; q < 4; ++q) {
                    const int k = 4 * q + l4;
                    x4 = mfma_f64(S.Ui[i][l16 * LT + k], sum[q], x4);
                }
            }
            X[i] = x4;
#pragma unroll
            for (int r = 0; r < 4; ++r) U[(16 * i + 4 * r + l4) * kNB + 16 * w + l16] = x4[r];
        }
    }
}

// An entry of x that is not there yet: a signalling NaN, which no arithmetic gives.  The first panel's launch fills x with it.
constexpr unsigned long long kNoValue = 0x7ff0dead00000001ull;

// Panel p (columns k0 .. k0 + kb - 1) together with the previous panel's trailing update
// (kp = k0 - 64; A22 -= L21 U12 with panel p-1's blocks), one launch per panel:
//   roles 0 .. 2 nrb (panel p): each applies panel p-1's update to the diagonal block A_pp (kept in
//     LDS; the diagonal blocks are never stored) and factors it (waves 0 .. 3) while the waves 4 .. 7,
//     one 16-wide strip each, apply the update to the role's own block A_ip (row roles) or A_pj
//     (column roles) and follow the factorisation with their forward substitution, one 16-row tile
//     behind; row roles leave L21_i = A_ip U11^{-1} and b_i -= L21_i y_p, column roles
//     U12_j = L11^{-1} A_pj, role 0 U11^{-1} and y_p = L11^{-1} b_p;
//   roles above 2 nrb: panel p-1's update of the trailing tiles (i, j), i, j > p, that no panel
//     role owns, an equal share of them each (lu_step_grid).
// Panel p's dependency chain (the diagonal block) thereby runs beside the bulk of the previous
// panel's update rather than after it.
__global__ __launch_bounds__(kLuThreads) void lu_step_kernel(LuArgs a, int k0) {
    __shared__ LuLds S;
    const LuView v = view(a);
    const int n = a.n, t = threadIdx.x;
    const int kb = min(kNB, n - k0);
    const int nrb = (n - k0 - kb + kNB - 1) / kNB;
    const int role = blockIdx.x;
    if (k0 == 0 && role == 0) {
        unsigned long long* x = reinterpret_cast<unsigned long long*>(v.x);
        for (int i = t; i < n; i += kLuThreads) x[i] = kNoValue;
    }
    if (role > 2 * nrb) {   // trailing tiles of panel p-1's update (only when k0 > 0)
        const int wgs = gridDim.x - 1 - 2 * nrb, i = role - 1 - 2 * nrb, tiles = nrb * nrb;
        update_tiles(v, n, k0 - kNB, k0 + kb, nrb, (int)((long long)tiles * i / wgs), (int)((long long)tiles * (i + 1) / wgs),
                     S.D, S.Lp, S.Up);
    } else {
        lu_panel(v, n, k0, kb, nrb, role, S);
    }
}

// Unblocked GEPP (first row of maximal |a|) and solve of A x = b by one workgroup of 256 threads.
__device__ void gepp_solve(int n, double* A, const double* b, double* x, int* piv, int* counters) {
    if (threadIdx.x == 0) atomicAdd(&counters[0], 1);
    __shared__ double rv[256];
    __shared__ int ri[256];
    const int t = threadIdx.x;
    for (int i = t; i < n; i += blockDim.x) x[i] = b[i];
    __syncthreads();
    for (int j = 0; j < n; ++j) {
        double best = -1.0;
        int bi = n;
        for (int i = j + t; i < n; i += blockDim.x) {
            const double vv = fabs(A[(long long)i * n + j]);
            if (vv > best) { best = vv; bi = i; }
        }
        rv[t] = best;
        ri[t] = bi;
        __syncthreads();
        for (int s = 128; s > 0; s >>= 1) {
            if (t < s) {
                if (rv[t + s] > rv[t] || (rv[t + s] == rv[t] && ri[t + s] < ri[t])) {
                    rv[t] = rv[t + s];
                    ri[t] = ri[t + s];
                }
            }
            __syncthreads();
        }
        const int pr = ri[0];
        if (t == 0) piv[j] = pr;
        if (pr != j && pr < n) {
            for (int c = t; c < n; c += blockDim.x) {
                const double tmp = A[(long long)j * n + c];
                A[(long long)j * n + c] = A[(long long)pr * n + c];
                A[(long long)pr * n + c] = tmp;
            }
            if (t == 0) {
                const double tmp = x[j];
                x[j] = x[pr];
                x[pr] = tmp;
            }
        }
        __syncthreads();
        const double d = A[(long long)j * n + j];
        if (d == 0.0) {   // exactly singular column: getrf records it and moves on
            __syncthreads();
            continue;
        }
        const double xj = x[j];
        for (int i = j + 1 + t; i < n; i += blockDim.x) {
            double* Ri = A + (long long)i * n;
            const double l = Ri[j] / d;
            Ri[j] = l;
            const double* Rj = A + (long long)j * n;
            for (int c = j + 1; c < n; ++c) Ri[c] -= l * Rj[c];
            x[i] -= l * xj;
        }
        __syncthreads();
    }
    for (int i = n - 1; i >= 0; --i) {
        if (t == 0) x[i] = x[i] / A[(long long)i * n + i];
        __syncthreads();
        const double xi = x[i];
        for (int r = t; r < i; r += blockDim.x) x[r] -= A[(long long)r * n + i] * xi;
        __syncthreads();
    }
}

// For a system of its own (A holds it as it was): run only when the interchange-free factorisation reported a
// multiplier above 1 (status[2 s] != 0).
__global__ __launch_bounds__(256) void gepp_fallback_kernel(const SurfDesc* sd, double* M, const double* bvec,
                                                            double* xvec, int* pivv, int* status,
                                                            int* counters) {
    const int s_ = blockIdx.x;
    if (status[2 * s_] == 0) return;
    const SurfDesc dsc = sd[s_];
    gepp_solve(dsc.n, M + dsc.moff, bvec + dsc.voff, xvec + dsc.voff, pivv + dsc.voff, counters);
}

// The stepper's fallback, by one workgroup: the matrix of surface s as assemble64_kernel forms it (createM.cuh:43-92),
// then the elimination with interchanges.
__device__ void fallback_solve(const LuFallback& f, int s) {
    const SurfDesc d = f.sd[s];
    const int n = d.n;
    const NodeTrig* tr = f.trig + d.voff;
    double* A = f.M + d.moff;
    const bool water = f.ph.kind == 0;
    const double c = water ? 0.25 * (1 - f.ph.rho) / kPi : 0.25 / kPi, ci = 0.25 / kPi;
    const double h = f.ph.depth, eh = exp(h), ehi = exp(-h);
    for (int k = 0; k < n; ++k) {
        const NodeTrig tk = tr[k];
        const double2 zp = f.Zp[d.voff + k];
        for (int j = threadIdx.x; j < n; j += 256) {
            double v;
            if (j == k) {
                v = (water ? 0.5 * (1 + f.ph.rho) : 0.5) + c * cdiv(f.Zpp[d.voff + k], zp).y;
                if (f.ph.image) v -= ci * cot64(0.0, f.Z[d.voff + k].y + h).y;
            } else {
                const CotParts cp = cot_parts(tk, tr[j]);
                v = cp.id * (c * zp.y * cp.p - c * zp.x * cp.q);
                if (f.ph.image) {
                    const CotParts cq = cot_image_parts(tk, tr[j], eh, ehi);
                    v += ci * (cq.q * cq.id);
                }
            }
            A[(long long)k * n + j] = v;
        }
    }
    __syncthreads();
    gepp_solve(n, A, f.b + d.voff, f.x + d.voff, f.piv + d.voff, f.counters);
}

// x_p = U_pp^{-1} (y_p - sum_{q>p} U_pq x_q).  Workgroup b handles block row p = P-1-b, so a workgroup only waits for
// workgroups dispatched before it; every wait is bounded.  The chain from x_{p+1} to x_p bounds the launch, so nothing
// else is on it: the entries of x are polled themselves (agent scope, past the XCDs' L2 caches; a flag would add a fence
// and a load behind it), thread (r, chunk) holds its 16 entries of U_pq in registers, loaded while it waits for the block
// before, and one barrier separates the blocks.  N = 2048 67 -> 52 us,
// N = 768 25 -> 21, N = 256 9.5 -> 7.7; with 8-byte loads of the rows 75 at N = 2048, as much as through LDS.
// FALLBACK: when the factorisation needed interchanges, the surface's first workgroup solves its system anew instead
// (fallback_solve); as launches of their own the two kernels of that cost every solve 9 us to find nothing to do.
template <bool FALLBACK>
__global__ __launch_bounds__(256) void lu_backsolve_kernel(LuArgs a, LuFallback f) {
    __shared__ double xq[2][kNB], part[4][kNB], sv[kNB];
    const LuView v = view(a);
    const int n = a.n, t = threadIdx.x;
    const int P = (n + kNB - 1) / kNB;
    const int p = P - 1 - blockIdx.x;
    const int R0 = p * kNB, rb = min(kNB, n - R0);
    const int r = t & 63, chunk = t >> 6;
    const int bad = FALLBACK ? v.status[0] : 0;
    // 16 entries of row r of block U_pq, one 128-byte line of it; a row or column beyond the matrix is read clamped and
    // meets a zero of x (or is not used).  n is even when there are several blocks: 16-byte loads.
    const double* Ar = v.A + (long long)(R0 + min(r, rb - 1)) * n;
    auto load = [&](int q, double (&u)[16]) {
        const int c0 = q * kNB + chunk * 16;
        if ((q + 1) * kNB <= n) {
#pragma unroll
            for (int c = 0; c < 16; c += 2) {
                const double2 w = *reinterpret_cast<const double2*>(Ar + c0 + c);
                u[c] = w.x;
                u[c + 1] = w.y;
            }
        } else {
#pragma unroll
            for (int c = 0; c < 16; ++c) u[c] = Ar[min(c0 + c, n - 1)];
        }
    };
    double ui[16], u[16], un[16];
    const double2* U = reinterpret_cast<const double2*>(v.uinv + (long long)p * kNB * kNB + r * kNB + chunk * 16);
#pragma unroll
    for (int c = 0; c < 8; ++c) {
        const double2 w = U[c];
        ui[2 * c] = w.x;
        ui[2 * c + 1] = w.y;
    }
    const double y = t < rb ? v.y[R0 + t] : 0.0;
    if (P > 1) load(P - 1, u);
    if (FALLBACK && bad) {
        if (blockIdx.x == 0) fallback_solve(f, f.first + blockIdx.z);
        return;
    }
    double acc[4] = {0.0, 0.0, 0.0, 0.0};
    for (int q = P - 1; q > p; --q) {
        load(max(q - 1, p), un);
        if (t < kNB) {
            unsigned long long bits = 0;   // 0.0 beyond the matrix
            if (q * kNB + t < n) {
                const unsigned long long* x = reinterpret_cast<const unsigned long long*>(v.x) + q * kNB + t;
                int spins = 0;
                while ((bits = __hip_atomic_load(x, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT)) == kNoValue) {
                    if (++spins > (1 << 22)) {
                        atomicOr(&v.status[1], 1);
                        break;
                    }
                }
            }
            xq[q & 1][t] = __longlong_as_double((long long)bits);
        }
        __syncthreads();   // two buffers: this one is written again only after the next barrier
#pragma unroll
        for (int c = 0; c < 16; ++c) acc[c & 3] += u[c] * xq[q & 1][chunk * 16 + c];
#pragma unroll
        for (int c = 0; c < 16; ++c) u[c] = un[c];
    }
    part[chunk][r] = (acc[0] + acc[1]) + (acc[2] + acc[3]);
    __syncthreads();
    if (t < kNB) sv[t] = t < rb ? y - (part[0][t] + part[1][t] + part[2][t] + part[3][t]) : 0.0;
    __syncthreads();
    {   // x_p = U_pp^{-1} sv, 4 threads per row
        double s[4] = {0.0, 0.0, 0.0, 0.0};
#pragma unroll
        for (int c = 0; c < 16; ++c) s[c & 3] += ui[c] * sv[chunk * 16 + c];
        part[chunk][r] = (s[0] + s[1]) + (s[2] + s[3]);
    }
    __syncthreads();
    if (t < rb)
        __hip_atomic_store(v.x + R0 + t, part[0][t] + part[1][t] + part[2][t] + part[3][t], __ATOMIC_RELAXED,
                           __HIP_MEMORY_SCOPE_AGENT);
}
template __global__ void lu_backsolve_kernel<false>(LuArgs, LuFallback);
template __global__ void lu_backsolve_kernel<true>(LuArgs, LuFallback);

}  // namespace sfh
