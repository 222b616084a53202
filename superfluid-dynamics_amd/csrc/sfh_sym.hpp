// sfh_sym.hpp -- pair sweeps of the per-surface workgroup kernel that evaluate every unordered node
// pair once.
//
// The pair kernel of the dipole matrix and of the velocity is antisymmetric,
// cot((z_j - z_k)/2) = -cot((z_k - z_j)/2): in the parts of cot_parts, p and q change sign with the
// order of the pair and id does not.  In the image cotangent cot((z_k - conj z_j)/2 + i h), p changes
// sign and q and id do not.  One evaluation therefore gives the matrix entries (k, j) and (j, k) and
// the pair's contributions to the sums of both rows, about half the arithmetic of a sweep over
// ordered pairs.
//
// Geometry.  The N nodes form nb = ceil(N / 64) blocks of 64.  A tile (I, J) pairs the rows of block
// I with the columns of block J; at offset r (0..63) lane l takes row I*64 + l and column
// J*64 + (l + r) % 64, so the 64 lanes of a wave touch 64 distinct columns.  Row sums accumulate in
// registers.  Column (mirror) sums accumulate in a register that moves one lane down after every
// offset (DPP wave rotate), so at offset r lane l holds the sum of column (l + r) % 64.
//
// Work split.  Each wave owns one block row I; with nb < 16 blocks, wpb = 16 / nb waves share a block
// row and split the offsets of each of its tiles.  Every pair of blocks is visited once: phase 0 takes
// the diagonal tile (I, I) at offsets 1..32 (at offset 32 lanes l and l + 32 take the same pair, so
// that offset adds no column sums), phases d = 1 .. (nb - 1) / 2 the tiles (I, I + d), and for even
// nb a last phase the tile (I, I + nb / 2) at offsets 1..32 when I < nb / 2 and 0..31 otherwise
// (together every pair of the two blocks once).  In any phase each block receives column sums from
// one block row only, so the column sums go into an LDS slot per sub-wave without atomics; a barrier
// separates the phases, and every sum is formed in a fixed order.
//
// Parts.  A surface's sweeps can be split into a few parts, each for a workgroup of its own (sfh_cluster.hpp):
// part p of P takes its share of every range of offsets, as if the sub-waves of a block row were P times as many.
//
// Stored matrix.  A wave keeps the entries it forms for its own products: the offset that is the q-th of
// block row I (phase 0's offsets, then phase 1's, ...) holds its 64 direct entries M_kj at row 2 q and the
// mirrored ones M_jk (0 where there are none) at row 2 q + 1 of the block row's 64 nb rows of 64 elements; lane l's are at element l.  The
// product repeats the sweep with loads in place of evaluations, so a wave reads what it wrote itself, in contiguous
// rows, and no other workgroup's stores.  Entries of nodes beyond N are 0; the diagonal stays in LDS.
#pragma once
#include <type_traits>

#include "sfh_cluster.hpp"
#include "sfh_wg.hpp"

namespace sfh {

// v from lane (l + 1) % 64 (wave rotate left by one lane; every lane active).
__device__ inline double dpp_rol1(double v) {
    const int lo = __builtin_amdgcn_mov_dpp(__double2loint(v), 0x134, 0xf, 0xf, false);
    const int hi = __builtin_amdgcn_mov_dpp(__double2hiint(v), 0x134, 0xf, 0xf, false);
    return __hiloint2double(hi, lo);
}

struct SymGeo {
    int nb;       // blocks of 64 nodes
    int wpb;      // waves per block row
    int I, sub;   // this wave's block row and its index among the wpb waves of that row
    int l;        // lane
    bool active;  // the wave takes part (waves beyond nb * wpb idle)
};

__device__ inline SymGeo sym_geo(int n) {
    SymGeo g;
    const int w = __builtin_amdgcn_readfirstlane(threadIdx.x / kTile);   // wave-uniform: scalar
    g.nb = (n + kTile - 1) / kTile;
    g.wpb = kBW / g.nb;
    g.I = w / g.wpb;
    g.sub = w % g.wpb;
    g.l = threadIdx.x % kTile;
    g.active = g.I < g.nb;
    return g;
}

// This wave's share of phase ph: offsets r0 .. r1 of block column J, of which those below rm have mirrored entries;
// offset r is number q0 + r of the block row.
struct SymRange {
    int J, r0, r1, rm, q0;
};
__device__ inline SymRange sym_range(const SymGeo& g, int ph, int part, int parts) {
    SymRange s;
    s.J = (g.I + ph) % g.nb;
    int lo, hi;
    if (ph == 0) {
        lo = 1;
        hi = 33;
    } else if (2 * ph < g.nb) {
        lo = 0;
        hi = kTile;
    } else {
        lo = g.I < g.nb / 2 ? 1 : 0;
        hi = lo + 32;
    }
    const int i = part * g.wpb + g.sub, m = parts * g.wpb;
    s.r0 = lo + ((hi - lo) * i) / m;
    s.r1 = lo + ((hi - lo) * (i + 1)) / m;
    // offset 32 of the diagonal tile (no column sums) is the last offset of its range
    s.rm = (ph == 0 && s.r1 == 33) ? 32 : s.r1;
    s.q0 = (ph == 0 ? 0 : 32 + kTile * (ph - 1)) - lo;
    return s;
}

// sym_sweep for n a multiple of 64 (FULL) or not.
template <int NA, bool FULL, class F>
__device__ inline void sym_sweep_impl(int n, double* const (&acc)[NA], F& pair, int part, int parts) {
    const SymGeo g = sym_geo(n);
    const int t = threadIdx.x;
    const int stride = g.nb * kTile;
#pragma unroll
    for (int a = 0; a < NA; ++a) acc[a][t] = 0.0;
    __syncthreads();
    double row[NA];
#pragma unroll
    for (int a = 0; a < NA; ++a) row[a] = 0.0;
    const int k = g.I * kTile + g.l;
    const int nphase = g.nb / 2 + 1;
    for (int ph = 0; ph < nphase; ++ph) {
        if (g.active) {
            const SymRange s = sym_range(g, ph, part, parts);
            double col[NA];
#pragma unroll
            for (int a = 0; a < NA; ++a) col[a] = 0.0;
            for (int r = s.r0; r < s.rm; ++r) {
                const int j = s.J * kTile + ((g.l + r) & (kTile - 1));
                pair(k, j, s.q0 + r, std::true_type{}, std::integral_constant<bool, FULL>{}, row, col);
#pragma unroll
                for (int a = 0; a < NA; ++a) col[a] = dpp_rol1(col[a]);
            }
            if (s.rm < s.r1) {
                const int j = s.J * kTile + ((g.l + 32) & (kTile - 1));
                pair(k, j, s.q0 + 32, std::false_type{}, std::integral_constant<bool, FULL>{}, row, col);
#pragma unroll
                for (int a = 0; a < NA; ++a) col[a] = dpp_rol1(col[a]);
            }
            if (s.r1 > s.r0) {
                const int c = s.J * kTile + ((g.l + s.r1) & (kTile - 1));
#pragma unroll
                for (int a = 0; a < NA; ++a) acc[a][g.sub * stride + c] += col[a];
            }
        }
        __syncthreads();
    }
    if (g.active) {
#pragma unroll
        for (int a = 0; a < NA; ++a) acc[a][g.sub * stride + k] += row[a];
    }
    __syncthreads();
}

// The sweep.  acc[a] (a < NA) are LDS arrays of kBT doubles: slot s of node i at s * nb * 64 + i.
// pair(k, j, q, mirror, full, row, col) is called by every lane of an active wave for row
// k = I*64 + l and column j = J*64 + (l + r) % 64, q the offset's number in the block row; it adds the pair's contribution to row k into
// row[] and, when mirror, to row j into col[].  mirror and full are std::integral_constant<bool>:
// mirror is false only at offset 32 of the diagonal tile, and full (n a multiple of 64) says that
// k and j are always < n, so the functor checks them only when it is false.  On return the total
// of node t is sym_total(acc[a], n); the caller synchronises before reusing acc.
template <int NA, class F>
__device__ inline void sym_sweep(int n, double* const (&acc)[NA], F& pair, int part, int parts) {
    if ((n & (kTile - 1)) == 0)
        sym_sweep_impl<NA, true>(n, acc, pair, part, parts);
    else
        sym_sweep_impl<NA, false>(n, acc, pair, part, parts);
}

// The total of node t (< n) over the slots of a sweep's accumulator.
__device__ inline double sym_total(const double* acc, int n) {
    const int nb = (n + kTile - 1) / kTile, wpb = kBW / nb, t = threadIdx.x;
    double s = 0.0;
    for (int q = 0; q < wpb; ++q) s += acc[q * nb * kTile + t];
    return s;
}

// This lane's row of the sweeps: k = I*64 + l (rows >= n are padding; k < 1024 always).
__device__ inline int sym_row(int n) {
    const SymGeo g = sym_geo(n);
    return g.I * kTile + g.l;
}

// Off-diagonal entries e = M_kj and em = M_jk of M = I/2 + K (createM.cuh:43-92) from one
// evaluation of the pair cotangents: with cot((z_k - z_j)/2) = (p - i q) id,
//   M_kj = c id (y'_k p - x'_k q) [+ ci q' id'],  M_jk = c id (x'_j q - y'_j p) [+ ci q' id'],
// where (p', q', id') are the image cotangent's parts (q' and id' symmetric in k, j).  czk = c Z'_k.
__device__ inline void entry_pair(const NodeTrig& tk, const NodeTrig& tj, double2 czk, double2 zj,
                                  const PairConst& pc, double& e, double& em) {
    const CotParts cp = cot_parts(tk, tj);
    e = cp.id * (czk.y * cp.p - czk.x * cp.q);
    em = (pc.c * cp.id) * (zj.x * cp.q - zj.y * cp.p);
    if (pc.image) {
        const CotParts cq = cot_image_parts(tk, tj, pc.eh, pc.ehi);
        const double im = pc.ci * (cq.q * cq.id);
        e += im;
        em += im;
    }
}

// The sums of a sweep over all parts of the surface: out[a] is the total of node t on threads t < n.  A workgroup
// sweeps its own parts; with several workgroups the parts' sums meet in the exchange buffer and every workgroup
// adds them in the parts' order.
template <int NA, class F>
__device__ inline void sym_sums(int n, double* const (&acc)[NA], F&& pair, Cluster& cl, double (&out)[NA]) {
    const int t = threadIdx.x;
    if (cl.parts == 1) {
        sym_sweep<NA>(n, acc, pair, 0, 1);
#pragma unroll
        for (int a = 0; a < NA; ++a) out[a] = t < n ? sym_total(acc[a], n) : 0.0;
        return;
    }
    for (int p = cl.rank; p < cl.parts; p += cl.members) {
        sym_sweep<NA>(n, acc, pair, p, cl.parts);
        if (t < n) {
#pragma unroll
            for (int a = 0; a < NA; ++a) cl.put(n, p * NA + a, sym_total(acc[a], n));
        }
        __syncthreads();
    }
    cl.exchange<NA>(n, out);
}

// (M v)_t evaluated matrix-free in FP64 (entry_pair and the diagonal), v in L.vs with the padding
// entries 0 (the caller has synchronised).  Returns the value on threads t < n, 0 elsewhere.
__device__ inline double mv_free_sym(int n, const PairConst& pc, Cluster& cl, BLds& L) {
    const int t = threadIdx.x;
    const int kr = sym_row(n);
    const NodeTrig tk = L.tr[kr];
    const double2 zq = L.zp[kr];
    const double2 czk = make_double2(pc.c * zq.x, pc.c * zq.y);
    const double vk = L.vs[kr];
    double* const acc[1] = {L.part};
    double w[1];
    sym_sums<1>(n, acc, [&](int k, int j, int, auto mirror, auto full, double (&row)[1], double (&col)[1]) {
        if (!decltype(full)::value && (k >= n || j >= n)) return;
        double e, em;
        entry_pair(tk, L.tr[j], czk, L.zp[j], pc, e, em);
        row[0] += e * L.vs[j];
        if constexpr (decltype(mirror)::value) col[0] += em * vk;
    }, cl, w);
    if (t < n) w[0] += L.diag[t] * L.vs[t];
    __syncthreads();
    return w[0];
}

// The cotangent sums of v (L.vs) that (M v)_t and the velocity share: out = sum_j v_j of Re and Im cot((z_t - z_j)/2)
// over j != t, and for the film (NA = 4) of cot((z_t - conj z_j)/2 + i h).  acc: NA LDS arrays of kBT doubles.
template <int NA>
__device__ inline void cot_sums(int n, double* const (&acc)[NA], const PairConst& pc, Cluster& cl, BLds& L, double (&out)[NA]) {
    static_assert(NA == 2 || NA == 4, "water or film");
    const int kr = sym_row(n);
    const NodeTrig tk = L.tr[kr];
    const double vk = L.vs[kr];
    sym_sums<NA>(n, acc, [&](int k, int j, int, auto mirror, auto full, double (&row)[NA], double (&col)[NA]) {
        if (!decltype(full)::value && (k >= n || j >= n)) return;
        const NodeTrig tj = L.tr[j];
        const double vj = L.vs[j];
        const CotParts cp = cot_parts(tk, tj);
        const double w = vj * cp.id;
        row[0] += w * cp.p;
        row[1] -= w * cp.q;
        if constexpr (decltype(mirror)::value) {   // p, p' change sign with the pair's order, q changes, q' not
            const double wk = vk * cp.id;
            col[0] -= wk * cp.p;
            col[1] += wk * cp.q;
        }
        if constexpr (NA == 4) {
            const CotParts cq = cot_image_parts(tk, tj, pc.eh, pc.ehi);
            const double wi = vj * cq.id;
            row[2] += wi * cq.p;
            row[3] -= wi * cq.q;
            if constexpr (decltype(mirror)::value) {
                const double wki = vk * cq.id;
                col[2] -= wki * cq.p;
                col[3] -= wki * cq.q;
            }
        }
    }, cl, out);
}
// (M v)_t from them; t < n.
template <int NA>
__device__ inline double product_of_sums(const double (&s)[NA], const PairConst& pc, double2 zp, double diag, double v) {
    double w = pc.c * (zp.x * s[1] + zp.y * s[0]) + diag * v;
    if constexpr (NA == 4) w -= pc.ci * s[3];
    return w;
}

// (M v)_t for the matrix that the waves stored (see above), v in L.vs with L.vs[j] = 0 for n <= j < nb*64
// (the caller has synchronised).  Returns the value on threads t < n, 0 elsewhere.
template <typename T>
__device__ inline double mv_pairs(const T* __restrict__ M, int n, Cluster& cl, BLds& L) {
    const SymGeo g = sym_geo(n);
    const int t = threadIdx.x, stride = g.nb * kTile, k = g.I * kTile + g.l;
    constexpr int U = sizeof(T) == 8 ? 8 : 16;   // offsets in flight per lane, two loads each
    const T* base = M + (long long)g.I * g.nb * kTileElems + g.l;
    double w[1] = {0.0};
    for (int p = cl.rank; p < cl.parts; p += cl.members) {
        L.part[t] = 0.0;
        __syncthreads();
        const double vk = L.vs[k];
        double row = 0.0;
        for (int ph = 0; ph <= g.nb / 2; ++ph) {
            if (g.active) {
                const SymRange s = sym_range(g, ph, p, cl.parts);
                double col = 0.0;
                auto chunk = [&](int r, auto whole) {
                    constexpr bool W = decltype(whole)::value;
                    T m[U], mm[U];
#pragma unroll
                    for (int u = 0; u < U; ++u) {   // clamped: no branch between the loads, nor around their uses
                        const unsigned q = 2 * (s.q0 + (W ? r + u : min(r + u, s.r1 - 1))) * kTile;
                        m[u] = base[q];
                        mm[u] = base[q + kTile];
                    }
#pragma unroll
                    for (int u = 0; u < U; ++u) {
                        const double vj = L.vs[s.J * kTile + ((g.l + r + u) & (kTile - 1))];
                        row += (double)m[u] * (W || r + u < s.r1 ? vj : 0.0);
                        col += (double)mm[u] * (W || r + u < s.r1 ? vk : 0.0);
                        col = dpp_rol1(col);
                    }
                };
                int r = s.r0;
                for (; r + U <= s.r1; r += U) chunk(r, std::true_type{});
                if (r < s.r1) {
                    chunk(r, std::false_type{});
                    r += U;
                }
                // the register has moved down once per offset taken
                if (r > s.r0) L.part[g.sub * stride + s.J * kTile + ((g.l + r) & (kTile - 1))] += col;
            }
            __syncthreads();
        }
        if (g.active) L.part[g.sub * stride + k] += row;
        __syncthreads();
        if (t < n) {
            w[0] = sym_total(L.part, n);
            if (cl.parts > 1) cl.put(n, p, w[0]);
        }
        __syncthreads();
    }
    if (cl.parts > 1) cl.exchange<1>(n, w);
    if (t < n) w[0] += (double)(T)L.diag[t] * L.vs[t];
    __syncthreads();
    return w[0];
}

}  // namespace sfh
