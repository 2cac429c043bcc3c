// nbx_knn.hip -- exact FP64 k-nearest-neighbour search and SPH densities.
//
// Replaces KDTree::FindNearest* (KDFindNearest.cxx:247-361, :444-564),
// SplitNode/LeafNode::FindNearestPos/Phase (KDSplitNode.cxx:15-95,
// KDLeafNode.cxx:15-57, :119-154), the periodic image passes
// (KDSplitNode.cxx:1119-1179), CalcDensity / CalcDensityParticle /
// CalcVelDensity (KDCalcSmoothQuantities.cxx:203-389, :768-844).
//
// Mapping to CDNA4: one wavefront owns 64 slot-consecutive queries (two
// sibling leaves).  The wave walks the implicit tree once for all 64 lanes
// (a node is opened when any lane's bound reaches it), so node boxes and
// leaf particles arrive through the scalar cache as 64-byte s_load bursts
// and are shared by the whole wave.  A leaf is consumed in two phases: (1)
// all lanes test every candidate against their current k-th distance,
// building a 32-bit accept mask; (2) lanes insert their accepted candidates
// one at a time from an LDS copy of the leaf, so the wave pays for as many
// insertions as its busiest lane, not the sum over lanes.
//
// Kept entries.  Each lane keeps its kh smallest d2 in LDS, laid out
// [position][lane] (conflict-free), in G groups of S positions, with every
// group's largest value and its position in registers.  An insertion stores
// over the largest kept value, reloads that one group and takes its maximum:
// one store, S independent loads and about 60 VALU, with a single LDS round
// trip.  The particles' slots go to a per-workgroup scratch block in device
// memory (a store nothing waits for), so LDS holds 8 bytes per entry and 9
// waves fit on a CU at k = 32.  The 4-ary heap of (d2, ID) pairs in LDS that
// this replaced held 12 bytes per entry (6 waves per CU) and took three
// dependent levels and about 135 VALU per insertion.  Measured, heap to
// groups: 0.5M clustered particles k = 8 1.68 -> 0.88 ms; with room for 18
// entries instead of 33, 16 waves on a CU, 2.1M 2.54 -> 1.79, 8.4M 9.9 -> 6.7
// ms.  More entries, lists, positions and 6-D trees are searched with a wave
// per query.
// The scratch is sized by the resident workgroups: the kernel is persistent
// and takes waves of queries from its XCD's share through an atomic counter,
// as the precision form does (nbx_mixed.hip).
//
// Exactness: distances are summed in the reference's order with no FMA
// (this file is built with -ffp-contract=off); pruning uses box_lb, which is
// never larger than a computed particle distance.  The neighbour set is the k
// smallest (d2, ID) pairs: ties at the k-th distance go to the smaller ID
// (the reference's choice there depends on its traversal order).  The search
// itself evicts any of several equal d2; a lane remembers the smallest value
// it discarded, and when that equals its final k-th distance a second walk
// collects the particles at exactly that distance and keeps the smallest IDs.
#include <atomic>

#include "nbx_kernels.h"

// v_max_f64 without the NaN canonicalisation fmax() adds: kept values are
// never NaN (a NaN d2 fails every test that leads here).
__device__ __forceinline__ double kmax(double a, double b) {
    double r;
    asm("v_max_f64 %0, %1, %2" : "=v"(r) : "v"(a), "v"(b));
    return r;
}

template <int KMAX>
struct KShape {
    static constexpr int G = 3;
    static constexpr int S = KMAX / G;
    static_assert(G * S == KMAX, "groups must tile KMAX");
};

#define HD(p) hd[(p) * NBX_WAVE + lane]  // kept d2 (LDS); unused positions hold -1
#define SL(p) sl[(p) * NBX_WAVE + lane]  // their slots (scratch)

// Per-lane search state.  kth: the largest kept d2 (NBX_MAXVALUE while fewer
// than kh are kept); gm, gp: each group's largest value and its position;
// lost: the smallest d2 discarded so far that was equal to kth when discarded.
template <int ND, int KMAX>
struct KnnCtx {
    double q[ND];
    double kth, lost;
    double gm[KShape<KMAX>::G];
    int gp[KShape<KMAX>::G];
    bool act, exz;
};

// Largest of the S values of group g and its (first) position.
template <int KMAX>
__device__ __forceinline__ void group_max(const double *hd, int lane, int base, double &m, int &at) {
    constexpr int S = KShape<KMAX>::S;
    double x[S];
#pragma unroll
    for (int u = 0; u < S; ++u) x[u] = HD(base + u);
    m = x[0];
#pragma unroll
    for (int u = 1; u < S; ++u) m = kmax(m, x[u]);
    uint32_t eq = 0;
#pragma unroll
    for (int u = S - 1; u >= 0; --u) eq = eq + eq + (x[u] == m ? 1u : 0u);
    at = base + __builtin_ctz(eq);
}

template <int ND, int KMAX>
__device__ __forceinline__ void knn_top(KnnCtx<ND, KMAX> &c) {
    c.kth = c.gm[0];
#pragma unroll
    for (int g = 1; g < KShape<KMAX>::G; ++g) c.kth = kmax(c.kth, c.gm[g]);
}

// Store (d2, slot) over the largest kept value in the lanes with ins set;
// the others store that value back, so only the slot's store branches.
template <int ND, int KMAX>
__device__ __forceinline__ void knn_replace(KnnCtx<ND, KMAX> &c, double *hd, int32_t *sl, int lane, bool ins,
                                            double d2, int32_t slot) {
    constexpr int G = KShape<KMAX>::G, S = KShape<KMAX>::S;
    int g0 = 0, p = c.gp[0];
#pragma unroll
    for (int g = 1; g < G; ++g) {
        const bool here = c.gm[g] == c.kth;
        g0 = here ? g : g0;
        p = here ? c.gp[g] : p;
    }
    HD(p) = ins ? d2 : c.kth;
    if (ins) SL(p) = slot;
    double m;
    int at;
    group_max<KMAX>(hd, lane, g0 * S, m, at);
#pragma unroll
    for (int g = 0; g < G; ++g) {
        c.gm[g] = g0 == g ? m : c.gm[g];
        c.gp[g] = g0 == g ? at : c.gp[g];
    }
    knn_top<ND, KMAX>(c);
}

template <int ND>
__device__ __forceinline__ double knn_d2(const double *q, const double *cx, int j) {
    double d2 = 0.0;
#pragma unroll
    for (int d = 0; d < ND; ++d) {
        const double t = q[d] - cx[d * NBX_LEAF + j];
        d2 += t * t;
    }
    return d2;
}

// Insert one accepted candidate (j of the LDS copy) per lane.  TIE 0: the
// search.  TIE 1: the candidate lies at exactly the k-th distance; entries at
// that distance hold -(2 + ID) (see knn_ties), the largest ID is the lowest
// value, and it gives way to a smaller ID.
template <int ND, int KMAX, int TIE>
__device__ __forceinline__ void knn_insert(const DevTree &T, KnnCtx<ND, KMAX> &c, double *hd, int32_t *sl,
                                           const double *cx, int lane, int kh, int base, int j, bool has) {
    if constexpr (TIE == 0) {
        const double d2 = knn_d2<ND>(c.q, cx, j);
        const bool in = has && d2 <= c.kth && (!c.exz || d2 > 0.0);
        c.lost = in ? c.kth : c.lost;  // the evicted value, or d2 itself when equal
        knn_replace<ND, KMAX>(c, hd, sl, lane, in && d2 < c.kth, d2, base + j);
    } else {
        const double mine = has ? -2.0 - (double)T.perm[base + j] : -1.0;
        double lo = 0.0;
        int at = 0;
        for (int p = 0; p < kh; ++p) {
            const double v = HD(p);
            at = v < lo ? p : at;
            lo = v < lo ? v : lo;
        }
        if (has && mine > lo) {
            HD(at) = mine;
            SL(at) = base + j;
        }
    }
}

// Consume one leaf for every active lane (two-phase insertion, see header).
template <int ND, int KMAX, int TIE>
__device__ __forceinline__ void knn_leaf(const DevTree &T, const double *const (&X)[ND], int leaf,
                                         KnnCtx<ND, KMAX> &c, double *hd, int32_t *sl, double *cx, int lane, int kh) {
    const int base = leaf * NBX_LEAF;
    double st[ND];
#pragma unroll
    for (int d = 0; d < ND; ++d) st[d] = X[d][base + (lane & (NBX_LEAF - 1))];
    uint32_t mask = 0;
    // candidates arrive in chunks through the scalar cache: 8 per dimension
    // (24 SGPR pairs)
    constexpr int CH = 8;
    typedef double dxc __attribute__((ext_vector_type(CH)));
    typedef const __attribute__((address_space(4))) dxc *cdcptr;
#pragma unroll
    for (int jj = 0; jj < NBX_LEAF; jj += CH) {
        dxc cv[ND];
#pragma unroll
        for (int d = 0; d < ND; ++d) cv[d] = *(cdcptr)(X[d] + base + jj);
#pragma unroll
        for (int u = 0; u < CH; ++u) {
            double d2 = 0.0;
#pragma unroll
            for (int d = 0; d < ND; ++d) {
                const double t = c.q[d] - cv[d][u];
                d2 += t * t;
            }
            mask = mask + mask + ((TIE ? d2 == c.kth : d2 <= c.kth) ? 1u : 0u);
        }
    }
    mask = __builtin_bitreverse32(mask);  // candidate j was shifted in at bit 31 - j
    if (!c.act) mask = 0;
    if (!ballot(mask != 0)) return;
    if (lane < NBX_LEAF) {
#pragma unroll
        for (int d = 0; d < ND; ++d) cx[d * NBX_LEAF + lane] = st[d];
    }
    __syncthreads();
    // as many steps as the lane with the most candidates needs (a counted
    // loop keeps the search state in place across steps)
    int nit = __popc(mask);
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) nit = max(nit, __shfl_xor(nit, off));
    nit = __builtin_amdgcn_readfirstlane(nit);
    for (int it = 0; it < nit; ++it) {
        const bool has = mask != 0;
        const int j = __builtin_ctz(mask | 0x80000000u);
        mask &= mask - 1;
        knn_insert<ND, KMAX, TIE>(T, c, hd, sl, cx, lane, kh, base, j, has);
    }
    __syncthreads();
}

// Uniform stackless depth-first walk of the heap-ordered tree.  It starts at
// the wave's own leaf node (anc; -1 when the queries are not tree particles or
// are image-shifted: then at the root), so every lane is filled from the
// query's own neighbourhood before anything else is opened; elsewhere
// children are taken nearest first from qc.  A node is
// opened when any active lane has box_lb <= its current k-th distance.
// State is uniform (SGPRs): node, depth and one "right child first" bit per
// depth; the tree's fields it reads are scalar values of their own (a field
// read from the wide argument block in the loop would bring back the block).
template <int ND, int KMAX, int TIE>
__device__ __forceinline__ void knn_walk(const DevTree &T, KnnCtx<ND, KMAX> &c, const float *qc, int anc, double *hd,
                                         int32_t *sl, double *cx, int lane, int kh) {
    int D = T.depth, nleafp = T.nleafp;
    const double *boxp = T.box;
    const float *planep = T.plane;
    asm volatile("" : "+s"(D), "+s"(nleafp), "+s"(boxp), "+s"(planep));
    const double *X[ND];
#pragma unroll
    for (int d = 0; d < ND; ++d) {
        X[d] = T.x[d];
        asm volatile("" : "+s"(X[d]));
    }
    int node = 1, dep = 0;
    uint64_t firstright = 0;
    if (anc >= 0) {
        // nothing is kept yet, so every node down to the wave's own leaf is
        // open: start there, the path's bits saying which child went first
        node = anc;
        dep = D;
        firstright = (uint64_t)(__builtin_bitreverse32((uint32_t)anc) >> (31 - D)) & ~1ULL;
    }
    for (;;) {
        cdptr bx = (cdptr)(boxp + (size_t)node * 2 * ND);
        const bool want = c.act && box_lb<ND>(c.q, bx) <= c.kth;
        if (ballot(want)) {
            if (dep == D) {
                knn_leaf<ND, KMAX, TIE>(T, X, node - nleafp, c, hd, sl, cx, lane, kh);
            } else {
                const int first = 2 * node + (first_is_right<ND>(planep, node, qc) ? 1 : 0);
                dep += 1;
                firstright = (firstright & ~(1ULL << dep)) | ((uint64_t)(first & 1) << dep);
                node = first;
                continue;
            }
        }
        // climb to the next unvisited sibling (it always exists in the padded tree)
        while (node != 1 && (uint64_t)(node & 1) != ((firstright >> dep) & 1ULL)) {
            node >>= 1;
            dep -= 1;
        }
        if (node == 1) break;
        node ^= 1;
    }
}

// The kept entries in ascending order of (value, ID, position): slots (or
// IDs; -1 for a missing one) to so, values to sd.  si: room for the IDs.
template <int KMAX>
__device__ __forceinline__ void knn_sort(const DevTree &T, const double *hd, const int32_t *sl, int32_t *so,
                                         double *sd, int32_t *si, int lane, int kh, bool ids) {
    auto put = [&](int p, double v, int r) {
        int32_t e = -1;
        if (v < NBX_MAXVALUE) {
            e = SL(p);
            if (ids) e = T.perm[e];
        }
        so[r * NBX_WAVE + lane] = e;
        sd[r * NBX_WAVE + lane] = v;
    };
    double x[KMAX];
#pragma unroll
    for (int p = 0; p < KMAX; ++p) x[p] = HD(p);
    int sum = 0;
    for (int p = 0; p < kh; ++p) {
        const double v = HD(p);
        // how many are smaller (positions past kh hold -1 and are not counted)
        int r = kh - KMAX;
#pragma unroll
        for (int u = 0; u < KMAX; ++u) r += x[u] < v ? 1 : 0;
        sum += r;
        put(p, v, r);
    }
    // equal values share a rank, which lowers the sum of the ranks; those
    // lanes rank again with the IDs (on a lattice every lane)
    if (sum != kh * (kh - 1) / 2) {
        for (int p = 0; p < kh; ++p) si[p * NBX_WAVE + lane] = HD(p) < NBX_MAXVALUE ? T.perm[SL(p)] : 0;
        for (int i = 0; i < kh; ++i) {
            const double v = HD(i);
            const int32_t id = si[i * NBX_WAVE + lane];
            int r = 0;
#pragma unroll 8
            for (int p = 0; p < kh; ++p) {
                const double w = HD(p);
                const int32_t ip = si[p * NBX_WAVE + lane];
                r += w < v || (w == v && (ip < id || (ip == id && p < i))) ? 1 : 0;
            }
            put(i, v, r);
        }
    }
}

// scratch of one workgroup, in 4-byte words: slots by position, the output
// rows in ascending order (entries and their d2), IDs by position
#define KNN_BLKW(KM) ((KM) * NBX_WAVE * 5)
#define KNN_CTR_STRIDE 16  // XCD counters 64 bytes apart

// One wave of 64 queries, wave index g.
template <int ND, int KMAX, int QSRC>
__device__ __forceinline__ void knn_task(const DevTree &T, const KnnArgs &A, double *hd, double *cx, int32_t *sl,
                                         int g, int lane) {
    int32_t *const so = sl + KMAX * NBX_WAVE;                  // sorted entries
    double *const sd = (double *)(so + KMAX * NBX_WAVE);       // their d2
    int32_t *const si = (int32_t *)(sd + KMAX * NBX_WAVE);     // IDs by position
    const int kh = A.kh;
    const int wend = A.wbeg + A.wcnt;
    const int nq = A.wcnt > 0 && wend < (T.n + NBX_WAVE - 1) / NBX_WAVE ? wend * NBX_WAVE : T.n;
    const int qi = g * NBX_WAVE + lane;
    const bool valid = qi < nq;
    double q0[ND];
#pragma unroll
    for (int d = 0; d < ND; ++d) q0[d] = valid ? T.x[d][qi] : 0.0;
    KnnCtx<ND, KMAX> c;
#pragma unroll
    for (int gr = 0; gr < KShape<KMAX>::G; ++gr) {
        constexpr int S = KShape<KMAX>::S;
        for (int u = 0; u < S; ++u) HD(gr * S + u) = gr * S + u < kh ? NBX_MAXVALUE : -1.0;
        c.gm[gr] = gr * S < kh ? NBX_MAXVALUE : -1.0;
        c.gp[gr] = gr * S;
    }
    c.exz = (QSRC == NBX_Q_SLOTS) && A.excl_zero;
    c.kth = NBX_MAXVALUE;
    c.lost = INFINITY;
    const int npass = (QSRC != NBX_Q_SLOTS && A.periodic) ? 8 : 1;
    uint32_t passes = 0;  // image passes the lane took part in
    auto pass_begin = [&](int pass, bool again, float(&qc)[ND]) -> bool {
#pragma unroll
        for (int d = 0; d < ND; ++d) c.q[d] = q0[d];
        c.act = valid;
        if (pass > 0) {
            double xp[3];
            const bool take = image_pass(pass, q0, A.period, c.kth, ND == 6, xp);
            c.act = valid && take;
            c.q[0] = xp[0]; c.q[1] = xp[1]; c.q[2] = xp[2];
        }
        if (again) c.act = (passes >> pass) & 1u;
        else passes |= c.act ? 1u << pass : 0u;
#pragma unroll
        for (int d = 0; d < ND; ++d) qc[d] = (float)readfirst_d(c.q[d]);
        return ballot(c.act) != 0;
    };
    const int own_leaves = T.nleafp + 2 * g;
    for (int pass = 0; pass < npass; ++pass) {
        float qc[ND];
        if (!pass_begin(pass, false, qc)) continue;
        knn_walk<ND, KMAX, 0>(T, c, qc, pass == 0 ? own_leaves : -1, hd, sl, cx, lane, kh);
    }
    const double kth = c.kth;

    // Ties at the k-th distance: something equal to it was discarded, so the
    // entries at that distance may not be the smallest IDs.  Those entries
    // are emptied (to the value of an ID past all others), every particle at
    // exactly that distance is met again, and the smallest IDs stay.
    const bool tied = valid && c.lost == kth && kth < NBX_MAXVALUE;
    if (ballot(tied)) {
        const uint32_t taken = passes;
        if (tied) {
            for (int p = 0; p < kh; ++p)
                if (HD(p) == kth) HD(p) = -2.0 - 2147483648.0;
        }
        passes = tied ? taken : 0u;
        for (int pass = 0; pass < npass; ++pass) {
            float qc[ND];
            if (!pass_begin(pass, true, qc)) continue;
            knn_walk<ND, KMAX, 1>(T, c, qc, pass == 0 ? own_leaves : -1, hd, sl, cx, lane, kh);
        }
        if (tied) {
            for (int p = 0; p < kh; ++p)
                if (HD(p) < -1.5) HD(p) = kth;
        }
    }
    __syncthreads();

    // ------------------------------------------------------------ densities
    // Symmetric scatter: contributions to the wave's own 64 queries are summed in LDS (over the leaf copy) and flushed with one
    // atomic per query.
    double *const racc = cx;
    const bool spline = ND == 3 && QSRC == NBX_Q_SLOTS && A.dens == NBX_DO_SPLINE;
    const bool sym = QSRC == NBX_Q_SLOTS && (A.dens == NBX_DO_SYM || spline);
    double racc_own = 0.0;
    if (sym) racc[lane] = 0.0;
    __syncthreads();
    // image-shifted queries take the gather forms only
    if (A.dens != NBX_DO_NONE && valid && (QSRC == NBX_Q_SLOTS || A.dens == NBX_DO_GATHER)) {
        const bool bad = !(kth < NBX_MAXVALUE);  // fewer than kh neighbours
        if (A.dens == NBX_DO_VEL || A.dens == NBX_DO_VELPHYS) {
            // CalcVelDensity: |dv| of the Nsearch physical neighbours, the
            // Nsmooth smallest of them, h_v = max/2, sum W(|dv|/h_v) h_v^-3.
            // |dv| takes the place of d2; the terms are summed in the order
            // of (|dv|, ID).
            const int ns = A.nsmooth;
            const double qvx = T.x[3][qi], qvy = T.x[4][qi], qvz = T.x[5][qi];
            if (!bad) {
                for (int p = 0; p < kh; ++p) {
                    const int32_t s = SL(p);
                    double vx = qvx - T.x[3][s], vy = qvy - T.x[4][s], vz = qvz - T.x[5][s];
                    HD(p) = sqrt(vx * vx + vy * vy + vz * vz);
                }
                knn_sort<KMAX>(T, hd, sl, so, sd, si, lane, kh, false);
                const double hv = 0.5 * sd[(ns - 1) * NBX_WAVE + lane];
                const double norm = 1.0 / pow(hv, 3.0);
                // CalcVelDensityWithPhysDensity (KDCalcSmoothQuantities.cxx:428-466):
                // each term times W(r_ij / h) h^-3 / rho_i * m_i, with
                // h = d2 of the Nsearch-th neighbour / 2 (no square root)
                const bool phys = A.dens == NBX_DO_VELPHYS;
                const double hp = 0.5 * kth;
                const double pnorm = phys ? 1.0 / pow(hp, 3.0) : 0.0;
                const double rhoi = phys ? A.rho_in[qi] : 1.0, mi = phys ? T.mass[qi] : 0.0;
                double den = 0.0;
                for (int p = 0; p < ns; ++p) {
                    const double v = sd[p * NBX_WAVE + lane];
                    const double vW = wsm_at(v, hv, T.kern, T.kernres) * norm;
                    if (!phys) {
                        den = den + vW;
                    } else {
                        const int32_t s = so[p * NBX_WAVE + lane];
                        double dx = T.x[0][qi] - T.x[0][s], dy = T.x[1][qi] - T.x[1][s], dz = T.x[2][qi] - T.x[2][s];
                        double r = sqrt(dx * dx + dy * dy + dz * dz);
                        double W = wsm_at(r, hp, T.kern, T.kernres) * pnorm;
                        den = den + vW * (W / rhoi * mi);
                    }
                }
                A.rho[qi] = den;
                if (A.hout) A.hout[A.hout_by_id ? T.perm[qi] : qi] = hv;
            }
        } else {
            const double hi = 0.5 * sqrt(kth);
            const double ih = 1.0 / hi;
            const double norm = spline ? NBX_SIGMA3 * ih * ih * ih : 1.0 / pow(hi, (double)ND);
            const double mi = QSRC == NBX_Q_SLOTS ? T.mass[qi] : 0.0;
            double acc = 0.0;
            // entries in groups of 8 so their slot/mass gathers are in flight
            // together; summed in position order
            for (int p0 = 0; p0 < kh; p0 += 8) {
                int32_t sv[8];
                double dv[8], mv[8];
#pragma unroll
                for (int u = 0; u < 8; ++u) {
                    const bool in = p0 + u < kh;
                    dv[u] = in ? HD(p0 + u) : NBX_MAXVALUE;
                    sv[u] = dv[u] < NBX_MAXVALUE ? SL(p0 + u) : 0;
                }
#pragma unroll
                for (int u = 0; u < 8; ++u) mv[u] = T.mass[sv[u]];
#pragma unroll
                for (int u = 0; u < 8; ++u) {
                    if (!(dv[u] < NBX_MAXVALUE)) continue;  // past the end, or missing
                    const int32_t s = sv[u];
                    const double r = sqrt(dv[u]);
                    const double W = spline ? w_cubic(r * ih) : wsm_at(r, hi, T.kern, T.kernres);
                    if (sym) {
                        const double Wij = 0.5 * W * norm;
                        acc = acc + Wij * mv[u];
                        const uint32_t r = (uint32_t)(s - g * NBX_WAVE);
                        if (r < NBX_WAVE) atomicAdd(&racc[r], Wij * mi);
                        else unsafeAtomicAdd(A.rho + s, Wij * mi);
                    } else {
                        acc += W * norm * mv[u];
                    }
                }
            }
            if (sym) racc_own = acc;
            else A.rho[qi] = acc;
            if (A.hout) A.hout[A.hout_by_id ? T.perm[qi] : qi] = hi;
        }
        if (bad) atomicOr(A.err, 1);
    }
    __syncthreads();
    if (sym && valid) unsafeAtomicAdd(A.rho + qi, racc_own + racc[lane]);

    // ------------------------------------------------------------ outputs
    // (rows of the search only: the velocity densities ask for none)
    if (A.nn == nullptr && A.d2 == nullptr) return;
    const bool ids = A.layout == 0;
    if (A.miss_self && valid && !(kth < NBX_MAXVALUE)) {
        atomicOr(A.err, 1);
        for (int p = 0; p < kh; ++p)
            if (!(HD(p) < NBX_MAXVALUE)) {
                HD(p) = 0.5 * NBX_MAXVALUE;
                SL(p) = qi;
            }
    }
    if (valid) knn_sort<KMAX>(T, hd, sl, so, sd, si, lane, kh, ids);
    __syncthreads();
    const int kout = A.kout;
    const int off = (A.drop == NBX_DROP_SMALLEST) ? 1 : 0;
    const int total = NBX_WAVE * kout;
    for (int e = lane; e < total; e += NBX_WAVE) {
        int r = e / kout, t = e - r * kout;
        int qr = g * NBX_WAVE + r;
        if (qr >= nq) break;
        const int64_t row = A.layout == 1 ? qr - A.row0 : T.perm[qr];
        if (A.nn) A.nn[row * kout + t] = so[(t + off) * NBX_WAVE + r];
        if (A.d2) A.d2[row * kout + t] = sd[(t + off) * NBX_WAVE + r];
    }
    __syncthreads();  // the scratch is written again by the next wave of queries
}

// Persistent kernel, one wave per workgroup: workgroup b stays on XCD
// (b mod 8), takes waves of queries from that XCD's contiguous share through
// its counter, then from the other shares in turn, and owns one scratch
// block.  Every ticket names one wave; a workgroup exits when all eight
// counters have passed their shares' ends.
template <int ND, int KMAX, int QSRC>
__global__ __launch_bounds__(64) void k_knn(DevTree T, KnnArgs A, int nw, int32_t *scratch, int32_t *ctr) {
    __shared__ double hd[KMAX * NBX_WAVE];
    __shared__ double cx[ND * NBX_LEAF];  // leaf copy; then the symmetric scatter
    static_assert(ND * NBX_LEAF >= NBX_WAVE, "the scatter lies over the leaf copy");
    const int lane = threadIdx.x;
    int32_t *sl = scratch + (size_t)blockIdx.x * KNN_BLKW(KMAX);
    // in a VGPR pair: a scalar base would be spilled and reloaded per store
    asm volatile("" : "+v"(sl));
    const int x = blockIdx.x & 7, q8 = nw >> 3, r8 = nw & 7;
    for (int s = 0; s < 8; ++s) {
        const int y = (x + s) & 7;
        const int ybeg = y * q8 + (y < r8 ? y : r8), ycnt = q8 + (y < r8 ? 1 : 0);
        for (;;) {
            int t = 0;
            if (lane == 0) t = atomicAdd(ctr + y * KNN_CTR_STRIDE, 1);
            t = __builtin_amdgcn_readfirstlane(t);
            if (t >= ycnt) break;
            knn_task<ND, KMAX, QSRC>(T, A, hd, cx, sl, A.wbeg + ybeg + t, lane);
        }
    }
}

// Resident workgroups of one instance over the device, a multiple of 8.
template <int ND, int KMAX, int QSRC>
static int knn_resident() {
    static std::atomic<int> grid{0};
    int g = grid.load();
    if (g == 0) {
        int dev = 0, ncu = 0, per = 0;
        if (hipGetDevice(&dev) != hipSuccess) dev = 0;
        if (hipDeviceGetAttribute(&ncu, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess || ncu <= 0) ncu = 256;
        if (hipOccupancyMaxActiveBlocksPerMultiprocessor(&per, k_knn<ND, KMAX, QSRC>, NBX_WAVE, 0) != hipSuccess ||
            per <= 0)
            per = 1;
        g = (per * ncu) & ~7;
        g = g < 8 ? 8 : g;
        grid.store(g);
    }
    return g;
}

// Which kernel serves a search.  A lane per query shares each node and leaf
// among 64 neighbours and wins for few kept entries over many queries; a wave
// per query (nbx_knn_wave.hip) keeps its entries in registers and needs few
// queries to fill the device.  Measured in ms, lanes / waves, density: 0.3M
// clustered particles k = 1 0.24 / 0.38, k = 4 0.40 / 0.41, k = 8 0.51 / 0.42,
// k = 17 0.69 / 0.46; 0.5M k = 4 0.49 / 0.68, k = 8 0.59 / 0.72, k = 17 0.77 /
// 0.79; 1M k = 8 0.91 / 1.44, k = 17 1.24 / 1.60; with room for 33 entries in
// the lanes' kernel, 2.1M k = 20 3.6 / 3.4, k = 32 4.4 / 3.7.  So the line moves
// with the entries kept.
// Up to 7 entries it lies lower.  There a wave is slow on a lattice, where
// nearly every merge meets equal distances: 262144 particles, density, lattice
// k = 2 0.24 / 0.57, k = 4 0.26 / 0.58, k = 6 0.30 / 0.62 (k = 8 0.48 / 0.66);
// uniform k = 4 0.28 / 0.38, k = 6 0.32 / 0.40; clustered k = 4 0.35 / 0.38, k =
// 6 0.38 / 0.39, rows 0.34 / 0.28 and 0.39 / 0.29.  Of 195112: lattice k = 2
// 0.32 / 0.46, clustered 0.26 / 0.29, rows 0.23 / 0.22.
#define KNN_KM 18
bool nbx_knn_by_waves(int nd, int kh, int qsrc, bool listed, int64_t nqueries) {
    if (nd == 6 || kh > KNN_KM || qsrc == NBX_Q_POINTS || listed) return true;
    return nqueries <= (kh <= 7 ? 139264 + 16384 * kh : 163840 + 24576 * kh);
}

static const size_t KNN_CTR_BYTES = 8 * KNN_CTR_STRIDE * sizeof(int32_t);
static const size_t KNN_BLOCK_BYTES = (size_t)KNN_BLKW(KNN_KM) * sizeof(int32_t);

// workgroups for nw waves: no more than are resident (or than there are waves)
static int knn_grid(int qsrc, int64_t nw) {
    const int res = qsrc == NBX_Q_PERIODIC ? knn_resident<3, KNN_KM, NBX_Q_PERIODIC>()
                                           : knn_resident<3, KNN_KM, NBX_Q_SLOTS>();
    const int64_t want = (nw + 7) & ~(int64_t)7;
    return (int)(want < res ? want : res);
}

size_t nbx_knn_scratch_bytes(int nd, int kh, int qsrc, bool listed, int64_t nqueries) {
    if (nbx_knn_by_waves(nd, kh, qsrc, listed, nqueries)) return 0;
    return KNN_CTR_BYTES + (size_t)knn_grid(qsrc, (nqueries + NBX_WAVE - 1) / NBX_WAVE) * KNN_BLOCK_BYTES;
}

hipError_t nbx_launch_knn(const DevTree &T, const KnnArgs &A, int nqueries, hipStream_t st, void *work,
                          size_t work_bytes) {
    const int nw = (nqueries + NBX_WAVE - 1) / NBX_WAVE;
    if (nw == 0) return hipSuccess;
    if (A.kh < 1 || A.kh > 129) return hipErrorInvalidValue;
    const bool listed = A.qsrc != NBX_Q_POINTS && A.qlist;
    if (nbx_knn_by_waves(T.nd, A.kh, A.qsrc, listed, nqueries)) return nbx_launch_knn_wave(T, A, nqueries, st);
    int grid = knn_grid(A.qsrc, nw);
    void *mem = work;
    if (mem) {
        // as many workgroups as the scratch given has blocks for
        if (work_bytes < KNN_CTR_BYTES + 8 * KNN_BLOCK_BYTES) return hipErrorInvalidValue;
        const size_t fit = (work_bytes - KNN_CTR_BYTES) / KNN_BLOCK_BYTES;
        if (fit < (size_t)grid) grid = (int)fit & ~7;
    } else {
        const hipError_t e = hipMallocAsync(&mem, KNN_CTR_BYTES + (size_t)grid * KNN_BLOCK_BYTES, st);
        if (e != hipSuccess) return e;
    }
    int32_t *ctr = (int32_t *)mem, *scr = (int32_t *)((char *)mem + KNN_CTR_BYTES);
    hipLaunchKernelGGL(k_fill_i32, dim3(1), dim3(256), 0, st, ctr, 0, (int64_t)(8 * KNN_CTR_STRIDE));
    {
        ProfScope ps("k_knn_fp64", st);
        if (A.qsrc == NBX_Q_PERIODIC)
            hipLaunchKernelGGL((k_knn<3, KNN_KM, NBX_Q_PERIODIC>), dim3(grid), dim3(NBX_WAVE), 0, st, T, A, nw, scr, ctr);
        else
            hipLaunchKernelGGL((k_knn<3, KNN_KM, NBX_Q_SLOTS>), dim3(grid), dim3(NBX_WAVE), 0, st, T, A, nw, scr, ctr);
    }
    const hipError_t e = hipGetLastError();
    if (!work) hipFreeAsync(mem, st);
    return e;
}
