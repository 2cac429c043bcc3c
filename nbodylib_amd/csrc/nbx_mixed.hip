// nbx_mixed.hip -- precision form of kNN + SPH density (FP32 search, FP64
// re-check band, exact neighbour sets).
//
// Same call as CalcDensity (KDCalcSmoothQuantities.cxx:203-305) and the
// target-based FindNearest / FindNearestPhase (KDFindNearest.cxx:247-318,
// :347-361) on a non-periodic search, in 3-D or on the 6-D phase-space
// tree, with the same wave/leaf structure as the FP64 kernel (nbx_knn.hip).
//
// Search: particle coordinates are stored as FP32 offsets from their leaf's
// FP64 centre; a query is re-expressed per leaf as fl32(q - centre) so every
// difference is formed between two small FP32 numbers.  Each lane keeps the
// k+1 smallest FP32 d2: their bits in LDS (4 bytes per entry, so LDS does
// not limit how many waves a CU holds) and their particle slots in a
// per-workgroup scratch array in device memory.  The kernel is persistent:
// each workgroup takes waves of queries from its XCD's share of the tree
// order through an atomic counter, so the scratch is sized by the resident
// workgroups, not by n.
//
// Error bound: with u = 2^-24 and E the half-diagonal of the leaf a
// candidate came from, |dist32 - dist64| <= 12 u dist32 + 5 u E.  Per
// component the two offset roundings and the difference add at most
// u(|q - o| + |x - o| + |t|) <= u(dist + 2E + dist); the FMA chain over ND
// <= 6 squares adds ND u relative to the sum, sqrt halves it and adds u:
// at most (2 + ND/2 + 1) u dist + 2 u E = 6 u dist + 2 u E in 6-D, so the
// constants keep a factor 2 of margin.  A kept key adds its tag error (2^TB
// u dist, see the kept keys below) to the 12 u dist term.  Each lane tracks E_max over the leaves it evaluated
// as reachable or accepted a candidate from (candidates of other leaves are
// outside by the FP64 node bound).
//
// Re-check band: after the walk the k+1 keys are sorted; the candidates
// whose distance interval overlaps the k-th one's (plus any that could be a
// d2 == 0 duplicate) are recomputed in FP64 and the k-th neighbour is chosen
// among them by (d2, ID) as in the FP64 form.  Certificate: the largest
// selected FP64 d2 must be strictly below the squared lower bound of every
// particle outside the heap (bounded through the (k+1)-th key).  Lanes that
// fail it (the bound is loose when a lane has evaluated a very large leaf)
// are verified exactly: the k smallest (d2, ID) of the k+1 candidates are
// taken in FP64 and an FP64 walk of that ball counts the particles below the
// k-th; exactly k-1 proves the set.  Only lanes that fail this too are
// appended to a fallback list and recomputed by the FP64 kernel, so
// neighbour sets are always exact.
// h = |x - x_k| / 2 comes from the FP64 k-th distance, and the kernel
// weights of the k selected neighbours use FP64 distances (an FP32 offset
// carries a storage error proportional to its leaf's size, which in
// clustered data can reach 1e-5 of the neighbour distance); the search --
// every candidate test and heap operation -- stays in FP32.
#include <algorithm>
#include <atomic>

#include "nbx_kernels.h"

typedef float fx8 __attribute__((ext_vector_type(8)));
typedef const __attribute__((address_space(4))) fx8 *cf8ptr;

#define MX_PLOG 5  // a wave's queries go to at most 32 waves
#define MX_U 5.9604644775390625e-8  // 2^-24
#define MX_DB 4               // neighbours gathered together in the density pass
#define MX_EMPTY 0x7F7FFFFFu  // empty kept entry: the bits of FLT_MAX

#define HK(p) hk[(p) * NBX_WAVE + lane]   // kept keys (LDS)
typedef __attribute__((address_space(1))) uint16_t gu16;
typedef __attribute__((address_space(1))) uint32_t gu32;
#define SLH(p) ((gu16 *)sl + lane)[(p) * NBX_WAVE]  // their handles (scratch, by position)
#define MX_V 2048  // leaves a wave can record: handle = leaf's visit number << 5 | index in leaf

// Kept keys.  The kh = k+1 kept candidates of a lane sit at positions
// p < kh of KMAX = G * S (G groups of S positions; positions p >= kh hold
// 0, which never outranks a key).  A kept key is the FP32 d2's bits with the
// low TB bits replaced by a tag: its position p when KMAX <= 33 (keys are
// then unique), else its position within its group (the group holding the
// largest key is found among the group maxima).  Keys compare as unsigned
// integers in d2 order up to the TB replaced bits, and the largest key names
// its own position.  A key overstates or understates d2 by less than 2^TB
// ulps -- a relative 2^TB * 2^-23 in d2, 2^TB * u in the distance -- which
// the error bound below carries.  Each group's largest key stays in a
// register; replacing the largest kept key is one LDS store, one scratch
// store and one S-wide LDS reload of its group.
template <int KMAX>
struct GShape {
    static constexpr int G = KMAX <= 33 ? 3 : 5;
    static constexpr int S = KMAX / G;
    static constexpr bool GT = KMAX <= 33;    // tag = position p (else position in group)
    static constexpr int TB = GT ? 6 : 4;      // tag bits
    static constexpr uint32_t TM = (1u << TB) - 1u;
    static_assert(G * S == KMAX && (GT ? KMAX : S) <= (1 << TB), "group shape must tile KMAX");
};

__device__ __forceinline__ uint32_t umax3(uint32_t a, uint32_t b, uint32_t c) { return max(max(a, b), c); }

// Batcher's odd-even merge sorting network over 64 inputs, keeping only the
// comparators whose inputs are both below lim (the inputs from lim on are
// +inf, which those comparators would leave in place).  Built at compile
// time; a fully unrolled pass over it sorts keys held in registers.
struct SortNet {
    int n;
    uint8_t a[256], b[256];
};
constexpr void sn_add(SortNet &s, int i, int j, int lim) {
    if (j < lim) {
        s.a[s.n] = (uint8_t)i;
        s.b[s.n] = (uint8_t)j;
        s.n += 1;
    }
}
constexpr void sn_merge(SortNet &s, int lo, int hi, int r, int lim) {
    const int step = 2 * r;
    if (step < hi - lo) {
        sn_merge(s, lo, hi, step, lim);
        sn_merge(s, lo + r, hi, step, lim);
        for (int i = lo + r; i < hi - r; i += step) sn_add(s, i, i + r, lim);
    } else {
        sn_add(s, lo, lo + r, lim);
    }
}
constexpr void sn_sort(SortNet &s, int lo, int hi, int lim) {
    if (hi - lo >= 1) {
        const int mid = lo + (hi - lo) / 2;
        sn_sort(s, lo, mid, lim);
        sn_sort(s, mid + 1, hi, lim);
        sn_merge(s, lo, hi, 1, lim);
    }
}
constexpr SortNet sort_net(int lim) {
    SortNet s{};
    sn_sort(s, 0, 63, lim);
    return s;
}
constexpr SortNet MX_NET33 = sort_net(33);  // 246 comparators

// Largest of S keys (a max tree).
template <int S>
__device__ __forceinline__ uint32_t gmaxu(const uint32_t (&x)[S]) {
    uint32_t v[S];
#pragma unroll
    for (int u = 0; u < S; ++u) v[u] = x[u];
#pragma unroll
    for (int w = 1; w < S; w *= 3)
#pragma unroll
        for (int u = 0; u + w < S; u += 3 * w) v[u] = u + 2 * w < S ? umax3(v[u], v[u + w], v[u + 2 * w]) : max(v[u], v[u + w]);
    return v[0];
}

template <int KMAX>
__device__ __forceinline__ uint32_t gtop_init(uint32_t *hk, int lane, int kh, uint32_t (&gm)[GShape<KMAX>::G]) {
    constexpr int G = GShape<KMAX>::G, S = GShape<KMAX>::S;
    constexpr uint32_t TM = GShape<KMAX>::TM;
#pragma unroll
    for (int g = 0; g < G; ++g) {
        uint32_t m = 0u;
        for (int u = 0; u < S; ++u) {
            const int p = g * S + u;
            const uint32_t v = p < kh ? ((MX_EMPTY & ~TM) | (uint32_t)(GShape<KMAX>::GT ? p : u)) : 0u;
            HK(p) = v;
            m = max(m, v);
        }
        gm[g] = m;
    }
    return gmaxu<G>(gm);
}

// Replace the largest kept key (root) by key in the lanes with ins set (key
// carries the root's position); the others store the root back, so nothing
// but the handle store branches.  slot is the candidate's 16-bit handle.
// Returns the new largest key.
template <int KMAX>
__device__ __forceinline__ uint32_t gtop_replace(uint32_t *hk, uint32_t *sl, int lane,
                                                 uint32_t (&gm)[GShape<KMAX>::G], bool ins, uint32_t key,
                                                 int32_t slot, uint32_t root) {
    constexpr int G = GShape<KMAX>::G, S = GShape<KMAX>::S;
    constexpr uint32_t TM = GShape<KMAX>::TM;
    int g0 = 0, p;
    if constexpr (GShape<KMAX>::GT) {
        p = (int)(root & TM);
#pragma unroll
        for (int g = 1; g < G; ++g) g0 += p >= g * S ? 1 : 0;
    } else {
#pragma unroll
        for (int g = G - 1; g > 0; --g) g0 = gm[g] == root ? g : g0;
        p = g0 * S + (int)(root & TM);
    }
    const int b = g0 * S;
    HK(p) = ins ? key : root;
    if (ins) SLH(p) = (uint16_t)slot;
    uint32_t x[S];
#pragma unroll
    for (int u = 0; u < S; ++u) x[u] = HK(b + u);
    const uint32_t bc = gmaxu<S>(x);
#pragma unroll
    for (int g = 0; g < G; ++g) gm[g] = g0 == g ? bc : gm[g];
    return gmaxu<G>(gm);
}

template <int ND>
struct MixCtx {
    double q[ND];
    bool act;
    int32_t self;
    uint32_t root;  // largest kept key
    double emax;    // largest leaf half-diagonal that matters for this lane
    int nvis;       // leaves recorded (wave-uniform), the next handle's visit number
    int fillkh;     // kh while the heap is still empty and kh >= 32 (wave-uniform), else 0
};

// The leaf data a visit reads, each base a value of its own (see mix_walk):
// origins and half-diagonals (scalar loads), and the FP32 offsets, 3-D
// interleaved (scalar and vector loads) or 6-D per dimension (vector loads
// only, so those bases are held in vector registers).
template <int ND>
struct MixSrc {
    const double *org, *ext;
    const float4 *xq;
    const float *xf[ND == 6 ? 6 : 1];
};

// What a leaf visit reads in 6-D, loaded a leaf ahead: this lane's candidate,
// and the leaf's origin.
struct MixPre {
    float st[6];
    double o[6];
};
__device__ __forceinline__ void mix_load(const MixSrc<6> &S, int leaf, int lane, MixPre &p) {
#pragma unroll
    for (int d = 0; d < 6; ++d) p.st[d] = S.xf[d][leaf * NBX_LEAF + (lane & (NBX_LEAF - 1))];
    const double2 *op = (const double2 *)(S.org + (size_t)leaf * 6);
#pragma unroll
    for (int i = 0; i < 3; ++i) {
        const double2 v = op[i];
        p.o[2 * i] = v.x;
        p.o[2 * i + 1] = v.y;
    }
}

// A query in LDS for a transposed test: its coordinates and its threshold, 4
// floats in 3-D and 8 in 6-D (16-byte accesses), at most MX_QMAX of them
// (even, so that an odd count has room for one that passes nothing).
#define MX_FEW 24  // 3-D: wanting lanes up to which a leaf is scanned transposed (see mix_leaf)
#define MX_QW(ND) ((ND) == 6 ? 8 : 4)
#define MX_QMAX(ND) ((ND) == 6 ? NBX_WAVE : MX_FEW + 2)
template <int ND>
__device__ __forceinline__ void mix_put_query(float *qb, int at, const float *q, float th) {
    float4 *p = (float4 *)qb + (MX_QW(ND) / 4) * at;
    if constexpr (ND == 6) {
        p[0] = make_float4(q[0], q[1], q[2], q[3]);
        p[1] = make_float4(q[4], q[5], th, 0.0f);
    } else {
        p[0] = make_float4(q[0], q[1], q[2], th);
    }
}

template <int ND, int KMAX>
__device__ __forceinline__ void mix_leaf(const MixSrc<ND> &S, int leaf, MixCtx<ND> &c, bool want,
                                         uint32_t *hk, uint32_t *sl, float *cx, int lane,
                                         uint32_t (&gm)[GShape<KMAX>::G], const MixPre &pre) {
    const int base = leaf * NBX_LEAF;
    // A kept candidate is stored as a 16-bit handle, its leaf's visit number
    // << 5 | its index in the leaf; the wave's visit table (vt, right after
    // the handles in scratch) maps visit numbers to leaves.  A 3-D wave
    // numbers every leaf it visits (about 36); a 6-D wave visits hundreds,
    // so it numbers only the leaves where some lane accepts a candidate.
    uint32_t *vt = sl + KMAX * (NBX_WAVE / 2);
    int rbase = c.nvis << 5;
    if constexpr (ND == 3) {
        if (lane == 0) vt[c.nvis] = (uint32_t)leaf;
        c.nvis += 1;
    }
    // candidate (lane mod 32) of this leaf: the tested point in phase 1 and
    // this lane's part of the LDS copy used in phase 2 (6-D: loaded ahead)
    float st[ND];
    if constexpr (ND == 3) {
        const float4 v = S.xq[base + (lane & (NBX_LEAF - 1))];
        st[0] = v.x;
        st[1] = v.y;
        st[2] = v.z;
    } else {
#pragma unroll
        for (int d = 0; d < ND; ++d) st[d] = pre.st[d];
    }
    // query relative to this leaf's centre, rounded once to FP32
    const double *o = S.org + (size_t)leaf * ND;
    float qv[ND];
#pragma unroll
    for (int d = 0; d < ND; ++d) qv[d] = (float)(c.q[d] - (ND == 6 ? pre.o[d] : ((cdptr)o)[d]));
    const float th = __uint_as_float(c.root);
    uint32_t mask = 0u;
    const uint64_t wm = ballot(want);
    const int nwq = __popcll(wm);
    if (ND == 3 && nwq > MX_FEW) {
        // Phase 1: every lane tests the 32 candidates, read in 64-byte scalar
        // loads, in the expanded form
        //     w + 2 qv.p >= |p|^2,  w = th + m - |qv|^2
        // (|p|^2 stored per slot): three FMAs and a compare per candidate,
        // the accept bit shifted in with a carry.  In exact arithmetic this
        // is |qv - p|^2 <= th + m.  Phase 2 accepts only candidates whose
        // difference-form d2 (3 roundings, relative error < 6u, u = 2^-24)
        // is <= th, i.e. with |qv - p|^2 <= th (1 + 6u); the rounding of the
        // expanded form is below 11u th + 5u m + 7u (|qv| + |p|)^2, so the
        // margin m = 2^-20 (th + (|qv| + e)^2) (e >= |p|: the leaf's
        // half-diagonal) lets every such candidate through.  The few extra
        // ones fail phase 2's test, so the kept keys are those of the
        // difference form alone.
        typedef float fxc __attribute__((ext_vector_type(16)));
        typedef const __attribute__((address_space(4))) fxc *cfcptr;
        const float q2 = __builtin_fmaf(qv[2], qv[2], __builtin_fmaf(qv[1], qv[1], qv[0] * qv[0]));
        const float r = sqrtf(q2) + (float)(((cdptr)S.ext)[leaf] * (1.0 + 0x1p-20));
        const float m = 0x1p-20f * __builtin_fmaf(r, r, th);
        // FLT_MAX (no bound yet): every real candidate passes
        const float w = fminf((th + m) - q2, 3.402823466e38f);
        const float a0 = 2.0f * qv[0], a1 = 2.0f * qv[1], a2 = 2.0f * qv[2];
        // two halves of 16 candidates (x, y, z, |p|^2), 64 scalar registers
        // each (the whole leaf at once would not fit the scalar register file)
        const cfcptr lp = (cfcptr)(S.xq + base);
#pragma unroll 1
        for (int h = 0; h < 2; ++h) {
            fxc c4[4];
#pragma unroll
            for (int i = 0; i < 4; ++i) c4[i] = lp[4 * h + i];
#pragma unroll
            for (int u = 0; u < 16; ++u) {
                const int i = u >> 2, o = (u & 3) * 4;
                float v = __builtin_fmaf(a0, c4[i][o], w);
                v = __builtin_fmaf(a1, c4[i][o + 1], v);
                v = __builtin_fmaf(a2, c4[i][o + 2], v);
                mask = mask + mask + (v >= c4[i][o + 3] ? 1u : 0u);
            }
        }
        // candidate j was shifted in at bit 31 - j
        mask = __builtin_bitreverse32(mask);
    } else {
        // Phase 1, transposed: the lanes that want this leaf put their query
        // offsets and thresholds in LDS (over cx), and each step tests two of
        // them against the 32 candidates, one candidate per lane; the
        // ballot's halves are the two queries' accept masks, left in LDS for
        // their lanes.  Lanes that do not want the leaf have no candidate in
        // it: their bound already exceeds their largest kept key.  In 6-D
        // always; in 3-D, where the scan by lanes takes 200 VALU and 57% of
        // the leaves are wanted by at most 16 lanes, up to MX_FEW of them:
        // 16.8M particles, k = 32, 18.58 ms without, 17.89 up to 12, 17.83
        // up to 24, 17.91 up to 32, 18.06 up to 48.
        const int wr = __builtin_amdgcn_mbcnt_hi((uint32_t)(wm >> 32), __builtin_amdgcn_mbcnt_lo((uint32_t)wm, 0u));
        if (want) mix_put_query<ND>(cx, wr, qv, th);
        if ((nwq & 1) && lane == 0) {
            // an odd count's last step tests a second query that passes nothing
            const float none[6] = {0.0f, 0.0f, 0.0f, 0.0f, 0.0f, 0.0f};
            mix_put_query<ND>(cx, nwq, none, -1.0f);
        }
        __syncthreads();
        constexpr int Q4 = MX_QW(ND) / 4;
        const float4 *qm = (const float4 *)cx + Q4 * (lane >> 5);
        uint32_t *mb = (uint32_t *)(cx + MX_QW(ND) * MX_QMAX(ND));
        for (int it = 0; it < nwq; it += 2) {
            const float4 a = qm[Q4 * it];
            const float t0 = a.x - st[0], t1 = a.y - st[1], t2 = a.z - st[2];
            float dd = t0 * t0;
            dd = __builtin_fmaf(t1, t1, dd);
            dd = __builtin_fmaf(t2, t2, dd);
            float lim = a.w;
            if constexpr (ND == 6) {
                const float4 b = qm[Q4 * it + 1];
                const float t3 = a.w - st[3], t4 = b.x - st[4], t5 = b.y - st[5];
                dd = __builtin_fmaf(t3, t3, dd);
                dd = __builtin_fmaf(t4, t4, dd);
                dd = __builtin_fmaf(t5, t5, dd);
                lim = b.z;
            }
            const uint64_t pm = ballot(dd <= lim);
            if (lane == 0) *(uint64_t *)(mb + it) = pm;
        }
        __syncthreads();
        mask = want ? mb[wr] : 0u;
    }
    if (c.self >= base && c.self < base + NBX_LEAF) mask &= ~(1u << (c.self - base));
    if (!c.act) mask = 0;
    if (c.act && (want || mask)) c.emax = fmax(c.emax, ((cdptr)S.ext)[leaf]);
    if constexpr (ND == 6) {
        // no lane accepts anything: nothing to insert, no visit number
        if (!ballot(mask != 0)) return;
        if (lane == 0) vt[c.nvis] = (uint32_t)leaf;
        c.nvis += 1;
    }
    if (lane < NBX_LEAF) {
#pragma unroll
        for (int d = 0; d < ND; ++d) cx[d * NBX_LEAF + lane] = st[d];
    }
    __syncthreads();
    if constexpr (GShape<KMAX>::GT) {
        if (c.fillkh) {
            // First leaf of the walk, every heap still empty and at least 32
            // positions: the replacement would put the m-th accepted
            // candidate at position kh - 1 - m (the largest empty key's), so
            // the keys go straight there in one pass over the leaf, and the
            // group maxima are taken once at the end.
            const int kh = c.fillkh;
            c.fillkh = 0;
            constexpr uint32_t TM = GShape<KMAX>::TM;
            constexpr int G = GShape<KMAX>::G, S = GShape<KMAX>::S;
            int cnt = 0;
            for (int j = 0; j < NBX_LEAF; ++j) {
                float t = qv[0] - cx[j];
                float dd = t * t;
#pragma unroll
                for (int d = 1; d < ND; ++d) {
                    t = qv[d] - cx[d * NBX_LEAF + j];
                    dd = __builtin_fmaf(t, t, dd);
                }
                const int p = kh - 1 - cnt;
                const uint32_t key = (__float_as_uint(dd) & ~TM) | (uint32_t)p;
                const bool ins = ((mask >> j) & 1u) && key < ((MX_EMPTY & ~TM) | (uint32_t)p);
                if (ins) {
                    HK(p) = key;
                    SLH(p) = (uint16_t)(rbase + j);
                }
                cnt += ins ? 1 : 0;
            }
#pragma unroll
            for (int g = 0; g < G; ++g) {
                uint32_t x[S];
#pragma unroll
                for (int u = 0; u < S; ++u) x[u] = HK(g * S + u);
                gm[g] = gmaxu<S>(x);
            }
            c.root = gmaxu<G>(gm);
            __syncthreads();
            return;
        }
    }
    // as many steps as the lane with the most candidates needs (a counted
    // loop keeps the kept-key state in place across steps)
    const int nmine = __popc(mask);
    int nit = 0;
#pragma unroll
    for (int b = 32; b > 0; b >>= 1) nit += ballot(nmine >= nit + b) ? b : 0;
    for (int it = 0; it < nit; ++it) {
        const bool has = mask != 0;
        const int j = __builtin_ctz(mask | 0x80000000u);
        mask &= mask - 1;
        float t = qv[0] - cx[j];
        float dd = t * t;
#pragma unroll
        for (int d = 1; d < ND; ++d) {
            t = qv[d] - cx[d * NBX_LEAF + j];
            dd = __builtin_fmaf(t, t, dd);
        }
        constexpr uint32_t TM = GShape<KMAX>::TM;
        const uint32_t key = (__float_as_uint(dd) & ~TM) | (c.root & TM);
        c.root = gtop_replace<KMAX>(hk, sl, lane, gm, has && key < c.root, key, rbase + j, c.root);
    }
    __syncthreads();
}

// The 8 nodes three levels below an opened node, tested at once (6-D).  A
// wave of 64 queries opens about 600 leaves there, each wanted by 10 of them
// on average, so testing one node at a time for all 64 lanes spends 2500 box
// tests, each behind a load of its own, mostly on lanes that ruled the node
// out above.  Here the lanes that want the node are compacted into LDS and
// each step tests 8 of them against the 8 boxes, one pair per lane; the 7
// planes that order them are evaluated one per lane.  The tests use the
// bounds from before the first of the 8 is entered, so they never miss one
// that the walk by single nodes opens.
// Measured on 2.1M particles, k = 64: 51.9 -> 42.4 ms with the leaves under a
// height-3 node tested so, 39.2 with the queries and masks of this test and
// of the leaf scan in 16-byte LDS rows, 37.1 with the height-3 nodes under a
// height-6 node tested the same way and the leaf data loaded a leaf ahead
// (308,000 -> 273,000 VALU per wave over the last two).  It still waits for
// half its cycles: 18.9 KB of LDS a wave leave 2 waves per SIMD.
// order: the 8 in visiting order, 3 bits each; todo: bit i set when the i-th
// of that order is open; returns the lane's own mask, by child.
template <int ND>
__device__ __forceinline__ uint32_t mix_test8(const float *boxp, const float *planep, int node, int height, float th,
                                              const float *q32, const float *qc, int anc, bool want, float *cx,
                                              int lane, uint32_t &order, uint32_t &todo) {
    const int l8 = lane & 7;
    // the box of this lane's child
    const float4 *bp = (const float4 *)(boxp + (size_t)(8 * node + l8) * 2 * ND);
    float bx[2 * ND];
#pragma unroll
    for (int i = 0; i < ND / 2; ++i) {
        const float4 v = bp[i];
        bx[4 * i] = v.x;
        bx[4 * i + 1] = v.y;
        bx[4 * i + 2] = v.z;
        bx[4 * i + 3] = v.w;
    }
    // which half comes first: bit 0 the node's, bits 1-2 its children's,
    // bits 3-6 its grandchildren's
    uint32_t right;
    {
        const int lv = l8 == 0 ? 0 : (l8 < 3 ? 1 : 2);
        const int nid = (node << lv) + (l8 == 7 ? 0 : l8 + 1 - (1 << lv));
        const float4 *pp = (const float4 *)(planep + (size_t)nid * 8);
        const float4 p0 = pp[0], p1 = pp[1];
        float s = __builtin_fmaf(p0.x, qc[0], 0.0f);
        s = __builtin_fmaf(p0.y, qc[1], s);
        s = __builtin_fmaf(p0.z, qc[2], s);
        s = __builtin_fmaf(p0.w, qc[3], s);
        s = __builtin_fmaf(p1.x, qc[4], s);
        s = __builtin_fmaf(p1.y, qc[5], s);
        bool r = s > p1.z;
        if ((anc >> (height - lv)) == nid) r = (anc >> (height - 1 - lv)) & 1;  // the wave's own leaves first
        right = (uint32_t)ballot(r) & 0x7fu;
    }
    const uint64_t wm = ballot(want);
    const int nwq = __popcll(wm);
    const int rank = __builtin_amdgcn_mbcnt_hi((uint32_t)(wm >> 32), __builtin_amdgcn_mbcnt_lo((uint32_t)wm, 0u));
    if (want) mix_put_query<ND>(cx, rank, q32, th);
    __syncthreads();
    // the step's ballot holds 8 bits per query: byte r of mb is the mask of
    // the query with rank r
    uint8_t *mb = (uint8_t *)(cx + MX_QW(ND) * NBX_WAVE);
    const float4 *qm = (const float4 *)cx;
    uint64_t any = 0;
    for (int it = 0; it < nwq; it += 8) {
        const int qs = it + (lane >> 3);
        const int q = qs < nwq ? qs : it;
        const float4 a = qm[2 * q], b = qm[2 * q + 1];
        const float x[6] = {a.x, a.y, a.z, a.w, b.x, b.y};
        float s = 0.0f;
#pragma unroll
        for (int d = 0; d < ND; ++d) {  // box_lb32
            const float t = fmaxf(bx[d] - x[d], x[d] - bx[ND + d]);
            const float tl = fmaxf(__builtin_fmaf(t, 1.0f - 0x1p-20f, -0x1p-20f * fabsf(x[d])), 0.0f);
            s = __builtin_fmaf(tl, tl, s);
        }
        const uint64_t pm = ballot(qs < nwq && s <= b.z);
        if (lane == 0) *(uint64_t *)(mb + it) = pm;
        any |= pm;
    }
    __syncthreads();
    const uint32_t mine = want ? mb[rank] : 0u;
    uint32_t open = (uint32_t)(any | (any >> 32));
    open |= open >> 16;
    open = (open | (open >> 8)) & 0xffu;
    uint32_t od = 0, td = 0;
#pragma unroll
    for (int i = 0; i < 8; ++i) {
        const uint32_t a = (uint32_t)(i >> 2) ^ (right & 1u);
        const uint32_t b = 2u * a + (((uint32_t)(i >> 1) & 1u) ^ ((right >> (1u + a)) & 1u));
        const uint32_t l = 2u * b + (((uint32_t)i & 1u) ^ ((right >> (3u + b)) & 1u));
        od |= l << (3 * i);
        td |= ((open >> l) & 1u) << i;
    }
    order = __builtin_amdgcn_readfirstlane(od);
    todo = __builtin_amdgcn_readfirstlane(td);
    return mine;
}
__device__ __forceinline__ int mix_next8(uint32_t order, uint32_t todo) {
    return (int)((order >> (3 * __builtin_ctz(todo))) & 7u);
}

// An opened node of height 3: its leaves, each loaded while the one before
// it is consumed.
template <int ND, int KMAX>
__device__ __forceinline__ void mix_sub8(const MixSrc<ND> &S, const float *boxp, const float *planep, int node,
                                         int nleafp, MixCtx<ND> &c, const float *q32, const float *qc, int anc,
                                         bool want, uint32_t *hk, uint32_t *sl, float *cx, int lane,
                                         uint32_t (&gm)[GShape<KMAX>::G]) {
    uint32_t order, todo;
    const uint32_t mine = mix_test8<ND>(boxp, planep, node, 3, __uint_as_float(c.root), q32, qc, anc, want, cx, lane,
                                        order, todo);
    if (!todo) return;
    const int leaf0 = 8 * node - nleafp;
    int l = mix_next8(order, todo);
    MixPre pre;
    mix_load(S, leaf0 + l, lane, pre);
    for (;;) {
        todo &= todo - 1;
        const int ln = todo ? mix_next8(order, todo) : l;
        MixPre nxt;
        mix_load(S, leaf0 + ln, lane, nxt);
        if (c.nvis >= MX_V) return;  // visit table full: lanes fall back
        mix_leaf<ND, KMAX>(S, leaf0 + l, c, (mine >> l) & 1u, hk, sl, cx, lane, gm, pre);
        if (!todo) return;
        l = ln;
        pre = nxt;
    }
}

// Stackless depth-first walk, begun at the wave's own leaf (3-D) or its
// ancestor three or six levels up (6-D): elsewhere the child nearer to the
// wave's first query comes first; firstright[dep] records
// which child was entered first at each depth.  Two loop forms visit the
// nodes in the same order; the compiler schedules them differently, and the
// measured faster one is used for each dimensionality (3-D: climb to the
// next unvisited sibling in an inner loop; 6-D: one node step per trip).
template <int ND, int KMAX>
__device__ __forceinline__ void mix_walk(const DevTree &T, const double *ext, MixCtx<ND> &c, const float *qc, int anc,
                                         uint32_t *hk, uint32_t *sl, float *cx, int lane,
                                         uint32_t (&gm)[GShape<KMAX>::G]) {
    // The depth and the box and plane bases as scalar values of their own.
    // The tree view arrives as wide blocks of scalar registers, and the
    // register allocator spills and restores such a block whole: a field
    // read from it in the loop brought back 16 registers (16 v_readlane)
    // per node in 6-D.
    int D = T.depth, nleafp = T.nleafp;
    const float *boxp = T.boxf;
    const float *planep = T.plane;
    asm volatile("" : "+s"(D), "+s"(nleafp), "+s"(boxp), "+s"(planep));
    // node tests in FP32 on the outward-rounded boxes: never above the FP64
    // bound, so every node the FP64 test opens is opened (a lane past the end
    // sits at 1e30, beyond every box)
    float q32[ND];
#pragma unroll
    for (int d = 0; d < ND; ++d) q32[d] = c.act ? (float)c.q[d] : NBX_PAD_COORD_F;
    MixSrc<ND> S;
    S.org = T.org;
    S.ext = ext;
    asm volatile("" : "+s"(S.org), "+s"(S.ext));
    if constexpr (ND == 3) {
        S.xq = T.xq;
        asm volatile("" : "+s"(S.xq));
    } else {
#pragma unroll
        for (int d = 0; d < ND; ++d) {
            S.xf[d] = T.xf[d];
            asm volatile("" : "+v"(S.xf[d]));
        }
    }
    // The walk starts where the first descent ends: every node on the way to
    // the wave's own leaf is open (nothing is kept yet), and its child toward
    // the leaf goes first.  Bit d of firstright is that child's last bit at
    // depth d, the path's bits from the root down.
    int node = anc, dep = D;
    uint64_t firstright = (uint64_t)(__builtin_bitreverse32((uint32_t)anc) >> (31 - D)) & ~1ULL;
    if constexpr (ND == 3) {
        for (;;) {
            cfptr bx = (cfptr)(boxp + (size_t)node * 2 * ND);
            const bool want = box_lb32<ND>(q32, bx) <= __uint_as_float(c.root);
            if (ballot(want)) {
                if (dep == D) {
                    if (c.nvis >= MX_V) break;  // visit table full: lanes fall back
                    mix_leaf<ND, KMAX>(S, node - nleafp, c, want, hk, sl, cx, lane, gm, MixPre());
                } else {
                    const int first = 2 * node + (first_is_right<ND>(planep, node, qc) ? 1 : 0);
                    dep += 1;
                    firstright = (firstright & ~(1ULL << dep)) | ((uint64_t)(first & 1) << dep);
                    node = first;
                    continue;
                }
            }
            while (node != 1 && (uint64_t)(node & 1) != ((firstright >> dep) & 1ULL)) {
                node >>= 1;
                dep -= 1;
            }
            if (node == 1) break;
            node ^= 1;
        }
    } else {
        if (D >= 6) {  // (below the node of height 6 in mix_test8's order)
            node = anc >> 6;
            dep = D - 6;
        } else if (D >= 3) {
            node = anc >> 3;
            dep = D - 3;
        }
        bool down = true;
        for (;;) {
            if (down) {
                cfptr bx = (cfptr)(boxp + (size_t)node * 2 * ND);
                const bool want = box_lb32<ND>(q32, bx) <= __uint_as_float(c.root);
                if (ballot(want)) {
                    if (dep == D) {
                        // trees of fewer than 8 leaves only: the rest end in mix_sub8
                        if (c.nvis >= MX_V) break;  // visit table full: lanes fall back
                        MixPre pre;
                        mix_load(S, node - nleafp, lane, pre);
                        mix_leaf<ND, KMAX>(S, node - nleafp, c, want, hk, sl, cx, lane, gm, pre);
                        down = false;
                    } else if (dep == D - 3 || dep == D - 6) {
                        // height 3, or height 6: the height-3 nodes under it in turn
                        uint32_t order = 0, todo = 1, mine = want ? 1u : 0u;
                        const int n0 = dep == D - 6 ? 8 * node : node;
                        if (dep == D - 6)
                            mine = mix_test8<ND>(boxp, planep, node, 6, __uint_as_float(c.root), q32, qc, anc, want, cx,
                                                 lane, order, todo);
                        while (todo) {
                            const int l = mix_next8(order, todo);
                            todo &= todo - 1;
                            mix_sub8<ND, KMAX>(S, boxp, planep, n0 + l, nleafp, c, q32, qc, anc, (mine >> l) & 1u, hk, sl,
                                               cx, lane, gm);
                            if (c.nvis >= MX_V) break;
                        }
                        if (c.nvis >= MX_V) break;
                        down = false;
                    } else {
                        const int first = 2 * node + (first_is_right<ND>(planep, node, qc) ? 1 : 0);
                        dep += 1;
                        if (first & 1) firstright |= (1ULL << dep);
                        else firstright &= ~(1ULL << dep);
                        node = first;
                        continue;
                    }
                } else {
                    down = false;
                }
            }
            if (node == 1) break;
            if ((uint64_t)(node & 1) == ((firstright >> dep) & 1ULL)) {
                node ^= 1;
                down = true;
            } else {
                node >>= 1;
                dep -= 1;
            }
        }
    }
}

template <int ND>
__device__ __forceinline__ double d64(const DevTree &T, const double *q, int32_t s) {
    double d2 = 0.0;
#pragma unroll
    for (int d = 0; d < ND; ++d) {
        double t = q[d] - T.x[d][s];
        d2 += t * t;
    }
    return d2;
}

// Exact FP64 check of a candidate set: counts the particles whose key
// (d2, ID) is below (Dk, IDk) -- self and d2 == 0 excluded, as in the target
// search -- within the ball of radius^2 Dk, for the lanes with act set.
// Wave-uniform left-first walk; leaves through 64-byte scalar loads.
template <int ND>
__device__ __forceinline__ int verify_walk(const DevTree &T, const double *q, bool act, double Dk, int32_t IDk,
                                           int32_t self) {
    constexpr int CH = ND == 6 ? 4 : 8;
    typedef double dxc __attribute__((ext_vector_type(CH)));
    typedef const __attribute__((address_space(4))) dxc *cdcptr;
    int cnt = 0;
    int node = 1;
    bool down = true;
    for (;;) {
        if (down) {
            cdptr bx = (cdptr)node_box(T, node, ND);
            bool want = act && box_lb<ND>(q, bx) <= Dk;
            if (ballot(want)) {
                if (node >= T.nleafp) {
                    const int base = (node - T.nleafp) * NBX_LEAF;
#pragma unroll
                    for (int jj = 0; jj < NBX_LEAF; jj += CH) {
                        dxc cv[ND];
#pragma unroll
                        for (int d = 0; d < ND; ++d) cv[d] = *(cdcptr)(T.x[d] + base + jj);
#pragma unroll
                        for (int u = 0; u < CH; ++u) {
                            double d2 = 0.0;
#pragma unroll
                            for (int d = 0; d < ND; ++d) {
                                const double t = q[d] - cv[d][u];
                                d2 += t * t;
                            }
                            const int32_t cs = base + jj + u;
                            bool below = d2 < Dk;
                            if (d2 == Dk && act && cs != self) below = T.perm[cs] < IDk;
                            cnt += (act && want && d2 > 0.0 && cs != self && below) ? 1 : 0;
                        }
                    }
                    down = false;
                } else {
                    node = 2 * node;
                    continue;
                }
            } else {
                down = false;
            }
        }
        if (node == 1) break;
        if (!(node & 1)) {
            node ^= 1;
            down = true;
        } else {
            node >>= 1;
        }
    }
    return cnt;
}

// After the sort: kept keys in ascending order (SKC) and their slots (SLOT).
// When KMAX <= 33 the keys are sorted in place in LDS and a key's tag is
// its slot's scratch position; else keys and slots are sorted into two more
// scratch regions.
#define SKC(p) kb[(p) * NBX_WAVE + lane]
#define SLB(p) slb[(p) * NBX_WAVE + lane]

// What an instance does with the neighbours it found.  Instances of their
// own, because code in the table instance changes its register allocation.
//  * EXACT orders the rows before they leave LDS and computes d2 as they are
//    written, coalesced.  A kernel that read the rows back, one thread per
//    row, and sorted them in per-thread arrays (scratch memory) took 1.53 ms
//    for 1M rows of 20; here they cost under 0.1 ms.
//  * SPLINE sums the differentiation form's forward over the neighbours while
//    their slots are in LDS, so no list is written or read.
#define MX_TABLE 0   // the table densities, rows in key order
#define MX_EXACT 1   // no density; rows in ascending (d2, ID) order, with d2 when asked for
#define MX_SPLINE 2  // the analytic-spline symmetric density (NBX_DO_SPLINE), no rows

// One wave of 64 consecutive queries (tree order), wave index g.
// k = kh - 1 neighbours; A.dens: NBX_DO_NONE / NBX_DO_SYM / NBX_DO_GATHER, or
// as MODE says.
template <int ND, int KMAX, int MODE>
__device__ __forceinline__ void mix_task(const DevTree &T, const KnnArgs &A, const double *ext, int32_t *fb_list,
                                         int32_t *fb_count, uint32_t *hk, float *cx, double *racc, uint32_t *sl,
                                         uint32_t *slb, uint32_t *skc, int g, int part, int plog, int lane) {
    constexpr bool GT = GShape<KMAX>::GT;
    constexpr uint32_t TM = GShape<KMAX>::TM;
    uint32_t *const kb = GT ? hk : skc;
    // slot of sorted entry p; move sorted entry src to dst
    uint32_t *const vt = sl + KMAX * (NBX_WAVE / 2);  // visit table
    auto slot_at = [&](int p) -> int32_t {
        if constexpr (GT) {
            const uint32_t h = SLH(SKC(p) & TM);
            return (int32_t)(vt[h >> 5] * NBX_LEAF + (h & 31u));
        } else {
            return (int32_t)SLB(p);
        }
    };
    auto move_entry = [&](int dst, int src) {
        if constexpr (GT) SKC(dst) = SKC(src);
        else SLB(dst) = SLB(src);
    };
    // k + 1, opaque to the compiler so nothing derived from it is hoisted
    // out of the workgroup's loop into registers
    int kh = A.kh;
    asm volatile("" : "+s"(kh));
    const int k = kh - 1;
    const int qi = g * NBX_WAVE + lane;
    const bool valid = qi < T.n && lane >> (6 - plog) == part;
    const int kres = T.kernres;
    MixCtx<ND> c;
    // A lane past the end, or of another part, queries from the padding sentinel: node boxes
    // bound real particles only, so every box bound from there is +inf and
    // the walk needs no activity test (the leaf code still masks the lane).
    float qc[ND];
#pragma unroll
    for (int d = 0; d < ND; ++d) {
        const double x = qi < T.n ? T.x[d][qi] : NBX_PAD_COORD;
        qc[d] = (float)readfirst_d(x);  // the order of the walk is the whole wave's
        c.q[d] = valid ? x : NBX_PAD_COORD;
    }
    c.act = valid;
    c.self = qi;
    c.root = 0u;
    c.emax = 0.0;
    uint32_t gm[GShape<KMAX>::G];
    c.root = gtop_init<KMAX>(hk, lane, kh, gm);
    // every slot read later is a valid index: handle 0 names the leaf in
    // visit table entry 0, first the wave's own leaf, then the first leaf
    // with an accepted candidate
    for (int p = 0; p < kh; ++p) SLH(p) = 0;
    if (lane == 0) vt[0] = (uint32_t)(2 * g);
    c.nvis = 0;
    c.fillkh = (GT && kh >= NBX_LEAF) ? kh : 0;
    mix_walk<ND, KMAX>(T, ext, c, qc, T.nleafp + 2 * g, hk, sl, cx, lane, gm);

    // ---------------------------------------------------------------- band
    const bool ovf = c.nvis >= MX_V;  // walk stopped early: no certificate
    bool ok = valid && !ovf;
    if (valid) {
        // rank sort of the kh kept keys: keys to SKC, slots to SLB
        if constexpr (GT) {
            // unique keys (unused positions +inf) sorted in registers by the
            // network, then stored back in order
            static_assert(KMAX == 33, "the sorting network is built for 33 keys");
            uint32_t kq[KMAX];
#pragma unroll
            for (int p = 0; p < KMAX; ++p) kq[p] = p < kh ? HK(p) : 0xffffffffu;
#pragma unroll
            for (int e = 0; e < MX_NET33.n; ++e) {
                const uint32_t x = kq[MX_NET33.a[e]], y = kq[MX_NET33.b[e]];
                kq[MX_NET33.a[e]] = min(x, y);
                kq[MX_NET33.b[e]] = max(x, y);
            }
#pragma unroll
            for (int p = 0; p < KMAX; ++p)
                if (p < kh) HK(p) = kq[p];
        } else {
            // ties (possible only between groups) by position
            uint32_t kq[KMAX];
#pragma unroll
            for (int p = 0; p < KMAX; ++p) kq[p] = p < kh ? HK(p) : 0xffffffffu;
            for (int i = 0; i < kh; ++i) {
                const uint32_t ki = HK(i);
                int r = 0;
#pragma unroll
                for (int j = 0; j < KMAX; ++j) r += (kq[j] < ki || (kq[j] == ki && j < i)) ? 1 : 0;
                const uint32_t h = SLH(i);
                SKC(r) = ki;
                SLB(r) = vt[h >> 5] * NBX_LEAF + (h & 31u);
            }
        }
        if ((SKC(kh - 1) & ~GShape<KMAX>::TM) == (MX_EMPTY & ~GShape<KMAX>::TM)) ok = false;  // < k+1 candidates
    }
    // FP32 search error plus the key's position bits, or the caller's
    // re-check band where that is wider (a wider band only sends more
    // entries to the FP64 re-check and the exact verification)
    const double eu = fmax((12.0 + (double)(1 << GShape<KMAX>::TB)) * MX_U, A.band_rel), ea = 5.0 * MX_U * c.emax;
    int i0 = k - 1;
    int32_t bs[4];
    uint32_t bk[4];
    double bd[4];
    double Dk = 0.0;
    if (ok) {
        // band: entries whose interval overlaps the k-th entry's
        double dk = sqrt((double)__uint_as_float(SKC(k - 1)));
        double lo_k = dk - (eu * dk + ea);
        while (i0 > 0) {
            double di = sqrt((double)__uint_as_float(SKC(i0 - 1)));
            if (di + (eu * di + ea) < lo_k) break;
            --i0;
        }
        // a certain entry that could be an exact duplicate (d2 == 0) must be checked too
        double d0 = sqrt((double)__uint_as_float(SKC(0)));
        if (d0 - (eu * d0 + ea) <= 0.0 && i0 > 0) ok = false;
        if (kh - i0 > 4) ok = false;
    }
    if (ok) {
        // recompute the band in FP64; drop one entry: a d2 == 0 duplicate if
        // present, else the largest (d2, ID)
        const int nb = kh - i0;
        int drop = -1, nzero = 0;
#pragma unroll
        for (int b = 0; b < 4; ++b) {
            bs[b] = -1;
            bd[b] = 0.0;
            if (b < nb) {
                bk[b] = SKC(i0 + b);
                bs[b] = slot_at(i0 + b);
                bd[b] = d64<ND>(T, c.q, bs[b]);
                if (bd[b] == 0.0) { nzero++; drop = b; }
            }
        }
        if (nzero > 1) ok = false;
        if (drop < 0) {
            // the largest (d2, ID) of the band (static indices only)
            drop = 0;
            double dd = bd[0];
            int32_t pd = T.perm[bs[0]];
#pragma unroll
            for (int b = 1; b < 4; ++b) {
                const int32_t pb = b < nb ? T.perm[bs[b]] : 0;
                if (b < nb && (bd[b] > dd || (bd[b] == dd && pb > pd))) {
                    drop = b;
                    dd = bd[b];
                    pd = pb;
                }
            }
        }
        Dk = 0.0;
#pragma unroll
        for (int b = 0; b < 4; ++b)
            if (b < nb && b != drop && bd[b] > Dk) Dk = bd[b];
        // certificate against everything outside the heap
        double dl = sqrt((double)__uint_as_float(SKC(kh - 1)));
        double lout = dl - (eu * dl + ea);
        if (!(lout > 0.0 && Dk < lout * lout)) ok = false;
        if (ok) {
            // the kept band entries fill positions i0 .. k-1 (FP32 order)
#pragma unroll
            for (int b = 0; b < 4; ++b)
                if (b < nb && b != drop) {
                    const int dst = i0 + b - (b > drop ? 1 : 0);
                    if constexpr (GT) SKC(dst) = bk[b];
                    else SLB(dst) = (uint32_t)bs[b];
                }
        }
    }
    // exact verification for lanes the error bound could not decide: keep
    // the k smallest (d2, ID) of the k+1 candidates in FP64, then count in
    // FP64 the particles below the k-th of them
    bool verify = valid && !ok && !ovf && (SKC(kh - 1) & ~GShape<KMAX>::TM) != (MX_EMPTY & ~GShape<KMAX>::TM);
    int32_t IDk = 0;
    if (verify) {
        int zero_at = -1, nzero = 0, maxp = -1;
        double dmax = -1.0;
        int32_t imax = -1;
        for (int p = 0; p < kh; ++p) {
            int32_t s = slot_at(p);
            double d = d64<ND>(T, c.q, s);
            if (d == 0.0) {
                nzero++;
                zero_at = p;
                continue;
            }
            int32_t id = T.perm[s];
            if (maxp < 0 || d > dmax || (d == dmax && id > imax)) { maxp = p; dmax = d; imax = id; }
        }
        const int drop = nzero == 1 ? zero_at : maxp;
        if (nzero > 1) verify = false;
        if (verify) {
            for (int p = drop; p < kh - 1; ++p) move_entry(p, p + 1);
            Dk = 0.0;
            IDk = -1;
            for (int p = 0; p < k; ++p) {
                int32_t s = slot_at(p);
                double d = d64<ND>(T, c.q, s);
                int32_t id = T.perm[s];
                if (d > Dk || (d == Dk && id > IDk)) { Dk = d; IDk = id; }
            }
        }
    }
    if (ballot(verify)) {
        int cnt = verify_walk<ND>(T, c.q, verify, Dk, IDk, qi);
        if (verify && cnt == k - 1) ok = true;
    }
    // fallback list for the FP64 kernel
    uint64_t fbm = ballot(valid && !ok);
    if (fbm) {
        int base = 0;
        if (lane == 0) base = atomicAdd(fb_count, __popcll(fbm));
        base = __shfl(base, 0);
        if (valid && !ok) fb_list[base + __popcll(fbm & ((1ULL << lane) - 1))] = qi;
    }

    // k <= 32: the slots of the k kept entries, decoded in one batch (every
    // handle load, then every visit-table load, instead of a dependent pair
    // per entry) and stored over their keys, which nothing reads after this;
    // the density and the output rows take them from there
    if constexpr (GT) {
        if (ok) {
            const gu32 *vtg = (const gu32 *)vt;
            uint32_t hv[KMAX];
#pragma unroll
            for (int p = 0; p < KMAX; ++p) hv[p] = p < k ? (uint32_t)SLH(SKC(p) & TM) : 0u;
#pragma unroll
            for (int p = 0; p < KMAX; ++p)
                if (p < k) SKC(p) = vtg[hv[p] >> 5] * NBX_LEAF + (hv[p] & 31u);
        }
    }
    auto slot_final = [&](int p) -> int32_t {
        if constexpr (GT) return (int32_t)SKC(p);
        else return (int32_t)SLB(p);
    };

    // ---------------------------------------------------------------- density
    // Symmetric scatter: contributions to the wave's own 64 queries (about
    // half of all neighbour entries) are summed in LDS and flushed with one
    // atomic per query; the rest go straight to HBM.
    const bool sym = MODE == MX_SPLINE || (MODE == MX_TABLE && A.dens == NBX_DO_SYM);
    double racc_own = 0.0;
    const bool dens_here = MODE != MX_EXACT && ok && A.dens != NBX_DO_NONE;
    if (sym) racc[lane] = 0.0;
    __syncthreads();
    if (dens_here) {
        // weights from FP64 distances of the k selected neighbours (the FP32
        // offsets carry a storage error proportional to the leaf size)
        const double hi = 0.5 * sqrt(Dk);
        double norm, ih = 0.0;
        if constexpr (MODE == MX_SPLINE) {
            ih = 1.0 / hi;
            norm = 0.5 * NBX_SIGMA3 * ih * ih * ih;
        } else {
            norm = 1.0 / pow(hi, (double)ND);
        }
        const double mi = T.mass[qi];
        // the table lookup of Wsm (KDCalcSmoothQuantities.cxx:12-15) with
        // its division by the table step turned into a product: index
        // floor(r/h * c), c = (kernres - 1) / 2 = 1 / step, and the linear
        // weight of the next entry the index's fraction.  r/h stays a
        // division, so the k-th neighbour's is exactly 2 and it takes the
        // table's last entry, as in the reference.
        const double ck = 0.5 * (kres - 1);
        double acc = 0.0;
        // neighbours in groups of MX_DB so their coordinate/mass gathers are in
        // flight together
        for (int p0 = 0; p0 < k; p0 += MX_DB) {
            int32_t sv[MX_DB];
            double d2v[MX_DB], mv[MX_DB];
#pragma unroll
            for (int u = 0; u < MX_DB; ++u) {
                sv[u] = p0 + u < k ? slot_final(p0 + u) : qi;
                d2v[u] = d64<ND>(T, c.q, sv[u]);
                mv[u] = T.mass[sv[u]];
            }
#pragma unroll
            for (int u = 0; u < MX_DB; ++u) {
                if (p0 + u >= k) break;
                const int32_t s = sv[u];
                double W;
                if constexpr (MODE == MX_SPLINE) {
                    W = w_cubic(sqrt(d2v[u]) * ih);
                } else {
                    const double fi = sqrt(d2v[u]) / hi * ck;
                    if (!(fi < (double)(kres - 1))) {
                        W = T.kern[kres - 1];
                    } else {
                        const int i = (int)fi;
                        W = T.kern[i] + (T.kern[i + 1] - T.kern[i]) * (fi - (double)i);
                    }
                }
                if (sym) {
                    const double Wij = MODE == MX_SPLINE ? W * norm : 0.5 * W * norm;
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
    __syncthreads();
    if (sym && (valid || (qi < T.n && racc[lane] != 0.0))) unsafeAtomicAdd(A.rho + qi, racc_own + racc[lane]);

    // ---------------------------------------------------------------- outputs
    if constexpr (MODE == MX_SPLINE) return;
    if (A.nn == nullptr && (MODE != MX_EXACT || A.d2 == nullptr)) return;
    if constexpr (MODE == MX_EXACT) {
        // The entries come in key order, which departs from (d2, ID) order
        // only between neighbouring keys.  Passes that carry the larger of
        // two neighbours along run until one changes nothing (one or two
        // passes; as many as a shell has members on a lattice).
        auto slot_put = [&](int p, int32_t s) {
            if constexpr (GT) SKC(p) = (uint32_t)s;
            else SLB(p) = (uint32_t)s;
        };
        for (bool again = ok; ballot(again);) {
            if (again) {
                again = false;
                int32_t sc = slot_final(0);
                double dc = d64<ND>(T, c.q, sc);
                for (int p0 = 1; p0 < k; p0 += MX_DB) {
                    int32_t sv[MX_DB];
                    double dv[MX_DB];
#pragma unroll
                    for (int u = 0; u < MX_DB; ++u) {
                        sv[u] = p0 + u < k ? slot_final(p0 + u) : qi;
                        dv[u] = d64<ND>(T, c.q, sv[u]);
                    }
#pragma unroll
                    for (int u = 0; u < MX_DB; ++u) {
                        if (p0 + u >= k) break;
                        bool below = dv[u] < dc;
                        if (dv[u] == dc) below = T.perm[sv[u]] < T.perm[sc];
                        slot_put(p0 + u - 1, below ? sv[u] : sc);
                        sc = below ? sc : sv[u];
                        dc = below ? dc : dv[u];
                        again |= below;
                    }
                }
                slot_put(k - 1, sc);
            }
        }
    }
    const uint64_t okm = ballot(ok);
    __syncthreads();
    if constexpr (ND == 3 && MODE == MX_TABLE && GT) {
        if (A.layout == 1) {
            // rows by slot: the wave's rows are one run of memory, entry e =
            // lane + 64 i at its e-th place; only the LDS index (row r,
            // column t) has to be stepped (16.8M particles, k = 32: the search
            // 17.60 -> 17.35 ms)
            const int q64 = NBX_WAVE / k, m64 = NBX_WAVE - q64 * k;
            int r = lane / k, t = lane - r * k;
            int32_t *out = A.nn + (int64_t)(g * NBX_WAVE - A.row0) * k + lane;
            asm volatile("" : "+v"(out));
            for (int i = 0; i < k; ++i, out += NBX_WAVE, t += m64, r += q64) {
                if (t >= k) {
                    t -= k;
                    r += 1;
                }
                if ((okm >> r) & 1ULL) *out = (int32_t)hk[t * NBX_WAVE + r];
            }
            return;
        }
    }
    // entry e = lane + 64 i of the wave's rows is row r = e / k, column
    // t = e % k: stepped without a division in 3-D, divided in 6-D (each the
    // measured faster form of its instance)
    const int q64 = NBX_WAVE / k, m64 = NBX_WAVE - q64 * k;
    int r = lane / k, t = lane - (lane / k) * k;
    for (int i = 0; i < k; ++i, t += m64, r += q64) {
        if constexpr (ND == 3) {
            if (t >= k) {
                t -= k;
                r += 1;
            }
        } else {
            const int e = lane + NBX_WAVE * i;
            r = e / k;
            t = e - r * k;
        }
        int qr = g * NBX_WAVE + r;
        if (qr >= T.n) break;
        if (!((okm >> r) & 1ULL)) continue;
        int32_t s;
        if constexpr (GT) s = (int32_t)hk[t * NBX_WAVE + r];  // decoded above
        else s = (int32_t)slb[t * NBX_WAVE + r];
        int64_t row = A.layout == 1 ? qr - A.row0 : T.perm[qr];
        if (MODE != MX_EXACT || A.nn) A.nn[row * k + t] = A.layout == 1 ? s : T.perm[s];
        if constexpr (MODE == MX_EXACT) {
            if (A.d2) {
                double q[ND];
#pragma unroll
                for (int d = 0; d < ND; ++d) q[d] = T.x[d][qr];
                A.d2[row * k + t] = d64<ND>(T, q, s);
            }
        }
    }
}

// Persistent precision-form kernel, one wave per workgroup.  Workgroup b
// stays on XCD (b mod 8) (workgroups are dealt to XCDs round robin), takes
// waves of queries from that XCD's contiguous share of the tree order (the
// xcd_wave split) through the XCD's counter, and owns one scratch block of
// MX_BLKW(KMAX) words (16-bit handles by position and the visit table; for
// KMAX > 33 also slots and keys in ascending order) for its whole life, so
// the scratch is sized by the resident workgroups and only ever touched from
// one XCD.  Once its own
// share is drained a workgroup takes waves from the other XCDs' counters in
// turn (each ticket names one wave, so every wave runs once), which evens out
// shares of unequal cost; it exits when all eight counters have passed their
// shares' ends.
#define MX_CTR_STRIDE 16  // XCD counters 64 bytes apart
// scratch words per workgroup: 16-bit handles and the visit table, and for
// KMAX > 33 the slots and keys in ascending order
#define MX_BLKW(KM) ((KM) * (NBX_WAVE / 2) + MX_V + ((KM) <= 33 ? 0 : 2 * (KM) * NBX_WAVE))
// (6-D, k <= 32: LDS allows 15 waves per CU, so the registers are held to the
// 128 that four waves per SIMD leave)
template <int ND, int KMAX, int MODE>
__global__ __launch_bounds__(64, ND == 6 && KMAX == 33 ? 4 : 1)
void k_knn_mixed(DevTree T, KnnArgs A, const double *ext, int32_t *fb_list, int32_t *fb_count, uint32_t *scratch,
                 int32_t *ctr, int plog) {
    __shared__ uint32_t hk[KMAX * NBX_WAVE];
    // one buffer for three uses at different times: the leaf copy (phase 2),
    // the compacted queries and their masks (6-D node tests and phase 1) and
    // the symmetric scatter into the wave's own queries (density)
    constexpr int UB1 = (MX_QW(ND) + 1) * MX_QMAX(ND);
    constexpr int UBN = UB1 > ND * NBX_LEAF + 2 * NBX_WAVE ? UB1 : ND * NBX_LEAF + 2 * NBX_WAVE;
    __shared__ __attribute__((aligned(16))) float ub[UBN];
    float *cx = ub;
    double *racc = (double *)(ub + ND * NBX_LEAF);
    const int lane = threadIdx.x;
    uint32_t *sl = scratch + (size_t)blockIdx.x * MX_BLKW(KMAX);
    // kept in a VGPR pair: the scalar registers are oversubscribed, and a
    // scalar base would be reloaded from its spill slot at every handle store
    asm volatile("" : "+v"(sl));
    uint32_t *slb = sl + KMAX * (NBX_WAVE / 2) + MX_V, *skc = slb + KMAX * NBX_WAVE;
    const int nw = (A.wcnt > 0 ? A.wcnt : (T.n + NBX_WAVE - 1) / NBX_WAVE) << plog;
    const int x = blockIdx.x & 7, q8 = nw >> 3, r8 = nw & 7;
    for (int s = 0; s < 8; ++s) {
        const int y = (x + s) & 7;
        const int ybeg = y * q8 + (y < r8 ? y : r8), ycnt = q8 + (y < r8 ? 1 : 0);
        for (;;) {
            int t = 0;
            if (lane == 0) t = atomicAdd(ctr + y * MX_CTR_STRIDE, 1);
            t = __builtin_amdgcn_readfirstlane(__shfl(t, 0));
            if (t >= ycnt) break;
            const int v = ybeg + t;
            mix_task<ND, KMAX, MODE>(T, A, ext, fb_list, fb_count, hk, cx, racc, sl, slb, skc, A.wbeg + (v >> plog),
                                     v & ((1 << plog) - 1), plog, lane);
        }
    }
}

__global__ void k_mx_zero(int32_t *p, int cnt) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i < cnt) p[i] = 0;
}

// Resident workgroups of one instance over the device, a multiple of 8
// (every XCD gets workgroups) and at least 8.
template <int ND, int KMAX, int MODE>
static int mx_grid() {
    static std::atomic<int> grid{0};
    if (grid.load() == 0) {
        int dev = 0, ncu = 0, per = 0;
        if (hipGetDevice(&dev) != hipSuccess) dev = 0;
        if (hipDeviceGetAttribute(&ncu, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess || ncu <= 0) ncu = 256;
        if (hipOccupancyMaxActiveBlocksPerMultiprocessor(&per, k_knn_mixed<ND, KMAX, MODE>, NBX_WAVE, 0) != hipSuccess ||
            per <= 0)
            per = 8;
        const int gsz = (per * ncu) & ~7;
        grid.store(gsz < 8 ? 8 : gsz);
    }
    return grid.load();
}

// (more than 33 kept entries: rows in key order only, see mixed_by_waves)
static int mx_launch_grid(int nd, int km, int mode) {
    if (km == 65) return nd == 3 ? mx_grid<3, 65, MX_TABLE>() : mx_grid<6, 65, MX_TABLE>();
    if (nd == 3 && mode == MX_SPLINE) return mx_grid<3, 33, MX_SPLINE>();
    if (mode == MX_EXACT) return nd == 3 ? mx_grid<3, 33, MX_EXACT>() : mx_grid<6, 33, MX_EXACT>();
    return nd == 3 ? mx_grid<3, 33, MX_TABLE>() : mx_grid<6, 33, MX_TABLE>();
}
static int mx_mode(const KnnArgs &A) {
    return A.dens == NBX_DO_SPLINE ? MX_SPLINE : (A.exact_rows || A.d2 ? MX_EXACT : MX_TABLE);
}

size_t nbx_mixed_scratch_bytes(int nd, int kh) {
    const int km = kh <= 33 ? 33 : 65;
    int g = 0;  // enough for any instance
    for (int mode = 0; mode < 3; ++mode) g = std::max(g, mx_launch_grid(nd, km, mode));
    return (size_t)g * MX_BLKW(km) * sizeof(uint32_t) + 8 * MX_CTR_STRIDE * sizeof(int32_t);
}

hipError_t nbx_launch_knn_mixed(const DevTree &T, const KnnArgs &A, const double *ext, int32_t *fallback_list,
                                int32_t *fallback_count, hipStream_t st, void *work, size_t work_bytes) {
    const int nw = A.wcnt > 0 ? A.wcnt : (T.n + NBX_WAVE - 1) / NBX_WAVE;
    if (nw == 0) return hipSuccess;
    if ((T.nd != 3 && T.nd != 6) || A.kh > 65 || A.kh < 2 || !T.kernf || !T.org || !T.boxf || !ext)
        return hipErrorInvalidValue;
    const int km = A.kh <= 33 ? 33 : 65;
    const int mode = mx_mode(A);
    // densities and exact rows do not come together; the spline is 3-D; both keep at most 33
    if ((mode != MX_TABLE && km > 33) || (mode == MX_EXACT && A.dens != NBX_DO_NONE) ||
        (mode == MX_SPLINE && (T.nd != 3 || A.nn || A.d2)))
        return hipErrorInvalidValue;
    const int grid = mx_launch_grid(T.nd, km, mode);
    // Few waves leave the device idle while each works through the union of
    // its queries' neighbourhoods, so a wave's 64 queries are split among as
    // many waves as there is room for.  The walk keeps the whole wave's order,
    // so every lane meets its candidates as before and the rows are the same.
    // Rows and density of 4096 clustered particles, k = 32, 0.26 -> 0.18 ms (a
    // query per wave: 0.22), of 10001 0.40 -> 0.25, of 32768 0.37 -> 0.33, 6-D
    // 1.65 -> 1.21; from 65536 on no difference in 3-D.
    int plog = 0;
    while (plog < MX_PLOG && ((int64_t)nw << (plog + 1)) <= grid) ++plog;
    const int ngrid = (int)std::min<int64_t>(grid, (((int64_t)nw << plog) + 7) & ~(int64_t)7);
    const size_t nscr = (size_t)grid * MX_BLKW(km);
    const size_t need = nscr * sizeof(uint32_t) + 8 * MX_CTR_STRIDE * sizeof(int32_t);
    void *mem = work;
    hipError_t e = hipSuccess;
    if (mem) {
        if (work_bytes < need) return hipErrorInvalidValue;
    } else {
        e = hipMallocAsync(&mem, need, st);
        if (e != hipSuccess) return e;
    }
    uint32_t *scr = (uint32_t *)mem;
    int32_t *ctr = (int32_t *)(scr + nscr);
    hipLaunchKernelGGL(k_mx_zero, dim3(1), dim3(8 * MX_CTR_STRIDE), 0, st, ctr, 8 * MX_CTR_STRIDE);
    {
        ProfScope ps("k_knn_mixed", st);
#define MIXL(ND, KM, MODE)                                                                                       \
    hipLaunchKernelGGL((k_knn_mixed<ND, KM, MODE>), dim3(ngrid), dim3(NBX_WAVE), 0, st, T, A, ext, fallback_list, \
                       fallback_count, scr, ctr, plog)
        if (T.nd == 3) {
            if (km == 65) MIXL(3, 65, MX_TABLE);
            else if (mode == MX_TABLE) MIXL(3, 33, MX_TABLE);
            else if (mode == MX_EXACT) MIXL(3, 33, MX_EXACT);
            else MIXL(3, 33, MX_SPLINE);
        } else {
            if (km == 65) MIXL(6, 65, MX_TABLE);
            else if (mode == MX_TABLE) MIXL(6, 33, MX_TABLE);
            else MIXL(6, 33, MX_EXACT);
        }
#undef MIXL
    }
    e = hipGetLastError();
    if (!work) hipFreeAsync(mem, st);
    return e;
}
