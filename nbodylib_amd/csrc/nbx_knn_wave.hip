// nbx_knn_wave.hip -- exact FP64 nearest neighbours, one query per wave.
//
// The same searches, densities and results as nbx_knn.hip (the reference's
// lines are cited there).  There a wave walks the tree for 64 queries, opens
// what any of them needs and pays for its busiest lane at every insertion; in
// 6-D, for many kept entries, for queries that are not one another's
// neighbours and for few queries most of that is waste.
//
// Here the 64 lanes work on one query.
//  * Nodes: an opened node has its 64 descendants six levels below tested at
//    once, one per lane; the lanes keep the bounds, and the nearest open one
//    is taken next (a minimum over the wave), so the kept distances shrink as
//    fast as they can and few leaves are read.
//  * Leaves: the four nearest at a time, two particles per lane: the address
//    unit takes 16 cycles for a load of 64 lanes whether each asks for 4 or 16
//    bytes, and with one particle per lane it, not the arithmetic, bounded the
//    6-D search (93% busy; 6.6 -> 5.6 ms for 0.5M queries, k = 64).
//  * Kept entries: sorted by (d2, ID) across the lanes (E to a lane), so ties
//    need no care, and rows leave in order and coalesced.  One to three
//    accepted particles are inserted (a compare, a shift by one lane); more
//    are sorted and merged by bitonic networks of 32-bit keys, three
//    instructions a stage, through DPP and lane swaps.  Networks of whole
//    entries took six times as many (0.5M queries, k = 32: 1.54 ms, and 0.77
//    with keys).
//  * No scratch, no counters: a call is one launch.
// Vector issue bounds it: 892 instructions a query with the density at k = 32 in
// 3-D (2.1M clustered particles; 972 of 16.8M), of which the merges are about
// half, at 73 to 79% of the peak rate under the profiler.  So the common path
// is kept short (the last few open nodes are taken without a minimum, a group's
// leaves share one scalar base address, padding needs no test of its own and
// the query's own entry is sorted out after something was accepted): 6-D, 0.5M,
// k = 64 5.68 -> 5.4 ms.
// Measured, a lane per query -> this: 4096 particles, k = 32, periodic 266 ->
// 23 us; 100k positions among 1M particles 6.17 -> 0.52 ms; 2.1M clustered
// particles, density at k = 32 4.5 -> 3.9 ms; 0.5M particles k = 64 3.8 -> 1.0,
// k = 128 17.7 -> 2.0 ms; 6-D 0.5M k = 32 21.7 -> 3.9 ms, 2.1M k = 64 (from the
// FP32 form) 36 -> 22 ms.
#include <algorithm>

#include "nbx_kernels.h"

#define WV_NOID 0x7fffffff
#define WV_LEVELS 5  // opened levels of a tree of at most 2^26 leaves

template <int CTRL>
__device__ __forceinline__ uint32_t dpp(uint32_t v) {
    return (uint32_t)__builtin_amdgcn_mov_dpp((int)v, CTRL, 0xf, 0xf, true);
}
// minimum over the wave
__device__ __forceinline__ uint32_t wave_umin(uint32_t v) {
#define WV_MIN(ctrl) v = min(v, (uint32_t)__builtin_amdgcn_update_dpp((int)0xffffffffu, (int)v, ctrl, 0xf, 0xf, false))
    WV_MIN(0x111);  // row_shr:1, 2, 4, 8, then rows 0 into 1 and 2 into 3, then the lower half into the upper
    WV_MIN(0x112);
    WV_MIN(0x114);
    WV_MIN(0x118);
    WV_MIN(0x142);
    WV_MIN(0x143);
#undef WV_MIN
    return (uint32_t)__builtin_amdgcn_readlane((int)v, 63);
}
// the lane below's value (lane 0: any; its place is never taken from below)
__device__ __forceinline__ int32_t lane_below(int32_t v) {
    return __builtin_amdgcn_update_dpp(v, v, 0x138, 0xf, 0xf, false);  // wave_shr:1
}
// sum over the wave, in lane 63
__device__ __forceinline__ double wave_sum(double v) {
    union {
        double d;
        int32_t w[2];
    } a, b;
    a.d = v;
#define WV_SUM(ctrl)                                                             \
    b.w[0] = __builtin_amdgcn_update_dpp(0, a.w[0], ctrl, 0xf, 0xf, false);      \
    b.w[1] = __builtin_amdgcn_update_dpp(0, a.w[1], ctrl, 0xf, 0xf, false);      \
    a.d += b.d
    WV_SUM(0x111);  // as wave_umin; the broadcasts reach the rows above only
    WV_SUM(0x112);
    WV_SUM(0x114);
    WV_SUM(0x118);
#undef WV_SUM
#define WV_SUM(ctrl, rows)                                                       \
    b.w[0] = __builtin_amdgcn_update_dpp(0, a.w[0], ctrl, rows, 0xf, false);     \
    b.w[1] = __builtin_amdgcn_update_dpp(0, a.w[1], ctrl, rows, 0xf, false);     \
    a.d += b.d
    WV_SUM(0x142, 0xa);
    WV_SUM(0x143, 0xc);
#undef WV_SUM
    return a.d;
}
// h^3 or h^6 to about half a unit in the last place, from the exact errors of
// the products (pow takes more instructions than the rest of the density)
template <int ND>
__device__ __forceinline__ double wv_pow(double h) {
    const double p = h * h, pe = fma(h, h, -p);
    double r = p * h, re = fma(p, h, -r) + pe * h;  // r + re = h^3
    if (ND == 3) {
        const double f = r + re;
        return f == f ? f : r;  // (an infinite h)
    }
    const double s = r * r, se = fma(r, r, -s);
    return s + (se + 2.0 * r * re);
}
__device__ __forceinline__ bool before(double da, int32_t ia, double db, int32_t ib) {
    return (da < db) | ((da == db) & (ia < ib));
}

// Kept entries of the wave's query: position p = 64 e + lane, ascending in
// (d2, ID); kth, kslot: the entry at position kh - 1, lim: its key.  IDs decide
// only between equal distances, and are looked up then.
template <int E>
struct WvKept {
    union Dbl {
        double d;
        int32_t w[2];
    } d[E];
    int32_t slot[E];
    double kth;
    int32_t kslot;
    uint32_t lim;
};
template <int E>
struct WvShared {
    uint32_t stk[WV_LEVELS][NBX_WAVE];
    double d[NBX_WAVE * (E + 1)];
    int32_t slot[NBX_WAVE * (E + 1)];
};

// (one unit above the distance's own key: a bound's last bits are free)
__device__ __forceinline__ uint32_t wv_lim(double kth) {
    return ((uint32_t)__builtin_amdgcn_readfirstlane((int)__float_as_uint((float)kth)) | 63u) + 64u;
}
template <int E>
__device__ __forceinline__ void wv_kth(WvKept<E> &k, int kh) {
    const int l = (kh - 1) & 63, at = (kh - 1) >> 6;
    double d = k.d[0].d;
    int32_t i = k.slot[0];
#pragma unroll
    for (int e = 1; e < E; ++e) {
        d = at == e ? k.d[e].d : d;
        i = at == e ? k.slot[e] : i;
    }
    k.kth = lane_d(d, l);
    k.kslot = __builtin_amdgcn_readlane(i, l);
    k.lim = wv_lim(k.kth);
}

// ID of a kept entry; an empty one comes after all others
__device__ __forceinline__ int32_t wv_id(const DevTree &T, int32_t slot) { return slot >= 0 ? T.perm[slot] : WV_NOID; }

// Insert one entry (uniform values).
template <int E>
__device__ __forceinline__ void wv_insert(const DevTree &T, WvKept<E> &k, double d, int32_t slot, int lane) {
    typename WvKept<E>::Dbl n;
    n.d = d;
    // (what leaves a block at its top enters the next one at its bottom)
#pragma unroll
    for (int e = 0; e < E; ++e) {
        uint64_t less = ballot(k.d[e].d < n.d);
        const uint64_t same = ballot(k.d[e].d == n.d);
        if (same) {
            const int32_t id = wv_id(T, slot), ki = wv_id(T, k.slot[e]);
            less |= same & ballot(ki < id);
        }
        const int p = __builtin_popcountll(less);
        if (p == NBX_WAVE) continue;
        const bool stay = lane < p;
        typename WvKept<E>::Dbl top;
        top.d = lane_d(k.d[e].d, NBX_WAVE - 1);
        const int32_t tslot = __builtin_amdgcn_readlane(k.slot[e], NBX_WAVE - 1);
        auto put = [&](int32_t v, int32_t x) {
            const int32_t below = lane_below(v);
            return lane == p ? x : (stay ? v : below);
        };
        k.d[e].w[0] = put(k.d[e].w[0], n.w[0]);
        k.d[e].w[1] = put(k.d[e].w[1], n.w[1]);
        k.slot[e] = put(k.slot[e], slot);
        n = top;
        slot = tslot;
    }
}

// ------------------------------------------------- merging by short keys
// A key is a distance rounded to FP32 (monotone) with its lowest bits
// replaced by where the entry is: two keys that differ above those bits are in
// the exact order, equal ones are found afterwards and settled exactly.
template <int E>
struct WvKey {
    static constexpr uint32_t TAGS = E == 1 ? 128 : 256, NONE = ~(TAGS - 1);
    static __device__ __forceinline__ uint32_t of(double d, bool some, uint32_t tag) {
        const uint32_t u = (__float_as_uint((float)d) << 1) & NONE;
        return (some ? u : NONE) | tag;
    }
};
// the smaller of each pair of lanes that differ in bit J to the lane with the
// bit clear; o: the partner's key
template <int J>
__device__ __forceinline__ uint32_t key_pick(uint32_t v, uint32_t o, int lane) {
    const uint32_t lo = min(v, o), hi = max(v, o);
    return (lane & J) ? hi : lo;
}
template <int J>
__device__ __forceinline__ uint32_t key_stage(uint32_t v, int lane) {
    if constexpr (J == 32 || J == 16) {
        const auto r = J == 32 ? __builtin_amdgcn_permlane32_swap(v, v, false, false)
                               : __builtin_amdgcn_permlane16_swap(v, v, false, false);
        return key_pick<J>(r[0], r[1], lane);
    } else if constexpr (J == 8) {
        return key_pick<8>(v, dpp<0x128>(v), lane);  // row_ror:8
    } else if constexpr (J == 4) {
        return key_pick<4>(v, dpp<0x1B>(dpp<0x141>(v)), lane);  // the half row reversed, then each four
    } else if constexpr (J == 2) {
        return key_pick<2>(v, dpp<0x4E>(v), lane);
    } else {
        return key_pick<1>(v, dpp<0xB1>(v), lane);
    }
}
// a bitonic sequence of 2 J keys into ascending order
template <int J>
__device__ __forceinline__ uint32_t key_merge(uint32_t v, int lane) {
    v = key_stage<J>(v, lane);
    if constexpr (J > 1) v = key_merge<J / 2>(v, lane);
    return v;
}
// the wave's keys in reverse
__device__ __forceinline__ uint32_t key_reverse(uint32_t v, int lane) {
    return (uint32_t)__builtin_amdgcn_ds_bpermute((lane ^ 63) << 2, (int)v);
}
__device__ __forceinline__ uint32_t key_sort_row(uint32_t v, int lane) {
    v = key_stage<1>(v, lane);
    v = key_merge<1>(key_pick<2>(v, dpp<0x1B>(v), lane), lane);   // a four reversed
    v = key_merge<2>(key_pick<4>(v, dpp<0x141>(v), lane), lane);  // half a row
    return key_merge<4>(key_pick<8>(v, dpp<0x140>(v), lane), lane);  // a row
}
__device__ __forceinline__ uint32_t key_sort_half(uint32_t v, int lane) {
    v = key_sort_row(v, lane);
    return key_merge<8>(key_pick<16>(v, (uint32_t)__builtin_amdgcn_ds_swizzle((int)v, 0x7c1f), lane), lane);  // lane ^ 31
}
__device__ __forceinline__ uint32_t key_sort(uint32_t v, int lane) {
    v = key_sort_half(v, lane);
    return key_merge<16>(key_pick<32>(v, key_reverse(v, lane), lane), lane);
}

// One exact compare-exchange stage between lanes that differ in bit j: the
// smaller entry to the lane with that bit clear (up) or set (!up).
template <class D>
__device__ __forceinline__ void wv_exchange(D &d, int32_t &id, int32_t &slot, int j, bool up, int lane) {
    const double od = __shfl_xor(d.d, j);
    const int32_t oi = __shfl_xor(id, j), os = __shfl_xor(slot, j);
    const bool low = (lane & j) == 0;
    const bool less = before(od, oi, d.d, id), more = before(d.d, id, od, oi);
    const bool take = low == up ? less : more;
    d.d = take ? od : d.d;
    id = take ? oi : id;
    slot = take ? os : slot;
}

// Merge 64 entries, one per lane in any order, into the kept ones, exactly:
// for entries whose keys do not tell them apart.
template <int E>
__device__ __forceinline__ void wv_merge_exact(const DevTree &T, WvKept<E> &k, double nd, int32_t slot, int lane) {
    typename WvKept<E>::Dbl d;
    d.d = nd;
    int32_t id = wv_id(T, slot);
#pragma unroll 1
    for (int n = 2; n <= NBX_WAVE; n <<= 1)
#pragma unroll 1
        for (int j = n >> 1; j > 0; j >>= 1) wv_exchange(d, id, slot, j, (lane & n) != 0, lane);
    // descending now; from the last block down, the 64 smaller of a block and
    // these go on, the larger stay in the block above
#pragma unroll
    for (int e = E - 1; e >= 0; --e) {
        const int32_t ki = wv_id(T, k.slot[e]);
        const bool take = before(d.d, id, k.d[e].d, ki);
        typename WvKept<E>::Dbl hd = take ? k.d[e] : d;
        int32_t hi = take ? ki : id, hs = take ? k.slot[e] : slot;
        d = take ? d : k.d[e];
        id = take ? id : ki;
        slot = take ? slot : k.slot[e];
#pragma unroll 1
        for (int j = 32; j > 0; j >>= 1) {
            if (e + 1 < E) wv_exchange(hd, hi, hs, j, true, lane);
            wv_exchange(d, id, slot, j, e == 0, lane);
        }
        if (e + 1 < E) {
            k.d[e + 1 < E ? e + 1 : 0] = hd;
            k.slot[e + 1 < E ? e + 1 : 0] = hs;
        }
    }
    k.d[0] = d;
    k.slot[0] = slot;
}

// Merge cnt entries, staged from sh.d[0] on in any order, into the kept ones.
template <int E>
__device__ __forceinline__ void wv_merge(const DevTree &T, WvKept<E> &k, int cnt, int kh, WvShared<E> &sh, int lane) {
    typedef WvKey<E> Key;
    __syncthreads();
    const bool in = lane < cnt;
    const bool empty = !(lane_d(k.d[0].d, 0) < NBX_MAXVALUE);
    uint32_t v = Key::of(in ? sh.d[lane] : 0.0, in, (uint32_t)lane), x[E], out = ~0u;
    v = cnt <= 16 ? key_sort_row(v, lane) : cnt <= 32 ? key_sort_half(v, lane) : key_sort(v, lane);
#pragma unroll
    for (int e = E - 1; e >= 0; --e) {
        const uint32_t kk = Key::of(k.d[e].d, k.d[e].d < NBX_MAXVALUE, (uint32_t)(NBX_WAVE * (e + 1) + lane));
        if (e == 0 && E == 1 && empty) break;
        const uint32_t r = key_reverse(v, lane), hi = max(kk, r);
        v = key_merge<32>(min(kk, r), lane);
        if (e + 1 < E) x[e + 1 < E ? e + 1 : 0] = key_merge<32>(hi, lane);
        else out = hi;
    }
    x[0] = v;
    // neighbours in the order that only their tags tell apart
    uint64_t tie = 0;
#pragma unroll
    for (int e = 0; e < E; ++e) {
        const uint32_t prev = e ? (uint32_t)__builtin_amdgcn_readlane((int)x[e ? e - 1 : 0], 63) : ~x[0];
        const uint32_t b = (uint32_t)lane_below((int32_t)x[e]), a = lane ? b : prev;
        tie |= ballot(((x[e] ^ a) < Key::TAGS) & (x[e] < Key::NONE));
    }
    if (kh == E * NBX_WAVE) {  // the last kept and the first left out
        const uint32_t a = (uint32_t)__builtin_amdgcn_readlane((int)x[E - 1], 63), b = wave_umin(out);
        tie |= (uint64_t)((a ^ b) < Key::TAGS && a < Key::NONE);
    }
    if (!in) {
        sh.d[lane] = NBX_MAXVALUE;
        sh.slot[lane] = -1;
    }
    if (tie) {
        wv_merge_exact(T, k, sh.d[lane], sh.slot[lane], lane);
        __syncthreads();
        return;
    }
#pragma unroll
    for (int e = 0; e < E; ++e) {
        sh.d[NBX_WAVE * (e + 1) + lane] = k.d[e].d;
        sh.slot[NBX_WAVE * (e + 1) + lane] = k.slot[e];
    }
    __syncthreads();
#pragma unroll
    for (int e = 0; e < E; ++e) {
        const uint32_t t = x[e] & (Key::TAGS - 1);
        k.d[e].d = sh.d[t];
        k.slot[e] = sh.slot[t];
    }
    __syncthreads();
}
#define WV_MERGE 4  // accepted entries from which on a merge takes fewer instructions than insertions

// Before anything is kept more particles are accepted than a merge takes at
// once.  A distance that at least kh and at most a wave of them lie within,
// found by bisection, leaves the rest out: they are not among the kh nearest.
// A few compares instead of a second merge: 2.1M particles, density, k = 32
// 3.86 -> 3.73 ms; 4096 particles 19 -> 17 us.
#define WV_CUT 56  // kh up to which it is tried: a narrow target takes too many steps
__device__ __forceinline__ void wv_cut(const double (&d2)[2], uint64_t (&acc)[2], int kh, int lane) {
    float top = (acc[0] >> lane) & 1ULL ? (float)d2[0] : 0.0f;
    top = fmaxf(top, (acc[1] >> lane) & 1ULL ? (float)d2[1] : 0.0f);
    float lo = 0.0f, hi = __uint_as_float(~wave_umin(~__float_as_uint(top)));
    for (int i = 0; i < 10; ++i) {
        const float m = 0.5f * (lo + hi);
        const uint64_t a = acc[0] & ballot(d2[0] <= (double)m), b = acc[1] & ballot(d2[1] <= (double)m);
        const int c = __builtin_popcountll(a) + __builtin_popcountll(b);
        if (c < kh) lo = m;
        else if (c > NBX_WAVE) hi = m;
        else {
            acc[0] = a;
            acc[1] = b;
            return;
        }
    }
}

// The walk for one position q.  A node's key is its bound rounded to FP32
// with the lane in the lowest bits: its least is the nearest node, and a node
// whose key is above lim cannot hold a neighbour.
template <int ND, int E>
__device__ __forceinline__ void wv_walk(const DevTree &T, const double (&q)[ND], WvKept<E> &k, int kh, bool exz,
                                        WvShared<E> &sh, int lane) {
    // levels opened by the first step; every later one opens six
    const int first = T.depth == 0 ? 0 : (T.depth - 1) % 6 + 1;
    int sp = 0, height = T.depth, step = first;
    uint32_t node = 1, base = 0, key = ~0u;
    bool expand = true;
    // nearest of the descendants (its lane), which is then marked taken
    auto take = [&]() -> int {
        const uint32_t m = wave_umin(key);
        if (key == m) key = ~0u;
        return (int)(m & 63u);
    };
    int staged = 0;  // accepted entries in sh that are not kept yet
    auto flush = [&]() {
        if (staged < WV_MERGE) {
            __syncthreads();
            for (int j = 0; j < staged; ++j)
                wv_insert(T, k, readfirst_d(sh.d[j]), __builtin_amdgcn_readfirstlane(sh.slot[j]), lane);
            __syncthreads();
        } else {
            wv_merge(T, k, staged, kh, sh, lane);
        }
        wv_kth(k, kh);
        staged = 0;
    };
    for (;;) {
        if (expand) {
            height -= step;
            base = node << step;
            const bool mine = lane < (1 << step);
            const double2 *bp = (const double2 *)node_box(T, (int)base, ND) + (mine ? lane * ND : 0);
            double bx[2 * ND];
#pragma unroll
            for (int i = 0; i < ND; ++i) {
                const double2 v = bp[i];
                bx[2 * i] = v.x;
                bx[2 * i + 1] = v.y;
            }
            double s = 0.0;
#pragma unroll
            for (int d = 0; d < ND; ++d) {
                const double t = fmax(fmax(bx[d] - q[d], q[d] - bx[ND + d]), 0.0);
                s = fma(t, t, s);
            }
            key = mine ? (__float_as_uint((float)s) & ~63u) | (uint32_t)lane : ~0u;
            expand = false;
        }
        if (height == 0) {
            // the four nearest open leaves, two particles per lane
            uint64_t open = ballot(key <= k.lim);
            if (open) {
                int li = 0;
                uint64_t has = ~0ULL;  // the lanes with a leaf, 16 for each
                const int nopen = __builtin_popcountll(open);
                if (nopen <= 4) {  // all of them, in any order
                    if (key <= k.lim) key = ~0u;
                    has >>= 64 - 16 * nopen;
#pragma unroll
                    for (int j = 0; j < 4; ++j) {
                        if (!open) break;
                        li = lane >> 4 == j ? __builtin_ctzll(open) : li;
                        open &= open - 1;
                    }
                } else {
#pragma unroll
                    for (int j = 0; j < 4; ++j) {
                        const int i = take();
                        li = lane >> 4 == j ? i : li;
                    }
                }
                const int32_t s0 = ((int)base - T.nleafp) * NBX_LEAF;  // the first of the 64 leaves
                const uint32_t ls = (uint32_t)(li * NBX_LEAF + 2 * (lane & 15));
                const int32_t sl = s0 + (int32_t)ls;
                double d2[2] = {0.0, 0.0};
#pragma unroll
                for (int d = 0; d < ND; ++d) {
                    const double2 x = *(const double2 *)((const char *)(T.x[d] + s0) + ls * 8u);
                    const double t0 = q[d] - x.x, t1 = q[d] - x.y;
                    d2[0] += t0 * t0;
                    d2[1] += t1 * t1;
                }
                // (padding slots lie at 1e300, so their d2 is infinite)
                uint64_t acc[2] = {ballot(d2[0] <= k.kth) & has, ballot(d2[1] <= k.kth) & has};
                if (!(acc[0] | acc[1])) continue;
                // equally far as the last kept: only a smaller ID counts; the
                // query itself has d2 == 0
                const uint64_t tie[2] = {acc[0] & ballot(d2[0] == k.kth), acc[1] & ballot(d2[1] == k.kth)};
                if (tie[0] | tie[1]) {
                    const int2 ids = *(const int2 *)((const char *)(T.perm + s0) + ls * 4u);
                    const int32_t kid = wv_id(T, k.kslot);
                    acc[0] &= ~tie[0] | ballot(ids.x < kid);
                    acc[1] &= ~tie[1] | ballot(ids.y < kid);
                }
                if (exz) {
                    acc[0] &= ballot(d2[0] > 0.0);
                    acc[1] &= ballot(d2[1] > 0.0);
                }
                if (!(k.kth < NBX_MAXVALUE) && kh <= WV_CUT &&
                    __builtin_popcountll(acc[0]) + __builtin_popcountll(acc[1]) > NBX_WAVE)
                    wv_cut(d2, acc, kh, lane);
#pragma unroll
                for (int p = 0; p < 2; ++p) {
                    const int cnt = __builtin_popcountll(acc[p]);
                    if (cnt == 0) continue;
                    if (staged + cnt > NBX_WAVE) flush();
                    if ((acc[p] >> lane) & 1ULL) {
                        const int at = staged + __builtin_amdgcn_mbcnt_hi((uint32_t)(acc[p] >> 32),
                                                                          __builtin_amdgcn_mbcnt_lo((uint32_t)acc[p], 0));
                        sh.d[at] = d2[p];
                        sh.slot[at] = sl + p;
                    }
                    staged += cnt;
                }
                if (staged) flush();
                continue;
            }
        } else {
            const uint64_t open = ballot(key <= k.lim);
            if (open) {
                int i = __builtin_ctzll(open);
                if (open & (open - 1)) i = take();
                else if (lane == i) key = ~0u;
                sh.stk[sp][lane] = key;
                ++sp;
                node = base + (uint32_t)i;
                step = 6;
                expand = true;
                continue;
            }
        }
        if (sp == 0) break;
        --sp;  // back to the level above: base's ancestor six levels up is among its nodes
        key = sh.stk[sp][lane];
        const int opened = sp == 0 ? first : 6;
        base = (base >> 6 >> opened) << opened;
        height += 6;
    }
}

template <int ND, int E, int QSRC>
__global__ __launch_bounds__(64) void k_knn_wave(DevTree T, KnnArgs A, int first) {
    __shared__ WvShared<E> sh;
    const int lane = threadIdx.x;
    const int g = first + xcd_wave(blockIdx.x, gridDim.x);
    const int kh = A.kh;
    const bool listed = A.qlist != nullptr;
    const int qi = listed ? A.qlist[g] : A.wbeg * NBX_WAVE + g;
    double q0[ND], q[ND];
#pragma unroll
    for (int d = 0; d < ND; ++d)
        q0[d] = QSRC == NBX_Q_POINTS ? (d < 3 ? A.q[d][qi] : A.qv[d - 3][qi]) : T.x[d][qi];
    const bool exz = QSRC == NBX_Q_SLOTS && A.excl_zero;
    WvKept<E> k;
#pragma unroll
    for (int e = 0; e < E; ++e) {
        k.d[e].d = NBX_MAXVALUE;
        k.slot[e] = -1;
    }
    k.kth = NBX_MAXVALUE;
    k.kslot = -1;
    k.lim = wv_lim(k.kth);
#pragma unroll
    for (int d = 0; d < ND; ++d) q[d] = q0[d];
    wv_walk<ND, E>(T, q, k, kh, exz, sh, lane);
    if (QSRC != NBX_Q_SLOTS && A.periodic) {
        // image p in lane p: all are tested at once, and again as kth shrinks
        double xp[3];
        uint64_t todo = 0xfeULL;
        for (;;) {
            todo &= ballot(image_pass(lane, q0, A.period, k.kth, ND == 6, xp));
            if (!todo) break;
            const int p = __builtin_ctzll(todo);
            todo &= todo - 1;
#pragma unroll
            for (int d = 0; d < 3; ++d) q[d] = lane_d(xp[d], p);
            wv_walk<ND, E>(T, q, k, kh, exz, sh, lane);
        }
    }
    const double kth = k.kth;
    const bool bad = !(kth < NBX_MAXVALUE);  // fewer than kh neighbours

    // ------------------------------------------------------------ densities
    // (position queries take the gather forms only)
    if (A.dens != NBX_DO_NONE &&
        (QSRC == NBX_Q_SLOTS || A.dens == NBX_DO_GATHER || (QSRC == NBX_Q_POINTS && A.dens == NBX_DO_VEL))) {
        double hi;
        if (A.dens == NBX_DO_VEL || A.dens == NBX_DO_VELPHYS) {
            // |dv| of the Nsearch neighbours, the Nsmooth smallest by (|dv|,
            // ID), h_v = max / 2, sum W(|dv| / h_v) h_v^-3 in that order (see
            // nbx_knn.hip)
            const int ns = A.nsmooth;
            const bool pts = QSRC == NBX_Q_POINTS, phys = A.dens == NBX_DO_VELPHYS;
            const double qvx = pts ? A.qv[0][qi] : T.x[3][qi], qvy = pts ? A.qv[1][qi] : T.x[4][qi],
                         qvz = pts ? A.qv[2][qi] : T.x[5][qi];
            __shared__ double sv[E * NBX_WAVE];
            __shared__ int32_t di[E * NBX_WAVE];
            double *dv = sh.d;
            int32_t *ss = sh.slot;
            if (!bad) {
                double v[E];
                int32_t vi[E];
#pragma unroll
                for (int e = 0; e < E; ++e) {
                    const int p = e * NBX_WAVE + lane;
                    const int32_t s = p < kh ? k.slot[e] : 0;
                    const double vx = qvx - T.x[3][s], vy = qvy - T.x[4][s], vz = qvz - T.x[5][s];
                    v[e] = sqrt(vx * vx + vy * vy + vz * vz);
                    dv[p] = v[e];
                    vi[e] = T.perm[s];
                    di[p] = vi[e];
                    sv[p] = v[e];  // (ranks of unordered values, NaN, may leave places unwritten)
                    ss[p] = s;
                }
                __syncthreads();
#pragma unroll
                for (int e = 0; e < E; ++e) {
                    const int p = e * NBX_WAVE + lane;
                    if (p >= kh) continue;
                    int r = 0;
                    for (int j = 0; j < kh; ++j)
                        r += before(dv[j], di[j], v[e], vi[e]) || (dv[j] == v[e] && di[j] == vi[e] && j < p) ? 1 : 0;
                    sv[r] = v[e];
                    ss[r] = k.slot[e];
                }
                __syncthreads();
                hi = 0.5 * sv[ns - 1];
                const double norm = 1.0 / wv_pow<3>(hi), hp = 0.5 * kth, pnorm = phys ? 1.0 / wv_pow<3>(hp) : 0.0;
                const double rhoi = phys ? A.rho_in[qi] : 1.0, mi = phys ? T.mass[qi] : 0.0;
                for (int p = lane; p < ns; p += NBX_WAVE) {
                    double t = wsm_at(sv[p], hi, T.kern, T.kernres) * norm;
                    if (phys) {
                        const int32_t s = ss[p];
                        const double dx = T.x[0][qi] - T.x[0][s], dy = T.x[1][qi] - T.x[1][s],
                                     dz = T.x[2][qi] - T.x[2][s];
                        const double W = wsm_at(sqrt(dx * dx + dy * dy + dz * dz), hp, T.kern, T.kernres) * pnorm;
                        t = t * (W / rhoi * mi);
                    }
                    dv[p] = t;
                }
                __syncthreads();
                double den = 0.0;
                for (int p = 0; p < ns; ++p) den = den + dv[p];
                if (lane == 0) {
                    A.rho[qi] = den;
                    if (A.hout) A.hout[A.hout_by_id ? T.perm[qi] : qi] = hi;
                }
            }
        } else {
            const bool spline = ND == 3 && QSRC == NBX_Q_SLOTS && A.dens == NBX_DO_SPLINE;
            const bool sym = QSRC == NBX_Q_SLOTS && (A.dens == NBX_DO_SYM || spline);
            hi = 0.5 * sqrt(kth);
            const double ih = 1.0 / hi;
            const double norm = spline ? NBX_SIGMA3 * ih * ih * ih : 1.0 / wv_pow<ND>(hi);
            const double mi = QSRC == NBX_Q_SLOTS ? T.mass[qi] : 0.0;
            double acc = 0.0;
#pragma unroll
            for (int e = 0; e < E; ++e) {
                if (e * NBX_WAVE + lane < kh && k.d[e].d < NBX_MAXVALUE) {
                    const int32_t s = k.slot[e];
                    const double r = sqrt(k.d[e].d);
                    const double W = spline ? w_cubic(r * ih) : wsm_at(r, hi, T.kern, T.kernres);
                    const double Wij = sym ? 0.5 * W * norm : W * norm;
                    acc += Wij * T.mass[s];
                    if (sym) unsafeAtomicAdd(A.rho + s, Wij * mi);
                }
            }
            acc = wave_sum(acc);
            if (lane == NBX_WAVE - 1) {
                if (sym) unsafeAtomicAdd(A.rho + qi, acc);
                else A.rho[qi] = acc;
                if (A.hout) A.hout[A.hout_by_id ? T.perm[qi] : qi] = hi;
            }
        }
        if (bad && lane == 0) atomicOr(A.err, 1);
    }

    // ------------------------------------------------------------ outputs
    if (A.nn == nullptr && A.d2 == nullptr) return;
    int64_t row;
    if (QSRC == NBX_Q_POINTS) row = qi;
    else if (listed && A.list_rows) row = g;
    else if (A.layout == 1) row = qi - A.row0;
    else row = T.perm[qi];
    if (A.miss_self && bad && lane == 0) atomicOr(A.err, 1);
    const bool ids = QSRC == NBX_Q_POINTS || A.layout == 0;
    const int off = (A.drop == NBX_DROP_SMALLEST) ? 1 : 0;
#pragma unroll
    for (int e = 0; e < E; ++e) {
        const int t = e * NBX_WAVE + lane - off;
        if (t < 0 || t >= A.kout) continue;
        const bool miss = !(k.d[e].d < NBX_MAXVALUE);
        const bool self = miss && A.miss_self;  // (a missing entry that names the query)
        if (A.nn) A.nn[row * A.kout + t] = self ? (ids ? T.perm[qi] : qi) : miss ? -1 : (ids ? T.perm[k.slot[e]] : k.slot[e]);
        if (A.d2) A.d2[row * A.kout + t] = self ? 0.5 * NBX_MAXVALUE : k.d[e].d;
    }
}

// A launch holds fewer than 2^32 threads, hence the runs of queries.
#define WV_RUN (1 << 25)
template <int ND, int E>
static void wave_start(const DevTree &T, const KnnArgs &A, int nq, hipStream_t st) {
    for (int64_t q0 = 0; q0 < nq; q0 += WV_RUN) {
        const dim3 grid((unsigned)std::min<int64_t>(WV_RUN, nq - q0));
        if (A.qsrc == NBX_Q_SLOTS)
            hipLaunchKernelGGL((k_knn_wave<ND, E, NBX_Q_SLOTS>), grid, dim3(NBX_WAVE), 0, st, T, A, (int)q0);
        else if (A.qsrc == NBX_Q_PERIODIC)
            hipLaunchKernelGGL((k_knn_wave<ND, E, NBX_Q_PERIODIC>), grid, dim3(NBX_WAVE), 0, st, T, A, (int)q0);
        else
            hipLaunchKernelGGL((k_knn_wave<ND, E, NBX_Q_POINTS>), grid, dim3(NBX_WAVE), 0, st, T, A, (int)q0);
    }
}

hipError_t nbx_launch_knn_wave(const DevTree &T, const KnnArgs &A, int nqueries, hipStream_t st) {
    // particle queries by runs of whole waves: the last wave may be partial
    int nq = nqueries;
    if (A.qsrc != NBX_Q_POINTS && !A.qlist) nq = std::min<int64_t>(nq, (int64_t)T.n - (int64_t)A.wbeg * NBX_WAVE);
    if (nq <= 0) return hipSuccess;
    ProfScope ps(A.qsrc != NBX_Q_POINTS && A.qlist ? "k_knn_fallback" : "k_knn_fp64", st);
    if (T.nd == 6) {
        if (A.kh <= 64) wave_start<6, 1>(T, A, nq, st);
        else if (A.kh <= 128) wave_start<6, 2>(T, A, nq, st);
        else wave_start<6, 3>(T, A, nq, st);
    } else {
        if (A.kh <= 64) wave_start<3, 1>(T, A, nq, st);
        else if (A.kh <= 128) wave_start<3, 2>(T, A, nq, st);
        else wave_start<3, 3>(T, A, nq, st);
    }
    return hipGetLastError();
}
