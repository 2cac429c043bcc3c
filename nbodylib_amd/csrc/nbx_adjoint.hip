// nbx_adjoint.hip -- differentiation form: SPH density over a frozen
// neighbour list and its hand-written adjoint.
//
// No reference counterpart: NBodylib allocates derKernel but never fills it
// (KDTree.cxx:1150, :1345).  The forward is CalcDensity's symmetric formula
// (KDCalcSmoothQuantities.cxx:260-286) with the table replaced by the
// analytic cubic spline WSPH (SmoothingKernels.h:32-37), 3-D norm 1/pi
// (KDTree.cxx:1158-1164), so the derivative is continuous:
//   w_ij = (sigma/2) W(r_ij/h_i) h_i^-3,  rho_i += w_ij m_j,  rho_j += w_ij m_i,
//   h_i  = |x_i - x_K(i)| / 2  (K(i) = last column of the list).
// Adjoint, with a_ij = g_i m_j + g_j m_i and q = r/h:
//   dL/dm_j += w_ij g_i,  dL/dm_i += w_ij g_j,
//   dL/dx_i += a_ij (sigma/2) W'(q) h^-4 (x_i-x_j)/r   (and minus on x_j),
//   dL/dh_i  = sum_j a_ij (-(sigma/2) h^-4 (q W'(q) + 3 W(q))),
//   dL/dx_i += dL/dh_i (x_i-x_K)/(2 r_iK)               (and minus on x_K).
// One thread per particle i; contributions to other particles use FP64
// atomics (LDS ones for particles of the same block).
#include "nbx_kernels.h"

// Contributions to particles of the same 1024-particle block (most of them
// when the arrays are in tree order) are summed in LDS and flushed with one
// atomic per particle and component; the rest go straight to HBM.
#define ADJ_B 1024
#define ADJ_G 8   // neighbours whose gathers are issued together (forward)
#define ADJ_GB 4  // (adjoint: more live values per neighbour)

__global__ __launch_bounds__(ADJ_B) void k_sph_fwd(const double *__restrict__ X, const double *__restrict__ Y,
                                                   const double *__restrict__ Z, const double *__restrict__ mass,
                                                   const int32_t *__restrict__ nbr, int64_t n,
                                                   int k, double *rho, double *hout) {
    __shared__ double lrho[ADJ_B];
    const int t = threadIdx.x;
    const int64_t i0 = (int64_t)blockIdx.x * ADJ_B;
    const int64_t i = i0 + t;
    lrho[t] = 0.0;
    __syncthreads();
    double acc = 0.0;
    if (i < n) {
        const double xi = X[i], yi = Y[i], zi = Z[i], mi = mass[i];
        const int32_t *row = nbr + i * k;
        const int64_t K = row[k - 1];
        const double dx = xi - X[K], dy = yi - Y[K], dz = zi - Z[K];
        const double h = 0.5 * sqrt(dx * dx + dy * dy + dz * dz);
        if (hout) hout[i] = h;
        const double ih = 1.0 / h;
        const double norm = 0.5 * NBX_SIGMA3 * ih * ih * ih;
        for (int j0 = 0; j0 < k; j0 += ADJ_G) {
            int64_t qv[ADJ_G];
            double rv[ADJ_G], mv[ADJ_G];
#pragma unroll
            for (int u = 0; u < ADJ_G; ++u) {
                qv[u] = j0 + u < k ? row[j0 + u] : i;
                const double ex = xi - X[qv[u]], ey = yi - Y[qv[u]], ez = zi - Z[qv[u]];
                rv[u] = sqrt(ex * ex + ey * ey + ez * ez);
                mv[u] = mass[qv[u]];
            }
#pragma unroll
            for (int u = 0; u < ADJ_G; ++u) {
                if (j0 + u >= k) break;
                const double w = norm * w_cubic(rv[u] * ih);
                acc += w * mv[u];
                const uint64_t r = (uint64_t)(qv[u] - i0);
                if (r < ADJ_B) atomicAdd(&lrho[r], w * mi);
                else unsafeAtomicAdd(rho + qv[u], w * mi);
            }
        }
    }
    __syncthreads();
    if (i < n) unsafeAtomicAdd(rho + i, acc + lrho[t]);
}

__global__ __launch_bounds__(ADJ_B) void k_sph_adj(const double *__restrict__ X, const double *__restrict__ Y,
                                                   const double *__restrict__ Z, const double *__restrict__ mass,
                                                   const int32_t *__restrict__ nbr, int64_t n,
                                                   int k, const double *__restrict__ g, double *DX, double *DY,
                                                   double *DZ, double *dmass) {
    __shared__ double lx[ADJ_B], ly[ADJ_B], lz[ADJ_B], lm[ADJ_B];
    const int t = threadIdx.x;
    const int64_t i0 = (int64_t)blockIdx.x * ADJ_B;
    const int64_t i = i0 + t;
    lx[t] = 0.0;
    ly[t] = 0.0;
    lz[t] = 0.0;
    lm[t] = 0.0;
    __syncthreads();
    double gx = 0.0, gy = 0.0, gz = 0.0, gm = 0.0;
    if (i < n) {
        const double xi = X[i], yi = Y[i], zi = Z[i], mi = mass[i], gi = g[i];
        const int32_t *row = nbr + i * k;
        const int64_t K = row[k - 1];
        const double kx = xi - X[K], ky = yi - Y[K], kz = zi - Z[K];
        const double rk = sqrt(kx * kx + ky * ky + kz * kz);
        const double h = 0.5 * rk;
        const double ih = 1.0 / h;
        const double ih3 = ih * ih * ih, ih4 = ih3 * ih;
        double Hs = 0.0;
        for (int j0 = 0; j0 < k; j0 += ADJ_GB) {
            int64_t qv[ADJ_GB];
            double exv[ADJ_GB], eyv[ADJ_GB], ezv[ADJ_GB], mv[ADJ_GB], gv[ADJ_GB];
#pragma unroll
            for (int u = 0; u < ADJ_GB; ++u) {
                qv[u] = j0 + u < k ? row[j0 + u] : i;
                exv[u] = xi - X[qv[u]];
                eyv[u] = yi - Y[qv[u]];
                ezv[u] = zi - Z[qv[u]];
                mv[u] = mass[qv[u]];
                gv[u] = g[qv[u]];
            }
#pragma unroll
            for (int u = 0; u < ADJ_GB; ++u) {
                if (j0 + u >= k) break;
                const int64_t q = qv[u];
                const double ex = exv[u], ey = eyv[u], ez = ezv[u];
                const double r = sqrt(ex * ex + ey * ey + ez * ez);
                const double qq = r * ih;
                const double W = w_cubic(qq), dW = dw_cubic(qq);
                const double w = 0.5 * NBX_SIGMA3 * W * ih3;
                const double a = gi * mv[u] + gv[u] * mi;
                const uint64_t lr = (uint64_t)(q - i0);
                const bool loc = lr < ADJ_B;
                if (loc) atomicAdd(&lm[lr], w * gi);
                else unsafeAtomicAdd(dmass + q, w * gi);
                gm += w * gv[u];
                Hs += a * (-0.5 * NBX_SIGMA3 * (qq * dW + 3.0 * W) * ih4);
                if (r > 0.0) {
                    const double f = a * 0.5 * NBX_SIGMA3 * dW * ih4 / r;
                    gx += f * ex;
                    gy += f * ey;
                    gz += f * ez;
                    if (loc) {
                        atomicAdd(&lx[lr], -f * ex);
                        atomicAdd(&ly[lr], -f * ey);
                        atomicAdd(&lz[lr], -f * ez);
                    } else {
                        unsafeAtomicAdd(DX + q, -f * ex);
                        unsafeAtomicAdd(DY + q, -f * ey);
                        unsafeAtomicAdd(DZ + q, -f * ez);
                    }
                }
            }
        }
        if (rk > 0.0) {
            const double f = Hs * 0.5 / rk;
            gx += f * kx;
            gy += f * ky;
            gz += f * kz;
            const uint64_t lr = (uint64_t)(K - i0);
            if (lr < ADJ_B) {
                atomicAdd(&lx[lr], -f * kx);
                atomicAdd(&ly[lr], -f * ky);
                atomicAdd(&lz[lr], -f * kz);
            } else {
                unsafeAtomicAdd(DX + K, -f * kx);
                unsafeAtomicAdd(DY + K, -f * ky);
                unsafeAtomicAdd(DZ + K, -f * kz);
            }
        }
    }
    __syncthreads();
    if (i < n) {
        unsafeAtomicAdd(DX + i, gx + lx[t]);
        unsafeAtomicAdd(DY + i, gy + ly[t]);
        unsafeAtomicAdd(DZ + i, gz + lz[t]);
        unsafeAtomicAdd(dmass + i, gm + lm[t]);
    }
}

hipError_t nbx_launch_sph_fwd(const double *pos, const double *mass, const int32_t *nbr, int64_t n, int k, double *rho,
                              double *h, hipStream_t st) {
    ProfScope ps("k_sph_fwd", st);
    hipLaunchKernelGGL(k_sph_fwd, dim3((unsigned)((n + ADJ_B - 1) / ADJ_B)), dim3(ADJ_B), 0, st, pos, pos + n,
                       pos + 2 * n, mass, nbr, n, k, rho, h);
    return hipGetLastError();
}

hipError_t nbx_launch_sph_adj(const double *pos, const double *mass, const int32_t *nbr, int64_t n, int k,
                              const double *g, double *dpos, double *dmass, hipStream_t st) {
    ProfScope ps("k_sph_adj", st);
    hipLaunchKernelGGL(k_sph_adj, dim3((unsigned)((n + ADJ_B - 1) / ADJ_B)), dim3(ADJ_B), 0, st, pos, pos + n,
                       pos + 2 * n, mass, nbr, n, k, g, dpos, dpos + n, dpos + 2 * n, dmass);
    return hipGetLastError();
}

// ------------------------------------------------------------------ packed records, rows in an order
// The kernels above work on the caller's arrays alone: five 8-byte gathers per
// neighbour from five arrays, and a device-scope atomic per component for each
// neighbour outside the block.  With room for records (32 bytes of position
// and mass per particle) a neighbour is one gather, and the adjoint's four
// sums of a particle lie together, so a contribution leaves as one 32-byte
// transaction (sph_scatter): backward of 1M particles in tree order, k = 32,
// 1.14 -> 0.49 ms.  That is bound by the transactions still, so what counts is
// how many neighbours fall outside a row's block of 1024: 19% in tree order,
// but 78% in a snapshot's own order (background particles at random, halo
// members shuffled).  There the rows are taken in Morton order of the
// positions (30-bit keys, one radix sort, 0.12 ms): forward and backward of
// 1M particles 7.2 -> 2.8 ms with records alone, 1.47 ms in Morton order.

#define SPH_BITS 10  // key bits per dimension: cells of a thousandth of the box, a few rows each in dense cores

struct SphWork {
    uint64_t *bounds;  // 6: smallest and largest coordinate per dimension, as ordered integers
    uint32_t *key, *key2;
    int32_t *idx, *rank;
    double4 *rec;  // x, y, z, mass, by rank
    double *g;     // dL/drho by rank
    double *acc;   // adjoint sums by rank, 4 per particle
    void *sort;
    size_t sort_bytes, fwd, total;  // fwd: what the order and the forward need
    SphWork(void *base, int64_t n) {
        char *at = (char *)base;
        auto carve = [&](size_t b) {
            char *p = at;
            at += (b + 255) & ~(size_t)255;
            return p;
        };
        bounds = (uint64_t *)carve(6 * sizeof(uint64_t));
        rank = (int32_t *)carve(sizeof(int32_t) * n);
        rec = (double4 *)carve(sizeof(double4) * n);
        const size_t end_rec = (size_t)(at - (char *)base);
        g = (double *)carve(sizeof(double) * n);
        acc = (double *)carve(4 * sizeof(double) * n);
        // the sort's arrays are done with before the records are written
        at = (char *)rec;
        key = (uint32_t *)carve(sizeof(uint32_t) * n);
        key2 = (uint32_t *)carve(sizeof(uint32_t) * n);
        idx = (int32_t *)carve(sizeof(int32_t) * n);
        sort_bytes = 0;
        nbx_sort_pairs_u32(nullptr, sort_bytes, key, key2, idx, rank, n, 3 * SPH_BITS, nullptr);
        sort = carve(sort_bytes);
        const size_t end_sort = (size_t)(at - (char *)base);
        const size_t end_acc = (size_t)((char *)(acc + 4 * n) - (char *)base);
        fwd = (end_sort > end_rec ? end_sort : end_rec) + 256;
        total = (end_sort > end_acc ? end_sort : end_acc) + 256;
    }
};
size_t nbx_sph_work_size(int64_t n) { return SphWork(nullptr, n).total; }
size_t nbx_sph_fwd_work_size(int64_t n) { return SphWork(nullptr, n).fwd; }

// Rows and columns are stepped without a division.  The waves of a block meet in LDS and blocks are few: with three atomics per
// wave of 4096 blocks the pass took 582 us on 1M x 32, all of it atomics on
// one line; so it takes 47 us, a read of the list at 2.9 TB/s.
#define SPH_CHECK_BLOCKS 512
__global__ __launch_bounds__(1024) void k_sph_list_check(const int32_t *__restrict__ nbr, int64_t n, int k,
                                                         unsigned long long *stats) {
    __shared__ int blo[16], bhi[16];
    __shared__ unsigned long long bloc[16];
    const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
    int lo = 0x7fffffff, hi = (int)0x80000000;
    unsigned long long loc = 0;
    const int64_t total = n * k, step = (int64_t)gridDim.x * 1024;
    int64_t e = (int64_t)blockIdx.x * 1024 + threadIdx.x;
    int64_t row = e / k;
    int64_t col = e - row * k;
    const int64_t drow = step / k, dcol = step - drow * k;
    for (; e < total; e += step, row += drow, col += dcol) {
        if (col >= k) {
            col -= k;
            row += 1;
        }
        const int j = nbr[e];
        lo = min(lo, j);
        hi = max(hi, j);
        loc += (uint32_t)j / ADJ_B == (uint32_t)row / ADJ_B ? 1u : 0u;
    }
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) {
        lo = min(lo, __shfl_xor(lo, off));
        hi = max(hi, __shfl_xor(hi, off));
        loc += __shfl_xor(loc, off);
    }
    if (lane == 0) {
        blo[wv] = lo;
        bhi[wv] = hi;
        bloc[wv] = loc;
    }
    __syncthreads();
    if (threadIdx.x == 0) {
        for (int w = 1; w < 16; ++w) {
            lo = min(lo, blo[w]);
            hi = max(hi, bhi[w]);
            loc += bloc[w];
        }
        atomicMin((long long *)stats, (long long)lo);
        atomicMax((long long *)stats + 1, (long long)hi);
        atomicAdd(stats + 2, loc);
    }
}
__global__ void k_sph_stats_init(long long *s) {
    if (threadIdx.x == 0) {
        s[0] = 0x7fffffffffffffffLL;
        s[1] = -0x7fffffffffffffffLL;
        s[2] = 0;
    }
}
hipError_t nbx_launch_sph_list_check(const int32_t *nbr, int64_t n, int k, int64_t *stats, hipStream_t st) {
    const int64_t blocks = (n * k + 1023) / 1024;
    hipLaunchKernelGGL(k_sph_stats_init, dim3(1), dim3(64), 0, st, (long long *)stats);
    hipLaunchKernelGGL(k_sph_list_check, dim3((unsigned)(blocks < SPH_CHECK_BLOCKS ? blocks : SPH_CHECK_BLOCKS)),
                       dim3(1024), 0, st, nbr, n, k, (unsigned long long *)stats);
    return hipGetLastError();
}

// doubles as integers in the same order
__device__ __forceinline__ uint64_t d_ordered(double v) {
    const uint64_t b = (uint64_t)__double_as_longlong(v);
    return b >> 63 ? ~b : b | 0x8000000000000000ULL;
}
__device__ __forceinline__ double d_from_ordered(uint64_t b) {
    return __longlong_as_double((long long)(b >> 63 ? b & 0x7fffffffffffffffULL : ~b));
}
__global__ void k_sph_bounds_init(unsigned long long *b) {
    if (threadIdx.x < 6) b[threadIdx.x] = threadIdx.x < 3 ? ~0ULL : 0ULL;
}
__global__ __launch_bounds__(1024) void k_sph_bounds(const double *__restrict__ pos, int64_t n,
                                                     unsigned long long *b) {
    __shared__ unsigned long long part[6][16];
    const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
#pragma unroll
    for (int d = 0; d < 3; ++d) {
        unsigned long long lo = ~0ULL, hi = 0;
        for (int64_t i = (int64_t)blockIdx.x * 1024 + threadIdx.x; i < n; i += (int64_t)gridDim.x * 1024) {
            const unsigned long long v = d_ordered(pos[d * n + i]);
            lo = v < lo ? v : lo;
            hi = v > hi ? v : hi;
        }
#pragma unroll
        for (int off = 32; off > 0; off >>= 1) {
            const unsigned long long a = __shfl_xor(lo, off), c = __shfl_xor(hi, off);
            lo = a < lo ? a : lo;
            hi = c > hi ? c : hi;
        }
        if (lane == 0) {
            part[d][wv] = lo;
            part[3 + d][wv] = hi;
        }
    }
    __syncthreads();
    if (threadIdx.x < 6) {
        const int c = threadIdx.x;
        unsigned long long v = part[c][0];
        for (int w = 1; w < 16; ++w) v = c < 3 ? min(v, part[c][w]) : max(v, part[c][w]);
        if (c < 3) atomicMin(b + c, v);
        else atomicMax(b + c, v);
    }
}
__global__ __launch_bounds__(256) void k_sph_keys(const double *__restrict__ pos, int64_t n, const uint64_t *b,
                                                  uint32_t *key, int32_t *idx) {
    const int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x;
    if (i >= n) return;
    const double top = (double)((1 << SPH_BITS) - 1);
    uint32_t v = 0;
#pragma unroll
    for (int d = 0; d < 3; ++d) {
        const double lo = d_from_ordered(b[d]), ext = d_from_ordered(b[3 + d]) - lo;
        const double t = ext > 0.0 ? (pos[d * n + i] - lo) * (top / ext) : 0.0;
        const uint32_t cell = (uint32_t)fmin(fmax(t, 0.0), top);  // NaN: the first cell
#pragma unroll
        for (int bit = 0; bit < SPH_BITS; ++bit) v |= ((cell >> bit) & 1u) << (3 * bit + d);
    }
    key[i] = v;
    idx[i] = (int32_t)i;
}
hipError_t nbx_launch_sph_order(const double *pos, int64_t n, int32_t *order, void *work, hipStream_t st) {
    SphWork W(work, n);
    const int nb = (int)((n + 255) / 256);
    ProfScope ps("k_sph_order", st);
    hipLaunchKernelGGL(k_sph_bounds_init, dim3(1), dim3(64), 0, st, (unsigned long long *)W.bounds);
    hipLaunchKernelGGL(k_sph_bounds, dim3(nb < 256 ? (nb + 3) / 4 : 64), dim3(1024), 0, st, pos, n,
                       (unsigned long long *)W.bounds);
    hipLaunchKernelGGL(k_sph_keys, dim3(nb), dim3(256), 0, st, pos, n, W.bounds, W.key, W.idx);
    hipError_t e = hipGetLastError();
    size_t tb = W.sort_bytes;
    if (e == hipSuccess)
        e = nbx_sort_pairs_u32(W.sort, tb, W.key, W.key2, W.idx, order, n, 3 * SPH_BITS, st);
    return e;
}

// Records by rank, ranks by index, and with g (the adjoint) the cotangents by
// rank and the sums cleared.  No order: rank and index are the same (rank is
// not written).  gidx: where the cotangents of a rank are (null: at its index).
__global__ __launch_bounds__(256) void k_sph_pack(const double *__restrict__ X, const double *__restrict__ Y,
                                                  const double *__restrict__ Z, const double *__restrict__ mass,
                                                  const double *__restrict__ g, const int32_t *__restrict__ gidx,
                                                  const int32_t *__restrict__ order, int64_t n, double4 *rec,
                                                  double *gs, int32_t *rank, double4 *acc) {
    const int64_t s = (int64_t)blockIdx.x * 256 + threadIdx.x;
    if (s >= n) return;
    const int64_t i = order ? order[s] : s;
    rec[s] = make_double4(X[i], Y[i], Z[i], mass[i]);
    if (order) rank[i] = (int32_t)s;
    if (g) {
        gs[s] = g[gidx ? gidx[s] : i];
        acc[s] = make_double4(0.0, 0.0, 0.0, 0.0);
    }
}

// G neighbours of a row from column j0 (their ranks; past the row's end: s).
// V: four columns per load (rows 16-byte aligned).
// ORD: indices go through rank.
template <int G, bool V, bool ORD>
__device__ __forceinline__ void sph_ranks(const int32_t *row, const int32_t *rank, int j0, int k, int32_t s,
                                          int32_t (&r)[G]) {
    if constexpr (V) {
        int4 c[G / 4];
#pragma unroll
        for (int u = 0; u < G / 4; ++u) c[u] = j0 + 4 * u < k ? ((const int4 *)(row + j0))[u] : make_int4(-1, -1, -1, -1);
#pragma unroll
        for (int u = 0; u < G; ++u) {
            const int32_t j = u % 4 == 0 ? c[u / 4].x : u % 4 == 1 ? c[u / 4].y : u % 4 == 2 ? c[u / 4].z : c[u / 4].w;
            r[u] = j < 0 ? s : (ORD ? rank[j] : j);
        }
    } else {
#pragma unroll
        for (int u = 0; u < G; ++u) r[u] = j0 + u >= k ? s : (ORD ? rank[row[j0 + u]] : row[j0 + u]);
    }
}

template <bool V, bool ORD>
__global__ __launch_bounds__(ADJ_B) void k_sph_fwd_ordered(const double4 *__restrict__ rec,
                                                           const int32_t *__restrict__ rank,
                                                           const int32_t *__restrict__ order,
                                                           const int32_t *__restrict__ nbr, int64_t n, int k,
                                                           double *rho, double *hout) {
    __shared__ double lrho[ADJ_B];
    const int t = threadIdx.x;
    const int64_t s0 = (int64_t)xcd_wave(blockIdx.x, gridDim.x) * ADJ_B;
    const int64_t s = s0 + t;
    lrho[t] = 0.0;
    __syncthreads();
    double acc = 0.0;
    int64_t i = 0;
    if (s < n) {
        i = ORD ? order[s] : s;
        const double4 me = rec[s];
        const int32_t *row = nbr + i * k;
        const double4 far = rec[ORD ? rank[row[k - 1]] : row[k - 1]];
        const double dx = me.x - far.x, dy = me.y - far.y, dz = me.z - far.z;
        const double h = 0.5 * sqrt(dx * dx + dy * dy + dz * dz);
        if (hout) hout[i] = h;
        const double ih = 1.0 / h;
        const double norm = 0.5 * NBX_SIGMA3 * ih * ih * ih;
        for (int j0 = 0; j0 < k; j0 += ADJ_G) {
            int32_t r[ADJ_G];
            double rv[ADJ_G], mv[ADJ_G];
            sph_ranks<ADJ_G, V, ORD>(row, rank, j0, k, (int32_t)s, r);
#pragma unroll
            for (int u = 0; u < ADJ_G; ++u) {
                const double4 o = rec[r[u]];
                const double ex = me.x - o.x, ey = me.y - o.y, ez = me.z - o.z;
                rv[u] = sqrt(ex * ex + ey * ey + ez * ez);
                mv[u] = o.w;
            }
#pragma unroll
            for (int u = 0; u < ADJ_G; ++u) {
                if (j0 + u >= k) break;
                const double w = norm * w_cubic(rv[u] * ih);
                acc += w * mv[u];
                const uint64_t l = (uint64_t)(r[u] - s0);
                if (l < ADJ_B) atomicAdd(&lrho[l], w * me.w);
                else unsafeAtomicAdd(rho + (ORD ? order[r[u]] : r[u]), w * me.w);
            }
        }
    }
    __syncthreads();
    if (s < n) unsafeAtomicAdd(rho + i, acc + lrho[t]);
}

// Contributions outside the block: the lanes that have one put their four
// components and the target in LDS, and four neighbouring lanes add one
// target's components, so a particle's 32 bytes leave as one transaction.
struct SphOut {
    double v[NBX_WAVE][4];
    int32_t to[NBX_WAVE];
};
__device__ __forceinline__ void sph_scatter(SphOut &o, double *acc, bool has, int32_t to, double vx, double vy,
                                            double vz, double vm) {
    const uint64_t m = ballot(has);
    if (!m) return;
    const int lane = threadIdx.x & 63;
    if (has) {
        const int at = __builtin_amdgcn_mbcnt_hi((uint32_t)(m >> 32), __builtin_amdgcn_mbcnt_lo((uint32_t)m, 0u));
        o.v[at][0] = vx;
        o.v[at][1] = vy;
        o.v[at][2] = vz;
        o.v[at][3] = vm;
        o.to[at] = to;
    }
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
    const int cnt = 4 * __popcll(m);
    for (int e = lane; e < cnt; e += NBX_WAVE) unsafeAtomicAdd(acc + 4 * (int64_t)o.to[e >> 2] + (e & 3), o.v[e >> 2][e & 3]);
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
}

template <bool V, bool ORD>
__global__ __launch_bounds__(ADJ_B) void k_sph_adj_ordered(const double4 *__restrict__ rec,
                                                           const int32_t *__restrict__ rank,
                                                           const int32_t *__restrict__ order,
                                                           const double *__restrict__ gs,
                                                           const int32_t *__restrict__ nbr, int64_t r0, int64_t rend,
                                                           int k, double *sums) {
    __shared__ double lx[ADJ_B], ly[ADJ_B], lz[ADJ_B], lm[ADJ_B];
    __shared__ SphOut out[ADJ_B / NBX_WAVE];
    const int t = threadIdx.x;
    const int64_t s0 = r0 + (int64_t)xcd_wave(blockIdx.x, gridDim.x) * ADJ_B;
    const int64_t s = s0 + t;
    lx[t] = 0.0;
    ly[t] = 0.0;
    lz[t] = 0.0;
    lm[t] = 0.0;
    __syncthreads();
    SphOut &o = out[t / NBX_WAVE];
    const bool in = s < rend;
    double gx = 0.0, gy = 0.0, gz = 0.0, gm = 0.0;
    const int64_t i = in ? (ORD ? order[s] : s - r0) : 0;
    const double4 me = in ? rec[s] : make_double4(0.0, 0.0, 0.0, 0.0);
    const double gi = in ? gs[s] : 0.0;
    const int32_t *row = nbr + i * k;
    const int32_t rK = in ? (ORD ? rank[row[k - 1]] : row[k - 1]) : 0;
    const double4 far = rec[rK];
    const double kx = me.x - far.x, ky = me.y - far.y, kz = me.z - far.z;
    const double rk = sqrt(kx * kx + ky * ky + kz * kz);
    const double h = 0.5 * rk;
    const double ih = 1.0 / h;
    const double ih3 = ih * ih * ih, ih4 = ih3 * ih;
    double Hs = 0.0;
    for (int j0 = 0; j0 < k; j0 += ADJ_GB) {  // every lane of a wave takes every step (sph_scatter)
        int32_t r[ADJ_GB];
        double exv[ADJ_GB], eyv[ADJ_GB], ezv[ADJ_GB], mv[ADJ_GB], gv[ADJ_GB];
        if (in) sph_ranks<ADJ_GB, V, ORD>(row, rank, j0, k, (int32_t)s, r);
        else {
#pragma unroll
            for (int u = 0; u < ADJ_GB; ++u) r[u] = 0;
        }
#pragma unroll
        for (int u = 0; u < ADJ_GB; ++u) {
            const double4 q = rec[r[u]];
            exv[u] = me.x - q.x;
            eyv[u] = me.y - q.y;
            ezv[u] = me.z - q.z;
            mv[u] = q.w;
            gv[u] = gs[r[u]];
        }
#pragma unroll
        for (int u = 0; u < ADJ_GB; ++u) {
            if (j0 + u >= k) break;
            const double ex = exv[u], ey = eyv[u], ez = ezv[u];
            const double d = sqrt(ex * ex + ey * ey + ez * ez);
            const double qq = d * ih;
            const double W = w_cubic(qq), dW = dw_cubic(qq);
            const double w = 0.5 * NBX_SIGMA3 * W * ih3;
            const double a = gi * mv[u] + gv[u] * me.w;
            gm += w * gv[u];
            Hs += a * (-0.5 * NBX_SIGMA3 * (qq * dW + 3.0 * W) * ih4);
            const double f = d > 0.0 ? a * 0.5 * NBX_SIGMA3 * dW * ih4 / d : 0.0;
            const bool pull = d > 0.0;  // at one point the direction is undefined: no force
            const double fx = pull ? f * ex : 0.0, fy = pull ? f * ey : 0.0, fz = pull ? f * ez : 0.0;
            gx += fx;
            gy += fy;
            gz += fz;
            const uint64_t l = (uint64_t)(r[u] - s0);
            const bool loc = l < ADJ_B;
            if (in && loc) {
                atomicAdd(&lm[l], w * gi);
                if (pull) {
                    atomicAdd(&lx[l], -fx);
                    atomicAdd(&ly[l], -fy);
                    atomicAdd(&lz[l], -fz);
                }
            }
            sph_scatter(o, sums, in && !loc, r[u], -fx, -fy, -fz, w * gi);
        }
    }
    {
        const bool pull = in && rk > 0.0;
        const double f = pull ? Hs * 0.5 / rk : 0.0;
        const double fx = pull ? f * kx : 0.0, fy = pull ? f * ky : 0.0, fz = pull ? f * kz : 0.0;
        gx += fx;
        gy += fy;
        gz += fz;
        const uint64_t l = (uint64_t)(rK - s0);
        if (pull && l < ADJ_B) {
            atomicAdd(&lx[l], -fx);
            atomicAdd(&ly[l], -fy);
            atomicAdd(&lz[l], -fz);
        }
        sph_scatter(o, sums, pull && l >= ADJ_B, rK, -fx, -fy, -fz, 0.0);
    }
    __syncthreads();
    if (in) {
        double *a = sums + 4 * s;
        unsafeAtomicAdd(a, gx + lx[t]);
        unsafeAtomicAdd(a + 1, gy + ly[t]);
        unsafeAtomicAdd(a + 2, gz + lz[t]);
        unsafeAtomicAdd(a + 3, gm + lm[t]);
    }
}

__global__ __launch_bounds__(256) void k_sph_unpack(const double4 *__restrict__ sums, const int32_t *__restrict__ rank,
                                                    int64_t n, double *dpos, double *dmass) {
    const int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x;
    if (i >= n) return;
    const double4 v = sums[rank ? rank[i] : i];
    dpos[i] = v.x;
    dpos[n + i] = v.y;
    dpos[2 * n + i] = v.z;
    dmass[i] = v.w;
}

static bool sph_vec(const int32_t *nbr, int k) { return k % 4 == 0 && ((uintptr_t)nbr & 15) == 0; }

// order null: the rows as they lie
hipError_t nbx_launch_sph_fwd_ordered(const double *pos, const double *mass, const int32_t *nbr, const int32_t *order,
                                      int64_t n, int k, double *rho, double *h, void *work, hipStream_t st) {
    SphWork W(work, n);
    const dim3 nb((unsigned)((n + 255) / 256)), blocks((unsigned)((n + ADJ_B - 1) / ADJ_B));
    ProfScope ps("k_sph_fwd", st);
    hipLaunchKernelGGL(k_fill_f64, nb, dim3(256), 0, st, rho, 0.0, n);
    hipLaunchKernelGGL(k_sph_pack, nb, dim3(256), 0, st, pos, pos + n, pos + 2 * n, mass, (const double *)nullptr,
                       (const int32_t *)nullptr, order, n, W.rec, (double *)nullptr, W.rank, (double4 *)nullptr);
#define SPH_F(V, ORD)                                                                                                  \
    hipLaunchKernelGGL((k_sph_fwd_ordered<V, ORD>), blocks, dim3(ADJ_B), 0, st, W.rec, W.rank, order, nbr, n, k, rho, h)
    const bool v = sph_vec(nbr, k);
    if (order) { if (v) SPH_F(true, true); else SPH_F(false, true); }
    else { if (v) SPH_F(true, false); else SPH_F(false, false); }
#undef SPH_F
    return hipGetLastError();
}

void nbx_sph_adj_begin(const double *const *X, const double *mass, const int32_t *order, int64_t n, const double *g,
                       const int32_t *gidx, void *work, hipStream_t st) {
    SphWork W(work, n);
    hipLaunchKernelGGL(k_sph_pack, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, st, X[0], X[1], X[2], mass, g, gidx,
                       order, n, W.rec, W.g, W.rank, (double4 *)W.acc);
}
void nbx_sph_adj_rows(const int32_t *nbr, const int32_t *order, int64_t n, int64_t r0, int64_t nr, int k, void *work,
                      hipStream_t st) {
    SphWork W(work, n);
    const dim3 blocks((unsigned)((nr + ADJ_B - 1) / ADJ_B));
#define SPH_A(V, ORD)                                                                                              \
    hipLaunchKernelGGL((k_sph_adj_ordered<V, ORD>), blocks, dim3(ADJ_B), 0, st, W.rec, W.rank, order, W.g, nbr, r0, \
                       r0 + nr, k, W.acc)
    const bool v = sph_vec(nbr, k);
    if (order) { if (v) SPH_A(true, true); else SPH_A(false, true); }
    else { if (v) SPH_A(true, false); else SPH_A(false, false); }
#undef SPH_A
}
// rank: where the sums of an index are (null: at the index)
void nbx_sph_adj_end(const int32_t *rank, int64_t n, double *dpos, double *dmass, void *work, hipStream_t st) {
    SphWork W(work, n);
    hipLaunchKernelGGL(k_sph_unpack, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, st, (const double4 *)W.acc, rank, n,
                       dpos, dmass);
}

hipError_t nbx_launch_sph_adj_ordered(const double *pos, const double *mass, const int32_t *nbr, const int32_t *order,
                                      int64_t n, int k, const double *g, double *dpos, double *dmass, void *work,
                                      hipStream_t st) {
    const double *X[3] = {pos, pos + n, pos + 2 * n};
    ProfScope ps("k_sph_adj", st);
    nbx_sph_adj_begin(X, mass, order, n, g, nullptr, work, st);
    nbx_sph_adj_rows(nbr, order, n, 0, n, k, work, st);
    nbx_sph_adj_end(order ? SphWork(work, n).rank : nullptr, n, dpos, dmass, work, st);
    return hipGetLastError();
}
