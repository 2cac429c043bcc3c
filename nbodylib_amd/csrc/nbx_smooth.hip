// nbx_smooth.hip -- smoothed velocity mean and dispersion on gfx950.
//
// Replaces KDTree::CalcSmoothVel (KDCalcSmoothQuantities.cxx:480-540),
// CalcSmoothVelDisp (:542-614), CalcSmoothVelSkew (:617-690) and
// CalcSmoothVelKurtosis (:692-767) on TPHYS trees, and the local mean and
// dispersion of a per-particle scalar (k_smooth_local).  For every particle i the
// reference takes the non-periodic target kNN of CalcDensity, h_i = r_k / 2,
// and for each neighbour j adds half-weight shares to both ends:
//   mean_i += W_ij / rho_j * m_j * v_j,   mean_j += W_ij / rho_i * m_i * v_i,
// with W_ij = W(r_ij / h_i) h_i^-3 / 2 from the kernel table (the weights of
// CalcDensity's symmetric sum).  The dispersion adds the same weights times
// (v - mean)(v - mean)^T about the receiving particle's finished mean.
//
// The neighbour lists come from the fused kNN + density pass (rows by slot,
// entries slots), with h.  One thread per particle walks its row: its own
// share sums in registers, the other end's share goes to LDS when that
// particle is in the same block and to FP64 atomics otherwise.  Sums are
// order-independent up to rounding.
//
// What bounds these kernels is memory transactions.  So what a neighbour gives
// lies in one record (k_smooth_pack: 64 bytes in two aligned halves) and what
// it receives in another, whose components leave a wave side by side
// (smooth_scatter), one transaction per share instead of one per component;
// 19% of the shares of 1024 rows in tree order go to other blocks.  Separate
// arrays, and a first loop over the row for h, took 1.17 ms (means) and 1.33 ms
// (dispersions) for 0.5M particles, k = 32; these take 0.23 and 0.43 ms.
#include "nbx_kernels.h"

__device__ __forceinline__ double smooth_d2(const DevTree &T, const double *xi, int32_t j) {
    double s = 0.0;
#pragma unroll
    for (int d = 0; d < 3; ++d) {
        const double t = xi[d] - T.x[d][j];
        s += t * t;
    }
    return s;
}

// Records by slot of what a particle gives: position and mass, velocity and
// density; and its h.
__global__ __launch_bounds__(256) void k_smooth_pack(DevTree T, const double *rho_by_id, const double *h_by_id,
                                                     SmoothRec *rec, double *h) {
    const int64_t s = (int64_t)blockIdx.x * 256 + threadIdx.x;
    if (s >= T.n) return;
    const int64_t id = T.perm[s];
    SmoothRec r;
    r.x = make_double4(T.x[0][s], T.x[1][s], T.x[2][s], T.mass[s]);
    r.v = make_double4(T.x[3][s], T.x[4][s], T.x[5][s], rho_by_id[id]);
    rec[s] = r;
    h[s] = h_by_id[id];
}

// Blocks of SM_B consecutive slots: a share for a particle of the same block
// (most neighbours are) is summed with LDS atomics, and each particle's total
// goes out with one global atomic per component; shares for particles of
// other blocks go out as global atomics at once.
#define SM_B 1024
// neighbours whose records are in flight together (a block of 1024 threads has
// 128 registers a thread)
#define SM_GB(STAGE) ((STAGE) == SM_VEL ? 4 : (STAGE) == SM_DISP ? 2 : 1)

// Shares of NC components on their way to sums[slot][W] from one wave, so many
// at a time that the atomics of a round take two instructions.
template <int NC>
struct SmoothOut {
    static constexpr int CAP = 128 / NC;
    double v[CAP * NC];
    int32_t to[CAP];
};
template <int NC, int W>
__device__ __forceinline__ void smooth_scatter(SmoothOut<NC> &o, double *sums, bool has, int32_t to,
                                               const double (&v)[NC]) {
    constexpr int CAP = SmoothOut<NC>::CAP;
    const uint64_t m = ballot(has);
    if (!m) return;
    const int lane = threadIdx.x & 63, cnt = __popcll(m);
    const int at = __builtin_amdgcn_mbcnt_hi((uint32_t)(m >> 32), __builtin_amdgcn_mbcnt_lo((uint32_t)m, 0u));
    for (int b = 0; b < cnt; b += CAP) {
        if (has && at >= b && at < b + CAP) {
#pragma unroll
            for (int c = 0; c < NC; ++c) o.v[(at - b) * NC + c] = v[c];
            o.to[at - b] = to;
        }
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
        __builtin_amdgcn_wave_barrier();
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
        const int e1 = NC * (cnt - b < CAP ? cnt - b : CAP);
        for (int e = lane; e < e1; e += NBX_WAVE) unsafeAtomicAdd(sums + (int64_t)o.to[e / NC] * W + e % NC, o.v[e]);
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
        __builtin_amdgcn_wave_barrier();
    }
}

// One pass over the rows.
// SM_VEL: the means.
// SM_DISP: dispersions about the finished means.  The 3x3 products are
// symmetric (dv_a * dv_b == dv_b * dv_a exactly), so six are summed.
// SM_MOM: per-component skewness and kurtosis (CalcSmoothVelSkew,
// KDCalcSmoothQuantities.cxx:617-690; CalcSmoothVelKurtosis, :692-767) about
// the receiving particle's mean, scaled by its dispersion diagonal s:
// share * dv^3 / s^1.5 and share * dv^4 / (s * s) - 3, the 3 taken off every
// share as the reference does.
#define SM_VEL 0
#define SM_DISP 1
#define SM_MOM 2
template <int STAGE, bool V>
__global__ __launch_bounds__(SM_B) void k_smooth(DevTree T, SmoothArgs A, double *sums) {
    constexpr int NC = STAGE == SM_VEL ? 3 : 6, W = STAGE == SM_VEL ? 4 : 8, GB = SM_GB(STAGE);
    typedef int32_t rowv __attribute__((ext_vector_type(GB == 1 ? 2 : GB)));
    __shared__ double ls[NC][SM_B];
    __shared__ SmoothOut<NC> out[SM_B / NBX_WAVE];
    const int tid = threadIdx.x;
    const int64_t i0 = (int64_t)xcd_wave(blockIdx.x, gridDim.x) * SM_B, i = i0 + tid;
    const int64_t n = T.n;
    const bool valid = i < n;
    SmoothOut<NC> &o = out[tid / NBX_WAVE];
#pragma unroll
    for (int c = 0; c < NC; ++c) ls[c][tid] = 0.0;
    __syncthreads();
    double acc[NC];
#pragma unroll
    for (int c = 0; c < NC; ++c) acc[c] = 0.0;
    const int k = A.k;
    const int32_t *row = A.nn + (valid ? i : 0) * k;
    const double4 xi = A.rec[valid ? i : 0].x, vr = A.rec[valid ? i : 0].v;
    const double vi[3] = {vr.x, vr.y, vr.z}, hi = A.h[valid ? i : 0], mi = xi.w, rhoi = vr.w;
    const double norm = 1.0 / pow(hi, 3.0);
    double ui[3], si[3], pi[3];
    if (STAGE != SM_VEL) {
        const double4 u = A.mean[valid ? i : 0];
        ui[0] = u.x; ui[1] = u.y; ui[2] = u.z;
    }
    if (STAGE == SM_MOM) {
        const SmoothSum &q = A.disp[valid ? i : 0];
#pragma unroll
        for (int d = 0; d < 3; ++d) {
            si[d] = q.c[SM_DIAG(d)];
            pi[d] = pow(si[d], 1.5);
        }
    }
    for (int t0 = 0; t0 < k; t0 += GB) {  // every lane of a wave takes every step (smooth_scatter)
        int32_t r[GB];
        double4 xj[GB], vj[GB], uj[GB];
        if constexpr (V && GB > 1) {
            const rowv q = *(const rowv *)(row + t0);
#pragma unroll
            for (int u = 0; u < GB; ++u) r[u] = q[u];
        } else {
#pragma unroll
            for (int u = 0; u < GB; ++u) r[u] = row[t0 + u < k ? t0 + u : k - 1];
        }
#pragma unroll
        for (int u = 0; u < GB; ++u) {
            xj[u] = A.rec[r[u]].x;
            vj[u] = A.rec[r[u]].v;
            if (STAGE != SM_VEL) uj[u] = A.mean[r[u]];
        }
#pragma unroll
        for (int u = 0; u < GB; ++u) {
            if (t0 + u >= k) break;
            const double dx = xi.x - xj[u].x, dy = xi.y - xj[u].y, dz = xi.z - xj[u].z;
            const double rij = sqrt(dx * dx + dy * dy + dz * dz);
            const double w = 0.5 * wsm_at(rij, hi, T.kern, T.kernres) * norm;
            const double tj = w / vj[u].w * xj[u].w, ti = w / rhoi * mi;
            const double wj[3] = {vj[u].x, vj[u].y, vj[u].z};
            double v[NC];  // the neighbour's share
            if constexpr (STAGE == SM_VEL) {
#pragma unroll
                for (int d = 0; d < 3; ++d) {
                    acc[d] += tj * wj[d];
                    v[d] = ti * vi[d];
                }
            } else {
                const double mj[3] = {uj[u].x, uj[u].y, uj[u].z};
                double a[3], b[3];
#pragma unroll
                for (int d = 0; d < 3; ++d) {
                    a[d] = wj[d] - ui[d];  // neighbour about my mean
                    b[d] = vi[d] - mj[d];  // me about the neighbour's mean
                }
                if constexpr (STAGE == SM_DISP) {
                    int c = 0;
#pragma unroll
                    for (int p = 0; p < 3; ++p)
#pragma unroll
                        for (int q = p; q < 3; ++q, ++c) {
                            acc[c] += tj * a[p] * a[q];
                            v[c] = ti * b[p] * b[q];
                        }
                } else {
#pragma unroll
                    for (int d = 0; d < 3; ++d) {
                        const double sj = A.disp[r[u]].c[SM_DIAG(d)];
                        acc[d] += tj * a[d] * a[d] * a[d] / pi[d];
                        acc[3 + d] += tj * a[d] * a[d] * a[d] * a[d] / (si[d] * si[d]) - 3.;
                        v[d] = ti * b[d] * b[d] * b[d] / pow(sj, 1.5);
                        v[3 + d] = ti * b[d] * b[d] * b[d] * b[d] / (sj * sj) - 3.;
                    }
                }
            }
            const uint64_t l = (uint64_t)(r[u] - i0);
            const bool near = l < SM_B;
            if (valid && near) {
#pragma unroll
                for (int c = 0; c < NC; ++c) atomicAdd(&ls[c][l], v[c]);
            }
            smooth_scatter<NC, W>(o, sums, valid && !near, r[u], v);
        }
    }
    __syncthreads();
    if (valid) {
#pragma unroll
        for (int c = 0; c < NC; ++c) unsafeAtomicAdd(sums + i * W + c, acc[c] + ls[c][tid]);
    }
}

// CalcSmoothLocalMeanParticle / CalcSmoothLocalDispParticle (:1539-1617) and
// the Position forms (:1619-1693): the gather sum over a row with the full
// weight W(r/h) h^-3 (no half, no scatter), each neighbour counting
// W / rho_j * m_j * w_j, and for the dispersion W / rho_j * m_j * (w_j - mean)^2.
__global__ __launch_bounds__(256) void k_smooth_local(DevTree T, LocalArgs A) {
    const int64_t r = (int64_t)blockIdx.x * 256 + threadIdx.x;
    if (r >= A.m) return;
    const int k = A.k;
    const int32_t *row = A.nn + r * k;
    double xi[3];
#pragma unroll
    for (int d = 0; d < 3; ++d) xi[d] = A.q[0] ? A.q[d][r] : T.x[d][r];
    double m2 = 0.0;
    for (int t = 0; t < k; ++t) {
        const int32_t j = A.nn_ids ? T.inv[row[t]] : row[t];
        m2 = fmax(m2, smooth_d2(T, xi, j));
    }
    const double hi = 0.5 * sqrt(m2);
    const double norm = 1.0 / pow(hi, 3.0);
    const double mu = A.mean_in ? A.mean_in[r] : 0.0;
    double mean = 0.0, disp = 0.0;
    for (int t = 0; t < k; ++t) {
        const int32_t j = A.nn_ids ? T.inv[row[t]] : row[t];
        const double rij = sqrt(smooth_d2(T, xi, j));
        const double w = wsm_at(rij, hi, T.kern, T.kernres) * norm;
        const double temp = w / A.rho[j] * T.mass[j];
        mean += temp * A.w[j];
        const double delta = A.w[j] - mu;
        disp += temp * delta * delta;
    }
    if (A.mean) A.mean[r] = mean;
    if (A.disp && A.mean_in) A.disp[r] = disp;
}

hipError_t nbx_launch_smooth_local(const DevTree &T, const LocalArgs &A, hipStream_t st) {
    if (A.m == 0) return hipSuccess;
    ProfScope ps("k_smooth_local", st);
    hipLaunchKernelGGL(k_smooth_local, dim3((unsigned)((A.m + 255) / 256)), dim3(256), 0, st, T, A);
    return hipGetLastError();
}

// Sums by slot ([n][w]) to ID-major rows of ncomp values: from the w-wide
// record's place from0 on, or the six of a dispersion to 3x3 (ncomp 9).
__global__ __launch_bounds__(256) void k_smooth_out(const double *in, const int32_t *perm, int64_t n, int w, int from0,
                                                    int ncomp, double *out) {
    const int64_t s = (int64_t)blockIdx.x * 256 + threadIdx.x;
    if (s >= n) return;
    const int64_t id = perm[s];
    for (int c = 0; c < ncomp; ++c) {
        int src = from0 + c;
        if (ncomp == 9) {
            const int p = c / 3 < c % 3 ? c / 3 : c % 3, q = c / 3 < c % 3 ? c % 3 : c / 3;
            src = p * (5 - p) / 2 + q;
        }
        out[id * ncomp + c] = in[s * w + src];
    }
}
// The reverse, of the caller's means (ncomp 3) or dispersions (ncomp 9).
__global__ __launch_bounds__(256) void k_smooth_in(const double *rows, const int32_t *perm, int64_t n, int w, int ncomp,
                                                   double *out) {
    const int64_t s = (int64_t)blockIdx.x * 256 + threadIdx.x;
    if (s >= n) return;
    const int64_t id = perm[s];
    for (int c = 0; c < ncomp; ++c) {
        const int p = c / 3, q = c % 3;
        if (ncomp == 9 && p > q) continue;
        out[s * w + (ncomp == 9 ? p * (5 - p) / 2 + q : c)] = rows[id * ncomp + c];
    }
}

__global__ __launch_bounds__(256) void k_gather_by_id(const double *by_id, const int32_t *perm, int64_t n,
                                                      double *by_slot) {
    const int64_t s = (int64_t)blockIdx.x * 256 + threadIdx.x;
    if (s < n) by_slot[s] = by_id[perm[s]];
}

static inline int nblk(int64_t n) { return (int)((n + 255) / 256); }

hipError_t nbx_launch_smooth(const DevTree &T, const SmoothArgs &A, bool with_mean, bool with_disp, hipStream_t st) {
    const int64_t n = T.n;
    if (n == 0) return hipSuccess;
    if (T.nd != 3 || !T.x[3] || A.k < 1) return hipErrorInvalidValue;
    if ((with_disp || A.mom) && !A.disp) return hipErrorInvalidValue;
    const dim3 grid((unsigned)((n + SM_B - 1) / SM_B));
    const bool v = A.k % 4 == 0 && ((uintptr_t)A.nn & 15) == 0;
#define SM_RUN(STAGE, sums)                                                                               \
    do {                                                                                                  \
        if (v) hipLaunchKernelGGL((k_smooth<STAGE, true>), grid, dim3(SM_B), 0, st, T, A, (double *)sums); \
        else hipLaunchKernelGGL((k_smooth<STAGE, false>), grid, dim3(SM_B), 0, st, T, A, (double *)sums);  \
    } while (0)
    if (with_mean) {
        ProfScope ps("k_smooth_vel", st);
        SM_RUN(SM_VEL, A.mean);
    }
    if (with_disp) {
        ProfScope ps("k_smooth_disp", st);
        SM_RUN(SM_DISP, A.disp);
    }
    if (A.mom) {
        ProfScope ps("k_smooth_moments", st);
        SM_RUN(SM_MOM, A.mom);
    }
#undef SM_RUN
    return hipGetLastError();
}
