// pp_batch.hip -- batched persistent IC(0)-preconditioned CG over many
// independent SPD systems of uneven size.  k_batch_pcg solves the whole batch
// in one launch: workgroup s owns system s for the entire solve (SpMV, both
// triangular sweeps level by level with workgroup barriers, workgroup
// reductions, the FP64 refinement loop), so no grid-wide synchronisation is
// ever needed and ~256 systems fill the 256 CUs.  The launch is captured in a
// hipGraph and replayed.  The workgroup size (the row tile each SpMV / sweep
// step covers) is chosen per batch by a small timing autotuner.  Mixed solves
// whose systems all have the reduced form spread each system over tiles
// instead (k_tile_cg, k_step_* below).
#include <hip/hip_runtime.h>

#include <algorithm>
#include <atomic>
#include <chrono>
#include <cmath>
#include <cstring>

#include "pp_internal.h"

namespace pp {

struct DevBatchSweep {
    uint32_t *perm = nullptr;     // global row processed at global position k
    uint32_t *rp = nullptr;       // [ntot+1] positions (level order within each system)
    uint32_t *ci = nullptr;       // global dependency rows
    double *val64 = nullptr;
    float *val32 = nullptr;
    double *diag64 = nullptr;     // by global row
    float *diag32 = nullptr;
    uint32_t *lev = nullptr;      // concatenated level pointers (global positions)
    uint32_t *lev_off = nullptr;  // [nsys+1] offsets into lev
    void free_all() {
        dfree(perm); dfree(rp); dfree(ci); dfree(val64); dfree(val32);
        dfree(diag64); dfree(diag32); dfree(lev); dfree(lev_off);
        perm = rp = ci = lev = lev_off = nullptr;
        val64 = diag64 = nullptr;
        val32 = diag32 = nullptr;
    }
};

// Everything the persistent kernel reads, by value.
struct BatchArgs {
    uint32_t nsys;
    const uint32_t *roff;  // [nsys+1]
    const uint32_t *rp, *ci;
    const double *v64;
    const float *v32;
    DevBatchSweep lo, up;
    const double *b;
    double *x;
    double *r64;
    float *r32, *e32, *q32, *w32, *d32, *p32;  // rhs, solution, residual, M^-1 r, direction, A d
    double *rr64, *w64, *d64, *p64;             // FP64 mode: residual, M^-1 r, direction, A d
    double tol, inner_tol;
    uint32_t maxit, max_outer;
    // reduced form of every system's two-colour IC(0) (mixed inner solves),
    // or red_n0 == nullptr: per system its n0 first-colour rows come first;
    // kab: KA rows (first colour) then KB rows (second colour), kfe: KE rows
    // then KF rows, all in batch row and column numbering; s1, dt over the
    // second colour's positions
    const uint32_t *red_n0;
    const uint32_t *kab_rp, *kab_ci, *kfe_rp, *kfe_ci;
    const float *kab_v, *kfe_v, *red_s1, *red_dt;
    int32_t *iters;       // [nsys] total inner iterations
    int32_t *outer;       // [nsys]
    int32_t *conv;        // [nsys]
    double *relres;       // [nsys] final ||b - A x|| / ||b||
};

namespace {

template <int BS>
__device__ inline double block_reduce(double v, double *sh) {
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) v += __shfl_down(v, off, 64);
    const int lane = threadIdx.x & 63, wid = threadIdx.x >> 6;
    __syncthreads();
    if (lane == 0) sh[wid] = v;
    __syncthreads();
    double t = 0.0;
#pragma unroll
    for (int w = 0; w < BS / 64; ++w) t += sh[w];
    return t;  // every thread holds the total (fixed order)
}

// Rows handled per thread and pass: their index, entry and vector loads are
// issued together (a system's workgroup is alone on its CU, so its
// latency is hidden by loads in flight, not by other waves).
constexpr int kRowsInFlight = 4;

// y = A x on the rows [r0, r1) with values V (FP64 or FP32); each row's sum
// in storage order
template <class T, class V>
__device__ inline void sys_spmv(const uint32_t *rp, const uint32_t *ci, const V *val, const T *x, T *y,
                                uint32_t r0, uint32_t r1) {
    constexpr int U = kRowsInFlight;
    const uint32_t step = blockDim.x;
    for (uint32_t i0 = r0 + threadIdx.x; i0 < r1; i0 += U * step) {
        uint32_t k[U], e[U];
        T sum[U];
#pragma unroll
        for (int u = 0; u < U; ++u) {
            const uint32_t i = i0 + u * step;
            k[u] = i < r1 ? rp[i] : 0;
            e[u] = i < r1 ? rp[i + 1] : 0;
            sum[u] = 0;
        }
        for (bool more = true; more;) {
            more = false;
#pragma unroll
            for (int u = 0; u < U; ++u)
                if (k[u] < e[u]) {
                    sum[u] += (T)val[k[u]] * x[ci[k[u]]];
                    ++k[u];
                    more = true;
                }
        }
#pragma unroll
        for (int u = 0; u < U; ++u) {
            const uint32_t i = i0 + u * step;
            if (i < r1) y[i] = sum[u];
        }
    }
}

// Level-by-level sweep of one system; y may alias b (rows of a level only read
// rows of earlier levels, finished before the barrier, and each row reads its
// own b before writing its y).  mode 0: divide by diag (IC(0) both sweeps).
template <class T>
__device__ inline void sys_sweep(const uint32_t *perm, const uint32_t *rp, const uint32_t *ci, const T *val,
                                 const T *diag, const uint32_t *lev, uint32_t l0, uint32_t l1, const T *b, T *y) {
    constexpr int U = kRowsInFlight;
    const uint32_t step = blockDim.x;
    for (uint32_t l = l0; l < l1; ++l) {
        const uint32_t k1 = lev[l + 1];
        for (uint32_t k0 = lev[l] + threadIdx.x; k0 < k1; k0 += U * step) {
            uint32_t row[U], e[U], f[U];
            T sum[U];
#pragma unroll
            for (int u = 0; u < U; ++u) {
                const uint32_t k = k0 + u * step;
                const bool ok = k < k1;
                row[u] = ok ? perm[k] : 0;
                e[u] = ok ? rp[k] : 0;
                f[u] = ok ? rp[k + 1] : 0;
                sum[u] = ok ? b[row[u]] : (T)0;
            }
            for (bool more = true; more;) {
                more = false;
#pragma unroll
                for (int u = 0; u < U; ++u)
                    if (e[u] < f[u]) {
                        sum[u] -= val[e[u]] * y[ci[e[u]]];
                        ++e[u];
                        more = true;
                    }
            }
#pragma unroll
            for (int u = 0; u < U; ++u)
                if (k0 + u * step < k1) y[row[u]] = sum[u] / diag[row[u]];
        }
        __syncthreads();
    }
}

template <class T>
struct Pick;
template <>
struct Pick<float> {
    __device__ static const float *v(const BatchArgs &a) { return a.v32; }
    __device__ static const float *lv(const DevBatchSweep &s) { return s.val32; }
    __device__ static const float *dg(const DevBatchSweep &s) { return s.diag32; }
};
template <>
struct Pick<double> {
    __device__ static const double *v(const BatchArgs &a) { return a.v64; }
    __device__ static const double *lv(const DevBatchSweep &s) { return s.val64; }
    __device__ static const double *dg(const DevBatchSweep &s) { return s.diag64; }
};

// FlexibleCG (source/Solver/CG.cpp:33-83) on one system in precision T,
// x0 = 0 in x, stopping on the recursive residual.  Returns iterations in the
// reference convention (m + 1).
template <class T, int BS>
__device__ int sys_pcg(const BatchArgs &a, uint32_t s, uint32_t r0, uint32_t r1, const T *b, T *x, T *r, T *w,
                       T *d, T *v, double tol, uint32_t maxit, double *sh, int *converged) {
    const T *A = Pick<T>::v(a);
    // system s owns level pointers lev[off[s] .. off[s+1]-1] (nlev + 1 of them)
    const uint32_t L0 = a.lo.lev_off[s], L1 = a.lo.lev_off[s + 1] - 1;
    const uint32_t U0 = a.up.lev_off[s], U1 = a.up.lev_off[s + 1] - 1;
    auto apply = [&](const T *in, T *out) {
        sys_sweep<T>(a.lo.perm, a.lo.rp, a.lo.ci, Pick<T>::lv(a.lo), Pick<T>::dg(a.lo), a.lo.lev, L0, L1, in, out);
        sys_sweep<T>(a.up.perm, a.up.rp, a.up.ci, Pick<T>::lv(a.up), Pick<T>::dg(a.up), a.up.lev, U0, U1, out, out);
    };
    // r = b (x0 = 0), w = M^{-1} r, d = w, v = A d
    double bb = 0.0;
    for (uint32_t i = r0 + threadIdx.x; i < r1; i += BS) {
        r[i] = b[i];
        x[i] = 0;
        bb += (double)b[i] * (double)b[i];
    }
    const double normb = sqrt(block_reduce<BS>(bb, sh));
    __syncthreads();
    apply(r, w);
    double dr = 0.0;
    for (uint32_t i = r0 + threadIdx.x; i < r1; i += BS) {
        d[i] = w[i];
        dr += (double)(w[i] * r[i]);
    }
    dr = block_reduce<BS>(dr, sh);
    __syncthreads();
    sys_spmv<T, T>(a.rp, a.ci, A, d, v, r0, r1);
    __syncthreads();
    double dv = 0.0;
    for (uint32_t i = r0 + threadIdx.x; i < r1; i += BS) dv += (double)(d[i] * v[i]);
    dv = block_reduce<BS>(dv, sh);
    uint32_t m = maxit;
    *converged = 0;
    if (normb == 0.0) {
        *converged = 1;
        return 1;
    }
    for (uint32_t it = 0;; ++it) {
        // x += alpha d ; r -= alpha v ; (r, r)
        const T alpha = (T)(dr / dv);
        double rr = 0.0;
        for (uint32_t i = r0 + threadIdx.x; i < r1; i += BS) {
            x[i] += alpha * d[i];
            const T rn = r[i] - alpha * v[i];
            r[i] = rn;
            rr += (double)(rn * rn);
        }
        rr = block_reduce<BS>(rr, sh);
        const uint32_t check = it + 1;
        if (check >= maxit) break;
        const double norm = sqrt(rr) / normb;
        if (!(norm == norm)) break;
        if (norm < tol) {
            *converged = 1;
            m = check;
            break;
        }
        __syncthreads();
        apply(r, w);
        double wv = 0.0;
        for (uint32_t i = r0 + threadIdx.x; i < r1; i += BS) wv += (double)(w[i] * v[i]);
        wv = block_reduce<BS>(wv, sh);
        const T beta = (T)(wv / dv);
        dr = 0.0;
        for (uint32_t i = r0 + threadIdx.x; i < r1; i += BS) {
            const T dn = w[i] - beta * d[i];
            d[i] = dn;
            dr += (double)(dn * r[i]);
        }
        dr = block_reduce<BS>(dr, sh);
        __syncthreads();
        sys_spmv<T, T>(a.rp, a.ci, A, d, v, r0, r1);
        __syncthreads();
        dv = 0.0;
        for (uint32_t i = r0 + threadIdx.x; i < r1; i += BS) dv += (double)(d[i] * v[i]);
        dv = block_reduce<BS>(dv, sh);
        if (dv == 0.0 || !(dv == dv)) break;
    }
    __syncthreads();
    return (int)m + 1;
}

// three sums at once (fixed order); sh holds 3 * BS / 64 doubles
template <int BS>
__device__ inline void block_reduce3(double &a, double &b, double &c, double *sh) {
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) {
        a += __shfl_down(a, off, 64);
        b += __shfl_down(b, off, 64);
        c += __shfl_down(c, off, 64);
    }
    const int lane = threadIdx.x & 63, wid = threadIdx.x >> 6;
    __syncthreads();
    if (lane == 0) {
        sh[wid] = a;
        sh[BS / 64 + wid] = b;
        sh[2 * BS / 64 + wid] = c;
    }
    __syncthreads();
    a = b = c = 0.0;
#pragma unroll
    for (int w = 0; w < BS / 64; ++w) {
        a += sh[w];
        b += sh[BS / 64 + w];
        c += sh[2 * BS / 64 + w];
    }
}

// CG on the reduced system of system s's two-colour IC(0) (the same
// iteration as the single-system reduced CG: single-reduction recurrence,
// u = r): solves A e = rin approximately to the relative reduction tol of
// the inner system's true residual sqrt(sum Dt r^2) / ||rin||.  z holds
// y0 = KA r on the first colour and r on the second; x accumulates in e's
// second-colour part.  Returns the number of residual checks.
template <int BS>
__device__ int sys_red_cg(const BatchArgs &a, uint32_t s, uint32_t r0, uint32_t r1, const float *rin, float *e,
                          float *z, float *w, float *p, float *sv, double tol, uint32_t maxit, double *sh,
                          double *sh3, int *converged) {
    constexpr int U = kRowsInFlight;
    const uint32_t m0 = r0 + a.red_n0[s];
    // r = KF rin (second colour); x = p = s = 0; ||rin||
    sys_spmv<float, float>(a.kfe_rp, a.kfe_ci, a.kfe_v, rin, z, m0, r1);
    double bb = 0.0;
    for (uint32_t i = r0 + threadIdx.x; i < r1; i += BS) bb += (double)rin[i] * (double)rin[i];
    for (uint32_t i = m0 + threadIdx.x; i < r1; i += BS) {
        e[i] = 0.f;
        p[i] = 0.f;
        sv[i] = 0.f;
    }
    const double normb = sqrt(block_reduce<BS>(bb, sh));
    __syncthreads();
    *converged = 0;
    uint32_t m = maxit;
    double gold = 0.0, aold = 1.0;
    bool first = true;
    for (uint32_t c = 1;; ++c) {
        sys_spmv<float, float>(a.kab_rp, a.kab_ci, a.kab_v, z, z, r0, m0);  // y0 = KA r
        __syncthreads();
        // w = KB [y0; r] with (r, w), (r, r) and sum Dt r^2
        double delta = 0.0, gamma = 0.0, rho = 0.0;
        for (uint32_t i0 = m0 + threadIdx.x; i0 < r1; i0 += U * BS) {
            uint32_t k[U], f[U];
            float sum[U], ri[U], di[U];
#pragma unroll
            for (int u = 0; u < U; ++u) {
                const uint32_t i = i0 + u * BS;
                const bool ok = i < r1;
                k[u] = ok ? a.kab_rp[i] : 0;
                f[u] = ok ? a.kab_rp[i + 1] : 0;
                ri[u] = ok ? z[i] : 0.f;
                di[u] = ok ? a.red_dt[i] : 0.f;
                sum[u] = 0.f;
            }
            for (bool more = true; more;) {
                more = false;
#pragma unroll
                for (int u = 0; u < U; ++u)
                    if (k[u] < f[u]) {
                        sum[u] += a.kab_v[k[u]] * z[a.kab_ci[k[u]]];
                        ++k[u];
                        more = true;
                    }
            }
#pragma unroll
            for (int u = 0; u < U; ++u) {
                const uint32_t i = i0 + u * BS;
                if (i < r1) {
                    w[i] = sum[u];
                    delta += (double)(ri[u] * sum[u]);
                    gamma += (double)(ri[u] * ri[u]);
                    rho += (double)di[u] * (double)(ri[u] * ri[u]);
                }
            }
        }
        block_reduce3<BS>(delta, gamma, rho, sh3);
        if (c >= maxit) break;
        const double norm = normb > 0.0 ? sqrt(rho) / normb : 0.0;
        if (!(norm == norm) || isinf(norm)) break;
        if (norm < tol) {
            *converged = 1;
            m = c;
            break;
        }
        const double beta = first ? 0.0 : gamma / gold;
        const double den = first ? delta : delta - beta * gamma / aold;
        if (den == 0.0 || !(den == den)) break;
        const double alpha = gamma / den;
        gold = gamma;
        aold = alpha;
        first = false;
        const float fa = (float)alpha, fb = (float)beta;
        for (uint32_t i0 = m0 + threadIdx.x; i0 < r1; i0 += U * BS) {
            float zr[U], wr[U], pr[U], sr[U], er[U];
#pragma unroll
            for (int u = 0; u < U; ++u) {
                const uint32_t i = i0 + u * BS;
                if (i < r1) {
                    zr[u] = z[i];
                    wr[u] = w[i];
                    pr[u] = p[i];
                    sr[u] = sv[i];
                    er[u] = e[i];
                }
            }
#pragma unroll
            for (int u = 0; u < U; ++u) {
                const uint32_t i = i0 + u * BS;
                if (i < r1) {
                    const float pn = zr[u] + fb * pr[u];
                    const float sn = wr[u] + fb * sr[u];
                    p[i] = pn;
                    sv[i] = sn;
                    e[i] = er[u] + fa * pn;
                    z[i] = zr[u] - fa * sn;
                }
            }
        }
        __syncthreads();
    }
    // e = [KE [rin_0; e_1]; e_1], e_1 = s1 x
    __syncthreads();
    for (uint32_t i = m0 + threadIdx.x; i < r1; i += BS) {
        const float ei = a.red_s1[i] * e[i];
        e[i] = ei;
        z[i] = ei;
    }
    for (uint32_t i = r0 + threadIdx.x; i < m0; i += BS) z[i] = rin[i];
    __syncthreads();
    sys_spmv<float, float>(a.kfe_rp, a.kfe_ci, a.kfe_v, z, e, r0, m0);
    __syncthreads();
    return (int)m;
}

// One workgroup per system.  MIXED: FP64 residual r = b - A x, FP32 inner
// FlexibleCG on A e = r / ||r|| (or the reduced CG where every system has
// the two-colour structure), x += ||r|| e, until ||b - A x|| / ||b|| < tol.
template <int BS, bool MIXED>
__global__ __launch_bounds__(BS) void k_batch_pcg(BatchArgs a) {
    __shared__ double sh[BS / 64];
    __shared__ double sh3[3 * (BS / 64)];
    const uint32_t s = blockIdx.x;
    if (s >= a.nsys) return;
    const uint32_t r0 = a.roff[s], r1 = a.roff[s + 1];
    int conv = 0, total = 0, outer = 0;
    double rel = 1.0;
    if (!MIXED) {
        total = sys_pcg<double, BS>(a, s, r0, r1, a.b, a.x, a.rr64, a.w64, a.d64, a.p64, a.tol, a.maxit, sh, &conv);
        outer = 1;
        __syncthreads();
        sys_spmv<double, double>(a.rp, a.ci, a.v64, a.x, a.r64, r0, r1);
        __syncthreads();
        double rr = 0.0, bb = 0.0;
        for (uint32_t i = r0 + threadIdx.x; i < r1; i += BS) {
            const double t = a.b[i] - a.r64[i];
            rr += t * t;
            bb += a.b[i] * a.b[i];
        }
        rr = block_reduce<BS>(rr, sh);
        bb = block_reduce<BS>(bb, sh);
        rel = bb > 0 ? sqrt(rr) / sqrt(bb) : 0.0;
    } else {
        double bb = 0.0;
        for (uint32_t i = r0 + threadIdx.x; i < r1; i += BS) {
            bb += a.b[i] * a.b[i];
            a.x[i] = 0.0;
        }
        const double normb = sqrt(block_reduce<BS>(bb, sh));
        for (;;) {
            __syncthreads();
            sys_spmv<double, double>(a.rp, a.ci, a.v64, a.x, a.r64, r0, r1);
            __syncthreads();
            double rr = 0.0;
            for (uint32_t i = r0 + threadIdx.x; i < r1; i += BS) {
                const double t = a.b[i] - a.r64[i];
                a.r64[i] = t;
                rr += t * t;
            }
            const double rn = sqrt(block_reduce<BS>(rr, sh));
            rel = normb > 0 ? rn / normb : 0.0;
            if (rel < a.tol || !(rel == rel)) {
                conv = rel < a.tol;
                break;
            }
            if ((uint32_t)outer >= a.max_outer || (uint32_t)total >= a.maxit) break;
            const float sc = (float)(1.0 / rn);
            for (uint32_t i = r0 + threadIdx.x; i < r1; i += BS) a.r32[i] = (float)a.r64[i] * sc;
            __syncthreads();
            const double want = fmax(a.inner_tol, 0.5 * a.tol * normb / rn);
            int ic = 0;
            if (a.red_n0)
                total += sys_red_cg<BS>(a, s, r0, r1, a.r32, a.e32, a.q32, a.w32, a.d32, a.p32, want,
                                        a.maxit - (uint32_t)total, sh, sh3, &ic);
            else
                total += sys_pcg<float, BS>(a, s, r0, r1, a.r32, a.e32, a.q32, a.w32, a.d32, a.p32, want,
                                            a.maxit - (uint32_t)total, sh, &ic);
            ++outer;
            for (uint32_t i = r0 + threadIdx.x; i < r1; i += BS) a.x[i] += rn * (double)a.e32[i];
        }
    }
    if (threadIdx.x == 0) {
        a.iters[s] = total;
        a.outer[s] = outer;
        a.conv[s] = conv;
        a.relres[s] = rel;
    }
}

// ---------------------------------------------------------------------------
// The mixed solve of a batch in reduced form with every system's inner CG
// spread over tiles, a workgroup each (k_tile_cg), and the refinement steps
// around it over slices of rows (k_step_*).
//
// One workgroup per system left the largest system alone on one compute unit
// (65,536 rows: 135 us an iteration, 4.4 MB of operators and vectors streamed
// at the 33 GB/s one unit draws, while the small systems' units idled).  A
// tile of at most 2048 second-colour rows keeps everything in the unit: the
// operators' values and the vectors p, s, e in registers, r and y0 = KA r in
// LDS.  It owns its rows and computes what it reads of its neighbours' twice:
// F = the first-colour rows its own rows touch, R = its own rows and those F
// touches (r and s are kept for all of R).  So one exchange an iteration
// remains: w on R's halo, and the tiles' three partial sums.  Every word
// carries its iteration's number beside 32 bits of payload, so it is its own
// ready flag and nothing is reset; two buffers alternate, since a tile may
// run one iteration ahead of another's reads but not two.
// Tiles of one system are neighbours in the launch, no more than the chip
// holds, and workgroups start in order, so the first unfinished system has all
// its tiles running.  Should other work keep them out all the same, a wait
// past the deadline raises the abort word, which ends every tile, and the
// batch is solved by k_batch_pcg instead.
// A solve of 256 systems of 32^2 to 256^2 rows: 88 ms with one workgroup a
// system, 7.3 ms now, 6.5 of it here.  There are 1,664 tiles, and the 512 places
// are taken until 0.75 to 0.9 of the time, 5.6 us a tile-iteration: the tiles'
// number sets it, not the largest systems, which start first and end after a
// third.  Two workgroups of 256 threads a unit
// hide each other's exchange: one of 512 threads, the same rows and registers
// a thread, took 0.3 ms more (24 systems of 60^2 to 200^2: 2.72 against 2.51).
// ---------------------------------------------------------------------------
constexpr int kTileThreads = 256;
// rows of F, owned rows, halo rows of a thread, by the entries of a row
template <int W>
struct TileShape {
    static constexpr int kF = W <= 4 ? 10 : 8, kS = W <= 4 ? 8 : 5, kH = W <= 4 ? 3 : 5;
};
constexpr uint32_t kNoSlot = 0xffffffffu;

struct Tile {
    uint32_t sys, tile0, ntile;     // its system, the system's first tile and count
    uint32_t row0, ns, nf, nh;      // first owned row; owned, F, halo rows
    uint32_t f, h;                  // F's rows in `rows`, then the halo's; the halo's slots in `slots`
    uint32_t ka, kb;                // local words of F's and the owned rows' entries in `loc` (W a row, by entry)
    uint32_t out;                   // the owned rows' slots in `slots`
};

struct TileArgs {
    const Tile *tiles;
    const uint32_t *rows, *slots;
    const uint16_t *loc;
    unsigned long long *xw, *xp;    // exchanged w (two buffers of nslot), partial sums (two of 6 * ntiles)
    uint32_t nslot, ntiles;
    int *abort;
    long long deadline;
    const int32_t *active;          // per system, set by k_step_test
    const double *want, *rin_norm;
    const uint32_t *left;           // iterations the system may still take
    const uint32_t *kab_rp;
    const float *kab_v, *red_s1, *red_dt;
    float *z, *e;
    int32_t *iters;
};

__device__ inline unsigned long long tagged(uint32_t tag, uint32_t v) { return (unsigned long long)tag << 32 | v; }
__device__ inline void put_word(unsigned long long *p, unsigned long long v) {
    __hip_atomic_store(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ inline unsigned long long get_word(const unsigned long long *p) {
    return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

// v, but nothing computed from it leaves the loop it is used in (unpacked
// addresses kept across iterations would not fit the registers)
__device__ inline uint32_t here(uint32_t v) {
    asm volatile("" : "+v"(v));
    return v;
}

template <int W>
__global__ __launch_bounds__(kTileThreads) void k_tile_cg(TileArgs a) {
    using Sh = TileShape<W>;
    constexpr int F = Sh::kF, S = Sh::kS, H = Sh::kH, BS = kTileThreads;
    constexpr uint32_t kWords = BS / 6 * 6;  // partial-sum words read at a time, one a thread
    __shared__ float zr[(S + H) * BS], zy[F * BS];
    __shared__ double sh3[3 * (BS / 64)];
    __shared__ uint32_t part[kWords];
    __shared__ int stop;
    const Tile t = a.tiles[blockIdx.x];
    if (!a.active[t.sys]) return;
    const uint32_t tid = threadIdx.x;
    // operators and vectors of this thread's rows
    float kav[F][W], kbv[S][W + 1];
    uint32_t kai[F][W / 2], kbi[S][W / 2];
#pragma unroll
    for (int k = 0; k < F; ++k) {
        const uint32_t f = tid + k * BS;
        const bool ok = f < t.nf;
        const uint32_t i = ok ? a.rows[t.f + f] : 0;
        const uint32_t e0 = ok ? a.kab_rp[i] : 0, e1 = ok ? a.kab_rp[i + 1] : 0;
#pragma unroll
        for (int j = 0; j < W; ++j) {
            kav[k][j] = e0 + j < e1 ? a.kab_v[e0 + j] : 0.f;
            const uint32_t w = ok ? a.loc[t.ka + j * t.nf + f] : 0;
            kai[k][j / 2] = (j & 1) ? kai[k][j / 2] | w << 16 : w;
        }
    }
    float p[S], sv[S], e[S], dt[S];
    uint32_t to[S];
#pragma unroll
    for (int k = 0; k < S; ++k) {
        const uint32_t q = tid + k * BS;
        const bool ok = q < t.ns;
        const uint32_t i = t.row0 + (ok ? q : 0);
        const uint32_t e0 = ok ? a.kab_rp[i] : 0, e1 = ok ? a.kab_rp[i + 1] : 0;
#pragma unroll
        for (int j = 0; j < W; ++j) {
            kbv[k][j] = e0 + j + 1 < e1 ? a.kab_v[e0 + j] : 0.f;
            const uint32_t w = ok ? a.loc[t.kb + j * t.ns + q] : 0;
            kbi[k][j / 2] = (j & 1) ? kbi[k][j / 2] | w << 16 : w;
        }
        kbv[k][W] = ok ? a.kab_v[e1 - 1] : 0.f;  // the diagonal, last
        p[k] = sv[k] = e[k] = 0.f;
        dt[k] = ok ? a.red_dt[i] : 0.f;
        to[k] = ok ? a.slots[t.out + q] : kNoSlot;
        if (ok) zr[q] = a.z[i];
    }
    float hs[H];
    uint32_t from[H];
#pragma unroll
    for (int k = 0; k < H; ++k) {
        const uint32_t h = tid + k * BS;
        hs[k] = 0.f;
        from[k] = kNoSlot;
        if (h < t.nh) {
            from[k] = a.slots[t.h + h];
            zr[t.ns + h] = a.z[a.rows[t.f + t.nf + h]];
        }
    }
    if (tid == 0) stop = 0;
    const double tol = a.want[t.sys], normb = a.rin_norm[t.sys];
    const uint32_t maxit = a.left[t.sys];
    const bool shared = t.ntile > 1;
    uint32_t m = maxit;
    double gold = 0.0, aold = 1.0;
    bool first = true;
    __syncthreads();
    for (uint32_t c = 1;; ++c) {
        // y0 = KA r on F
#pragma unroll
        for (int k = 0; k < F; ++k) {
            float sum = 0.f;
#pragma unroll
            for (int j = 0; j < W; j += 2) {
                const uint32_t pair = here(kai[k][j / 2]);
                sum += kav[k][j] * zr[pair & 0xffffu];
                sum += kav[k][j + 1] * zr[pair >> 16];
            }
            if (tid + k * BS < t.nf) zy[tid + k * BS] = sum;
        }
        __syncthreads();
        // w = KB [y0; r] with (r, w), (r, r) and sum Dt r^2
        const uint32_t par = c & 1;
        unsigned long long *xw = a.xw + (size_t)par * a.nslot, *xp = a.xp + (size_t)par * 6 * a.ntiles;
        double delta = 0.0, gamma = 0.0, rho = 0.0;
        float w[S], r[S];
#pragma unroll
        for (int k = 0; k < S; ++k) {
            const bool ok = tid + k * BS < t.ns;
            r[k] = ok ? zr[tid + k * BS] : 0.f;
            float sum = 0.f;
#pragma unroll
            for (int j = 0; j < W; j += 2) {
                const uint32_t pair = here(kbi[k][j / 2]);
                sum += kbv[k][j] * zy[pair & 0xffffu];
                sum += kbv[k][j + 1] * zy[pair >> 16];
            }
            sum += kbv[k][W] * r[k];
            w[k] = sum;
            if (to[k] != kNoSlot) put_word(xw + to[k], tagged(c, __float_as_uint(sum)));
            if (ok) {
                delta += (double)(r[k] * sum);
                gamma += (double)(r[k] * r[k]);
                rho += (double)dt[k] * (double)(r[k] * r[k]);
            }
        }
        block_reduce3<BS>(delta, gamma, rho, sh3);
        float hw[H] = {};
        if (shared) {
            // this tile's sums out, all tiles' sums and the halo's w in
            if (tid < 6) {
                const double v = tid < 2 ? delta : tid < 4 ? gamma : rho;
                const uint32_t half = (tid & 1) ? (uint32_t)__double2hiint(v) : (uint32_t)__double2loint(v);
                put_word(xp + 6 * (size_t)blockIdx.x + tid, tagged(c, half));
            }
            const uint32_t nw = 6 * t.ntile;
            double td = 0.0, tg = 0.0, tr = 0.0;
            bool wait_h[H];
#pragma unroll
            for (int k = 0; k < H; ++k) wait_h[k] = from[k] != kNoSlot;
            for (uint32_t w0 = 0; w0 < nw; w0 += kWords) {
                const uint32_t cnt = min(nw - w0, kWords);
                bool wait_p = tid < cnt;
                const unsigned long long *src = xp + 6 * (size_t)t.tile0 + w0 + tid;
                WaitClock clock;
                for (uint32_t iter = 1;; ++iter) {
                    bool more = false;
                    const unsigned long long v = wait_p ? get_word(src) : 0;
                    unsigned long long hv[H];
#pragma unroll
                    for (int k = 0; k < H; ++k) hv[k] = wait_h[k] ? get_word(xw + from[k]) : 0;
                    if (wait_p && (uint32_t)(v >> 32) == c) {
                        part[tid] = (uint32_t)v;
                        wait_p = false;
                    }
                    more = wait_p;
#pragma unroll
                    for (int k = 0; k < H; ++k) {
                        if (wait_h[k] && (uint32_t)(hv[k] >> 32) == c) {
                            hw[k] = __uint_as_float((uint32_t)hv[k]);
                            wait_h[k] = false;
                        }
                        more = more || wait_h[k];
                    }
                    if (!__any(more)) break;
                    if (WaitClock::due(iter, a.deadline) &&
                        (clock.expired(a.deadline) ||
                         __hip_atomic_load(a.abort, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT))) {
                        atomicOr(a.abort, 1);
                        stop = 1;
                        break;
                    }
                }
                __syncthreads();
                for (uint32_t q = 0; q < cnt / 6; ++q) {  // in tile order, the same in every tile
                    td += __hiloint2double((int)part[6 * q + 1], (int)part[6 * q]);
                    tg += __hiloint2double((int)part[6 * q + 3], (int)part[6 * q + 2]);
                    tr += __hiloint2double((int)part[6 * q + 5], (int)part[6 * q + 4]);
                }
                if (w0 + kWords < nw) __syncthreads();
            }
            delta = td;
            gamma = tg;
            rho = tr;
            if (stop) break;
        }
        if (c >= maxit) break;
        const double norm = normb > 0.0 ? sqrt(rho) / normb : 0.0;
        if (!(norm == norm) || isinf(norm)) break;
        if (norm < tol) {
            m = c;
            break;
        }
        const double beta = first ? 0.0 : gamma / gold;
        const double den = first ? delta : delta - beta * gamma / aold;
        if (den == 0.0 || !(den == den)) break;
        const double alpha = gamma / den;
        gold = gamma;
        aold = alpha;
        first = false;
        const float fa = (float)alpha, fb = (float)beta;
#pragma unroll
        for (int k = 0; k < S; ++k) {
            p[k] = r[k] + fb * p[k];
            sv[k] = w[k] + fb * sv[k];
            e[k] = e[k] + fa * p[k];
            if (tid + k * BS < t.ns) zr[tid + k * BS] = r[k] - fa * sv[k];
        }
#pragma unroll
        for (int k = 0; k < H; ++k)
            if (tid + k * BS < t.nh) {
                hs[k] = hw[k] + fb * hs[k];
                zr[t.ns + tid + k * BS] -= fa * hs[k];
            }
        __syncthreads();
    }
    // e_1 = s1 x
#pragma unroll
    for (int k = 0; k < S; ++k)
        if (tid + k * BS < t.ns) {
            const uint32_t i = t.row0 + tid + k * BS;
            const float v = a.red_s1[i] * e[k];
            a.e[i] = v;
            a.z[i] = v;
        }
    if (tid == 0 && blockIdx.x == t.tile0) a.iters[t.sys] += (int32_t)m;
}

// One refinement step of the batch: the last inner solve's correction (not in
// the first step), the FP64 residual and its test, then the next inner
// solve's right-hand side r = KF rin, rin = (b - A x) / ||b - A x||.  It
// streams the operators once, so the rows go over all of the chip in slices
// of kSliceRows, and each of its three sums or row couplings across slices is
// the end of a launch.  A workgroup per system in one launch took 565 us for
// 256 systems of 32^2 to 256^2 rows, the largest system's 64 rows a thread
// behind one another; the five launches take 232 us (residual 127).
constexpr int kSliceThreads = 256;
constexpr uint32_t kSliceRows = kSliceThreads, kSliceWidth = 7;  // entries of a row at most (batch_build_tiles)
struct Slice {
    uint32_t sys, i0, i1;
};
struct StepState {
    const Slice *slices;
    const uint32_t *first;  // [nsys + 1] slices of a system
    double *part;           // two sums of a slice
    int32_t *active;
    double *want, *rin_norm, *rn, *normb;
    uint32_t *left;
    int *any;  // set when a system goes on
};

// Row i0 + thread of K x for the slice's rows [i0, i1): the entries and what
// they gather come in coalesced and go through LDS, a thread then adds its
// row's in order (row by row from memory the residual took 329 us, its lanes
// 40 bytes apart).
template <class T>
struct SliceStage {
    T v[kSliceRows * kSliceWidth], x[kSliceRows * kSliceWidth];
};
template <class T>
__device__ inline T slice_row(const uint32_t *__restrict__ rp, const uint32_t *__restrict__ ci,
                              const T *__restrict__ val, const T *x, uint32_t i0, uint32_t i1, SliceStage<T> &st) {
    if (i0 >= i1) return (T)0;
    const uint32_t e0 = rp[i0], cnt = rp[i1] - e0, i = i0 + threadIdx.x;
    uint32_t c[kSliceWidth];
    T v[kSliceWidth], g[kSliceWidth];
#pragma unroll
    for (uint32_t u = 0; u < kSliceWidth; ++u) {
        const uint32_t k = min(threadIdx.x + u * kSliceThreads, cnt - 1);  // every row holds its diagonal
        c[u] = ci[e0 + k];
        v[u] = val[e0 + k];
    }
#pragma unroll
    for (uint32_t u = 0; u < kSliceWidth; ++u) g[u] = x[c[u]];
#pragma unroll
    for (uint32_t u = 0; u < kSliceWidth; ++u) {
        const uint32_t k = threadIdx.x + u * kSliceThreads;
        if (k < cnt) {
            st.v[k] = v[u];
            st.x[k] = g[u];
        }
    }
    __syncthreads();
    T sum = 0;
    if (i < i1)
        for (uint32_t k = rp[i] - e0, e = rp[i + 1] - e0; k < e; ++k) sum += st.v[k] * st.x[k];
    return sum;
}

// The sum of a system's slices (q: which of the two), in every thread.
__device__ inline double slice_sum(const StepState &st, uint32_t s, int q, double *sh) {
    double v = 0.0;
    for (uint32_t k = st.first[s] + threadIdx.x; k < st.first[s + 1]; k += kSliceThreads) v += st.part[2 * (size_t)k + q];
    return block_reduce<kSliceThreads>(v, sh);
}

// x = 0 and (b, b); or e = [KE [rin_0; e_1]; e_1] (a KE row holds its diagonal
// and second-colour columns, so it reads rin_0 in its own row only) and x += rn e
__global__ __launch_bounds__(kSliceThreads) void k_step_correct(BatchArgs a, StepState st, int begin) {
    __shared__ double sh[kSliceThreads / 64];
    __shared__ SliceStage<float> stage;
    const Slice c = st.slices[blockIdx.x];
    const uint32_t m0 = min(c.i1, a.roff[c.sys] + a.red_n0[c.sys]), i = c.i0 + threadIdx.x;
    if (begin) {
        double bb = 0.0;
        if (i < c.i1) {
            bb = a.b[i] * a.b[i];
            a.x[i] = 0.0;
        }
        bb = block_reduce<kSliceThreads>(bb, sh);
        if (threadIdx.x == 0) st.part[2 * (size_t)blockIdx.x] = bb;
        return;
    }
    if (!st.active[c.sys]) return;
    if (i < m0) a.q32[i] = a.r32[i];
    __syncthreads();
    const float e0 = slice_row<float>(a.kfe_rp, a.kfe_ci, a.kfe_v, a.q32, c.i0, m0, stage);
    if (i < c.i1) a.x[i] += st.rn[c.sys] * (double)(i < m0 ? e0 : a.e32[i]);
}

// b - A x and its squares' sum
__global__ __launch_bounds__(kSliceThreads) void k_step_residual(BatchArgs a, StepState st, int begin) {
    __shared__ double sh[kSliceThreads / 64];
    __shared__ SliceStage<double> stage;
    const Slice c = st.slices[blockIdx.x];
    if (!begin && !st.active[c.sys]) return;
    const uint32_t i = c.i0 + threadIdx.x;
    const double ax = slice_row<double>(a.rp, a.ci, a.v64, a.x, c.i0, c.i1, stage);
    double rr = 0.0;
    if (i < c.i1) {
        const double t = a.b[i] - ax;
        a.r64[i] = t;
        rr = t * t;
    }
    rr = block_reduce<kSliceThreads>(rr, sh);
    if (threadIdx.x == 0) st.part[2 * (size_t)blockIdx.x + 1] = rr;
}

// The test, a workgroup per system.
__global__ __launch_bounds__(kSliceThreads) void k_step_test(BatchArgs a, StepState st, int begin) {
    __shared__ double sh[kSliceThreads / 64];
    const uint32_t s = blockIdx.x;
    if (!begin && !st.active[s]) return;
    const double normb = begin ? sqrt(slice_sum(st, s, 0, sh)) : st.normb[s];
    const double rn = sqrt(slice_sum(st, s, 1, sh));
    if (threadIdx.x != 0) return;
    const int outer = begin ? 0 : a.outer[s] + 1;
    const uint32_t total = begin ? 0 : (uint32_t)a.iters[s];
    const double rel = normb > 0 ? rn / normb : 0.0;
    const bool done = rel < a.tol || !(rel == rel) || (uint32_t)outer >= a.max_outer || total >= a.maxit;
    a.iters[s] = (int32_t)total;
    a.outer[s] = outer;
    a.conv[s] = rel < a.tol;
    a.relres[s] = rel;
    st.active[s] = !done;
    st.normb[s] = normb;
    st.rn[s] = rn;
    st.want[s] = fmax(a.inner_tol, 0.5 * a.tol * normb / rn);
    st.left[s] = a.maxit - total;
    if (!done) *st.any = 1;
}

// rin and its squares' sum
__global__ __launch_bounds__(kSliceThreads) void k_step_scale(BatchArgs a, StepState st) {
    __shared__ double sh[kSliceThreads / 64];
    const Slice c = st.slices[blockIdx.x];
    if (!st.active[c.sys]) return;
    const float sc = (float)(1.0 / st.rn[c.sys]);
    const uint32_t i = c.i0 + threadIdx.x;
    double bb = 0.0;
    if (i < c.i1) {
        const float v = (float)a.r64[i] * sc;
        a.r32[i] = v;
        bb = (double)v * (double)v;
    }
    bb = block_reduce<kSliceThreads>(bb, sh);
    if (threadIdx.x == 0) st.part[2 * (size_t)blockIdx.x] = bb;
}

// r = KF rin; a system's first slice also leaves ||rin||
__global__ __launch_bounds__(kSliceThreads) void k_step_rhs(BatchArgs a, StepState st) {
    __shared__ double sh[kSliceThreads / 64];
    __shared__ SliceStage<float> stage;
    const Slice c = st.slices[blockIdx.x];
    if (!st.active[c.sys]) return;
    const uint32_t m0 = max(c.i0, a.roff[c.sys] + a.red_n0[c.sys]);
    const float q = slice_row<float>(a.kfe_rp, a.kfe_ci, a.kfe_v, a.r32, m0, c.i1, stage);
    if (m0 + threadIdx.x < c.i1) a.q32[m0 + threadIdx.x] = q;
    if (blockIdx.x != st.first[c.sys]) return;
    const double nin = sqrt(slice_sum(st, c.sys, 0, sh));
    if (threadIdx.x == 0) st.rin_norm[c.sys] = nin;
}

}  // namespace
}  // namespace pp

// ============================================================================ host side
struct pp_batch {
    pp_ctx *ctx = nullptr;
    uint32_t nsys = 0, ntot = 0, nnz = 0;
    std::vector<uint32_t> h_roff, h_rp, h_ci;
    std::vector<double> h_v;
    uint32_t *roff = nullptr, *rp = nullptr, *ci = nullptr;
    double *v64 = nullptr;
    float *v32 = nullptr;
    pp::DevBatchSweep lo, up;
    double *r64 = nullptr, *rr64 = nullptr, *w64 = nullptr, *d64 = nullptr, *p64 = nullptr;
    float *r32 = nullptr, *e32 = nullptr, *q32 = nullptr, *w32 = nullptr, *d32 = nullptr, *p32 = nullptr;
    int32_t *iters = nullptr, *outer = nullptr, *conv = nullptr;
    double *relres = nullptr;
    int block = 256;
    bool symmetric = true;
    uint32_t max_levels = 0;
    // PP_ORDER_MULTICOLOR: every system is solved as P_s A_s P_s^T (rows
    // grouped by colour, so its IC(0) sweeps have one level per colour);
    // the kernel works on the permuted copy below, b and x are permuted once
    // per solve.  Position k of the permuted batch holds original row gperm[k];
    // permuted entry e holds original entry vmap[e].
    int ordering = PP_ORDER_NATURAL;
    std::vector<uint32_t> h_gperm, h_prp, h_pci, vmap;
    uint32_t *gperm = nullptr, *prp = nullptr, *pci = nullptr;
    double *pv64 = nullptr, *bp = nullptr, *xp = nullptr;
    float *pv32 = nullptr;
    // the reduced form of every system's two-colour IC(0) (multicolour order
    // only, and only when every system has the structure; see BatchArgs)
    uint32_t *red_n0 = nullptr, *kab_rp = nullptr, *kab_ci = nullptr, *kfe_rp = nullptr, *kfe_ci = nullptr;
    float *kab_v = nullptr, *kfe_v = nullptr, *red_s1 = nullptr, *red_dt = nullptr;
    // numeric re-factorization on the device (batch_refresh_build): where the
    // values of the permuted copy, of the sweeps and of the pivots come from
    int refresh = 0;  // 0 not built yet, 1 in use, -1 this batch factors on the host
    uint32_t *dvmap = nullptr, *pos = nullptr, *lo_src = nullptr, *dsrc = nullptr, *up_map = nullptr;
    uint32_t lo_nnz = 0;
    int *flag = nullptr;
    uint32_t device_refactors = 0;
    // the values before the last ones set, an array swapped with v64; after
    // values whose factorization failed: those of the factor still in use
    double *v64_before = nullptr;
    bool factor_before = false;
    bool h_v_stale = false;  // h_v predates the values in v64
    // the reduced form's tiles (batch_build_tiles); tile_width 0: none
    int tile_width = 0;
    uint32_t ntiles = 0, nslot = 0;
    pp::Tile *tiles = nullptr;
    uint32_t *tile_rows = nullptr, *tile_slots = nullptr;
    uint16_t *tile_loc = nullptr;
    unsigned long long *tile_w = nullptr, *tile_sums = nullptr;  // exchanged w, partial sums
    int32_t *active = nullptr;
    double *state = nullptr;   // want, rin_norm, rn, normb: nsys each
    uint32_t *left = nullptr;
    int *tile_flag = nullptr;  // any, abort
    pp::Slice *slices = nullptr;   // of the refinement steps' rows
    uint32_t *slice0 = nullptr, nslice = 0;
    double *slice_sums = nullptr;
};

namespace pp {
namespace {

// ---------------------------------------------------------------------------
// New values on a known pattern, factored on the device: one workgroup per
// system, every row's operations those of the host construction in its order
// (factor_ic0, reduced_host), so the factor and the reduced operators are the
// same bit for bit.  Bound by a workgroup's load latency (each row merges
// short rows of the factor): 256 systems of 32^2 to 256^2 rows take 1.6 ms,
// against 0.31 s for the host's factorization and its uploads.
// ---------------------------------------------------------------------------
constexpr int kRefreshThreads = 1024;

// pos[row] = position of the row in the forward sweep; flag |= 1 when a row of
// the matrix is not strictly ascending or lacks its diagonal
__global__ __launch_bounds__(256) void k_batch_rows(uint32_t n, const uint32_t *__restrict__ perm,
                                                    const uint32_t *__restrict__ rp, const uint32_t *__restrict__ ci,
                                                    uint32_t *pos, uint32_t *dsrc, int *flag) {
    const uint32_t k = blockIdx.x * 256 + threadIdx.x;
    if (k >= n) return;
    pos[perm[k]] = k;
    uint32_t d = UINT32_MAX;
    bool good = true;
    for (uint32_t e = rp[k]; e < rp[k + 1]; ++e) {
        if (e > rp[k]) good = good && ci[e - 1] < ci[e];
        if (ci[e] == k) d = e;
    }
    dsrc[k] = d;
    if (!good || d == UINT32_MAX) atomicOr(flag, 1);
}

// lo_src: the matrix entry each entry of L starts from; up_map: the entry of
// L each entry of the backward sweep holds; flag |= 2 when one is missing or
// a row of L is not ascending
__global__ __launch_bounds__(256) void k_batch_maps(uint32_t n, DevBatchSweep lo, DevBatchSweep up,
                                                    const uint32_t *__restrict__ rp, const uint32_t *__restrict__ ci,
                                                    const uint32_t *__restrict__ pos, uint32_t *lo_src,
                                                    uint32_t *up_map, int *flag) {
    const uint32_t k = blockIdx.x * 256 + threadIdx.x;
    if (k >= n) return;
    bool good = true;
    {
        const uint32_t i = lo.perm[k];
        uint32_t e = rp[i];
        for (uint32_t t = lo.rp[k]; t < lo.rp[k + 1]; ++t) {
            const uint32_t c = lo.ci[t];
            if (t > lo.rp[k]) good = good && lo.ci[t - 1] < c;
            while (e < rp[i + 1] && ci[e] < c) ++e;
            const bool found = e < rp[i + 1] && ci[e] == c;
            lo_src[t] = found ? e : 0;
            good = good && found;
        }
    }
    {
        const uint32_t j = up.perm[k];
        for (uint32_t t = up.rp[k]; t < up.rp[k + 1]; ++t) {
            const uint32_t q = pos[up.ci[t]];
            uint32_t u = lo.rp[q];
            while (u < lo.rp[q + 1] && lo.ci[u] != j) ++u;
            const bool found = u < lo.rp[q + 1];
            up_map[t] = found ? u : 0;
            good = good && found;
        }
    }
    if (!good) atomicOr(flag, 2);
}

// out64[e] = in[map ? map[e] : e], out32 the same rounded; out64 may be null
__global__ __launch_bounds__(256) void k_batch_values(uint32_t n, const uint32_t *__restrict__ map,
                                                      const double *__restrict__ in, double *out64, float *out32) {
    for (uint32_t e = blockIdx.x * 256 + threadIdx.x; e < n; e += gridDim.x * 256) {
        const double v = in[map ? map[e] : e];
        if (out64) out64[e] = v;
        out32[e] = (float)v;
    }
}

struct RefreshArgs {
    const uint32_t *roff, *rp, *ci;  // the (permuted) matrix
    const double *av;
    DevBatchSweep lo, up;
    const uint32_t *pos, *lo_src, *dsrc, *up_map;
    const uint32_t *red_n0, *kab_rp, *kfe_rp;  // red_n0 null: no reduced form
    float *kab_v, *kfe_v, *red_s1, *red_dt;
    double *dt;   // work, by row
    int *flag;    // |= 4: a pivot is not positive (the host reports it)
};

__global__ __launch_bounds__(kRefreshThreads) void k_batch_refresh(RefreshArgs a) {
#pragma clang fp contract(off)
    const uint32_t s = blockIdx.x, r0 = a.roff[s], r1 = a.roff[s + 1];
    double *lv = a.lo.val64, *dg = a.lo.diag64;
    bool good = true;
    for (uint32_t l = a.lo.lev_off[s]; l + 1 < a.lo.lev_off[s + 1]; ++l) {
        for (uint32_t k = a.lo.lev[l] + threadIdx.x; k < a.lo.lev[l + 1]; k += kRefreshThreads) {
            const uint32_t i = a.lo.perm[k], i0 = a.lo.rp[k], i1 = a.lo.rp[k + 1];
            double sq = a.av[a.dsrc[i]];
            for (uint32_t t = i0; t < i1; ++t) {
                const uint32_t c = a.lo.ci[t], q = a.pos[c];
                double v = a.av[a.lo_src[t]];
                uint32_t p = i0;
                for (uint32_t u = a.lo.rp[q]; u < a.lo.rp[q + 1]; ++u) {
                    const uint32_t cu = a.lo.ci[u];
                    while (p < t && a.lo.ci[p] < cu) ++p;
                    if (p < t && a.lo.ci[p] == cu) v -= lv[p] * lv[u];
                }
                v = v / dg[c];
                lv[t] = v;
                a.lo.val32[t] = (float)v;
            }
            for (uint32_t t = i0; t < i1; ++t) sq -= lv[t] * lv[t];
            good = good && sq > 0.0;
            const double d = sqrt(sq > 0.0 ? sq : 1.0);
            dg[i] = d;
            a.lo.diag32[i] = (float)d;
            a.up.diag64[i] = d;
            a.up.diag32[i] = (float)d;
        }
        __syncthreads();
    }
    // the backward sweep's entries (positions r0 .. r1 are this system's)
    for (uint32_t t = a.up.rp[r0] + threadIdx.x; t < a.up.rp[r1]; t += kRefreshThreads) {
        const double v = lv[a.up_map[t]];
        a.up.val64[t] = v;
        a.up.val32[t] = (float)v;
    }
    if (a.red_n0) {
        const uint32_t m0 = r0 + a.red_n0[s];
        for (uint32_t i = r0 + threadIdx.x; i < r1; i += kRefreshThreads) {
            const double d = a.av[a.dsrc[i]];
            good = good && d > 0.0;
            if (i < m0) continue;
            double t = d;
            for (uint32_t k = a.rp[i]; k < a.rp[i + 1]; ++k) {
                const uint32_t c = a.ci[k];
                if (c < m0) t -= a.av[k] * a.av[k] / a.av[a.dsrc[c]];
            }
            a.dt[i] = t;
            good = good && t > 0.0 && isfinite(t);
        }
        __syncthreads();
        for (uint32_t i = r0 + threadIdx.x; i < r1; i += kRefreshThreads) {
            const double d = a.av[a.dsrc[i]];
            uint32_t p = a.kab_rp[i], q = a.kfe_rp[i];
            if (i < m0) {
                a.kfe_v[q++] = (float)(1.0 / d);
                for (uint32_t k = a.rp[i]; k < a.rp[i + 1]; ++k) {
                    const uint32_t j = a.ci[k];
                    if (j == i) continue;
                    a.kab_v[p++] = (float)(a.av[k] / sqrt(d * a.dt[j]));
                    a.kfe_v[q++] = (float)(-a.av[k] / d);
                }
            } else {
                const double t = a.dt[i], rs = 1.0 / sqrt(t);
                for (uint32_t k = a.rp[i]; k < a.rp[i + 1]; ++k) {
                    const uint32_t j = a.ci[k];
                    if (j == i) continue;
                    const double dj = a.av[a.dsrc[j]];
                    a.kab_v[p++] = (float)(-a.av[k] / sqrt(dj * t));
                    a.kfe_v[q++] = (float)(-a.av[k] / dj * rs);
                }
                a.kab_v[p] = (float)(d / t);
                a.kfe_v[q] = (float)rs;
                a.red_s1[i] = (float)rs;
                a.red_dt[i] = (float)t;
            }
        }
    }
    if (!good) atomicOr(a.flag, 4);
}

struct HostBatchSweep {
    std::vector<uint32_t> perm, rp{0}, ci, lev, lev_off{0};
    std::vector<double> val, diag;
};

// Append the gather-form sweep of one system (local CSR `R`, rows offset by
// goff): rows grouped by dependency level, dependencies in storage order.
void append_sweep(HostBatchSweep &H, const HostCsr &R, bool lower, bool diag_first_in_row, uint32_t goff,
                  uint32_t &nlev_out) {
    const uint32_t n = R.n;
    std::vector<uint32_t> lev(n, 0), rp(n + 1, 0), ci;
    std::vector<double> val, dg(n, 1.0);
    for (uint32_t i = 0; i < n; ++i) {
        for (uint32_t k = R.rp[i]; k < R.rp[i + 1]; ++k) {
            if (R.ci[k] == i) {
                dg[i] = R.v[k];
                continue;
            }
            ci.push_back(R.ci[k]);
            val.push_back(R.v[k]);
        }
        rp[i + 1] = (uint32_t)ci.size();
    }
    (void)diag_first_in_row;
    uint32_t maxl = 0;
    auto visit = [&](uint32_t i) {
        uint32_t l = 0;
        for (uint32_t k = rp[i]; k < rp[i + 1]; ++k) l = std::max(l, lev[ci[k]] + 1);
        lev[i] = l;
        maxl = std::max(maxl, l);
    };
    if (lower)
        for (uint32_t i = 0; i < n; ++i) visit(i);
    else
        for (uint32_t i = n; i-- > 0;) visit(i);
    const uint32_t nlev = n ? maxl + 1 : 0;
    std::vector<uint32_t> lp(nlev + 1, 0);
    for (uint32_t i = 0; i < n; ++i) lp[lev[i] + 1]++;
    for (uint32_t l = 0; l < nlev; ++l) lp[l + 1] += lp[l];
    std::vector<uint32_t> fill(lp.begin(), lp.end() - (nlev ? 1 : 0)), perm(n);
    for (uint32_t i = 0; i < n; ++i) perm[fill[lev[i]]++] = i;
    const uint32_t base = (uint32_t)H.perm.size();
    for (uint32_t q = 0; q < n; ++q) {
        const uint32_t i = perm[q];
        H.perm.push_back(goff + i);
        for (uint32_t k = rp[i]; k < rp[i + 1]; ++k) {
            H.ci.push_back(goff + ci[k]);
            H.val.push_back(val[k]);
        }
        H.rp.push_back((uint32_t)H.ci.size());
    }
    for (uint32_t l = 0; l <= nlev; ++l) H.lev.push_back(base + lp[l]);
    H.lev_off.push_back((uint32_t)H.lev.size());
    H.diag.insert(H.diag.end(), dg.begin(), dg.end());
    nlev_out = nlev;
}

// Concatenate a part built by append_sweep into an empty HostBatchSweep
// onto H (positions, entry offsets and level pointers shifted).
void append_parts(HostBatchSweep &H, const HostBatchSweep &P) {
    const uint32_t bp = (uint32_t)H.perm.size(), be = (uint32_t)H.ci.size(), bl = (uint32_t)H.lev.size();
    H.perm.insert(H.perm.end(), P.perm.begin(), P.perm.end());
    H.ci.insert(H.ci.end(), P.ci.begin(), P.ci.end());
    H.val.insert(H.val.end(), P.val.begin(), P.val.end());
    H.diag.insert(H.diag.end(), P.diag.begin(), P.diag.end());
    for (size_t q = 1; q < P.rp.size(); ++q) H.rp.push_back(be + P.rp[q]);
    for (uint32_t l : P.lev) H.lev.push_back(bp + l);
    for (size_t q = 1; q < P.lev_off.size(); ++q) H.lev_off.push_back(bl + P.lev_off[q]);
}

template <class T>
T *upload(const std::vector<T> &h) {
    T *d = dalloc<T>(h.size());
    if (!h.empty()) PP_HIP(hipMemcpy(d, h.data(), h.size() * sizeof(T), hipMemcpyHostToDevice));
    return d;
}

std::vector<float> to_f32(const std::vector<double> &v) { return std::vector<float>(v.begin(), v.end()); }

void upload_batch_sweep(const HostBatchSweep &H, DevBatchSweep &D) {
    D.free_all();
    D.perm = upload(H.perm);
    D.rp = upload(H.rp);
    D.ci = upload(H.ci);
    D.val64 = upload(H.val);
    D.val32 = upload(to_f32(H.val));
    D.diag64 = upload(H.diag);
    D.diag32 = upload(to_f32(H.diag));
    D.lev = upload(H.lev);
    D.lev_off = upload(H.lev_off);
}

// The permuted pattern of every system (multicolour order within each
// diagonal block) and the entry map; values follow through vmap.
void batch_build_order(pp_batch *B) {
    B->h_gperm.assign(B->ntot, 0);
    B->h_prp.assign(B->ntot + 1, 0);
    B->h_pci.assign(B->nnz, 0);
    B->vmap.assign(B->nnz, 0);
    // a system's permuted entries occupy the same range as its original ones
    parallel_for(B->nsys, 1, [&](size_t s0, size_t s1) {
        std::vector<std::pair<uint32_t, uint32_t>> row;  // (new column, original entry)
        for (size_t s = s0; s < s1; ++s) {
            const uint32_t r0 = B->h_roff[s], r1 = B->h_roff[s + 1], n = r1 - r0;
            HostCsr A;
            A.n = n;
            A.rp.assign(n + 1, 0);
            for (uint32_t i = 0; i < n; ++i) A.rp[i + 1] = B->h_rp[r0 + i + 1] - B->h_rp[r0];
            A.ci.resize(A.rp[n]);
            A.v.assign(A.rp[n], 0.0);
            for (uint32_t k = 0; k < A.rp[n]; ++k) A.ci[k] = B->h_ci[B->h_rp[r0] + k] - r0;
            uint32_t ncol = 0;
            const std::vector<uint32_t> order = multicolor_order(A, ncol);
            std::vector<uint32_t> inv(n);
            for (uint32_t k = 0; k < n; ++k) inv[order[k]] = k;
            uint32_t q = B->h_rp[r0];
            for (uint32_t k = 0; k < n; ++k) {
                const uint32_t i = order[k];
                B->h_gperm[r0 + k] = r0 + i;
                row.clear();
                for (uint32_t e = B->h_rp[r0 + i]; e < B->h_rp[r0 + i + 1]; ++e)
                    row.emplace_back(inv[B->h_ci[e] - r0], e);
                std::sort(row.begin(), row.end());
                for (const auto &pe : row) {
                    B->h_pci[q] = r0 + pe.first;
                    B->vmap[q++] = pe.second;
                }
                B->h_prp[r0 + k + 1] = q;
            }
        }
    });
}

// values of the permuted copy from the original values
void batch_upload_permuted_values(pp_batch *B) {
    std::vector<double> pv(B->nnz);
    parallel_for(B->nnz, 1u << 16, [&](size_t e0, size_t e1) {
        for (size_t e = e0; e < e1; ++e) pv[e] = B->h_v[B->vmap[e]];
    });
    if (!B->pv64) B->pv64 = dalloc<double>(B->nnz);
    if (!B->pv32) B->pv32 = dalloc<float>(B->nnz);
    PP_HIP(hipMemcpy(B->pv64, pv.data(), B->nnz * sizeof(double), hipMemcpyHostToDevice));
    const std::vector<float> p32 = to_f32(pv);
    PP_HIP(hipMemcpy(B->pv32, p32.data(), B->nnz * sizeof(float), hipMemcpyHostToDevice));
}

void batch_free_reduced(pp_batch *B) {
    dfree(B->red_n0); dfree(B->kab_rp); dfree(B->kab_ci); dfree(B->kfe_rp); dfree(B->kfe_ci);
    dfree(B->kab_v); dfree(B->kfe_v); dfree(B->red_s1); dfree(B->red_dt);
    B->red_n0 = B->kab_rp = B->kab_ci = B->kfe_rp = B->kfe_ci = nullptr;
    B->kab_v = B->kfe_v = B->red_s1 = B->red_dt = nullptr;
}

// The systems' reduced operators in batch numbering (FP32 values: they run
// only in the mixed solves' inner iterations).
void batch_upload_reduced(pp_batch *B, const std::vector<ReducedHost> &reds) {
    const uint32_t ns = B->nsys, nt = B->ntot;
    std::vector<uint32_t> n0(ns), ab_rp(nt + 1, 0), fe_rp(nt + 1, 0);
    for (uint32_t s = 0; s < ns; ++s) {
        const ReducedHost &H = reds[s];
        const uint32_t r0 = B->h_roff[s];
        n0[s] = H.n0;
        for (uint32_t i = 0; i < H.n0; ++i) {
            ab_rp[r0 + i + 1] = ab_rp[r0 + i] + (H.ka_rp[i + 1] - H.ka_rp[i]);
            fe_rp[r0 + i + 1] = fe_rp[r0 + i] + (H.ke_rp[i + 1] - H.ke_rp[i]);
        }
        for (uint32_t q = 0; q < H.n1; ++q) {
            const uint32_t i = r0 + H.n0 + q;
            ab_rp[i + 1] = ab_rp[i] + (H.kb_rp[q + 1] - H.kb_rp[q]);
            fe_rp[i + 1] = fe_rp[i] + (H.kf_rp[q + 1] - H.kf_rp[q]);
        }
    }
    std::vector<uint32_t> ab_ci(ab_rp[nt]), fe_ci(fe_rp[nt]);
    std::vector<float> ab_v(ab_rp[nt]), fe_v(fe_rp[nt]), s1(nt, 0.f), dt(nt, 0.f);
    parallel_for(ns, 1, [&](size_t s0, size_t s1e) {
        for (size_t s = s0; s < s1e; ++s) {
            const ReducedHost &H = reds[s];
            const uint32_t r0 = B->h_roff[s];
            auto put = [&](const std::vector<uint32_t> &rp, const std::vector<uint32_t> &ci,
                           const std::vector<double> &v, uint32_t rows, uint32_t row0, const std::vector<uint32_t> &grp,
                           std::vector<uint32_t> &gci, std::vector<float> &gv) {
                for (uint32_t i = 0; i < rows; ++i)
                    for (uint32_t k = rp[i], q = grp[row0 + i]; k < rp[i + 1]; ++k, ++q) {
                        gci[q] = r0 + ci[k];
                        gv[q] = (float)v[k];
                    }
            };
            put(H.ka_rp, H.ka_ci, H.ka_v, H.n0, r0, ab_rp, ab_ci, ab_v);
            put(H.kb_rp, H.kb_ci, H.kb_v, H.n1, r0 + H.n0, ab_rp, ab_ci, ab_v);
            put(H.ke_rp, H.ke_ci, H.ke_v, H.n0, r0, fe_rp, fe_ci, fe_v);
            put(H.kf_rp, H.kf_ci, H.kf_v, H.n1, r0 + H.n0, fe_rp, fe_ci, fe_v);
            for (uint32_t q = 0; q < H.n1; ++q) {
                s1[r0 + H.n0 + q] = (float)H.s1[q];
                dt[r0 + H.n0 + q] = (float)H.dt[q];
            }
        }
    });
    B->red_n0 = upload(n0);
    B->kab_rp = upload(ab_rp);
    B->kab_ci = upload(ab_ci);
    B->kab_v = upload(ab_v);
    B->kfe_rp = upload(fe_rp);
    B->kfe_ci = upload(fe_ci);
    B->kfe_v = upload(fe_v);
    B->red_s1 = upload(s1);
    B->red_dt = upload(dt);
}

void batch_free_refresh(pp_batch *B) {
    dfree(B->dvmap); dfree(B->pos); dfree(B->lo_src); dfree(B->dsrc); dfree(B->up_map); dfree(B->flag);
    B->dvmap = B->pos = B->lo_src = B->dsrc = B->up_map = nullptr;
    B->flag = nullptr;
    B->refresh = 0;
}

void batch_free_tiles(pp_batch *B) {
    dfree(B->tiles); dfree(B->tile_rows); dfree(B->tile_slots); dfree(B->tile_loc); dfree(B->tile_w);
    dfree(B->tile_sums); dfree(B->active); dfree(B->state); dfree(B->left); dfree(B->tile_flag);
    dfree(B->slices); dfree(B->slice0); dfree(B->slice_sums);
    B->slices = nullptr;
    B->slice0 = nullptr;
    B->slice_sums = nullptr;
    B->nslice = 0;
    B->tiles = nullptr;
    B->tile_rows = B->tile_slots = B->left = nullptr;
    B->tile_loc = nullptr;
    B->tile_w = B->tile_sums = nullptr;
    B->active = nullptr;
    B->state = nullptr;
    B->tile_flag = nullptr;
    B->tile_width = 0;
    B->ntiles = B->nslot = 0;
}

// The tiles of one system: its second-colour rows cut into ntile ranges.
struct SystemTiles {
    std::vector<Tile> tiles;               // f, h, ka, kb, out relative to the vectors below
    std::vector<uint32_t> rows;            // F's rows and the halo's
    std::vector<uint32_t> slots;           // halo: the row, to be replaced by its slot; owned: kNoSlot or the slot
    std::vector<uint16_t> loc;
    uint32_t nslot = 0;
    bool fits = false;
};

SystemTiles tiles_of_system(const ReducedHost &H, uint32_t r0, int W, uint32_t ntile, uint32_t maxf, uint32_t maxs,
                            uint32_t maxh) {
    SystemTiles T;
    const uint32_t n0 = H.n0, n1 = H.n1;
    std::vector<uint32_t> fpos(n0, kNoSlot), rpos(n1, kNoSlot), slot(n1, kNoSlot);
    // rows exported: those some other tile reads (numbered after the tiles are known)
    std::vector<uint8_t> exported(n1, 0);
    for (uint32_t k = 0; k < ntile; ++k) {
        const uint32_t q0 = (uint32_t)((uint64_t)n1 * k / ntile), q1 = (uint32_t)((uint64_t)n1 * (k + 1) / ntile);
        Tile t{};
        t.row0 = r0 + n0 + q0;
        t.ns = q1 - q0;
        t.f = (uint32_t)T.rows.size();
        std::vector<uint32_t> F, R;
        for (uint32_t q = q0; q < q1; ++q)
            for (uint32_t e = H.kb_rp[q]; e + 1 < H.kb_rp[q + 1]; ++e)
                if (fpos[H.kb_ci[e]] == kNoSlot) {
                    fpos[H.kb_ci[e]] = 0;
                    F.push_back(H.kb_ci[e]);
                }
        std::sort(F.begin(), F.end());
        for (uint32_t f = 0; f < F.size(); ++f) fpos[F[f]] = f;
        for (uint32_t q = q0; q < q1; ++q) rpos[q] = q - q0;
        for (uint32_t i : F)
            for (uint32_t e = H.ka_rp[i]; e < H.ka_rp[i + 1]; ++e) {
                const uint32_t q = H.ka_ci[e] - n0;
                if (rpos[q] == kNoSlot) {
                    rpos[q] = t.ns + (uint32_t)R.size();
                    R.push_back(q);
                    exported[q] = 1;
                }
            }
        t.nf = (uint32_t)F.size();
        t.nh = (uint32_t)R.size();
        if (t.nf > maxf || t.ns > maxs || t.nh > maxh) return T;
        t.ka = (uint32_t)T.loc.size();
        T.loc.resize(T.loc.size() + (size_t)W * t.nf, 0);
        for (uint32_t f = 0; f < t.nf; ++f)
            for (uint32_t e = H.ka_rp[F[f]], j = 0; e < H.ka_rp[F[f] + 1]; ++e, ++j)
                T.loc[t.ka + (size_t)j * t.nf + f] = (uint16_t)rpos[H.ka_ci[e] - n0];
        t.kb = (uint32_t)T.loc.size();
        T.loc.resize(T.loc.size() + (size_t)W * t.ns, 0);
        for (uint32_t q = q0; q < q1; ++q)
            for (uint32_t e = H.kb_rp[q], j = 0; e + 1 < H.kb_rp[q + 1]; ++e, ++j)
                T.loc[t.kb + (size_t)j * t.ns + (q - q0)] = (uint16_t)fpos[H.kb_ci[e]];
        for (uint32_t i : F) T.rows.push_back(r0 + i);
        for (uint32_t q : R) T.rows.push_back(r0 + n0 + q);
        t.h = (uint32_t)T.slots.size();
        for (uint32_t q : R) T.slots.push_back(q);
        t.out = (uint32_t)T.slots.size();
        for (uint32_t q = q0; q < q1; ++q) T.slots.push_back(q);
        for (uint32_t i : F) fpos[i] = kNoSlot;
        for (uint32_t q : R) rpos[q] = kNoSlot;
        for (uint32_t q = q0; q < q1; ++q) rpos[q] = kNoSlot;
        T.tiles.push_back(t);
    }
    for (uint32_t q = 0; q < n1; ++q)
        if (exported[q]) slot[q] = T.nslot++;
    for (uint32_t &v : T.slots) v = slot[v];
    T.fits = true;
    return T;
}

// The tiles of every system (largest first), when all their rows are short
// enough: rows of at most 4 or 6 off-diagonal entries (5- and 7-point
// stencils).  Two tiles of kS * kTileThreads rows fill a unit's registers;
// batches that would leave units idle take tiles down to 1024 rows (smaller
// ones wait on one another more than they compute: 24 systems of 60^2 to
// 200^2 2.9 ms with 512 rows, 2.5 with 1024).  false (nothing kept): a system
// does not fit, or all are small.
bool batch_build_tiles(pp_batch *B, const std::vector<ReducedHost> &reds) {
    batch_free_tiles(B);
    const uint32_t ns = B->nsys;
    uint32_t width = 1;
    for (const ReducedHost &H : reds) {
        for (uint32_t i = 0; i < H.n0; ++i) width = std::max(width, H.ka_rp[i + 1] - H.ka_rp[i]);
        for (uint32_t q = 0; q < H.n1; ++q) width = std::max(width, H.kb_rp[q + 1] - H.kb_rp[q] - 1);
    }
    if (width > 6) return false;
    for (uint32_t i = 0; i < B->ntot; ++i)  // a row's diagonal beside them (k_step_*)
        if (B->h_prp[i + 1] - B->h_prp[i] > kSliceWidth) return false;
    for (const ReducedHost &H : reds) {
        for (uint32_t i = 0; i < H.n0; ++i)
            if (H.ke_rp[i + 1] - H.ke_rp[i] > kSliceWidth) return false;
        for (uint32_t q = 0; q < H.n1; ++q)
            if (H.kf_rp[q + 1] - H.kf_rp[q] > kSliceWidth) return false;
    }
    const int W = width <= 4 ? 4 : 6;
    // Small systems stay with k_batch_pcg, one launch for the whole solve: the
    // refinement steps' launches and waits take 170 us more than it does, and an
    // iteration saves only as the largest system grows.  16 (1000) equal systems,
    // us a solve in k_batch_pcg and over tiles: 5-point 22^2 380, 422 (601, 692);
    // 24^2 451, 440 (788, 754) and 389, 417 (688, 704) with constant
    // coefficients; 26^2 479, 459 (938, 793).  7-point 9^3 290, 341 (627, 539),
    // 10^3 324, 351 (782, 599), 11^3 409, 391 (1156, 693).
    uint32_t largest = 0;
    for (const ReducedHost &H : reds) largest = std::max(largest, H.n0 + H.n1);
    if (largest < (W == 4 ? 600u : 1100u)) return false;
    const uint32_t maxf = kTileThreads * (W == 4 ? TileShape<4>::kF : TileShape<6>::kF);
    const uint32_t maxs = kTileThreads * (W == 4 ? TileShape<4>::kS : TileShape<6>::kS);
    const uint32_t maxh = kTileThreads * (W == 4 ? TileShape<4>::kH : TileShape<6>::kH);
    const auto count = [&](uint32_t cap) {
        uint64_t c = 0;
        for (const ReducedHost &H : reds) c += std::max(1u, (H.n1 + cap - 1) / cap);
        return c;
    };
    // a system's tiles wait for one another, so all of them must run at a time
    const uint32_t max_tiles = (uint32_t)B->ctx->cu_count;
    uint32_t cap = maxs;
    while (cap > 1024 && count(cap / 2) <= (uint64_t)B->ctx->cu_count) cap /= 2;
    std::vector<SystemTiles> T(ns);
    std::atomic<bool> fits{true};
    parallel_for(ns, 1, [&](size_t s0, size_t s1) {
        for (size_t s = s0; s < s1 && fits; ++s) {
            uint32_t nt = std::max(1u, (reds[s].n1 + cap - 1) / cap);
            for (;; nt += std::max(1u, nt / 4)) {  // more tiles until F and the halo fit
                T[s] = tiles_of_system(reds[s], B->h_roff[s], W, nt, maxf, maxs, maxh);
                if (T[s].fits) break;
                if (nt > max_tiles || nt > reds[s].n1) break;
            }
            if (!T[s].fits || nt > max_tiles) fits = false;
        }
    });
    if (!fits) return false;
    std::vector<uint32_t> order(ns);
    for (uint32_t s = 0; s < ns; ++s) order[s] = s;
    std::stable_sort(order.begin(), order.end(), [&](uint32_t x, uint32_t y) { return reds[x].n1 > reds[y].n1; });
    std::vector<Tile> tiles;
    std::vector<uint32_t> rows, slots;
    std::vector<uint16_t> loc;
    uint32_t nslot = 0;
    for (uint32_t s : order) {
        SystemTiles &q = T[s];
        const uint32_t tile0 = (uint32_t)tiles.size();
        for (Tile t : q.tiles) {
            t.sys = s;
            t.tile0 = tile0;
            t.ntile = (uint32_t)q.tiles.size();
            t.f += (uint32_t)rows.size();
            t.h += (uint32_t)slots.size();
            t.out += (uint32_t)slots.size();
            t.ka += (uint32_t)loc.size();
            t.kb += (uint32_t)loc.size();
            tiles.push_back(t);
        }
        rows.insert(rows.end(), q.rows.begin(), q.rows.end());
        for (uint32_t v : q.slots) slots.push_back(v == kNoSlot ? kNoSlot : v + nslot);
        loc.insert(loc.end(), q.loc.begin(), q.loc.end());
        nslot += q.nslot;
    }
    auto up = [](const void *src, size_t bytes) {
        unsigned char *d = dalloc<unsigned char>(std::max<size_t>(16, bytes));
        if (bytes) PP_HIP(hipMemcpy(d, src, bytes, hipMemcpyHostToDevice));
        return d;
    };
    B->tiles = (Tile *)up(tiles.data(), tiles.size() * sizeof(Tile));
    B->tile_rows = upload(rows);
    B->tile_slots = upload(slots);
    B->tile_loc = (uint16_t *)up(loc.data(), loc.size() * 2);
    B->ntiles = (uint32_t)tiles.size();
    B->nslot = nslot;
    B->tile_w = dalloc<unsigned long long>(2 * (size_t)std::max(1u, nslot));
    B->tile_sums = dalloc<unsigned long long>(12 * (size_t)B->ntiles);
    B->active = dalloc<int>(ns);
    B->state = dalloc<double>(4 * (size_t)ns);
    B->left = dalloc<uint32_t>(ns);
    B->tile_flag = dalloc<int>(2);
    std::vector<Slice> slices;
    std::vector<uint32_t> slice0;
    for (uint32_t s = 0; s < ns; ++s) {
        slice0.push_back((uint32_t)slices.size());
        for (uint32_t i = B->h_roff[s]; i < B->h_roff[s + 1]; i += kSliceRows)
            slices.push_back({s, i, std::min(B->h_roff[s + 1], i + kSliceRows)});
    }
    slice0.push_back((uint32_t)slices.size());
    B->slices = (Slice *)up(slices.data(), slices.size() * sizeof(Slice));
    B->slice0 = upload(slice0);
    B->nslice = (uint32_t)slices.size();
    B->slice_sums = dalloc<double>(2 * slices.size());
    B->tile_width = W;
    return true;
}

// IC(0) of every diagonal block (of the permuted copy under multicolour
// ordering), as two gather-form sweeps.
void batch_factor(pp_batch *B) {
    const bool perm = B->ordering == PP_ORDER_MULTICOLOR;
    const std::vector<uint32_t> &Rp = perm ? B->h_prp : B->h_rp;
    const std::vector<uint32_t> &Ci = perm ? B->h_pci : B->h_ci;
    std::vector<HostBatchSweep> los(B->nsys), ups(B->nsys);
    std::vector<uint32_t> nlev(B->nsys, 0), fail_row(B->nsys, 0);
    std::vector<int> status(B->nsys, PP_OK);
    std::vector<ReducedHost> reds(perm ? B->nsys : 0);
    std::atomic<bool> red_ok{perm};
    // systems factor independently; their sweeps are concatenated in order
    parallel_for(B->nsys, 1, [&](size_t s0, size_t s1) {
        for (size_t s = s0; s < s1; ++s) {
            const uint32_t r0 = B->h_roff[s], r1 = B->h_roff[s + 1], n = r1 - r0;
            HostCsr A;
            A.n = n;
            A.rp.assign(n + 1, 0);
            for (uint32_t i = 0; i < n; ++i) A.rp[i + 1] = Rp[r0 + i + 1] - Rp[r0];
            A.ci.resize(A.rp[n]);
            A.v.resize(A.rp[n]);
            for (uint32_t k = 0; k < A.rp[n]; ++k) {
                const uint32_t e = Rp[r0] + k;
                A.ci[k] = Ci[e] - r0;
                A.v[k] = B->h_v[perm ? B->vmap[e] : e];
            }
            HostCsr lt;
            status[s] = factor_ic0(A, lt, fail_row[s]);
            if (status[s] != PP_OK) continue;
            if (red_ok && !reduced_host(n, A.rp, A.ci, A.v, reds[s])) red_ok = false;
            const HostCsr L = transpose(lt);
            uint32_t nl = 0, nu = 0;
            append_sweep(los[s], L, true, false, r0, nl);
            append_sweep(ups[s], lt, false, true, r0, nu);
            nlev[s] = std::max(nl, nu);
        }
    });
    for (uint32_t s = 0; s < B->nsys; ++s)  // the first failing system, as a serial loop reports it
        if (status[s] != PP_OK)
            throw Error(status[s], "batch system " + std::to_string(s) + ": IC(0) pivot not positive at row " +
                                       std::to_string(fail_row[s]));
    HostBatchSweep lo, up;
    B->max_levels = 0;
    for (uint32_t s = 0; s < B->nsys; ++s) {
        append_parts(lo, los[s]);
        append_parts(up, ups[s]);
        B->max_levels = std::max(B->max_levels, nlev[s]);
    }
    B->factor_before = false;
    upload_batch_sweep(lo, B->lo);
    upload_batch_sweep(up, B->up);
    B->lo_nnz = (uint32_t)lo.ci.size();
    batch_free_refresh(B);  // its maps belong to the sweeps just replaced
    batch_free_reduced(B);
    batch_free_tiles(B);
    if (red_ok) {
        batch_upload_reduced(B, reds);
        batch_build_tiles(B, reds);
    }
}

void batch_ensure_host_values(pp_batch *B) {
    if (!B->h_v_stale) return;
    PP_HIP(hipMemcpy(B->h_v.data(), B->v64, B->nnz * sizeof(double), hipMemcpyDeviceToHost));
    B->h_v_stale = false;
}

int read_flag(pp_batch *B) {
    int f = 0;
    PP_HIP(hipMemcpyAsync(&f, B->flag, sizeof(int), hipMemcpyDeviceToHost, B->ctx->stream));
    PP_HIP(hipStreamSynchronize(B->ctx->stream));
    return f;
}

// The maps of the device re-factorization, from the sweeps and operators of
// the batch's last host factorization.  Batches whose rows are not sorted or
// lack a diagonal, and colour-ordered ones without the reduced form (whose
// host construction looks at the values again), keep the host factorization.
void batch_refresh_build(pp_batch *B) {
    pp_ctx *ctx = B->ctx;
    const bool perm = B->ordering == PP_ORDER_MULTICOLOR;
    B->refresh = -1;
    if (perm && !B->red_n0) return;
    const uint32_t n = B->ntot, g = (n + 255) / 256;
    const uint32_t *rp = perm ? B->prp : B->rp, *ci = perm ? B->pci : B->ci;
    if (!n) return;
    if (perm) B->dvmap = upload(B->vmap);
    B->pos = dalloc<uint32_t>(n);
    B->dsrc = dalloc<uint32_t>(n);
    B->lo_src = dalloc<uint32_t>(std::max(1u, B->lo_nnz));
    B->up_map = dalloc<uint32_t>(std::max(1u, B->lo_nnz));
    B->flag = dalloc<int>(1);
    launch_fill_zero(ctx, B->flag, sizeof(int));
    k_batch_rows<<<g, 256, 0, ctx->stream>>>(n, B->lo.perm, rp, ci, B->pos, B->dsrc, B->flag);
    k_batch_maps<<<g, 256, 0, ctx->stream>>>(n, B->lo, B->up, rp, ci, B->pos, B->lo_src, B->up_map, B->flag);
    PP_HIP(hipGetLastError());
    if (read_flag(B)) {
        batch_free_refresh(B);
        B->refresh = -1;
        return;
    }
    B->refresh = 1;
}

// the copies the solves multiply with, from the values v
void batch_refresh_values(pp_batch *B, const double *v) {
    pp_ctx *ctx = B->ctx;
    const unsigned g = std::max(1u, std::min<uint32_t>((B->nnz + 1023) / 1024, 16384u));
    k_batch_values<<<g, 256, 0, ctx->stream>>>(B->nnz, nullptr, v, nullptr, B->v32);
    if (B->ordering == PP_ORDER_MULTICOLOR)
        k_batch_values<<<g, 256, 0, ctx->stream>>>(B->nnz, B->dvmap, v, B->pv64, B->pv32);
    PP_HIP(hipGetLastError());
}

// Factors the values v on the device; false: a pivot is not positive.
bool batch_refresh(pp_batch *B, const double *v) {
    pp_ctx *ctx = B->ctx;
    const bool perm = B->ordering == PP_ORDER_MULTICOLOR;
    batch_refresh_values(B, v);
    RefreshArgs a;
    a.roff = B->roff;
    a.rp = perm ? B->prp : B->rp;
    a.ci = perm ? B->pci : B->ci;
    a.av = perm ? B->pv64 : v;
    a.lo = B->lo;
    a.up = B->up;
    a.pos = B->pos;
    a.lo_src = B->lo_src;
    a.dsrc = B->dsrc;
    a.up_map = B->up_map;
    a.red_n0 = perm ? B->red_n0 : nullptr;
    a.kab_rp = B->kab_rp;
    a.kfe_rp = B->kfe_rp;
    a.kab_v = B->kab_v;
    a.kfe_v = B->kfe_v;
    a.red_s1 = B->red_s1;
    a.red_dt = B->red_dt;
    a.dt = B->r64;  // a work vector of the solves
    a.flag = B->flag;
    launch_fill_zero(ctx, B->flag, sizeof(int));
    k_batch_refresh<<<B->nsys, kRefreshThreads, 0, ctx->stream>>>(a);
    PP_HIP(hipGetLastError());
    return read_flag(B) == 0;
}

BatchArgs make_args(pp_batch *B, const pp_solve_opts &o, const double *b, double *x) {
    BatchArgs a;
    std::memset(&a, 0, sizeof(a));
    a.nsys = B->nsys;
    a.roff = B->roff;
    const bool perm = B->ordering == PP_ORDER_MULTICOLOR;
    a.rp = perm ? B->prp : B->rp;
    a.ci = perm ? B->pci : B->ci;
    a.v64 = perm ? B->pv64 : B->v64;
    a.v32 = perm ? B->pv32 : B->v32;
    a.lo = B->lo;
    a.up = B->up;
    a.b = b;
    a.x = x;
    a.r64 = B->r64;
    a.r32 = B->r32; a.e32 = B->e32; a.q32 = B->q32; a.w32 = B->w32; a.d32 = B->d32; a.p32 = B->p32;
    a.rr64 = B->rr64; a.w64 = B->w64; a.d64 = B->d64; a.p64 = B->p64;
    a.tol = o.tol;
    a.inner_tol = o.inner_tol > 0 ? o.inner_tol : 1e-6;
    a.maxit = o.maxit;
    a.max_outer = o.max_outer ? o.max_outer : 20;
    a.red_n0 = perm ? B->red_n0 : nullptr;
    a.kab_rp = B->kab_rp;
    a.kab_ci = B->kab_ci;
    a.kab_v = B->kab_v;
    a.kfe_rp = B->kfe_rp;
    a.kfe_ci = B->kfe_ci;
    a.kfe_v = B->kfe_v;
    a.red_s1 = B->red_s1;
    a.red_dt = B->red_dt;
    a.iters = B->iters;
    a.outer = B->outer;
    a.conv = B->conv;
    a.relres = B->relres;
    return a;
}

void launch_batch(hipStream_t st, int block, bool mixed, const BatchArgs &a) {
    const unsigned g = a.nsys;
#define PP_BATCH_CASE(BS)                                                          \
    if (block == BS) {                                                             \
        if (mixed) k_batch_pcg<BS, true><<<g, BS, 0, st>>>(a);                      \
        else k_batch_pcg<BS, false><<<g, BS, 0, st>>>(a);                           \
        PP_HIP(hipGetLastError());                                                 \
        return;                                                                    \
    }
    PP_BATCH_CASE(256)
    PP_BATCH_CASE(512)
    PP_BATCH_CASE(1024)
#undef PP_BATCH_CASE
    throw Error(PP_ERR_INVALID, "batch workgroup size must be 256, 512 or 1024");
}

// The single persistent launch, captured into a graph and replayed.
void run_batch(pp_ctx *ctx, pp_batch *B, bool mixed, const BatchArgs &a) {
    Graph G;
    PP_HIP(hipStreamBeginCapture(ctx->stream, hipStreamCaptureModeThreadLocal));
    try {
        launch_batch(ctx->stream, B->block, mixed, a);
    } catch (...) {
        hipGraph_t tmp;
        (void)hipStreamEndCapture(ctx->stream, &tmp);
        if (tmp) (void)hipGraphDestroy(tmp);
        throw;
    }
    PP_HIP(hipStreamEndCapture(ctx->stream, &G.g));
    PP_HIP(hipGraphInstantiate(&G.exec, G.g, nullptr, nullptr, 0));
    PP_HIP(hipGraphLaunch(G.exec, ctx->stream));
    PP_HIP(hipStreamSynchronize(ctx->stream));
}

// The mixed solve over tiles: refinement steps until no system goes on;
// false: a tile gave up waiting.
bool run_tiles(pp_ctx *ctx, pp_batch *B, const BatchArgs &a) {
    const uint32_t ns = B->nsys;
    StepState st;
    st.slices = B->slices;
    st.first = B->slice0;
    st.part = B->slice_sums;
    st.active = B->active;
    st.want = B->state;
    st.rin_norm = B->state + ns;
    st.rn = B->state + 2 * (size_t)ns;
    st.normb = B->state + 3 * (size_t)ns;
    st.left = B->left;
    st.any = B->tile_flag;
    TileArgs t;
    t.tiles = B->tiles;
    t.rows = B->tile_rows;
    t.slots = B->tile_slots;
    t.loc = B->tile_loc;
    t.xw = B->tile_w;
    t.xp = B->tile_sums;
    t.nslot = B->nslot;
    t.ntiles = B->ntiles;
    t.abort = B->tile_flag + 1;
    t.deadline = ctx->spin_deadline;
    t.active = B->active;
    t.want = st.want;
    t.rin_norm = st.rin_norm;
    t.left = B->left;
    t.kab_rp = B->kab_rp;
    t.kab_v = B->kab_v;
    t.red_s1 = B->red_s1;
    t.red_dt = B->red_dt;
    t.z = B->q32;
    t.e = B->e32;
    t.iters = B->iters;
    for (int begin = 1;; begin = 0) {
        launch_fill_zero(ctx, B->tile_flag, (begin ? 2 : 1) * sizeof(int));  // the abort word stays
        k_step_correct<<<B->nslice, kSliceThreads, 0, ctx->stream>>>(a, st, begin);
        k_step_residual<<<B->nslice, kSliceThreads, 0, ctx->stream>>>(a, st, begin);
        k_step_test<<<ns, kSliceThreads, 0, ctx->stream>>>(a, st, begin);
        k_step_scale<<<B->nslice, kSliceThreads, 0, ctx->stream>>>(a, st);
        k_step_rhs<<<B->nslice, kSliceThreads, 0, ctx->stream>>>(a, st);
        PP_HIP(hipGetLastError());
        int flag[2];
        PP_HIP(hipMemcpyAsync(flag, B->tile_flag, sizeof(flag), hipMemcpyDeviceToHost, ctx->stream));
        PP_HIP(hipStreamSynchronize(ctx->stream));
        if (flag[1]) return false;
        if (!flag[0]) return true;
        launch_fill_zero(ctx, B->tile_w, 2 * (size_t)std::max(1u, B->nslot) * 8);
        launch_fill_zero(ctx, B->tile_sums, 12 * (size_t)B->ntiles * 8);
        if (B->tile_width == 4) k_tile_cg<4><<<B->ntiles, kTileThreads, 0, ctx->stream>>>(t);
        else k_tile_cg<6><<<B->ntiles, kTileThreads, 0, ctx->stream>>>(t);
        PP_HIP(hipGetLastError());
    }
}

void batch_free(pp_batch *B) {
    batch_free_tiles(B);
    dfree(B->roff); dfree(B->rp); dfree(B->ci); dfree(B->v64); dfree(B->v32); dfree(B->v64_before);
    B->lo.free_all();
    B->up.free_all();
    dfree(B->r64); dfree(B->rr64); dfree(B->w64); dfree(B->d64); dfree(B->p64);
    dfree(B->r32); dfree(B->e32); dfree(B->q32); dfree(B->w32); dfree(B->d32); dfree(B->p32);
    dfree(B->iters); dfree(B->outer); dfree(B->conv); dfree(B->relres);
    batch_free_refresh(B);
    dfree(B->gperm); dfree(B->prp); dfree(B->pci); dfree(B->pv64); dfree(B->pv32); dfree(B->bp); dfree(B->xp);
    batch_free_reduced(B);
}

}  // namespace
}  // namespace pp

using namespace pp;

template <class F>
static int guarded_batch(pp_ctx *ctx, F &&f) {
    try {
        PP_HIP(hipSetDevice(ctx->device));
        f();
        return PP_OK;
    } catch (const pp::Error &e) {
        ctx->err = e.what();
        return e.status;
    } catch (const std::exception &e) {
        ctx->err = e.what();
        return PP_ERR_INVALID;
    }
}

extern "C" {

int pp_batch_create(pp_ctx *ctx, uint32_t nsys, const uint32_t *row_off, const uint32_t *rowptr,
                    const uint32_t *colidx, const double *values, pp_batch **out) {
    if (!ctx) return PP_ERR_INVALID;
    return guarded_batch(ctx, [&] {
        PP_CHECK(nsys > 0 && row_off && rowptr && colidx && values && out, PP_ERR_INVALID, "NULL argument");
        PP_CHECK(row_off[0] == 0, PP_ERR_INVALID, "row_off[0] must be 0");
        std::unique_ptr<pp_batch> B(new pp_batch);
        B->ctx = ctx;
        B->nsys = nsys;
        B->ntot = row_off[nsys];
        B->nnz = rowptr[B->ntot];
        B->h_roff.assign(row_off, row_off + nsys + 1);
        B->h_rp.assign(rowptr, rowptr + B->ntot + 1);
        B->h_ci.assign(colidx, colidx + B->nnz);
        B->h_v.assign(values, values + B->nnz);
        // block-diagonal and symmetric (IC(0)-CG needs SPD blocks)
        for (uint32_t s = 0; s < nsys; ++s)
            PP_CHECK(row_off[s] <= row_off[s + 1], PP_ERR_INVALID, "row_off not monotone");
        parallel_for(nsys, 1, [&](size_t s0, size_t s1) {
            for (size_t s = s0; s < s1; ++s)
                for (uint32_t i = row_off[s]; i < row_off[s + 1]; ++i)
                    for (uint32_t k = rowptr[i]; k < rowptr[i + 1]; ++k)
                        PP_CHECK(colidx[k] >= row_off[s] && colidx[k] < row_off[s + 1], PP_ERR_INVALID,
                                 "entry outside its system's diagonal block");
        });
        B->roff = upload(B->h_roff);
        B->rp = upload(B->h_rp);
        B->ci = upload(B->h_ci);
        B->v64 = upload(B->h_v);
        B->v32 = upload(to_f32(B->h_v));
        batch_factor(B.get());
        const size_t n = B->ntot;
        B->r64 = dalloc<double>(n); B->rr64 = dalloc<double>(n); B->w64 = dalloc<double>(n);
        B->d64 = dalloc<double>(n); B->p64 = dalloc<double>(n);
        B->r32 = dalloc<float>(n); B->e32 = dalloc<float>(n); B->q32 = dalloc<float>(n);
        B->w32 = dalloc<float>(n); B->d32 = dalloc<float>(n); B->p32 = dalloc<float>(n);
        B->iters = dalloc<int>(nsys); B->outer = dalloc<int>(nsys); B->conv = dalloc<int>(nsys);
        B->relres = dalloc<double>(nsys);
        *out = B.release();
    });
}

int pp_batch_info_get(const pp_batch *B, pp_batch_info *info) {
    if (!B || !info) return PP_ERR_INVALID;
    std::memset(info, 0, sizeof(*info));
    info->nsys = B->nsys;
    info->rows = B->ntot;
    info->nnz = B->nnz;
    info->tiles = B->tile_width ? B->ntiles : 0;
    info->device_refactors = B->device_refactors;
    return PP_OK;
}

int pp_batch_set_values(pp_ctx *ctx, pp_batch *B, const double *values, int on_device) {
    if (!ctx) return PP_ERR_INVALID;
    return guarded_batch(ctx, [&] {
        PP_CHECK(B && values, PP_ERR_INVALID, "NULL argument");
        if (B->refresh == 0) batch_refresh_build(B);
        // the factorization on the device overwrites the factor: the values it
        // came from are kept until it has succeeded
        const bool keep = B->refresh == 1 && !B->factor_before;
        if (keep && !B->v64_before) B->v64_before = dalloc<double>(B->nnz);
        PP_HIP(hipMemcpy(keep ? B->v64_before : B->v64, values, B->nnz * sizeof(double),
                         on_device ? hipMemcpyDeviceToDevice : hipMemcpyHostToDevice));
        PP_HIP(hipStreamSynchronize(nullptr));  // a device copy may return before it is done
        if (keep) std::swap(B->v64, B->v64_before);
        B->h_v_stale = true;
        if (B->refresh == 1) {
            B->factor_before = !batch_refresh(B, B->v64);
            if (!B->factor_before) {
                ++B->device_refactors;
                return;
            }
            // the factor in use comes back, as the host path leaves it where it fails
            batch_refresh(B, B->v64_before);
            batch_refresh_values(B, B->v64);
            PP_HIP(hipStreamSynchronize(B->ctx->stream));
        }
        // on the host (it also names the first failing system)
        batch_ensure_host_values(B);
        std::vector<float> v32 = to_f32(B->h_v);
        PP_HIP(hipMemcpy(B->v32, v32.data(), B->nnz * sizeof(float), hipMemcpyHostToDevice));
        if (B->ordering == PP_ORDER_MULTICOLOR) batch_upload_permuted_values(B);
        batch_factor(B);
    });
}

int pp_batch_set_ordering(pp_ctx *ctx, pp_batch *B, int ordering) {
    if (!ctx) return PP_ERR_INVALID;
    return guarded_batch(ctx, [&] {
        PP_CHECK(B, PP_ERR_INVALID, "NULL batch");
        PP_CHECK(ordering == PP_ORDER_NATURAL || ordering == PP_ORDER_MULTICOLOR, PP_ERR_INVALID, "unknown ordering");
        PP_HIP(hipStreamSynchronize(ctx->stream));
        batch_ensure_host_values(B);
        B->ordering = ordering;
        if (ordering == PP_ORDER_MULTICOLOR && !B->gperm) {
            batch_build_order(B);
            B->gperm = upload(B->h_gperm);
            B->prp = upload(B->h_prp);
            B->pci = upload(B->h_pci);
            B->bp = dalloc<double>(B->ntot);
            B->xp = dalloc<double>(B->ntot);
        }
        // also where the order had been used before: the values may have come since
        if (ordering == PP_ORDER_MULTICOLOR) batch_upload_permuted_values(B);
        batch_factor(B);
    });
}

static int batch_solve_impl(pp_ctx *ctx, pp_batch *B, const pp_solve_opts *opts, const double *b, double *x,
                            int32_t *iters_out, pp_solve_report *rep) {
    return guarded_batch(ctx, [&] {
        PP_CHECK(B && opts && b && x, PP_ERR_INVALID, "NULL argument");
        PP_CHECK(opts->tol > 0 && opts->maxit >= 1, PP_ERR_INVALID, "bad tolerance / maxit");
        const bool mixed = opts->precision == PP_MIXED;
        const bool perm = B->ordering == PP_ORDER_MULTICOLOR;
        BatchArgs a = make_args(B, *opts, perm ? B->bp : b, perm ? B->xp : x);
        PP_HIP(hipEventRecord(ctx->ev0, ctx->stream));
        if (perm) launch_permute(ctx, B->ntot, B->gperm, PP_F64, b, B->bp, true);
        const bool tiled = mixed && a.red_n0 && B->tile_width && run_tiles(ctx, B, a);
        if (!tiled) run_batch(ctx, B, mixed, a);
        if (perm) {
            launch_permute(ctx, B->ntot, B->gperm, PP_F64, B->xp, x, false);
            PP_HIP(hipStreamSynchronize(ctx->stream));
        }
        PP_HIP(hipEventRecord(ctx->ev1, ctx->stream));
        PP_HIP(hipEventSynchronize(ctx->ev1));
        float ms = 0;
        PP_HIP(hipEventElapsedTime(&ms, ctx->ev0, ctx->ev1));
        std::vector<int32_t> it(B->nsys), ou(B->nsys), cv(B->nsys);
        std::vector<double> rr(B->nsys);
        PP_HIP(hipMemcpy(it.data(), B->iters, B->nsys * sizeof(int32_t), hipMemcpyDeviceToHost));
        PP_HIP(hipMemcpy(ou.data(), B->outer, B->nsys * sizeof(int32_t), hipMemcpyDeviceToHost));
        PP_HIP(hipMemcpy(cv.data(), B->conv, B->nsys * sizeof(int32_t), hipMemcpyDeviceToHost));
        PP_HIP(hipMemcpy(rr.data(), B->relres, B->nsys * sizeof(double), hipMemcpyDeviceToHost));
        if (iters_out) std::copy(it.begin(), it.end(), iters_out);
        if (rep) {
            std::memset(rep, 0, sizeof(*rep));
            rep->iters = *std::max_element(it.begin(), it.end());
            rep->inner_iters = 0;
            for (int32_t v : it) rep->inner_iters += v;
            rep->outer_iters = *std::max_element(ou.begin(), ou.end());
            rep->converged = std::all_of(cv.begin(), cv.end(), [](int32_t c) { return c != 0; });
            rep->true_relres = *std::max_element(rr.begin(), rr.end());
            rep->final_error = rep->true_relres;
            rep->solve_ms = ms;
            rep->status = PP_OK;
            rep->cg_variant = mixed && a.red_n0 ? PP_CG_REDUCED : PP_CG_REFERENCE;
            rep->batch_tiles = tiled ? B->ntiles : 0;
        }
    });
}

int pp_batch_solve(pp_ctx *ctx, pp_batch *B, const pp_solve_opts *opts, const double *b, double *x,
                   int32_t *iters_out, pp_solve_report *rep) {
    if (!ctx) return PP_ERR_INVALID;
    return batch_solve_impl(ctx, B, opts, b, x, iters_out, rep);
}

// IC(0)-CG needs SPD blocks, so A^T = A and the adjoint system is the same one.
int pp_batch_solve_t(pp_ctx *ctx, pp_batch *B, const pp_solve_opts *opts, const double *g, double *lambda,
                     int32_t *iters_out, pp_solve_report *rep) {
    if (!ctx) return PP_ERR_INVALID;
    return batch_solve_impl(ctx, B, opts, g, lambda, iters_out, rep);
}

// Times a bounded number of mixed-precision iterations for each workgroup
// size and keeps the fastest.
int pp_batch_tune(pp_ctx *ctx, pp_batch *B, int *chosen) {
    if (!ctx) return PP_ERR_INVALID;
    return guarded_batch(ctx, [&] {
        PP_CHECK(B, PP_ERR_INVALID, "NULL batch");
        pp_solve_opts o;
        pp_solve_opts_default(&o, PP_SOLVER_CG);
        o.precision = PP_MIXED;
        o.maxit = 12;
        o.tol = 1e-30;
        double *b = dalloc<double>(B->ntot);
        double *x = dalloc<double>(B->ntot);
        std::vector<double> ones(B->ntot, 1.0);
        PP_HIP(hipMemcpy(b, ones.data(), B->ntot * sizeof(double), hipMemcpyHostToDevice));
        BatchArgs a = make_args(B, o, b, x);
        float best = 1e30f;
        int best_bs = B->block;
        for (int bs : {256, 512, 1024}) {
            launch_batch(ctx->stream, bs, true, a);  // warm-up
            PP_HIP(hipEventRecord(ctx->ev0, ctx->stream));
            for (int rep = 0; rep < 3; ++rep) launch_batch(ctx->stream, bs, true, a);
            PP_HIP(hipEventRecord(ctx->ev1, ctx->stream));
            PP_HIP(hipEventSynchronize(ctx->ev1));
            float ms = 0;
            PP_HIP(hipEventElapsedTime(&ms, ctx->ev0, ctx->ev1));
            if (ms < best) {
                best = ms;
                best_bs = bs;
            }
        }
        dfree(b);
        dfree(x);
        B->block = best_bs;
        if (chosen) *chosen = best_bs;
    });
}

void pp_batch_destroy(pp_batch *B) {
    if (!B) return;
    (void)hipSetDevice(B->ctx->device);
    (void)hipStreamSynchronize(B->ctx->stream);
    batch_free(B);
    delete B;
}

}  // extern "C"

namespace pp {
namespace {
__global__ void k_batch_outer(uint32_t n, const uint32_t *rp, const uint32_t *ci, double scale, const double *lam,
                              const double *x, double *g) {
    for (uint32_t i = blockIdx.x * blockDim.x + threadIdx.x; i < n; i += gridDim.x * blockDim.x) {
        const double li = scale * lam[i];
        for (uint32_t k = rp[i]; k < rp[i + 1]; ++k) g[k] = li * x[ci[k]];
    }
}
}  // namespace
}  // namespace pp

extern "C" int pp_batch_outer_on_pattern(pp_ctx *ctx, const pp_batch *B, double scale, const double *lambda,
                                         const double *x, double *grad) {
    if (!ctx) return PP_ERR_INVALID;
    return guarded_batch(ctx, [&] {
        PP_CHECK(B && lambda && x && grad, PP_ERR_INVALID, "NULL argument");
        const unsigned g = std::min<uint32_t>((B->ntot + 255) / 256, 4096);
        pp::k_batch_outer<<<std::max(1u, g), 256, 0, ctx->stream>>>(B->ntot, B->rp, B->ci, scale, lambda, x, grad);
        PP_HIP(hipGetLastError());
        PP_HIP(hipStreamSynchronize(ctx->stream));
    });
}
