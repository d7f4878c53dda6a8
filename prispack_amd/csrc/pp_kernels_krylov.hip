// pp_kernels_krylov.hip -- tall-skinny GEMV kernels of the GMRES orthogonalisation
// (classical Gram-Schmidt, applied twice) and mixed-precision glue kernels.
#include <hip/hip_runtime.h>

#include <algorithm>

#include "pp_internal.h"

namespace pp {

namespace {
constexpr int kGemvBlocks = 2048;  // at most (the partials' rows)
constexpr int kMaxCols = 257;
constexpr int kTailThreads = 1024;

// x plus its value CTRL lanes over (0 where none; MASK: the 16-lane rows that take it)
template <int CTRL, int MASK>
__device__ inline double dpp_add(double x) {
    const int2 b = __builtin_bit_cast(int2, x);
    int2 y;
    y.x = __builtin_amdgcn_update_dpp(0, b.x, CTRL, MASK, 0xf, false);
    y.y = __builtin_amdgcn_update_dpp(0, b.y, CTRL, MASK, 0xf, false);
    return x + __builtin_bit_cast(double, y);
}

// Sum over the wavefront, in its last lane: four shifts inside the rows of
// 16 lanes and two broadcasts across them, all in the vector unit (shuffles
// go through the LDS: 12 instructions and six waits a sum, and a GEMV^T over
// 30 columns ends in 30 sums per wavefront).
constexpr int kLastLane = 63;
__device__ inline double wsum(double v) {
    v = dpp_add<0x111, 0xf>(v);  // row_shr:1, 2, 4, 8
    v = dpp_add<0x112, 0xf>(v);
    v = dpp_add<0x114, 0xf>(v);
    v = dpp_add<0x118, 0xf>(v);
    v = dpp_add<0x142, 0xa>(v);  // row_bcast:15 into rows 1 and 3
    return dpp_add<0x143, 0xc>(v);  // row_bcast:31 into rows 2 and 3
}

// Workgroups of k_gemv_sub where it leaves the partials of a norm.
unsigned gemv_sub_blocks(uint32_t n) { return std::max(1u, std::min((n + 255) / 256, (unsigned)kGemvBlocks)); }

// The sum over a workgroup of 256, in every thread (sh: 4 values).
__device__ inline double bsum(double v, double *sh) {
    v = wsum(v);
    if ((threadIdx.x & 63) == kLastLane) sh[threadIdx.x >> 6] = v;
    __syncthreads();
    return ((sh[0] + sh[1]) + sh[2]) + sh[3];
}

// Workgroups of a pass over ncol columns of the basis: four per CU, eight
// where a row has too few loads for that many wavefronts to cover the memory
// latency.
unsigned gemv_blocks(const pp_ctx *ctx, uint32_t n, uint32_t ncol) {
    const unsigned full = (ncol <= 8 ? 8u : 4u) * (unsigned)ctx->cu_count;
    return std::max(1u, std::min((n + 255) / 256, std::min((unsigned)kGemvBlocks, full)));
}
}  // namespace

// Buffer of GMRES coefficients on the device: [0,320) h, [320, 640) y or a copy of h, and
// the per-column partials of the GEMV^T behind it.
double *gmres_coeff_buffer(pp_ctx *ctx) {
    return (double *)ws_get(ctx, kWsGmresCoeff, (size_t)(640 + (size_t)kMaxCols * kGemvBlocks) * sizeof(double));
}

// partial[c][block] = sum over the block's rows of V[r, c] * w[r] for more
// columns than k_gemv_cgs holds.  The columns go in groups of NG: one pass
// over the block's rows accumulates the whole group in registers (every
// column's loads in flight together, no barrier per column), then one
// reduction per group.
template <int NG, class TV>
__global__ __launch_bounds__(256) void k_gemv_t_partial(uint32_t n, uint32_t ncol, const TV *__restrict__ V,
                                                        size_t ld, const TV *__restrict__ w, double *partial,
                                                        const int *stop) {
    __shared__ double sh[NG][4];
    if (stop && *stop) return;
    const uint32_t chunk = (n + gridDim.x - 1) / gridDim.x;
    const uint32_t r0 = blockIdx.x * chunk, r1 = min(n, r0 + chunk);
    for (uint32_t c0 = 0; c0 < ncol; c0 += NG) {
        const uint32_t nc = min((uint32_t)NG, ncol - c0);
        double acc[NG];
#pragma unroll
        for (int c = 0; c < NG; ++c) acc[c] = 0.0;
        for (uint32_t r = r0 + threadIdx.x; r < r1; r += blockDim.x) {
            const double wr = w[r];
            // every slot's load is unconditional (slots past the group's
            // last column reread that column, a cache hit, and their sums are
            // never used), so the loads issue back to back instead of one
            // behind each branch
            double vv[NG];
#pragma unroll
            for (int c = 0; c < NG; ++c) vv[c] = (double)V[ld * (c0 + min((uint32_t)c, nc - 1)) + r];
#pragma unroll
            for (int c = 0; c < NG; ++c) acc[c] += vv[c] * wr;
        }
#pragma unroll
        for (int c = 0; c < NG; ++c)
            if ((uint32_t)c < nc) {
                const double v = wsum(acc[c]);
                if ((threadIdx.x & 63) == kLastLane) sh[c][threadIdx.x >> 6] = v;
            }
        __syncthreads();
        if (threadIdx.x < nc)
            partial[(size_t)(c0 + threadIdx.x) * gridDim.x + blockIdx.x] =
                ((sh[threadIdx.x][0] + sh[threadIdx.x][1]) + sh[threadIdx.x][2]) + sh[threadIdx.x][3];
        __syncthreads();
    }
}

// h[c] = sum_b partial[c][b] in block order (deterministic)
__global__ __launch_bounds__(256) void k_gemv_t_reduce(uint32_t nb, const double *partial, double *h,
                                                       const int *stop) {
    __shared__ double sh[4];
    if (stop && *stop) return;
    const uint32_t c = blockIdx.x;
    double v[kGemvBlocks / 256], acc = 0.0;
#pragma unroll
    for (int k = 0; k < kGemvBlocks / 256; ++k) {  // the loads overlap
        const uint32_t b = threadIdx.x + 256 * k;
        v[k] = b < nb ? partial[(size_t)c * nb + b] : 0.0;
    }
#pragma unroll
    for (int k = 0; k < kGemvBlocks / 256; ++k) acc += v[k];
    acc = bsum(acc, sh);
    if (threadIdx.x == 0) h[c] = acc;
}

// A pass of the orthogonalisation over up to kFuseCols columns.  SUB: w[r] -=
// sum_c V[r, c] h[c] first, the row's basis entries kept in registers between
// the two uses (one read of V fewer).  Then partial[c][block] of V[r, c] *
// w[r].  Bound by the reads of V: a wavefront has a row's NC loads in flight,
// four workgroups a CU fit the registers, and the rows go in as few
// workgroups as that fills, because each ends in NC sums over its wavefronts.
// NC: the columns rounded up to four (slots past the last column reread it
// and their sums are not used).  28 columns of 10^6 rows, FP64: 31.7 us
// without and 30.7 us with SUB (7.1, 7.8 TB/s, part of V in the last-level
// cache); 47 us where the compiler may move products between the loads; the
// mean over 30 steps was 31 and 43 us with 2048 workgroups, shuffles and
// slots for 8, 16 or 32 columns, and is 20 and 20 us.
constexpr int kFuseCols = 32;
template <int NC, bool SUB, class TV>
__global__ __launch_bounds__(256) void k_gemv_cgs(uint32_t n, uint32_t ncol, const TV *__restrict__ V, size_t ld,
                                                  const double *__restrict__ h, TV *__restrict__ w,
                                                  double *partial, const int *stop) {
    __shared__ double sh[NC][4];
    if (stop && *stop) return;
    const uint32_t chunk = (n + gridDim.x - 1) / gridDim.x;
    const uint32_t r0 = blockIdx.x * chunk, r1 = min(n, r0 + chunk);
    double acc[NC];
#pragma unroll
    for (int c = 0; c < NC; ++c) acc[c] = 0.0;
    for (uint32_t r = r0 + threadIdx.x; r < r1; r += blockDim.x) {
        TV v[NC];
        // loads unconditional, so they issue back to back
        TV wt = w[r];
#pragma unroll
        for (int c = 0; c < NC; ++c) v[c] = V[ld * min((uint32_t)c, ncol - 1) + r];
        __builtin_amdgcn_sched_barrier(0);  // all of them, before the first product waits
        if constexpr (SUB) {
            double a = 0.0;
#pragma unroll
            for (int c = 0; c < NC; ++c)
                if ((uint32_t)c < ncol) a += (double)v[c] * h[c];
            wt = (TV)((double)wt - a);
            w[r] = wt;
        }
        const double wr = (double)wt;
#pragma unroll
        for (int c = 0; c < NC; ++c) acc[c] += (double)v[c] * wr;
    }
#pragma unroll
    for (int c = 0; c < NC; ++c) {
        const double t = wsum(acc[c]);
        if ((threadIdx.x & 63) == kLastLane) sh[c][threadIdx.x >> 6] = t;
    }
    __syncthreads();
    if (threadIdx.x < ncol)
        partial[(size_t)threadIdx.x * gridDim.x + blockIdx.x] =
            ((sh[threadIdx.x][0] + sh[threadIdx.x][1]) + sh[threadIdx.x][2]) + sh[threadIdx.x][3];
}

template <bool SUB, class TV>
static void launch_gemv_cgs(pp_ctx *ctx, unsigned g, uint32_t n, uint32_t ncol, const TV *V, size_t ld,
                            const double *h, TV *w, double *partial) {
#define PP_CGS(NC)                                                                                                 \
    case NC / 4:                                                                                                   \
        k_gemv_cgs<NC, SUB, TV><<<g, 256, 0, ctx->stream>>>(n, ncol, V, ld, h, w, partial, ctx->stop_word);         \
        break
    switch ((ncol + 3) / 4) {
        PP_CGS(4);
        PP_CGS(8);
        PP_CGS(12);
        PP_CGS(16);
        PP_CGS(20);
        PP_CGS(24);
        PP_CGS(28);
        PP_CGS(32);
    }
#undef PP_CGS
}

template <class TV>
void launch_gemv_t(pp_ctx *ctx, uint32_t n, uint32_t ncol, const TV *V, size_t ld, const TV *w, double *dest) {
    PP_CHECK(ncol >= 1 && ncol <= kMaxCols, PP_ERR_UNSUPPORTED, "too many columns");
    double *buf = gmres_coeff_buffer(ctx);
    double *partial = buf + 640;
    const unsigned g = gemv_blocks(ctx, n, ncol);
    if (ncol <= (uint32_t)kFuseCols)
        launch_gemv_cgs<false, TV>(ctx, g, n, ncol, V, ld, nullptr, const_cast<TV *>(w), partial);
    else k_gemv_t_partial<16, TV><<<g, 256, 0, ctx->stream>>>(n, ncol, V, ld, w, partial, ctx->stop_word);
    k_gemv_t_reduce<<<ncol, 256, 0, ctx->stream>>>(g, partial, dest ? dest : buf, ctx->stop_word);
    PP_HIP(hipGetLastError());
}

// w[r] -= sum_c V[r, c] h[c] (the sum in FP64 for either storage type);
// norm_partials != NULL: also each workgroup's sum of w[r]^2 of the new w
template <class TV>
__global__ __launch_bounds__(256) void k_gemv_sub(uint32_t n, uint32_t ncol, const TV *__restrict__ V,
                                                  size_t ld, const double *__restrict__ h, TV *__restrict__ w,
                                                  double *norm_partials, const int *stop) {
    __shared__ double sh[4];
    if (stop && *stop) return;
    constexpr int kU = 8;
    double sq = 0.0;
    for (uint32_t r = blockIdx.x * blockDim.x + threadIdx.x; r < n; r += gridDim.x * blockDim.x) {
        const TV w0 = w[r];
        double acc = 0.0;
        // the columns eight at a time: the loads first (past the last
        // column they reread it), then the products in column order
        for (uint32_t c0 = 0; c0 < ncol; c0 += kU) {
            TV vv[kU];
#pragma unroll
            for (int u = 0; u < kU; ++u) vv[u] = V[ld * min(c0 + u, ncol - 1) + r];
#pragma unroll
            for (int u = 0; u < kU; ++u)
                if (c0 + u < ncol) acc += (double)vv[u] * h[c0 + u];
        }
        const TV wt = (TV)((double)w0 - acc);
        w[r] = wt;
        sq += (double)wt * (double)wt;
    }
    if (!norm_partials) return;
    sq = bsum(sq, sh);
    if (threadIdx.x == 0) norm_partials[blockIdx.x] = sq;
}

template <class TV>
void launch_gemv_sub(pp_ctx *ctx, uint32_t n, uint32_t ncol, const TV *V, size_t ld, const double *h, TV *w,
                     double *norm_partials) {
    const unsigned g = norm_partials ? gemv_sub_blocks(n) : std::min<uint32_t>((n + 255) / 256, 8192);
    k_gemv_sub<TV><<<g, 256, 0, ctx->stream>>>(n, ncol, V, ld, h, w, norm_partials, ctx->stop_word);
    PP_HIP(hipGetLastError());
}

// w -= V h1, then dest = V^T w: fused where the columns fit the registers
template <class TV>
void launch_gemv_sub_t(pp_ctx *ctx, uint32_t n, uint32_t ncol, const TV *V, size_t ld, const double *h1, TV *w,
                       double *dest) {
    if (ncol > (uint32_t)kFuseCols) {
        launch_gemv_sub<TV>(ctx, n, ncol, V, ld, h1, w, nullptr);
        launch_gemv_t(ctx, n, ncol, V, ld, w, dest);
        return;
    }
    double *buf = gmres_coeff_buffer(ctx);
    double *partial = buf + 640;
    const unsigned g = gemv_blocks(ctx, n, ncol);
    launch_gemv_cgs<true, TV>(ctx, g, n, ncol, V, ld, h1, w, partial);
    k_gemv_t_reduce<<<ncol, 256, 0, ctx->stream>>>(g, partial, dest ? dest : buf, ctx->stop_word);
    PP_HIP(hipGetLastError());
}
template void launch_gemv_t<double>(pp_ctx *, uint32_t, uint32_t, const double *, size_t, const double *, double *);
template void launch_gemv_t<float>(pp_ctx *, uint32_t, uint32_t, const float *, size_t, const float *, double *);
template void launch_gemv_sub<double>(pp_ctx *, uint32_t, uint32_t, const double *, size_t, const double *, double *,
                                      double *);
template void launch_gemv_sub<float>(pp_ctx *, uint32_t, uint32_t, const float *, size_t, const double *, float *,
                                     double *);
template void launch_gemv_sub_t<double>(pp_ctx *, uint32_t, uint32_t, const double *, size_t, const double *,
                                        double *, double *);
template void launch_gemv_sub_t<float>(pp_ctx *, uint32_t, uint32_t, const float *, size_t, const double *, float *,
                                       double *);


// x[r] += sum_c Z[r, c] y[c] (Z in FP32 or FP64), columns in ascending order
// like DenseMatrix::MatVec (DenseMatrix.cpp:208-224).  A column whose
// coefficient is zero adds nothing and is not read: the columns past a
// converged cycle's last step hold whatever the early-exit kernels left.
template <class T>
__global__ __launch_bounds__(256) void k_gemv_add(uint32_t n, uint32_t ncol, const T *__restrict__ Z, size_t ld,
                                                  const double *__restrict__ y, double *__restrict__ x) {
    for (uint32_t r = blockIdx.x * blockDim.x + threadIdx.x; r < n; r += gridDim.x * blockDim.x) {
        double acc = 0.0;
        for (uint32_t c = 0; c < ncol; ++c)
            if (y[c] != 0.0) acc += (double)Z[ld * c + r] * y[c];
        x[r] += acc;
    }
}

void launch_gemv_add(pp_ctx *ctx, uint32_t n, uint32_t ncol, const float *Z32, const double *Z64, size_t ld,
                     const double *y, double *x) {
    unsigned g = std::min<uint32_t>((n + 255) / 256, 8192);
    if (Z32) k_gemv_add<float><<<g, 256, 0, ctx->stream>>>(n, ncol, Z32, ld, y, x);
    else k_gemv_add<double><<<g, 256, 0, ctx->stream>>>(n, ncol, Z64, ld, y, x);
    PP_HIP(hipGetLastError());
}

__global__ void k_scale_convert(uint32_t n, const double *s, double a, float *d) {
    for (uint32_t i = blockIdx.x * blockDim.x + threadIdx.x; i < n; i += gridDim.x * blockDim.x)
        d[i] = (float)(s[i] * a);
}

void launch_scale_convert(pp_ctx *ctx, uint32_t n, const double *src, double scale, float *dst) {
    unsigned g = std::min<uint32_t>((n + 255) / 256, 4096);
    k_scale_convert<<<g, 256, 0, ctx->stream>>>(n, src, scale, dst);
    PP_HIP(hipGetLastError());
}

__global__ void k_axpy_f32_f64(uint32_t n, double a, const float *x, double *y) {
    for (uint32_t i = blockIdx.x * blockDim.x + threadIdx.x; i < n; i += gridDim.x * blockDim.x)
        y[i] += a * (double)x[i];
}

void launch_axpy_f32_to_f64(pp_ctx *ctx, uint32_t n, double a, const float *x, double *y) {
    unsigned g = std::min<uint32_t>((n + 255) / 256, 4096);
    k_axpy_f32_f64<<<g, 256, 0, ctx->stream>>>(n, a, x, y);
    PP_HIP(hipGetLastError());
}

// first == -1: the GMRES coefficient buffer; else device scalar slots.
void read_slots(pp_ctx *ctx, int first, int count, double *out) {
    const double *src = first < 0 ? gmres_coeff_buffer(ctx) : ctx->scal + first;
    PP_CHECK(count <= 320, PP_ERR_INVALID, "too many slots");
    PP_HIP(hipMemcpyAsync(ctx->pinned, src, count * sizeof(double), hipMemcpyDeviceToHost, ctx->stream));
    PP_HIP(hipStreamSynchronize(ctx->stream));
    std::copy(ctx->pinned, ctx->pinned + count, out);
}

}  // namespace pp

// ---------------------------------------------------------------------------
// Device-resident least-squares of FlexibleGMRES(m): the Hessenberg column,
// the Givens rotations (GMRES.cpp:72-101), the convergence test and the
// back substitution (GMRES.cpp:103-119) run on the stream, so an Arnoldi cycle is issued without any host round trip; the
// stop word ends the cycle's remaining kernels once the estimate converges.
// ---------------------------------------------------------------------------
namespace pp {

GmresDev gmres_state(pp_ctx *ctx, uint32_t mm) {
    const size_t ld = mm + 1;
    const size_t total = ld * mm + 6 * ld + kGmMisc + kGemvBlocks;
    double *base = (double *)ws_get(ctx, kWsGmresState, total * sizeof(double));
    GmresDev st;
    st.mm = mm;
    st.H = base;
    st.c = st.H + ld * mm;
    st.s = st.c + ld;
    st.g = st.s + ld;
    st.h1 = st.g + ld;
    st.h2 = st.h1 + ld;
    st.gb = st.h2 + ld;
    st.misc = st.gb + ld;
    st.norm = st.misc + kGmMisc;
    return st;
}

namespace {

__global__ void k_gmres_cycle_init(GmresDev st, double beta, double bnorm, double tol, uint32_t hist_base) {
    if (threadIdx.x != 0 || blockIdx.x != 0) return;
    for (uint32_t i = 0; i < st.mm; ++i) st.g[i] = 0.0;  // g[mm] keeps its value (GMRES.cpp:160)
    st.g[0] = beta;
    st.gb[0] = beta;
    st.misc[GM_M] = st.mm;
    st.misc[GM_STATUS] = 0.0;
    st.misc[GM_CONVCYC] = 0.0;
    st.misc[GM_NREC] = 0.0;
    st.misc[GM_HBASE] = (double)hist_base;
    st.misc[GM_BNORM] = bnorm;
    st.misc[GM_TOL] = tol;
}

// The end of an Arnoldi step: h_{j+1,j} = ||w|| from its partials, the
// Hessenberg column's Givens rotations (GMRES.cpp:72-101), the convergence
// test, and v_{j+1} = (1/h_{j+1,j}) w, evaluated like HostVector::add with
// b = 0.  Whether v_{j+1} is written hangs on the test, so every workgroup
// runs the rotations itself (thread 0, operands in LDS: about 1 us for 30
// columns) and workgroup 0 alone writes the state.  Of what the others read it
// writes the stop word alone (the right-hand side before the rotations is kept
// in gb, next to g), which one thread of a workgroup reads for all of it: where
// that thread finds this very step's stop, the workgroup ends as the test would
// have had it end.  One launch instead of four (sum, finish, a
// single-thread step with its operands in device memory, scaling): 21.5 us
// on 100^3 rows, now 6.7 us.
template <class TV>
__global__ __launch_bounds__(kTailThreads) void k_gmres_step(GmresDev st, uint32_t j, int quirks,
                                                             const double *__restrict__ norm_partials, unsigned np,
                                                             int *ctl, double *hist, uint32_t hist_idx,
                                                             uint32_t hist_cap, uint32_t n,
                                                             const TV *__restrict__ w, TV *__restrict__ v) {
#pragma clang fp contract(off)
    __shared__ double sh[kTailThreads / 64], col[kMaxCols + 1], cs[kMaxCols], sn[kMaxCols], inv;
    __shared__ int go, stopped;
    const uint32_t step = gridDim.x * kTailThreads, t = threadIdx.x;
    if (t == 0) stopped = ctl[C_STOP];
    uint32_t i = blockIdx.x * kTailThreads + t;
    TV wi = 0;
    if (i < n) wi = w[i];
    double nrm = 0.0;
    for (unsigned q = t; q < np; q += kTailThreads) nrm += norm_partials[q];
    nrm = wsum(nrm);
    if ((t & 63) == kLastLane) sh[t >> 6] = nrm;
    if (t <= j) col[t] = st.h1[t] + st.h2[t];
    if (t < j) {
        cs[t] = st.c[t];
        sn[t] = st.s[t];
    }
    __syncthreads();
    if (stopped) return;
    if (t == 0) {
        const uint32_t ld = st.mm + 1;
        double *H = st.H + (size_t)j * ld;
        double wn2 = 0.0;
        for (int q = 0; q < kTailThreads / 64; ++q) wn2 += sh[q];
        const double hn = sqrt(wn2);
        const double bnorm = st.misc[GM_BNORM], tol = st.misc[GM_TOL], gj = st.gb[j];
        const bool bad = !(hn == hn), breakdown = !bad && fabs(hn) == 0.0;
        double c = 0.0, s = 0.0, hj = 0.0, gn = 0.0, rnorm = 0.0, relerr = 0.0;
        const bool rotate = !bad && !(breakdown && quirks);
        if (rotate) {
            double h1 = col[0];
            for (uint32_t k = 0; k < j; ++k) {
                const double h2 = col[k + 1];
                col[k] = cs[k] * h1 + sn[k] * h2;
                h1 = cs[k] * h2 - sn[k] * h1;
            }
            const double h2 = hn;
            if (fabs(h1) > fabs(h2)) {
                const double u = h2 / h1;
                c = 1.0 / sqrt(fabs(1.0 + u * u));
                s = c * u;
            } else {
                const double u = h1 / h2;
                s = 1.0 / sqrt(fabs(1.0 + u * u));
                c = s * u;
            }
            hj = c * h1 + s * h2;
            gn = -s * gj;
            rnorm = fabs(gn);
            relerr = rnorm / bnorm;
        }
        const bool conv = !bad && !breakdown && relerr < tol;
        go = !bad && !breakdown && !conv;
        inv = 1.0 / hn;
        if (blockIdx.x == 0) {
            for (uint32_t k = 0; k < j; ++k) H[k] = col[k];
            if (rotate) {
                H[j] = hj;
                H[j + 1] = 0.0;
                st.c[j] = c;
                st.s[j] = s;
                st.g[j + 1] = st.gb[j + 1] = gn;
                st.g[j] = c * gj;
                st.misc[GM_RNORM] = rnorm;
                st.misc[GM_RELERR] = relerr;
            } else {
                H[j] = col[j];
                H[j + 1] = hn;
            }
            if (bad) {
                st.misc[GM_STATUS] = PP_ERR_NOT_FINITE;
                st.misc[GM_M] = j;
            } else if (breakdown) {  // happy breakdown (GMRES.cpp:183-186)
                st.misc[GM_M] = quirks ? j : j + 1;
                if (!quirks) st.misc[GM_CONVCYC] = 1.0;
            } else {
                // hist_idx counts from the cycle's first step (a captured cycle is replayed unchanged)
                const uint32_t hidx = (uint32_t)st.misc[GM_HBASE] + hist_idx;
                if (hist && hidx < hist_cap) hist[hidx] = relerr;
                st.misc[GM_NREC] += 1.0;
                if (conv) {
                    st.misc[GM_M] = quirks ? j : j + 1;  // the reference drops column j
                    st.misc[GM_CONVCYC] = 1.0;
                }
            }
            if (!go) ctl[C_STOP] = 1;
        }
    }
    __syncthreads();
    if (!go) return;
    const double a = inv;
    while (i < n) {
        const double t1 = a * (double)wi;
        const double t2 = 0.0 * (double)wi;
        v[i] = (TV)(t1 + t2);
        i += step;
        if (i < n) wi = w[i];
    }
}

// Back substitution by columns of H (column-major), thread k with the entry k
// of the right-hand side: a solved entry goes through LDS to the rows above
// it, the loads of eight columns run ahead.  A single thread walking the rows
// took 49 us for 30 columns, a chain of device-memory latencies; now 7.8 us.
__global__ __launch_bounds__(256) void k_gmres_backsolve(GmresDev st, int quirks, double *y) {
#pragma clang fp contract(off)
    __shared__ double sol[2];
    constexpr int kAhead = 8;
    const uint32_t ld = st.mm + 1, k = threadIdx.x;
    const uint32_t m = (uint32_t)st.misc[GM_M];  // at most 256
    double t = k < m ? st.g[k] : 0.0;
    for (int i1 = (int)m - 1; i1 >= 0; i1 -= kAhead) {
        double h[kAhead];
#pragma unroll
        for (int u = 0; u < kAhead; ++u) h[u] = st.H[(size_t)max(i1 - u, 0) * ld + min(k, st.mm)];
#pragma unroll
        for (int u = 0; u < kAhead; ++u) {
            const int i = i1 - u;
            if (i >= 0) {  // the same in every thread
                if ((int)k == i) sol[u & 1] = t = t / h[u];
                __syncthreads();
                if ((int)k < i) t -= h[u] * sol[u & 1];
            }
        }
    }
    if (k < m) st.g[k] = t;
    if (k == 0) st.g[m] = 0.0;
    __syncthreads();
    for (uint32_t i = k; i <= st.mm; i += blockDim.x) y[i] = (!quirks && i >= m) ? 0.0 : st.g[i];
}

}  // namespace

void launch_gmres_cycle_init(pp_ctx *ctx, const GmresDev &st, double beta, double bnorm, double tol,
                             uint32_t hist_base) {
    k_gmres_cycle_init<<<1, 64, 0, ctx->stream>>>(st, beta, bnorm, tol, hist_base);
    PP_HIP(hipGetLastError());
}

template <class TV>
void launch_gmres_step(pp_ctx *ctx, const GmresDev &st, uint32_t j, int quirks, double *hist, uint32_t hist_idx,
                       uint32_t hist_cap, uint32_t n, const TV *w, TV *vnext) {
    const unsigned g = std::max(1u, std::min((n + kTailThreads - 1) / kTailThreads, 2u * (unsigned)ctx->cu_count));
    k_gmres_step<TV><<<g, kTailThreads, 0, ctx->stream>>>(st, j, quirks, st.norm, gemv_sub_blocks(n), ctx->ctl, hist,
                                                          hist_idx, hist_cap, n, w, vnext);
    PP_HIP(hipGetLastError());
}
template void launch_gmres_step<double>(pp_ctx *, const GmresDev &, uint32_t, int, double *, uint32_t, uint32_t,
                                        uint32_t, const double *, double *);
template void launch_gmres_step<float>(pp_ctx *, const GmresDev &, uint32_t, int, double *, uint32_t, uint32_t,
                                       uint32_t, const float *, float *);

void launch_gmres_backsolve(pp_ctx *ctx, const GmresDev &st, int quirks, double *y) {
    k_gmres_backsolve<<<1, 256, 0, ctx->stream>>>(st, quirks, y);
    PP_HIP(hipGetLastError());
}

}  // namespace pp
