// Restarted GMRES(m) on gfx950, device resident.
//
// Replaces Solver<T>::solve of the reference's external solver library
// (call sites src/mesh.h:740-746, src/impl/slaplace_impl.h:171).  One restart
// cycle = m Arnoldi steps; each cycle begins from the true FP64 residual
// r = b - A x, so the same driver gives
//   * the plain FP64 form (vectors, matrix and Krylov basis in FP64), and
//   * the mixed form: Krylov basis, work vector and Arnoldi SpMV in FP32
//     (matrix values stored as FP32 or BF16), with FP64 kept for the
//     residual r = b - A x, every dot/norm accumulation, the Hessenberg
//     matrix and its Givens rotations, and the update x += V y.  Restarting
//     from the FP64 residual makes each cycle one step of iterative
//     refinement.
//
// Orthogonalisation: modified Gram-Schmidt (the reference form) or classical
// Gram-Schmidt with one re-orthogonalisation pass (CGS2).  The dots of a pass
// are computed together in both.  For modified Gram-Schmidt that needs the
// basis vectors' own products, which the step before has computed: see
// mgs_solve in krylov.h.
//
// Up to 262,144 rows and m <= 32 a restart cycle is one persistent launch
// (persist.hip).  Here are the driver and the form with a launch per pass, for
// larger matrices and restarts.  Its kernels per Arnoldi step: the SpMV with
// the first pass's dots, the update with the dots of the next pass or of the next
// basis vector and the norm (twice for CGS2), and after each of them one
// workgroup that adds the block partials and does the step's small dense
// work.  Every pass reads the basis once: the update keeps a row's basis
// entries in registers for the dots of the updated row.  Level 8 (257
// workgroups): 1217 steps in 63 ms, against 125 ms with a pass per basis
// vector; 52 us a step, of which reading the basis and the matrix takes 51
// at a copy's rate.  A restart cycle is captured once in a hipGraph and replayed;
// kernels of a finished cycle return at once.
//
// Reductions are deterministic: every block writes one partial per dot, and
// they are added in block order.  Results depend only on the inputs and the
// launch shape, never on timing, and both forms give the same bits.
#include <cmath>
#include <cstdlib>
#include <cstring>
#include <type_traits>
#include <vector>

#include "krylov.h"
#include "persist.h"
#include "phg_internal.h"

namespace phg {

constexpr int GM_MAXM = 64;
constexpr int GM_MAXN = 1 << 20; // most rows
constexpr int GM_RED = 1024;      // threads of the reducing workgroup
constexpr int GM_BS = KR_STRIDE;  // threads of the others
constexpr int GM_HALF = 32;       // basis entries of a row in registers at once

struct GmresState {
    double R[GM_MAXM * GM_MAXM];  // rotated (upper triangular) columns
    double L[GM_MAXM * GM_MAXM];  // <v_i, v_k>, k < i (MGS)
    double cs[2 * GM_MAXM];       // cos and sin of each rotation
    double g[GM_MAXM];            // rotated right-hand side, final entries
    double carry[GM_MAXM + 1];    // carry[j+1] = last entry after step j
    double y[GM_MAXM];
    double hc[GM_MAXM];           // coefficients of the current pass
    double hcol[GM_MAXM];         // Hessenberg column of the step
    double beta, bnorm, rel, hn, rtol, inner_rtol;
    int m, active, k, iters, iters0, max_iters, converged, cycles;
    const double* b;  // the caller's arrays: one captured cycle serves them all
    double* x;
};

struct GmresWork {
    int n = 0, m = 0, R = 0, G = 0, S = 0, prec = 0;
    size_t ldv = 0;
    PersistWork persist;
    // the launch-per-pass form (allocated when it first runs)
    DevBuf<char> V, W;     // m x ldv and 2 x ldv vectors of the Krylov type
    DevBuf<double> part;   // G x S block partials
    DevBuf<GmresState> st;
    GmresState* host = nullptr;  // pinned mirror
    // captured restart cycle, in parts
    hipStream_t cap = nullptr;
    hipGraphExec_t exec[4] = {};  // a cycle's chunks and its end, or all in one
    bool captured = false;
    const void* key[2] = {nullptr, nullptr};
    int key_m = 0, key_ortho = -1;
    void drop_graphs()
    {
        for (auto& e : exec)
            if (e) (void)hipGraphExecDestroy(e), e = nullptr;
        captured = false;
    }
    ~GmresWork()
    {
        drop_graphs();
        if (cap) (void)hipStreamDestroy(cap);
        if (host) (void)hipHostFree(host);
    }
};

void destroy_gmres_work(GmresWork* w) { delete w; }

namespace {

// Block partials part[block * S + value] of the tiers of eight values that
// reduce8 leaves in sh[wavefront][value], values 0..nv-1, and of the norm
// (sh[.][GM_MAXM]) as value S - 1.  All threads of the block.
__device__ __forceinline__ void write_partials(const double (*sh)[GM_MAXM + 1], int nv, bool norm,
                                               int S, double* __restrict__ part)
{
    __syncthreads();
    const int t = threadIdx.x;
    const int v = norm && t == GM_MAXM ? S - 1 : t;
    if (t < nv || (norm && t == GM_MAXM)) {
        double r = 0.0;
#pragma unroll
        for (int p = 0; p < GM_BS / 64; p += 4) r += krylov_half(sh[p][t], sh[p + 1][t], sh[p + 2][t], sh[p + 3][t]);
        part[(size_t)lblock() * S + v] = r;
    }
}

// a thread's sum of squares as the norm's partial
__device__ __forceinline__ void norm_partial(double a, double (*sh)[GM_MAXM + 1])
{
    a = wave_sum(a);
    if ((threadIdx.x & 63) == 0) sh[threadIdx.x >> 6][GM_MAXM] = a;
}
// a thread's dots as the partials of values 0..NV-1 (those up to j)
template <int NV>
__device__ __forceinline__ void dot_partials(const double (&acc)[NV], int j,
                                             double (*sh)[GM_MAXM + 1])
{
    const int lane = threadIdx.x & 63;
#pragma unroll
    for (int i0 = 0; i0 < NV; i0 += KR_T) {
        if (i0 > j) break;
        double p[KR_T];
#pragma unroll
        for (int q = 0; q < KR_T; ++q) p[q] = acc[i0 + q];
        const double s = reduce8(p);
        if ((lane & 7) == 0) sh[threadIdx.x >> 6][i0 + reduce8_value(lane)] = s;
    }
}

// ---------------------------------------------------------------- kernels --
// v_i(row) by a 32-bit offset from the basis (at most 64 x 2^20 x 8 bytes):
// 32 loads in flight do not need 32 scalar base addresses.
template <typename VT>
__device__ __forceinline__ VT basis_at(const VT* V, size_t ldv, int i, int row)
{
    const unsigned o = (unsigned)i * ((unsigned)ldv * (unsigned)sizeof(VT)) +
                       (unsigned)row * (unsigned)sizeof(VT);
    return *(const VT*)((const char*)V + o);
}

// A block owns R x GM_BS rows, a thread rows base + r * GM_BS, r < R.
//
// r = b - A x in FP64 (the refinement residual); W0 = r; partial ||r||^2.
template <typename VT>
__global__ void __launch_bounds__(GM_BS)
k_residual(int n, int R, int width, const int* __restrict__ col, const double* __restrict__ val,
           VT* __restrict__ W0, int S, double* __restrict__ part, const GmresState* __restrict__ st)
{
    __shared__ double sh[GM_BS / 64][GM_MAXM + 1];
    if (st->converged) return;
    const double *b = st->b, *x = st->x;
    const int base = lblock() * GM_BS * R + threadIdx.x;
    double a = 0.0;
    for (int r = 0; r < R; ++r) {
        const int row = base + r * GM_BS;
        double xo, ax;
        krylov_rows<double, double, false, 1>(n, width, row, col, val, x, 1, 1.0, &xo, &ax);
        if (row >= n) break;
        const double res = b[row] - ax;
        W0[row] = (VT)res;
        a = fma(res, res, a);
    }
    norm_partial(a, sh);
    write_partials(sh, 0, true, S, part);
}

__global__ void __launch_bounds__(GM_BS)
k_sumsq(int n, int R, const double* __restrict__ b, int S, double* __restrict__ part)
{
    __shared__ double sh[GM_BS / 64][GM_MAXM + 1];
    const int base = lblock() * GM_BS * R + threadIdx.x;
    double a = 0.0;
    for (int r = 0; r < R; ++r) {
        const int row = base + r * GM_BS;
        if (row >= n) break;
        a = fma(b[row], b[row], a);
    }
    norm_partial(a, sh);
    write_partials(sh, 0, true, S, part);
}

// Arnoldi step j < NV: v_j = W_src / h (stored), W_dst = A v_j, and the block
// partials of <W_dst, v_i>, i <= j.  Row by row; a row's basis entries are
// loaded without a branch (past j - 1 the last one again, not used), so that
// all of them are in flight, GM_HALF at a time.  SHORT: matrix rows of 1 to
// ELL_MAXW entries, tested at run time all the same (with the wide rows' loop
// behind the test instead of one entry by entry a level-8 solve took 0.7 %
// longer, without the test 6 %: the branch keeps the basis loads and the
// gathers in their order).
template <typename VT, typename MT, int NV, bool SHORT>
__global__ void __launch_bounds__(GM_BS)
k_step_spmv(int n, int R, int width, const int* __restrict__ col, const MT* __restrict__ val,
            const VT* __restrict__ Wsrc, VT* __restrict__ V, size_t ldv, VT* __restrict__ Wdst,
            int j, int S, double* __restrict__ part, const GmresState* __restrict__ st)
{
    __shared__ double sh[GM_BS / 64][GM_MAXM + 1];
    if (!st->active) return;
    constexpr int N1 = NV < GM_HALF ? NV : GM_HALF;
    const VT inv = (VT)(1.0 / (j == 0 ? st->beta : st->hn));
    const int base = lblock() * GM_BS * R + threadIdx.x;
    double acc[NV];
#pragma unroll
    for (int i = 0; i < NV; ++i) acc[i] = 0.0;
#pragma unroll 1
    for (int r = 0; r < R; ++r) {
        const int row = base + r * GM_BS;
        if (row >= n) break;
        VT v[N1], vj, w;
#pragma unroll
        for (int i = 0; i < N1; ++i) v[i] = basis_at(V, ldv, max(min(i, j - 1), 0), row);
        if (SHORT && width >= 1 && width <= ELL_MAXW)
            krylov_rows<VT, MT, false, 1, true>(n, width, row, col, val, Wsrc, 1, inv, &vj, &w);
        else if (SHORT)
            krylov_rows_each<VT, MT, false, 1>(n, width, row, col, val, Wsrc, 1, inv, &vj, &w);
        else
            krylov_rows_loop<VT, MT, false, 1>(n, width, row, col, val, Wsrc, 1, inv, &vj, &w);
        vj = vj * inv;
        V[(size_t)j * ldv + row] = vj;
        Wdst[row] = w;
#pragma unroll
        for (int i = 0; i < N1; ++i) acc[i] = fma(to_d(w), to_d(i == j ? vj : v[i]), acc[i]);
        if constexpr (NV > N1) {
#pragma unroll
            for (int i = N1; i < NV; ++i) v[i - N1] = basis_at(V, ldv, max(min(i, j - 1), 0), row);
#pragma unroll
            for (int i = N1; i < NV; ++i)
                acc[i] = fma(to_d(w), to_d(i == j ? vj : v[i - N1]), acc[i]);
        }
    }
    dot_partials<NV>(acc, j, sh);
    write_partials(sh, j + 1, false, S, part);
}

// w -= sum_{i<=j} hc_i v_i, then the block partials of <w, v_i>, i <= j
// (DOTS) and of ||w||^2 (norm).  Row by row, with the row's v_0..v_j kept in
// registers from the update to the dots: the basis is read once.  The loads
// have no branch between them (past j row j again, with a coefficient of 0):
// with one, level 8's updates with 32 vectors took 95 us instead of 30.
// Above GM_HALF vectors (restarts above 32) the first GM_HALF are read again
// for their dots: 64 in registers do not fit beside their 64 sums.  A level-7
// FP64 CGS2 solve with restart 64: 5.46 ms, with the whole basis read twice,
// eight vectors at a time, 6.41 ms.
template <typename VT, int NV, bool DOTS>
__global__ void __launch_bounds__(GM_BS)
k_update(int n, int R, VT* __restrict__ w, const VT* __restrict__ V, size_t ldv, int j, int norm,
         int S, double* __restrict__ part, const GmresState* __restrict__ st)
{
    __shared__ double sh[GM_BS / 64][GM_MAXM + 1];
    __shared__ VT hs[NV];
    if (!st->active) return;
    if ((int)threadIdx.x < NV)
        hs[threadIdx.x] = (int)threadIdx.x <= j ? (VT)st->hc[threadIdx.x] : VT(0);
    __syncthreads();
    constexpr int N1 = NV < GM_HALF ? NV : GM_HALF;
    const int base = lblock() * GM_BS * R + threadIdx.x;
    double acc[NV], nrm = 0.0;
#pragma unroll
    for (int i = 0; i < NV; ++i) acc[i] = 0.0;
#pragma unroll 1
    for (int r = 0; r < R; ++r) {
        const int row = base + r * GM_BS;
        if (row >= n) break;
        VT v[N1];
        VT wr = w[row];
#pragma unroll
        for (int i = 0; i < N1; ++i) v[i] = basis_at(V, ldv, min(i, j), row);
#pragma unroll
        for (int i = 0; i < N1; ++i) wr = kfma(-hs[i], v[i], wr);
        if constexpr (NV > N1) {
#pragma unroll
            for (int i = N1; i < NV; ++i) v[i - N1] = basis_at(V, ldv, min(i, j), row);
#pragma unroll
            for (int i = N1; i < NV; ++i) wr = kfma(-hs[i], v[i - N1], wr);
        }
        w[row] = wr;
        nrm = fma(to_d(wr), to_d(wr), nrm);
        if (DOTS) {
            if constexpr (NV > N1) {
#pragma unroll
                for (int i = N1; i < NV; ++i) acc[i] = fma(to_d(wr), to_d(v[i - N1]), acc[i]);
                const int again = opaque(row);  // loaded again, not kept
#pragma unroll
                for (int i = 0; i < N1; ++i) v[i] = basis_at(V, ldv, i, again);
            }
#pragma unroll
            for (int i = 0; i < N1; ++i) acc[i] = fma(to_d(wr), to_d(v[i]), acc[i]);
        }
    }
    if (DOTS) dot_partials<NV>(acc, j, sh);
    if (norm) norm_partial(nrm, sh);
    write_partials(sh, DOTS ? j + 1 : 0, norm, S, part);
}

// Adds the block partials of a pass and does the step's small dense work, in
// one workgroup: 32 running sums per value (block g to sum g mod 32), added
// in the persistent form's order.  The loads of a value's sum are the
// kernel's time: 8 per thread at level 8's 257 blocks, all in flight, 4.8 us
// (641 blocks, 20 per thread: 6.9 us).
enum { RED_BNORM, RED_START, RED_FIRST, RED_AGAIN, RED_NORM };
__global__ void __launch_bounds__(GM_RED)
k_reduce(int what, int mgs, int j, int nv, int norm, int S, const double* __restrict__ part, int G,
         GmresState* __restrict__ st, int* __restrict__ host_active)
{
    __shared__ double s32[2][32][33];
    __shared__ double s_cs[2 * GM_MAXM], s_g[GM_MAXM], s_carry[GM_MAXM + 1], s_h[GM_MAXM + 8];
    if (what == RED_START ? st->converged : (what != RED_BNORM && !st->active)) return;
    const int t = threadIdx.x, i = t & 31, c = t >> 5;
    if (what == RED_NORM && t >= GM_RED - 128) {
        const int e = t - (GM_RED - 128);
        s_cs[e] = st->cs[e];
        if (e <= GM_MAXM) s_carry[e] = st->carry[e];
        if (e < GM_MAXM) s_h[e] = st->hcol[e];
    }
    for (int v0 = 0; v0 < S; v0 += 32) {
        const int v = v0 + i;
        const bool mine = v < nv || (norm && v == S - 1);
        double a = 0.0;
        if (mine) {
            int g = c;
            for (; g + 7 * 32 < G; g += 8 * 32) {
                double u[8];
#pragma unroll
                for (int q = 0; q < 8; ++q) u[q] = part[(size_t)(g + 32 * q) * S + v];
#pragma unroll
                for (int q = 0; q < 8; ++q) a += u[q];
            }
            for (; g < G; g += 32) a += part[(size_t)g * S + v];
        }
        s32[v0 / 32][c][i] = a;
    }
    __syncthreads();
    if (t >= 64) return;
    // lane l: the total of value l (l < S)
    const int lane = t;
    double tot = 0.0;
    if (lane < S) {
        const double(*p)[33] = s32[lane >> 5];
        tot = p[0][i] + p[16][i];
#pragma unroll
        for (int q = 1; q < 16; ++q) tot += p[q][i] + p[q + 16][i];
    }
    const double last = readlane_d(tot, S - 1);
    if (what == RED_BNORM) {
        if (lane == 0) {
            const double bn = sqrt(last);
            st->bnorm = bn > 0.0 ? bn : 1.0;
        }
    } else if (what == RED_START) {
        if (lane == 0) {
            const double beta = sqrt(last);
            st->beta = beta;
            st->rel = beta / st->bnorm;
            st->k = 0;
            st->iters0 = st->iters;
            if (st->rel <= st->rtol || beta == 0.0) {
                st->converged = 1;
                st->active = 0;
            } else if (st->iters >= st->max_iters) {
                st->active = 0;
            } else {
                st->active = 1;
                st->carry[0] = beta;
                st->cycles += 1;
            }
        }
    } else if (what == RED_FIRST) {
        const double h = mgs ? mgs_solve<GM_MAXM>(tot, j, st->L, GM_MAXM, lane) : tot;
        if (lane <= j) {
            st->hc[lane] = h;
            st->hcol[lane] = h;
        }
    } else if (what == RED_AGAIN) {
        if (lane <= j) {
            st->hc[lane] = tot;
            st->hcol[lane] += tot;
        }
    } else {
        const double hn = sqrt(last);
        // the products of the next basis vector, w / hn rounded as it is stored
        if (mgs && lane < nv) {
            const double inv = 1.0 / hn;
            st->L[(j + 1) * GM_MAXM + lane] = tot * (mgs == 2 ? to_d((float)inv) : inv);
        }
        const double stop = fmax(st->rtol * st->bnorm, st->inner_rtol * st->beta);
        const GivensOut o = krylov_givens(j, st->m, s_h, hn, stop, st->iters0, st->max_iters, s_cs,
                                          s_g, s_carry, st->R, GM_MAXM);
        if (lane == 0) {
            st->cs[2 * j] = s_cs[2 * j];
            st->cs[2 * j + 1] = s_cs[2 * j + 1];
            st->g[j] = s_g[j];
            st->carry[j + 1] = s_carry[j + 1];
            st->hn = hn;
            st->k = j + 1;
            st->iters = o.iters;
            if (!o.cont) {
                st->active = 0;
                *host_active = 0;
            }
        }
    }
}

// y = R^{-1} g at the end of a cycle.
__global__ void __launch_bounds__(64)
k_solve_y(GmresState* __restrict__ st)
{
    if (st->converged) return;
    const int k = st->k;
    const double y = krylov_solve_y(k, st->R, GM_MAXM, st->g);
    if ((int)threadIdx.x < k) st->y[threadIdx.x] = y;
    if (threadIdx.x == 0) st->active = 0;
}

// x += sum_i y_i v_i, accumulated in FP64.
template <typename VT>
__global__ void __launch_bounds__(GM_BS)
k_xupdate(int n, const VT* __restrict__ V, size_t ldv, const GmresState* __restrict__ st)
{
    __shared__ double ys[GM_MAXM];
    if (st->converged) return;
    const int k = st->k;
    if (k == 0) return;
    if ((int)threadIdx.x < k) ys[threadIdx.x] = st->y[threadIdx.x];
    __syncthreads();
    const int row = lblock() * GM_BS + threadIdx.x;
    if (row >= n) return;
    double s = 0.0;
    int i = 0;
    for (; i + 8 <= k; i += 8) {
        VT v[8];
#pragma unroll
        for (int q = 0; q < 8; ++q) v[q] = V[(size_t)(i + q) * ldv + row];
#pragma unroll
        for (int q = 0; q < 8; ++q) s = fma(to_d(v[q]), ys[i + q], s);
    }
    for (; i < k; ++i) s = fma(to_d(V[(size_t)i * ldv + row]), ys[i], s);
    st->x[row] += s;
}

__global__ void k_fill0(int n, double* __restrict__ x)
{
    const int i = lblock() * blockDim.x + threadIdx.x;
    if (i < n) x[i] = 0.0;
}

// ---------------------------------------------------------------- driver --
int prepare_work(phg_matrix_s* A, int prec, int m, int ortho, GmresWork** out)
{
    auto& slot = A->work[2 * prec + (ortho == PHG_MGS ? 0 : 1)];
    const int n = A->n_rows;
    // The persistent form's rows per thread where it runs.  Above, as many as
    // leave about one workgroup per CU: the sums have few partials and the
    // workgroups end together (level 8, 5 rows on 257 workgroups: the
    // reducing workgroup took 4.8 us instead of 6.9 with 641 partials).
    const int R = n <= GM_BS * KR_RPT * KR_MAXG
                      ? KR_RPT
                      : std::max(KR_RPT, (int)std::lround((double)n / (GM_BS * KR_MAXG)));
    const int G = (int)(((long)n + GM_BS * R - 1) / (GM_BS * R));
    if (n > GM_MAXN) {
        set_error("gmres: matrix too large for one device workspace");
        return PHG_ERR_ARG;
    }
    if (!slot || slot->m < m) {
        std::unique_ptr<GmresWork> w(new GmresWork());
        w->n = n;
        w->m = m;
        w->prec = prec;
        w->R = R;
        w->G = G;
        w->ldv = ((size_t)n + 63) / 64 * 64;
        slot.reset(w.release());
    }
    *out = slot.get();
    return PHG_OK;
}

// What the launch-per-pass form needs beside: not allocated where every
// cycle is a persistent launch.
int prepare_passes(GmresWork* w)
{
    if (w->host) return PHG_OK;
    const size_t es = w->prec == PHG_F64 ? 8 : 4;
    w->S = w->m <= 32 ? 32 : 64;
    PHG_HIP(w->V.alloc((size_t)w->m * w->ldv * es));
    PHG_HIP(w->W.alloc(2 * w->ldv * es));
    PHG_HIP(w->part.alloc((size_t)w->G * w->S));
    PHG_HIP(w->st.alloc(1));
    PHG_HIP(hipHostMalloc((void**)&w->host, sizeof(GmresState), hipHostMallocDefault));
    return PHG_OK;
}

template <typename VT, typename MT, int NV, bool SHORT>
void step_nv(const Ell<MT>& E, GmresWork* w, const VT* src, VT* dst, int j, hipStream_t s)
{
    hipLaunchKernelGGL(HIP_KERNEL_NAME(k_step_spmv<VT, MT, NV, SHORT>), dim3(w->G), dim3(GM_BS), 0, s,
                       w->n, w->R, E.width, E.col.p, E.val.p, src, (VT*)w->V.p, w->ldv, dst, j,
                       w->S, w->part.p, w->st.p);
}
template <typename VT, int NV>
void update_nv(GmresWork* w, VT* dst, int j, bool dots, bool norm, hipStream_t s)
{
    const VT* V = (const VT*)w->V.p;
    const dim3 grid(w->G), block(GM_BS);
    if (dots)
        hipLaunchKernelGGL(HIP_KERNEL_NAME(k_update<VT, NV, true>), grid, block, 0, s, w->n, w->R,
                           dst, V, w->ldv, j, (int)norm, w->S, w->part.p, w->st.p);
    else
        hipLaunchKernelGGL(HIP_KERNEL_NAME(k_update<VT, NV, false>), grid, block, 0, s, w->n, w->R,
                           dst, V, w->ldv, j, (int)norm, w->S, w->part.p, w->st.p);
}

// f(vectors of the kernel for step j, as a constant)
template <typename F>
void by_step(int j, F f)
{
    switch (j / 8) {
    case 0: return f(std::integral_constant<int, 8>());
    case 1: return f(std::integral_constant<int, 16>());
    case 2: return f(std::integral_constant<int, 24>());
    case 3: return f(std::integral_constant<int, 32>());
    case 4: return f(std::integral_constant<int, 40>());
    case 5: return f(std::integral_constant<int, 48>());
    case 6: return f(std::integral_constant<int, 56>());
    default: return f(std::integral_constant<int, 64>());
    }
}

template <typename VT, typename MT>
void step(const Ell<MT>& E, GmresWork* w, const VT* src, VT* dst, int j, hipStream_t s)
{
    by_step(j, [&](auto nv) {
        constexpr int NV = decltype(nv)::value;
        if (E.width >= 1 && E.width <= ELL_MAXW) step_nv<VT, MT, NV, true>(E, w, src, dst, j, s);
        else step_nv<VT, MT, NV, false>(E, w, src, dst, j, s);
    });
}

template <typename VT>
void update(GmresWork* w, VT* dst, int j, bool dots, bool norm, hipStream_t s)
{
    by_step(j, [&](auto nv) { update_nv<VT, decltype(nv)::value>(w, dst, j, dots, norm, s); });
}

// Steps j0 .. j1-1 of a cycle of m, then with `end` the cycle's end.
template <typename VT, typename MT>
void enqueue_cycle(phg_matrix_s* A, const Ell<MT>& E, GmresWork* w, int m, int j0, int j1, bool end,
                   bool cgs, hipStream_t s)
{
    const int n = w->n, G = w->G, S = w->S;
    const size_t ldv = w->ldv;
    VT* V = (VT*)w->V.p;
    VT* W0 = (VT*)w->W.p;
    VT* W1 = W0 + ldv;
    double* part = w->part.p;
    GmresState* st = w->st.p;
    const int mgs = cgs ? 0 : (sizeof(VT) == 4 ? 2 : 1);
    const dim3 grid(G), block(GM_BS), one(1), red(GM_RED);
    for (int j = j0; j < j1; ++j) {
        VT* src = (j & 1) ? W1 : W0;
        VT* dst = (j & 1) ? W0 : W1;
        step<VT, MT>(E, w, src, dst, j, s);
        hipLaunchKernelGGL(k_reduce, one, red, 0, s, (int)RED_FIRST, mgs, j, j + 1, 0, S, part, G,
                           st, &w->host->active);
        if (cgs) {
            update<VT>(w, dst, j, true, false, s);
            hipLaunchKernelGGL(k_reduce, one, red, 0, s, (int)RED_AGAIN, mgs, j, j + 1, 0, S, part,
                               G, st, &w->host->active);
        }
        const bool dots = !cgs && j + 1 < m;
        update<VT>(w, dst, j, dots, true, s);
        hipLaunchKernelGGL(k_reduce, one, red, 0, s, (int)RED_NORM, mgs, j, dots ? j + 1 : 0, 1, S,
                           part, G, st, &w->host->active);
    }
    if (!end) return;
    hipLaunchKernelGGL(k_solve_y, one, dim3(64), 0, s, st);
    hipLaunchKernelGGL(HIP_KERNEL_NAME(k_xupdate<VT>), dim3((n + GM_BS - 1) / GM_BS), block, 0, s,
                       n, V, ldv, st);
    hipLaunchKernelGGL(HIP_KERNEL_NAME(k_residual<VT>), grid, block, 0, s, n, w->R, A->ell64.width,
                       A->ell64.col.p, A->ell64.val.p, W0, S, part, st);
    hipLaunchKernelGGL(k_reduce, one, red, 0, s, (int)RED_START, mgs, 0, 0, 1, S, part, G, st,
                       &w->host->active);
}

// iters, cycles: what a solve that is continued from x has done.
template <typename VT, typename MT>
int gmres_passes(phg_matrix_s* A, const Ell<MT>& E, GmresWork* w, const double* b, double* x,
                 const phg_gmres_opts& o, int iters, int cycles, phg_gmres_info* info, hipStream_t s)
{
    int rc = prepare_passes(w);
    if (rc) return rc;
    const int n = w->n, m = o.restart, G = w->G, S = w->S;
    VT* W0 = (VT*)w->W.p;
    double* part = w->part.p;
    GmresState* st = w->st.p;
    const dim3 grid(G), block(GM_BS), one(1), red(GM_RED);
    const bool cgs = o.ortho == PHG_CGS2;

    // parameters of the solve
    GmresState& init = *w->host;
    memset(&init, 0, sizeof init);
    init.m = m;
    init.rtol = o.rtol;
    init.inner_rtol = (o.precision == PHG_F64) ? 0.0 : o.inner_rtol;
    init.max_iters = o.max_iters;
    init.iters = iters;
    init.cycles = cycles;
    init.b = b;
    init.x = x;
    PHG_HIP(hipMemcpyAsync(st, &init, sizeof init, hipMemcpyHostToDevice, s));
    if (!o.use_x0) hipLaunchKernelGGL(k_fill0, dim3((n + 255) / 256), dim3(256), 0, s, n, x);
    hipLaunchKernelGGL(k_sumsq, grid, block, 0, s, n, w->R, b, S, part);
    hipLaunchKernelGGL(k_reduce, one, red, 0, s, (int)RED_BNORM, 0, 0, 0, 1, S, part, G, st,
                       &w->host->active);
    hipLaunchKernelGGL(HIP_KERNEL_NAME(k_residual<VT>), grid, block, 0, s, n, w->R, A->ell64.width,
                       A->ell64.col.p, A->ell64.val.p, W0, S, part, st);
    hipLaunchKernelGGL(k_reduce, one, red, 0, s, (int)RED_START, 0, 0, 0, 1, S, part, G, st,
                       &w->host->active);
    PHG_HIP(hipGetLastError());

    // the cycle in parts: steps from[c] .. from[c + 1] - 1, the last with its
    // end.  Above 32 steps chunks end at steps 16, 32 (with 16 or more left)
    // and m, and after each but the last the host looks whether the solve still
    // runs: an idle step is 4 or 6 launches of 1.5 us, a look costs 20 us.
    // Level 5, restart 64, FP64 CGS2 of 25 steps: 1072 -> 810 us.
    const int parts = m <= 32 ? 1 : m < 48 ? 3 : 4;
    const int from[5] = {0, parts == 1 ? m : 16, parts == 3 ? m : 32, m, m};
    const auto enqueue = [&](int c, hipStream_t cs) {
        enqueue_cycle<VT, MT>(A, E, w, m, from[c], from[c + 1], c == parts - 1, cgs, cs);
    };
    // captured; replayed only when built (or found current) here
    if (o.graph) {
        const void* key[2] = {E.val.p, A->ell64.val.p};
        const bool same = w->captured && w->key_m == m && w->key_ortho == o.ortho &&
                          !memcmp(key, w->key, sizeof key);
        if (!same) {
            w->drop_graphs();
            // recorded on the caller's stream; the null stream cannot be
            // captured, so for it on a stream of the workspace (a stream
            // per workspace would also take a share of the process's few
            // hardware queues from the caller's own streams)
            hipStream_t cs = s;
            if (!cs) {
                if (!w->cap) PHG_HIP(hipStreamCreateWithFlags(&w->cap, hipStreamNonBlocking));
                cs = w->cap;
            }
            for (int c = 0; c < parts; ++c) {
                hipGraph_t g = nullptr;
                PHG_HIP(hipStreamBeginCapture(cs, hipStreamCaptureModeThreadLocal));
                enqueue(c, cs);
                PHG_HIP(hipStreamEndCapture(cs, &g));
                hipError_t e = hipGraphInstantiate(&w->exec[c], g, nullptr, nullptr, 0);
                (void)hipGraphDestroy(g);
                PHG_HIP(e);
            }
            w->captured = true;
            memcpy(w->key, key, sizeof key);
            w->key_m = m;
            w->key_ortho = o.ortho;
        }
    }

    for (;;) {
        PHG_HIP(hipMemcpyAsync(w->host, st, sizeof(GmresState), hipMemcpyDeviceToHost, s));
        PHG_HIP(hipStreamSynchronize(s));
        if (w->host->converged || !w->host->active) break;
        for (int c = 0; c < parts; ++c) {
            if (o.graph) {
                PHG_HIP(hipGraphLaunch(w->exec[c], s));
            } else {
                enqueue(c, s);
                PHG_HIP(hipGetLastError());
            }
            if (c < parts - 2) {
                PHG_HIP(hipStreamSynchronize(s));
                if (!*(volatile int*)&w->host->active) c = parts - 2;  // the end is next
            }
        }
    }
    const GmresState& h = *w->host;
    if (info) {
        info->iterations = h.iters;
        info->restarts = h.cycles;
        info->rel_residual = h.rel;
        info->converged = h.converged;
    }
    return h.converged ? PHG_OK : PHG_ERR_NOCONV;
}

}  // namespace

int gmres_solve(phg_matrix_s* A, const double* b, double* x, const phg_gmres_opts* opts,
                phg_gmres_info* info, hipStream_t s)
{
    phg_gmres_opts o = *opts;
    if (o.restart < 1 || o.restart > GM_MAXM) {
        set_error("gmres: restart must be in 1..64");
        return PHG_ERR_ARG;
    }
    if (o.ortho != PHG_MGS && o.ortho != PHG_CGS2) {
        set_error("gmres: ortho must be PHG_MGS or PHG_CGS2");
        return PHG_ERR_ARG;
    }
    if (A->n_rows != A->n_cols) {
        set_error("gmres: matrix is not square");
        return PHG_ERR_ARG;
    }
    if (info) memset(info, 0, sizeof *info);
    if (A->n_rows == 0) {
        if (info) info->converged = 1;
        return PHG_OK;
    }
    int rc = ensure_ell64(A, s);
    if (rc) return rc;
    GmresWork* w = nullptr;
    rc = prepare_work(A, o.precision, o.restart, o.ortho, &w);
    if (rc) return rc;
    if (o.precision == PHG_F32) rc = ensure_ell32(A, s);
    else if (o.precision != PHG_F64) rc = ensure_ell16(A, s);
    if (rc) return rc;

    rc = PERSIST_NOT_HERE;
    int iters = 0, cycles = 0;
    if (o.persistent) {
        // one launch per restart cycle
        int launches = 0;
        double ms = 0.0;
        rc = persist_solve(A, &w->persist, 1, b, x, o, false, false, 1, 1, &launches, &ms, s);
        const PState* st = w->persist.host;
        if (rc == PERSIST_NO_START) {
            // the launches per pass need no CUs at the same time; they give
            // the same bits from here
            if (st->cycles > 0) o.use_x0 = 1;
            iters = st->iters, cycles = std::max(0, st->cycles - 1);
            if (info) info->cycle_launches = launches, info->cycle_ms = ms;
        }
        if (rc == PHG_OK) {
            const PState& h = *st;
            if (info) {
                info->iterations = h.iters;
                info->restarts = h.cycles;
                info->rel_residual = h.rel;
                info->converged = h.converged;
                info->cycle_launches = launches;
                info->cycle_ms = ms;
            }
            rc = h.converged ? PHG_OK : PHG_ERR_NOCONV;
        }
    }
    if (rc == PERSIST_NOT_HERE || rc == PERSIST_NO_START) {
        if (o.precision == PHG_F64)
            rc = gmres_passes<double, double>(A, A->ell64, w, b, x, o, iters, cycles, info, s);
        else if (o.precision == PHG_F32)
            rc = gmres_passes<float, float>(A, A->ell32, w, b, x, o, iters, cycles, info, s);
        else
            rc = gmres_passes<float, uint16_t>(A, A->ell16, w, b, x, o, iters, cycles, info, s);
    }
    if (info) info->refinements = o.precision == PHG_F64 ? 0 : info->restarts;
    return rc;
}

}  // namespace phg
