// Batched restarted GMRES(m): K <= 64 independent systems A x_q = b_q that
// share one matrix, on gfx950.
//
// Each column keeps its own Krylov space, Hessenberg matrix, Givens
// rotations and stopping test, exactly as K separate solves would (no block
// Krylov coupling), while every matrix read of an Arnoldi step serves all K
// columns (one SpMM instead of K SpMVs).  It is the form the callers with
// several right-hand sides per operator need: the eight mass solves of one
// SphereJacobian::calc2 (src/sjacobian.cpp:136-362: 16 idt_.solve calls with
// 8 distinct right-hand sides) and the implicit-step solves of the ensemble
// members that share one mesh level.
//
// Layout: vectors are n x KP row-major (entry (i, q) at i * KP + q), KP = K
// rounded up to a power of two; a thread owns one (row, column) pair, so a
// wavefront covers 64 / KP consecutive rows and the gathers of one ELL entry
// read KP consecutive words.  The caller's B and X are n x K, row-major.
//
// Orthogonalisation: classical Gram-Schmidt with one re-orthogonalisation
// pass (CGS2), or a single pass (CGS1) for well-conditioned operators such
// as the mass matrix.  Precision: FP64 throughout, or the mixed form (FP32
// basis, FP32/BF16 matrix values, FP64 dots, Hessenberg, Givens, update and
// a true FP64 residual at every restart, i.e. iterative refinement).
//
// Reductions are deterministic and do not depend on the column's position
// or on the other columns: a column's result is bit-identical whatever else
// is in the batch, provided K is the same.  In the persistent form below it is the
// same bits for every K, in the launches for every K of one KP; which form
// runs depends on K too.  A restart cycle is captured in
// one hipGraph and replayed; the host reads a K-entry summary per cycle.
//
// Where the columns' rows fit the chip in few enough launches, the solve runs
// as persistent launches instead (persist.hip; persistent_rounds below has
// the rule and what both sides measured).
#include <cmath>
#include <cstdlib>
#include <cstring>
#include <map>
#include <mutex>
#include <type_traits>

#include "ell.h"
#include "persist.h"
#include "phg_internal.h"

namespace phg {

constexpr int BB_BS = 256;
constexpr int BB_MAXM = 32;
constexpr int BB_MAXK = 64;
constexpr int BB_RPT = 16;  // largest rows per thread of a launch shape

// A restart cycle runs its Arnoldi steps in chunks ending at steps 4, 8, 16,
// 24 and 32; after each chunk but the last the host reads how many columns
// are still running and, when none is, ends the cycle there.  The steps
// skipped would have found every column stopped: same results, without the
// launches (and the preconditioner applications) of a full cycle, which
// matters for solves that stop after a few steps (multigrid-preconditioned,
// warm-started).
constexpr int BB_NCHUNK = 5;
__host__ __device__ constexpr int bb_chunk_end(int c) { return c < 2 ? 4 * (c + 1) : 8 * c; }

struct BCol {
    double H[(BB_MAXM + 1) * BB_MAXM];  // unrotated Hessenberg, H[i * BB_MAXM + j]
    double R[BB_MAXM * BB_MAXM];        // rotated, upper triangular
    double cs[BB_MAXM], sn[BB_MAXM], g[BB_MAXM], carry[BB_MAXM + 1], y[BB_MAXM];
    double hc[BB_MAXM + 1];             // coefficients of the current CGS pass
    double beta, bnorm, rel, hn;
    int k, active, converged, iters, iters0, cycles, pad0, pad1;
};

struct BSum {
    double rel;
    int active, converged, iters, cycles;
};

// The caller's arrays, read by the kernels of the captured cycle: a graph
// serves every pair of them (capturing one again takes 2 ms and more, as long
// as a whole preconditioned solve at level 7).
struct BIo {
    const double* B;
    double* X;
};

struct BatchWork {
    int n = 0, m = 0, kp = 0, G = 0, prec = 0, rpt = 0;
    DevBuf<char> V, W;    // (m+1) x n x kp and 2 x n x kp of the Krylov type
    DevBuf<char> Z;       // m x n x kp preconditioned vectors (with a preconditioner)
    DevBuf<double> part;  // (m+2) x kp x G block partials
    DevBuf<BCol> cols;    // kp
    DevBuf<BSum> sum;     // kp
    DevBuf<BIo> io;
    BSum* host = nullptr;
    DevBuf<int> nact;      // columns still running in the current cycle
    int* hnact = nullptr;  // its host copy (pinned)
    hipStream_t cap = nullptr;
    // one graph per chunk of Arnoldi steps of a cycle, then the cycle's end
    hipGraphExec_t exec[BB_NCHUNK + 1] = {};
    bool captured = false;
    const void* key[2] = {nullptr, nullptr};
    int key_m = 0, key_ortho = -1, key_k = 0, key_maxit = 0;
    const void* key_pc = nullptr;
    double key_rtol = 0.0, key_inner = 0.0;
    void drop_graphs()
    {
        for (auto& e : exec)
            if (e) (void)hipGraphExecDestroy(e), e = nullptr;
        captured = false;
    }
    ~BatchWork()
    {
        drop_graphs();
        if (cap) (void)hipStreamDestroy(cap);
        if (host) (void)hipHostFree(host);
        if (hnact) (void)hipHostFree(hnact);
    }
};

void batch_destroy(BatchWork* w) { delete w; }

namespace {

__device__ __forceinline__ double wave_sum64(double v)
{
    for (int off = 32; off > 0; off >>= 1) v += __shfl_xor(v, off, 64);
    return v;
}

// Sum over the lanes of a wavefront that hold the same column (lane % KP).
__device__ __forceinline__ double col_wave_sum(double v, int KP)
{
    for (int off = KP; off < 64; off <<= 1) v += __shfl_xor(v, off, 64);
    return v;
}

// Fixed-order sum of np partials by one wavefront; every lane returns it.
__device__ __forceinline__ double wave_sum_partials(const double* __restrict__ p, int np)
{
    const int lane = threadIdx.x & 63;
    double s = 0.0;
    int b = lane;
    for (; b + 64 * 7 < np; b += 64 * 8) {
        double v[8];
#pragma unroll
        for (int u = 0; u < 8; ++u) v[u] = p[b + 64 * u];
#pragma unroll
        for (int u = 0; u < 8; ++u) s += v[u];
    }
    for (; b < np; b += 64) s += p[b];
    return wave_sum64(s);
}

__device__ __forceinline__ double readlane_d(double v, int lane)
{
    const unsigned long long u = __double_as_longlong(v);
    const unsigned lo = __builtin_amdgcn_readlane((unsigned)u, lane);
    const unsigned hi = __builtin_amdgcn_readlane((unsigned)(u >> 32), lane);
    return __longlong_as_double((long long)(((unsigned long long)hi << 32) | lo));
}

template <typename T>
__device__ __forceinline__ double dd(T v) { return (double)v; }

// One term of a row's sum: r + val * (x * s) in FP64 (no fused multiply-add),
// fmaf(val, x * s, r) in FP32.
template <typename VT, typename MT>
struct BTerm;
template <>
struct BTerm<double, double> {
    __device__ __forceinline__ static double add(double r, double v, double x, double s)
    {
        return r + v * (x * s);
    }
};
template <typename MT>
struct BTerm<float, MT> {
    __device__ __forceinline__ static float add(float r, MT v, float x, float s)
    {
        return fmaf(ell_val_f32(v), x * s, r);
    }
};

// Row `row` of A times column q of X (row-major, ldx columns), X scaled by s.
// ELL_MAXW entries at a time: their slots are loaded first (past the width
// the last one again, in bounds), then their gathers.  280,000 rows of 27
// entries, 9 FP32 columns: bk_step_spmm 83 us, entry by entry 247.
template <typename VT, typename MT>
__device__ __forceinline__ VT brow(int n, int width, int row, const int* __restrict__ col,
                                   const MT* __restrict__ val, const VT* __restrict__ X, int ldx,
                                   int q, VT s)
{
    VT r = VT(0);
#pragma unroll 1
    for (int k0 = 0; k0 < width; k0 += ELL_MAXW) {
        int c[ELL_MAXW];
        MT v[ELL_MAXW];
        VT xv[ELL_MAXW];
#pragma unroll
        for (int k = 0; k < ELL_MAXW; ++k) {
            const size_t o = ell_slot(k0 + k, width, n, row);
            c[k] = col[o];
            v[k] = val[o];
        }
#pragma unroll
        for (int k = 0; k < ELL_MAXW; ++k) xv[k] = X[(size_t)c[k] * ldx + q];
#pragma unroll
        for (int k = 0; k < ELL_MAXW; ++k) {
            const VT t = BTerm<VT, MT>::add(r, v[k], xv[k], s);
            r = k0 + k < width ? t : r;
        }
    }
    return r;
}

// A thread's dots acc[i], i <= j (inactive threads: zeros), as block partials
// part[((out0 + i) * KP + q) * G + block].  All threads of the block call it.
template <int NV>
__device__ __forceinline__ void put_partials(const double (&acc)[NV], int last, int KP, int out0,
                                             double* __restrict__ part, int G)
{
    constexpr int LB = NV < 8 ? NV : 8;  // dots per round through LDS
    __shared__ double sh[BB_BS / 64][LB][BB_MAXK];
    const int wid = threadIdx.x >> 6, lane = threadIdx.x & 63;
#pragma unroll
    for (int i0 = 0; i0 < NV; i0 += LB) {
        if (i0 > last) break;
#pragma unroll
        for (int u = 0; u < LB; ++u) {
            const double s = col_wave_sum(acc[i0 + u], KP);
            if (lane < KP) sh[wid][u][lane] = s;
        }
        __syncthreads();
        for (int e = threadIdx.x; e < LB * KP; e += BB_BS) {
            const int u = e / KP, qq = e % KP;
            if (i0 + u <= last) {
                double s = 0.0;
#pragma unroll
                for (int ww = 0; ww < BB_BS / 64; ++ww) s += sh[ww][u][qq];
                part[((size_t)(out0 + i0 + u) * KP + qq) * G + lblock()] = s;
            }
        }
        __syncthreads();
    }
}

// brow of this thread's rows base + t * RB (t < RPT) of column q, and xo[t]
// = X(row, q); w[t] = xo[t] = 0 for rows at or past n and inactive columns.
// For rows of at most ELL_MAXW entries, RG rows at a time: every row's own
// entry and column/value slots (ell_slot: past the width the last slot
// again, in bounds) are loaded first, then every row's gathers, then the
// sums in brow's order; two memory round trips per group instead of three
// per row.  (Scalar loads of the slots, where 64 columns share a row, were
// slower: 265 instead of 242 us at level 7, FP32.)
template <typename VT, typename MT, int RPT, int RG>
__device__ __forceinline__ void brows(int n, int width, int KP, int q, int base, int RB, bool act,
                                      const int* __restrict__ col, const MT* __restrict__ val,
                                      const VT* __restrict__ X, VT s, VT (&xo)[RPT],
                                      VT (&w)[RPT])
{
    if (width >= 1 && width <= ELL_MAXW) {
#pragma unroll
        for (int g = 0; g < RPT; g += RG) {
            int c[RG][ELL_MAXW];
            MT v[RG][ELL_MAXW];
            VT xv[RG][ELL_MAXW];
#pragma unroll
            for (int u = 0; u < RG; ++u) {
                const int row = min(base + (g + u) * RB, n - 1);  // in bounds; unused past n
                xo[g + u] = X[(size_t)row * KP + q];
#pragma unroll
                for (int k = 0; k < ELL_MAXW; ++k) {
                    const size_t o = ell_slot(k, width, n, row);
                    c[u][k] = col[o];
                    v[u][k] = val[o];
                }
            }
#pragma unroll
            for (int u = 0; u < RG; ++u)
#pragma unroll
                for (int k = 0; k < ELL_MAXW; ++k) xv[u][k] = X[(size_t)c[u][k] * KP + q];
#pragma unroll
            for (int u = 0; u < RG; ++u) {
                VT r = VT(0);
#pragma unroll
                for (int k = 0; k < ELL_MAXW; ++k) {
                    const VT t = BTerm<VT, MT>::add(r, v[u][k], xv[u][k], s);
                    r = k < width ? t : r;
                }
                const bool in = act && base + (g + u) * RB < n;
                w[g + u] = in ? r : VT(0);
                xo[g + u] = in ? xo[g + u] : VT(0);
            }
        }
    } else {
#pragma unroll
        for (int t = 0; t < RPT; ++t) {
            const int row = base + t * RB;
            w[t] = VT(0);
            xo[t] = VT(0);
            if (act && row < n) {
                xo[t] = X[(size_t)row * KP + q];
                w[t] = brow<VT, MT>(n, width, row, col, val, X, KP, q, s);
            }
        }
    }
}

// Partial dots of w with v_0..v_j (v_j from `own` where given) of a thread's
// rows, V_LB vectors of all its rows at a time.  FP32 loads have no branch
// between them (past the last vector that one again, unused: steps with few
// vectors 55 instead of 67 us at level 7 x 64); FP64 ones stop at the last
// vector (180 instead of 187 us there).  With a test of every row and column
// before each load the steps with few vectors took 92 us.
constexpr int V_LB = 4;
template <typename VT, int RPT>
__device__ __forceinline__ void bdots(int j, const VT* own, const VT* __restrict__ V, size_t bs,
                                      int n, int KP, int q, int base, int RB, bool act,
                                      const VT* w, double* __restrict__ part, int G)
{
    const int last = own ? max(j - 1, 0) : j;
    for (int i0 = 0; i0 <= j; i0 += V_LB) {
        double acc[V_LB];
#pragma unroll
        for (int u = 0; u < V_LB; ++u) acc[u] = 0.0;
        if (act) {
            VT vb[V_LB][RPT];
#pragma unroll
            for (int u = 0; u < V_LB; ++u)
#pragma unroll
                for (int t = 0; t < RPT; ++t)
                    vb[u][t] = sizeof(VT) == 4 || i0 + u <= last
                                   ? V[(size_t)min(i0 + u, last) * bs +
                                       (size_t)min(base + t * RB, n - 1) * KP + q]
                                   : VT(0);
#pragma unroll
            for (int u = 0; u < V_LB; ++u)
#pragma unroll
                for (int t = 0; t < RPT; ++t)
                    acc[u] += dd(w[t]) * dd(own && i0 + u == j ? own[t] : vb[u][t]);
        }
        put_partials<V_LB>(acc, j - i0, KP, i0, part, G);
    }
}

// ---------------------------------------------------------------- kernels --
// The row kernels: a thread owns RPT (or R) rows base + t * RB of column q.
//
// Arnoldi step j: v_j = W_src / h (stored), W_dst = A v_j, partial dots of
// W_dst with v_0..v_j (first CGS pass).  PC: W_dst = A z_j (X = z_j = M^-1 v_j,
// the preconditioned vector), v_j has been stored.
template <typename VT, typename MT, int RPT, bool PC>
__global__ void __launch_bounds__(BB_BS)
bk_step_spmm(int n, int KP, int K, int width, const int* __restrict__ col,
             const MT* __restrict__ val, const VT* __restrict__ X, VT* __restrict__ V, size_t bs,
             VT* __restrict__ Wdst, int j, double* __restrict__ part, int G,
             const BCol* __restrict__ cols)
{
    const int q = threadIdx.x & (KP - 1);
    const int RB = BB_BS / KP;
    const int base = lblock() * RB * RPT + (int)threadIdx.x / KP;
    const bool act = q < K && cols[q].active;
    VT w[RPT], vj[RPT];
    if (act) {
        const double h = PC ? 1.0 : (j == 0 ? cols[q].beta : cols[q].hn);
        const VT inv = (VT)(1.0 / h);
        brows<VT, MT, RPT, (RPT < 4 ? RPT : 4)>(n, width, KP, q, base, RB, act, col, val, X, inv,
                                                vj, w);
#pragma unroll
        for (int t = 0; t < RPT; ++t) {
            const int row = base + t * RB;
            vj[t] = vj[t] * inv;
            if (row < n) {
                const size_t o = (size_t)row * KP + q;
                if (!PC) V[(size_t)j * bs + o] = vj[t];
                Wdst[o] = w[t];
            }
        }
    }
    bdots<VT, RPT>(j, PC ? nullptr : vj, V, bs, n, KP, q, base, RB, act, w, part, G);
}

// Right-preconditioned step: v_j = W_src / h (stored) for the preconditioner.
template <typename VT>
__global__ void __launch_bounds__(BB_BS)
bk_scale(int n, int KP, int K, const VT* __restrict__ Wsrc, VT* __restrict__ Vj, int j,
         const BCol* __restrict__ cols)
{
    const size_t e = (size_t)lblock() * BB_BS + threadIdx.x;
    if (e >= (size_t)n * KP) return;
    const int q = (int)(e % KP);
    if (q >= K || !cols[q].active) return;
    const double h = j == 0 ? cols[q].beta : cols[q].hn;
    Vj[e] = Wsrc[e] * (VT)(1.0 / h);
}

// Sums the partials of the nd dots of a pass, one wavefront per (i, column):
// pass 0 sets H(i, j), pass 1 adds the re-orthogonalisation correction.
__global__ void __launch_bounds__(BB_BS)
bk_reduce(int KP, int K, int nd, int j, int pass, const double* __restrict__ part, int G,
          BCol* __restrict__ cols)
{
    const int wv = lblock() * (BB_BS / 64) + ((int)threadIdx.x >> 6);
    if (wv >= nd * KP) return;
    const int i = wv / KP, q = wv % KP;
    if (q >= K || !cols[q].active) return;
    const double s = wave_sum_partials(part + ((size_t)i * KP + q) * G, G);
    if ((threadIdx.x & 63) == 0) {
        cols[q].hc[i] = s;
        if (pass == 0) cols[q].H[i * BB_MAXM + j] = s;
        else cols[q].H[i * BB_MAXM + j] += s;
    }
}

// w -= sum_{i<=j} hc_i v_i, then with `norm` the partial of ||w||^2 as value
// j + 1.  V_LB vectors of all a thread's rows at a time: level 7, 64 columns
// FP32, 15.5 vectors on average, 148 us, 5.0 TB/s, what a copy reaches here
// (row by row with all vectors of a row in flight 4.4 TB/s).
template <typename VT, int RPT>
__global__ void __launch_bounds__(BB_BS)
bk_update(int n, int KP, int K, VT* __restrict__ W, const VT* __restrict__ V, size_t bs, int j,
          int norm, double* __restrict__ part, int G, const BCol* __restrict__ cols)
{
    const int q = threadIdx.x & (KP - 1);
    const int RB = BB_BS / KP;
    const int base = lblock() * RB * RPT + (int)threadIdx.x / KP;
    const bool act = q < K && cols[q].active;
    double nrm[1] = {0.0};
    if (act) {
        VT w[RPT];
#pragma unroll
        for (int t = 0; t < RPT; ++t) w[t] = W[(size_t)min(base + t * RB, n - 1) * KP + q];
        for (int i0 = 0; i0 <= j; i0 += V_LB) {
            VT vb[V_LB][RPT], hv[V_LB];
#pragma unroll
            for (int u = 0; u < V_LB; ++u) {
                hv[u] = i0 + u <= j ? (VT)cols[q].hc[i0 + u] : VT(0);
#pragma unroll
                for (int t = 0; t < RPT; ++t)
                    vb[u][t] = i0 + u <= j ? V[(size_t)(i0 + u) * bs +
                                               (size_t)min(base + t * RB, n - 1) * KP + q]
                                           : VT(0);
            }
#pragma unroll
            for (int u = 0; u < V_LB; ++u)
#pragma unroll
                for (int t = 0; t < RPT; ++t) w[t] = w[t] - hv[u] * vb[u][t];
        }
#pragma unroll
        for (int t = 0; t < RPT; ++t) {
            const int row = base + t * RB;
            if (row < n) {
                W[(size_t)row * KP + q] = w[t];
                nrm[0] += dd(w[t]) * dd(w[t]);
            }
        }
    }
    if (norm) put_partials<1>(nrm, 0, KP, j + 1, part, G);
}

// The first CGS2 pass fused with the dots of the second (UPD): w -= sum hc_i
// v_i row by row, the row's v_0..v_j (j < NV, past j the last one again) kept in
// registers for the partial dots of the updated w: one read of the basis
// instead of two, the same bits.  Without UPD the dots alone.
template <typename VT, int NV, bool UPD>
__global__ void __launch_bounds__(BB_BS)
bk_update_dots(int n, int KP, int K, int R, VT* __restrict__ W, const VT* __restrict__ V, size_t bs,
               int j, double* __restrict__ part, int G, const BCol* __restrict__ cols)
{
    const int q = threadIdx.x & (KP - 1);
    const int RB = BB_BS / KP;
    const int base = lblock() * RB * R + (int)threadIdx.x / KP;
    const bool act = q < K && cols[q].active;
    double acc[NV];
#pragma unroll
    for (int i = 0; i < NV; ++i) acc[i] = 0.0;
    if (act) {
        VT hv[NV];
#pragma unroll
        for (int i = 0; i < NV; ++i) {
            const VT h = (VT)cols[q].hc[min(i, j)];
            hv[i] = UPD && i <= j ? h : VT(0);
        }
#pragma unroll 1
        for (int t = 0; t < R; ++t) {
            const int row = base + t * RB;
            if (row >= n) break;
            const size_t o = (size_t)row * KP + q;
            VT v[NV];
            VT w = W[o];
#pragma unroll
            for (int i = 0; i < NV; ++i) v[i] = V[(size_t)min(i, j) * bs + o];
            if (UPD) {
#pragma unroll
                for (int i = 0; i < NV; ++i) w = w - hv[i] * v[i];
                W[o] = w;
            }
#pragma unroll
            for (int i = 0; i < NV; ++i) acc[i] += dd(w) * dd(v[i]);
        }
    }
    put_partials<NV>(acc, j, KP, 0, part, G);
}

// Givens rotation of step j for each column (one wavefront per column) from
// H(0..j, j) and the norm partials; decides whether the column goes on.
__global__ void __launch_bounds__(BB_BS)
bk_givens(int KP, int K, int j, int m, const double* __restrict__ part, int G,
          BCol* __restrict__ cols, double rtol, double inner_rtol, int max_iters)
{
    const int q = lblock() * (BB_BS / 64) + ((int)threadIdx.x >> 6);
    if (q >= K) return;
    BCol* c = cols + q;
    if (!c->active) return;
    const int lane = threadIdx.x & 63;
    const double s = wave_sum_partials(part + ((size_t)(j + 1) * KP + q) * G, G);
    const double hreg = lane <= j ? c->H[lane * BB_MAXM + j] : 0.0;
    const double creg = lane < j ? c->cs[lane] : 0.0;
    const double sreg = lane < j ? c->sn[lane] : 0.0;
    const double hn = sqrt(s);
    double cur = readlane_d(hreg, 0);
    for (int i = 0; i < j; ++i) {
        const double cc = readlane_d(creg, i), sn = readlane_d(sreg, i);
        const double nxt = readlane_d(hreg, i + 1);
        const double t = cc * cur + sn * nxt;
        cur = -sn * cur + cc * nxt;
        if (lane == 0) c->R[i * BB_MAXM + j] = t;
    }
    const double r = hypot(cur, hn);
    const double cj = cur / r, sj = hn / r;
    const double carry = c->carry[j];
    const double gj = cj * carry, cn = -sj * carry;
    const int iters = c->iters0 + j + 1;
    const double stop = fmax(rtol * c->bnorm, inner_rtol * c->beta);
    const bool cont = !(fabs(cn) <= stop || !(hn > 0.0) || iters >= max_iters || j + 1 == m);
    if (lane == 0) {
        c->R[j * BB_MAXM + j] = r;
        c->H[(j + 1) * BB_MAXM + j] = hn;
        c->hn = hn;
        c->cs[j] = cj;
        c->sn[j] = sj;
        c->g[j] = gj;
        c->carry[j + 1] = cn;
        c->k = j + 1;
        c->iters = iters;
        if (!cont) c->active = 0;
    }
}

// y = R^{-1} g for each column that ran this cycle (one wavefront each:
// R staged in LDS by all lanes, back substitution by lane 0).
__global__ void __launch_bounds__(BB_BS)
bk_solve_y(int K, BCol* __restrict__ cols)
{
    __shared__ double Rs[BB_BS / 64][BB_MAXM * BB_MAXM];
    const int wid = threadIdx.x >> 6, lane = threadIdx.x & 63;
    const int q = lblock() * (BB_BS / 64) + wid;
    if (q >= K) return;
    BCol* c = cols + q;
    const int k = c->k;
    if (c->converged || k == 0) return;
    double* R = Rs[wid];
    for (int e = lane; e < k * k; e += 64) R[e] = c->R[(e / k) * BB_MAXM + (e % k)];
    const double gl = lane < k ? c->g[lane] : 0.0;
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    double y[BB_MAXM];
    for (int i = k - 1; i >= 0; --i) {
        double s = readlane_d(gl, i);
        for (int l = i + 1; l < k; ++l) s -= R[i * k + l] * y[l];
        y[i] = s / R[i * k + i];
    }
    if (lane == 0)
        for (int i = 0; i < k; ++i) c->y[i] = y[i];
}

// X += D (V y) per column (FP64 accumulation; D = dscale, or 1 when null: the
// diagonal right preconditioner); X is n x K (the caller's layout).  Eight
// vectors' loads at a time.
template <typename VT>
__global__ void __launch_bounds__(BB_BS)
bk_xupdate(int n, int KP, int K, int R, const VT* __restrict__ V, size_t bs,
           const BIo* __restrict__ io, const BCol* __restrict__ cols,
           const double* __restrict__ dscale)
{
    __shared__ double ys[BB_MAXM][BB_MAXK];
    for (int e = threadIdx.x; e < BB_MAXM * KP; e += BB_BS) {
        const int i = e / KP, qq = e % KP;
        ys[i][qq] = qq < K && i < cols[qq].k ? cols[qq].y[i] : 0.0;
    }
    __syncthreads();
    const int q = threadIdx.x & (KP - 1);
    const int RB = BB_BS / KP;
    const int base = lblock() * RB * R + (int)threadIdx.x / KP;
    if (q >= K) return;
    const int k = cols[q].k;
    if (cols[q].converged || k == 0) return;
    double* __restrict__ X = io->X;
    for (int t = 0; t < R; ++t) {
        const int row = base + t * RB;
        if (row >= n) break;
        const size_t o = (size_t)row * KP + q;
        double s = 0.0;
        for (int i0 = 0; i0 < k; i0 += 8) {
            VT v[8];
#pragma unroll
            for (int u = 0; u < 8; ++u) v[u] = V[(size_t)min(i0 + u, k - 1) * bs + o];
#pragma unroll
            for (int u = 0; u < 8; ++u) s += dd(v[u]) * ys[min(i0 + u, BB_MAXM - 1)][q];
        }
        X[(size_t)row * K + q] += dscale ? dscale[row] * s : s;
    }
}

// r = b - A x (FP64), W0 = r in the Krylov type, partial ||r||^2 per column.
template <typename VT>
__global__ void __launch_bounds__(BB_BS)
bk_residual(int n, int KP, int K, int R, int width, const int* __restrict__ col,
            const double* __restrict__ val, const BIo* __restrict__ io, VT* __restrict__ W0,
            double* __restrict__ part, int G, const BCol* __restrict__ cols)
{
    const double* __restrict__ B = io->B;
    const double* __restrict__ X = io->X;
    const int q = threadIdx.x & (KP - 1);
    const int RB = BB_BS / KP;
    const int base = lblock() * RB * R + (int)threadIdx.x / KP;
    double a[1] = {0.0};
    if (q < K && !cols[q].converged) {
        for (int t = 0; t < R; ++t) {
            const int row = base + t * RB;
            if (row >= n) break;
            const double s = brow<double, double>(n, width, row, col, val, X, K, q, 1.0);
            const VT w = (VT)(B[(size_t)row * K + q] - s);
            W0[(size_t)row * KP + q] = w;
            a[0] += dd(w) * dd(w);
        }
    }
    put_partials<1>(a, 0, KP, 0, part, G);
}

// ||b_q||^2 partials: the same reduction with B read as the vector.
__global__ void __launch_bounds__(BB_BS)
bk_sumsq(int n, int KP, int K, int R, const double* __restrict__ B, double* __restrict__ part,
         int G)
{
    const int q = threadIdx.x & (KP - 1);
    const int RB = BB_BS / KP;
    const int base = lblock() * RB * R + (int)threadIdx.x / KP;
    double a[1] = {0.0};
    if (q < K) {
        for (int t = 0; t < R; ++t) {
            const int row = base + t * RB;
            if (row >= n) break;
            const double b = B[(size_t)row * K + q];
            a[0] += b * b;
        }
    }
    put_partials<1>(a, 0, KP, 0, part, G);
}

// from: the columns of a solve that is continued from X (persist.h), or null.
__global__ void bk_set_bnorm(int KP, int K, const double* __restrict__ part, int G,
                             BCol* __restrict__ cols, BIo arrays, BIo* __restrict__ io,
                             const PState* __restrict__ from)
{
    if (lblock() == 0 && threadIdx.x == 0) *io = arrays;
    const int q = lblock() * (BB_BS / 64) + ((int)threadIdx.x >> 6);
    if (q >= K) return;
    const double s = wave_sum_partials(part + (size_t)q * G, G);
    if ((threadIdx.x & 63) == 0) {
        BCol* c = cols + q;
        const double bn = sqrt(s);
        c->bnorm = bn > 0.0 ? bn : 1.0;
        c->iters = from ? from[q].iters : 0;
        c->iters0 = c->iters;
        c->cycles = from ? max(0, from[q].cycles - 1) : 0;  // before the next one
        c->converged = from && !from[q].active;  // complete: left alone
        c->active = 0;
        c->k = 0;
    }
}

// Start of a restart cycle from the residual partials; writes the summary.
__global__ void bk_cycle_start(int KP, int K, const double* __restrict__ part, int G,
                               BCol* __restrict__ cols, BSum* __restrict__ sum, double rtol,
                               int max_iters)
{
    const int q = lblock() * (BB_BS / 64) + ((int)threadIdx.x >> 6);
    if (q >= K) return;
    BCol* c = cols + q;
    const bool done = c->converged;
    const double s = done ? 0.0 : wave_sum_partials(part + (size_t)q * G, G);
    if ((threadIdx.x & 63) != 0) return;
    if (!done) {
        const double beta = sqrt(s);
        // a whole restart cycle that lowered the true residual by less than
        // 1 % means it sits at its rounding floor above rtol: the column
        // stops there (not converged)
        const bool stalled = c->cycles > 0 && c->iters > c->iters0 && beta > 0.99 * c->beta;
        c->beta = beta;
        c->rel = beta / c->bnorm;
        c->k = 0;
        c->iters0 = c->iters;
        if (c->rel <= rtol || beta == 0.0) {
            c->converged = 1;
            c->active = 0;
        } else if (c->iters >= max_iters || stalled || !isfinite(beta)) {
            c->active = 0;
        } else {
            c->active = 1;
            c->carry[0] = beta;
            c->cycles += 1;
        }
    }
    BSum o;
    o.rel = c->rel;
    o.active = c->active;
    o.converged = c->converged;
    o.iters = c->iters;
    o.cycles = c->cycles;
    sum[q] = o;
}

// x = 0, of a continued solve only the columns that have not begun
__global__ void bk_fill0(size_t n, int K, double* __restrict__ x, const PState* __restrict__ from)
{
    const size_t i = (size_t)lblock() * blockDim.x + threadIdx.x;
    if (i >= n) return;
    if (!from || (from[i % K].active && from[i % K].cycles == 0)) x[i] = 0.0;
}

// ---------------------------------------------------------------- driver --
// The preconditioner works on FP64 vectors (the form it is used with).
template <typename VT>
void precond_apply(BatchPrecond* pc, int KP, const VT* v, VT* z, hipStream_t s);
template <>
void precond_apply<double>(BatchPrecond* pc, int KP, const double* v, double* z, hipStream_t s)
{
    pc->apply(KP, v, z, s);
}
template <>
void precond_apply<float>(BatchPrecond* pc, int KP, const float* v, float* z, hipStream_t s)
{
    pc->apply_f32(KP, v, z, s);
}

// The fused first-pass kernel (default on; PHG_BATCH_FUSED=0 selects the
// two-read form, which gives the same bits).
bool fused_update_dots()
{
    static const bool on = [] {
        const char* e = getenv("PHG_BATCH_FUSED");
        return !(e && e[0] == '0');
    }();
    return on;
}

int next_pow2(int k)
{
    int p = 1;
    while (p < k) p <<= 1;
    return p;
}

int blocks_for(int n, int kp, int rpt)
{
    const int rows_per_block = (BB_BS / kp) * rpt;
    return std::max(1, (n + rows_per_block - 1) / rows_per_block);
}

int prepare_batch(phg_matrix_s* A, int slot, int prec, int m, int kp, int rpt, bool pc,
                  BatchWork** out)
{
    BatchWork*& w = A->batch[slot];
    const int n = A->n_rows;
    if (!w || w->m < m || w->kp != kp || w->prec != prec) {
        batch_destroy(w);
        w = nullptr;
        std::unique_ptr<BatchWork> b(new BatchWork());
        b->n = n;
        b->m = m;
        b->kp = kp;
        b->prec = prec;
        const size_t es = prec == PHG_F64 ? 8 : 4;
        const size_t bs = (size_t)n * kp;
        PHG_HIP(b->V.alloc((size_t)(m + 1) * bs * es));
        PHG_HIP(b->W.alloc(2 * bs * es));
        // sized for the smallest rows-per-thread (most blocks)
        PHG_HIP(b->part.alloc((size_t)(m + 2) * kp * blocks_for(n, kp, 1)));
        PHG_HIP(b->cols.alloc(kp));
        PHG_HIP(b->sum.alloc(kp));
        PHG_HIP(b->io.alloc(1));
        PHG_HIP(hipHostMalloc((void**)&b->host, sizeof(BSum) * kp, hipHostMallocDefault));
        PHG_HIP(b->nact.alloc(1));
        PHG_HIP(hipHostMalloc((void**)&b->hnact, sizeof(int), hipHostMallocDefault));
        w = b.release();
    }
    if (w->rpt != rpt) {  // another launch shape: new block count, new graph
        w->rpt = rpt;
        w->G = blocks_for(n, kp, rpt);
        w->drop_graphs();
    }
    if (pc && !w->Z.p) PHG_HIP(w->Z.alloc((size_t)w->m * w->n * w->kp * (prec == PHG_F64 ? 8 : 4)));
    *out = w;
    return PHG_OK;
}

// Number of columns still running in the cycle, for the host's early exit.
__global__ void bk_count_active(int K, const BCol* __restrict__ cols, int* __restrict__ out)
{
    const int lane = threadIdx.x;
    int a = 0;
    for (int q = lane; q < K; q += 64) a += cols[q].active ? 1 : 0;
    for (int off = 32; off > 0; off >>= 1) a += __shfl_xor(a, off, 64);
    if (lane == 0) out[0] = a;
}

// f(rows per thread as a constant)
template <typename F>
void by_rpt(int rpt, F f)
{
    switch (rpt) {
    case 1: return f(std::integral_constant<int, 1>());
    case 2: return f(std::integral_constant<int, 2>());
    case 4: return f(std::integral_constant<int, 4>());
    case 8: return f(std::integral_constant<int, 8>());
    default: return f(std::integral_constant<int, BB_RPT>());
    }
}

template <typename VT, typename MT, bool PC>
void step(const Ell<MT>& E, BatchWork* w, int K, const VT* X, VT* dst, int j, hipStream_t s)
{
    const dim3 grid(w->G), block(BB_BS);
    const size_t bs = (size_t)w->n * w->kp;
    by_rpt(w->rpt, [&](auto r) {
        constexpr int RPT = decltype(r)::value;
        hipLaunchKernelGGL(HIP_KERNEL_NAME(bk_step_spmm<VT, MT, RPT, PC>), grid, block, 0, s, w->n,
                           w->kp, K, E.width, E.col.p, E.val.p, X, (VT*)w->V.p, bs, dst, j,
                           w->part.p, w->G, w->cols.p);
    });
}
template <typename VT>
void update(BatchWork* w, int K, VT* dst, int j, bool norm, hipStream_t s)
{
    by_rpt(w->rpt, [&](auto r) {
        hipLaunchKernelGGL(HIP_KERNEL_NAME(bk_update<VT, decltype(r)::value>), dim3(w->G),
                           dim3(BB_BS), 0, s, w->n, w->kp, K, dst, (const VT*)w->V.p,
                           (size_t)w->n * w->kp, j, (int)norm, w->part.p, w->G, w->cols.p);
    });
}
template <typename VT, bool UPD, int NV>
void launch_update_dots(BatchWork* w, int K, VT* dst, int j, hipStream_t s)
{
    hipLaunchKernelGGL(HIP_KERNEL_NAME(bk_update_dots<VT, NV, UPD>), dim3(w->G), dim3(BB_BS), 0, s,
                       w->n, w->kp, K, w->rpt, dst, (const VT*)w->V.p, (size_t)w->n * w->kp, j,
                       w->part.p, w->G, w->cols.p);
}
template <typename VT, bool UPD>
void update_dots(BatchWork* w, int K, VT* dst, int j, hipStream_t s)
{
    if (j < 4) launch_update_dots<VT, UPD, 4>(w, K, dst, j, s);
    else if (j < 8) launch_update_dots<VT, UPD, 8>(w, K, dst, j, s);
    else if (j < 16) launch_update_dots<VT, UPD, 16>(w, K, dst, j, s);
    else if (j < 24) launch_update_dots<VT, UPD, 24>(w, K, dst, j, s);
    else launch_update_dots<VT, UPD, 32>(w, K, dst, j, s);
}

// Arnoldi steps j0 .. j1-1 of a cycle of m steps (chunk c: steps up to
// bb_chunk_end(c)); a chunk that is not the cycle's last ends by counting
// the columns still running.
template <typename VT, typename MT>
void enqueue_batch_steps(phg_matrix_s* A, const Ell<MT>& E, BatchWork* w, int K, int j0, int j1,
                         int m, int passes, double rtol, double inner_rtol, int max_iters,
                         BatchPrecond* pc, hipStream_t s)
{
    (void)A;
    const int n = w->n, KP = w->kp, G = w->G;
    const size_t bs = (size_t)n * KP;
    VT* V = (VT*)w->V.p;
    VT* W0 = (VT*)w->W.p;
    VT* W1 = W0 + bs;
    double* part = w->part.p;
    BCol* cols = w->cols.p;
    const dim3 grid(G), block(BB_BS);
    const int cb = (K + 3) / 4;  // blocks of one wavefront per column
    for (int j = j0; j < j1; ++j) {
        VT* src = (j & 1) ? W1 : W0;
        VT* dst = (j & 1) ? W0 : W1;
        if (pc) {
            // right preconditioning (flexible form): z_j = M^-1 v_j kept for the update
            VT* Vj = V + (size_t)j * bs;
            VT* Zj = (VT*)w->Z.p + (size_t)j * bs;
            hipLaunchKernelGGL(HIP_KERNEL_NAME(bk_scale<VT>), dim3((unsigned)((bs + BB_BS - 1) / BB_BS)),
                               block, 0, s, n, KP, K, src, Vj, j, cols);
            precond_apply<VT>(pc, KP, Vj, Zj, s);
            step<VT, MT, true>(E, w, K, Zj, dst, j, s);
        } else {
            step<VT, MT, false>(E, w, K, src, dst, j, s);
        }
        for (int p = 0; p < passes; ++p) {
            const int nd = j + 1;
            hipLaunchKernelGGL(bk_reduce, dim3((nd * KP + 3) / 4), block, 0, s, KP, K, nd, j, p,
                               part, G, cols);
            if (p == passes - 1) {
                update<VT>(w, K, dst, j, true, s);
            } else if (fused_update_dots()) {
                update_dots<VT, true>(w, K, dst, j, s);
            } else {
                update<VT>(w, K, dst, j, false, s);
                update_dots<VT, false>(w, K, dst, j, s);
            }
        }
        hipLaunchKernelGGL(bk_givens, dim3(cb), block, 0, s, KP, K, j, m, part, G, cols, rtol,
                           inner_rtol, max_iters);
    }
    if (j1 < m) hipLaunchKernelGGL(bk_count_active, dim3(1), dim3(64), 0, s, K, cols, w->nact.p);
}

// The end of a cycle: y, the x update, the true residual and the next
// cycle's start (the host summary).
template <typename VT, typename MT>
void enqueue_batch_finish(phg_matrix_s* A, const Ell<MT>& E, BatchWork* w, int K, double rtol,
                          int max_iters, BatchPrecond* pc, hipStream_t s)
{
    const int n = w->n, KP = w->kp, G = w->G;
    const size_t bs = (size_t)n * KP;
    VT* V = (VT*)w->V.p;
    VT* W0 = (VT*)w->W.p;
    double* part = w->part.p;
    BCol* cols = w->cols.p;
    const dim3 grid(G), block(BB_BS);
    const int cb = (K + 3) / 4;
    hipLaunchKernelGGL(bk_solve_y, dim3(cb), block, 0, s, K, cols);
    hipLaunchKernelGGL(HIP_KERNEL_NAME(bk_xupdate<VT>), grid, block, 0, s, n, KP, K, w->rpt,
                       pc ? (const VT*)w->Z.p : (const VT*)V, bs, w->io.p, cols,
                       (!pc && (const void*)E.val.p == (const void*)A->ell64d.val.p)
                           ? A->dinv.p : (const double*)nullptr);
    hipLaunchKernelGGL(HIP_KERNEL_NAME(bk_residual<VT>), grid, block, 0, s, n, KP, K, w->rpt,
                       A->ell64.width, A->ell64.col.p, A->ell64.val.p, w->io.p, W0, part, G, cols);
    hipLaunchKernelGGL(bk_cycle_start, dim3(cb), block, 0, s, KP, K, part, G, cols, w->sum.p,
                       rtol, max_iters);
}

template <typename VT, typename MT>
int batch_run(phg_matrix_s* A, const Ell<MT>& E, BatchWork* w, int K, const double* B, double* X,
              const phg_gmres_opts& o, phg_gmres_info* infos, BatchPrecond* pc,
              const PersistWork* from, hipStream_t s)
{
    const int n = w->n, KP = w->kp, G = w->G, m = o.restart;
    const size_t bs = (size_t)n * KP;
    VT* W0 = (VT*)w->W.p;
    double* part = w->part.p;
    BCol* cols = w->cols.p;
    const dim3 grid(G), block(BB_BS);
    const int cb = (K + 3) / 4;
    const int passes = o.ortho == PHG_CGS1 ? 1 : 2;
    const double inner = o.precision == PHG_F64 ? 0.0 : o.inner_rtol;
    (void)bs;

    const PState* state = nullptr;
    if (from) {
        state = from->st.p;
        PHG_HIP(hipMemcpyAsync(from->st.p, from->host, sizeof(PState) * K, hipMemcpyHostToDevice, s));
    }
    if (!o.use_x0) {
        const size_t tot = (size_t)n * K;
        hipLaunchKernelGGL(bk_fill0, dim3((unsigned)((tot + 255) / 256)), dim3(256), 0, s, tot, K, X,
                           state);
    }
    hipLaunchKernelGGL(bk_sumsq, grid, block, 0, s, n, KP, K, w->rpt, B, part, G);
    hipLaunchKernelGGL(bk_set_bnorm, dim3(cb), block, 0, s, KP, K, part, G, cols,
                       BIo{B, X}, w->io.p, state);
    hipLaunchKernelGGL(HIP_KERNEL_NAME(bk_residual<VT>), grid, block, 0, s, n, KP, K, w->rpt,
                       A->ell64.width, A->ell64.col.p, A->ell64.val.p, w->io.p, W0, part, G, cols);
    hipLaunchKernelGGL(bk_cycle_start, dim3(cb), block, 0, s, KP, K, part, G, cols, w->sum.p,
                       o.rtol, o.max_iters);
    PHG_HIP(hipGetLastError());

    int nch = 0;  // chunks of the cycle
    while (nch < BB_NCHUNK && (nch == 0 || bb_chunk_end(nch - 1) < m)) ++nch;
    auto chunk_lo = [&](int c) { return c == 0 ? 0 : std::min(m, bb_chunk_end(c - 1)); };
    auto chunk_hi = [&](int c) { return c == nch - 1 ? m : std::min(m, bb_chunk_end(c)); };
    if (o.graph) {
        const void* key[2] = {E.val.p, A->ell64.val.p};
        const bool same = w->captured && w->key_m == m && w->key_ortho == o.ortho &&
                          w->key_k == K && w->key_rtol == o.rtol && w->key_inner == inner &&
                          w->key_maxit == o.max_iters && w->key_pc == (const void*)pc &&
                          !memcmp(key, w->key, sizeof key);
        if (!same) {
            w->drop_graphs();
            // recorded on the caller's stream, or for the null stream (which
            // cannot be captured) on a stream of the workspace
            hipStream_t cs = s;
            if (!cs) {
                if (!w->cap) PHG_HIP(hipStreamCreateWithFlags(&w->cap, hipStreamNonBlocking));
                cs = w->cap;
            }
            for (int c = 0; c <= nch; ++c) {
                hipGraph_t g = nullptr;
                PHG_HIP(hipStreamBeginCapture(cs, hipStreamCaptureModeThreadLocal));
                if (c < nch)
                    enqueue_batch_steps<VT, MT>(A, E, w, K, chunk_lo(c), chunk_hi(c), m,
                                                     passes, o.rtol, inner, o.max_iters, pc,
                                                     cs);
                else
                    enqueue_batch_finish<VT, MT>(A, E, w, K, o.rtol, o.max_iters, pc, cs);
                PHG_HIP(hipStreamEndCapture(cs, &g));
                hipError_t e = hipGraphInstantiate(&w->exec[c], g, nullptr, nullptr, 0);
                (void)hipGraphDestroy(g);
                PHG_HIP(e);
            }
            w->captured = true;
            memcpy(w->key, key, sizeof key);
            w->key_m = m;
            w->key_ortho = o.ortho;
            w->key_k = K;
            w->key_rtol = o.rtol;
            w->key_inner = inner;
            w->key_maxit = o.max_iters;
            w->key_pc = pc;
        }
    }
    for (;;) {
        PHG_HIP(hipMemcpyAsync(w->host, w->sum.p, sizeof(BSum) * K, hipMemcpyDeviceToHost, s));
        PHG_HIP(hipStreamSynchronize(s));
        bool any = false;
        for (int q = 0; q < K; ++q) any = any || w->host[q].active;
        if (!any) break;
        for (int c = 0; c < nch; ++c) {
            if (o.graph) {
                PHG_HIP(hipGraphLaunch(w->exec[c], s));
            } else {
                enqueue_batch_steps<VT, MT>(A, E, w, K, chunk_lo(c), chunk_hi(c), m, passes,
                                                 o.rtol, inner, o.max_iters, pc, s);
                PHG_HIP(hipGetLastError());
            }
            if (c < nch - 1) {
                PHG_HIP(hipMemcpyAsync(w->hnact, w->nact.p, sizeof(int), hipMemcpyDeviceToHost, s));
                PHG_HIP(hipStreamSynchronize(s));
                if (*w->hnact == 0) break;
            }
        }
        if (o.graph) {
            PHG_HIP(hipGraphLaunch(w->exec[nch], s));
        } else {
            enqueue_batch_finish<VT, MT>(A, E, w, K, o.rtol, o.max_iters, pc, s);
            PHG_HIP(hipGetLastError());
        }
    }
    bool all = true;
    for (int q = 0; q < K; ++q) {
        BSum h = w->host[q];
        if (from && !from->host[q].active) {
            const PState& p = from->host[q];
            h.rel = p.rel, h.converged = p.converged, h.iters = p.iters, h.cycles = p.cycles;
        }
        all = all && h.converged;
        if (infos) {
            const int launches = from ? infos[q].cycle_launches : 0;
            memset(&infos[q], 0, sizeof infos[q]);
            infos[q].iterations = h.iters;
            infos[q].restarts = h.cycles;
            infos[q].refinements = o.precision == PHG_F64 ? 0 : h.cycles;
            infos[q].rel_residual = h.rel;
            infos[q].converged = h.converged;
            infos[q].cycle_launches = launches;
        }
    }
    return all ? PHG_OK : PHG_ERR_NOCONV;
}

// ------------------------------------------------------- launch shapes --
// Rows per thread of the row kernels for an (n, KP, precision) shape.  A
// shape's value fixes the block partials of every dot product, so it is kept
// per process: every matrix of that shape uses the same value and a column's
// result does not depend on which object solved it.  Untuned shapes take
// the largest value that still gives >= 1024 workgroups (4 per CU), or 1.
struct ShapeKey {
    int n, kp, prec;
    bool operator<(const ShapeKey& o) const
    {
        return n != o.n ? n < o.n : kp != o.kp ? kp < o.kp : prec < o.prec;
    }
};
std::mutex g_shape_mu;
std::map<ShapeKey, int> g_shape_rpt;

int default_rpt(int n, int kp)
{
    for (int r = 8; r > 1; r >>= 1)
        if (blocks_for(n, kp, r) >= 1024) return r;
    return 1;
}

int shape_rpt(int n, int kp, int prec)
{
    std::lock_guard<std::mutex> g(g_shape_mu);
    auto it = g_shape_rpt.find({n, kp, prec});
    return it == g_shape_rpt.end() ? default_rpt(n, kp) : it->second;
}

void set_shape_rpt(int n, int kp, int prec, int rpt)
{
    std::lock_guard<std::mutex> g(g_shape_mu);
    g_shape_rpt[{n, kp, prec}] = rpt;
}

// How many persistent launches (persist.hip) the K columns may take for that
// form to be the faster one, from the time per Arnoldi step of both.  The
// kernels here: 26 us for the four launches of a step with one Gram-Schmidt
// pass, 43 us for the six with two, and the vectors that they read and write
// at 6 TB/s, less for 32 and 64 columns and beyond 0.5 GB a step (level 7 x 64:
// 3.9 to 4.4).  A persistent launch: 7 to 13 us, and 0.006 us per workgroup of
// a column.  Of 292 shapes measured in both forms, 10,000 to 250,000 rows and
// 1 to 64 columns, the model picks the faster one in 291 (the other: 7 %); its
// times are off by up to 31 % (launches) and 72 % (persistent mass solves of one
// column), far from the line.  It takes K as it is, not KP: 24 mass columns
// at level 6 are faster in four persistent launches, 32 and 48 as launches.
// Per step, here and persistent: level 5 x 8 columns FP64 CGS2 48 and 12 us,
// level 6 x 64 262 and 138, level 7 x 1 55 and 14, x 16 244 and 224, x 64 1036 and
// 898; level 7 FP32 CGS2 x 10 136 and 112, x 14 136 and 158, x 33 576 and 377,
// x 64 598 and 730; mass solves (restart 8, CGS1) level 6 x 24 60 and 49, x 48
// 90 and 98.
int persistent_rounds(int n, int kp, int m, bool f64, bool twice)
{
    const double passes = twice ? 2.0 : 1.0, es = f64 ? 8.0 : 4.0;
    const double vectors = 0.5 * (m + 1) * (passes + 1.0) + 5.0 + 16.0 / m;
    const double bytes = (double)n * kp * es * vectors;
    const double rate = 6e6 / (1.0 + 0.12 * std::max(0.0, std::log2(kp / 16.0))) /  // bytes per us
                        (1.0 + 0.03 * std::max(0.0, std::log2(bytes / 0.5e9)));
    const double here = 9.0 + 17.0 * passes + bytes / rate;
    const double there = (f64 ? 9.2 : 6.2) + (passes - 1.0) * (f64 ? 3.0 : 2.7) +
                         0.006 * n / 1024.0 + 24.0 / m;
    return (int)(here / there);
}

// The columns as persistent launches, where that is the faster form;
// PERSIST_NOT_HERE otherwise, PERSIST_NO_START where the launches go on with
// what w->host has.
int batch_persistent(phg_matrix_s* A, int K, const double* B, double* X, const phg_gmres_opts& o,
                     phg_gmres_info* infos, hipStream_t s)
{
    const int rounds = persistent_rounds(A->n_rows, next_pow2(K), o.restart,
                                         o.precision == PHG_F64, o.ortho == PHG_CGS2);
    PersistWork*& w = A->pbatch[o.precision == PHG_F64 ? 0 : 1];
    if (!w) w = new PersistWork();
    // a launch ends after some 4,000 Arnoldi steps (50 ms) for the host to look
    const int max_cycles = std::max(1, 4096 / o.restart);
    int launches = 0;
    const int rc = persist_solve(A, w, K, B, X, o, o.precision == PHG_F64 && o.diag_scale, true,
                                 max_cycles, rounds, &launches, nullptr, s);
    if (rc == PERSIST_NO_START && infos)
        for (int q = 0; q < K; ++q) infos[q].cycle_launches = launches;
    if (rc) return rc;
    bool all = true;
    for (int q = 0; q < K; ++q) {
        const PState& h = w->host[q];
        all = all && h.converged;
        if (infos) {
            memset(&infos[q], 0, sizeof infos[q]);
            infos[q].iterations = h.iters;
            infos[q].restarts = h.cycles;
            infos[q].refinements = o.precision == PHG_F64 ? 0 : h.cycles;
            infos[q].rel_residual = h.rel;
            infos[q].converged = h.converged;
            infos[q].cycle_launches = launches;
        }
    }
    return all ? PHG_OK : PHG_ERR_NOCONV;
}

// Deterministic right-hand sides for timing: values in [-1, 1) from a hash.
__global__ void bk_fill_hash(size_t n, double* __restrict__ x)
{
    const size_t i = (size_t)lblock() * blockDim.x + threadIdx.x;
    if (i >= n) return;
    unsigned long long h = (i + 1) * 0x9E3779B97F4A7C15ull;
    h ^= h >> 31;
    h *= 0xBF58476D1CE4E5B9ull;
    h ^= h >> 29;
    x[i] = (double)(h >> 11) * (2.0 / 9007199254740992.0) - 1.0;
}

}  // namespace

int gmres_batch_solve(phg_matrix_s* A, int K, const double* B, double* X,
                      const phg_gmres_opts* opts, phg_gmres_info* infos, hipStream_t s,
                      phg_mg_s* mg)
{
    return gmres_batch_solve_pc(A, K, B, X, opts, infos, s, mg ? mg_precond(mg) : nullptr);
}

int gmres_batch_solve_pc(phg_matrix_s* A, int K, const double* B, double* X,
                         const phg_gmres_opts* opts, phg_gmres_info* infos, hipStream_t s,
                         BatchPrecond* pc)
{
    phg_gmres_opts o = *opts;
    if (K < 1 || K > BB_MAXK) {
        set_error("gmres_batch: nrhs must be in 1..64");
        return PHG_ERR_ARG;
    }
    if (o.restart < 1 || o.restart > BB_MAXM) {
        set_error("gmres_batch: restart must be in 1..32");
        return PHG_ERR_ARG;
    }
    if (o.ortho != PHG_CGS2 && o.ortho != PHG_CGS1) {
        set_error("gmres_batch: ortho must be PHG_CGS2 or PHG_CGS1");
        return PHG_ERR_ARG;
    }
    if (o.precision < PHG_F64 || o.precision > PHG_BF16) {
        set_error("gmres_batch: bad precision");
        return PHG_ERR_ARG;
    }
    if (A->n_rows != A->n_cols) {
        set_error("gmres_batch: matrix is not square");
        return PHG_ERR_ARG;
    }
    if (A->n_rows == 0) {
        if (infos)
            for (int q = 0; q < K; ++q) memset(&infos[q], 0, sizeof infos[q]), infos[q].converged = 1;
        return PHG_OK;
    }
    int rc = ensure_ell64(A, s);
    if (rc) return rc;
    const int kp = next_pow2(K);
    if (pc) {
        if ((o.precision != PHG_F64 && !pc->f32()) || pc->rows() != A->n_rows) {
            set_error("gmres_batch: the preconditioner does not fit the matrix or the precision");
            return PHG_ERR_ARG;
        }
        rc = o.precision == PHG_F64 ? pc->reserve(kp) : pc->reserve_f32(kp);
        if (rc) return rc;
    }
    const bool diag = o.precision == PHG_F64 && o.diag_scale && !pc;
    if (diag) rc = ensure_ell64_diag(A, s);
    else if (o.precision == PHG_F32) rc = ensure_ell32(A, s);
    else if (o.precision == PHG_BF16) rc = ensure_ell16(A, s);
    if (rc) return rc;
    const int slot = o.precision == PHG_F64 ? 0 : 1;
    const PersistWork* from = nullptr;
    if (!pc && o.persistent) {
        rc = batch_persistent(A, K, B, X, o, infos, s);
        if (rc == PERSIST_NO_START) from = A->pbatch[slot];
        else if (rc != PERSIST_NOT_HERE) return rc;
    }
    BatchWork* w = nullptr;
    // the autotuner times the plain form, so a preconditioned solve keeps the
    // untuned default shape: its speed and bits do not depend on which
    // tunings ran earlier in the process
    const int rpt = pc ? default_rpt(A->n_rows, kp) : shape_rpt(A->n_rows, kp, o.precision);
    rc = prepare_batch(A, slot, o.precision == PHG_F64 ? PHG_F64 : PHG_F32, o.restart, kp, rpt,
                       pc != nullptr, &w);
    if (rc) return rc;
    // diag: right preconditioning by D^-1: solve (A D^-1) y = b, x = D^-1 y
    if (o.precision == PHG_F64)
        return batch_run<double, double>(A, diag ? A->ell64d : A->ell64, w, K, B, X, o, infos, pc,
                                         from, s);
    if (o.precision == PHG_F32)
        return batch_run<float, float>(A, A->ell32, w, K, B, X, o, infos, pc, from, s);
    return batch_run<float, uint16_t>(A, A->ell16, w, K, B, X, o, infos, pc, from, s);
}

int batch_shape_get(int n, int K, int prec)
{
    return shape_rpt(n, next_pow2(K), prec);
}

int batch_shape_set(int n, int K, int prec, int rpt)
{
    if (n < 1 || K < 1 || K > BB_MAXK || prec < PHG_F64 || prec > PHG_BF16 ||
        (rpt != 0 && rpt != 1 && rpt != 2 && rpt != 4 && rpt != 8 && rpt != 16)) {
        set_error("gmres_batch_set_shape: bad argument (rows per thread 0, 1, 2, 4, 8 or 16)");
        return PHG_ERR_ARG;
    }
    if (rpt == 0) {
        std::lock_guard<std::mutex> g(g_shape_mu);
        g_shape_rpt.erase({n, next_pow2(K), prec});
    } else {
        set_shape_rpt(n, next_pow2(K), prec, rpt);
    }
    return PHG_OK;
}

// Autotuner: times one restart cycle of `K` hash-valued right-hand sides for
// each rows-per-thread value and keeps the fastest for the shape.
int gmres_batch_tune(phg_matrix_s* A, int K, const phg_gmres_opts* opts, hipStream_t s,
                     int* best_out, double* ms_out)
{
    static const int cand[5] = {1, 2, 4, 8, 16};
    const int n = A->n_rows;
    if (K < 1 || K > BB_MAXK || n < 1) {
        set_error("gmres_batch_tune: nrhs must be in 1..64 and the matrix non-empty");
        return PHG_ERR_ARG;
    }
    phg_gmres_opts o = *opts;
    o.max_iters = o.restart;   // exactly one cycle of `restart` steps per column
    o.rtol = 0.0;
    o.inner_rtol = 0.0;
    o.use_x0 = 0;
    o.graph = 1;
    o.persistent = 0;  // the form whose shape is being chosen
    DevBuf<double> B, X;
    PHG_HIP(B.alloc((size_t)n * K));
    PHG_HIP(X.alloc((size_t)n * K));
    const size_t tot = (size_t)n * K;
    hipLaunchKernelGGL(bk_fill_hash, dim3((unsigned)((tot + 255) / 256)), dim3(256), 0, s, tot,
                       B.p);
    PHG_HIP(hipGetLastError());
    hipEvent_t e0 = nullptr, e1 = nullptr;
    PHG_HIP(hipEventCreate(&e0));
    hipError_t he = hipEventCreate(&e1);
    if (he != hipSuccess) {
        (void)hipEventDestroy(e0);
        PHG_HIP(he);
    }
    const int kp = next_pow2(K);
    int best = BB_RPT, rc = PHG_OK;
    float best_ms = 0.0f;
    for (int c = 0; c < 5 && rc == PHG_OK; ++c) {
        set_shape_rpt(n, kp, o.precision, cand[c]);
        float t = 0.0f;
        for (int rep = 0; rep < 4 && rc == PHG_OK; ++rep) {  // rep 0 captures the graph
            if (hipEventRecord(e0, s) != hipSuccess) rc = PHG_ERR_HIP;
            int r = gmres_batch_solve(A, K, B.p, X.p, &o, nullptr, s);
            if (r != PHG_OK && r != PHG_ERR_NOCONV) rc = r;
            if (rc == PHG_OK && (hipEventRecord(e1, s) != hipSuccess ||
                                 hipEventSynchronize(e1) != hipSuccess))
                rc = PHG_ERR_HIP;
            float ms = 0.0f;
            if (rc == PHG_OK && hipEventElapsedTime(&ms, e0, e1) != hipSuccess) rc = PHG_ERR_HIP;
            if (rc == PHG_OK && rep > 0 && (rep == 1 || ms < t)) t = ms;
        }
        if (rc == PHG_OK) {
            if (ms_out) ms_out[c] = t;
            if (c == 0 || t < best_ms) {
                best_ms = t;
                best = cand[c];
            }
        }
    }
    (void)hipEventDestroy(e0);
    (void)hipEventDestroy(e1);
    if (rc == PHG_ERR_HIP) set_error("gmres_batch_tune: HIP event error");
    set_shape_rpt(n, kp, o.precision, rc == PHG_OK ? best : default_rpt(n, kp));
    if (best_out) *best_out = best;
    return rc;
}

}  // namespace phg
