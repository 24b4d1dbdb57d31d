// The persistent solve (see persist.hip) for workgroups of PS_BS threads:
// included once per size, each in a source of its own so that they compile
// side by side.
#pragma once
#include <unistd.h>

#include <chrono>
#include <cstdlib>
#include <cstring>
#include <thread>

#include "krylov.h"
#include "persist.h"
#include "phg_internal.h"

namespace phg {
namespace {

// Workgroup pair p of 256 threads owns the 1024 rows of workgroup p of 512,
// wavefronts 0..3 of it the first of the pair.  Every sum has the same order
// in both sizes (the halves of a workgroup or pair, then the pairs): the size
// is a matter of speed alone, and results don't depend on it.
constexpr int BS = PS_BS, ROWS = BS * KR_RPT, GRP = BS / 32;
constexpr int PAIR = KR_STRIDE / BS;  // workgroups of 1024 rows
static_assert(PAIR == 1 || PAIR == 2, "workgroups of 512 or 256 threads");
__host__ __device__ inline int first_row(int bid)
{
    return bid / PAIR * (KR_STRIDE * KR_RPT) + bid % PAIR * BS;
}
inline int workgroups(int n) { return persist_workgroups(n, BS); }
// a workgroup's slot of a row of Gp: second ones of a pair in the upper half
__host__ __device__ inline int slot_of(int bid, int Gp) { return bid / PAIR + bid % PAIR * (Gp / PAIR); }
typedef unsigned long long xch_t;
constexpr xch_t XCH_EMPTY = 0x7FF4DEADBEEF0001ull;  // a signalling-NaN pattern no partial takes
constexpr long XCH_SPIN = 1L << 22;                  // polls before a wait gives up
// polls of a launch's first exchange (some 0.1 s), and launches until it
// succeeds or the solve goes on without them: 1.6 s for another process's
// work to end
constexpr long XCH_START = 1L << 17;
constexpr int XCH_TRIES = 16;
// (PHG_XCH_SPIN and PHG_XCH_START override the two limits: the tests of the
// failure paths force a give-up with a few polls; every workgroup still exits
// normally)
enum { ABORT_WAIT = 1, ABORT_START = 2 };  // bits of the host's abort word
constexpr int XCH_RING = 4;   // rows of a column's ring
constexpr int XCH_V = 32;     // values of a slot
constexpr int PS_M = 32;      // largest restart

// ------------------------------------------------------------- exchange --
// Exchange e of a column: every workgroup stores up to 32 block partials
// into its slot (32 words) of row e mod 4 with agent-scope stores, and every
// workgroup reads all G slots until none holds XCH_EMPTY, then adds them in
// krylov_join's order.  All of a thread's loads are issued before the first
// test, with no branch between them: 2.65 us among 161 workgroups, 32 values
// as fast as one; with a bounds test before each load the same exchange took
// 8.7 us.  A slot is one coalesced 256-byte store and load.  A row has one
// of a few lengths (hop_slots), so that the loads have fixed offsets; the
// slots past the last workgroup hold 0.
//
// A row is used again four exchanges later.  When a workgroup has finished
// exchange e - 1, every workgroup has stored into row e - 1 and has
// therefore finished reading row e - 2: each clears its own slot of row
// e - 2 then.  The clearing is complete before it stores into row e + 1 (the
// wait at the start of an exchange), and whoever polls row e + 2 has seen
// that store.  The rows of the ring start out clear: a launch uses one of two
// rings and clears its slots of the other one.
//
// Vectors that other workgroups gather (the next Arnoldi vector, x before the
// residual) are written with agent-scope stores that complete (s_waitcnt
// vmcnt(0)) before the partial that announces them is stored, and are
// gathered with agent-scope loads; no cache-wide write-back or invalidation
// is needed.  Every wait is bounded: after `spin` polls a workgroup raises
// the abort flag and leaves, and the others leave at their next look at it.
//
// The first exchange of a launch shows that a column's workgroups are resident
// together: each stays until it has seen the others' slots.  If something
// else holds the CUs (another process's launch, half of it waiting for this
// one's other half), that exchange ends after start_spin polls, and the host
// launches the column again.  A workgroup that gives up has stored its slot,
// and its CU may go to the one that was missing, so others may still pass the
// first exchange; none passes the second, which the one that gave up never
// stores.  So nothing that a repeated launch reads (W, the state, x when it is
// a start vector) is written before the second exchange: a launch that
// continues a solve begins with an exchange of no values, whose 1.7 to 2.7 us
// are 1 to 2 % of a cycle.  The abort flag is the column's own: the other
// columns of the launch, which may be far along, go on.  Within a process
// only launches that fit the device together run at the same time
// (persist_turns.h).  A cooperative launch would give the same guarantee but
// is refused to every process of a GPU except the first that asks.
struct Hop {
    xch_t* ring;
    int G, slot, e;  // G: slots of a row (padded workgroup count)
    long spin, start_spin;
    int* abort_dev;   // the column's
    int* abort_host;  // the solve's
};

inline int hop_slots(int G)
{
    return G <= 16 ? 16 : G <= 48 ? 48 : G <= 96 ? 96 : G <= 176 ? 176 : 256;
}

struct HopLds {
    double w[BS / 64][33];  // partials of the wavefronts
    double g[16][33];       // sums of the thread groups
    int bad, cont;
};

template <int NQ>
__device__ __forceinline__ bool hop_poll(const Hop& h, const xch_t* row, int val, double* sum)
{
    const long spin = h.e == 0 ? h.start_spin : h.spin;
    const unsigned off = ((threadIdx.x >> 5) * XCH_V + val) * (unsigned)sizeof(xch_t);
    xch_t u[NQ];
    bool ok = false, left = false;
    for (long it = 0; it < spin; ++it) {
#pragma unroll
        for (int q = 0; q < NQ; ++q)
            u[q] = ld_agent((const xch_t*)((const char*)(row + GRP * q * XCH_V) + off));
        bool all = true;
#pragma unroll
        for (int q = 0; q < NQ; ++q) all = all & (u[q] != XCH_EMPTY);
        if (__all(all)) {
            ok = true;
            break;
        }
        if ((it & 63) == 63 && ld_agent(h.abort_dev)) {
            left = true;
            break;
        }
    }
    if (!ok && !left) {
        st_agent(h.abort_dev, 1);
        __hip_atomic_fetch_or(h.abort_host, h.e == 0 ? ABORT_START : ABORT_WAIT, __ATOMIC_RELAXED,
                              __HIP_MEMORY_SCOPE_SYSTEM);
    }
    // the running sums grp + GRP k, and with them the sums q and q + 16
    double a[32 / GRP];
#pragma unroll
    for (int k = 0; k < 32 / GRP; ++k) a[k] = 0.0;
#pragma unroll
    for (int q = 0; q < NQ / PAIR; ++q) {
        double s = __longlong_as_double((long long)u[q]);
        if (PAIR == 2) s += __longlong_as_double((long long)u[q + NQ / PAIR]);
        a[q % (32 / GRP)] += s;
    }
#pragma unroll
    for (int k = 0; k < 16 / GRP; ++k) sum[k] = a[k] + a[k + 16 / GRP];
    return ok;
}

enum { HOP_OK = 0, HOP_STOP = 1, HOP_FAIL = 2 };

// The exchange of values 0..nv-1 and, with `last`, of value 31, from the
// wavefronts' partials in l->w; lane i of every wavefront returns the total
// of value i & 31.  The last wavefront runs `meanwhile` once the partials are
// on their way, and polls after it.  HOP_STOP when l->cont is 0, with `early`
// before the exchange, with `check` after it (meanwhile may write it): every
// workgroup of the column decides the same.
template <typename F>
__device__ __forceinline__ int hop(Hop& h, int nv, bool last, bool early, bool check, HopLds* l,
                                   double* tot, F meanwhile)
{
    const int t = threadIdx.x, i = t & 31;
    __builtin_amdgcn_s_waitcnt(0x0F70);  // vmcnt(0): this thread's stores are complete
    __syncthreads();
    if (early && !l->cont) return HOP_STOP;
    xch_t* row = h.ring + (size_t)(h.e & (XCH_RING - 1)) * h.G * XCH_V;
    const bool mine = i < nv || (last && i == 31);
    if (t < 32 && mine) {
        double r = 0.0;
#pragma unroll
        for (int p = 0; p < BS / 256; ++p)
            r += krylov_half(l->w[4 * p][i], l->w[4 * p + 1][i], l->w[4 * p + 2][i], l->w[4 * p + 3][i]);
        st_agent(row + (size_t)h.slot * XCH_V + i, (xch_t)__double_as_longlong(r));
    }
    if (t >= 64 && t < 96)
        st_agent(h.ring + ((size_t)((h.e + 2) & (XCH_RING - 1)) * h.G + h.slot) * XCH_V + i, XCH_EMPTY);
    if (t >= BS - 64) meanwhile();
    const int val = mine ? i : (nv > 0 ? 0 : 31);
    double sum[16 / GRP];
    bool ok;
    if (h.G == 16) ok = hop_poll<16 / GRP>(h, row, val, sum);
    else if (h.G == 48) ok = hop_poll<48 / GRP>(h, row, val, sum);
    else if (h.G == 96) ok = hop_poll<96 / GRP>(h, row, val, sum);
    else if (h.G == 176) ok = hop_poll<176 / GRP>(h, row, val, sum);
    else ok = hop_poll<256 / GRP>(h, row, val, sum);
#pragma unroll
    for (int k = 0; k < 16 / GRP; ++k) l->g[(t >> 5) + GRP * k][i] = sum[k];
    if (!ok) l->bad = 1;
    __syncthreads();
    *tot = krylov_join(l->g, i);
    ++h.e;
    return l->bad ? HOP_FAIL : check && !l->cont ? HOP_STOP : HOP_OK;
}
__device__ __forceinline__ int hop(Hop& h, int nv, bool last, HopLds* l, double* tot)
{
    return hop(h, nv, last, false, false, l, tot, [] {});
}

// --------------------------------------------------------------- kernel --
template <typename VT, typename MT>
struct PArgs {
    int n, ld, G, Gp, m, width;  // of both forms of the matrix
    const int* col;
    const MT* val;
    const int* col64;
    const double* val64;
    const double* dscale;  // x += dscale * (V y), or null
    const double* B;       // row-major, ld columns; column q at q
    double* X;
    VT* W;                 // a vector of ldw per column
    size_t ldw;
    xch_t *ring, *other;   // XCH_RING rows of Gp slots per column
    PState *st, *host;
    int *abort_dev, *abort_host;  // a word per column; one for the host
    long spin, start_spin;
    double rtol, inner_rtol;
    int max_iters, max_cycles, first, use_x0, stall;
};

// ||.||^2 of a thread's rows, as the block partial of value `i`
template <typename T>
__device__ __forceinline__ void put_norm(const T (&w)[KR_RPT], int i, HopLds* l)
{
    double a = 0.0;
#pragma unroll
    for (int r = 0; r < KR_RPT; ++r) a = fma(to_d(w[r]), to_d(w[r]), a);
    a = wave_sum(a);
    if ((threadIdx.x & 63) == 0) l->w[threadIdx.x >> 6][i] = a;
}

// A thread's rows of the basis, in tiers of KR_T vectors: in LDS what fits
// 128 of its 160 KB (all 32 vectors of 512 rows or of 1024 FP32 rows, 16 of
// 1024 FP64 rows), the others in registers.  All 32 in registers spilled 409
// of them.
template <typename VT>
struct Basis {
    static constexpr int TIERS = PS_M / KR_T;
    static constexpr int LDS_TIERS = PS_M * sizeof(VT) * ROWS <= (128 << 10) ? TIERS : TIERS / 2;
    static constexpr int REG_TIERS = TIERS > LDS_TIERS ? TIERS - LDS_TIERS : 1;
    VT* lds;  // [vector][row of the workgroup], this thread's first row
    VT reg[REG_TIERS][KR_T][KR_RPT];

    __device__ __forceinline__ VT at(int t, int i, int r) const
    {
        return t < LDS_TIERS ? lds[(t * KR_T + i) * ROWS + r * BS]
                             : reg[t < LDS_TIERS ? 0 : t - LDS_TIERS][i][r];
    }
    // zeros: tiers are read whole, and what is not a basis vector yet must be
    // finite there (a vector w / ||w|| with ||w|| = 0 is put as zeros too)
    __device__ __forceinline__ void clear()
    {
#pragma unroll
        for (int i = 0; i < LDS_TIERS * KR_T; ++i)
#pragma unroll
            for (int r = 0; r < KR_RPT; ++r) lds[i * ROWS + r * BS] = VT(0);
#pragma unroll
        for (int u = 0; u < REG_TIERS; ++u)
#pragma unroll
            for (int i = 0; i < KR_T; ++i)
#pragma unroll
                for (int r = 0; r < KR_RPT; ++r) reg[u][i][r] = VT(0);
    }
    __device__ __forceinline__ void put(int j, const VT (&v)[KR_RPT])
    {
        if (j < LDS_TIERS * KR_T) {
#pragma unroll
            for (int r = 0; r < KR_RPT; ++r) lds[j * ROWS + r * BS] = v[r];
        } else {
#pragma unroll
            for (int u = 0; u < TIERS - LDS_TIERS; ++u) {
                if (u + LDS_TIERS != j / KR_T) continue;
#pragma unroll
                for (int i = 0; i < KR_T; ++i)
#pragma unroll
                    for (int r = 0; r < KR_RPT; ++r)
                        reg[u][i][r] = i == j % KR_T ? v[r] : reg[u][i][r];
            }
        }
    }
};

// partials of the dots of w with v_0..v_j
template <typename VT>
__device__ __forceinline__ void put_dots(int j, const VT (&w)[KR_RPT], const Basis<VT>& V,
                                         HopLds* l)
{
    const int lane = threadIdx.x & 63;
#pragma unroll
    for (int t = 0; t < Basis<VT>::TIERS; ++t) {
        if (t * KR_T > j) break;
        VT v[KR_T][KR_RPT];
        double p[KR_T];
#pragma unroll
        for (int i = 0; i < KR_T; ++i)
#pragma unroll
            for (int r = 0; r < KR_RPT; ++r) v[i][r] = V.at(t, i, r);
        dots_tier<VT>(w, v, p);
        const double s = reduce8(p);
        const int i = t * KR_T + reduce8_value(lane);
        if ((lane & 7) == 0 && i <= j) l->w[threadIdx.x >> 6][i] = s;
    }
}

// w -= sum_{i<=j} h_i v_i (lane i of the wavefront holds h_i)
template <typename VT>
__device__ __forceinline__ void take_off(int j, double h, VT (&w)[KR_RPT], const Basis<VT>& V)
{
    // entries past j (finite: see put) take no part
    h = (int)(threadIdx.x & 31) <= j ? h : 0.0;
#pragma unroll
    for (int t = 0; t < Basis<VT>::TIERS; ++t) {
        if (t * KR_T > j) break;
        VT v[KR_T][KR_RPT];
#pragma unroll
        for (int i = 0; i < KR_T; ++i)
#pragma unroll
            for (int r = 0; r < KR_RPT; ++r) v[i][r] = V.at(t, i, r);
#pragma unroll
        for (int i = 0; i < KR_T; ++i) {
            const VT hv = (VT)readlane_d(h, t * KR_T + i);
#pragma unroll
            for (int r = 0; r < KR_RPT; ++r) w[r] = kfma(-hv, v[i][r], w[r]);
        }
    }
}

// PRE: rows of 1 to ELL_MAXW entries, the thread's matrix rows in registers
// throughout; otherwise rows of any width, read anew in every product.  With
// PRE `pre` is always true; the test at run time and the loop behind it keep
// the compiler's schedule of a step (the test left out: level 7 FP64 MGS 5.30
// instead of 5.06 ms, in six forms that were tried, 36,503 rows FP32 CGS2 1.80
// instead of 1.77).  256 threads with FP64 vectors are faster without it
// (level 4 287 instead of 293 us).
template <typename VT, typename MT, int ORTHO, bool PRE>
__global__ void __launch_bounds__(BS)
k_persist(PArgs<VT, MT> a)
{
    __shared__ VT sV[Basis<VT>::LDS_TIERS * KR_T * ROWS];
    __shared__ HopLds l;
    __shared__ double sL[PS_M * 33];  // <v_i, v_k>, k < i
    __shared__ double sR[PS_M * 33];
    __shared__ double s_cs[2 * PS_M], s_g[PS_M], s_carry[PS_M + 1], s_y[PS_M];
    __shared__ double s_h[PS_M + 8];  // Hessenberg column of the last step
    const int t = threadIdx.x, lane = t & 63, li = lane & 31;
    const int q = (int)blockIdx.x / a.G, bid = (int)blockIdx.x % a.G;
    // (512 threads with FP64 vectors spill 160 registers with it: 10.1 ms
    // instead of 5.0 at level 7)
    constexpr bool LATE = BS == 256 || sizeof(VT) == 4;
    const int n = a.n, ld = a.ld, m = a.m, slot = slot_of(bid, a.Gp);
    Hop h{a.ring + (size_t)q * XCH_RING * a.Gp * XCH_V, a.Gp, slot, 0, a.spin, a.start_spin,
          a.abort_dev + q, a.abort_host};
    if (t < XCH_RING * XCH_V)
        st_agent(a.other + (size_t)q * XCH_RING * a.Gp * XCH_V +
                     ((size_t)(t >> 5) * a.Gp + slot) * XCH_V + (t & 31), XCH_EMPTY);
    if (t == 0) l.bad = 0;
    const int base = first_row(bid) + t;
    const double* B = a.B + q;
    double* X = a.X + q;
    VT* W = a.W + (size_t)q * a.ldw;

    VT w[KR_RPT];
    double bnorm = 1.0, beta = 0.0, rel = 0.0, tot = 0.0;
    int iters = 0, cycles = 0, converged = 0, active = 0;
    if (a.first) {
        // x, ||b|| and the first residual; with x = 0 that is b
        double b[KR_RPT], r0[KR_RPT], xo[KR_RPT], ax[KR_RPT];
#pragma unroll
        for (int r = 0; r < KR_RPT; ++r) {
            const int rr = base + r * KR_STRIDE;
            b[r] = rr < n ? B[(size_t)rr * ld] : 0.0;
            r0[r] = b[r];
        }
        if (a.use_x0) {
            krylov_rows<double, double, false, KR_RPT, PRE>(n, a.width, base, a.col64, a.val64, X,
                                                            ld, 1.0, xo, ax);
#pragma unroll
            for (int r = 0; r < KR_RPT; ++r) r0[r] = b[r] - ax[r];
        }
#pragma unroll
        for (int r = 0; r < KR_RPT; ++r) {
            const int rr = base + r * KR_STRIDE;
            if (rr < n && !a.use_x0) st_agent(X + (size_t)rr * ld, 0.0);
            w[r] = (VT)r0[r];
            if (rr < n) st_agent(W + rr, w[r]);
        }
        put_norm(b, 0, &l);
        put_norm(r0, 1, &l);
    } else {
        const PState s = a.st[q];
        bnorm = s.bnorm, beta = s.beta, rel = s.rel;
        iters = s.iters, cycles = s.cycles, converged = s.converged, active = s.active;
#pragma unroll
        for (int r = 0; r < KR_RPT; ++r) {
            const int rr = base + r * KR_STRIDE;
            w[r] = rr < n ? W[rr] : VT(0);
        }
        if (lane < 2) l.w[t >> 6][lane] = 0.0;
    }
    if ((a.first || active) && hop(h, 2, false, &l, &tot) != HOP_OK) return;
    if (a.first) {
        bnorm = sqrt(readlane_d(tot, 0));
        if (!(bnorm > 0.0)) bnorm = 1.0;
        beta = sqrt(readlane_d(tot, 1));
        rel = beta / bnorm;
        if (rel <= a.rtol || beta == 0.0) converged = 1;
        else active = iters < a.max_iters && (!a.stall || isfinite(beta));
        if (active) ++cycles;
    }

    // the thread's matrix rows (past a row's width its last slot with the
    // value 0, past row n row n - 1: every load is in bounds), and its rows of the basis
    unsigned sc[KR_RPT][ELL_MAXW];  // byte offsets into W
    MT sv[KR_RPT][ELL_MAXW];
    const bool pre = PRE && ((BS == 256 && sizeof(VT) == 8) ||
                             (a.width >= 1 && a.width <= ELL_MAXW));
    if (pre && active) {
#pragma unroll
        for (int r = 0; r < KR_RPT; ++r) {
            const int rr = min(base + r * KR_STRIDE, n - 1);
#pragma unroll
            for (int k = 0; k < ELL_MAXW; ++k) {
                const size_t o = ell_slot(k, a.width, n, rr);
                sc[r][k] = (unsigned)a.col[o] * (unsigned)sizeof(VT);
                sv[r][k] = k < a.width ? a.val[o] : MT(0);
            }
        }
    }
    Basis<VT> V;
    V.lds = sV + t;
    V.clear();

    for (int run = 0; active && run < a.max_cycles; ++run) {
        const int iters0 = iters;
        const double stop = fmax(a.rtol * bnorm, a.inner_rtol * beta);
        if (t == 0) s_carry[0] = beta;
        double hn = beta;
        int j = 0, rc = HOP_OK;
        for (;; ++j) {
            // v_j = w / hn; w = A v_j.  The column of step j - 1 is rotated
            // while the dots are exchanged (level 4 FP64 MGS 305 -> 292 us a
            // solve, 36,503 rows FP32 CGS2 1.88 -> 1.73 ms), or by the first
            // wavefront while the gathers are in flight
            const VT inv = (VT)(1.0 / hn);
            VT vj[KR_RPT], xv[KR_RPT][ELL_MAXW];
            if (j < m) {
#pragma unroll
                for (int r = 0; r < KR_RPT; ++r) vj[r] = hn > 0.0 ? w[r] * inv : VT(0);
                if (pre) {
#pragma unroll
                    for (int r = 0; r < KR_RPT; ++r)
#pragma unroll
                        for (int k = 0; k < ELL_MAXW; ++k) xv[r][k] = ld_agent((const VT*)((const char*)W + sc[r][k]));
                }
            }
            const auto rotate = [&] {
                if (j == 0) return;
                const GivensOut g = krylov_givens(j - 1, m, s_h, hn, stop, iters0, a.max_iters,
                                                  s_cs, s_g, s_carry, sR, 33);
                if (lane == 0) l.cont = g.cont;
            };
            if (j == m || !LATE) {
                if (t < 64) rotate();
                if (j == m) break;
            }
            if (pre) {
#pragma unroll
                for (int r = 0; r < KR_RPT; ++r) {
                    VT s = VT(0);
#pragma unroll
                    for (int k = 0; k < ELL_MAXW; ++k)
                        s = RowTerm<VT, MT>::add(s, sv[r][k], xv[r][k], inv);
                    w[r] = base + r * KR_STRIDE < n ? s : VT(0);
                }
            } else {
                VT xo[KR_RPT];
                if constexpr (PRE)
                    krylov_rows_each<VT, MT, true, KR_RPT>(n, a.width, opaque(base), a.col, a.val,
                                                           W, 1, inv, xo, w);
                else
                    krylov_rows_loop<VT, MT, true, KR_RPT>(n, a.width, opaque(base), a.col, a.val,
                                                           W, 1, inv, xo, w);
            }
            V.put(j, vj);
            put_dots<VT>(j, w, V, &l);
            rc = hop(h, j + 1, false, !LATE && j > 0, LATE && j > 0, &l, &tot, [&] {
                if (LATE) rotate();
            });
            if (rc != HOP_OK) break;
            double hcol = tot;
            if (ORTHO == PHG_MGS) hcol = mgs_solve<PS_M>(tot, j, sL, 33, li);
            take_off<VT>(j, hcol, w, V);
            if (ORTHO == PHG_CGS2) {
                put_dots<VT>(j, w, V, &l);
                rc = hop(h, j + 1, false, &l, &tot);
                if (rc != HOP_OK) break;
                take_off<VT>(j, tot, w, V);
                hcol += tot;
            }
            if (t < PS_M) s_h[t] = hcol;
#pragma unroll
            for (int r = 0; r < KR_RPT; ++r) {
                const int rr = base + r * KR_STRIDE;
                if (rr < n) st_agent(W + rr, w[r]);
            }
            const bool more = ORTHO == PHG_MGS && j + 1 < m;
            put_norm(w, 31, &l);
            if (more) put_dots<VT>(j, w, V, &l);
            rc = hop(h, more ? j + 1 : 0, true, &l, &tot);
            if (rc != HOP_OK) break;
            hn = sqrt(readlane_d(tot, 31));
            if (more && t <= j) sL[(j + 1) * 33 + t] = tot * to_d((VT)(1.0 / hn));
        }
        if (rc == HOP_FAIL) return;
        // j steps are complete: y = R^-1 g, x += V y
        iters = iters0 + j;
        __syncthreads();
        if (t < 64) {
            const double y = krylov_solve_y(j, sR, 33, s_g);
            if (lane < PS_M) s_y[lane] = y;
        }
        __syncthreads();
#pragma unroll
        for (int r = 0; r < KR_RPT; ++r) {
            const int rr = opaque(base) + r * KR_STRIDE;
            double s = 0.0;  // y is 0 past step j
#pragma unroll
            for (int i = 0; i < PS_M; ++i) s = fma(to_d(V.at(i / KR_T, i % KR_T, r)), s_y[i], s);
            if (rr < n) {
                if (a.dscale) s = a.dscale[rr] * s;
                double* x = X + (size_t)rr * ld;
                st_agent(x, ld_agent(x) + s);
            }
        }
        if (lane == 0) l.w[t >> 6][0] = 0.0;
        if (hop(h, 1, false, &l, &tot) != HOP_OK) return;
        // r = b - A x in FP64, the next cycle's vector
        double res[KR_RPT], xo[KR_RPT];
        const int rb = opaque(base);
        krylov_rows<double, double, true, KR_RPT, PRE>(n, a.width, rb, a.col64, a.val64, X, ld,
                                                       1.0, xo, res);
#pragma unroll
        for (int r = 0; r < KR_RPT; ++r) {
            const int rr = rb + r * KR_STRIDE;
            res[r] = rr < n ? B[(size_t)rr * ld] - res[r] : 0.0;
            w[r] = (VT)res[r];
            if (rr < n) st_agent(W + rr, w[r]);
        }
        put_norm(res, 0, &l);
        if (hop(h, 1, false, &l, &tot) != HOP_OK) return;
        const double now = sqrt(readlane_d(tot, 0));
        const bool stalled = a.stall && iters > iters0 && now > 0.99 * beta;
        beta = now;
        rel = beta / bnorm;
        if (rel <= a.rtol || beta == 0.0) {
            converged = 1;
            active = 0;
        } else if (iters >= a.max_iters || stalled || (a.stall && !isfinite(beta))) {
            active = 0;
        } else {
            ++cycles;
        }
    }
    if (bid == 0 && t == 0) {
        PState s;
        s.bnorm = bnorm, s.beta = beta, s.rel = rel;
        s.iters = iters, s.cycles = cycles, s.converged = converged, s.active = active;
        a.st[q] = s;
        a.host[q] = s;
    }
}

// whether one of G workgroups has the slot
__device__ inline bool slot_used(int slot, int G, int Gp)
{
    const int half = slot / (Gp / PAIR), p = slot % (Gp / PAIR);
    return p * PAIR + half < G;
}

// Clears both rings (slots past the last workgroup: 0) and the nab columns'
// abort flags (nab at most a ring's slots).
__global__ void k_ring_reset(xch_t* ring, size_t count, int G, int Gp, int* abort_dev, int nab)
{
    const size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i < count) ring[i] = slot_used((int)(i / XCH_V % Gp), G, Gp) ? XCH_EMPTY : 0;
    if (i < (size_t)nab) abort_dev[i] = 0;
}

// Workgroups of the kernel that the device holds at once, per template
// instance, computed once (thread-safe static initialisation).
template <typename VT, typename MT, int ORTHO, bool PRE>
int capacity()
{
    static const int n = [] {
        int dev = 0, cus = 0, per = 0;
        if (hipGetDevice(&dev) != hipSuccess ||
            hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess ||
            hipOccupancyMaxActiveBlocksPerMultiprocessor(
                &per, (const void*)k_persist<VT, MT, ORTHO, PRE>, BS, 0) != hipSuccess)
            return 0;
        return cus * per;
    }();
    return n;
}

inline long poll_limit(const char* name, long limit)
{
    const char* e = getenv(name);
    return e ? std::max(1L, atol(e)) : limit;
}

// Columns q0 .. q0 + K - 1 of the ld in B and X.
template <typename VT, typename MT, int ORTHO, bool PRE>
int launch(phg_matrix_s* A, const Ell<MT>& E, PersistWork* w, int q0, int K, int ld, const double* B,
           double* X, const phg_gmres_opts& o, const double* dscale, bool stall, int max_cycles,
           int first, hipStream_t s)
{
    const int n = A->n_rows, G = workgroups(n), Gp = hop_slots(G);
    const size_t ldw = ((size_t)n + 63) / 64 * 64, slots = (size_t)K * XCH_RING * Gp * XCH_V;
    if (w->ring_k != K || w->ring_g != G) {
        // another shape than the last launch's, or after a give-up
        hipLaunchKernelGGL(k_ring_reset, dim3((unsigned)((2 * slots + 255) / 256)), dim3(256), 0, s,
                           w->xch.p(), 2 * slots, G, Gp, w->abort_dev.p, w->host_k);
        PHG_HIP(hipGetLastError());
        w->ring_k = K;
        w->ring_g = G;
    }
    PArgs<VT, MT> a;
    a.n = n, a.ld = ld, a.G = G, a.Gp = Gp, a.m = o.restart, a.width = E.width;
    a.col = E.col.p, a.val = E.val.p, a.col64 = A->ell64.col.p, a.val64 = A->ell64.val.p;
    a.dscale = dscale, a.B = B + q0, a.X = X + q0, a.W = (VT*)w->W.p + (size_t)q0 * ldw, a.ldw = ldw;
    a.ring = w->xch.p() + (w->parity ? slots : 0);
    a.other = w->xch.p() + (w->parity ? 0 : slots);
    w->parity ^= 1;
    a.st = w->st.p + q0, a.host = w->host + q0;
    a.abort_dev = w->abort_dev.p + q0, a.abort_host = (int*)(w->host + w->host_k);
    a.spin = poll_limit("PHG_XCH_SPIN", XCH_SPIN);
    a.start_spin = poll_limit("PHG_XCH_START", XCH_START);
    a.rtol = o.rtol;
    a.inner_rtol = o.precision == PHG_F64 ? 0.0 : o.inner_rtol;
    a.max_iters = o.max_iters, a.max_cycles = max_cycles, a.use_x0 = o.use_x0;
    a.stall = stall, a.first = first;
    for (int q = q0; q < q0 + K; ++q) w->host[q].active = -1;  // until the kernel writes it
    hipLaunchKernelGGL(HIP_KERNEL_NAME(k_persist<VT, MT, ORTHO, PRE>), dim3(G * K), dim3(BS), 0, s, a);
    PHG_HIP(hipGetLastError());
    return PHG_OK;
}

// The launches that a stream runs from begin to end, one after the other, of
// at most so many workgroups each.
struct Turn {
    PersistTurns& turns;
    int workgroups;
    bool in = false;
    Turn(PersistTurns& t, int w) : turns(t), workgroups(w) {}
    Turn(const Turn&) = delete;
    Turn& operator=(const Turn&) = delete;
    ~Turn() { end(); }
    hipError_t begin(hipStream_t s)
    {
        hipError_t e = hipSuccess;
        if (!turns.try_enter(workgroups)) {
            // other threads' launches run: wait for this stream's earlier work
            // first, so that nobody waits for that while it is this one's turn
            e = hipStreamSynchronize(s);
            if (e != hipSuccess) return e;
            turns.enter(workgroups);
        }
        in = true;
        return e;
    }
    void end()
    {
        if (in) turns.leave(workgroups);
        in = false;
    }
};

template <typename VT, typename MT, int ORTHO, bool PRE>
int run(phg_matrix_s* A, const Ell<MT>& E, PersistWork* w, int K, const double* B, double* X,
        const phg_gmres_opts& o, const double* dscale, bool stall, int max_cycles, int max_rounds,
        int* launches, double* ms, hipStream_t s)
{
    const int n = A->n_rows, G = workgroups(n);
    // columns of a launch, and launches for all columns, of equal size
    const int fit = std::min(capacity<VT, MT, ORTHO, PRE>(), KR_MAXG) / G;
    if (fit < 1) return PERSIST_NOT_HERE;
    const int rounds = (K + fit - 1) / fit, per = (K + rounds - 1) / rounds;
    if (rounds > max_rounds) return PERSIST_NOT_HERE;
    const size_t ldw = ((size_t)n + 63) / 64 * 64;
    const size_t slots = (size_t)per * XCH_RING * hop_slots(G) * XCH_V;
    const size_t bytes = (size_t)K * ldw * sizeof(VT);
    if (w->W.n < bytes) PHG_HIP(w->W.alloc(bytes));
    if (w->host_k < K) {
        if (w->host) (void)hipHostFree(w->host);
        w->host = nullptr;
        w->host_k = 0;
        PHG_HIP(w->st.alloc(K));
        PHG_HIP(w->abort_dev.alloc(K));
        w->ring_k = 0;  // they are cleared with the rings
        // K states, then the abort word
        PHG_HIP(hipHostMalloc((void**)&w->host, sizeof(PState) * (K + 1), hipHostMallocDefault));
        w->host_k = K;
    }
    if (w->ring_slots < slots) {
        w->ring_slots = 0;
        PHG_HIP(w->xch.alloc(2 * slots));
        w->ring_slots = slots;
        w->ring_k = 0;
    }
    if (ms && !w->ev[0]) {
        PHG_HIP(hipEventCreate(&w->ev[0]));
        PHG_HIP(hipEventCreate(&w->ev[1]));
    }
    int dev = 0;
    PHG_HIP(hipGetDevice(&dev));
    PersistTurns& turns = persist_turns(dev);
    volatile int* abort_host = (int*)(w->host + w->host_k);
    int tries = 0;
    for (int first = 1;; first = 0) {
        for (int q = 0; q < K; ++q)
            if (first) w->host[q] = PState{0.0, 0.0, 0.0, 0, 0, 0, 1};
        // the columns still running, and one by one those of a launch that
        // did not start
        for (bool again = false;; again = true) {
            *abort_host = 0;
            const int step = again ? 1 : per;
            Turn turn(turns, G * step);
            PHG_HIP(turn.begin(s));
            if (ms) PHG_HIP(hipEventRecord(w->ev[0], s));
            for (int q0 = 0; q0 < K; q0 += step) {
                const int kq = std::min(step, K - q0);
                bool any = false;
                for (int q = q0; q < q0 + kq; ++q)
                    any = any || (again ? w->host[q].active == -1 : w->host[q].active == 1);
                if (!any) continue;
                const int rc = launch<VT, MT, ORTHO, PRE>(A, E, w, q0, kq, K, B, X, o, dscale, stall,
                                                     max_cycles, first, s);
                if (rc) {
                    (void)hipStreamSynchronize(s);  // those before it, in this turn
                    return rc;
                }
                if (launches) ++*launches;
            }
            if (ms) PHG_HIP(hipEventRecord(w->ev[1], s));
            const hipError_t e = hipStreamSynchronize(s);
            if (e != hipSuccess) w->ring_k = 0;
            PHG_HIP(e);
            turn.end();
            if (ms) {
                float t = 0.0f;
                PHG_HIP(hipEventElapsedTime(&t, w->ev[0], w->ev[1]));
                *ms += t;
            }
            if (!*abort_host) break;
            w->ring_k = 0;
            if (*abort_host & ABORT_WAIT) {
                set_error("gmres: a workgroup of the persistent solve timed out waiting for the "
                          "others");
                return PHG_ERR_HIP;
            }
            if (++tries >= XCH_TRIES) {
                for (int q = 0; q < K; ++q)
                    if (w->host[q].active == -1) w->host[q].active = 1;
                return PERSIST_NO_START;
            }
            // two processes that collided do not try again at the same moment
            std::this_thread::sleep_for(std::chrono::microseconds(100 * (1 + (getpid() * 7 + tries) % 32)));
        }
        bool any = false;
        for (int q = 0; q < K; ++q) any = any || w->host[q].active;
        if (!any) break;
    }
    return PHG_OK;
}

template <typename VT, typename MT, typename... Rest>
int run_ortho(phg_matrix_s* A, const Ell<MT>& E, PersistWork* w, int K, const double* B, double* X,
              const phg_gmres_opts& o, Rest... rest)
{
    const bool pre = E.width >= 1 && E.width <= ELL_MAXW;
    switch (o.ortho) {
    case PHG_MGS:
        return pre ? run<VT, MT, PHG_MGS, true>(A, E, w, K, B, X, o, rest...)
                   : run<VT, MT, PHG_MGS, false>(A, E, w, K, B, X, o, rest...);
    case PHG_CGS2:
        return pre ? run<VT, MT, PHG_CGS2, true>(A, E, w, K, B, X, o, rest...)
                   : run<VT, MT, PHG_CGS2, false>(A, E, w, K, B, X, o, rest...);
    default:
        return pre ? run<VT, MT, PHG_CGS1, true>(A, E, w, K, B, X, o, rest...)
                   : run<VT, MT, PHG_CGS1, false>(A, E, w, K, B, X, o, rest...);
    }
}

int solve(phg_matrix_s* A, PersistWork* w, int K, const double* B, double* X,
          const phg_gmres_opts& o, bool diag, bool stall, int max_cycles, int max_rounds,
          int* launches, double* ms, hipStream_t s)
{
    if (o.restart > PS_M || workgroups(A->n_rows) > KR_MAXG) return PERSIST_NOT_HERE;
    const double* none = nullptr;
    if (o.precision == PHG_F64)
        return run_ortho<double, double>(A, diag ? A->ell64d : A->ell64, w, K, B, X, o,
                                         diag ? (const double*)A->dinv.p : none, stall, max_cycles,
                                         max_rounds, launches, ms, s);
    if (o.precision == PHG_F32)
        return run_ortho<float, float>(A, A->ell32, w, K, B, X, o, none, stall, max_cycles,
                                       max_rounds, launches, ms, s);
    return run_ortho<float, uint16_t>(A, A->ell16, w, K, B, X, o, none, stall, max_cycles,
                                      max_rounds, launches, ms, s);
}

}  // namespace
}  // namespace phg
