// Device functions that the single right-hand-side GMRES (gmres.hip) and the
// persistent solve (persist.hip) share: lane sums, the dots of one vector
// with a tier of basis vectors, the Arnoldi product of a thread's rows, the
// triangular solve of the modified Gram-Schmidt coefficients and the Givens
// rotation.  Both forms run these functions over the same rows per thread
// and add their block partials in the same order (krylov_total), so they
// give the same bits.
#pragma once
#include <hip/hip_runtime.h>

#include "ell.h"

namespace phg {

constexpr int KR_RPT = 2;       // rows per thread
constexpr int KR_STRIDE = 512;  // between a thread's rows
constexpr int KR_T = 8;         // basis vectors per tier of dots
constexpr int KR_MAXG = 256;    // most workgroups of a persistent launch

// A double moved between lanes by a DPP pattern (both 32-bit halves).
template <int CTRL>
__device__ __forceinline__ double dpp_d(double v)
{
    const unsigned long long u = (unsigned long long)__double_as_longlong(v);
    const int lo = __builtin_amdgcn_update_dpp(0, (int)(unsigned)u, CTRL, 0xF, 0xF, false);
    const int hi = __builtin_amdgcn_update_dpp(0, (int)(unsigned)(u >> 32), CTRL, 0xF, 0xF, false);
    return __longlong_as_double((long long)(((unsigned long long)(unsigned)hi << 32) | (unsigned)lo));
}

// a of this lane plus a of the partner in the lower half (ROWS 32) or even
// 16-lane row (16), b plus b of the partner in the others: one swap per
// 32-bit half serves two sums.
template <int ROWS>
__device__ __forceinline__ double swap_add(double a, double b)
{
    const unsigned long long ua = (unsigned long long)__double_as_longlong(a);
    const unsigned long long ub = (unsigned long long)__double_as_longlong(b);
    const auto lo = ROWS == 16
                        ? __builtin_amdgcn_permlane16_swap((unsigned)ua, (unsigned)ub, false, false)
                        : __builtin_amdgcn_permlane32_swap((unsigned)ua, (unsigned)ub, false, false);
    const auto hi = ROWS == 16 ? __builtin_amdgcn_permlane16_swap(
                                     (unsigned)(ua >> 32), (unsigned)(ub >> 32), false, false)
                               : __builtin_amdgcn_permlane32_swap(
                                     (unsigned)(ua >> 32), (unsigned)(ub >> 32), false, false);
    const double x = __longlong_as_double((long long)(((unsigned long long)hi[0] << 32) | lo[0]));
    const double y = __longlong_as_double((long long)(((unsigned long long)hi[1] << 32) | lo[1]));
    return x + y;
}

// Sum over the 64 lanes of a wavefront, all active, the same bits in every
// lane: lane pairs 32, 16 and 8 apart, then the mirror lane within 8, the
// lane 2 and the lane 1 apart (VALU lane moves, no LDS).
__device__ __forceinline__ double wave_sum(double v)
{
    v = swap_add<32>(v, v);
    v = swap_add<16>(v, v);
    v += dpp_d<0x128>(v);  // row_ror:8
    v += dpp_d<0x141>(v);  // row_half_mirror
    v += dpp_d<0x4E>(v);   // quad_perm [2,3,0,1]
    v += dpp_d<0xB1>(v);   // quad_perm [1,0,3,2]
    return v;
}

// Eight such sums at once: every step of the first three halves the values a
// lane carries, so the eight cost 34 instructions instead of 8 x 21.  Lane l
// returns the sum of value reduce8_value(l), in wave_sum's order.
__device__ __forceinline__ int reduce8_value(int lane) { return lane >> 3; }
__device__ __forceinline__ double reduce8(const double (&p)[KR_T])
{
    const int lane = threadIdx.x & 63;
    double a[4], b[2];
    // after the 32-lane swap lanes 0..31 hold values 0..3, the others 4..7,
    // after the 16-lane one odd rows the upper two of those
#pragma unroll
    for (int i = 0; i < 4; ++i) a[i] = swap_add<32>(p[i], p[i + 4]);
#pragma unroll
    for (int i = 0; i < 2; ++i) b[i] = swap_add<16>(a[i], a[i + 2]);
    const bool up = lane & 8;
    const double keep = up ? b[1] : b[0], send = up ? b[0] : b[1];
    double v = keep + dpp_d<0x128>(send);
    v += dpp_d<0x141>(v);
    v += dpp_d<0x4E>(v);
    v += dpp_d<0xB1>(v);
    return v;
}

// Value of v in lane `lane` (wave-uniform index): two v_readlane_b32.
__device__ __forceinline__ double readlane_d(double v, int lane)
{
    const unsigned long long u = __double_as_longlong(v);
    const unsigned lo = __builtin_amdgcn_readlane((unsigned)u, lane);
    const unsigned hi = __builtin_amdgcn_readlane((unsigned)(u >> 32), lane);
    return __longlong_as_double((long long)(((unsigned long long)hi << 32) | lo));
}

template <typename T>
__device__ __forceinline__ double to_d(T v) { return (double)v; }

__device__ __forceinline__ double kfma(double a, double b, double c) { return fma(a, b, c); }
__device__ __forceinline__ float kfma(float a, float b, float c) { return fmaf(a, b, c); }

// Agent-scope relaxed accesses: for values that other workgroups of the same
// launch write or read (they do not stay in this XCD's L2).
template <typename T>
__device__ __forceinline__ T ld_agent(const T* p)
{
    return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
template <typename T>
__device__ __forceinline__ void st_agent(T* p, T v)
{
    __hip_atomic_store(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
// v as a value the compiler knows nothing about: addresses that depend on it
// are formed where they are used instead of being kept in registers across a
// loop (the persistent kernel has none to spare).
__device__ __forceinline__ int opaque(int v)
{
    asm volatile("" : "+v"(v));
    return v;
}

template <bool AGENT, typename T>
__device__ __forceinline__ T ld_x(const T* p)
{
    if constexpr (AGENT) return ld_agent(p);
    else return *p;
}

// One term of a row's sum: s + val * (x * inv) in FP64 (no fused
// multiply-add), fmaf(val, x * inv, s) in FP32, as ell_row_f64 and
// ell_row_f32 add them.
template <typename VT, typename MT>
struct RowTerm;
template <>
struct RowTerm<double, double> {
    __device__ __forceinline__ static double add(double s, double v, double x, double inv)
    {
        return s + v * (x * inv);
    }
};
template <typename MT>
struct RowTerm<float, MT> {
    __device__ __forceinline__ static float add(float s, MT v, float x, float inv)
    {
        return fmaf(ell_val_f32(v), x * inv, s);
    }
};

// Rows of any width: base + r * KR_STRIDE (r < RG) of A x, ELL_MAXW entries of
// a row at a time: their slots, then their gathers, then the sums in slot
// order.  163,841 rows of 11 and of 27 entries, a step of the FP64 persistent
// solve: 13.8 and 19.9 us, entry by entry 17.6 and 38.7.
template <typename VT, typename MT, bool AGENT, int RG>
__device__ __forceinline__ void krylov_rows_loop(int n, int width, int base,
                                                 const int* __restrict__ col,
                                                 const MT* __restrict__ val, const VT* x, int ldx,
                                                 VT inv, VT* xo, VT* w)
{
#pragma unroll
    for (int q = 0; q < RG; ++q) {
        const int rr = base + q * KR_STRIDE;
        xo[q] = VT(0);
        w[q] = VT(0);
        if (rr < n) {
            xo[q] = ld_x<AGENT>(x + (size_t)rr * ldx);
            VT s = VT(0);
#pragma unroll 1
            for (int k0 = 0; k0 < width; k0 += ELL_MAXW) {
                int c[ELL_MAXW];
                MT v[ELL_MAXW];
                VT xv[ELL_MAXW];
#pragma unroll
                for (int k = 0; k < ELL_MAXW; ++k) {
                    const size_t o = ell_slot(k0 + k, width, n, rr);
                    c[k] = col[o];
                    v[k] = val[o];
                }
#pragma unroll
                for (int k = 0; k < ELL_MAXW; ++k) xv[k] = ld_x<AGENT>(x + (size_t)c[k] * ldx);
#pragma unroll
                for (int k = 0; k < ELL_MAXW; ++k) {
                    const VT t = RowTerm<VT, MT>::add(s, v[k], xv[k], inv);
                    s = k0 + k < width ? t : s;
                }
            }
            w[q] = s;
        }
    }
}

// The same entry by entry (k_step_spmv and k_persist have the reason).
template <typename VT, typename MT, bool AGENT, int RG>
__device__ __forceinline__ void krylov_rows_each(int n, int width, int base,
                                                 const int* __restrict__ col,
                                                 const MT* __restrict__ val, const VT* x, int ldx,
                                                 VT inv, VT* xo, VT* w)
{
#pragma unroll
    for (int q = 0; q < RG; ++q) {
        const int rr = base + q * KR_STRIDE;
        xo[q] = VT(0);
        w[q] = VT(0);
        if (rr < n) {
            xo[q] = ld_x<AGENT>(x + (size_t)rr * ldx);
            VT s = VT(0);
            for (int k = 0; k < width; ++k) {
                const size_t o = (size_t)k * n + rr;
                s = RowTerm<VT, MT>::add(s, val[o], ld_x<AGENT>(x + (size_t)col[o] * ldx), inv);
            }
            w[q] = s;
        }
    }
}

// Rows base + r * KR_STRIDE (r < RG) of A x (x scaled by inv): xo[r] = x[row],
// w[r] = the row's sum, both 0 at and past row n; x entry i at x[i * ldx].
// SHORT: rows of 1 to ELL_MAXW entries; every row's own entry and slots are
// loaded first, then every gather, then the sums in slot order: two memory
// round trips for the group.
template <typename VT, typename MT, bool AGENT, int RG, bool SHORT>
__device__ __forceinline__ void krylov_rows(int n, int width, int base, const int* __restrict__ col,
                                            const MT* __restrict__ val, const VT* x, int ldx,
                                            VT inv, VT* xo, VT* w)
{
    if constexpr (SHORT) {
        int c[RG][ELL_MAXW];
        MT v[RG][ELL_MAXW];
        VT xv[RG][ELL_MAXW];
#pragma unroll
        for (int q = 0; q < RG; ++q) {
            const int rr = min(base + q * KR_STRIDE, n - 1);  // in bounds; unused past n
            xo[q] = ld_x<AGENT>(x + (size_t)rr * ldx);
#pragma unroll
            for (int k = 0; k < ELL_MAXW; ++k) {
                const size_t o = ell_slot(k, width, n, rr);
                c[q][k] = col[o];
                v[q][k] = val[o];
            }
        }
#pragma unroll
        for (int q = 0; q < RG; ++q)
#pragma unroll
            for (int k = 0; k < ELL_MAXW; ++k) xv[q][k] = ld_x<AGENT>(x + (size_t)c[q][k] * ldx);
#pragma unroll
        for (int q = 0; q < RG; ++q) {
            VT s = VT(0);
#pragma unroll
            for (int k = 0; k < ELL_MAXW; ++k) {
                const VT t = RowTerm<VT, MT>::add(s, v[q][k], xv[q][k], inv);
                s = k < width ? t : s;
            }
            const bool in = base + q * KR_STRIDE < n;
            w[q] = in ? s : VT(0);
            xo[q] = in ? xo[q] : VT(0);
        }
    } else {
        krylov_rows_loop<VT, MT, AGENT, RG>(n, width, base, col, val, x, ldx, inv, xo, w);
    }
}
template <typename VT, typename MT, bool AGENT, int RG>
__device__ __forceinline__ void krylov_rows(int n, int width, int base, const int* __restrict__ col,
                                            const MT* __restrict__ val, const VT* x, int ldx,
                                            VT inv, VT* xo, VT* w)
{
    if (width >= 1 && width <= ELL_MAXW)
        krylov_rows<VT, MT, AGENT, RG, true>(n, width, base, col, val, x, ldx, inv, xo, w);
    else
        krylov_rows<VT, MT, AGENT, RG, false>(n, width, base, col, val, x, ldx, inv, xo, w);
}

// A thread's share of the dots of w with KR_T basis vectors.
template <typename VT>
__device__ __forceinline__ void dots_tier(const VT (&w)[KR_RPT], const VT (&v)[KR_T][KR_RPT],
                                          double (&p)[KR_T])
{
#pragma unroll
    for (int q = 0; q < KR_T; ++q) {
        double a = 0.0;
#pragma unroll
        for (int r = 0; r < KR_RPT; ++r) a = fma(to_d(w[r]), to_d(v[q][r]), a);
        p[q] = a;
    }
}

// Wavefronts' sums 0..3 or 4..7 of a block of 1024 rows; the block's partial
// is the sum of the two halves.
__device__ __forceinline__ double krylov_half(double a, double b, double c, double d)
{
    return ((a + b) + c) + d;
}

// Block partials g = 0..G-1 are added as 32 running sums (g mod 32, in g
// order), then the sums q and q + 16, then the sixteen results in order.
__device__ __forceinline__ double krylov_join(const double (*s)[33], int i)
{
    double r = s[0][i];
#pragma unroll
    for (int q = 1; q < 16; ++q) r += s[q][i];
    return r;
}

// Modified Gram-Schmidt coefficients from the dots r_i = <v_i, w> (lane i)
// and the basis vectors' products L(i, k) = <v_i, v_k>, k < i: subtracting
// h_0 v_0 from w before the dot with v_1, and so on, gives h_i = r_i -
// sum_{k<i} L(i, k) h_k, a triangular solve.  All 64 lanes of a wavefront;
// lane i (li = its row, at most j) returns h_i.
template <int MAXM>
__device__ __forceinline__ double mgs_solve(double r, int j, const double* L, int ldl, int li)
{
#pragma unroll
    for (int k0 = 0; k0 < MAXM; k0 += 8) {
        if (k0 >= j) break;
        double l[8];
#pragma unroll
        for (int q = 0; q < 8; ++q) l[q] = L[li * ldl + k0 + q];  // used for k < li only
#pragma unroll
        for (int q = 0; q < 8; ++q) {
            const double h = readlane_d(r, k0 + q);
            r = k0 + q < j && li > k0 + q ? fma(-l[q], h, r) : r;
        }
    }
    return r;
}

// Givens rotation of step j (j < 64) from the Hessenberg column h[0..j] (in
// LDS, written by this wavefront before) and ||w||.  All 64 lanes of a
// wavefront compute the same values from broadcast reads, so that the chain
// is one fused multiply-add per rotation; the state is written by lane 0
// (R's column by the lane of each row).  cs: cos and sin of each rotation,
// one pair after the other.  Arrays hold a multiple of 8 entries.
struct GivensOut {
    bool cont;
    int iters;
};
__device__ __forceinline__ GivensOut krylov_givens(int j, int m, const double* h, double hn,
                                                   double stop, int iters0, int max_iters,
                                                   double* cs, double* g, double* carry, double* R,
                                                   int ldr)
{
    const int lane = threadIdx.x & 63;
    double cur = h[0];
    const double cy = carry[j];
    double tv = 0.0;  // lane i keeps R(i, j): one store per lane after the loop
    for (int i0 = 0; i0 < j; i0 += 8) {
        double c[8], s[8], a[8], b[8];
#pragma unroll
        for (int q = 0; q < 8; ++q) {
            const double up = h[i0 + q + 1];
            c[q] = cs[2 * (i0 + q)], s[q] = cs[2 * (i0 + q) + 1];
            a[q] = c[q] * up, b[q] = s[q] * up;
        }
#pragma unroll
        for (int q = 0; q < 8; ++q) {
            if (i0 + q >= j) break;
            const double t = fma(c[q], cur, b[q]);
            cur = fma(-s[q], cur, a[q]);
            tv = lane == i0 + q ? t : tv;
        }
    }
    // away from overflow and underflow of the squares, hypot's value directly
    const double big = fmax(fabs(cur), hn);
    const double r = big > 1e-140 && big < 1e140 ? sqrt(fma(cur, cur, hn * hn)) : hypot(cur, hn);
    const double cj = cur / r, sj = hn / r;
    const double gj = cj * cy, cn = -sj * cy;
    const int iters = iters0 + j + 1;
    const bool cont = !(fabs(cn) <= stop || !(hn > 0.0) || iters >= max_iters || j + 1 == m);
    if (lane < j) R[lane * ldr + j] = tv;
    if (lane == 0) {
        R[j * ldr + j] = r;
        cs[2 * j] = cj;
        cs[2 * j + 1] = sj;
        g[j] = gj;
        carry[j + 1] = cn;
    }
    return GivensOut{cont, iters};
}

// y = R^-1 g, one wavefront, lane i the row i: column by column from the
// last, so each step is one division and one update of every row above.
__device__ __forceinline__ double krylov_solve_y(int k, const double* R, int ldr, const double* g)
{
    const int lane = threadIdx.x & 63;
    double s = lane < k ? g[lane] : 0.0, y = 0.0;
    for (int l = k - 1; l >= 0; --l) {
        const double col = lane <= l ? R[lane * ldr + l] : 0.0;
        const double yl = readlane_d(s, l) / readlane_d(col, l);
        y = lane == l ? yl : y;
        s = lane < l ? fma(-col, yl, s) : s;
    }
    return y;
}

}  // namespace phg
