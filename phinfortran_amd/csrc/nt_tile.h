// nt_tile.h -- complex FP64 matrices of up to 128 held in the registers of a
// workgroup, one wave for every 16 columns.
//
// A wave's columns are in the layout in which v_mfma_f64_16x16x4 returns its
// result: row 4 r + lane / 16 of a tile is element r, and that is the layout in
// which the same instruction takes its B operand, so a chain of products needs
// no exchange between lanes or waves; only A operands come from memory.
#pragma once

#include <type_traits>

#include "nt_device.h"

namespace {

using namespace nt;

typedef double2 C2;

// ------------------------------------------------- one wave's 16 columns
// The lane's number as a value the compiler takes for a new one at every use:
// addresses and masks formed from it are formed where they are used instead of
// being kept, by the hundred, in registers across the solver kernels' loops.
__device__ __forceinline__ int lane_new()
{
    int l = lane_id();
    asm volatile("" : "+v"(l));
    return l;
}

template <int NT>
struct Blk {
    v4d re[NT], im[NT];
};

template <int NT>
__device__ __forceinline__ void blk_zero(Blk<NT>& x)
{
#pragma unroll
    for (int t = 0; t < NT; ++t) x.re[t] = x.im[t] = v4d{0, 0, 0, 0};
}

// Operands in memory: element (cm + lm, ck + lk) of a column-major matrix, of
// its transpose, of its adjoint, and of Gamma^T = (i (S - S^+))^T.  cm, ck are
// the same for all lanes and lm, lk for all uses, so the address is a scalar
// base and one 32-bit lane offset (in LDS an immediate offset).
template <class P>
__device__ __forceinline__ C2 at(P p, int uni, int lane)
{
    return p[uni + lane];
}
template <>
__device__ __forceinline__ C2 at<const C2*>(const C2* p, int uni, int lane)
{
    return *reinterpret_cast<const C2*>(reinterpret_cast<const char*>(p + uni) + (unsigned)(lane * 16));
}
struct LdN {
    const C2* p;
    int ld;
    __device__ __forceinline__ C2 operator()(int cm, int ck, int lm, int lk) const
    {
        return at(p, cm + ck * ld, lm + lk * ld);
    }
};
struct LdT {
    const C2* p;
    int ld;
    __device__ __forceinline__ C2 operator()(int cm, int ck, int lm, int lk) const
    {
        return at(p, ck + cm * ld, lk + lm * ld);
    }
};
struct LdC {
    const C2* p;
    int ld;
    __device__ __forceinline__ C2 operator()(int cm, int ck, int lm, int lk) const
    {
        const C2 v = at(p, ck + cm * ld, lk + lm * ld);
        return make_double2(v.x, -v.y);
    }
};
struct LdGamT {
    const C2* p;
    int ld;
    __device__ __forceinline__ C2 operator()(int cm, int ck, int lm, int lk) const
    {
        const C2 a = at(p, ck + cm * ld, lk + lm * ld), b = at(p, cm + ck * ld, lm + lk * ld);   // S[k][m], S[m][k]
        return make_double2(-(a.y + b.y), a.x - b.x);
    }
};
struct LdNc {           // conjugate
    const C2* p;
    int ld;
    __device__ __forceinline__ C2 operator()(int cm, int ck, int lm, int lk) const
    {
        const C2 v = at(p, cm + ck * ld, lm + lk * ld);
        return make_double2(v.x, -v.y);
    }
};
struct LdGam {          // Gamma
    const C2* p;
    int ld;
    __device__ __forceinline__ C2 operator()(int cm, int ck, int lm, int lk) const
    {
        const C2 a = at(p, cm + ck * ld, lm + lk * ld), b = at(p, ck + cm * ld, lk + lm * ld);   // S[m][k], S[k][m]
        return make_double2(-(a.y + b.y), a.x - b.x);
    }
};
struct LsN {            // the same in LDS
    const C2* p;
    int ld;
    __device__ __forceinline__ C2 operator()(int cm, int ck, int lm, int lk) const { return p[cm + ck * ld + lm + lk * ld]; }
};
struct LsT {
    const C2* p;
    int ld;
    __device__ __forceinline__ C2 operator()(int cm, int ck, int lm, int lk) const { return p[ck + cm * ld + lk + lm * ld]; }
};

// this wave's number, known to be the same in all its lanes
__device__ __forceinline__ int wave_id() { return __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6)); }

// columns 16 w .. 16 w + 15 of a matrix given by a loader
template <int NT, class F>
__device__ __forceinline__ void blk_load(Blk<NT>& x, F ld, int w)
{
    const int lane = lane_new(), l15 = lane & 15, q = lane >> 4;
#pragma unroll
    for (int t = 0; t < NT; ++t)
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            const C2 v = ld(16 * t + 4 * r, 16 * w, q, l15);
            x.re[t][r] = v.x;
            x.im[t][r] = v.y;
        }
    __builtin_amdgcn_sched_barrier(0);
}

template <int NT>
__device__ __forceinline__ void blk_store(const Blk<NT>& x, C2* p, int ld, int w)
{
    const int lane = lane_new(), l15 = lane & 15, q = lane >> 4;
    const unsigned off = (unsigned)(q + l15 * ld) * 16;
#pragma unroll
    for (int t = 0; t < NT; ++t)
#pragma unroll
        for (int r = 0; r < 4; ++r)
            *reinterpret_cast<C2*>(reinterpret_cast<char*>(p + (16 * t + 4 * r + 16 * w * ld)) + off) =
                make_double2(x.re[t][r], x.im[t][r]);
    __builtin_amdgcn_sched_barrier(0);
}

// y += A x; A by a loader, 16 NT square.  The A operands of a step are loaded
// during the step before; the scheduling barrier keeps the compiler from
// loading all of them first, which takes the registers of a second wave.
// Bit NT i + t of mask is clear where A's rows 16 t .. 16 t + 15 are zero in
// its columns 4 i .. 4 i + 3 (such a piece is neither loaded nor multiplied).
template <int NT, bool MASK = false, class F>
__device__ __forceinline__ void blk_mul(Blk<NT>& y, F A, const Blk<NT>& x, unsigned long long mask = ~0ull)
{
    const int lane = lane_new(), l15 = lane & 15, q = lane >> 4;
    C2 a[2][NT];
    auto on = [&](int i, int t) __attribute__((always_inline)) { return !MASK || ((mask >> (NT * i + t)) & 1); };
#pragma unroll
    for (int t = 0; t < NT; ++t)
        if (on(0, t)) a[0][t] = A(16 * t, 0, l15, q);
#pragma unroll
    for (int i = 0; i < 4 * NT; ++i) {
        const int s = i / 4, r = i % 4, c = i & 1;
        if (i + 1 < 4 * NT) {
#pragma unroll
            for (int t = 0; t < NT; ++t)
                if (on(i + 1, t)) a[c ^ 1][t] = A(16 * t, 4 * (i + 1), l15, q);
        }
        const double xr = x.re[s][r], xi = x.im[s][r];
        if (MASK) {
#pragma unroll
            for (int t = 0; t < NT; ++t)
                if (on(i, t)) {
                    y.re[t] = mfma16x16x4(a[c][t].x, xr, y.re[t]);
                    y.im[t] = mfma16x16x4(a[c][t].x, xi, y.im[t]);
                    y.re[t] = mfma16x16x4(-a[c][t].y, xi, y.re[t]);
                    y.im[t] = mfma16x16x4(a[c][t].y, xr, y.im[t]);
                }
        } else {
#pragma unroll
            for (int t = 0; t < NT; ++t) {
                y.re[t] = mfma16x16x4(a[c][t].x, xr, y.re[t]);
                y.im[t] = mfma16x16x4(a[c][t].x, xi, y.im[t]);
            }
#pragma unroll
            for (int t = 0; t < NT; ++t) {
                y.re[t] = mfma16x16x4(-a[c][t].y, xi, y.re[t]);
                y.im[t] = mfma16x16x4(a[c][t].y, xr, y.im[t]);
            }
        }
        __builtin_amdgcn_sched_barrier(0);
    }
}

// y += A x where x's rows 4 i .. 4 i + 3 are zero unless bit NT i of mask is set
template <int NT, class F>
__device__ __forceinline__ void blk_mul_rows(Blk<NT>& y, F A, const Blk<NT>& x, unsigned long long mask)
{
    const int lane = lane_new(), l15 = lane & 15, q = lane >> 4;
#pragma unroll
    for (int i = 0; i < 4 * NT; ++i) {
        if (!((mask >> (NT * i)) & 1)) continue;
        const int s = i / 4, r = i % 4;
        C2 a[NT];
#pragma unroll
        for (int t = 0; t < NT; ++t) a[t] = A(16 * t, 4 * i, l15, q);
        const double xr = x.re[s][r], xi = x.im[s][r];
#pragma unroll
        for (int t = 0; t < NT; ++t) {
            y.re[t] = mfma16x16x4(a[t].x, xr, y.re[t]);
            y.im[t] = mfma16x16x4(a[t].x, xi, y.im[t]);
        }
#pragma unroll
        for (int t = 0; t < NT; ++t) {
            y.re[t] = mfma16x16x4(-a[t].y, xi, y.re[t]);
            y.im[t] = mfma16x16x4(a[t].y, xr, y.im[t]);
        }
        __builtin_amdgcn_sched_barrier(0);
    }
}

__device__ __forceinline__ double read_lane(double v, int lane)
{
    const long long b = __double_as_longlong(v);
    const unsigned lo = __builtin_amdgcn_readlane((int)(b & 0xffffffffll), lane);
    const unsigned hi = __builtin_amdgcn_readlane((int)(b >> 32), lane);
    return __longlong_as_double(((long long)hi << 32) | lo);
}

// largest of 64 lanes' values, in every lane
__device__ __forceinline__ unsigned wave_max(unsigned v)
{
    auto step = [](unsigned x, unsigned y) { return x > y ? x : y; };
    v = step(v, (unsigned)__builtin_amdgcn_update_dpp(0, (int)v, 0x111, 0xf, 0xf, false));   // row_shr:1
    v = step(v, (unsigned)__builtin_amdgcn_update_dpp(0, (int)v, 0x112, 0xf, 0xf, false));   // row_shr:2
    v = step(v, (unsigned)__builtin_amdgcn_update_dpp(0, (int)v, 0x114, 0xf, 0xf, false));   // row_shr:4
    v = step(v, (unsigned)__builtin_amdgcn_update_dpp(0, (int)v, 0x118, 0xf, 0xf, false));   // row_shr:8
    v = step(v, (unsigned)__builtin_amdgcn_update_dpp(0, (int)v, 0x142, 0xa, 0xf, false));   // row_bcast:15
    v = step(v, (unsigned)__builtin_amdgcn_update_dpp(0, (int)v, 0x143, 0xc, 0xf, false));   // row_bcast:31
    return (unsigned)__builtin_amdgcn_readlane((int)v, 63);
}

// Inverse of the matrix of 16 NT rows whose columns NT waves hold in m;
// element (i, j) of it goes to out(i, j, value).  Blocked Gauss-Jordan with
// partial pivoting, rows never exchanged: panel J is the 16 columns of wave J,
// swept with one row per lane (two from 65 rows on; the pivot row reaches the
// other lanes through scalar registers); the other waves then add panel x
// pivot rows by MFMA.  The implicit exchanges are undone by the indexes of the
// final store.  A pivot is the largest |re| + |im| of the free rows to 13 bits
// (the first one of those).  Contains barriers: all waves call it.  work (2
// panels of LD = 16 NT + 1 and 256 elements per wave) must be free, i.e. there
// was a barrier since its last reader; a barrier ends the call.
struct InvLds {
    int *piv;              // pivot row of every column
    int *cinv;             // column a row was the pivot of, or -1
    int *info;             // first zero pivot (1-based) or -1 (NaN, or a pivot over big)
    double big = INFINITY; // bound of |pivot|^2
};

template <int NT, class Out>
__device__ __forceinline__ void wg_inverse(C2* work, const InvLds& s, Blk<NT>& m, Out out)
{
    constexpr int NP = 16 * NT, LD = NP + 1, RPL = (NP + 63) / 64, KM = RPL > 1 ? 255 : 127;
    const int lane = lane_new(), l15 = lane & 15, q = lane >> 4, w = wave_id();
    if (threadIdx.x < NP) s.cinv[threadIdx.x] = -1;
    __syncthreads();
    C2* pb = work + 2 * 16 * LD + w * 256;
#pragma unroll 1
    for (int J = 0; J < NT; ++J) {
        C2* wb = work + (J & 1) * 16 * LD;
        if (w == J) {
            // columns -> rows
#pragma unroll
            for (int t = 0; t < NT; ++t)
#pragma unroll
                for (int r = 0; r < 4; ++r)
                    wb[l15 * LD + 16 * t + 4 * r + q] = make_double2(m.re[t][r], m.im[t][r]);
            __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
            __builtin_amdgcn_wave_barrier();
            double xr[RPL][16], xi[RPL][16];
            double svr = 0.0, svi = 0.0;     // 1 / pivot of a row that became one here
            bool free_row[RPL], here = false;
            int row[RPL];
#pragma unroll
            for (int l = 0; l < RPL; ++l) {
                row[l] = lane + 64 * l < NP ? lane + 64 * l : NP - 1;
                free_row[l] = lane + 64 * l < NP && s.cinv[row[l]] < 0;
#pragma unroll
                for (int c = 0; c < 16; ++c) {
                    const C2 v = wb[c * LD + row[l]];
                    xr[l][c] = v.x;
                    xi[l][c] = v.y;
                }
            }
            // largest |re| + |im| of column 0's free rows, the row in the low bits
            auto pivot_key = [&]() __attribute__((always_inline)) {
                unsigned key = 0;
#pragma unroll
                for (int l = 0; l < RPL; ++l) {
                    const unsigned hi =
                        (unsigned)(__double_as_longlong(fabs(xr[l][0]) + fabs(xi[l][0])) >> 32);
                    const unsigned k = free_row[l] ? ((hi & ~(unsigned)KM) | (unsigned)(64 * RPL - 64 * l - lane)) : 0u;
                    key = k > key ? k : key;
                }
                return wave_max(key) & (unsigned)KM;
            };
            // Column c is always element 0: the columns move down by one per
            // step and the finished one goes to the end, so the loop needs no
            // register indexing.  One wave works here and the steps follow on
            // one another, so what counts is the chain from pivot to pivot.
            // With one row per lane (NP <= 64) the pivot row is read into
            // scalars at once, the next column is updated first and its pivot
            // search overlaps the other columns' updates, the pivot row is
            // scaled after the panel (a row's multipliers scale with it) and
            // no branch is taken in a step: 4096 matrices of 48 take 268 us
            // (293 with the step below), of 64 542 (603).  With two rows per
            // lane the registers do not hold that row beside the panel: the
            // same order spills (96: 2830 us, against 2557), so there the
            // pivot row is read as it is used and scaled in its step.
            if constexpr (RPL == 1) {
                unsigned key = pivot_key();
                int pv = 0;          // lane c: pivot row of column c and its |pivot|^2
                double dn = 1.0;
#pragma unroll 1
                for (int c = 0; c < 16; ++c) {
                    const int pl = __builtin_amdgcn_readfirstlane(64 - (int)key);
                    const double dr = read_lane(xr[0][0], pl), di = read_lane(xi[0][0], pl);
                    double pr[16], pim[16];
#pragma unroll
                    for (int j = 1; j < 16; ++j) {
                        pr[j] = read_lane(xr[0][j], pl);
                        pim[j] = read_lane(xi[0][j], pl);
                    }
                    const double den = dr * dr + di * di;
                    // 1 / den: the instruction's estimate and two Newton steps
                    double rc = __builtin_amdgcn_rcp(den);
                    rc = fma(rc, fma(-den, rc, 1.0), rc);
                    rc = fma(rc, fma(-den, rc, 1.0), rc);
                    double vr = dr * rc, vi = -di * rc;      // 1 / pivot
                    // where 1 / den has no double, or den is zero or not finite
                    if (__builtin_expect(!(den > 1e-290 && den < 1e290), 0)) {
                        vr = den != 0.0 ? dr / den : 0.0;
                        vi = den != 0.0 ? -di / den : 0.0;
                    }
                    const bool own = lane == pl;
                    const double fr = xr[0][0], fi = xi[0][0];
                    const double tr = fr * vr - fi * vi, ti = fr * vi + fi * vr;
                    const double gxr = own ? 0.0 : tr, gxi = own ? 0.0 : ti;    // multiplier f / pivot
                    free_row[0] = free_row[0] && !own;
                    here = here || own;
                    svr = own ? vr : svr;
                    svi = own ? vi : svi;
                    xr[0][0] = fma(gxi, pim[1], fma(-gxr, pr[1], xr[0][1]));
                    xi[0][0] = fma(-gxi, pr[1], fma(-gxr, pim[1], xi[0][1]));
                    pv = lane == c ? pl : pv;
                    dn = lane == c ? den : dn;
                    key = pivot_key();
#pragma unroll
                    for (int j = 2; j < 16; ++j) {
                        xr[0][j - 1] = fma(-gxr, pr[j], xr[0][j]);
                        xi[0][j - 1] = fma(-gxr, pim[j], xi[0][j]);
                    }
#pragma unroll
                    for (int j = 2; j < 16; ++j) {
                        xr[0][j - 1] = fma(gxi, pim[j], xr[0][j - 1]);
                        xi[0][j - 1] = fma(-gxi, pr[j], xi[0][j - 1]);
                    }
                    xr[0][15] = own ? 1.0 : -gxr;
                    xi[0][15] = own ? 0.0 : -gxi;
                }
                // the panel's pivots: their record, the first bad one, their rows' scale
                if (lane < 16) {
                    s.piv[16 * J + lane] = pv;
                    s.cinv[pv] = 16 * J + lane;
                }
                const unsigned long long bad = __ballot(lane < 16 && (!(dn > 0.0) || dn > s.big));
                if (bad && *s.info == 0) {
                    const int c = __ffsll((long long)bad) - 1;
                    if (lane == c) *s.info = dn == 0.0 ? 16 * J + c + 1 : -1;
                }
            } else {
#pragma unroll 1
                for (int c = 0; c < 16; ++c) {
                    const int p = __builtin_amdgcn_readfirstlane(64 * RPL - (int)pivot_key()), pl = p & 63;
                    // the step with the pivot row in slot SL of its lane
                    auto step = [&](auto slot) __attribute__((always_inline)) {
                        constexpr int SL = decltype(slot)::value;
                        const double dr = read_lane(xr[SL][0], pl), di = read_lane(xi[SL][0], pl);
                        const double den = dr * dr + di * di;
                        double vr = 0.0, vi = 0.0;      // 1 / pivot
                        if (den != 0.0) {
                            const double rc = 1.0 / den;
                            vr = dr * rc;
                            vi = -di * rc;
                        }
                        // (where 1 / den has no double)
                        if (__builtin_expect(den != 0.0 && !(den > 1e-290 && den < 1e290), 0)) {
                            vr = dr / den;
                            vi = -di / den;
                        }
                        if (lane == 0) {
                            s.piv[16 * J + c] = p;
                            s.cinv[p] = 16 * J + c;
                            if (!(den > 0.0) || den > s.big) {
                                if (*s.info == 0) *s.info = den == 0.0 ? 16 * J + c + 1 : -1;
                            }
                        }
                        // multiplier f / pivot; the pivot row becomes row / pivot
                        double gxr[RPL], gxi[RPL], keep[RPL];
#pragma unroll
                        for (int l = 0; l < RPL; ++l) {
                            const bool own = l == SL && lane == pl;
                            if (own) free_row[l] = false;
                            const double fr = xr[l][0], fi = xi[l][0];
                            gxr[l] = own ? -vr : fr * vr - fi * vi;
                            gxi[l] = own ? -vi : fr * vi + fi * vr;
                            keep[l] = own ? 0.0 : 1.0;
                        }
#pragma unroll
                        for (int j = 1; j < 16; ++j) {
                            const double pr = read_lane(xr[SL][j], pl), pim = read_lane(xi[SL][j], pl);
#pragma unroll
                            for (int l = 0; l < RPL; ++l) {
                                const double a = l == SL ? xr[l][j] * keep[l] : xr[l][j];
                                const double b = l == SL ? xi[l][j] * keep[l] : xi[l][j];
                                xr[l][j - 1] = a - gxr[l] * pr + gxi[l] * pim;
                                xi[l][j - 1] = b - gxr[l] * pim - gxi[l] * pr;
                            }
                        }
#pragma unroll
                        for (int l = 0; l < RPL; ++l) {
                            xr[l][15] = -gxr[l];
                            xi[l][15] = -gxi[l];
                        }
                    };
                    if (p < 64) step(std::integral_constant<int, 0>{});
                    else step(std::integral_constant<int, RPL - 1>{});
                }
            }
#pragma unroll
            for (int l = 0; l < RPL; ++l)
                if (lane + 64 * l < NP) {
#pragma unroll
                    for (int c = 0; c < 16; ++c) {
                        C2 v = make_double2(xr[l][c], xi[l][c]);
                        if (RPL == 1 && here) v = make_double2(v.x * svr - v.y * svi, v.x * svi + v.y * svr);
                        wb[c * LD + row[l]] = v;
                    }
                }
            // (a barrier in either branch: m is not live while its wave sweeps)
            __syncthreads();
#pragma unroll
            for (int t = 0; t < NT; ++t)
#pragma unroll
                for (int r = 0; r < 4; ++r) {
                    const C2 v = wb[l15 * LD + 16 * t + 4 * r + q];
                    m.re[t][r] = v.x;
                    m.im[t][r] = v.y;
                }
        } else {
            __syncthreads();
            // the panel's pivot rows of this wave's columns, in pivot order;
            // the rows themselves start from zero
#pragma unroll
            for (int t = 0; t < NT; ++t)
#pragma unroll
                for (int r = 0; r < 4; ++r) {
                    const int k = s.cinv[16 * t + 4 * r + q] - 16 * J;
                    if (k >= 0 && k < 16) {
                        pb[k * 16 + l15] = make_double2(m.re[t][r], m.im[t][r]);
                        m.re[t][r] = 0.0;
                        m.im[t][r] = 0.0;
                    }
                }
            __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
            __builtin_amdgcn_wave_barrier();
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                const C2 pv = pb[(4 * r + q) * 16 + l15];
                C2 a[NT];
#pragma unroll
                for (int t = 0; t < NT; ++t) a[t] = wb[(4 * r + q) * LD + 16 * t + l15];
#pragma unroll
                for (int t = 0; t < NT; ++t) {
                    m.re[t] = mfma16x16x4(a[t].x, pv.x, m.re[t]);
                    m.im[t] = mfma16x16x4(a[t].x, pv.y, m.im[t]);
                }
#pragma unroll
                for (int t = 0; t < NT; ++t) {
                    m.re[t] = mfma16x16x4(-a[t].y, pv.y, m.re[t]);
                    m.im[t] = mfma16x16x4(a[t].y, pv.x, m.im[t]);
                }
                __builtin_amdgcn_sched_barrier(0);
            }
        }
    }
    __syncthreads();
    const int oc = s.piv[16 * w + l15];
#pragma unroll
    for (int t = 0; t < NT; ++t)
#pragma unroll
        for (int r = 0; r < 4; ++r) out(s.cinv[16 * t + 4 * r + q], oc, make_double2(m.re[t][r], m.im[t][r]));
    __syncthreads();
}

// largest v of NW waves, in every lane (two barriers)
template <int NW>
__device__ __forceinline__ double wg_max(double* red, double v)
{
#pragma unroll
    for (int o = 32; o; o >>= 1) v = fmax(v, __shfl_xor(v, o));
    __syncthreads();
    if (lane_id() == 0) red[wave_id()] = v;
    __syncthreads();
    double r = red[0];
#pragma unroll
    for (int i = 1; i < NW; ++i) r = fmax(r, red[i]);
    return r;
}

// largest modulus of a wave's columns, infinite with a NaN among them
template <int NT>
__device__ __forceinline__ double blk_maxabs(const Blk<NT>& x)
{
    double v = 0.0;
#pragma unroll
    for (int t = 0; t < NT; ++t)
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            const double a = sqrt(x.re[t][r] * x.re[t][r] + x.im[t][r] * x.im[t][r]);
            v = a > v || a != a ? (a != a ? INFINITY : a) : v;      // NaN never converges
        }
    return v;
}

}  // namespace
