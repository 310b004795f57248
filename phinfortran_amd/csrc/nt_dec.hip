// nt_dec.hip -- Lopez-Sancho decimation (negf/surface.f90:479-497) of dense
// leads of at most 64 degrees of freedom, one kernel for the whole recursion.
#include "nt_kernels.h"
#include "nt_tile.h"

namespace nt {

namespace {

constexpr int DEC_MAXNT = 4;
constexpr int DEC_SLOTS = 5;        // matrices of NP^2 per item: alpha twice, beta, e, g

// One workgroup per item, NT waves of 16 columns each.  A step inverts z - e in
// the registers (nt_tile.h) and forms
//   e += alpha (g beta) + beta (g alpha), es += alpha (g beta),
//   alpha' = alpha (g alpha), beta' = beta (g beta)
// from the wave's own columns of alpha and beta: the products in brackets stay
// in registers, so six products need two barriers and no pass over memory but
// the A operands, which come from L2.  As launches a step was an inverse and
// four products, each reading and writing every matrix, with the smaller ones
// padded to an output tile.  Bound by the pivot chain of the inverse for few
// items and by the MFMAs and L2 reads for many: two items of n = 48 take 0.19 ms
// (as launches 0.9, mostly gaps), 5978 of them 13.6 ms (21).  Three waves per
// SIMD up to n = 48, at the price of 100 bytes of scratch: 13.6 ms against 16.5
// with two; at n = 64 the columns alone take the registers of two.
template <int NT>
__global__ __launch_bounds__(64 * NT, NT < 4 ? 3 : 2) void k_dec_tile(DecTileArgs a)
{
    constexpr int NP = 16 * NT, NN = NP * NP, LD = NP + 1;
    const int p = blockIdx.x;
    if (!a.active[p]) return;
    __shared__ C2 work[2 * 16 * LD + NT * 256];
    __shared__ int piv[NP], cinv[NP], info;
    __shared__ double red[NT];
    if (threadIdx.x == 0) info = 0;
    const InvLds il{piv, cinv, &info};
    const int n = a.n, w = wave_id();
    const double zr = a.z[2 * p], zi = a.z[2 * p + 1];
    C2* sc = reinterpret_cast<C2*>(a.scratch) + (long)p * DEC_SLOTS * NN;
    C2 *al = sc, *aln = sc + NN, *be = sc + 2 * NN, *e = sc + 3 * NN, *G = sc + 4 * NN;
    C2* es = reinterpret_cast<C2*>(bptr(a.es, p, 0));
    const int lds = a.es.ld;
    Blk<NT> x, y, u;
    auto load = [&](Blk<NT>& b, const C2* m) __attribute__((always_inline)) { blk_load<NT>(b, LdN{m, NP}, w); };
    auto store = [&](const Blk<NT>& b, C2* m) __attribute__((always_inline)) { blk_store<NT>(b, m, NP, w); };
    // es += v or es = v on the n x n of it
    auto to_es = [&](const Blk<NT>& v, bool add) __attribute__((always_inline)) {
        const int lane = lane_new(), q = lane >> 4, col = 16 * w + (lane & 15);
#pragma unroll
        for (int t = 0; t < NT; ++t)
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                const int row = 16 * t + 4 * r + q;
                if (row < n && col < n) {
                    C2 o = make_double2(v.re[t][r], v.im[t][r]);
                    if (add) {
                        const C2 s = es[row + (long)col * lds];
                        o.x += s.x;
                        o.y += s.y;
                    }
                    es[row + (long)col * lds] = o;
                }
            }
    };
    // n x n input, dagger: its adjoint; zero beyond n
    auto input = [&](const BMat<double>& M, bool dagger) __attribute__((always_inline)) {
        const double* m = bptr(M, p, 0);
        const int lane = lane_new(), q = lane >> 4, col = 16 * w + (lane & 15);
#pragma unroll
        for (int t = 0; t < NT; ++t)
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                const int row = 16 * t + 4 * r + q;
                x.re[t][r] = x.im[t][r] = 0.0;
                if (row < n && col < n) {
                    const double* s = m + 2 * (dagger ? col + (long)row * M.ld : row + (long)col * M.ld);
                    x.re[t][r] = s[0];
                    x.im[t][r] = dagger ? -s[1] : s[1];
                }
            }
    };
    input(a.H00, false);
    store(x, e);
    to_es(x, false);
    input(a.V, !a.alpha_dagger);
    store(x, be);
    input(a.V, a.alpha_dagger);
    store(x, al);
    double amax = wg_max<NT>(red, blk_maxabs<NT>(x));     // its barriers also publish the slots
    int it = 0, dead = 0;
    bool still = amax > a.conv;
    while (still && it < a.max_iter) {
        load(x, e);
        {
            const int lane = lane_new(), q = lane >> 4, col = 16 * w + (lane & 15);
#pragma unroll
            for (int t = 0; t < NT; ++t)
#pragma unroll
                for (int r = 0; r < 4; ++r) {
                    const int row = 16 * t + 4 * r + q;
                    const bool in = row < n && col < n, dg = row == col;
                    x.re[t][r] = in ? (dg ? zr : 0.0) - x.re[t][r] : (dg ? 1.0 : 0.0);
                    x.im[t][r] = in ? (dg ? zi : 0.0) - x.im[t][r] : 0.0;
                }
        }
        wg_inverse<NT>(work, il, x, [&](int i, int j, C2 v) { G[i + j * NP] = v; });
        // beta's side: u = beta' (held back: the others still read beta)
        load(x, be);
        blk_zero<NT>(y);
        blk_mul<NT>(y, LdN{G, NP}, x);
        blk_zero<NT>(x);
        blk_mul<NT>(x, LdN{al, NP}, y);
        to_es(x, true);
        load(u, e);
#pragma unroll
        for (int t = 0; t < NT; ++t) u.re[t] += x.re[t], u.im[t] += x.im[t];
        store(u, e);
        blk_zero<NT>(u);
        blk_mul<NT>(u, LdN{be, NP}, y);
        // alpha's side
        load(x, al);
        blk_zero<NT>(y);
        blk_mul<NT>(y, LdN{G, NP}, x);
        load(x, e);
        blk_mul<NT>(x, LdN{be, NP}, y);
        store(x, e);
        blk_zero<NT>(x);
        blk_mul<NT>(x, LdN{al, NP}, y);
        store(x, aln);
        double v = blk_maxabs<NT>(x);
#pragma unroll
        for (int o = 32; o; o >>= 1) v = fmax(v, __shfl_xor(v, o));
        __syncthreads();
        store(u, be);
        if (lane_id() == 0) red[w] = v;
        __syncthreads();
        amax = red[0];
#pragma unroll
        for (int i = 1; i < NT; ++i) amax = fmax(amax, red[i]);
        C2* sw = al;
        al = aln;
        aln = sw;
        ++it;
        still = amax > a.conv;
        // a decimation that left the finite numbers ends at once
        if (still && amax > 1.7976931348623157e308 && it + 2 <= a.max_iter) {
            still = false;
            dead = 1;
        }
    }
    if (threadIdx.x == 0) {
        a.iters[p] = dead ? a.max_iter : it;
        a.active[p] = still;
        const int st = info ? info : dead ? -1 : 0;
        if (st && a.status[p] == 0) a.status[p] = st;
    }
}

}  // namespace

size_t dec_tile_scratch(int n)
{
    const int np = (n + 15) / 16 * 16;
    return np <= 16 * DEC_MAXNT ? sizeof(C2) * DEC_SLOTS * np * np : 0;
}

hipError_t launch_dec_tile(const DecTileArgs& a, hipStream_t s)
{
    if (a.batch <= 0 || a.n <= 0) return hipSuccess;
    switch ((a.n + 15) / 16) {
        case 1: hipLaunchKernelGGL(k_dec_tile<1>, dim3(a.batch), dim3(64), 0, s, a); break;
        case 2: hipLaunchKernelGGL(k_dec_tile<2>, dim3(a.batch), dim3(128), 0, s, a); break;
        case 3: hipLaunchKernelGGL(k_dec_tile<3>, dim3(a.batch), dim3(192), 0, s, a); break;
        case 4: hipLaunchKernelGGL(k_dec_tile<4>, dim3(a.batch), dim3(256), 0, s, a); break;
        default: return hipErrorInvalidValue;
    }
    return hipGetLastError();
}

}  // namespace nt
