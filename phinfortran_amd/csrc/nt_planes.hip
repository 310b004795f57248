// nt_planes.hip -- batched solve on the planes of the principal layers.
//
// Force constants and hoppings of short range couple a principal layer to the
// next one through a few of its degrees of freedom only, and inside the layer
// they couple neighbours.  The degrees of freedom of every layer, sorted by
// their distance (in couplings) from the ones the previous layer touches, then
// form planes that couple to the plane before and after only: a diamond layer
// one conventional cell thick has four, of a quarter of its size.  The same
// block elimination (lead decimation, both sweeps, Caroli T) on these smaller
// blocks gives the same Green's functions with (planes per layer)^2 fewer
// operations: b = 192, L = 40 takes 1.9 GFLOP per point instead of 29.
//
//   k_pl_pattern  which elements of the blocks are nonzero at any k-point
//   k_pl_levels   per layer: distances from the previous layer, plane counts
//   k_pl_plan     plane size class (16, 32, 48, 64, 96), plane offsets, validity
//   k_pl_perm     degrees of freedom of every plane
//   k_pl_pack     diagonal and coupling blocks of the planes, per k-point,
//                 zero padded to the class size
//   k_pl_decimate one workgroup per (point, lead): the lead's self-energy
//   k_pl_sweep    one workgroup per (point, direction): the whole sweep and T
//   k_pl_finish   statuses, iteration counts, clamps
//
// The plan stays on the device: no kernel needs the host to know it, so a
// solve can be captured in a HIP graph.  Blocks without zeros form one plane
// per layer and are left to the block path, as are planes over 96.
//
// The solver kernels work on matrices held in registers (nt_tile.h).
#include <type_traits>

#include "nt_host.h"
#include "nt_kernels.h"
#include "nt_planes.h"
#include "nt_tile.h"

namespace {

constexpr int PL_MAXNT = 4;         // planes of up to 64: both solver kernels
constexpr int PL_BIGNT = 6;         // planes of up to 96: the sweep's (planes_big_leads decimates)
constexpr int PL_NCLS = 5;          // plane size classes 16, 32, 48, 64, 96
constexpr int PL_PERM = 16 * PL_BIGNT;
__host__ __device__ constexpr int class_nt(int t) { return t < PL_MAXNT ? t + 1 : PL_BIGNT; }
constexpr int PL_WAVES = 2;          // waves per SIMD the solver kernels are built for
constexpr int PL_NLV = 128;         // levels a layer may have
// Where planes and layers lose digits, they lose different ones, and the planes
// are not to move the results: what lost digits is done on the layers.
// Leads: steps whose cell is nearly singular at E lose digits that the later
// steps do not bring back, on planes and on layers alike (planes about a third
// of what the layers lose, against an 80-bit recursion).  The self-energy's own
// equation shows the loss: the recursion adds up es = e + Sigma, and Sigma = V^+
// (z - es)^-1 V.  Where the residual, over Sigma's largest element, passes the
// bound, the layers' self-energy takes its place.  Films of 192, 20 times 1024
// points, largest differences of planes and layers by residual: T 7e-7 up to
// 3e-7, 2e-6 up to 1e-6, 1e-5 beyond (2 points); the gradient of a point, over
// its norm, 2e-7 up to 3e-8, 2e-6 up to 3e-7, 1e-5 up to 1e-6, 7e-5 beyond.  The
// leads of a few points of 192 take 30 ms on the layers (80: 13), whence not
// less: 0.1 of 1024 points are beyond the bound of T, one beyond the gradient's.
constexpr double PL_RESIDUAL = 1.0e-6, PL_RESIDUAL_ADJ = 1.0e-7;
// A loss beyond the broadening may make the recursion grow without end instead:
// of 360,000 energies of ribbons at eta = 1e-8 eV the layers' did at 47 where the
// planes' did not, all with residuals of 2 eta / scale and more, 46 of 5 and
// more; of 740,000 frequencies of films, 117 with more than eta / scale, none
// did.  Whether a recursion ends is decided on the layers from the bound
// PL_RESIDUAL_ETA eta / scale on (0.1 of 1024 points of the film), from eta / scale
// itself where that is less than PL_SMALL_ETA: the electrons' calls have such
// leads anyway (31 of 2048 points of the ribbon), and a few more take no longer.
constexpr double PL_RESIDUAL_ETA = 5.0, PL_SMALL_ETA = 1.0e-8;
// Planes inside a lead cell and of the device are eliminated with pivots from
// one plane only, and a plane may be nearly singular at E where its layer is
// not.  With kappa = |G|max scale of the eliminated planes, G between the leads
// then is off by 1e-16 to 5e-16 kappa (where all layers have such planes at one
// energy up to ten times that): layers of 13 + 14 + 13 degrees of freedom,
// the middle ones uncoupled sites at E, eta = 1e-8: kappa 3e7, error of T 3e-8
// (on layers 3e-11), at kappa 2e5 3e-10.  T changes by 2 sqrt(T) times as much,
// and by no less than its square: what is bounded is kappa sqrt(T), with T from
// this floor (kappa <= 1e9: 1e-13) to 1, in a gradient, which is of first order
// in G, from 0.01.  Films reach 1.2e5 (40,000 points), the wire 2e5, the ribbon
// 1.5e5 and, in its gap, 2e6; a point on layers of 192 takes 100 ms.
constexpr double PL_T_FLOOR = 1.0e-8, PL_T_FLOOR_ADJ = 0.01;
constexpr double PL_KAPPA = 3.0e5;

// need[p]: 0 solved on the planes, else why it is not (yet)
enum { NEED_LAYERS = 1, NEED_AFTER_SWEEP = 2, NEED_LEADS = 3 };
// counters of a solve (device ints; the first three of a chunk)
enum { CNT_LAYERS = 0, CNT_AFTER_SWEEP = 1, CNT_LEADS = 2, CNT_STEPS = 3, CNT_SAME = 4, CNT_N = 5 };

// ------------------------------------------------------------------ the plan
// Device arrays of the plan (ints), carved from one buffer.
struct PlanView {
    PlanHdr* h;
    unsigned* adj;      // (layer, dof) rows of adjacency bits, W words each
    unsigned* cbits;    // (layer) W words: dofs coupled to the previous layer
    unsigned* rbits;    // (layer) W words: dofs coupled to the next layer
    int* bad;           // leads not Hermitian
    int* level;         // (layer, dof)
    int* nlev;          // (layer)
    int* cnt;           // (layer, PL_NLV) dofs per level
    int* npl;           // (layer, PL_NCLS) planes per class, -1: a level does not fit
    int* poff;          // (layer + 1) first plane
    int* psize;         // (plane)
    int* player;        // (plane) layer
    int* perm;          // (plane, PL_PERM) dof of the layer at each place
};

// sizes a plan depends on
struct PlanDims {
    int nl, nr, b, L, nk;
    int nmax, W, Mcap;
};

PlanDims plan_dims(int nl, int nr, int b, int L, int nk)
{
    PlanDims d{nl, nr, b, L, nk, 0, 0, 0};
    d.nmax = std::max(b, std::max(nl, nr));
    d.W = (d.nmax + 31) / 32;
    // two neighbouring planes of a layer hold more than 16 dofs together
    d.Mcap = (2 * (nl / 16) + 2) + (2 * (nr / 16) + 2) + L * (2 * (b / 16) + 2);
    return d;
}

PlanView plan_carve(Arena& a, const PlanDims& d)
{
    const size_t nL = d.L + 2, i4 = sizeof(int);
    PlanView v;
    // zeroed region first: header, bits, flags
    const size_t oh = a.take(sizeof(PlanHdr)), oa = a.take(i4 * nL * d.nmax * d.W), oc = a.take(i4 * nL * d.W),
                 orr = a.take(i4 * nL * d.W), ob = a.take(i4);
    const size_t ol = a.take(i4 * nL * d.nmax), on = a.take(i4 * nL), oq = a.take(i4 * nL * PL_NLV),
                 op = a.take(i4 * nL * PL_NCLS), oo = a.take(i4 * (nL + 1)), os = a.take(i4 * d.Mcap),
                 oy = a.take(i4 * d.Mcap), om = a.take(i4 * (size_t)d.Mcap * PL_PERM);
    v.h = a.ptr<PlanHdr>(oh);
    v.adj = a.ptr<unsigned>(oa);
    v.cbits = a.ptr<unsigned>(oc);
    v.rbits = a.ptr<unsigned>(orr);
    v.bad = a.ptr<int>(ob);
    v.level = a.ptr<int>(ol);
    v.nlev = a.ptr<int>(on);
    v.cnt = a.ptr<int>(oq);
    v.npl = a.ptr<int>(op);
    v.poff = a.ptr<int>(oo);
    v.psize = a.ptr<int>(os);
    v.player = a.ptr<int>(oy);
    v.perm = a.ptr<int>(om);
    return v;
}

// the caller's blocks
struct BlocksIn {
    const C2 *Haml, *Hamlv, *Hamr, *Hamrv, *Hamd, *Hamdv, *Hamld, *Hamrd;
};

__device__ __forceinline__ int layer_size(const PlanDims& d, int layer)
{
    return layer == 0 ? d.nl : layer == d.L + 1 ? d.nr : d.b;
}

// diagonal block of a layer at k-point k (ld = its size)
__device__ __forceinline__ const C2* layer_H(const PlanDims& d, const BlocksIn& B, int layer, int k)
{
    if (layer == 0) return B.Haml + (long)k * d.nl * d.nl;
    if (layer == d.L + 1) return B.Hamr + (long)k * d.nr * d.nr;
    return B.Hamd + ((long)k * d.L + layer - 1) * d.b * d.b;
}

__device__ __forceinline__ void set_bit(unsigned* w, int i)
{
    const unsigned m = 1u << (i & 31);
    if (!(w[i >> 5] & m)) atomicOr(&w[i >> 5], m);
}

// blockIdx.y: the L + 2 diagonal blocks, then the couplings lead-lead (left),
// lead-device, device-device, device-lead, lead-lead (right); blockIdx.z: k
__global__ void k_pl_pattern(PlanDims d, PlanView v, BlocksIn B, int k0)
{
    // (more k-points only add nonzeros: a plan refused stays refused)
    if (k0 && !v.h->ok) return;
    const int k = k0 + blockIdx.z, nL = d.L + 2;
    const long step = (long)gridDim.x * blockDim.x, e0 = (long)blockIdx.x * blockDim.x + threadIdx.x;
    int m = blockIdx.y;
    if (m < nL) {
        const int n = layer_size(d, m);
        const C2* H = layer_H(d, B, m, k);
        unsigned* adj = v.adj + (long)m * d.nmax * d.W;
        const bool lead = m == 0 || m == nL - 1;
        for (long e = e0; e < (long)n * n; e += step) {
            const int r = (int)(e % n), c = (int)(e / n);
            const C2 x = H[e];
            if (!(x.x == 0.0 && x.y == 0.0) && r != c) {
                set_bit(adj + (long)r * d.W, c);
                set_bit(adj + (long)c * d.W, r);
            }
            if (lead && r <= c) {
                // the left lead is decimated at E - i eta and daggered: only
                // for a Hermitian lead is that its retarded function
                const C2 y = H[c + (long)r * n], hr = H[r + (long)r * n], hc = H[c + (long)c * n];
                const double df = fabs(x.x - y.x) + fabs(x.y + y.y);
                const double off = fabs(x.x) + fabs(x.y), dg = fabs(hr.x) + fabs(hc.x);
                if (df > 1e-10 * off && df > 1e-13 * dg) *v.bad = 1;
            }
        }
        return;
    }
    m -= nL;
    const C2* V;
    int rows, cols;
    unsigned *rb, *cb;
    auto R = [&](int layer) { return v.rbits + (long)layer * d.W; };
    auto Cc = [&](int layer) { return v.cbits + (long)layer * d.W; };
    if (m == 0) {                    // V_{-1,0}: rows face the device, columns the lead
        V = B.Hamlv + (long)k * d.nl * d.nl, rows = cols = d.nl, rb = R(0), cb = Cc(0);
    } else if (m == 1) {             // V_{0,1}
        V = B.Hamld + (long)k * d.nl * d.b, rows = d.nl, cols = d.b, rb = R(0), cb = Cc(1);
    } else if (m <= d.L) {           // V_{i,i+1}
        V = B.Hamdv + ((long)k * (d.L > 1 ? d.L - 1 : 1) + m - 2) * d.b * d.b, rows = cols = d.b, rb = R(m - 1),
        cb = Cc(m);
    } else if (m == d.L + 1) {       // V_{N+1,N}
        V = B.Hamrd + (long)k * d.nr * d.b, rows = d.nr, cols = d.b, rb = Cc(d.L + 1), cb = R(d.L);
    } else {                         // V_{N+2,N+1}: rows face the device, columns the lead
        V = B.Hamrv + (long)k * d.nr * d.nr, rows = cols = d.nr, rb = Cc(d.L + 1), cb = R(d.L + 1);
    }
    for (long e = e0; e < (long)rows * cols; e += step) {
        const C2 x = V[e];
        if (!(x.x == 0.0 && x.y == 0.0)) {
            set_bit(rb, (int)(e % rows));
            set_bit(cb, (int)(e / rows));
        }
    }
}

// whether a level begins a plane: it does not fit into the one before, or it
// is the last of a lead cell that has one plane so far (the decimation works
// on a cell's first and last plane)
__device__ __forceinline__ bool plane_starts(bool full, bool lead, bool last, int planes)
{
    return full || (lead && last && planes == 1);
}

// One workgroup per layer: level of every dof = distance from the dofs that
// face the previous layer; everything from the first dof that faces the next
// layer on is one level (the next layer couples to the last plane only).
__global__ __launch_bounds__(256) void k_pl_levels(PlanDims d, PlanView v)
{
    const int layer = blockIdx.x, n = layer_size(d, layer), t = threadIdx.x;
    const unsigned* adj = v.adj + (long)layer * d.nmax * d.W;
    const unsigned* cb = v.cbits + (long)layer * d.W;
    const unsigned* rb = v.rbits + (long)layer * d.W;
    __shared__ short lev[1024];
    __shared__ unsigned front[32];
    __shared__ int found, last, cnt[PL_NLV];
    for (int i = t; i < n; i += 256) lev[i] = (cb[i >> 5] >> (i & 31)) & 1 ? 0 : -1;
    if (t < PL_NLV) cnt[t] = 0;
    if (t == 0) last = PL_NLV - 1;
    int lv = 0;
    for (; lv < PL_NLV - 1; ++lv) {
        if (t < 32) front[t] = 0;
        if (t == 0) found = 0;
        __syncthreads();
        for (int i = t; i < n; i += 256)
            if (lev[i] == lv) atomicOr(&front[i >> 5], 1u << (i & 31));
        __syncthreads();
        for (int i = t; i < n; i += 256) {
            if (lev[i] >= 0) continue;
            unsigned hit = 0;
            for (int w = 0; w < d.W; ++w) hit |= adj[(long)i * d.W + w] & front[w];
            if (hit) {
                lev[i] = (short)(lv + 1);
                found = 1;
            }
        }
        __syncthreads();
        const int f = found;
        __syncthreads();
        if (!f) break;
    }
    for (int i = t; i < n; i += 256)
        if (((rb[i >> 5] >> (i & 31)) & 1) && lev[i] >= 0) atomicMin(&last, (int)lev[i]);
    __syncthreads();
    const int m = min(last, lv);
    for (int i = t; i < n; i += 256) {
        const int l = lev[i] < 0 || lev[i] > m ? m : lev[i];
        v.level[(long)layer * d.nmax + i] = l;
        atomicAdd(&cnt[l], 1);
    }
    __syncthreads();
    if (t < PL_NLV) v.cnt[(long)layer * PL_NLV + t] = cnt[t];
    if (t == 0) v.nlev[layer] = m + 1;
    if (t < PL_NCLS) {
        // planes of at most the class's size: consecutive levels merged while they
        // fit (plane_starts); a lead cell keeps two at least
        const int lim = 16 * class_nt(t);
        const bool lead = layer == 0 || layer == d.L + 1;
        int planes = 0, fill = lim + 1;
        for (int l = 0; l <= m; ++l) {
            const int k = cnt[l];
            if (k > lim) {
                planes = -1;
                break;
            }
            if (plane_starts(fill + k > lim, lead, l == m, planes)) {
                ++planes;
                fill = k;
            } else {
                fill += k;
            }
        }
        v.npl[layer * PL_NCLS + t] = planes;
    }
}

// One workgroup: wave t sums the planes of class t, the cheapest of the first
// ncls classes wins: per plane about five products of the class size and as
// many pivots as it has columns (5120 SIMD cycles per 16^3 of products and
// 12000 per 16 pivots, of the inverse's 53 us at 64 and the products' rate).
__global__ __launch_bounds__(64 * PL_NCLS) void k_pl_plan(PlanDims d, PlanView v, int ncls)
{
    const int nL = d.L + 2, w = threadIdx.x >> 6, lane = threadIdx.x & 63;
    __shared__ int tot[PL_NCLS];
    __shared__ int pick;
    int s = 0, bad = 0;
    for (int i = lane; i < nL; i += 64) {
        const int p = v.npl[i * PL_NCLS + w];
        bad |= p < 0;
        s += p;
    }
    for (int o = 32; o; o >>= 1) {
        s += __shfl_xor(s, o);
        bad |= __shfl_xor(bad, o);
    }
    if (lane == 0) tot[w] = bad ? -1 : s;
    __syncthreads();
    if (threadIdx.x == 0) {
        double best = 0.0;
        int cl = -1;
        for (int t = 0; t < ncls; ++t) {
            if (tot[t] < 0) continue;
            const double u = class_nt(t), c = tot[t] * (5120.0 * u * u * u + 12000.0 * u);
            if (cl < 0 || c < best) {
                best = c;
                cl = t;
            }
        }
        pick = cl;
        const int M = cl < 0 ? 0 : tot[cl], m0 = cl < 0 ? 0 : v.npl[cl], m1 = cl < 0 ? 0 : v.npl[(nL - 1) * PL_NCLS + cl];
        v.h->nt = cl < 0 ? 0 : class_nt(cl);
        v.h->M = M;
        v.h->m0 = m0;
        v.h->m1 = m1;
        // one plane per layer: nothing is gained over the layers themselves; a
        // lead cell of one plane: not written for that; the large class's
        // leads: both cells of two to four planes
        v.h->ok = cl >= 0 && !*v.bad && M <= d.Mcap && M > nL && m0 > 1 && m1 > 1 &&
                  (cl < PL_MAXNT || (m0 == m1 && m0 <= 4));
    }
    __syncthreads();
    const int cl = pick;
    if (cl < 0 || w) return;
    int base = 0;
    for (int i0 = 0; i0 < nL; i0 += 64) {
        const int i = i0 + lane;
        int x = i < nL ? v.npl[i * PL_NCLS + cl] : 0, inc = x;
        for (int o = 1; o < 64; o <<= 1) {
            const int y = __shfl_up(inc, o);
            if (lane >= o) inc += y;
        }
        if (i < nL) v.poff[i] = base + inc - x;
        base += __shfl(inc, 63);
    }
    if (lane == 0) v.poff[nL] = base;
}

// One workgroup per layer: plane and place of every dof (in dof order)
__global__ __launch_bounds__(256) void k_pl_perm(PlanDims d, PlanView v)
{
    if (!v.h->ok) return;
    const int layer = blockIdx.x, n = layer_size(d, layer), t = threadIdx.x;
    const int lim = 16 * v.h->nt, p0 = v.poff[layer], np = v.poff[layer + 1] - p0;
    __shared__ short pl[1024];
    __shared__ short of_level[PL_NLV];
    if (t == 0) {
        const int nlev = v.nlev[layer];
        int p = -1, fill = lim + 1;
        for (int l = 0; l < nlev; ++l) {
            const int k = v.cnt[(long)layer * PL_NLV + l];
            if (plane_starts(fill + k > lim, layer == 0 || layer == d.L + 1, l == nlev - 1, p + 1)) {
                ++p;
                fill = k;
            } else {
                fill += k;
            }
            of_level[l] = (short)p;
        }
    }
    __syncthreads();
    for (int i = t; i < n; i += 256) pl[i] = of_level[v.level[(long)layer * d.nmax + i]];
    __syncthreads();
    for (int i = t; i < n; i += 256) {
        int pos = 0;
        for (int j = 0; j < i; ++j) pos += pl[j] == pl[i];
        v.perm[(long)(p0 + pl[i]) * PL_PERM + pos] = i;
    }
    for (int p = t; p < np; p += 256) {
        int c = 0;
        for (int j = 0; j < n; ++j) c += pl[j] == p;
        v.psize[p0 + p] = c;
        v.player[p0 + p] = layer;
    }
}

// blockIdx.x: plane, blockIdx.y: k, blockIdx.z: 0 diagonal block, 1 coupling
// to the next plane, 2 coupling from it (and the two's masks), 3 the leads' cell coupling (planes 0
// and M - 1 only)
__global__ __launch_bounds__(256) void k_pl_pack(PlanDims d, PlanView v, BlocksIn B, C2* H, C2* U, C2* Lw, C2* LV,
                                                 unsigned long long* masks)
{
    const PlanHdr& h = *v.h;
    const int pl = blockIdx.x, k = blockIdx.y, what = blockIdx.z, M = h.M;
    if (!h.ok || pl >= M) return;
    const int NP = 16 * h.nt, NN = NP * NP;
    const int la = v.player[pl], na = layer_size(d, la), sa = v.psize[pl];
    const int* pa = v.perm + (long)pl * PL_PERM;
    if (what == 3) {
        if (pl != 0 && pl != M - 1) return;
        // V from the plane that faces the device (rows) to the one that faces
        // the lead (columns) of the next cell
        const int side = pl != 0;
        const int fb = side ? M - h.m1 : h.m0 - 1;        // plane facing the device
        const int* pb = v.perm + (long)fb * PL_PERM;
        const int sb = v.psize[fb];
        const C2* V = side ? B.Hamrv + (long)k * na * na : B.Hamlv + (long)k * na * na;
        C2* o = LV + ((long)k * 2 + side) * NN;
        for (int e = threadIdx.x; e < NN; e += 256) {
            const int r = e % NP, c = e / NP;
            C2 x = make_double2(0.0, 0.0);
            if (r < sb && c < sa) x = V[pb[r] + (long)pa[c] * na];
            o[e] = x;
        }
        return;
    }
    C2* o = (what == 0 ? H : what == 1 ? U : Lw) + ((long)k * M + pl) * NN;
    if (what == 0) {
        const C2* S = layer_H(d, B, la, k);
        for (int e = threadIdx.x; e < NN; e += 256) {
            const int r = e % NP, c = e / NP;
            C2 x = make_double2(0.0, 0.0);
            if (r < sa && c < sa) x = S[pa[r] + (long)pa[c] * na];
            o[e] = x;
        }
        return;
    }
    if (pl + 1 >= M) return;
    const int lb = v.player[pl + 1], nb = layer_size(d, lb), sb = v.psize[pl + 1];
    const int* pb = v.perm + (long)(pl + 1) * PL_PERM;
    // U (rows of this plane, columns of the next), Lw (rows of the next)
    const C2* S = nullptr;
    int ld = 0;
    bool dag = false;              // element (r, c) is conj(S[c, r])
    if (la == lb) {
        S = layer_H(d, B, la, k);
        ld = na;
    } else if (lb == d.L + 1) {    // V_{N,N+1} = V_{N+1,N}^+
        S = B.Hamrd + (long)k * d.nr * d.b;
        ld = d.nr;
        dag = what == 1;
    } else {
        S = la == 0 ? B.Hamld + (long)k * d.nl * d.b
                    : B.Hamdv + ((long)k * (d.L > 1 ? d.L - 1 : 1) + la - 1) * d.b * d.b;
        ld = na;
        dag = what == 2;
    }
    // which of its 4 x 16 and 16 x 4 pieces are not zero (blk_mul's masks)
    __shared__ unsigned long long piece[2];
    if (threadIdx.x < 2) piece[threadIdx.x] = 0;
    __syncthreads();
    const int* pr = what == 1 ? pa : pb;
    const int* pc = what == 1 ? pb : pa;
    const int sr = what == 1 ? sa : sb, sc = what == 1 ? sb : sa;
    for (int e = threadIdx.x; e < NN; e += 256) {
        const int r = e % NP, c = e / NP;
        C2 x = make_double2(0.0, 0.0);
        if (r < sr && c < sc) {
            if (dag) {
                x = S[pc[c] + (long)pr[r] * ld];
                x.y = -x.y;
            } else {
                x = S[pr[r] + (long)pc[c] * ld];
            }
        }
        o[e] = x;
        if (h.nt <= PL_MAXNT && !(x.x == 0.0 && x.y == 0.0)) {
            atomicOr(&piece[0], 1ull << (h.nt * (r / 4) + c / 16));
            atomicOr(&piece[1], 1ull << (h.nt * (c / 4) + r / 16));
        }
    }
    __syncthreads();
    if (threadIdx.x < 2) masks[(((long)k * M + pl) * 2 + (what - 1)) * 2 + threadIdx.x] = piece[threadIdx.x];
}

// ------------------------------------------------------------- LDS of a workgroup
// One region holds either an inverse (column-major, ld = NP + 1: rows and
// columns both read without bank conflicts) or, while a matrix is being
// inverted in registers, two panels and one pivot-row buffer per wave.
template <int NT>
struct PlSmem {
    static constexpr int NP = 16 * NT, LD = NP + 1;
    static constexpr int MAT = NP * LD, WORK = 2 * 16 * LD + NT * 256;
    C2 g[MAT > WORK ? MAT : WORK];
    int piv[NP], cinv[NP], info;
    double red[NT];
};

// m = z - m on the n x n block, the identity on the padding
template <int NT>
__device__ __forceinline__ void blk_shift(Blk<NT>& m, double zr, double zi, int n, int w)
{
    const int lane = lane_new(), q = lane >> 4, col = 16 * w + (lane & 15);
#pragma unroll
    for (int t = 0; t < NT; ++t)
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            const int row = 16 * t + 4 * r + q;
            const bool in = row < n && col < n, dg = row == col;
            m.re[t][r] = in ? (dg ? zr : 0.0) - m.re[t][r] : (dg ? 1.0 : 0.0);
            m.im[t][r] = in ? (dg ? zi : 0.0) - m.im[t][r] : 0.0;
        }
}

// ------------------------------------------------------------------ decimation
// Lopez-Sancho decimation (negf/surface.f90:479-497) of a lead cell whose
// couplings run from its plane B (facing the device) to plane A of the next
// cell: alpha = V^+ lives on A x B, beta = V on B x A, so of
//   e += alpha g beta + beta g alpha, es += alpha g beta,
//   alpha' = alpha g alpha, beta' = beta g beta
// only the A and B blocks of e and g enter.  The planes between A and B are
// eliminated once per point, two at a time; every step then inverts the cell
// of two planes as one matrix, with pivots from both (inverting the planes one
// after the other takes as many operations but lost 10 to 50 times the digits:
// 1.8e-8 against 3.2e-10 at the 99th percentile of the ribbon's energies, the
// full cell's inverse 2.7e-10).  The elements of alpha are the ones of the
// full recursion, so the count of steps to max|alpha| <= convergence is too.
// 2 NT waves: the first NT own the columns of A, the others those of B.
// Bound by the inverse's pivot chain; from NT = 3 on one workgroup has a CU to
// itself, and its waves' registers spill.  2048 leads of a film of 192 (four
// planes of 48): 29.8 ms.
constexpr int DEC_SLOTS = 19;       // matrices of NP^2 per item

template <int NT>
struct DecSmem {
    static constexpr int NP2 = 32 * NT;
    C2 work[2 * 16 * (NP2 + 1) + 2 * NT * 256];
    int piv[NP2], cinv[NP2], info;
    double red[2 * NT];
};

template <int NT>
__global__ __launch_bounds__(128 * NT, PL_WAVES) void k_pl_decimate(DecPlArgs a)
{
    constexpr int NP = 16 * NT, NN = NP * NP, NP2 = 2 * NP;
    const PlanHdr& h = *a.h;
    if (!h.ok || h.nt != NT) return;
    __shared__ DecSmem<NT> s;
    const InvLds il{s.piv, s.cinv, &s.info, 1.0e300};
    const int item = blockIdx.x, p = item >> 1, side = item & 1;
    const int w = wave_id(), half = w >= NT, wc = half ? w - NT : w;
    const int l15 = lane_id() & 15, q = lane_id() >> 4;
    const int k = a.kidx ? a.kidx[p] : 0, M = h.M, mc = side ? h.m1 : h.m0;
    const double E = a.E[p], et = a.eta_mode == NT_ETA_RELATIVE ? E * a.eta + a.eta0 : a.eta;
    const double zr = E, zi = side ? et : -et;
    // plane j of the cell counted from A; couplings j -> j + 1 and back
    auto plane = [&](int j) { return side ? M - 1 - j : j; };
    const C2* Hk = a.H + (long)k * M * NN;
    const C2* Uk = a.U + (long)k * M * NN;
    const C2* Lk = a.Lw + (long)k * M * NN;
    auto Hp = [&](int j) { return Hk + (long)plane(j) * NN; };
    auto Fp = [&](int j) { return side ? Lk + (long)(M - 2 - j) * NN : Uk + (long)j * NN; };
    auto Bp = [&](int j) { return side ? Uk + (long)(M - 2 - j) * NN : Lk + (long)j * NN; };
    const C2* V = a.LV + ((long)k * 2 + side) * NN;       // rows B, columns A
    C2* sc = a.scratch + (long)item * DEC_SLOTS * NN;
    auto slot = [&](int i) { return sc + (long)i * NN; };
    C2 *eA = slot(0), *eB = slot(1), *esA = slot(2), *eB0 = slot(3), *al = slot(4), *be = slot(5), *aln = slot(6),
       *ben = slot(7), *cf = slot(8), *cb = slot(9), *cfn = slot(10);
    C2 *T1 = slot(11), *T2 = slot(13), *G = slot(15);     // NP x 2 NP twice, 2 NP square
    C2* cbn = T1;                                         // (before the steps)
    if (threadIdx.x == 0) s.info = 0;
    double mid = 0.0;              // |G|max of the planes inside the cell, the wave's columns
    Blk<NT> x, y;
    auto load = [&](Blk<NT>& b, const C2* m) __attribute__((always_inline)) { blk_load<NT>(b, LdN{m, NP}, wc); };
    auto store = [&](const Blk<NT>& b, C2* m) __attribute__((always_inline)) { blk_store<NT>(b, m, NP, wc); };
    auto copy = [&](C2* to, const C2* from) __attribute__((always_inline)) {
        load(x, from);
        store(x, to);
    };
    int it = 0, j = 1, mode = mc > 2 ? 0 : 1;
    // G = (z - [[a, b], [c, d]])^-1 of planes of n1 and n2; no second plane
    // where n2 = 0.  Wave w holds column 16 w + lane % 16 of the 2 NP.
    auto invert = [&](const C2* ma, const C2* mb, const C2* mcc, const C2* md, int n1, int n2) __attribute__((always_inline)) {
        Blk<2 * NT> m;
        {
            Blk<NT> u, v;
            load(u, half ? mb : ma);
            load(v, half ? md : mcc);
#pragma unroll
            for (int t = 0; t < NT; ++t) m.re[t] = u.re[t], m.im[t] = u.im[t], m.re[NT + t] = v.re[t], m.im[NT + t] = v.im[t];
        }
        const int lane = lane_new(), q = lane >> 4, c0 = 16 * wc + (lane & 15);
        const bool cin = c0 < (half ? n2 : n1);
#pragma unroll
        for (int t = 0; t < 2 * NT; ++t)
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                const int r0 = 16 * (t % NT) + 4 * r + q;
                const bool in = cin && r0 < (t < NT ? n1 : n2), dg = (t >= NT) == (half != 0) && r0 == c0;
                m.re[t][r] = in ? (dg ? zr : 0.0) - m.re[t][r] : (dg ? 1.0 : 0.0);
                m.im[t][r] = in ? (dg ? zi : 0.0) - m.im[t][r] : 0.0;
            }
        __syncthreads();
        wg_inverse<2 * NT>(s.work, il, m, [&](int i, int j, C2 v) {
            G[i + j * NP2] = v;
            auto in = [&](int r) { return r < NP ? r < n1 : r - NP < n2; };
            if (mode == 0 && in(i) && in(j)) mid = fmax(mid, fabs(v.x) + fabs(v.y));
        });
    };
    const C2 *G11 = G, *G21 = G + NP, *G12 = G + (long)NP * NP2, *G22 = G + NP + (long)NP * NP2;
    const int nA = a.psize[plane(0)], nB = a.psize[plane(mc - 1)];
    // alpha0 = V^+, beta0 = V
    blk_load<NT>(x, LdC{V, NP}, wc);
    store(x, al);
    double amax = blk_maxabs<NT>(x);
    copy(be, V);
    copy(eA, Hp(0));
    double scale = fmax(amax, blk_maxabs<NT>(x));
    copy(cf, Fp(0));
    copy(cb, Bp(0));
    copy(eB, Hp(1));
    __syncthreads();
    // One inverse per pass: the elimination of planes j (and j + 1) between A
    // and B (cf = A -> j, cb = j -> A) while there are any, then the steps,
    // then the last one with es (one copy of the inverse's code, and the
    // registers of one).
    auto steps_begin = [&]() __attribute__((always_inline)) {
        if (cbn != T1) {              // T1's slot is needed by the steps
            copy(cbn, cb);
            cb = cbn;
        }
        copy(eB0, eB);
        copy(esA, eA);
        copy(cfn, eA);                // (a free slot from here on)
        if (mc > 2) mid = wg_max<2 * NT>(s.red, mid);
        amax = wg_max<2 * NT>(s.red, half ? 0.0 : amax);      // its barriers also publish the slots
    };
    if (mode) steps_begin();
    for (;;) {
        if (mode == 1 && !(it < a.max_iter && amax > a.conv && s.info == 0)) mode = 2;
        const bool two = j + 2 < mc;
        const C2 *ma = mode == 0 ? eB : mode == 1 ? eA : esA, *mb = mode ? cf : two ? Fp(j) : eB,
                 *mcc = mode ? cb : two ? Bp(j) : eB, *md = mode == 0 ? (two ? Hp(j + 1) : eB) : mode == 1 ? eB : eB0;
        const int n1 = mode ? nA : a.psize[plane(j)], n2 = mode ? nB : two ? a.psize[plane(j + 1)] : 0;
        invert(ma, mb, mcc, md, n1, n2);
        if (mode == 2) break;
        if (mode == 0) {
            const int o = two ? j + 1 : j;
            // half 0, through A:  e_AA += cf (g cb),  cb' = B_o (g cb)
            // half 1, onward:     cf' = cf (g F_o),   e = H_{o + 1} + B_o (g F_o)
            Blk<NT> u;
            load(x, half ? Fp(o) : cb);
            blk_zero<NT>(y);
            blk_mul<NT>(y, LdN{half && two ? G12 : G11, NP2}, x);
            if (half) blk_zero<NT>(u);
            else load(u, eA);
            blk_mul<NT>(u, LdN{cf, NP}, y);
            store(u, half ? cfn : eA);
            blk_zero<NT>(y);
            blk_mul<NT>(y, LdN{two ? (half ? G22 : G21) : G11, NP2}, x);
            if (half) load(u, Hp(o + 1));
            else blk_zero<NT>(u);
            blk_mul<NT>(u, LdN{Bp(o), NP}, y);
            store(u, half ? eB : cbn);
            C2* v = cf;
            cf = cfn;
            cfn = v;
            v = cb;
            cb = cbn;
            cbn = v;
            __syncthreads();
            j = o + 1;
            if (j + 1 >= mc) {
                mode = 1;
                steps_begin();
            }
            continue;
        }
        // T1 = alpha [g_BA, g_BB], T2 = beta [g_AA, g_AB]
        blk_load<NT>(x, LdN{G21, NP2}, w);
        blk_zero<NT>(y);
        blk_mul<NT>(y, LdN{al, NP}, x);
        blk_store<NT>(y, T1, NP, w);
        blk_load<NT>(x, LdN{G11, NP2}, w);
        blk_zero<NT>(y);
        blk_mul<NT>(y, LdN{be, NP}, x);
        blk_store<NT>(y, T2, NP, w);
        __syncthreads();
        // half 0: alpha g_BB beta to es and e_AA, alpha' = alpha g_BA alpha
        // half 1: beta g_AA alpha to e_BB, beta' = beta g_AB beta
        load(x, half ? al : be);
        blk_zero<NT>(y);
        blk_mul<NT>(y, LdN{half ? T2 : T1 + (long)NN, NP}, x);
        if (!half) {
            load(x, esA);
#pragma unroll
            for (int t = 0; t < NT; ++t) x.re[t] += y.re[t], x.im[t] += y.im[t];
            store(x, esA);
        }
        load(x, half ? eB : eA);
#pragma unroll
        for (int t = 0; t < NT; ++t) x.re[t] += y.re[t], x.im[t] += y.im[t];
        store(x, half ? eB : eA);
        load(x, half ? be : al);
        blk_zero<NT>(y);
        blk_mul<NT>(y, LdN{half ? T2 + (long)NN : T1, NP}, x);
        store(y, half ? ben : aln);
        C2* sw = al;
        al = aln;
        aln = sw;
        sw = be;
        be = ben;
        ben = sw;
        ++it;
        amax = wg_max<2 * NT>(s.red, half ? 0.0 : blk_maxabs<NT>(y));
    }
    const int not_conv = amax > a.conv;
    // Sigma = V^+ g_BB V on A with g = (z - es)^-1, and its difference to what
    // the steps added up
    double smax = 0.0, rmax = 0.0;
    if (!half) {
        load(x, V);
        blk_zero<NT>(y);
        blk_mul<NT>(y, LdN{G22, NP2}, x);
        blk_zero<NT>(x);
        blk_mul<NT>(x, LdC{V, NP}, y);
        C2* out = a.sigma + (long)item * NN;
        smax = blk_maxabs<NT>(x);
        load(y, cfn);
#pragma unroll
        for (int t = 0; t < NT; ++t) y.re[t] += x.re[t], y.im[t] += x.im[t];
        {
            Blk<NT> u;
            load(u, esA);
#pragma unroll
            for (int t = 0; t < NT; ++t) y.re[t] -= u.re[t], y.im[t] -= u.im[t];
        }
        rmax = blk_maxabs<NT>(y);
        if (side) {
            store(x, out);
        } else {
            // retarded = adjoint of the advanced
#pragma unroll
            for (int t = 0; t < NT; ++t)
#pragma unroll
                for (int r = 0; r < 4; ++r)
                    out[16 * wc + l15 + (16 * t + 4 * r + q) * NP] = make_double2(x.re[t][r], -x.im[t][r]);
        }
    }
    smax = wg_max<2 * NT>(s.red, smax);
    rmax = wg_max<2 * NT>(s.red, rmax);
    scale = fmax(wg_max<2 * NT>(s.red, scale), fabs(E));
    if (threadIdx.x == 0) {
        a.iters[item] = it;
        a.status[item] = s.info ? s.info : not_conv ? NT_ERR_NOT_CONVERGED : 0;
        // (a Sigma that is not finite: no number)
        a.loss[item] = LeadLoss{mid * scale, rmax == 0.0 ? 0.0 : rmax / smax, scale};
    }
}

// ----------------------------------------------------------------------- sweep
// One direction of one point: system 0 left to right (left lead planes at the
// lead's broadening, everything else at the device's), system 1 right to left
// (the roles swapped), negf/lesser.f90:556-793 on the planes.  Step i:
//   A = z_i - H_i - L X,  X = G U            (U, L: couplings to and from step i)
//   G = A^-1                                  in LDS
//   R = G_{first,i}^T = G^T (U^T R)           in registers
// and at the end T = Re Tr[(R^T Gamma_e)(R^* Gamma_s)].
// Bound by the pivot chains of the inverses (other workgroups fill the CU
// meanwhile) and by L2 reads of H, U and L.  Both directions go through as
// points of one launch: the corner correction that saves the second one on
// layers costs inverses here as well.  The couplings' zero pieces (4 columns by
// 16 rows) are skipped by a mask, and up to 48 three waves per SIMD are built
// for: film of 168 planes of 48, 1024 points, 54.6 -> 43.9 ms from both, 38.3
// with the shorter pivot chain, 39.5 with the measure of the planes' inverses.  The whole solve of
// them: 748 ms on layers of 192, 71 on planes, 30 of them the decimation.
template <int NT>
__global__ __launch_bounds__(64 * NT, NT < 4 ? 3 : 2) void k_pl_sweep(SweepPlArgs a)
{
    constexpr int NP = 16 * NT, LD = NP + 1, NN = NP * NP;
    const PlanHdr& h = *a.h;
    if (!h.ok || h.nt != NT) return;
    __shared__ PlSmem<NT> s;
    const InvLds il{s.piv, s.cinv, &s.info, 1.0e300};
    const int item = blockIdx.x, p = item >> 1, sys = item & 1;
    const int w = wave_id();
    const int k = a.kidx ? a.kidx[p] : 0, M = h.M;
    const double E = a.E[p], et = a.eta_mode == NT_ETA_RELATIVE ? E * a.eta + a.eta0 : a.eta;
    if (a.need[p]) return;
    const int lead_planes = sys ? h.m1 : h.m0;
    const C2* Hk = a.H + (long)k * M * NN;
    const C2* Uk = a.U + (long)k * M * NN;
    const C2* Lk = a.Lw + (long)k * M * NN;
    // self-energies of the starting and of the closing lead
    const C2* Ss = a.sigma + (long)(2 * p + sys) * NN;
    const C2* Se = a.sigma + (long)(2 * p + 1 - sys) * NN;
    if (threadIdx.x == 0) s.info = 0;
    unsigned gmax = 0;             // upper word of |G|max, the wave's columns
    Blk<NT> R;
    blk_zero<NT>(R);
#pragma unroll 1
    for (int i = 0; i < M; ++i) {
        const int j = sys ? M - 1 - i : i;
        Blk<NT> m;
        blk_load<NT>(m, LdN{Hk + (long)j * NN, NP}, w);
        if (j == 0 || j == M - 1) {
            Blk<NT> sg;
            blk_load<NT>(sg, LdN{j || !a.left ? a.sigma + (long)(2 * p + (j != 0)) * NN : a.left + (long)p * NN, NP}, w);
#pragma unroll
            for (int t = 0; t < NT; ++t) m.re[t] += sg.re[t], m.im[t] += sg.im[t];
        }
        if (i) {
            const C2* U = sys ? Lk + (long)j * NN : Uk + (long)(j - 1) * NN;      // step i - 1 -> i
            const C2* Lo = sys ? Uk + (long)j * NN : Lk + (long)(j - 1) * NN;     // step i -> i - 1
            // masks of U's 4 x 16 pieces and of Lo's 16 x 4 pieces
            const unsigned long long* mk = a.masks + ((long)k * M + (sys ? j : j - 1)) * 4;
            const unsigned long long mu = mk[sys ? 2 : 0], ml = mk[sys ? 1 : 3];
            Blk<NT> t2;
            blk_zero<NT>(t2);
            // (a mask has room for the pieces of classes up to 64)
            blk_mul<NT, NT <= PL_MAXNT>(t2, LdT{U, NP}, R, mu);
            R = t2;
            blk_load<NT>(t2, LdN{U, NP}, w);
            Blk<NT> X;
            blk_zero<NT>(X);
            if constexpr (NT <= PL_MAXNT) blk_mul_rows<NT>(X, LsN{s.g, LD}, t2, mu >> w);
            else blk_mul<NT>(X, LsN{s.g, LD}, t2);
            blk_mul<NT, NT <= PL_MAXNT>(m, LdN{Lo, NP}, X, ml);
        }
        blk_shift<NT>(m, E, i < lead_planes ? et : a.dev_factor * et, a.psize[j], w);
        __syncthreads();
        double g = 0.0;
        const int n = a.psize[j];
        wg_inverse<NT>(s.g, il, m, [&](int r, int c, C2 v) {
            s.g[r + c * LD] = v;
            if (r < n && c < n) g = fmax(g, fabs(v.x) + fabs(v.y));
        });
        const unsigned gh = wave_max((unsigned)(__double_as_longlong(g) >> 32));
        gmax = gh > gmax ? gh : gmax;
        if (i) {
            Blk<NT> n;
            blk_zero<NT>(n);
            blk_mul<NT>(n, LsT{s.g, LD}, R);
            R = n;
        } else {
            blk_load<NT>(R, LsT{s.g, LD}, w);
        }
        if (a.keep && !sys && j >= *a.keep_from) {
            C2* kp = a.keep + (p * a.keep_stride + 2 * (j - *a.keep_from)) * NN;
            Blk<NT> g;
            blk_load<NT>(g, LsN{s.g, LD}, w);
            blk_store<NT>(g, kp, NP, w);
            blk_store<NT>(R, kp + NN, NP, w);
        }
    }
    // Y^T = Gamma_e^T R into LDS, Q = Y^T Gamma_s^T, T = Re sum conj(R) Q
    Blk<NT> y;
    blk_zero<NT>(y);
    blk_mul<NT>(y, LdGamT{Se, NP}, R);
    __syncthreads();
    blk_store<NT>(y, s.g, LD, w);
    Blk<NT> gs;
    blk_load<NT>(gs, LdGamT{Ss, NP}, w);
    __syncthreads();
    blk_zero<NT>(y);
    blk_mul<NT>(y, LsN{s.g, LD}, gs);
    double tr = 0.0;
#pragma unroll
    for (int t = 0; t < NT; ++t)
#pragma unroll
        for (int r = 0; r < 4; ++r) tr += R.re[t][r] * y.re[t][r] + R.im[t][r] * y.im[t][r];
#pragma unroll
    for (int o = 32; o; o >>= 1) tr += __shfl_xor(tr, o);
    __syncthreads();
    if (lane_id() == 0) s.red[w] = tr;
    __syncthreads();
    if (threadIdx.x == 0) {
        double t = 0.0;
        for (int i = 0; i < NT; ++i) t += s.red[i];
        a.T[item] = t;
        a.status[item] = s.info;
    }
    const double g = wg_max<NT>(s.red, __longlong_as_double((long long)gmax << 32));
    if (threadIdx.x == 0) a.grow[item] = g;
}

// --------------------------------------------------------------------- adjoint
// Column and row of the full Green's function on the window's planes, one
// workgroup per point, from the left-connected blocks the sweep kept:
//   C_j = G^L_j U_j C_{j+1},  R_j^T = (G^L_{0,j})^T + (G^L_j)^T L_j^T R_{j+1}^T
// from C_{M-1} = G_{M-1,M-1} A, A = w Gamma_R G_{0,M-1}^+ Gamma_L, so that
// X_{j,i} = C_j R_i (the block path's adjoint_backward).  No LDS and no
// barrier: every wave works on its own columns, all A operands are read from
// memory.  The window's blocks are written in the layers' own order, the rows
// of R of all points above one another and the columns of C beside one
// another: the sums over the points of X_{j,i}^+ = R_i^+ C_j^+ are then one
// product per layer and k-point, over 16 NT rows per point instead of a b x b
// block of each point summed afterwards.  Bound by L2 and HBM reads of the kept
// blocks.  Gradient of 512 points over 16 layers of 192, all of it: 465 ms on
// layers, 59 on planes: 43 forward, 10 the three products of the sums, 5 here.
template <int NT>
__global__ __launch_bounds__(64 * NT, PL_WAVES) void k_pl_adjoint(AdjPlArgs a)
{
    constexpr int NP = 16 * NT, NN = NP * NP;
    const PlanHdr& h = *a.h;
    if (!h.ok || h.nt != NT) return;
    const int p = blockIdx.x, w = wave_id(), M = h.M;
    const int k = a.kidx ? a.kidx[p] : 0;
    const C2* Uk = a.U + (long)k * M * NN;
    const C2* Lk = a.Lw + (long)k * M * NN;
    const int jw = a.poff[a.lo + 1], je = a.poff[a.hi1 + 2];       // the window's planes
    const C2* keep = a.keep + (long)p * a.keep_stride * NN;
    auto gl = [&](int j) { return keep + 2L * (j - jw) * NN; };
    auto g0 = [&](int j) { return keep + (2L * (j - jw) + 1) * NN; };
    const bool on = !a.need[p] && !a.status[2 * p] && !a.status[2 * p + 1] && !a.dstatus[2 * p] &&
                    !a.dstatus[2 * p + 1] && !(a.first && a.first[p]);
    const C2* Ss = a.sigma + (long)(2 * p) * NN;
    const C2* Se = Ss + NN;
    Blk<NT> C, R, y;
    blk_zero<NT>(C);
    blk_zero<NT>(R);
    if (on) {
        blk_load<NT>(y, LdGam{Ss, NP}, w);
        blk_mul<NT>(R, LdNc{g0(M - 1), NP}, y);
        blk_zero<NT>(y);
        blk_mul<NT>(y, LdGam{Se, NP}, R);
        const double f = a.w[p];
#pragma unroll
        for (int t = 0; t < NT; ++t) y.re[t] *= f, y.im[t] *= f;
        blk_mul<NT>(C, LdN{gl(M - 1), NP}, y);
        blk_load<NT>(R, LdN{g0(M - 1), NP}, w);
    }
    const int place = a.place ? a.place[p] : p;
    // rows of a point: its place among the points, NP each
#pragma unroll 1
    for (int j = M - 2; j >= jw; --j) {
        if (on) {
            blk_zero<NT>(y);
            const unsigned long long* mk = a.masks + ((long)k * M + j) * 4;
            blk_mul<NT, NT <= PL_MAXNT>(y, LdN{Uk + (long)j * NN, NP}, C, mk[1]);
            blk_zero<NT>(C);
            blk_mul<NT>(C, LdN{gl(j), NP}, y);
            blk_zero<NT>(y);
            blk_mul<NT, NT <= PL_MAXNT>(y, LdT{Lk + (long)j * NN, NP}, R, mk[2]);
            blk_load<NT>(R, LdN{g0(j), NP}, w);
            blk_mul<NT>(R, LdT{gl(j), NP}, y);
        }
        if (j < je) {
            const int lane = lane_new(), q = lane >> 4, n = a.psize[j], l = a.player[j] - 1 - a.lo;
            const long cc = (long)place * NP + 16 * w + (lane & 15);
            C2* CA = a.CA + l * a.K * a.b + cc * a.b;
            C2* RW = a.RW + l * a.K * a.b + cc;
            const int* pm = a.perm + (long)j * PL_PERM;
#pragma unroll
            for (int t = 0; t < NT; ++t)
#pragma unroll
                for (int r = 0; r < 4; ++r) {
                    const int row = 16 * t + 4 * r + q;
                    if (row < n) {
                        const int d = pm[row];
                        CA[d] = make_double2(C.re[t][r], C.im[t][r]);
                        RW[d * a.K] = make_double2(R.re[t][r], R.im[t][r]);
                    }
                }
        }
    }
}

// NEED_LAYERS: plan refused, a singular or nearly singular plane of a lead;
// lossy: what a point needs whose leads lost digits or left the finite numbers
__global__ void k_pl_check(const PlanHdr* h, int P, const int* dst, const LeadLoss* loss, const double* E, double eta,
                           double eta0, int mode, double res_max, int lossy, int* need, int* count)
{
    const int p = blockIdx.x * blockDim.x + threadIdx.x;
    if (p >= P) return;
    int why = h->ok ? 0 : NEED_LAYERS;
    if (!why) {
        const double e = E[p], et = mode == NT_ETA_RELATIVE ? e * eta + eta0 : eta;
        bool bad = false, lost = false;
        for (int i = 0; i < 2; ++i) {
            const int d = dst[2 * p + i];
            const LeadLoss l = loss[2 * p + i];
            // (the sweep goes through the planes inside the cell as well)
            bad = bad || (d != 0 && d != -1 && d != NT_ERR_NOT_CONVERGED) || (d == 0 && l.mid > PL_KAPPA);
            const double r = fabs(et) / l.scale, b = fmin(res_max, r < PL_SMALL_ETA ? r : PL_RESIDUAL_ETA * r);
            lost = lost || d == -1 || (d == 0 && !(l.res <= b && l.mid <= PL_KAPPA));
        }
        why = bad ? NEED_LAYERS : lost ? lossy : 0;
    }
    need[p] = why;
    if (why) atomicAdd(count + (why == NEED_LEADS ? CNT_LEADS : CNT_LAYERS), 1);
}

// *same stays 1 where the planes of both lead cells hold the same degrees of
// freedom in the same places as the stored ones (sizes, then PL_PERM places of
// every plane); store: written instead.  One workgroup per plane.
__global__ void k_pl_lead_planes(const PlanHdr* h, const int* psize, const int* perm, int* stored, int store, int* same)
{
    const int q = blockIdx.x, pl = q < h->m0 ? q : h->M - h->m1 + (q - h->m0), n = psize[pl];
    int* o = stored + (long)q * (PL_PERM + 1);
    for (int i = threadIdx.x; i <= n; i += blockDim.x) {
        const int v = i ? perm[(long)pl * PL_PERM + i - 1] : n;
        if (store) o[i] = v;
        else if (o[i] != v) *same = 0;
    }
}

__global__ void k_pl_count(int n, const int* need, int* count)
{
    const int p = blockIdx.x * blockDim.x + threadIdx.x;
    if (p < n && need[p] == NEED_LAYERS) atomicAdd(count + CNT_LAYERS, 1);
}

// Self-energies of the layers (layers_sigma) of the points idx onto the planes
// that face the leads, with their statuses and step counts; a point with a
// singular matrix on the layers is left to them.  The layers' sweep begins
// with the left lead's es and closes with V^+ g V of the right one, which differ
// by the digits lost: left takes the former.  blockIdx.y: item.
__global__ void k_pl_put_sigma(PlanDims d, PlanView v, BlocksIn B, const int* idx, const int* kidx, const C2* S,
                               const C2* ES, long stride, const int* st, const int* it, C2* sigma, C2* left, int* dst,
                               int* dit, int* need, int* count)
{
    const int q = blockIdx.y, p = idx[q / 2], side = q & 1, M = v.h->M, NP = 16 * v.h->nt;
    const int pl = side ? M - 1 : 0, n = v.psize[pl], ld = side ? d.nr : d.nl;
    const int* pm = v.perm + (long)pl * PL_PERM;
    const C2 *s = S + q * stride, *es = ES + q * stride;
    const C2* H = layer_H(d, B, side ? d.L + 1 : 0, kidx ? kidx[q / 2] : 0);
    for (int e = blockIdx.x * blockDim.x + threadIdx.x; e < NP * NP; e += gridDim.x * blockDim.x) {
        const int r = e % NP, c = e / NP;
        C2 x = make_double2(0.0, 0.0), y = x;
        if (r < n && c < n) {
            // (retarded = adjoint of the left lead's advanced)
            const long o = side ? pm[r] + (long)pm[c] * ld : pm[c] + (long)pm[r] * ld;
            x = s[o];
            y = make_double2(es[o].x - H[o].x, es[o].y - H[o].y);
            if (!side) x.y = -x.y, y.y = -y.y;
        }
        sigma[(long)(2 * p + side) * NP * NP + e] = x;
        if (!side) left[(long)p * NP * NP + e] = y;
    }
    if (blockIdx.x || threadIdx.x) return;
    dst[2 * p + side] = st[q];
    dit[2 * p + side] = it[q];
    if (!side) {
        bool bad = false;
        for (int i = 0; i < 2; ++i)
            bad = bad || (st[q + i] != 0 && st[q + i] != -1 && st[q + i] != NT_ERR_NOT_CONVERGED);
        need[p] = bad ? NEED_LAYERS : 0;
        if (bad) atomicAdd(count + CNT_LAYERS, 1);
    }
}

// Points solved on the planes: statuses, iteration counts, clamps.  A singular
// or nearly singular plane in the sweep sets need[p] too; count[CNT_STEPS] sums
// the decimation steps.
__global__ void k_pl_finish(int P, const int* dst, const int* dit, const int* sst, const double* T,
                            const LeadLoss* loss, const double* grow, double T_floor, const int* first_mask, int* need,
                            int* count, double* T_LR, double* T_RL, int* status, int* iters)
{
    const int p = blockIdx.x * blockDim.x + threadIdx.x;
    if (p >= P || need[p]) return;
    double tl = T[2 * p], tr = T[2 * p + 1];
    // a lead's recursion that left the finite numbers on the layers: no T
    const bool none = dst[2 * p] == -1 || dst[2 * p + 1] == -1;
    if (none) tl = tr = __longlong_as_double(0x7ff8000000000000LL);
    const double kappa = fmax(grow[2 * p], grow[2 * p + 1]) * fmax(loss[2 * p].scale, loss[2 * p + 1].scale);
    if (!none && (sst[2 * p] || sst[2 * p + 1] || tl != tl || tr != tr ||
        !(kappa * sqrt(fmin(fmax(fmax(tl, tr), T_floor), 1.0)) <= PL_KAPPA))) {
        need[p] = NEED_AFTER_SWEEP;
        atomicAdd(count + CNT_AFTER_SWEEP, 1);
        return;
    }
    atomicAdd(count + CNT_STEPS, dit[2 * p] + dit[2 * p + 1]);
    if (tl < 1.0e-60) tl = 0.0;       // negf/lesser.f90:795-800
    if (tr < 1.0e-60) tr = 0.0;
    if (first_mask && first_mask[p]) tl = tr = 0.0;      // negf/lesser.f90:802-807
    T_LR[p] = tl;
    T_RL[p] = tr;
    if (status) status[p] = dst[2 * p] ? dst[2 * p] : dst[2 * p + 1];
    if (iters) iters[p] = (dit[2 * p] + dit[2 * p + 1] + 1) / 2;
}

// the points with need[p] == which, in order, at most `most` of them: their
// indexes and inputs.  One workgroup.
__global__ __launch_bounds__(1024) void k_pl_gather(int P, const int* need, int which, int most, const double* E,
                                                    const int* kidx, const int* first, int* idx, double* gE, int* gk,
                                                    int* gf, const double* wt, double* gw)
{
    __shared__ int wsum[16];
    int base = 0;
    const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
    for (int p0 = 0; p0 < P; p0 += 1024) {
        const int p = p0 + threadIdx.x;
        const bool on = p < P && need[p] == which;
        const unsigned long long m = __ballot(on);
        if (lane == 0) wsum[w] = __popcll(m);
        __syncthreads();
        int off = base, all = 0;
        for (int i = 0; i < 16; ++i) {
            if (i < w) off += wsum[i];
            all += wsum[i];
        }
        const int o = off + __popcll(m & ((1ull << lane) - 1));
        if (on && o < most) {
            idx[o] = p;
            gE[o] = E[p];
            if (kidx) gk[o] = kidx[p];
            if (first) gf[o] = first[p];
            if (wt) gw[o] = wt[p];
        }
        base += all;
        __syncthreads();
    }
}

// out += the sum of S parts
__global__ void k_pl_add_parts(long n, int S, const C2* part, C2* out)
{
    const long i = (long)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    C2 v = out[i];
    for (int g = 0; g < S; ++g) {
        const C2 x = part[(long)g * n + i];
        v.x += x.x;
        v.y += x.y;
    }
    out[i] = v;
}

__global__ void k_pl_scatter(int n, const int* idx, const double* Tl, const double* Tr, const int* st, const int* it,
                             double* T_LR, double* T_RL, int* status, int* iters)
{
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    const int p = idx[i];
    T_LR[p] = Tl[i];
    T_RL[p] = Tr[i];
    if (status) status[p] = st[i];
    if (iters) iters[p] = it[i];
}

}  // namespace

namespace {

void ensure_plan_buf(nt_ctx* c, size_t bytes)
{
    if (c->plan_bytes >= bytes) return;
    if (c->plan_buf) {
        hipcheck(c, hipStreamSynchronize(c->stream), "hipStreamSynchronize");
        unreg_region(c, c->plan_buf);
        hipcheck(c, hipFree(c->plan_buf), "hipFree");
        c->plan_buf = nullptr;
        c->plan_bytes = 0;
    }
    hipcheck(c, hipMalloc(&c->plan_buf, bytes), "hipMalloc plan");
    c->plan_bytes = bytes;
    reg_region(c, c->plan_buf, bytes);
}

double free_bytes(nt_ctx* c)
{
    size_t free_b = 0, total_b = 0;
    hipcheck(c, hipMemGetInfo(&free_b, &total_b), "hipMemGetInfo");
    return (double)free_b;
}

// gathered inputs and results of the points left to the layers
void ensure_left_buf(nt_ctx* w, size_t bytes)
{
    unreg_region(w, w->left_buf);
    if (w->left_bytes < bytes) {
        if (w->left_buf) {
            hipcheck(w, hipStreamSynchronize(w->stream), "hipStreamSynchronize");
            hipcheck(w, hipFree(w->left_buf), "hipFree");
            w->left_buf = nullptr;
            w->left_bytes = 0;
        }
        hipcheck(w, hipMalloc(&w->left_buf, bytes), "hipMalloc points");
        w->left_bytes = bytes;
    }
    reg_region(w, w->left_buf, w->left_bytes);
}

// per point of a chunk: the two leads' decimation slots and self-energies,
// statuses, counts, digits lost, T of both directions
struct ChunkView {
    C2 *scratch, *sigma, *left;
    int *dst, *dit, *sst;
    LeadLoss* loss;
    double *T, *grow;
    C2 *keep = nullptr, *CA = nullptr, *RW = nullptr;      // adjoint
    int* place = nullptr;
};

ChunkView chunk_carve(Arena& a, int P, int NN)
{
    const size_t it = 2 * (size_t)P;
    ChunkView v;
    v.scratch = a.ptr<C2>(a.take(NN <= 256 * PL_MAXNT * PL_MAXNT ? sizeof(C2) * it * DEC_SLOTS * NN : 0));
    v.sigma = a.ptr<C2>(a.take(sizeof(C2) * it * NN));
    v.left = a.ptr<C2>(a.take(sizeof(C2) * P * NN));
    v.dst = a.ptr<int>(a.take(sizeof(int) * it));
    v.dit = a.ptr<int>(a.take(sizeof(int) * it));
    v.sst = a.ptr<int>(a.take(sizeof(int) * it));
    v.loss = a.ptr<LeadLoss>(a.take(sizeof(LeadLoss) * it));
    v.grow = a.ptr<double>(a.take(sizeof(double) * it));
    v.T = a.ptr<double>(a.take(sizeof(double) * it));
    return v;
}

// what devices with the same leads share (PlanesLeads): per point the leads'
// self-energies, digits lost, statuses, step counts and need, and the lead
// cells' planes
struct LeadsView {
    C2 *sigma, *left;
    LeadLoss* loss;
    int *dst, *dit, *need, *planes;
};
LeadsView leads_carve(Arena& a, int npts, int NN, int planes)
{
    LeadsView v;
    v.sigma = a.ptr<C2>(a.take(sizeof(C2) * 2 * NN * (size_t)npts));
    v.left = a.ptr<C2>(a.take(sizeof(C2) * NN * (size_t)npts));
    v.loss = a.ptr<LeadLoss>(a.take(sizeof(LeadLoss) * 2 * (size_t)npts));
    v.dst = a.ptr<int>(a.take(sizeof(int) * 2 * (size_t)npts));
    v.dit = a.ptr<int>(a.take(sizeof(int) * 2 * (size_t)npts));
    v.need = a.ptr<int>(a.take(sizeof(int) * (size_t)npts));
    v.planes = a.ptr<int>(a.take(sizeof(int) * (PL_PERM + 1) * (size_t)planes));
    return v;
}

// ---------------------------------------- leads whose planes hold more than 64
// The two planes of a lead cell, as one matrix, no longer fit the decimation
// kernel's registers: their cell (the planes between eliminated by one batched
// inverse and four products) goes through the layers' decimation instead, as a
// lead of 2 NP degrees of freedom of its own (half of the layer's: an eighth
// of its operations).

// shift and (k, lead) of item 2 p + lead
__global__ void k_pl_items(int P, const double* E, const int* kidx, double eta, double eta0, int mode, double* z,
                           int* idx)
{
    const int q = blockIdx.x * blockDim.x + threadIdx.x;
    if (q >= 2 * P) return;
    const double e = E[q / 2], et = mode == NT_ETA_RELATIVE ? e * eta + eta0 : eta;
    z[2 * q] = e;
    z[2 * q + 1] = q & 1 ? et : -et;
    idx[q] = 2 * (kidx ? kidx[q / 2] : 0) + (q & 1);
}

// packed block of a lead cell's planes counted from A: 0 diagonal block of
// plane j, 1 coupling j -> j + 1, 2 coupling back
__device__ __forceinline__ const C2* cell_block(const C2* H, const C2* U, const C2* Lw, int M, long NN, int k, int side,
                                                int what, int j)
{
    const long o = (long)k * M;
    if (what == 0) return H + (o + (side ? M - 1 - j : j)) * NN;
    return ((what == 1) != (side != 0) ? U : Lw) + (o + (side ? M - 2 - j : j)) * NN;
}

// per (k, lead): F_0, B_0, F_l, B_l (l the last coupling) and V as a 2 NP square
__global__ void k_pl_cell_stack(int M, int NP, int mc, const C2* H, const C2* U, const C2* Lw, const C2* LV, C2* CP,
                                C2* VS)
{
    const int ks = blockIdx.y, k = ks / 2, side = ks & 1;
    const long NN = (long)NP * NP;
    for (long e = (long)blockIdx.x * blockDim.x + threadIdx.x; e < 4 * NN; e += (long)gridDim.x * blockDim.x) {
        const int m = (int)(e / NN);
        const long i = e % NN;
        CP[(long)ks * 4 * NN + e] = cell_block(H, U, Lw, M, NN, k, side, 1 + (m & 1), m < 2 ? 0 : mc - 2)[i];
        const int r = (int)(e % (2 * NP)), c = (int)(e / (2 * NP));
        VS[(long)ks * 4 * NN + e] =
            r >= NP && c < NP ? LV[(long)ks * NN + (r - NP) + (long)c * NP] : make_double2(0.0, 0.0);
    }
}

// z - the planes between A and B (one or two), the identity on the padding
__global__ void k_pl_cell_mid(int M, int NP, int mc, const int* psize, const C2* H, const C2* U, const C2* Lw,
                              const int* idx, const double* z, C2* W)
{
    const int q = blockIdx.y, ks = idx[q], k = ks / 2, side = ks & 1, N2 = 2 * NP;
    const long NN = (long)NP * NP;
    for (long e = (long)blockIdx.x * blockDim.x + threadIdx.x; e < 4 * NN; e += (long)gridDim.x * blockDim.x) {
        const int r = (int)(e % N2), c = (int)(e / N2), hr = r >= NP, hc = c >= NP, r0 = r - hr * NP, c0 = c - hc * NP;
        const int nr = hr && mc < 4 ? 0 : psize[side ? M - 2 - hr : 1 + hr];
        const int ncl = hc && mc < 4 ? 0 : psize[side ? M - 2 - hc : 1 + hc];
        C2 x = make_double2(r == c ? 1.0 : 0.0, 0.0);
        if (r0 < nr && c0 < ncl) {
            const C2 b = cell_block(H, U, Lw, M, NN, k, side, hr == hc ? 0 : hr < hc ? 1 : 2, hr == hc ? 1 + hr : 1)[
                r0 + (long)c0 * NP];
            x = make_double2((r == c ? z[2 * q] : 0.0) - b.x, (r == c ? z[2 * q + 1] : 0.0) - b.y);
        }
        W[(long)q * 4 * NN + e] = x;
    }
}

// the cell's own blocks added to He (cleared first where add = 0); the padding's
// diagonal is 0, or -1 at E = 0: the decimation inverts z - He, and z without
// real part may be nothing, while z - (z - 1) is 0 from |E| = 2^53 on
__global__ void k_pl_cell_own(int M, int NP, int mc, const int* psize, const C2* H, const C2* U, const C2* Lw,
                              const int* idx, const double* z, int add, C2* He)
{
    const int q = blockIdx.y, ks = idx[q], k = ks / 2, side = ks & 1, N2 = 2 * NP;
    const long NN = (long)NP * NP;
    for (long e = (long)blockIdx.x * blockDim.x + threadIdx.x; e < 4 * NN; e += (long)gridDim.x * blockDim.x) {
        const int r = (int)(e % N2), c = (int)(e / N2), hr = r >= NP, hc = c >= NP, r0 = r - hr * NP, c0 = c - hc * NP;
        C2 x = add ? He[(long)q * 4 * NN + e] : make_double2(0.0, 0.0);
        if (hr == hc || mc == 2) {
            const C2 b = cell_block(H, U, Lw, M, NN, k, side, hr == hc ? 0 : hr < hc ? 1 : 2,
                                    hr == hc ? hr * (mc - 1) : 0)[r0 + (long)c0 * NP];
            x.x += b.x;
            x.y += b.y;
        }
        const int pl = hr ? mc - 1 : 0;
        if (r == c && r0 >= psize[side ? M - 1 - pl : pl]) x = make_double2(z[2 * q] == 0.0 ? -1.0 : 0.0, 0.0);
        He[(long)q * 4 * NN + e] = x;
    }
}

// retarded self-energy on plane A: the right lead's own, the left's adjoint
__global__ void k_pl_cell_sigma(int NP, const C2* S, C2* sigma)
{
    const int q = blockIdx.y, N2 = 2 * NP;
    const long NN = (long)NP * NP;
    for (long e = (long)blockIdx.x * blockDim.x + threadIdx.x; e < NN; e += (long)gridDim.x * blockDim.x) {
        const int r = (int)(e % NP), c = (int)(e / NP);
        const C2* s = S + (long)q * 4 * NN;
        C2 x = q & 1 ? s[r + (long)c * N2] : s[c + (long)r * N2];
        if (!(q & 1)) x.y = -x.y;
        sigma[(long)q * NN + e] = x;
    }
}

// LeadLoss of the cells but for the residual: the middle planes' inverse G1
// (mc > 2), the cell's first plane, its coupling and E.  One workgroup per item.
__global__ __launch_bounds__(256) void k_pl_cell_loss(int M, int NP, int mc, const int* psize, const C2* H,
                                                      const C2* VS, const C2* G1, const int* idx, const double* z,
                                                      LeadLoss* loss)
{
    const int q = blockIdx.x, ks = idx[q], side = ks & 1, N2 = 2 * NP, N4 = N2 * N2, t = threadIdx.x;
    auto size_of = [&](C2 x) { const double a = fabs(x.x) + fabs(x.y); return a == a ? a : INFINITY; };
    double g = 0.0, e = 0.0;
    if (mc > 2) {
        const int n1 = psize[side ? M - 2 : 1], n2 = mc == 4 ? psize[side ? M - 3 : 2] : 0;
        auto in = [&](int r) { return r < NP ? r < n1 : r - NP < n2; };
        const C2* m = G1 + (long)q * N4;
        for (int i = t; i < N4; i += 256)
            if (in(i % N2) && in(i / N2)) g = fmax(g, size_of(m[i]));
    }
    const C2 *A = cell_block(H, nullptr, nullptr, M, (long)NP * NP, ks / 2, side, 0, 0), *V = VS + (long)ks * N4;
    for (int i = t; i < NP * NP; i += 256) e = fmax(e, size_of(A[i]));
    for (int i = t; i < N4; i += 256) e = fmax(e, size_of(V[i]));
    __shared__ double wg[4], we[4];
    for (int o = 32; o; o >>= 1) {
        g = fmax(g, __shfl_xor(g, o));
        e = fmax(e, __shfl_xor(e, o));
    }
    if ((t & 63) == 0) {
        wg[t >> 6] = g;
        we[t >> 6] = e;
    }
    __syncthreads();
    if (t == 0) {
        for (int i = 1; i < 4; ++i) {
            g = fmax(g, wg[i]);
            e = fmax(e, we[i]);
        }
        e = fmax(e, fabs(z[2 * q]));
        loss[q].mid = g * e;
        loss[q].scale = e;
    }
}

struct BigView {
    C2 *CP, *VS, *W, *G1, *He, *S;
    double* z;
    int* idx;
    size_t dec_off;
};

BigView big_carve(Arena& a, int P, int nk, int NP)
{
    const size_t N2 = 2 * (size_t)NP, mb = sizeof(C2) * N2 * N2, Q = 2 * (size_t)P;
    BigView v;
    v.CP = a.ptr<C2>(a.take(mb * 2 * nk));
    v.VS = a.ptr<C2>(a.take(mb * 2 * nk));
    v.W = a.ptr<C2>(a.take(mb * Q));
    v.G1 = a.ptr<C2>(a.take(mb * Q));
    v.He = a.ptr<C2>(a.take(mb * Q));
    v.S = a.ptr<C2>(a.take(mb * Q));
    v.z = a.ptr<double>(a.take(sizeof(double) * 2 * Q));
    v.idx = a.ptr<int>(a.take(sizeof(int) * Q));
    v.dec_off = a.off;
    a.take(lead_sigma_scratch((int)N2, (int)Q));
    return v;
}

// bytes a chunk of points may take (with the batch limit of the context, its
// workspace cap and the free memory); where the host does not know the planes,
// the packed blocks included
constexpr double PL_CHUNK_BYTES = 6.0 * 1024 * 1024 * 1024;
constexpr double PL_ADJ_BYTES = 24.0 * 1024 * 1024 * 1024;
constexpr double PL_SHARE_BYTES = 1.0 * 1024 * 1024 * 1024;      // self-energies kept for devices with the same leads
constexpr int PL_MAX_GRID_Y = 65535;    // a launch's second and third dimensions
constexpr int PL_MAX_ITER = 20000;      // decimation steps inside one kernel

// self-energies of a chunk's points on leads of large planes
void planes_big_leads(nt_ctx* c, const nt_params* prm, const TdbArgs& a, const PlanView& v, const PlanHdr& h,
                      const BigView& g, Arena& ar, const C2* pH, const C2* pU, const C2* pL, const C2* pV, int p0, int n,
                      const ChunkView& cv)
{
    typedef double T;
    hipStream_t s = c->stream;
    const int NP = 16 * h.nt, N2 = 2 * NP, Q = 2 * n, mc = h.m0, nk2 = 2 * a.nk;
    const long NN = (long)NP * NP, N4 = 4 * NN;
    const unsigned gx = nblk(N4, 1024);
    auto R = [](const C2* p) { return reinterpret_cast<const T*>(p); };
    auto W = [](C2* p) { return reinterpret_cast<T*>(p); };
    launch(c, NT_K_ELEM, 0, "cell items", [&] {
        hipLaunchKernelGGL(k_pl_items, dim3(nblk(Q)), dim3(256), 0, s, n, a.E + p0, a.kidx ? a.kidx + p0 : nullptr,
                           prm->eta, prm->eta0, prm->eta_mode, g.z, g.idx);
        hipLaunchKernelGGL(k_pl_cell_stack, dim3(gx, nk2), dim3(256), 0, s, h.M, NP, mc, pH, pU, pL, pV, g.CP, g.VS);
        return hipGetLastError();
    });
    zero_dev(c, cv.dst, sizeof(int) * Q, s);
    if (mc > 2) {
        launch(c, NT_K_ELEM, 0, "cell mid", [&] {
            hipLaunchKernelGGL(k_pl_cell_mid, dim3(gx, Q), dim3(256), 0, s, h.M, NP, mc, v.psize, pH, pU, pL, g.idx, g.z,
                               g.W);
            return hipGetLastError();
        });
        inverse<T>(c, N2, bw(W(g.W), N4, N2), none<T>(), nullptr, bw(W(g.G1), N4, N2), cv.dst, Q);
        // T = G [B_0, F_l] (into W), He = [F_0 T; B_l T]
        const int r = mc == 4 ? NP : 0;
        auto blk = [&](int m) { return bm<T>(R(g.CP) + 2 * m * NN, N4, NP, g.idx, 0, nk2); };
        gemm<T>(c, N2, NP, NP, OP_N, bm<T>(R(g.G1), N4, N2), OP_N, blk(1), bw(W(g.W), N4, N2), 1.0, none<T>(), 0.0,
                nullptr, Q);
        gemm<T>(c, N2, NP, NP, OP_N, bm<T>(R(g.G1) + 2L * r * N2, N4, N2), OP_N, blk(2),
                bw(W(g.W) + 2L * NP * N2, N4, N2), 1.0, none<T>(), 0.0, nullptr, Q);
        gemm<T>(c, NP, N2, NP, OP_N, blk(0), OP_N, bm<T>(R(g.W), N4, N2), bw(W(g.He), N4, N2), 1.0, none<T>(), 0.0,
                nullptr, Q);
        gemm<T>(c, NP, N2, NP, OP_N, blk(3), OP_N, bm<T>(R(g.W) + 2 * r, N4, N2), bw(W(g.He) + 2 * NP, N4, N2), 1.0,
                none<T>(), 0.0, nullptr, Q);
    }
    launch(c, NT_K_ELEM, 0, "cell own", [&] {
        hipLaunchKernelGGL(k_pl_cell_own, dim3(gx, Q), dim3(256), 0, s, h.M, NP, mc, v.psize, pH, pU, pL, g.idx, g.z,
                           mc > 2, g.He);
        return hipGetLastError();
    });
    launch(c, NT_K_ELEM, 0, "cell loss", [&] {
        hipLaunchKernelGGL(k_pl_cell_loss, dim3(Q), dim3(256), 0, s, h.M, NP, mc, v.psize, pH, g.VS, g.G1, g.idx,
                           g.z, cv.loss);
        return hipGetLastError();
    });
    lead_sigma(c, N2, Q, bm<T>(R(g.He), N4, N2), bm<T>(R(g.VS), N4, N2, g.idx, 0, nk2), g.z, prm->convergence,
               prm->max_iter, bw(W(g.G1), N4, N2), bw(W(g.S), N4, N2), cv.dst, cv.dit, &cv.loss->res,
               sizeof(LeadLoss) / sizeof(double), ar, g.dec_off);
    launch(c, NT_K_ELEM, 0, "cell sigma", [&] {
        hipLaunchKernelGGL(k_pl_cell_sigma, dim3(nblk(NN, 1024), Q), dim3(256), 0, s, NP, g.S, cv.sigma);
        return hipGetLastError();
    });
}

template <int NT>
void launch_adjoint(const AdjPlArgs& a, int n, hipStream_t s)
{
    hipLaunchKernelGGL(k_pl_adjoint<NT>, dim3(n), dim3(64 * NT), 0, s, a);
}

// Gradients of one chunk's points, added to a's dHd and dHdv.
void planes_adjoint(nt_ctx* c, const TdbArgs& a, const PlanView& v, const PlanHdr& h,
                    const ChunkView& cv, const C2* pU, const C2* pL, const unsigned long long* pM, int p0, int n, const std::vector<int>& hk,
                    const int* need, long kept, int hi1)
{
    typedef double T;
    hipStream_t s = c->stream;
    const int NP = 16 * h.nt, b = a.b, lo = a.adj_lo, hi = a.adj_hi, nw = hi - lo + 1, hc = std::min(hi, a.L - 2),
              nc = hc - lo + 1;
    const long K = (long)n * NP;
    // points of one k-point stand together
    std::vector<int> place, k0(a.nk + 1, 0);
    if (a.nk > 1) {
        for (int i = 0; i < n; ++i) ++k0[hk[p0 + i] + 1];
        for (int k = 0; k < a.nk; ++k) k0[k + 1] += k0[k];
        std::vector<int> at(k0.begin(), k0.end() - 1);
        place.resize(n);
        for (int i = 0; i < n; ++i) place[i] = at[hk[p0 + i]]++;
        hipcheck(c, hipMemcpyAsync(cv.place, place.data(), sizeof(int) * n, hipMemcpyHostToDevice, s), "H2D");
        hipcheck(c, hipStreamSynchronize(s), "sync");
    } else {
        k0[1] = n;
    }
    const AdjPlArgs aa{v.h, v.psize, v.player, v.poff, v.perm, pU, pL, pM, cv.sigma, cv.keep, kept,
                       a.kidx ? a.kidx + p0 : nullptr, need, cv.sst, cv.dst, a.first_mask ? a.first_mask + p0 : nullptr,
                       a.adj_w + p0, a.nk > 1 ? cv.place : nullptr, lo, hi1, b, K, cv.CA, cv.RW};
    check_range(c, a.adj_w + p0, sizeof(double) * n, "adjoint weights");
    const double m = NP;
    launch(c, NT_K_PLANES, 4.0 * 8 * m * m * m * n * (kept / 2), "plane adjoint", [&] {
        if (h.nt == 1) launch_adjoint<1>(aa, n, s);
        if (h.nt == 2) launch_adjoint<2>(aa, n, s);
        if (h.nt == 3) launch_adjoint<3>(aa, n, s);
        if (h.nt == 4) launch_adjoint<4>(aa, n, s);
        if (h.nt == PL_BIGNT) launch_adjoint<PL_BIGNT>(aa, n, s);
        return hipGetLastError();
    });
    // dHd_l += 2 sum_p R_l^+ C_l^+, dHdv_l += 2 sum_p (R_l^+ C_{l+1}^+ + C_l R_{l+1}),
    // one launch for all layers of the window
    const long bb = (long)b * b, per = K * b;
    const T* CA = reinterpret_cast<const T*>(cv.CA);
    const T* RW = reinterpret_cast<const T*>(cv.RW);
    // A product has the depth of all points but few tiles (17 layers of 192: 153
    // workgroups on 256 CUs, 6.4 ms each): parts of the points are summed side by
    // side, up to four workgroups per CU of them, into the decimation's scratch,
    // which is free by now, and then added up; the points beyond equal parts
    // form one more product.  The three products 19 -> 10 ms at 512 points.
    T* part = h.nt <= PL_MAXNT ? reinterpret_cast<T*>(cv.scratch) : nullptr;
    const long room = part ? 2L * n * DEC_SLOTS * NP * NP : 0;
    const long tiles = (long)((b + 63) / 64) * ((b + 63) / 64);
    for (int k = 0; k < a.nk; ++k) {
        const int nk = k0[k + 1] - k0[k];
        if (!nk) continue;
        // out += 2 (A1 B1 + A2 B2) over the k-point's points, layers of the window
        auto sum = [&](T* out, int layers, auto term, int terms) {
            const long want = std::min<long>({8, (4 * 256 + tiles * layers - 1) / (tiles * layers),
                                              room / ((long)layers * bb), (long)nk * NP / 512});
            const int S = (int)std::max<long>(1, want), q = nk / S, rest = S > 1 ? nk - q * S : 0;
            if (S > 1) check_range(c, part, sizeof(C2) * S * layers * bb, "gradient parts");
            for (int i = 0; i < terms; ++i) {
                const BMatW<T> to = S > 1 ? bw(part, bb, b, nullptr, (long)layers * bb) : bw(out, bb, b);
                term(i, k0[k], q, to, S > 1 && i == 0 ? none<T>() : ro(to), layers, S);
                if (rest) term(i, k0[k] + q * S, rest, bw(out, bb, b), bm<T>(out, bb, b), layers, 1);
            }
            if (S > 1) {
                hipLaunchKernelGGL(k_pl_add_parts, dim3(nblk(layers * bb)), dim3(256), 0, s, layers * bb, S,
                                   reinterpret_cast<const C2*>(part), reinterpret_cast<C2*>(out));
                hipcheck(c, hipGetLastError(), "add parts");
            }
        };
        // i of 0: R_l^+ C_l^+, 1: R_l^+ C_{l+1}^+, 2: C_l R_{l+1} over np points from p on
        auto product = [&](int what, int p, int np, BMatW<T> to, BMat<T> from, int layers, int S) {
            const long q0 = (long)p * NP, up = what == 0 ? 0 : per;
            const BMat<T> Rm = bm<T>(RW + 2 * (q0 + (what == 2 ? up : 0)), per, (int)K, nullptr, (long)np * NP);
            const BMat<T> Cm = bm<T>(CA + 2 * (q0 * b + (what == 1 ? up : 0)), per, b, nullptr, (long)np * NP * b);
            if (what == 2)
                gemm<T>(c, b, b, np * NP, OP_N, Cm, OP_N, Rm, to, 2.0, from, 1.0, nullptr, layers, -1, nullptr, S);
            else
                gemm<T>(c, b, b, np * NP, OP_C, Rm, OP_C, Cm, to, 2.0, from, 1.0, nullptr, layers, -1, nullptr, S);
        };
        sum(reinterpret_cast<T*>(a.dHd) + 2 * (long)k * nw * bb, nw,
            [&](int, int p, int np, BMatW<T> to, BMat<T> from, int layers, int S) {
                product(0, p, np, to, from, layers, S);
            }, 1);
        if (nc > 0 && a.dHdv)
            sum(reinterpret_cast<T*>(a.dHdv) + 2 * (long)k * nc * bb, nc,
                [&](int i, int p, int np, BMatW<T> to, BMat<T> from, int layers, int S) {
                    product(1 + i, p, np, to, from, layers, S);
                }, 2);
    }
}

template <int NT>
void launch_decimate(const DecPlArgs& a, int items, hipStream_t s)
{
    hipLaunchKernelGGL(k_pl_decimate<NT>, dim3(items), dim3(128 * NT), 0, s, a);
}
template <int NT>
void launch_sweep(const SweepPlArgs& a, int items, hipStream_t s)
{
    hipLaunchKernelGGL(k_pl_sweep<NT>, dim3(items), dim3(64 * NT), 0, s, a);
}

}  // namespace

namespace {
// inverses by panels only while it lives, as on the layers before the planes
struct PanelsOnly {
    nt_ctx* c;
    explicit PanelsOnly(nt_ctx* ctx) : c(ctx) { c->inv_panels = true; }
    ~PanelsOnly() { c->inv_panels = false; }
};
}  // namespace

// The n points of a's points [p0, p0 + P) with need == which, on the layers.
// beside: on a worker context, from where c's stream stands at chk[0] (the
// decimation's end) on, c's stream waiting for it; else on c's stream.
static void solve_left(nt_ctx* c, const nt_params* prm, const TdbArgs& a, int p0, int P, const int* need, int which,
                       int n, bool beside)
{
    nt_ctx* w = c;
    if (beside) {
        if (const int st = prepare_workers(c, 1)) {
            c->err = "could not set up a worker context";
            throw Fail{st};
        }
        w = c->subs[0];
        hipcheck(c, hipStreamWaitEvent(w->stream, c->chk[0], 0), "wait check");
    }
    const size_t nd = sizeof(double) * n, ni = sizeof(int) * n;
    hipStream_t s = w->stream;
    TdbArgs g = a;
    g.no_planes = true;
    g.siblings.clear();
    Arena la;
    const size_t oi = la.take(ni), oe = la.take(nd), ok = la.take(ni), of = la.take(ni), ol = la.take(nd),
                 orr = la.take(nd), os = la.take(ni), ot = la.take(ni), ow = la.take(nd);
    if (w != c) {
        w->regions = c->regions;
        if (w->ws) reg_region(w, w->ws, w->ws_bytes);
    }
    ensure_left_buf(w, 2 * la.off);
    la.base = static_cast<char*>(w->left_buf);
    int *idx = la.ptr<int>(oi), *gk = la.ptr<int>(ok), *gf = la.ptr<int>(of);
    double* gE = la.ptr<double>(oe);
    hipLaunchKernelGGL(k_pl_gather, dim3(1), dim3(1024), 0, s, P, need, which, n, a.E + p0,
                       a.kidx ? a.kidx + p0 : nullptr, a.first_mask ? a.first_mask + p0 : nullptr, idx, gE, gk, gf,
                       a.adj_w ? a.adj_w + p0 : nullptr, la.ptr<double>(ow));
    hipcheck(w, hipGetLastError(), "gather");
    if (a.adj_w) g.adj_w = la.ptr<double>(ow);
    g.npts = n;
    g.E = gE;
    g.kidx = a.kidx ? gk : nullptr;
    g.first_mask = a.first_mask ? gf : nullptr;
    g.T_LR = la.ptr<double>(ol);
    g.T_RL = la.ptr<double>(orr);
    g.status = la.ptr<int>(os);
    g.iters = la.ptr<int>(ot);
    try {
        const PanelsOnly panels(w);
        solve_tdb_dev(w, prm, g);
    } catch (const Fail&) {
        if (w != c) c->err = w->err;
        throw;
    }
    if (w != c) {
        hipcheck(c, hipEventRecord(w->join, s), "event join");
        hipcheck(c, hipStreamWaitEvent(c->stream, w->join, 0), "wait join");
        if (w->prof) harvest_profile(w);
        for (int k = 0; k < NT_K_COUNT; ++k) {
            c->launches[k] += w->launches[k];
            c->ms[k] += w->ms[k];
            c->flops[k] += w->flops[k];
            w->launches[k] = 0;
            w->ms[k] = 0;
            w->flops[k] = 0;
        }
        for (int k = 0; k < 3; ++k) {
            c->mixed_counts[k] += w->mixed_counts[k];
            w->mixed_counts[k] = 0;
        }
    }
    hipLaunchKernelGGL(k_pl_scatter, dim3(nblk(n)), dim3(256), 0, c->stream, n, idx, g.T_LR, g.T_RL, g.status, g.iters,
                       a.T_LR + p0, a.T_RL + p0, a.status ? a.status + p0 : nullptr, a.iters ? a.iters + p0 : nullptr);
    hipcheck(c, hipGetLastError(), "scatter");
}

// bytes the layers' self-energies of some of a chunk's points may take
constexpr double PL_LEADS_BYTES = 512.0 * 1024 * 1024;

// The leads of the m points with need == NEED_LEADS among a chunk's n, on the
// layers.  Returns how many points are left to the layers since then.
static int planes_redo_leads(nt_ctx* c, const nt_params* prm, const TdbArgs& a, const PlanDims& d, const PlanView& v,
                             const BlocksIn& B, const ChunkView& cv, int NP, int p0, int n, int m, int* need, int* cnt, int had)
{
    hipStream_t s = c->stream;
    Arena la;
    int *idx = nullptr, *gk = nullptr, *st = nullptr, *it = nullptr;
    double *gE = nullptr, *sig = nullptr, *es = nullptr;
    size_t scr = 0;
    auto carve = [&](int P) {
        la.off = 0;
        idx = la.ptr<int>(la.take(sizeof(int) * P));
        gk = la.ptr<int>(la.take(sizeof(int) * P));
        st = la.ptr<int>(la.take(sizeof(int) * 2 * P));
        it = la.ptr<int>(la.take(sizeof(int) * 2 * P));
        gE = la.ptr<double>(la.take(sizeof(double) * P));
        sig = la.ptr<double>(la.take(sizeof(C2) * 2 * sigma_stride(a) * P));
        es = la.ptr<double>(la.take(sizeof(C2) * 2 * sigma_stride(a) * P));
        scr = la.off;
        la.off += layers_sigma_scratch(a, P);
        return la.off;
    };
    const double one = ((double)carve(65) - (double)carve(1)) / 64;
    int P = std::max(1.0, std::min<double>({(double)m, (double)c->batch_limit, PL_LEADS_BYTES / one, PL_MAX_GRID_Y / 2}));
    if (carve(P) > c->left_bytes)          // no further than the memory reaches
        P = std::max(1.0, std::min<double>(P, 0.8 * (free_bytes(c) + (double)c->left_bytes) / one));
    carve(P);
    ensure_left_buf(c, la.off);
    la.base = static_cast<char*>(c->left_buf);
    carve(P);
    const size_t row = sizeof(C2) * NP * NP;
    hipcheck(c, hipMemcpy2DAsync(cv.left, row, cv.sigma, 2 * row, row, n, hipMemcpyDeviceToDevice, s), "copy sigma");
    for (int q = 0; q < m; q += P) {
        const int k = std::min(P, m - q);
        // (the points of earlier passes no longer need it)
        hipLaunchKernelGGL(k_pl_gather, dim3(1), dim3(1024), 0, s, n, need, NEED_LEADS, k, a.E + p0,
                           a.kidx ? a.kidx + p0 : nullptr, (const int*)nullptr, idx, gE, gk, (int*)nullptr,
                           (const double*)nullptr, (double*)nullptr);
        hipcheck(c, hipGetLastError(), "gather");
        {
            const PanelsOnly panels(c);
            layers_sigma(c, prm, a, k, gE, a.kidx ? gk : nullptr, sig, es, st, it, la, scr);
        }
        hipLaunchKernelGGL(k_pl_put_sigma, dim3(nblk((long)NP * NP, 8), 2 * k), dim3(256), 0, s, d, v, B, idx,
                           a.kidx ? gk : nullptr, reinterpret_cast<const C2*>(sig), reinterpret_cast<const C2*>(es),
                           sigma_stride(a), st, it, cv.sigma, cv.left, cv.dst, cv.dit, need, cnt);
        hipcheck(c, hipGetLastError(), "put sigma");
    }
    hipcheck(c, hipMemcpyAsync(c->host_plan, cnt, sizeof(int), hipMemcpyDeviceToHost, s), "count D2H");
    hipcheck(c, hipStreamSynchronize(s), "count sync");
    return c->host_plan[0] - had;
}

bool planes_candidate(const nt_ctx* c, const nt_params* prm, const TdbArgs& a)
{
    const nt_solve_extras& x = a.ex;
    const bool extras = x.gl_adv || x.gr_ret || x.gl_plus || x.gr_minus || x.gml_adv || x.gmr_ret || x.sl_adv ||
                        x.sr_ret || x.G_D_LR || x.G_D_RL || x.G_L || x.G_R || x.sdos_l || x.sdos_r || x.ldos ||
                        x.ddos;
    // (an adjoint solve needs the plan's sizes on the host)
    return c->planes && !a.no_planes && !a.mask && !(a.adj_w && c->dec_check == 0) && !a.probe && !extras &&
           !(prm->circular && prm->n_bloch_x * prm->n_bloch_y > 1) && c->one_sweep && !c->gemm_m3 &&
           prm->max_iter <= PL_MAX_ITER && a.nk <= PL_MAX_GRID_Y && 2 * a.L + 5 <= PL_MAX_GRID_Y;
}

// Solve a's points on their planes.  False: the blocks do not fall into planes
// of at most 96 (nothing was written).  Points the planes are no good for (a
// singular or nearly singular plane) are solved by the block path before it
// returns, leads whose decimation lost digits are decimated by it.
bool planes_solve(nt_ctx* c, const nt_params* prm, const TdbArgs& a, PlanesLeads* share)
{
    const bool wait = c->dec_check > 0;        // the host may wait for the device
    const PlanDims d = plan_dims(a.nl, a.nr, a.b, a.L, a.nk);
    hipStream_t s = c->stream;
    // the plan, the mask of points left to the block path, the counters
    Arena pa;
    plan_carve(pa, d);
    const size_t o_need = pa.take(sizeof(int) * (size_t)a.npts), o_cnt = pa.take(sizeof(int) * CNT_N);
    const size_t plan_need = pa.off;
    size_t scratch_bytes = 0;
    char* scratch = static_cast<char*>(scratch_region(c->device, &scratch_bytes));
    size_t reserve = 0;
    if (a.noalloc) {
        // at the end of the static scratch, which the block path then keeps off
        reserve = (plan_need + 4095) / 4096 * 4096;
        if (!scratch || 2 * reserve > scratch_bytes) return false;
        pa = Arena();
        pa.base = scratch + (scratch_bytes - reserve);
    } else {
        ensure_plan_buf(c, plan_need);
        pa = Arena();
        pa.base = static_cast<char*>(c->plan_buf);
    }
    const PlanView v = plan_carve(pa, d);
    int* need = pa.ptr<int>(o_need);
    int* cnt = pa.ptr<int>(o_cnt);
    if (c->ws_poison) poison_dev(c, pa.base, plan_need, s);
    zero_dev(c, v.h, (char*)v.level - (char*)v.h, s);
    zero_dev(c, cnt, sizeof(int) * CNT_N, s);
    const BlocksIn B{reinterpret_cast<const C2*>(a.Haml), reinterpret_cast<const C2*>(a.Hamlv),
                     reinterpret_cast<const C2*>(a.Hamr), reinterpret_cast<const C2*>(a.Hamrv),
                     reinterpret_cast<const C2*>(a.Hamd), reinterpret_cast<const C2*>(a.Hamdv),
                     reinterpret_cast<const C2*>(a.Hamld), reinterpret_cast<const C2*>(a.Hamrd)};
    const size_t z = sizeof(C2);
    check_range(c, B.Haml, z * a.nl * a.nl * a.nk, "planes Haml");
    check_range(c, B.Hamlv, z * a.nl * a.nl * a.nk, "planes Hamlv");
    check_range(c, B.Hamr, z * a.nr * a.nr * a.nk, "planes Hamr");
    check_range(c, B.Hamrv, z * a.nr * a.nr * a.nk, "planes Hamrv");
    check_range(c, B.Hamd, z * a.b * a.b * a.L * a.nk, "planes Hamd");
    if (a.L > 1) check_range(c, B.Hamdv, z * a.b * a.b * (a.L - 1) * a.nk, "planes Hamdv");
    check_range(c, B.Hamld, z * a.nl * a.b * a.nk, "planes Hamld");
    check_range(c, B.Hamrd, z * a.nr * a.b * a.nk, "planes Hamrd");
    check_range(c, a.E, sizeof(double) * a.npts, "planes E");
    check_range(c, a.kidx, sizeof(int) * a.npts, "planes kidx");
    check_range(c, a.first_mask, sizeof(int) * a.npts, "planes first mask");
    check_range(c, a.T_LR, sizeof(double) * a.npts, "planes T_LR");
    check_range(c, a.T_RL, sizeof(double) * a.npts, "planes T_RL");
    check_range(c, a.status, sizeof(int) * a.npts, "planes status");
    check_range(c, a.iters, sizeof(int) * a.npts, "planes iters");
    const int nL = a.L + 2;
    // the large class where the host may wait, with workspace, with a launch's
    // second dimension for the leads of all k-points, and not at a
    // fixed broadening (the electrons' eta = 1e-8 eV: only phonons were measured)
    const bool large = wait && !a.noalloc && 2L * a.nk <= PL_MAX_GRID_Y && prm->eta_mode == NT_ETA_RELATIVE;
    const int ncls = large ? PL_NCLS : PL_MAXNT;
    launch(c, NT_K_ELEM, 0, "plane pattern", [&] {
        const unsigned gx = nblk((long)d.nmax * d.nmax, 1024);
        // the first k-point's pattern alone refuses dense blocks (49 k-points
        // of b = 48, L = 2 took 1.1 ms to be refused together)
        for (int k0 = 0; k0 < a.nk; k0 += k0 ? a.nk : 1) {
            hipLaunchKernelGGL(k_pl_pattern, dim3(gx, 2 * a.L + 5, k0 ? a.nk - 1 : 1), dim3(256), 0, s, d, v, B, k0);
            hipLaunchKernelGGL(k_pl_levels, dim3(nL), dim3(256), 0, s, d, v);
            hipLaunchKernelGGL(k_pl_plan, dim3(1), dim3(64 * PL_NCLS), 0, s, d, v, ncls);
        }
        hipLaunchKernelGGL(k_pl_perm, dim3(nL), dim3(256), 0, s, d, v);
        return hipGetLastError();
    });
    // sizes: the plan's when the host may wait for it, else their bounds
    PlanHdr h{1, PL_MAXNT, d.Mcap, 0, 0};
    if (wait) {
        hipcheck(c, hipMemcpyAsync(c->host_plan, v.h, sizeof(PlanHdr), hipMemcpyDeviceToHost, s), "plan D2H");
        hipcheck(c, hipStreamSynchronize(s), "plan sync");
        h = *reinterpret_cast<const PlanHdr*>(c->host_plan);
        if (!h.ok) return false;
        if (h.nt < 1 || h.nt > PL_BIGNT || h.M < 3 || h.M > d.Mcap) {
            c->err = "plane plan out of range";
            throw Fail{NT_ERR_HIP};
        }
    }
    const int NN = 256 * h.nt * h.nt;
    // adjoint: planes from the window's first on are kept
    const bool adj = a.adj_w != nullptr;
    const int hi1 = adj ? std::min(a.adj_hi + 1, a.L - 1) : 0, nw1 = hi1 - a.adj_lo + 1;
    int jw = 0;
    std::vector<int> hk;
    if (adj) {
        hipcheck(c, hipMemcpyAsync(c->host_plan, v.poff + a.adj_lo + 1, sizeof(int), hipMemcpyDeviceToHost, s), "D2H");
        if (a.nk > 1) {
            hk.resize(a.npts);
            hipcheck(c, hipMemcpyAsync(hk.data(), a.kidx, sizeof(int) * a.npts, hipMemcpyDeviceToHost, s), "D2H");
        }
        hipcheck(c, hipStreamSynchronize(s), "sync");
        jw = c->host_plan[0];
        if (jw < 0 || jw >= h.M) {
            c->err = "plane plan out of range";
            throw Fail{NT_ERR_HIP};
        }
    }
    const long kept = 2L * (h.M - jw);      // matrices per point
    // packed blocks, then one chunk of points
    Arena w;
    const size_t blk = z * NN * (size_t)h.M * a.nk;
    const size_t oH = w.take(blk), oU = w.take(blk), oL = w.take(blk), oV = w.take(z * NN * 2 * a.nk),
                 oM = w.take(sizeof(unsigned long long) * 4 * (size_t)h.M * a.nk);
    const size_t fixed = w.off;
    const int NP = 16 * h.nt;
    const bool big = h.nt > PL_MAXNT;
    BigView bv{};
    auto carve = [&](Arena& ar, int P) {
        ChunkView cv = chunk_carve(ar, P, NN);
        if (adj) {
            cv.keep = ar.ptr<C2>(ar.take(z * NN * kept * P));
            cv.CA = ar.ptr<C2>(ar.take(z * NP * a.b * nw1 * P));
            cv.RW = ar.ptr<C2>(ar.take(z * NP * a.b * nw1 * P));
            cv.place = ar.ptr<int>(ar.take(sizeof(int) * (size_t)P));
        }
        if (big) bv = big_carve(ar, P, a.nk, NP);
        return cv;
    };
    Arena one;
    carve(one, 64);
    const double per_pt = (double)one.off / 64;
    double room = adj ? PL_ADJ_BYTES : PL_CHUNK_BYTES;
    if (a.noalloc) room = (double)scratch_bytes - reserve - fixed - 65536.0;
    else if (!wait) room -= fixed;         // (the bound of blocks whose planes the host does not know)
    if (!a.noalloc && c->ws_cap) room = std::min(room, (double)c->ws_cap - fixed);
    int P = std::min({(double)a.npts, (double)c->batch_limit, room / per_pt});
    if (P < 1) {
        if (a.noalloc || !wait || c->ws_cap) return false;
        P = 1;
    }
    carve(w, P);
    if (!a.noalloc && w.off > c->ws_bytes) {
        // the workspace has to grow: no further than the memory reaches (ensure_ws
        // adds an eighth)
        const double have = 8.0 / 9.0 * (free_bytes(c) + (double)c->ws_bytes);
        if ((double)w.off > have) {
            const int q = std::min((double)P, (have - fixed) / per_pt) - 1;
            if (q < 1) return false;
            P = q;
            w.off = fixed;
            carve(w, P);
        }
    }
    if (a.noalloc) {
        if (w.off > scratch_bytes - reserve) return false;
        if (c->ws_poison) poison_dev(c, scratch, w.off, s);
    } else {
        ensure_ws(c, w.off);
    }
    const size_t total = w.off;
    w = Arena();
    w.base = a.noalloc ? scratch : static_cast<char*>(c->ws);
    check_range(c, w.base, total, "planes workspace");
    w.off = fixed;
    C2 *pH = w.ptr<C2>(oH), *pU = w.ptr<C2>(oU), *pL = w.ptr<C2>(oL), *pV = w.ptr<C2>(oV);
    unsigned long long* pM = w.ptr<unsigned long long>(oM);
    const ChunkView own = carve(w, P);
    launch(c, NT_K_ELEM, 0, "plane pack", [&] {
        hipLaunchKernelGGL(k_pl_pack, dim3(h.M, a.nk, 4), dim3(256), 0, s, d, v, B, pH, pU, pL, pV, pM);
        return hipGetLastError();
    });
    // Leads that another device of the call has or may want: the first one keeps
    // its self-energies for those whose lead cells have the same planes (the
    // couplings to the device take part in the plan)
    LeadsView lv{};
    bool reuse = false, keep_leads = false;
    if (share && wait && !a.noalloc && !adj && h.m0 + h.m1 <= 4 * PL_NLV) {
        Arena sa;
        leads_carve(sa, a.npts, NN, h.m0 + h.m1);
        const bool alike = share->have && share->nt == h.nt && share->m0 == h.m0 && share->m1 == h.m1;
        if (!share->have && (double)sa.off <= PL_SHARE_BYTES &&
            (sa.off <= c->leads_bytes || (double)sa.off <= 0.25 * (free_bytes(c) + (double)c->leads_bytes))) {
            if (c->leads_bytes < sa.off) {
                if (c->leads_buf) {
                    hipcheck(c, hipStreamSynchronize(s), "hipStreamSynchronize");
                    hipcheck(c, hipFree(c->leads_buf), "hipFree");
                    c->leads_buf = nullptr;
                    c->leads_bytes = 0;
                }
                hipcheck(c, hipMalloc(&c->leads_buf, sa.off), "hipMalloc leads");
                c->leads_bytes = sa.off;
            }
            keep_leads = true;
        }
        if (alike || keep_leads) {
            sa = Arena();
            sa.base = static_cast<char*>(c->leads_buf);
            lv = leads_carve(sa, a.npts, NN, h.m0 + h.m1);
            launch(c, NT_K_ELEM, 0, "fill", [&] { return launch_fill_int(cnt + CNT_SAME, 1, 1, s); });
            hipLaunchKernelGGL(k_pl_lead_planes, dim3(h.m0 + h.m1), dim3(128), 0, s, v.h, v.psize, v.perm, lv.planes,
                               keep_leads ? 1 : 0, cnt + CNT_SAME);
            hipcheck(c, hipGetLastError(), "lead planes");
        }
        if (alike) {
            hipcheck(c, hipMemcpyAsync(c->host_plan, cnt + CNT_SAME, sizeof(int), hipMemcpyDeviceToHost, s), "D2H");
            hipcheck(c, hipStreamSynchronize(s), "sync");
            reuse = c->host_plan[0] != 0;
        }
    }
    auto copy = [&](void* to, const void* from, size_t bytes) {
        hipcheck(c, hipMemcpyAsync(to, from, bytes, hipMemcpyDeviceToDevice, s), "copy leads");
    };
    int left = 0, later[2] = {0, 0};      // points solved on the layers, those not beside the sweep
    for (int p0 = 0; p0 < a.npts; p0 += P) {
        const int n = std::min(P, a.npts - p0);
        const int* kidx = a.kidx ? a.kidx + p0 : nullptr;
        const int* first = a.first_mask ? a.first_mask + p0 : nullptr;
        ChunkView cv = own;
        if (reuse) {
            cv.sigma = lv.sigma + 2L * p0 * NN;
            cv.left = lv.left + (long)p0 * NN;
            cv.loss = lv.loss + 2L * p0;
            cv.dst = lv.dst + 2L * p0;
            cv.dit = lv.dit + 2L * p0;
        }
        const DecPlArgs da{v.h, v.psize, pH, pU, pL, pV, a.E + p0, kidx, prm->eta, prm->eta0, prm->convergence,
                           prm->eta_mode, prm->max_iter, cv.scratch, cv.sigma, cv.dst, cv.dit, cv.loss};
        SweepPlArgs sa{v.h, v.psize, pH, pU, pL, pM, a.E + p0, kidx, prm->eta, prm->eta0, prm->device_eta_factor,
                       prm->eta_mode, need + p0, cv.sigma, nullptr, cv.T, cv.grow, cv.sst, cv.keep,
                       v.poff + a.adj_lo + 1, kept};
        if (p0) zero_dev(c, cnt, sizeof(int) * CNT_STEPS, s);
        if (reuse) {
            copy(need + p0, lv.need + p0, sizeof(int) * n);
            hipLaunchKernelGGL(k_pl_count, dim3(nblk(n)), dim3(256), 0, s, n, need + p0, cnt);
            hipcheck(c, hipGetLastError(), "count");
            sa.left = cv.left;
        } else if (big) planes_big_leads(c, prm, a, v, h, bv, w, pH, pU, pL, pV, p0, n, cv);
        else launch(c, NT_K_PLANES, 0, "plane decimation", [&] {
            if (!wait || h.nt == 1) launch_decimate<1>(da, 2 * n, s);
            if (!wait || h.nt == 2) launch_decimate<2>(da, 2 * n, s);
            if (!wait || h.nt == 3) launch_decimate<3>(da, 2 * n, s);
            if (!wait || h.nt == 4) launch_decimate<4>(da, 2 * n, s);
            return hipGetLastError();
        });
        // leads that lost digits: once more on the layers, where the host may wait
        // for their count and the call may allocate (else the whole point)
        const int lossy = wait && !a.noalloc ? NEED_LEADS : NEED_LAYERS;
        if (!reuse)
            hipLaunchKernelGGL(k_pl_check, dim3(nblk(n)), dim3(256), 0, s, v.h, n, cv.dst, cv.loss, a.E + p0, prm->eta,
                           prm->eta0, prm->eta_mode, adj ? PL_RESIDUAL_ADJ : PL_RESIDUAL, lossy, need + p0, cnt);
        hipcheck(c, hipGetLastError(), "plane check");
        int n1 = 0;                        // points for the layers
        if (wait) {
            hipcheck(c, hipMemcpyAsync(c->host_plan, cnt, 3 * sizeof(int), hipMemcpyDeviceToHost, s), "count D2H");
            hipcheck(c, hipStreamSynchronize(s), "count sync");
            n1 = c->host_plan[CNT_LAYERS];
            if (const int m = c->host_plan[CNT_LEADS]) {
                n1 += planes_redo_leads(c, prm, a, d, v, B, cv, NP, p0, n, m, need + p0, cnt, n1);
                sa.left = cv.left;
            }
            if (keep_leads) {
                const size_t row = z * NN;
                copy(lv.sigma + 2L * p0 * NN, cv.sigma, 2 * row * n);
                if (sa.left) copy(lv.left + (long)p0 * NN, cv.left, row * n);
                else
                    hipcheck(c, hipMemcpy2DAsync(lv.left + (long)p0 * NN, row, cv.sigma, 2 * row, row, n,
                                                 hipMemcpyDeviceToDevice, s), "copy leads");
                copy(lv.loss + 2L * p0, cv.loss, sizeof(LeadLoss) * 2 * n);
                copy(lv.dst + 2L * p0, cv.dst, sizeof(int) * 2 * n);
                copy(lv.dit + 2L * p0, cv.dit, sizeof(int) * 2 * n);
                copy(lv.need + p0, need + p0, sizeof(int) * n);
            }
            hipcheck(c, hipEventRecord(c->chk[0], s), "event check");
        }
        const double m = 16.0 * h.nt;
        launch(c, NT_K_PLANES, wait ? 2.0 * n * h.M * 5 * 8 * m * m * m : 0.0, "plane sweep", [&] {
            if (!wait || h.nt == 1) launch_sweep<1>(sa, 2 * n, s);
            if (!wait || h.nt == 2) launch_sweep<2>(sa, 2 * n, s);
            if (!wait || h.nt == 3) launch_sweep<3>(sa, 2 * n, s);
            if (!wait || h.nt == 4) launch_sweep<4>(sa, 2 * n, s);
            if (big) launch_sweep<PL_BIGNT>(sa, 2 * n, s);
            return hipGetLastError();
        });
        hipLaunchKernelGGL(k_pl_finish, dim3(nblk(n)), dim3(256), 0, s, n, cv.dst, cv.dit, cv.sst, cv.T, cv.loss,
                           cv.grow, adj ? PL_T_FLOOR_ADJ : PL_T_FLOOR, first, need + p0, cnt, a.T_LR + p0,
                           a.T_RL + p0, a.status ? a.status + p0 : nullptr, a.iters ? a.iters + p0 : nullptr);
        hipcheck(c, hipGetLastError(), "plane finish");
        if (adj) planes_adjoint(c, a, v, h, cv, pU, pL, pM, p0, n, hk, need + p0, kept, hi1);
        if (!wait) continue;
        // the points for the layers are known: they are solved beside the sweep, on
        // a worker context
        // (an adjoint solve of them adds to the same gradients: afterwards)
        const bool beside = !c->worker && !a.noalloc && !adj;
        if (n1 && beside) solve_left(c, prm, a, p0, n, need + p0, NEED_LAYERS, n1, true);
        hipcheck(c, hipMemcpyAsync(c->host_plan, cnt, CNT_N * sizeof(int), hipMemcpyDeviceToHost, s), "count D2H");
        hipcheck(c, hipStreamSynchronize(s), "count sync");
        left += n1 + c->host_plan[CNT_AFTER_SWEEP];
        later[0] += beside ? 0 : n1;
        later[1] += c->host_plan[CNT_AFTER_SWEEP];
    }
    if (keep_leads) *share = PlanesLeads{true, h.nt, h.m0, h.m1};
    const double steps = wait ? (double)c->host_plan[CNT_STEPS] : 0.0;
    // of a decimation step: the inverse of two planes and eight products of one
    if (c->prof && !big && !reuse) c->flops_pending[NT_K_PLANES] += steps * 16 * 8 * (16.0 * h.nt) * (16.0 * h.nt) * (16.0 * h.nt);
    // (the layers count theirs)
    if (prm->precision == NT_PREC_MIXED && wait && !adj) c->mixed_counts[0] += a.npts - (a.noalloc ? 0 : left);
    TdbArgs g = a;
    g.siblings.clear();
    g.no_planes = true;
    g.scratch_reserve = reserve;
    if (!wait || (a.noalloc && left)) {
        // every point whose need is set, masked inside the layers' kernels; in FP64,
        // as the mixed-precision kernels have no mask
        nt_params p64 = *prm;
        p64.precision = NT_PREC_FP64;
        g.mask = need;
        const PanelsOnly panels(c);
        solve_tdb_dev(c, &p64, g);
    } else {
        // (in c's own workspace, which the planes have no use for any more)
        for (int i = 0; i < 2; ++i)
            if (later[i]) solve_left(c, prm, a, 0, a.npts, need, i ? NEED_AFTER_SWEEP : NEED_LAYERS, later[i], false);
    }
    c->last_mean_iters = !wait ? -1.0 : left < a.npts ? steps / (2.0 * (a.npts - left)) : 0.0;
    return true;
}
