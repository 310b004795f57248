// The plane solver's argument blocks and host entry (nt_planes.hip).
#pragma once
#include "nt_solve.h"

struct PlanHdr {
    int ok;        // every layer falls into planes of one size class
    int nt;        // class: planes padded to 16 nt
    int M;         // planes of the whole system
    int m0, m1;    // planes of the left and right lead cell
};

// What tells how many digits a lead's decimation lost
struct LeadLoss {
    double mid;    // |G|max of the planes eliminated inside the cell, times scale
    double res;    // residual of the self-energy's own equation, over its largest element
    double scale;  // energy scale: largest of |E|, a cell's block and the cells' coupling
};

struct DecPlArgs {
    const PlanHdr* h;
    const int* psize;
    const double2 *H, *U, *Lw, *LV;
    const double* E;
    const int* kidx;
    double eta, eta0, conv;
    int eta_mode, max_iter;
    double2* scratch;      // DEC_SLOTS matrices per item
    double2* sigma;        // retarded self-energy per item (point, lead)
    int *status, *iters;
    LeadLoss* loss;
};

struct SweepPlArgs {
    const PlanHdr* h;
    const int* psize;
    const double2 *H, *U, *Lw;
    const unsigned long long* masks;       // per (k, plane): U's 4 x 16 and 16 x 4 pieces, Lw's
    const double* E;
    const int* kidx;
    double eta, eta0, dev_factor;
    int eta_mode;
    const int* need;       // points left out
    const double2* sigma;
    const double2* left;   // per point: the left lead's in the system's matrix (null: sigma's; redone leads)
    double* T;             // per item (point, direction)
    double* grow;          // |G|max of its planes
    int* status;
    // adjoint: G^L_j and (G^L_{0,j})^T of the planes from *keep_from on, two
    // matrices per plane, keep_stride matrices per point (null: not kept)
    double2* keep;
    const int* keep_from;
    long keep_stride;
};

struct AdjPlArgs {
    const PlanHdr* h;
    const int *psize, *player, *poff, *perm;
    const double2 *U, *Lw;
    const unsigned long long* masks;
    const double2 *sigma, *keep;
    long keep_stride;
    const int* kidx;
    const int *need, *status, *dstatus, *first;
    const double* w;
    const int* place;      // place of a point among the points of its chunk, by k
    int lo, hi1;           // window layers (device layers, 0-based), with the one after
    int b;
    long K;                // rows of the gathered row matrices: points of the chunk x NP
    double2 *CA, *RW;      // per window layer: b x K and K x b
};

// n worker contexts of c set up for a call (nt_workers.hip)
int prepare_workers(nt_ctx* c, int n);

// Decimation of Q leads (H00 of its own for every item) at the shifts z, as the
// layers' (nt_engine.hip): g = (z - es)^-1, sigma = V^+ g V; residual of item q
// (LeadLoss::res) to res[q * res_stride]; scratch from scratch_off of ar on.
size_t lead_sigma_scratch(int n, int Q);
void lead_sigma(nt_ctx* c, int n, int Q, BMat<double> H00, BMat<double> V, const double* z, double conv, int max_iter,
                BMatW<double> g, BMatW<double> sigma, int* status, int* iters, double* res, int res_stride, Arena& ar,
                size_t scratch_off);

// Self-energies of both leads of a's system on the layers, at the P points (E,
// kidx): sigma = V^+ g V, es = the cell with the self-energy that the recursion
// added up (item 2 p + lead, sigma_stride(a) elements apart, ld = the lead's
// size; the left ones advanced), statuses and step counts per item.
inline long sigma_stride(const TdbArgs& a)
{
    const long n = a.nl > a.nr ? a.nl : a.nr;
    return n * n;
}
size_t layers_sigma_scratch(const TdbArgs& a, int P);
void layers_sigma(nt_ctx* c, const nt_params* prm, const TdbArgs& a, int P, const double* E, const int* kidx,
                  double* sigma, double* es, int* status, int* iters, Arena& ar, size_t scratch_off);
