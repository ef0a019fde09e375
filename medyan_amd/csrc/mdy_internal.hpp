// mdy_internal.hpp -- device-side tables and the library context.
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

#include <string>
#include <vector>

#include "mdy.h"

namespace mdy {

constexpr int kNFF = MDY_NFF;
constexpr int kBlock = 256;          // threads per block, where a kernel has no size of its own
constexpr int kQueueCap = 4096;      // excluded-volume quadrature fallback queue
constexpr int kOneShot = 16;         // qn words of the one-shot calls: energy, force queue counts, two flags, ticket; zero between calls
// words of Ctx::h_out: host energies; queued force pairs; error word; rebuild totals from there on
constexpr int kOutForce = 16, kOutErr = 17, kOutSolve = 18, kOutNl = 24;
constexpr int kRed = 32;             // 8-byte words per block in a reduction record

// Interaction tables on the device. The evaluation index space is
// [EV | FS | FB | LM | BS | BB | BDH | BP | BD]: excluded volume first so its
// costly items are packed densely into the first waves of the grid.
// Force slots (3 doubles each) follow the reference force-field order
// FS, FB, LS, MS, BS, BB, EV, BD, so the per-bead gather adds contributions in
// the order ForceFieldManager::computeForces would.
struct Dev {
    int nb, ndof;
    int n_ev, n_fs, n_fb, n_lm, n_ls, n_bs, n_bb, n_bdh, n_bp, n_bd;
    const int4 *ev_bs; const double *ev_kr;   // monomer-sum form: ev_kr holds kvol * seg1 * seg2
    int ev_mon;                               // excluded volume as the monomer-pair sum
    int bdh_quad;                             // branching dihedral E = k theta^2 (else k (1 - cos theta))
    const int2 *ev_cyl;                       // monomer-sum form: the pair's cylinders
    const int4 *cyl_mon;                      // per cylinder: minus serial, plus serial, interval
    const int2 *fs_bs; const double *fs_k, *fs_l0;
    const int *fb_bs; const double *fb_k, *fb_th, *fb_ct, *fb_st;   // ct/st: cos/sin(theta0) from the host
    const int4 *lm_bs; const double *lm_k, *lm_l0, *lm_p1, *lm_p2;
    const int *bs_bs; const double *bs_k, *bs_l0, *bs_p;
    const int4 *bb_bs; const double *bb_k, *bb_th, *bb_ct, *bb_st;
    const int4 *bdh_bs; const double *bdh_k, *bdh_pos;           // branching dihedral
    const int *bp_bs; const double *bp_k, *bp_pos;               // branching position
    const int *bd_bead; const int *bd_plane; const double *bd_k, *bd_sl; const double *planes;
    int slot_fs, slot_fb, slot_lm, slot_bs, slot_bb, slot_bdh, slot_bp, slot_ev, slot_bd, n_slots;
    // bead -> its slots in slot order, as offsets 3 * slot in groups of four (the last one filled
    // up with 3 * n_slots): bead b's groups are row[b].x .. row[b].y - 1
    const int2 *row; const int4 *row_idx;
    int coplanar_mode;
    const unsigned char *evq;     // quadrature mode: per excluded-volume pair, 1 = evaluated by quadrature
    double cq, sq;                // cos and sin of pi/2 (C library), branching position
    // excluded-volume quadrature fallback queues (pair indices)
    int *qe, *qe_n;               // energy
    int *qf, *qf_n;               // force
    int *err;                     // sticky device error word (MDY_ERR_*)
    __host__ __device__ int n_items() const { return n_ev + n_fs + n_fb + n_lm + n_bs + n_bb + n_bdh + n_bp + n_bd; }
    // lanes of a sweep: two per excluded-volume pair of the integral form, one per other interaction
    __host__ __device__ int n_duo_lanes() const { return ev_mon ? 0 : 2 * n_ev; }
    __host__ __device__ int n_lanes() const { return n_items() + (ev_mon ? 0 : n_ev); }
};

template <class T>
struct DBuf {
    T *p = nullptr;
    size_t n = 0;
};

struct Ctx {
    int device = 0;
    hipStream_t stream = nullptr;
    mdy_opts opts{};
    std::string msg;
    int num_cu = 0;
    // system
    bool have_sys = false, have_nl = false;
    int nb = 0;
    int ncyl = 0;
    // host copies needed for rebuilds
    std::vector<int> h_static_counts;
    // device tables (static part)
    DBuf<int2> fs_bs; DBuf<double> fs_k, fs_l0;
    DBuf<int> fb_bs; DBuf<double> fb_k, fb_th, fb_ct, fb_st;
    DBuf<int4> lm_bs; DBuf<double> lm_k, lm_l0, lm_p1, lm_p2;
    DBuf<int> bs_bs; DBuf<double> bs_k, bs_l0, bs_p;
    DBuf<int4> bb_bs; DBuf<double> bb_k, bb_th, bb_ct, bb_st;
    DBuf<int4> bdh_bs; DBuf<double> bdh_k, bdh_pos;
    DBuf<int> bp_bs; DBuf<double> bp_k, bp_pos;
    DBuf<int> st_off, st_idx;   // bead -> bonded / cross-link slots
    int n_fs = 0, n_fb = 0, n_ls = 0, n_ms = 0, n_bs = 0, n_bb = 0, n_bdh = 0, n_bp = 0;
    // cylinders
    DBuf<int> c_b1, c_b2, c_fil, c_pos, c_child; DBuf<long long> c_id; DBuf<short> c_type;
    DBuf<double> c_eq, c_ek; DBuf<unsigned char> c_minus, c_plus;   // c_plus: last cylinder of its filament
    int ev_mon = 0;                // monomer-sum excluded volume
    int bdh_quad = 0;              // quadratic branching dihedral
    DBuf<int4> c_mon;              // minus serial, plus serial, interval, 0
    DBuf<double> c_seg;            // interval * monomer size
    float ev_cut = 0, bd_cut = 0;
    int ev_on = 0, bd_on = 0;
    int n_planes = 0;
    DBuf<double> planes, plane_k, plane_sl;
    // neighbor-list work
    DBuf<double> mid;       // 3 * ncyl: midpoints
    DBuf<int> cell_cnt, cell_rank, near; DBuf<int2> cell_range; DBuf<int4> cell_list;
    DBuf<unsigned long long> row_cnt, row_off;   // per cylinder: pairs << 32 | kept pairs
    DBuf<int> pairs, pair_tmp;    // 2 * npairs (NL, before mother-daughter filtering); npairs
    long long n_pairs = 0;
    DBuf<int4> ev_bs; DBuf<double> ev_kr; int n_ev = 0;
    DBuf<int2> ev_cyl;            // monomer-sum form: cylinders of each pair
    DBuf<int> bd_flag, bd_off, bd_bead, bd_plane; DBuf<double> bd_k, bd_sl; int n_bd = 0;
    std::vector<int> h_bd_nneigh;
    DBuf<int> row_cur; DBuf<int2> row; DBuf<int4> row_idx, row_tmp;   // bead -> all slots (Dev::row_idx)
    int n_static = 0;             // entries of st_idx
    DBuf<unsigned char> evq;      // quadrature mode: per-pair flags of the current evaluation
    DBuf<int> qpan, qcnt, qoff, qmap; // quadrature mode: panels, record counts, first records, record -> pair
    DBuf<unsigned long long> qtot;    // quadrature mode: running record totals (zero between calls)
    DBuf<double> qpart, qpe;      // quadrature mode: records, per-pair values
    DBuf<int> scan_tmp;
    // evaluation scratch
    DBuf<double> x, xt, f, contrib;
    DBuf<double> red;             // per-block partials
    DBuf<double> out;             // small results
    DBuf<int> qe, qf, qn, err;    // qn: 16 words of the minimizer's phases, 16 of the one-shot calls (kOneShot)
    long long *h_out = nullptr;   // pinned: what a call's last kernel tells the host
    size_t h_out_n = 0;
    DBuf<double> qe_u, simpson_part;
    DBuf<double> solve;           // linear solve: its scalars, block sums of p.Hp and of r.r
    // CG state
    DBuf<double> F0, F1, S0, S1, xmin;
    DBuf<unsigned long long> bar, acc;
    DBuf<double> cg_out;          // result block
    DBuf<double> tr_lam, tr_e, tr_mf, tr_beta; DBuf<int> tr_safe;
    long long trace_cap = 0, trace_n = 0;
    DBuf<long long> prof; DBuf<int> prof_kind; long long prof_cap = 0, prof_n = 0;
    DBuf<unsigned char> batch_args;  // batched launch: per-network kernel arguments
    DBuf<int2> batch_map;            // batched launch: (network, block within its cluster)
    DBuf<int> batch_done;            // batched launch: finished minimizations (passes by completions)
    double last_ms = 0;
    // the last minimization's search direction (CGMethod::searchDir): the CG
    // buffer that holds it (0 F0, 1 F1, 2 S0, 3 S1) or, when its final update
    // s = F + beta d is still pending, the current force buffer, d and beta
    bool have_dir = false, dir_pend = false;
    int dir_buf = -1, dir_cur = 0, dir_prev = -1;
    double dir_beta = 0;
    int coop_blocks = 0, coop_threads = 0;   // the last minimization's grid
    Dev dev() const;
};

}  // namespace mdy
