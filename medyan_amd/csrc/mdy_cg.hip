// mdy_cg.hip -- CGMethod::minimize<method> with the backtracking or the
// quadratic line search, resident on the device for the whole minimization
// (src/Mechanics/Minimizer/CGMethod.hpp:238-373, 522-765, 826-1743;
// CGMethod.cpp:43-360).
//
// One cooperative launch; every block runs the same control flow and derives
// every decision from grid reductions that all blocks evaluate in the same
// fixed order (exact sums), so decisions are identical without a broadcast.
// Phases are separated by a grid barrier.
//
// Every line-search trial evaluates energy AND force slots at the trial point,
// so an accepted trial needs no second pass over the interactions. An
// accepted iteration costs two barriers:
//   [gather F at the accepted point, x += lam*d, max|F|, F.F, F.Fprev]
//   | [beta, s = F + beta*d, s.F, energy+forces at x + lam0*s (the next
//      line search's first trial)]
// The energy at the accepted point is the trial energy of the same
// coordinates (bitwise), so E(x) is never recomputed.
#include "mdy_eval.hpp"
#include "mdy_launch.hpp"

#include <algorithm>
#include <cstring>
#include <utility>
#include <vector>

namespace mdy {

struct CgArgs {
    Dev D;
    double *x, *F0, *F1, *S0, *S1, *xmin, *contrib;
    double *red;          // 3 * nblk * kRed
    double *qe_u;         // 3 * kQueueCap
    double *spart;        // 6 * nblk * kRed
    int *qe, *qf, *qn;    // 3 * kQueueCap each; qn: 3 x 4 counters
    unsigned long long *bar;  // [0] abort flag, [16] arrivals
    unsigned long long *acc;  // 3 x kAccWords phase accumulators
    double *out;          // result record
    long long *prof;      // phase profile, 5 words per phase: barrier exit (block 0), latest
                          // arrival (all blocks), block 0's work start, end of its item
                          // loop, and its arrival
    int *prof_kind;       // phase kind code
    long long prof_cap;
    double *tr_lam, *tr_e, *tr_mf, *tr_beta;
    int *tr_safe;
    long long tr_cap;
    // parameters
    int method, line_search, try_recover, energy_call_limit, force_call_limit, report_call_limit;
    double max_dist, lambda_max, grad_tol, energy_rel_tol;
    long long spin_limit;
    int grid;             // blocks of this minimization's cluster (batched launch)
    // batched passes: suspend at the top of an iteration once this many force
    // calls are done (0: never), and resume from the state a suspension saved
    int suspend_calls, resume;
    int other;            // blocks of the launch that takes over from this one; 0: none
    int poll_sleep;       // barrier: 128-clock sleeps between two polls
};

// result record layout (doubles)
enum {
    R_EB = 0,              // energies before [kNFF] + total
    R_EA = R_EB + kNFF + 1,  // energies after
    R_FLAGS = R_EA + kNFF + 1,
    R_NEC, R_NFC, R_NIT, R_GIN, R_ERC, R_NEE, R_NSM, R_NREC, R_STATUS, R_TRN, R_LAST, R_FOUT, R_NPH,
    R_T0, R_T1,            // 100 MHz wall clock at the leader's start and end
    R_DIR, R_PEND, R_BETA, R_DPREV,   // search direction at the end (buffer ids 0 F0, 1 F1, 2 S0, 3 S1)
    R_SUSP,                // 1: the run suspended and resumes in another launch; kWants: on more blocks
    R_RS                   // the CgState a suspension saves
};

__device__ __forceinline__ int ld_i(const int *p) { return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT); }

// phase accumulator sets: 3 rotating sets of kAccWords 64-bit words
constexpr int kAccWords = 32;
constexpr int kAcc0 = 0, kAcc1 = 8, kAccMax = 16, kAccDone = 19;

// phase kinds recorded by the profile
enum { PK_ENERGY = 1, PK_EFALLBACK, PK_EVAL, PK_FFALLBACK, PK_GATHER, PK_REDUCE, PK_RESTORE };

template <bool MIXED>
struct Cg {
    using Slot = typename SlotT<MIXED>::T;   // force records: double, or float in the mixed form
    const CgArgs &A;
    double *lds;
    XBlock &xb;                  // the block's exact sums of the current phase
    unsigned long long *accl;    // LDS copy of the words a phase's decisions read
    int G, blk, tid, gtid, gs;
    int ph = 0;                  // phase counter (uniform)
    // batched passes by completions: the launch's count of finished
    // minimizations (nullable)
    int *done_ctr = nullptr;
    int status = MDY_OK;         // set by a collective step, the same in every thread
    bool leave = false;          // likewise: the launch ends, to be taken up by one of more blocks

    // blk: this block's index within the cluster of G blocks that runs the
    // minimization (the whole grid, or one network's share of a batch)
    __device__ Cg(const CgArgs &a, double *l, XBlock &x, unsigned long long *al, int blk_, int G_)
        : A(a), lds(l), xb(x), accl(al) {
        G = G_; blk = blk_; tid = threadIdx.x;
        gtid = blk * blockDim.x + tid; gs = G * blockDim.x;
    }
    __device__ long long *ldsl() const { return reinterpret_cast<long long *>(lds); }
    __device__ Slot *slots() const { return reinterpret_cast<Slot *>(A.contrib); }
    __device__ Dev dv(int b) const {
        Dev d = A.D;
        d.qe = A.qe + b * kQueueCap; d.qe_n = A.qn + 4 * b;
        d.qf = A.qf + b * kQueueCap; d.qf_n = A.qn + 4 * b + 1;
        return d;
    }
    __device__ double *red(int p) const { return A.red + (size_t)(p % 3) * G * kRed; }
    __device__ double *qeu(int b) const { return A.qe_u + (size_t)b * kQueueCap; }

    // Grid barrier, run by the block's first wave. Arrival: one agent-scope
    // release, then one added to the cluster's count. Departure: lane 0 polls the
    // count until every block has arrived in this phase, then one agent-scope
    // acquire. A watchdog on the poll sets the shared abort flag; every waiting
    // block sees it and leaves. Returns false on abort. The block's other waves
    // wait at a __syncthreads.
    __attribute__((always_inline)) __device__ bool barrier(int kind) {
        const unsigned long long target = (unsigned long long)(ph + 1) * (unsigned long long)G;
        unsigned long long *count = A.bar + 16;
        if (tid == 0 && ph < A.prof_cap) {
            const unsigned long long t = wall_clock64();
            atomicMax(reinterpret_cast<unsigned long long *>(A.prof) + 5 * (size_t)ph + 1, t);
            if (blk == 0) A.prof[5 * (size_t)ph + 4] = (long long)t;
        }
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "agent");
        bool ab = false;
        if (tid == 0) {
            __hip_atomic_fetch_add(count, 1ull, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            long long spins = 0;
            while (__hip_atomic_load(count, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) < target) {
                for (int q = 0; q < A.poll_sleep; q++) __builtin_amdgcn_s_sleep(2);
                if (__builtin_expect((++spins & 255) == 0, 0)) {
                    if (__hip_atomic_load(A.bar, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT)) { ab = true; break; }
                    if (spins > A.spin_limit) {
                        __hip_atomic_store(A.bar, 1ull, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                        ab = true;
                        break;
                    }
                }
            }
        }
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "agent");
        if (blk == 0 && tid == 0 && ph < A.prof_cap) {
            A.prof[5 * (size_t)ph] = wall_clock64();
            A.prof_kind[ph] = kind;
        }
        // recycle the queue counters of phase ph + 2: last written two phases ago,
        // read by every block before the barrier just passed
        if (blk == 0 && tid < 4) A.qn[4 * ((ph + 2) % 3) + tid] = 0;
        // and the accumulator set of that phase (read by every block right
        // after its barrier, which every block has since left)
        if (blk == 0 && tid < kAccWords)
            __hip_atomic_store(A.acc + (size_t)((ph + 2) % 3) * kAccWords + tid, 0ull, __ATOMIC_RELAXED,
                               __HIP_MEMORY_SCOPE_AGENT);
        return __ballot(ab) == 0;
    }
    // a whole block's barrier: what it wrote before is visible to every block after
    __attribute__((always_inline)) __device__ bool sync(int kind) {
        __shared__ int s_ok;
        __builtin_amdgcn_s_waitcnt(0);
        __syncthreads();
        if (tid < 64) {
            const bool ok = barrier(kind);
            if (tid == 0) s_ok = ok ? 1 : 0;
        }
        ph++;
        __syncthreads();
        return s_ok != 0;
    }

    // profile marks of block 0 inside a phase: 0 = work start, 1 = end of the main loop
    __device__ void mark(int i) const {
        if (blk == 0 && tid == 0 && ph < A.prof_cap) A.prof[5 * (size_t)ph + 2 + i] = wall_clock64();
    }

    // ---- phase accumulators. Every exact sum a decision needs (energy, s.F,
    // F.F, F.Fprev) is reduced per block, then added digit by digit with
    // 64-bit integer atomics into one of three rotating sets (phase % 3):
    // integer addition is associative, so the total is independent of the
    // arrival order and every block reads the same bits right after the
    // barrier. Max |F| uses an integer max on the bit pattern (values >= 0).
    // A set is read right after its phase's barrier and zeroed by block 0 one
    // barrier later.
    __device__ unsigned long long *accs(int p) const { return A.acc + (size_t)(p % 3) * kAccWords; }
    // the block's sums and maximum into the set of phase p (after a __syncthreads)
    __attribute__((always_inline)) __device__ void acc_push(int p) const {
        const unsigned long long v = xblock_take(xb);
        if (tid < 17 && v != 0) {
            unsigned long long *w = accs(p) + tid;
            if (tid == kAccMax) atomicMax(w, v);
            else if ((tid & 7) == 7) atomicOr(w, v);
            else atomicAdd(w, v);
        }
    }
    // After a barrier the first wave loads the words its decisions read into LDS.
    // extra0..2 (nullable): counters loaded into words 17 to 19. Lane t < 2 returns
    // the value of sum t.
    __attribute__((always_inline)) __device__ double acc_fetch(int p, const int *extra0, const int *extra1) const {
        const unsigned long long *base = accs(p);
        if (tid < 17 || tid == kAccDone)
            accl[tid] = __hip_atomic_load(base + tid, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        else if (tid == 17 && extra0) accl[17] = (unsigned long long)(unsigned)ld_i(extra0);
        else if (tid == 18 && extra1) accl[18] = (unsigned long long)(unsigned)ld_i(extra1);
        __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "workgroup");   // LDS of one wave: in order
        __builtin_amdgcn_wave_barrier();
        if (tid >= 2) return 0.0;
        const mdy_xsum X = acc_local(8 * tid);
        return mdy_xs_value(&X);
    }
    __attribute__((always_inline)) __device__ mdy_xsum acc_local(int off) const {
        mdy_xsum X;
#pragma unroll
        for (int k = 0; k < MDY_XS_N; k++) X.d[k] = (long long)accl[off + k];
        X.flags = (int)accl[off + 7];
        X.cnt = 0;
        return X;
    }
    __attribute__((always_inline)) __device__ mdy_xsum acc_read(const unsigned long long *base) const {
        mdy_xsum X;
#pragma unroll
        for (int k = 0; k < MDY_XS_N; k++)
            X.d[k] = (long long)__hip_atomic_load(base + k, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        X.flags = (int)__hip_atomic_load(base + 7, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        X.cnt = 0;
        return X;
    }

    // ---- quadrature fallback energies of the pairs queued in buffer qb, one
    // block per pair (CylinderExclVolRepulsion.cpp:884-999, 442-481)
    __attribute__((always_inline)) __device__ bool energy_fallback(const PosAny &pos, const Dev &d, int nqe, int qb) {
        const int N = 400;
        for (int q = blk; q < nqe; q += G) {
            const int i = ld_i(d.qe + q);
            int4 b = d.ev_bs[i];
            SimpsonGeo g = simpson_geo(pos(b.x), pos(b.y), pos(b.z), pos(b.w));
            mdy_xsum Y;
            mdy_xs_zero(&Y);
            if (tid == 0) mdy_xs_add(&Y, simpson_e_corners(g));
            for (int node = tid; node < (N + 1) * (N + 1); node += blockDim.x)
                simpson_e_node(g, node / (N + 1), node % (N + 1), N, Y);
            block_reduce_xsum(Y, ldsl());
            if (tid == 0) {
                const double ds = 1.0 / ((double)N);
                qeu(qb)[q] = d.ev_kr[i] * (ds * ds / 9.0) * mdy_xs_value(&Y);
            }
        }
        return sync(PK_EFALLBACK);
    }

    // ---- hot loop: all interactions at `pos`, energy (the block's first sum)
    // and force slots
    __attribute__((always_inline)) __device__ void eval(const PosAny &pos) {
        const Dev d = dv(ph % 3);
        mark(0);
        sweep<MIXED, false>(d, pos, blk, G, nullptr, &xb, slots(), false, true);
        mark(1);
    }

    // ---- computeIndividualEnergies at x (energies only, per force field):
    // out[0..7] per force field, out[8] their sum; returns the computeEnergy
    // total (+inf sentinel) in E and the plain total in Eplain.
    __attribute__((always_inline)) __device__ bool eval_ff(const PosAny &pos, double *out, double &E, double &Eplain) {
        const int p0 = ph, qb = p0 % 3;
        Dev d = dv(qb);
        double acc[kNFF];
#pragma unroll
        for (int k = 0; k < kNFF; k++) acc[k] = 0.0;
        sweep<MIXED, false>(d, pos, blk, G, acc, &xb, nullptr, true, false);
        double *r = red(p0);
        block_reduce<kNFF>(acc, lds);
        if (tid < kNFF) r[(size_t)blk * kRed + tid] = acc[tid];
        acc_push(p0);
        if (!sync(PK_ENERGY)) return false;
        mdy_xsum X = acc_read(accs(p0) + kAcc0);
        const int nqe = ld_i(d.qe_n);
        if (nqe > kQueueCap) {
            status = MDY_ERR_CAPACITY;
            return true;
        }
        if (nqe > G && A.other > G) {   // the larger grid repeats this evaluation
            leave = true;
            return true;
        }
        if (__builtin_expect(nqe > 0, 0) && !energy_fallback(pos, d, nqe, qb)) return false;
        double v[kNFF], e[kNFF + 2];
        grid_partials_reduce<kNFF>(r, G, v, lds);
        energy_finish(X, v, nqe, d.qe, qeu(qb), e);
        if (blk == 0 && tid == 0) {
            for (int k = 0; k < kNFF; k++) out[k] = e[k];
            out[kNFF] = e[kNFF + 1];
        }
        E = e[kNFF];
        Eplain = e[kNFF + 1];
        return true;
    }

    // ---- quadrature forces for the pairs an accepted evaluation queued
    // (CylinderExclVolRepulsion.cpp:1001-1254, 1017-1022 retry with the first
    // cylinder moved off the plane). The slots are written by block 0.
    __attribute__((always_inline)) __device__ bool force_fallback(const PosAny &pos, int nqf, int qb) {
        const int *qf = A.qf + qb * kQueueCap;
        for (int q = 0; q < nqf; q++) {
            const int i = ld_i(qf + q);
            int4 b = A.D.ev_bs[i];
            bool done = false;
            for (int moved = 0; moved < 2 && !done; moved++) {
                d3 c1 = pos(b.x), c2 = pos(b.y), c3 = pos(b.z), c4 = pos(b.w);
                const bool inplane = are_in_plane(c1, c2, c3, c4);
                if (moved) {
                    d3 n2 = moved_off_plane(c1, c2, c3, c2, 0.01), n1 = moved_off_plane(c1, c2, c3, c1, 0.01);
                    c1 = n1; c2 = n2;
                }
                SimpsonGeo g = simpson_geo(c1, c2, c3, c4);
                const int N = 10000;
                const long long nodes = (long long)(N + 1) * (N + 1);
                for (int comp = 0; comp < 6; comp++) {
                    mdy_xsum X;
                    mdy_xs_zero(&X);
                    if (gtid == 0) simpson_f_corners(g, comp, X);
                    for (long long nd = gtid; nd < nodes; nd += gs)
                        simpson_f_node(g, (int)(nd / (N + 1)), (int)(nd % (N + 1)), N, comp, X);
                    block_reduce_xsum(X, ldsl());
                    if (tid == 0) store_xsum(A.spart + (size_t)comp * G * kRed, blk, 0, X);
                }
                if (!sync(PK_FFALLBACK)) return false;
                double T0 = 0, T1 = 0, T2 = 0, T3 = 0, T4 = 0, T5 = 0;
#pragma clang loop unroll(disable)
                for (int comp = 0; comp < 6; comp++) {
                    mdy_xsum X;
                    grid_reduce_xsum(A.spart + (size_t)comp * G * kRed, G, 0, X, ldsl());
                    const double t = mdy_xs_value(&X);
                    T0 = comp == 0 ? t : T0; T1 = comp == 1 ? t : T1; T2 = comp == 2 ? t : T2;
                    T3 = comp == 3 ? t : T3; T4 = comp == 4 ? t : T4; T5 = comp == 5 ? t : T5;
                }
                const double T[6] = {T0, T1, T2, T3, T4, T5};
                d3 f[4];
                simpson_f_assemble(g, T, A.D.ev_kr[i], N, f);
                const bool ok = finite_d3(f[0]) && finite_d3(f[1]) && finite_d3(f[2]) && finite_d3(f[3]);
                if (ok) {
                    if (blk == 0 && tid == 0) {
                        int s = A.D.slot_ev + 4 * i;
                        put3(slots(), s, f[0]); put3(slots(), s + 1, f[1]);
                        put3(slots(), s + 2, f[2]); put3(slots(), s + 3, f[3]);
                    }
                    done = true;
                } else if (moved || !inplane) {
                    status = MDY_ERR_FORCE;   // the reference exits here
                    return true;
                }
                if (!sync(PK_FFALLBACK)) return false;   // spart reuse / slot visibility
            }
        }
        return true;
    }

    // ---- forces from the slots into Fout, one lane per coordinate; x += lam*d
    // when `move`. The block's sums: F.F and F.Fprev (Fprev may be null), and max|F_i|.
    template <bool BATCH>
    __attribute__((always_inline)) __device__ void gather(double *Fout, const double *Fprev, bool move,
                                                          const double *dvec, double lam) {
        const int ndof = A.D.ndof;
        double m = 0.0;
        mark(0);
        int turn = 0;
        for (int base = blk * blockDim.x; base < ndof; base += gs) {
            if (turn == kXTurns) { xblock_norm(xb); turn = 0; }
            turn++;
            const int o = base + tid;
            if (o < ndof) {
                const double f = gather_coord(A.D, slots(), o);
                Fout[o] = f;
                m = fmax(m, fabs(f));
                XAdd{&xb, 0}(f * f);
                if (Fprev) XAdd{&xb, 8}(f * Fprev[o]);
                if (move) A.x[o] = A.x[o] + lam * dvec[o];
            }
            if (ndof - base <= gs) break;
        }
        xblock_max(xb, m);
        mark(1);
        // the cluster's blocks all read the launch's completion count as one
        // block saw it, through this phase's accumulators
        if (BATCH && done_ctr && blk == 0 && tid == 0)
            atomicMax(accs(ph) + kAccDone, (unsigned long long)(unsigned)ld_i(done_ctr));
    }
};

// s = F + beta * d for every coordinate into Sn, and s.F into the block's
// second sum (reduced with the phase's energy, or on its own without a trial)
template <bool MIXED>
__device__ __attribute__((always_inline)) void spec_direction(Cg<MIXED> &K, const double *Fn, const double *dprev,
                                                              double beta, double *Sn) {
    int turn = 0;
    for (int base = K.blk * blockDim.x; base < K.A.D.ndof; base += K.gs) {
        if (turn == kXTurns) { xblock_norm(K.xb); turn = 0; }
        turn++;
        const int o = base + K.tid;
        if (o < K.A.D.ndof) {
            const double f = Fn[o], s = f + beta * dprev[o];
            Sn[o] = s;
            XAdd{&K.xb, 8}(s * f);
        }
        if (K.A.D.ndof - base <= K.gs) break;
    }
}

// The minimizer as a state machine: every turn performs one kind of device
// work (each with a single call site, so each is inlined once), and one thread
// of every block then advances the CGMethod::minimize control flow
// (CGMethod.hpp:826-1743, backtrackingLineSearch CGMethod.cpp:43-360) from the
// reduced sums, which are the same bits in every block. Its state and the next
// work's operands are in LDS: held in registers by every thread, as the same
// value 64 times per wave, they left room for one wave per SIMD.
// The first trial of a line search that follows an accepted step is taken
// along s = F + beta*d while s itself is formed in the same phase; if s.F <= 0
// (resetCGParams) that trial is discarded and redone along F.
constexpr int kWants = 1 << 20;   // in a batch's count of finished networks: above all counts
constexpr int kQuiet = 16;   // force calls without a fallback after which the larger grid hands back (run_minimize)
enum Op { OP_NONE, OP_EVAL_FF, OP_EVAL, OP_EFALLBACK, OP_GATHER, OP_MINSTEP, OP_SDONLY, OP_RESTORE, OP_EXIT };
enum Stage {
    ST_INIT_FF, ST_INIT_F, ST_INIT_G, ST_ITER, ST_TRIAL, ST_SD, ST_QUAD, ST_QUAD_EVAL, ST_QUAD_DONE, ST_QUAD_AT,
    ST_LS_DONE, ST_ACCEPT, ST_REC_STEP, ST_REC_EVAL, ST_REC_GATHER, ST_FINAL, ST_FINAL_DONE, ST_FINISH
};

// vectors by number: 0 F0, 1 F1, 2 S0, 3 S1, -1 none
struct CgState {
    // the next device work: its kind and positions (PosAny along vector d, or
    // F + beta d), the gather's output and previous force, the new direction
    int op, mode, pd, pF, gOut, gPrev, gMove, sNew, ffAfter, saveMin;
    int nqe, nqf, qb;           // fallback queues of the last evaluation
    double plam, pbeta;
    // results of collective work
    double Eff, Effp, stepRec;
    // control
    int stage, status, cur, sidx, dv, dprev, safeMode, haveMin, pendingSpec, after, suspended, quadLS;
    unsigned flags;
    int susp;                   // force calls at which an iteration suspends
    int nEC, nFC, nIter, nEE, nSM, nRec, doneSeen;
    long long trn;
    double gradInf, relE, maxF, FF, FFp, FFcur, E, xa, E0, prevEnergy, lastFDotF, slope, minimumE, lam, newE, armijo,
        reducedSlope, sdF, beta, lamEval, Eacc;
    // quadratic line search (quadraticLineSearchV2): trial count, the last
    // rejected trial, the first record, the highest later record, the
    // parabola's bracket, its refinement count, and the last evaluated step
    int qIter, qRef;
    double qPrevL, qPrevE, qL0, qE0, qMax, qBt, qx0, qx1, qx2, qy0, qy1, qy2, qLam;

    __device__ void at_x() { mode = PosAny::X; pd = pF = -1; plam = pbeta = 0.0; }
    __device__ void line(int d, double l) { mode = PosAny::LINE; pd = d; pF = -1; plam = l; pbeta = 0.0; }
    __device__ void spec(int F, int d, double b, double l) { mode = PosAny::SPEC; pd = d; pF = F; plam = l; pbeta = b; }
    __device__ void eval_line(int d, double l, int st) { op = OP_EVAL; line(d, l); stage = st; }
    __device__ void gather_step(int st) {
        op = OP_GATHER;
        gOut = 1 - cur; gPrev = cur; gMove = 1;
        stage = st;
    }
    __device__ void reset() { dv = cur; lastFDotF = FFcur; slope = FFcur; }   // resetCGParams
    __device__ void stop(int code) { status = code; after = 0; stage = ST_FINISH; }
    // This launch ends; another one takes up the work next_op and then next_stage. Everything the
    // minimization carries on is saved here or in the network's buffers (x, forces, directions,
    // minimum-energy backup, trace). The phase counter restarts at 0 with cleared accumulators,
    // which changes no value.
    __device__ void suspend(double *R, bool leader, int next_op, int next_stage, int why = 1) {
        op = next_op; stage = next_stage;
        doneSeen = 0;
        if (leader) {
            *reinterpret_cast<CgState *>(R + R_RS) = *this;
            R[R_SUSP] = why;
        }
        suspended = why;
        after = 0;
        op = OP_NONE;
        stage = ST_FINISH;
    }
};
constexpr int R_SIZE = R_RS + (int)((sizeof(CgState) + sizeof(double) - 1) / sizeof(double));

// One block's thread 0: the control flow from the work just done to the next
// (s.op). Returns nothing; s.op = OP_EXIT at the end.
template <bool QUAD, bool BATCH>
__device__ __attribute__((always_inline)) void cg_control(CgState &s, const CgArgs &A, bool leader, int suspend_done) {
    double *R = A.out;
    auto callLimit = [&]() {
        return (A.energy_call_limit != 0 && s.nEC > A.energy_call_limit) ||
               (A.force_call_limit != 0 && s.nFC > A.force_call_limit);
    };
    auto converged = [&]() { return s.gradInf < A.grad_tol || s.relE < A.energy_rel_tol; };
    auto trace = [&](double l, double e, double b) {
        if (leader && s.trn < A.tr_cap) {
            A.tr_lam[s.trn] = l; A.tr_e[s.trn] = e; A.tr_mf[s.trn] = s.gradInf; A.tr_beta[s.trn] = b;
            A.tr_safe[s.trn] = s.safeMode;
        }
        s.trn++;
    };
    s.op = OP_NONE;
    if (__builtin_expect(s.status != 0, 0) && s.stage != ST_FINISH) { s.after = 0; s.stage = ST_FINISH; }
    while (s.op == OP_NONE) {
        switch (s.stage) {
        case ST_INIT_FF:   // energiesBefore = computeIndividualEnergies(x); E(x) for the first line search
            s.nEC++; s.nEE++;
            s.E0 = s.Eff; s.prevEnergy = s.Effp;
            s.op = OP_EVAL; s.at_x(); s.stage = ST_INIT_F;
            break;
        case ST_INIT_F:    // forces at x
            s.op = OP_GATHER; s.gOut = s.cur; s.gPrev = -1; s.gMove = 0; s.stage = ST_INIT_G;
            break;
        case ST_INIT_G:
            s.nFC++;
            s.gradInf = s.maxF;
            if (__builtin_expect(!isfinite(s.gradInf), 0)) { s.stop(MDY_ERR_NONFINITE); break; }
            s.FFcur = s.FF;
            s.reset();
            s.stage = ST_ITER;
            break;
        case ST_ITER:
            if (callLimit() || converged()) {
                if (callLimit() && s.haveMin && A.report_call_limit) s.op = OP_RESTORE;
                s.stage = ST_FINAL;
                break;
            }
            if (s.nFC >= s.susp || (BATCH && suspend_done > 0 && s.doneSeen >= suspend_done)) {
                s.suspend(R, leader, OP_NONE, ST_ITER);
                break;
            }
            s.nIter++;
            s.armijo = s.safeMode ? 0.0 : 0.4;
            s.quadLS = QUAD && A.line_search == MDY_LS_QUADRATIC && !s.safeMode;
            s.qIter = 0;
            s.qMax = -INFINITY;
            s.lam = 0.0; s.newE = 0.0;
            if (s.maxF != 0.0) {
                s.lam = smin(A.lambda_max, A.max_dist / s.maxF);
                s.nEC++;   // currentEnergy = computeEnergy(x): E0, known bitwise from the accepting trial
                s.op = OP_EVAL;
                if (s.pendingSpec) s.spec(s.cur, s.dprev, s.beta, s.lam);
                else s.line(s.dv, s.lam);
                s.reducedSlope = s.armijo * s.slope;
                s.stage = ST_TRIAL;
            } else if (s.pendingSpec) {
                s.op = OP_SDONLY; s.spec(s.cur, s.dprev, s.beta, 0.0); s.stage = ST_SD;
            } else {
                s.stage = ST_LS_DONE;
            }
            break;
        case ST_SD:        // s.F without a trial (max|F| = 0)
            s.pendingSpec = 0;
            s.sdF = s.xa;
            if (s.sdF <= 0) s.reset();
            else { s.dv = s.sNew; s.slope = s.sdF; }
            s.stage = ST_LS_DONE;
            break;
        case ST_TRIAL: {   // one backtracking step
            if (s.mode == PosAny::SPEC) {
                s.pendingSpec = 0;
                s.sdF = s.xa;
                if (s.sdF <= 0) {   // resetCGParams: redo this trial along F
                    s.reset();
                    s.reducedSlope = s.armijo * s.slope;
                    s.eval_line(s.dv, s.lam, ST_TRIAL);
                    break;
                }
                s.dv = s.sNew; s.slope = s.sdF;
                s.reducedSlope = s.armijo * s.slope;
            }
            double Et = s.E;
            s.nEC++;
            if (QUAD && s.quadLS) {   // CGMethod.hpp:567-617: Armijo slope 0.4, every trial recorded
                s.lamEval = s.lam; s.Eacc = Et;
                s.qIter++;
                const double idealq = -0.4 * s.lam * s.slope;
                if (idealq > 0) { s.stop(MDY_ERR_QUADRATIC); break; }
                bool conv = false;
                if (Et - s.E0 <= idealq) conv = true;
                else { s.qPrevL = s.lam; s.qPrevE = Et; s.lam *= 0.5; }
                double recL, recE;
                if (s.lam <= 0.0 || s.lam <= 1e-8) { conv = true; s.lam = 0.0; recL = 0.0; recE = s.E0; }
                else if (conv) { recL = s.lam; recE = Et; }
                else { recL = s.qPrevL; recE = s.qPrevE; }
                if (s.qIter == 1) { s.qL0 = recL; s.qE0 = recE; }
                else s.qMax = fmax(s.qMax, recE);
                if (!conv) { s.eval_line(s.dv, s.lam, ST_TRIAL); break; }
                s.newE = Et;
                // CGMethod.hpp:621-645: refine when an earlier record lies above
                // the accepted energy; the third point is the first record
                if (s.lam > 0.0 && s.qIter > 1 && Et < s.E0 && Et < s.qMax) {
                    s.qx0 = 0.0; s.qx1 = s.lam; s.qx2 = s.qL0; s.qy0 = s.E0; s.qy1 = Et; s.qy2 = s.qE0;
                    s.qBt = s.lam; s.qRef = 0;
                    s.stage = ST_QUAD;
                } else {
                    s.stage = ST_LS_DONE;
                }
                break;
            }
            const double ideal = -s.reducedSlope * s.lam;
            bool done = false;
            if (s.lam < 0 || ideal > 0) { done = true; s.lam = 0.0; }
            const double change = Et - s.E0;
            if (change <= ideal) done = true;
            else s.lam *= 0.5;
            if (s.lam <= 0.0 || s.lam <= 1e-8) { done = true; s.lam = 0.0; Et = s.E0; }
            if (!done) { s.eval_line(s.dv, s.lam, ST_TRIAL); break; }
            s.newE = Et;
            s.stage = ST_LS_DONE;
            break;
        }
        case ST_QUAD: {   // quadraticoptimization, CGMethod.hpp:663-765 (at most 200 refinements)
            if constexpr (!QUAD) break;
            if (s.qRef >= 200) { s.qLam = s.qx1; s.stage = ST_QUAD_DONE; break; }
            s.qRef++;
            const double d = (s.qx0 - s.qx1) * (s.qx0 - s.qx2) * (s.qx1 - s.qx2);
            const double a = s.qy0 * (s.qx1 - s.qx2) - s.qy1 * (s.qx0 - s.qx2) + s.qy2 * (s.qx0 - s.qx1);
            const double b = -(s.qy0 * (s.qx1 + s.qx2) * (s.qx1 - s.qx2) - s.qy1 * (s.qx0 + s.qx2) * (s.qx0 - s.qx2) +
                               s.qy2 * (s.qx0 + s.qx1) * (s.qx0 - s.qx1));
            s.qLam = -b / (2 * a);
            if (fabs(s.qLam - s.qx1) / s.qx1 < 1e-3) { s.stage = ST_QUAD_DONE; break; }
            if (a / d < 0) { s.qLam = s.qBt; s.stage = ST_QUAD_DONE; break; }
            s.eval_line(s.dv, s.qLam, ST_QUAD_EVAL);
            break;
        }
        case ST_QUAD_EVAL: {
            if constexpr (!QUAD) break;
            const double eq = s.E;
            s.nEC++;
            s.lamEval = s.qLam; s.Eacc = eq;
            if (fabs(eq - s.qy1) / s.qy1 < 1e-3) { s.stage = ST_QUAD_DONE; break; }
            if (s.qLam < s.qx1) {
                if (eq < s.qy0 && eq < s.qy1) { s.qx1 = s.qLam; s.qy1 = eq; }
                else { s.qx0 = s.qLam; s.qy0 = eq; }
            } else if (s.qx1 < s.qLam) {
                if (eq < s.qy1 && eq < s.qy2) { s.qx1 = s.qLam; s.qy1 = eq; }
                else { s.qx2 = s.qLam; s.qy2 = eq; }
            } else {
                s.qLam = s.qx1; s.stage = ST_QUAD_DONE; break;
            }
            s.stage = ST_QUAD;
            break;
        }
        case ST_QUAD_DONE:   // newE stays the backtracking energy (CGMethod.hpp:655)
            if constexpr (!QUAD) break;
            s.lam = (s.qLam <= 0.0 || s.qLam <= 1e-8) ? 0.0 : s.qLam;
            if (s.lam != 0.0 && s.lam != s.lamEval) {   // forces and energy at the accepted point
                s.eval_line(s.dv, s.lam, ST_QUAD_AT);
                break;
            }
            s.stage = ST_LS_DONE;
            break;
        case ST_QUAD_AT:
            if constexpr (!QUAD) break;
            s.Eacc = s.E;
            s.stage = ST_LS_DONE;
            break;
        case ST_LS_DONE:
            if (s.lam == 0.0) {
                if (!A.try_recover) {
                    s.flags |= MDY_ERROR_LINESEARCH;
                    trace(0.0, s.newE, 0.0);
                    s.after = 0;   // the reference returns before energiesAfter / ptrOutForce
                    s.stage = ST_FINISH;
                } else if (s.safeMode) {
                    s.op = OP_MINSTEP; s.stage = ST_REC_STEP;
                } else {
                    s.reset();
                    s.safeMode = 1;
                    s.nSM++;
                    trace(0.0, s.newE, 0.0);
                    s.stage = ST_ITER;
                }
            } else {   // accepted: the force slots hold the forces at x + lam*d
                s.line(s.dv, s.lam);
                s.gather_step(ST_ACCEPT);
            }
            break;
        case ST_REC_STEP:
            if (s.stepRec == INFINITY) { s.stop(MDY_ERR_RECOVERY); break; }
            s.eval_line(s.dv, s.stepRec, ST_REC_EVAL);
            break;
        case ST_REC_EVAL:
            s.gather_step(ST_REC_GATHER);
            break;
        case ST_REC_GATHER:
            s.nFC++; s.nRec++;
            s.gradInf = s.maxF;
            if (__builtin_expect(!isfinite(s.gradInf), 0)) { s.stop(MDY_ERR_NONFINITE); break; }
            s.cur = 1 - s.cur;
            s.FFcur = s.FF;
            s.reset();
            s.safeMode = 0;
            s.E0 = s.E;   // computeEnergy at the moved coordinates
            trace(0.0, s.newE, 0.0);
            s.stage = ST_ITER;
            break;
        case ST_ACCEPT: {
            s.nFC++;
            s.gradInf = s.maxF;
            if (__builtin_expect(!isfinite(s.gradInf), 0)) { s.stop(MDY_ERR_NONFINITE); break; }
            s.E0 = QUAD && s.quadLS ? s.Eacc : s.newE;   // E(x) of the next line search
            s.relE = fabs(s.newE - s.prevEnergy) / fabs(s.prevEnergy);
            s.prevEnergy = s.newE;
            const double newGrad = s.FF, prevGrad = s.FFp;
            s.beta = 0.0;
            if (A.method == MDY_CG_FLETCHER_RIEVES) s.beta = newGrad / s.lastFDotF;
            else if (A.method == MDY_CG_POLAK_RIBIERE) s.beta = smax(0.0, (newGrad - prevGrad) / s.lastFDotF);
            s.cur = 1 - s.cur;
            s.FFcur = newGrad;
            s.dprev = s.dv; s.sNew = 2 + (1 - s.sidx); s.sidx = 1 - s.sidx;
            s.pendingSpec = 1;   // s = F + beta*d is formed with the next trial
            // forceBelowRelaxedTolerance(10) && numIter > forceCallLimit/2 -> keep lowest-energy coordinates
            if (s.maxF <= 10 * A.grad_tol && s.nIter > A.force_call_limit / 2 && s.newE <= s.minimumE) {
                s.minimumE = s.newE;
                s.haveMin = 1;
                s.saveMin = 1;   // copied before the next work moves anything
            }
            if (A.method != MDY_CG_STEEPEST) s.lastFDotF = newGrad;
            trace(s.lam, s.newE, s.beta);
            s.stage = ST_ITER;
            break;
        }
        case ST_FINAL:
            if (s.after) { s.op = OP_EVAL_FF; s.at_x(); s.ffAfter = 1; s.stage = ST_FINAL_DONE; }
            else s.stage = ST_FINISH;
            break;
        case ST_FINAL_DONE:
            s.nEC++; s.nEE++;
            s.stage = ST_FINISH;
            break;
        default:   // ST_FINISH
            s.op = OP_EXIT;
            break;
        }
    }
}

// One minimization run by a cluster of G blocks (blk = index within it).
// QUAD: compiled with the quadratic line-search stages.
// BATCH: the batched launch's passes ended by completions.
template <bool MIXED, bool QUAD, bool BATCH>
__device__ __attribute__((always_inline)) void cg_run(const CgArgs &A, double *lds, int blk, int G,
                                                      int *done = nullptr, int suspend_done = 0) {
    __shared__ unsigned long long accl[24];
    __shared__ XBlock xb;
    __shared__ CgState S;
    xblock_zero(xb);
    atan_table_fill();
    Cg<MIXED> K(A, lds, xb, accl, blk, G);
    if (BATCH) K.done_ctr = done;
    double *R = A.out;
    const int tid = K.tid;
    const bool leader = (K.blk == 0 && tid == 0);
    if (leader) { R[R_T0] = (double)wall_clock64(); R[R_SUSP] = 0.0; }
    if (tid == 0) {
        if (A.resume) {
            S = *reinterpret_cast<const CgState *>(R + R_RS);
        } else {
            S = CgState{};
            S.op = OP_EVAL_FF; S.at_x(); S.stage = ST_INIT_FF;
            S.gradInf = S.relE = S.minimumE = INFINITY;
            S.after = 1;
            S.dv = S.dprev = S.sNew = -1;
        }
        S.susp = A.suspend_calls > 0 ? A.suspend_calls : 0x7fffffff;
        if (A.other && A.other < G) S.susp = S.nFC + kQuiet;
    }
    auto vec = [&](int id) -> double * {
        return id == 0 ? A.F0 : id == 1 ? A.F1 : id == 2 ? A.S0 : id == 3 ? A.S1 : nullptr;
    };
    auto uni = [](int v) { return __builtin_amdgcn_readfirstlane(v); };
    auto unid = [](double v) {
        return __hiloint2double(__builtin_amdgcn_readfirstlane(__double2hiint(v)),
                                __builtin_amdgcn_readfirstlane(__double2loint(v)));
    };
    for (;;) {
        __syncthreads();
        const int op = uni(S.op);
        if (__builtin_expect(uni(S.saveMin), 0))   // read back by the same threads (OP_RESTORE)
            for (int o = K.gtid; o < A.D.ndof; o += K.gs) A.xmin[o] = A.x[o];
        if (op == OP_EXIT) break;
        const PosAny P{A.x, vec(uni(S.pd)), vec(uni(S.pF)), unid(S.plam), unid(S.pbeta), uni(S.mode)};
        bool ok = true, failed = false;
        if (op == OP_GATHER) {
            const int nqf = uni(S.nqf);
            if (__builtin_expect(nqf != 0, 0)) {
                if (A.other > G) {   // the larger grid repeats the evaluation: its slots stay here, its queue does not
                    __syncthreads();   // S is read
                    if (tid == 0) {
                        S.nEE--;
                        S.suspend(R, leader, OP_EVAL, S.stage == ST_INIT_G ? ST_INIT_F
                                                      : S.stage == ST_ACCEPT ? ST_LS_DONE : ST_REC_EVAL, kWants);
                    }
                    failed = true;
                } else {
                    ok = K.force_fallback(P, nqf, uni(S.qb));
                    if (!ok) break;
                    failed = K.status != 0;
                    if (tid == 0 && A.other) S.susp = S.nFC + kQuiet;
                }
            }
        }
        if (__builtin_expect((op == OP_EVAL || op == OP_GATHER || op == OP_SDONLY) && !failed, 1)) {
            if (op != OP_GATHER) {
                if (P.mode == PosAny::SPEC) spec_direction(K, P.F, P.d, P.beta, vec(uni(S.sNew)));
                if (op == OP_EVAL) K.eval(P);
            } else {
                K.template gather<BATCH>(vec(uni(S.gOut)), vec(uni(S.gPrev)), uni(S.gMove) != 0, P.d, P.lam);
            }
            // end of the phase: the block's sums, the barrier, and what the
            // decision reads; the other waves wait at the top of the loop
            const int p1 = K.ph;
            __builtin_amdgcn_s_waitcnt(0);
            __syncthreads();
            if (tid < 64) {
                K.acc_push(p1);
                ok = K.barrier(op == OP_EVAL ? PK_EVAL : op == OP_GATHER ? PK_GATHER : PK_REDUCE);
                const double v = K.acc_fetch(p1, A.qn + 4 * (p1 % 3), A.qn + 4 * (p1 % 3) + 1);
                const double v1 = __shfl(v, 1, 64);
                if (tid == 0) {
                    if (op == OP_GATHER) {
                        S.maxF = __longlong_as_double((long long)accl[kAccMax]);
                        S.FF = v;
                        S.FFp = S.gPrev >= 0 ? v1 : 0.0;
                        if (BATCH) S.doneSeen = (int)accl[kAccDone];
                    } else {
                        S.xa = v1;
                        if (op == OP_EVAL) {
                            const int nqe = (int)accl[17], nqf = (int)accl[18];
                            S.nEE++;
                            S.E = v;
                            S.nqe = nqe; S.nqf = nqf; S.qb = p1 % 3;
                            if (__builtin_expect(nqe > kQueueCap || nqf > kQueueCap, 0)) {
                                S.status = MDY_ERR_CAPACITY;
                            } else if (__builtin_expect(nqe > 0, 0)) {
                                if (nqe > G && A.other > G) {   // the larger grid repeats this turn
                                    S.nEE--;
                                    S.suspend(R, leader, OP_EVAL, S.stage, kWants);
                                } else {
                                    S.op = OP_EFALLBACK;
                                    if (A.other && nqe > A.other) S.susp = S.nFC + kQuiet;
                                }
                            }
                        }
                    }
                }
            }
            K.ph++;
        } else if (op == OP_NONE) {
            // a resume's first turn has no phase and so no barrier of its own: every
            // wave has read S before thread 0 writes the first operation into it
            __syncthreads();
        } else if (op != OP_GATHER) {
            // collective work: every thread takes part beyond the barrier
            double Eff = 0.0, Effp = 0.0, step = 0.0;
            if (op == OP_EVAL_FF) {
                ok = K.eval_ff(P, R + (uni(S.ffAfter) ? R_EA : R_EB), Eff, Effp);
                if (__builtin_expect(K.leave, 0) && tid == 0) S.suspend(R, leader, OP_EVAL_FF, S.stage, kWants);
            } else if (op == OP_EFALLBACK) {
                ok = K.energy_fallback(P, K.dv(uni(S.qb)), uni(S.nqe), uni(S.qb));
            } else if (op == OP_MINSTEP) {
                // MController::moveAlongDirectionLimitingBeadMove_: step = min maxDist/|d_i|
                const double *dvec = vec(uni(S.dv));
                double v[1] = {INFINITY};
                for (int o = K.gtid; o < A.D.ndof; o += K.gs) v[0] = smin(v[0], A.max_dist / fabs(dvec[o]));
                block_reduce<1>(v, lds, 0u, 0x1u);
                const int p1 = K.ph;
                if (tid == 0) K.red(p1)[(size_t)K.blk * kRed] = v[0];
                ok = K.sync(PK_REDUCE);
                if (ok) {
                    grid_partials_reduce<1>(K.red(p1), K.G, v, lds, 0u, 0x1u);
                    step = v[0];
                }
            } else {   // OP_RESTORE
                for (int o = K.gtid; o < A.D.ndof; o += K.gs) A.x[o] = A.xmin[o];
                ok = K.sync(PK_RESTORE);
            }
            if (tid == 0) {
                S.Eff = Eff; S.Effp = Effp; S.stepRec = step;
                if (op == OP_EFALLBACK) {
                    double e[kNFF + 2];
                    energy_finish(K.acc_local(kAcc0), nullptr, S.nqe, A.qe + S.qb * kQueueCap, K.qeu(S.qb), e);
                    S.E = e[kNFF];
                    S.op = OP_NONE;
                }
            }
        }
        if (tid == 0) {
            S.saveMin = 0;
            if (K.status) S.status = K.status;
            if (__builtin_expect(!ok, 0)) { S.op = OP_EXIT; S.status = MDY_ERR_TIMEOUT; }
            else if (S.op != OP_EFALLBACK) cg_control<QUAD, BATCH>(S, A, leader, suspend_done);
        }
    }
    if (leader) {
        if (S.status == MDY_ERR_TIMEOUT || S.op != OP_EXIT) { R[R_STATUS] = MDY_ERR_TIMEOUT; return; }
        R[R_FLAGS] = S.flags; R[R_NEC] = S.nEC; R[R_NFC] = S.nFC; R[R_NIT] = S.nIter; R[R_GIN] = S.gradInf;
        R[R_ERC] = S.relE; R[R_NEE] = S.nEE; R[R_NSM] = S.nSM; R[R_NREC] = S.nRec; R[R_STATUS] = S.status;
        R[R_TRN] = (double)S.trn; R[R_LAST] = S.after ? 1.0 : 0.0; R[R_FOUT] = (double)S.cur; R[R_NPH] = (double)K.ph;
        // the reference shifts the direction right after an accepted step; here
        // that shift is pending until the next trial
        R[R_DIR] = S.dv; R[R_PEND] = S.pendingSpec; R[R_BETA] = S.beta; R[R_DPREV] = S.dprev;
        R[R_T1] = (double)wall_clock64();
        if (BATCH && done) {
            if (S.suspended == kWants) atomicOr(done, kWants);
            else if (!S.suspended) atomicAdd(done, 1);
        }
    }
}

// The arguments come by value: pointers read from the kernel-argument segment
// are known to be global, so every access is a global (not flat) access.
constexpr int kCgLds = 17 * 16;    // words of the block reductions
constexpr int kCgBlock = 768;      // threads per block: three waves per SIMD

template <bool MIXED, bool QUAD>
__global__ void __launch_bounds__(kCgBlock) k_cg(const CgArgs Av) {
    __shared__ double lds[kCgLds];
    cg_run<MIXED, QUAD, false>(Av, lds, blockIdx.x, gridDim.x);
}

// Batched form: independent minimizations in one cooperative launch. Block b
// belongs to network map[b].x as its block map[b].y; each network's cluster
// runs its own state machine with its own barrier, reductions and buffers.
// Pointers loaded from generic memory are flat to the compiler; loaded from
// the constant address space (as kernel arguments are) they are known to be
// global, so the arguments are read through a constant-space view and every
// access through them uses global instructions, as in the single-network
// kernel.
// done (nullable): the launch's count of finished minimizations; each
// suspends at the top of an iteration once the count reaches suspend_done (>0).
template <bool MIXED, bool QUAD>
__global__ void __launch_bounds__(kCgBlock) k_cg_batch(const CgArgs *__restrict__ all, const int2 *__restrict__ map,
                                                     int *done, int suspend_done) {
    __shared__ double lds[kCgLds];
    const int2 m = map[blockIdx.x];
#if defined(__HIP_DEVICE_COMPILE__)
    typedef __attribute__((address_space(4))) const CgArgs ConstArgs;
    CgArgs A = ((ConstArgs *)all)[m.x];
#else
    CgArgs A = all[m.x];
#endif
    cg_run<MIXED, QUAD, true>(A, lds, m.y, A.grid, done, suspend_done);
}

static const void *cg_kernel(bool mixed, bool quad) {
    if (mixed) return quad ? reinterpret_cast<const void *>(k_cg<true, true>)
                           : reinterpret_cast<const void *>(k_cg<true, false>);
    return quad ? reinterpret_cast<const void *>(k_cg<false, true>)
                : reinterpret_cast<const void *>(k_cg<false, false>);
}
static const void *cg_batch_kernel(bool mixed, bool quad) {
    if (mixed) return quad ? reinterpret_cast<const void *>(k_cg_batch<true, true>)
                           : reinterpret_cast<const void *>(k_cg_batch<true, false>);
    return quad ? reinterpret_cast<const void *>(k_cg_batch<false, true>)
                : reinterpret_cast<const void *>(k_cg_batch<false, false>);
}

// ---------------------------------------------------------------------------
// Buffers and arguments of one minimization run by a cluster of G blocks on
// stream st (the counters and flags it relies on are cleared there; the error
// word where it starts, not where it resumes).
static int prepare_cg(Ctx &c, const mdy_cg_params *p, double *d_x, int G, bool resume, hipStream_t st, CgArgs &A) {
    const int ndof = 3 * c.nb;
    MDY_TRY(ensure(c.F0, ndof)); MDY_TRY(ensure(c.F1, ndof));
    MDY_TRY(ensure(c.S0, ndof)); MDY_TRY(ensure(c.S1, ndof));
    MDY_TRY(ensure(c.xmin, ndof));
    MDY_TRY(ensure(c.prof, 5 * (size_t)c.prof_cap + 5));
    MDY_TRY(ensure(c.prof_kind, c.prof_cap + 1));
    MDY_TRY(ensure(c.cg_out, R_SIZE));
    MDY_TRY(ensure(c.qe, 3 * kQueueCap)); MDY_TRY(ensure(c.qf, 3 * kQueueCap));
    MDY_TRY(ensure(c.qn, 16));
    MDY_TRY(ensure(c.qe_u, 3 * kQueueCap));
    MDY_TRY(ensure(c.tr_lam, c.trace_cap + 1)); MDY_TRY(ensure(c.tr_e, c.trace_cap + 1));
    MDY_TRY(ensure(c.tr_mf, c.trace_cap + 1)); MDY_TRY(ensure(c.tr_beta, c.trace_cap + 1));
    MDY_TRY(ensure(c.tr_safe, c.trace_cap + 1));
    MDY_TRY(ensure(c.bar, 32));
    MDY_TRY(ensure(c.acc, 3 * (size_t)kAccWords));
    MDY_TRY(ensure(c.red, (size_t)3 * G * kRed));
    MDY_TRY(ensure(c.simpson_part, (size_t)6 * G * kRed));
    MDY_HIP(hipMemsetAsync(c.bar.p, 0, 32 * sizeof(unsigned long long), st));
    MDY_HIP(hipMemsetAsync(c.qn.p, 0, 16 * sizeof(int), st));
    MDY_HIP(hipMemsetAsync(c.acc.p, 0, 3 * kAccWords * sizeof(unsigned long long), st));
    if (!resume) MDY_HIP(hipMemsetAsync(c.err.p, 0, sizeof(int), st));
    if (c.prof_cap > 0) MDY_HIP(hipMemsetAsync(c.prof.p, 0, (5 * (size_t)c.prof_cap + 5) * sizeof(long long), st));
    A.D = c.dev();
    A.x = d_x; A.F0 = c.F0.p; A.F1 = c.F1.p; A.S0 = c.S0.p; A.S1 = c.S1.p; A.xmin = c.xmin.p;
    A.contrib = c.contrib.p; A.red = c.red.p; A.qe_u = c.qe_u.p; A.spart = c.simpson_part.p;
    A.qe = c.qe.p; A.qf = c.qf.p; A.qn = c.qn.p; A.bar = c.bar.p; A.acc = c.acc.p; A.out = c.cg_out.p;
    A.tr_lam = c.tr_lam.p; A.tr_e = c.tr_e.p; A.tr_mf = c.tr_mf.p; A.tr_beta = c.tr_beta.p; A.tr_safe = c.tr_safe.p;
    A.tr_cap = c.trace_cap;
    A.prof = c.prof.p; A.prof_kind = c.prof_kind.p; A.prof_cap = c.prof_cap;
    A.method = p->method; A.line_search = p->line_search; A.try_recover = p->try_to_recover; A.energy_call_limit = p->energy_call_limit;
    A.force_call_limit = p->force_call_limit > 3 * p->n_beads_limit ? p->force_call_limit : 3 * p->n_beads_limit;
    A.max_dist = p->max_dist; A.lambda_max = p->lambda_max; A.grad_tol = p->grad_tol;
    A.energy_rel_tol = p->energy_rel_tol;
    A.report_call_limit = p->report_on_call_limit;
    A.spin_limit = 20000000LL;   // polls (tens of seconds) before the watchdog fires
    A.grid = G;
    A.suspend_calls = 0;
    A.resume = resume;
    A.other = 0;
    // Polls go past L2. Below 64 blocks their traffic is small and the shorter wait wins; at 256
    // blocks 2k clocks measured best (40k cylinders: 81.7 / 79.7 / 85.8 us per iteration at 512 /
    // 2k / 8k clocks)
    A.poll_sleep = G > 64 ? 16 : 4;
    return MDY_OK;
}

// MinimizationResult from a result record
static void collect(Ctx &c, const double *R, const mdy_cg_params *p, const CgArgs &A, mdy_min_result *res) {
    std::memset(res, 0, sizeof(*res));
    for (int k = 0; k <= kNFF; k++) { res->energies_before[k] = R[R_EB + k]; res->energies_after[k] = R[R_EA + k]; }
    res->error_flags = (uint32_t)R[R_FLAGS];
    res->num_energy_call = (int32_t)R[R_NEC];
    res->energy_call_limit = p->energy_call_limit;
    res->num_force_call = (int32_t)R[R_NFC];
    res->force_call_limit = A.force_call_limit;
    res->num_iter = (int32_t)R[R_NIT];
    res->grad_inf_norm = R[R_GIN];
    res->grad_tol = p->grad_tol;
    res->energy_rel_change = R[R_ERC];
    res->energy_rel_tol = p->energy_rel_tol;
    res->num_energy_eval = (int32_t)R[R_NEE];
    res->num_safe_mode = (int32_t)R[R_NSM];
    res->num_recovery = (int32_t)R[R_NREC];
    res->status = (int32_t)R[R_STATUS];
    c.trace_n = (long long)R[R_TRN];
    c.prof_n = (long long)R[R_NPH];
    c.have_dir = res->status == MDY_OK;
    c.dir_buf = (int)R[R_DIR]; c.dir_pend = R[R_PEND] != 0.0; c.dir_beta = R[R_BETA];
    c.dir_prev = (int)R[R_DPREV]; c.dir_cur = (int)R[R_FOUT];
}

// s = F + beta d and the exact s.F, in one block (cgShiftSearchDir and
// resetCGParams, CGMethod.cpp:325-360: the same expression and the same exact
// sum as the kernel's direction update)
__global__ void __launch_bounds__(1024) k_final_dir(const double *__restrict__ F, const double *__restrict__ d,
                                                     double beta, int n, double *__restrict__ s, double *sf) {
    __shared__ long long lds[136];
    mdy_xsum x;
    mdy_xs_zero(&x);
    for (int i = threadIdx.x; i < n; i += blockDim.x) {
        const double v = F[i] + beta * d[i];
        s[i] = v;
        mdy_xs_add(&x, v * F[i]);
    }
    block_reduce_xsum(x, lds);
    if (threadIdx.x == 0) sf[0] = mdy_xs_value(&x);
}

int final_search_dir(Ctx &c, double *h_out) {
    if (!c.have_dir) return MDY_ERR_STATE;
    hipStream_t st = c.stream;
    const size_t n = 3 * (size_t)c.nb;
    auto buf = [&](int id) -> const double * {
        return id == 0 ? c.F0.p : id == 1 ? c.F1.p : id == 2 ? c.S0.p : id == 3 ? c.S1.p : nullptr;
    };
    const double *src = buf(c.dir_buf);
    if (c.dir_pend) {
        const double *F = buf(c.dir_cur), *d = buf(c.dir_prev);
        if (!F || !d) return MDY_ERR_STATE;
        MDY_TRY(ensure(c.xt, n));
        MDY_TRY(ensure(c.out, 8));
        hipLaunchKernelGGL(k_final_dir, dim3(1), dim3(1024), 0, st, F, d, c.dir_beta, (int)n, c.xt.p, c.out.p);
        MDY_HIP(hipGetLastError());
        double sf = 0;
        MDY_HIP(hipMemcpyAsync(&sf, c.out.p, sizeof(double), hipMemcpyDeviceToHost, st));
        MDY_HIP(hipStreamSynchronize(st));
        src = (sf <= 0) ? F : c.xt.p;   // resetCGParams when s.F <= 0
    }
    if (!src) return MDY_ERR_STATE;
    MDY_HIP(hipMemcpyAsync(h_out, src, sizeof(double) * n, hipMemcpyDeviceToHost, st));
    MDY_HIP(hipStreamSynchronize(st));
    return MDY_OK;
}

static int copy_force_out(Ctx &c, const double *R, double *d_force_out, hipStream_t st) {
    if (d_force_out && R[R_LAST] != 0.0) {
        const double *src = ((int)R[R_FOUT] == 0) ? c.F0.p : c.F1.p;
        MDY_HIP(hipMemcpyAsync(d_force_out, src, sizeof(double) * 3 * (size_t)c.nb, hipMemcpyDeviceToDevice, st));
    }
    return MDY_OK;
}

// two timing events, destroyed on every return path
struct EventPair {
    hipEvent_t a = nullptr, b = nullptr;
    ~EventPair() {
        if (a) (void)hipEventDestroy(a);
        if (b) (void)hipEventDestroy(b);
    }
};

int run_minimize(Ctx &c, const mdy_cg_params *p, double *d_x, double *d_force_out, mdy_min_result *res) {
    hipStream_t st = c.stream;
    // persistent grid: all blocks resident
    int per_cu = 0;
    const bool mixed = c.opts.precision == MDY_PREC_MIXED;
    const bool quad = p->line_search == MDY_LS_QUADRATIC;
    const void *kern = cg_kernel(mixed, quad);
    MDY_HIP(hipOccupancyMaxActiveBlocksPerMultiprocessor(&per_cu, kern, kCgBlock, 0));
    if (per_cu < 1) return MDY_ERR_LAUNCH;
    if (c.opts.blocks_per_cu > 0 && c.opts.blocks_per_cu < per_cu) per_cu = c.opts.blocks_per_cu;
    // One lane per thread where the network has fewer lanes than that: a phase's
    // barrier, and the L2 write-back and invalidation that go with it, get slower
    // with the block count (500 cylinders: 27 us per iteration on 8 blocks, 43 on
    // 256; 4k: 43 on 48 blocks, 80 on 256; fewer blocks than lanes / 512 lose more
    // than they save: 50 on 24). Blocks of 512 threads while one turn covers the
    // lanes, of 768 (three waves per SIMD) beyond: 200k cylinders 191 against 195.
    const int lanes = c.dev().n_lanes();
    const int threads = lanes > c.num_cu * 512 ? kCgBlock : 512;
    // The fallbacks' quadratures want every CU: 260 us for a turn of queued
    // energies, a block each, and 155 ms per queued force on 8 blocks (5 on 256). An
    // evaluation that queues more energies than there are blocks, or a force
    // that is needed, suspends the launch; one on all blocks repeats it and hands
    // back after kQuiet force calls without another. 60 force calls from 64
    // parallel pairs: 3.5 ms, 6.9 on 8 blocks alone, 4.1 on 256 alone; 2 force
    // calls with both of 2 pairs by quadrature: 31 ms, 928 on 8 blocks alone.
    const int all = per_cu * c.num_cu;
    const int few = c.opts.blocks_per_cu > 0 ? all : std::min(all, std::max(8, (lanes + threads - 1) / threads));
    int G = few;
    EventPair ev;
    MDY_HIP(hipEventCreate(&ev.a));
    MDY_HIP(hipEventCreate(&ev.b));
    CgArgs A;
    double R[R_SIZE];
    c.last_ms = 0;
    for (bool resume = false;; resume = true, G = G == few ? all : few) {
        MDY_TRY(prepare_cg(c, p, d_x, G, resume, st, A));
        if (few < all && c.prof_cap == 0) A.other = G == few ? all : few;   // a profile is one launch's
        MDY_HIP(hipEventRecord(ev.a, st));
        void *args[] = {&A};
        if (hipLaunchCooperativeKernel(kern, dim3(G), dim3(threads), args, 0, st) != hipSuccess) return MDY_ERR_LAUNCH;
        MDY_HIP(hipEventRecord(ev.b, st));
        MDY_HIP(hipMemcpyAsync(R, c.cg_out.p, sizeof(R), hipMemcpyDeviceToHost, st));
        MDY_HIP(hipStreamSynchronize(st));
        float ms = 0;
        (void)hipEventElapsedTime(&ms, ev.a, ev.b);
        c.last_ms += ms;
        if (R[R_SUSP] == 0.0 || R[R_STATUS] != MDY_OK) break;
    }
    c.coop_blocks = G;
    c.coop_threads = threads;
    collect(c, R, p, A, res);
    MDY_TRY(copy_force_out(c, R, d_force_out, st));
    MDY_HIP(hipStreamSynchronize(st));
    return res->status == MDY_ERR_TIMEOUT ? MDY_ERR_TIMEOUT : MDY_OK;
}

// Batched minimizations: the resident blocks are split into one cluster per
// network, in proportion to its weight (by default its per-evaluation work,
// interactions + 2 x beads), at least one block each; networks beyond the
// resident block count run in further launches. With first_pass_calls > 0 the minimizations run in passes: pass
// k suspends every minimization at the top of its first iteration after
// first_pass_calls * 4^(k-1) force calls (one below its own limit and not
// converged), saving its state; the next pass resumes it exactly there, with
// all the blocks shared among the networks still running; a pass in which
// every network gets at least kUncappedShare threads runs uncapped. A
// minimization's trajectory does not depend on its cluster size, so the
// results equal those of one uncapped pass; the passes only move the blocks
// of finished networks to the slow ones. With first_pass_calls = -k < 0 the
// passes end by completions instead: a launch of m > 1 networks counts its
// finished minimizations on the device, and once max(1, m / k) have finished
// the others suspend at the top of their next iteration (each reads the
// count once per iteration); the next pass re-splits all the blocks among
// them, down to one network on the whole grid. Quadrature fallbacks that want
// more blocks than a network has lanes for (run_minimize) end a pass as well:
// from the next one on the network gets some that nobody has lanes for, up to
// kWideThreads (8 networks of 128 cylinders, 64 parallel pairs and 60 force
// calls each: 4.2 ms, 36 on the two blocks that their lanes fill; 4 networks
// with 2 force calls by 2 quadratures each: 232 ms and 7310 on one block).
// cs[i] owns network i's tables, neighbor lists and CG buffers; cs[0] the
// launch arrays.
constexpr int kUncappedShare = 4096;   // threads per network at which a pass runs uncapped
constexpr int kCapGrowth = 4;          // force-call cap growth from one pass to the next (x2 measured slower)
constexpr int kWideThreads = 16384;    // threads of a network with quadrature fallbacks, at most
constexpr int kBatchBlock = 512;       // threads per block while every network gets a block
int run_minimize_batch(Ctx **cs, int n, const mdy_cg_params *p, double *const *d_x, double *const *d_force_out,
                       mdy_min_result *res, double *net_ms, int threads_per_block, const double *weights,
                       int first_pass_calls, hipStream_t st, double *total_ms) {
    Ctx &c0 = *cs[0];
    const bool mixed = c0.opts.precision == MDY_PREC_MIXED;
    bool quad = false;
    for (int i = 0; i < n; i++) quad = quad || p[i].line_search == MDY_LS_QUADRATIC;
    const void *kern = cg_batch_kernel(mixed, quad);
    // Blocks of threads_per_block threads; for 64, the default, of 512 while every
    // network gets one, then half as many, down to 64: every block of a launch
    // writes its XCD's L2 back and invalidates it once per phase of its network,
    // for all the others too, so fewer and larger ones win (32 networks of 500 to
    // 5000 cylinders, kernel time: 156 ms with 64 threads, 67 with 256, 53 with 512;
    // 256 networks: 333, 147, 112). The results do not depend on it.
    const bool chosen = threads_per_block > 64;
    int tpb = chosen ? threads_per_block : kBatchBlock, per_cu = 0;
    for (;; tpb /= 2) {
        MDY_HIP(hipOccupancyMaxActiveBlocksPerMultiprocessor(&per_cu, kern, tpb, 0));
        if (chosen || tpb <= 64 || per_cu * c0.num_cu >= n) break;
    }
    if (per_cu < 1) return MDY_ERR_LAUNCH;
    const int Gmax = per_cu * c0.num_cu;
    std::vector<char> resume(n, 0), wide(n, 0);   // suspended in an earlier pass; for its fallbacks
    EventPair ev;
    MDY_HIP(hipEventCreate(&ev.a));
    MDY_HIP(hipEventCreate(&ev.b));
    hipEvent_t e0 = ev.a, e1 = ev.b;
    double kernel_ms = 0;
    double t_origin = -1.0;   // device clock at the first launch's start
    std::vector<CgArgs> args;
    std::vector<int2> map;
    std::vector<int> gsz, todo(n), next;
    for (int i = 0; i < n; i++) todo[i] = i;
    long long cap = first_pass_calls > 0 ? first_pass_calls : 0;
    const int by_done = first_pass_calls < 0 ? -first_pass_calls : 0;
    int rc = MDY_OK;
    rc = ensure(c0.batch_done, 1);
    while (!todo.empty() && rc == MDY_OK) {
        next.clear();
        const int nt = (int)todo.size();
        // few networks left: each gets enough blocks that a larger cluster
        // would not be faster, so this pass runs them to the end
        if ((long long)nt * kUncappedShare <= (long long)Gmax * tpb) cap = 0;
        for (int lo = 0; lo < nt && rc == MDY_OK; lo += Gmax) {
            const int m = (nt - lo < Gmax) ? nt - lo : Gmax;
            // cluster sizes: proportional shares of the blocks left after one each
            double tot = 0;
            std::vector<double> w(m);
            for (int i = 0; i < m; i++) {
                const int k = todo[lo + i];
                const Ctx &ci = *cs[k];
                w[i] = weights ? weights[k] : (double)ci.dev().n_items() + 2.0 * ci.nb;
                if (!(w[i] > 0.0)) w[i] = 0.0;
                tot += w[i];
            }
            gsz.assign(m, 1);
            const int spare = Gmax - m;
            int used = 0;
            std::vector<std::pair<double, int>> frac;
            for (int i = 0; i < m; i++) {
                const double share = tot > 0 ? spare * w[i] / tot : 0.0;
                const int whole = (int)share;
                gsz[i] += whole;
                used += whole;
                frac.push_back({share - whole, i});
            }
            std::sort(frac.begin(), frac.end(),
                      [](const std::pair<double, int> &a, const std::pair<double, int> &b) {
                          return a.first > b.first || (a.first == b.first && a.second < b.second);
                      });
            for (int k = 0; k < spare - used && k < m; k++) gsz[frac[k].second]++;
            // one lane per thread: more blocks only slow a cluster's barrier down
            int nwide = 0;
            used = 0;
            for (int i = 0; i < m; i++) {
                gsz[i] = std::min(gsz[i], std::max(1, (cs[todo[lo + i]]->dev().n_lanes() + tpb - 1) / tpb));
                used += gsz[i];
                nwide += wide[todo[lo + i]];
            }
            // what that leaves is for the fallbacks: split among the networks that asked, or there to be asked for
            std::vector<int> other(m, 0);
            bool may_want = false;
            const int left = Gmax - used, each = nwide ? left / nwide : 0;
            for (int i = 0; i < m; i++) {
                const int room = std::max(0, kWideThreads / tpb - gsz[i]);
                if (wide[todo[lo + i]]) {
                    gsz[i] += std::min(room, each);
                } else if (std::min(room, left) > 0) {
                    other[i] = gsz[i] + std::min(room, left);
                    may_want = true;
                }
            }
            args.assign(m, CgArgs{});
            map.clear();
            for (int i = 0; i < m && rc == MDY_OK; i++) {
                const int k = todo[lo + i];
                rc = prepare_cg(*cs[k], &p[k], d_x[k], gsz[i], resume[k] != 0, st, args[i]);
                args[i].other = other[i];
                if (cap > 0 && cap < (long long)args[i].force_call_limit) args[i].suspend_calls = (int)cap;
                for (int b = 0; b < gsz[i]; b++) map.push_back(make_int2(i, b));
            }
            if (rc != MDY_OK) break;
            const int G = (int)map.size();
            rc = ensure(c0.batch_args, (size_t)m * sizeof(CgArgs));
            if (rc == MDY_OK) rc = ensure(c0.batch_map, (size_t)G);
            if (rc != MDY_OK) break;
            if (hipMemcpyAsync(c0.batch_args.p, args.data(), (size_t)m * sizeof(CgArgs), hipMemcpyHostToDevice,
                               st) != hipSuccess ||
                hipMemcpyAsync(c0.batch_map.p, map.data(), (size_t)G * sizeof(int2), hipMemcpyHostToDevice, st) !=
                    hipSuccess) {
                rc = MDY_ERR_HIP;
                break;
            }
            if (hipMemsetAsync(c0.batch_done.p, 0, sizeof(int), st) != hipSuccess) {
                rc = MDY_ERR_HIP;
                break;
            }
            const CgArgs *pa = reinterpret_cast<const CgArgs *>(c0.batch_args.p);
            const int2 *pm = c0.batch_map.p;
            int *done = (by_done || may_want) && m > 1 ? c0.batch_done.p : nullptr;
            int suspend_done = !done ? 0 : by_done ? std::max(1, m / by_done) : kWants;
            void *kargs[] = {&pa, &pm, &done, &suspend_done};
            (void)hipEventRecord(e0, st);
            if (hipLaunchCooperativeKernel(kern, dim3(G), dim3(tpb), kargs, 0, st) != hipSuccess) {
                rc = MDY_ERR_LAUNCH;
                break;
            }
            (void)hipEventRecord(e1, st);
            // the host arrays are reused by the next launch: wait for this one
            if (hipStreamSynchronize(st) != hipSuccess) { rc = MDY_ERR_HIP; break; }
            float ms = 0;
            (void)hipEventElapsedTime(&ms, e0, e1);
            kernel_ms += ms;
            for (int i = 0; i < m && rc == MDY_OK; i++) {
                const int k = todo[lo + i];
                Ctx &ci = *cs[k];
                double R[R_SIZE];
                if (hipMemcpy(R, ci.cg_out.p, sizeof(R), hipMemcpyDeviceToHost) != hipSuccess) {
                    rc = MDY_ERR_HIP;
                    break;
                }
                if (t_origin < 0 || R[R_T0] < t_origin) t_origin = R[R_T0];
                ci.coop_blocks = gsz[i];
                ci.coop_threads = tpb;
                if (R[R_SUSP] != 0.0 && R[R_STATUS] == MDY_OK) {   // resumes in the next pass
                    resume[k] = 1;
                    wide[k] |= R[R_SUSP] == kWants;
                    next.push_back(k);
                    continue;
                }
                collect(ci, R, &p[k], args[i], &res[k]);
                if (net_ms) net_ms[k] = (R[R_T1] - t_origin) * 1e-5;   // 100 MHz ticks
                rc = copy_force_out(ci, R, d_force_out ? d_force_out[k] : nullptr, st);
            }
        }
        todo.swap(next);
        if (cap > 0) cap *= kCapGrowth;
    }
    (void)hipStreamSynchronize(st);
    if (total_ms) *total_ms = kernel_ms;
    return rc;
}

}  // namespace mdy
