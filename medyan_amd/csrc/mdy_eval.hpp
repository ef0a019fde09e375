// mdy_eval.hpp -- evaluation of all interactions over the unified index space,
// per-bead force gather, exact block/grid reductions and the quadrature
// fallbacks. Used both by the one-shot kernels (mdy_eval.hip) and by the
// persistent conjugate-gradient kernel (mdy_cg.hip).
#pragma once
#include "mdy_device.hpp"
#include "mdy_internal.hpp"

namespace mdy {

// ---- where bead positions come from ---------------------------------------
// get: the positions of N beads, every load issued before the first use, so N
// beads cost one memory round trip.
struct PosX {  // x
    const double *__restrict__ x;
    __device__ __forceinline__ d3 operator()(int o) const { return d3{x[o], x[o + 1], x[o + 2]}; }
    template <int N> __device__ __forceinline__ void get(const int (&o)[N], d3 (&c)[N]) const {
#pragma unroll
        for (int k = 0; k < N; k++) c[k] = (*this)(o[k]);
    }
};
// One functor for the minimizer's three kinds (uniform runtime mode), so that a
// single inlined copy of the interaction code serves every evaluation: x,
// x + lam * d (CGMethod::calcCoordLineSearch, CGMethod.cpp:43-46), or
// x + lam * (F + beta * d), the trial along the not-yet-stored new direction.
// One branch per item: with one per component each was a dependent round trip
// (a linker's four beads took 21 us of a 50 us sweep at 40k cylinders).
struct PosAny {
    enum { X = 0, LINE = 1, SPEC = 2 };
    const double *__restrict__ x;
    const double *__restrict__ d;
    const double *__restrict__ F;
    double lam, beta;
    int mode;
    template <int N> __device__ __forceinline__ void get(const int (&o)[N], d3 (&c)[N]) const {
        const PosX px{x};
        px.get(o, c);
        if (mode == X) return;
        d3 s[N];
        PosX{d}.get(o, s);
        if (mode == SPEC) {
            d3 f[N];
            PosX{F}.get(o, f);
#pragma unroll
            for (int k = 0; k < N; k++)
                s[k] = d3{f[k].x + beta * s[k].x, f[k].y + beta * s[k].y, f[k].z + beta * s[k].z};
        }
#pragma unroll
        for (int k = 0; k < N; k++)
            c[k] = d3{c[k].x + lam * s[k].x, c[k].y + lam * s[k].y, c[k].z + lam * s[k].z};
    }
    __device__ __forceinline__ d3 operator()(int o) const {
        const int q[1] = {o};
        d3 c[1];
        get(q, c);
        return c[0];
    }
};

__device__ __forceinline__ void set_err(int *err, int code) { atomicCAS(err, 0, code); }

__device__ __forceinline__ void enqueue(int *q, int *qn, int v, int *err) {
    int s = atomicAdd(qn, 1);
    if (s < kQueueCap) q[s] = v;
    else set_err(err, MDY_ERR_CAPACITY);
}

__device__ __forceinline__ void put3(double *__restrict__ c, int slot, d3 v) {
    c[3 * slot] = v.x; c[3 * slot + 1] = v.y; c[3 * slot + 2] = v.z;
}
// mixed-precision force records: 3 floats per slot
__device__ __forceinline__ void put3(float *__restrict__ c, int slot, d3 v) {
    c[3 * slot] = (float)v.x; c[3 * slot + 1] = (float)v.y; c[3 * slot + 2] = (float)v.z;
}
__device__ __forceinline__ void put3(float *__restrict__ c, int slot, f3 v) {
    c[3 * slot] = v.x; c[3 * slot + 1] = v.y; c[3 * slot + 2] = v.z;
}
template <class S> __device__ __forceinline__ V3<S> vec3_none() { return V3<S>{S(-0.0), S(-0.0), S(-0.0)}; }
// force-record element type of each form
template <bool MIXED> struct SlotT { using T = double; };
template <> struct SlotT<true> { using T = float; };

// ---- exact block sums in LDS -------------------------------------------------
// Two exact sums (mdy_xsum's digits) and a maximum per block, accumulated as the
// terms arise: each term adds its two or three digits with LDS integer atomics,
// in any order with the same result, so no thread carries an accumulator (14
// registers each) through the sweep and the end of a phase combines 16 copies
// of 17 words instead of every thread's. Copy = thread % 16.
// A block of at most 1024 threads may add kXTurns terms per thread and sum
// between two calls of xblock_norm: 1024 * 16 terms below 2^48 stay below 2^63.
constexpr int kXRep = 16, kXTurns = 16;
struct XBlock {
    unsigned long long w[17][kXRep];   // sum 0: digits 0..6, flags; sum 1: the same; maximum
};
struct XAdd {   // this thread's copy of sum 0 or 1
    XBlock *x;
    int row;
    __device__ __forceinline__ void put(int k, unsigned long long v) const {
        __hip_atomic_fetch_add(&x->w[row + k][threadIdx.x & (kXRep - 1)], v, __ATOMIC_RELAXED,
                               __HIP_MEMORY_SCOPE_WORKGROUP);
    }
    __device__ __forceinline__ void flag(int v) const {
        __hip_atomic_fetch_or(&x->w[row + 7][threadIdx.x & (kXRep - 1)], (unsigned long long)v, __ATOMIC_RELAXED,
                              __HIP_MEMORY_SCOPE_WORKGROUP);
    }
    // mdy_xs_add
    __device__ __forceinline__ void operator()(double v) const {
        const unsigned long long b = mdy_dbits(v);
        const bool neg = (b >> 63) != 0;
        const int ex = (int)((b >> 52) & 0x7ff);
        unsigned long long m = b & 0xFFFFFFFFFFFFFull;
        if (__builtin_expect(ex == 0x7ff, 0)) {
            flag(m ? MDY_XS_NAN : (neg ? MDY_XS_NINF : MDY_XS_PINF));
            return;
        }
        if (ex) m |= 0x10000000000000ull;
        int p = (ex ? ex - 1075 : -1074) + MDY_XS_BIAS;
        if (p < 0) {
            m = (-p >= 64) ? 0 : (m >> (-p));
            p = 0;
        }
        if (m == 0) return;
        if (__builtin_expect(p + 53 > 48 * (MDY_XS_N - 1) + 47, 0)) {
            flag(neg ? MDY_XS_NINF : MDY_XS_PINF);
            return;
        }
        const int j = p / 48, sh = p - 48 * j;
        const unsigned long long lo = (m << sh) & (unsigned long long)MDY_XS_MASK;
        const unsigned long long mid = (sh == 0 ? (m >> 48) : (m >> (48 - sh))) & (unsigned long long)MDY_XS_MASK;
        const unsigned long long hi = (96 - sh < 64) ? m >> (96 - sh) : 0;   // 0 in the last digits: the sum's bound
        put(j, neg ? 0 - lo : lo);
        put(j + 1, neg ? 0 - mid : mid);
        if (hi) put(j + 2, neg ? 0 - hi : hi);
    }
};
__device__ __forceinline__ void xblock_zero(XBlock &x) {
    for (int k = threadIdx.x; k < 17 * kXRep; k += blockDim.x) (&x.w[0][0])[k] = 0;
}
__device__ __forceinline__ void xblock_max(XBlock &x, double m) {   // m >= 0 or NaN: ordered as integers
    __hip_atomic_fetch_max(&x.w[16][threadIdx.x & (kXRep - 1)], (unsigned long long)__double_as_longlong(m),
                           __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
}
// carries of every copy into [0, 2^48) digits (all threads of the block)
__device__ __forceinline__ void xblock_norm(XBlock &x) {
    __syncthreads();
    if (threadIdx.x < 2 * kXRep) {
        const int row = 8 * (threadIdx.x / kXRep), r = threadIdx.x % kXRep;
        long long c = 0;
        for (int k = 0; k < MDY_XS_N; k++) {
            const long long d = (long long)x.w[row + k][r] + c;
            c = d >> 48;
            x.w[row + k][r] = k < MDY_XS_N - 1 ? (unsigned long long)(d & MDY_XS_MASK) : (unsigned long long)d;
        }
    }
    __syncthreads();
}
// Word t (t = 0..16, one per thread of the first wave) of the block's sums, its
// copies cleared for the next phase: digits below 2^49, so that the words of
// 2^14 blocks can be added. Every thread calls it after a __syncthreads();
// threads t >= 17 get 0.
__device__ __forceinline__ unsigned long long xblock_take(XBlock &x) {
    const int t = threadIdx.x;
    if (t >= 64) return 0;
    unsigned long long r = 0;
    if (t < 17) {
        const bool isor = (t & 7) == 7, ismax = t == 16;
#pragma unroll
        for (int k = 0; k < kXRep; k++) {   // rotated: the lanes read different banks
            unsigned long long &e = x.w[t][(k + t) & (kXRep - 1)];
            const unsigned long long v = e;
            e = 0;
            r = isor ? (r | v) : ismax ? (v > r ? v : r) : r + v;
        }
    }
    // one carry step: each digit keeps its low 48 bits and takes its neighbor's rest
    const long long carry = (long long)r >> 48, up = __shfl_up(carry, 1, 64);
    const int k = t & 7;
    if (t < 16 && k < 7) {
        if (k < MDY_XS_N - 1) r &= (unsigned long long)MDY_XS_MASK;
        if (k > 0) r += (unsigned long long)up;
    }
    return r;
}

// ---- the interaction sweep -------------------------------------------------
// The sweep's index space is one of lanes: two for every excluded-volume pair
// of the integral form, then one for every other interaction,
// [EV x 2 | FS | FB | LM | BS | BB | BDH | BP | BD]. Starts and strides are
// multiples of the wave, so a pair's lanes are neighbors in one.
// IT_EVM: an excluded-volume pair of the monomer-sum form (one lane, same table and slots)
enum { IT_EVM = 0, IT_FS, IT_FB, IT_LM, IT_BS, IT_BB, IT_BDH, IT_BP, IT_BD, IT_NONE };
struct ItemRec {
    int type, j;      // kind and index within its table
    int4 b;           // bead offsets (x3); unused entries repeat the first
    double p0, p1, p2, p3;
};
// record of lane i >= n_duo_lanes()
__device__ __forceinline__ ItemRec fetch_rec(const Dev &D, int i) {
    ItemRec r;
    r.p0 = r.p1 = r.p2 = r.p3 = 0.0;
    i -= D.n_duo_lanes();
    const int n_evm = D.ev_mon ? D.n_ev : 0;
    if (i < n_evm) {
        r.type = IT_EVM; r.j = i;
        r.b = D.ev_bs[i];
        r.p0 = D.ev_kr[i];
    } else if ((i -= n_evm) < D.n_fs) {
        r.type = IT_FS; r.j = i;
        const int2 b = D.fs_bs[i];
        r.b = make_int4(b.x, b.y, b.x, b.x);
        r.p0 = D.fs_k[i]; r.p1 = D.fs_l0[i];
    } else if ((i -= D.n_fs) < D.n_fb) {
        r.type = IT_FB; r.j = i;
        const int *b = D.fb_bs + 3 * i;
        r.b = make_int4(b[0], b[1], b[2], b[0]);
        r.p0 = D.fb_k[i]; r.p1 = D.fb_th[i]; r.p2 = D.fb_ct[i]; r.p3 = D.fb_st[i];
    } else if ((i -= D.n_fb) < D.n_lm) {
        r.type = IT_LM; r.j = i;
        r.b = D.lm_bs[i];
        r.p0 = D.lm_k[i]; r.p1 = D.lm_l0[i]; r.p2 = D.lm_p1[i]; r.p3 = D.lm_p2[i];
    } else if ((i -= D.n_lm) < D.n_bs) {
        r.type = IT_BS; r.j = i;
        const int *b = D.bs_bs + 3 * i;
        r.b = make_int4(b[0], b[1], b[2], b[0]);
        r.p0 = D.bs_k[i]; r.p1 = D.bs_l0[i]; r.p2 = D.bs_p[i];
    } else if ((i -= D.n_bs) < D.n_bb) {
        r.type = IT_BB; r.j = i;
        r.b = D.bb_bs[i];
        r.p0 = D.bb_k[i]; r.p1 = D.bb_th[i]; r.p2 = D.bb_ct[i]; r.p3 = D.bb_st[i];
    } else if ((i -= D.n_bb) < D.n_bdh) {
        r.type = IT_BDH; r.j = i;
        r.b = D.bdh_bs[i];
        r.p0 = D.bdh_k[i]; r.p1 = D.bdh_pos[i];
    } else if ((i -= D.n_bdh) < D.n_bp) {
        r.type = IT_BP; r.j = i;
        const int *b = D.bp_bs + 3 * i;
        r.b = make_int4(b[0], b[1], b[2], b[0]);
        r.p0 = D.bp_k[i]; r.p1 = D.bp_pos[i];
    } else if ((i -= D.n_bp) < D.n_bd) {
        r.type = IT_BD; r.j = i;
        const int bead = D.bd_bead[i];
        r.b = make_int4(bead, D.bd_plane[i], bead, bead);
        r.p0 = D.bd_k[i]; r.p1 = D.bd_sl[i];
    } else {
        r.type = IT_NONE; r.j = 0;
        r.b = make_int4(0, 0, 0, 0);
    }
    return r;
}
__device__ __forceinline__ int rec_nbeads(int type) {
    return type == IT_EVM || type == IT_LM || type == IT_BB || type == IT_BDH ? 4
         : type == IT_FB || type == IT_BS || type == IT_BP ? 3
         : type == IT_FS ? 2 : type == IT_BD ? 1 : 0;
}
// Mixed-precision form: a pair's force runs in FP32 only when the squared
// normalized triple product q = -JJ / (a b c) of the two cylinders is at
// least this; nearer-coplanar pairs amplify FP32 rounding as ~6e-8 / q (at
// 0.03 the FP32 pair force stays within ~6e-5 of its FP64 value, about 3/4 of
// the pairs of a random network qualify).
constexpr double kMixedMinQ = 0.03;

// ---- an excluded-volume pair on its two lanes, each having loaded its
// cylinder's beads: energy (counted by lane 0) and, if FORCES, the four slots.
// QUAD: the pairs flagged in D.evq are skipped (the quadrature kernels evaluate them).
template <bool MIXED, bool QUAD, class P>
__device__ __forceinline__ void ev_duo_item(const Dev &D, int i, const P &pos, double acc[kNFF], const XAdd &xs,
                                            typename SlotT<MIXED>::T *__restrict__ contrib, const bool PER_FF,
                                            const bool FORCES) {
    const int j = i >> 1;
    const bool h = (i & 1) != 0;
    if (QUAD && D.evq[j]) return;
    const int2 o = reinterpret_cast<const int2 *>(D.ev_bs)[i];
    const double kr = D.ev_kr[j];
    const int oo[2] = {o.x, o.y};
    d3 mm[2];
    pos.get(oo, mm);
    const d3 m0 = mm[0];
    d3 m1 = mm[1];
    EvDuoT<double> v;
    double U = 0.0;
    // pass 0: the pair as given (energy, and force unless coplanar);
    // pass 1: the coplanar perturbation of the reference force path,
    // c2 moved off the plane (CylinderExclVolRepulsion.cpp:610-626)
#pragma clang loop unroll(disable)
    for (int pass = 0; pass < 2; pass++) {
        const d3 c1 = duo_get<0>(m0), c2 = duo_get<0>(m1), c3 = duo_get<1>(m0), c4 = duo_get<1>(m1);
        double block;
        ev_duo_invariants(h, c1, c2, c3, c4, v, block);
        if (pass == 0) {
            U = ev_duo_energy(v, block, kr);
            if (!FORCES || !(D.coplanar_mode == MDY_COPLANAR_REFERENCE && are_in_plane(c1, c2, c3, c4))) break;
            const d3 c2e = moved_off_plane(c1, c2, c3, c2, 0.01);
            m1 = pick3(h, m1, c2e);
        }
    }
    // a pair is queued for its quadrature energy only where energies are summed:
    // nothing takes the entries of a sweep for forces alone out of the queue
    if (!h && (xs.x || PER_FF)) {
        if (ev_energy_bad(U)) {
            enqueue(D.qe, D.qe_n, j, D.err);
        } else {
            if (xs.x) xs(U);
            if (PER_FF) acc[MDY_FF_EV] += U;
        }
    }
    if (FORCES) {
        const int s = D.slot_ev + 2 * i;
        const d3 c1 = duo_get<0>(m0), c2 = duo_get<0>(m1), c3 = duo_get<1>(m0), c4 = duo_get<1>(m1);
        if constexpr (MIXED) {
            if (-v.JJ / (v.a * v.b * v.c) >= kMixedMinQ) {
                // well-conditioned pair: derivative blocks in FP32
                f3 f[2];
                ev_duo_force<float>(h, v, c1, c2, c3, c4, kr, f);
                if (!duo_any(!(finite_d3(f[0]) && finite_d3(f[1])))) {
                    put3(contrib, s, f[0]); put3(contrib, s + 1, f[1]);
                    return;
                }
            }
        }
        d3 f[2];
        ev_duo_force<double>(h, v, c1, c2, c3, c4, kr, f);
        if (duo_any(!(finite_d3(f[0]) && finite_d3(f[1])))) {
            if (!h) enqueue(D.qf, D.qf_n, j, D.err);
        } else {
            put3(contrib, s, f[0]); put3(contrib, s + 1, f[1]);
        }
    }
}

// ---- one other interaction from its record and positions: energy (into the
// exact total and, if PER_FF, into the per-force-field double sums) and, if
// FORCES, its per-bead force slots. One accumulation site keeps the inlined
// code small (it runs from the instruction cache of every CU).
template <bool MIXED = false>
__device__ __forceinline__ void item_compute(const Dev &D, const ItemRec &r, const d3 c[4], double acc[kNFF],
                                             const XAdd &xs, typename SlotT<MIXED>::T *__restrict__ contrib,
                                             const bool PER_FF, const bool FORCES) {
    double U = 0.0;
    int ff = 0;
    bool add = true;
    const int j = r.j;
    if (r.type == IT_EVM) {   // monomer-pair sum, in FP64 in both forms; no fallbacks
        ff = MDY_FF_EV;
        const int2 cc = D.ev_cyl[j];
        const int4 m1 = D.cyl_mon[cc.x], m2 = D.cyl_mon[cc.y];
        d3 f[4];
        if (FORCES) {
            U = evm_eval<double, true>(c[0], c[1], c[2], c[3], m1, m2, r.p0, f);
            const int s = D.slot_ev + 4 * j;
            put3(contrib, s, f[0]); put3(contrib, s + 1, f[1]); put3(contrib, s + 2, f[2]); put3(contrib, s + 3, f[3]);
        } else {
            U = evm_eval<double, false>(c[0], c[1], c[2], c[3], m1, m2, r.p0, f);
        }
    } else if (r.type == IT_FS) {
        ff = MDY_FF_FS;
        U = fs_energy(c[0], c[1], r.p0, r.p1);
        if (FORCES) {
            d3 f1, f2;
            fs_force(c[0], c[1], r.p0, r.p1, f1, f2);
            int s = D.slot_fs + 2 * j;
            put3(contrib, s, f1); put3(contrib, s + 1, f2);
        }
    } else if (r.type == IT_FB) {
        ff = MDY_FF_FB;
        U = fb_energy(c[0], c[1], c[2], r.p0, r.p1, r.p2, r.p3);
        if (FORCES) {
            d3 f1, f2, f3;
            fb_force(c[0], c[1], c[2], r.p0, r.p1, r.p2, r.p3, f1, f2, f3);
            int s = D.slot_fb + 3 * j;
            put3(contrib, s, f1); put3(contrib, s + 1, f2); put3(contrib, s + 2, f3);
        }
    } else if (r.type == IT_LM) {
        ff = (j < D.n_ls) ? MDY_FF_LS : MDY_FF_MS;
        U = ls_energy(c[0], c[1], c[2], c[3], r.p0, r.p1, r.p2, r.p3);
        if (FORCES) {
            d3 f1, f2, f3, f4;
            ls_force(c[0], c[1], c[2], c[3], r.p0, r.p1, r.p2, r.p3, f1, f2, f3, f4);
            int s = D.slot_lm + 4 * j;
            put3(contrib, s, f1); put3(contrib, s + 1, f2); put3(contrib, s + 2, f3); put3(contrib, s + 3, f4);
        }
    } else if (r.type == IT_BS) {
        ff = MDY_FF_BS;
        U = bs_energy(c[0], c[1], c[2], r.p0, r.p1, r.p2);
        if (FORCES) {
            d3 f1, f2, f3;
            bs_force(c[0], c[1], c[2], r.p0, r.p1, r.p2, f1, f2, f3);
            int s = D.slot_bs + 3 * j;
            put3(contrib, s, f1); put3(contrib, s + 1, f2); put3(contrib, s + 2, f3);
        }
    } else if (r.type == IT_BB) {
        ff = MDY_FF_BB;
        U = bb_energy(c[0], c[1], c[2], c[3], r.p0, r.p1, r.p2, r.p3);
        if (FORCES) {
            d3 f1, f2, f3, f4;
            bb_force(c[0], c[1], c[2], c[3], r.p0, r.p1, r.p2, r.p3, f1, f2, f3, f4);
            int s = D.slot_bb + 4 * j;
            put3(contrib, s, f1); put3(contrib, s + 1, f2); put3(contrib, s + 2, f3); put3(contrib, s + 3, f4);
        }
    } else if (r.type == IT_BDH) {
        ff = MDY_FF_BDH;
        U = D.bdh_quad ? bdhq_energy(c[0], c[1], c[2], c[3], r.p0, r.p1) : bdh_energy(c[0], c[1], c[2], c[3], r.p0, r.p1);
        if (FORCES) {
            d3 f1, f2, f3, f4;
            if (D.bdh_quad) bdhq_force(c[0], c[1], c[2], c[3], r.p0, r.p1, f1, f2, f3, f4);
            else bdh_force(c[0], c[1], c[2], c[3], r.p0, r.p1, f1, f2, f3, f4);
            int s = D.slot_bdh + 4 * j;
            put3(contrib, s, f1); put3(contrib, s + 1, f2); put3(contrib, s + 2, f3); put3(contrib, s + 3, f4);
        }
    } else if (r.type == IT_BP) {
        ff = MDY_FF_BP;
        U = bp_energy(c[0], c[1], c[2], r.p0, r.p1, D.cq, D.sq);
        if (FORCES) {
            d3 f1, f2, f3;
            bp_force(c[0], c[1], c[2], r.p0, r.p1, D.cq, D.sq, f1, f2, f3);
            int s = D.slot_bp + 3 * j;
            put3(contrib, s, f1); put3(contrib, s + 1, f2); put3(contrib, s + 2, f3);
        }
    } else if (r.type == IT_BD) {
        const double *pl = D.planes + 4 * r.b.y;
        ff = MDY_FF_BD;
        U = bd_energy(pl, c[0], r.p0, r.p1);
        if (FORCES) put3(contrib, D.slot_bd + j, bd_force(pl, c[0], r.p0, r.p1));
    } else {
        add = false;
    }
    if (add) {
        if (xs.x) xs(U);
        if (PER_FF) {
#pragma unroll
            for (int k = 0; k < kNFF; k++) acc[k] += (k == ff) ? U : 0.0;
        }
    }
}

// lane i of the sweep's index space
template <bool MIXED = false, bool QUAD = false, class P>
__device__ __forceinline__ void item(const Dev &D, int i, const P &pos, double acc[kNFF], const XAdd &xs,
                                     typename SlotT<MIXED>::T *__restrict__ contrib, const bool PER_FF,
                                     const bool FORCES) {
    if (i < D.n_duo_lanes()) {
        ev_duo_item<MIXED, QUAD>(D, i, pos, acc, xs, contrib, PER_FF, FORCES);
        return;
    }
    const ItemRec r = fetch_rec(D, i);
    d3 c[4];
    const int o1 = r.type == IT_BD ? r.b.x : r.b.y;   // a boundary record's second entry is its plane
    if (__any(rec_nbeads(r.type) > 2)) {
        const int o[4] = {r.b.x, o1, r.b.z, r.b.w};
        pos.get(o, c);
    } else {   // a wave of stretching or boundary terms
        const int o[2] = {r.b.x, o1};
        d3 q[2];
        pos.get(o, q);
        c[0] = c[2] = c[3] = q[0];
        c[1] = q[1];
    }
    item_compute<MIXED>(D, r, c, acc, xs, contrib, PER_FF, FORCES);
}

// Block blk of nblk's lanes of the index space at positions pos. Chunks of 64
// lanes (a wave) go to the blocks in turn, chunk c to block c % nblk, so that
// every CU gets its share of each kind of item: the kinds are contiguous in the
// index space and differ by a factor of five in time. The terms go into sum 0
// of x (null: forces only).
template <bool MIXED, bool QUAD, class P>
__device__ __forceinline__ void sweep(const Dev &D, const P &pos, int blk, int nblk, double acc[kNFF], XBlock *x,
                                      typename SlotT<MIXED>::T *__restrict__ contrib, const bool PER_FF,
                                      const bool FORCES) {
    const int total = D.n_lanes(), stride = nblk * (int)blockDim.x;
    const int first = (((int)threadIdx.x >> 6) * nblk + blk) * 64 + ((int)threadIdx.x & 63);
    if (FORCES && first == 0) put_none(D, contrib);
    int turn = 0;
    for (int base = 0; base < total; base += stride) {
        if (x && turn == kXTurns) { xblock_norm(*x); turn = 0; }
        turn++;
        const int i = base + first;
        if (i < total) item<MIXED, QUAD>(D, i, pos, acc, XAdd{x, 0}, contrib, PER_FF, FORCES);
        if (total - base <= stride) break;   // base + stride may pass the range of int
    }
}

// Force on one coordinate, o = 3 * bead + axis: its bead's slots in reference
// order, starting from 0.0 (ForceFieldManager::computeForces zero-fills, then
// each force field adds). One lane per coordinate: three lanes share a bead's
// row and read neighboring words of its records, so a wave's loads touch
// about 21 beads' lines instead of 64, and the vectors that the caller reads
// and writes next to it are contiguous. The row comes in groups of four slot
// offsets, filled up with the offset of a record of -0.0, the addition that
// changes nothing; sixteen values are in flight at a time.
constexpr int kRowGroups = 4;
template <class S>
__device__ __forceinline__ double gather_coord(const Dev &D, const S *__restrict__ contrib, int o) {
    const int b = o / 3, c = o - 3 * b;
    const int2 r = D.row[b];
    const int g1 = r.y;
    double f = 0.0;
    for (int g = r.x; g < g1; g += kRowGroups) {
        int4 id[kRowGroups];
        const int none = 3 * D.n_slots;
#pragma unroll
        for (int m = 0; m < kRowGroups; m++) {
            id[m] = D.row_idx[min(g + m, g1 - 1)];
            if (g + m >= g1) id[m] = make_int4(none, none, none, none);
        }
        S v[4 * kRowGroups];
#pragma unroll
        for (int m = 0; m < kRowGroups; m++) {
            v[4 * m] = contrib[id[m].x + c]; v[4 * m + 1] = contrib[id[m].y + c];
            v[4 * m + 2] = contrib[id[m].z + c]; v[4 * m + 3] = contrib[id[m].w + c];
        }
#pragma unroll
        for (int m = 0; m < 4 * kRowGroups; m++) f += v[m];
    }
    return f;
}
// the record that fills up the rows
template <class S>
__device__ __forceinline__ void put_none(const Dev &D, S *__restrict__ contrib) {
    put3(contrib, D.n_slots, vec3_none<S>());
}

// ---- block reductions (fixed butterfly + fixed wave order: deterministic) ----
__device__ __forceinline__ double wave_sum(double v) {
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) v += __shfl_xor(v, o, 64);
    return v;
}
__device__ __forceinline__ double wave_max(double v) {
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) v = fmax(v, __shfl_xor(v, o, 64));
    return v;
}
__device__ __forceinline__ double wave_min(double v) {
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) v = fmin(v, __shfl_xor(v, o, 64));
    return v;
}
__device__ __forceinline__ long long wave_sum_i64(long long v) {
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) v += __shfl_xor(v, o, 64);
    return v;
}
__device__ __forceinline__ int wave_or(int v) {
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) v |= __shfl_xor(v, o, 64);
    return v;
}
// N doubles per thread -> N block results (all threads). Entries whose bit is
// set in max_mask / min_mask are max / min reduced, the rest summed.
// lds: >= 17 * N doubles.
template <int N>
__device__ __forceinline__ void block_reduce(double v[N], double *lds, unsigned max_mask = 0, unsigned min_mask = 0) {
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, nw = blockDim.x >> 6;
#pragma unroll
    for (int k = 0; k < N; k++) {
        double r = ((max_mask >> k) & 1) ? wave_max(v[k]) : ((min_mask >> k) & 1) ? wave_min(v[k]) : wave_sum(v[k]);
        if (lane == 0) lds[wave * N + k] = r;
    }
    __syncthreads();
    if (threadIdx.x < N) {
        int k = threadIdx.x;
        double r = lds[k];
        for (int w = 1; w < nw; w++) {
            double o = lds[w * N + k];
            r = ((max_mask >> k) & 1) ? fmax(r, o) : ((min_mask >> k) & 1) ? fmin(r, o) : r + o;
        }
        lds[16 * N + k] = r;
    }
    __syncthreads();
#pragma unroll
    for (int k = 0; k < N; k++) v[k] = lds[16 * N + k];
    __syncthreads();
}
// Exact block sum of per-thread accumulators (integer digit sums are
// associative, so any tree gives the same result). lds: >= 17 * 8 int64.
__device__ __forceinline__ void block_reduce_xsum(mdy_xsum &s, long long *lds) {
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, nw = blockDim.x >> 6;
    mdy_xs_norm(&s);
#pragma unroll
    for (int k = 0; k < MDY_XS_N; k++) {
        long long r = wave_sum_i64(s.d[k]);
        if (lane == 0) lds[wave * 8 + k] = r;
    }
    int f = wave_or(s.flags);
    if (lane == 0) lds[wave * 8 + 7] = f;
    __syncthreads();
    if (threadIdx.x < 8) {
        int k = threadIdx.x;
        long long r = lds[k];
        for (int w = 1; w < nw; w++) r = (k == 7) ? (r | lds[w * 8 + k]) : r + lds[w * 8 + k];
        lds[128 + k] = r;
    }
    __syncthreads();
#pragma unroll
    for (int k = 0; k < MDY_XS_N; k++) s.d[k] = lds[128 + k];
    s.flags = (int)lds[128 + 7];
    mdy_xs_norm(&s);
    __syncthreads();
}
// per-block partial records: [blk * kRed + off .. off+7] hold a normalized accumulator
__device__ __forceinline__ void store_xsum(double *red, int blk, int off, const mdy_xsum &s) {
    long long *r = reinterpret_cast<long long *>(red) + (size_t)blk * kRed + off;
#pragma unroll
    for (int k = 0; k < MDY_XS_N; k++) r[k] = s.d[k];
    r[7] = s.flags;
}
__device__ __forceinline__ void grid_reduce_xsum(const double *red, int nblk, int off, mdy_xsum &s, long long *lds) {
    mdy_xs_zero(&s);
    const long long *r = reinterpret_cast<const long long *>(red);
    for (int b = threadIdx.x; b < nblk; b += blockDim.x) {
        const long long *q = r + (size_t)b * kRed + off;
#pragma unroll
        for (int k = 0; k < MDY_XS_N; k++) s.d[k] += __builtin_nontemporal_load(q + k);
        s.flags |= (int)__builtin_nontemporal_load(q + 7);
    }
    block_reduce_xsum(s, lds);
}

// Reduce per-block partials red[blk * kRed + off + k] for k < N over nblk
// blocks in a fixed order; every calling block obtains bit-identical results.
template <int N>
__device__ __forceinline__ void grid_partials_reduce(const double *red, int nblk, double v[N], double *lds,
                                                     unsigned max_mask = 0, unsigned min_mask = 0, int off = 0) {
#pragma unroll
    for (int k = 0; k < N; k++) v[k] = ((max_mask >> k) & 1) ? -INFINITY : ((min_mask >> k) & 1) ? INFINITY : 0.0;
    for (int blk = threadIdx.x; blk < nblk; blk += blockDim.x) {
#pragma unroll
        for (int k = 0; k < N; k++) {
            double o = __builtin_nontemporal_load(red + (size_t)blk * kRed + off + k);
            v[k] = ((max_mask >> k) & 1) ? fmax(v[k], o) : ((min_mask >> k) & 1) ? fmin(v[k], o) : v[k] + o;
        }
    }
    block_reduce<N>(v, lds, max_mask, min_mask);
}

// Energy epilogue, shared by the one-shot and persistent kernels. X holds the
// exact total of the analytic energies; v (per_ff) the per-force-field double
// sums. Quadrature-fallback energies (queue qe, values qe_u) are added to
// both, in increasing pair order. e[0..7] per FF (reported values), e[8] =
// computeEnergy total (+inf when a force field returned its -1 sentinel),
// e[9] = the sum without the sentinel.
constexpr int kXsE = 16;   // exact energy total in a reduction record (after the kNFF per-FF sums)
constexpr int kXsA = 24;   // second exact accumulator in a reduction record
static_assert(kNFF <= kXsE && kXsA + 8 <= kRed, "reduction record layout");
__device__ __forceinline__ void energy_finish(mdy_xsum X, const double v_in[kNFF], int nq, const int *qe,
                                              const double *qe_u, double e[kNFF + 2]) {
    double v[kNFF];
    for (int k = 0; k < kNFF; k++) v[k] = v_in ? v_in[k] : 0.0;
    nq = min(nq, kQueueCap);
    bool bad = false;
    if (nq > 0) {
        double add = 0.0;
        int last = -1;
        for (int r = 0; r < nq; r++) {
            int best = -1, bi = 0x7fffffff;
            for (int q = 0; q < nq; q++) {
                int pi = __hip_atomic_load(qe + q, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                if (pi > last && pi < bi) { bi = pi; best = q; }
            }
            if (best < 0) break;
            last = bi;
            double U = qe_u[best];
            if (ev_energy_bad(U)) bad = true;
            else mdy_xs_add(&X, U);
            add += U;
        }
        v[MDY_FF_EV] = bad ? -1.0 : v[MDY_FF_EV] + add;
    }
    for (int k = 0; k < kNFF; k++) e[k] = v[k];
    const double tot = mdy_xs_value(&X);
    e[kNFF] = bad ? INFINITY : tot;
    e[kNFF + 1] = bad ? tot - 1.0 : tot;
}
// The blocks' records added up word by word by one block of kTailBlock threads:
// v the per-FF doubles at [0, kNFF), X (EXACT) the exact total at kXsE; both
// valid in thread 0. Thirty-two lanes read a record's words, 32 records at a
// time with eight loads each in flight (a lane per record held one 256-byte
// stride per load: 33 us for 2048 records).
constexpr int kTailBlock = 1024;
template <bool EXACT>
__device__ __forceinline__ void sum_records(const double *red, int nblk, double v[kNFF], mdy_xsum &X) {
    constexpr int kRows = kTailBlock / kRed, kDeep = 8;
    __shared__ long long part[kRows][kRed];
    const int w = threadIdx.x % kRed, r0 = threadIdx.x / kRed;
    const bool is_d = w < kNFF, is_x = EXACT && w >= kXsE && w < kXsE + 8, is_f = w == kXsE + 7;
    const long long *q = reinterpret_cast<const long long *>(red) + w;
    double d = 0.0;
    long long x = 0;
    if (is_d || is_x)
        for (int r = r0; r < nblk; r += kDeep * kRows) {
            long long u[kDeep];
#pragma unroll
            for (int j = 0; j < kDeep; j++) u[j] = r + j * kRows < nblk ? q[(size_t)(r + j * kRows) * kRed] : 0;
#pragma unroll
            for (int j = 0; j < kDeep; j++) {
                d += __longlong_as_double(u[j]);
                x = is_f ? (x | u[j]) : x + u[j];
            }
        }
    part[r0][w] = is_d ? __double_as_longlong(d) : x;
    __syncthreads();
    if (threadIdx.x < kRed) {
        d = 0.0;
        x = 0;
        for (int r = 0; r < kRows; r++) {
            const long long u = part[r][w];
            d += __longlong_as_double(u);
            x = is_f ? (x | u) : x + u;
        }
        part[0][w] = is_d ? __double_as_longlong(d) : x;
    }
    __syncthreads();
    if (threadIdx.x != 0) return;
    for (int k = 0; k < kNFF; k++) v[k] = __longlong_as_double(part[0][k]);
    if (EXACT) {
        for (int k = 0; k < MDY_XS_N; k++) X.d[k] = part[0][kXsE + k];
        X.flags = (int)part[0][kXsE + 7];
        mdy_xs_norm(&X);
    }
}

// ---- Simpson quadrature fallbacks (CylinderExclVolRepulsion.cpp:884-1254) ----
// The reference advances its abscissae before first use, so interior node i
// sits at (i+1)/N; node values are formed here as (i+1)*(1/N). Sums are exact
// (mdy_xsum), like the CPU path in exact mode.
struct SimpsonGeo { double a, b, c, d, e, F; d3 vA, vB, vC; };
__device__ __forceinline__ SimpsonGeo simpson_geo(d3 c1, d3 c2, d3 c3, d3 c4) {
    SimpsonGeo g;
    g.a = sprod(c1, c2, c1, c2); g.b = sprod(c3, c4, c3, c4); g.c = sprod(c3, c1, c3, c1);
    g.d = sprod(c1, c2, c3, c4); g.e = sprod(c1, c2, c3, c1); g.F = sprod(c3, c4, c3, c1);
    g.vA = sub(c1, c2); g.vB = sub(c3, c4); g.vC = sub(c3, c1);
    return g;
}
__device__ __forceinline__ double eint(const SimpsonGeo &g, double s, double t) {
    double r2 = ev_r2(g.a, g.b, g.c, g.d, g.e, g.F, s, t);
    return (1.0 / (r2 * r2));
}
// energy: terms that node (i, j) adds to Termset2/3/4 (CylinderExclVolRepulsion.cpp:923-958)
__device__ __forceinline__ void simpson_e_node(const SimpsonGeo &g, int i, int j, int N, mdy_xsum &X) {
    const double ds = 1.0 / ((double)N);
    double s = (double)(i + 1) * ds, t = (double)(j + 1) * ds;
    double fs = (i % 2 == 0) ? 2.0 : 4.0, ft = (j % 2 == 0) ? 2.0 : 4.0;
    double v = 0.0;
    if (j == 0 && i > 0 && i < N) v = fs * (eint(g, s, 0.0) + eint(g, s, 1.0));
    if (j > 0 && j < N) {
        if (i == 0) v = ft * (eint(g, 0.0, t) + eint(g, 1.0, t));
        else if (i < N) v = fs * ft * eint(g, s, t);
    }
    mdy_xs_add(&X, v);   // adding an exact 0.0 changes nothing
}
__device__ __forceinline__ double simpson_e_corners(const SimpsonGeo &g) {
    return eint(g, 0.0, 0.0) + eint(g, 0.0, 1.0) + eint(g, 1.0, 0.0) + eint(g, 1.0, 1.0);
}
// force: component q of the six integrands {1, s, s^2, st, t, t^2}/r^6
__device__ __forceinline__ double fint_q(const SimpsonGeo &g, double s, double t, int q) {
    double r2 = ev_r2(g.a, g.b, g.c, g.d, g.e, g.F, s, t);
    double x = (1.0 / (r2 * r2 * r2));
    return q == 0 ? x : q == 1 ? s * x : q == 2 ? s * s * x : q == 3 ? s * t * x : q == 4 ? t * x : t * t * x;
}
__device__ __forceinline__ void simpson_f_node(const SimpsonGeo &g, int i, int j, int N, int q, mdy_xsum &X) {
    const double ds = 1.0 / ((double)N);
    double s = (double)(i + 1) * ds, t = (double)(j + 1) * ds;
    double fs = (i % 2 == 0) ? 2.0 : 4.0, ft = (j % 2 == 0) ? 2.0 : 4.0;
    double v1 = 0.0, v2 = 0.0;   // the node's terms (an exact 0.0 adds nothing)
    if (j == 0 && i > 0 && i < N) {
        v1 = fs * fint_q(g, s, 0.0, q);
        v2 = fs * fint_q(g, s, 1.0, q);
    }
    if (j > 0 && j < N) {
        if (i == 0) {
            v1 = ft * fint_q(g, 0.0, t, q);
            v2 = ft * fint_q(g, 1.0, t, q);
        } else if (i < N) {
            v1 = fs * ft * fint_q(g, s, t, q);
        }
    }
    mdy_xs_add(&X, v1);
    mdy_xs_add(&X, v2);
}
__device__ __forceinline__ void simpson_f_corners(const SimpsonGeo &g, int q, mdy_xsum &X) {
    mdy_xs_add(&X, fint_q(g, 0.0, 0.0, q));
    mdy_xs_add(&X, fint_q(g, 0.0, 1.0, q));
    mdy_xs_add(&X, fint_q(g, 1.0, 0.0, q));
    mdy_xs_add(&X, fint_q(g, 1.0, 1.0, q));
}
__device__ __forceinline__ void simpson_f_assemble(const SimpsonGeo &g, const double T[6], double kr, int N, d3 f[4]) {
    const double ds = 1.0 / ((double)N);
    double in[6];
    for (int q = 0; q < 6; q++) in[q] = (ds * ds / 9.0) * T[q];
    const double A[3] = {g.vA.x, g.vA.y, g.vA.z}, B[3] = {g.vB.x, g.vB.y, g.vB.z}, Cv[3] = {g.vC.x, g.vC.y, g.vC.z};
    double o[4][3];
    for (int k = 0; k < 3; k++) {
        o[0][k] = 4.0 * kr * (-in[0] * Cv[k] + in[1] * (Cv[k] - A[k]) + in[2] * A[k] + in[4] * B[k] - in[3] * B[k]);
        o[1][k] = 4.0 * kr * (-in[1] * Cv[k] - in[2] * A[k] + in[3] * B[k]);
        o[2][k] = 4.0 * kr * (in[0] * Cv[k] + in[1] * A[k] - in[4] * (B[k] + Cv[k]) - in[3] * A[k] + in[5] * B[k]);
        o[3][k] = 4.0 * kr * (in[4] * Cv[k] + in[3] * A[k] - in[5] * B[k]);
    }
    for (int q = 0; q < 4; q++) f[q] = d3{o[q][0], o[q][1], o[q][2]};
}

}  // namespace mdy
