// mdy_hvp.hip -- derivatives of the exact-gradient force field (no coplanar
// perturbation, no Simpson fallback; in the quadrature mode the flagged
// excluded-volume pairs come from mdy_quad.hip) for implicit differentiation
// of minimized structures:
//   * Hessian-vector products H v, by forward-mode differentiation of the
//     force code: bead positions are the dual numbers x + t v, every
//     interaction's forces are evaluated in dual arithmetic and the tangent
//     parts d/dt F(x + t v) = -H v are written (negated) to the interaction's
//     force slots, then gathered per bead in the reference order;
//   * per-force-field directional derivatives grad E_k(x) . w of the
//     energies, from the interaction forces dotted with w at their beads.
#include "mdy_eval.hpp"
#include "mdy_launch.hpp"

namespace mdy {

// Forces of one interaction on its beads in scalar type T (f[0..nbeads));
// returns the force-field index, or -1 for an empty record.
template <class T>
__device__ __forceinline__ int item_forces(const Dev &D, const ItemRec &r, const V3<T> c[4], V3<T> f[4]) {
    if (r.type == IT_EVM) {
        const int2 cc = D.ev_cyl[r.j];
        (void)evm_eval<T, true>(c[0], c[1], c[2], c[3], D.cyl_mon[cc.x], D.cyl_mon[cc.y], r.p0, f);
        return MDY_FF_EV;
    } else if (r.type == IT_FS) {
        fs_force(c[0], c[1], r.p0, r.p1, f[0], f[1]);
        return MDY_FF_FS;
    } else if (r.type == IT_FB) {
        fb_force(c[0], c[1], c[2], r.p0, r.p1, r.p2, r.p3, f[0], f[1], f[2]);
        return MDY_FF_FB;
    } else if (r.type == IT_LM) {
        ls_force(c[0], c[1], c[2], c[3], r.p0, r.p1, r.p2, r.p3, f[0], f[1], f[2], f[3]);
        return r.j < D.n_ls ? MDY_FF_LS : MDY_FF_MS;
    } else if (r.type == IT_BS) {
        bs_force(c[0], c[1], c[2], r.p0, r.p1, r.p2, f[0], f[1], f[2]);
        return MDY_FF_BS;
    } else if (r.type == IT_BB) {
        bb_force(c[0], c[1], c[2], c[3], r.p0, r.p1, r.p2, r.p3, f[0], f[1], f[2], f[3]);
        return MDY_FF_BB;
    } else if (r.type == IT_BDH) {
        if (D.bdh_quad) bdhq_force(c[0], c[1], c[2], c[3], r.p0, r.p1, f[0], f[1], f[2], f[3]);
        else bdh_force(c[0], c[1], c[2], c[3], r.p0, r.p1, f[0], f[1], f[2], f[3]);
        return MDY_FF_BDH;
    } else if (r.type == IT_BP) {
        bp_force(c[0], c[1], c[2], r.p0, r.p1, D.cq, D.sq, f[0], f[1], f[2]);
        return MDY_FF_BP;
    } else if (r.type == IT_BD) {
        f[0] = bd_force(D.planes + 4 * r.b.y, c[0], r.p0, r.p1);
        return MDY_FF_BD;
    }
    return -1;
}

__device__ __forceinline__ int item_slot(const Dev &D, const ItemRec &r) {
    switch (r.type) {
        case IT_EVM: return D.slot_ev + 4 * r.j;
        case IT_FS: return D.slot_fs + 2 * r.j;
        case IT_FB: return D.slot_fb + 3 * r.j;
        case IT_LM: return D.slot_lm + 4 * r.j;
        case IT_BS: return D.slot_bs + 3 * r.j;
        case IT_BB: return D.slot_bb + 4 * r.j;
        case IT_BDH: return D.slot_bdh + 4 * r.j;
        case IT_BP: return D.slot_bp + 3 * r.j;
        default: return D.slot_bd + r.j;
    }
}

__device__ __forceinline__ int bead_off(const ItemRec &r, int k) {
    return k == 0 ? r.b.x : k == 1 ? r.b.y : k == 2 ? r.b.z : r.b.w;
}

// Two waves per SIMD (the compiler fits 256 registers with ~15 words per
// lane spilled; at one wave the kernel needed 286): 13 % faster at 50k.
__global__ void __launch_bounds__(kBlock, 2) k_hvp(Dev D, const double *__restrict__ x, const double *__restrict__ v,
                                                 double *__restrict__ contrib) {
    const int total = D.n_lanes(), gs = gridDim.x * blockDim.x;
    atan_table_fill();
    __syncthreads();
    if (blockIdx.x == 0 && threadIdx.x == 0) put_none(D, contrib);
    for (int i = blockIdx.x * blockDim.x + threadIdx.x; i < total; i += gs) {
        if (i < D.n_duo_lanes()) {   // an excluded-volume pair's two lanes, one per cylinder
            if (D.evq && D.evq[i >> 1]) continue;   // evaluated by the quadrature kernels
            const bool h = (i & 1) != 0;
            const int2 o = reinterpret_cast<const int2 *>(D.ev_bs)[i];
            auto at = [&](int k) {
                return V3<Dual>{Dual(x[k], v[k]), Dual(x[k + 1], v[k + 1]), Dual(x[k + 2], v[k + 2])};
            };
            const V3<Dual> m0 = at(o.x), m1 = at(o.y);
            const V3<Dual> c1 = duo_get<0>(m0), c2 = duo_get<0>(m1), c3 = duo_get<1>(m0), c4 = duo_get<1>(m1);
            EvDuoT<Dual> inv;
            Dual block;
            ev_duo_invariants(h, c1, c2, c3, c4, inv, block);
            V3<Dual> f[2];
            ev_duo_force<Dual>(h, inv, c1, c2, c3, c4, D.ev_kr[i >> 1], f);
#pragma unroll
            for (int k = 0; k < 2; k++) {
                const d3 hv{-f[k].x.d, -f[k].y.d, -f[k].z.d};
                if (!finite_d3(hv)) set_err(D.err, MDY_ERR_FORCE);
                put3(contrib, D.slot_ev + 2 * i + k, hv);
            }
            continue;
        }
        const ItemRec r = fetch_rec(D, i);
        const int nb = rec_nbeads(r.type);
        V3<Dual> c[4], f[4];
#pragma unroll
        for (int k = 0; k < 4; k++) {
            const int o = bead_off(r, k < nb ? k : 0);
            c[k] = V3<Dual>{Dual(x[o], v[o]), Dual(x[o + 1], v[o + 1]), Dual(x[o + 2], v[o + 2])};
        }
        if (item_forces<Dual>(D, r, c, f) < 0) continue;
        const int s = item_slot(D, r);
        bool ok = true;
#pragma unroll
        for (int k = 0; k < 4; k++) {
            if (k < nb) {
                const d3 h{-f[k].x.d, -f[k].y.d, -f[k].z.d};   // -dF/dt = H v
                ok = ok && finite_d3(h);
                put3(contrib, s + k, h);
            }
        }
        // a degenerate excluded-volume pair has no analytic second derivative
        if (!ok) set_err(D.err, MDY_ERR_FORCE);
    }
}

__global__ void __launch_bounds__(kBlock) k_hvp_gather(Dev D, const double *__restrict__ contrib,
                                                        double *__restrict__ hv, long long *told) {
    if (told && blockIdx.x == 0 && threadIdx.x == 0) *told = *D.err;
    for (int o = blockIdx.x * blockDim.x + threadIdx.x; o < D.ndof; o += gridDim.x * blockDim.x)
        hv[o] = gather_coord(D, contrib, o);
}

// per-block partial sums of grad E_k . w = -sum over an interaction's beads of F . w
__global__ void __launch_bounds__(kBlock) k_energy_jvp(Dev D, const double *__restrict__ x,
                                                        const double *__restrict__ w, double *red) {
    __shared__ double lds[17 * kNFF + 8];
    double acc[kNFF];
#pragma unroll
    for (int k = 0; k < kNFF; k++) acc[k] = 0.0;
    const int total = D.n_lanes(), gs = gridDim.x * blockDim.x;
    bool ok = true;
    atan_table_fill();
    __syncthreads();
    for (int i = blockIdx.x * blockDim.x + threadIdx.x; i < total; i += gs) {
        if (i < D.n_duo_lanes()) {   // an excluded-volume pair's two lanes, one per cylinder
            if (D.evq && D.evq[i >> 1]) continue;   // evaluated by the quadrature kernels
            const bool h = (i & 1) != 0;
            const int2 o = reinterpret_cast<const int2 *>(D.ev_bs)[i];
            const d3 m0 = ld3(x + o.x), m1 = ld3(x + o.y);
            const d3 c1 = duo_get<0>(m0), c2 = duo_get<0>(m1), c3 = duo_get<1>(m0), c4 = duo_get<1>(m1);
            EvDuoT<double> inv;
            double block;
            ev_duo_invariants(h, c1, c2, c3, c4, inv, block);
            d3 f[2];
            ev_duo_force<double>(h, inv, c1, c2, c3, c4, D.ev_kr[i >> 1], f);
            ok = ok && finite_d3(f[0]) && finite_d3(f[1]);
            acc[MDY_FF_EV] -= f[0].x * w[o.x] + f[0].y * w[o.x + 1] + f[0].z * w[o.x + 2] + f[1].x * w[o.y] +
                              f[1].y * w[o.y + 1] + f[1].z * w[o.y + 2];
            continue;
        }
        const ItemRec r = fetch_rec(D, i);
        const int nb = rec_nbeads(r.type);
        d3 c[4], f[4];
#pragma unroll
        for (int k = 0; k < 4; k++) {
            const int o = bead_off(r, k < nb ? k : 0);
            c[k] = d3{x[o], x[o + 1], x[o + 2]};
        }
        const int ff = item_forces<double>(D, r, c, f);
        if (ff < 0) continue;
        double s = 0.0;
#pragma unroll
        for (int k = 0; k < 4; k++) {
            if (k < nb) {
                const int o = bead_off(r, k);
                ok = ok && finite_d3(f[k]);
                s -= f[k].x * w[o] + f[k].y * w[o + 1] + f[k].z * w[o + 2];
            }
        }
#pragma unroll
        for (int k = 0; k < kNFF; k++) acc[k] += (k == ff) ? s : 0.0;
    }
    if (!ok) set_err(D.err, MDY_ERR_FORCE);
    block_reduce<kNFF>(acc, lds);
    if (threadIdx.x < kNFF) red[(size_t)blockIdx.x * kRed + threadIdx.x] = acc[threadIdx.x];
}

// err, told: the error word and where the host reads it
__global__ void __launch_bounds__(kTailBlock) k_energy_jvp_final(const double *red, int nblk, double *out, const int *err,
                                                                 long long *told) {
    double v[kNFF];
    mdy_xsum none;
    sum_records<false>(red, nblk, v, none);
    if (threadIdx.x == 0) {
        double t = 0.0;
        for (int k = 0; k < kNFF; k++) {
            out[k] = v[k];
            t += v[k];
        }
        out[kNFF] = t;
        *told = *err;
    }
}

__global__ void k_tell_err(const int *err, long long *told) { *told = *err; }
__global__ void k_clear_err(int *err) { *err = 0; }

static int grid_of(const Ctx &c, long long n) {
    long long g = (n + kBlock - 1) / kBlock, cap = (long long)c.num_cu * 8;
    return (int)(g > cap ? cap : g < 1 ? 1 : g);
}

// The error word after the stream's work, from pinned memory, where the last
// kernel has written it (a copy to pageable memory took 9 us more); cleared if set.
static int told_errors(Ctx &c, hipStream_t st) {
    if (hipGetLastError() != hipSuccess) return MDY_ERR_HIP;
    if (hipStreamSynchronize(st) != hipSuccess) return MDY_ERR_HIP;
    const int e = (int)c.h_out[kOutErr];
    if (e) {
        hipLaunchKernelGGL(k_clear_err, dim3(1), dim3(1), 0, st, c.err.p);
        if (hipStreamSynchronize(st) != hipSuccess) return MDY_ERR_HIP;
    }
    return e;
}
int sync_errors(Ctx &c, hipStream_t st) {
    hipLaunchKernelGGL(k_tell_err, dim3(1), dim3(1), 0, st, c.err.p, c.h_out + kOutErr);
    return told_errors(c, st);
}

// H v's slots; the quadrature pairs' classification stays for another product with `keep`
static int hvp_slots(Ctx &c, const Dev &D, const double *d_x, const double *d_v, hipStream_t st, bool keep) {
    hipLaunchKernelGGL(k_hvp, dim3(grid_of(c, D.n_lanes())), dim3(kBlock), 0, st, D, d_x, d_v, c.contrib.p);
    return quad_on(c) ? launch_quad(c, D, 2, d_x, d_v, c.contrib.p, 0, st, keep) : MDY_OK;
}

int launch_hvp(Ctx &c, const double *d_x, const double *d_v, double *d_hv, hipStream_t st, bool sync) {
    Dev D = c.dev();
    if (quad_on(c)) MDY_TRY(quad_classify(c, D, d_x, st));
    MDY_TRY(hvp_slots(c, D, d_x, d_v, st, false));
    hipLaunchKernelGGL(k_hvp_gather, dim3(grid_of(c, D.ndof)), dim3(kBlock), 0, st, D, c.contrib.p, d_hv,
                       sync ? c.h_out + kOutErr : nullptr);
    if (!sync) return hipGetLastError() == hipSuccess ? MDY_OK : MDY_ERR_HIP;
    return told_errors(c, st);
}

// ---------------------------------------------------------------------------
// (H + shift I) w = b by conjugate gradients. An iteration is H p's slots and
// three kernels: the gather with p.Hp, the step along p with r.r, and the next
// direction. Each sums the block sums of the one before, in a fixed order, so
// the scalars stay on the device and no iteration waits for the host, which
// enqueues kSolveAhead iterations ahead of the last one it has seen end; after the
// stop, the kernels of those do nothing to w, r and p. No kernel writes a scalar
// that its own blocks test: k_solve_dir writes the stop, which the next gather
// hands on to the next k_solve_dir, so every block of a launch sees the same. Bound by the latency of
// its kernels (six with quadrature pairs) at a few thousand cylinders: 32 us
// per iteration at 5k; one product with a host wait and its own classification
// of the pairs, two dot products read back and five vector kernels took 126.
// ---------------------------------------------------------------------------
constexpr int kSolveAhead = 2;
// scalars: r.r of even and odd iterations, the reason to stop, iterations done, the last p.(H + shift I)p,
// the stop as the iteration's gather saw it
enum { S_RR = 0, S_STOP = 2, S_ITER, S_PHP, S_SEEN, S_SUMS = 8 };
enum { STOP_CONVERGED = 1, STOP_CURVATURE, STOP_ERROR };

__global__ void k_solve_begin(double *s, double rr) {
    s[S_RR] = rr;
    s[S_STOP] = s[S_ITER] = s[S_PHP] = s[S_SEEN] = 0.0;
}

// the blocks' sums added up by every block alike
__device__ __forceinline__ double sum_of_blocks(const double *__restrict__ part, int n, double *lds) {
    double v[1] = {0.0};
    for (int k = threadIdx.x; k < n; k += blockDim.x) v[0] += part[k];
    block_reduce<1>(v, lds);
    return v[0];
}

__global__ void __launch_bounds__(kBlock) k_solve_gather(Dev D, const double *__restrict__ contrib,
                                                         const double *__restrict__ p, double shift,
                                                         double *__restrict__ hp, double *s,
                                                         double *__restrict__ part) {
    __shared__ double lds[24];
    const double stop = s[S_STOP];
    if (blockIdx.x == 0 && threadIdx.x == 0) s[S_SEEN] = stop;
    if (stop != 0.0) return;
    double v[1] = {0.0};
    for (int o = blockIdx.x * blockDim.x + threadIdx.x; o < D.ndof; o += gridDim.x * blockDim.x) {
        const double q = p[o], h = __builtin_fma(shift, q, gather_coord(D, contrib, o));
        hp[o] = h;
        v[0] = __builtin_fma(q, h, v[0]);
    }
    block_reduce<1>(v, lds);
    if (threadIdx.x == 0) part[blockIdx.x] = v[0];
}

__global__ void __launch_bounds__(kBlock) k_solve_step(int n, int odd, double *s, const double *__restrict__ php_part,
                                                       int nphp, const double *__restrict__ p,
                                                       const double *__restrict__ hp, double *__restrict__ w,
                                                       double *__restrict__ r, double *__restrict__ rr_part) {
    __shared__ double lds[24];
    if (s[S_STOP] != 0.0) return;
    const double php = sum_of_blocks(php_part, nphp, lds);   // the same in every block
    if (blockIdx.x == 0 && threadIdx.x == 0) s[S_PHP] = php;
    if (!(php > 0.0)) return;
    const double a = s[S_RR + odd] / php;
    double v[1] = {0.0};
    for (int o = blockIdx.x * blockDim.x + threadIdx.x; o < n; o += gridDim.x * blockDim.x) {
        w[o] = __builtin_fma(a, p[o], w[o]);
        const double q = __builtin_fma(-a, hp[o], r[o]);
        r[o] = q;
        v[0] = __builtin_fma(q, q, v[0]);
    }
    block_reduce<1>(v, lds);
    if (threadIdx.x == 0) rr_part[blockIdx.x] = v[0];
}

// told: pinned, the reason to stop
__global__ void __launch_bounds__(kBlock) k_solve_dir(int n, int odd, double *s, const double *__restrict__ rr_part,
                                                      int nrr, const double *__restrict__ r, double *__restrict__ p,
                                                      double tol, const int *err, long long *told) {
    __shared__ double lds[24];
    const bool first = blockIdx.x == 0 && threadIdx.x == 0;
    if (s[S_SEEN] != 0.0) return;
    if (!(s[S_PHP] > 0.0)) {   // no step was taken; p is the direction to report
        if (first) {
            s[S_STOP] = STOP_CURVATURE;
            *told = *err ? STOP_ERROR : STOP_CURVATURE;
        }
        return;
    }
    const double rr = sum_of_blocks(rr_part, nrr, lds), beta = rr / s[S_RR + odd];
    for (int o = blockIdx.x * blockDim.x + threadIdx.x; o < n; o += gridDim.x * blockDim.x)
        p[o] = __builtin_fma(p[o], beta, r[o]);
    if (first) {
        s[S_RR + 1 - odd] = rr;
        s[S_ITER] += 1.0;
        const int why = *err ? STOP_ERROR : !(rr > tol) ? STOP_CONVERGED : 0;
        if (why) {
            s[S_STOP] = why;
            *told = why;
        }
    }
}

static int solve_loop(Ctx &c, const Dev &D, const double *d_x, double *d_w, double *d_r, double *d_p, double *d_hp,
                      double tol, int maxiter, double shift, hipStream_t st, hipEvent_t *ended) {
    const int n = D.ndof, ng = grid_of(c, n), nv = ng < c.num_cu ? ng : c.num_cu;
    double *s = c.solve.p, *php = s + S_SUMS, *rr = php + ng;
    volatile long long *told = c.h_out + kOutSolve;
    for (int it = 0; it < maxiter && *told == 0; it++) {
        if (it >= kSolveAhead) {
            MDY_HIP(hipEventSynchronize(ended[it % kSolveAhead]));
            if (*told != 0) break;
        }
        MDY_TRY(hvp_slots(c, D, d_x, d_p, st, true));
        hipLaunchKernelGGL(k_solve_gather, dim3(ng), dim3(kBlock), 0, st, D, c.contrib.p, d_p, shift, d_hp, s, php);
        hipLaunchKernelGGL(k_solve_step, dim3(nv), dim3(kBlock), 0, st, n, it & 1, s, php, ng, d_p, d_hp, d_w, d_r, rr);
        hipLaunchKernelGGL(k_solve_dir, dim3(nv), dim3(kBlock), 0, st, n, it & 1, s, rr, nv, d_r, d_p, tol, c.err.p,
                           c.h_out + kOutSolve);
        MDY_HIP(hipGetLastError());
        MDY_HIP(hipEventRecord(ended[it % kSolveAhead], st));
    }
    return MDY_OK;
}

int solve_hessian(Ctx &c, const double *d_x, double *d_w, double *d_r, double *d_p, double *d_hp, double rr, double tol,
                  int maxiter, double shift, hipStream_t st, mdy_solve_result *res) {
    Dev D = c.dev();
    MDY_TRY(ensure(c.solve, S_SUMS + 2 * (size_t)grid_of(c, D.ndof)));
    hipEvent_t ended[kSolveAhead] = {};
    int rc = MDY_OK;
    for (hipEvent_t &e : ended)
        if (hipEventCreateWithFlags(&e, hipEventDisableTiming) != hipSuccess) rc = MDY_ERR_HIP;
    c.h_out[kOutSolve] = 0;
    const bool quad = quad_on(c);
    if (rc == MDY_OK) {
        hipLaunchKernelGGL(k_solve_begin, dim3(1), dim3(1), 0, st, c.solve.p, rr);
        if (quad) rc = quad_classify(c, D, d_x, st);
        if (rc == MDY_OK) {
            rc = solve_loop(c, D, d_x, d_w, d_r, d_p, d_hp, tol, maxiter, shift, st, ended);
            if (quad && quad_end(c, st) != MDY_OK) rc = MDY_ERR_HIP;
        }
    }
    // errors of the products, and the end of everything enqueued
    const int e = sync_errors(c, st);
    if (rc == MDY_OK) rc = e;
    for (hipEvent_t &v : ended)
        if (v) (void)hipEventDestroy(v);
    if (rc != MDY_OK) return rc;
    double s[S_SUMS];
    MDY_HIP(hipMemcpy(s, c.solve.p, sizeof(s), hipMemcpyDeviceToHost));
    res->iterations = (int32_t)s[S_ITER];
    res->residual_sq = s[S_RR + (res->iterations & 1)];
    res->curvature = s[S_PHP];
    res->not_positive = s[S_STOP] == STOP_CURVATURE;
    return MDY_OK;
}

int launch_energy_jvp(Ctx &c, const double *d_x, const double *d_w, double *d_out, hipStream_t st) {
    Dev D = c.dev();
    const int nblk = grid_of(c, D.n_lanes());
    const bool quad = quad_on(c);
    const int nqb = quad ? quad_blocks(c) : 0;   // the quadrature pairs' block records follow the others
    MDY_TRY(ensure(c.red, (size_t)kRed * (nblk + nqb)));
    if (quad) MDY_TRY(quad_classify(c, D, d_x, st));
    hipLaunchKernelGGL(k_energy_jvp, dim3(nblk), dim3(kBlock), 0, st, D, d_x, d_w, c.red.p);
    if (quad) MDY_TRY(launch_quad(c, D, 3, d_x, d_w, c.red.p, nblk, st));
    hipLaunchKernelGGL(k_energy_jvp_final, dim3(1), dim3(kTailBlock), 0, st, c.red.p, nblk + nqb, d_out, c.err.p,
                       c.h_out + kOutErr);
    return told_errors(c, st);
}

}  // namespace mdy
