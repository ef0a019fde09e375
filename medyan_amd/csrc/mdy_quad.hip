// mdy_quad.hip -- excluded-volume pairs evaluated by quadrature of their
// defining integral (MDY_COPLANAR_QUADRATURE).
//
// The cylinder-cylinder excluded-volume energy is
//     E = kr * Int_0^1 Int_0^1 ds dt / |P(s) - Q(t)|^4,
//     P(s) = c1 + s (c2 - c1),  Q(t) = c3 + t (c4 - c3),
// which CylinderExclVolRepulsion::energy (CylinderExclVolRepulsion.cpp:
// 28-120) evaluates in closed form. For nearly coplanar or nearly parallel
// cylinders that closed form is a difference of nearly equal atan terms
// divided by a vanishing triple product: the rounding of its FP64 terms is
// amplified as ~5e-14 / q, where q is the squared normalized triple product
// (v1 x v2 . v3)^2 / (|v1|^2 |v2|^2 |v3|^2), so its second derivatives are
// dominated by rounding noise there. In this mode the pairs with q < 1e-3
// (about 2-5% of the pairs of a random network; closed-form force error
// below ~5e-11 elsewhere) are evaluated instead by a composite 16-point
// Gauss-Legendre rule in s and t: m equal panels per cylinder, m =
// ceil(max length / segment distance) (at most 64), so every panel is no
// longer than the distance to the other segment and the rule's error is
// below ~1e-19 of the integral. Energy, forces, Hessian-vector products and
// directional derivatives of a pair all differentiate the same discrete
// rule, so they are mutually consistent to rounding.
//
// Work is split by tiles, a panel of s times a panel of t (16 x 16 nodes). A
// pair of up to 8 x 8 panels is split into pieces of 4 tiles, each one wave's
// work; a larger one into at most 16 pieces of at least 64 tiles, each one
// block's, whose waves take its tiles in turn (so the closest pair does not
// set the kernel's time). k_ev_classify flags the pairs and places their
// pieces, k_quad_nodes sums each one's nodes (each lane a fixed subset in a
// fixed order, then a fixed tree) into a record, and one thread per pair adds
// its records in order. Results are reproducible bit for bit. The closed-form
// kernels skip the flagged pairs.
#include <algorithm>
#include <cmath>

#include "mdy_eval.hpp"
#include "mdy_launch.hpp"

namespace mdy {

constexpr double kQuadMaxQ = 1e-3;   // pairs with q below this are integrated numerically
constexpr int kQuadPanels = 64;      // at most this many panels per cylinder
constexpr int kWavePanels = 8;       // pairs of up to this many panels go to waves, others to blocks
constexpr int kWaveTiles = 4;        // a wave's piece
constexpr int kBlockTiles = 64;      // a block's piece, at least
constexpr int kPieces = 16;          // at most this many pieces per pair
constexpr int kQuadBlock = 1024;     // threads per block of k_quad_nodes
constexpr int kQuadWaves = kQuadBlock / 64;
static_assert(kWavePanels * kWavePanels <= kPieces * kWaveTiles, "pieces of the largest wave pair");

// tiles in a piece of a pair of m panels
__device__ __forceinline__ int piece_tiles(int m) {
    return m <= kWavePanels ? kWaveTiles : max(kBlockTiles, (m * m + kPieces - 1) / kPieces);
}

// 16-point Gauss-Legendre nodes and weights on [0, 1], ascending
struct GL16 {
    double t[16], w[16];
};

// Newton iteration on the Legendre polynomial P_16 in long double from the
// standard cosine initial guesses; weights 2 / ((1 - x^2) P_16'(x)^2).
static GL16 make_gl16() {
    GL16 g;
    const int n = 16;
    for (int i = 0; i < n; i++) {
        long double x = cosl(3.14159265358979323846264338327950288L * (i + 0.75L) / (n + 0.5L));
        long double p0 = 1, p1 = x, dp = 1;
        for (int it = 0; it < 100; it++) {
            p0 = 1;
            p1 = x;
            for (int k = 2; k <= n; k++) {
                const long double p2 = ((2 * k - 1) * x * p1 - (k - 1) * p0) / k;
                p0 = p1;
                p1 = p2;
            }
            dp = n * (x * p1 - p0) / (x * x - 1);
            const long double dx = p1 / dp;
            x -= dx;
            if (fabsl(dx) < 1e-30L) break;
        }
        p0 = 1;
        p1 = x;
        for (int k = 2; k <= n; k++) {
            const long double p2 = ((2 * k - 1) * x * p1 - (k - 1) * p0) / k;
            p0 = p1;
            p1 = p2;
        }
        dp = n * (x * p1 - p0) / (x * x - 1);
        g.t[i] = (double)(0.5L * (1 - x));
        g.w[i] = (double)(1 / ((1 - x * x) * dp * dp));   // (2 / ...) * 1/2 for [0, 1]
    }
    return g;
}

static const GL16 &gl16() {
    static const GL16 g = make_gl16();
    return g;
}

__device__ __forceinline__ d3 ld3(const double *x, int o) { return d3{x[o], x[o + 1], x[o + 2]}; }
__device__ __forceinline__ double dot3(d3 a, d3 b) { return a.x * b.x + a.y * b.y + a.z * b.z; }

// q = (v1 x v2 . v3)^2 / (|v1|^2 |v2|^2 |v3|^2); NaN (degenerate pair) counts as flagged
__device__ __forceinline__ bool needs_quadrature(d3 c1, d3 c2, d3 c3, d3 c4) {
    const d3 v1 = sub(c2, c1), v2 = sub(c4, c3), v3 = sub(c3, c1);
    const d3 n{v1.y * v2.z - v1.z * v2.y, v1.z * v2.x - v1.x * v2.z, v1.x * v2.y - v1.y * v2.x};
    const double tp = dot3(n, v3);
    const double q = tp * tp / (dot3(v1, v1) * dot3(v2, v2) * dot3(v3, v3));
    return !(q >= kQuadMaxQ);
}

// the distance helper is defined below; declared here for the classifier
__device__ __forceinline__ double segment_distance(d3 c1, d3 c2, d3 c3, d3 c4);

// panels per cylinder: each no longer than the segments' distance (at most kQuadPanels)
__device__ __forceinline__ int quad_panels(d3 c1, d3 c2, d3 c3, d3 c4) {
    const d3 v1 = sub(c2, c1), v2 = sub(c4, c3);
    const double L = sqrt(fmax(dot3(v1, v1), dot3(v2, v2)));
    const double dm = segment_distance(c1, c2, c3, c4);
    const double mr = dm > 0.0 ? ceil(L / dm) : (double)kQuadPanels;
    return mr >= (double)kQuadPanels ? kQuadPanels : mr <= 1.0 ? 1 : (int)mr;
}

// flag[j]; for a flagged pair the panel count pan[j], its record count cnt[j]
// and its first record off[j], and the record -> pair map. Blocks' pieces take
// records from the front of the cap records, waves' from the back: tot holds the
// blocks' count in its low and the waves' in its high half, taken
// atomically (the order of pairs among the records changes no result, since
// each record's nodes and each pair's sum over its records are fixed).
__global__ void __launch_bounds__(kBlock) k_ev_classify(Dev D, const double *__restrict__ x,
                                                         unsigned char *__restrict__ flag, int *__restrict__ pan,
                                                         int *__restrict__ cnt, int *__restrict__ off,
                                                         int *__restrict__ map, unsigned long long *__restrict__ tot,
                                                         int cap) {
    // one atomic per block and sweep turn: the block's counts are scanned in
    // LDS (wave prefix sums, then the wave totals), both halves at once
    __shared__ unsigned long long wsum[kBlock / 64];
    __shared__ unsigned long long bbase;
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    for (int j0 = blockIdx.x * blockDim.x; j0 < D.n_ev; j0 += gridDim.x * blockDim.x) {
        const int j = j0 + threadIdx.x;
        int nc = 0, m = 0;
        if (j < D.n_ev) {
            const int4 b = D.ev_bs[j];
            const d3 c1 = ld3(x, b.x), c2 = ld3(x, b.y), c3 = ld3(x, b.z), c4 = ld3(x, b.w);
            const bool f = needs_quadrature(c1, c2, c3, c4);
            flag[j] = f ? 1 : 0;
            if (f) {
                m = quad_panels(c1, c2, c3, c4);
                const int pt = piece_tiles(m);
                nc = (m * m + pt - 1) / pt;
            }
        }
        const bool to_waves = m <= kWavePanels;
        const unsigned long long mine = to_waves ? (unsigned long long)nc << 32 : (unsigned long long)nc;
        unsigned long long incl = mine;   // inclusive prefix within the wave
#pragma unroll
        for (int o = 1; o < 64; o <<= 1) {
            const unsigned long long v = __shfl_up(incl, o, 64);
            if (lane >= o) incl += v;
        }
        if (lane == 63) wsum[wave] = incl;
        __syncthreads();
        if (threadIdx.x == 0) {
            unsigned long long s = 0;
            for (int w = 0; w < kBlock / 64; w++) { const unsigned long long v = wsum[w]; wsum[w] = s; s += v; }
            bbase = s ? atomicAdd(tot, s) : 0;
        }
        __syncthreads();
        if (j < D.n_ev) {
            if (nc) {
                const unsigned long long at = bbase + wsum[wave] + incl - mine;
                const long long base = to_waves ? (long long)cap - nc - (long long)(at >> 32) : (long long)(at & 0xffffffffull);
                pan[j] = m;
                if (base >= 0 && base + nc <= cap) {
                    off[j] = (int)base;
                    for (int q = 0; q < nc; q++) map[base + q] = j;
                } else {   // cannot happen with a cleared total (kPieces records per pair at most)
                    nc = 0;
                    set_err(D.err, MDY_ERR_CAPACITY);
                }
            }
            cnt[j] = nc;
        }
        __syncthreads();   // wsum and bbase are rewritten by the next turn
    }
}

__global__ void k_quad_zero(unsigned long long *tot) { *tot = 0; }

__device__ __forceinline__ double clamp01(double v) { return v < 0.0 ? 0.0 : v > 1.0 ? 1.0 : v; }

// Distance between the segments c1-c2 and c3-c4: the minimum over the unit
// square of |c1 + s d1 - c3 - t d2|, from the stationary point of that
// quadratic, clamped to the square edge by edge (for parallel segments s
// starts at 0).
__device__ __forceinline__ double segment_distance(d3 c1, d3 c2, d3 c3, d3 c4) {
    const d3 d1 = sub(c2, c1), d2 = sub(c4, c3), r = sub(c1, c3);
    const double a = dot3(d1, d1), e = dot3(d2, d2), f = dot3(d2, r), c = dot3(d1, r), b = dot3(d1, d2);
    const double den = a * e - b * b;
    double s = den > 1e-14 * a * e ? clamp01((b * f - c * e) / den) : 0.0;
    double t = (b * s + f) / e;
    if (t < 0.0) {
        t = 0.0;
        s = clamp01(-c / a);
    } else if (t > 1.0) {
        t = 1.0;
        s = clamp01((b - c) / a);
    }
    const d3 p{r.x + s * d1.x - t * d2.x, r.y + s * d1.y - t * d2.y, r.z + s * d1.z - t * d2.z};
    return sqrt(dot3(p, p));
}

enum { Q_ENERGY = 0, Q_FORCE = 1, Q_HVP = 2, Q_JVP = 3 };
template <int W> struct QuadAcc { static constexpr int N = W == Q_ENERGY ? 1 : 9; };

// Sum over the wave, the same bits in every lane: 16 lanes by data-parallel
// moves (no LDS), then the four rows.
template <int CTRL> __device__ __forceinline__ double dpp_add(double v) {
    const int hi = __builtin_amdgcn_update_dpp(0, __double2hiint(v), CTRL, 0xf, 0xf, true);
    const int lo = __builtin_amdgcn_update_dpp(0, __double2loint(v), CTRL, 0xf, 0xf, true);
    return v + __hiloint2double(hi, lo);
}
__device__ __forceinline__ double wave_total(double v) {
    v = dpp_add<0xB1>(v);    // lanes 1 0 3 2
    v = dpp_add<0x4E>(v);    // lanes 2 3 0 1
    v = dpp_add<0x141>(v);   // 7 - lane, within eight
    v = dpp_add<0x140>(v);   // 15 - lane, within sixteen
    v += __shfl_xor(v, 16, 64);
    return v + __shfl_xor(v, 32, 64);
}

// The nodes of one lane: s node lane % 16 and the four t nodes lane / 16 + 4 q of a tile.
// The t nodes stay in LDS (tw: node and weight): in registers they made H v spill.
struct LaneNodes { double s, ws; const double2 *tw; };

// Tiles k0, k0 + step, ... below k1 of pair j by one wave, summed into acc in
// every lane: for Q_ENERGY the sum of W |r|^-4; otherwise G, sum of s h, sum
// of t h with h = W r/|r|^6 (Q_FORCE, Q_JVP: minus the gradient of |r|^-4, but
// for its factor 4) or h = W grad^2 |r|^-4 dr / 4 (Q_HVP, dr the direction v
// along r). What depends on s only leaves the loop over t.
template <int W>
__device__ __forceinline__ void quad_tiles(const Dev &D, const double *__restrict__ x, const double *__restrict__ v,
                                           const LaneNodes &L, int j, int m, int k0, int k1, int step,
                                           double acc[QuadAcc<W>::N]) {
    constexpr int NA = QuadAcc<W>::N;
    const int4 b = D.ev_bs[j];
    const d3 c1 = ld3(x, b.x), c2 = ld3(x, b.y), c3 = ld3(x, b.z), c4 = ld3(x, b.w);
    const d3 v1 = sub(c2, c1), v2 = sub(c4, c3), c13 = sub(c1, c3);
    d3 e1{0, 0, 0}, e2{0, 0, 0}, e13{0, 0, 0};   // HVP: the direction at (c2 - c1), (c4 - c3), (c1 - c3)
    if (W == Q_HVP) {
        const d3 u1 = ld3(v, b.x), u2 = ld3(v, b.y), u3 = ld3(v, b.z), u4 = ld3(v, b.w);
        e1 = sub(u2, u1);
        e2 = sub(u4, u3);
        e13 = sub(u1, u3);
    }
    auto at = [](d3 o, double k, d3 d) {
        return d3{__builtin_fma(k, d.x, o.x), __builtin_fma(k, d.y, o.y), __builtin_fma(k, d.z, o.z)};
    };
    const double im = 1.0 / (double)m;
    int ps = k0 / m, pt = k0 - ps * m;
    for (int k = k0; k < k1; k += step) {
        const double s = ((double)ps + L.s) * im;
        const d3 rs = at(c13, s, v1), es = at(e13, s, e1);
        double g[NA == 1 ? 1 : 6];
#pragma unroll
        for (int q = 0; q < (NA == 1 ? 1 : 6); q++) g[q] = 0.0;
#pragma unroll 2
        for (int q = 0; q < 4; q++) {
            const double2 nt = L.tw[4 * q];
            const double t = ((double)pt + nt.x) * im;
            const d3 r = at(rs, -t, v2);
            const double d2 = __builtin_fma(r.z, r.z, __builtin_fma(r.y, r.y, r.x * r.x));
            const double inv = 1.0 / d2, inv2 = inv * inv;
            if (W == Q_ENERGY) {
                g[0] = __builtin_fma(nt.y, inv2, g[0]);
            } else {
                const double a = nt.y * (inv2 * inv);
                d3 h;
                if (W == Q_HVP) {
                    // d/dt of the gradient of |r|^-4 along dr, over 4: -dr/|r|^6 + 6 (r.dr) r/|r|^8
                    const d3 dr = at(es, -t, e2);
                    const double rd = __builtin_fma(r.z, dr.z, __builtin_fma(r.y, dr.y, r.x * dr.x));
                    const double c = 6.0 * (a * inv) * rd;
                    h = d3{__builtin_fma(c, r.x, -a * dr.x), __builtin_fma(c, r.y, -a * dr.y),
                           __builtin_fma(c, r.z, -a * dr.z)};
                } else {
                    h = d3{a * r.x, a * r.y, a * r.z};
                }
                g[0] += h.x; g[1] += h.y; g[2] += h.z;
                g[3] = __builtin_fma(t, h.x, g[3]); g[4] = __builtin_fma(t, h.y, g[4]); g[5] = __builtin_fma(t, h.z, g[5]);
            }
        }
        acc[0] += g[0];
        if constexpr (NA > 1) {
            acc[1] += g[1]; acc[2] += g[2];
            acc[3] = __builtin_fma(s, g[0], acc[3]); acc[4] = __builtin_fma(s, g[1], acc[4]);
            acc[5] = __builtin_fma(s, g[2], acc[5]);
            acc[6] += g[3]; acc[7] += g[4]; acc[8] += g[5];
        }
        for (pt += step; pt >= m; pt -= m) ps++;
    }
    // the weights' common factors: w_s / m^2, and the gradient's 4
    const double f = (W == Q_ENERGY ? 1.0 : 4.0) * L.ws * (im * im);
#pragma unroll
    for (int q = 0; q < NA; q++) acc[q] = wave_total(acc[q] * f);
}

// The records' sums: the blocks' pieces first, one per block and turn, then the
// waves', one per wave and turn. Bound by FP64 instruction issue on the CUs
// that hold the closest pairs, and by a wave's chain of about 16 nodes; a lane
// keeps its s node through a tile, and pieces are small so that they spread
// over the CUs. At 66k pairs, 1.5k of them flagged, H v / force / energy take
// 32 / 26 / 17 us; 107 / 89 / 67 with one block of 256 threads per 65536 nodes,
// a division of the node's number into s and t and a block reduction per pair;
// 49 / 41 / 28 with pieces of 16 tiles per wave and 256 per block.
template <int W>
__global__ void __launch_bounds__(kQuadBlock) k_quad_nodes(Dev D, const double *__restrict__ x,
                                                           const double *__restrict__ v, GL16 g,
                                                           const int *__restrict__ off, const int *__restrict__ map,
                                                           const int *__restrict__ pan,
                                                           const unsigned long long *__restrict__ tot, int cap,
                                                           double *__restrict__ part) {
    constexpr int NA = QuadAcc<W>::N;
    __shared__ double sum[kQuadWaves][NA];
    __shared__ double2 tw[16];   // the rule, indexed per lane (no dynamic indexing of kernel arguments)
    if (threadIdx.x < 16) tw[threadIdx.x] = make_double2(g.t[threadIdx.x], g.w[threadIdx.x]);
    __syncthreads();
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const LaneNodes L{tw[lane & 15].x, tw[lane & 15].y, tw + (lane >> 4)};
    const unsigned long long n = *tot;
    const int nb = (int)min(n & 0xffffffffull, (unsigned long long)cap);
    const int nw = (int)min(n >> 32, (unsigned long long)(cap - nb));
    for (int at = blockIdx.x; at < nb; at += gridDim.x) {
        const int j = map[at], m = pan[j], size = piece_tiles(m), k0 = (at - off[j]) * size;
        double acc[NA] = {};
        quad_tiles<W>(D, x, v, L, j, m, k0 + wave, min(m * m, k0 + size), kQuadWaves, acc);
        if (lane == 0)
#pragma unroll
            for (int k = 0; k < NA; k++) sum[wave][k] = acc[k];
        __syncthreads();
        if (threadIdx.x < NA) {
            double r = 0.0;
            for (int w = 0; w < kQuadWaves; w++) r += sum[w][threadIdx.x];
            part[(size_t)at * NA + threadIdx.x] = r;
        }
        __syncthreads();   // sum is rewritten by the next turn
    }
    // to the blocks in turn, so that few pieces spread over all CUs
    for (int q = wave * gridDim.x + blockIdx.x; q < nw; q += kQuadWaves * gridDim.x) {
        const int at = cap - 1 - q, j = map[at], m = pan[j], k0 = (at - off[j]) * kWaveTiles;
        double acc[NA] = {};
        quad_tiles<W>(D, x, v, L, j, m, k0, min(m * m, k0 + kWaveTiles), 1, acc);
        if (lane == 0)
#pragma unroll
            for (int k = 0; k < NA; k++) part[(size_t)at * NA + k] = acc[k];
    }
}

// One thread per pair: its records added in order. Q_FORCE /
// Q_HVP: the pair's four slots; Q_ENERGY: pe[j] = its energy; Q_JVP:
// pe[j] = grad E_pair . w (pe[j] = 0 for pairs left to the closed form).
// The running totals are cleared for the next call (this kernel follows
// k_quad_nodes on the stream, so every record is written).
template <int W>
__global__ void __launch_bounds__(kBlock) k_quad_finish(Dev D, const double *__restrict__ v,
                                                        const int *__restrict__ off, const int *__restrict__ cnt,
                                                        const double *__restrict__ part, double *__restrict__ slots,
                                                        double *__restrict__ pe,
                                                        unsigned long long *__restrict__ tot) {
    if (tot && blockIdx.x == 0 && threadIdx.x == 0) *tot = 0;
    constexpr int NA = QuadAcc<W>::N;
    bool ok = true;
    for (int j = blockIdx.x * blockDim.x + threadIdx.x; j < D.n_ev; j += gridDim.x * blockDim.x) {
        if (!D.evq[j]) {
            if (W == Q_ENERGY || W == Q_JVP) pe[j] = 0.0;
            continue;
        }
        double acc[NA];
#pragma unroll
        for (int k = 0; k < NA; k++) acc[k] = 0.0;
        for (int q = off[j], qe = off[j] + cnt[j]; q < qe; q++)
#pragma unroll
            for (int k = 0; k < NA; k++) acc[k] += part[(size_t)q * NA + k];
        const double kr = D.ev_kr[j];
        if constexpr (W == Q_ENERGY) {
            pe[j] = kr * acc[0];
        } else {
            // bead weights of r = P(s) - Q(t): c1 (1 - s), c2 s, c3 -(1 - t), c4 -t. For
            // Q_FORCE / Q_JVP the terms were -W grad |r|^-4 (f = forces); for Q_HVP
            // W grad^2 |r|^-4 dr (f = H v)
            const d3 G{acc[0], acc[1], acc[2]}, Gs{acc[3], acc[4], acc[5]}, Gt{acc[6], acc[7], acc[8]};
            d3 f[4];
            f[0] = d3{kr * (G.x - Gs.x), kr * (G.y - Gs.y), kr * (G.z - Gs.z)};
            f[1] = d3{kr * Gs.x, kr * Gs.y, kr * Gs.z};
            f[2] = d3{-kr * (G.x - Gt.x), -kr * (G.y - Gt.y), -kr * (G.z - Gt.z)};
            f[3] = d3{-kr * Gt.x, -kr * Gt.y, -kr * Gt.z};
            ok = ok && finite_d3(f[0]) && finite_d3(f[1]) && finite_d3(f[2]) && finite_d3(f[3]);
            if constexpr (W == Q_JVP) {
                const int4 b = D.ev_bs[j];
                const int o[4] = {b.x, b.y, b.z, b.w};
                double sdot = 0.0;
#pragma unroll
                for (int q = 0; q < 4; q++) sdot -= f[q].x * v[o[q]] + f[q].y * v[o[q] + 1] + f[q].z * v[o[q] + 2];
                pe[j] = sdot;
            } else {
                const int s0 = D.slot_ev + 4 * j;
#pragma unroll
                for (int q = 0; q < 4; q++) put3(slots, s0 + q, f[q]);
            }
        }
    }
    if (!ok) set_err(D.err, MDY_ERR_FORCE);
}

// Block records [rec0 + block] of the per-pair values: pairs j = block * 256
// + thread + k * (grid * 256), each thread's share summed in order, then the
// block's fixed tree; EV entry = that double sum, and for Q_ENERGY the exact
// total in the record's accumulator.
template <int W>
__global__ void __launch_bounds__(kBlock) k_quad_records(Dev D, const double *__restrict__ pe, double *__restrict__ out,
                                                         int rec0) {
    __shared__ double lds[17 * 8 + 8];
    double s[1] = {0.0};
    mdy_xsum X;
    mdy_xs_zero(&X);
    for (int j = blockIdx.x * blockDim.x + threadIdx.x; j < D.n_ev; j += gridDim.x * blockDim.x) {
        if (!D.evq[j]) continue;
        s[0] += pe[j];
        if (W == Q_ENERGY) mdy_xs_add(&X, pe[j]);
    }
    block_reduce<1>(s, lds);
    if (W == Q_ENERGY) block_reduce_xsum(X, reinterpret_cast<long long *>(lds));
    if (threadIdx.x == 0) {
        double *r = out + (size_t)(rec0 + blockIdx.x) * kRed;
        for (int k = 0; k < kNFF; k++) r[k] = k == MDY_FF_EV ? s[0] : 0.0;
        if (W == Q_ENERGY) store_xsum(out, rec0 + blockIdx.x, kXsE, X);
    }
}

// ---------------------------------------------------------------------------
// host side
// ---------------------------------------------------------------------------
bool quad_on(const Ctx &c) {
    return c.opts.coplanar_mode == MDY_COPLANAR_QUADRATURE && !c.ev_mon && c.n_ev > 0;
}

// one pair per thread up to one block per CU: more blocks only give the total
// more records to read (4 per CU: k_energy_tail 10.4 us at
// 66k pairs; so: 7.3)
int quad_blocks(const Ctx &c) {
    const int g = (c.n_ev + kBlock - 1) / kBlock;
    return g < c.num_cu ? (g < 1 ? 1 : g) : c.num_cu;
}

int quad_classify(Ctx &c, Dev &D, const double *d_x, hipStream_t st) {
    const size_t n = (size_t)c.n_ev;
    MDY_TRY(ensure(c.evq, n));
    MDY_TRY(ensure(c.qpan, n));
    MDY_TRY(ensure(c.qcnt, n));
    MDY_TRY(ensure(c.qoff, n));
    MDY_TRY(ensure(c.qmap, kPieces * n));
    // everything the quadrature kernels use is allocated before the totals
    // are taken, so nothing fails between this call and the kernel that clears them
    MDY_TRY(ensure(c.qpart, kPieces * n * 9));
    MDY_TRY(ensure(c.qpe, n));
    if (!c.qtot.p) {
        MDY_TRY(ensure(c.qtot, 1));
        hipLaunchKernelGGL(k_quad_zero, dim3(1), dim3(1), 0, st, c.qtot.p);
    }
    long long g = ((long long)n + kBlock - 1) / kBlock, cap = (long long)c.num_cu * 8;
    const dim3 grid((int)(g > cap ? cap : g < 1 ? 1 : g));
    hipLaunchKernelGGL(k_ev_classify, grid, dim3(kBlock), 0, st, D, d_x, c.evq.p, c.qpan.p, c.qcnt.p, c.qoff.p,
                       c.qmap.p, c.qtot.p, (int)(kPieces * n));
    D.evq = c.evq.p;
    return hipGetLastError() == hipSuccess ? MDY_OK : MDY_ERR_HIP;
}

template <int W>
static void quad_launch(Ctx &c, const Dev &D, const double *d_x, const double *d_v, double *out, int rec0,
                        hipStream_t st, bool keep) {
    const long long n = c.n_ev;
    const dim3 blk(kBlock);
    long long g = (n + kBlock - 1) / kBlock, cap = (long long)c.num_cu * 8;
    const dim3 pairs((int)(g > cap ? cap : g < 1 ? 1 : g));
    const int rcap = (int)(kPieces * n);
    // one block per CU, fewer where the table cannot hold as many flagged pairs
    const int nodes = (int)std::min<long long>(c.num_cu, std::max<long long>(n / 8, 16));
    hipLaunchKernelGGL(k_quad_nodes<W>, dim3(nodes), dim3(kQuadBlock), 0, st, D, d_x, d_v, gl16(), c.qoff.p, c.qmap.p,
                       c.qpan.p, c.qtot.p, rcap, c.qpart.p);
    hipLaunchKernelGGL(k_quad_finish<W>, pairs, blk, 0, st, D, d_v, c.qoff.p, c.qcnt.p, c.qpart.p, out, c.qpe.p,
                       keep ? nullptr : c.qtot.p);
    if (W == Q_ENERGY || W == Q_JVP)
        hipLaunchKernelGGL(k_quad_records<W>, dim3(quad_blocks(c)), blk, 0, st, D, c.qpe.p, out, rec0);
}

int launch_quad(Ctx &c, const Dev &D, int what, const double *d_x, const double *d_v, double *out, int rec0,
                hipStream_t st, bool keep) {
    switch (what) {
        case 0: quad_launch<Q_ENERGY>(c, D, d_x, d_v, out, rec0, st, keep); break;
        case 1: quad_launch<Q_FORCE>(c, D, d_x, d_v, out, rec0, st, keep); break;
        case 2: quad_launch<Q_HVP>(c, D, d_x, d_v, out, rec0, st, keep); break;
        default: quad_launch<Q_JVP>(c, D, d_x, d_v, out, rec0, st, keep); break;
    }
    return hipGetLastError() == hipSuccess ? MDY_OK : MDY_ERR_HIP;
}

int quad_end(Ctx &c, hipStream_t st) {
    hipLaunchKernelGGL(k_quad_zero, dim3(1), dim3(1), 0, st, c.qtot.p);
    return hipGetLastError() == hipSuccess ? MDY_OK : MDY_ERR_HIP;
}

int quad_pair_count(Ctx &c, const double *d_x, hipStream_t st, int *count) {
    *count = 0;
    if (!quad_on(c)) return MDY_OK;
    Dev D = c.dev();
    MDY_TRY(quad_classify(c, D, d_x, st));
    MDY_TRY(quad_end(c, st));   // no quadrature follows
    std::vector<unsigned char> h((size_t)c.n_ev);
    MDY_HIP(hipMemcpyAsync(h.data(), c.evq.p, h.size(), hipMemcpyDeviceToHost, st));
    MDY_HIP(hipStreamSynchronize(st));
    int n = 0;
    for (unsigned char f : h) n += f;
    *count = n;
    return MDY_OK;
}

}  // namespace mdy
