// mdy_nl.hip -- binned cylinder neighbor-list rebuild and the vectorization of
// the excluded-volume and boundary force fields, all on the device.
//
// Pair predicate: HybridCylinderCylinderNL::updateNeighborsbin
// (src/Structure/HybridNeighborListImpl.cpp:405-441): keep (c, n) iff
// id(c) > id(n), not (same filament and |pos(c) - pos(n)| <= 2), and the
// squared midpoint distance (double) lies in [(float)rMin^2, (float)rMax^2].
// The reference's bins (edge 1.125 rMax) only prune candidates; the cells used
// here have edge >= the float cutoff, so the pair SET is the same. Rows are
// sorted by neighbour index, making the list deterministic.
// CylinderExclVolume::vectorize (CylinderExclVolume.cpp:34-179) then drops
// pairs whose neighbour is the cylinder's mother (getBranchingCylinder()).
#include <hipcub/hipcub.hpp>

#include <cmath>

#include "mdy_device.hpp"
#include "mdy_eval.hpp"
#include "mdy_launch.hpp"

namespace mdy {

// start of the n entries that this thread takes from *total, one atomic per
// block of 1024 threads (same-address atomics are served every 11 ns: one per
// wave took 95 us at 200k cylinders). Every thread of the block calls it.
constexpr int kRoomBlock = 1024;
__device__ __forceinline__ int block_room(int n, int *total) {
    __shared__ int part[kRoomBlock / 64], base;
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    int incl = n;
#pragma unroll
    for (int o = 1; o < 64; o <<= 1) {
        const int u = __shfl_up(incl, o, 64);
        if (lane >= o) incl += u;
    }
    if (lane == 63) part[wave] = incl;
    __syncthreads();
    if (threadIdx.x == 0) {
        int s = 0;
        for (int w = 0; w < kRoomBlock / 64; w++) { const int v = part[w]; part[w] = s; s += v; }
        base = s ? atomicAdd(total, s) : 0;
    }
    __syncthreads();
    return base + part[wave] + incl - n;
}

// Cells of edge h in a hash table of nb = 2^k buckets, at least two per
// cylinder: no bounding box, so the host does not wait for one, and the table
// does not grow with the box. A bucket's cylinders are contiguous in `list`
// with their cells; a reader skips those of other cells in the same bucket.
// Cells that follow one another in x have neighbouring buckets: the 27 around a
// cylinder lie in nine lines instead of 27.
struct Cells {
    double h;
    unsigned mask;
    __device__ __forceinline__ int3 cell(const double *m) const {
        return make_int3((int)floor(m[0] / h), (int)floor(m[1] / h), (int)floor(m[2] / h));   // saturates
    }
    __device__ __forceinline__ unsigned bucket(int3 c) const {
        const unsigned u = ((unsigned)c.y * 0x9E3779B1u) ^ ((unsigned)c.z * 0x85EBCA6Bu);
        return ((u ^ (u >> 15)) * 0xC2B2AE35u + (unsigned)c.x) & mask;
    }
};

__global__ void k_nl_zero(int *a, int na, int *b, int nb) {
    for (int i = blockIdx.x * blockDim.x + threadIdx.x; i < na + nb; i += gridDim.x * blockDim.x)
        if (i < na) a[i] = 0;
        else b[i - na] = 0;
}

// flags[0]: an infinite midpoint; flags[1..3]: a number on that axis (plain
// stores of 1: nothing to order, no atomics on one word)
__global__ void __launch_bounds__(kBlock) k_nl_cells(int ncyl, const int *__restrict__ b1, const int *__restrict__ b2,
                                                     const double *__restrict__ x, Cells g, double *__restrict__ mid,
                                                     int *__restrict__ rank, int *cnt, int *flags) {
    int f = 0;
    for (int c = blockIdx.x * blockDim.x + threadIdx.x; c < ncyl; c += gridDim.x * blockDim.x) {
        const double *p1 = x + b1[c], *p2 = x + b2[c];
        double m[3];
        for (int k = 0; k < 3; k++) {
            m[k] = 0.5 * (p1[k] + p2[k]);   // Cylinder::updateCoordinate (Cylinder.cpp:45-49)
            mid[3 * c + k] = m[k];
            if (m[k] == m[k]) f |= 2 << k;
            if (fabs(m[k]) == INFINITY) f |= 1;
        }
        rank[c] = atomicAdd(cnt + g.bucket(g.cell(m)), 1);
    }
    f = wave_or(f);
    if ((threadIdx.x & 63) < 4 && ((f >> (threadIdx.x & 63)) & 1)) flags[threadIdx.x & 63] = 1;
}

// a bucket's range, start and end (the buckets' order in the list does not matter)
__global__ void __launch_bounds__(kRoomBlock) k_nl_ranges(const int *__restrict__ cnt, int2 *__restrict__ range,
                                                          int *total) {
    const int i = blockIdx.x * kRoomBlock + threadIdx.x;   // the bucket count is a multiple of the block
    const int n = cnt[i], at = block_room(n, total);
    range[i] = make_int2(at, at + n);
}

struct CylView {
    const int *b1, *b2, *fil, *pos, *child;
    const long long *id;
    const short *type;
    const double *eq, *ek;
    const double *seg;   // monomer-sum form: interval * monomer size
    int mon;             // monomer-sum excluded volume
};

// What the search reads of a cylinder, 64 bytes each, in the order of
// the buckets: candidates of a bucket are read in full lines.
struct CellEntry {
    double m[3];
    int c, fil;
    long long id;
    int pos, child;
    int3 cell;
    int pad;
};
static_assert(sizeof(CellEntry) == 64, "");
__device__ __forceinline__ CellEntry cell_entry(const CylView &C, const Cells &g, const double *__restrict__ mid, int c) {
    CellEntry e;
    for (int k = 0; k < 3; k++) e.m[k] = mid[3 * c + k];
    e.c = c; e.fil = C.fil[c]; e.id = C.id[c]; e.pos = C.pos[c]; e.child = C.child[c];
    e.cell = g.cell(e.m);
    e.pad = 0;
    return e;
}

__global__ void k_nl_fill(int ncyl, CylView C, Cells g, const double *__restrict__ mid, const int *__restrict__ rank,
                          const int2 *__restrict__ range, CellEntry *__restrict__ list) {
    for (int c = blockIdx.x * blockDim.x + threadIdx.x; c < ncyl; c += gridDim.x * blockDim.x) {
        const CellEntry e = cell_entry(C, g, mid, c);
        list[range[g.bucket(e.cell)].x + rank[c]] = e;
    }
}

// Pairs the excluded-volume force field drops: the integral form skips a
// neighbour that is the cylinder's branching mother
// (cin->getBranchingCylinder() == ci, CylinderExclVolume.cpp:85, 116); the
// monomer-sum form skips mother-daughter pairs in either order
// (CylinderVolumeMon.hpp:134-136).
__device__ __forceinline__ bool ev_dropped(const CylView &C, const CellEntry &c, const CellEntry &n) {
    return n.child == c.c || (C.mon && c.child == n.c);
}

// The candidates of cylinder c that pass the reference predicate, found by the
// kGroup lanes of a group, each looking into its share of the 27 cells around
// c. fn(n) is called by the lane that finds n. One lane per cylinder followed
// 27 cells' dependent loads in a row (113 us at 40k cylinders for the count).
constexpr int kGroup = 16;
template <class F>
__device__ __forceinline__ void for_neighbors(const Cells &g, const int2 *__restrict__ range,
                                              const CellEntry *__restrict__ list, const CellEntry &me, double rminsq,
                                              double rmaxsq, F &&fn) {
    constexpr int kCells = (27 + kGroup - 1) / kGroup;   // cells per lane
    int3 cell[kCells];
    int2 r[kCells];
#pragma unroll
    for (int j = 0; j < kCells; j++) {   // every range is on its way before the first is used
        const int k = (int)(threadIdx.x & (kGroup - 1)) + j * kGroup;
        cell[j] = make_int3(me.cell.x + k % 3 - 1, me.cell.y + (k / 3) % 3 - 1, me.cell.z + k / 9 - 1);
        r[j] = k < 27 ? range[g.bucket(cell[j])] : make_int2(0, 0);
    }
#pragma unroll
    for (int j = 0; j < kCells; j++) {
        for (int a = r[j].x; a < r[j].y; a++) {
            const CellEntry &n = list[a];
            double d2 = (n.m[0] - me.m[0]) * (n.m[0] - me.m[0]);
            d2 += (n.m[1] - me.m[1]) * (n.m[1] - me.m[1]);
            d2 += (n.m[2] - me.m[2]) * (n.m[2] - me.m[2]);
            if (d2 < rminsq || d2 > rmaxsq) continue;
            if (n.cell.x != cell[j].x || n.cell.y != cell[j].y || n.cell.z != cell[j].z) continue;
            if (me.id <= n.id) continue;
            if (me.fil == n.fil) {
                const int ds = me.pos - n.pos;
                if ((ds < 0 ? -ds : ds) <= 2) continue;   // ChemParams::minCylinderDistanceSameFilament (SysParams.h:315)
            }
            fn(n);
        }
    }
}

// Row counts, pairs in the upper and kept pairs in the lower half (row[ncyl] =
// 0), and the first kNear neighbours found (2 n, + 1 if dropped) in any order.
// Cylinders are taken in the order of the cells' list, so that the groups of a
// block share their cells' lines: 77 us at 200k cylinders (105 in cylinder
// order with every field from its own array), bound by the reads of the buckets.
constexpr int kNear = kGroup;
__global__ void __launch_bounds__(kBlock) k_pair_count(int ncyl, CylView C, Cells g, const int2 *range,
                                                       const CellEntry *list, double rminsq, double rmaxsq,
                                                       unsigned long long *row, int *near) {
    __shared__ int found[kBlock / kGroup];
    const int i = blockIdx.x * (kBlock / kGroup) + threadIdx.x / kGroup, lane = threadIdx.x & (kGroup - 1);
    const int grp = threadIdx.x / kGroup;
    if (lane == 0) found[grp] = 0;
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "workgroup");   // the group's lanes are one wave's
    __builtin_amdgcn_wave_barrier();
    if (i < ncyl) {
        const CellEntry me = list[i];
        const int c = me.c;
        int keep = 0;
        for_neighbors(g, range, list, me, rminsq, rmaxsq, [&](const CellEntry &n) {
            const int drop = ev_dropped(C, me, n) ? 1 : 0, at = atomicAdd(found + grp, 1);
            if (at < kNear) near[(size_t)kNear * c + at] = 2 * n.c + drop;
            keep += 1 - drop;
        });
#pragma unroll
        for (int o = 1; o < kGroup; o <<= 1) keep += __shfl_xor(keep, o, kGroup);
        __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "workgroup");
        __builtin_amdgcn_wave_barrier();
        if (lane == 0) row[c] = ((unsigned long long)(unsigned)found[grp] << 32) | (unsigned)keep;
    } else if (i == ncyl && lane == 0) {
        row[i] = 0;
    }
}

// The rows: each entry placed by counting the smaller ones of its row. Rows of
// up to kNear come from the count; the longer ones are searched again, into
// tmp. beads: slots per bead so far. 23 us at 200k cylinders; 93
// with every row searched again.
__global__ void __launch_bounds__(kBlock) k_pair_emit(int ncyl, CylView C, Cells g, const double *mid, const int2 *range,
                                                      const CellEntry *list, double rminsq, double rmaxsq,
                                                      const unsigned long long *row_off, const int *near,
                                                      int *tmp, int2 *pairs, int4 *ev_bs, double *ev_kr, int2 *ev_cyl,
                                                      int *beads) {
    __shared__ int found[kBlock / kGroup];
    const int q = threadIdx.x & (kGroup - 1), grp = threadIdx.x / kGroup;
    const int c = blockIdx.x * (kBlock / kGroup) + grp;
    if (c < ncyl) {
        const unsigned long long r0 = row_off[c], r1 = row_off[c + 1];
        const int o = (int)(r0 >> 32), len = (int)(r1 >> 32) - o, ok = (int)(unsigned)r0;
        const int *keys = near + (size_t)kNear * c;
        if (len > kNear) {
            if (q == 0) found[grp] = 0;
            __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "workgroup");   // the group's lanes are one wave's
            __builtin_amdgcn_wave_barrier();
            const CellEntry me = cell_entry(C, g, mid, c);
            for_neighbors(g, range, list, me, rminsq, rmaxsq, [&](const CellEntry &n) {
                tmp[o + atomicAdd(found + grp, 1)] = 2 * n.c + (ev_dropped(C, me, n) ? 1 : 0);
            });
            __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "workgroup");
            __builtin_amdgcn_wave_barrier();
            keys = tmp + o;
        }
        for (int e = q; e < len; e += kGroup) {
            const int key = keys[e];
            int rank = 0, krank = 0;
            for (int m = 0; m < len; m++) {
                const int k = keys[m];
                if (k < key) { rank++; krank += 1 - (k & 1); }
            }
            const int n = key >> 1;
            pairs[o + rank] = make_int2(c, n);
            if (key & 1) continue;
            const int4 bs = make_int4(C.b1[c], C.b2[c], C.b1[n], C.b2[n]);
            const int at = ok + krank;
            ev_bs[at] = bs;
            if (C.mon) {
                // kvol = max of the two constants; coeff = kvol * segEqLen1 * segEqLen2
                // (CylinderVolumeMon.hpp:43, 160-163)
                ev_kr[at] = smax(C.ek[c], C.ek[n]) * C.seg[c] * C.seg[n];
                ev_cyl[at] = make_int2(c, n);
            } else {
                const double krep = (C.type[c] != C.type[n]) ? smax(C.ek[c], C.ek[n]) : C.ek[c];
                ev_kr[at] = krep * C.eq[c] * C.eq[n];
            }
            atomicAdd(beads + bs.x / 3, 1); atomicAdd(beads + bs.y / 3, 1);
            atomicAdd(beads + bs.z / 3, 1); atomicAdd(beads + bs.w / 3, 1);
        }
    }
}

// BoundaryCylinderNL (NeighborListImpl.cpp:738-751): plane distance of
// Cylinder::coordinate = midPointCoordinate(b1, b2, 0.5) below the float cutoff.
// One block per plane and kBlock cylinders; cnt: its terms (two for a minus end).
__global__ void __launch_bounds__(kBlock) k_bd_flag(int ncyl, int nchunk, const int *__restrict__ b1,
                                                    const int *__restrict__ b2, const unsigned char *__restrict__ minus,
                                                    const double *__restrict__ x, const double *__restrict__ planes,
                                                    float cutoff, int *__restrict__ flag, int *__restrict__ cnt) {
    __shared__ int part[kBlock / 64];
    const int p = blockIdx.x / nchunk, c = (blockIdx.x % nchunk) * kBlock + threadIdx.x;
    int f = 0;
    if (c < ncyl) {
        const double *p1 = x + b1[c], *p2 = x + b2[c];
        d3 m = d3{p1[0] * (1.0 - 0.5) + 0.5 * p2[0], p1[1] * (1.0 - 0.5) + 0.5 * p2[1],
                  p1[2] * (1.0 - 0.5) + 0.5 * p2[2]};
        const double dist = plane_dist(planes + 4 * p, m);
        f = (dist < (double)cutoff) ? (minus[c] ? 2 : 1) : 0;
        flag[(size_t)p * ncyl + c] = f;
    }
    const int n = __popcll(__ballot(f > 0)) + __popcll(__ballot(f > 1));
    if ((threadIdx.x & 63) == 0) part[threadIdx.x >> 6] = n;
    __syncthreads();
    if (threadIdx.x == 0) {
        int t = 0;
        for (int w = 0; w < kBlock / 64; w++) t += part[w];
        cnt[blockIdx.x] = t;
    }
}

// One block: the chunks' offsets, in place, and what the host needs to size the
// tables: out = pair totals (packed as in row), midpoints fit for cells, then the offset
// of each plane's first term and their total.
__global__ void __launch_bounds__(1024) k_nl_totals(int nplanes, int nchunk, int *cnt, const unsigned long long *pairs,
                                                    const int *flags, long long *out) {
    __shared__ int part[16];
    const int n = nplanes * nchunk, lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    int run = 0;
    if (threadIdx.x == 0) {
        out[0] = pairs ? (long long)*pairs : 0;
        out[1] = flags ? (!flags[0] && flags[1] && flags[2] && flags[3] ? 1 : 0) : 1;
    }
    for (int i0 = 0; i0 < n; i0 += 1024) {
        const int i = i0 + threadIdx.x;
        const int v = i < n ? cnt[i] : 0;
        int incl = v;
#pragma unroll
        for (int o = 1; o < 64; o <<= 1) {
            const int u = __shfl_up(incl, o, 64);
            if (lane >= o) incl += u;
        }
        if (lane == 63) part[wave] = incl;
        __syncthreads();
        int before = 0, all = 0;
        for (int w = 0; w < 16; w++) { before += w < wave ? part[w] : 0; all += part[w]; }
        const int at = run + before + incl - v;
        if (i < n) {
            cnt[i] = at;
            if (i % nchunk == 0) out[2 + i / nchunk] = at;
        }
        run += all;
        __syncthreads();
    }
    if (threadIdx.x == 0) out[2 + nplanes] = run;
}

// BoundaryCylinderRepulsion::vectorize (BoundaryCylinderRepulsion.cpp:33-88)
__global__ void __launch_bounds__(kBlock) k_bd_emit(int ncyl, int nchunk, const int *__restrict__ b1,
                                                    const int *__restrict__ b2, const int *__restrict__ flag,
                                                    const int *__restrict__ off, const double *__restrict__ pk,
                                                    const double *__restrict__ psl, int *bd_bead, int *bd_plane,
                                                    double *bd_k, double *bd_sl, int *beads) {
    __shared__ int part[kBlock / 64];
    const int p = blockIdx.x / nchunk, c = (blockIdx.x % nchunk) * kBlock + threadIdx.x;
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int f = c < ncyl ? flag[(size_t)p * ncyl + c] : 0;
    const unsigned long long one = __ballot(f > 0), two = __ballot(f > 1), below = (1ull << lane) - 1;
    if (lane == 0) part[wave] = __popcll(one) + __popcll(two);
    __syncthreads();
    if (!f) return;
    int o = off[blockIdx.x] + __popcll(one & below) + __popcll(two & below);
    for (int w = 0; w < wave; w++) o += part[w];
    auto put = [&](int bead) {
        bd_bead[o] = bead; bd_plane[o] = p; bd_k[o] = pk[p]; bd_sl[o] = psl[p];
        atomicAdd(beads + bead / 3, 1);
        o++;
    };
    if (f == 2) put(b1[c]);
    put(b2[c]);
}

// The gather's rows (Dev::row_idx): a bead's bonded slots, then its
// excluded-volume and boundary slots in slot order.
__device__ __forceinline__ int dyn_slot_bead(const Dev &D, int j, int &slot) {
    const int nev4 = 4 * D.n_ev;
    if (j < nev4) {
        slot = D.slot_ev + j;
        return reinterpret_cast<const int *>(D.ev_bs)[j] / 3;
    }
    j -= nev4;
    slot = D.slot_bd + j;
    return D.bd_bead[j] / 3;
}
// room for the rows, in groups of four (their order does not matter); the
// counters restart for the fill
__global__ void __launch_bounds__(kRoomBlock) k_row_ranges(int nb, const int *__restrict__ st_off, int *__restrict__ cur,
                                                       int2 *__restrict__ row, int *total) {
    const int b = blockIdx.x * kRoomBlock + threadIdx.x;
    const int n = b < nb ? (st_off[b + 1] - st_off[b] + cur[b] + 3) / 4 : 0;
    const int base = block_room(n, total);
    if (b < nb) {
        row[b] = make_int2(base, base + n);
        cur[b] = 0;
    }
}
// dynamic slots in any order, after the room of the bonded ones
__global__ void k_row_fill(Dev D, const int *__restrict__ st_off, int *cur, int *tmp) {
    const int tot = 4 * D.n_ev + D.n_bd;
    for (int j = blockIdx.x * blockDim.x + threadIdx.x; j < tot; j += gridDim.x * blockDim.x) {
        int s;
        const int b = dyn_slot_bead(D, j, s);
        tmp[4 * D.row[b].x + (st_off[b + 1] - st_off[b]) + atomicAdd(cur + b, 1)] = s;
    }
}
// Eight lanes per bead: the bonded slots copied, each dynamic slot placed by
// counting the smaller ones of its row (rows hold ~10, all in cache), the last
// group filled up.
__global__ void k_row_place(Dev D, const int *__restrict__ st_off, const int *__restrict__ st_idx,
                            const int *__restrict__ cur, const int *__restrict__ tmp, int *__restrict__ out) {
    const int q = threadIdx.x & 7;
    for (int b = (blockIdx.x * blockDim.x + threadIdx.x) >> 3; b < D.nb; b += (gridDim.x * blockDim.x) >> 3) {
        const int s0 = st_off[b], ns = st_off[b + 1] - s0, nd = cur[b];
        const int r0 = 4 * D.row[b].x, r1 = 4 * D.row[b].y;
        for (int k = q; k < ns; k += 8) out[r0 + k] = 3 * st_idx[s0 + k];
        const int *row = tmp + r0 + ns;
        for (int k = q; k < nd; k += 8) {
            const int v = row[k];
            int rank = 0;
            for (int m = 0; m < nd; m++) rank += row[m] < v ? 1 : 0;
            out[r0 + ns + rank] = 3 * v;
        }
        for (int k = r0 + ns + nd + q; k < r1; k += 8) out[k] = 3 * D.n_slots;
    }
}

// ---------------------------------------------------------------------------
static int grid1(const Ctx &c, long long n) {
    long long g = (n + kBlock - 1) / kBlock;
    long long cap = (long long)c.num_cu * 8;
    return (int)(g < 1 ? 1 : (g > cap ? cap : g));
}

int build_neighbors(Ctx &c, const double *d_x) {
    hipStream_t st = c.stream;
    const int ncyl = c.ncyl, nb = c.nb;
    c.n_ev = 0;
    c.n_bd = 0;
    c.n_pairs = 0;
    CylView C{c.c_b1.p, c.c_b2.p, c.c_fil.p, c.c_pos.p, c.c_child.p, c.c_id.p, c.c_type.p, c.c_eq.p, c.c_ek.p,
              c.c_seg.p, c.ev_mon};
    const bool ev = c.ev_on && ncyl > 1, bd = c.bd_on && c.n_planes > 0 && ncyl > 0;
    // counters that start at zero: bucket counts, then list total, row total, four midpoint flags
    int nbuckets = 1024;
    while (nbuckets < 2LL * ncyl && nbuckets < (1 << 29)) nbuckets *= 2;
    const int nzero = (ev ? nbuckets : 0) + 6;
    MDY_TRY(ensure(c.cell_cnt, (size_t)nzero));
    MDY_TRY(ensure(c.row_cur, (size_t)nb + 1));
    int *misc = c.cell_cnt.p + (nzero - 6);
    hipLaunchKernelGGL(k_nl_zero, dim3(grid1(c, (long long)nzero + nb)), dim3(kBlock), 0, st, c.cell_cnt.p, nzero,
                       c.row_cur.p, nb);
    const float rmaxsq_f = c.ev_cut * c.ev_cut;   // float, HybridNeighborListImpl.h:78-80
    const float rminsq_f = 0.0f * 0.0f;
    const double rmin2 = (double)rminsq_f, rmax2 = (double)rmaxsq_f;
    const Cells g{std::sqrt(rmax2) * (1.0 + 1e-6) + 1e-6, (unsigned)nbuckets - 1};
    // a group per cylinder without a cap: each is one chain of dependent loads
    const dim3 groups((unsigned)(((long long)kGroup * (ncyl + 1) + kBlock - 1) / kBlock)), blk(kBlock);
    if (ev) {
        MDY_TRY(ensure(c.mid, (size_t)3 * ncyl));
        MDY_TRY(ensure(c.cell_rank, ncyl));
        MDY_TRY(ensure(c.cell_range, nbuckets));
        MDY_TRY(ensure(c.cell_list, sizeof(CellEntry) / sizeof(int4) * (size_t)ncyl));
        CellEntry *list = reinterpret_cast<CellEntry *>(c.cell_list.p);
        MDY_TRY(ensure(c.near, (size_t)kNear * ncyl));
        MDY_TRY(ensure(c.row_cnt, (size_t)ncyl + 1));
        MDY_TRY(ensure(c.row_off, (size_t)ncyl + 1));
        const dim3 cyl(grid1(c, ncyl));
        hipLaunchKernelGGL(k_nl_cells, cyl, blk, 0, st, ncyl, c.c_b1.p, c.c_b2.p, d_x, g, c.mid.p, c.cell_rank.p,
                           c.cell_cnt.p, misc + 2);
        hipLaunchKernelGGL(k_nl_ranges, dim3(nbuckets / kRoomBlock), dim3(kRoomBlock), 0, st, c.cell_cnt.p,
                           c.cell_range.p, misc);
        hipLaunchKernelGGL(k_nl_fill, cyl, blk, 0, st, ncyl, C, g, c.mid.p, c.cell_rank.p, c.cell_range.p, list);
        hipLaunchKernelGGL(k_pair_count, groups, blk, 0, st, ncyl, C, g, c.cell_range.p, list, rmin2,
                           rmax2, c.row_cnt.p, c.near.p);
        size_t tmp = 0;
        MDY_HIP(hipcub::DeviceScan::ExclusiveSum(nullptr, tmp, c.row_cnt.p, c.row_off.p, ncyl + 1, st));
        MDY_TRY(ensure(c.scan_tmp, tmp / sizeof(int) + 1));
        size_t cap = c.scan_tmp.n * sizeof(int);
        MDY_HIP(hipcub::DeviceScan::ExclusiveSum(c.scan_tmp.p, cap, c.row_cnt.p, c.row_off.p, ncyl + 1, st));
    }
    const int nchunk = (ncyl + kBlock - 1) / kBlock, np = bd ? c.n_planes : 0;
    if (bd) {
        MDY_TRY(ensure(c.bd_flag, (size_t)np * ncyl));
        MDY_TRY(ensure(c.bd_off, (size_t)np * nchunk));
        hipLaunchKernelGGL(k_bd_flag, dim3(np * nchunk), blk, 0, st, ncyl, nchunk, c.c_b1.p, c.c_b2.p, c.c_minus.p, d_x,
                           c.planes.p, c.bd_cut, c.bd_flag.p, c.bd_off.p);
    }
    MDY_TRY(ensure_host_out(c, kOutNl + (size_t)c.n_planes + 3));
    const long long *tot = c.h_out + kOutNl;
    hipLaunchKernelGGL(k_nl_totals, dim3(1), dim3(1024), 0, st, np, nchunk, c.bd_off.p,
                       ev ? c.row_off.p + ncyl : nullptr, ev ? misc + 2 : nullptr, c.h_out + kOutNl);
    MDY_HIP(hipGetLastError());
    MDY_HIP(hipStreamSynchronize(st));
    if (!tot[1]) return MDY_ERR_NONFINITE;   // an infinite midpoint, or an axis without a number
    c.n_pairs = (unsigned long long)tot[0] >> 32;
    c.n_ev = (int)(unsigned)tot[0];
    c.n_bd = (int)tot[2 + np];
    c.h_bd_nneigh.assign(c.n_planes, 0);
    for (int p = 0; p < np; p++) c.h_bd_nneigh[p] = (int)(tot[3 + p] - tot[2 + p]);
    MDY_TRY(ensure(c.ev_bs, (size_t)c.n_ev + 1));
    MDY_TRY(ensure(c.ev_kr, (size_t)c.n_ev + 1));
    if (c.ev_mon) MDY_TRY(ensure(c.ev_cyl, (size_t)c.n_ev + 1));
    MDY_TRY(ensure(c.bd_bead, (size_t)c.n_bd + 1));
    MDY_TRY(ensure(c.bd_plane, (size_t)c.n_bd + 1));
    MDY_TRY(ensure(c.bd_k, (size_t)c.n_bd + 1));
    MDY_TRY(ensure(c.bd_sl, (size_t)c.n_bd + 1));
    const int ndyn = 4 * c.n_ev + c.n_bd;
    // every row's last group may be filled up with three entries
    const size_t rows = ((size_t)c.n_static + ndyn) / 4 + nb + 1;
    MDY_TRY(ensure(c.row, (size_t)nb + 1));
    MDY_TRY(ensure(c.row_idx, rows));
    MDY_TRY(ensure(c.row_tmp, rows));
    if (c.n_pairs > 0) {
        MDY_TRY(ensure(c.pairs, 2 * (size_t)c.n_pairs));
        MDY_TRY(ensure(c.pair_tmp, (size_t)c.n_pairs));
        hipLaunchKernelGGL(k_pair_emit, groups, blk, 0, st, ncyl, C, g, c.mid.p, c.cell_range.p,
                           reinterpret_cast<const CellEntry *>(c.cell_list.p), rmin2, rmax2, c.row_off.p, c.near.p, c.pair_tmp.p, (int2 *)c.pairs.p,
                           c.ev_bs.p, c.ev_kr.p, c.ev_mon ? c.ev_cyl.p : nullptr, c.row_cur.p);
    }
    if (c.n_bd > 0)
        hipLaunchKernelGGL(k_bd_emit, dim3(np * nchunk), blk, 0, st, ncyl, nchunk, c.c_b1.p, c.c_b2.p, c.bd_flag.p,
                           c.bd_off.p, c.plane_k.p, c.plane_sl.p, c.bd_bead.p, c.bd_plane.p, c.bd_k.p, c.bd_sl.p,
                           c.row_cur.p);
    c.have_nl = true;
    const Dev D = c.dev();
    hipLaunchKernelGGL(k_row_ranges, dim3((nb + kRoomBlock - 1) / kRoomBlock), dim3(kRoomBlock), 0, st, nb, c.st_off.p,
                       c.row_cur.p, c.row.p, misc + 1);
    if (ndyn > 0)
        hipLaunchKernelGGL(k_row_fill, dim3(grid1(c, ndyn)), blk, 0, st, D, c.st_off.p, c.row_cur.p,
                           reinterpret_cast<int *>(c.row_tmp.p));
    hipLaunchKernelGGL(k_row_place, dim3(grid1(c, 8LL * nb)), blk, 0, st, D, c.st_off.p, c.st_idx.p, c.row_cur.p,
                       reinterpret_cast<const int *>(c.row_tmp.p), reinterpret_cast<int *>(c.row_idx.p));
    MDY_HIP(hipGetLastError());
    // evaluation scratch sized for the new slot count
    MDY_TRY(ensure(c.contrib, (size_t)3 * D.n_slots + 3));
    return MDY_OK;
}

}  // namespace mdy
