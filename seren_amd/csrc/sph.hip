// sph.hip -- grad-h smoothing-length / density solve, neighbour lists,
// isothermal thermal update and grad-h hydro pair forces on gfx950.
//
// Each wave owns 64 consecutive particles in tree order (a compact leaf
// group) and walks the hydro tree once per pass for all of them with
// group_walk; every lane keeps its own state machine of all_sph_gradh.
// Sums run over the walk's leaves in DFS order, which is the order of the
// reference's potential-neighbour list, and use the reference's operation
// order (built without FMA contraction), so h, rho, Omega, zeta and the
// neighbour lists come out identical to the reference.
#include <algorithm>
#include <cstring>
#include <rocprim/rocprim.hpp>

#include "walk.h"

namespace serenx {

namespace {

constexpr int TB = 256;
inline int nblk(long n, int tb = TB) { return (int)((n + tb - 1) / tb); }

// Compact 32-byte records for the per-lane candidate loops of the h solve,
// in the record buffer (which the hydro pass later rewrites): rec[i] =
// (x, y, z, m) and rec[n + i] = (vx, vy, vz, 0).  Four particles share a
// cache line, so a leaf's candidates are two lines, and the loops' working
// set stays in L2.
__global__ void k_pack_hsolve(int n, const double *__restrict__ x, const double *__restrict__ y,
                              const double *__restrict__ z, const double *__restrict__ vx,
                              const double *__restrict__ vy, const double *__restrict__ vz,
                              const double *__restrict__ m, double4 *__restrict__ rec) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    rec[i] = make_double4(x[i], y[i], z[i], m[i]);
    rec[(size_t)n + i] = make_double4(vx[i], vy[i], vz[i], 0.0);
}

// [x y z h] records of the particles, and hrangemax of the nodes in BFS order
// (update_hmax leaves it in DFS order; bn null: not wanted)
__global__ void k_pack_xyzh(int n, const double *__restrict__ x, const double *__restrict__ y,
                            const double *__restrict__ z, const double *__restrict__ h,
                            double4 *__restrict__ rec, int nc, const int *__restrict__ bfs2dfs,
                            const HNode *__restrict__ hn, BNode *__restrict__ bn) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) rec[i] = make_double4(x[i], y[i], z[i], h[i]);
    if (bn && i < nc) bn[i].hrangemax = hn[bfs2dfs[i]].hrangemax;
}

// Squared distance from the point at offset (dx, dy, dz) from a node's box
// centre to the node's (grown) bounding box: a lower bound of the distance to
// any particle of the subtree.
__device__ __forceinline__ double box_dist2(const HNode &nd, double dx, double dy, double dz) {
    const double ex = fmax(fabs(dx) - (double)nd.half[0], 0.0);
    const double ey = fmax(fabs(dy) - (double)nd.half[1], 0.0);
    const double ez = fmax(fabs(dz) - (double)nd.half[2], 0.0);
    return ex * ex + ey * ey + ez * ez;
}

// HNode visit of BHhydrowalk_hgather.F90:40 for a search radius R (the
// reference's bounding-sphere test, so the leaves it yields are the
// reference's potential list, whose size the h solve reads)
__device__ __forceinline__ int hgather_visit(const HNode &nd, double rpx, double rpy, double rpz,
                                             double R) {
    const double dx = nd.r[0] - rpx, dy = nd.r[1] - rpy, dz = nd.r[2] - rpz;
    const double drsqd = dx * dx + dy * dy + dz * dz;
    const double lim = (R + nd.rmax) * (R + nd.rmax);
    if (!(drsqd <= lim)) return WALK_SKIP;
    return nd.leaf == 0 ? WALK_DESCEND : WALK_LEAF;
}

// Whether a leaf of that list can hold a particle within R: with fresh boxes
// (box) a leaf whose box lies farther than R holds none, and its particles
// are left out of the candidate lists (they cannot contribute, so the
// candidates that remain come in the reference's order)
__device__ __forceinline__ bool leaf_near(const HNode &nd, double rpx, double rpy, double rpz,
                                          double R, bool box) {
    if (!box) return true;
    return box_dist2(nd, nd.r[0] - rpx, nd.r[1] - rpy, nd.r[2] - rpz) <= R * R * (1.0 + 1.0e-12);
}

// Loops every summing lane over its own potential-neighbour list, leaf by
// leaf in DFS order, calling use(j, load(j)) for each listed particle j != p.
// Each lane walks its own stream of candidates and issues the load of the
// next candidate (and the next list slot) before using the current one, so
// the record's memory latency overlaps the current candidate's table lookup
// and arithmetic.  The order of the candidates is the list order.
template <class Load, class Use>
__device__ __forceinline__ void list_loop(const int *__restrict__ wl, int nslot, bool sum, int p,
                                          Load &&load, Use &&use) {
    int sl = 0, jcur = 0, jend = 0;
    // moves to the next listed particle; false when the list is done
    auto advance = [&]() -> bool {
        while (jcur >= jend) {
            if (sl >= nslot) return false;
            const int d = wl[sl * WAVE];
            sl++;
            jcur = d >> 4;
            jend = jcur + (d & 15);
        }
        return true;
    };
    bool have = sum && advance();
    decltype(load(0)) next{};
    if (have) next = load(jcur);
    while (any_lane(have)) {
        const auto cur = next;
        const int jc = jcur;
        const bool hc = have;
        if (have) {
            jcur++;
            have = advance();
            if (have) next = load(jcur);
        }
        if (hc && jc != p) use(jc, cur);
    }
}

// appends the particles of the lanes with pred set to the queue, one atomic
// per wave
__device__ __forceinline__ void queue_lanes(bool pred, int p, int *__restrict__ q,
                                            int *__restrict__ len) {
    const unsigned long long m = ballot(pred);
    if (m == 0) return;
    const int lane = (int)(threadIdx.x & (WAVE - 1));
    int at = 0;
    if (lane == 0) at = atomicAdd(len, __popcll(m));
    at = __shfl(at, 0, WAVE);
    if (pred) q[at + __popcll(m & ((1ull << lane) - 1ull))] = p;
}

// all_sph_gradh.F90:103-309, the h iteration, for every active particle.
//
// Potential-neighbour lists (BHhydrowalk_hgather) are recorded once per
// change of search radius: a group walk stores, for every lane, the leaves
// its own walk opens, in DFS order, as (first << 4) | count in HL_SLOTS
// slots per lane (slot-major, so the lanes of a wave read one contiguous row
// per step).  The iterations loop over each lane's own list, which is the
// reference's pp_potlist in the reference's order, so every sum is formed
// exactly as the reference forms it.  A lane whose list does not fit leaves
// its particle to k_hsolve_wave (hq) and stops: summed here over the tree
// walk, it held its wave in walks of the whole cloud (one particle on its
// way through the bisection took 1 s of a 131k-particle step).  On exit
// every other lane leaves rhotemp in rho, h_high in hhigh and its list
// length in nlist (-1: left to k_hsolve_wave) for k_hsolve_final; its list
// stays in hlist (a lane joins no walk after it has converged).
//
// WAVES > 0 holds the kernel to WAVES waves per SIMD (64 VGPRs at 8, with a
// few spills outside the candidate loops): more waves in flight hide more of
// the walks' memory latency, at the cost of issue slots taken from kernels
// running beside it.  0 leaves the register budget to the compiler
// (92 VGPRs, 5 waves).
template <int WAVES>
__global__ void __launch_bounds__(256)
__attribute__((amdgpu_waves_per_eu(WAVES > 0 ? WAVES : 1, WAVES > 0 ? WAVES : 8))) k_hsolve_iter(
    KGeom kg, bool box, int n, int nc, const HNode *__restrict__ hn, const double4 *__restrict__ rec,
    const int *__restrict__ cid, const int2 *__restrict__ root_range,
    const double *__restrict__ roots, int *__restrict__ hlist, int hl_cap,
    const uint8_t *__restrict__ active, const double *__restrict__ ktab,
    double h_fac, int pp_gather, double *__restrict__ h,
    double *__restrict__ rho, double *__restrict__ hhigh, int *__restrict__ nlist,
    int *__restrict__ hq, int *__restrict__ hq_len, unsigned long long *__restrict__ wstat) {
    const int p = xcd_block() * blockDim.x + threadIdx.x;
    const bool valid = p < n && active[p];
    int *wl = hlist + (size_t)(p / WAVE) * (HL_SLOTS * WAVE) + (threadIdx.x & (WAVE - 1));
    const double *w0 = ktab + T_W0 * KT;
    const double *wh = ktab + T_WH * KT;
    const double *h4 = ktab + KT_H4_OFF;   // (w0, wh, w4, wg) per index
    double rpx = 0, rpy = 0, rpz = 0, mp = 0, hp = 1, rextent = 0.0;
    int2 rr = make_int2(nc, nc);
    if (valid) {
        const double4 a = rec[p];
        rpx = a.x; rpy = a.y; rpz = a.z; mp = a.w;
        hp = h[p];
        const int k = cid[p];
        rr = root_range[k];
        rextent = roots[11 * k + 4];   // the particle's own cloud (bounding_box.F90:39)
    }
    double h_high = 0.0, h_old = hp, h_lower = 0.0, h_upper = rextent;
    double rhotemp = 0.0;
    int iteration = 0;
    bool iterating = valid;
    unsigned passes = 0, vis = 0, lvis = 0, walks = 0;
    int nslot = 0, cnt = 0, slot_max = 0;
    bool have_list = false, my_ovf = false;

    while (any_lane(iterating)) {
        passes++;
        bool newlist = false;
        if (iterating && hp > h_high) {
            h_high = hp * HMULT;
            newlist = true;
        }
        const double R = kg.range * h_high;
        const double invhp = 1.0 / hp;
        const double hfactor_p = cr_pow3(invhp);
        const double hrangesqd = kg.rangesqd * hp * hp;
        double srho = mp * w0[0] * hfactor_p;                  // :209-210
        double som = mp * hfactor_p * invhp * wh[0];
        // :214-231 for one potential neighbour
        auto pair = [&](double xj, double yj, double zj, double mj) {
            const double ex = xj - rpx, ey = yj - rpy, ez = zj - rpz;
            const double dsq = ex * ex + ey * ey + ez * ez;
            if (dsq >= hrangesqd) return;                       // :223
            const double drmag = sqrt(dsq) + SMALL_NUMBER;
            const int kern = (int)(kg.half * drmag * invhp);
            if (kern >= KERNTOT) return;                        // :227
            const double2 w = *reinterpret_cast<const double2 *>(h4 + 4 * (size_t)kern);
            srho = srho + mj * hfactor_p * w.x;
            som = som + mj * hfactor_p * invhp * w.y;
        };

        if (!have_list || any_lane(newlist)) {
            // record every iterating lane's list (unchanged radii give the same
            // lists); converged lanes keep theirs
            if (iterating) {
                nslot = 0;
                cnt = 0;
            }
            bool lovf = false;   // the list is full: the lane passes over the rest
            vis += group_walk(hn, nc, iterating, rr.x, rr.y, lvis,
                              [&](const HNode &nd, bool) {
                                  return lovf ? WALK_SKIP : hgather_visit(nd, rpx, rpy, rpz, R);
                              },
                              [&](const HNode &nd, bool mine) {
                if (mine) {
                    cnt += nd.leaf;                       // the reference's pp_pot
                    if (leaf_near(nd, rpx, rpy, rpz, R, box)) {
                        if (nslot < hl_cap)
                            wl[nslot * WAVE] = (nd.first << 4) | nd.leaf;
                        else
                            lovf = true;
                        nslot++;
                    }
                }
            });
            if (iterating) {
                slot_max = max(slot_max, nslot);
                my_ovf = lovf;
                if (lovf) iterating = false;
            }
            have_list = true;
            walks++;
        }
        // too few potential neighbours: grow h and gather again (:185-189)
        const bool grow = iterating && newlist && cnt < pp_gather;
        const bool sum = iterating && !grow;
        list_loop(wl, nslot, sum, p, [&](int j) { return rec[j]; },
                  [&](int, const double4 &a) { pair(a.x, a.y, a.z, a.w); });

        if (grow) {
            h_high = 0.0;
            hp = hp * HMULT;
        } else if (iterating) {
            rhotemp = srho;
            const double hnew = h_fac * ref_pow_third(mp / rhotemp);
            if (fabs(hp - hnew) / hp < H_CON && iteration >= 1) {  // :246
                iterating = false;
            } else if (iteration < GRADH_ITERATION_MAX) {           // :252
                hp = hnew;
                iteration++;
            } else if (iteration == GRADH_ITERATION_MAX) {          // :256
                h_upper = rextent;
                h_lower = 0.0;
                hp = 0.5 * (h_lower + h_upper);
                iteration++;
            } else if (iteration < 2 * GRADH_ITERATION_MAX) {       // :262
                double fb;
                if (rhotemp > SMALL_NUMBER)
                    fb = cr_pow3(hp) - cr_pow3(h_fac) * mp / rhotemp;
                else
                    fb = 1.0;
                if (fb > 0.0)
                    h_upper = hp;
                else
                    h_lower = hp;
                hp = 0.5 * (h_lower + h_upper);
                iteration++;
            } else {                                                // :276-279
                iterating = false;
            }
        }
    }
    (void)h_old;   // the final h is formed from rhotemp alone (:317)
    if (valid) {
        rho[p] = rhotemp;
        hhigh[p] = h_high;
        nlist[p] = my_ovf ? -1 : nslot;
    }
    queue_lanes(my_ovf, p, hq, hq_len);
    // walk statistics: cells visited / lane visits, passes, lane iterations,
    // list walks, longest list
    wave_stats(wstat, 2, vis, lvis);
    unsigned long long it = valid ? (unsigned long long)iteration : 0ull;
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) it += __shfl_xor(it, o, 64);
    const int smx = wave_max_int(slot_max);
    if ((threadIdx.x & 63) == 0) {
        unsigned long long *ws = ctr_row(wstat);
        atomicAdd(ws + 4, (unsigned long long)passes);
        atomicMax(ws + 5, (unsigned long long)passes);
        atomicAdd(ws + 6, it);
        atomicAdd(ws + 7, 1ull);
        atomicAdd(ws + 10, (unsigned long long)walks);
        atomicMax(ws + 12, (unsigned long long)smx);
    }
}

// all_sph_gradh.F90:310-489: with h from the converged density, the gather
// sums rho, Omega, div v and zeta over the last potential-neighbour list, for
// the particles whose list k_hsolve_iter holds; k_hsolve_wave does the others.
__global__ void __launch_bounds__(256) k_hsolve_final(
    KGeom kg, bool box, int n, const double4 *__restrict__ rec, const int *__restrict__ hlist, const uint8_t *__restrict__ active,
    const double *__restrict__ ktab, double h_fac, const double *__restrict__ hhigh,
    const int *__restrict__ nlist, double *__restrict__ h, double *__restrict__ zeta,
    double *__restrict__ rho, double *__restrict__ omega, double *__restrict__ divv,
    double *__restrict__ drhodt, int *__restrict__ hq, int *__restrict__ hq_len,
    int *__restrict__ err) {
    const int p = xcd_block() * blockDim.x + threadIdx.x;
    bool valid = p < n && active[p];
    const int *wl = hlist + (size_t)(p / WAVE) * (HL_SLOTS * WAVE) + (threadIdx.x & (WAVE - 1));
    const double *w0 = ktab + T_W0 * KT;
    const double *wh = ktab + T_WH * KT;
    const double *wg = ktab + T_WG * KT;
    const double *h4 = ktab + KT_H4_OFF;   // (w0, wh, w4, wg) per index
    const double4 *vrec = rec + n;
    double rpx = 0, rpy = 0, rpz = 0, mp = 0, vpx = 0, vpy = 0, vpz = 0, hp = 1;
    int nslot = 0;
    bool beyond = false;
    if (valid) nslot = nlist[p];
    valid = valid && nslot >= 0;
    if (valid) {
        const double4 a = rec[p], b = vrec[p];
        rpx = a.x; rpy = a.y; rpz = a.z; mp = a.w;
        vpx = b.x; vpy = b.y; vpz = b.z;
        hp = h_fac * ref_pow_third(mp / rho[p]);                 // :317
        // a final h beyond the list's radius can reach particles past it in
        // leaves the box test left out: left to k_hsolve_wave as well
        beyond = box && kg.range * hp > kg.range * hhigh[p];
        valid = !beyond;
    }
    queue_lanes(beyond, p, hq, hq_len);
    const double invhp = 1.0 / hp;
    const double hfactor_p = cr_pow3(invhp);
    const double hrangesqd = kg.rangesqd * hp * hp;
    // self contributions (:323-346)
    double srho = mp * w0[0] * hfactor_p;
    double som = mp * hfactor_p * invhp * wh[0];
    double sdiv = 0.0;
    double szeta = mp * invhp * invhp * wg[0];
    // :356-381 for one potential neighbour
    auto pair = [&](double xj, double yj, double zj, double mj, int j) {
        const double ex = xj - rpx, ey = yj - rpy, ez = zj - rpz;
        const double dsq = ex * ex + ey * ey + ez * ez;
        if (dsq > hrangesqd) return;                            // :364
        const double drmag = sqrt(dsq) + SMALL_NUMBER;
        const int kern = (int)(kg.half * drmag * invhp);
        if (kern > KERNTOT) return;                             // :368
        const double4 vj = vrec[j];
        const double dvx = vj.x - vpx, dvy = vj.y - vpy, dvz = vj.z - vpz;
        const double dvdr = dvx * ex + dvy * ey + dvz * ez;
        const double4 w = *reinterpret_cast<const double4 *>(h4 + 4 * (size_t)kern);
        srho = srho + mj * hfactor_p * w.x;
        som = som + mj * hfactor_p * invhp * w.y;
        sdiv = sdiv - mj * dvdr * w.z * hfactor_p * invhp / drmag;
        szeta = szeta + mj * invhp * invhp * w.w;
    };
    list_loop(wl, nslot, valid, p, [&](int j) { return rec[j]; },
              [&](int j, const double4 &a) { pair(a.x, a.y, a.z, a.w, j); });
    if (valid) {
        const double om = 1.0 + ((hp * som) / (3.0 * srho));
        const double dv = sdiv / srho;
        rho[p] = srho;
        omega[p] = om;
        divv[p] = dv;
        drhodt[p] = -srho * dv / om;
        h[p] = hp;
        zeta[p] = -(hp * szeta) / (3.0 * srho * om);
        if (hp < 0.0) atomicOr(err, 1);
    }
}

// ---- searches of one particle by a whole wave ------------------------------
//
// The lane kernels give a particle to a lane, and a wave's time is its
// slowest lane's; with few waves in the launch (small clouds) or one particle
// with a long search (far outskirts, the bisection of the h solve) the
// serial chain of one lane's loads is what the launch takes.  Here a wave
// serves one particle: 64 nodes are tested at once, the candidates are
// evaluated 64 at once, and only the additions of the terms inside the
// kernel range are serial, because the sums keep the order of the
// reference's list (DFS order) and with it its rounding.

// nodes of a search front, and leaves of a list, held in LDS.  512 entries
// hold a front of the largest chain of a resumed search (7 siblings on each
// of LMAX levels) and the lists of all but a few particles; 8 KB per wave
// leave room for 20 waves on a CU.
constexpr int WS_CAP = 512;
static_assert(WS_CAP >= 8 * (LMAX + 1), "a resumed search's first front must fit");

// batches of 64 candidates that a density pass has in flight
constexpr int WS_U = 4;

struct WaveSearch {
    int front[2][WS_CAP];
    int leaf[WS_CAP];      // leaves found: (first particle << 4) | particles
    double4 term[WAVE];    // terms in list order: of one batch, or the densities of WS_U
};
static_assert(sizeof(double4) == WS_U * sizeof(double), "the densities fit");

// inclusive prefix sum over the lanes of a wave
__device__ __forceinline__ int wave_prefix(int v, int lane) {
#pragma unroll
    for (int d = 1; d < WAVE; d <<= 1) {
        const int u = __shfl_up(v, d, WAVE);
        if (lane >= d) v += u;
    }
    return v;
}

// The leaves below root, from the subtree at resume on (DFS order), that
// test() passes together with all their ancestors at or below the start, in
// DFS order into L.leaf; returns their number.  The front is expanded level
// by level, each branch's children in its place.  A front that would pass
// WS_CAP is cut: resume then names the first node left out (another call
// continues there), else it is -1.  Every call moves resume on or ends the
// search: the node it starts at is expanded until it is a leaf or fails.
//
// MASKED: a search for several particles, whose tests of a node are the bits
// of test().  masks holds, beside the two fronts, the particles that passed
// every ancestor of an entry: a leaf's test does not imply its ancestors'
// (its sphere need not lie within theirs), so the particles that open it are
// those of its entry's mask and its own test.  They are left in
// masks[0 .. number of leaves).  all: the particles searched for.
template <bool MASKED, class Test>
__device__ __forceinline__ int wave_leaves(WaveSearch &L, uint8_t *masks, unsigned all,
                                           const BNode *__restrict__ bn, int root, int &resume,
                                           unsigned &visits, Test &&test) {
    const int lane = (int)(threadIdx.x & (WAVE - 1));
    int len = 0, cur = 0;
    if (resume == root) {
        if (lane == 0) {
            L.front[0][0] = root;
            if (MASKED) masks[0] = (uint8_t)all;
        }
        len = 1;
    } else {
        // the rest of the tree in DFS order: resume and its later siblings,
        // then the later siblings of each ancestor
        int c = resume, p = bn[c].parent;
        for (;;) {
            const int end = bn[p].fc - bn[p].k;
            if (c + lane < end) L.front[0][len + lane] = c + lane;
            len += max(end - c, 0);
            if (p == root) break;
            c = p + 1;
            p = bn[p].parent;
        }
        if (MASKED) {   // their ancestors' tests again, one entry per lane
            wave_lds_fence();
            for (int e = lane; e < len; e += WAVE) {
                unsigned mk = all;
                for (int a = bn[L.front[0][e]].parent;; a = bn[a].parent) {
                    mk &= test(bn[a]);
                    if (a == root) break;
                }
                masks[e] = (uint8_t)mk;
            }
        }
    }
    resume = -1;
    bool branches = true;
    while (branches) {
        branches = false;
        int out = 0;
        const int *in = L.front[cur];
        int *dst = L.front[cur ^ 1];
        wave_lds_fence();
        for (int base = 0; base < len; base += WAVE) {
            const int e = base + lane;
            int v = 0, nout = 0, first = 0;   // a leaf that passed is kept as ~id
            unsigned mk = 0;
            bool branch = false;
            if (e < len) {
                v = in[e];
                if (MASKED) mk = masks[cur * WS_CAP + e];
                if (v < 0) {
                    nout = 1;
                    first = v;
                } else {
                    const BNode nd = bn[v];
                    mk = MASKED ? mk & test(nd) : (unsigned)test(nd);
                    if (mk) {
                        branch = nd.k < 0;
                        nout = branch ? -nd.k : 1;
                        first = branch ? nd.fc : ~v;
                    }
                }
            }
            visits += (unsigned)min(WAVE, len - base);
            const int incl = wave_prefix(nout, lane);
            const unsigned long long over = ballot(nout > 0 && out + incl > WS_CAP);
            const int cutlane = over ? __ffsll((long long)over) - 1 : WAVE;
            if (lane < cutlane) {
                const int o = out + incl - nout;
                for (int i = 0; i < nout; i++) {
                    dst[o + i] = first + i;
                    if (MASKED) masks[(cur ^ 1) * WS_CAP + o + i] = (uint8_t)mk;
                }
            }
            branches = branches || ballot(branch && lane < cutlane) != 0;
            if (over) {
                const int r = __shfl(v, cutlane, WAVE);
                resume = r < 0 ? ~r : r;
                if (cutlane > 0) out += __shfl(incl, cutlane - 1, WAVE);
                break;
            }
            out += __shfl(incl, WAVE - 1, WAVE);
        }
        wave_lds_fence();
        len = out;
        cur ^= 1;
    }
    // the nodes kept are all leaves now
    for (int e = lane; e < len; e += WAVE) {
        const BNode &nd = bn[~L.front[cur][e]];
        L.leaf[e] = (nd.fc << 4) | nd.k;
        if (MASKED) masks[e] = masks[cur * WS_CAP + e];
    }
    wave_lds_fence();
    return len;
}

template <class Test>
__device__ __forceinline__ int wave_leaves(WaveSearch &L, const BNode *__restrict__ bn, int root,
                                           int &resume, unsigned &visits, Test &&test) {
    return wave_leaves<false>(L, nullptr, 0u, bn, root, resume, visits, test);
}

// Calls use(j, record, ok) for the particles of the leaves found, 64 slots
// at a time in list order: 8 leaves, lane l the particle l & 7 of leaf l >> 3
// (ok: that particle exists).  The loads of four batches are in flight
// together.  use(j, record, ok, e) has the list entry e too, and returns true to
// stop.
template <class Use>
__device__ __forceinline__ void wave_candidates(const WaveSearch &L, int nleaf,
                                                const double4 *__restrict__ rec, int p,
                                                Use &&use) {
    const int lane = (int)(threadIdx.x & (WAVE - 1)), sub = lane >> 3, k = lane & 7;
    constexpr int U = 4;
    for (int e0 = 0; e0 < nleaf; e0 += 8 * U) {
        double4 a[U];
        int j[U];
        bool ok[U];
#pragma unroll
        for (int u = 0; u < U; u++) {
            const int e = e0 + 8 * u + sub;
            const int d = e < nleaf ? L.leaf[e] : 0;
            ok[u] = k < (d & 15);
            j[u] = ok[u] ? (d >> 4) + k : p;
            a[u] = rec[j[u]];
        }
#pragma unroll
        for (int u = 0; u < U; u++)
            if (e0 + 8 * u < nleaf && use(j[u], a[u], ok[u], e0 + 8 * u + sub)) return;
    }
}

// all_sph_gradh.F90:103-489 for one particle per wave: the state machine of
// k_hsolve_iter and the sums of k_hsolve_final, with the same arithmetic in
// the same order, so both give the same bits.  Runs over the particles
// hq[0 .. *hq_len) when hq is given, else over all n.
//
// While the bisection runs, a pass only decides whether h is too large.  Its
// density sum grows with every term (masses and kernel are not negative), so
// the pass ends as soon as the sum shows that h exceeds the h of that density
// by more than the convergence test's 2 % (2.1 % here, which covers the
// rounding of the powers): the rest of the sum cannot change the decision.
// The bisection starts at half the cloud's extent, where the full sum takes
// in most of the cloud.
//
// Bound by the latency of the front's node loads and of the serial sums
// (about a microsecond each per pass), hidden by the 12 waves on a CU.
// Measured (steady evaluation, beside the gravity walk): 60 us at 2,048
// particles, 232 us at 16,384 and 4.4 ms at 131,072, against 680, 980 and
// 3,560 us of the lane kernels, which keep 64 particles' worth of work per
// wave (first evaluation of a 2,053-particle Plummer sphere, whose outskirts
// go through the bisection: 21 -> 3.2 ms).  Contexts of up to HSOLVE_WAVE_MAX
// particles take this kernel, larger ones the lane kernels.  The profiles
// cross at different sizes, and the line lies between them.  Steady
// evaluations, waves / lanes (ms), FP64: uniform 2.6 / 2.7 at 32,768, 3.3 / 3.0
// at 49,152, 3.8 / 3.2 at 65,536, 5.5 / 4.3 at 98,304; r^-2 2.2 / 3.8, 3.4 /
// 3.8, 4.0 / 4.4, 5.2 / 5.7 (6.6 / 6.4 at 131,071); Plummer 2.6 / 2.9, 3.4 /
// 3.2, 4.1 / 3.8, 5.8 / 4.7.  Mixed: uniform 2.1 / 2.5, 2.5 / 2.5, 2.8 / 2.4,
// 4.0 / 3.2; r^-2 2.0 / 3.5, 3.0 / 3.4, 3.6 / 3.9, 4.5 / 5.1; Plummer 2.2 /
// 2.6, 2.7 / 2.8, 3.1 / 3.2, 4.3 / 3.6.  Held to 4 or 5 waves per SIMD instead
// of the compiler's 149 registers (three) it was slower (242 and 289 us at
// 16,384).
constexpr int HSOLVE_WAVE_MAX = 1 << 16;

__global__ void __launch_bounds__(256) k_hsolve_wave(
    KGeom kg, bool box, int n, const BNode *__restrict__ bn, const double4 *__restrict__ rec,
    const int *__restrict__ cid, const double *__restrict__ roots,
    const uint8_t *__restrict__ active, const double *__restrict__ ktab, double h_fac,
    int pp_gather, int list_cap, const int *__restrict__ hq, const int *__restrict__ hq_len,
    double *__restrict__ h, double *__restrict__ zeta, double *__restrict__ rho,
    double *__restrict__ omega, double *__restrict__ divv, double *__restrict__ drhodt,
    int *__restrict__ err, unsigned long long *__restrict__ wstat) {
    __shared__ WaveSearch lds[256 / WAVE];
    WaveSearch &L = lds[threadIdx.x / WAVE];
    const int lane = (int)(threadIdx.x & (WAVE - 1)), wv = (int)(threadIdx.x / WAVE);
    const double *w0 = ktab + T_W0 * KT;
    const double *wh = ktab + T_WH * KT;
    const double *wg = ktab + T_WG * KT;
    const double *h4 = ktab + KT_H4_OFF;   // (w0, wh, w4, wg) per index
    const double4 *vrec = rec + n;
    const int total = hq ? uniform(*hq_len) : n;
    // each block a contiguous run of the particles, its waves in turn
    const int nb = (int)gridDim.x, blk = xcd_block();
    const int lo = (int)((long long)blk * total / nb), hi = (int)((long long)(blk + 1) * total / nb);
    unsigned passes = 0, passmax = 0, iters = 0, nwave = 0, walks = 0, streamed = 0, longest = 0,
             vis = 0;
    for (int t = lo + wv; t < hi; t += 256 / WAVE) {
        const int p = hq ? uniform(hq[t]) : t;
        if (!active[p]) continue;
        const double4 self = rec[p];
        const double rpx = self.x, rpy = self.y, rpz = self.z, mp = self.w;
        const int root = uniform(cid[p]);   // a cloud's root has the cloud's BFS id
        const double rextent = roots[11 * root + 4];
        double hp = h[p], h_high = 0.0, h_lower = 0.0, h_upper = rextent, rhotemp = 0.0;
        int iteration = 0, nleaf = 0;
        unsigned mypasses = 0;
        bool complete = false;   // L.leaf holds the whole list of radius h_high
        // BHhydrowalk_hgather.F90:40 at radius R, and with fresh boxes the
        // nodes that can hold a particle within Rb
        auto near = [&](const BNode &nd, double R, double Rb) {
            const double dx = nd.r[0] - rpx, dy = nd.r[1] - rpy, dz = nd.r[2] - rpz;
            const double drsqd = dx * dx + dy * dy + dz * dz;
            if (!(drsqd <= (R + nd.rmax) * (R + nd.rmax))) return false;
            if (!box) return true;
            const double ex = fmax(fabs(dx) - (double)nd.half[0], 0.0);
            const double ey = fmax(fabs(dy) - (double)nd.half[1], 0.0);
            const double ez = fmax(fabs(dz) - (double)nd.half[2], 0.0);
            return ex * ex + ey * ey + ez * ez <= Rb * Rb * (1.0 + 1.0e-12);
        };
        // f(nleaf) over the candidates within Rb (of the list of radius
        // h_high): from the list when it is complete, else searched anew in
        // pieces of at most WS_CAP leaves.  f returns true to stop.
        auto sweep = [&](double Rb, bool from_list, auto &&f) {
            if (from_list) {
                f(nleaf);
                return;
            }
            streamed++;
            complete = false;
            const double R = kg.range * h_high;
            int resume = root;
            do {
                const int m = wave_leaves(L, bn, root, resume, vis,
                                          [&](const BNode &nd) { return near(nd, R, Rb); });
                if (f(m)) break;
            } while (resume >= 0);
        };
        bool iterating = true;
        while (iterating) {
            passes++;
            mypasses++;
            if (hp > h_high) {
                h_high = hp * HMULT;
                const double R = kg.range * h_high;
                walks++;
                int resume = root;
                nleaf = wave_leaves(L, bn, root, resume, vis,
                                    [&](const BNode &nd) { return near(nd, R, R); });
                complete = resume < 0 && nleaf <= list_cap;
                longest = max(longest, (unsigned)nleaf);
                // the particles of the reference's list (:185-189): those of
                // the leaves found are a part of it
                auto count = [&](int m) {
                    int s = 0;
                    for (int e = lane; e < m; e += WAVE) s += L.leaf[e] & 15;
                    return uniform(__shfl(wave_prefix(s, lane), WAVE - 1, WAVE));
                };
                int cnt = count(nleaf);
                if (cnt < pp_gather && (box || resume >= 0)) {
                    // by the sphere test alone
                    complete = false;
                    cnt = 0;
                    resume = root;
                    do {
                        const int m = wave_leaves(L, bn, root, resume, vis, [&](const BNode &nd) {
                            const double dx = nd.r[0] - rpx, dy = nd.r[1] - rpy,
                                         dz = nd.r[2] - rpz;
                            return dx * dx + dy * dy + dz * dz <= (R + nd.rmax) * (R + nd.rmax);
                        });
                        cnt += count(m);
                    } while (resume >= 0 && cnt < pp_gather);
                }
                if (cnt < pp_gather) {   // grow h and gather again
                    h_high = 0.0;
                    hp = hp * HMULT;
                    continue;
                }
            }
            const double invhp = 1.0 / hp;
            const double hfactor_p = cr_pow3(invhp);
            const double hrangesqd = kg.rangesqd * hp * hp;
            double srho = mp * w0[0] * hfactor_p;                  // :209-210
            const bool bisecting = iteration > GRADH_ITERATION_MAX &&
                                   iteration < 2 * GRADH_ITERATION_MAX;
            const double hq1 = h_fac / (0.979 * hp);
            const double enough = mp * hq1 * hq1 * hq1;
            bool decided = bisecting && srho >= enough;
            if (!decided) {
                sweep(kg.range * hp, complete, [&](int m) {
                    // WS_U batches of 64 at once: their records, then their
                    // table entries are in flight together (a particle of a
                    // Plummer sphere's outskirts sums 2,000 terms in each of
                    // 40 passes, one after the other: 1,343 -> 1,145 us there)
                    double *term = reinterpret_cast<double *>(L.term);
                    const int sub = lane >> 3, k8 = lane & 7;
                    for (int e0 = 0; e0 < m && !decided; e0 += 8 * WS_U) {
                        double4 a[WS_U];
                        double w[WS_U];
                        bool in[WS_U];
#pragma unroll
                        for (int u = 0; u < WS_U; u++) {
                            const int e = e0 + 8 * u + sub;
                            const int d = e < m ? L.leaf[e] : 0;
                            const int j = (d >> 4) + k8;
                            in[u] = k8 < (d & 15) && j != p;
                            a[u] = rec[in[u] ? j : p];
                        }
#pragma unroll
                        for (int u = 0; u < WS_U; u++) {   // :214-231
                            const double ex = a[u].x - rpx, ey = a[u].y - rpy, ez = a[u].z - rpz;
                            const double dsq = ex * ex + ey * ey + ez * ez;
                            const double drmag = sqrt(dsq) + SMALL_NUMBER;
                            const int kern = (int)(kg.half * drmag * invhp);
                            in[u] = in[u] && !(dsq >= hrangesqd) && !(kern >= KERNTOT);
                            w[u] = in[u] ? h4[4 * (size_t)kern] : 0.0;
                        }
                        int cnt = 0;
#pragma unroll
                        for (int u = 0; u < WS_U; u++) {
                            const unsigned long long mask = ballot(in[u]);
                            if (in[u])
                                term[cnt + __popcll(mask & ((1ull << lane) - 1ull))] =
                                    a[u].w * hfactor_p * w[u];
                            cnt += __popcll(mask);
                        }
                        wave_lds_fence();
#pragma unroll 16
                        for (int i = 0; i < cnt; i++) srho = srho + term[i];
                        wave_lds_fence();
                        decided = bisecting && srho >= enough;
                    }
                    return decided;
                });
            }
            rhotemp = srho;
            if (decided) {   // fb > 0 (:262) and not converged
                h_upper = hp;
                hp = 0.5 * (h_lower + h_upper);
                iteration++;
                continue;
            }
            const double hnew = h_fac * ref_pow_third(mp / rhotemp);
            if (fabs(hp - hnew) / hp < H_CON && iteration >= 1) {  // :246
                iterating = false;
            } else if (iteration < GRADH_ITERATION_MAX) {           // :252
                hp = hnew;
                iteration++;
            } else if (iteration == GRADH_ITERATION_MAX) {          // :256
                h_upper = rextent;
                h_lower = 0.0;
                hp = 0.5 * (h_lower + h_upper);
                iteration++;
            } else if (iteration < 2 * GRADH_ITERATION_MAX) {       // :262
                double fb;
                if (rhotemp > SMALL_NUMBER)
                    fb = cr_pow3(hp) - cr_pow3(h_fac) * mp / rhotemp;
                else
                    fb = 1.0;
                if (fb > 0.0)
                    h_upper = hp;
                else
                    h_lower = hp;
                hp = 0.5 * (h_lower + h_upper);
                iteration++;
            } else {                                                // :276-279
                iterating = false;
            }
        }
        // :310-489 with h from the converged density
        hp = h_fac * ref_pow_third(mp / rhotemp);                   // :317
        const double4 vself = vrec[p];
        const double invhp = 1.0 / hp;
        const double hfactor_p = cr_pow3(invhp);
        const double hrangesqd = kg.rangesqd * hp * hp;
        double srho = mp * w0[0] * hfactor_p;
        double som = mp * hfactor_p * invhp * wh[0];
        double sdiv = 0.0;
        double szeta = mp * invhp * invhp * wg[0];
        const bool from_list = complete && !(box && kg.range * hp > kg.range * h_high);
        sweep(kg.range * hp, from_list, [&](int m) {
            wave_candidates(L, m, rec, p, [&](int j, const double4 &a, bool ok, int) {
                const double ex = a.x - rpx, ey = a.y - rpy, ez = a.z - rpz;
                const double dsq = ex * ex + ey * ey + ez * ez;
                const double drmag = sqrt(dsq) + SMALL_NUMBER;
                const int kern = (int)(kg.half * drmag * invhp);
                const bool in = ok && j != p && !(dsq > hrangesqd) && !(kern > KERNTOT);
                const unsigned long long mask = ballot(in);
                if (in) {
                    const double4 vj = vrec[j];
                    const double dvx = vj.x - vself.x, dvy = vj.y - vself.y, dvz = vj.z - vself.z;
                    const double dvdr = dvx * ex + dvy * ey + dvz * ez;
                    const double4 w = *reinterpret_cast<const double4 *>(h4 + 4 * (size_t)kern);
                    L.term[__popcll(mask & ((1ull << lane) - 1ull))] =
                        make_double4(a.w * hfactor_p * w.x, a.w * hfactor_p * invhp * w.y,
                                     a.w * dvdr * w.z * hfactor_p * invhp / drmag,
                                     a.w * invhp * invhp * w.w);
                }
                wave_lds_fence();
                const int cnt = __popcll(mask);
#pragma unroll 4
                for (int i = 0; i < cnt; i++) {
                    const double4 v = L.term[i];
                    srho = srho + v.x;
                    som = som + v.y;
                    sdiv = sdiv - v.z;
                    szeta = szeta + v.w;
                }
                wave_lds_fence();
                return false;
            });
            return false;
        });
        if (lane == 0) {
            const double om = 1.0 + ((hp * som) / (3.0 * srho));
            const double dv = sdiv / srho;
            rho[p] = srho;
            omega[p] = om;
            divv[p] = dv;
            drhodt[p] = -srho * dv / om;
            h[p] = hp;
            zeta[p] = -(hp * szeta) / (3.0 * srho * om);
            if (hp < 0.0) atomicOr(err, 1);
        }
        iters += (unsigned)iteration;
        passmax = max(passmax, mypasses);
        nwave++;
    }
    if (nwave > 0 && lane == 0) {
        unsigned long long *ws = ctr_row(wstat);
        atomicAdd(ws + 2, (unsigned long long)((vis + WAVE - 1) / WAVE));
        atomicAdd(ws + 3, (unsigned long long)vis);
        atomicAdd(ws + 4, (unsigned long long)passes);
        atomicMax(ws + 5, (unsigned long long)passmax);
        atomicAdd(ws + 6, (unsigned long long)iters);
        atomicAdd(ws + 7, (unsigned long long)nwave);
        atomicAdd(ws + 10, (unsigned long long)walks);
        atomicAdd(ws + 11, (unsigned long long)streamed);
        atomicMax(ws + 12, (unsigned long long)longest);
    }
}

constexpr int OVF_PER_WAVE = 1;

// get_neib.F90:46-118: gather-or-scatter neighbours in walk (DFS) order.
// Rows of pp_limit ids; particles with more neighbours only get their count
// here (the reference does not store their list either, :115-118) and are
// listed completely by the OVERFLOW_PASS instance.
template <bool OVERFLOW_PASS>
__global__ void __launch_bounds__(256) k_neib(KGeom kg, bool box, int n, const int *__restrict__ ovf_idx,
                                              int nc,
                                              const HNode *__restrict__ hn,
                                              const double4 *__restrict__ rec,
                                              const int *__restrict__ cid,
                                              const int2 *__restrict__ root_range,
                                              const uint8_t *__restrict__ active, int pp_limit,
                                              int *__restrict__ pptot, int *__restrict__ pplist,
                                              const int *__restrict__ ovf_off,
                                              int *__restrict__ ovf_list,
                                              int *__restrict__ ovf_count,
                                              unsigned long long *__restrict__ wstat) {
    // the overflow pass runs over the list of overflow particles (n of them),
    // OVF_PER_WAVE to a wave: their walks are long, and a wave walks the union
    // of its lanes' walks, so a few lanes per wave keep many waves in flight
    const int t = xcd_block() * blockDim.x + threadIdx.x;
    const int ot = (t / WAVE) * OVF_PER_WAVE + (t % WAVE);
    const bool ovf_lane = (t % WAVE) < OVF_PER_WAVE && ot < n;
    const int p = OVERFLOW_PASS ? (ovf_lane ? ovf_idx[ot] : 0) : t;
    const bool valid = OVERFLOW_PASS ? ovf_lane : (p < n && active[p]);
    double rpx = 0, rpy = 0, rpz = 0, hp = 0;
    if (valid) {
        const double4 a = rec[p];
        rpx = a.x; rpy = a.y; rpz = a.z;
        hp = a.w;
    }
    const double hrangesqd_p = kg.rangesqd * hp * hp;
    const double R = kg.range * hp;
    int tot = 0;
    int *row = nullptr;
    int lim = pp_limit;   // entries this lane may store
    if (valid) {
        row = OVERFLOW_PASS ? ovf_list + ovf_off[p] : pplist + (size_t)p * pp_limit;
        if (OVERFLOW_PASS) lim = pptot[p];
    }
    unsigned lvis = 0;
    const int2 rr = valid ? root_range[cid[p]] : make_int2(nc, nc);
    const unsigned vis = group_walk(
        hn, nc, valid, rr.x, rr.y, lvis,
        [&](const HNode &nd, bool) -> int {
            const double dx = nd.r[0] - rpx, dy = nd.r[1] - rpy, dz = nd.r[2] - rpz;
            const double drsqd = dx * dx + dy * dy + dz * dz;
            const double m1 = (R + nd.rmax) * (R + nd.rmax);
            const double m2 = (nd.hrangemax + nd.rmax) * (nd.hrangemax + nd.rmax);
            if (!(drsqd <= m1 || drsqd <= m2)) return WALK_SKIP;   // BHhydro_walk.F90:43
            // and the box test at the larger of the two radii (hgather_visit)
            const double Rb = fmax(R, nd.hrangemax);
            if (box && box_dist2(nd, dx, dy, dz) > Rb * Rb * (1.0 + 1.0e-12)) return WALK_SKIP;
            return nd.leaf == 0 ? WALK_DESCEND : WALK_LEAF;
        },
        [&](const HNode &nd, bool mine) {
            const int k = nd.leaf, f0 = nd.first;
            for (int i = 0; i < k; i++) {
                const int j = f0 + i;
                const double4 aj = rec[j];   // one scalar load per candidate
                const double xj = aj.x, yj = aj.y, zj = aj.z, hj = aj.w;
                if (!mine || j == p) continue;
                const double hrangesqd_pp = kg.rangesqd * hj * hj;
                const double ex = xj - rpx, ey = yj - rpy, ez = zj - rpz;
                const double dsq = ex * ex + ey * ey + ez * ez;
                if (dsq <= hrangesqd_p || dsq <= hrangesqd_pp) {
                    if (tot < lim) row[tot] = j;
                    tot++;
                }
            }
        });
    if (valid && !OVERFLOW_PASS) {
        pptot[p] = tot;
        if (tot > pp_limit) atomicAdd(ovf_count, 1);
    }
    if (!OVERFLOW_PASS) wave_stats(wstat, 8, vis, lvis);
}

// a lane's value in scalar registers
__device__ __forceinline__ double lane_value(double v, int from) {
    return __hiloint2double(__builtin_amdgcn_readlane(__double2hiint(v), from),
                            __builtin_amdgcn_readlane(__double2loint(v), from));
}

// get_neib.F90:46-118 from searches by whole waves: a wave takes NW_T
// consecutive particles (one: a row above pp_limit).
//
// Every particle j with r^2 <= KERNRANGESQD h_p^2 or r^2 <= KERNRANGESQD
// h_j^2 lies in a leaf that the reference's BHhydro_walk opens for p: every
// ancestor's bounding sphere holds j, so |r_p - r_c| <= |r_p - r_j| + rmax_c,
// and hrangemax_c >= KERNRANGE h_j.  The reference keeps exactly those
// particles, in DFS order.  Any search that finds a superset of those leaves,
// in DFS order, therefore yields the reference's lists once each candidate
// passes the reference's pair test (formed as get_neib.F90:89-95 forms it).
//
// The leaves come from a front of 64 nodes at a time (wave_leaves), in DFS
// order.  With fresh boxes, those whose box lies within max(KERNRANGE h_p,
// hrangemax) of any of the particles: that box holds every neighbour in it.
// With stale ones (particles moved since the tree was stocked) a neighbour
// can lie outside its leaf's and its leaf's ancestors' spheres, and the
// reference's list is what its walk opens: each particle's path is followed
// by itself (BHhydro_walk.F90:36-43 on the leaf and on all its ancestors), so
// that the rows, and the counts of both passes, are those of its own walk.
// 64 candidates at a time are put to each particle's pair test, and the
// matches are placed by their rank among the lanes.
//
// Why: a wave that walks node by node for 64 particles needs 0.3 us per cell
// and 0.1 us per candidate, one after the other: 275 us at 2,048 particles and
// 525 us at 16,384, on the way to the hydro forces; now 40 and 90 us.  1M r^-2
// sphere: 1.80 -> 1.73 ms, bound by the vector ALU and the rows' stores (7.2e8
// instructions).  Eight particles share a search and its candidates; their own
// tests, not one of their common box, keep a wave that straddles two branches
// of the tree from opening all that lies between (1M: 17.8 ms).
constexpr int NW_T = 8;

template <bool OVERFLOW_PASS, bool BOX>
__global__ void __launch_bounds__(256) k_neib_wave(
    KGeom kg, int n, const int *__restrict__ ovf_idx, const BNode *__restrict__ bn,
    const double4 *__restrict__ rec, const int *__restrict__ cid,
    const uint8_t *__restrict__ active, int pp_limit, int *__restrict__ pptot,
    int *__restrict__ pplist, const int *__restrict__ ovf_off, int *__restrict__ ovf_list,
    int *__restrict__ ovf_count, unsigned long long *__restrict__ wstat) {
    constexpr int T = OVERFLOW_PASS ? 1 : NW_T;
    __shared__ WaveSearch lds[256 / WAVE];
    WaveSearch &L = lds[threadIdx.x / WAVE];
    // the particles whose own walk opens a node, for several on stale boxes
    constexpr bool MASKED = !BOX && T > 1;
    static_assert(NW_T <= 8, "a mask is a byte");
    __shared__ uint8_t masks_all[256 / WAVE][MASKED ? 2 * WS_CAP : 1];
    uint8_t *masks = masks_all[threadIdx.x / WAVE];
    const int lane = (int)(threadIdx.x & (WAVE - 1));
    const int t0 = (xcd_block() * (256 / WAVE) + (int)(threadIdx.x / WAVE)) * T;
    if (t0 >= n) return;
    const int mine = OVERFLOW_PASS ? ovf_idx[t0] : t0 + lane;   // lanes below T
    const bool valid = lane < T && t0 + lane < n && (OVERFLOW_PASS || active[mine]);
    double4 a = make_double4(0.0, 0.0, 0.0, 0.0);
    int cloud = -1;
    if (valid) {
        a = rec[mine];
        cloud = cid[mine];
    }
    unsigned long long todo = ballot(valid);
    unsigned vis = 0;
    int mytot = 0;
    while (todo) {   // the particles of one cloud at a time
        const int lead = __ffsll((long long)todo) - 1;
        const int root = __builtin_amdgcn_readlane(cloud, lead);
        const bool in = valid && cloud == root;
        const unsigned long long im = ballot(in);
        todo &= ~im;
        int tot[T];
        double tx[T], ty[T], tz[T], tr[T], th[T];
#pragma unroll
        for (int t = 0; t < T; t++) {
            const int from = (im >> t) & 1ull ? t : lead;   // (others repeat the first)
            tot[t] = 0;
            tx[t] = lane_value(a.x, from);
            ty[t] = lane_value(a.y, from);
            tz[t] = lane_value(a.z, from);
            const double hp = lane_value(a.w, from);
            tr[t] = kg.range * hp;
            th[t] = kg.rangesqd * hp * hp;
        }
        int resume = root;
        do {
            // the particles (bit t) whose cell test passes a node
            auto test = [&](const BNode &nd) -> unsigned {
                unsigned pass = 0;
#pragma unroll
                for (int t = 0; t < T; t++) {
                    const double dx = nd.r[0] - tx[t], dy = nd.r[1] - ty[t], dz = nd.r[2] - tz[t];
                    bool ok;
                    if (BOX) {
                        const double ex = fmax(fabs(dx) - (double)nd.half[0], 0.0);
                        const double ey = fmax(fabs(dy) - (double)nd.half[1], 0.0);
                        const double ez = fmax(fabs(dz) - (double)nd.half[2], 0.0);
                        const double Rb = fmax(tr[t], nd.hrangemax);
                        ok = ex * ex + ey * ey + ez * ez <= Rb * Rb * (1.0 + 1.0e-12);
                    } else {
                        const double dsq = dx * dx + dy * dy + dz * dz;
                        ok = dsq <= (tr[t] + nd.rmax) * (tr[t] + nd.rmax) ||
                             dsq <= (nd.hrangemax + nd.rmax) * (nd.hrangemax + nd.rmax);
                    }
                    pass |= ok ? 1u << t : 0u;
                }
                return pass;
            };
            const int m =
                wave_leaves<MASKED>(L, masks, (unsigned)im, bn, root, resume, vis, test);
            wave_candidates(L, m, rec, 0, [&](int j, const double4 &aj, bool ok, int e) {
                const unsigned own = MASKED && ok ? masks[e] : ~0u;
                const double hrangesqd_pp = kg.rangesqd * aj.w * aj.w;
#pragma unroll
                for (int t = 0; t < T; t++) {
                    if (!((im >> t) & 1ull)) continue;
                    const int p = OVERFLOW_PASS ? mine : t0 + t;
                    const double qx = aj.x - tx[t], qy = aj.y - ty[t], qz = aj.z - tz[t];
                    const double dsq = qx * qx + qy * qy + qz * qz;
                    const bool hit = ok && ((own >> t) & 1u) && j != p &&
                                     (dsq <= th[t] || dsq <= hrangesqd_pp);
                    const unsigned long long hm = ballot(hit);
                    if (hm == 0) continue;
                    const int o = tot[t] + __popcll(hm & ((1ull << lane) - 1ull));
                    if (hit) {
                        if (OVERFLOW_PASS) {
                            if (o < pptot[p]) ovf_list[ovf_off[p] + o] = j;
                        } else if (o < pp_limit) {
                            pplist[(size_t)p * pp_limit + o] = j;
                        }
                    }
                    tot[t] += __popcll(hm);
                }
                return false;
            });
        } while (resume >= 0);
#pragma unroll
        for (int t = 0; t < T; t++)
            if (lane == t && in) mytot = tot[t];
    }
    if (!OVERFLOW_PASS) {
        if (valid) {
            pptot[mine] = mytot;
            if (mytot > pp_limit) atomicAdd(ovf_count, 1);
        }
        wave_stats(wstat, 8, (vis + WAVE - 1) / WAVE, vis);
    } else if (valid && mytot < pptot[mine]) {
        pptot[mine] = mytot;   // a row's readers go as far as it was written
    }
}

// The same rows by one walk per wave of 64 particles, for large clouds with
// fresh boxes: it visits a cell's children when the box test at any lane's
// larger radius passes the cell, and a lane takes the candidates of the
// leaves its own test passes.  Slower alone in small clouds (275 against 40 us at
// 2,048 particles) and equal at 300,007, but 5.7e8 instead of 7.2e8 VALU
// instructions at 1M, where the walk's pair phase beside it wants the same
// units: 3.9 against 4.8 ms there, so clouds above NEIB_WAVE_MAX particles take it.
constexpr int NEIB_WAVE_MAX = 1 << 18;

__global__ void __launch_bounds__(256) k_neib_group(KGeom kg, int n, int nc,
                                                    const HNode *__restrict__ hn,
                                                    const double4 *__restrict__ rec,
                                                    const int *__restrict__ cid,
                                                    const int2 *__restrict__ root_range,
                                                    const uint8_t *__restrict__ active,
                                                    int pp_limit, int *__restrict__ pptot,
                                                    int *__restrict__ pplist,
                                                    int *__restrict__ ovf_count,
                                                    unsigned long long *__restrict__ wstat) {
    const int p = xcd_block() * blockDim.x + threadIdx.x;
    const bool valid = p < n && active[p];
    if (ballot(valid) == 0) return;
    double rpx = 0, rpy = 0, rpz = 0, hp = 0;
    if (valid) {
        const double4 a = rec[p];
        rpx = a.x; rpy = a.y; rpz = a.z;
        hp = a.w;
    }
    const double hrangesqd_p = kg.rangesqd * hp * hp;
    const double R = kg.range * hp;
    int tot = 0;
    int *row = pplist + (size_t)(valid ? p : 0) * pp_limit;
    const int2 rr = valid ? root_range[cid[p]] : make_int2(nc, nc);
    int c = uniform(wave_min_int(rr.x));
    const int cend = uniform(wave_max_int(valid ? rr.y : 0));
    unsigned vis = 0, lvis = 0;
    while (c < cend) {
        const HNode nd = hn[c];
        vis++;
        const double Rb = fmax(R, nd.hrangemax);
        const bool pass = valid && c >= rr.x && c < rr.y &&
                          box_dist2(nd, nd.r[0] - rpx, nd.r[1] - rpy, nd.r[2] - rpz) <=
                              Rb * Rb * (1.0 + 1.0e-12);
        lvis += lanes(pass);
        if (ballot(pass) == 0) {
            c = nd.next;
            continue;
        }
        if (nd.leaf == 0) {
            c = c + 1;
            continue;
        }
        const int k = nd.leaf, f0 = nd.first;
        for (int i = 0; i < k; i++) {
            const int j = f0 + i;
            const double4 aj = rec[j];   // one scalar load per candidate
            if (!pass || j == p) continue;
            const double hrangesqd_pp = kg.rangesqd * aj.w * aj.w;
            const double qx = aj.x - rpx, qy = aj.y - rpy, qz = aj.z - rpz;
            const double dsq = qx * qx + qy * qy + qz * qz;
            if (dsq <= hrangesqd_p || dsq <= hrangesqd_pp) {
                if (tot < pp_limit) row[tot] = j;
                tot++;
            }
        }
        c = nd.next;
    }
    if (valid) {
        pptot[p] = tot;
        if (tot > pp_limit) atomicAdd(ovf_count, 1);
    }
    wave_stats(wstat, 8, vis, lvis);
}

__global__ void k_ovf_sizes(int n, int pp_limit, const int *__restrict__ pptot,
                            const uint8_t *__restrict__ active, int *__restrict__ sz,
                            int *__restrict__ is_ovf) {
    int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    const bool o = active[i] && pptot[i] > pp_limit;
    sz[i] = o ? pptot[i] : 0;
    is_ovf[i] = o ? 1 : 0;
}

// overflow particles in tree order: ovf_idx[pos[i]] = i
__global__ void k_ovf_compact(int n, const int *__restrict__ is_ovf, const int *__restrict__ pos,
                              int *__restrict__ ovf_idx) {
    int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n && is_ovf[i]) ovf_idx[pos[i]] = i;
}

// thermal.F90:52-60 with the sound speed given: P = cs^2 rho, c = cs
__global__ void k_thermal_iso(int n, double cs, const uint8_t *__restrict__ active,
                              const double *__restrict__ rho, double *__restrict__ press,
                              double *__restrict__ sound) {
    int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n || !active[i]) return;
    press[i] = cs * cs * rho[i];
    sound[i] = cs;
}

// Per-particle record of everything a hydro pair reads from the neighbour,
// 128 bytes (one cache line) per particle, so that each neighbour costs one
// line instead of one line per field.  The per-particle factors are formed
// with the reference's operations (hydro_gradh.F90:90-96, :178, :195-196),
// so the pair terms use the same values bit for bit:
//   [0] x y z h   [1] vx vy vz m   [2] rho pfactor sound invh   [3] hfactor
__global__ void k_pack_hydro(int n, const double *__restrict__ x, const double *__restrict__ y,
                             const double *__restrict__ z, const double *__restrict__ h,
                             const double *__restrict__ vx, const double *__restrict__ vy,
                             const double *__restrict__ vz, const double *__restrict__ m,
                             const double *__restrict__ rho, const double *__restrict__ omega,
                             const double *__restrict__ press, const double *__restrict__ sound,
                             double4 *__restrict__ rec) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    const double hi = h[i], rh = rho[i];
    const double invh = 1.0 / hi;
    const double pf = press[i] / rh / rh / omega[i];
    double4 *r = rec + 4 * (size_t)i;
    r[0] = make_double4(x[i], y[i], z[i], hi);
    r[1] = make_double4(vx[i], vy[i], vz[i], m[i]);
    r[2] = make_double4(rh, pf, sound[i], invh);
    r[3] = make_double4(cr_pow4(invh), 0.0, 0.0, 0.0);
}

// hydro_gradh.F90:87-297 (AB viscosity, beta := 2 alpha).  ENERGY: the
// INTERNAL_ENERGY terms, du/dt = sum 0.5 m_j visc W_mean (dv.dr) / |dr|
// (:258-259) - P div v / (Omega rho) (:326-332)
//
// HYD_LPP lanes take a particle, each every HYD_LPP-th neighbour.  The factors
// of eight neighbours' terms then go through LDS to the lanes that add them in
// list order, one lane per sum (three of the pressure force, three of the
// viscous one, du/dt), so the sums are those of one lane bit for bit.
//
// One lane per particle went through its row in a chain of gather, square root
// and divisions, and the longest row held the launch: 115 -> 40 us at 2,048 particles,
// 650 -> 95 us on a Plummer sphere of 2,053 (rows of thousands), 569 -> 337 us on
// an r^-2 sphere of 300,007, where eight gathers of a particle in flight hide
// the L2 misses that bound it.
constexpr int HYD_LPP = 8;

// per wave [f_p, f_pp, f_visc, e1, e2, ux, uy, uz][lane], one column of
// padding: the eight lanes of a particle read one lane's entries
using HydXch = double[8][WAVE + 1];

// The calling lane's sum with eight neighbours' terms f u added in their
// order: f_p u and f_pp u (lanes 0-2, the components of the pressure force),
// f_visc u (lanes 3-5), e1 and e2 (lane 6, du/dt).  A neighbour without a
// term has zeros: they leave the sum (never -0) as it is.
__device__ __forceinline__ double hyd_add(HydXch &x, int lane, int sub, double acc, double f1,
                                          double f2, double f3, double e1, double e2, double ux,
                                          double uy, double uz) {
    x[0][lane] = f1;
    x[1][lane] = f2;
    x[2][lane] = f3;
    x[3][lane] = e1;
    x[4][lane] = e2;
    x[5][lane] = ux;
    x[6][lane] = uy;
    x[7][lane] = uz;
    wave_lds_fence();
    const int l0 = lane & ~(HYD_LPP - 1);
    const int ra = sub < 3 ? 0 : sub < 6 ? 2 : 3, rb = sub < 3 ? 1 : 4,
              ru = 5 + (sub < 3 ? sub : sub < 6 ? sub - 3 : 0);
    double fa[HYD_LPP], fb[HYD_LPP], fu[HYD_LPP];
#pragma unroll
    for (int k = 0; k < HYD_LPP; k++) {
        fa[k] = x[ra][l0 + k];
        fb[k] = x[rb][l0 + k];
        fu[k] = x[ru][l0 + k];
    }
    wave_lds_fence();
#pragma unroll
    for (int k = 0; k < HYD_LPP; k++) {
        const double u = sub < 6 ? fu[k] : 1.0;
        acc = acc + fa[k] * u;
        acc = acc + (sub >= 3 && sub < 6 ? 0.0 : fb[k] * u);
    }
    return acc;
}

template <bool ENERGY>
__global__ void __launch_bounds__(256) k_hydro(
    KGeom kg, int n, const double4 *__restrict__ rec, const uint8_t *__restrict__ active,
    const int *__restrict__ pptot, const int *__restrict__ pplist, const int *__restrict__ ovf_off,
    const int *__restrict__ ovf_list, int pp_limit, const double *__restrict__ ktab, double alpha,
    double *__restrict__ ax, double *__restrict__ ay, double *__restrict__ az,
    const double *__restrict__ press, const double *__restrict__ divv,
    const double *__restrict__ omega, double *__restrict__ dudt) {
    __shared__ HydXch xch_all[256 / WAVE];
    HydXch &xch = xch_all[threadIdx.x / WAVE];
    const int t = xcd_block() * blockDim.x + threadIdx.x, sub = t % HYD_LPP;
    const int lane = (int)(threadIdx.x & (WAVE - 1));
    const bool valid = t / HYD_LPP < n && active[t / HYD_LPP];
    if (ballot(valid) == 0) return;
    const int p = valid ? t / HYD_LPP : 0;   // (lanes without a particle: an empty row)
    const double *w1 = ktab + T_W1 * KT;
    const double4 *rp = rec + 4 * (size_t)p;
    const double4 r0 = rp[0], r1 = rp[1], r2 = rp[2], r3 = rp[3];
    const double rpx = r0.x, rpy = r0.y, rpz = r0.z, hp = r0.w;
    const double vpx = r1.x, vpy = r1.y, vpz = r1.z;
    const double rho_p = r2.x, pfactor_p = r2.y, sound_p = r2.z, invhp = r2.w;
    const double hfactor_p = r3.x;
    const double beta = 2.0 * alpha;
    double acc = 0.0;
    const int nn = valid ? pptot[p] : 0;
    const int *lst = (nn <= pp_limit) ? pplist + (size_t)p * pp_limit : ovf_list + ovf_off[p];
    for (int i0 = 0; any_lane(i0 < nn); i0 += HYD_LPP) {
        double f1 = 0.0, f2 = 0.0, f3 = 0.0, e1 = 0.0, ux = 0.0, uy = 0.0, uz = 0.0;
        if (i0 + sub < nn) {
            const double4 *rq = rec + 4 * (size_t)lst[i0 + sub];
            const double4 q0 = rq[0], q1 = rq[1], q2 = rq[2];
            const double hpp = q0.w, mpp = q1.w, rho_pp = q2.x;
            const double dx = q0.x - rpx, dy = q0.y - rpy, dz = q0.z - rpz;
            const double drsqd = dx * dx + dy * dy + dz * dz;
            if (!(drsqd >= kg.rangesqd * hp * hp) || !(drsqd >= kg.rangesqd * hpp * hpp)) {
                const double drmag = sqrt(drsqd) + SMALL_NUMBER;
                const double dvx = q1.x - vpx, dvy = q1.y - vpy, dvz = q1.z - vpz;
                const double dvdr = dvx * dx + dvy * dy + dvz * dz;
                const double invdrmag = 1.0 / drmag;
                double wmean = 0.0;
                ux = dx * invdrmag;
                uy = dy * invdrmag;
                uz = dz * invdrmag;
                if (drmag < kg.range * hp) {
                    const int kern = min((int)(kg.half * drmag * invhp), KERNTOT);
                    const double wk = w1[kern];
                    wmean = 0.5 * hfactor_p * wk;
                    f1 = mpp * pfactor_p * hfactor_p * wk;
                }
                if (drmag < kg.range * hpp) {
                    const double invhpp = q2.w, hfactor_pp = rq[3].x, pfactor_pp = q2.y;
                    const int kern = min((int)(kg.half * drmag * invhpp), KERNTOT);
                    const double wk = w1[kern];
                    wmean = wmean + 0.5 * hfactor_pp * wk;
                    f2 = mpp * pfactor_pp * hfactor_pp * wk;
                }
                if (dvdr < 0.0) {
                    const double rhomean = 0.5 * (rho_p + rho_pp);
                    const double vsignal = 0.5 * (sound_p + q2.z);
                    const double mu = 0.5 * (hp + hpp) * dvdr /
                                      (drmag * drmag + 0.25 * ETA_SQD * (hp + hpp) * (hp + hpp));
                    const double visc = (-alpha * vsignal * mu + beta * mu * mu) / rhomean;
                    f3 = mpp * visc * wmean;
                    if (ENERGY) e1 = 0.5 * mpp * visc * wmean * dvdr * invdrmag;
                }
            }
        }
        acc = hyd_add(xch, lane, sub, acc, f1, f2, f3, e1, 0.0, ux, uy, uz);
    }
    // the pressure force's lane takes the viscous one's sum; lane 6 has du/dt
    const double ad = __shfl(acc, lane + 3, WAVE), du = __shfl(acc, lane + 6, WAVE);
    if (!valid || sub > 2) return;
    (sub == 0 ? ax : sub == 1 ? ay : az)[p] = acc + ad;
    if (ENERGY && sub == 0)
        dudt[p] = (0.0 + du) - press[p] * divv[p] / omega[p] / rho_p;
}

// Mixed-precision hydro record, 64 bytes per particle: the position in FP64
// (the offsets are formed in FP64, then rounded), everything else in FP32,
// with the per-particle factors of k_pack_hydro formed in FP64 first.
struct __attribute__((aligned(64))) HydroRecF {
    double x, y, z;
    float h, vx, vy, vz, m, rho, pf, sound, invh, hfac;
};
static_assert(sizeof(HydroRecF) == 64, "HydroRecF layout");

__global__ void k_pack_hydro_mixed(int n, const double *__restrict__ x,
                                   const double *__restrict__ y, const double *__restrict__ z,
                                   const double *__restrict__ h, const double *__restrict__ vx,
                                   const double *__restrict__ vy, const double *__restrict__ vz,
                                   const double *__restrict__ m, const double *__restrict__ rho,
                                   const double *__restrict__ omega,
                                   const double *__restrict__ press,
                                   const double *__restrict__ sound,
                                   HydroRecF *__restrict__ rec) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    const double hi = h[i], rh = rho[i];
    const double invh = 1.0 / hi;
    HydroRecF r;
    r.x = x[i];
    r.y = y[i];
    r.z = z[i];
    r.h = (float)hi;
    r.vx = (float)vx[i];
    r.vy = (float)vy[i];
    r.vz = (float)vz[i];
    r.m = (float)m[i];
    r.rho = (float)rh;
    r.pf = (float)(press[i] / rh / rh / omega[i]);
    r.sound = (float)sound[i];
    r.invh = (float)invh;
    r.hfac = (float)cr_pow4(invh);
    rec[i] = r;
}

// hydro_gradh.F90:87-297 as k_hydro computes it, in FP32 on the
// FP64-formed offsets (mixed precision): half the record bytes of the FP64
// kernel, whose neighbour gathers miss L2 and bound it.  |r| and 1/|r| come
// from one reciprocal square root, the divisions from reciprocals; the
// accelerations are summed in FP32 over the particle's neighbours (tens of
// terms) and stored in FP64.  ENERGY: du/dt as k_hydro, the P div v term in
// FP64.
//
// HYD_LPP lanes take a particle, each every HYD_LPP-th neighbour.  The factors
// of eight neighbours' terms then go through LDS to the lanes that add them in
// list order, one lane per sum (three of the pressure force, three of the
// viscous one, du/dt), so the FP32 sums are those of one lane; every
// multiply-add is written out for the same reason.  r^-2 spheres: 120 -> 30 us
// at 16,384 particles, 1,408 -> 686 us at 1M (10 M record gathers of 64 B).
template <bool ENERGY>
__global__ void __launch_bounds__(256) k_hydro_mixed(
    KGeom kg, int n, const HydroRecF *__restrict__ rec, const uint8_t *__restrict__ active,
    const int *__restrict__ pptot, const int *__restrict__ pplist, const int *__restrict__ ovf_off,
    const int *__restrict__ ovf_list, int pp_limit, const float *__restrict__ w1, float alpha,
    double *__restrict__ ax, double *__restrict__ ay, double *__restrict__ az,
    const double *__restrict__ press, const double *__restrict__ divv,
    const double *__restrict__ omega, const double *__restrict__ rho,
    double *__restrict__ dudt) {
#pragma clang fp contract(off)
    static_assert(HYD_LPP == 8, "eight lanes, seven sums");
    // per wave [f_p, f_pp, f_visc, e, ux, uy, uz, 1/|r|][lane], one column of
    // padding: the eight lanes of a particle read one lane's entries
    __shared__ float xch_all[256 / WAVE][8][WAVE + 1];
    float(*xch)[WAVE + 1] = xch_all[threadIdx.x / WAVE];
    const int t = xcd_block() * blockDim.x + threadIdx.x, p = t / HYD_LPP, sub = t % HYD_LPP;
    const int lane = (int)(threadIdx.x & (WAVE - 1));
    const bool valid = p < n && active[p];
    if (ballot(valid) == 0) return;
    HydroRecF s{};
    int nn = 0;
    const int *lst = nullptr;
    if (valid) {
        s = rec[p];
        nn = pptot[p];
        lst = (nn <= pp_limit) ? pplist + (size_t)p * pp_limit : ovf_list + ovf_off[p];
    }
    const double rpx = s.x, rpy = s.y, rpz = s.z;
    const float hp = s.h;
    const float rangesqd = (float)kg.rangesqd, range = (float)kg.range, half = (float)kg.half;
    const float beta = alpha + alpha;
    const float lim_p = hp * (hp * rangesqd), rng_p = hp * range;
    // this lane's sum: its factors' rows
    const int arow = sub < 3 ? 0 : sub < 6 ? 2 : 3;
    const int urow = sub < 3 ? 4 + sub : sub < 6 ? 1 + sub : 7;
    float acc = 0.0f;
    for (int i0 = 0; any_lane(i0 < nn); i0 += HYD_LPP) {
        float f1 = 0.0f, f2 = 0.0f, f3 = 0.0f, e = 0.0f, ux = 0.0f, uy = 0.0f, uz = 0.0f,
              ir = 0.0f;
        if (i0 + sub < nn) {
            const HydroRecF q = rec[lst[i0 + sub]];
            const float hpp = q.h, mpp = q.m;
            const float ex = (float)(q.x - rpx), ey = (float)(q.y - rpy), ez = (float)(q.z - rpz);
            const float dr2 = __builtin_fmaf(ez, ez, __builtin_fmaf(ex, ex, ey * ey));
            if (!(dr2 >= lim_p) || !(dr2 >= hpp * (hpp * rangesqd))) {
                ir = __builtin_amdgcn_rsqf(dr2 + 1.0e-30f);
                const float drmag = dr2 * ir;
                const float dvx = q.vx - s.vx, dvy = q.vy - s.vy, dvz = q.vz - s.vz;
                const float dvdr = __builtin_fmaf(dvz, ez, __builtin_fmaf(dvx, ex, dvy * ey));
                ux = ir * ex;
                uy = ir * ey;
                uz = ir * ez;
                float wmean = 0.0f;
                if (drmag < rng_p) {
                    const float wk = w1[min((int)(s.invh * (drmag * half)), KERNTOT)];
                    wmean = (0.5f * s.hfac) * wk;
                    f1 = (s.hfac * (s.pf * mpp)) * wk;
                }
                if (drmag < hpp * range) {
                    const float wk = w1[min((int)((drmag * half) * q.invh), KERNTOT)];
                    wmean = __builtin_fmaf(0.5f * q.hfac, wk, wmean);
                    f2 = ((mpp * q.pf) * q.hfac) * wk;
                }
                if (dvdr < 0.0f) {
                    const float hs = hp + hpp;
                    const float vsignal = 0.5f * (s.sound + q.sound);
                    const float den =
                        __builtin_fmaf(hs, hs * (0.25f * (float)ETA_SQD), drmag * drmag);
                    const float mu = ((0.5f * hs) * dvdr) * __builtin_amdgcn_rcpf(den);
                    const float visc =
                        __builtin_amdgcn_rcpf(0.5f * (s.rho + q.rho)) *
                        __builtin_fmaf(mu, beta * mu, -((alpha * vsignal) * mu));
                    f3 = (mpp * visc) * wmean;
                    if (ENERGY) e = dvdr * (((0.5f * mpp) * visc) * wmean);
                }
            }
        }
        xch[0][lane] = f1;
        xch[1][lane] = f2;
        xch[2][lane] = f3;
        if (ENERGY) xch[3][lane] = e;
        xch[4][lane] = ux;
        xch[5][lane] = uy;
        xch[6][lane] = uz;
        if (ENERGY) xch[7][lane] = ir;
        wave_lds_fence();
        // a neighbour without a term adds 0 u, which leaves the sum (never -0)
        // as it is
        const int l0 = lane & ~(HYD_LPP - 1);
        float fa[HYD_LPP], fb[HYD_LPP], fu[HYD_LPP];
#pragma unroll
        for (int k = 0; k < HYD_LPP; k++) {
            fa[k] = xch[arow][l0 + k];
            fb[k] = xch[1][l0 + k];
            fu[k] = xch[urow][l0 + k];
        }
        wave_lds_fence();
#pragma unroll
        for (int k = 0; k < HYD_LPP; k++) {
            acc = __builtin_fmaf(fu[k], fa[k], acc);
            acc = __builtin_fmaf(fu[k], sub < 3 ? fb[k] : 0.0f, acc);
        }
    }
    // the pressure force's lane takes the viscous one's sum; lane 6 has du/dt
    const float ad = __shfl(acc, lane + 3, WAVE), du = __shfl(acc, lane + 6, WAVE);
    if (!valid || sub > 2) return;
    (sub == 0 ? ax : sub == 1 ? ay : az)[p] = (double)(ad + acc);
    if (ENERGY && sub == 0)
        dudt[p] = (0.0 + (double)du) - press[p] * divv[p] / omega[p] / rho[p];
}

// thermal.F90:108-113 (INTERNAL_ENERGY, ideal gas): P = (gamma - 1) rho u,
// c = sqrt(P / rho), for every particle: update_thermal_properties.F90:76-81
// loops over all particles once any is active (its active-list loop is
// commented out), so inactive particles take P and c from their advanced u.
// The temperature is not used on the force path.
__global__ void k_thermal_energy(int n, double gamma, const double *__restrict__ rho,
                                 const double *__restrict__ u, double *__restrict__ press,
                                 double *__restrict__ sound) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    const double rho_p = rho[i];
    const double press_p = (gamma - 1.0) * rho_p * u[i];
    press[i] = press_p;
    sound[i] = sqrt(press_p / rho_p);
}

// ---- standard SPH (SPH=STANDARD, HFIND=NUMBER) ---------------------------
//
// h_gather.F90:13-203 for every active particle.  The reference brackets h
// between h_low and h_high = HMULT h_low until pp_low < pp_gather <= pp_tot
// (the counts of other particles with r^2 below KERNRANGESQD h_low^2 and
// h_high^2), sorts the r^2 of the band between them and takes element
// pp_gather - pp_low: h = INVKERNRANGE sqrt(r^2 of the pp_gather-th nearest
// other particle), which does not depend on the path the bracketing took.
// Here each lane brackets the same way over its own potential-neighbour leaf
// list (recorded by a group walk at radius KERNRANGE h_search whenever h_high
// outgrows h_search, as the reference re-walks), narrows a band of more than
// BAND_MAX values by bisection in r^2, copies the band to its slice of the
// band buffer and sorts it there.  r^2 is formed as distance2.F90 forms it,
// so h is the reference's bit for bit.  A lane that cannot bracket within
// HG_ITER_MAX passes (fewer than pp_gather other particles) sets *err.
constexpr int HG_ITER_MAX = 400;

__global__ void __launch_bounds__(256) k_hgather(
    KGeom kg, bool box, int n, int nc, const HNode *__restrict__ hn, const double4 *__restrict__ rec,
    const int *__restrict__ cid, const int2 *__restrict__ root_range, int *__restrict__ hlist,
    int hl_cap, double *__restrict__ band, const uint8_t *__restrict__ active, int pp_gather,
    double *__restrict__ h, int *__restrict__ err, unsigned long long *__restrict__ wstat) {
    const int p = xcd_block() * blockDim.x + threadIdx.x;
    const bool valid = p < n && active[p];
    const int lane = threadIdx.x & (WAVE - 1);
    int *wl = hlist + (size_t)(p / WAVE) * (HL_SLOTS * WAVE) + lane;
    double *bl = band + (size_t)(p / WAVE) * (BAND_MAX * WAVE) + lane;
    double rpx = 0, rpy = 0, rpz = 0, h_old = 1.0;
    int2 rr = make_int2(nc, nc);
    if (valid) {
        const double4 a = rec[p];
        rpx = a.x; rpy = a.y; rpz = a.z;
        h_old = h[p];
        rr = root_range[cid[p]];
    }
    double h_high = HMULT * h_old, h_low = h_old / HMULT, h_search = 0.0;
    bool iterating = valid;
    int nslot = 0, cnt = 0, pp_low = 0, pp_tot = 0, passes = 0;
    bool my_ovf = false, wave_ovf = false, have_list = false, failed = false;
    unsigned vis = 0, lvis = 0, walked = 0;   // walked: passes over the tree walk
    auto dist2 = [&](const double4 &a) {   // distance2.F90, no contraction
        const double dx = a.x - rpx, dy = a.y - rpy, dz = a.z - rpz;
        return dx * dx + dy * dy + dz * dz;
    };
    // one pass over the lane's candidates: f(j, r^2) for each other particle
    auto for_each = [&](bool on, auto &&f) {
        if (!wave_ovf) {
            list_loop(wl, nslot, on, p, [&](int j) { return rec[j]; },
                      [&](int j, const double4 &a) { f(j, dist2(a)); });
        } else {
            const double R = kg.range * h_search;
            walked++;
            vis += group_walk(hn, nc, on, rr.x, rr.y, lvis,
                              [&](const HNode &nd, bool) {
                                  return hgather_visit(nd, rpx, rpy, rpz, R);
                              },
                              [&](const HNode &nd, bool mine) {
                const bool use = mine && leaf_near(nd, rpx, rpy, rpz, R, box);
                for (int i = 0; i < nd.leaf; i++) {
                    const int j = nd.first + i;
                    const double4 a = rec[j];
                    if (use && j != p) f(j, dist2(a));
                }
            });
        }
    };

    // bracketing (h_gather.F90:57-175)
    while (any_lane(iterating)) {
        passes++;
        bool newlist = false;
        if (iterating && h_high > h_search) {
            h_search = HMULT * h_high;
            newlist = true;
        }
        if (!have_list || any_lane(newlist)) {
            if (iterating) {
                nslot = 0;
                cnt = 0;
            }
            bool lovf = false;
            const double R = kg.range * h_search;
            vis += group_walk(hn, nc, iterating, rr.x, rr.y, lvis,
                              [&](const HNode &nd, bool) {
                                  return hgather_visit(nd, rpx, rpy, rpz, R);
                              },
                              [&](const HNode &nd, bool mine) {
                if (mine) {
                    cnt += nd.leaf;                       // the reference's pp_pot
                    if (leaf_near(nd, rpx, rpy, rpz, R, box)) {
                        if (nslot < hl_cap)
                            wl[nslot * WAVE] = (nd.first << 4) | nd.leaf;
                        else
                            lovf = true;
                        nslot++;
                    }
                }
            });
            if (iterating) my_ovf = lovf;
            have_list = true;
            wave_ovf = any_lane(my_ovf);   // lanes that stopped keep their lists
        }
        // too few potential neighbours: grow and walk again (:93-99)
        const bool grow = iterating && newlist && cnt <= pp_gather;
        const bool count = iterating && !grow;
        const double hr2_high = kg.rangesqd * h_high * h_high;
        const double hr2_low = kg.rangesqd * h_low * h_low;
        int lo = 0, tot = 0;
        for_each(count, [&](int, double r2) {
            if (r2 < hr2_high) {
                tot++;
                if (r2 < hr2_low) lo++;
            }
        });
        if (grow) {
            h_search = 0.0;
            h_low = h_high;
            h_high = HMULT * h_high;
        } else if (count) {
            pp_low = lo;
            pp_tot = tot;
            if (tot < pp_gather) {                    // :143-147
                h_low = h_high;
                h_high = HMULT * h_high;
            } else if (lo >= pp_gather) {             // :150-153
                h_high = h_low;
                h_low = h_low / HMULT;
            } else {                                  // :156-158
                iterating = false;
            }
        }
        if (iterating && passes >= HG_ITER_MAX) {
            iterating = false;
            failed = true;
        }
    }

    // band [lo2, hi2) of r^2 with count(r^2 < lo2) = pp_low < pp_gather <=
    // count(r^2 < hi2) = pp_tot; narrow it to BAND_MAX values at most
    double lo2 = kg.rangesqd * h_low * h_low, hi2 = kg.rangesqd * h_high * h_high;
    bool narrowing = valid && !failed && pp_tot - pp_low > BAND_MAX;
    // tie: the band [lo2, hi2) holds one double only (lo2 and hi2 adjacent),
    // so every band value is lo2 -- more than BAND_MAX particles at exactly
    // that r^2, as in a lattice shell -- and the pp_gather-th is lo2 itself
    bool tie = false;
    int nb = 0;
    while (any_lane(narrowing)) {
        const double mid = 0.5 * (lo2 + hi2);
        const bool split = mid > lo2 && mid < hi2;
        int c = 0;
        for_each(narrowing && split, [&](int, double r2) {
            if (r2 < mid) c++;
        });
        if (narrowing && !split) {
            narrowing = false;
            tie = true;
        } else if (narrowing) {
            if (c >= pp_gather) {
                hi2 = mid;
                pp_tot = c;
            } else {
                lo2 = mid;
                pp_low = c;
            }
            if (pp_tot - pp_low <= BAND_MAX) narrowing = false;
            if (++nb >= HG_ITER_MAX) {
                narrowing = false;
                failed = true;
            }
        }
    }
    // copy the band and sort it (insertion_sort.F90:4-30)
    if (tie) h[p] = kg.invrange * sqrt(lo2);
    const bool fill = valid && !failed && !tie;
    int m = 0;
    for_each(fill, [&](int, double r2) {
        if (r2 < hi2 && !(r2 < lo2) && m < BAND_MAX) {
            bl[m * WAVE] = r2;
            m++;
        }
    });
    if (fill) {
        for (int j = 1; j < m; j++) {
            const double raux = bl[j * WAVE];
            int i = j - 1;
            for (; i >= 0; i--) {
                const double ri = bl[i * WAVE];
                if (ri <= raux) break;
                bl[(i + 1) * WAVE] = ri;
            }
            bl[(i + 1) * WAVE] = raux;
        }
        const int k = pp_gather - pp_low - 1;
        if (k >= 0 && k < m)
            h[p] = kg.invrange * sqrt(bl[k * WAVE]);
        else
            failed = true;
    }
    if (failed) atomicOr(err, 1);
    wave_stats(wstat, 2, vis, lvis);
    if (walked && (threadIdx.x & 63) == 0) atomicAdd(ctr_row(wstat) + 11, (unsigned long long)walked);
}

// all_sph.F90:11-167 (standard SPH) for every active particle: rho, div v
// and drho/dt over the gather neighbours (r < KERNRANGE h_p) of its list, in
// list order.  rec holds [2i] x y z m and [2i+1] vx vy vz 0.
__global__ void __launch_bounds__(256) k_all_sph(
    KGeom kg, int n, const double4 *__restrict__ rec, const uint8_t *__restrict__ active,
    const int *__restrict__ pptot, const int *__restrict__ pplist, const int *__restrict__ ovf_off,
    const int *__restrict__ ovf_list, int pp_limit, const double *__restrict__ ktab,
    const double *__restrict__ h, double *__restrict__ rho, double *__restrict__ divv,
    double *__restrict__ drhodt) {
    const int p = xcd_block() * blockDim.x + threadIdx.x;
    if (p >= n || !active[p]) return;
    const double *w0 = ktab + T_W0 * KT, *w4 = ktab + T_W4 * KT;
    const double4 a = rec[2 * (size_t)p], b = rec[2 * (size_t)p + 1];
    const double rpx = a.x, rpy = a.y, rpz = a.z;
    const double vpx = b.x, vpy = b.y, vpz = b.z;
    const double hp = h[p], invhp = 1.0 / hp, hfactor = cr_pow3(invhp);
    const double range_p = kg.range * hp;
    double rhotemp = a.w * w0[0] * hfactor;
    double div_v_p = 0.0;
    const int nn = pptot[p];
    const int *lst = (nn <= pp_limit) ? pplist + (size_t)p * pp_limit : ovf_list + ovf_off[p];
    for (int i = 0; i < nn; i++) {
        const int j = lst[i];
        const double4 q = rec[2 * (size_t)j], qv = rec[2 * (size_t)j + 1];
        const double dvx = qv.x - vpx, dvy = qv.y - vpy, dvz = qv.z - vpz;
        const double mpp = q.w;
        const double dx = q.x - rpx, dy = q.y - rpy, dz = q.z - rpz;
        const double drsqd = dx * dx + dy * dy + dz * dz;
        const double dvdr = dvx * dx + dvy * dy + dvz * dz;
        const double drmag = sqrt(drsqd) + SMALL_NUMBER;
        if (drmag >= range_p) continue;                        // all_sph.F90:103
        const double invdrmag = 1.0 / drmag;
        const int kern = min((int)(kg.half * drmag * invhp), KERNTOT);
        rhotemp = rhotemp + mpp * hfactor * w0[kern];
        div_v_p = div_v_p - mpp * dvdr * w4[kern] * hfactor * invhp * invdrmag;
    }
    rho[p] = rhotemp;
    div_v_p = div_v_p / rhotemp;
    divv[p] = div_v_p;
    drhodt[p] = -rhotemp * div_v_p;
}

__global__ void k_pack_sph(int n, const double *__restrict__ x, const double *__restrict__ y,
                           const double *__restrict__ z, const double *__restrict__ vx,
                           const double *__restrict__ vy, const double *__restrict__ vz,
                           const double *__restrict__ m, double4 *__restrict__ rec) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    rec[2 * (size_t)i] = make_double4(x[i], y[i], z[i], m[i]);
    rec[2 * (size_t)i + 1] = make_double4(vx[i], vy[i], vz[i], 0.0);
}

// Hydro record of standard SPH (hydro.F90:83-98, :180-188): [0] x y z h
// [1] vx vy vz m  [2] rho pfactor sound invh  [3] hfactor P/(rho rho), with
// pfactor = P / rho / rho, invh = 1 / h and hfactor = invh**3 formed as the
// reference forms them.
__global__ void k_pack_hydro_std(int n, const double *__restrict__ x, const double *__restrict__ y,
                                 const double *__restrict__ z, const double *__restrict__ h,
                                 const double *__restrict__ vx, const double *__restrict__ vy,
                                 const double *__restrict__ vz, const double *__restrict__ m,
                                 const double *__restrict__ rho, const double *__restrict__ press,
                                 const double *__restrict__ sound, double4 *__restrict__ rec) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    double4 *r = rec + 4 * (size_t)i;
    const double hi = h[i], invh = 1.0 / hi, rho_i = rho[i], p_i = press[i];
    r[0] = make_double4(x[i], y[i], z[i], hi);
    r[1] = make_double4(vx[i], vy[i], vz[i], m[i]);
    r[2] = make_double4(rho_i, p_i / rho_i / rho_i, sound[i], invh);
    r[3] = make_double4(cr_pow3(invh), p_i / (rho_i * rho_i), 0.0, 0.0);
}

// hydro.F90:11-323 (standard SPH, AB viscosity): the kernel gradient
// averaged over h_p and h_pp (wmean) weighs both the pressure term
// (P_p/rho_p^2 + P_pp/rho_pp^2) and the viscous term.  ENERGY adds du/dt,
// the same pair terms projected on dv.dr / |dr| (hydro.F90:206-208, :262-264).
// HYD_LPP lanes per particle, as k_hydro.
template <bool ENERGY>
__global__ void __launch_bounds__(256) k_hydro_std(
    KGeom kg, int n, const double4 *__restrict__ rec, const uint8_t *__restrict__ active,
    const int *__restrict__ pptot, const int *__restrict__ pplist, const int *__restrict__ ovf_off,
    const int *__restrict__ ovf_list, int pp_limit, const double *__restrict__ ktab, double alpha,
    double *__restrict__ ax, double *__restrict__ ay, double *__restrict__ az,
    double *__restrict__ dudt_out) {
    __shared__ HydXch xch_all[256 / WAVE];
    HydXch &xch = xch_all[threadIdx.x / WAVE];
    const int t = xcd_block() * blockDim.x + threadIdx.x, sub = t % HYD_LPP;
    const int lane = (int)(threadIdx.x & (WAVE - 1));
    const bool valid = t / HYD_LPP < n && active[t / HYD_LPP];
    if (ballot(valid) == 0) return;
    const int p = valid ? t / HYD_LPP : 0;   // (lanes without a particle: an empty row)
    const double *w1 = ktab + T_W1 * KT;
    const double4 *rp = rec + 4 * (size_t)p;
    const double4 r0 = rp[0], r1 = rp[1], r2 = rp[2], r3 = rp[3];
    const double rpx = r0.x, rpy = r0.y, rpz = r0.z, hp = r0.w;
    const double vpx = r1.x, vpy = r1.y, vpz = r1.z;
    const double rho_p = r2.x, pfactor_p = r2.y, sound_p = r2.z, invhp = r2.w;
    const double hfactor_p = r3.x;
    double acc = 0.0;
    const int nn = valid ? pptot[p] : 0;
    const int *lst = (nn <= pp_limit) ? pplist + (size_t)p * pp_limit : ovf_list + ovf_off[p];
    for (int i0 = 0; any_lane(i0 < nn); i0 += HYD_LPP) {
        double f1 = 0.0, f3 = 0.0, e1 = 0.0, e2 = 0.0, ux = 0.0, uy = 0.0, uz = 0.0;
        if (i0 + sub < nn) {
            const double4 *rq = rec + 4 * (size_t)lst[i0 + sub];
            const double4 q0 = rq[0], q1 = rq[1], q2 = rq[2];
            const double hpp = q0.w, mpp = q1.w, rho_pp = q2.x;
            const double dx = q0.x - rpx, dy = q0.y - rpy, dz = q0.z - rpz;
            const double drsqd = dx * dx + dy * dy + dz * dz;
            if (!(drsqd >= kg.rangesqd * hp * hp) || !(drsqd >= kg.rangesqd * hpp * hpp)) {
                const double drmag = sqrt(drsqd) + SMALL_NUMBER;
                const double invdrmag = 1.0 / drmag;
                ux = dx * invdrmag;
                uy = dy * invdrmag;
                uz = dz * invdrmag;
                const double dvx = q1.x - vpx, dvy = q1.y - vpy, dvz = q1.z - vpz;
                const double dvdr = dvx * dx + dvy * dy + dvz * dz;
                double wmean = 0.0;
                if (drmag < kg.range * hp) {
                    const int kern = min((int)(kg.half * drmag * invhp), KERNTOT);
                    wmean = 0.5 * hfactor_p * invhp * w1[kern];
                }
                if (drmag < kg.range * hpp) {
                    const double invhpp = q2.w, hfactor_pp = rq[3].x;
                    const int kern = min((int)(kg.half * drmag * invhpp), KERNTOT);
                    wmean = wmean + 0.5 * hfactor_pp * invhpp * w1[kern];
                }
                const double pf = pfactor_p + rq[3].y;
                f1 = mpp * wmean * pf;
                if (ENERGY) e1 = 0.5 * mpp * wmean * dvdr * invdrmag * pf;
                if (dvdr < 0.0) {                              // hydro.F90:221-224
                    const double rhomean = 0.5 * (rho_p + rho_pp);
                    const double beta = 2 * alpha;
                    const double vsignal = 0.5 * (sound_p + q2.z);
                    const double mu = 0.5 * (hp + hpp) * dvdr /
                                      (drsqd + 0.25 * ETA_SQD * (hp + hpp) * (hp + hpp));
                    const double visc = (-alpha * vsignal * mu + beta * mu * mu) / rhomean;
                    f3 = mpp * visc * wmean;
                    if (ENERGY) e2 = 0.5 * mpp * visc * wmean * dvdr * invdrmag;
                }
            }
        }
        acc = hyd_add(xch, lane, sub, acc, f1, 0.0, f3, e1, e2, ux, uy, uz);
    }
    const double ad = __shfl(acc, lane + 3, WAVE), du = __shfl(acc, lane + 6, WAVE);
    if (!valid || sub > 2) return;
    (sub == 0 ? ax : sub == 1 ? ay : az)[p] = acc + ad;
    if (ENERGY && sub == 0) dudt_out[p] = du;
}

// sph_update.F90:107-109 (HFIND=CONSTANT): parray(SMOO,1:ptot) = hmin
__global__ void k_fill_h(int n, double hmin, double *__restrict__ h) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) h[i] = hmin;
}

__global__ void k_pow_third(int n, const double *__restrict__ x, double *__restrict__ y) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) y[i] = ref_pow_third(x[i]);
}

}  // namespace

int eval_pow_third(Ctx &c, int n, const double *x, double *y) {
    hipLaunchKernelGGL(k_pow_third, dim3(nblk(n)), dim3(TB), 0, c.stream, n, x, y);
    SX_HIP(hipGetLastError());
    return SERENX_OK;
}

int sph_hsolve(Ctx &c) {
    if (c.n < c.pp_gather)
        return set_error(SERENX_EFEW, "fewer particles than pp_gather: the grad-h solve "
                                      "cannot reach its neighbour number");
    SX_TRY(zero_words(c.flag, 1, c.stream));
    double4 *rec = reinterpret_cast<double4 *>(c.hrec);
    hipLaunchKernelGGL(k_pack_hsolve, dim3(nblk(c.n)), dim3(TB), 0, c.stream, c.n, c.x, c.y, c.z,
                       c.vx, c.vy, c.vz, c.m, rec);
    SX_HIP(hipGetLastError());
    // leaves a particle may list (the tuning knob's slots, when lowered)
    const int list_cap = c.hl_cap < HL_SLOTS ? c.hl_cap : WS_CAP;
    const bool by_waves = c.n <= HSOLVE_WAVE_MAX;
    if (!by_waves) {
        SX_TRY(zero_words(c.hq_len, 1, c.stream));
        // h_high per particle in the permutation scratch, list lengths in tmpi
        // the h solve at 8 waves per SIMD in mixed precision, where it is on the
        // critical path; beside the FP64 walk (issue-bound) at the compiler's 5
        const bool w8 =
            c.hsolve_waves == 8 || (c.hsolve_waves < 0 && c.opt.precision == SERENX_MIXED);
        hipLaunchKernelGGL(w8 ? k_hsolve_iter<8> : k_hsolve_iter<0>, dim3(nblk(c.n)), dim3(TB), 0,
                           c.stream, c.kg, c.box_ok, c.n, c.nc, c.hn, rec, c.cid, c.root_range,
                           c.root, c.hlist, c.hl_cap, c.active, c.ktab, c.opt.h_fac, c.pp_gather,
                           c.h, c.rho, c.tmpd, c.tmpi, c.hq, c.hq_len, c.wstat);
        SX_HIP(hipGetLastError());
        hipLaunchKernelGGL(k_hsolve_final, dim3(nblk(c.n)), dim3(TB), 0, c.stream, c.kg, c.box_ok,
                           c.n, rec, c.hlist, c.active, c.ktab, c.opt.h_fac, c.tmpd, c.tmpi, c.h,
                           c.zeta, c.rho, c.omega, c.divv, c.drhodt, c.hq, c.hq_len, c.flag);
        SX_HIP(hipGetLastError());
    }
    // all particles of a small cloud, or those the lanes left
    const int blocks = std::min(nblk(c.n, 256 / WAVE), 5 * c.ncu);
    hipLaunchKernelGGL(k_hsolve_wave, dim3(blocks), dim3(256), 0, c.stream, c.kg, c.box_ok, c.n,
                       c.bn, rec, c.cid, c.root, c.active, c.ktab, c.opt.h_fac, c.pp_gather,
                       list_cap, by_waves ? nullptr : c.hq, c.hq_len, c.h, c.zeta, c.rho, c.omega,
                       c.divv, c.drhodt, c.flag, c.wstat);
    SX_HIP(hipGetLastError());
    SX_HIP(hipMemcpyAsync(c.hostpin + 8, c.flag, sizeof(int), hipMemcpyDeviceToHost, c.stream));
    return SERENX_OK;
}

int sph_hgather(Ctx &c) {
    if (c.opt.hfind == SERENX_HFIND_CONSTANT) {
        hipLaunchKernelGGL(k_fill_h, dim3(nblk(c.n)), dim3(TB), 0, c.stream, c.n, c.opt.hmin,
                           c.h);
        SX_HIP(hipGetLastError());
        c.hostpin[8] = 0;   // no h solve ran: sph_neighbours reads slot 8 as its error flag
        return SERENX_OK;
    }
    if (c.n <= c.pp_gather)
        return set_error(SERENX_EFEW, "h_gather needs more than pp_gather particles");
    const size_t need = ((size_t)c.cap + TB - 1) / TB * TB;   // whole blocks, as hlist
    if (c.band_cap < need) {
        c.graph_epoch++;
        if (c.band) (void)hipFree(c.band);
        c.band = nullptr;
        c.band_cap = 0;
        if (hipMalloc((void **)&c.band, sizeof(double) * need * BAND_MAX) != hipSuccess)
            return set_error(SERENX_ENOMEM, "hipMalloc failed for the h_gather band buffer");
        c.band_cap = need;
    }
    SX_TRY(zero_words(c.flag, 1, c.stream));
    double4 *rec = reinterpret_cast<double4 *>(c.hrec);
    hipLaunchKernelGGL(k_pack_hsolve, dim3(nblk(c.n)), dim3(TB), 0, c.stream, c.n, c.x, c.y, c.z,
                       c.vx, c.vy, c.vz, c.m, rec);
    hipLaunchKernelGGL(k_hgather, dim3(nblk(c.n)), dim3(TB), 0, c.stream, c.kg, c.box_ok, c.n, c.nc, c.hn,
                       rec, c.cid, c.root_range, c.hlist, c.hl_cap, c.band, c.active,
                       c.pp_gather, c.h,
                       c.flag, c.wstat);
    SX_HIP(hipGetLastError());
    SX_HIP(hipMemcpyAsync(c.hostpin + 8, c.flag, sizeof(int), hipMemcpyDeviceToHost, c.stream));
    SX_HIP(hipStreamSynchronize(c.stream));
    if (c.hostpin[8] != 0)
        return set_error(SERENX_EFEW, "h_gather could not bracket pp_gather neighbours "
                                      "(a cloud with too few particles)");
    c.hostpin[8] = 0;   // sph_neighbours reads it as the h-solve error flag
    return SERENX_OK;
}

int sph_density(Ctx &c) {
    double4 *rec = reinterpret_cast<double4 *>(c.hrec);
    hipLaunchKernelGGL(k_pack_sph, dim3(nblk(c.n)), dim3(TB), 0, c.stream, c.n, c.x, c.y, c.z,
                       c.vx, c.vy, c.vz, c.m, rec);
    hipLaunchKernelGGL(k_all_sph, dim3(nblk(c.n)), dim3(TB), 0, c.stream, c.kg, c.n, rec,
                       c.active, c.pptot, c.pplist, c.ovf_off, c.ovf_list, c.pp_limit, c.ktab,
                       c.h, c.rho, c.divv, c.drhodt);
    SX_HIP(hipGetLastError());
    return SERENX_OK;
}

// The neighbour rows of sph_neighbours, launches only: rows of up to
// pp_limit ids, every particle's count, and the number of particles above
// pp_limit copied to pinned slot 9 (read by sph_neib_finish once the stream
// has got there).
int sph_neib_rows(Ctx &c) {
    hipStream_t s = c.stream;
    double4 *rec = reinterpret_cast<double4 *>(c.hrec);
    // [0] x y z h with the solved h
    hipLaunchKernelGGL(k_pack_xyzh, dim3(nblk(std::max(c.n, c.nc))), dim3(TB), 0, s, c.n, c.x, c.y,
                       c.z, c.h, rec, c.nc, c.bfs2dfs, c.hn, c.neib_group ? c.bn : nullptr);
    SX_TRY(zero_words(c.ovf_count, 1, s));
    if (c.neib_group && c.box_ok && c.n > NEIB_WAVE_MAX) {
        hipLaunchKernelGGL(k_neib_group, dim3(nblk(c.n)), dim3(TB), 0, s, c.kg, c.n, c.nc, c.hn, rec,
                           c.cid, c.root_range, c.active, c.pp_limit, c.pptot, c.pplist,
                           c.ovf_count, c.wstat);
    } else if (c.neib_group) {
        auto k = c.box_ok ? k_neib_wave<false, true> : k_neib_wave<false, false>;
        hipLaunchKernelGGL(k, dim3(nblk((c.n + NW_T - 1) / NW_T, 256 / WAVE)),
                           dim3(256), 0, s, c.kg, c.n, c.ovf_idx, c.bn, rec, c.cid, c.active,
                           c.pp_limit, c.pptot, c.pplist, c.ovf_off, c.ovf_list, c.ovf_count,
                           c.wstat);
    } else {
        hipLaunchKernelGGL(k_neib<false>, dim3(nblk(c.n)), dim3(TB), 0, s, c.kg, c.box_ok, c.n,
                           c.ovf_idx, c.nc, c.hn, rec, c.cid, c.root_range, c.active, c.pp_limit,
                           c.pptot, c.pplist, c.ovf_off, c.ovf_list, c.ovf_count, c.wstat);
    }
    SX_HIP(hipGetLastError());
    SX_HIP(hipMemcpyAsync(c.hostpin + 9, c.ovf_count, sizeof(int), hipMemcpyDeviceToHost, s));
    return SERENX_OK;
}

int sph_neighbours(Ctx &c) {
    SX_TRY(sph_neib_rows(c));
    SX_HIP(hipStreamSynchronize(c.stream));
    return sph_neib_finish(c);
}

// The host part of sph_neighbours, after the stream has run sph_neib_rows:
// the h solve's status (slot 8) and the complete lists of the particles
// above pp_limit (the rows get_neib_on_fly.F90 would walk for).
int sph_neib_finish(Ctx &c) {
    hipStream_t s = c.stream;
    double4 *rec = reinterpret_cast<double4 *>(c.hrec);
    if (c.hostpin[8] != 0)
        return set_error(SERENX_EHNEG, "Negative smoothing lengths (all_sph_gradh)");
    if (c.hostpin[9] > 0) {
        // complete lists for particles above pp_limit, packed by offset
        // sizes (flag) and overflow marks (incl; both tree-build scratch)
        hipLaunchKernelGGL(k_ovf_sizes, dim3(nblk(c.n)), dim3(TB), 0, s, c.n, c.pp_limit, c.pptot,
                           c.active, c.flag, c.incl);
        SX_TRY(zero_words(c.flag + c.n, 1, s));
        size_t tb = c.sorttmp_bytes;
        SX_HIP(rocprim::exclusive_scan(c.sorttmp, tb, c.flag, c.ovf_off, 0, (size_t)c.n + 1,
                                       rocprim::plus<int>(), s));
        tb = c.sorttmp_bytes;
        SX_HIP(rocprim::exclusive_scan(c.sorttmp, tb, c.incl, c.cellof, 0, (size_t)c.n,
                                       rocprim::plus<int>(), s));
        hipLaunchKernelGGL(k_ovf_compact, dim3(nblk(c.n)), dim3(TB), 0, s, c.n, c.incl, c.cellof,
                           c.ovf_idx);
        SX_HIP(hipMemcpyAsync(c.hostpin + 10, c.ovf_off + c.n, sizeof(int),
                              hipMemcpyDeviceToHost, s));
        SX_HIP(hipStreamSynchronize(s));
        const size_t need = (size_t)c.hostpin[10];
        if (need > c.ovf_cap) {
            c.graph_epoch++;   // a captured hydro pass holds the old address
            if (c.ovf_list) (void)hipFree(c.ovf_list);
            c.ovf_list = nullptr;
            c.ovf_cap = need + need / 4 + 1024;
            if (hipMalloc(&c.ovf_list, sizeof(int) * c.ovf_cap) != hipSuccess)
                return set_error(SERENX_ENOMEM, "hipMalloc failed for overflow neighbour lists");
        }
        const int nov = c.hostpin[9];   // overflow particles, counted by k_neib<false>
        if (c.neib_group) {
            auto k = c.box_ok ? k_neib_wave<true, true> : k_neib_wave<true, false>;
            hipLaunchKernelGGL(k, dim3(nblk(nov, 256 / WAVE)), dim3(256), 0, s, c.kg, nov,
                               c.ovf_idx, c.bn, rec, c.cid, c.active, c.pp_limit, c.pptot,
                               c.pplist, c.ovf_off, c.ovf_list, c.ovf_count, c.wstat);
        } else {
            const long threads = (long)((nov + OVF_PER_WAVE - 1) / OVF_PER_WAVE) * WAVE;
            hipLaunchKernelGGL(k_neib<true>, dim3(nblk(threads)), dim3(TB), 0, s, c.kg, c.box_ok,
                               nov, c.ovf_idx, c.nc, c.hn, rec, c.cid, c.root_range, c.active,
                               c.pp_limit, c.pptot, c.pplist, c.ovf_off, c.ovf_list, c.ovf_count,
                               c.wstat);
        }
        SX_HIP(hipGetLastError());
    }
    return SERENX_OK;
}

int sph_thermal(Ctx &c) {
    if (c.opt.thermal == SERENX_THERMAL_ENERGY_EQN) {
        hipLaunchKernelGGL(k_thermal_energy, dim3(nblk(c.n)), dim3(TB), 0, c.stream, c.n,
                           c.opt.gamma, c.rho, c.u, c.press, c.sound);
        SX_HIP(hipGetLastError());
        return SERENX_OK;
    }
    return sph_thermal_iso(c, c.opt.sound_speed);
}

int sph_thermal_iso(Ctx &c, double cs) {
    hipLaunchKernelGGL(k_thermal_iso, dim3(nblk(c.n)), dim3(TB), 0, c.stream, c.n, cs, c.active,
                       c.rho, c.press, c.sound);
    SX_HIP(hipGetLastError());
    return SERENX_OK;
}

int hydro_forces(Ctx &c) {
    double4 *rec = reinterpret_cast<double4 *>(c.hrec);
    if (c.opt.sph == SERENX_SPH_STANDARD) {
        hipLaunchKernelGGL(k_pack_hydro_std, dim3(nblk(c.n)), dim3(TB), 0, c.stream, c.n, c.x,
                           c.y, c.z, c.h, c.vx, c.vy, c.vz, c.m, c.rho, c.press, c.sound, rec);
        if (c.opt.thermal == SERENX_THERMAL_ENERGY_EQN)
            hipLaunchKernelGGL(k_hydro_std<true>, dim3(nblk((long)c.n * HYD_LPP)), dim3(TB), 0, c.stream, c.kg,
                               c.n, rec, c.active, c.pptot, c.pplist, c.ovf_off, c.ovf_list,
                               c.pp_limit, c.ktab, c.opt.alpha, c.ax, c.ay, c.az, c.dudt);
        else
            hipLaunchKernelGGL(k_hydro_std<false>, dim3(nblk((long)c.n * HYD_LPP)), dim3(TB), 0, c.stream, c.kg,
                               c.n, rec, c.active, c.pptot, c.pplist, c.ovf_off, c.ovf_list,
                               c.pp_limit, c.ktab, c.opt.alpha, c.ax, c.ay, c.az, c.dudt);
        SX_HIP(hipGetLastError());
        return SERENX_OK;
    }
    if (c.opt.precision == SERENX_MIXED) {
        // mixed precision: FP32 pair terms on 64-byte records
        HydroRecF *rf = reinterpret_cast<HydroRecF *>(c.hrec);
        const float *w1f = reinterpret_cast<const float *>(c.ktab + KT_F32_OFF) + T_W1 * KT;
        hipLaunchKernelGGL(k_pack_hydro_mixed, dim3(nblk(c.n)), dim3(TB), 0, c.stream, c.n, c.x,
                           c.y, c.z, c.h, c.vx, c.vy, c.vz, c.m, c.rho, c.omega, c.press, c.sound,
                           rf);
        if (c.opt.thermal == SERENX_THERMAL_ENERGY_EQN)
            hipLaunchKernelGGL(k_hydro_mixed<true>, dim3(nblk((long)c.n * HYD_LPP)), dim3(TB), 0, c.stream, c.kg,
                               c.n, rf, c.active, c.pptot, c.pplist, c.ovf_off, c.ovf_list,
                               c.pp_limit, w1f, (float)c.opt.alpha, c.ax, c.ay, c.az, c.press,
                               c.divv, c.omega, c.rho, c.dudt);
        else
            hipLaunchKernelGGL(k_hydro_mixed<false>, dim3(nblk((long)c.n * HYD_LPP)), dim3(TB), 0, c.stream, c.kg,
                               c.n, rf, c.active, c.pptot, c.pplist, c.ovf_off, c.ovf_list,
                               c.pp_limit, w1f, (float)c.opt.alpha, c.ax, c.ay, c.az, c.press,
                               c.divv, c.omega, c.rho, c.dudt);
        SX_HIP(hipGetLastError());
        return SERENX_OK;
    }
    hipLaunchKernelGGL(k_pack_hydro, dim3(nblk(c.n)), dim3(TB), 0, c.stream, c.n, c.x, c.y, c.z,
                       c.h, c.vx, c.vy, c.vz, c.m, c.rho, c.omega, c.press, c.sound, rec);
    SX_HIP(hipGetLastError());
    if (c.opt.thermal == SERENX_THERMAL_ENERGY_EQN)
        hipLaunchKernelGGL(k_hydro<true>, dim3(nblk((long)c.n * HYD_LPP)), dim3(TB), 0, c.stream, c.kg, c.n, rec,
                           c.active, c.pptot, c.pplist, c.ovf_off, c.ovf_list, c.pp_limit, c.ktab,
                           c.opt.alpha, c.ax, c.ay, c.az, c.press, c.divv, c.omega, c.dudt);
    else
        hipLaunchKernelGGL(k_hydro<false>, dim3(nblk((long)c.n * HYD_LPP)), dim3(TB), 0, c.stream, c.kg, c.n, rec,
                           c.active, c.pptot, c.pplist, c.ovf_off, c.ovf_list, c.pp_limit, c.ktab,
                           c.opt.alpha, c.ax, c.ay, c.az, c.press, c.divv, c.omega, c.dudt);
    SX_HIP(hipGetLastError());
    return SERENX_OK;
}

}  // namespace serenx
