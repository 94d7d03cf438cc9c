// grav.hip -- Barnes-Hut gravity walk with monopole/quadrupole/octupole cell
// terms and the grad-h kernel-softened near field, plus the FP64
// kernel-softened direct sum, on gfx950.
//
// The tree is walked for groups of 64 consecutive (tree-ordered) particles, by a
// block that opens it level by level (k_grav_list) or, in large clouds, begun by
// a wave cell by cell (k_grav_cells_*).  In FP64 every particle applies its own
// MAC (BHgrav_accel.F90:154-158): cells it accepts add a multipole term, leaves
// it opens add kernel-softened pair terms (gravity_gradh.F90), branches it opens
// descend.  Each particle therefore sees exactly the reference particle's
// interaction set; MAC tests use the reference's arithmetic (no contraction)
// so that accept/open decisions are identical.  The reference sums all cell
// terms first and the near-field pairs at the end (BHgrav_accel.F90:272-290);
// here cells and pairs go to two accumulators added at the end, so results
// agree with the reference to rounding.
//
// Mixed precision (SERENX_MIXED): the cell offset rp - rc is formed in FP64
// and the multipole and pair terms are evaluated in FP32 on that
// cell-relative offset; cell terms are summed in FP32 batches added to FP64
// sums, pair terms in FP32 per leaf, each leaf's sum added to
// Neumaier-compensated FP32 sums.  Its walk uses a group MAC (see
// group_accepts).
#include <algorithm>
#include <cstring>
#include <rocprim/rocprim.hpp>

#include "walk.h"

namespace serenx {

namespace {

constexpr int TB = 256;
inline int nblk(long n, int tb = TB) { return (int)((n + tb - 1) / tb); }

// BHgrav_accel.F90:97-116: the walk's MAC factor from the previous
// evaluation's |a| (GADGET, GADGET2) or potential (EIGEN); zero while |a| is
// not yet known
template <int MACT>
__device__ __forceinline__ double mac_afactor(double agravmag, double gpot) {
    if (!(agravmag > SMALL_NUMBER)) return 0.0;
    if (MACT == SERENX_MAC_GADGET) return pow(agravmag, -ONETHIRD);
    if (MACT == SERENX_MAC_GADGET2) return 1.0 / sqrt(agravmag);
    return pow(1.0 / gpot, 2.0 * ONETHIRD);
}

// the kernel-range constants in FP32
struct KGeomF {
    float half, range, invrange;
};

// The gravity walks take the kernel range as a template argument (QUINTIC:
// the quintic's range 3, else M4's 2), so that the constants are immediates:
// as kernel arguments they cost the walks 2-6 VGPRs and a wave of occupancy.
template <bool QUINTIC>
__host__ __device__ constexpr KGeom walk_geom() {
    return kernel_geom(QUINTIC ? SERENX_KERNEL_QUINTIC : SERENX_KERNEL_M4);
}

// dx^2 + dy^2 + dz^2 in the reference's operation order with no fused
// multiply-add, also when inlined into code compiled with contraction on
__device__ __forceinline__ double dist2_unfused(double dx, double dy, double dz) {
#pragma clang fp contract(off)
    return dx * dx + dy * dy + dz * dz;
}

// 1/d for d > 0 to a few ulp: the hardware estimate refined by two Newton
// steps y <- y + y (1 - d y) (each squares the relative error).
__device__ __forceinline__ double rcp_fp64(double d) {
#pragma clang fp contract(fast)
    double y = __builtin_amdgcn_rcp(d);
#pragma unroll
    for (int k = 0; k < 2; k++) y = __fma_rn(y, __fma_rn(-d, y, 1.0), y);
    return y;
}

// gravity_gradh.F90:42-86 for one pair, (dx, dy, dz) = r_j - r_p; t4 holds
// (w4, w5, w6, 0) per table index; rangehj = KERNRANGE h_j (the reference's
// product), invhj = 1/h_j.  The kernel index uses the reference's drmag =
// sqrt(r^2) + 1e-20; 1/drmag comes from rcp_fp64.  The pair adds
// f (dx, dy, dz) to the acceleration and m_j / 2 dpot to the potential, each
// by one fused multiply-add; both tables' entries are loaded before either
// is used.
// Returns bit 0: r inside the kernel range of h_p, bit 1: of h_j.
__device__ __forceinline__ unsigned pair_terms(const KGeom &kg, const double4 *__restrict__ t4,
                                               double invhp, double zo_p, double dx, double dy,
                                               double dz, double mj, double rangehj, double invhj,
                                               double zetaj, double &f, double &dpot) {
#pragma clang fp contract(off)
    // r^2 unfused, as the reference forms it: standard SPH's h_gather puts
    // the pp_gather-th neighbour at r = KERNRANGE h_p exactly, and a fused
    // sum can move r across that boundary
    const double drsqd = dist2_unfused(dx, dy, dz);
    const double drmag = sqrt(drsqd) + SMALL_NUMBER;
    const double invdrmag = rcp_fp64(drmag);
    const double id2 = invdrmag * invdrmag;
    const bool in_p = invdrmag > kg.invrange * invhp;
    const bool in_j = drmag < rangehj;
    double4 wp = make_double4(0.0, 0.0, 0.0, 0.0), wj = wp;
    if (in_p) wp = t4[min((int)(kg.half * drmag * invhp), KERNTOT)];
    if (in_j) wj = t4[min((int)(kg.half * drmag * invhj), KERNTOT)];
    double gp = id2, pp = invdrmag, gj = id2, pj = invdrmag;
    if (in_p) {
        gp = invhp * invhp * __fma_rn(zo_p * wp.x * invhp, invhp, wp.y);
        pp = invhp * wp.z;
    }
    if (in_j) {
        gj = invhj * invhj * __fma_rn(zetaj * wj.x * invhj, invhj, wj.y);
        pj = invhj * wj.z;
    }
    f = 0.5 * mj * invdrmag * (gp + gj);
    dpot = pp + pj;
    return (in_p ? 1u : 0u) | (in_j ? 2u : 0u);
}

// the pair's terms added to a lane's own sums; the same bits returned
__device__ __forceinline__ unsigned pair_fp64(const KGeom &kg, const double4 *__restrict__ t4,
                                              double invhp, double zo_p, double dx, double dy,
                                              double dz, double mj, double rangehj, double invhj,
                                              double zetaj, double &ax, double &ay, double &az,
                                              double &pot) {
    double f, dpot;
    const unsigned in_ =
        pair_terms(kg, t4, invhp, zo_p, dx, dy, dz, mj, rangehj, invhj, zetaj, f, dpot);
    ax = __fma_rn(f, dx, ax);
    ay = __fma_rn(f, dy, ay);
    az = __fma_rn(f, dz, az);
    pot = __fma_rn(0.5 * mj, dpot, pot);
    return in_;
}

// Gravity source record of particle j, 64 bytes in a buffer of its own (the
// walk runs beside the neighbour and hydro kernels, which use theirs):
// [0] x y z m  [1] h 1/h zeta KERNRANGE*h
__global__ void k_pack_grav(int n, double kernrange, const double *__restrict__ x,
                            const double *__restrict__ y,
                            const double *__restrict__ z, const double *__restrict__ m,
                            const double *__restrict__ h, const double *__restrict__ zeta,
                            double4 *__restrict__ rec) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    double4 *r = rec + 2 * (size_t)i;
    r[0] = make_double4(x[i], y[i], z[i], m[i]);
    r[1] = make_double4(h[i], 1.0 / h[i], zeta[i], kernrange * h[i]);
}

// Gravity source records of the mixed walk, 32 bytes per particle, written
// per leaf of the gravity tree (one thread per node; leaves partition the
// particles):
//   [0] x - x_f, y - y_f, z - z_f (FP32), m / 2   [1] KERNRANGE h, 1/h, 1/h^2, zeta/h^2
// where (x_f, y_f, z_f) is the leaf's first particle.  A pair term then
// takes the offset r_j - r_p as (r_j - r_f) + (r_f - r_p): the second term is
// formed in FP64 once per leaf and lane, so no FP64 work remains per pair.
__global__ void k_pack_grav_mixed(int nc, double kernrange, const GNodeF *__restrict__ gn,
                                  const double *__restrict__ x, const double *__restrict__ y,
                                  const double *__restrict__ z, const double *__restrict__ m,
                                  const double *__restrict__ h, const double *__restrict__ zeta,
                                  float4 *__restrict__ rec) {
    const int c = blockIdx.x * blockDim.x + threadIdx.x;
    if (c >= nc) return;
    const int k = gn[c].leaf, f = gn[c].first;
    if (k <= 0) return;
    const double xf = x[f], yf = y[f], zf = z[f];
    for (int i = 0; i < k; i++) {
        const int j = f + i;
        const double hj = h[j], ih = 1.0 / hj;
        rec[2 * (size_t)j] = make_float4((float)(x[j] - xf), (float)(y[j] - yf),
                                         (float)(z[j] - zf), (float)(0.5 * m[j]));
        rec[2 * (size_t)j + 1] = make_float4((float)(kernrange * hj), (float)ih,
                                             (float)(ih * ih), (float)(zeta[j] * ih * ih));
    }
}

// a += a_grav for the active particles: the one addition sph_grav_forces.F90
// makes (a holds the hydro acceleration)
__global__ void k_add_grav(int n, const uint8_t *__restrict__ active,
                           const double *__restrict__ gx, const double *__restrict__ gy,
                           const double *__restrict__ gz, double *__restrict__ ax,
                           double *__restrict__ ay, double *__restrict__ az) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n || !active[i]) return;
    ax[i] = ax[i] + gx[i];
    ay[i] = ay[i] + gy[i];
    az[i] = az[i] + gz[i];
}

// 1/sqrt(a) for a > 0 to about one ulp: the hardware estimate (relative
// error below 2^-23) refined by one third-order step
//   y <- y (1 + e/2 + 3e^2/8),  e = 1 - a y^2,
// whose truncation error (5/16) e^3 is below 2^-66.
__device__ __forceinline__ double rsqrt_fp64(double a) {
#pragma clang fp contract(fast)
    const double y = __builtin_amdgcn_rsq(a);
    const double e = __fma_rn(-a * y, y, 1.0);
    return __fma_rn(y * e, __fma_rn(0.375, e, 0.5), y);
}

// Multipole terms of one accepted cell at offset (x, y, z) = r_p - r_cell:
// the monopole, quadrupole and octupole terms of BHgrav_accel.F90:159-222,
// evaluated in factored form.  With Q the traceless quadrupole,
// S(r) = sum_k s_k m_k(r) the octupole cubic and H = grad(S) / 2,
//   a   = -m r / r^3 + Q r / r^5 - 5/2 (r.Q.r) r / r^7
//         + H / r^7 - 7/3 (r.H) r / r^9,
//   phi = m / r + (r.Q.r) / (2 r^5) + (r.H) / (3 r^7),
// term for term the reference's expressions (its octupole force terms are
// the components of H); S is formed as 2 (r.H) / 3 (Euler's identity for a
// homogeneous cubic).  q = [xx xy yy zx zy zz]; oc holds H's coefficients on
// the monomials (xx xy xz yy zz yz), stocked per node.
//
// The factors of the terms, so that a wave can form them and another add them
// (add_cell): a += Q ir5 + H ir7 + crad r, phi.  Every multiply-add is written
// out, as in cell_terms_s.
struct CellFactors {
    double Q[3], ir5, H[3], ir7, crad, phi;
};

template <int OCT>
__device__ __forceinline__ CellFactors cell_factors(double x, double y, double z, double ir,
                                                    double m, const double *q,
                                                    const double *oc) {
#pragma clang fp contract(off)
    CellFactors f;
    const double ir2 = ir * ir;
    const double ir3 = ir * ir2;
    f.ir5 = ir2 * ir3;
    f.ir7 = ir2 * f.ir5;
    f.Q[0] = __fma_rn(q[3], z, __fma_rn(q[1], y, q[0] * x));
    f.Q[1] = __fma_rn(q[4], z, __fma_rn(q[2], y, q[1] * x));
    f.Q[2] = __fma_rn(q[5], z, __fma_rn(q[4], y, q[3] * x));
    // (r.Q.r) / r^5
    const double t5 = f.ir5 * __fma_rn(z, f.Q[2], __fma_rn(y, f.Q[1], x * f.Q[0]));
    f.crad = __fma_rn(ir2, -2.5 * t5, -(m * ir3));
    f.phi = __fma_rn(m, ir, 0.5 * t5);
    f.H[0] = f.H[1] = f.H[2] = 0.0;
    if (OCT) {
        const double xx = x * x, yy = y * y, zz = z * z;
        const double xy = x * y, xz = x * z, yz = y * z;
#pragma unroll
        for (int k = 0; k < 3; k++) {
            const double *o = oc + 6 * k;
            f.H[k] = __fma_rn(
                o[5], yz,
                __fma_rn(o[4], zz,
                         __fma_rn(o[3], yy, __fma_rn(o[2], xz, __fma_rn(o[1], xy, o[0] * xx)))));
        }
        // (r.H) / r^7
        const double rh = f.ir7 * __fma_rn(z, f.H[2], __fma_rn(y, f.H[1], x * f.H[0]));
        f.crad = __fma_rn(ir2, (-7.0 / 3.0) * rh, f.crad);
        f.phi = __fma_rn(1.0 / 3.0, rh, f.phi);
    }
    return f;
}

// one component of the acceleration
template <int OCT>
__device__ __forceinline__ double add_cell(double a, double Q, double ir5, double H, double ir7,
                                           double crad, double x) {
    a = __fma_rn(ir5, Q, a);
    if (OCT) a = __fma_rn(ir7, H, a);
    return __fma_rn(x, crad, a);
}

// The same terms from the moments themselves (the FP32 walk, whose nodes keep
// 10 moments instead of 18 coefficients to stay at two cache lines):
// G = grad S = 2 H, S formed as (r.G) / 3.
//   s = [x^3 x^2y y^2x y^3 z^2x z^2y z^3 x^2z y^2z xyz]
// Every multiply-add is written out: left to the compiler, which of two
// products is rounded changes from one caller to the next, and with it the
// FP32 rounding of the results.
template <int OCT>
__device__ __forceinline__ void cell_terms_s(float x, float y, float z, float ir, float m,
                                             const float *q, const float *s, float &ax, float &ay,
                                             float &az, float &pot) {
#pragma clang fp contract(off)
    const float ir2 = ir * ir;
    const float ir3 = ir * ir2;
    const float ir5 = ir2 * ir3;
    const float ir7 = ir2 * ir5;
    auto dot = [](float a0, float b0, float a1, float b1, float a2, float b2) {
        return __builtin_fmaf(a2, b2, __builtin_fmaf(a1, b1, a0 * b0));
    };
    const float Qx = dot(q[0], x, q[1], y, q[3], z);
    const float Qy = dot(q[1], x, q[2], y, q[4], z);
    const float Qz = dot(q[3], x, q[4], y, q[5], z);
    const float qs = dot(Qx, x, Qy, y, Qz, z);
    float crad = __builtin_fmaf(ir7, -2.5f * qs, -(m * ir3));
    float phi = __builtin_fmaf(m, ir, ir5 * (0.5f * qs));
    float fx, fy, fz;
    if (OCT) {
        const float xx = x * x, yy = y * y, zz = z * z;
        const float xy = x * y, xz = x * z, yz = y * z;
        const float xx3 = 3.0f * xx, yy3 = 3.0f * yy, zz3 = 3.0f * zz;
        const float xy2 = xy + xy, xz2 = xz + xz, yz2 = yz + yz;
        auto dot3 = [](float v, float a0, float b0, float a1, float b1, float a2, float b2) {
            return __builtin_fmaf(a2, b2, __builtin_fmaf(a1, b1, __builtin_fmaf(a0, b0, v)));
        };
        const float Gx = dot3(dot(s[0], xx3, s[1], xy2, s[7], xz2), s[2], yy, s[4], zz, s[9], yz);
        const float Gy = dot3(dot(s[1], xx, s[2], xy2, s[3], yy3), s[5], zz, s[9], xz, s[8], yz2);
        const float Gz = dot3(dot(s[7], xx, s[8], yy, s[6], zz3), s[4], xz2, s[5], yz2, s[9], xy);
        const float rg = dot(Gx, x, Gy, y, Gz, z);   // 3 S
        const float h7 = 0.5f * ir7;
        crad = __builtin_fmaf(ir2, ir7 * ((-3.5f / 3.0f) * rg), crad);
        phi = __builtin_fmaf(ir7, (0.5f / 3.0f) * rg, phi);
        fx = __builtin_fmaf(crad, x, __builtin_fmaf(h7, Gx, Qx * ir5));
        fy = __builtin_fmaf(crad, y, __builtin_fmaf(h7, Gy, Qy * ir5));
        fz = __builtin_fmaf(crad, z, __builtin_fmaf(h7, Gz, Qz * ir5));
    } else {
        fx = __builtin_fmaf(ir5, Qx, crad * x);
        fy = __builtin_fmaf(ir5, Qy, crad * y);
        fz = __builtin_fmaf(ir5, Qz, crad * z);
    }
    ax = ax + fx;
    ay = ay + fy;
    az = az + fz;
    pot = pot + phi;
}

template <int OCT>
__device__ __forceinline__ void cell_fp64(const GNode &g, const double dr[3], double drsqd,
                                          double &ax, double &ay, double &az, double &pot) {
    const CellFactors f =
        cell_factors<OCT>(dr[0], dr[1], dr[2], rsqrt_fp64(drsqd + SMALL_NUMBER), g.m, g.q, g.oc);
    ax = add_cell<OCT>(ax, f.Q[0], f.ir5, f.H[0], f.ir7, f.crad, dr[0]);
    ay = add_cell<OCT>(ay, f.Q[1], f.ir5, f.H[1], f.ir7, f.crad, dr[1]);
    az = add_cell<OCT>(az, f.Q[2], f.ir5, f.H[2], f.ir7, f.crad, dr[2]);
    pot = pot + f.phi;
}

// Near-field lists: per group, the leaves its walk opened, in DFS order, as
// (first particle << 4) | particle count, with the mask of the lanes that
// opened each.  Phase 1 of the walk writes them, phase 2 reads them.  Entries
// lie in pages of a pool (a group knows its number of leaves before it takes
// its pages, so the pool serves lists of any length without waste).
struct NearList {
    int *leaf;                    // npage x PL_PAGE entries
    unsigned long long *mask;     // their lane masks
    int *page;                    // per group: PL_PAGES page numbers
    int *next;                    // next free page
    int *len;                     // per group: entries (NEAR_DROPPED: not stored)
    int cap;                      // entries a group may store (<= PL_PAGES PL_PAGE)
    int npage;                    // pages of the pool
    __device__ __forceinline__ size_t slot(int g, int e) const {
        return (size_t)page[(size_t)g * PL_PAGES + e / PL_PAGE] * PL_PAGE + e % PL_PAGE;
    }
};
constexpr int NEAR_DROPPED = 0x7FFFFFFF;

// Ordered FP64 sums (clouds of up to LW_ORDERED particles): waves of a block,
// in the pair phase targets of a wave and lanes of a target
constexpr int OW_WAVES = 16, OW_TB = OW_WAVES * WAVE;
constexpr int OW_T = WAVE / OW_WAVES, OW_L = WAVE / OW_T;
static_assert(OW_L == 2 * LEAFMAX, "two leaves on a target's lanes");

// The walk in two phases, so that the traversal and the cell terms -- which
// need only the positions, the tree stocked with the previous h (Q2:
// BHgrav_stock runs before sph_update) and the previous |a| -- run beside
// the h solve, and only the kernel-softened pair terms wait for the new h
// and zeta.  The reference sums the cell terms of the walk first and the
// near-field pairs of its list afterwards (BHgrav_accel.F90:225-226,
// 272-290); so does this split, in the same orders.
//
// Phase 1 is k_grav_list below.  FP64: each target applies its own MAC
// (BHgrav_accel.F90:154-158); cells it accepts add a multipole term, leaves it
// opens go to the group's near-field list, branches it opens descend.

// Phase 2: the pair terms of gravity_gradh.F90 over each particle's opened
// leaves, in list order, added to the cell sums of phase 1.
//
// A block takes a group: every wave has all its targets, one per lane, and
// takes the list's batches of PF_STAGE leaves in turn: lane l copies particle
// l of the batch's leaves into LDS (the loads of a batch are in flight at
// once), then the wave goes through the leaves and the lanes that opened one
// add its terms.  The waves' sums are added in wave order at the end.
//
// Why: the chain of record load, square root, reciprocal and table load takes
// half a microsecond per source, so a wave that has a group's list alone takes
// as long as the longest list (the centre of a uniform sphere, where
// |a| -> 0, opens 10,000 leaves).  Uniform sphere of 131,071 particles: 10.6 ->
// 0.9 ms, of 2,048: 128 -> 60 us (four lanes per target, a wave per 16
// targets); r^-2 sphere of 300,007, which fills the device: 1.7 -> 1.3 ms.
//
// A group whose list was not stored walks again, all its targets in every
// wave (the same MAC decisions: they read the stocked tree and the previous
// |a| and potential, which the block overwrites only when all its waves are
// done), so the batches and the sums are the same.
//
// ORDERED: clouds of up to LW_ORDERED particles, whose terms are added in list
// order (see k_grav_list): a wave has OW_T targets with OW_L lanes each, which
// take the particles of the target's next two leaves and send their factors
// through LDS to the lanes that add them: 349 us on an r^-2 sphere of 4,096
// (153 us with the sums in wave order), bound by the steps of the target with
// the most leaves; with 16 targets and four lanes each 361 us, with a leaf per
// wave and the adding left to four waves 456 us.
constexpr int PF_STAGE = WAVE / LEAFMAX;
constexpr int PF_WAVES = 8;
constexpr int PF_TB = PF_WAVES * WAVE;

template <int MACT, bool QUINTIC, bool ORDERED>
__global__ void __launch_bounds__(ORDERED ? OW_TB : PF_TB) k_grav_pairs_fp64(
    int nc, const GNode *__restrict__ gn, const double4 *__restrict__ rec,
    const int *__restrict__ cid, const int2 *__restrict__ root_range,
    const uint8_t *__restrict__ active, const double4 *__restrict__ t4,
    double *__restrict__ ax, double *__restrict__ ay, double *__restrict__ az,
    const double *__restrict__ cp, double *__restrict__ gpot, double *__restrict__ agm,
    NearList near, unsigned long long *__restrict__ icount, const int2 *__restrict__ grp,
    const int *__restrict__ cloud_off, GroupQueue queue) {
    // persistent over the walk's queue: the groups of each XCD range
    // longest-first (by the previous walk's cost), as phase 1 takes them
    __builtin_amdgcn_s_setprio(2);
    // per wave: the records of a batch; in their place at the end, the sums.
    // Ordered sums: per component, the lanes' factor pairs (one slot of padding)
    __shared__ union {
        double4 stage[ORDERED ? 1 : PF_WAVES][2 * WAVE];
        double2 xch[ORDERED ? OW_WAVES : 1][4][WAVE + 1];
    } lds;
    auto &stage_all = lds.stage;
    __shared__ int job;
    constexpr KGeom kg = walk_geom<QUINTIC>();
    const int lane = (int)(threadIdx.x & (WAVE - 1));
    const int wave = uniform((int)(threadIdx.x / WAVE));
    double4 *stage = stage_all[wave];
    unsigned npp = 0, nin_p = 0, nin_j = 0;   // wave totals
    const int home = blockIdx.x % NXCD;
    int qdone = 0;
    for (;;) {
        __syncthreads();
        if (wave == 0) {
            const int t = next_group(queue, home, qdone);
            if (lane == 0) job = t;
        }
        __syncthreads();
        const int g = uniform(job);
        if (g < 0) break;
        const int2 gr = grp[g];
        const int p = gr.x + lane;
        const bool valid = p < gr.y && active[p];
        if (ballot(valid) == 0) continue;   // the whole block
        double rpx = 0, rpy = 0, rpz = 0, invhp = 1.0, zo_p = 0.0;
        double gx = 0, gy = 0, gz = 0, gp = 0;
        if (valid) {
            const double4 a = rec[2 * (size_t)p], b = rec[2 * (size_t)p + 1];
            rpx = a.x; rpy = a.y; rpz = a.z;
            invhp = b.y;
            zo_p = b.z;
        }
        // one leaf, its records at a (wave-uniform)
        auto leaf_pairs = [&](const double4 *src, int first, int count, bool mine) {
            for (int i = 0; i < count; i++) {
                const double4 a = src[2 * i], b = src[2 * i + 1];
                const bool act = mine && first + i != p;
                unsigned in_ = 0;
                if (act)
                    in_ = pair_fp64(kg, t4, invhp, zo_p, a.x - rpx, a.y - rpy, a.z - rpz, a.w,
                                    b.w, b.y, b.z, gx, gy, gz, gp);
                npp += lanes(act);
                nin_p += lanes(in_ & 1);
                nin_j += lanes(in_ & 2);
            }
        };
        const int len = uniform(near.len[g]);
        const int root = __builtin_amdgcn_readlane(valid ? cid[p] : 0,
                                                   __ffsll((long long)ballot(valid)) - 1);
        if ((cloud_off[root + 1] - cloud_off[root] <= LW_ORDERED) != ORDERED)
            continue;   // the other launch's group
        constexpr bool ordered = ORDERED;
        if (ordered && len == NEAR_DROPPED && valid && wave == 0) {
            gx = ax[p]; gy = ay[p]; gz = az[p]; gp = cp[p];   // wave 0 walks alone
        }
        if (ordered && len != NEAR_DROPPED) {
            // the wave's targets go through their own leaves, a target's lanes
            // on the leaf's particles; the factors of the terms go through LDS
            // to the lane that adds a component (0-2, potential 3, in gx)
            double2(*xch)[WAVE + 1] = lds.xch[wave];
            const int sub = lane % OW_L, l0 = lane & ~(OW_L - 1);
            const int tg = wave * OW_T + lane / OW_L, pt = gr.x + tg;
            const bool mine = pt < gr.y && active[pt];
            double qx = 0.0, qy = 0.0, qz = 0.0, ihq = 1.0, zoq = 0.0;
            if (mine) {
                const double4 a = rec[2 * (size_t)pt], b = rec[2 * (size_t)pt + 1];
                qx = a.x; qy = a.y; qz = a.z;
                ihq = b.y;
                zoq = b.z;
                if (sub < 4) gx = (sub == 0 ? ax : sub == 1 ? ay : sub == 2 ? az : cp)[pt];
            }
            for (int e0 = 0; e0 < len; e0 += WAVE) {
                const bool have = e0 + lane < len;
                const size_t at = near.slot(g, e0) + lane;   // a chunk lies in one page
                const int d = have ? near.leaf[at] : 0;
                const unsigned long long m = have ? near.mask[at] : 0ull;
                // the chunk's leaves that the lane's target opened
                const unsigned mm = (unsigned)(m >> (wave * OW_T));
                unsigned long long word = 0;
#pragma unroll
                for (int t = 0; t < OW_T; t++) {
                    const unsigned long long b = ballot((mm >> t) & 1u);
                    if (lane / OW_L == t) word = b;
                }
                if (!mine) word = 0;
                // the lane's source of the target's next two leaves, if any
                auto next = [&](int &j) -> bool {
                    const unsigned long long rest = word & (word - 1);
                    const unsigned long long own = sub < LEAFMAX ? word : rest;
                    const int e = own ? __ffsll((long long)own) - 1 : 0;
                    const int de = __shfl(d, e, WAVE), i = sub % LEAFMAX;
                    const bool act = own != 0 && i < (de & 15);
                    j = act ? (de >> 4) + i : gr.x;
                    word = rest & (rest - 1);
                    return act && j != pt;
                };
                bool more = any_lane(word != 0);
                int j;
                bool act = next(j);
                double4 a = rec[2 * (size_t)j], b = rec[2 * (size_t)j + 1];
                while (more) {
                    more = any_lane(word != 0);
                    // the next sources' records are in flight while these are used
                    int jn;
                    const bool actn = next(jn);
                    const double4 an = rec[2 * (size_t)jn], bn = rec[2 * (size_t)jn + 1];
                    double dx = 0.0, dy = 0.0, dz = 0.0, f = 0.0, hm = 0.0, dpot = 0.0;
                    unsigned in_ = 0;
                    if (act) {
                        dx = a.x - qx;
                        dy = a.y - qy;
                        dz = a.z - qz;
                        hm = 0.5 * a.w;
                        in_ = pair_terms(kg, t4, ihq, zoq, dx, dy, dz, a.w, b.w, b.y, b.z, f,
                                         dpot);
                    }
                    npp += lanes(act);
                    nin_p += lanes(in_ & 1);
                    nin_j += lanes(in_ & 2);
                    // a lane without a source adds 0 * 0, which leaves the sum
                    // (never -0) as it is
                    xch[0][lane] = make_double2(f, dx);
                    xch[1][lane] = make_double2(f, dy);
                    xch[2][lane] = make_double2(f, dz);
                    xch[3][lane] = make_double2(hm, dpot);
                    wave_lds_fence();
                    if (sub < 4) {
#pragma unroll
                        for (int i0 = 0; i0 < OW_L; i0 += 4) {
                            double2 t[4];
#pragma unroll
                            for (int i = 0; i < 4; i++) t[i] = xch[sub][l0 + i0 + i];
#pragma unroll
                            for (int i = 0; i < 4; i++) gx = __fma_rn(t[i].x, t[i].y, gx);
                        }
                    }
                    wave_lds_fence();
                    a = an;
                    b = bn;
                    act = actn;
                }
            }
            const double sx = __shfl(gx, l0, WAVE), sy = __shfl(gx, l0 + 1, WAVE),
                         sz = __shfl(gx, l0 + 2, WAVE);
            __syncthreads();   // every wave is done
            if (mine && sub < 4) {
                (sub == 0 ? ax : sub == 1 ? ay : sub == 2 ? az : gpot)[pt] = gx;
                if (MACT != SERENX_MAC_GEOMETRIC && sub == 0)
                    agm[pt] = sqrt(sx * sx + sy * sy + sz * sz);
            }
            continue;
        } else if (len != NEAR_DROPPED) {
            for (int e0 = wave * PF_STAGE; e0 < len; e0 += PF_WAVES * PF_STAGE) {
                const int nb = min(PF_STAGE, len - e0);
                const size_t at = near.slot(g, e0);   // a batch lies in one page
                const int e = lane / LEAFMAX, i = lane % LEAFMAX;
                const int dl = e < nb ? near.leaf[at + e] : 0;
                const unsigned long long ml = e < nb ? near.mask[at + e] : 0ull;
                if (i < (dl & 15)) {
                    const size_t j = (size_t)(dl >> 4) + i;
                    stage[2 * lane] = rec[2 * j];
                    stage[2 * lane + 1] = rec[2 * j + 1];
                }
                wave_lds_fence();
                for (int k = 0; k < nb; k++) {
                    const int d = __builtin_amdgcn_readlane(dl, k * LEAFMAX);
                    const unsigned long long m =
                        (unsigned)__builtin_amdgcn_readlane((int)ml, k * LEAFMAX) |
                        (unsigned long long)(unsigned)__builtin_amdgcn_readlane(
                            (int)(ml >> 32), k * LEAFMAX) << 32;
                    leaf_pairs(stage + 2 * LEAFMAX * k, d >> 4, d & 15,
                               __builtin_amdgcn_inverse_ballot_w64(m));
                }
                wave_lds_fence();   // every read before the next batch's writes
            }
        } else {
            // the group's walk again; the wave takes its own batches
            double afactor = 0.0;
            if (valid && MACT != SERENX_MAC_GEOMETRIC)
                afactor = mac_afactor<MACT>(agm[p], gpot[p]);
            const int2 rr = valid ? root_range[cid[p]] : make_int2(nc, nc);
            unsigned lv = 0;
            int e = 0;
            (void)group_walk(
                gn, nc, valid, rr.x, rr.y, lv,
                [&](const GNode &nd, bool) -> int {
                    const double dr[3] = {rpx - nd.r[0], rpy - nd.r[1], rpz - nd.r[2]};
                    const double drsqd = dr[0] * dr[0] + dr[1] * dr[1] + dr[2] * dr[2];
                    bool accept;
                    if (MACT == SERENX_MAC_GEOMETRIC)
                        accept = drsqd > nd.dminsqd;
                    else
                        accept = drsqd > nd.mac * afactor && drsqd > nd.dminsqd;
                    accept = accept && nd.leaf != 1;
                    if (accept) return WALK_SKIP;
                    return nd.leaf > 0 ? WALK_LEAF : WALK_DESCEND;
                },
                [&](const GNode &nd, bool mine) {
                    if ((ordered ? 0 : e / PF_STAGE % PF_WAVES) == wave)
                        leaf_pairs(rec + 2 * (size_t)nd.first, nd.first, nd.leaf, mine);
                    e++;
                });
        }
        // every wave is done with its stage and with the previous |a|
        __syncthreads();
        double *sums = reinterpret_cast<double *>(&lds);   // [wave][component][lane]
        sums[(wave * 4 + 0) * WAVE + lane] = gx;
        sums[(wave * 4 + 1) * WAVE + lane] = gy;
        sums[(wave * 4 + 2) * WAVE + lane] = gz;
        sums[(wave * 4 + 3) * WAVE + lane] = gp;
        __syncthreads();
        if (wave == 0 && valid) {
            if (!ordered) {
                gx = ax[p]; gy = ay[p]; gz = az[p]; gp = cp[p];   // the cell sums
                for (int w = 0; w < PF_WAVES; w++) {
                    gx += sums[(w * 4 + 0) * WAVE + lane];
                    gy += sums[(w * 4 + 1) * WAVE + lane];
                    gz += sums[(w * 4 + 2) * WAVE + lane];
                    gp += sums[(w * 4 + 3) * WAVE + lane];
                }
            }
            ax[p] = gx;   // the gravity acceleration; k_add_grav adds it to a
            ay[p] = gy;
            az[p] = gz;
            gpot[p] = gp;
            if (MACT != SERENX_MAC_GEOMETRIC) agm[p] = sqrt(gx * gx + gy * gy + gz * gz);
        }
    }
    if (lane == 0) {
        unsigned long long *ic = ctr_row(icount);
        atomicAdd(ic + 1, (unsigned long long)npp);
        atomicAdd(ic + 2, (unsigned long long)nin_p);
        atomicAdd(ic + 3, (unsigned long long)nin_j);
    }
}

// ---- mixed precision ------------------------------------------------------
// Neumaier compensated FP32 sum
struct CSum {
    float s = 0.0f, c = 0.0f;
    __device__ __forceinline__ void add(float v) {
        const float t = s + v;
        c += (fabsf(s) >= fabsf(v)) ? ((s - t) + v) : ((v - t) + s);
        s = t;
    }
    __device__ __forceinline__ double value() const { return (double)s + (double)c; }
};

// The target's side of a mixed pair term, per lane: 1/h_p, 1/h_p^2,
// zeta_p/h_p^2, the kernel-range limit on 1/r (KERNRANGE h_p)^-1 and the
// table scale KERNTOT / (KERNRANGE h_p)
struct PairTarget {
    float ih, ih2, zi2, lim, hk;
};

// gravity_gradh.F90:42-86 for one pair in FP32 on the offset (dx, dy, dz) =
// r_j - r_p, with the source record of k_pack_grav_mixed (hm = m_j / 2, rh =
// KERNRANGE h_j, ih = 1/h_j, ih2 = 1/h_j^2, zi2 = zeta_j/h_j^2).  |r| and 1/|r|
// come from one reciprocal square root.  The softened terms are selected per
// lane under wave-uniform branches (taken when any lane is inside the
// range), so that the wave runs no divergent branches; a lane with act
// unset adds nothing.  The terms
// are added to FP32 sums (the caller's per-leaf partial sums).  mact is the
// wave's mask of the lanes with act set; the wave counts the pairs inside
// the kernel range of h_p (nin_p) and of h_j (nin_j) from the masks of the
// two comparisons themselves.
__device__ __forceinline__ void pair_f32(const KGeomF &kg, const float4 *__restrict__ t4,
                                         const PairTarget &tp, bool act,
                                         unsigned long long mact, float dx, float dy,
                                         float dz, float hm, float rh, float ih, float ih2,
                                         float zi2, float &ax, float &ay, float &az, float &pot,
                                         unsigned &nin_p, unsigned &nin_j) {
#pragma clang fp contract(fast)
    // written out: which product the compiler rounds depends on the caller
    const float d2 = __builtin_fmaf(dz, dz, __builtin_fmaf(dx, dx, dy * dy));
    const float ir = __builtin_amdgcn_rsqf(d2 + 1.0e-30f);
    const float dr = d2 * ir;
    const float ir2 = ir * ir;
    const bool in_p = act && ir > tp.lim;
    const bool in_j = act && dr < rh;
    const unsigned long long mp = ballot(ir > tp.lim) & mact, mj = ballot(dr < rh) & mact;
    nin_p += (unsigned)__popcll(mp);
    nin_j += (unsigned)__popcll(mj);
    float grav = ir2, dpot = ir;
    // the kernel-softened parts only when a lane needs them (wave-uniform
    // branches); unsigned table indices (at most KERNTOT) give 32-bit offsets
    if (mp) {
        const float4 wp = t4[(unsigned)min((int)(tp.hk * dr), KERNTOT)];
        grav = in_p ? tp.ih2 * (wp.y + tp.zi2 * wp.x) : grav;
        dpot = in_p ? tp.ih * wp.z : dpot;
    }
    float gj = ir2, pj = ir;
    if (mj) {
        const float4 wj = t4[(unsigned)min((int)(kg.half * dr * ih), KERNTOT)];
        gj = in_j ? ih2 * (wj.y + zi2 * wj.x) : gj;
        pj = in_j ? ih * wj.z : pj;
    }
    grav = grav + gj;
    dpot = dpot + pj;
    const float f = act ? hm * ir * grav : 0.0f;
    ax = ax + f * dx;
    ay = ay + f * dy;
    az = az + f * dz;
    pot = pot + (act ? hm * dpot : 0.0f);
}

// FP32 multipole terms on the FP32 cell offset, added to an FP32 batch sum
template <int OCT>
__device__ __forceinline__ void cell_fp32(const GNodeF &g, const float dr[3], float &ax,
                                          float &ay, float &az, float &pot) {
#pragma clang fp contract(off)
    const float drsqd =
        __builtin_fmaf(dr[2], dr[2], __builtin_fmaf(dr[0], dr[0], dr[1] * dr[1]));
    const float ir = __builtin_amdgcn_rsqf(drsqd + 1.0e-30f);
    cell_terms_s<OCT>(dr[0], dr[1], dr[2], ir, g.m, g.q, g.s, ax, ay, az, pot);
}

// Cell terms are summed in FP32 over batches of CELL_BATCH cell visits of the
// wave and each batch is added to FP64 sums: a batch sum carries at most a
// few FP32 roundings per term, and the conversions and FP64 additions are
// paid once per batch instead of once per cell.
constexpr int CELL_BATCH = 8;

// The mixed walk uses a group MAC: a wave of 64 tree-ordered particles
// accepts a cell only when the MAC of BHgrav_accel.F90:154-158 accepts it for
// every one of its particles, and otherwise opens it for all of them (leaves
// give pair terms to all).  Every accepted cell therefore satisfies each
// particle's own MAC, so the truncation error is at most the per-particle
// walk's; the walk is wave-uniform (no per-lane resume state), and no cell
// term is issued for a cell that only some lanes use.  The FP64 walk keeps
// the reference's per-particle interaction sets.  As the FP64 walk, it runs
// in two phases: cells (beside the h solve), then pairs.
//
// A group lies in one cloud (its walk covers that cloud's DFS range), so
// the lanes taking part are the same at every cell: vmask, the valid lanes.
// The test forms each comparison's lane mask directly and combines the
// masks in scalar registers.
template <int MACT>
__device__ __forceinline__ bool group_accepts(const GNodeF &nd, unsigned long long vmask,
                                              double rpx, double rpy, double rpz, double afactor,
                                              double &d0, double &d1, double &d2) {
    d0 = rpx - nd.r[0];
    d1 = rpy - nd.r[1];
    d2 = rpz - nd.r[2];
    const double drsqd = d0 * d0 + d1 * d1 + d2 * d2;
    unsigned long long ok = ballot(drsqd > nd.dminsqd);
    if (MACT != SERENX_MAC_GEOMETRIC) ok &= ballot(drsqd > nd.mac * afactor);
    return nd.leaf != 1 && (vmask & ~ok) == 0;       // :128-136; every lane accepts
}

// ---- the list walk ---------------------------------------------------------
// Phase 1 of the walk (traversal, cell terms, near lists) by a block of
// LW_WAVES waves per group, in three steps:
//  1. the tree is opened level by level, one cell per lane: the lane tests its
//     cell's MAC against the sphere that holds the group's targets and, where
//     that does not decide it, against every target (in LDS); it appends an
//     opened branch's children to the block's list of cells to visit;
//  2. two bit maps over the cloud's cells (accepted cells, opened leaves) give
//     every entry its rank in DFS order, so both lists come out in the order
//     of a walk, whatever order the lanes appended in;
//  3. each wave forms the terms of its share of the accepted cells, one
//     target per lane, the nodes through the scalar cache.
//
// Why: a wave that walks alone visits a cell in 0.4 to 1 us (scalar load, test,
// vote and term one after the other), so a launch took as long as its largest
// walk: 16.6 ms on a uniform sphere of 131,071 particles whose central groups,
// where |a| -> 0, visit 15,000 cells.  Here 64 tests run at once and the cells
// to come are known before their terms are formed: 3.5 ms there; 300 -> 62 us
// on 2,048 particles (FP64, quadrupole), 1,454 -> 332 us on an r^-2 sphere of
// 16,384 and 5.3 -> 0.7 ms on a uniform one of 65,536 (mixed).  Bound by the
// vector ALU: on the 1M r^-2 sphere 89 instructions per accepted cell and
// wave, and 1.1e9 of 8.1e9 in steps 1 and 2 (2.2e9 with every cell tested
// against every target, without the sphere).
//
// Results.  The accepted cells, their order and (mixed) their batches of
// CELL_BATCH are the serial walk's; the waves' FP64 sums are added in wave
// order at the end.  A group's sums depend only on its own cloud.  In clouds of
// up to LW_ORDERED particles the terms themselves are added in the walk's
// order, so their results are those of a walk by one wave bit for bit: small
// clouds are the ones followed over many steps, and a collapsing core of 4,096
// particles makes 1e-8 of a last bit in 60 steps.  Mixed: the sums of a batch
// go through LDS to four waves, one component each.  FP64: a launch of its own
// with 16 waves a block; a round of 16 cells' factors (6.6 KB a cell) goes
// through LDS to four waves that add them: 311 us on an r^-2 sphere of 4,096
// particles, 188 us with the sums in wave order, 849 us by one wave.
//
// A window of the cloud's DFS range is walked at a time: at most LW_BITS
// cells, halved when the block's LW_CAP entries overflow (cells outside the
// window are dropped untested, its ancestors are tested and not counted).
constexpr int LW_TB = LW_WAVES * WAVE;

template <int NW>
struct ListWalk {
    // cells of a window (a block of ordered sums, whose factors need the room,
    // walks small clouds)
    static constexpr int CELLS = NW == LW_WAVES ? LW_BITS : LW_BITS / 4;
    double x[WAVE], y[WAVE], z[WAVE], af[WAVE];   // targets
    unsigned bits[2][CELLS / 32];                 // accepted cells, opened leaves
    int pre[2][CELLS / 128];                    // their ranks at every 128th cell
    unsigned short und[LW_CAP];                   // entries of a level left to all targets
    double c[3], rad, afmin, afmax;               // sphere of the targets, range of af
    int job, cnt[3], nund[3], page0;
    unsigned long long wsum[NW];
};
// the waves' sums take the place of the accepted cells' bits at the end
static_assert(sizeof(unsigned) * LW_BITS / 32 >= sizeof(double) * 4 * LW_TB, "sums fit");
// Walks that one wave began and left to the list walk (k_grav_cells_*): their
// groups, where each goes on, their number and how many have been taken.
// A null group: the list walk takes every group of the queue from its root.
struct LongWalks {
    int *group, *at, *n, *taken;
    int budget;      // visits of a walk by one wave
    int alone;       // clouds of at most this many particles are left whole
};

struct ListScratch {
    int *ids;                    // BFS ids of the cells to visit, then the outcome bits
    unsigned long long *in;      // lanes that visit the cell, then those that accept it
    unsigned long long *open;    // lanes that open it
    int *list;                   // accepted cells in DFS order
    unsigned long long *mask;    // the lanes that accept them
    int cap;
};
constexpr int LW_ACC = 1 << 30, LW_LEAF = (int)(1u << 31), LW_ID = LW_ACC - 1;

// MAC tests of one cell against N targets from t0 on; bit k of the result:
// target t0 + k accepts.  The reference's arithmetic (BHgrav_accel.F90:154-158).
template <int MACT, int N, int NW>
__device__ __forceinline__ unsigned mac_bits(const ListWalk<NW> &L, int t0, const GMac &nd,
                                             double mac) {
    unsigned b = 0;
#pragma unroll 8
    for (int k = 0; k < N; k++) {
        const int t = t0 + k;
        const double dx = L.x[t] - nd.r[0], dy = L.y[t] - nd.r[1], dz = L.z[t] - nd.r[2];
        const double d2 = dist2_unfused(dx, dy, dz);
        bool ok = d2 > nd.dminsqd;
        if (MACT != SERENX_MAC_GEOMETRIC) ok = ok && d2 > mac * L.af[t];
        b = __builtin_amdgcn_alignbit(ok ? 1u : 0u, b, 1);
    }
    return b >> (32 - N);
}

// number of set bits before a bit
template <int NW>
__device__ __forceinline__ int lw_rank(const ListWalk<NW> &L, int which, int bit) {
    const int w = bit >> 5, g = w >> 2;
    int r = L.pre[which][g];
#pragma unroll
    for (int k = 0; k < 4; k++) {
        const unsigned v = L.bits[which][4 * g + k];
        if (4 * g + k < w) r += __popc(v);
        if (4 * g + k == w) r += __popc(v & ((1u << (bit & 31)) - 1u));
    }
    return r;
}

// What one walk of a block counts and needs in every level
struct LevelState {
    int ws, we;          // window
    unsigned nvalid;
    unsigned vis, lvis, ncell;
    int hi, slot;        // end of the level's entries, its counter
};

// The outcome of an entry on the lanes with lead set: am, om are the lanes of
// the group that accept the cell and that open it (mixed: 1 or 0).  The
// children of opened branches are appended, with one counter update per wave.
template <bool MIXED, int NW>
__device__ __forceinline__ void lw_outcome(ListWalk<NW> &L, const ListScratch &sc, LevelState &st,
                                           bool lead, int e, int id, const GMac &nd,
                                           unsigned long long in, unsigned long long am,
                                           unsigned long long om) {
    const int lane = (int)(threadIdx.x & (WAVE - 1));
    int kids = 0;
    if (lead) {
        int f = id;
        if (nd.c >= st.ws) {
            st.vis++;
            st.lvis += MIXED ? st.nvalid : (unsigned)__popcll(in);
            st.ncell += MIXED ? (am ? st.nvalid : 0u) : (unsigned)__popcll(am);
            const int bit = nd.c - st.ws;
            if (am) {
                f |= LW_ACC;
                atomicOr(&L.bits[0][bit >> 5], 1u << (bit & 31));
            }
            if (om && nd.k > 0) {
                f |= LW_LEAF;
                atomicOr(&L.bits[1][bit >> 5], 1u << (bit & 31));
            }
        }
        sc.ids[e] = f;
        if (!MIXED) {
            sc.in[e] = am;
            sc.open[e] = om;
        }
        if (om && nd.k < 0) kids = -nd.k;
    }
    if (!any_lane(kids != 0)) return;
    int at = kids;
#pragma unroll
    for (int d = 1; d < WAVE; d *= 2) {
        const int v = __shfl_up(at, d, WAVE);
        if (lane >= d) at += v;
    }
    int base = 0;
    if (lane == WAVE - 1) base = atomicAdd(&L.cnt[st.slot], at);
    base = st.hi + __shfl(base, WAVE - 1, WAVE) + at - kids;
    for (int k = 0; k < kids; k++)
        if (base + k < sc.cap) {
            sc.ids[base + k] = nd.fc + k;
            if (!MIXED) sc.in[base + k] = om;
        }
}

// One level's entries from lo on, one per lane, against the targets' sphere.
// Every target lies within rad of c, so its distance from the cell lies within
// rad of c's: the cell is accepted by all (opened by all) when that holds
// with 1e-9 to spare, which is far more than the tests' rounding.  Mixed: a
// cell that the first or the last target refuses is opened.  The other
// entries go to L.und.
template <bool MIXED, int MACT, int NW>
__device__ __forceinline__ void lw_sphere(ListWalk<NW> &L, const ListScratch &sc, LevelState &st,
                                          const GMac *__restrict__ gmac, double macscale, int lo) {
    const int lane = (int)(threadIdx.x & (WAVE - 1));
    const double rad = L.rad;
    for (int e = lo + (int)threadIdx.x; any_lane(e < st.hi); e += NW * WAVE) {
        bool has = e < st.hi;
        GMac nd{};
        int id = 0;
        if (has) {
            id = sc.ids[e];
            nd = gmac[id];
        }
        has = has && nd.c < st.we && nd.next > st.ws;
        unsigned long long in = 1;
        if (!MIXED && has) in = sc.in[e];
        const double mac = nd.mac * macscale;
        const double dx = L.c[0] - nd.r[0], dy = L.c[1] - nd.r[1], dz = L.c[2] - nd.r[2];
        const double d2 = dx * dx + dy * dy + dz * dz;
        double far2 = nd.dminsqd, near2 = nd.dminsqd;   // largest and smallest limit on d^2
        bool fine = true;
        if (MACT != SERENX_MAC_GEOMETRIC) {
            far2 = fmax(far2, mac * L.afmax);
            near2 = fmax(near2, mac * L.afmin);
            fine = mac < 1.0e300;
        }
        const double sf = (sqrt(far2) + rad) * (1.0 + 1.0e-9);
        const double sn = (sqrt(near2) - rad) * (1.0 - 1.0e-9);
        const bool all = fine && d2 > sf * sf;
        bool none = (fine && sn > 0.0 && d2 < sn * sn) || nd.k == 1;   // :128-136
        if (MIXED) {
#pragma unroll
            for (int t = 0; t < WAVE; t += WAVE - 1) {
                const double q2 = dist2_unfused(L.x[t] - nd.r[0], L.y[t] - nd.r[1],
                                                L.z[t] - nd.r[2]);
                bool ok = q2 > nd.dminsqd;
                if (MACT != SERENX_MAC_GEOMETRIC) ok = ok && q2 > mac * L.af[t];
                none = none || !ok;
            }
        }
        const bool und = has && !none && !all;
        lw_outcome<MIXED>(L, sc, st, has && !und, e, id, nd, in, none ? 0ull : in,
                          none ? in : 0ull);
        const unsigned long long um = ballot(und);
        if (um) {
            int base = 0;
            if (lane == 0) base = atomicAdd(&L.nund[st.slot], __popcll(um));
            base = __shfl(base, 0, WAVE);
            if (und)
                L.und[base + __popcll(um & ((1ull << lane) - 1ull))] = (unsigned short)e;
        }
    }
}

// The nu entries of L.und against every target, S lanes per entry
template <bool MIXED, int MACT, int S, int NW>
__device__ __forceinline__ void lw_targets(ListWalk<NW> &L, const ListScratch &sc, LevelState &st,
                                           const GMac *__restrict__ gmac, double macscale,
                                           int nu) {
    const int sub = (int)threadIdx.x % S;
    for (int u = (int)threadIdx.x / S; any_lane(u < nu); u += NW * WAVE / S) {
        const bool has = u < nu;
        GMac nd{};
        int id = 0, e = 0;
        unsigned long long in = 1, acc;
        if (has) {
            e = L.und[u];
            id = sc.ids[e];
            nd = gmac[id];
            if (!MIXED) in = sc.in[e];
        }
        const double mac = nd.mac * macscale;
        constexpr int N = WAVE / S;
        if (S == 1) {
            acc = (unsigned long long)mac_bits<MACT, 32>(L, 0, nd, mac) |
                  (unsigned long long)mac_bits<MACT, 32>(L, 32, nd, mac) << 32;
        } else {
            acc = (unsigned long long)mac_bits<MACT, (N < 32 ? N : 32)>(L, sub * N, nd, mac)
                  << (sub * N);
#pragma unroll
            for (int d = 1; d < S; d *= 2) acc |= __shfl_xor(acc, d, WAVE);
        }
        if (MIXED) acc = acc == ~0ull ? 1 : 0;
        lw_outcome<MIXED>(L, sc, st, has && sub == 0, e, id, nd, in, in & acc, in & ~acc);
    }
}

// (four waves per SIMD: two blocks of a CU hide each other's barriers)
//
// LEAN: registers for 6 (FP64) or 8 (mixed) waves per SIMD, where LDS admits
// four, and no raised priority.  The others are the h solve's: with 114 to 128
// registers the walk's two blocks filled a CU's register files, and where there
// are groups for every CU the h solve had to wait until the walk was done.  Some
// values are spilled (56 in FP64, 53 mixed).  Forests of 4,096 to 262,144
// particles a cloud, an evaluation: mixed 14.4M particles 194 -> 171 ms (walk
// and h solve beside each other 134 -> 107), FP64 6.1M 235 -> 219; one cloud,
// mixed uniform 131,071 4.1 -> 3.6, r^-2 390,000 10.4 -> 8.9, FP64 Plummer
// 200,000 10.5 -> 8.0, r^-2 16,384 1.80 -> 1.78.  FP64 walks of fewer groups than
// CUs, which leave the h solve room anyway, keep their registers (uniform 8,192:
// 1.19, 1.22 lean); mixed ones gain there too (1.03 -> 0.98).
template <bool MIXED, bool ORDERED, bool LEAN, int OCT, int MACT>
__global__ void __launch_bounds__(ORDERED ? OW_TB : LW_TB)
__attribute__((amdgpu_waves_per_eu(!LEAN ? 4 : MIXED ? 8 : 6))) k_grav_list(
    int nc, const GMac *__restrict__ gmac, double macscale, const GNode *__restrict__ gn,
    const GNodeF *__restrict__ gnf, const double *__restrict__ x,
    const double *__restrict__ y, const double *__restrict__ z, const int *__restrict__ cid,
    const int2 *__restrict__ root_range, const uint8_t *__restrict__ active,
    const double *__restrict__ gpot, const double *__restrict__ agm, double *__restrict__ cx,
    double *__restrict__ cy, double *__restrict__ cz, double *__restrict__ cp, NearList near,
    ListScratch all, unsigned long long *__restrict__ icount,
    unsigned long long *__restrict__ wstat, GroupQueue queue, int *__restrict__ cost,
    const int2 *__restrict__ grp, const int *__restrict__ cloud_off, LongWalks lw) {
    constexpr int NW = ORDERED ? OW_WAVES : LW_WAVES, NT = NW * WAVE;
    // (given at the launch: the compiler would keep the registers of no more waves
    // than its LDS admits)
    extern __shared__ double list_walk_lds[];
    ListWalk<NW> &L = *reinterpret_cast<ListWalk<NW> *>(list_walk_lds);
    // a round's factors [wave][dx, Q, H, ir5, ir7, crad, phi][lane]
    __shared__ double xc[ORDERED ? NW : 1][13][ORDERED ? WAVE : 1];
    // a walk of few groups is the critical path while the SPH kernels run beside
    // it: its waves take issue priority over theirs on shared SIMDs
    if (!LEAN) __builtin_amdgcn_s_setprio(2);
    const int tid = threadIdx.x, lane = tid & (WAVE - 1), wave = uniform(tid / WAVE);
    ListScratch sc = all;
    sc.ids += (size_t)blockIdx.x * all.cap;
    sc.in += (size_t)blockIdx.x * all.cap;
    sc.open += (size_t)blockIdx.x * all.cap;
    sc.list += (size_t)blockIdx.x * (all.cap + CELL_BATCH);
    sc.mask += (size_t)blockIdx.x * (all.cap + CELL_BATCH);
    LevelState st{};   // counts per thread
    const int home = blockIdx.x % NXCD;
    int qdone = 0;
    for (;;) {
        __syncthreads();   // the previous group's use of L
        if (wave == 0) {
            int g = -1;
            if (!lw.group) {
                g = next_group(queue, home, qdone);
            } else if (lane == 0) {
                const int t = atomicAdd(lw.taken, 1);
                if (t < *lw.n) g = lw.group[t];
            }
            if (lane == 0) L.job = g;
        }
        __syncthreads();
        const int g = uniform(L.job);
        if (g < 0) break;
        const int2 gr = grp[g];
        const int p = gr.x + lane;
        const bool valid = p < gr.y && active[p];
        const unsigned long long vmask = ballot(valid);
        if (vmask == 0) {
            if (tid == 0) {
                cost[g] = 0;
                near.len[g] = 0;
            }
            continue;
        }
        const unsigned nvalid = (unsigned)__popcll(vmask);
        // the other lanes repeat the first valid lane's target: they change
        // no vote and store nothing
        const int q = valid ? p : gr.x + __ffsll((long long)vmask) - 1;
        const double rpx = x[q], rpy = y[q], rpz = z[q];
        if (wave == 0) {
            const double af =
                MACT != SERENX_MAC_GEOMETRIC ? mac_afactor<MACT>(agm[q], gpot[q]) : 0.0;
            L.x[lane] = rpx;
            L.y[lane] = rpy;
            L.z[lane] = rpz;
            L.af[lane] = af;
            double lo[4] = {rpx, rpy, rpz, af}, hi[4] = {rpx, rpy, rpz, af};
#pragma unroll
            for (int d = 1; d < WAVE; d *= 2)
#pragma unroll
                for (int k = 0; k < (MACT != SERENX_MAC_GEOMETRIC ? 4 : 3); k++) {
                    lo[k] = fmin(lo[k], __shfl_xor(lo[k], d, WAVE));
                    hi[k] = fmax(hi[k], __shfl_xor(hi[k], d, WAVE));
                }
            double r2 = 0.0, slack = 0.0;   // slack: the rounding of the centre
#pragma unroll
            for (int k = 0; k < 3; k++) {
                const double half = 0.5 * (hi[k] - lo[k]);
                r2 += half * half;
                slack += 1.0e-15 * fmax(fabs(lo[k]), fabs(hi[k]));
                if (lane == 0) L.c[k] = lo[k] + half;
            }
            // an infinite or undefined factor decides nothing by the sphere
            const bool odd = any_lane(!(af < 1.0e300));
            if (lane == 0) {
                L.rad = odd ? 1.0e300 : sqrt(r2) * (1.0 + 1.0e-9) + slack;
                L.afmin = lo[3];
                L.afmax = hi[3];
            }
        }
        const int root = uniform(cid[q]);   // BFS id of the cloud's root
        const int2 rr = root_range[root];
        double gx = 0, gy = 0, gz = 0, gp = 0;   // the wave's share of the terms
        int len = 0, carry = 0;                  // near list so far; cells left of a batch
        int npage = 0;                           // pages of the near list
        bool dropped = false;                    // the near list did not fit
        int gvis = 0;
        const bool ordered = cloud_off[root + 1] - cloud_off[root] <= LW_ORDERED;
        if (!MIXED && ordered != ORDERED) continue;   // the other launch's group
        int ws = rr.x;
        if (lw.group) {   // the rest of a walk that one wave began
            ws = uniform(lw.at[g]);
            len = uniform(near.len[g]);
            dropped = len == NEAR_DROPPED;
            if (dropped) len = 0;
            npage = (len + PL_PAGE - 1) / PL_PAGE;
            gvis = uniform(cost[g]);
            if (wave == 0 && valid && !ordered) {   // (ordered walks begin here)
                gx = cx[p];
                gy = cy[p];
                gz = cz[p];
                gp = cp[p];
            }
        }
        int we = min(rr.y, ws + L.CELLS);
        while (ws < rr.y) {
            const int words = (we - ws + 127) / 128 * 4;
            for (int i = tid; i < words; i += NT) L.bits[0][i] = L.bits[1][i] = 0u;
            if (tid == 0) {
                sc.ids[0] = root;
                if (!MIXED) sc.in[0] = vmask;
                for (int k = 0; k < 3; k++) L.cnt[k] = L.nund[k] = 0;
            }
            st.ws = ws;
            st.we = we;
            st.nvalid = nvalid;
            __syncthreads();
            // step 1.  Three counters in turn: one is cleared only after
            // every wave has read it
            int lo = 0, hi = 1, slot = 0;
            const LevelState st0 = st;
            while (lo < hi && hi <= sc.cap) {
                st.hi = hi;
                st.slot = slot;
                lw_sphere<MIXED, MACT>(L, sc, st, gmac, macscale, lo);
                __syncthreads();
                const int nu = uniform(L.nund[slot]);
                if (nu) {
                    // the more lanes an entry has, the sooner it is done and
                    // the more is spent on it besides the tests
                    if (nu * 8 <= NT)
                        lw_targets<MIXED, MACT, 8>(L, sc, st, gmac, macscale, nu);
                    else if (nu * 2 <= NT)
                        lw_targets<MIXED, MACT, 2>(L, sc, st, gmac, macscale, nu);
                    else
                        lw_targets<MIXED, MACT, 1>(L, sc, st, gmac, macscale, nu);
                    __syncthreads();
                }
                lo = hi;
                hi = hi + uniform(L.cnt[slot]);
                const int old = slot == 0 ? 2 : slot - 1;
                if (tid == 0) L.cnt[old] = L.nund[old] = 0;
                slot = slot == 2 ? 0 : slot + 1;
            }
            if (hi > sc.cap) {   // too many entries: a window of half the cells
                st = st0;
                we = ws + (we - ws) / 2;
                __syncthreads();
                continue;
            }
            gvis += hi;
            // step 2
            int nacc = 0, nleaf = 0;
            {
                unsigned long long run = 0;   // accepted | leaves << 32, of groups of 128 cells
                for (int k0 = 0; k0 < words / 4; k0 += NT) {
                    const int k = k0 + tid;
                    unsigned long long v = 0;
                    if (k < words / 4) {
                        int a = 0, b = 0;
#pragma unroll
                        for (int i = 0; i < 4; i++) {
                            a += __popc(L.bits[0][4 * k + i]);
                            b += __popc(L.bits[1][4 * k + i]);
                        }
                        v = (unsigned)a | (unsigned long long)(unsigned)b << 32;
                    }
                    unsigned long long s = v;
#pragma unroll
                    for (int d = 1; d < WAVE; d *= 2) {
                        const unsigned long long o = __shfl_up(s, d, WAVE);
                        if (lane >= d) s += o;
                    }
                    if (lane == WAVE - 1) L.wsum[wave] = s;
                    __syncthreads();
                    unsigned long long before = run, sum = 0;
#pragma unroll
                    for (int w = 0; w < NW; w++) {
                        if (w < wave) before += L.wsum[w];
                        sum += L.wsum[w];
                    }
                    if (k < words / 4) {
                        const unsigned long long ex = before + s - v;
                        L.pre[0][k] = (int)(unsigned)ex;
                        L.pre[1][k] = (int)(ex >> 32);
                    }
                    run += sum;
                    __syncthreads();
                }
                nacc = uniform((int)(unsigned)run);
                nleaf = uniform((int)(run >> 32));
            }
            // pages for the leaves of this window
            const int pages = (len + nleaf + PL_PAGE - 1) / PL_PAGE;
            if (len + nleaf > near.cap) dropped = true;
            if (!dropped && pages > npage) {
                if (tid == 0) L.page0 = atomicAdd(near.next, pages - npage);
                __syncthreads();
                const int first = uniform(L.page0);
                if (first + pages - npage > near.npage)
                    dropped = true;
                else
                    for (int i = npage + tid; i < pages; i += NT)
                        near.page[(size_t)g * PL_PAGES + i] = first + i - npage;
                npage = pages;
                __syncthreads();
            }
            for (int e = tid; e < hi; e += NT) {
                const int f = sc.ids[e];
                if (!(f & (LW_ACC | LW_LEAF))) continue;
                const GMac &nd = gmac[f & LW_ID];
                const int bit = nd.c - ws;
                if (f & LW_ACC) {
                    const int r = carry + lw_rank(L, 0, bit);
                    sc.list[r] = nd.c;
                    if (!MIXED) sc.mask[r] = sc.in[e];
                }
                if ((f & LW_LEAF) && !dropped) {
                    const size_t at = near.slot(g, len + lw_rank(L, 1, bit));
                    near.leaf[at] = (nd.fc << 4) | nd.k;
                    near.mask[at] = MIXED ? vmask : sc.open[e];
                }
            }
            len += nleaf;
            __syncthreads();
            // step 3: whole batches, the last window's remainder too; each
            // wave takes a run of them
            const int have = carry + nacc;
            const bool last = we >= rr.y;
            const int nb = last ? (have + CELL_BATCH - 1) / CELL_BATCH : have / CELL_BATCH;
            const int i0 = (int)((long long)nb * wave / NW) * CELL_BATCH;
            const int i1 = min(have, (int)((long long)nb * (wave + 1) / NW) * CELL_BATCH);
            if (ordered) {
                const int n1 = min(have, nb * CELL_BATCH);
                float(*xb)[4][WAVE] = reinterpret_cast<float(*)[4][WAVE]>(L.bits);
                for (int j0 = 0; j0 < n1; j0 += WAVE) {
                    const int m = min(WAVE, n1 - j0);
                    const int mine = sc.list[j0 + min(lane, m - 1)];
                    if (MIXED) {
                        // wave w < 3 has component w of the acceleration, wave 3
                        // the potential (in gx); WAVE entries are at most LW_WAVES
                        // batches
                        static_assert(WAVE == CELL_BATCH * LW_WAVES, "a batch a wave");
                        float bx = 0.0f, by = 0.0f, bz = 0.0f, bp = 0.0f;
                        const int b0 = wave * CELL_BATCH;
                        for (int i = b0; i < min(m, b0 + CELL_BATCH); i++) {
                            const GNodeF nd = gnf[__builtin_amdgcn_readlane(mine, i)];
                            const float dr[3] = {(float)(rpx - nd.r[0]), (float)(rpy - nd.r[1]),
                                                 (float)(rpz - nd.r[2])};
                            cell_fp32<OCT>(nd, dr, bx, by, bz, bp);
                        }
                        xb[wave][0][lane] = bx;
                        xb[wave][1][lane] = by;
                        xb[wave][2][lane] = bz;
                        xb[wave][3][lane] = bp;
                        __syncthreads();
                        if (wave < 4)
                            for (int b = 0; b * CELL_BATCH < m; b++)
                                gx += (double)xb[b][wave][lane];
                        __syncthreads();
                    } else {
                        // wave w < 3: component w, wave 3: the potential (gx)
                        const unsigned long long mm = sc.mask[j0 + min(lane, m - 1)];
                        for (int r = 0; r < m; r += NW) {
                            if (r + wave < m) {
                                const GNode nd = gn[__builtin_amdgcn_readlane(mine, r + wave)];
                                const double dr[3] = {rpx - nd.r[0], rpy - nd.r[1],
                                                      rpz - nd.r[2]};
                                const double d2 = dist2_unfused(dr[0], dr[1], dr[2]);
                                const CellFactors f =
                                    cell_factors<OCT>(dr[0], dr[1], dr[2],
                                                      rsqrt_fp64(d2 + SMALL_NUMBER), nd.m, nd.q,
                                                      nd.oc);
#pragma unroll
                                for (int k = 0; k < 3; k++) {
                                    xc[wave][k][lane] = dr[k];
                                    xc[wave][3 + k][lane] = f.Q[k];
                                    if (OCT) xc[wave][6 + k][lane] = f.H[k];
                                }
                                xc[wave][9][lane] = f.ir5;
                                xc[wave][10][lane] = f.ir7;
                                xc[wave][11][lane] = f.crad;
                                xc[wave][12][lane] = f.phi;
                            }
                            __syncthreads();
                            if (wave < 4)
#pragma unroll
                                for (int k = 0; k < NW; k++) {
                                    if (r + k >= m) break;
                                    const int e = r + k;
                                    const unsigned long long em =
                                        (unsigned)__builtin_amdgcn_readlane((int)mm, e) |
                                        (unsigned long long)(unsigned)__builtin_amdgcn_readlane(
                                            (int)(mm >> 32), e) << 32;
                                    if (!__builtin_amdgcn_inverse_ballot_w64(em)) continue;
                                    if (wave == 3)
                                        gx = gx + xc[k][12][lane];
                                    else
                                        gx = add_cell<OCT>(gx, xc[k][3 + wave][lane],
                                                           xc[k][9][lane],
                                                           OCT ? xc[k][6 + wave][lane] : 0.0,
                                                           xc[k][10][lane], xc[k][11][lane],
                                                           xc[k][wave][lane]);
                                }
                            __syncthreads();
                        }
                    }
                }
            } else for (int j0 = i0; j0 < i1; j0 += WAVE) {
                const int m = min(WAVE, i1 - j0);
                const int mine = sc.list[j0 + min(lane, m - 1)];
                unsigned mlo = 0, mhi = 0;
                if (!MIXED) {
                    const unsigned long long mm = sc.mask[j0 + min(lane, m - 1)];
                    mlo = (unsigned)mm;
                    mhi = (unsigned)(mm >> 32);
                }
                if (MIXED) {
                    for (int b0 = 0; b0 < m; b0 += CELL_BATCH) {
                        float bx = 0.0f, by = 0.0f, bz = 0.0f, bp = 0.0f;
                        const int be = min(m, b0 + CELL_BATCH);
                        for (int i = b0; i < be; i++) {
                            const GNodeF nd = gnf[__builtin_amdgcn_readlane(mine, i)];
                            const float dr[3] = {(float)(rpx - nd.r[0]), (float)(rpy - nd.r[1]),
                                                 (float)(rpz - nd.r[2])};
                            cell_fp32<OCT>(nd, dr, bx, by, bz, bp);
                        }
                        gx += (double)bx; gy += (double)by; gz += (double)bz; gp += (double)bp;
                    }
                } else {
                    for (int i = 0; i < m; i++) {
                        const GNode nd = gn[__builtin_amdgcn_readlane(mine, i)];
                        const unsigned long long mm =
                            (unsigned)__builtin_amdgcn_readlane((int)mlo, i) |
                            (unsigned long long)(unsigned)__builtin_amdgcn_readlane((int)mhi, i)
                                << 32;
                        const double dr[3] = {rpx - nd.r[0], rpy - nd.r[1], rpz - nd.r[2]};
                        const double d2 = dist2_unfused(dr[0], dr[1], dr[2]);
                        if (__builtin_amdgcn_inverse_ballot_w64(mm)) cell_fp64<OCT>(nd, dr, d2, gx, gy, gz, gp);
                    }
                }
            }
            // the cells of an unfinished batch come first in the next window
            carry = have - min(have, nb * CELL_BATCH);
            int keep = 0;
            unsigned long long keepm = 0;
            if (tid < carry) {
                keep = sc.list[nb * CELL_BATCH + tid];
                if (!MIXED) keepm = sc.mask[nb * CELL_BATCH + tid];
            }
            __syncthreads();
            if (tid < carry) {
                sc.list[tid] = keep;
                if (!MIXED) sc.mask[tid] = keepm;
            }
            ws = we;
            we = min(rr.y, ws + L.CELLS);
        }
        if (ordered) {
            if (wave < 4 && valid) (wave == 0 ? cx : wave == 1 ? cy : wave == 2 ? cz : cp)[p] = gx;
        } else {
        // the waves' sums, added in wave order
        double *sum = reinterpret_cast<double *>(L.bits[0]);   // [component][wave][lane]
        sum[(0 * NW + wave) * WAVE + lane] = gx;
        sum[(1 * NW + wave) * WAVE + lane] = gy;
        sum[(2 * NW + wave) * WAVE + lane] = gz;
        sum[(3 * NW + wave) * WAVE + lane] = gp;
        __syncthreads();
        if (wave < 4) {
            double s = sum[wave * NW * WAVE + lane];
#pragma unroll
            for (int w = 1; w < NW; w++) s += sum[(wave * NW + w) * WAVE + lane];
            if (valid) (wave == 0 ? cx : wave == 1 ? cy : wave == 2 ? cz : cp)[p] = s;
        }
        }
        if (tid == 0) {
            cost[g] = gvis;
            near.len[g] = dropped ? NEAR_DROPPED : len;
        }
    }
#pragma unroll
    for (int d = 1; d < WAVE; d *= 2) {
        st.ncell += __shfl_xor(st.ncell, d, WAVE);
        st.vis += __shfl_xor(st.vis, d, WAVE);
        st.lvis += __shfl_xor(st.lvis, d, WAVE);
    }
    if (lane == 0) atomicAdd(ctr_row(icount) + 0, (unsigned long long)st.ncell);
    wave_stats(wstat, 0, st.vis, st.lvis);
}

// ---- the walk of one wave --------------------------------------------------
// In a cloud of more than LW_ALONE particles a wave walks for its group alone,
// up to LW_BUDGET visits; the list walk takes what is left, from the cell where
// the wave stopped.  With that many groups the waves hide each other's
// latency, and the walk by one wave issues slightly fewer instructions: an
// evaluation of an r^-2 sphere of 1M takes (waves / list walk, ms) 22.0 / 22.8
// mixed, 31.6 / 32.9 in FP64.  Elsewhere the list walk, with the registers it
// has now, is ahead: r^-2 12.4 / 11.5 at 524k, 10.0 / 9.3 at 400k (mixed), 17.4 /
// 17.0 and 13.9 / 13.3 (FP64); uniform 28.9 / 26.6 at 1M, 17.8 / 12.7 at 524k, 13.3
// / 10.4 at 400k (mixed); Plummer 39.4 / 37.1, 25.8 / 18.8, 20.1 / 15.0 (FP64).
// The line was drawn where the gains balanced when two blocks of the list walk
// filled a CU's registers (r^-2 12.7 / 13.8 at 524k, 9.7 / 10.9 at 400k, uniform
// 14.8 / 11.2 at 400k), and stays below the 1M steps that the knobs are tuned
// for, which have been measured by waves only.  The budget keeps the
// long walks of a large uniform cloud from their waves (1M: 75 -> 30 ms;
// budgets of 3,000, 8,192 and 16,384 differ by 2 % there, and 3,000 costs the
// r^-2 sphere 10 %).
// The near list of the group that a wave walks (wave-uniform): entries found
// and the page that takes the next ones, -1 once none could be had
struct NearWriter {
    int len = 0, page = 0;
    __device__ __forceinline__ void append(const NearList &L, int g, int first, int count,
                                           unsigned long long mask) {
        if (len % PL_PAGE == 0 && page >= 0) {
            int pg = L.npage;
            if (len < PL_PAGES * PL_PAGE && (threadIdx.x & 63) == 0) pg = atomicAdd(L.next, 1);
            page = uniform(pg);
            if (page >= L.npage)
                page = -1;
            else if ((threadIdx.x & 63) == 0)
                L.page[(size_t)g * PL_PAGES + len / PL_PAGE] = page;
        }
        if (page >= 0 && (threadIdx.x & 63) == 0) {
            const size_t at = (size_t)page * PL_PAGE + len % PL_PAGE;
            L.leaf[at] = (first << 4) | count;
            L.mask[at] = mask;
        }
        len++;
    }
    __device__ __forceinline__ int stored(const NearList &L) const {
        return page < 0 || len > L.cap ? NEAR_DROPPED : len;
    }
};

// visits that one wave may make for its group: none in a small cloud
__device__ __forceinline__ unsigned walk_budget(const LongWalks &lw, bool valid, int p,
                                                const int *__restrict__ cid,
                                                const int *__restrict__ cloud_off) {
    const unsigned long long vm = ballot(valid);
    if (vm == 0) return 0;
    const int k = __builtin_amdgcn_readlane(valid ? cid[p] : 0, __ffsll((long long)vm) - 1);
    return cloud_off[k + 1] - cloud_off[k] > lw.alone ? (unsigned)lw.budget : 0u;
}

template <int OCT, int MACT>
__global__ void __launch_bounds__(256) k_grav_cells_fp64(
    int nc, const GNode *__restrict__ gn, const double *__restrict__ x,
    const double *__restrict__ y, const double *__restrict__ z, const int *__restrict__ cid,
    const int2 *__restrict__ root_range, const uint8_t *__restrict__ active,
    const double *__restrict__ gpot, const double *__restrict__ agm, double *__restrict__ cx,
    double *__restrict__ cy, double *__restrict__ cz, double *__restrict__ cp, NearList near,
    unsigned long long *__restrict__ icount, unsigned long long *__restrict__ wstat,
    GroupQueue queue, int *__restrict__ cost, const int2 *__restrict__ grp,
    const int *__restrict__ cloud_off, LongWalks lw) {
    // the walk is the critical path while the SPH kernels run beside it: its
    // waves take issue priority over theirs on shared SIMDs
    __builtin_amdgcn_s_setprio(2);
    unsigned ncell = 0, vis = 0, lvis = 0;   // wave totals
    const int home = blockIdx.x % NXCD;
    int qdone = 0;
    for (int g = next_group(queue, home, qdone); g >= 0; g = next_group(queue, home, qdone)) {
        const int2 gr = grp[g];
        const int p = gr.x + (int)(threadIdx.x & (WAVE - 1));
        const bool valid = p < gr.y && active[p];
        double rpx = 0, rpy = 0, rpz = 0, afactor = 0.0;
        if (valid) {
            rpx = x[p]; rpy = y[p]; rpz = z[p];
            if (MACT != SERENX_MAC_GEOMETRIC) afactor = mac_afactor<MACT>(agm[p], gpot[p]);
        }
        double gx = 0, gy = 0, gz = 0, gp = 0;
        NearWriter nw;
        const int2 rr = valid ? root_range[cid[p]] : make_int2(nc, nc);
        const unsigned budget = walk_budget(lw, valid, p, cid, cloud_off);
        unsigned gv = 0;
        int resume = valid ? rr.x : nc;
        int c = uniform(wave_min_int(resume));
        while (c < nc && gv < budget) {
            gv++;
            group_step(gn, nc, rr.y, c, resume, lvis,
            [&](const GNode &nd, bool here) -> int {
                const double dr[3] = {rpx - nd.r[0], rpy - nd.r[1], rpz - nd.r[2]};
                const double drsqd = dr[0] * dr[0] + dr[1] * dr[1] + dr[2] * dr[2];
                bool accept;
                if (MACT == SERENX_MAC_GEOMETRIC)
                    accept = drsqd > nd.dminsqd;
                else
                    accept = drsqd > nd.mac * afactor && drsqd > nd.dminsqd;
                accept = accept && nd.leaf != 1;                   // :128-136, no MAC test
                ncell += lanes(here && accept);
                if (here && accept) cell_fp64<OCT>(nd, dr, drsqd, gx, gy, gz, gp);
                if (accept) return WALK_SKIP;
                return nd.leaf > 0 ? WALK_LEAF : WALK_DESCEND;     // :242-258
            },
            [&](const GNode &nd, bool mine) {
                nw.append(near, g, nd.first, nd.leaf, ballot(mine));
            });
        }
        vis += gv;
        if ((threadIdx.x & 63) == 0) {
            cost[g] = (int)gv;
            near.len[g] = nw.stored(near);
            if (c < nc) {
                lw.at[g] = c;
                lw.group[atomicAdd(lw.n, 1)] = g;
            }
        }
        if (valid) {
            cx[p] = gx;
            cy[p] = gy;
            cz[p] = gz;
            cp[p] = gp;
        }
    }
    if ((threadIdx.x & 63) == 0) atomicAdd(ctr_row(icount) + 0, (unsigned long long)ncell);
    wave_stats(wstat, 0, vis, lvis);
}

template <int OCT, int MACT>
__global__ void __launch_bounds__(256) k_grav_cells_mixed(
    int nc, const GNodeF *__restrict__ gn, const double *__restrict__ x,
    const double *__restrict__ y, const double *__restrict__ z, const int *__restrict__ cid,
    const int2 *__restrict__ root_range, const uint8_t *__restrict__ active,
    const double *__restrict__ gpot, const double *__restrict__ agm, double *__restrict__ ox,
    double *__restrict__ oy, double *__restrict__ oz, double *__restrict__ op, NearList near,
    unsigned long long *__restrict__ icount, unsigned long long *__restrict__ wstat,
    GroupQueue queue, int *__restrict__ cost, const int2 *__restrict__ grp,
    const int *__restrict__ cloud_off, LongWalks lw) {
    __builtin_amdgcn_s_setprio(2);
    unsigned ncell = 0, vis = 0, lvis = 0;   // wave totals
    const int home = blockIdx.x % NXCD;
    int qdone = 0;
    for (int g = next_group(queue, home, qdone); g >= 0; g = next_group(queue, home, qdone)) {
        const int2 gr = grp[g];
        const int p = gr.x + (int)(threadIdx.x & (WAVE - 1));
        const bool valid = p < gr.y && active[p];
        double rpx = 0, rpy = 0, rpz = 0, afactor = 0.0;
        if (valid) {
            rpx = x[p]; rpy = y[p]; rpz = z[p];
            if (MACT != SERENX_MAC_GEOMETRIC) afactor = mac_afactor<MACT>(agm[p], gpot[p]);
        }
        double cx = 0.0, cy = 0.0, cz = 0.0, cp = 0.0;   // cell terms
        float bx = 0.0f, by = 0.0f, bz = 0.0f, bp = 0.0f; // current batch of cell terms
        int nbatch = 0;                                   // wave-uniform
        NearWriter nw;
        unsigned gv = 0;
        // the walk covers the tree of the group's cloud (groups never straddle
        // clouds); every valid lane takes part at every cell, and the cell
        // terms of the other lanes are formed and never stored
        const unsigned long long vmask = ballot(valid);
        const unsigned nvalid = (unsigned)__popcll(vmask);
        const int2 rr = valid ? root_range[cid[p]] : make_int2(nc, nc);
        int c = uniform(wave_min_int(valid ? rr.x : nc));
        const int cend = uniform(wave_max_int(valid ? rr.y : 0));
        const unsigned budget = walk_budget(lw, valid, p, cid, cloud_off);
        int stop = budget ? cend : c;   // the walk ends here
        while (c < stop) {
            const GNodeF nd = gn[c];
            gv++;
            lvis += nvalid;
            double d0, d1, d2;
            if (group_accepts<MACT>(nd, vmask, rpx, rpy, rpz, afactor, d0, d1, d2)) {
                ncell += nvalid;
                const float dr[3] = {(float)d0, (float)d1, (float)d2};
                cell_fp32<OCT>(nd, dr, bx, by, bz, bp);
                if (++nbatch == CELL_BATCH) {
                    cx += (double)bx; cy += (double)by; cz += (double)bz; cp += (double)bp;
                    bx = by = bz = bp = 0.0f;
                    nbatch = 0;
                    if (gv >= budget) stop = 0;   // only between batches
                }
                c = nd.next;
            } else if (nd.leaf > 0) {
                nw.append(near, g, nd.first, nd.leaf, vmask);
                c = nd.next;
            } else {
                c = c + 1;
            }
        }
        cx += (double)bx; cy += (double)by; cz += (double)bz; cp += (double)bp;
        vis += gv;
        if ((threadIdx.x & 63) == 0) {
            cost[g] = (int)gv;
            near.len[g] = nw.stored(near);
            if (c < cend) {
                lw.at[g] = c;
                lw.group[atomicAdd(lw.n, 1)] = g;
            }
        }
        if (valid) {
            ox[p] = cx;
            oy[p] = cy;
            oz[p] = cz;
            op[p] = cp;
        }
    }
    if ((threadIdx.x & 63) == 0) atomicAdd(ctr_row(icount) + 0, (unsigned long long)ncell);
    wave_stats(wstat, 0, vis, lvis);
}

// The mixed pair phase: a block of PM_WAVES waves takes a group; each wave
// has all its targets, one per lane, and takes the list's batches of PL_STAGE
// leaves (staged in LDS) in turn.  The waves' compensated sums are added in
// wave order at the end, in FP64.  One wave per group left the longest lists
// (5,000 to 20,000 leaves at the centre of a uniform sphere) to one wave:
// r^-2 sphere of 16,384 particles 957 -> 163 us, uniform sphere of 1M 27.3 ->
// 4.6 ms, r^-2 sphere of 1M, which fills the device, 3.1 ms either way.
constexpr int PL_STAGE = 16;
constexpr int PM_WAVES = 8;
constexpr int PM_LEAVES = 4;   // leaves per wave and round of ordered sums

template <int MACT, bool QUINTIC, int NW>
__device__ __forceinline__ void pairs_group_mixed(
    int g, int wave, int nc, const GNodeF *__restrict__ gn, const float4 *__restrict__ rec,
    float4 *__restrict__ stage, double *__restrict__ sums, float *__restrict__ xsum,
    const int *__restrict__ cloud_off,
    const double *__restrict__ x, const double *__restrict__ y, const double *__restrict__ z,
    const double *__restrict__ h, const double *__restrict__ zeta,
    const int *__restrict__ cid, const int2 *__restrict__ root_range,
    const uint8_t *__restrict__ active, const float4 *__restrict__ t4,
    double *__restrict__ ax, double *__restrict__ ay, double *__restrict__ az,
    const double *__restrict__ cpot, double *__restrict__ gpot, double *__restrict__ agm,
    NearList near, const int2 *__restrict__ grp, unsigned &npp_out, unsigned &nin_p_out,
    unsigned &nin_j_out) {
    constexpr int SHARES = PM_WAVES / NW;   // a wave's, taken one after the other
    static_assert(SHARES <= 2, "one share's sums held");
    constexpr KGeom kg64 = walk_geom<QUINTIC>();
    constexpr KGeomF kg{(float)kg64.half, (float)kg64.range, (float)kg64.invrange};
    const int lane = (int)(threadIdx.x & (WAVE - 1));
    const int2 gr = grp[g];
    const int p = gr.x + lane;
    const bool valid = p < gr.y && active[p];
    if (ballot(valid) == 0) return;   // the whole block
    double rpx = 0, rpy = 0, rpz = 0, afactor = 0.0;
    PairTarget tp{1.0f, 1.0f, 0.0f, 0.0f, 0.0f};
    if (valid) {
        rpx = x[p]; rpy = y[p]; rpz = z[p];
        const double ih = 1.0 / h[p];
        tp.ih = (float)ih;
        tp.ih2 = (float)(ih * ih);
        tp.zi2 = (float)(zeta[p] * ih * ih);
        tp.lim = (float)(kg64.invrange * ih);
        tp.hk = (float)(kg64.half * ih);
        if (MACT != SERENX_MAC_GEOMETRIC) afactor = mac_afactor<MACT>(agm[p], gpot[p]);
    }
    CSum px, py, pz, pq;   // pair terms, one compensated addition per leaf
    double held[4] = {0.0, 0.0, 0.0, 0.0};   // the first share's sums
    unsigned npp = 0, nin_p = 0, nin_j = 0;
    auto leaf_pairs = [&](int first, int count, bool mine) {
        // r_f - r_p in FP64, once per leaf (r_f: the leaf's first particle)
        const float ox = (float)(x[first] - rpx), oy = (float)(y[first] - rpy),
                    oz = (float)(z[first] - rpz);
        float bx = 0.0f, by = 0.0f, bz = 0.0f, bp = 0.0f;
        const unsigned long long mm = ballot(mine);
        // the next source's record is loaded (scalar loads) before the
        // current pair is formed; after the leaf's last particle that is
        // particle first + count <= n, within the buffer's n + 1 records
        float4 a = rec[2 * (size_t)first], b = rec[2 * (size_t)first + 1];
        for (int i = 0; i < count; i++) {
            const int j = first + i;
            const float4 an = rec[2 * (size_t)(j + 1)], bn = rec[2 * (size_t)(j + 1) + 1];
            // the lanes taking the pair: those that opened the leaf, less the
            // one whose particle is j
            const unsigned sl = (unsigned)(j - gr.x);
            const unsigned long long mact = mm & ~(sl < WAVE ? 1ull << sl : 0ull);
            npp += (unsigned)__popcll(mact);
            pair_f32(kg, t4, tp, mine && j != p, mact, a.x + ox, a.y + oy, a.z + oz, a.w, b.x,
                     b.y, b.z, b.w, bx, by, bz, bp, nin_p, nin_j);
            a = an;
            b = bn;
        }
        if (mine) {
            px.add(bx);
            py.add(by);
            pz.add(bz);
            pq.add(bp);
        }
    };
    // one leaf's sums over the valid lanes, stored (ordered sums)
    auto leaf_sums = [&](const float4 *src, int first, int count, float *out) {
        const float ox = (float)(x[first] - rpx), oy = (float)(y[first] - rpy),
                    oz = (float)(z[first] - rpz);
        float bx = 0.0f, by = 0.0f, bz = 0.0f, bp = 0.0f;
        const unsigned long long mm = ballot(valid);
        for (int i = 0; i < count; i++) {
            const int j = first + i;
            const float4 a = src[2 * i], b = src[2 * i + 1];
            const unsigned sl = (unsigned)(j - gr.x);
            const unsigned long long mact = mm & ~(sl < WAVE ? 1ull << sl : 0ull);
            npp += (unsigned)__popcll(mact);
            pair_f32(kg, t4, tp, valid && j != p, mact, a.x + ox, a.y + oy, a.z + oz, a.w, b.x,
                     b.y, b.z, b.w, bx, by, bz, bp, nin_p, nin_j);
        }
        wave_lds_fence();   // the last leaf's sums take the stage's place
        out[0 * WAVE] = bx;
        out[1 * WAVE] = by;
        out[2 * WAVE] = bz;
        out[3 * WAVE] = bp;
    };
    // the same terms with the leaf's records read from the wave's LDS stage
    // (src: the leaf's LEAFMAX slots of two float4)
    auto leaf_pairs_staged = [&](const float4 *src, int first, int count, bool mine) {
        const float ox = (float)(x[first] - rpx), oy = (float)(y[first] - rpy),
                    oz = (float)(z[first] - rpz);
        float bx = 0.0f, by = 0.0f, bz = 0.0f, bp = 0.0f;
        const unsigned long long mm = ballot(mine);
        for (int i = 0; i < count; i++) {
            const int j = first + i;
            const float4 a = src[2 * i], b = src[2 * i + 1];
            const unsigned sl = (unsigned)(j - gr.x);
            const unsigned long long mact = mm & ~(sl < WAVE ? 1ull << sl : 0ull);
            npp += (unsigned)__popcll(mact);
            pair_f32(kg, t4, tp, mine && j != p, mact, a.x + ox, a.y + oy, a.z + oz, a.w, b.x,
                     b.y, b.z, b.w, bx, by, bz, bp, nin_p, nin_j);
        }
        if (mine) {
            px.add(bx);
            py.add(by);
            pz.add(bz);
            pq.add(bp);
        }
    };
    const int len = uniform(near.len[g]);
    const int root =
        __builtin_amdgcn_readlane(valid ? cid[p] : 0, __ffsll((long long)ballot(valid)) - 1);
    const bool ordered = cloud_off[root + 1] - cloud_off[root] <= LW_ORDERED;
    auto stored_pairs = [&](int share) {
        // the near list in batches of PL_STAGE leaves: lane l copies the
        // records of the batch's leaf l into the wave's LDS stage (all the
        // batch's loads in flight at once), then the wave forms the pairs
        // leaf by leaf in list order from LDS
        for (int e0 = share * PL_STAGE; e0 < len; e0 += PM_WAVES * PL_STAGE) {
            const int nb = min(PL_STAGE, len - e0);
            const size_t at = near.slot(g, e0);   // a batch lies in one page
            int dl = 0;
            if (lane < nb) {
                dl = near.leaf[at + lane];
                const int f = dl >> 4, k = dl & 15;
                float4 *dst = stage + 2 * LEAFMAX * lane;
                for (int i = 0; i < k; i++) {
                    dst[2 * i] = rec[2 * (size_t)(f + i)];
                    dst[2 * i + 1] = rec[2 * (size_t)(f + i) + 1];
                }
            }
            wave_lds_fence();   // lanes read other lanes' slots
            for (int e = 0; e < nb; e++) {
                const int d = __builtin_amdgcn_readlane(dl, e);
                const unsigned long long m = near.mask[at + e];
                leaf_pairs_staged(stage + 2 * LEAFMAX * e, d >> 4, d & 15,
                                  valid && ((m >> lane) & 1ull));
            }
            wave_lds_fence();   // every read before the next batch's writes
        }
    };
    auto walked_pairs = [&](int share) {
        // the list was not stored: the same wave-uniform walk again, pairs of
        // the share's batches only
        int e = 0;
        const int2 rr = valid ? root_range[cid[p]] : make_int2(nc, nc);
        int c = uniform(wave_min_int(valid ? rr.x : nc));
        const int cend = uniform(wave_max_int(valid ? rr.y : 0));
        const unsigned long long vmask = ballot(valid);
        while (c < cend) {
            const GNodeF nd = gn[c];
            double d0, d1, d2;
            if (group_accepts<MACT>(nd, vmask, rpx, rpy, rpz, afactor, d0, d1, d2)) {
                c = nd.next;
            } else if (nd.leaf > 0) {
                if ((ordered ? 0 : e / PL_STAGE % PM_WAVES) == share)
                    leaf_pairs(nd.first, nd.leaf, valid);
                e++;
                c = nd.next;
            } else {
                c = c + 1;
            }
        }
    };
    if (ordered && len != NEAR_DROPPED) {
        // PM_LEAVES leaves per wave and round; their sums go to the four waves
        // that add them in list order, one component each (px).  The sums fill
        // the waves' LDS; the leaves are staged where the last one's sums go
        float4 *last = stage + (PM_LEAVES - 1) * WAVE;
        for (int r = 0; r < len; r += NW * PM_LEAVES) {
            const int e0 = r + wave * PM_LEAVES, nb = max(0, min(PM_LEAVES, len - e0));
            int dl = 0;
            if (lane < nb) {
                dl = near.leaf[near.slot(g, e0) + lane];   // in one page
                const int f = dl >> 4, k = dl & 15;
                float4 *dst = last + 2 * LEAFMAX * lane;
                for (int i = 0; i < k; i++) {
                    dst[2 * i] = rec[2 * (size_t)(f + i)];
                    dst[2 * i + 1] = rec[2 * (size_t)(f + i) + 1];
                }
            }
            wave_lds_fence();
            for (int e = 0; e < nb; e++) {
                const int d = __builtin_amdgcn_readlane(dl, e);
                leaf_sums(last + 2 * LEAFMAX * e, d >> 4, d & 15,
                          xsum + ((wave * PM_LEAVES + e) * 4) * WAVE + lane);
            }
            __syncthreads();
            if (wave < 4)
                for (int e = 0; e < min(NW * PM_LEAVES, len - r); e++)
                    px.add(xsum[(e * 4 + wave) * WAVE + lane]);
            __syncthreads();
        }
    } else {
        // the wave's shares of the list: the batches of PL_STAGE leaves go to
        // PM_WAVES shares in turn
        for (int share = wave; share < PM_WAVES; share += NW) {
            if (share != wave) {
                held[0] = px.value();
                held[1] = py.value();
                held[2] = pz.value();
                held[3] = pq.value();
                px = py = pz = pq = CSum{};
            }
            if (len != NEAR_DROPPED)
                stored_pairs(share);
            else
                walked_pairs(share);
        }
    }
    // every wave is done with its stage and with the previous |a|
    __syncthreads();
    const int at = wave + PM_WAVES - NW;   // the last share (ordered: the wave's sum)
    sums[(at * 4 + 0) * WAVE + lane] = px.value();
    sums[(at * 4 + 1) * WAVE + lane] = py.value();
    sums[(at * 4 + 2) * WAVE + lane] = pz.value();
    sums[(at * 4 + 3) * WAVE + lane] = pq.value();
    if (SHARES > 1)
        for (int k = 0; k < 4; k++) sums[(wave * 4 + k) * WAVE + lane] = held[k];
    __syncthreads();
    if (wave == 0 && valid) {
        double gx = ax[p], gy = ay[p], gz = az[p], gp = cpot[p];
        if (ordered && len != NEAR_DROPPED) {   // component w is wave w's px
            gx += sums[((at + 0) * 4 + 0) * WAVE + lane];
            gy += sums[((at + 1) * 4 + 0) * WAVE + lane];
            gz += sums[((at + 2) * 4 + 0) * WAVE + lane];
            gp += sums[((at + 3) * 4 + 0) * WAVE + lane];
        } else for (int w = 0; w < (ordered ? 1 : PM_WAVES); w++) {
            gx += sums[(w * 4 + 0) * WAVE + lane];
            gy += sums[(w * 4 + 1) * WAVE + lane];
            gz += sums[(w * 4 + 2) * WAVE + lane];
            gp += sums[(w * 4 + 3) * WAVE + lane];
        }
        ax[p] = gx;   // the gravity acceleration; k_add_grav adds it to a
        ay[p] = gy;
        az[p] = gz;
        gpot[p] = gp;
        if (MACT != SERENX_MAC_GEOMETRIC) agm[p] = sqrt(gx * gx + gy * gy + gz * gz);
    }
    npp_out += npp;
    nin_p_out += nin_p;
    nin_j_out += nin_j;
}

template <int MACT, bool QUINTIC, int NW>
__global__ void __launch_bounds__(NW * WAVE) k_grav_pairs_mixed(
    int nc, const GNodeF *__restrict__ gn, const float4 *__restrict__ rec,
    const double *__restrict__ x, const double *__restrict__ y, const double *__restrict__ z,
    const double *__restrict__ h, const double *__restrict__ zeta,
    const int *__restrict__ cid, const int2 *__restrict__ root_range,
    const uint8_t *__restrict__ active, const float4 *__restrict__ t4,
    double *__restrict__ ax, double *__restrict__ ay, double *__restrict__ az,
    const double *__restrict__ cpot, double *__restrict__ gpot, double *__restrict__ agm,
    NearList near, unsigned long long *__restrict__ icount, const int2 *__restrict__ grp,
    const int *__restrict__ cloud_off, GroupQueue queue) {
    // persistent over the walk's queue: the groups of each XCD range
    // longest-first (by the previous walk's cost), as phase 1 takes them
    __builtin_amdgcn_s_setprio(2);
    // each wave's LDS stage: PL_STAGE leaves of LEAFMAX two-float4 records;
    // in its place the leaves' sums where they are added in list order, and the
    // waves' sums at the end
    __shared__ float4 stage_all[NW * PL_STAGE * LEAFMAX * 2];
    static_assert(sizeof(stage_all) >= sizeof(double) * 4 * PM_WAVES * WAVE, "sums fit");
    static_assert(sizeof(stage_all) == sizeof(float) * NW * PM_LEAVES * 4 * WAVE &&
                      PM_LEAVES * LEAFMAX * 2 <= WAVE, "leaves' sums fit, their stage in one's");
    __shared__ int job;
    const int wave = uniform((int)(threadIdx.x / WAVE));
    float4 *stage = stage_all + wave * (PL_STAGE * LEAFMAX * 2);
    unsigned npp = 0, nin_p = 0, nin_j = 0;   // wave totals
    const int home = blockIdx.x % NXCD;
    int qdone = 0;
    for (;;) {
        __syncthreads();
        if (wave == 0) {
            const int t = next_group(queue, home, qdone);
            if (threadIdx.x == 0) job = t;
        }
        __syncthreads();
        const int g = uniform(job);
        if (g < 0) break;
        pairs_group_mixed<MACT, QUINTIC, NW>(
            g, wave, nc, gn, rec, stage, reinterpret_cast<double *>(stage_all),
            reinterpret_cast<float *>(stage_all), cloud_off, x, y, z, h, zeta, cid, root_range,
            active, t4, ax, ay, az, cpot, gpot, agm, near, grp, npp, nin_p, nin_j);
    }
    if ((threadIdx.x & 63) == 0) {
        unsigned long long *ic = ctr_row(icount);
        atomicAdd(ic + 1, (unsigned long long)npp);
        atomicAdd(ic + 2, (unsigned long long)nin_p);
        atomicAdd(ic + 3, (unsigned long long)nin_j);
    }
}

// Work-queue order of the walk's groups: keys (range, ~cost) so that an
// ascending sort lists every XCD range's groups by decreasing cost of their
// previous walk; with no cost yet the keys are the ranges alone (a stable
// sort keeps tree order within each)
__global__ void k_queue_keys(int ngroups, const int *__restrict__ cost, int have_cost,
                             uint64_t *__restrict__ keys, int *__restrict__ vals) {
    const int g = blockIdx.x * blockDim.x + threadIdx.x;
    if (g >= ngroups) return;
    const uint64_t range = (uint64_t)(((long long)NXCD * g) / ngroups);
    const uint32_t c = have_cost ? (uint32_t)max(cost[g], 0) : 0u;
    keys[g] = (range << 32) | (uint64_t)(0xFFFFFFFFu - c);
    vals[g] = g;
}

// the queue in tree order (each XCD range's groups in order)
__global__ void k_queue_identity(int ngroups, int *__restrict__ order) {
    const int g = blockIdx.x * blockDim.x + threadIdx.x;
    if (g < ngroups) order[g] = g;
}

__global__ void k_zero_ints(int n, int *__restrict__ a) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) a[i] = 0;
}

// direct_sph_gravity.F90:63-79: sum of gravity_gradh over all other
// particles, FP64, sources staged through LDS
__global__ void __launch_bounds__(256) k_direct(KGeom kg, int n, int nt,
                                                const int *__restrict__ targets,
                                                const double *__restrict__ x,
                                                const double *__restrict__ y,
                                                const double *__restrict__ z,
                                                const double *__restrict__ m,
                                                const double *__restrict__ h,
                                                const double *__restrict__ zeta,
                                                const int *__restrict__ cid,
                                                const int *__restrict__ cloud_off,
                                                const double4 *__restrict__ t4,
                                                double *__restrict__ acc, double *__restrict__ pot) {
    __shared__ double sx[256], sy[256], sz[256], sm[256], sh[256], sih[256], szt[256];
    const int t = blockIdx.x * blockDim.x + threadIdx.x;
    const bool valid = t < nt;
    const int p = valid ? targets[t] : 0;
    const double rpx = x[p], rpy = y[p], rpz = z[p], invhp = 1.0 / h[p], zo_p = zeta[p];
    // sources: the target's own cloud
    const int lo = cloud_off[cid[p]], hi = cloud_off[cid[p] + 1];
    double gx = 0, gy = 0, gz = 0, gp = 0;
    for (int base = 0; base < n; base += 256) {
        const int j = base + threadIdx.x;
        if (j < n) {
            sx[threadIdx.x] = x[j];
            sy[threadIdx.x] = y[j];
            sz[threadIdx.x] = z[j];
            sm[threadIdx.x] = m[j];
            sh[threadIdx.x] = kg.range * h[j];
            sih[threadIdx.x] = 1.0 / h[j];
            szt[threadIdx.x] = zeta[j];
        }
        __syncthreads();
        const int lim = min(256, n - base);
        if (valid) {
            for (int k = 0; k < lim; k++) {
                if (base + k == p || base + k < lo || base + k >= hi) continue;
                (void)pair_fp64(kg, t4, invhp, zo_p, sx[k] - rpx, sy[k] - rpy, sz[k] - rpz, sm[k],
                          sh[k], sih[k], szt[k], gx, gy, gz, gp);
            }
        }
        __syncthreads();
    }
    if (valid) {
        acc[3 * t] = gx;
        acc[3 * t + 1] = gy;
        acc[3 * t + 2] = gz;
        pot[t] = gp;
    }
}

// Blocks per CU of the walk launch: the knob's value (default: as many as
// fit).  Fewer blocks leave wave slots to the SPH kernels that run beside
// the walk; the device's vector ALUs are the bound both share, and the best
// split depends on the workload (seren_amd/autotune.py times a few
// candidates on it).  A walk with nothing beside it (serenx_grav_forces)
// takes all that fit.
int walk_cap(const Ctx &c) { return c.walk_alone ? 64 : c.walk_queue; }

// Blocks per CU of the pair phase: its own knob when set.  The pair phase
// runs beside the neighbour and hydro kernels, which need less of the
// device than the h solve beside the cell phase.
int pair_cap(const Ctx &c) {
    if (c.walk_alone) return 64;
    return c.pair_blocks > 0 ? c.pair_blocks : c.walk_queue;
}

// Blocks of a walk launch that has `groups` groups per block at a time: as many
// as the device holds at once and at most cap per CU, where the knob counts
// blocks of TB threads (rounded up to whole blocks: at 3 of them the pair phase
// of a mixed 1M step keeps 16 waves a CU: 14.8 ms, 16.1 with the 8 of rounding
// down, each one run).
template <class K>
int walk_blocks(Ctx &c, K kernel, int cap, int tb, int groups = 1, size_t lds = 0) {
    int per_cu = 0;
    if (hipOccupancyMaxActiveBlocksPerMultiprocessor(&per_cu, kernel, tb, lds) != hipSuccess ||
        per_cu <= 0)
        per_cu = 1;
    if (c.walk_queue != 0) per_cu = std::min(per_cu, (cap * TB + tb - 1) / tb);
    return std::max(1, std::min((c.gq.ngroups + groups - 1) / groups, per_cu * c.ncu));
}

// near_cap bounds a group's list; its largest value leaves that to the pool
NearList near_list(Ctx &c) {
    const int cap = c.near_cap < PL_CAP ? c.near_cap : PL_PAGES * PL_PAGE;
    return NearList{c.pl_leaf, c.pl_mask, c.pl_page, c.gq.ctr + 2 * NXCD, c.pl_len, cap,
                    c.pl_npage};
}

// particles of the smallest and the largest cloud
void cloud_sizes(const Ctx &c, int &least, int &most) {
    least = most = c.cloud_off_h[1] - c.cloud_off_h[0];
    for (int i = 1; i < c.ncloud; i++) {
        least = std::min(least, c.cloud_off_h[i + 1] - c.cloud_off_h[i]);
        most = std::max(most, c.cloud_off_h[i + 1] - c.cloud_off_h[i]);
    }
}

// phase 1 of the walk (traversal and cell terms), persistent over the
// queue, on stream s with at most cap blocks per CU
template <int OCT, int MACT>
void launch_cells(Ctx &c, hipStream_t s, int cap) {
    GroupQueue q{c.gq.ctr, c.gq.order, c.gq.ngroups};
    const bool mixed = c.opt.precision == SERENX_MIXED;
    int least, most;
    cloud_sizes(c, least, most);
    const bool waves = most > LW_ALONE;
    int *cont = c.gq.ctr + 2 * NXCD + 1;
    const LongWalks lw{waves ? c.lw_group : nullptr, c.lw_at, cont, cont + 1, LW_BUDGET, LW_ALONE};
    if (waves && mixed) {
        auto kw = k_grav_cells_mixed<OCT, MACT>;
        hipLaunchKernelGGL(kw, dim3(walk_blocks(c, kw, cap, TB, TB / WAVE)), dim3(TB), 0, s, c.nc, c.gnf,
                           c.x, c.y, c.z, c.cid, c.root_range, c.active, c.gpot, c.agm, c.gax,
                           c.gay, c.gaz, c.gpc, near_list(c), c.icount, c.wstat, q, c.gq.cost,
                           c.grp, c.cloud_off, lw);
    } else if (waves) {
        auto kw = k_grav_cells_fp64<OCT, MACT>;
        hipLaunchKernelGGL(kw, dim3(walk_blocks(c, kw, cap, TB, TB / WAVE)), dim3(TB), 0, s, c.nc, c.gn,
                           c.x, c.y, c.z, c.cid, c.root_range, c.active, c.gpot, c.agm, c.gax,
                           c.gay, c.gaz, c.gpc, near_list(c), c.icount, c.wstat, q, c.gq.cost,
                           c.grp, c.cloud_off, lw);
    }
    const ListScratch sc{c.lw_ids, c.lw_in, c.lw_open, c.lw_list, c.lw_mask, c.lw_cap};
    auto launch = [&](auto k, int tb, const GroupQueue &gq, const LongWalks &walks) {
        const size_t lds =
            tb == OW_TB ? sizeof(ListWalk<OW_WAVES>) : sizeof(ListWalk<LW_WAVES>);
        const int nb = std::min(walk_blocks(c, k, cap, tb, 1, lds), c.lw_blocks);
        hipLaunchKernelGGL(k, dim3(nb), dim3(tb), lds, s, c.nc, c.gmac,
                           mixed ? mixed_mac_scale(c) : 1.0, c.gn, c.gnf, c.x, c.y, c.z, c.cid,
                           c.root_range, c.active, c.gpot, c.agm, c.gax, c.gay, c.gaz, c.gpc,
                           near_list(c), sc, c.icount, c.wstat, gq, c.gq.cost, c.grp,
                           c.cloud_off, walks);
    };
    if (mixed) {
        launch(k_grav_list<true, false, true, OCT, MACT>, LW_TB, q, lw);
        return;
    }
    if (most > LW_ORDERED && q.ngroups >= c.ncu)
        launch(k_grav_list<false, false, true, OCT, MACT>, LW_TB, q, lw);
    else if (most > LW_ORDERED)
        launch(k_grav_list<false, false, false, OCT, MACT>, LW_TB, q, lw);
    if (least <= LW_ORDERED) {
        LongWalks lo = lw;
        lo.taken = cont + 2;
        launch(k_grav_list<false, true, false, OCT, MACT>, OW_TB, GroupQueue{cont + 3, q.order, q.ngroups},
               lo);
    }
}

// Whether the mixed pair phase takes blocks of half its waves (each wave two of
// the eight shares of a list, so the sums are the same).  The knob counts blocks
// of four waves; of blocks of eight two fit a CU, so 3 is the odd number above
// one that they round up.  At 3 the pair phase of a 1M r^-2 step at the tuned
// tolerance kept 16 waves a CU where 12 were asked for, and the neighbour rows
// beside it, on the way to the hydro forces, took 3.6 instead of 2.9 ms (step
// 15.4 -> 14.8 ms).  In smaller clouds the longest lists bound the phase, and
// four waves take longer over them (uniform 131,071: 4.8 against 4.1 ms), so
// only clouds whose walks single waves begin are halved.
bool pairs_halved(const Ctx &c, int cap) {
    int least, most;
    cloud_sizes(c, least, most);
    return c.walk_queue != 0 && cap == 3 && most > LW_ALONE;
}

// phase 2 (pair terms), persistent over the same queue order (its second
// set of counters), on stream s with at most cap blocks per CU
template <int MACT, bool QUINTIC>
void launch_pairs(Ctx &c, const double4 *rec, hipStream_t s, int cap) {
    GroupQueue q{c.gq.ctr + NXCD, c.gq.order, c.gq.ngroups};
    if (c.opt.precision == SERENX_MIXED) {
        auto launch = [&](auto k, int tb) {
            hipLaunchKernelGGL(k, dim3(walk_blocks(c, k, cap, tb)), dim3(tb), 0, s, c.nc, c.gnf,
                               reinterpret_cast<const float4 *>(rec), c.x, c.y, c.z, c.h, c.zeta,
                               c.cid, c.root_range, c.active,
                               reinterpret_cast<const float4 *>(c.ktab + KT_G4F_OFF), c.gax, c.gay,
                               c.gaz, c.gpc, c.gpot, c.agm, near_list(c), c.icount, c.grp,
                               c.cloud_off, q);
        };
        constexpr int NW = PM_WAVES, HALF = PM_WAVES / 2;
        if (pairs_halved(c, cap))
            launch(k_grav_pairs_mixed<MACT, QUINTIC, HALF>, HALF * WAVE);
        else
            launch(k_grav_pairs_mixed<MACT, QUINTIC, NW>, NW * WAVE);
    } else {
        int least, most;
        cloud_sizes(c, least, most);
        auto launch = [&](auto k, int tb, const GroupQueue &gq) {
            hipLaunchKernelGGL(k, dim3(walk_blocks(c, k, cap, tb)), dim3(tb), 0, s, c.nc, c.gn, rec,
                               c.cid, c.root_range, c.active,
                               reinterpret_cast<const double4 *>(c.ktab + KT_G4_OFF), c.gax, c.gay,
                               c.gaz, c.gpc, c.gpot, c.agm, near_list(c), c.icount, c.grp,
                               c.cloud_off, gq);
        };
        if (most > LW_ORDERED) launch(k_grav_pairs_fp64<MACT, QUINTIC, false>, PF_TB, q);
        if (least <= LW_ORDERED)
            launch(k_grav_pairs_fp64<MACT, QUINTIC, true>, OW_TB,
                   GroupQueue{c.gq.ctr + 3 * NXCD + 6, q.order, q.ngroups});
    }
}

// Whether a launch takes its groups in tree order: forests with many groups for
// every block of the device have no long last walk to fear, and groups that are
// neighbours share the cells in L2.  The forests' evaluations with a build,
// longest first / in tree order (ms): FP64 33.6 / 34.2 at 19,000 groups, 50.8 /
// 48.6 at 28,000, 98 / 91 at 43,000, 153 / 137 at 67,000, 535 / 461 at 224,000
// (519 when single waves took the walks longest first); mixed 10.4 / 11.7 at 9,000,
// 22.5 / 22.0 at 19,000, 55.4 / 52.4 at 67,000, 186 / 168 at 224,000.  A cloud
// that single waves walk keeps longest first (uniform 2M FP64 82.7 / 88.3, r^-2
// 64.1 / 63.4).
bool tree_order(const Ctx &c) {
    int least, most;
    cloud_sizes(c, least, most);
    return c.gq.ngroups >= 100 * c.ncu && most <= LW_ALONE;
}

// sorts the queue order from the costs of the last walk, on the gravity
// stream
int sort_queue(Ctx &c) {
    Ctx::WalkQueue &q = c.gq;
    const int ng = q.ngroups;
    if (tree_order(c)) {
        hipLaunchKernelGGL(k_queue_identity, dim3(nblk(ng)), dim3(TB), 0, c.gstream, ng, q.order);
        return SERENX_OK;
    }
    hipLaunchKernelGGL(k_queue_keys, dim3(nblk(ng)), dim3(TB), 0, c.gstream, ng, q.cost,
                       (int)(q.have_cost && c.walk_queue != 0), q.keys, q.vals);
    size_t tb = q.tmp_bytes;
    SX_HIP(rocprim::radix_sort_pairs(q.tmp, tb, q.keys, q.keys2, q.vals, q.order, (unsigned)ng,
                                     0, 35, c.gstream));
    return SERENX_OK;
}

// the queue order of this walk (from the previous walk's costs) and zeroed
// counters, on the gravity stream.  The order is normally sorted at the end
// of the previous walk (grav_pairs), where the sort runs beside the hydro
// kernels; here it is sorted only when that order is missing or stale.
int prepare_queue(Ctx &c) {
    Ctx::WalkQueue &q = c.gq;
    const int ng = c.ngrp;
    if (ng != q.ngroups) {   // another group layout
        q.have_cost = false;
        q.order_ready = false;
    }
    q.ngroups = ng;
    if (c.capturing) {
        // a walk recorded into a graph takes its groups in tree order: the
        // sort library clears its buffers with memset nodes, which graphs
        // here must not hold (they have given wrong results on replays)
        hipLaunchKernelGGL(k_queue_identity, dim3(nblk(ng)), dim3(TB), 0, c.gstream, ng, q.order);
    } else if (!q.order_ready) {
        SX_TRY(sort_queue(c));
    }
    q.order_ready = false;   // used by this walk
    hipLaunchKernelGGL(k_zero_ints, dim3(1), dim3(64), 0, c.gstream, 4 * NXCD + 6, q.ctr);
    SX_HIP(hipGetLastError());
    return SERENX_OK;
}

// the cell phase on the gravity stream: queue prepared, then the walk
template <int OCT, int MACT>
int launch_grav_cells(Ctx &c) {
    SX_TRY(prepare_queue(c));
    launch_cells<OCT, MACT>(c, c.gstream, walk_cap(c));
    return SERENX_OK;
}

int cells_dispatch(Ctx &c) {
    const bool oct = c.opt.multipole != SERENX_QUADRUPOLE;
    switch (c.opt.mac) {
    case SERENX_MAC_GEOMETRIC:
        return oct ? launch_grav_cells<1, SERENX_MAC_GEOMETRIC>(c)
                   : launch_grav_cells<0, SERENX_MAC_GEOMETRIC>(c);
    case SERENX_MAC_GADGET:
        return oct ? launch_grav_cells<1, SERENX_MAC_GADGET>(c)
                   : launch_grav_cells<0, SERENX_MAC_GADGET>(c);
    case SERENX_MAC_EIGEN:
        return oct ? launch_grav_cells<1, SERENX_MAC_EIGEN>(c)
                   : launch_grav_cells<0, SERENX_MAC_EIGEN>(c);
    default:
        return oct ? launch_grav_cells<1, SERENX_MAC_GADGET2>(c)
                   : launch_grav_cells<0, SERENX_MAC_GADGET2>(c);
    }
}

// the pair phase on the gravity stream: source records packed, then the
// walk
template <int MACT>
int launch_grav_pairs(Ctx &c) {
    double4 *rec = reinterpret_cast<double4 *>(c.grec);
    if (c.opt.precision == SERENX_MIXED)
        hipLaunchKernelGGL(k_pack_grav_mixed, dim3(nblk(c.nc)), dim3(TB), 0, c.gstream, c.nc,
                           c.kg.range, c.gnf, c.x, c.y, c.z, c.m, c.h, c.zeta,
                           reinterpret_cast<float4 *>(c.grec));
    else
        hipLaunchKernelGGL(k_pack_grav, dim3(nblk(c.n)), dim3(TB), 0, c.gstream, c.n, c.kg.range,
                           c.x, c.y, c.z, c.m, c.h, c.zeta, rec);
    if (c.kg.range == walk_geom<true>().range)
        launch_pairs<MACT, true>(c, rec, c.gstream, pair_cap(c));
    else
        launch_pairs<MACT, false>(c, rec, c.gstream, pair_cap(c));
    return SERENX_OK;
}

int pairs_dispatch(Ctx &c) {
    switch (c.opt.mac) {
    case SERENX_MAC_GEOMETRIC: return launch_grav_pairs<SERENX_MAC_GEOMETRIC>(c);
    case SERENX_MAC_GADGET: return launch_grav_pairs<SERENX_MAC_GADGET>(c);
    case SERENX_MAC_EIGEN: return launch_grav_pairs<SERENX_MAC_EIGEN>(c);
    default: return launch_grav_pairs<SERENX_MAC_GADGET2>(c);
    }
}

}  // namespace

// The gravity walk runs on the context's gravity stream in two phases.
// grav_launch, queued after the tree is stocked, forks the gravity stream
// and runs phase 1 (traversal and cell terms: they read the tree, the
// positions and the previous |a| and potential) beside the h solve.
// grav_pairs, queued after the h solve, makes the gravity stream wait for
// it and runs phase 2 (pair terms, which need the new h and zeta), beside
// the neighbour lists, thermal and hydro forces.  grav_join adds the walk's
// acceleration to a on the main stream.
int grav_launch(Ctx &c) {
    SX_HIP(hipEventRecord(c.evfork, c.stream));
    SX_HIP(hipStreamWaitEvent(c.gstream, c.evfork, 0));
    SX_HIP(hipEventRecord(c.evg[0], c.gstream));
    SX_TRY(zero_words(c.icount, 2 * CTR_WORDS, c.gstream));
    SX_TRY(cells_dispatch(c));
    SX_HIP(hipGetLastError());
    SX_HIP(hipEventRecord(c.evg[1], c.gstream));
    c.grav_timed = false;
    return SERENX_OK;
}

int grav_pairs(Ctx &c) {
    SX_HIP(hipEventRecord(c.evfork2, c.stream));
    SX_HIP(hipStreamWaitEvent(c.gstream, c.evfork2, 0));
    SX_HIP(hipEventRecord(c.evg[2], c.gstream));
    SX_TRY(pairs_dispatch(c));
    SX_HIP(hipGetLastError());
    SX_HIP(hipEventRecord(c.evg[3], c.gstream));
    c.gq.have_cost = true;
    c.grav_timed = true;
    // the next walk's order, from this walk's costs: it runs beside the
    // main stream's hydro kernels, and the join waits for it, so that no
    // work of the walk outlives the evaluation
    if (!c.capturing && c.gq.ngroups == c.ngrp) {
        SX_TRY(sort_queue(c));
        SX_HIP(hipGetLastError());
        c.gq.order_ready = true;
    }
    SX_HIP(hipEventRecord(c.evjoin, c.gstream));
    return SERENX_OK;
}

int grav_join(Ctx &c) {
    SX_HIP(hipStreamWaitEvent(c.stream, c.evjoin, 0));
    hipLaunchKernelGGL(k_add_grav, dim3(nblk(c.n)), dim3(TB), 0, c.stream, c.n, c.active, c.gax,
                       c.gay, c.gaz, c.ax, c.ay, c.az);
    SX_HIP(hipGetLastError());
    return SERENX_OK;
}

int direct_gravity(Ctx &c, int nt, const int *dtargets, double *dacc, double *dpot) {
    hipLaunchKernelGGL(k_direct, dim3(nblk(nt)), dim3(256), 0, c.stream, c.kg, c.n, nt, dtargets, c.x,
                       c.y, c.z, c.m, c.h, c.zeta, c.cid, c.cloud_off,
                       reinterpret_cast<const double4 *>(c.ktab + KT_G4_OFF), dacc, dpot);
    SX_HIP(hipGetLastError());
    return SERENX_OK;
}

}  // namespace serenx
