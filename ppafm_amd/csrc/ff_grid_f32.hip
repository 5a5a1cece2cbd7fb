// FP32 force-field grid kernel on gfx950 (the float4 grid of the OpenCL
// path, FF.cl:366-423 evalLJC_QZs_noPos, and an FP32 variant of the
// ProbeParticle grid, Forces.h:120-132 / 237-244): bound by VALU issue.
//
//   * Orthogonal cells: boxes of 16^3 points with the far atoms on Chebyshev
//     nodes (box_f32).  Sheared cells: brick mapping as the FP64 kernel (4x4
//     grid columns x 64 z points per 256-thread block, 4 z points per lane,
//     z fastest stores), every atom at every point.
//   * Atoms are staged through LDS, box- or brick-local, as FP32 hi + lo parts
//     (x = hi + lo within FP32 rounding of the FP64 offset), so a pair
//     distance keeps FP32 relative accuracy 40 A from the grid origin.
//   * One v_rsq_f32 per pair serves the LJ term and the Coulomb point at
//     zero z offset; orthogonal cells share dx, dy and dx^2 + dy^2 + R2SAFE
//     across a lane's 4 z points.
//   * Coulomb stencils with z offsets (tip charges Qs at QZs, or the pz /
//     dz2 probe kinds) are finite differences whose terms cancel by orders
//     of magnitude (the dz2-like -10/+20/-10 tip: ~10^3).  They are summed
//     relative to the zero-offset distance r0 without forming the
//     differences in floating point: with W = sum w_s,
//       sum w_s / r_s   = W / r0   + sum w_s (1/r_s - 1/r0),
//       1/r_s - 1/r0    = (r0^2 - r_s^2) / (r0 r_s (r0 + r_s)),
//       r0^2 - r_s^2    = -dz_s (2 dz + dz_s)            (exact offsets),
//       1/r_s^3 - 1/r0^3 = (1/r_s - 1/r0)(1/r_s^2 + 1/(r_s r0) + 1/r0^2),
//     and the z offsets' own term sum w_s dz_s / r_s^3 the same way, so the
//     FP32 rounding is relative to the stencil's sum, not to its terms.
//   * The OpenCL model (mode 1) sums LJ and Coulomb into one force scale per
//     pair (one set of 3 FMAs); the ProbeParticle model (mode 0) keeps the
//     two fields apart for their separate clamps (io.py:766-778).
//   * FP32 partial sums over 32 atoms are folded into FP64 accumulators.
//   * Overflow guard: where a pair comes so close that an FP32 intermediate
//     overflows (r^-14 of the repulsion, below ~0.005 A), the point's sums
//     are no longer finite; such points (rare: an atom on a grid node) are
//     summed again over all atoms in FP64 after the loop.  Every other pair
//     is FP32.
// The epilogue clamps and combines as the FP64 kernel does.

#include <cmath>

#include "ff_grid.hpp"

#pragma clang fp contract(off)

namespace pp {

namespace {

// One atom against a lane's K points (ALL: the first nk of them).  SEP:
// separate LJ and Coulomb accumulators sL, sE (mode 0), else one, sL (mode 1).
// ORTHO: the points share x and y (orthogonal cell axes).
template <bool LJ, int NS, bool Z0, bool WE, bool QS, bool ORTHO, bool SEP, bool ALL, int K>
__device__ __forceinline__ void atom_f32(const FFArgs &A, const AtomLds &a, const float *px, const float *py,
                                         const float *pz, int nk, float sL[K][4], float sE[K][4])
{
    const float4 hi = a.hi;
    const float4 lo = a.lo;
    const float4 lj = a.lj;
    // uniform over the wave (every lane reads the same atom)
    const bool charged = NS > 0 && (!QS || hi.w != 0.f);
    float dx0 = 0.f, dy0 = 0.f, dxy2 = 0.f;
    if (ORTHO) {
        dx0 = (px[0] - hi.x) - lo.x;
        dy0 = (py[0] - hi.y) - lo.y;
        dxy2 = __fmaf_rn(dx0, dx0, __fmaf_rn(dy0, dy0, A.r2safe));
    }
#pragma unroll
    for (int k = 0; k < K; k++) {
        if (!ALL && k >= nk) break;
        const float dx = ORTHO ? dx0 : (px[k] - hi.x) - lo.x;
        const float dy = ORTHO ? dy0 : (py[k] - hi.y) - lo.y;
        // (pz - hi) is exact for a close atom (the operands are
        // within a factor of 2), which the near pairs' r^-13 needs
        const float dz = (pz[k] - hi.z) - lo.z;
        const float r2 = ORTHO ? __fmaf_rn(dz, dz, dxy2) : r2_f32(dx, dy, dz, A.r2safe);
        float ir0 = 0.f, ir20 = 0.f;
        if (LJ || NS > 0) {
            ir0 = __builtin_amdgcn_rsqf(r2);
            ir20 = ir0 * ir0;
        }
        // s: force over distance at zero z offset; e: energy;
        // sc, ec, fzc: the Coulomb stencil's force scale, energy
        // and extra z force
        // s = s0 * ir8 and e = e0 * ir6; the combined sum folds
        // these products into the additions of the Coulomb terms
        float s0 = 0.f, e0 = 0.f, ir6 = 0.f, ir8 = 0.f, sc = 0.f, ec = 0.f, fzc = 0.f;
        if (LJ) {
            ir6 = ir20 * ir20 * ir20;
            ir8 = ir6 * ir20;
            s0 = __fmaf_rn(lj.y, ir6, -lj.x);
            if (WE) e0 = __fmaf_rn(lj.w, ir6, -lj.z);
        }
        if (charged && NS == 1 && Z0) {  // one point at zero offset
            ec = (hi.w * A.sw[0]) * ir0;
            sc = ec * ir20;
        } else if (charged) {  // stencil with offsets, cancellation free
            const float r0 = r2 * ir0;
            float s1 = 0.f, s3 = 0.f, s3z = 0.f;
#pragma unroll
            for (int s_ = Z0 ? 1 : 0; s_ < NS; s_++) {
                const float dzs = dz + A.sdz[s_];
                const float r2s = ORTHO ? __fmaf_rn(dzs, dzs, dxy2) : r2_f32(dx, dy, dzs, A.r2safe);
                const float irs = __builtin_amdgcn_rsqf(r2s);
                const float rs = r2s * irs;
                const float dr2 = -A.sdz[s_] * (dz + dz + A.sdz[s_]);  // r0^2 - rs^2
                const float d1 = (dr2 * ir0) * (irs * __builtin_amdgcn_rcpf(r0 + rs));
                const float d3 = d1 * __fmaf_rn(irs, irs, __fmaf_rn(irs, ir0, ir20));
                s1 = __fmaf_rn(A.sw[s_], d1, s1);
                s3 = __fmaf_rn(A.sw[s_], d3, s3);
                s3z = __fmaf_rn(A.sw[s_] * A.sdz[s_], d3, s3z);
            }
            const float ir30 = ir0 * ir20;
            ec = hi.w * __fmaf_rn(A.swsum, ir0, s1);
            sc = hi.w * __fmaf_rn(A.swsum, ir30, s3);
            fzc = hi.w * __fmaf_rn(A.swdz, ir30, s3z);
        }
        if (SEP) {
            if (LJ) {
                const float s = s0 * ir8;
                sL[k][0] = __fmaf_rn(dx, s, sL[k][0]);
                sL[k][1] = __fmaf_rn(dy, s, sL[k][1]);
                sL[k][2] = __fmaf_rn(dz, s, sL[k][2]);
                if (WE) sL[k][3] = __fmaf_rn(e0, ir6, sL[k][3]);
            }
            if (charged) {
                sE[k][0] = __fmaf_rn(dx, sc, sE[k][0]);
                sE[k][1] = __fmaf_rn(dy, sc, sE[k][1]);
                sE[k][2] = __fmaf_rn(dz, sc, NS == 1 && Z0 ? sE[k][2] : sE[k][2] + fzc);
                if (WE) sE[k][3] += ec;
            }
        } else if (LJ || charged) {
            // s0 ir8 + ec ir20 = (s0 ir6 + ec) ir20 (one Coulomb point)
            const float st = LJ ? (NS == 1 && Z0 ? __fmaf_rn(s0, ir6, ec) * ir20 : __fmaf_rn(s0, ir8, sc)) : sc;
            sL[k][0] = __fmaf_rn(dx, st, sL[k][0]);
            sL[k][1] = __fmaf_rn(dy, st, sL[k][1]);
            sL[k][2] = __fmaf_rn(dz, st, NS == 1 && Z0 ? sL[k][2] : sL[k][2] + fzc);
            if (WE) sL[k][3] += LJ ? __fmaf_rn(e0, ir6, ec) : ec;
        }
    }
}

// Sums over the atoms lds[first], lds[first + step], ... (n of them) at the
// lane's points: FP32 partial sums of FOLD atoms folded into FP64.
template <bool LJ, int NS, bool Z0, bool WE, bool QS, bool ORTHO, bool SEP, bool ALL, int K = kK, int FOLD = kFold>
__device__ __forceinline__ void sum_f32(const FFArgs &A, const AtomLds *lds, int first, int step, int n, const float *px,
                                        const float *py, const float *pz, int nk, double aL[K][4], double aE[K][4])
{
    for (int j0 = 0; j0 < n; j0 += FOLD) {
        const int j1 = min(n, j0 + FOLD);
        float sL[K][4], sE[K][4];
#pragma unroll
        for (int k = 0; k < K; k++)
#pragma unroll
            for (int c = 0; c < 4; c++) { sL[k][c] = 0.f; sE[k][c] = 0.f; }
        for (int j = j0; j < j1; j++)
            atom_f32<LJ, NS, Z0, WE, QS, ORTHO, SEP, ALL, K>(A, lds[first + j * step], px, py, pz, nk, sL, sE);
#pragma unroll
        for (int k = 0; k < K; k++)
#pragma unroll
            for (int c = 0; c < 4; c++) {
                aL[k][c] += (double)sL[k][c];
                if (SEP) aE[k][c] += (double)sE[k][c];
            }
    }
}

// Atom a relative to (cx, cy, cz), as FP32 hi + lo parts.
__device__ __forceinline__ AtomLds atom_record(const AtomRec &a, double rx, double ry, double rz)
{
    const float hx = (float)rx, hy = (float)ry, hz = (float)rz;
    AtomLds r;
    r.hi = make_float4(hx, hy, hz, (float)a.q);
    r.lo = make_float4((float)(rx - hx), (float)(ry - hy), (float)(rz - hz), 0.f);
    r.lj = make_float4((float)(6.0 * a.c6), (float)(12.0 * a.c12), (float)a.c6, (float)a.c12);
    return r;
}

// The grid value at a point (qx, qy, qz): sums aL, aE of every atom there,
// again in FP64 where an FP32 term overflowed, clamped and combined.
template <bool LJ, int NS, bool WE, bool SEP>
__device__ __forceinline__ float4 point_value(const FFArgs &A, const AtomRec *__restrict__ atoms, double qx, double qy,
                                              double qz, double aL[4], double aE[4])
{
    bool finite = true;
#pragma unroll
    for (int c = 0; c < 4; c++) finite = finite && isfinite(aL[c]) && (!SEP || isfinite(aE[c]));
    if (!finite) {  // overflow guard: this point again, every pair in FP64
#pragma unroll
        for (int c = 0; c < 4; c++) { aL[c] = 0; aE[c] = 0; }
        for (int j = 0; j < A.natoms; j++) {
            const AtomRec a = atoms[j];
            pair_fp64<LJ, NS, WE>(A, qx - a.x, qy - a.y, qz - a.z, a.q, a.c6, a.c12, aL, SEP ? aE : aL);
        }
    }
    double gx, gy, gz, en;
    if (SEP) {
        clamp_vec(aL[0], aL[1], aL[2], A.fmax);
        clamp_vec(aE[0], aE[1], aE[2], A.fmax);
        gx = aL[0] + A.probe_q * aE[0];
        gy = aL[1] + A.probe_q * aE[1];
        gz = aL[2] + A.probe_q * aE[2];
        en = aL[3] + A.probe_q * aE[3];
    } else {
        gx = aL[0]; gy = aL[1]; gz = aL[2]; en = aL[3];
    }
    return make_float4((float)gx, (float)gy, (float)gz, WE ? (float)en : 0.f);
}

// Sheared cells: a 4x4-column x 64-point brick, every atom at every point.
template <bool LJ, int NS, bool Z0, bool WE, bool QS, bool SEP>
__device__ __forceinline__ void brick_f32(const FFArgs &A, const AtomRec *__restrict__ atoms, float4 *__restrict__ out,
                                          int b, AtomLds *lds)
{
    const int t = threadIdx.x;
    const int col = t / kZLanes;
    const int zl = t % kZLanes;
    const int bz = b % A.nbz; b /= A.nbz;
    const int by = b % A.nby;
    const int bx = b / A.nby;
    const int ix = bx * kColsX + (col % kColsX);
    const int iy = by * kColsY + (col / kColsX);
    const int z0 = bz * kZBrick;
    const double cx = bx * kColsX + 0.5 * (kColsX - 1);
    const double cy = by * kColsY + 0.5 * (kColsY - 1);
    const double cz = z0 + 0.5 * (kZBrick - 1);
    const double *D = A.dcell;
    const double ccx = D[0] * cx + D[3] * cy + D[6] * cz;
    const double ccy = D[1] * cx + D[4] * cy + D[7] * cz;
    const double ccz = D[2] * cx + D[5] * cy + D[8] * cz;
    const double fx = ix - cx, fy = iy - cy;
    float px[kK], py[kK], pz[kK];
#pragma unroll
    for (int k = 0; k < kK; k++) {
        const double fz = (z0 + zl + kZLanes * k) - cz;
        px[k] = (float)(D[0] * fx + D[3] * fy + D[6] * fz);
        py[k] = (float)(D[1] * fx + D[4] * fy + D[7] * fz);
        pz[k] = (float)(D[2] * fx + D[5] * fy + D[8] * fz);
    }
    const int nk = min(kK, (A.n[2] - z0 + kZLanes - 1) / kZLanes);

    double aL[kK][4], aE[kK][4];  // aE: mode 0 only
#pragma unroll
    for (int k = 0; k < kK; k++)
#pragma unroll
        for (int c = 0; c < 4; c++) { aL[k][c] = 0; aE[k][c] = 0; }

    for (int i0 = 0; i0 < A.natoms; i0 += kTile) {
        const int nt = min(kTile, A.natoms - i0);
        __syncthreads();
        for (int j = t; j < nt; j += kThreads) {
            const AtomRec a = atoms[i0 + j];
            lds[j] = atom_record(a, a.x - ccx, a.y - ccy, a.z - ccz);
        }
        __syncthreads();
        // bricks with all of a lane's points inside the grid (all but the
        // top ones) need no per-point test
        if (nk == kK) sum_f32<LJ, NS, Z0, WE, QS, false, SEP, true>(A, lds, 0, 1, nt, px, py, pz, nk, aL, aE);
        else sum_f32<LJ, NS, Z0, WE, QS, false, SEP, false>(A, lds, 0, 1, nt, px, py, pz, nk, aL, aE);
    }

    if (ix >= A.n[0] || iy >= A.n[1]) return;
#pragma unroll
    for (int k = 0; k < kK; k++) {
        const int iz = z0 + zl + kZLanes * k;
        if (iz >= A.n[2]) break;
        const double fz = iz - cz;
        out[((long)ix * A.n[1] + iy) * A.n[2] + iz] =
            point_value<LJ, NS, WE, SEP>(A, atoms, ccx + (D[0] * fx + D[3] * fy + D[6] * fz),
                                         ccy + (D[1] * fx + D[4] * fy + D[7] * fz),
                                         ccz + (D[2] * fx + D[5] * fy + D[8] * fz), aL[k], aE[k]);
    }
}

// Orthogonal cells: a block computes a box of 16^3 points.  The field of an
// atom farther from the box than kFarRatio half widths (with the Coulomb
// stencil's points, which lie up to maxdz above and below it), and so far that
// its repulsion is below 1/24 of its attraction, is smooth over it: such far atoms
// are summed at the box's kP^3 Chebyshev nodes only, and the sums are carried
// to the 4096 points by the nodes' tensor-product polynomial in FP64; atoms
// nearer are summed at every point.  A far pair costs 1/8 of a near one.  With
// more atoms than one LDS tile, those beyond kVeryFarRatio half widths are
// summed at kP2^3 nodes (1/33), whose polynomial is added to the values at the
// kP^3 nodes.  Bound by VALU issue, in the near pairs for a molecule, in the
// nodes for a slab: of a wave's time 53 % is issue (slab; 49 % molecule), 30 %
// (35 %) waiting for a slot that another wave holds, 17 % (16 %) for loads, LDS
// and barriers, 0.04 % (0.5 %) LDS bank conflicts; 2.8 (2.3) waves on a SIMD, a
// VALU instruction every 3.1 (4.4) cycles.
// Interpolation error at 0.1 A steps, against the far atom's own force at the
// point, largest over a box that faces the atom (an atom off its edges or
// corners: a tenth), in FP64: order 8 at ratio 8 (6 A) 5.9e-7 for H, 4.1e-7 O,
// 2.7e-7 N, 1.3e-7 C (6.1 A), 3e-8 Au (6.9 A), 4e-9 of the Coulomb force; its
// root mean square over the box is a third of that.  Order 5 at ratio 40 (30 A):
// 3.5e-7 of the Lennard-Jones force, 5e-9 of the Coulomb force.  An FP32 pair is
// rounded by as much, which is why the grid's error as a whole may not grow:
// the nodes are stretched to the box's ends, where the polynomial would
// otherwise scale a node's rounding by up to 1.4 an axis (now at most 1.02), and
// their FP32 sums are 8 atoms long, not 32.  Over 17 grids (slabs and molecules,
// both tips) the error against FP64 is 0.90 (median) and 0.95 (99th percentile)
// of the sum over every pair, 0.92 and 0.90 for the energy; without these two
// changes it was 1.02 and 1.08, 1.18 and 1.17.  Node coordinates are FP32 while
// the weights assume exact nodes: 3e-8 A at 0.75 A, 4e-8 of the force at 6 A.
// Measured (grid kernel, before: every atom at every point): 60 atoms, dz2
// tip, 256x256x192 points 1254 -> 368 us; 16 such grids of 8-120 atoms
// 24.1 -> 6.8 ms; 17,928 atoms, 400x400x300 points 319 -> 43 ms with one set of
// nodes, 15.4 ms with two.
constexpr int kBox = 16;
constexpr int kP = 8;
constexpr double kFarRatio = 8.0;
constexpr double kFarForces = 24.0;  // attraction over repulsion
constexpr int kP2 = 5;
constexpr double kVeryFarRatio = 40.0;
constexpr int kGroups = 10;  // lane groups of kP2^2 that share the atoms, kP2 nodes along z a lane
// Far atoms a box needs before the polynomial (56 FP64 FMAs per point) costs
// less than their pair sums; below it every atom of the box counts as near.
// 256x256x192 points, all near against far ones at the nodes: dz2 tip, 12 atoms
// 238 and 123 us; one Coulomb point, 12 atoms 84 and 89, 20 atoms 123 and 100.
template <int NS, bool Z0>
constexpr int kFarMin = NS == 0 || (NS == 1 && Z0) ? 16 : 12;
constexpr int kNodeFold = 8;  // FP32 partial-sum length at the nodes
constexpr int kBoxTile = kThreads;  // atoms per LDS tile, one per thread
constexpr int kNearCap = 512;       // near atoms listed; beyond, every atom is staged for each slab
constexpr int kWPad = kP + 1;       // row stride against LDS bank conflicts

// Chebyshev nodes, stretched so that the first and last are -1 and 1, and the
// values of their Lagrange polynomials at the box's equidistant points (the
// ends at -1 and 1).
struct FarTable {
    double x[kP];
    double w[kBox * kP];
    double x2[kP2];
    double w2[kP * kP2];  // the second set's polynomials at the first set's nodes
};

template <int NG>  // fields summed together: force, and energy where it is wanted
struct BoxLds {
    double w[kBox * kWPad];
    union {
        AtomLds rec[kBoxTile];
        struct {
            double after_rec[kBoxTile * sizeof(AtomLds) / sizeof(double)];
            double node2[NG][kP2 * kP2 * kP2];
        };
        struct {
            double t1[NG][4 * kP * kP];         // slab of 4 x: (x, node y, node z)
            double t2[NG][4 * kBox * kWPad];    // (x, y, node z)
        };
    };
    int list[kNearCap];
    int count[2][kThreads / 64];
};

template <bool LJ, int NS, bool Z0, bool WE, bool SEP>
__device__ __forceinline__ void box_f32(const FFArgs &A, const FarTable &F, const AtomRec *__restrict__ atoms,
                                        float4 *__restrict__ out, int b, int slab0, int slab1)
{
    constexpr int NG = WE ? 4 : 3;
    constexpr int G = SEP ? 2 : 1;
    constexpr bool QS = LJ && NS > 0;  // skip uncharged atoms' Coulomb terms
    __shared__ BoxLds<NG> L;
    __shared__ double node[G][NG][kP * kP * kP];
    const int t = threadIdx.x, lane = t & 63, wave = t >> 6;
    const int bz = b % A.nbz; b /= A.nbz;
    const int by = b % A.nby;
    const int bx = b / A.nby;
    if (bx * kBox + slab0 * 4 >= A.n[0]) return;  // uniform
    const double dcx = A.dcell[0], dcy = A.dcell[4], dcz = A.dcell[8];
    constexpr double half = 0.5 * (kBox - 1);
    const double cx = bx * kBox + half, cy = by * kBox + half, cz = bz * kBox + half;
    const double ccx = dcx * cx, ccy = dcy * cy, ccz = dcz * cz;
    const double hx = half * fabs(dcx), hy = half * fabs(dcy), hz = half * fabs(dcz);
    const double hmax = fmax(hx, fmax(hy, hz));
    // 0 near, 1 far, 2 very far
    const bool two_sets = A.natoms > kBoxTile;
    auto range = [&](const AtomRec &a) {
        const double rx = a.x - ccx, ry = a.y - ccy, rz = a.z - ccz;
        // the stencil's Coulomb points act as charges up to maxdz above and
        // below the atom: the distance is that of the nearest of them
        const double ex = fmax(fabs(rx) - hx, 0.0), ey = fmax(fabs(ry) - hy, 0.0), ez = fmax(fabs(rz) - (hz + A.maxdz), 0.0);
        const double d2 = (ex * ex + ey * ey + ez * ez);
        // force terms 12 c12 r^-13 and 6 c6 r^-7
        const bool far = d2 >= kFarRatio * kFarRatio * (hmax * hmax) &&
                         (!LJ || d2 * d2 * d2 * a.c6 >= 2.0 * kFarForces * fabs(a.c12)) &&
                         isfinite(rx) && isfinite(ry) && isfinite(rz);
        return !far ? 0 : two_sets && d2 >= kVeryFarRatio * kVeryFarRatio * (hmax * hmax) ? 2 : 1;
    };
    for (int e = t; e < kBox * kP; e += kThreads) L.w[(e / kP) * kWPad + e % kP] = F.w[e];

    // ---- far atoms at the nodes.  128 lanes hold the nodes, 4 along z each;
    // the block's halves take alternate atoms.
    const int u = t & 127;
    float nx[kK], ny[kK], nz[kK];
    nx[0] = (float)(F.x[u >> 4] * half * dcx);
    ny[0] = (float)(F.x[(u >> 1) & 7] * half * dcy);
#pragma unroll
    for (int k = 0; k < kK; k++) {
        nx[k] = nx[0]; ny[k] = ny[0];
        nz[k] = (float)(F.x[(u & 1) * kK + k] * half * dcz);
    }
    bool use_far = true;
    int nnear = 0;
    {
        double aL[kK][4], aE[kK][4];
#pragma unroll
        for (int k = 0; k < kK; k++)
#pragma unroll
            for (int c = 0; c < 4; c++) { aL[k][c] = 0; aE[k][c] = 0; }
        for (int i0 = 0; i0 < A.natoms; i0 += kBoxTile) {
            const bool in = i0 + t < A.natoms;
            AtomRec a = {};
            int rg = -1;
            if (in) {
                a = atoms[i0 + t];
                rg = range(a);
            }
            const bool far = rg == 1;
            const unsigned long long mf = __ballot(far), mn = __ballot(rg == 0);
            if (lane == 0) {
                L.count[0][wave] = __popcll(mf);
                L.count[1][wave] = __popcll(mn);
            }
            __syncthreads();
            int nf = 0, pf = 0, pn = nnear;
#pragma unroll
            for (int q = 0; q < kThreads / 64; q++) {
                if (q < wave) { pf += L.count[0][q]; pn += L.count[1][q]; }
                nf += L.count[0][q];
                nnear += L.count[1][q];
            }
            const unsigned long long below = (1ull << lane) - 1;
            if (A.natoms <= kBoxTile && nf < kFarMin<NS, Z0>) {  // uniform: too few far atoms
                use_far = false;
                nnear = A.natoms;
                if (in && t < kNearCap) L.list[t] = t;
                break;
            }
            if (far) L.rec[pf + __popcll(mf & below)] = atom_record(a, a.x - ccx, a.y - ccy, a.z - ccz);
            else if (rg == 0) {
                const int p = pn + __popcll(mn & below);
                if (p < kNearCap) L.list[p] = i0 + t;
            }
            __syncthreads();
            const int first = t >> 7;
            sum_f32<LJ, NS, Z0, WE, QS, true, SEP, true, kK, kNodeFold>(A, L.rec, first, 2, (nf - first + 1) / 2, nx, ny, nz, kK,
                                                                        aL, aE);
            __syncthreads();
        }
        if (use_far) {
            if (t >= 128) {
#pragma unroll
                for (int k = 0; k < kK; k++)
#pragma unroll
                    for (int c = 0; c < NG; c++) {
                        node[0][c][u * kK + k] = aL[k][c];
                        if (SEP) node[G - 1][c][u * kK + k] = aE[k][c];
                    }
            }
            __syncthreads();
            if (t < 128) {
#pragma unroll
                for (int k = 0; k < kK; k++)
#pragma unroll
                    for (int c = 0; c < NG; c++) {
                        node[0][c][u * kK + k] += aL[k][c];
                        if (SEP) node[G - 1][c][u * kK + k] += aE[k][c];
                    }
            }
        }
    }
    __syncthreads();
    if (two_sets) {  // uniform
        // ---- very far atoms at the second set of nodes
        const int grp = t / (kP2 * kP2), c5 = t % (kP2 * kP2);
        const bool on = grp < kGroups;
        float nx[kP2], ny[kP2], nz[kP2];
        double aL[kP2][4], aE[kP2][4];
#pragma unroll
        for (int k = 0; k < kP2; k++) {
            nx[k] = (float)(F.x2[c5 / kP2] * half * dcx);
            ny[k] = (float)(F.x2[c5 % kP2] * half * dcy);
            nz[k] = (float)(F.x2[k] * half * dcz);
#pragma unroll
            for (int c = 0; c < 4; c++) { aL[k][c] = 0; aE[k][c] = 0; }
        }
        int any = 0;
        for (int i0 = 0; i0 < A.natoms; i0 += kBoxTile) {
            AtomRec a = {};
            bool vf = false;
            if (i0 + t < A.natoms) {
                a = atoms[i0 + t];
                vf = range(a) == 2;
            }
            const unsigned long long m = __ballot(vf);
            if (lane == 0) L.count[0][wave] = __popcll(m);
            __syncthreads();
            int n = 0, p = 0;
#pragma unroll
            for (int q = 0; q < kThreads / 64; q++) {
                if (q < wave) p += L.count[0][q];
                n += L.count[0][q];
            }
            if (vf) L.rec[p + __popcll(m & ((1ull << lane) - 1))] = atom_record(a, a.x - ccx, a.y - ccy, a.z - ccz);
            __syncthreads();
            if (on)
                sum_f32<LJ, NS, Z0, WE, QS, true, SEP, true, kP2, kNodeFold>(A, L.rec, grp, kGroups,
                                                                             (n - grp + kGroups - 1) / kGroups, nx, ny, nz, kP2,
                                                                             aL, aE);
            any += n;
            __syncthreads();
        }
        if (any > 0) {  // uniform
#pragma unroll
            for (int g = 0; g < G; g++) {
                for (int r = 0; r < kGroups; r++) {  // the groups' sums, in order
                    if (grp == r) {
#pragma unroll
                        for (int k = 0; k < kP2; k++)
#pragma unroll
                            for (int c = 0; c < NG; c++) {
                                const double v = g == 0 ? aL[k][c] : aE[k][c];
                                double &o = L.node2[c][c5 * kP2 + k];
                                o = r == 0 ? v : o + v;
                            }
                    }
                    __syncthreads();
                }
                for (int e = t; e < kP * kP * kP; e += kThreads) {
                    double v[NG];
#pragma unroll
                    for (int c = 0; c < NG; c++) v[c] = 0;
                    const double *wx = F.w2 + (e >> 6) * kP2, *wy = F.w2 + ((e >> 3) & 7) * kP2, *wz = F.w2 + (e & 7) * kP2;
                    for (int i = 0; i < kP2 * kP2; i++) {
                        const double wxy = wx[i / kP2] * wy[i % kP2];
                        for (int k = 0; k < kP2; k++) {
                            const double w = wxy * wz[k];
#pragma unroll
                            for (int c = 0; c < NG; c++) v[c] = __fma_rn(w, L.node2[c][i * kP2 + k], v[c]);
                        }
                    }
#pragma unroll
                    for (int c = 0; c < NG; c++) node[g][c][e] += v[c];
                }
                __syncthreads();
            }
        }
    }

    // ---- the points, in slabs of 4 x: a wave holds 4x4 columns, a lane 4 z
    // points of one.  Near pairs are summed in coordinates relative to the
    // centre of the wave's columns (and of 64 points along z), which keeps the
    // rounding of a point within 1e-8 A in x and y.
    const int col = lane >> 2, zl = lane & 3;
    const int xi = col >> 2, y = wave * 4 + (col & 3);
    const int c2 = xi * kBox + y;  // the column's row in t2
    const int iy = by * kBox + y;
    const double wcy = by * kBox + wave * 4 + 1.5, wcz = (bz * kBox / kZBrick) * kZBrick + 0.5 * (kZBrick - 1);
    const double fy = iy - wcy;
    const double oy = dcy * wcy, oz = dcz * wcz;
    for (int slab = slab0; slab < slab1; slab++) {
        if (bx * kBox + slab * 4 >= A.n[0]) break;  // uniform
        const int ix = bx * kBox + slab * 4 + xi;
        const double wcx = bx * kBox + slab * 4 + 1.5;
        const double fx = ix - wcx;
        const double ox = dcx * wcx;
        double aL[kK][4], aE[kK][4];
#pragma unroll
        for (int k = 0; k < kK; k++)
#pragma unroll
            for (int c = 0; c < 4; c++) { aL[k][c] = 0; aE[k][c] = 0; }
        if (use_far) {
#pragma unroll
            for (int g = 0; g < G; g++) {
                double v[NG];
#pragma unroll
                for (int c = 0; c < NG; c++) v[c] = 0;
#pragma unroll 2
                for (int q = 0; q < kP; q++) {
                    const double w = L.w[(slab * 4 + wave) * kWPad + q];
#pragma unroll
                    for (int c = 0; c < NG; c++) v[c] = __fma_rn(w, node[g][c][q * kP * kP + lane], v[c]);
                }
#pragma unroll
                for (int c = 0; c < NG; c++) L.t1[c][t] = v[c];
                __syncthreads();
#pragma unroll
                for (int r = 0; r < 2; r++) {
                    const int e = t + r * kThreads;
                    const int cc = e >> 3, kz = e & 7;
#pragma unroll
                    for (int c = 0; c < NG; c++) v[c] = 0;
#pragma unroll 2
                    for (int q = 0; q < kP; q++) {
                        const double w = L.w[(cc & 15) * kWPad + q];
#pragma unroll
                        for (int c = 0; c < NG; c++) v[c] = __fma_rn(w, L.t1[c][(cc >> 4) * kP * kP + q * kP + kz], v[c]);
                    }
#pragma unroll
                    for (int c = 0; c < NG; c++) L.t2[c][cc * kWPad + kz] = v[c];
                }
                __syncthreads();
#pragma unroll 2
                for (int q = 0; q < kP; q++) {
#pragma unroll
                    for (int c = 0; c < NG; c++) v[c] = L.t2[c][c2 * kWPad + q];
#pragma unroll
                    for (int k = 0; k < kK; k++) {
                        const double w = L.w[(zl + 4 * k) * kWPad + q];
#pragma unroll
                        for (int c = 0; c < NG; c++) {
                            if (g == 0) aL[k][c] = __fma_rn(w, v[c], aL[k][c]);
                            else aE[k][c] = __fma_rn(w, v[c], aE[k][c]);
                        }
                    }
                }
                __syncthreads();
            }
        }
        float px[kK], py[kK], pz[kK];
#pragma unroll
        for (int k = 0; k < kK; k++) {
            px[k] = (float)(dcx * fx);
            py[k] = (float)(dcy * fy);
            pz[k] = (float)(dcz * (bz * kBox + zl + 4 * k - wcz));
        }
        const bool listed = nnear <= kNearCap;
        const int total = listed ? nnear : A.natoms;
        AtomLds *rec = L.rec + wave * 64;  // each wave stages the atoms for itself
        for (int i0 = 0; i0 < total; i0 += 64) {
            const int nt = min(64, total - i0);
            if (lane < nt) {
                const AtomRec a = atoms[listed ? L.list[i0 + lane] : i0 + lane];
                AtomLds r = atom_record(a, a.x - ox, a.y - oy, a.z - oz);
                if (!listed && use_far && range(a) > 0) {  // in the polynomial already: its terms here are zeros
                    r.hi.w = 0.f;
                    r.lj = make_float4(0.f, 0.f, 0.f, 0.f);
                }
                rec[lane] = r;
            }
            __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
            __builtin_amdgcn_wave_barrier();
            sum_f32<LJ, NS, Z0, WE, QS, true, SEP, true>(A, rec, 0, 1, nt, px, py, pz, kK, aL, aE);
            __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
            __builtin_amdgcn_wave_barrier();
        }
        __syncthreads();  // the next slab's t1, t2 share the records' memory
        if (ix < A.n[0] && iy < A.n[1]) {
#pragma unroll
            for (int k = 0; k < kK; k++) {
                const int iz = bz * kBox + zl + 4 * k;
                if (iz >= A.n[2]) break;
                out[((long)ix * A.n[1] + iy) * A.n[2] + iz] =
                    point_value<LJ, NS, WE, SEP>(A, atoms, ox + dcx * fx, oy + dcy * fy, oz + dcz * (iz - wcz), aL[k], aE[k]);
            }
        }
    }
}

template <bool LJ, int NS, bool Z0, bool WE, bool SEP>
__global__ __launch_bounds__(kThreads) void ff_f32_kernel(FFArgs A, const AtomRec *__restrict__ atoms,
                                                          float4 *__restrict__ out)
{
    __shared__ AtomLds lds[kTile];
    brick_f32<LJ, NS, Z0, WE, false, SEP>(A, atoms, out, blockIdx.x, lds);
}

template <bool LJ, int NS, bool Z0, bool WE, bool QS, bool SEP>
__global__ __launch_bounds__(kThreads) void ff_f32_batch_kernel(FFArgs A0, const BatchGridItem *__restrict__ items,
                                                                const long long *__restrict__ prefix, int nitems,
                                                                const AtomRec *__restrict__ atoms, float4 *__restrict__ grid)
{
    __shared__ AtomLds lds[kTile];
    const long long bidx = blockIdx.x;
    const int m = find_item(prefix, nitems, bidx);
    const BatchGridItem it = items[m];
    const FFArgs A = batch_args(A0, it);
    brick_f32<LJ, NS, Z0, WE, QS, SEP>(A, atoms + it.atom_off, grid + it.grid_off, (int)(bidx - prefix[m]), lds);
}

__host__ __device__ inline void set_boxes(FFArgs &A)
{
    A.nbx = (A.n[0] + kBox - 1) / kBox;
    A.nby = (A.n[1] + kBox - 1) / kBox;
    A.nbz = (A.n[2] + kBox - 1) / kBox;
}

// One grid (items == nullptr) or every grid of a batch; split: blocks per box
// (box_split).  Three workgroups per CU: LDS (46 KB) allows no more, so the
// registers need not either.
template <bool LJ, int NS, bool Z0, bool WE, bool SEP>
__global__ __launch_bounds__(kThreads, SEP ? 2 : 3) void ff_box_kernel(FFArgs A, FarTable F,
                                                                       const BatchGridItem *__restrict__ items,
                                                                       const long long *__restrict__ prefix, int nitems,
                                                                       const AtomRec *__restrict__ atoms,
                                                                       float4 *__restrict__ out, int split)
{
    long long b = blockIdx.x / split;
    const int slabs = kBox / 4 / split, slab0 = (blockIdx.x % split) * slabs;
    if (items) {
        const int m = find_item(prefix, nitems, b);
        const BatchGridItem it = items[m];
        A = batch_args(A, it);
        set_boxes(A);
        b -= prefix[m];
        atoms += it.atom_off;
        out += it.grid_off;
    }
    box_f32<LJ, NS, Z0, WE, SEP>(A, F, atoms, out, (int)b, slab0, slab0 + slabs);
}

// Chebyshev points of the first kind, divided by the largest (which leaves
// their barycentric weights), x[n], and the values w[m][n] of their Lagrange
// polynomials at m points (barycentric form; unit weights at a node).
void cheb(int n, double *x, int m, const double *at, double *w)
{
    const double pi = 3.14159265358979323846;
    for (int k = 0; k < n; k++) x[k] = std::cos((2 * k + 1) * pi / (2 * n)) / std::cos(pi / (2 * n));
    for (int i = 0; i < m; i++) {
        int node = -1;
        for (int k = 0; k < n; k++)
            if (std::fabs(at[i] - x[k]) < 1e-12) node = k;
        if (node >= 0) {
            for (int k = 0; k < n; k++) w[i * n + k] = k == node;
            continue;
        }
        double sum = 0;
        for (int k = 0; k < n; k++)
            sum += w[i * n + k] = (k % 2 ? -1.0 : 1.0) * std::sin((2 * k + 1) * pi / (2 * n)) / (at[i] - x[k]);
        for (int k = 0; k < n; k++) w[i * n + k] /= sum;
    }
}

FarTable make_far_table()
{
    FarTable F;
    double pt[kBox];
    for (int i = 0; i < kBox; i++) pt[i] = 2.0 * i / (kBox - 1) - 1.0;
    cheb(kP, F.x, kBox, pt, F.w);
    cheb(kP2, F.x2, kP, F.x, F.w2);
    return F;
}

const FarTable &far_table()
{
    static const FarTable F = make_far_table();
    return F;
}

// Blocks per box.  A block takes as long on any grid (40 atoms, dz2 tip: 95 us),
// so a launch that leaves CUs without work gives the four slabs of a
// box to 2 or 4 blocks, each of which sums the nodes for itself; the points'
// sums are the same.  1 / 2 / 4 blocks a box and, before boxes, the 4x4x64 bricks
// over all atoms, us (dz2 tip, 40 atoms; one Coulomb point, 120 atoms):
//   64 boxes    95 / 50 / 27, bricks 25     65 / 38 / 25, 27
//   128         96 / 50 / 40, 40            65 / 38 / 31, 34
//   175         96 / 58 / 49, 71            65 / 41 / 37, 58
//   216         97 / 58 / 58, 88            66 / 43 / 50, 69
//   392         125 / 94 / 95, 88           76 / 67 / 79, 71
//   512         131 / 116 / 118, 138        78 / 81 / 92, 104
//   768         115 / 121 / 140, 201        80 / 93 / 120, 149
// With more than one tile of atoms, both sets of nodes and twice the passes over
// the atoms are repeated, and it pays up to half as many boxes only (400 atoms,
// dz2 tip): 64 boxes 243 / 174 / 140, 128 244 / 174 / 206, 216 263 / 230 / 359,
// 392 346 / 400 / 615.  (A batch's atoms are not known here.)
int box_split(unsigned boxes, bool two_sets)
{
    const unsigned cus = two_sets ? 128 : 256;
    return boxes <= cus * 3 / 4 ? 4 : boxes <= cus * 7 / 4 ? 2 : 1;
}

template <bool LJ, int NS, bool Z0, bool WE, bool SEP>
void launch_o(const FFArgs &A0, bool ortho, const AtomRec *atoms, void *out, const BatchLaunch *b, hipStream_t st)
{
    dim3 block(kThreads);
    FFArgs A = A0;
    if (ortho) set_boxes(A);
    dim3 grid(b ? (unsigned)b->nbricks : (unsigned)A.nbx * A.nby * A.nbz);
    if (ortho) {
        const int split = box_split(grid.x, !b && A.natoms > kBoxTile);
        grid.x *= split;
        hipLaunchKernelGGL((ff_box_kernel<LJ, NS, Z0, WE, SEP>), grid, block, 0, st, A, far_table(), b ? b->items : nullptr,
                           b ? b->prefix : nullptr, b ? b->nitems : 0, atoms, (float4 *)out, split);
    } else if (b) {
        if (LJ && NS > 0 && b->qskip)
            hipLaunchKernelGGL((ff_f32_batch_kernel<LJ, NS, Z0, WE, (LJ && NS > 0), SEP>), grid, block, 0, st, A, b->items,
                               b->prefix, b->nitems, atoms, (float4 *)out);
        else
            hipLaunchKernelGGL((ff_f32_batch_kernel<LJ, NS, Z0, WE, false, SEP>), grid, block, 0, st, A, b->items,
                               b->prefix, b->nitems, atoms, (float4 *)out);
    } else {
        hipLaunchKernelGGL((ff_f32_kernel<LJ, NS, Z0, WE, SEP>), grid, block, 0, st, A, atoms, (float4 *)out);
    }
}

template <bool LJ, int NS, bool Z0, bool WE>
void launch_s(const FFArgs &A, bool ortho, const AtomRec *atoms, void *out, const BatchLaunch *b, hipStream_t st)
{
    if (A.mode == 0) launch_o<LJ, NS, Z0, WE, true>(A, ortho, atoms, out, b, st);
    else launch_o<LJ, NS, Z0, WE, false>(A, ortho, atoms, out, b, st);
}

template <bool LJ, bool WE>
int launch_ns(int ns, bool z0, const FFArgs &A, bool ortho, const AtomRec *atoms, void *out, const BatchLaunch *b,
              hipStream_t st)
{
    switch (ns) {
    case 0: launch_s<LJ, 0, false, WE>(A, ortho, atoms, out, b, st); break;
    case 1: z0 ? launch_s<LJ, 1, true, WE>(A, ortho, atoms, out, b, st) : launch_s<LJ, 1, false, WE>(A, ortho, atoms, out, b, st); break;
    case 2: z0 ? launch_s<LJ, 2, true, WE>(A, ortho, atoms, out, b, st) : launch_s<LJ, 2, false, WE>(A, ortho, atoms, out, b, st); break;
    case 3: z0 ? launch_s<LJ, 3, true, WE>(A, ortho, atoms, out, b, st) : launch_s<LJ, 3, false, WE>(A, ortho, atoms, out, b, st); break;
    case 4: z0 ? launch_s<LJ, 4, true, WE>(A, ortho, atoms, out, b, st) : launch_s<LJ, 4, false, WE>(A, ortho, atoms, out, b, st); break;
    default: set_error("n_stencil must be 0..4"); return -2;
    }
    return 0;
}

}  // namespace

long long ff_boxes(const int n[3])
{
    long long m = 1;
    for (int k = 0; k < 3; k++) m *= (n[k] + kBox - 1) / kBox;
    return m;
}

int launch_ff_f32(const FFArgs &A, bool z0, bool with_lj, bool with_energy, const AtomRec *atoms, void *out,
                  const BatchLaunch *batch, bool ortho, hipStream_t st)
{
    if (with_lj) {
        if (with_energy) return launch_ns<true, true>(A.ns, z0, A, ortho, atoms, out, batch, st);
        return launch_ns<true, false>(A.ns, z0, A, ortho, atoms, out, batch, st);
    }
    if (with_energy) return launch_ns<false, true>(A.ns, z0, A, ortho, atoms, out, batch, st);
    return launch_ns<false, false>(A.ns, z0, A, ortho, atoms, out, batch, st);
}

}  // namespace pp
