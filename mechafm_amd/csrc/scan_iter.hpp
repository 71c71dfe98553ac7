// Fast scan, FP64, one whole minimiser iteration per loop trip.
//
// The kernels of scan_fast.hpp make one evaluation per trip and carry each
// group's phase in its state: right for many columns of large tables, but a
// trip outside the site sums then costs thousands of cycles (spilled state,
// scalar loads of the tables, both branches of the state machine).  A scan of
// up to a few tens of thousands of columns is bound by exactly that: each
// column is one chain of ~8 000 dependent evaluations.  Here
//   * the two evaluations of a midpoint iteration (four of RK4) follow each
//     other in straight code, all groups of a wave in step; a group whose
//     height is done takes its output evaluation with the others' first one;
//   * the molecule's constants are loaded once, into scalar registers as far as
//     those go (21 to 44 values of the site kernels, 55 to 61 of the force grids',
//     68 to 132 of the images' spill into lanes of vector registers); RES sites of
//     each lane sit in vector registers, the rest streams from LDS two sites ahead;
//   * groups of 16 and more lanes are summed on the FP64 matrix unit;
//   * a force grid is read by eight lanes a column, one corner each, kept in
//     registers until the cell changes.
// What bounds it now: FP64 issue (4 cycles an instruction; one that needs the
// last one's result waits 8, so two waves a SIMD fill the pipe) and, for few
// columns, the length of the longest column's chain, in which an iteration's
// evaluations follow each other although the midpoint step's two points are known
// together (of RK4's four, the first two).  The images' kernels use all 256
// vector registers and 84 to 112 B of scratch a lane, a few of the others 36 B.
// Measured (kernel ms, general kernels -> now):
//   one column over 96 sites                                      16.6 -> 3.0
//   101 x 101 columns x 41 heights, 96 charge-free flat sites     32.2 -> 12.6
//   33 x 33 x 41, RK4, 131 charged sites                          51 -> 16.5
//   128 x 128 x 36 through a force grid                           24.1 -> 6.9
//   128 x 128 x 30, 150 charged flat sites                        54.9 -> 18.3
//   64 flat molecules of 20 to 400 charged sites, 64 x 64 x 40    402 -> 359
//   64 x 64 x 40, 2000 sites with nine images and a potential     437 -> 244
// (as sites of different heights the flat ones took 13.2, 20.2 and 392 where the
// flat kernels took 12.5, 18.6 and 361).  Many columns over few sites stay with the
// general kernels, one lane a column (one_lane_is_faster, api.cpp).
// Tried and left out: flat or not decided in the kernel (RK4 17 -> 21: both
// bodies' code and registers), charge-free sites sharing a reciprocal by fours
// (the chain grows: one column 3.2 -> 3.9).
#pragma once
#include "../../include/mafm.h"
#include <type_traits>

#include "scan_fast.hpp"

namespace mafm {
namespace {

// One LJ (+ Coulomb) site as the pair term below reads it (48 B: three 16 B
// LDS reads, and 12 banks between the sites of neighbouring lanes, so eight
// lanes' 16 B reads never share a bank).
struct SiteLJ {
    double x, y, z;
    double q0, q1, qc;
};

// 1 / sqrt(x) and 1 / x from the hardware seeds (~5e-8) by one third-order
// step each: error far below an ulp before rounding, and a shorter chain than
// two Newton steps.
__device__ inline double rsq64h(double x) {
    const double y = __builtin_amdgcn_rsq(x);
    const double e = fma(-x * y, y, 1.0);
    return fma(y * e, fma(e, 0.375, 0.5), y);
}
__device__ inline double rcp64h(double x) {
    const double r = __builtin_amdgcn_rcp(x);
    const double e = fma(-x, r, 1.0);
    return fma(r, fma(e, e, e), r);
}

// Which lanes of a wave form pixel group `grp`, and a lane's place in it.
// Groups of 4 and 8 are neighbouring lanes.  Groups of 16 are the blocks of
// v_mfma_f64_4x4x4_4b (lanes that share bits 2-3: operand A holds row lane &
// 3, column lane >> 4 of its block, operand B and the result row lane >> 4,
// column lane & 3), groups of 32 two such blocks, 64 the wave.
template <int G>
struct Lanes {
    static __device__ int place(int lane) {
        if (G <= 8) return lane % G;
        if (G == 16) return (lane & 3) | (lane >> 4) << 2;
        if (G == 32) return (lane & 7) | (lane >> 4) << 3;
        return lane;
    }
    static __device__ int first(int lane) {   // the group's leading lane
        if (G <= 8) return lane - lane % G;
        if (G == 16) return lane & 12;
        if (G == 32) return lane & 8;
        return 0;
    }
};

// Sums of r[0 .. N-1] over the lanes of each group, the same values on each
// of them; all lanes of the wave active.
//   G <= 8: DPP butterflies, value by value in step (three instructions a
//   value and stage, and no wait between a write and its DPP read).
//   G >= 16: two contractions on the FP64 matrix unit, the first with 0 / 1 matrices.
//   The first puts value q's sum over a block's columns into column q of one
//   result (the values' matrices accumulate), the second adds the four rows;
//   the sums are then in lanes 0-3 of every quad and four DPP moves hand them
//   out.  Products with 0 and 1 are exact, except that 0 x inf is NaN: one
//   value's infinity makes the others NaN.  An iteration is lost either way (the
//   mixing's |f| is infinite).  PICK, for sums that a record may hold: the first
//   product is with ones, and the lanes pick the value of their column: the same
//   bits where they are finite; in every sum 0.999 of the time over 57 scans, but up
//   to 4 % more for the midpoint step over few sites, whose records alone take it.
//   16 lanes, 3 values: 4 matrix instructions (16 cycles of the FP64 pipe each) and
//   6 moves against 36 instructions of the butterflies.
//   No addition here may be contracted with the product a caller's value comes
//   from: a lane's a * b + (its neighbour's, rounded) is not its neighbour's sum,
//   the lanes of a column then carry different states, and a long relaxation
//   along a ridge drives them 1e-4 A apart.
template <int G, int N, bool PICK>
__device__ inline void group_sums(double* r) {
#pragma clang fp contract(off)
    if constexpr (G <= 8) {
#pragma unroll
        for (int q = 0; q < N; ++q) r[q] += dpp_f64<0xB1>(r[q]);
#pragma unroll
        for (int q = 0; q < N; ++q) r[q] += dpp_f64<0x4E>(r[q]);
        if (G >= 8) {
#pragma unroll
            for (int q = 0; q < N; ++q) r[q] += dpp_f64<0x141>(r[q]);
        }
    } else {
        const int lane = threadIdx.x & 63;
        double d = 0.0;
        if (PICK) {
            double row[N];
#pragma unroll
            for (int q = 0; q < N; ++q) row[q] = __builtin_amdgcn_mfma_f64_4x4x4f64(r[q], 1.0, 0.0, 0, 0, 0);
            const bool odd = lane & 1, high = lane & 2;
            const double lo = odd ? row[1] : row[0], hi = N > 3 && odd ? row[N - 1] : row[2];
            d = high ? hi : lo;
        } else {
#pragma unroll
            for (int q = 0; q < N; ++q)
                d = __builtin_amdgcn_mfma_f64_4x4x4f64(r[q], (lane & 3) == q ? 1.0 : 0.0, d, 0, 0, 0);
        }
        d = __builtin_amdgcn_mfma_f64_4x4x4f64(1.0, d, 0.0, 0, 0, 0);
        // blocks 0 + 1 and 2 + 3 (lane ^ 4 = half-row mirror of a mirrored quad),
        // then all four (lane ^ 8 = rotation by 8 within the row)
        if (G >= 32) d += dpp_f64<0x141>(dpp_f64<0x1B>(d));
        if (G >= 64) d += dpp_f64<0x128>(d);
        r[0] = dpp_f64<0x00>(d);
        r[1] = dpp_f64<0x55>(d);
        r[2] = dpp_f64<0xAA>(d);
        if (N > 3) r[3] = dpp_f64<0xFF>(d);
    }
}

// One site's force (acc 0-2) and, when E, energy (acc 3) on a tip at t.
// COUL: s = -2 / r comes out of the Newton step z0 (r2 z0^2 - 3) in three
// operations instead of four; its powers of two are folded into the site's
// constants (q0 = 6 es6 / 2^8, q1 = 12 es12 / 2^14, qc = -qq / 2^3, all
// exact), acc 3 collects 3 E.  Without Coulomb: q0 = 6 es6, q1 = 12 es12,
// acc 3 collects 12 E.
// FLAT: the sites have one height, and tz is the tip's above it, dz2 its square;
// acc 2 collects the force over tz (two instructions of 23 a charged site saved).
template <bool COUL, bool E, bool FLAT>
__device__ inline void pair_acc(const SiteLJ& st, double tx, double ty, double tz, double dz2, double* acc) {
    const double dx = tx - st.x, dy = ty - st.y, dz = FLAT ? tz : tz - st.z;
    const double r2 = fma(dx, dx, fma(dy, dy, FLAT ? dz2 : dz * dz));
    double fs;
    if (COUL) {
        const double z0 = __builtin_amdgcn_rsq(r2);
        const double s = z0 * fma(r2, z0 * z0, -3.0);
        const double A = s * s;
        const double B = A * A * A;
        const double fl = fma(st.q1, B, -st.q0);
        const double ec = st.qc * s;
        fs = fma(fl, B, ec) * A;
        if (E) acc[3] = fma(12.0, ec, fma(B, fl - st.q0, acc[3]));
    } else {
        const double ir2 = rcp64p(r2);
        const double ir6 = ir2 * ir2 * ir2;
        const double fl = fma(st.q1, ir6, -st.q0);
        fs = fl * ir6 * ir2;
        if (E) acc[3] = fma(ir6, fl - st.q0, acc[3]);
    }
    acc[0] = fma(fs, dx, acc[0]);
    acc[1] = fma(fs, dy, acc[1]);
    acc[2] = FLAT ? acc[2] + fs : fma(fs, dz, acc[2]);
}

// One charge-free site and its 3 x 3 images: ax[i] / ay[j] = tip minus the
// images' shift along x / y.  The squared distances are sums of three and
// three parts, the nine reciprocals come from one hardware reciprocal (the
// product of all, refined, times the products of the others: 30 instructions
// instead of 54), and the force's components are sums of row and column sums:
// 13.3 instructions a pair instead of 20.
template <bool E>
__device__ inline void images_acc(const double4& st, double q1, const double* ax, const double* ay, double pz, double* acc) {
    const double dz = pz - st.z, dz2 = dz * dz;
    double dx[3], dy[3], xz[3], yy[3];
#pragma unroll
    for (int i = 0; i < 3; ++i) {
        dx[i] = ax[i] - st.x;
        xz[i] = fma(dx[i], dx[i], dz2);
        dy[i] = ay[i] - st.y;
        yy[i] = dy[i] * dy[i];
    }
    double r2[3][3], p01[3], row[3];
#pragma unroll
    for (int i = 0; i < 3; ++i) {
#pragma unroll
        for (int j = 0; j < 3; ++j) r2[i][j] = xz[i] + yy[j];
        p01[i] = r2[i][0] * r2[i][1];
        row[i] = p01[i] * r2[i][2];
    }
    const double q01 = row[0] * row[1];
    const double all = rcp64h(q01 * row[2]);
    const double t2 = all * row[2];
    const double irow[3] = {t2 * row[1], t2 * row[0], all * q01};
    double cy[3], sum = 0, s6 = 0, sg = 0;
#pragma unroll
    for (int i = 0; i < 3; ++i) {
        const double t = irow[i] * r2[i][2];
        const double ir2[3] = {t * r2[i][1], t * r2[i][0], irow[i] * p01[i]};
        double rx = 0;
#pragma unroll
        for (int j = 0; j < 3; ++j) {
            const double ir6 = ir2[j] * ir2[j] * ir2[j];
            const double gl = fma(q1, ir6, -st.w) * ir6;
            const double fs = gl * ir2[j];
            rx = j ? rx + fs : fs;
            cy[j] = i ? cy[j] + fs : fs;
            if (E) {
                s6 += ir6;
                sg += gl;
            }
        }
        acc[0] = fma(dx[i], rx, acc[0]);
        sum += rx;
    }
#pragma unroll
    for (int j = 0; j < 3; ++j) acc[1] = fma(dy[j], cy[j], acc[1]);
    acc[2] = fma(dz, sum, acc[2]);
    if (E) acc[3] = fma(-st.w, s6, acc[3] + sg);   // 12 E = sum of ir6 (fl - 6 es6)
}
// x, or 1e15 with its sign where it is finite and larger
__device__ inline double keep_near(double x) {
    return fabs(x) > 1e15 && fabs(x) < INFINITY ? copysign(1e15, x) : x;
}

// Tip-dummy constants of the workgroup's molecule
struct Dummy {
    double p0, p1, qq, k, r0, kk;
    bool coul;
};

// tip_dummy for a Lennard-Jones dummy: VDW, Coulomb and the lateral spring
// (interactions.cpp:15-51, 252-266) at t with the dummy at d.  A spring with
// r0 = 0 is linear in the displacement and needs no root.
template <bool E>
__device__ inline void dummy_terms(const Dummy& D, double dx, double dy, double dz, double tx, double ty, double tz,
                                   double* o) {
    const double rx = tx - dx, ry = ty - dy, rz = tz - dz;
    const double rl2 = fma(rx, rx, ry * ry);
    const double r2 = fma(rz, rz, rl2);
    const double i2 = rcp64h(r2);
    const double i6 = i2 * i2 * i2;
    const double ta = D.p1 * i6 * i6, tb = D.p0 * i6;
    double s = fma(12.0, ta, -6.0 * tb) * i2;
    double e = ta - tb;
    if (D.coul) {
        asm volatile("");                 // a uniform branch, not eleven selected instructions
        const double ec = D.qq * rsq64h(r2);
        s = fma(ec, i2, s);
        if (E) e += ec;
    }
    double h = -D.kk;
    if (D.r0 == 0.0) {
        if (E) e = fma(D.k, rl2, e);
    } else if (rl2 > 1e-20) {
        const double irl = rsq64h(rl2);
        const double dr = fma(rl2, irl, -D.r0);
        h = -D.kk * dr * irl;
        if (E) e = fma(D.k * dr, dr, e);
    } else {
        h = 0.0;
        const double dr = sqrt(rl2) - D.r0;
        if (E) e = fma(D.k * dr, dr, e);
    }
    o[0] = (s + h) * rx;
    o[1] = (s + h) * ry;
    o[2] = s * rz;
    o[3] = e;
}

// A force grid's corner held by one lane of a group of eight: the lane's bits
// 2, 1, 0 choose the upper corner along x, y, z.  Against one lane a column
// that gathers all eight corners in each evaluation: 16 384 columns make 2 048
// waves instead of 256, and the gathers (99.6 % L2 hits, but ~700 cycles each)
// are left out while the tip stays in its 0.05 A cell.
struct Corner {
    double4 v;
    long idx;
};

// The workgroup's force grid, held in scalar registers (read through the
// table, each field would be a scalar load with its wait in every lookup).
// near: row and point numbers fit the 24-bit multiplier and 32 bits.
struct Grid {
    double off[3], inv[3];
    int n[3];
    bool diagonal, periodic, near;
    const double4* fe;
    cptr<DevGrid> d;
};

// What a column's tip-surface force is made of: the molecule's sites, a force
// grid, or the sites' 3 x 3 periodic images and, where the system has one, an
// external potential.
// ITER_FLAT: ITER_SITES where every molecule's sites have one height
enum { ITER_SITES = 0, ITER_GRID = 1, ITER_IMAGES = 2, ITER_FLAT = 3 };

// Sites of a lane that shares n sites with G - 1 others, padded: at least the
// resident ones, and a multiple of two past them (res = 1, the images' kernels:
// no padding of the share).
__host__ __device__ inline int padded_share(int n, int G, int res) {
    const int per = (n + G - 1) / G;
    if (res == 1) return per > 1 ? per : 1;
    return res + (per > res ? (per - res + 1) / 2 * 2 : 0);
}
// The resident count for molecules of n sites or more: a lane's whole share up
// to 6, else 8 where the registers of two waves a SIMD hold them (groups of up
// to 8 lanes with the midpoint step; 6 elsewhere, 8 would spill).
inline int resident_sites(int n, int G, bool mid) {
    const int per = (n + G - 1) / G, most = G <= 8 && mid ? 8 : 6;
    return per <= 2 ? 2 : (per <= 6 ? per : most);
}

// A branch that one trip in a hundred takes: laid out behind the others, so that
// the registers it needs are not spilled on their way (57 scans of all modes: 0.97 of
// the time).  Not in the images' kernels without the midpoint step, which it costs
// up to a third (Euler, 32 sites, 64 x 64 x 6: 1.05 -> 1.46 ms).
#define SELDOM(branch) (IMG && !MID ? (branch) : __builtin_expect((branch), 0))

// RES of a lane's sites stay in registers for the whole scan (the first RES
// of its share, loaded from the staged copy); the others stream from LDS two
// at a time.
template <int G, int RES, bool COUL, int MODE, bool MID>
__device__ __attribute__((always_inline)) inline void scan_iter_body(const ScanArgs& a) {
    constexpr bool GRID = MODE == ITER_GRID, IMG = MODE == ITER_IMAGES, FLAT = MODE == ITER_FLAT;
    const int lane = threadIdx.x & 63;
    const int gl = Lanes<G>::place(lane);
    const bool leader = gl == 0;
    const int n_cols = a.nx * a.ny;
    const uint64_t lt_mask = (lane == 0) ? 0ull : (~0ull >> (64 - lane));
    extern __shared__ double2 lds_iter[];
    __shared__ int next_shared;
    SiteLJ* const lsite = reinterpret_cast<SiteLJ*>(lds_iter);
    // the images' kernels: {x, y, z, q0} and, behind the most sites of a molecule, q1 (40 B a site)
    double4* const lxyz = reinterpret_cast<double4*>(lds_iter);
    double* const lq1 = reinterpret_cast<double*>(lds_iter) + 4 * (size_t)a.lds_sites;

    int rk = __builtin_amdgcn_readfirstlane(pick_rank(a, blockIdx.x, gridDim.x));
    int m = a.mol_order[rk];
    SiteLJ res[RES > 0 ? RES : 1];
    Dummy D;
    int per_lane = 0;                 // sites of a lane, a multiple of two past the resident ones
    double flat_z = 0;                // their height where they have one
    // the corners last read, for the half steps and the full steps apart: a
    // pair of points on both sides of a cell face does not reload each other's
    Corner cn0 = {{0, 0, 0, 0}, -1}, cn1 = cn0;
    Grid g;
    bool has_grid = false;
    double img_x[3], img_y[3];        // the images' shifts along x and y
    const int bit[3] = {gl >> 2 & 1, gl >> 1 & 1, gl & 1};
    const double wsign[3] = {bit[0] ? 1.0 : -1.0, bit[1] ? 1.0 : -1.0, bit[2] ? 1.0 : -1.0};
    const double wbase[3] = {1.0 - bit[0], 1.0 - bit[1], 1.0 - bit[2]};
    auto stage = [&](int mol) {
        cptr<DevMol> M = as_const(a.mols) + mol;
        D.p0 = M->td_p0; D.p1 = M->td_p1; D.qq = M->td_qq; D.k = M->td_k; D.r0 = M->td_r0;
        D.kk = 2 * D.k;
        D.coul = M->td_coul != 0;
        has_grid = GRID || (IMG && M->potential_grid >= 0);
        if (has_grid) {
            g.d = as_const(a.grids) + (GRID ? M->force_grid : M->potential_grid);
#pragma unroll
            for (int d = 0; d < 3; ++d) {
                g.off[d] = g.d->offset[d];
                g.inv[d] = g.d->inv[4 * d];
                g.n[d] = g.d->n[d];
            }
            g.diagonal = g.d->orthogonal;
            g.periodic = g.d->periodic;
            g.fe = g.d->fe64;
            g.near = (long)g.n[0] * g.n[1] < (1 << 24) && g.n[2] < (1 << 24) &&
                     (long)g.n[0] * g.n[1] * g.n[2] < INT32_MAX;
            cn0.idx = cn1.idx = -1;
        }
        if (GRID) return;
        if (IMG) {
#pragma unroll
            for (int d = 0; d < 3; ++d) {
                img_x[d] = M->shift[3 * d][0];
                img_y[d] = M->shift[d][1];
            }
        }
        const int n = M->n_seg[0] + M->n_seg[1];
        per_lane = padded_share(n, G, RES);
        if (FLAT) flat_z = n > 0 ? as_const(a.segf64)[M->seg_off].z + M->shift[0][2] : 0.0;
        __syncthreads();
        for (int t = threadIdx.x; t < per_lane * G; t += blockDim.x) {
            // padding: no force, at a distance that is finite and never zero (nine
            // images' squared distances are multiplied), where no scan goes
            SiteLJ s = {1e15, 1e15, 1e15, 0, 0, 0};
            if (t < n) {
                const SiteF64 f = a.segf64[M->seg_off + t];
                s.x = f.x; s.y = f.y; s.z = f.z;
                if (!IMG) { s.x += M->shift[0][0]; s.y += M->shift[0][1]; s.z += M->shift[0][2]; }
                s.q0 = COUL ? f.p0 * 0x1p-8 : f.p0;
                s.q1 = COUL ? f.p1 * 0x1p-14 : f.p1;
                s.qc = f.qq * -0x1p-3;
            }
            if (IMG) {
                lxyz[t] = make_double4(s.x, s.y, s.z, s.q0);
                lq1[t] = s.q1;
            } else {
                lsite[t] = s;
            }
        }
        __syncthreads();
#pragma unroll
        for (int u = 0; u < (IMG ? 0 : RES); ++u) res[u] = lsite[u * G + gl];
    };
    stage(m);

    // group state (identical on the G lanes of a group)
    int col = -1, k = 0, n_tot = 1, nnn = 0, flags = 0;
    bool out = false;                 // waits for the evaluation its record holds
    double dmx = 0, dmy = 0, dmz = 1.0e3, tx = 0, ty = 0, tz = 1.0e3, vx = 0, vy = 0, vz = 0;
    double e = 0, dt = a.dt, alpha = 0.1;
    const double dt_max = 10 * a.dt;
    // checkConvergence (minimiser.cpp:15-37): the part the minterm does not test always passes
    const bool any_e = a.minterm == 1, any_f = a.minterm == 0;
    const double ftol2 = a.ftol * a.ftol;
    const bool track = a.margins != nullptr;
    float mgf = INFINITY, mge = INFINITY, mgp = INFINITY;   // the height's decision margins
    int64_t trips = 0;
    int32_t active = 0;

    // this lane's corner of the grid cell around p: its weight, the samples in
    // cn.v; counts: the point is one of the column's evaluations, so leaving
    // the grid is noted
    auto corner = [&](Corner& cn, bool counts, double px, double py, double pz) {
        double q[3];
        if (g.diagonal) {
            q[0] = (px - g.off[0]) * g.inv[0];
            q[1] = (py - g.off[1]) * g.inv[1];
            q[2] = (pz - g.off[2]) * g.inv[2];
        } else {
            mat_vec(g.d->inv, px - g.off[0], py - g.off[1], pz - g.off[2], q[0], q[1], q[2]);
        }
        int gp[3], at[3], fl = 0;
        bool inside = true;
#pragma unroll
        for (int d = 0; d < 3; ++d) {
            gp[d] = (int)floor(q[d]);
            at[d] = gp[d] + bit[d];
            inside &= (unsigned)gp[d] < (unsigned)(g.n[d] - 1);
        }
        if (!inside) {   // the clamp and wrap rules of grid_lookup
#pragma unroll
            for (int d = 0; d < 3; ++d) {
                const int n = g.n[d];
                if (!g.periodic) {
                    if (gp[d] < 0) { gp[d] = 0; fl |= REC_GRID_CLAMP; }
                    else if (gp[d] >= n) { gp[d] = n - 1; fl |= REC_GRID_CLAMP; }
                    if (gp[d] + 1 >= n) fl |= REC_OUT_OF_GRID;
                }
                int i = gp[d] + bit[d];
                if (g.periodic && (i < 0 || i >= n)) i -= (int)floor((double)i / n) * n;
                at[d] = i < 0 ? 0 : (i >= n ? n - 1 : i);   // inside the grid even for non-finite positions
            }
            if (counts) flags |= fl;
        }
        // f on an upper corner, 1 - f on a lower one, each rounded once
        const double w = fma(q[0] - gp[0], wsign[0], wbase[0]) * fma(q[1] - gp[1], wsign[1], wbase[1]) *
                         fma(q[2] - gp[2], wsign[2], wbase[2]);
        long idx;
        if (g.near) idx = (int)(__umul24(__umul24(at[0], g.n[1]) + at[1], g.n[2]) + at[2]);
        else idx = ((long)at[0] * g.n[1] + at[1]) * g.n[2] + at[2];
        if (idx != cn.idx) {
            cn.v = g.fe[idx];
            cn.idx = idx;
        }
        return w;
    };
    // tip-surface force and energy at p, summed over the group's lanes; record:
    // for some group's record
    auto surface = [&](auto want_e, auto record, Corner& cn, bool counts, double px, double py, double pz, double* r) {
        constexpr bool E = decltype(want_e)::value, PICK = decltype(record)::value;
        r[3] = 0;
        if constexpr (GRID) {
            const double w = corner(cn, counts, px, py, pz);
            r[0] = w * cn.v.x;
            r[1] = w * cn.v.y;
            r[2] = w * cn.v.z;
            if (E) r[3] = w * cn.v.w;
            group_sums<G, E ? 4 : 3, PICK>(r);
        } else if constexpr (IMG) {
            r[0] = r[1] = r[2] = 0;
            if (has_grid && gl < 8) {   // eight of the column's lanes hold the potential's corners
                const double w = corner(cn, counts, px, py, pz);
                r[0] = w * cn.v.x;
                r[1] = w * cn.v.y;
                r[2] = w * cn.v.z;
                if (E) r[3] = 12.0 * w * cn.v.w;
            }
            // a tip thrown past 1e15 A feels nothing here; nearer, it keeps the
            // product of nine squared distances inside the exponent range
            if (__any(fmax(fmax(fabs(px), fabs(py)), fabs(pz)) > 1e15)) {
                px = keep_near(px);
                py = keep_near(py);
                pz = keep_near(pz);
            }
            const double ax[3] = {px - img_x[0], px - img_x[1], px - img_x[2]};
            const double ay[3] = {py - img_y[0], py - img_y[1], py - img_y[2]};
            int t = gl;
            double4 st = lxyz[t];
            double q1 = lq1[t];
            for (int u = 1; u < per_lane; ++u) {
                t += G;
                const double4 st2 = lxyz[t];
                const double q2 = lq1[t];
                images_acc<E>(st, q1, ax, ay, pz, r);
                st = st2;
                q1 = q2;
            }
            images_acc<E>(st, q1, ax, ay, pz, r);
            group_sums<G, E ? 4 : 3, PICK>(r);
            if (E) r[3] *= 1.0 / 12.0;
        } else {
            r[0] = r[1] = r[2] = 0;
            const double z = FLAT ? pz - flat_z : pz, dz2 = z * z;
#pragma unroll
            for (int u = 0; u < RES; ++u) pair_acc<COUL, E, FLAT>(res[u], px, py, z, dz2, r);
            if (per_lane > RES) {
                // two sites in flight while two are evaluated, in turn
                const SiteLJ* s = lsite + RES * G + gl;
                SiteLJ a0 = s[0], a1 = s[G];
                for (int left = per_lane - RES - 2;; left -= 4) {
                    SiteLJ b0, b1;
                    if (left > 0) {
                        b0 = s[2 * G];
                        b1 = s[3 * G];
                    }
                    pair_acc<COUL, E, FLAT>(a0, px, py, z, dz2, r);
                    pair_acc<COUL, E, FLAT>(a1, px, py, z, dz2, r);
                    if (left <= 0) break;
                    s += 4 * G;
                    if (left > 2) {
                        a0 = s[0];
                        a1 = s[G];
                    }
                    pair_acc<COUL, E, FLAT>(b0, px, py, z, dz2, r);
                    pair_acc<COUL, E, FLAT>(b1, px, py, z, dz2, r);
                    if (left <= 2) break;
                }
            }
            if (FLAT) r[2] *= z;
            group_sums<G, E ? 4 : 3, PICK>(r);
            if (E) r[3] *= COUL ? 1.0 / 3.0 : 1.0 / 12.0;
        }
    };
    // the whole list: tip-surface plus, where with_d, tip-dummy.  The sum is never
    // contracted with the product a dummy value comes from: it would be in the call
    // whose with_d is known and not in the other, and a column's rounding would
    // depend on whether a neighbour in its wave has a record to write.
    auto total = [&](auto want_e, auto record, Corner& cn, bool counts, bool with_d, double px, double py, double pz,
                     double* r) {
#pragma clang fp contract(off)
        constexpr bool E = decltype(want_e)::value;
        double d[4];
        dummy_terms<E>(D, dmx, dmy, dmz, px, py, pz, d);
        surface(want_e, record, cn, counts, px, py, pz, r);
#pragma unroll
        for (int q = 0; q < (E ? 4 : 3); ++q) r[q] += with_d ? d[q] : 0.0;
    };
    constexpr std::true_type yes{};
    constexpr std::false_type no{};
    auto begin_height = [&]() {
        n_tot = 1; dt = a.dt; alpha = 0.1; nnn = 0; flags = 0;
        mgf = mge = mgp = INFINITY;
        out = n_tot >= a.maxsteps;
    };
    // the record of a group whose height is done, from the tip-surface values
    // at the relaxed tip; then the next height, or no column
    auto emit = [&](const double* r) {
        if (leader) {
            const int i = col / a.ny, j = col - i * a.ny;
            DevRecord rec;
            rec.x = i * a.dx; rec.y = j * a.dy; rec.z = dmz;
            rec.fx = r[0]; rec.fy = r[1]; rec.fz = r[2];
            rec.rx = tx - dmx; rec.ry = ty - dmy; rec.rz = tz - dmz;
            rec.e = r[3];
            rec.n_steps = n_tot;
            rec.flags = flags | (n_tot >= a.maxsteps ? REC_UNCONVERGED : 0);
            const long ri = (as_const(a.mols) + m)->rec_off + ((long)col * a.nz + k);
            a.rec[ri] = rec;
            if (track) a.margins[ri] = make_float4(mgf, mge, mgp, 0.f);
            if (a.col_done) column_progress(a, (long)m * n_cols + col, k + 1);
        }
        dmz -= a.dz;
        tz -= a.dz;
        if (++k >= a.nz) {
            col = -1;
            out = false;
        } else {
            begin_height();
        }
    };
    // FIREMinimisation's iteration tail (minimiser.cpp:102-126) after a step
    // that left force f and energy en
    auto fire_tail = [&](double fx, double fy, double fz, double en) {
        const double f2 = fma(fx, fx, fma(fy, fy, fz * fz));
        const double de = fabs(en - e);
        e = en;
        if (track) test_margins(a, f2, de, mgf, mge);
        if ((any_e | (de < a.etol)) & (any_f | (f2 < ftol2))) {
            out = true;
            return;
        }
        const double p = fma(vx, fx, fma(vy, fy, vz * fz));
        const double v2 = fma(vx, vx, fma(vy, vy, vz * vz));
        if (track) fire_margin(p, v2, v2 > 0 ? rsq64h(v2) : 0.0, mgp);
        // |v| / |f| by one root; 0 where the force has no direction (vectors.hpp:107-114)
        // (beyond |f| = 2^200, where a tip was thrown off an atom, of the product over
        // 2^1000: it would overflow where its factors do not; 0 to 2 % of an iteration,
        // a branch to two roots 3 to 5)
        const bool thrown = f2 > 0x1p400;
        const double vf = v2 * (f2 * (thrown ? 0x1p-1000 : 1.0));
        const double s = (f2 > 1e-20 && vf > 1e-280) ? alpha * (thrown ? 0x1p-500 : 1.0) * v2 * rsq64h(vf) : 0.0;
        const double b = 1 - alpha;
        const bool up = !(p < 0);
        vx = up ? fma(s, fx, b * vx) : 0.0;
        vy = up ? fma(s, fy, b * vy) : 0.0;
        vz = up ? fma(s, fz, b * vz) : 0.0;
        if (up) {
            if (nnn > 5) {
                dt = fmin(dt * 1.1, dt_max);
                alpha *= 0.99;
            }
            ++nnn;
        } else {
            nnn = 0;
            dt *= 0.5;
            alpha = 0.1;
        }
        ++n_tot;
        out = n_tot >= a.maxsteps;
    };

    for (;;) {
        // ---- groups without a column steal one from molecule m
        if (SELDOM(__any(col < 0))) {
            const bool need = leader && col == -1;
            const uint64_t need_mask = __ballot(need);
            if (need_mask) {
                const int first = __ffsll((unsigned long long)need_mask) - 1;
                int base = 0;
                if (lane == first) base = atomicAdd(&a.next_col[m], __popcll(need_mask));
                base = __shfl(base, first, 64);
                int got = col;
                if (need) {
                    const int c = base + __popcll(need_mask & lt_mask);
                    got = c < n_cols ? c : -2;
                }
                got = __shfl(got, Lanes<G>::first(lane), 64);
                if (col == -1) {
                    col = got;
                    if (col >= 0) {   // System copy, setDummyXY, setDummyZ (simulation.cpp:93-101)
                        cptr<DevMol> M = as_const(a.mols) + m;
                        const int i = col / a.ny, j = col - i * a.ny;
                        const double x = i * a.dx, y = j * a.dy;
                        dmx = x; dmy = y;
                        if (M->tip_pbc) wrap_xy(M->cell, M->cell_inv, M->offset, x, y, dmx, dmy);
                        dmz = a.zhigh;
                        tx = dmx; ty = dmy; tz = a.zhigh - M->tip_dummy_d;
                        vx = vy = vz = 0;
                        e = 0;
                        k = 0;
                        begin_height();
                    }
                }
            }
            if (!__any(col >= 0)) {
                // molecule m exhausted: the workgroup's waves move on together
                __syncthreads();
                if (threadIdx.x == 0) next_shared = next_rank(a, rk);
                __syncthreads();
                const int nr = __builtin_amdgcn_readfirstlane(next_shared);
                if (nr < 0) break;
                rk = nr;
                m = a.mol_order[rk];
                col = -1;
                stage(m);
                continue;
            }
        }
        const bool live = col >= 0 && !out;
        const bool emits = col >= 0 && out;
        double r[4];
        if constexpr (MID) {
            // half step: every running group at its tip, and the groups with a
            // finished height at theirs (tip-surface terms only)
            const double hx = dt / 2 * vx, hy = dt / 2 * vy, hz = dt / 2 * vz;
            if (SELDOM(__any(emits))) {
                total(yes, yes, cn0, true, !emits, tx, ty, tz, r);
                if (emits) emit(r);
            } else {
                total(no, no, cn0, true, true, tx, ty, tz, r);
            }
            const double ax = fma(dt / 2, r[0], vx), ay = fma(dt / 2, r[1], vy), az = fma(dt / 2, r[2], vz);
            total(yes, no, cn1, live, true, tx + hx, ty + hy, tz + hz, r);
            if (live) {
                tx = fma(dt, ax, tx); ty = fma(dt, ay, ty); tz = fma(dt, az, tz);
                vx = fma(dt, r[0], vx); vy = fma(dt, r[1], vy); vz = fma(dt, r[2], vz);
                fire_tail(r[0], r[1], r[2], r[3]);
            }
            trips += 2;
            active += 2 * live + emits;
        } else {
            // SD, FIRE with Euler or RK4: the stages of one iteration
            const bool sd = a.minimiser == 0, rk4 = !sd && a.integrator == 2;
            double px = tx, py = ty, pz = tz, wx = vx, wy = vy, wz = vz;      // stage point and velocity
            double bx = 0, by = 0, bz = 0, cx = 0, cy = 0, cz = 0, ce = 0;    // sums over the stages
            const int ns = rk4 ? 4 : 1;
            const bool any_emits = __any(emits);
            for (int s = 0; s < ns; ++s) {
                const bool record = s == 0 && any_emits;
                total(yes, yes, cn0, s == 0 || live, s > 0 || !emits, px, py, pz, r);
                if (SELDOM(record)) {
                    if (emits) emit(r);
                    if (!__any(live)) break;
                }
                if (!rk4) break;
                const double wt = (s == 1 || s == 2) ? 2.0 : 1.0;
                bx = fma(wt, wx, bx); by = fma(wt, wy, by); bz = fma(wt, wz, bz);
                cx = fma(wt, r[0], cx); cy = fma(wt, r[1], cy); cz = fma(wt, r[2], cz); ce = fma(wt, r[3], ce);
                const double h = s < 2 ? dt / 2 : dt;
                px = fma(h, wx, tx); py = fma(h, wy, ty); pz = fma(h, wz, tz);
                wx = fma(h, r[0], vx); wy = fma(h, r[1], vy); wz = fma(h, r[2], vz);
            }
            if (live) {
                if (sd) {                                      // minimiser.cpp:39-65
                    const double f2 = fma(r[0], r[0], fma(r[1], r[1], r[2] * r[2]));
                    const double de = fabs(r[3] - e);
                    e = r[3];
                    if (track) test_margins(a, f2, de, mgf, mge);
                    if ((any_e | (de < a.etol)) & (any_f | (f2 < ftol2))) {
                        out = true;
                    } else {
                        tx = fma(a.dt, r[0], tx); ty = fma(a.dt, r[1], ty); tz = fma(a.dt, r[2], tz);
                        ++n_tot;
                        out = n_tot >= a.maxsteps;
                    }
                } else if (rk4) {
                    const double h = dt / 6;
                    tx = fma(h, bx, tx); ty = fma(h, by, ty); tz = fma(h, bz, tz);
                    vx = fma(h, cx, vx); vy = fma(h, cy, vy); vz = fma(h, cz, vz);
                    fire_tail(cx / 6, cy / 6, cz / 6, ce / 6);
                } else {
                    tx = fma(dt, vx, tx); ty = fma(dt, vy, ty); tz = fma(dt, vz, tz);
                    vx = fma(dt, r[0], vx); vy = fma(dt, r[1], vy); vz = fma(dt, r[2], vz);
                    fire_tail(r[0], r[1], r[2], r[3]);
                }
            }
            trips += ns;
            active += ns * live + emits;
        }
    }
    if (lane == 0) atomicAdd((unsigned long long*)&a.counters[4], (unsigned long long)(trips * (64 / G)));
    if (leader && active) atomicAdd((unsigned long long*)&a.counters[5], (unsigned long long)active);
}

template <int G, int RES, bool COUL, int MODE, bool MID>
__global__ void __launch_bounds__(512, 2) k_scan_iter(ScanArgs a) {
    scan_iter_body<G, RES, COUL, MODE, MID>(a);
}

inline size_t iter_site_bytes(int mode) { return mode == ITER_IMAGES ? 40 : sizeof(SiteLJ); }

}  // namespace

struct IterLaunch {
    const ScanArgs& a;
    int n_blocks, W, n_min, n_max;
    hipStream_t st;
};

namespace {

template <int G, int RES, bool COUL, int MODE, bool MID>
hipError_t launch_one(const IterLaunch& L) {
    const size_t lds = MODE == ITER_GRID ? 0 : iter_site_bytes(MODE) * (size_t)G * padded_share(L.n_max, G, RES);
    const auto fn = &k_scan_iter<G, RES, COUL, MODE, MID>;
    if (lds > 64 * 1024) {
        const hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void*>(fn),
                                                 hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
        if (e != hipSuccess) return e;
    }
    ScanArgs a = L.a;
    a.lds_sites = G * padded_share(L.n_max, G, RES);
    hipLaunchKernelGGL(fn, dim3(L.n_blocks), dim3(64 * L.W), lds, L.st, a);
    return hipGetLastError();
}

template <int G, bool COUL, int MODE, bool MID>
hipError_t launch_res(const IterLaunch& L) {
    switch (resident_sites(L.n_min, G, MID)) {
        case 2: return launch_one<G, 2, COUL, MODE, MID>(L);
        case 3: return launch_one<G, 3, COUL, MODE, MID>(L);
        case 4: return launch_one<G, 4, COUL, MODE, MID>(L);
        case 5: return launch_one<G, 5, COUL, MODE, MID>(L);
        case 6: return launch_one<G, 6, COUL, MODE, MID>(L);
        default:
            if constexpr (G <= 8 && MID) return launch_one<G, 8, COUL, MODE, MID>(L);
            return hipErrorInvalidValue;
    }
}

}  // namespace

// The kernels of site tables, MODE ITER_SITES or ITER_FLAT.  Each combination is
// instantiated in a file of few: the runtime loads a file's kernels whole when the
// first of them is launched, and a program's first scan needs one of them (32 x 32
// x 4 with all in one file 12.9 ms, now 3.4).
template <bool COUL, int MODE, bool MID>
hipError_t launch_iter_sites(const IterLaunch& L, int G) {
    switch (G) {
        case 4: return launch_res<4, COUL, MODE, MID>(L);
        case 8: return launch_res<8, COUL, MODE, MID>(L);
        case 16: return launch_res<16, COUL, MODE, MID>(L);
        case 32: return launch_res<32, COUL, MODE, MID>(L);
        case 64: return launch_res<64, COUL, MODE, MID>(L);
        default: return hipErrorInvalidValue;
    }
}

}  // namespace mafm
