// Flexible scan (flexible on) and the System-level operators: interaction lists
// over whole systems, every free atom moving.
//
// One workgroup of 1-4 wavefronts relaxes one pixel column (or one state) at a
// time; columns are handed out by an atomic counter.  The column's whole state
// lives with the workgroup -- in LDS when it fits (gfx950: up to 160 KiB), else
// in a per-block slice of HBM: positions, the evaluation point, stage
// velocities, velocities, forces and the term results.
//
// One integrator stage evaluates the interaction list in two phases:
//   1. term-parallel: each thread evaluates the terms the host's schedule
//      gives it (64 terms of one kind per wave-round, so a wave runs one
//      code path at a time, the rounds spread over the waves by cost) and
//      writes, per atom the term acts on, the force that atom receives
//      (interactions.cpp:15-51, 252-362; `forces[i] -= f` is stored as -f,
//      which adds with the same rounding) into a result slot.  A thread's
//      terms are the same in every stage: where the state lives in LDS the
//      first four stay in registers for the whole launch;
//   2. component-parallel: a thread sums one component of one atom's force
//      from the atom's slots in the interaction list's order, from zero -- the
//      order in which the reference's Interaction::eval calls accumulate
//      forces_[i] (integrators.cpp:8-111) -- so each force is the reference's to
//      the last bit given the same term arithmetic.  The thread owns that
//      component of the atom's position and velocity too, so the integrator's
//      update follows without a barrier.
// FIRE's power P = sum_i v_i . f_i (minimiser.cpp:107-109) is summed in atom
// order by one thread while the others evaluate the next iteration's terms at
// the new positions, which do not depend on it; the velocities it decides are
// applied after that evaluation.  Built with -ffp-contract=off; IEEE divisions
// and square roots.  The angle, dihedral and Morse terms call the device acos /
// sin / atan / exp, which may differ from glibc's in the last place.
//
// What bounds it: FP64 issue and the chain of one column -- a dihedral is three
// roots, divisions and an atan deep.  The 72-atom graphene job at its full window
// (12.8 M FIRE iterations, two columns a CU: their result slots fill the LDS):
// 2285 vector instructions a wave and iteration, 45 % of the issue slots used
// over the launch, the longest column 1.3 times the mean.  657 -> 473 ms, of
// which terms in registers and component-parallel sums 657 -> 494, slots in rows
// and shared divisions 494 -> 473; a relaxation of 300 states 20 -> 8.8 ms.
// Bounded to 256 registers: at 268 one column a CU is resident, 712 ms.
#include <algorithm>

#include "flex.hpp"
#include "ref_terms.hpp"

namespace mafm {
namespace {

constexpr double TOL = 1e-10;   // TOLERANCE, globals.hpp:11

__device__ inline V3 ld3(const double* a, int i) { return {a[3 * i], a[3 * i + 1], a[3 * i + 2]}; }
__device__ inline void st3(double* a, int i, V3 v) {
    a[3 * i] = v.x;
    a[3 * i + 1] = v.y;
    a[3 * i + 2] = v.z;
}
__device__ inline V3 sub(V3 a, V3 b) { return {a.x - b.x, a.y - b.y, a.z - b.z}; }
__device__ inline V3 add(V3 a, V3 b) { return {a.x + b.x, a.y + b.y, a.z + b.z}; }
__device__ inline V3 neg(V3 a) { return {-a.x, -a.y, -a.z}; }
__device__ inline V3 scl(double s, V3 v) { return {s * v.x, s * v.y, s * v.z}; }   // T * Vector3
__device__ inline V3 scr(V3 v, double s) { return {v.x * s, v.y * s, v.z * s}; }   // Vector3 * T
__device__ inline double dot(V3 a, V3 b) { return a.x * b.x + a.y * b.y + a.z * b.z; }   // vectors.hpp:116-118
__device__ inline V3 cross(V3 a, V3 b) {                                                   // vectors.hpp:120-122
    return {a.y * b.z - a.z * b.y, a.z * b.x - a.x * b.z, a.x * b.y - a.y * b.x};
}

// A term as a thread holds it: the atoms it acts on, the result slot of each
// (n_slots: nobody reads it), where the tip's energy list keeps its energy, and
// its numbers q (pair terms: p0, p1, p2, shift; the others: p).  Packed: 16-bit
// pairs, for lists whose state fits the LDS.
template <bool PACKED>
struct Term {
    int kind;
    uint32_t at[PACKED ? 2 : 4], sl[PACKED ? 2 : 4], en[PACKED ? 1 : 2];
    double q[6];
    __device__ static int get(const uint32_t* w, int r) {
        return PACKED ? (int)((w[r >> 1] >> (16 * (r & 1))) & 0xffff) : (int)w[r];
    }
    __device__ int atom(int r) const { return get(at, r); }
    __device__ int slot(int r) const { return get(sl, r); }
    __device__ int place(int r) const { return get(en, r); }
    __device__ void load(const FxTerm& t) {
        kind = t.kind;
        for (int r = 0; r < (PACKED ? 2 : 4); ++r) {
            at[r] = PACKED ? (uint32_t)(t.atom[2 * r] | t.atom[2 * r + 1] << 16) : (uint32_t)t.atom[r];
            sl[r] = PACKED ? (uint32_t)(t.slot[2 * r] | t.slot[2 * r + 1] << 16) : (uint32_t)t.slot[r];
        }
        en[0] = PACKED ? (uint32_t)(t.place[0] | t.place[1] << 16) : (uint32_t)t.place[0];
        if (!PACKED) en[1] = t.place[1];
#pragma unroll
        for (int k = 0; k < 6; ++k) q[k] = t.q[k];
    }
};

// Where results go.  The slots lie in rows: row q holds the q-th slot of every
// atom that has so many, the atoms by falling number of slots, three components
// a slot, so the threads that sum one component each read neighbouring values
// (an atom's slots side by side cost 6-way bank conflicts: 3300 against 900
// cycles a sum phase).  A term's slot is its first component's place.
//   E_TIP  energies of the tip's terms in their order, at tip[place]
//   E_ALL  every atom's, at all[slot / 3]
//   E_ONLY energies in a slot's first component, no forces
enum { E_TIP = 0, E_ALL = 1, E_ONLY = 2 };
struct Results {
    double* r;
    double* tip;
    double* all;
    int mode;
};

template <bool P>
__device__ inline void put(const Results& R, const Term<P>& t, int role, V3 f) {
    double* r = R.r + t.slot(role);
    if (R.mode == E_ONLY) return;
    r[0] = f.x;
    r[1] = f.y;
    r[2] = f.z;
}

// One Interaction::eval of the list at positions X: the force on each atom
// and the energy into the term's places in R.
template <bool PACKED>
__device__ inline void eval_term(const Term<PACKED>& t, const double* X, const Results& R) {
    double e_out = 0;
    int roles = 2;
    switch (t.kind) {
        case MAFM_FX_LJ:
        case MAFM_FX_MORSE: {   // interactions.cpp:15-40
            const V3 p2 = ld3(X, t.atom(1));
            const V3 r = sub(ld3(X, t.atom(0)), add(p2, {t.q[3], t.q[4], t.q[5]}));
            V3 f;
            vdw(t.kind == MAFM_FX_LJ ? 0 : 1, t.q[0], t.q[1], t.q[2], r, f, e_out);
            put(R, t, 0, f);
            put(R, t, 1, neg(f));
            break;
        }
        case MAFM_FX_COULOMB: {   // interactions.cpp:42-51
            V3 f;
            coulomb(t.q[0], sub(ld3(X, t.atom(0)), ld3(X, t.atom(1))), f, e_out);
            put(R, t, 0, f);
            put(R, t, 1, neg(f));
            break;
        }
        case MAFM_FX_TIP_HARMONIC: {   // interactions.cpp:252-266
            const V3 r = sub(ld3(X, t.atom(0)), ld3(X, t.atom(1)));
            const double rl = sqrt(sq(r.x) + sq(r.y));
            const double dr = rl - t.q[1];
            const double e = t.q[0] * dr * dr;
            V3 f = {0, 0, 0};
            if (rl > TOL) {
                const double s = -2 * t.q[0] * dr / rl;
                f = {s * r.x, s * r.y, 0};
            }
            e_out = e;
            put(R, t, 0, f);
            put(R, t, 1, neg(f));
            break;
        }
        case MAFM_FX_BOND: {   // HarmonicInteraction::eval, interactions.cpp:296-306
            const V3 r = sub(ld3(X, t.atom(0)), ld3(X, t.atom(1)));
            const double rl = len3(r);
            const double dr = rl - t.q[1];
            const double e = t.q[0] * sq(dr);
            const V3 f = scl(-2 * t.q[0] * dr / rl, r);
            e_out = e;
            put(R, t, 0, f);
            put(R, t, 1, neg(f));
            break;
        }
        case MAFM_FX_ANGLE: {   // HarmonicAngleInteraction::eval, interactions.cpp:308-332
            const V3 ps = ld3(X, t.atom(0));
            const V3 r1v = sub(ld3(X, t.atom(1)), ps), r2v = sub(ld3(X, t.atom(2)), ps);
            const double r1 = len3(r1v), r2 = len3(r2v);
            double cos_t = dot(r1v, r2v) / (r1 * r2);
            if (cos_t > 1) cos_t = 1;
            else if (cos_t < -1) cos_t = -1;
            const double theta = acos(cos_t);
            const double sin_t = sin(theta);
            const double d_theta = theta - t.q[1];
            const double fm = -2 * t.q[0] * d_theta / sin_t;
            const Divisor by1(r1), by2(r2);
            const V3 f1 = scl(by1(-fm), sub(by2(r2v), by1(scr(r1v, cos_t))));
            const V3 f2 = scl(by2(-fm), sub(by1(r1v), by2(scr(r2v, cos_t))));
            e_out = t.q[0] * sq(d_theta);
            put(R, t, 0, neg(add(f1, f2)));   // forces[shared] -= f1 + f2
            put(R, t, 1, f1);
            put(R, t, 2, f2);
            roles = 3;
            break;
        }
        case MAFM_FX_DIHEDRAL: {   // HarmonicDihedralInteraction::eval, interactions.cpp:334-362
            const V3 p2 = ld3(X, t.atom(1)), p3 = ld3(X, t.atom(2));
            const V3 r12 = sub(ld3(X, t.atom(0)), p2), r23 = sub(p2, p3), r43 = sub(ld3(X, t.atom(3)), p3);
            const double r23l = len3(r23);
            const V3 mv = cross(r12, r23), nv = cross(r43, r23);
            const double m = len3(mv), n = len3(nv);
            const double tan_s = dot(nv, r12) * r23l / dot(mv, nv);
            const double sigma = atan(tan_s);
            const double d_sigma = sigma - t.q[1];
            const double fm = 2 * t.q[0] * d_sigma;
            e_out = t.q[0] * sq(d_sigma);
            const Divisor by_m(m * m * r23l), by_n(n * n * r23l);
            put(R, t, 0, scl(-fm * r23l / (m * m), mv));
            put(R, t, 1, scl(-fm, sub(scl(by_n(dot(r43, r23)), nv), scl(by_m((r23l * r23l) + dot(r12, r23)), mv))));
            put(R, t, 2, scl(-fm, add(scl(by_m(dot(r12, r23)), mv), scl(by_n((r23l * r23l) - dot(r43, r23)), nv))));
            put(R, t, 3, scl(fm * r23l / (n * n), nv));
            roles = 4;
            break;
        }
        case MAFM_FX_SUBSTRATE: {   // SubstrateInteraction::eval, interactions.cpp:280-294
            // p: multiplier, ulj, ushift, z0, rc, sigma
            const double dz = X[3 * t.atom(0) + 2] - t.q[3];
            const Divisor by_dz(dz);
            const double sig_z = by_dz(t.q[5]);
            const double sig_z2 = sig_z * sig_z;
            const double sig_z4 = sig_z2 * sig_z2;
            const double sig_z10 = sig_z4 * sig_z4 * sig_z2;
            double eterm = 0.0, fterm = 0.0;
            if (dz <= t.q[4]) {
                eterm += t.q[0] * (2. / 5 * sig_z10 - sig_z4) + t.q[1] * dz * dz - t.q[2];
                fterm += by_dz(4 * t.q[0]) * (sig_z10 - sig_z4) + 2 * t.q[1] * dz;
            }
            // forces[i].z += fterm: the +0 added to x and y leaves them as they are
            put(R, t, 0, {0, 0, fterm});
            e_out = eterm;
            roles = 1;
            break;
        }
        default: {   // MAFM_FX_XY_HARMONIC, interactions.cpp:268-278: p = k, x0, y0
            const double rx = X[3 * t.atom(0)] - t.q[1], ry = X[3 * t.atom(0) + 1] - t.q[2];
            const double rl = sqrt(sq(rx) + sq(ry));
            const double e = t.q[0] * rl * rl;
            V3 f = {0, 0, 0};
            if (rl > TOL) f = {-2 * t.q[0] * rx, -2 * t.q[0] * ry, 0};
            e_out = e;
            put(R, t, 0, f);
            roles = 1;
            break;
        }
    }
    if (R.mode == E_TIP) {
        R.tip[t.place(0)] = e_out;
        R.tip[t.place(1)] = e_out;
    } else {
        for (int k = 0; k < roles; ++k) {
            if (R.mode == E_ALL) R.all[t.slot(k) / 3] = e_out;
            else R.r[t.slot(k)] = e_out;
        }
    }
}

// checkConvergence (minimiser.cpp:15-37)
template <typename A>
__device__ inline bool converged(const A& a, V3 f, double ediff) {
    switch (a.minterm) {
        case MAFM_TERM_E: return fabs(ediff) < a.etol;
        case MAFM_TERM_F: return len3(f) < a.ftol;
        default: return fabs(ediff) < a.etol && len3(f) < a.ftol;
    }
}

__device__ inline void block_sync() { __syncthreads(); }

// acc + v[q0] + ... + v[q1 - 1], in order.  The additions are one chain; the
// next eight values are in flight while eight are added.
__device__ inline double seq_sum(double acc, const double* v, int q0, int q1) {
    double r[8], s[8];
    int q = q0;
    if (q + 8 <= q1) {
#pragma unroll
        for (int j = 0; j < 8; ++j) r[j] = v[q + j];
        for (; q + 16 <= q1; q += 8) {
#pragma unroll
            for (int j = 0; j < 8; ++j) s[j] = v[q + 8 + j];
#pragma unroll
            for (int j = 0; j < 8; ++j) acc += r[j];
#pragma unroll
            for (int j = 0; j < 8; ++j) r[j] = s[j];
        }
#pragma unroll
        for (int j = 0; j < 8; ++j) acc += r[j];
        q += 8;
    }
    // up to seven left: loaded together, added where they exist
    const int left = q1 - q;
    if (left > 0) {
#pragma unroll
        for (int j = 0; j < 7; ++j) s[j] = j < left ? v[q + j] : 0.0;
#pragma unroll
        for (int j = 0; j < 7; ++j)
            if (j < left) acc += s[j];
    }
    return acc;
}

// acc + v[row[0] / div + p] + ... over the first nq rows, in order, as seq_sum.
// The rows' places are read with scalar loads (the table has eight more).
template <int DIV>
__device__ inline double row_sum(double acc, const double* v, cptr<int32_t> row, int nq, int p) {
    double r[8], s[8];
    int q = 0;
    if (nq >= 8) {
#pragma unroll
        for (int j = 0; j < 8; ++j) r[j] = v[row[j] / DIV + p];
        for (; q + 16 <= nq; q += 8) {
#pragma unroll
            for (int j = 0; j < 8; ++j) s[j] = v[row[q + 8 + j] / DIV + p];
#pragma unroll
            for (int j = 0; j < 8; ++j) acc += r[j];
#pragma unroll
            for (int j = 0; j < 8; ++j) r[j] = s[j];
        }
#pragma unroll
        for (int j = 0; j < 8; ++j) acc += r[j];
        q += 8;
    }
    const int left = nq - q;
    if (left > 0) {
#pragma unroll
        for (int j = 0; j < 7; ++j) s[j] = j < left ? v[row[q + j] / DIV + p] : 0.0;
#pragma unroll
        for (int j = 0; j < 7; ++j)
            if (j < left) acc += s[j];
    }
    return acc;
}

// The force components a thread owns: places p = 3 rank + component, t, t +
// block threads, ...; e = 3 atom + component, the entry in the state's arrays.
#define FOR_ENTRIES(p, e) \
    for (int p = t, e = entry_of(p); p < 3 * n; p += nthr, e = entry_of(p))

// Terms of a thread that stay in registers (lists whose state fits the LDS)
constexpr int HELD_TERMS = 4;

// The thread's terms of every round at positions X into R.
template <bool PACKED>
struct Evaluator {
    Term<PACKED> held[PACKED ? HELD_TERMS : 1];
    const FxTerm* terms;
    int rounds, t, nthr;
    __device__ void init(const FxTerm* terms_, int rounds_, int t_, int nthr_) {
        terms = terms_; rounds = rounds_; t = t_; nthr = nthr_;
        if (PACKED) {
#pragma unroll
            for (int r = 0; r < HELD_TERMS; ++r) {
                held[r].kind = -1;
                if (r < rounds) held[r].load(terms[r * nthr + t]);
            }
        }
    }
    __device__ void operator()(const double* X, const Results& R) const {
        Term<PACKED> cur;
        for (int r = 0; r < rounds; ++r) {
            // one instance of the term code; the copy picks the round's registers
            if (PACKED && r == 0) cur = held[0];
            else if (PACKED && r == 1) cur = held[1];
            else if (PACKED && r == 2) cur = held[2];
            else if (PACKED && r == 3) cur = held[3];
            else cur.load(terms[r * nthr + t]);
            if (cur.kind >= 0) eval_term(cur, X, R);
        }
    }
};

// Per-column state: positions, evaluation point, velocities, stage velocities
// (then the mixed velocities), forces, powers, energies of the tip, broadcast
// values, RK4's sums, results.
struct State {
    double *pos, *pev, *vel, *vst, *frc, *pdot, *tip, *bc, *facc, *vacc, *eacc, *ener, *all, *res;
    const int32_t *cnt, *order, *fixed;   // slots of each rank, its atom; fixed flags by atom
    // the tables behind the state, copied from the rows' end on
    __device__ void tables(const int32_t* idx, int n) {
        cnt = idx;
        order = idx + n;
        fixed = idx + 2 * n;
    }
};
__host__ __device__ inline size_t flex_doubles(int n, int n_slots, int n_tip, bool rk4) {
    return (size_t)(16 + (rk4 ? 6 : 0)) * n + (n_tip + 1) + 4 + 3 * ((size_t)n_slots + 1);
}
__device__ inline State flex_layout(double* p, int n, int n_tip, bool rk4) {
    State S;
    S.pos = p; p += 3 * n;
    S.pev = p; p += 3 * n;
    S.vel = p; p += 3 * n;
    S.vst = p; p += 3 * n;
    S.frc = p; p += 3 * n;
    S.pdot = p; p += n;
    S.tip = p; p += n_tip + 1;
    S.bc = p; p += 4;
    S.facc = p; p += rk4 ? 3 * n : 0;
    S.vacc = p; p += rk4 ? 3 * n : 0;
    S.eacc = S.ener = S.all = nullptr;
    S.res = p;
    return S;
}

// FIRE's velocity mixing (minimiser.cpp:112-118) of one component, and the
// atom's power.  normalized(): vectors.hpp:107-114.
__device__ inline double fire_mix(const State& S, int e, double alpha) {
    const int i = e / 3, c = e - 3 * i;
    const V3 v = ld3(S.vel, i), f = ld3(S.frc, i);
    const double fl = len3(f), fc = S.frc[e];
    const double fh = fl > 1e-10 ? fc / fl : 0;
    if (c == 0) S.pdot[i] = dot(v, f);
    return (1 - alpha) * S.vel[e] + alpha * fh * len3(v);
}

template <bool IN_LDS>
__global__ void __launch_bounds__(256, 2) k_scan_flex(FlexArgs a) {
    extern __shared__ double lds_flex[];
    __shared__ int col_shared;
    const int t = threadIdx.x;        // thread of the block (1-4 waves share a column)
    const int nthr = blockDim.x;
    const int n = a.n_atoms;
    const bool sd = a.minimiser == MAFM_MIN_SD, rk4 = !sd && a.integrator == MAFM_INT_RK4;
    const bool mid = !sd && a.integrator == MAFM_INT_MIDPOINT;
    const size_t nd = flex_doubles(n, a.n_slots, a.n_tip, rk4);
    double* base = IN_LDS ? lds_flex : a.work + (size_t)blockIdx.x * nd;
    State S = flex_layout(base, n, a.n_tip, rk4);
    const int32_t* idx = a.idx;
    if (IN_LDS) {
        int32_t* l = reinterpret_cast<int32_t*>(lds_flex + nd);
        for (int q = t; q < 3 * n; q += nthr) l[q] = a.idx[q];
        idx = l;
    }
    S.tables(idx, n);
    const cptr<int32_t> rows = as_const(a.idx) + 3 * n;
    const Results R = {S.res, S.tip, nullptr, E_TIP};
    Evaluator<IN_LDS> eval;
    eval.init(a.terms, a.rounds, t, nthr);
    block_sync();
    auto entry_of = [&](int p) { return p < 3 * n ? 3 * S.order[p / 3] + p % 3 : 0; };
    auto force = [&](int p) { return row_sum<1>(0.0, S.res, rows, S.cnt[p / 3], p); };
    const int tip_place = 3 * a.tip_rank;
    const int n_cols = a.nx * a.ny;
    for (;;) {
        if (t == 0) col_shared = atomicAdd(a.next_col, 1);
        block_sync();
        const int col = col_shared;
        block_sync();
        if (col >= n_cols) break;
        const int ci = col / a.ny, cj = col - ci * a.ny;
        const double x = ci * a.dx, y = cj * a.dy;   // simulation.cpp:80-83
        // System copy (simulation.cpp:93): initial positions, zero velocities
        for (int q = t; q < 3 * n; q += nthr) {
            S.pos[q] = a.pos0[q];
            S.vel[q] = 0;
        }
        block_sync();
        if (t == 0) {
            // setDummyXY / setDummyZ (system.cpp:139-162, system.hpp:47-50)
            double px = x, py = y;
            if (a.tip_pbc) wrap_xy(a.cell, a.cell_inv, a.offset, x, y, px, py);
            st3(S.pos, 0, {px, py, a.zhigh});
            st3(S.pos, 1, {px, py, a.zhigh - a.tip_dummy_d});
        }
        block_sync();
        double e_tip = 0;             // energies_[1] of the System copy: 0 until its first step
        // FIREMinimisation / SDMinimisation (minimiser.cpp:39-129), a stage per
        // trip; out: the tip-surface evaluation of the height's record
        int k = 0, s = 0, nnn = 0, n_tot = 1;
        double alpha = 0.1, dt = a.dt, e_acc = 0;
        bool pending = false;         // mixed velocities wait in vst for P
        bool out = n_tot >= a.maxsteps;
        for (;;) {
            if (pending && t == nthr - 1) S.bc[1] = seq_sum(0.0, S.pdot, 0, n);
            eval(s == 0 || out ? S.pos : S.pev, R);
            block_sync();
            if (pending) {            // minimiser.cpp:107-126
                const bool up = !(S.bc[1] < 0);
                FOR_ENTRIES(p, e)
                    if (S.fixed[e / 3] != 1) S.vel[e] = up ? S.vst[e] : 0.0;
                if (!up) {
                    nnn = 0;
                    dt *= 0.5;
                    alpha = 0.1;
                } else {
                    if (nnn > 5) {
                        dt = fmin(dt * 1.1, 10 * a.dt);
                        alpha *= 0.99;
                    }
                    ++nnn;
                }
                pending = false;
            }
            if (out) {
                // makeXYZFile of the state column (simulation.cpp:114-116), then
                // getOutput (system.cpp:28-51): the tip-surface terms only
                if (col == a.state_col && a.state)
                    for (int q = t; q < 3 * n; q += nthr) a.state[(size_t)k * 3 * n + q] = S.pos[q];
                if (t < 3) S.frc[3 + t] = row_sum<1>(0.0, S.res, rows, a.tip_ts_slots, tip_place + t);
                if (t == nthr - 1) S.bc[0] = seq_sum(0.0, S.tip, 0, a.tip_ts_terms);
                block_sync();
                if (t == 0) {
                    const V3 d = ld3(S.pos, 0), r = ld3(S.pos, 1), f = ld3(S.frc, 1);
                    DevRecord rec;
                    rec.x = x; rec.y = y; rec.z = d.z;
                    rec.fx = f.x; rec.fy = f.y; rec.fz = f.z;
                    rec.rx = r.x - d.x; rec.ry = r.y - d.y; rec.rz = r.z - d.z;
                    rec.e = S.bc[0];
                    rec.n_steps = n_tot;
                    rec.flags = n_tot >= a.maxsteps ? REC_UNCONVERGED : 0;
                    a.rec[(size_t)col * a.nz + k] = rec;
                    // lowerTip (system.hpp:51-54)
                    S.pos[2] -= a.dz;
                    S.pos[5] -= a.dz;
                }
                block_sync();
                if (++k >= a.nz) break;
                s = 0; nnn = 0; n_tot = 1;
                alpha = 0.1; dt = a.dt;
                out = n_tot >= a.maxsteps;
                continue;
            }
            // the tip's energy is read by the energy convergence test only
            if (t == nthr - 1 && a.minterm != MAFM_TERM_F && !(mid && s == 0)) S.bc[0] = seq_sum(0.0, S.tip, 0, a.n_tip);
            if (mid && s == 0) {            // midpointStep's half step
                FOR_ENTRIES(p, e) {
                    const double f = force(p), v = S.vel[e], x0 = S.pos[e];
                    const bool free_ = S.fixed[e / 3] != 1;
                    S.pev[e] = free_ ? x0 + dt / 2 * v : x0;
                    S.vst[e] = v + dt / 2 * f;
                }
                block_sync();
                s = 1;
                continue;
            }
            if (rk4) {                                // stages at pos, pos + dt/2 v1, pos + dt/2 v2, pos + dt v3
                FOR_ENTRIES(p, e) {
                    const double fs = force(p), vs = s == 0 ? S.vel[e] : S.vst[e];
                    const bool free_ = S.fixed[e / 3] != 1;
                    double fa, va;
                    if (s == 0) { fa = fs; va = vs; }
                    else if (s < 3) { fa = S.facc[e] + 2 * fs; va = S.vacc[e] + 2 * vs; }
                    else { fa = S.facc[e] + fs; va = S.vacc[e] + vs; }
                    if (s < 3) {
                        const double h = s < 2 ? dt / 2 : dt;
                        S.facc[e] = fa;
                        S.vacc[e] = va;
                        S.pev[e] = free_ ? S.pos[e] + h * vs : S.pos[e];
                        S.vst[e] = free_ ? S.vel[e] + h * fs : S.vel[e];
                    } else {
                        if (free_) {
                            S.pos[e] = S.pos[e] + dt / 6 * va;
                            S.vel[e] = S.vel[e] + dt / 6 * fa;
                        }
                        S.frc[e] = fa / 6;
                    }
                }
                block_sync();
                const double es = S.bc[0];
                e_acc = s == 0 ? es : e_acc + (s == 3 ? es : 2 * es);
                if (s < 3) {
                    block_sync();     // bc[0] is read before the next stage's is written
                    ++s;
                    continue;
                }
            } else {
                FOR_ENTRIES(p, e) {
                    const double f = force(p);
                    S.frc[e] = f;
                    if (S.fixed[e / 3] != 1 && !sd) {  // midpointStep, eulerStep; masses are 1
                        S.pos[e] = S.pos[e] + dt * (mid ? S.vst[e] : S.vel[e]);
                        S.vel[e] = S.vel[e] + dt * f;
                    }
                }
                block_sync();
            }
            const double prev_e = e_tip;
            e_tip = rk4 ? e_acc / 6 : S.bc[0];
            s = 0;
            if (converged(a, ld3(S.frc, 1), e_tip - prev_e)) {
                out = true;
                block_sync();         // the tip's force and energy are read before they are written again
                continue;
            }
            if (sd) {                                 // evaluate, test, move
                FOR_ENTRIES(p, e)
                    if (S.fixed[e / 3] != 1) S.pos[e] = S.pos[e] + a.dt * S.frc[e];
            } else {
                FOR_ENTRIES(p, e) S.vst[e] = fire_mix(S, e, alpha);
                pending = true;
            }
            out = ++n_tot >= a.maxsteps;
            block_sync();
        }
    }
}

// ---------------------------------------------------------------- System operators
// State of one system copy: as the scan's, with every atom's energy, and a
// fourth result component where the operator needs all energies of each
// evaluation (eval, one step, RK4).
__host__ __device__ inline bool sys_all_energies(const SysArgs& a) {
    return a.op != SYS_MINIMISE || (a.minimiser != MAFM_MIN_SD && a.integrator == MAFM_INT_RK4);
}
__host__ __device__ inline size_t sys_doubles(const SysArgs& a) {
    return (size_t)24 * a.n_atoms + (a.n_tip + 1) + 4 + (sys_all_energies(a) ? 4 : 3) * ((size_t)a.n_slots + 1);
}
__device__ inline State sys_layout(double* p, int n, int n_tip, int n_slots) {
    State S;
    S.pos = p; p += 3 * n;
    S.pev = p; p += 3 * n;
    S.vel = p; p += 3 * n;
    S.vst = p; p += 3 * n;
    S.frc = p; p += 3 * n;
    S.pdot = p; p += n;
    S.facc = p; p += 3 * n;
    S.vacc = p; p += 3 * n;
    S.eacc = p; p += n;
    S.ener = p; p += n;
    S.tip = p; p += n_tip + 1;
    S.bc = p; p += 4;
    S.res = p; p += 3 * (n_slots + 1);
    S.all = p;
    return S;
}

template <bool IN_LDS>
__global__ void __launch_bounds__(256, 2) k_system_op(SysArgs a) {
    extern __shared__ double lds_sys[];
    const int t = threadIdx.x, nthr = blockDim.x;
    const int n = a.n_atoms;
    const size_t nd = sys_doubles(a);
    double* base = IN_LDS ? lds_sys : a.work + (size_t)blockIdx.x * nd;
    State S = sys_layout(base, n, a.n_tip, a.n_slots);
    const int32_t* idx = a.idx;
    if (IN_LDS) {
        int32_t* l = reinterpret_cast<int32_t*>(lds_sys + nd);
        for (int q = t; q < 3 * n; q += nthr) l[q] = a.idx[q];
        idx = l;
    }
    S.tables(idx, n);
    const cptr<int32_t> rows = as_const(a.idx) + 3 * n;
    const bool minimise = a.op == SYS_MINIMISE, sd = minimise && a.minimiser == MAFM_MIN_SD;
    const bool rk4 = !sd && a.op != SYS_EVAL && a.integrator == MAFM_INT_RK4;
    const bool mid = !sd && a.op != SYS_EVAL && a.integrator == MAFM_INT_MIDPOINT;
    const bool all_e = sys_all_energies(a);
    Results R = {S.res, S.tip, S.all, all_e ? E_ALL : E_TIP};
    Evaluator<IN_LDS> eval;
    eval.init(a.terms, a.rounds, t, nthr);
    auto entry_of = [&](int p) { return p < 3 * n ? 3 * S.order[p / 3] + p % 3 : 0; };
    auto force = [&](int p, double f0) { return row_sum<1>(f0, S.res, rows, S.cnt[p / 3], p); };
    // every atom's energy from what `from` gives for it, into S.ener / S.eacc by `put`
    auto energies = [&](auto from, auto to) {
        for (int k = t; k < n; k += nthr) {
            const int i = S.order[k];
            to(i, row_sum<3>(from(i), S.all, rows, S.cnt[k], k));
        }
    };
    block_sync();
    for (int64_t st = blockIdx.x; st < a.n_states; st += gridDim.x) {
        const size_t o3 = (size_t)st * 3 * n, o1 = (size_t)st * n;
        for (int q = t; q < 3 * n; q += nthr) {
            S.pos[q] = S.pev[q] = a.pos[o3 + q];
            S.frc[q] = a.frc[o3 + q];
            S.vel[q] = a.op == SYS_EVAL ? 0.0 : a.vel[o3 + q];
        }
        for (int i = t; i < n; i += nthr) S.ener[i] = a.ener[o1 + i];
        block_sync();
        int s = 0, nnn = 0, n_tot = 1;
        double alpha = 0.1, dt = a.dt, e_tip = S.ener[1];
        bool pending = false;
        // the force a step's sums start from: eulerStep and Interaction::eval add
        // onto what is there, which the minimisers clear first
        const bool onto = a.op == SYS_EVAL || (a.op == SYS_STEP && !mid && !rk4);
        bool last = false;            // only the energies of the last evaluation are missing
        bool run = !minimise || n_tot < a.maxsteps;
        // minimiser.cpp:107-126, once P is there; P < 0 stops the fixed atoms too
        auto apply = [&]() {
            const bool up = !(S.bc[1] < 0);
            FOR_ENTRIES(p, e) {
                if (!up) S.vel[e] = 0;
                else if (S.fixed[e / 3] != 1) S.vel[e] = S.vst[e];
            }
            if (!up) {
                nnn = 0;
                dt *= 0.5;
                alpha = 0.1;
            } else {
                if (nnn > 5) {
                    dt = fmin(dt * 1.1, 10 * a.dt);
                    alpha *= 0.99;
                }
                ++nnn;
            }
            pending = false;
        };
        while (run) {
            if (pending && t == nthr - 1) S.bc[1] = seq_sum(0.0, S.pdot, 0, n);
            R.mode = last ? E_ONLY : (all_e ? E_ALL : E_TIP);
            eval(s == 0 && !last ? S.pos : S.pev, R);
            block_sync();
            if (pending) apply();
            if (last) {
                for (int k = t; k < n; k += nthr) S.ener[S.order[k]] = row_sum<1>(0.0, S.res, rows, S.cnt[k], 3 * k);
                break;
            }
            if (a.op == SYS_EVAL) {
                FOR_ENTRIES(p, e) S.frc[e] = force(p, S.frc[e]);
                energies([&](int i) { return S.ener[i]; }, [&](int i, double e) { S.ener[i] = e; });
                break;
            }
            if (mid && s == 0) {                      // midpointStep's half step
                FOR_ENTRIES(p, e) {
                    const double f = force(p, 0.0), v = S.vel[e], x0 = S.pos[e];
                    const bool free_ = S.fixed[e / 3] != 1;
                    S.pev[e] = free_ ? x0 + dt / 2 * v : x0;
                    S.vst[e] = free_ ? v + dt / 2 * f : v;
                }
                block_sync();
                s = 1;
                continue;
            }
            if (rk4) {                                // rk4Step
                FOR_ENTRIES(p, e) {
                    const double fs = force(p, 0.0), vs = s == 0 ? S.vel[e] : S.vst[e];
                    const bool free_ = S.fixed[e / 3] != 1;
                    double fa, va;
                    if (s == 0) { fa = fs; va = vs; }
                    else if (s < 3) { fa = S.facc[e] + 2 * fs; va = S.vacc[e] + 2 * vs; }
                    else { fa = S.facc[e] + fs; va = S.vacc[e] + vs; }
                    if (s < 3) {
                        const double h = s < 2 ? dt / 2 : dt;
                        S.facc[e] = fa;
                        S.vacc[e] = va;
                        S.pev[e] = free_ ? S.pos[e] + h * vs : S.pos[e];
                        S.vst[e] = free_ ? S.vel[e] + h * fs : S.vel[e];
                    } else {
                        if (free_) {
                            S.pos[e] = S.pos[e] + dt / 6 * va;
                            S.vel[e] = S.vel[e] + dt / 6 * fa;
                        }
                        S.frc[e] = fa / 6;
                    }
                }
                energies([](int) { return 0.0; }, [&](int i, double es) {
                    if (s == 0) S.eacc[i] = es;
                    else if (s < 3) S.eacc[i] = S.eacc[i] + 2 * es;
                    else S.ener[i] = (S.eacc[i] + es) / 6;
                });
                block_sync();
                if (s < 3) {
                    ++s;
                    continue;
                }
            } else {
                FOR_ENTRIES(p, e) {
                    const double f = force(p, onto ? S.frc[e] : 0.0);
                    S.frc[e] = f;
                    if (S.fixed[e / 3] != 1 && !sd) {
                        const double x0 = S.pos[e];
                        if (!mid) S.pev[e] = x0;      // where this step evaluated
                        S.pos[e] = x0 + dt * (mid ? S.vst[e] : S.vel[e]);
                        S.vel[e] = S.vel[e] + dt * f;
                    }
                }
                if (all_e) {
                    energies([&](int i) { return onto ? S.ener[i] : 0.0; }, [&](int i, double e) { S.ener[i] = e; });
                } else if (t == nthr - 1 && a.minterm != MAFM_TERM_F) {
                    S.bc[0] = seq_sum(0.0, S.tip, 0, a.n_tip);
                }
                block_sync();
            }
            s = 0;
            if (!minimise) break;
            const double prev = e_tip;
            e_tip = all_e ? S.ener[1] : S.bc[0];
            const bool done = converged(a, ld3(S.frc, 1), e_tip - prev);
            if (!done) {
                if (sd) {
                    FOR_ENTRIES(p, e)
                        if (S.fixed[e / 3] != 1) {
                            S.pev[e] = S.pos[e];
                            S.pos[e] = S.pos[e] + a.dt * S.frc[e];
                        }
                } else {
                    FOR_ENTRIES(p, e) S.vst[e] = fire_mix(S, e, alpha);
                    pending = true;
                }
                ++n_tot;
            } else if (sd) {
                FOR_ENTRIES(p, e) S.pev[e] = S.pos[e];
            }
            block_sync();
            if (done || n_tot >= a.maxsteps) {
                if (!all_e) {         // one more trip for every atom's energy
                    last = true;
                    continue;
                }
                if (pending) {
                    if (t == nthr - 1) S.bc[1] = seq_sum(0.0, S.pdot, 0, n);
                    block_sync();
                    apply();
                }
                break;
            }
        }
        block_sync();
        for (int q = t; q < 3 * n; q += nthr) {
            a.pos[o3 + q] = S.pos[q];
            a.frc[o3 + q] = S.frc[q];
            if (a.op != SYS_EVAL) a.vel[o3 + q] = S.vel[q];
        }
        for (int i = t; i < n; i += nthr) a.ener[o1 + i] = S.ener[i];
        if (t == 0 && minimise) a.steps[st] = n_tot;
        block_sync();
    }
}

}  // namespace

size_t flex_block_doubles(const FlexArgs& a) {
    return flex_doubles(a.n_atoms, a.n_slots, a.n_tip, a.minimiser == MAFM_MIN_FIRE && a.integrator == MAFM_INT_RK4);
}

size_t flex_block_lds(const FlexArgs& a) {
    return flex_block_doubles(a) * sizeof(double) + 3 * (size_t)a.n_atoms * sizeof(int32_t);
}

size_t sys_block_doubles(const SysArgs& a) { return sys_doubles(a); }

size_t sys_block_bytes(const SysArgs& a) {
    return sys_doubles(a) * sizeof(double) + 3 * (size_t)a.n_atoms * sizeof(int32_t);
}

hipError_t launch_system_op(const SysArgs& a, int waves, bool in_lds, hipStream_t st) {
    const unsigned blocks = (unsigned)std::min<int64_t>(a.n_states, 1 << 20);
    if (in_lds) {
        const size_t lds = sys_block_bytes(a);
        hipError_t e = hipFuncSetAttribute((const void*)k_system_op<true>,
                                           hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
        if (e != hipSuccess) return e;
        hipLaunchKernelGGL(k_system_op<true>, dim3(blocks), dim3(64 * waves), lds, st, a);
    } else {
        hipLaunchKernelGGL(k_system_op<false>, dim3(blocks), dim3(64 * waves), 0, st, a);
    }
    return hipGetLastError();
}

hipError_t launch_scan_flex(const FlexArgs& a, int n_blocks, int waves, bool in_lds, hipStream_t st) {
    if (in_lds) {
        const size_t lds = flex_block_lds(a);
        // above 64 KiB a workgroup asks for the larger allocation (gfx950: 160 KiB)
        hipError_t e = hipFuncSetAttribute((const void*)k_scan_flex<true>,
                                           hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
        if (e != hipSuccess) return e;
        hipLaunchKernelGGL(k_scan_flex<true>, dim3(n_blocks), dim3(64 * waves), lds, st, a);
    } else {
        hipLaunchKernelGGL(k_scan_flex<false>, dim3(n_blocks), dim3(64 * waves), 0, st, a);
    }
    return hipGetLastError();
}

}  // namespace mafm
