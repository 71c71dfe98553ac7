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
// What bounds it: one column's chain, FP64 operations that wait 8 cycles for the
// one before, shared by two columns a CU (their result slots fill the LDS) whose
// chains fill three quarters of the issue slots.  The 72-atom graphene job at its
// full window (12.8 M FIRE iterations): an iteration 31000 -> 24800 cycles, of
// which two evaluations take 16600 (an angle and a dihedral a lane each), force
// sums and updates 5800, the mixing 1800; 657 -> 388 ms.  A relaxation of 300
// states 19.7 -> 7.0 ms.  Measured on the way: an atom's slots side by side 494
// ms, in rows of single values 473, pairs and the powers and the tip's sums as
// padded lists 388; bounded to more than 256 registers (one column a CU) 712;
// eight waves a column (one column a CU) 500.
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
// (n_res: nobody reads it), where its energy goes if it acts on the tip, and
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

// Where results go: first the tip's slots, force and energy, which four lanes sum
// side by side (the tip has a term with every surface atom, twice the slots of
// the next); then the others' in rows: row q holds the slots 2 q and 2 q + 1 of
// every atom that has so many, the atoms by falling number of slots, three
// components a slot, so the threads that sum one component each read
// neighbouring pairs (an atom's slots side by side cost 6-way bank conflicts;
// values one by one, with their addresses, 46 instructions for eight against
// 20).  A slot's components are two apart, its pair's other slot between; an
// unpaired slot is paired with -0, which leaves every sum as it is.  A term's
// slot is its first component's place; r[n_res] on takes what nobody reads.
//   E_TIP  the tip's energies alone
//   E_ALL  every atom's, the others' at all_place(slot)
//   E_ONLY energies in a slot's first component, no forces
enum { E_TIP = 0, E_ALL = 1, E_ONLY = 2 };
struct Results {
    double* r;
    double* all;
    int others, n_res, mode;
    __device__ int all_place(int slot) const {
        const int q = (slot < others ? n_res : slot) - others;
        return q / 6 * 2 + (q & 1);
    }
};

template <bool P>
__device__ inline void put(const Results& R, const Term<P>& t, int role, V3 f) {
    double* r = R.r + t.slot(role);
    if (R.mode == E_ONLY) return;
    r[0] = f.x;
    r[2] = f.y;
    r[4] = f.z;
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
    if (R.mode == E_ONLY) {
        for (int k = 0; k < roles; ++k) R.r[t.slot(k)] = e_out;
        return;
    }
    R.r[t.place(0)] = e_out;
    R.r[t.place(1)] = e_out;
    if (R.mode == E_ALL)
        for (int k = 0; k < roles; ++k) R.all[R.all_place(t.slot(k))] = e_out;
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

// A list that one thread sums is padded to whole batches with -0, and the batch
// past its end may be read.
constexpr int BATCH = FLEX_BATCH;

// acc + the n values of a padded list, in order; its pairs are S apart.  One
// chain of additions, the next batch in flight while one is added.  (By one lane
// a masked or moved value costs as much as an addition: 95 cycles a value where
// the batches were guarded.)
template <int S>
__device__ inline double list_sum(double acc, const double* v, int n) {
    double2 r[BATCH / 2], s[BATCH / 2];
    auto load = [&](double2* x, int q) {
#pragma unroll
        for (int j = 0; j < BATCH / 2; ++j) x[j] = *reinterpret_cast<const double2*>(v + S * (q / 2 + j));
    };
    auto add = [&](const double2* x) {
#pragma unroll
        for (int j = 0; j < BATCH / 2; ++j) {
            acc += x[j].x;
            acc += x[j].y;
        }
    };
    load(r, 0);
    for (int q = 0; q < n; q += 2 * BATCH) {
        load(s, q + BATCH);
        add(r);
        if (q + BATCH >= n) break;
        load(r, q + 2 * BATCH);
        add(s);
    }
    return acc;
}

// acc + an atom's slots, in order: nq of them, pairs at v + row[0] / DIV + p,
// v + row[1] / DIV + p, ...  Four pairs and the places of the four after them are
// in flight while four are added; the table has twelve more rows, and past the
// last one v is read but not added.
template <int DIV>
__device__ inline double row_sum(double acc, const double* v, const int32_t* row, int nq, int p) {
    double2 r[4], s[4];
    int4 w = *reinterpret_cast<const int4*>(row);
    v += p;
    auto load = [&](double2* x) {
        x[0] = *reinterpret_cast<const double2*>(v + w.x / DIV);
        x[1] = *reinterpret_cast<const double2*>(v + w.y / DIV);
        x[2] = *reinterpret_cast<const double2*>(v + w.z / DIV);
        x[3] = *reinterpret_cast<const double2*>(v + w.w / DIV);
    };
    auto places = [&](int q) { w = *reinterpret_cast<const int4*>(row + q); };
    auto add = [&](const double2* x) {
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            acc += x[j].x;
            acc += x[j].y;
        }
    };
    const int n2 = (nq + 1) / 2;
    load(r);
    places(4);
    int q = 0;
    for (; q + 4 <= n2; q += 4) {
        load(s);
        places(q + 8);
        add(r);
#pragma unroll
        for (int j = 0; j < 4; ++j) r[j] = s[j];
    }
#pragma unroll
    for (int j = 0; j < 3; ++j) {
        acc += q + j < n2 ? r[j].x : -0.0;
        acc += q + j < n2 ? r[j].y : -0.0;
    }
    return acc;
}

// The force components a thread owns: of the other atoms the places p = 3 rank +
// component, t, t + block threads, ...; the tip's go to the fourth to second
// last thread, before its others (p past them all); the last thread has the tip's
// energy.  e = 3 atom + component, the entry in the state's arrays.  What a
// thread needs to know of its first place of the others stays in registers.
struct Own {
    int e, slots;
    bool moves;
};
struct Places {
    int t, nthr, n3, tip;    // tip: component of the tip, 3 its energy, < 0 neither
    __device__ Places(int t_, int nthr_, int n) : t(t_), nthr(nthr_), n3(3 * (n - 1)), tip(t_ - (nthr_ - 4)) {}
    __device__ int first() const { return (unsigned)tip < 3u ? n3 + tip : (t < n3 ? t : -1); }
    __device__ int next(int p) const { return p >= n3 ? (t < n3 ? t : -1) : (p + nthr < n3 ? p + nthr : -1); }
};
#define FOR_ENTRIES(p, o)                                            \
    for (int p = my.first(); p >= 0; p = my.next(p))                 \
        if (const Own o = p >= my.n3 ? tip_own : p == t ? first : S.own(p); true)

// Terms of a thread that stay in registers (lists whose state fits the LDS)
constexpr int HELD_TERMS = FLEX_HELD_ROUNDS;

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
// (then the mixed velocities), forces, powers, broadcast values, RK4's sums,
// results.
struct State {
    double *pos, *pev, *vel, *vst, *frc, *pdot, *bc, *facc, *vacc, *eacc, *ener, *all, *res;
    const int32_t *rows, *cnt, *order, *fixed;   // places of the rows; slots of each rank, its atom; fixed flags by atom
    __device__ void tables(const int32_t* idx, int n_rows, int n) {
        rows = idx;
        cnt = rows + n_rows;
        order = cnt + n;
        fixed = order + n;
    }
    // the -0 that pad the lists and pair the unpaired slots (with_all: of the energies too)
    __device__ void pad(int n, int n_tip, int others, bool with_all, int t, int nthr) {
        for (int q = n + t; q < flex_padded(n); q += nthr) pdot[q] = -0.0;
        for (int q = n_tip + t; q < flex_padded(n_tip); q += nthr)
            for (int c = 0; c < 4; ++c) res[8 * (q / 2) + 2 * c + (q & 1)] = -0.0;
        for (int k = t; k < n - 1; k += nthr) {
            const int last = cnt[k] / 2;
            if (cnt[k] % 2 == 0) continue;
            for (int c = 0; c < 3; ++c) res[others + rows[last] + 6 * k + 2 * c + 1] = -0.0;
            if (with_all) all[rows[last] / 3 + 2 * k + 1] = -0.0;
        }
    }
    __device__ Own own(int p) const {
        const int k = p / 3, i = order[k];
        return {3 * i + (p - 3 * k), cnt[k], fixed[i] != 1};
    }
};
__device__ inline State flex_layout(double* p, int n, int n_res, bool rk4) {
    State S;
    S.pdot = p; p += flex_padded(n);
    S.bc = p; p += 4;
    S.res = p; p += n_res + 8;
    S.pos = p; p += 3 * n;
    S.pev = p; p += 3 * n;
    S.vel = p; p += 3 * n;
    S.vst = p; p += 3 * n;
    S.frc = p; p += 3 * n;
    S.facc = p; p += rk4 ? 3 * n : 0;
    S.vacc = p;
    S.eacc = S.ener = S.all = nullptr;
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
    extern __shared__ __align__(16) double lds_flex[];
    __shared__ int col_shared;
    const int t = threadIdx.x;        // thread of the block (1-4 waves share a column)
    const int nthr = blockDim.x;
    const int n = a.n_atoms;
    const bool sd = a.minimiser == MAFM_MIN_SD, rk4 = !sd && a.integrator == MAFM_INT_RK4;
    const bool mid = !sd && a.integrator == MAFM_INT_MIDPOINT;
    const size_t nd = flex_block_doubles(a);
    double* base = IN_LDS ? lds_flex : a.work + (size_t)blockIdx.x * nd;
    State S = flex_layout(base, n, a.n_res, rk4);
    const int32_t* idx = a.idx;
    if (IN_LDS) {
        int32_t* l = reinterpret_cast<int32_t*>(lds_flex + nd);
        for (int q = t; q < a.n_rows + 3 * n; q += nthr) l[q] = a.idx[q];
        idx = l;
    }
    S.tables(idx, a.n_rows, n);
    const int others = 4 * flex_padded(a.n_tip);
    const Results R = {S.res, nullptr, others, a.n_res, E_TIP};
    Evaluator<IN_LDS> eval;
    eval.init(a.terms, a.rounds, t, nthr);
    block_sync();
    S.pad(n, a.n_tip, others, false, t, nthr);
    const Places my(t, nthr, n);
    const Own first = t < my.n3 ? S.own(t) : Own{0, 0, false};
    const Own tip_own = {3 + my.tip, 0, true};
    double tip_sum = 0;               // of the thread's component of the tip
    auto sum_tip = [&]() {
        if (my.tip >= 0) tip_sum = list_sum<8>(0.0, S.res + 2 * my.tip, a.n_tip);
        if (my.tip == 3) S.bc[0] = tip_sum;   // read by the energy convergence test
    };
    auto force = [&](const Own& o, int p) {
        return p >= my.n3 ? tip_sum : row_sum<1>(0.0, S.res + others, S.rows, o.slots, 2 * p);
    };
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
            if (pending && t == nthr - 1) S.bc[1] = list_sum<2>(0.0, S.pdot, n);
            eval(s == 0 || out ? S.pos : S.pev, R);
            block_sync();
            if (pending) {            // minimiser.cpp:107-126
                const bool up = !(S.bc[1] < 0);
                FOR_ENTRIES(p, o)
                    if (o.moves) S.vel[o.e] = up ? S.vst[o.e] : 0.0;
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
                if (my.tip >= 0) {
                    double v = 0;
#pragma unroll 8
                    for (int q = 0; q < a.tip_ts_slots; ++q) v += S.res[8 * (q / 2) + 2 * my.tip + (q & 1)];
                    *(my.tip == 3 ? S.bc : S.frc + 3 + my.tip) = v;
                }
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
            sum_tip();
            if (mid && s == 0) {            // midpointStep's half step
                FOR_ENTRIES(p, o) {
                    const int e = o.e;
                    const double f = force(o, p), v = S.vel[e], x0 = S.pos[e];
                    const bool free_ = o.moves;
                    S.pev[e] = free_ ? x0 + dt / 2 * v : x0;
                    S.vst[e] = v + dt / 2 * f;
                }
                block_sync();
                s = 1;
                continue;
            }
            if (rk4) {                                // stages at pos, pos + dt/2 v1, pos + dt/2 v2, pos + dt v3
                FOR_ENTRIES(p, o) {
                    const int e = o.e;
                    const double fs = force(o, p), vs = s == 0 ? S.vel[e] : S.vst[e];
                    const bool free_ = o.moves;
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
                FOR_ENTRIES(p, o) {
                    const int e = o.e;
                    const double f = force(o, p);
                    S.frc[e] = f;
                    if (o.moves && !sd) {  // midpointStep, eulerStep; masses are 1
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
                FOR_ENTRIES(p, o)
                    if (o.moves) S.pos[o.e] = S.pos[o.e] + a.dt * S.frc[o.e];
            } else {
                FOR_ENTRIES(p, o) S.vst[o.e] = fire_mix(S, o.e, alpha);
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
// evaluation.
__device__ inline State sys_layout(double* p, const SysArgs& a) {
    const int n = a.n_atoms;
    State S;
    S.pdot = p; p += flex_padded(n);
    S.bc = p; p += 4;
    S.res = p; p += a.n_res + 8;
    S.all = p; p += sys_energy_doubles(a);
    S.pos = p; p += 3 * n;
    S.pev = p; p += 3 * n;
    S.vel = p; p += 3 * n;
    S.vst = p; p += 3 * n;
    S.frc = p; p += 3 * n;
    S.facc = p; p += 3 * n;
    S.vacc = p; p += 3 * n;
    S.eacc = p; p += n;
    S.ener = p;
    return S;
}

template <bool IN_LDS>
__global__ void __launch_bounds__(256, 2) k_system_op(SysArgs a) {
    extern __shared__ __align__(16) double lds_sys[];
    const int t = threadIdx.x, nthr = blockDim.x;
    const int n = a.n_atoms;
    const size_t nd = sys_block_doubles(a);
    double* base = IN_LDS ? lds_sys : a.work + (size_t)blockIdx.x * nd;
    State S = sys_layout(base, a);
    const int32_t* idx = a.idx;
    if (IN_LDS) {
        int32_t* l = reinterpret_cast<int32_t*>(lds_sys + nd);
        for (int q = t; q < a.n_rows + 3 * n; q += nthr) l[q] = a.idx[q];
        idx = l;
    }
    S.tables(idx, a.n_rows, n);
    const bool minimise = a.op == SYS_MINIMISE, sd = minimise && a.minimiser == MAFM_MIN_SD;
    const bool rk4 = !sd && a.op != SYS_EVAL && a.integrator == MAFM_INT_RK4;
    const bool mid = !sd && a.op != SYS_EVAL && a.integrator == MAFM_INT_MIDPOINT;
    const bool all_e = sys_all_energies(a);
    const int others = 4 * flex_padded(a.n_tip);
    Results R = {S.res, S.all, others, a.n_res, all_e ? E_ALL : E_TIP};
    Evaluator<IN_LDS> eval;
    eval.init(a.terms, a.rounds, t, nthr);
    block_sync();
    S.pad(n, a.n_tip, others, all_e, t, nthr);
    const Places my(t, nthr, n);
    const Own first = t < my.n3 ? S.own(t) : Own{0, 0, false};
    const Own tip_own = {3 + my.tip, 0, S.fixed[1] != 1};
    double tip_sum = 0;               // of the thread's component of the tip, from f0 (its energy: e0)
    auto sum_tip = [&](bool onto) {
        if (my.tip < 0) return;
        const double from = !onto ? 0.0 : my.tip == 3 ? S.ener[1] : S.frc[3 + my.tip];
        tip_sum = list_sum<8>(from, S.res + 2 * my.tip, a.n_tip);
        if (my.tip == 3) S.bc[0] = tip_sum;
    };
    auto force = [&](const Own& o, int p, double f0) {
        return p >= my.n3 ? tip_sum : row_sum<1>(f0, S.res + others, S.rows, o.slots, 2 * p);
    };
    // every atom's energy into `to`, the others' from what `from` gives for them
    auto energies = [&](auto from, auto to) {
        if (my.tip == 3) to(1, tip_sum);
        for (int k = t; k < n - 1; k += nthr) {
            const int i = S.order[k];
            to(i, row_sum<3>(from(i), S.all, S.rows, S.cnt[k], 2 * k));
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
            FOR_ENTRIES(p, o) {
                const int e = o.e;
                if (!up) S.vel[e] = 0;
                else if (o.moves) S.vel[e] = S.vst[e];
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
            if (pending && t == nthr - 1) S.bc[1] = list_sum<2>(0.0, S.pdot, n);
            R.mode = last ? E_ONLY : (all_e ? E_ALL : E_TIP);
            eval(s == 0 && !last ? S.pos : S.pev, R);
            block_sync();
            if (pending) apply();
            if (last) {
                if (my.tip == 0) S.ener[1] = list_sum<8>(0.0, S.res, a.n_tip);
                for (int k = t; k < n - 1; k += nthr)
                    S.ener[S.order[k]] = row_sum<1>(0.0, S.res + others, S.rows, S.cnt[k], 6 * k);
                break;
            }
            sum_tip(onto);
            if (a.op == SYS_EVAL) {
                FOR_ENTRIES(p, o) S.frc[o.e] = force(o, p, S.frc[o.e]);
                energies([&](int i) { return S.ener[i]; }, [&](int i, double e) { S.ener[i] = e; });
                break;
            }
            if (mid && s == 0) {                      // midpointStep's half step
                FOR_ENTRIES(p, o) {
                    const int e = o.e;
                    const double f = force(o, p, 0.0), v = S.vel[e], x0 = S.pos[e];
                    const bool free_ = o.moves;
                    S.pev[e] = free_ ? x0 + dt / 2 * v : x0;
                    S.vst[e] = free_ ? v + dt / 2 * f : v;
                }
                block_sync();
                s = 1;
                continue;
            }
            if (rk4) {                                // rk4Step
                FOR_ENTRIES(p, o) {
                    const int e = o.e;
                    const double fs = force(o, p, 0.0), vs = s == 0 ? S.vel[e] : S.vst[e];
                    const bool free_ = o.moves;
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
                FOR_ENTRIES(p, o) {
                    const int e = o.e;
                    const double f = force(o, p, onto ? S.frc[e] : 0.0);
                    S.frc[e] = f;
                    if (o.moves && !sd) {
                        const double x0 = S.pos[e];
                        if (!mid) S.pev[e] = x0;      // where this step evaluated
                        S.pos[e] = x0 + dt * (mid ? S.vst[e] : S.vel[e]);
                        S.vel[e] = S.vel[e] + dt * f;
                    }
                }
                if (all_e) {
                    energies([&](int i) { return onto ? S.ener[i] : 0.0; }, [&](int i, double e) { S.ener[i] = e; });
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
                    FOR_ENTRIES(p, o)
                        if (o.moves) {
                            S.pev[o.e] = S.pos[o.e];
                            S.pos[o.e] = S.pos[o.e] + a.dt * S.frc[o.e];
                        }
                } else {
                    FOR_ENTRIES(p, o) S.vst[o.e] = fire_mix(S, o.e, alpha);
                    pending = true;
                }
                ++n_tot;
            } else if (sd) {
                FOR_ENTRIES(p, o) S.pev[o.e] = S.pos[o.e];
            }
            block_sync();
            if (done || n_tot >= a.maxsteps) {
                if (!all_e) {         // one more trip for every atom's energy
                    last = true;
                    continue;
                }
                if (pending) {
                    if (t == nthr - 1) S.bc[1] = list_sum<2>(0.0, S.pdot, n);
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
