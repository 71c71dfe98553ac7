// Device arguments of the flexible scan (scan_flex.hip), shared with the
// host side that fills them (api.cpp).
#pragma once
#include "../../include/mafm.h"
#include "device_common.hpp"

namespace mafm {

constexpr int FLEX_HELD_ROUNDS = 4;   // rounds whose terms a thread keeps in registers

// Lists that one thread sums (the atoms' powers, the tip's energies) are padded
// to whole batches.
constexpr int FLEX_BATCH = 16;
__host__ __device__ inline int flex_padded(int n) { return (n + FLEX_BATCH - 1) / FLEX_BATCH * FLEX_BATCH; }

// One interaction as the kernels read it.  Every term is evaluated once per
// integrator stage into result slots {fx, fy, fz}, one per atom it acts on,
// holding the signed force that atom receives (the reference's `forces[i] -= f`
// is `+= -f`, the same rounding).  An atom's slots are numbered in the
// interaction list's order, the order its force is summed in.  They lie in pairs,
// a slot's components two doubles apart: the tip's slot q, with its energy behind
// the force, at 8 (q / 2) + q % 2; slot q of the other atom of rank k (by falling
// number of slots) behind the tip's at row[q / 2] + 6 k + q % 2.
struct FxTerm {
    int32_t kind;                     // MAFM_FX_*; -1: nothing to evaluate
    int32_t atom[4];
    int32_t slot[4];                  // place of each atom's result slot; n_res: not read
    int32_t place[2];                 // place of its energy where it acts on the tip; n_res: not read
    int32_t pad;
    double q[6];                      // pair terms: p0, p1, p2, shift x, y, z; else mafm_flex_term::p
};

// The term records lie in schedule order: thread l of the block takes record
// r * block threads + l in rounds r < rounds.  The schedule only places the
// work; the slots are summed in list order.
struct FlexArgs {
    int32_t n_atoms, n_res, n_tip;    // doubles of results; slots of the tip
    int32_t tip_ts_slots;             // the tip's first slots, from tip-surface terms
    int32_t nx, ny, nz;
    double dx, dy, dz, zhigh;
    int32_t minimiser, integrator, minterm, maxsteps;
    double etol, ftol, dt;
    const FxTerm* terms;
    int32_t rounds;
    // index tables, back to back: the rows' places (n_rows: 12 more than rows,
    // rounded to whole fours), slots of each rank (none for fixed atoms; the last
    // place is unused), its atom, fixed flags by atom (n_atoms each)
    const int32_t* idx;
    int32_t n_rows;
    const double* pos0;               // n_atoms x 3
    int32_t tip_pbc;
    int32_t state_col;                // column whose positions are kept per height, -1 none
    double cell[9], cell_inv[9], offset[3];
    double tip_dummy_d;
    DevRecord* rec;
    int32_t* next_col;                // work counter, zero at launch
    double* state;                    // nz x n_atoms x 3
    double* work;                     // per-block state when it does not fit LDS
};

// The reference's System-level operators on n_states independent copies of
// one system (one workgroup each): the whole interaction list evaluated into
// every atom's force and energy, one integrator step, or a whole FIRE / SD
// minimisation from the given state.
enum { SYS_EVAL = 0, SYS_STEP = 1, SYS_MINIMISE = 2 };
struct SysArgs {
    int32_t n_atoms, n_res, n_tip, n_rows, op;
    int32_t minimiser, integrator, minterm, maxsteps;
    double etol, ftol, dt;
    int64_t n_states;
    const FxTerm* terms;              // as FlexArgs; every atom's roles have a slot
    int32_t rounds;
    const int32_t* idx;               // as FlexArgs
    double* pos;       // n_states x n_atoms x 3, in and out
    double* vel;       // n_states x n_atoms x 3, in and out (step, minimise)
    double* frc;       // n_states x n_atoms x 3: in (eval and the Euler step add to it), out
    double* ener;      // n_states x n_atoms: as frc; minimise reads energies[1] as the last tip energy
    int32_t* steps;    // n_states (minimise)
    double* work;      // per-block state when it does not fit LDS
};
hipError_t launch_system_op(const SysArgs& a, int waves, bool in_lds, hipStream_t st);

// Doubles of state a block keeps: the atoms' powers (a list), four broadcast
// values, the results and eight more, then positions, integrator stages,
// velocities and forces.  The sums load a batch past the end of a list and, of a
// row, what wider rows have: both fall on the state behind the results, except
// that with two or three atoms the tip's list needs more than there is.
// Even: the index tables behind the state are read four at a time.
__host__ __device__ inline size_t flex_state_doubles(int n, int n_res, int n_tip, size_t behind) {
    const size_t own = n_res + 8 + behind, list = 4 * (size_t)(flex_padded(n_tip) + FLEX_BATCH);
    const size_t all = flex_padded(n) + 4 + (own > list ? own : list);
    return all + (all & 1);
}
__host__ __device__ inline size_t flex_block_doubles(const FlexArgs& a) {
    const bool rk4 = a.minimiser == MAFM_MIN_FIRE && a.integrator == MAFM_INT_RK4;
    return flex_state_doubles(a.n_atoms, a.n_res, a.n_tip, (size_t)(15 + (rk4 ? 6 : 0)) * a.n_atoms);
}
// LDS bytes of one block when the state lives there (state + index tables).
inline size_t flex_block_lds(const FlexArgs& a) {
    return flex_block_doubles(a) * sizeof(double) + (a.n_rows + 3 * (size_t)a.n_atoms) * sizeof(int32_t);
}

// All energies of each evaluation are kept by eval, one step and RK4.
__host__ __device__ inline bool sys_all_energies(const SysArgs& a) {
    return a.op != SYS_MINIMISE || (a.minimiser != MAFM_MIN_SD && a.integrator == MAFM_INT_RK4);
}
__host__ __device__ inline size_t sys_energy_doubles(const SysArgs& a) {
    return sys_all_energies(a) ? (a.n_res - 4 * flex_padded(a.n_tip)) / 3 + 2 : 0;
}
__host__ __device__ inline size_t sys_block_doubles(const SysArgs& a) {
    return flex_state_doubles(a.n_atoms, a.n_res, a.n_tip, sys_energy_doubles(a) + (size_t)23 * a.n_atoms);
}
inline size_t sys_block_bytes(const SysArgs& a) {   // with the index tables
    return sys_block_doubles(a) * sizeof(double) + (a.n_rows + 3 * (size_t)a.n_atoms) * sizeof(int32_t);
}
// waves: wavefronts per workgroup (1-4); in_lds: the state lives in LDS (else
// in a.work, one slice per block).
hipError_t launch_scan_flex(const FlexArgs& a, int n_blocks, int waves, bool in_lds, hipStream_t st);

}  // namespace mafm
