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
size_t sys_block_doubles(const SysArgs& a);
size_t sys_block_bytes(const SysArgs& a);   // with the index tables
hipError_t launch_system_op(const SysArgs& a, int waves, bool in_lds, hipStream_t st);

// Doubles of per-column state one block keeps (positions, integrator
// stages, velocities, forces, term results).
size_t flex_block_doubles(const FlexArgs& a);
// LDS bytes of one block when the state lives there (state + index tables).
size_t flex_block_lds(const FlexArgs& a);
// waves: wavefronts per workgroup (1-4); in_lds: the state lives in LDS (else
// in a.work, one slice per block).
hipError_t launch_scan_flex(const FlexArgs& a, int n_blocks, int waves, bool in_lds, hipStream_t st);

}  // namespace mafm
