// Front program of the sparse LU: the numeric refactorisation and the two
// solves as small dense fronts on the elimination tree.
//
// The circuits' fill, once the supply and source rows are out of the way, is
// a tree of tiny dense blocks (65k-gate DAG: 25k fronts of at most 60 rows).
// A front holds k pivots and the s later rows (= columns: the structure of
// the LU pattern is made symmetric) that they update.  One wavefront
// assembles a front from matrix entries and its children's update blocks,
// eliminates its k pivots and leaves the s x s update block to its parent, so
// a pivot costs a few register operations in place of a level of indexed
// updates with a barrier.
//
// Singletons.  A column with one entry (the current of a source) and a row
// with one entry (a source's voltage) cause no fill; they are eliminated
// first and stay outside the fronts: the row singletons' columns are
// subtracted from the right-hand side, the column singletons' rows are summed
// after the solve.  That takes the supply rail, whose row and column touch
// most of the circuit, out of every front.
#pragma once

#include <cstdint>
#include <string>
#include <vector>

namespace vjx {

// Largest front (pivots + update rows): one wavefront holds it as an 8 x 8
// grid of lanes with at most 8 x 8 values each.
constexpr int kFrontMax = 64;
constexpr uint16_t kNoPos = 0xffff;

// One front of a block pattern.  Offsets named `block` count from the block
// instance's base (FrontInst), the others are absolute in the program.
struct FrontDesc {
  int32_t k, m;     // pivots, pivots + update rows
  int32_t r0;       // first pivot (block; permuted rows r0 .. r0 + k - 1)
  int32_t fac;      // factors (block): k columns of m values, then s columns of k
  int32_t cb;       // own update block, s x s column-major (block)
  int32_t cv;       // own s solve contributions (block)
  int32_t idx;      // s update rows (permuted, block) in FrontProgram::idx
  int32_t a0, na;   // matrix entries: FrontProgram::apos; sources at a0 + FrontInst::asrc
  int32_t c0, nc;   // children's update blocks: nc values from c0 (block) ...
  int32_t cpos;     // ... and their positions in FrontProgram::cpos
  int32_t v0, nv;   // children's solve contributions from v0 (block), at most nv per row
  int32_t vtab;     // row i's c-th contribution: v0 + FrontProgram::vtab[vtab + c * m + i]
  int32_t nt;       // ceil(m / 8)
  int32_t rounds;   // largest number of children's values on one position
                    // (above kMaxRounds: kMaxRounds + 1)
  int32_t pad0, pad1, pad2;
};

// cpos: position, and in the upper bits its number among the children's values
// on that position, in the children's order.
constexpr int kPosBits = 13;
constexpr int kPosMask = (1 << kPosBits) - 1;
constexpr int kMaxRounds = 7;  // numbers 0 .. 6 (7 marks kNoPos); later ones keep 6

// One diagonal block of the system.
struct FrontInst {
  int32_t row, fac, cb, cv, asrc, pad0, pad1, pad2;
};

// Leading dimension (and column count 8 nt) of a front in LDS: 8 times an odd
// number, so that four 8-value columns start on distinct bank groups.
constexpr int front_ld(int nt) { return 8 * (nt | 1); }
constexpr int front_lds(int nt) { return 8 * nt * front_ld(nt); }

struct FrontProgram {
  std::vector<FrontDesc> fronts;
  std::vector<FrontInst> inst;
  std::vector<int32_t> idx;
  std::vector<uint16_t> apos, cpos, vtab;
  std::vector<int32_t> asrc;  // per instance: matrix entry of each apos
  // Stages, one launch each: a task is a piece of the tree whose children
  // pieces belong to earlier stages.  Stage 0's tasks are subtrees of fronts
  // of at most 32 rows, walked level by level by one workgroup, one front per
  // wavefront; a task of a later stage is one front, or a chain of fronts
  // with no other child left, by a whole workgroup.
  std::vector<int32_t> stage_task;  // stage g: tasks [stage_task[g], stage_task[g + 1])
  std::vector<int32_t> stage_nt;    // largest nt of the stage
  std::vector<int32_t> task;        // 4 ints: instance, first level, levels, first in order
  std::vector<int32_t> level;       // level l: order[level[l] .. level[l + 1])
  std::vector<int32_t> order;       // front ids
  int32_t n_fac = 0, n_cb = 0, n_cv = 0;  // sizes over all instances
  // Singletons.  Values in the factor storage from n_fac on: value i is
  // matrix entry sg_src[i], divided by entry sg_div[i] where that is >= 0.
  std::vector<int32_t> sg_src, sg_div;
  // entries of row-singleton columns in permuted row r: [rs_ptr[r],
  // rs_ptr[r + 1]), value rs entry e = sg value e, times right-hand side row
  // rs_rhs[e]
  std::vector<int32_t> rs_ptr, rs_rhs;
  // row singletons {permuted row, value of the pivot}
  std::vector<int32_t> row_single;
  // column singletons {permuted row, value of the pivot, first entry, end};
  // entry e: value e, column us_col[e - us_first] (original numbering)
  std::vector<int32_t> col_single;
  std::vector<int32_t> us_col;
  int32_t us_first = 0;
  // chunks of the column singletons' rows {row's index, first entry, end, chunks of the row}
  std::vector<int32_t> us_chunk;
  bool on() const { return !inst.empty(); }
  // One task does it all (a small circuit): factors and solves are one launch
  // each, or one together, with everything in LDS.  Offsets in bytes, for
  // 8-byte values; 0 total: not that kind.
  struct Tiny {
    int32_t desc, level, idx, vtab, apos, cpos, av, fac, sg, cb, cv, y, z, front, total;
    int32_t n_fronts, n_level, n_idx, n_vtab, n_a, n_c, n_fac, n_rows, lds_wave;
  } tiny = {};
  int64_t storage() const { return (int64_t)n_fac + (int64_t)sg_src.size(); }
};

// Plan of one block pattern (positions as in FrontProgram, all block-relative).
struct FrontPlan {
  bool ok = false;
  int n_col_single = 0, n_row_single = 0;  // pivots [0, ncs), [ncs, ncs + nrs)
  std::vector<FrontDesc> fronts;
  std::vector<int32_t> parent;
  std::vector<int32_t> idx;
  std::vector<uint16_t> apos, cpos, vtab;
  std::vector<int32_t> asrc;  // local matrix entry
  std::vector<int32_t> rows_below;  // pivots in each front's subtree
  int32_t n_fac = 0, n_cb = 0, n_cv = 0;
};

struct LuSymbolic;

// Column and row singletons of a matrix: the pivot order starts with them.
// sc / sr: columns and rows of the column singletons, rc / rr: of the row
// singletons.
struct Singletons {
  std::vector<int32_t> sc, sr, rc, rr;
};
void find_singletons(int n, const int32_t* indptr, const int32_t* indices, const double* vals,
                     double pivot_tol, Singletons& out);

// Tree, fronts and a pivot order in which every front's pivots are
// consecutive, from the factors' pattern (L columns / U columns, permuted
// rows).  np[k]: new position of pivot k.  False (nothing written) when a
// front would exceed kFrontMax or the padding costs too much.
bool plan_fronts(int n, int n_single, const std::vector<int64_t>& lptr,
                 const std::vector<int32_t>& lidx, const std::vector<int64_t>& uptr,
                 const std::vector<int32_t>& uidx, FrontPlan& plan, std::vector<int32_t>& np);

// Matrix entries of the fronts: every entry (permuted row i, column j) with
// both in the core, local entry id e.
void plan_entries(const std::vector<int32_t>& rows, const std::vector<int32_t>& cols,
                  const std::vector<int32_t>& ids, FrontPlan& plan);

// Program of a system from its blocks' plans: block c uses plan
// plans[kind[c]], starts at permuted row row0[c] and reads matrix entry
// entry[c][e] for the plan's local entry e.
void assemble_program(const std::vector<const FrontPlan*>& plans, const std::vector<int32_t>& kind,
                      const std::vector<int32_t>& row0,
                      const std::vector<std::vector<int32_t>>& entry, int n,
                      FrontProgram& out);

// Largest number of fronts one workgroup takes by itself, and its wavefronts.
// A small circuit is all launches and waiting: a 200-section RC ladder (37
// fronts) as two stages of eight workgroups and one took 195 us a time step.
constexpr int kTinyFronts = 128;
constexpr int kTinyWaves = 8;
// The tiny form's LDS layout (F.tiny) when everything fits a workgroup.
void tiny_layout(FrontProgram& F, int n_rows);

// Offset in the factor storage of every LU slot (s.rowptr / s.col), given the
// program's fronts and singletons.
void front_slot_map(const LuSymbolic& s, std::vector<int32_t>& map);

// Checks of a program: every LU entry has its own place, every matrix entry
// reaches one place, levels and stages follow the tree.
bool check_fronts(const LuSymbolic& s, std::string& err);

template <typename T>
void fronts_refactor_host(const LuSymbolic& s, const double* a, T* fac);
template <typename T>
void fronts_solve_host(const LuSymbolic& s, const T* fac, const double* b, double* x);

}  // namespace vjx
