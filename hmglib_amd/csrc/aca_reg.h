// aca_reg.h -- the adaptive cross approximation with the block's factors held by its
// team (aca.hip states the method and its rules, and keeps the memory form for the
// blocks that this form does not take).
//
// A team of NW wavefronts runs one block.  Thread t holds row t of U_b and of the row
// cluster's points, and column t of V_b and of the column cluster's points, so blocks of
// up to 64 NW rows and columns fit.  The first NT rank terms (8 or 16) live in registers,
// the next eight in LDS, later ones in the factors' own storage.  A rank step reads none
// of the former from memory: the pivot row's U terms and the pivot column's V terms go to
// all threads through LDS, and the factors are written once, at the end.  Wider blocks
// keep V column-major in a slab of the workgroup, where the lanes of a wavefront read
// consecutive values.
//
// After a rejected row the norms of the next four are formed together (one pair of
// barriers).  A search for the next acceptable row that does not end soon is not run by
// the team: the block writes what it has, joins a queue, and a search over all
// queued blocks (one row per lane, every compute unit) finds the row with which the
// team resumes.
#pragma once
#include "hmg_internal.h"
#include "kernel_eval.h"

namespace hmg {

// Tolerance stop of the ACA (aca.hip)
struct AcaTol {
    int mode;
    double c;
};

// Operands of one ACA launch: list[] names the blocks, factors of block a start at
// ublk[a] / vblk[a], or at U + uoff[a] / V + voff[a] without them.
struct AcaArgs {
    Coords c1, c2;
    KernelParams kp;
    const int4* blk;
    const work_item* items;
    const int* list;
    const int* kb;
    const int64_t* uoff;
    const int* ldu;
    const int64_t* voff;
    const int* ldv;
    double* U;
    double* V;
    double* const* ublk;
    double* const* vblk;
    int* keff;
    int tie_last;
    int scan;
    AcaTol tol;
    int few;            // at most that many teams leave most of the chip idle
    int nlist;          // blocks in list[] (resumed ones: at most that many, *count of them)
    const int* count;
    int resume;         // the blocks of list[] were suspended
    // suspended blocks: the launch appends block indices to queue[] at *queued; row[a] is
    // the last row the block rejected, found[a] the row the search found (m1: none),
    // fro2[a] its tolerance sum
    int suspend;        // long searches suspend their block
    int tries;          // rejected rows in a row after which a block is suspended
    int* queue;
    int* queued;
    int* row;
    int* found;
    double* fro2;
    // wide teams: nslabs slabs of slab elements, one per workgroup, and the launch's work
    // counter
    double* slabs;
    int64_t slab;
    int nslabs;
    int* next;
};

constexpr int kRegSlots = 1;    // rows and columns per thread
static_assert(kRegSlots == 1, "the look-ahead over rejected rows takes the first slot only");
constexpr int kRegTail = 8;     // rank terms in LDS after the ones in registers
constexpr int kRegRank = 64;    // largest rank of the register form
// rows of one workgroup of the search over suspended blocks
constexpr int kSearchRows = kWave;

// Launches the g.nlist blocks of g.list[] on teams of nw wavefronts: 1, 2, 3, 4, 5, 8, 9, 12
// or 16 (every block within 64 nw rows and columns), or with wide set 4 or 8 (blocks of any
// size; a slab holds at least k x m2 elements of each).  Dimension 2 or 3; kmax: the
// largest rank among the blocks.  One translation unit per kernel kind.
template <int KIND>
hmg_status aca_reg_launch(const AcaArgs& g, int nw, bool wide, int kmax, hipStream_t s);
// g.found[a] of the *g.count suspended blocks in g.list[] becomes the first row after
// g.row[a] that may be acceptable at rank step g.keff[a] (m1 when there is none); maxm1:
// the largest row count among them
template <int KIND>
hmg_status aca_search_launch(const AcaArgs& g, int maxm1, hipStream_t s);

}  // namespace hmg
