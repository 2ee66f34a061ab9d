// The resident form of the fused engine's step loop (rk_resident.hip): one
// launch runs many attempts, its workgroups staying on the chip.
#pragma once
#include <hip/hip_runtime.h>

#include "qa_coef.h"
#include "qa_rk.h"

namespace qa {

constexpr int kResRing = 32;        // slots of the stage-input ring
constexpr int kResKept = 16;        // entries a lane keeps
constexpr int kResSyncWords = 2048; // control words of one launch (see rk_resident.hip)
constexpr int kResPolls = 1 << 20;  // polls of a wait, unless an engine sets them

// The combine lists of the tableau: x_{i+1} (or y_front, for the last step
// stage) = y_prev + sum_t dt tc[i][t] k_{tj[i][t]} + dt cs[i] k_i; the error
// takes te, ce of the last step stage.  List kMaxStages: the input of the
// first dense-output stage when it is not y_front.
struct ResTab {
    double tc[kMaxStages + 1][kMaxStages];
    double te[kMaxStages];
    double cs[kMaxStages + 1];
    double ce;
    double c[kMaxStages];                    // stage times
    double bi[kMaxStages][kMaxDenseOrder];   // dense-output table
    int tj[kMaxStages + 1][kMaxStages];
    int nt[kMaxStages + 1];
    int pad;
};

struct ResArgs {
    int n, nslices, threads, nwg, grid, nblk;  // nblk: 256-lane blocks (error partials)
    int64_t npad;
    int multi;  // workgroups on every XCD (0: on one)
    int rk_step, nk, dorder, has_bi, dense, first_front;
    // operator: SELL-C, coded SELL-C or diagonals
    const int *slice_ptr, *col;
    const void *vals;
    const uint2 *code;
    const double2 *vtab;
    const int *otab;
    int vbits, lanes, fp32;
    CoefSet td;
    // engine state
    RKCtl *ctl;
    double2 *y0, *y1, *K, *y_last;
    double2 *ring;
    double *parts;   // [2][nblk]
    unsigned *sync;  // kResSyncWords
    const ResTab *tab;
    // outputs: the states of rows with need[r] >= 0 go to yout[output -
    // out_base][need[r]]; at most out_cap outputs a launch
    const int *need;
    double2 *yout;
    int nneed, out_base, out_cap;
    int max_attempts;
    int polls;  // bound of every wait, in polls of 0.4 us or more
};

// RES_KEPT: at most kResKept entries a lane, kept in registers; the others
// read the operator every stage (time-dependent generators always: keeping
// their entries too made the coefficient programs spill, 6.9 against 5.2 ms
// on a driven chain of 4096 rows).
enum ResForm { RES_KEPT = 0, RES_SELL = 1, RES_SELL_F32 = 2, RES_CODED = 3, RES_CODED_TD = 4,
               RES_DIA = 5 };

// Dynamic LDS of a workgroup.
size_t res_lds_bytes(int form, int lanes, int threads, int nk, int vbits);
// Threads and workgroups for `lanes_total` lanes; false when the shape does
// not fit this device (compute units, XCDs, LDS).
bool res_plan(int form, int lanes, int64_t lanes_total, int nk, int vbits, ResArgs *P);
// Clears the control words and launches the loop on s.  On an error the
// state is as it was (at most the control words are cleared).
int res_launch(int form, const ResArgs &P, const DiaOp &D, hipStream_t s);

// The functionals of the outputs of a launch, from yout.
struct ResFunArgs {
    const RKCtl *ctl;
    const double2 *yout;
    int nneed, out_base, nfun;
    const int *fptr, *fkind, *frow, *fcol;  // entries by slot of yout
    const double2 *fw;
    double2 *fun_out;
};
int res_functionals(const ResFunArgs &A, int nout, hipStream_t s);

}  // namespace qa
