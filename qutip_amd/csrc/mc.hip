// Batched Monte-Carlo wave-function trajectories (mcsolve) on gfx950.
//
// One workgroup runs one trajectory from the first to the last output time
// (grid-stride over trajectories), with no host round trip: the explicit
// Runge-Kutta integrator in its "mcstep" form, the norm-based collapse
// search and the quantum jumps all run on the device.  Trajectories advance
// independently with their own step sizes and jump counts; a workgroup that
// finishes early simply picks up the next trajectory.
//
// Restated algorithms (qutip/solver/...):
//   RK step, step control, dense output     integrator/explicit_rk.pyx:204-467
//   integrate(t, step=True)  (mcstep)        explicit_rk.pyx:278-331
//   MCIntegrator.set_state / integrate       mcsolve.py:245-302
//   _find_collapse_time (log-ratio secant)   mcsolve.py:321-369
//   _do_collapse (channel choice, jump)      mcsolve.py:371-406
//   H_eff = -iH - 1/2 sum c^dag c            mcsolve.py:491-496 (built on host)
// Random numbers: the uniform draws of numpy's Generator (PCG64 seeded by
// SeedSequence(seed), multitraj.py:354-393) are produced on the host in the
// order the reference consumes them (mcsolve.py:276-279, 388, 405) and
// streamed in; a trajectory that uses up its draws stops with a status the
// host acts on.
//
// Layout: each thread owns one row of the state (d <= 1024).  The RK stage
// vectors stay on the chip for the whole trajectory, k_0..k_9 in registers
// and k_10..k_15 in LDS.  The vector an RHS product reads is staged in LDS.
// A vern7 run on an operator of few entries a row and few distinct values has
// it packed: 16-bit codes in registers, values in LDS, so a stage touches no
// other memory.  Else H_eff is a column-major ELL (entry u of row r at
// u d + r), so the 64 lanes of a wave, which own 64 consecutive rows, load 64
// consecutive columns and values per instruction, from L2; c_ops and e_ops
// (used at jumps and outputs only) are CSR.  Norms, error norms and
// expectation values accumulate in FP64; with the complex64 variant the
// state, stages and RHS products are FP32.
//
// What bounds it: a stage is a chain (sum of stages, LDS write, barrier,
// gathers, multiply-adds) of some 1700 clocks with one workgroup a CU, and
// with 16 waves a CU the instructions and the LDS bytes of the gathers.
// Measured against the ELL form with two rows a thread and a run-time
// tableau, Ising chains with vern7, kernel time: L = 10, 2048 trajectories:
// complex128 140 -> 51 ms, complex64 104 -> 69; L = 8, 500 of them: 4.2 ->
// 1.9 ms and 3.8 -> 2.4; L = 8, 8192: 62 -> 15 ms and 41 -> 21; whole solve of a 400-row
// Liouvillian: 5.5 -> 2.9 ms.  What gave it, for L = 10: no ELL in the
// stages, one row a thread and stages in registers (the spills gone from the
// stage loop) 140 -> 104, compile-time stage loops with step and dense output
// apart 104 -> 53.
#include <algorithm>
#include <math.h>
#include <string.h>

#include "qa_api_internal.h"
#include "qa_common.h"

using namespace qa;

namespace {

constexpr int kMcStages = 16;
constexpr int kMcOrder = 8;
constexpr int kMcMaxChan = 32;
constexpr int kMcMaxEops = 8;
constexpr int kMcThreads = 1024; // threads of a workgroup at most

// trajectory status codes (beside the RK codes of explicit_rk.pxd:5-12)
enum McStatus {
    MC_OK = 0,
    MC_TOO_MUCH_WORK = -1,
    MC_DT_UNDERFLOW = -2,
    MC_OUTSIDE_RANGE = -3,
    MC_COLLAPSE_NOT_FOUND = -10,  // mcsolve.py:363-367 RuntimeError
    MC_DRAWS_EXHAUSTED = -11,     // host re-runs with more pre-drawn numbers
    MC_NO_PROGRESS = -12
};
enum RkStatus { RK_AT_FRONT = 2, RK_INTERPOLATED = 1, RK_NORMAL = 0 };

struct McTableau {
    double a[kMcStages][kMcStages];
    double b[kMcStages];
    double c[kMcStages];
    double e[kMcStages];
    double bi[kMcStages][kMcOrder];
    int order, rk_step, rk_extra, dorder, interpolate, adaptive, fsal, pad;
};

struct McArgs {
    int d, ntraj, ntimes, nchan, neops, max_draws, max_jumps, traj_offset;
    int h_width;       // ELL width of H_eff
    const int *h_col;  // [h_width][d] column-major ELL (entry u of row r at u d + r)
    const void *h_vals;
    const int *c_rowptr, *c_col;  // nchan blocks of d + 1 row pointers (absolute)
    const void *c_vals;
    const int *e_rowptr, *e_col;
    const void *e_vals;
    const McTableau *tab;
    const double *times;
    const double2 *psi0;
    const double *draws;  // [ntraj][max_draws]
    double rtol, atol, first_step, min_step, max_step;
    int nsteps, norm_steps;
    double norm_t_tol, norm_tol, norm_min_step, mc_corr_eps;
    double2 *expect_out;  // [ntraj][ntimes][neops]
    double *col_times;    // [ntraj][max_jumps]
    int *col_which;
    int *info;  // [ntraj][4]: status, jumps, draws used, RK attempts
    // whole-solve mode (rk_small_kernel): per-system operator stride
    // (entries; 0 = one shared operator), start time, linear / quadratic
    // functionals of the state, outputs
    long long h_stride;
    double t0;
    int nfun;
    const int *f_kind, *f_ptr, *f_row, *f_col;
    const double2 *f_w;
    double2 *fun_out;  // [nsys][ntimes][nfun]
    double2 *y_final;  // [nsys][d] or null
    int fun_lds;       // LDS bytes reserved for the functionals and times (0: none)
    int x2;            // a second LDS copy of the product's input vector is reserved
    // packed operator (OP_PACKED, OP_PACKED_IM), or pk_width 0: the diagonal
    // [d], and up to kMcPack off-diagonal entries a row as 16-bit codes,
    // entry u of row r at u d + r: column | value index << pk_cbits; index 0
    // is the value 0
    const unsigned short *pk_code;
    const void *pk_diag, *pk_tab;
    int pk_width, pk_cbits, pk_ntab, pk_imag;
};

// Forms of the shared operator.  OP_ELL: columns and values from global
// memory (or LDS, rk_small_kernel's HL); OP_PACKED: codes and the diagonal
// in registers, the distinct values in LDS; OP_PACKED_IM: the same with
// purely imaginary off-diagonal values (-i H of a real H).
enum OpForm { OP_ELL = 0, OP_PACKED = 1, OP_PACKED_IM = 2 };
constexpr int kMcPack = 16;     // packed entries a row
constexpr int kMcPackTab = 256; // distinct packed values
constexpr int kPackStep = 10;   // stages of a step, and with the dense output,
constexpr int kPackExtra = 16;  // of the tableau that goes with a packed operator

// A double that every thread of the workgroup holds alike, kept in scalar
// registers: assignments go through lane 0.  The trajectory's times and
// norms would take some forty vector registers otherwise, and comparisons of
// them would mask lanes instead of branching.
__device__ __forceinline__ double uni(double v) {
    return __hiloint2double(__builtin_amdgcn_readfirstlane(__double2hiint(v)),
                            __builtin_amdgcn_readfirstlane(__double2loint(v)));
}
struct Uni {
    double v;
    __device__ __forceinline__ Uni() : v(0.0) {}
    __device__ __forceinline__ Uni(double x) : v(uni(x)) {}
    __device__ __forceinline__ operator double() const { return v; }
};

template <typename R>
struct cplx_t;
template <>
struct cplx_t<double> {
    using type = double2;
};
template <>
struct cplx_t<float> {
    using type = float2;
};

template <typename R>
using C2 = typename cplx_t<R>::type;

template <typename R>
__device__ __forceinline__ C2<R> mk(R x, R y) {
    C2<R> v;
    v.x = x;
    v.y = y;
    return v;
}
template <typename R>
__device__ __forceinline__ void cfmaR(C2<R> &acc, C2<R> a, C2<R> b) {
    acc.x = fma(a.x, b.x, acc.x);
    acc.x = fma(-a.y, b.y, acc.x);
    acc.y = fma(a.x, b.y, acc.y);
    acc.y = fma(a.y, b.x, acc.y);
}
template <typename R>
__device__ __forceinline__ void raxpyR(C2<R> &acc, R s, C2<R> v) {
    acc.x = fma(s, v.x, acc.x);
    acc.y = fma(s, v.y, acc.y);
}
template <typename R>
__device__ __forceinline__ double nrm2(C2<R> v) {
    return (double)v.x * (double)v.x + (double)v.y * (double)v.y;
}

// Stages k_0 .. k_9 (the step stages of vern7) live in registers, the rest in
// LDS: from LDS the sums over stages moved more bytes than the products, and
// with two rows a thread the registers spilled.
constexpr int kRegStages = 10;

// Per-workgroup LDS (dynamic): the vector an RHS product reads, the stage
// vectors k_10.. (the dense-output stages of vern7) and the FSAL slot, one
// entry per row, plus reduction scratch.
template <typename R>
struct McLds {
    C2<R> *x;      // [npad]
    C2<R> *xalt;   // [npad] the other input buffer, or null (one buffer)
    C2<R> *kd;     // [npad][kDenseSlots]: a row's stages, then its FSAL slot
    double *red;   // [2 * kFunGroup * threads / 64]
    double *probs; // [kMcMaxChan]
    double *bfs;   // [2][kMcStages] dense-output weights (two buffers, alternating)
    int bsel;      // the buffer the next interpolation writes
    double *rsum;  // [2][2 * threads / 64] block-sum partials (two buffers, alternating)
    int rsel;      // the buffer the next block sum writes
    const void *vt;  // packed operator: the table of values
    int npad;
};

// Slots of a row in kd: an odd number, so the 16-byte accesses of 16 lanes
// fall into different banks, with one address register for all of them.
constexpr int kDenseSlots = kMcStages - kRegStages + 1;

// Functionals summed per block reduction (one pair of barriers for each
// group) by the whole-solve kernel.
constexpr int kFunGroup = 4;

template <typename R>
inline size_t mc_lds_bytes(int threads) {
    return sizeof(C2<R>) * (size_t)threads * (1 + kDenseSlots) +
           sizeof(double) * ((2 * kFunGroup + 4) * (threads / 64) + kMcMaxChan + 2 * kMcStages) +
           64;
}

// Per-trajectory integrator state.  Vectors are per thread; scalars are
// uniform (every thread holds the same value).
template <typename R>
struct Traj {
    C2<R> k[kRegStages];
    C2<R> yprev, yfront, y;
    Uni t, t_prev, t_front, dt_safe, dt_int;
    int status;    // trajectory status (McStatus)
    int rk_state;  // last RK status (INTERPOLATED marks a prepared dense output)
    long long attempts;
    int ndense;  // dense-output preparations
};

template <typename R, int NT, int FM>
struct Ctx {
    const McArgs &A;
    McLds<R> &S;
    const double (*bi)[kMcOrder];  // the dense-output weights' polynomials, in LDS
    int wave0;          // the first row of this wave, uniform
    bool act;
    int rowc;  // the row clamped into [0, d) for the ELL loads
    const int *hcol;    // this system's H_eff ELL
    const void *hval;
    unsigned pk[FM == OP_ELL ? 1 : kMcPack / 2];  // this thread's codes, two a word
    C2<R> dg;                                     // and diagonal entry
    int dpos;  // complex64: the slot before which the diagonal is added
    int n_step, n_extra, is_fsal, is_adaptive, is_interp;  // of the tableau, uniform
    const __attribute__((address_space(4))) McTableau *tab;
    // Packed operators come with a tableau of vern7's shape (packed_args), so
    // the loops over stages have compile-time bounds: with run-time ones a
    // branch stood between any two stages of every sum, and the compiler
    // spilled the stage vectors.
    static constexpr bool kFix = FM != OP_ELL;
    __device__ __forceinline__ int rk_step() const { return kFix ? kPackStep : n_step; }
    __device__ __forceinline__ int rk_extra() const { return kFix ? kPackExtra : n_extra; }
    __device__ __forceinline__ bool fsal() const { return kFix ? false : is_fsal != 0; }
    __device__ __forceinline__ bool adaptive() const { return kFix ? true : is_adaptive != 0; }
    __device__ __forceinline__ bool interp() const { return kFix ? true : is_interp != 0; }
};

// This thread's row, formed anew at each use from the lane
// number: kept in a register across the trajectory loop it was spilled, and
// a scratch load (some 700 clocks) sat before every write to the LDS.
template <typename R, int NT, int FM>
__device__ __forceinline__ int row_of(const Ctx<R, NT, FM> &c) {
    int l;
    asm volatile("v_mbcnt_lo_u32_b32 %0, -1, 0\n\tv_mbcnt_hi_u32_b32 %0, -1, %0" : "=v"(l));
    return c.wave0 + l;
}

// Stage vector j; j is a compile-time constant after unrolling, so the
// register / LDS choice costs nothing.
template <typename R, int NT, int FM>
__device__ __forceinline__ C2<R> kget(Ctx<R, NT, FM> &c, Traj<R> &s, int j) {
    if (j < kRegStages) return s.k[j < kRegStages ? j : 0];
    return c.S.kd[row_of(c) * kDenseSlots + (j - kRegStages)];
}
template <typename R, int NT, int FM>
__device__ __forceinline__ void kset(Ctx<R, NT, FM> &c, Traj<R> &s, int j, const C2<R> &x) {
    if (j < kRegStages) {
        s.k[j < kRegStages ? j : 0] = x;
    } else {
        c.S.kd[row_of(c) * kDenseSlots + (j - kRegStages)] = x;
    }
}

// Block sums write their wave partials to one of two LDS buffers in turn,
// so one barrier per sum suffices: a buffer is written again only after the
// barrier of the sum in between, which every thread passes after its reads
// of it (the buffers serve nothing else).
template <typename R, int NT, int FM>
__device__ __forceinline__ double bsum(Ctx<R, NT, FM> &c, double v) {
    const int lane = threadIdx.x & (QA_WAVE - 1), wid = threadIdx.x / QA_WAVE;
    const int nw = blockDim.x / QA_WAVE;
    double *rb = c.S.rsum + 2 * nw * c.S.rsel;
    c.S.rsel ^= 1;
    v = wave_sum(v);
    if (lane == 0) rb[wid] = v;
    __syncthreads();
    double t = 0.0;
    for (int w = 0; w < nw; ++w) t += rb[w];
    return uni(t);
}

// Two block sums with one pair of barriers; each component is summed in
// the order bsum uses, so the results are bsum's bits.
template <typename R, int NT, int FM>
__device__ __forceinline__ double2 bsum2(Ctx<R, NT, FM> &c, double a, double b) {
    const int lane = threadIdx.x & (QA_WAVE - 1), wid = threadIdx.x / QA_WAVE;
    const int nw = blockDim.x / QA_WAVE;
    double *rb = c.S.rsum + 2 * nw * c.S.rsel;
    c.S.rsel ^= 1;
    a = wave_sum(a);
    b = wave_sum(b);
    if (lane == 0) {
        rb[wid] = a;
        rb[nw + wid] = b;
    }
    __syncthreads();
    double ta = 0.0, tb = 0.0;
    for (int w = 0; w < nw; ++w) {
        ta += rb[w];
        tb += rb[nw + w];
    }
    return make_double2(uni(ta), uni(tb));
}

// The input of a product (or of the functionals) into LDS, for every thread
// to gather from.  With two buffers the writes go to the one not read last,
// so only the barrier after them is needed: a thread still gathering from
// the other buffer has not reached that barrier, and every read of a
// buffer lies between the barrier after its writes and the barrier after
// the next input's, before the buffer is written again.
template <typename R, int NT, int FM>
__device__ __forceinline__ void stage_in(Ctx<R, NT, FM> &c, const C2<R> &x) {
    if (c.S.xalt) {  // uniform
        C2<R> *t = c.S.x;
        c.S.x = c.S.xalt;
        c.S.xalt = t;
    } else {
        __syncthreads();
    }
    c.S.x[row_of(c)] = x;
    __syncthreads();
}

// M ELL entries (u0 .. u0 + M - 1) of this thread's rows: all column and
// value loads first, then the LDS gathers and multiply-adds.
template <int M, typename R, int NT, int FM>
__device__ __forceinline__ void ell_chunk(Ctx<R, NT, FM> &c, int u0, C2<R> &acc) {
    const C2<R> *hv = (const C2<R> *)c.hval;
    const size_t d = (size_t)c.A.d;
    int cc[M];
    C2<R> vv[M];
#pragma unroll
    for (int w = 0; w < M; ++w) cc[w] = c.hcol[(size_t)(u0 + w) * d + c.rowc];
#pragma unroll
    for (int w = 0; w < M; ++w) vv[w] = hv[(size_t)(u0 + w) * d + c.rowc];
#pragma unroll
    for (int w = 0; w < M; ++w) cfmaR<R>(acc, vv[w], c.S.x[cc[w]]);
}

// M packed entries u0 .. u0 + M - 1 of this thread's rows: the gathers and
// the values (LDS, no other memory) together, then the multiply-adds.
template <int M, int U0, typename R, int NT, int FM>
__device__ __forceinline__ void packed_chunk(Ctx<R, NT, FM> &c, const C2<R> &x, C2<R> &acc) {
    const unsigned cm = (1u << c.A.pk_cbits) - 1u;
    C2<R> xv[M], vv[M];
#pragma unroll
    for (int w = 0; w < M; ++w) {
        const unsigned h = (c.pk[(U0 + w) / 2] >> (16 * ((U0 + w) & 1))) & 0xffffu;
        xv[w] = c.S.x[h & cm];
        if constexpr (FM == OP_PACKED_IM)
            vv[w].y = ((const R *)c.S.vt)[h >> c.A.pk_cbits];
        else
            vv[w] = ((const C2<R> *)c.S.vt)[h >> c.A.pk_cbits];
    }
#pragma unroll
    for (int w = 0; w < M; ++w) {
        if (sizeof(R) == 4 && c.dpos == U0 + w) cfmaR<R>(acc, c.dg, x);
        if constexpr (FM == OP_PACKED_IM) {
            acc.x = fma(-vv[w].y, xv[w].y, acc.x);
            acc.y = fma(vv[w].y, xv[w].x, acc.y);
        } else {
            cfmaR<R>(acc, vv[w], xv[w]);
        }
    }
}

template <int K, int U0, typename R, int NT, int FM>
__device__ __forceinline__ void packed_from(Ctx<R, NT, FM> &c, const C2<R> &x, C2<R> &acc) {
    if constexpr (U0 < kMcPack) {
        const int left = c.A.pk_width - U0;  // uniform, even
        if constexpr (K >= 8 && U0 + 8 <= kMcPack) {
            if (left >= 8) {
                packed_chunk<8, U0>(c, x, acc);
                packed_from<K, U0 + 8>(c, x, acc);
                return;
            }
        }
        if constexpr (U0 + 4 <= kMcPack) {
            if (left >= 4) {
                packed_chunk<4, U0>(c, x, acc);
                packed_from<4, U0 + 4>(c, x, acc);
                return;
            }
        }
        if (left == 2) packed_chunk<2, U0>(c, x, acc);
    }
}

// k = H_eff x for this thread's rows; x is staged in LDS first.  ELL: the
// width is a multiple of 4 (the host pads it), so entries go in chunks of 8
// (4 in 1024 threads with complex128 stages in registers, which leaves room
// for those) and at most one chunk of 4; no load is predicated.
// Packed: the entries in eights or fours and a last two, after the diagonal;
// complex64 adds the diagonal in its column's place, as the ELL form does: in
// another order the sums differ by 1e-7, and now and then a trajectory of
// 500 takes another jump (it costs 1.94 -> 2.37 ms for 500 of L = 8).
template <typename R, int NT, int FM>
__device__ __forceinline__ C2<R> rhs(Ctx<R, NT, FM> &c, const C2<R> &x) {
    stage_in(c, x);
    C2<R> acc = mk<R>(0, 0);
    constexpr int K = (NT > kMcThreads / 2 && sizeof(R) == 8) ? 4 : 8;
    if constexpr (FM == OP_ELL) {
        const int W = c.A.h_width;
        int u = 0;
        for (; u + K <= W; u += K) ell_chunk<K>(c, u, acc);
        if (K == 8 && u < W) ell_chunk<4>(c, u, acc);
    } else {
        // opaque here, or every slot's decoded addresses are kept in
        // registers for the whole kernel
#pragma unroll
        for (int w = 0; w < kMcPack / 2; ++w) asm volatile("" : "+v"(c.pk[w]));
        if (sizeof(R) == 8) cfmaR<R>(acc, c.dg, x);
        packed_from<K, 0>(c, x, acc);
        if (sizeof(R) == 4 && c.dpos >= c.A.pk_width) cfmaR<R>(acc, c.dg, x);
    }
    if constexpr (FM == OP_ELL) {
        if (!c.act) acc = mk<R>(0, 0);  // padding rows stay zero
    }
    return acc;
}

// (O x)_r for a CSR operator (c_ops / e_ops block); x already in LDS.
template <typename R, int NT, int FM>
__device__ __forceinline__ C2<R> op_rows(Ctx<R, NT, FM> &c, const int *rowptr, const int *col,
                                            const void *vals) {
    C2<R> acc = mk<R>(0, 0);
    const C2<R> *v = (const C2<R> *)vals;
    if (c.act)
        for (int p = rowptr[row_of(c)]; p < rowptr[row_of(c) + 1]; ++p)
            cfmaR<R>(acc, v[p], c.S.x[col[p]]);
    return acc;
}

template <typename R, int NT, int FM>
__device__ __forceinline__ double norm2(Ctx<R, NT, FM> &c, const C2<R> &x) {
    double s = 0.0;
    s += nrm2<R>(x);  // inactive rows hold zeros
    return bsum(c, s);
}

// The tableau's rows come through the constant address space: scalar loads
// into scalar registers (from LDS they took two vector registers each and
// spilled the stage vectors).
typedef const __attribute__((address_space(4))) McTableau McConstTab;
typedef const __attribute__((address_space(4))) double McCoef;

// The weight of a stage in dt sum_j coef_j k_j.  complex128 sums with the
// bare coefficient and multiplies by dt once; complex64 rounds the product
// for every stage (with rounded coefficients the sums of a row's weights are
// off by the same 1e-7 in every step, which adds up: the mean of 500
// trajectories moved by 1e-4).
__device__ __forceinline__ double weight(double coef, double, double) { return coef; }
__device__ __forceinline__ float weight(double coef, double dt, float) { return (float)(coef * dt); }

// yprev + dt sum_{j < n} coef[j] k_j (a zero coefficient adds nothing).
template <typename R, int NT, int FM>
__device__ __forceinline__ C2<R> combine(Ctx<R, NT, FM> &c, Traj<R> &s, McCoef *coef,
                                            int n, double dt) {
    constexpr bool once = sizeof(R) == 8;
    C2<R> o = once ? mk<R>(0, 0) : s.yprev;
#pragma unroll
    for (int j = 0; j < kMcStages; ++j) {
        if (j < n) {
            const C2<R> kj = kget(c, s, j);
            const R fj = weight(coef[j], dt, R());
            raxpyR<R>(o, fj, kj);
        }
    }
    if constexpr (!once) return o;
    C2<R> r = s.yprev;
    raxpyR<R>(r, (R)dt, o);
    return r;
}

// The stages I0 <= i < I1, of which i0 <= i < i1 are formed.
template <int I0, int I1, typename R, int NT, int FM>
__device__ __forceinline__ void stages(Ctx<R, NT, FM> &c, Traj<R> &s, int i0, int i1,
                                       double dt) {
#pragma unroll
    for (int i = I0; i < I1; ++i) {
        if (FM != OP_ELL || (i >= i0 && i < i1)) {
            const C2<R> x = combine(c, s, c.tab->a[i], i, dt);
            kset(c, s, i, rhs(c, x));
        }
    }
}

// The stages of _compute_step (explicit_rk.pyx:358-389) and those of the
// dense output (:399-410).
template <typename R, int NT, int FM>
__device__ __forceinline__ void step_stages(Ctx<R, NT, FM> &c, Traj<R> &s, double dt) {
    stages<0, FM != OP_ELL ? kPackStep : kMcStages>(c, s, c.fsal() ? 1 : 0, c.rk_step(), dt);
}
template <typename R, int NT, int FM>
__device__ __forceinline__ void dense_stages(Ctx<R, NT, FM> &c, Traj<R> &s) {
    stages<FM != OP_ELL ? kPackStep : 1, kMcStages>(c, s, c.rk_step(), c.rk_extra(), s.dt_int);
}

// The end of _compute_step: y_front and the error norm (:391-397), one pass
// over the stages for both sums.
template <typename R, int NT, int FM>
__device__ __forceinline__ double step_end(Ctx<R, NT, FM> &c, Traj<R> &s, double dt) {
    constexpr bool once = sizeof(R) == 8;
    McCoef *cb = c.tab->b, *ce = c.tab->e;
    C2<R> o = once ? mk<R>(0, 0) : s.yprev, ev = mk<R>(0, 0);
#pragma unroll
    for (int j = 0; j < kMcStages; ++j) {
        if (j < c.rk_step()) {
            const C2<R> kj = kget(c, s, j);
            const R fb = weight(cb[j], dt, R()), fe = weight(ce[j], dt, R());
            raxpyR<R>(o, fb, kj);
            raxpyR<R>(ev, fe, kj);
        }
    }
    s.yfront = once ? s.yprev : o;
    if constexpr (once) {
        raxpyR<R>(s.yfront, (R)dt, o);
    }
    s.t_front = s.t_prev + dt;
    if (!c.adaptive()) return 0.0;
    double qsum = 0.0;
    if (row_of(c) < c.A.d) {
        const double tol = c.A.atol + c.A.rtol * sqrt(nrm2<R>(s.yfront));
        const double ratio = (once ? dt : 1.0) * sqrt(nrm2<R>(ev)) / tol;
        qsum += ratio * ratio;
    }
    return sqrt(bsum(c, qsum) / (double)c.A.d);
}

// The weights b_i(tau) (explicit_rk.pyx:412-430) are formed by threads
// i < kMcStages, each with its row of the table loaded at once (a loop to
// the run-time order would wait on every load before the next step), and
// shared through LDS.  Two weight buffers alternate, so one barrier per
// interpolation suffices: a buffer is written again only after the barrier
// of the interpolation in between, which every thread passes after its
// reads of it.
template <typename R, int NT, int FM>
__device__ __forceinline__ C2<R> interpolate(Ctx<R, NT, FM> &c, Traj<R> &s, double t) {
    double *bw = c.S.bfs + kMcStages * c.S.bsel;
    c.S.bsel ^= 1;
    const int i = threadIdx.x;
    if (i < kMcStages) {
        const double tau = (t - s.t_prev) / s.dt_int;
        double bv[kMcOrder];
#pragma unroll
        for (int j = 0; j < kMcOrder; ++j) bv[j] = c.bi[i][j];
        double v = 0.0;
        if (i < c.rk_extra()) {
#pragma unroll
            for (int j = kMcOrder - 1; j >= 0; --j)
                if (j < c.tab->dorder) {  // Horner from j = dorder - 1 down
                    v += bv[j];
                    v *= tau;
                }
        }
        bw[i] = s.dt_int * v;
    }
    __syncthreads();
    C2<R> o = s.yprev;
#pragma unroll
    for (int j = 0; j < kMcStages; ++j) {
        if (j < c.rk_extra()) {
            const C2<R> kj = kget(c, s, j);
            const R fj = (R)bw[j];
            raxpyR<R>(o, fj, kj);
        }
    }
    return o;
}

template <typename R, int NT, int FM>
__device__ __forceinline__ double estimate_first_step(Ctx<R, NT, FM> &c, Traj<R> &s,
                                                      const C2<R> &y0) {
    McConstTab &T = *c.tab;
    if (!c.adaptive()) return 0.0;
    double norm = sqrt(norm2(c, y0));
    const double tol = c.A.atol + norm * c.A.rtol;
    // f(y0) and f(y0 + dt1/100 f(y0)) are local temporaries (the reference
    // borrows k[0] and k[1] for them; the next step overwrites both anyway)
    C2<R> f0;
    if (c.fsal()) {
        f0 = c.S.kd[row_of(c) * kDenseSlots + (kDenseSlots - 1)];
    } else {
        f0 = rhs(c, y0);
    }
    if (norm <= c.A.atol) norm = 1.0;
    double tmp = sqrt(norm2(c, f0));
    double factorial = 1.0;
    for (int i = 1; i <= T.order; ++i) factorial *= i;
    double dt1, dt2;
    if (tmp >= c.A.atol * 1e-6)
        dt1 = pow(tol * factorial * pow(norm, T.order), 1.0 / (T.order + 1)) / tmp;
    else
        dt1 = pow(tol * factorial, 1.0 / (T.order + 1)) * norm * 0.5;
    C2<R> yt = y0;
    raxpyR<R>(yt, (R)(dt1 / 100), f0);
    const C2<R> f1 = rhs(c, yt);
    tmp = sqrt(norm2(c, f1));
    if (tmp >= c.A.atol * 1e-6)
        dt2 = pow(tol * factorial * pow(norm, T.order), 1.0 / (T.order + 1)) / tmp;
    else
        dt2 = dt1;
    double dt = fmin(dt1, dt2);
    if (c.A.max_step != 0.0) dt = fmin(c.A.max_step, dt);
    if (c.A.min_step != 0.0) dt = fmax(c.A.min_step, dt);
    return dt;
}

// The stages in registers hold nothing from here on (no instruction): their
// registers are free until the next stages fill them.
template <typename R>
__device__ __forceinline__ void drop_stages(Traj<R> &s) {
#pragma unroll
    for (int j = 0; j < kRegStages; ++j)
        asm volatile("" : "=v"(s.k[j].x), "=v"(s.k[j].y));
}

// set_initial_value (explicit_rk.pyx:204-230)
template <typename R, int NT, int FM>
__device__ __forceinline__ void set_initial_value(Ctx<R, NT, FM> &c, Traj<R> &s,
                                                  const C2<R> &y0, double t0) {
    s.t = t0;
    s.t_prev = s.t;
    s.t_front = s.t;
    s.dt_int = 0.0;
    s.y = y0;
    s.yfront = y0;
    s.yprev = y0;
    s.rk_state = RK_NORMAL;
    drop_stages(s);
    if (c.fsal()) {
        const C2<R> kf = rhs(c, y0);
        c.S.kd[row_of(c) * kDenseSlots + (kDenseSlots - 1)] = kf;
    }
    s.dt_safe = c.A.first_step != 0.0 ? c.A.first_step : estimate_first_step(c, s, y0);
}

template <typename R, int NT, int FM>
__device__ __forceinline__ void recompute_safe_step(Ctx<R, NT, FM> &c, Traj<R> &s, double err,
                                                    double dt) {
    if (!c.adaptive()) return;
    double f;
    if (err == 0.0) {
        f = 10.0;
    } else {
        // square and cube roots for vern7's eighth root and tsit5's sixth: pow,
        // which every wave computes, took 3800 clocks of a step in one wave
        // and 13000 in 16 (600 tsit5 solves of 1024 rows 3.8 -> 3.25 ms)
        f = c.tab->order == 7   ? 0.9 / sqrt(sqrt(sqrt(err)))
            : c.tab->order == 5 ? 0.9 / sqrt(cbrt(err))
                                : 0.9 * pow(err, -1.0 / (c.tab->order + 1));
        f = fmin(10.0, f);
        f = fmax(0.2, f);
    }
    s.dt_safe = dt * f;
    if (c.A.max_step != 0.0) s.dt_safe = fmin(c.A.max_step, s.dt_safe);
    if (c.A.min_step != 0.0) s.dt_safe = fmax(c.A.min_step, s.dt_safe);
}

template <typename R, int NT, int FM>
__device__ __forceinline__ double get_timestep(Ctx<R, NT, FM> &c, Traj<R> &s, double t) {
    const double dt_needed = t - s.t_prev;
    if (!c.adaptive()) return dt_needed;
    if (c.interp()) return s.dt_safe;
    if (dt_needed <= s.dt_safe) return dt_needed;
    return dt_needed / (double)((long long)(dt_needed / s.dt_safe) + 1);
}

// integrate(t, step) (explicit_rk.pyx:278-331) with _step_in_err (:333-356):
// single: one accepted step at most (mcstep), else steps until t_front
// reaches t within one budget of nsteps attempts; then the state at t, by
// interpolation or y_front.
template <typename R, int NT, int FM>
__device__ __forceinline__ void advance(Ctx<R, NT, FM> &c, Traj<R> &s, double t,
                                        bool single) {
    if (t == s.t) return;
    if (t < s.t_prev) {
        s.status = MC_OUTSIDE_RANGE;
        return;
    }
    bool stepping = false, dense = false, interp = false;
    if (c.interp() && t < s.t_front) {
        dense = s.rk_state != RK_INTERPOLATED;
        interp = true;
    } else {
        s.rk_state = RK_NORMAL;
        if (single && s.t < s.t_front && t > s.t_front) t = s.t_front;
        stepping = s.t_front < t;
        if (!stepping) {
            s.rk_state = RK_AT_FRONT;
            s.t = s.t_front;
            s.y = s.yfront;
            return;
        }
        s.yprev = s.yfront;
        s.t_prev = s.t_front;
    }
    int nsteps_left = c.A.nsteps, n = 0;
    while (stepping) {
        drop_stages(s);
        const double dt = get_timestep(c, s, t);
        s.attempts++;
        if (c.fsal()) {
            C2<R> k0;
            k0 = c.S.kd[row_of(c) * kDenseSlots + (kDenseSlots - 1)];
            kset(c, s, 0, k0);
        }
        step_stages(c, s, dt);
        const double error = step_end(c, s, dt);
        s.dt_int = dt;
        recompute_safe_step(c, s, error, dt);
        n++;
        if (dt == c.A.min_step && error > 1.0)
            s.status = MC_DT_UNDERFLOW;
        else if (n > nsteps_left)
            s.status = MC_TOO_MUCH_WORK;
        if (error >= 1.0 && s.status >= 0) continue;
        if (c.fsal()) {
#pragma unroll
            for (int j = 0; j < kMcStages; ++j) {
                if (j == c.rk_step() - 1) {
                    const C2<R> kl = kget(c, s, j);
                    c.S.kd[row_of(c) * kDenseSlots + (kDenseSlots - 1)] = kl;
                }
            }
        }
        if (s.status < 0) return;
        nsteps_left -= n;
        n = 0;
        if (!single && s.t_front < t) {
            s.yprev = s.yfront;
            s.t_prev = s.t_front;
            continue;
        }
        stepping = false;
        interp = dense = s.t_front > t;
        if (!interp) {
            s.rk_state = RK_AT_FRONT;
            s.t = s.t_front;
            s.y = s.yfront;
        }
    }
    if (dense) {
        s.ndense++;
        dense_stages(c, s);
        s.rk_state = RK_INTERPOLATED;
    }
    if (interp) {
        s.y = interpolate(c, s, t);
        s.t = t;
    }
}

struct Rng {
    const double *d;
    int n, used;
};

template <typename D>
__device__ __forceinline__ bool draw(Rng &g, D &u) {
    if (g.used >= g.n) return false;
    u = g.d[g.used++];
    return true;
}

template <typename R, int NT, int FM>
__device__ __forceinline__ void write_expect(Ctx<R, NT, FM> &c, const C2<R> &y, double n2,
                                             int traj, int k) {
    stage_in(c, y);
    for (int e = 0; e < c.A.neops; ++e) {
        const int *rp = c.A.e_rowptr + (size_t)e * (c.A.d + 1);
        const C2<R> oy = op_rows(c, rp, c.A.e_col, c.A.e_vals);
        double re = 0.0, im = 0.0;  // conj(y_r) (O y)_r in FP64
        re += (double)y.x * oy.x + (double)y.y * oy.y;
        im += (double)y.x * oy.y - (double)y.y * oy.x;
        const double2 r = bsum2(c, re, im);
        if (threadIdx.x == 0)
            c.A.expect_out[((size_t)traj * c.A.ntimes + k) * c.A.neops + e] =
                make_double2(r.x / n2, r.y / n2);
    }
}

// p rounded up to 16 bytes as an offset from p itself, so the result keeps
// p's provenance: a pointer into the LDS stays one the compiler knows to be
// in the LDS (DS instructions, not FLAT ones, which wait on both the memory
// and the LDS counters).
template <typename T>
__device__ __forceinline__ unsigned char *align16(T *p) {
    unsigned char *b = (unsigned char *)p;
    return b + ((16 - ((uintptr_t)b & 15)) & 15);
}

// LDS carving, tableau copy and zeroing shared by the kernels of this file;
// returns the first free byte, aligned to 16.
template <typename R, int NT, int FM>
__device__ __forceinline__ unsigned char *kernel_prologue(const McArgs &A, unsigned char *lds,
                                                          double (*bi)[kMcOrder], McLds<R> &S) {
    const int nt = blockDim.x;
    const int npad = nt;
    unsigned char *p = lds;
    S.npad = npad;
    S.x = (C2<R> *)p;
    p += sizeof(C2<R>) * npad;
    S.kd = (C2<R> *)p;
    p += sizeof(C2<R>) * npad * kDenseSlots;
    S.red = (double *)p;
    p += sizeof(double) * 2 * kFunGroup * (nt / QA_WAVE);
    S.probs = (double *)p;
    p += sizeof(double) * kMcMaxChan;
    S.bfs = (double *)p;
    S.bsel = 0;
    p += sizeof(double) * 2 * kMcStages;
    S.rsum = (double *)p;
    S.rsel = 0;
    unsigned char *tail = align16(S.rsum + 4 * (nt / QA_WAVE));
    S.vt = tail;
    if constexpr (FM != OP_ELL) {  // the packed operator's values
        const int words = A.pk_ntab * (int)(sizeof(R) * (FM == OP_PACKED_IM ? 1 : 2) / 4);
        for (int i = threadIdx.x; i < words; i += nt) ((int *)tail)[i] = ((const int *)A.pk_tab)[i];
        tail = align16((int *)tail + words);
    }
    S.xalt = nullptr;
    if (A.x2) {  // the second input buffer, when the launcher reserved it
        S.xalt = (C2<R> *)tail;
        tail += sizeof(C2<R>) * (size_t)npad;
    }
    for (int i = threadIdx.x; i < kMcStages * kMcOrder; i += nt)
        (&bi[0][0])[i] = (&A.tab->bi[0][0])[i];
    for (int i = threadIdx.x; i < (1 + kDenseSlots) * npad; i += nt)
        S.x[i] = mk<R>(0, 0);  // x, the LDS stages and the FSAL slot start at zero
    __syncthreads();
    return tail;
}

// The rows of this thread, the operator it multiplies with, and the
// tableau's sizes as scalars.
template <typename R, int NT, int FM>
__device__ __forceinline__ void ctx_rows(Ctx<R, NT, FM> &c, const int *hcol, const void *hval) {
    c.hcol = hcol;
    c.hval = hval;
    c.wave0 = __builtin_amdgcn_readfirstlane((int)threadIdx.x & ~(QA_WAVE - 1));
    c.tab = (McConstTab *)c.A.tab;
    c.n_step = c.tab->rk_step;
    c.n_extra = c.tab->rk_extra;
    c.is_fsal = c.tab->fsal;
    c.is_adaptive = c.tab->adaptive;
    c.is_interp = c.tab->interpolate;
    const int row = row_of(c);
    c.act = row < c.A.d;
    c.rowc = c.act ? row : 0;
    if constexpr (FM != OP_ELL) {
        // padding rows: a zero diagonal and value 0 in every slot
        c.dpos = sizeof(R) == 4 && c.act ? c.A.pk_code[(size_t)c.A.pk_width * c.A.d + c.rowc] : 0;
        c.dg = c.act ? ((const C2<R> *)c.A.pk_diag)[c.rowc] : mk<R>(0, 0);
#pragma unroll
        for (int u = 0; u < kMcPack; ++u) {
            const unsigned h = u < c.A.pk_width && c.act
                                   ? c.A.pk_code[(size_t)u * c.A.d + c.rowc]
                                   : 0u;
            if (u & 1)
                c.pk[u / 2] |= h << 16;
            else
                c.pk[u / 2] = h;
        }
    }
}

// The functionals as the whole-solve kernel reads them: kind, CSR-style
// entry pointer, rows, columns and weights, in LDS when they were staged
// there, else in global memory.
struct FunView {
    const int *kind, *ptr, *row, *col;
    const double2 *w;
};

// Functionals of the state y (linear: sum w y[col]; quadratic:
// sum w conj(y[row]) y[col]), accumulated in FP64 in a fixed order, into
// out[0 .. nfun-1] (thread 0 writes).
template <typename R, int NT, int FM>
__device__ __forceinline__ void write_functionals(Ctx<R, NT, FM> &c, const C2<R> &y,
                                                  const FunView &fv, double2 *out) {
    stage_in(c, y);
    const int lane = threadIdx.x & (QA_WAVE - 1), wid = threadIdx.x / QA_WAVE;
    const int nw = blockDim.x / QA_WAVE;
    // kFunGroup functionals per block reduction: each wave's sums go to LDS
    // as they are formed (no array of them in registers), then one barrier,
    // and thread t < kFunGroup adds functional f0 + t over the waves in
    // order, which is bsum2's order, so the bits are bsum2's.  The barrier
    // after stage_in's writes (first group) or at the top of the loop (the
    // previous group's sums read) comes before a wave writes LDS sums.
    for (int f0 = 0; f0 < c.A.nfun; f0 += kFunGroup) {
        if (f0 > 0) __syncthreads();
#pragma unroll 1
        for (int g = 0; g < kFunGroup; ++g) {
            const int f = f0 + g;
            if (f >= c.A.nfun) break;  // uniform
            const int quad = fv.kind[f];
            const int e1 = fv.ptr[f + 1];
            double re = 0.0, im = 0.0;
            for (int e = fv.ptr[f] + threadIdx.x; e < e1; e += blockDim.x) {
                const C2<R> xc = c.S.x[fv.col[e]];
                const double2 w = fv.w[e];
                double vr = w.x * (double)xc.x - w.y * (double)xc.y;
                double vi = w.x * (double)xc.y + w.y * (double)xc.x;
                if (quad) {
                    const C2<R> xr = c.S.x[fv.row[e]];
                    const double lr = (double)xr.x, li = -(double)xr.y;
                    const double tr = lr * vr - li * vi;
                    vi = lr * vi + li * vr;
                    vr = tr;
                }
                re += vr;
                im += vi;
            }
            re = wave_sum(re);
            im = wave_sum(im);
            if (lane == 0) {
                c.S.red[(2 * g) * nw + wid] = re;
                c.S.red[(2 * g + 1) * nw + wid] = im;
            }
        }
        __syncthreads();
        if (threadIdx.x < kFunGroup && f0 + (int)threadIdx.x < c.A.nfun) {
            double ta = 0.0, tb = 0.0;
            for (int w = 0; w < nw; ++w) {
                ta += c.S.red[2 * threadIdx.x * nw + w];
                tb += c.S.red[(2 * threadIdx.x + 1) * nw + w];
            }
            out[f0 + threadIdx.x] = make_double2(ta, tb);
        }
    }
}

// One trajectory after another (grid-stride).  The loop holds one copy of
// each part: a start (of the trajectory, or after a jump), one advance (to
// the next output time, or to a guess of the collapse time), the search and
// the jump, the outputs.
template <typename R, int NT, int FM>
__global__ __launch_bounds__(NT) void mc_traj_kernel(McArgs A) {
    extern __shared__ __align__(16) unsigned char mc_dyn_lds[];
    __shared__ double bi[kMcStages][kMcOrder];
    McLds<R> S;
    kernel_prologue<R, NT, FM>(A, mc_dyn_lds, bi, S);
    Ctx<R, NT, FM> c{A, S, bi};
    ctx_rows(c, A.h_col, A.h_vals);

    for (int traj = blockIdx.x; traj < A.ntraj; traj += gridDim.x) {
        Traj<R> s;
        s.status = MC_OK;
        s.attempts = 0;
        s.ndense = 0;
#pragma unroll
        for (int j = 0; j < kRegStages; ++j) s.k[j] = mk<R>(0, 0);
        Rng g{A.draws + (size_t)traj * A.max_draws, A.max_draws, 0};
        int jumps = 0;
        Uni target;
        // s.y: the state of the next start
        const double2 p0 = c.act ? A.psi0[row_of(c)] : make_double2(0.0, 0.0);
        s.y = mk<R>((R)p0.x, (R)p0.y);
        if (!draw(g, target)) s.status = MC_DRAWS_EXHAUSTED;
        int k = 0;          // the next output
        int guard = 0;      // steps since the last output
        bool start = true, search = false;
        int tries = 0;
        Uni t_out = A.times[0];  // output k
        Uni t_start = t_out, t_old = t_start, norm_old = 1.0;
        Uni tp, tf, nold, nrm, t_guess;
        while (s.status == MC_OK) {
            // MCIntegrator.integrate (mcsolve.py:286-302); the state at t_old
            // is s.y outside of the search
            Uni n2 = -1.0;  // the norm of s.y once it is known
            bool found = false;
            if (start) {
                set_initial_value(c, s, s.y, t_start);
                start = false;
                t_old = s.t;
                norm_old = 1.0;  // after a jump (an output below sets it again)
            } else {
                if (!search && ++guard > 100000) {  // a search has its own bound
                    s.status = MC_NO_PROGRESS;
                    break;
                }
                advance(c, s, search ? (double)t_guess : (double)t_out, true);
                if (s.status < 0) break;
                n2 = norm2(c, s.y);
                if (search) {
                    if (fabs(target - n2) < A.norm_tol * target) {
                        found = true;
                    } else if (n2 < target) {
                        tf = t_guess;
                        nrm = n2;
                    } else {
                        tp = t_guess;
                        nold = n2;
                    }
                } else if (n2 <= target) {
                    search = true;
                    tries = 0;
                    tp = t_old;
                    tf = s.t;
                    nold = norm_old;
                    nrm = n2;
                    t_guess = tf;
                } else {
                    t_old = s.t;
                    norm_old = n2;
                }
            }
            if (search) {
                // _find_collapse_time (mcsolve.py:321-369)
                if (!found) {
                    if (tries >= A.norm_steps) {
                        s.status = MC_COLLAPSE_NOT_FOUND;
                        break;
                    }
                    tries++;
                    if (tf - tp < A.norm_t_tol) {
                        t_guess = tf;
                        found = true;
                    } else {
                        const double dtc = tf - tp;
                        double ratio = log(nold / target) / log(nold / nrm);
                        if (ratio < A.norm_min_step) ratio = A.norm_min_step;
                        if (ratio > 1.0 - A.norm_min_step) ratio = 1.0 - A.norm_min_step;
                        t_guess = tp + dtc * ratio;
                        if (t_guess - tp < A.norm_t_tol) t_guess = tp + A.norm_t_tol;
                        continue;
                    }
                }
                if (tries >= A.norm_steps) {
                    s.status = MC_COLLAPSE_NOT_FOUND;
                    break;
                }
                // _do_collapse (mcsolve.py:371-406); the state is s.y
                search = false;
                const C2<R> psi = s.y;
                stage_in(c, psi);
                int which = 0;
                if (A.nchan > 1) {
                    double tot = 0.0;
                    for (int ch = 0; ch < A.nchan; ++ch) {
                        const int *rp = A.c_rowptr + (size_t)ch * (A.d + 1);
                        const double pr = norm2(c, op_rows(c, rp, A.c_col, A.c_vals));
                        if (threadIdx.x == 0) S.probs[ch] = pr;
                        tot += pr;
                    }
                    __syncthreads();
                    Uni u;
                    if (!draw(g, u)) {
                        s.status = MC_DRAWS_EXHAUSTED;
                        break;
                    }
                    double tg = tot * u - S.probs[0];
                    while (tg > 0.0 && which < A.nchan - 1) {
                        which++;
                        tg -= S.probs[which];
                    }
                }
                const int *rp = A.c_rowptr + (size_t)which * (A.d + 1);
                C2<R> ynew = op_rows(c, rp, A.c_col, A.c_vals);
                const double nn = sqrt(norm2(c, ynew));
                if (nn < A.mc_corr_eps) {
                    const double np = sqrt(norm2(c, psi));
                    ynew.x = (R)(psi.x / np);
                    ynew.y = (R)(psi.y / np);
                } else {
                    ynew.x = (R)(ynew.x / nn);
                    ynew.y = (R)(ynew.y / nn);
                    if (threadIdx.x == 0 && jumps < A.max_jumps) {
                        A.col_times[(size_t)traj * A.max_jumps + jumps] = t_guess;
                        A.col_which[(size_t)traj * A.max_jumps + jumps] = which;
                    }
                    jumps++;
                    if (!draw(g, target)) {
                        s.status = MC_DRAWS_EXHAUSTED;
                        break;
                    }
                }
                s.y = ynew;
                start = true;
                t_start = t_guess;
                continue;
            }
            // the outputs reached (the first one at the start)
            while (k < A.ntimes && (k == 0 || !(t_old < t_out))) {
                if (n2 < 0.0) n2 = norm2(c, s.y);
                write_expect(c, s.y, n2, traj, k);
                norm_old = n2;
                guard = 0;
                if (++k < A.ntimes) t_out = A.times[k];
            }
            if (k >= A.ntimes) break;
        }
        if (threadIdx.x == 0) {
            A.info[(size_t)traj * 4 + 0] = s.status;
            A.info[(size_t)traj * 4 + 1] = jumps;
            A.info[(size_t)traj * 4 + 2] = g.used;
            A.info[(size_t)traj * 4 + 3] = (int)s.attempts;
        }
        __syncthreads();
    }
}

// Whole solves of small systems (sesolve / mesolve with n <= 1024): one
// workgroup integrates one system from t0 through every output time (the
// integrate(t) loop of the reference with interpolation), evaluating the
// functionals at each time, with no host round trip.  Systems are
// independent initial states (and optionally operators, h_stride apart),
// picked up grid-stride.  HL: the one operator of every system (h_stride
// 0) is copied into LDS after the other arrays once per workgroup, so the
// RHS products read it there instead of from L2 (the launcher picks this
// when it fits the configuration's LDS budget).
template <typename R, int NT, int FM, bool HL>
__global__ __launch_bounds__(NT) void rk_small_kernel(McArgs A) {
    extern __shared__ __align__(16) unsigned char mc_dyn_lds[];
    __shared__ double bi[kMcStages][kMcOrder];
    McLds<R> S;
    unsigned char *tail = kernel_prologue<R, NT, FM>(A, mc_dyn_lds, bi, S);
    Ctx<R, NT, FM> c{A, S, bi};
    const int *lcol = nullptr;
    const C2<R> *lval = nullptr;
    if constexpr (HL) {
        const int nent = A.h_width * A.d;
        C2<R> *v = (C2<R> *)tail;
        int *col = (int *)(tail + sizeof(C2<R>) * (size_t)nent);
        const C2<R> *gv = (const C2<R> *)A.h_vals;
        for (int i = threadIdx.x; i < nent; i += blockDim.x) {
            v[i] = gv[i];
            col[i] = A.h_col[i];
        }
        lcol = col;
        lval = v;
        tail = align16(col + nent);
    }
    // The functionals, then the output times, into the fun_lds bytes the
    // launcher reserved after the arrays above, each when it fits there
    // (the sizes are checked here, where the entry count is known).
    FunView fv{A.f_kind, A.f_ptr, A.f_row, A.f_col, A.f_w};
    const double *times = A.times;
    if (A.fun_lds > 0) {
        size_t used = 0;
        if (A.nfun > 0) {
            const int nfun = A.nfun, nnz = A.f_ptr[nfun];
            const size_t need = sizeof(double2) * (size_t)nnz +
                                sizeof(int) * (2 * (size_t)nnz + 2 * (size_t)nfun + 1);
            if (nnz >= 0 && need <= (size_t)A.fun_lds) {
                double2 *w = (double2 *)tail;
                int *ptr = (int *)(w + nnz);
                int *kind = ptr + nfun + 1;
                int *row = kind + nfun;
                int *col = row + nnz;
                for (int i = threadIdx.x; i < nnz; i += blockDim.x) {
                    w[i] = A.f_w[i];
                    row[i] = A.f_row[i];
                    col[i] = A.f_col[i];
                }
                for (int i = threadIdx.x; i <= nfun; i += blockDim.x) {
                    ptr[i] = A.f_ptr[i];
                    if (i < nfun) kind[i] = A.f_kind[i];
                }
                fv = FunView{kind, ptr, row, col, w};
                used = (size_t)(align16(col + nnz) - tail);
            }
        }
        if (used + sizeof(double) * (size_t)A.ntimes <= (size_t)A.fun_lds) {
            double *tl = (double *)(tail + used);
            for (int i = threadIdx.x; i < A.ntimes; i += blockDim.x) tl[i] = A.times[i];
            times = tl;
        }
    }
    __syncthreads();
    for (int sys = blockIdx.x; sys < A.ntraj; sys += gridDim.x) {
        const size_t hoff = (size_t)sys * (size_t)A.h_stride;
        if constexpr (HL)
            ctx_rows(c, lcol, (const void *)lval);
        else
            ctx_rows(c, A.h_col + hoff, (const void *)((const C2<R> *)A.h_vals + hoff));
        Traj<R> s;
        s.status = MC_OK;
        s.attempts = 0;
        s.ndense = 0;
#pragma unroll
        for (int j = 0; j < kRegStages; ++j) s.k[j] = mk<R>(0, 0);
        C2<R> y0;
        const double2 p0 =
            c.act ? A.psi0[(size_t)sys * A.d + row_of(c)] : make_double2(0.0, 0.0);
        y0 = mk<R>((R)p0.x, (R)p0.y);
        set_initial_value(c, s, y0, A.t0);
        int k = 0;
        for (; k < A.ntimes && s.status >= 0; ++k) {
            advance(c, s, times[k], false);
            if (s.status < 0) break;
            write_functionals(c, s.y, fv, A.fun_out + ((size_t)sys * A.ntimes + k) * A.nfun);
        }
        if (A.y_final) {
            if (c.act)
                A.y_final[(size_t)sys * A.d + row_of(c)] =
                    make_double2((double)s.y.x, (double)s.y.y);
        }
        if (threadIdx.x == 0) {
            A.info[(size_t)sys * 4 + 0] = s.status;
            A.info[(size_t)sys * 4 + 1] = k;  // outputs written
            A.info[(size_t)sys * 4 + 2] = s.ndense;
            A.info[(size_t)sys * 4 + 3] = (int)s.attempts;
        }
        __syncthreads();
    }
}

constexpr size_t kLdsBudget = 160 * 1024;  // LDS of one gfx950 CU
constexpr int kChipCUs = 256;

constexpr size_t kFunLdsMax = 16 * 1024;  // LDS for the functionals and times

// Static LDS of both kernels (the dense-output polynomials), rounded up to
// the 16-byte granule the dynamic part starts on.  Every budget below counts
// it: a workgroup's LDS is the static part plus the dynamic bytes.
constexpr size_t kLdsStatic = (sizeof(double) * kMcStages * kMcOrder + 15) & ~(size_t)15;

// The LDS plan of one launch: dynamic bytes, the operator in LDS (HL), and
// the bytes reserved for functionals and times.
struct McPlan {
    size_t lds;   // dynamic LDS bytes per workgroup
    bool hl;      // the shared ELL operator is staged in LDS
    int fun_lds;  // bytes for the functionals and times (0: none)
    bool x2;      // a second input buffer (one barrier per product instead of two)
    bool pk;      // the packed operator is used (its values in LDS)
};

inline size_t mc_lds_cap() { return kLdsBudget - kLdsStatic; }

template <typename R>
McPlan plan_mc(const McArgs &A, int threads, bool small) {
    McPlan P;
    P.lds = mc_lds_bytes<R>(threads);
    P.hl = false;
    P.fun_lds = 0;
    P.x2 = false;
    const size_t cap = mc_lds_cap();
    P.pk = false;
    if (A.pk_code) {
        const size_t tab = 16 + 2 * sizeof(R) * (size_t)A.pk_ntab;
        if (P.lds + tab <= cap) {
            P.lds += tab;
            P.pk = true;
        }
    }
    if (small && !P.pk && A.h_stride == 0 && A.h_width > 0) {
        // the shared operator in LDS when it fits, beside a second workgroup
        // where the systems are more than the CUs
        const size_t ell = (size_t)A.h_width * A.d * (sizeof(C2<R>) + sizeof(int));
        if (P.lds + ell <= (A.ntraj > kChipCUs ? kLdsBudget / 2 - kLdsStatic : cap)) {
            P.lds += ell;
            P.hl = true;
        }
    }
    {
        // the second input buffer (with 16 bytes for its alignment) when it
        // fits and keeps the number of workgroups an LDS-limited CU holds
        const size_t xb = 16 + sizeof(C2<R>) * (size_t)threads;
        if (P.lds + xb <= cap &&
            kLdsBudget / (P.lds + xb + kLdsStatic) == kLdsBudget / (P.lds + kLdsStatic)) {
            P.lds += xb;
            P.x2 = true;
        }
    }
    if (small) {
        if (A.nfun > 0 || A.ntimes > 0) {
            // room for the functionals and times, up to kFunLdsMax, that
            // keeps the number of workgroups an LDS-limited CU holds
            const size_t per_wg = P.lds + kLdsStatic;
            const size_t nwg = kLdsBudget / per_wg;  // >= 1: P.lds <= cap
            const size_t lim = std::min(kLdsBudget / nwg - kLdsStatic, cap);
            const size_t room = lim > P.lds ? std::min(lim - P.lds, kFunLdsMax + 16) : 0;
            if (room >= 16 + 256) {
                P.fun_lds = (int)((room - 16) & ~(size_t)15);
                P.lds += 16 + (size_t)P.fun_lds;
            }
        }
    }
    return P;
}

template <typename R, int NT, bool SMALL>
int launch_mc_cfg(const McArgs &A0, int threads, int blocks, hipStream_t s) {
    McArgs A = A0;
    const McPlan P = plan_mc<R>(A, threads, SMALL);
    if (P.lds > mc_lds_cap()) {
        qa::set_error("trajectory kernel: %zu B of dynamic LDS exceed the %zu B budget", P.lds,
                      mc_lds_cap());
        return QA_ERR_ARG;
    }
    A.fun_lds = P.fun_lds;
    A.x2 = P.x2 ? 1 : 0;
    const size_t lds = P.lds;
    const bool hl = P.hl;
    const int fm = !P.pk ? OP_ELL : A.pk_imag ? OP_PACKED_IM : OP_PACKED;
    const void *fn;
    if constexpr (!SMALL && NT < kMcThreads)
        fn = (const void *)mc_traj_kernel<R, NT, OP_ELL>;  // not for packed operators (launch_mc)
    else if constexpr (!SMALL)
        fn = fm == OP_PACKED_IM ? (const void *)mc_traj_kernel<R, NT, OP_PACKED_IM>
             : fm == OP_PACKED  ? (const void *)mc_traj_kernel<R, NT, OP_PACKED>
                                : (const void *)mc_traj_kernel<R, NT, OP_ELL>;
    else
        fn = fm == OP_PACKED_IM ? (const void *)rk_small_kernel<R, NT, OP_PACKED_IM, false>
             : fm == OP_PACKED  ? (const void *)rk_small_kernel<R, NT, OP_PACKED, false>
             : hl               ? (const void *)rk_small_kernel<R, NT, OP_ELL, true>
                                : (const void *)rk_small_kernel<R, NT, OP_ELL, false>;
    QA_HIP(hipFuncSetAttribute(fn, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds));
    void *args[] = {(void *)&A};
    QA_HIP(hipLaunchKernel(fn, dim3(blocks), dim3(threads), args, lds, s));
    QA_CHECK_LAUNCH();
    return QA_OK;
}

// Threads for d rows, one row each; false when d does not fit.
template <typename R>
bool shape_mc(int d, int *threads) {
    const int t = ((d + QA_WAVE - 1) / QA_WAVE) * QA_WAVE;
    if (t > kMcThreads) return false;
    *threads = t;
    return mc_lds_bytes<R>(t) <= mc_lds_cap();
}

// The kernels are compiled for up to 1024 threads (128 vector registers each,
// so 16 waves a CU), and some also for up to 512 (256 registers, 8 waves a CU,
// nothing spilled).  The whole-solve kernel takes that form where no CU gets a
// second workgroup (400 rows, one system: 2.96 ms against 3.23).
// Trajectories of a packed operator come in numbers: 512 of 512 rows 3.3 ms
// with 1024, 4.2 with 512, and 8192 of 256 rows 16 against 24 ms; 500 of them
// are equal.  Those of an ELL operator in complex128 load eight entries at a
// time with 256 registers and four with 128, and wide rows are bound by those
// loads: with 512 while the 8 waves a CU then holds are enough for every
// trajectory at once (ms with 512 / 1024, width = rows: 64 of 512 rows 41.9 /
// 50.9, 512 of 256 15.7 / 16.4, 256 of 128 4.2 / 4.9; beyond it 1500 of 128
// 11.0 / 9.1, and with 16 to 20 entries a row 500 of 300 8.9 / 6.1).
template <typename R, bool SMALL = false>
int launch_mc(const McArgs &A, int blocks, hipStream_t s) {
    int threads;
    if (!shape_mc<R>(A.d, &threads)) {
        qa::set_error("qa_mc_run: d = %d does not fit the trajectory kernel", A.d);
        return QA_ERR_ARG;
    }
    constexpr int kWaves = kMcThreads / 2 / QA_WAVE;  // a CU's with 256 registers
    if constexpr (SMALL || sizeof(R) == 8)
        if (threads <= kMcThreads / 2 &&
            (SMALL ? blocks <= kChipCUs
                   : !A.pk_code && blocks <= kChipCUs * (kWaves / (threads / QA_WAVE))))
            return launch_mc_cfg<R, kMcThreads / 2, SMALL>(A, threads, blocks, s);
    return launch_mc_cfg<R, kMcThreads, SMALL>(A, threads, blocks, s);
}

}  // namespace

extern "C" {

int qa_mc_tableau_size(void) { return (int)sizeof(McTableau); }

int qa_mc_lds_plan(int d, int h_width, int nfun, int ntimes, int fp32, int small,
                   long long *out) {
    QA_REQUIRE(out != nullptr, "qa_mc_lds_plan: null output");
    QA_REQUIRE(d >= 1 && h_width >= 0 && nfun >= 0 && ntimes >= 0, "qa_mc_lds_plan: bad size");
    McArgs A;
    memset(&A, 0, sizeof(A));
    A.d = d;
    A.h_width = h_width;
    A.nfun = nfun;
    A.ntimes = ntimes;
    int threads;
    const bool ok = fp32 ? shape_mc<float>(d, &threads) : shape_mc<double>(d, &threads);
    if (!ok) {
        qa::set_error("qa_mc_lds_plan: d = %d does not fit the trajectory kernel", d);
        return QA_ERR_ARG;
    }
    const McPlan P = fp32 ? plan_mc<float>(A, threads, small != 0)
                          : plan_mc<double>(A, threads, small != 0);
    out[0] = threads;
    out[1] = 1;  // rows per thread
    out[2] = kRegStages;
    out[3] = (long long)P.lds;
    out[4] = (long long)kLdsStatic;
    out[5] = P.hl ? 1 : 0;
    out[6] = P.fun_lds;
    out[7] = (long long)mc_lds_cap();
    return QA_OK;
}

// Pack a tableau (host arrays as for qa_rk_create) into the device layout
// the trajectory kernel reads; `out` is a host buffer of
// qa_mc_tableau_size() bytes to be copied to the device by the caller.
int qa_mc_pack_tableau(void *out, int order, int rk_step, int rk_extra, int dorder,
                       const double *a, const double *b, const double *c, const double *e,
                       const double *bi, int interpolate) {
    QA_REQUIRE(out && a && b && c, "qa_mc_pack_tableau: null argument");
    QA_REQUIRE(rk_step >= 1 && rk_step <= rk_extra && rk_extra <= kMcStages,
               "qa_mc_pack_tableau: 1 <= rk_step <= rk_extra <= %d", kMcStages);
    QA_REQUIRE(!bi || (dorder >= 1 && dorder <= kMcOrder), "qa_mc_pack_tableau: dense order");
    McTableau *T = (McTableau *)out;
    memset(T, 0, sizeof(McTableau));
    for (int i = 0; i < rk_extra; ++i) {
        for (int j = 0; j < rk_extra; ++j) T->a[i][j] = a[(size_t)i * rk_extra + j];
        T->c[i] = c[i];
        if (bi)
            for (int j = 0; j < dorder; ++j) T->bi[i][j] = bi[(size_t)i * dorder + j];
    }
    for (int i = 0; i < rk_step; ++i) {
        T->b[i] = b[i];
        T->e[i] = e ? e[i] : 0.0;
    }
    T->order = order;
    T->rk_step = rk_step;
    T->rk_extra = (bi && interpolate) ? rk_extra : rk_step;
    T->dorder = bi ? dorder : 0;
    T->interpolate = (bi && interpolate) ? 1 : 0;
    T->adaptive = e != nullptr;
    int fsal = 1;
    for (int j = 0; j < rk_step; ++j) {
        const double x = a[(size_t)(rk_step - 1) * rk_extra + j], y = b[j];
        if (fabs(x - y) > 1e-14 + 1e-5 * fabs(y)) fsal = 0;
    }
    T->fsal = fsal;
    return QA_OK;
}

static int packed_args(McArgs &A, const qa_packed_op *op) {
    A.pk_code = nullptr;
    A.pk_diag = A.pk_tab = nullptr;
    A.pk_width = A.pk_cbits = A.pk_ntab = A.pk_imag = 0;
    if (!op) return QA_OK;
    QA_REQUIRE(op->code && op->diag && op->table, "packed operator: null pointer");
    QA_REQUIRE(op->width >= 0 && op->width <= kMcPack && op->width % 2 == 0,
               "packed operator: width must be even, at most %d", kMcPack);
    QA_REQUIRE(op->cbits >= 1 && op->cbits <= 15 && A.d <= (1 << op->cbits),
               "packed operator: columns must fit cbits");
    QA_REQUIRE(op->ntab >= 1 && op->ntab <= kMcPackTab && op->ntab <= (1 << (16 - op->cbits)),
               "packed operator: 1 <= ntab <= %d", kMcPackTab);
    QA_REQUIRE(op->rk_step == kPackStep && op->rk_extra == kPackExtra,
               "packed operator: for tableaus of %d stages, %d with the dense output", kPackStep,
               kPackExtra);
    A.pk_code = (const unsigned short *)op->code;
    A.pk_diag = op->diag;
    A.pk_tab = op->table;
    A.pk_width = op->width;
    A.pk_cbits = op->cbits;
    A.pk_ntab = op->ntab;
    A.pk_imag = op->imag;
    return QA_OK;
}

int qa_mc_run(int d, int ntraj, int ntimes, const double *times_dev, const void *psi0_dev,
              int h_width, const int *h_col, const void *h_vals, int nchan,
              const int *c_rowptr, const int *c_col, const void *c_vals, int neops,
              const int *e_rowptr, const int *e_col, const void *e_vals,
              const void *tableau_dev, const double *draws_dev, int max_draws,
              double rtol, double atol, int nsteps, double first_step, double min_step,
              double max_step, int norm_steps, double norm_t_tol, double norm_tol,
              double norm_min_step, double mc_corr_eps, int fp32, void *expect_out_dev,
              double *col_times_dev, int *col_which_dev, int max_jumps, int *info_dev,
              int grid, void *stream) {
    return qa_mc_run_packed(nullptr, d, ntraj, ntimes, times_dev, psi0_dev, h_width, h_col, h_vals,
                            nchan, c_rowptr, c_col, c_vals, neops, e_rowptr, e_col, e_vals,
                            tableau_dev, draws_dev, max_draws, rtol, atol, nsteps, first_step,
                            min_step, max_step, norm_steps, norm_t_tol, norm_tol, norm_min_step,
                            mc_corr_eps, fp32, expect_out_dev, col_times_dev, col_which_dev,
                            max_jumps, info_dev, grid, stream);
}

int qa_mc_run_packed(const qa_packed_op *packed, int d, int ntraj, int ntimes,
              const double *times_dev, const void *psi0_dev, int h_width, const int *h_col, const void *h_vals, int nchan,
              const int *c_rowptr, const int *c_col, const void *c_vals, int neops,
              const int *e_rowptr, const int *e_col, const void *e_vals,
              const void *tableau_dev, const double *draws_dev, int max_draws,
              double rtol, double atol, int nsteps, double first_step, double min_step,
              double max_step, int norm_steps, double norm_t_tol, double norm_tol,
              double norm_min_step, double mc_corr_eps, int fp32, void *expect_out_dev,
              double *col_times_dev, int *col_which_dev, int max_jumps, int *info_dev,
              int grid, void *stream) {
    QA_REQUIRE(d >= 1 && d <= kMcThreads, "qa_mc_run: 1 <= d <= %d (rows held per thread)",
               kMcThreads);
    QA_REQUIRE(ntraj >= 0 && ntimes >= 1, "qa_mc_run: need ntimes >= 1");
    QA_REQUIRE(nchan >= 1 && nchan <= kMcMaxChan, "qa_mc_run: 1 <= nchan <= %d", kMcMaxChan);
    QA_REQUIRE(neops >= 0 && neops <= kMcMaxEops, "qa_mc_run: neops <= %d", kMcMaxEops);
    QA_REQUIRE(max_draws >= 1 && max_jumps >= 1, "qa_mc_run: need max_draws, max_jumps >= 1");
    QA_REQUIRE(norm_steps >= 1 && nsteps >= 0, "qa_mc_run: bad step limits");
    QA_REQUIRE(h_width >= 0 && h_width % 4 == 0 && h_width <= d + 3,
               "qa_mc_run: h_width must be a multiple of 4, at most d + 3");
    QA_REQUIRE(times_dev && psi0_dev && tableau_dev && draws_dev && info_dev &&
                   expect_out_dev && col_times_dev && col_which_dev && c_rowptr &&
                   (h_width == 0 || (h_col && h_vals)),
               "qa_mc_run: null pointer");
    if (ntraj == 0) return QA_OK;
    McArgs A;
    memset(&A, 0, sizeof(A));
    A.d = d;
    QA_CHECK(packed_args(A, packed));
    A.ntraj = ntraj;
    A.ntimes = ntimes;
    A.nchan = nchan;
    A.neops = neops;
    A.max_draws = max_draws;
    A.max_jumps = max_jumps;
    A.traj_offset = 0;
    A.h_width = h_width;
    A.h_col = h_col;
    A.h_vals = h_vals;
    A.c_rowptr = c_rowptr;
    A.c_col = c_col;
    A.c_vals = c_vals;
    A.e_rowptr = e_rowptr;
    A.e_col = e_col;
    A.e_vals = e_vals;
    A.tab = (const McTableau *)tableau_dev;
    A.times = times_dev;
    A.psi0 = (const double2 *)psi0_dev;
    A.draws = draws_dev;
    A.rtol = rtol;
    A.atol = atol;
    A.first_step = first_step;
    A.min_step = min_step != 0.0 ? min_step : 1e-15;
    A.max_step = max_step;
    A.nsteps = nsteps;
    A.norm_steps = norm_steps;
    A.norm_t_tol = norm_t_tol;
    A.norm_tol = norm_tol;
    A.norm_min_step = norm_min_step;
    A.mc_corr_eps = mc_corr_eps;
    A.expect_out = (double2 *)expect_out_dev;
    A.col_times = col_times_dev;
    A.col_which = col_which_dev;
    A.info = info_dev;
    if (grid <= 0) grid = ntraj;
    if (grid > ntraj) grid = ntraj;
    hipStream_t s = (hipStream_t)stream;
    return fp32 ? launch_mc<float>(A, grid, s) : launch_mc<double>(A, grid, s);
}


int qa_rk_small_run(int n, int nsys, double t0, int ntimes, const double *times_dev,
                    const void *y0_dev, int h_width, const int *h_col, const void *h_vals,
                    long long h_stride, int nfun, const int *fkind, const int *fptr,
                    const int *frows, const int *fcols, const void *fw, const void *tableau_dev,
                    double rtol, double atol, int nsteps, double first_step, double min_step,
                    double max_step, int fp32, void *fun_out_dev, void *y_final_dev,
                    int *info_dev, int grid, void *stream) {
    return qa_rk_small_run_packed(nullptr, n, nsys, t0, ntimes, times_dev, y0_dev, h_width, h_col,
                                  h_vals, h_stride, nfun, fkind, fptr, frows, fcols, fw,
                                  tableau_dev, rtol, atol, nsteps, first_step, min_step, max_step,
                                  fp32, fun_out_dev, y_final_dev, info_dev, grid, stream);
}

int qa_rk_small_run_packed(const qa_packed_op *packed, int n, int nsys, double t0, int ntimes,
                    const double *times_dev, const void *y0_dev, int h_width, const int *h_col, const void *h_vals,
                    long long h_stride, int nfun, const int *fkind, const int *fptr,
                    const int *frows, const int *fcols, const void *fw, const void *tableau_dev,
                    double rtol, double atol, int nsteps, double first_step, double min_step,
                    double max_step, int fp32, void *fun_out_dev, void *y_final_dev,
                    int *info_dev, int grid, void *stream) {
    QA_REQUIRE(n >= 1 && n <= kMcThreads, "qa_rk_small_run: 1 <= n <= %d", kMcThreads);
    QA_REQUIRE(nsys >= 0 && ntimes >= 0 && nfun >= 0, "qa_rk_small_run: negative size");
    QA_REQUIRE(h_width >= 0 && h_width % 4 == 0 && h_width <= n + 3 && h_stride >= 0,
               "qa_rk_small_run: h_width must be a multiple of 4, at most n + 3");
    QA_REQUIRE(y0_dev && tableau_dev && info_dev && (ntimes == 0 || times_dev) &&
                   (h_width == 0 || (h_col && h_vals)) &&
                   (nfun == 0 || (fkind && fptr && frows && fcols && fw && fun_out_dev)),
               "qa_rk_small_run: null pointer");
    QA_REQUIRE(nsteps >= 0, "qa_rk_small_run: nsteps >= 0");
    if (nsys == 0) return QA_OK;
    McArgs A;
    memset(&A, 0, sizeof(A));
    A.d = n;
    QA_REQUIRE(!packed || h_stride == 0, "qa_rk_small_run_packed: one operator for every system");
    QA_CHECK(packed_args(A, packed));
    A.ntraj = nsys;
    A.ntimes = ntimes;
    A.h_width = h_width;
    A.h_col = h_col;
    A.h_vals = h_vals;
    A.h_stride = h_stride;
    A.tab = (const McTableau *)tableau_dev;
    A.times = times_dev;
    A.t0 = t0;
    A.psi0 = (const double2 *)y0_dev;
    A.rtol = rtol;
    A.atol = atol;
    A.first_step = first_step;
    A.min_step = min_step;
    A.max_step = max_step;
    A.nsteps = nsteps;
    A.nfun = nfun;
    A.f_kind = fkind;
    A.f_ptr = fptr;
    A.f_row = frows;
    A.f_col = fcols;
    A.f_w = (const double2 *)fw;
    A.fun_out = (double2 *)fun_out_dev;
    A.y_final = (double2 *)y_final_dev;
    A.info = info_dev;
    if (grid <= 0 || grid > nsys) grid = nsys;
    hipStream_t s = (hipStream_t)stream;
    return fp32 ? launch_mc<float, true>(A, grid, s) : launch_mc<double, true>(A, grid, s);
}

}  // extern "C"
