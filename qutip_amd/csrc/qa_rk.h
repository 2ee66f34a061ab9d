// Pieces shared by the translation units of the fused Runge-Kutta engine: the
// control block and its device-side transitions (step control, output
// routing), and the banded right-hand side.
#pragma once
#include <hip/hip_runtime.h>

#include "qa_common.h"

namespace qa {

enum Phase { PH_IDLE = 0, PH_STEP = 1, PH_DENSE = 2, PH_OUTPUT = 3, PH_DONE = 4, PH_ERROR = 5 };
// integrator status codes: qutip/solver/integrator/explicit_rk.pxd:5-12
enum Status {
    ST_AT_FRONT = 2,
    ST_INTERPOLATED = 1,
    ST_NORMAL = 0,
    ST_TOO_MUCH_WORK = -1,
    ST_DT_UNDERFLOW = -2,
    ST_OUTSIDE_RANGE = -3,
    ST_NOT_INITIATED = -4
};

constexpr int kMaxStages = 16;
constexpr int kMaxPending = 4;     // output times handled per output launch
constexpr int kOutChunk = 16;      // functional entries per output workgroup
constexpr int kOutThreads = 64;    // one wavefront per output workgroup
constexpr int kStepBlocks = 256;   // threads per stage workgroup
constexpr int kMaxChunk = 64;      // loop iterations per host chunk
constexpr int kGraphBatch = 8;     // loop iterations per batch graph
constexpr int kBatchAfter = 128;   // iterations an engine runs before it batches

enum Resident { RES_NONE = 0, RES_RUNNING = 1, RES_DONE = 2 };

struct RKCtl {
    double t_prev, t_front, dt_safe, dt_int, dt_try, err, t_last;
    double rtol, atol, min_step, max_step;
    double *times;  // mutable copy of the requested output times
    double2 *fun_out;
    double2 *states_out;
    int ntimes, phase, cur, out_idx, nsteps_left, nsteps_call, dense_ready, status;
    int order, max_numsteps, interpolate, adaptive, single_step, nfun;
    // resident loop (rk_resident.hip): RES_RUNNING from the launch until the
    // kernel has written its state back (RES_DONE)
    int resident, pad;
    long long n_attempts, n_accepted, n_dense, n_outputs;
};

// ---- step control (executed by one thread) ---------------------------------
__device__ inline double get_timestep(const RKCtl *c, double t) {
    // explicit_rk.pyx:439-449
    const double dt_needed = t - c->t_prev;
    if (!c->adaptive) return dt_needed;
    if (c->interpolate) return c->dt_safe;
    if (dt_needed <= c->dt_safe) return dt_needed;
    return dt_needed / (double)((long long)(dt_needed / c->dt_safe) + 1);
}

__device__ inline void recompute_safe_step(RKCtl *c, double err, double dt) {
    // explicit_rk.pyx:451-467
    if (!c->adaptive) return;
    double factor;
    if (err == 0.0) {
        factor = 10.0;
    } else {
        factor = 0.9 * pow(err, -1.0 / (c->order + 1));
        factor = fmin(10.0, factor);
        factor = fmax(0.2, factor);
    }
    c->dt_safe = dt * factor;
    if (c->max_step != 0.0) c->dt_safe = fmin(c->max_step, c->dt_safe);
    if (c->min_step != 0.0) c->dt_safe = fmax(c->min_step, c->dt_safe);
}

// y_prev <- y_front, t_prev <- t_front, then a fresh _step_in_err
// (explicit_rk.pyx:312-316).
__device__ inline void start_step(RKCtl *c, double target) {
    c->cur ^= 1;
    c->t_prev = c->t_front;
    c->dense_ready = 0;
    c->nsteps_call = 0;
    c->dt_try = get_timestep(c, target);
    c->phase = PH_STEP;
}

// Decide what the next output time needs (explicit_rk.pyx:288-331).
__device__ inline void route(RKCtl *c) {
    if (c->out_idx >= c->ntimes) {
        c->phase = PH_DONE;
        return;
    }
    double target = c->times[c->out_idx];
    if (target < c->t_prev) {
        c->status = ST_OUTSIDE_RANGE;
        c->phase = PH_ERROR;
        return;
    }
    if (target < c->t_front) {
        if (!c->interpolate) {
            c->status = ST_OUTSIDE_RANGE;
            c->phase = PH_ERROR;
            return;
        }
        c->phase = c->dense_ready ? PH_OUTPUT : PH_DENSE;
        return;
    }
    if (c->single_step && c->t_last < c->t_front && target > c->t_front) {
        // integrate(t, step=True) clamps to the front (explicit_rk.pyx:309-311)
        c->times[c->out_idx] = c->t_front;
        target = c->t_front;
    }
    if (target == c->t_front) {
        c->phase = PH_OUTPUT;
        return;
    }
    c->nsteps_left = c->max_numsteps;
    c->status = ST_NORMAL;
    start_step(c, target);
}

// After one attempt of _compute_step (explicit_rk.pyx:333-356).
__device__ inline void after_attempt(RKCtl *c, double err) {
    const double dt = c->dt_try;
    c->err = err;
    c->n_attempts++;
    c->dt_int = dt;
    recompute_safe_step(c, err, dt);
    if (dt == c->min_step && err > 1.0) {
        c->status = ST_DT_UNDERFLOW;
        c->phase = PH_ERROR;
        return;
    }
    c->nsteps_call++;
    if (c->nsteps_call > c->nsteps_left) {
        c->status = ST_TOO_MUCH_WORK;
        c->phase = PH_ERROR;
        return;
    }
    double target = c->times[c->out_idx];
    if (err >= 1.0) {
        c->dt_try = get_timestep(c, target);
        c->phase = PH_STEP;
        return;
    }
    c->t_front = c->t_prev + dt;
    c->nsteps_left -= c->nsteps_call;
    c->nsteps_call = 0;
    c->n_accepted++;
    c->dense_ready = 0;
    if (c->single_step && c->t_front < target) {
        // integrate(t, step=True) stops after one step at the front
        c->times[c->out_idx] = c->t_front;
        target = c->t_front;
    }
    if (c->t_front < target) {
        start_step(c, target);
    } else if (c->t_front > target) {
        if (c->interpolate) {
            c->phase = PH_DENSE;
        } else {
            c->status = ST_OUTSIDE_RANGE;
            c->phase = PH_ERROR;
        }
    } else {
        c->phase = PH_OUTPUT;
    }
}

// Completion of an output (thread 0 of one workgroup): the time and status
// of the last output, the counters, and the next phase (route).
__device__ inline void finish_outputs(RKCtl *c, int ph, int nq, const int *front) {
    if (nq == 0) {
        // a non-finite step left no output time inside [t_prev, t_front]
        c->status = ST_OUTSIDE_RANGE;
        c->phase = PH_ERROR;
        return;
    }
    if (ph == PH_DENSE) {
        c->dense_ready = 1;
        c->n_dense++;
    }
    c->t_last = c->times[c->out_idx + nq - 1];
    c->status = front[nq - 1] ? ST_AT_FRONT : ST_INTERPOLATED;
    c->n_outputs += nq;
    c->out_idx += nq;
    route(c);
}

// One entry of a functional: w y, or conj(l) w y for a quadratic one (l the
// row's value).  Explicit fused multiply-adds, so every kernel that sums
// functionals forms the same bits.
__device__ __forceinline__ double2 fun_term(double2 w, double2 y, int quad, double2 l) {
    const double2 v = make_double2(fma(-w.y, y.y, w.x * y.x), fma(w.y, y.x, w.x * y.y));
    if (!quad) return v;
    return make_double2(fma(l.y, v.y, l.x * v.x), fma(-l.y, v.x, l.x * v.y));
}

constexpr int kMaxDenseOrder = 8;

// Operator forms of rk_stage_kernel.
enum StageForm { FORM_PLAIN = 0, FORM_CODED = 1, FORM_CODED_UNIFORM = 2 };

// ---- banded (DIA) Lindblad right-hand side ----------------------------------
// The matrix-form RHS k = Hm X + X Hp + sum_c C_c X Cd_c (Hm = -i H_nh,
// Hp = i H_nh^dag, Cd_c = C_c^dag) for banded operators, as LindbladMatrix-
// Form computes it with Dia products (lindblad_matrix_form.pyx:105-203 over
// matmul_dia_dense_dense, matmul.pyx:429-507), in FP64.  Every product is a
// list of terms acc += A[i, i+o] x[i+o, j-p] B[j-p, j]: a diagonal of Hm
// (B = 1), of Hp (A = 1), or a pair of diagonals of C_c and Cd_c.  Values
// are rows of `val` (row d: the diagonal's entries by row index; the last
// row all ones).  One thread per element (i, j) of the column-major N x N
// state, i fastest: the x and A loads of a wavefront are coalesced and its
// B load is one value.  Terms go in chunks of at most eight, each a body of
// exactly its length, so a chunk's loads are issued together; out-of-range
// neighbours are clamped and their terms dropped by a select.
constexpr int kDiaMaxTerms = 96;

struct DiaTerm {
    int o, p, a, b;
};

struct DiaOp {
    int N, nterms;
    const double2 *val;  // [rows][N]
    DiaTerm t[kDiaMaxTerms];
};

template <int M>
__device__ __forceinline__ void dia_terms(const DiaOp &D, const double2 *__restrict__ x, int i,
                                          int j, int t0, double2 &acc) {
    const int N = D.N;
    double2 av[M], bv[M], xv[M];
    bool ok[M];
#pragma unroll
    for (int u = 0; u < M; ++u) {
        const DiaTerm T = D.t[t0 + u];
        const int ii = i + T.o, jj = j - T.p;
        ok[u] = (unsigned)ii < (unsigned)N && (unsigned)jj < (unsigned)N;
        const int iic = ok[u] ? ii : i, jjc = ok[u] ? jj : j;
        av[u] = D.val[(int64_t)T.a * N + i];
        bv[u] = D.val[(int64_t)T.b * N + jjc];
        xv[u] = x[(int64_t)jjc * N + iic];
    }
#pragma unroll
    for (int u = 0; u < M; ++u) {
        const double2 t = cmul(cmul(av[u], xv[u]), bv[u]);
        if (ok[u]) acc = cadd(acc, t);
    }
}

__device__ __forceinline__ double2 dia_rhs_at(const DiaOp &D, const double2 *__restrict__ x,
                                              int i, int j) {
    double2 acc = make_double2(0.0, 0.0);
    int t = 0;
    for (; t + 8 <= D.nterms; t += 8) dia_terms<8>(D, x, i, j, t, acc);
    switch (D.nterms - t) {
        case 7: dia_terms<7>(D, x, i, j, t, acc); break;
        case 6: dia_terms<6>(D, x, i, j, t, acc); break;
        case 5: dia_terms<5>(D, x, i, j, t, acc); break;
        case 4: dia_terms<4>(D, x, i, j, t, acc); break;
        case 3: dia_terms<3>(D, x, i, j, t, acc); break;
        case 2: dia_terms<2>(D, x, i, j, t, acc); break;
        case 1: dia_terms<1>(D, x, i, j, t, acc); break;
        default: break;
    }
    return acc;
}

}  // namespace qa
