// The resident step loop of the fused Runge-Kutta engine.
//
// The launched loop (rk.hip) runs an attempt as a dozen kernels; each pays
// its launch, the control block, its operator slice and the earlier stages'
// k again (3.6 to 5.4 us a stage, whatever the size).  Here the workgroups
// stay on the chip for many attempts: a lane keeps its operator entries in
// registers (up to kResKept; longer rows are read again every stage), its
// k_0 .. k_15 in LDS and y_prev / y_front in registers, so a stage writes
// x_{i+1}, crosses one barrier and gathers it; the terms of the next combine
// that are known are summed while the barrier fills.  The product of y_front
// is both the next step's k_0 and the first dense-output stage, and a
// rejected attempt keeps its k_0, so an attempt with an output crosses 15
// barriers where the launched loop has 18 kernels.
//
// Measured, us per right-hand side of a whole run (outputs and step control
// included), launched -> resident: 2116 rows of 7 entries 4.6 -> 2.2, 4096
// of 13-18 5.6 -> 2.6, 16384 of 15 6.7 -> 3.2, 65536 of 13-24 6.5 -> 4.4,
// 131072 of 18 16.6 -> 6.6, the banded matrix form of 256 x 256 5.9 -> 4.5,
// a driven chain of 4096 rows (coefficients once an attempt instead of in
// every stage launch) 16.5 -> 4.3.
//
// Bound by that barrier and the two trips around it (measured with 19
// gathers a row: barrier alone / store, barrier and gather):
//   up to 32 workgroups on one XCD     0.58 us / 1.4 - 1.7 us
//   256 workgroups on every XCD        2.5 us  / 3.8 us
//     (every workgroup polling all flags 3.5 / 6.1, one counter 4.0 / 5.8)
//   the same stage as launches         -       / 2.6 us (8192 rows), 3.9 us (65536)
// hence one XCD wherever the rows fit its 32 compute units, and above that a
// barrier in two levels.
//
// Visibility.  Stage inputs go round a ring of kResRing slots, so a load
// never meets an older copy of its line in L1 or L2 except after the ring
// wraps, where one buffer_inv drops them.  On one XCD the slots are written
// and read through its L2 by plain accesses (the L1 writes through; the wait
// for the stores comes before the arrival).  Across XCDs the stores are
// write-through (sc1), so no L2 write-back is needed.  Flags and error
// partials are read past the L1 with sc1 loads.
//
// Every workgroup runs the step control itself, from the same partials in
// the same order, on its own copy of the control block.  Arithmetic and
// summation orders are those of the launched kernels: the same bits.
//
// Every wait is bounded.  A workgroup whose wait runs out (its peers did not
// become resident) leaves without writing the state back; the state, control
// block and y as of the launch then stand and the host goes on with the
// launched loop.  Workgroup 0 decides through the commit word, so either all
// of them write back or none does.
#include <string.h>

#include <algorithm>

#include "qa_api_internal.h"
#include "rk_resident.h"

namespace qa {
namespace {

constexpr int kResThreads = 512;      // at most; two waves per SIMD
constexpr int kResChunk = 12;         // entries of a longer plain row in flight (registers)
constexpr int kResTimes = 256;        // output times kept in LDS

// control words, a line (32 words) or more apart
constexpr int kSyElected = 0;    // XCD + 1 of the first workgroup to arrive
constexpr int kSyTicket = 32;    // workgroups of the elected XCD
constexpr int kSyCommit = 64;    // 1: write back, 2: given up
constexpr int kSyRegister = 96;  // arrivals of the registration
constexpr int kSyCount = 128;    // [16] workgroups per XCD
constexpr int kSyFlags = 192;    // [32] one XCD: arrivals
constexpr int kSyGlobal = 256;   // [16][32] for each XCD: the XCDs that have arrived
constexpr int kSyLocal = 768;    // [16][32] per XCD: arrivals of its workgroups
static_assert(kSyLocal + 512 <= kResSyncWords, "control words");

typedef unsigned u32x4 __attribute__((ext_vector_type(4)));

__device__ __forceinline__ unsigned xcc_id() {
    return __builtin_amdgcn_s_getreg((3 << 11) | 20) & 15u;  // HW_REG_XCC_ID[3:0]
}
// past the L1 (and, across XCDs, coherent): agent-scope relaxed accesses
__device__ __forceinline__ unsigned ld_agent(const unsigned *p) {
    return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ __forceinline__ void st_agent(unsigned *p, unsigned v) {
    __hip_atomic_store(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ __forceinline__ void wait_stores() { asm volatile("s_waitcnt vmcnt(0)" ::: "memory"); }
__device__ __forceinline__ void drop_caches() {
    asm volatile("buffer_inv sc1\n\ts_waitcnt vmcnt(0)" ::: "memory");
}

struct ResShared {
    RKCtl c;
    double f[kMaxStages + 1][kMaxStages];  // dt tc
    double fs[kMaxStages + 1];             // dt cs
    double fe[kMaxStages], fes;            // dt te, dt ce
    double c_stage[kMaxStages];
    double w[kMaxPending][kMaxStages];     // output weights
    double red[kResThreads / QA_WAVE], red2[4];
    double2 cf[kMaxStages + 2][kMaxCoef];  // coefficients at the stage times
    double times[kResTimes];
    double bi[kMaxStages][kMaxDenseOrder];
    CoefSet td;
    alignas(16) int koff[kMaxStages + 1][kMaxStages];  // byte offsets of the lists' k
    int nt[kMaxStages + 1];
    int front[kMaxPending], okq[kMaxPending];
    int wg, xcc, lidx, nloc, xccs, ok, commit, polls;
};

// Dynamic LDS beside it.
constexpr size_t kResLdsMax = 160 * 1024 - (sizeof(ResShared) + 255) / 256 * 256;
static_assert(sizeof(double2) * kMaxStages * kResThreads <= kResLdsMax,
              "16 stages of one row a thread fit");

struct Where {  // this workgroup's place in the barrier
    int wg, nwg, multi, xcc, lidx, nloc;
    unsigned xccs;  // XCDs that take part
    unsigned *sync;
    const int *polls;  // of a wait, at least one
};

// Lanes 0 .. of wave 0 wait until every word (lane < cnt, at p + stride lane)
// has reached g.
__device__ __forceinline__ bool poll_words(const unsigned *p, bool mine, unsigned g,
                                           const int *polls) {
    for (int k = 1;; ++k) {
        const bool ok = !mine || (int)(ld_agent(p) - g) >= 0;
        if (__all(ok)) return true;
        if (k >= *polls) return false;  // in LDS: read while the next poll would wait anyway
    }
}

// Wave 0, lane 0: this workgroup has arrived at barrier g.
__device__ __forceinline__ void arrive(const Where &W, unsigned g) {
    unsigned *p = W.multi ? W.sync + kSyLocal + 32 * W.xcc + W.lidx : W.sync + kSyFlags + W.wg;
    __hip_atomic_store(p, g, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
}

// Wave 0: true when every workgroup has arrived at barrier g.  Across XCDs
// the first workgroup of each collects its XCD's arrivals in that L2 and
// tells every XCD; all workgroups wait for their XCD's line of those words.
__device__ __forceinline__ bool wait_all(const Where &W, unsigned g) {
    const int lane = threadIdx.x;
    unsigned *y = W.sync;
    if (!W.multi) return poll_words(y + kSyFlags + (lane & 31), lane < W.nwg, g, W.polls);
    const bool part = lane < 16 && ((W.xccs >> (lane & 15)) & 1u);
    if (W.lidx == 0) {
        if (!poll_words(y + kSyLocal + 32 * W.xcc + (lane & 31), lane < W.nloc, g, W.polls))
            return false;
        if (part) st_agent(y + kSyGlobal + 32 * lane + W.xcc, g);
    }
    return poll_words(y + kSyGlobal + 32 * W.xcc + (lane & 15), part, g, W.polls);
}

// x[r] = v, seen by every workgroup after the next barrier.
__device__ __forceinline__ void publish(double2 *x, int r, double2 v, int multi) {
    if (multi) {
        const __amdgpu_buffer_rsrc_t rs =
            __builtin_amdgcn_make_buffer_rsrc(x, 0, 0x7fffffff, 0x00027000);
        u32x4 w;
        memcpy(&w, &v, 16);
        __builtin_amdgcn_raw_buffer_store_b128(w, rs, r * 16, 0, 16);  // sc1
    } else {
        x[r] = v;
    }
}

// o += sum_t f[t] k over NT terms of a list, the loads issued together (the
// terms and order of epi_terms of the launched kernels; four at a time, the
// sum is hidden in the barrier).  Kr: this row of
// the k in LDS; the list holds byte offsets from it.  Every list but the
// last step stage's holds non-zero coefficients only; there a factor 0 (a
// stage that only enters the error, or only y_front) leaves the sum alone.
template <int NT>
__device__ __forceinline__ void list_terms(const ResShared &S, const char *Kr, int i, int t0,
                                           bool fin, double2 &o, double2 &er) {
    double2 kv[NT];
#pragma unroll
    for (int t = 0; t < NT; ++t) kv[t] = *(const double2 *)(Kr + S.koff[i][t0 + t]);
    if (!fin) {
#pragma unroll
        for (int t = 0; t < NT; ++t) raxpy(o, S.f[i][t0 + t], kv[t]);
    } else {
#pragma unroll
        for (int t = 0; t < NT; ++t) {
            const double f = S.f[i][t0 + t], fe = S.fe[t0 + t];
            double2 p = o, q = er;
            raxpy(p, f, kv[t]);
            raxpy(q, fe, kv[t]);
            o.x = f != 0.0 ? p.x : o.x;
            o.y = f != 0.0 ? p.y : o.y;
            er.x = fe != 0.0 ? q.x : er.x;
            er.y = fe != 0.0 ? q.y : er.y;
        }
    }
}

__device__ __forceinline__ void list_sum(const ResShared &S, const char *Kr, int i, bool fin,
                                         double2 &o, double2 &er) {
    int t = 0;
    const int n = S.nt[i];
    for (; t + 4 <= n; t += 4) list_terms<4>(S, Kr, i, t, fin, o, er);
    switch (n - t) {
        case 3: list_terms<3>(S, Kr, i, t, fin, o, er); break;
        case 2: list_terms<2>(S, Kr, i, t, fin, o, er); break;
        case 1: list_terms<1>(S, Kr, i, t, fin, o, er); break;
        default: break;
    }
}

// A lane's entries kept in registers: values and byte offsets into x.  The terms and order of sell_row_dot: even entries into a0, odd
// ones into a1.
template <int M>
__device__ __forceinline__ void kept_terms(const unsigned (&off)[kResKept],
                                           const double2 (&val)[kResKept], const char *x,
                                           double2 &a0, double2 &a1) {
    double2 xv[M];
#pragma unroll
    for (int u = 0; u < M; ++u) xv[u] = *(const double2 *)(x + off[u]);
#pragma unroll
    for (int u = 0; u < M; ++u) cfma((u & 1) ? a1 : a0, val[u], xv[u]);
}

__device__ __forceinline__ double2 kept_dot(const unsigned (&off)[kResKept],
                                            const double2 (&val)[kResKept], int steps,
                                            const char *x) {
    double2 a0 = make_double2(0.0, 0.0), a1 = make_double2(0.0, 0.0);
    switch (steps) {
#define QA_RES_CASE(m) \
        case m: kept_terms<m>(off, val, x, a0, a1); break;
        QA_RES_CASE(1) QA_RES_CASE(2) QA_RES_CASE(3) QA_RES_CASE(4) QA_RES_CASE(5)
        QA_RES_CASE(6) QA_RES_CASE(7) QA_RES_CASE(8) QA_RES_CASE(9) QA_RES_CASE(10)
        QA_RES_CASE(11) QA_RES_CASE(12) QA_RES_CASE(13) QA_RES_CASE(14) QA_RES_CASE(15)
        QA_RES_CASE(16)
#undef QA_RES_CASE
        default: break;
    }
    static_assert(kResKept == 16, "the cases above");
    return cadd(a0, a1);
}

// Row i of cf: the coefficients at stage time i of a step from tp by dt; row
// kMaxStages: at tpub.  Out of line: the stack machine is large, and a call
// an attempt costs less than its registers in the loop.
__device__ __noinline__ void res_coefs(ResShared *S, int nk, double tp, double dt, double tpub) {
    const int nc = S->td.ncoef;
    for (int q = threadIdx.x; q < nc * (kMaxStages + 1); q += blockDim.x) {
        const int e = q % nc, i = q / nc;
        if (i < nk || i == kMaxStages)
            S->cf[i][e] = coef_eval(S->td, e, i == kMaxStages ? tpub : tp + S->c_stage[i] * dt);
    }
}

template <typename V, int FORM>
__global__ __launch_bounds__(kResThreads) void rk_resident_kernel(ResArgs P, DiaOp D) {
    constexpr bool KEPT = FORM == RES_KEPT;
    constexpr bool TD = FORM == RES_CODED_TD;  // the value table is scaled every stage
    constexpr bool CODED = FORM == RES_CODED || TD;  // tables in LDS
    const int L = FORM == RES_DIA ? 1 : P.lanes;
    extern __shared__ __align__(16) unsigned char res_lds[];
    __shared__ ResShared S;
    const int tid = threadIdx.x, nt = blockDim.x;

    // ---- the workgroups that take part -------------------------------------
    if (tid == 0) {
        const unsigned x = xcc_id();
        int wg = blockIdx.x;
        S.lidx = 0;
        if (!P.multi) {
            const unsigned old = atomicCAS(P.sync + kSyElected, 0u, x + 1u);
            wg = -1;
            if (old == 0u || old == x + 1u) {
                const unsigned tk = atomicAdd(P.sync + kSyTicket, 1u);
                wg = tk < (unsigned)P.nwg ? (int)tk : -1;
            }
        } else {
            S.lidx = (int)atomicAdd(P.sync + kSyCount + x, 1u);
        }
        S.polls = P.polls;
        S.wg = wg;
        S.xcc = (int)x;
    }
    __syncthreads();
    if (S.wg < 0 || P.polls < 1) return;  // another XCD's, or one too many: uniform
    Where W;
    W.wg = S.wg;
    W.nwg = P.nwg;
    W.multi = P.multi;
    W.xcc = S.xcc;
    W.lidx = S.lidx;
    W.nloc = 0;
    W.xccs = 0;
    W.sync = P.sync;
    W.polls = &S.polls;
    if (P.multi) {
        // every workgroup has registered: the XCDs' counts are final
        if (tid == 0) {
            wait_stores();
            atomicAdd(P.sync + kSyRegister, 1u);
            int ok = 0;
            for (int k = 0; k < P.polls && !ok; ++k)
                ok = ld_agent(P.sync + kSyRegister) >= (unsigned)P.nwg;
            unsigned m = 0;
            for (int i = 0; i < 16; ++i) {
                const unsigned c = ld_agent(P.sync + kSyCount + i);
                if (c) m |= 1u << i;
                if (i == W.xcc) S.nloc = (int)c;
                if (c > 32u) ok = 0;  // more than the local flags hold
            }
            S.xccs = (int)m;
            S.ok = ok;
        }
        __syncthreads();
        if (!S.ok) return;  // uniform; nobody can pass the first barrier without this one
        W.nloc = S.nloc;
        W.xccs = (unsigned)S.xccs;
    }

    // ---- rows, operator, tables, control block --------------------------------
    const int rows = nt / L;
    double2 *K = (double2 *)res_lds;
    double2 *vt = K + (size_t)P.nk * rows;
    const int nv = CODED ? 1 << P.vbits : 0, no = CODED ? 1 << (16 - P.vbits) : 0;
    double2 *vts = TD ? vt + nv : vt;  // the table the products read
    int *ot = (int *)(vts + nv);
    const int64_t t = (int64_t)W.wg * nt + tid;
    const int slice = (int)(t / QA_WAVE), lane = (int)(t % QA_WAVE);
    const int r = slice * (QA_WAVE / L) + lane / L;
    const int lr = tid / L;
    const bool live = FORM == RES_DIA ? r < P.n : slice < P.nslices;
    const bool owner = live && lane % L == 0;
    const int di = FORM == RES_DIA ? r % D.N : 0, dj = FORM == RES_DIA ? r / D.N : 0;
    int sp0 = 0, steps = 0;
    unsigned koffs[KEPT ? kResKept : 1];
    double2 kval[KEPT ? kResKept : 1];
    if constexpr (FORM != RES_DIA) {
        const int sl = live ? slice : P.nslices - 1;
        sp0 = P.slice_ptr[sl];
        steps = (P.slice_ptr[sl + 1] - sp0) / QA_WAVE;
    }
    if constexpr (KEPT) {
        // decode this lane's entries (coded: four to a word)
        const bool coded = P.code != nullptr;
        const int ne = steps;  // words or entries a lane
        if (coded) steps *= 4;
#pragma unroll
        for (int u = 0; u < kResKept; ++u) {
            double2 v = make_double2(0.0, 0.0);
            int c = min(r, P.n - 1);
            if (coded && u / 4 < ne) {
                const uint2 w = P.code[sp0 + lane + (u / 4) * QA_WAVE];
                const unsigned h = (((u & 2) ? w.y : w.x) >> (16 * (u & 1))) & 0xffffu;
                v = P.vtab[h & ((1u << P.vbits) - 1u)];
                c = min(max(r + P.otab[h >> P.vbits], 0), P.n - 1);
            } else if (!coded && u < ne) {
                const int at = sp0 + lane + u * QA_WAVE;
                c = P.col[at];
                v = P.fp32 ? ld((const float2 *)P.vals, at) : ((const double2 *)P.vals)[at];
            }
            koffs[u] = (unsigned)c * 16u;
            kval[u] = v;
        }
    }
    if constexpr (CODED) {
        for (int i = tid; i < nv; i += nt) vt[i] = P.vtab[i];
        for (int i = tid; i < no; i += nt) ot[i] = P.otab[i];
    }
    {
        const int *src = (const int *)P.ctl;
        for (int i = tid; i < (int)(sizeof(RKCtl) / 4); i += nt) ((int *)&S.c)[i] = src[i];
        for (int q = tid; q < (kMaxStages + 1) * kMaxStages; q += nt) {
            const int i = q / kMaxStages, u = q % kMaxStages;
            S.koff[i][u] = P.tab->tj[i][u] * rows * (int)sizeof(double2);
            if (u == 0) S.nt[i] = P.tab->nt[i];
            if (i == 0) S.c_stage[u] = P.tab->c[u];
            if (q < kMaxStages * kMaxDenseOrder) S.bi[q / kMaxDenseOrder][q % kMaxDenseOrder] =
                P.tab->bi[q / kMaxDenseOrder][q % kMaxDenseOrder];
        }
    }
    if (TD && tid == 0) S.td = P.td;
    __syncthreads();
    double *const times_mem = S.c.times;
    double *const times = S.c.ntimes <= kResTimes ? S.times : times_mem;
    if (S.c.ntimes <= kResTimes)
        for (int i = tid; i < S.c.ntimes; i += nt) S.times[i] = times_mem[i];
    int cur = S.c.cur;
    const int phase0 = S.c.phase;
    const CodeSplit cs = {CODED ? (1u << P.vbits) - 1u : 0u, P.vbits};
    double2 yprev = make_double2(0.0, 0.0), yfront = yprev;
    if (owner) {
        yprev = (cur ? P.y1 : P.y0)[r];
        yfront = (cur ? P.y0 : P.y1)[r];
        if (phase0 != PH_STEP)
            for (int j = 0; j < P.nk; ++j) K[j * rows + lr] = P.K[(int64_t)j * P.npad + r];
    }
    __syncthreads();
    if (tid == 0) S.c.times = times;

    unsigned g = 0;           // barriers passed
    int slot = kResRing - 1;  // the slot last published
    const double2 *x = P.ring;

    // One barrier: x (published by every row before) is readable after it;
    // cfrow: the coefficient row the next product's table is scaled by.
    // next >= 0: the stage whose product comes next; the terms of its combine
    // that are known by now are summed while the barrier fills.
    char *const Kr = (char *)(K + lr);
    double2 on = make_double2(0.0, 0.0), ern = on;
    auto barrier = [&](int cfrow, int next) {
        ++g;
        wait_stores();
        __syncthreads();
        bool ok = true;
        if (tid == 0) arrive(W, g);
        if (next >= 0) {
            on = yprev;
            ern = make_double2(0.0, 0.0);
            if (owner) list_sum(S, Kr, next, next == P.rk_step - 1, on, ern);
        }
        if (tid < QA_WAVE) {
            ok = wait_all(W, g);
            if (slot == 0) drop_caches();  // the ring has wrapped
        } else if constexpr (TD) {
            const int v1 = S.td.vstart[S.td.ncoef];
            for (int i = tid - QA_WAVE; i < nv; i += nt - QA_WAVE) {
                double2 v = vt[i];
                if (i >= S.td.vstart[0] && i < v1) {
                    int e = 0;
                    while (e + 1 < S.td.ncoef && i >= S.td.vstart[e + 1]) ++e;
                    v = cmul_fixed(v, S.cf[cfrow][e]);
                }
                vts[i] = v;
            }
        }
        if (tid == 0) S.ok = ok;
        __syncthreads();
        asm volatile("" ::: "memory");
        return S.ok != 0;
    };
    // The combine factors of a step of dt; TD: the coefficients at its stage
    // times from tp, row kMaxStages at tpub (the time of the vector that is
    // published at the step's end).
    auto factors = [&](double tp, double dt, double tpub) {
        for (int q = tid; q < (kMaxStages + 1) * kMaxStages; q += nt) {
            const int i = q / kMaxStages, u = q % kMaxStages;
            S.f[i][u] = dt * P.tab->tc[i][u];
            if (u == 0) S.fs[i] = dt * P.tab->cs[i];
            if (i == 0) S.fe[u] = dt * P.tab->te[u];
            if (q == 0) S.fes = dt * P.tab->ce;
        }
        if constexpr (TD) res_coefs(&S, P.nk, tp, dt, tpub);
        __syncthreads();
    };

    // The loop publishes a vector o, crosses the barrier, takes the product
    // of the vector and decides the next one.  i: the stage whose product is
    // wanted, or
    enum { AT_END = -1, AT_DECIDE = -2, AT_FIRST_DENSE = kMaxStages };
    // AT_END: the product of a step's end (or of the vector at hand at the
    // launch) is kf, the next step's k_0 and the first dense stage;
    // AT_FIRST_DENSE: o is that stage's own input.
    factors(S.c.t_prev, S.c.dt_int, phase0 == PH_STEP ? S.c.t_prev : S.c.t_front);
    int i = AT_END, cfrow = kMaxStages, attempts = 0, nq = 0;
    bool alive, control = false, k0_new = true;
    double2 o = phase0 == PH_STEP ? yprev : yfront;
    double2 kf = make_double2(0.0, 0.0), acc;
    for (;;) {
        slot = slot + 1 == kResRing ? 0 : slot + 1;
        x = P.ring + (int64_t)slot * P.npad;
        if (owner) publish((double2 *)x, r, o, P.multi);
        const int next =
            control || i == AT_END ? -1 : i == AT_FIRST_DENSE ? P.rk_step : i + 1;
        alive = barrier(cfrow, next);
        if (!alive) break;
        double v = 0.0;  // the error partials, requested with the gathers
        if (control && tid < kStepBlocks)
            for (int k = tid; k < P.nblk; k += kStepBlocks)
                v += __hip_atomic_load(P.parts + (attempts & 1) * P.nblk + k, __ATOMIC_RELAXED,
                                       __HIP_MEMORY_SCOPE_AGENT);
        acc = make_double2(0.0, 0.0);
        if (live) {
            if constexpr (FORM == RES_DIA)
                acc = dia_rhs_at(D, x, di, dj);
            else if constexpr (KEPT)
                acc = kept_dot(koffs, kval, steps, (const char *)x);
            else if constexpr (CODED)
                acc = sell_coded_row_dot<1>(P.code, vts, ot, cs, x, sp0, steps, lane, r, P.n - 1);
            else
                acc = sell_row_dot<1, V, kResChunk>(P.col, (const V *)P.vals, x, sp0, steps, lane);
        }
        for (int d = L / 2; d > 0; d >>= 1) {
            acc.x += __shfl_xor(acc.x, d, QA_WAVE);
            acc.y += __shfl_xor(acc.y, d, QA_WAVE);
        }
        if (control) {
            if (tid < kStepBlocks) {
                v = wave_sum(v);
                if (lane == 0) S.red2[tid / QA_WAVE] = v;
            }
            const long long acc0 = S.c.n_accepted;
            __syncthreads();
            if (tid == 0) {
                double tot = 0.0;
                for (int w = 0; w < kStepBlocks / QA_WAVE; ++w) tot += S.red2[w];
                after_attempt(&S.c, S.c.adaptive ? sqrt(tot / (double)P.n) : 0.0);
            }
            __syncthreads();
            k0_new = S.c.n_accepted != acc0;
            control = false;
            if (k0_new) kf = acc;  // else k_0 stands: the same y_prev
            i = AT_DECIDE;
        } else if (i == AT_END) {
            kf = acc;
            i = AT_DECIDE;
        } else {
            i = next;
        }
        bool stop = false, summed = next >= 0;
        for (;;) {
            if (i >= 0) {  // acc = k_i
                if (owner) K[i * rows + lr] = acc;
                if (i + 1 < P.nk || i == P.rk_step - 1) {
                    const bool fin = i == P.rk_step - 1;
                    if (!summed) {
                        on = yprev;
                        ern = make_double2(0.0, 0.0);
                        if (owner) list_sum(S, Kr, i, fin, on, ern);
                    }
                    double2 er = ern;
                    o = on;
                    const double fb = S.fs[i];
                    if (fb != 0.0) raxpy(o, fb, acc);
                    cfrow = i + 1;
                    if (fin) {
                        if (S.fes != 0.0) raxpy(er, S.fes, acc);
                        yfront = o;
                        double part = 0.0;
                        if (owner && r < P.n) {
                            const double q =
                                sqrt(cabs2(er)) / (S.c.atol + S.c.rtol * sqrt(cabs2(o)));
                            part = q * q;
                        }
                        part = wave_sum(part);
                        if (lane == 0) S.red[tid / QA_WAVE] = part;
                        __syncthreads();
                        const int blk = (int)(t / kStepBlocks);
                        if (tid % kStepBlocks == 0 && blk < P.nblk) {
                            double s = 0.0;
                            for (int w = 0; w < kStepBlocks / QA_WAVE; ++w)
                                s += S.red[tid / QA_WAVE + w];
                            __hip_atomic_store(P.parts + (attempts & 1) * P.nblk + blk, s,
                                               __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                        }
                        cfrow = kMaxStages;
                        control = true;
                    }
                    break;
                }
            } else {
                if (S.c.cur != cur) {  // a step begins where the last one ended
                    cur = S.c.cur;
                    yprev = yfront;
                    k0_new = true;
                }
                const int phase = S.c.phase;
                if (phase == PH_STEP && attempts < P.max_attempts) {
                    ++attempts;
                    factors(S.c.t_prev, S.c.dt_try, S.c.t_prev + S.c.dt_try);
                    i = 0;
                    summed = false;
                    acc = kf;
                    if (!k0_new && owner) acc = K[lr];
                    continue;
                }
                if (phase != PH_DENSE && phase != PH_OUTPUT) {
                    stop = true;
                    break;
                }
                // pending outputs and their weights (pending_outputs of rk.hip)
                if (tid < kMaxPending * kMaxStages) {
                    const int q = tid / kMaxStages, j = tid % kMaxStages;
                    const int idx = S.c.out_idx + q;
                    const bool in_range = idx < S.c.ntimes;
                    const double tq = in_range ? times[idx] : 0.0;
                    const bool ok = in_range && tq <= S.c.t_front;
                    double w = 0.0;
                    if (ok && tq != S.c.t_front && P.has_bi && j < P.nk) {
                        const double tau = (tq - S.c.t_prev) / S.c.dt_int;
#pragma unroll
                        for (int m = kMaxDenseOrder - 1; m >= 0; --m)
                            if (m < P.dorder) {
                                w += S.bi[j][m];
                                w *= tau;
                            }
                        w *= S.c.dt_int;
                    }
                    S.w[q][j] = w;
                    if (j == 0) {
                        S.okq[q] = ok;
                        S.front[q] = ok && tq == S.c.t_front;
                    }
                }
                __syncthreads();
                nq = 0;
                while (nq < kMaxPending && S.okq[nq]) ++nq;
                if (S.c.out_idx - P.out_base + nq > P.out_cap) {  // the host takes these first
                    stop = true;
                    break;
                }
                if (phase == PH_DENSE && P.dense) {
                    if (P.first_front) {
                        i = P.rk_step;
                        summed = false;
                        acc = kf;
                        continue;
                    }
                    o = yprev;
                    double2 er;
                    if (owner) list_sum(S, Kr, kMaxStages, false, o, er);
                    i = AT_FIRST_DENSE;
                    cfrow = P.rk_step;
                    break;
                }
            }
            // the stages of this step are complete: its outputs
            if (owner) {
                const int o0 = S.c.out_idx;
                const int nd = P.need ? P.need[r] : -1;
#pragma unroll 1
                for (int q = 0; q < nq; ++q) {
                    const int idx = o0 + q;
                    const bool last = idx == S.c.ntimes - 1;
                    if (nd < 0 && !last && !S.c.states_out) continue;
                    double2 y = yfront;
                    if (!S.front[q]) {
                        y = yprev;
#pragma unroll 4
                        for (int j = 0; j < kMaxStages; ++j) {
                            const double wj = j < P.nk ? S.w[q][j] : 0.0;
                            const double2 kk = K[min(j, P.nk - 1) * rows + lr];
                            raxpy(y, wj, make_double2(wj != 0.0 ? kk.x : 0.0, wj != 0.0 ? kk.y : 0.0));
                        }
                    }
                    if (nd >= 0) P.yout[(int64_t)(idx - P.out_base) * P.nneed + nd] = y;
                    if (S.c.states_out) S.c.states_out[(int64_t)idx * P.npad + r] = y;
                    if (last) P.y_last[r] = y;
                }
            }
            __syncthreads();
            if (tid == 0) finish_outputs(&S.c, S.c.phase, nq, S.front);
            __syncthreads();
            i = AT_DECIDE;
        }
        if (stop) break;
    }

    // ---- write back, all or none -----------------------------------------------
    if (alive) alive = barrier(kMaxStages, -1);
    if (tid == 0) {
        unsigned d;
        d = 0;
        if (alive && W.wg != 0)
            for (int k = 0; k / 4 < P.polls && d == 0; ++k) d = ld_agent(P.sync + kSyCommit);
        if (d == 0) {
            // workgroup 0 past the last barrier, or a wait that ran out: the
            // first to set the word decides for all.  (Write back can only
            // be set once every workgroup has arrived at that barrier.)
            const unsigned want = alive && W.wg == 0 ? 1u : 2u;
            const unsigned old = atomicCAS(P.sync + kSyCommit, 0u, want);
            d = old ? old : want;
        }
        // a word of its own: a wave may still have to read S.ok of the wait
        // that ended the loop
        S.commit = (int)d;
    }
    __syncthreads();
    if (S.commit != 1) return;
    if (owner) {
        (cur ? P.y1 : P.y0)[r] = yprev;
        (cur ? P.y0 : P.y1)[r] = yfront;
        for (int j = 0; j < P.nk; ++j) P.K[(int64_t)j * P.npad + r] = K[j * rows + lr];
    }
    if (W.wg == 0) {
        if (tid == 0) {
            S.c.times = times_mem;
            S.c.resident = RES_DONE;
        }
        __syncthreads();
        int *dst = (int *)P.ctl;
        for (int i = tid; i < (int)(sizeof(RKCtl) / 4); i += nt) dst[i] = ((int *)&S.c)[i];
    }
}

__global__ __launch_bounds__(256) void res_prepare_kernel(unsigned *sync, RKCtl *ctl) {
    for (int i = threadIdx.x; i < kResSyncWords; i += blockDim.x) sync[i] = 0;
    if (threadIdx.x == 0) ctl->resident = RES_RUNNING;
}

// Functional f of output out_base + k (grid: outputs, functionals) from the
// states kept in yout, summed as rk_output_kernel sums: chunks of kOutChunk
// entries (a row of 16 lanes each), the chunk sums strided over 64 lanes,
// then the wave tree.
__device__ __forceinline__ double row16_sum(double v) {
    v += dpp_move<0xB1>(v);
    v += dpp_move<0x4E>(v);
    v += dpp_move<0x141>(v);
    v += dpp_move<0x140>(v);
    return v;
}

__global__ __launch_bounds__(256) void res_functionals_kernel(ResFunArgs A) {
    const int out = A.out_base + (int)blockIdx.x, f = blockIdx.y;
    if (out >= A.ctl->out_idx) return;  // uniform
    __shared__ double2 part[64];
    const double2 *y = A.yout + (int64_t)blockIdx.x * A.nneed;
    const int fbeg = A.fptr[f], fend = A.fptr[f + 1], quad = A.fkind[f];
    const int nch = (fend - fbeg + kOutChunk - 1) / kOutChunk;
    const int tid = threadIdx.x;
    double re = 0.0, im = 0.0;  // wave 0: lane k's chunks
    for (int c0 = 0; c0 < nch; c0 += 64) {
        double2 v[4];
#pragma unroll
        for (int s = 0; s < 4; ++s) {
            const int e = fbeg + (c0 + 16 * s + tid / 16) * kOutChunk + tid % 16;
            const bool has = e < fend;
            const int ec = has ? e : fbeg;
            const double2 yc = y[A.fcol[ec]];
            v[s] = fun_term(A.fw[ec], yc, quad, quad ? y[A.frow[ec]] : yc);
            if (!has) v[s] = make_double2(0.0, 0.0);
        }
        __syncthreads();
#pragma unroll
        for (int s = 0; s < 4; ++s) {
            const double a = row16_sum(v[s].x), b = row16_sum(v[s].y);
            if (tid % 16 == 0) part[16 * s + tid / 16] = make_double2(a, b);
        }
        __syncthreads();
        if (tid < 64 && c0 + tid < nch) {
            re += part[tid].x;
            im += part[tid].y;
        }
    }
    if (tid < 64) {
        re = wave_sum(re);
        im = wave_sum(im);
        if (tid == 0) A.fun_out[(int64_t)out * A.nfun + f] = make_double2(re, im);
    }
}

const void *res_kernel(int form) {
    switch (form) {
        case RES_KEPT: return (const void *)rk_resident_kernel<double2, RES_KEPT>;
        case RES_SELL: return (const void *)rk_resident_kernel<double2, RES_SELL>;
        case RES_SELL_F32: return (const void *)rk_resident_kernel<float2, RES_SELL_F32>;
        case RES_CODED: return (const void *)rk_resident_kernel<double2, RES_CODED>;
        case RES_CODED_TD: return (const void *)rk_resident_kernel<double2, RES_CODED_TD>;
        case RES_DIA: return (const void *)rk_resident_kernel<double2, RES_DIA>;
        default: return nullptr;
    }
}

}  // namespace

size_t res_lds_bytes(int form, int lanes, int threads, int nk, int vbits) {
    size_t b = sizeof(double2) * (size_t)nk * (threads / lanes);
    if (form == RES_CODED || form == RES_CODED_TD)
        b += sizeof(double2) * ((size_t)1 << vbits) * (form == RES_CODED_TD ? 2 : 1) +
             sizeof(int) * ((size_t)1 << (16 - vbits));
    return b;
}

bool res_plan(int form, int lanes, int64_t lanes_total, int nk, int vbits, ResArgs *P) {
    int dev = 0, cus = 0;
    if (hipGetDevice(&dev) != hipSuccess ||
        hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess)
        return false;
    if (cus < 8) return false;
    const int per_xcd = std::min(cus / 8, 32);
    const void *fn = res_kernel(form);
    if (!fn) return false;
    for (int threads : {256, kResThreads}) {
        const size_t lds = res_lds_bytes(form, lanes, threads, nk, vbits);
        if (lds > kResLdsMax) continue;
        const int64_t nwg = (lanes_total + threads - 1) / threads;
        if (nwg > 8 * per_xcd) continue;
        const bool multi = nwg > per_xcd;
        // a smaller workgroup that needs every XCD gives way to a larger one
        // that fits one
        if (multi && threads < kResThreads &&
            (lanes_total + kResThreads - 1) / kResThreads <= per_xcd &&
            res_lds_bytes(form, lanes, kResThreads, nk, vbits) <= kResLdsMax)
            continue;
        int occ = 0;
        if (hipFuncSetAttribute(fn, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds) !=
                hipSuccess ||
            hipOccupancyMaxActiveBlocksPerMultiprocessor(&occ, fn, threads, lds) != hipSuccess ||
            occ < 1) {
            (void)hipGetLastError();
            continue;
        }
        P->threads = threads;
        P->nwg = (int)nwg;
        P->multi = multi ? 1 : 0;
        P->lanes = lanes;
        P->grid = multi ? (int)nwg : (int)nwg * 8;
        return true;
    }
    return false;
}

int res_launch(int form, const ResArgs &P, const DiaOp &D, hipStream_t s) {
    const void *fn = res_kernel(form);
    QA_REQUIRE(fn != nullptr, "resident loop: no kernel for this operator");
    QA_REQUIRE(P.polls >= 0, "resident loop: not launched");
    const size_t lds = res_lds_bytes(form, P.lanes, P.threads, P.nk, P.vbits);
    QA_HIP(hipFuncSetAttribute(fn, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds));
    hipLaunchKernelGGL(res_prepare_kernel, dim3(1), dim3(256), 0, s, P.sync, P.ctl);
    QA_CHECK_LAUNCH();
    void *args[] = {(void *)&P, (void *)&D};
    // An ordinary launch: the grid fits the chip (res_plan) and every wait is
    // bounded.  A cooperative one makes the runtime open a queue of its own
    // for the rest of the process, and with it kernels of different streams
    // overlap less: the solve server after one such launch took 34.4 s for
    // 1000 requests that take 28.4 s without, and 28.0 with this one.
    QA_HIP(hipLaunchKernel(fn, dim3(P.grid), dim3(P.threads), args, (unsigned)lds, s));
    return QA_OK;
}

int res_functionals(const ResFunArgs &A, int nout, hipStream_t s) {
    if (A.nfun < 1 || nout < 1) return QA_OK;
    hipLaunchKernelGGL(res_functionals_kernel, dim3(nout, A.nfun), dim3(256), 0, s, A);
    QA_CHECK_LAUNCH();
    return QA_OK;
}

}  // namespace qa
