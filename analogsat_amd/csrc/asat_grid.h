// Persistent integrator over a few workgroups, for problems too big for one
// workgroup's LDS (asat_small.h) and too small for 13 kernels per attempt to
// pay: those take 60 to 80 us an attempt whatever the size, nearly all of it the
// kernels' own start and end.
//
// Every workgroup owns the variables of some groups of 64 and keeps a copy of
// every clause that names one of them, with the clause's auxiliary state and
// stage derivatives in registers.  A clause of K literals is then carried by up
// to K workgroups, which compute the same bits; in return a stage needs one
// exchange between workgroups, the stage spins, and none for the contributions:
//   clause phase: factors from the spins of all variables in LDS, K_m, the aux
//     stage input, k_J(a); terms of the workgroup's own variables into LDS
//   var phase:    own variables add their terms (rows of 64 entries, -0.0 where
//     one is missing) in the reference's accumulation order and form their
//     next stage input (J = 6: x_new)
//   exchange:     own spins to a global buffer, a barrier, everyone's spins back
//     into LDS.  The last one carries the workgroups' error maxima, the first
//     one of a step the violated-clause counts where they are due; every
//     workgroup then takes the same decision.
// Spins travel by agent-scope relaxed atomics, which bypass the caches that are
// not coherent between XCDs; an agent-scope acquire fence (an invalidation per
// wave) would cost 1 to 7 us more per exchange at 64 to 256 workgroups.  Measured
// alone, a store, the barrier and four loads take 2.2 us with 8 workgroups, 2.8
// with 32, 4.3 with 64 and 6.9 with 256.  Two buffers alternate: no workgroup can
// write one again before all have passed the barrier after reading it.
//
// The arithmetic is that of the multi-kernel path (clause_tile / var_stage),
// operation for operation, so states, step sizes and counters are the same bits.
// Clauses of 3 or 4 literals, CTDS family, no bias term; the solver loop of
// SatSolver runs on the device as in asat_small.h.
//
// One workgroup alone (SOLO, up to 1024 variables) keeps the same layout and
// exchanges through LDS.  It is bound by the latency of its phases, and holding
// the state in registers and reading a variable's terms as rows without bank
// conflicts leaves fewer of them than asat_small.h, which has every vector in
// LDS (us per attempt, FP64: N = 200, M = 852 7.0 against 10.7, N = 240 7.3
// against 12.0).  With 256 threads, up to 512 clauses, it was no faster (N = 50:
// 4.7-5.1 against 4.6), so those keep asat_small.h.
//
// The layout is used where the device holds all its workgroups at once, and the
// launch is cooperative where the runtime grants it. Where they wait for each other all the same (another
// process keeps part of the CUs busy), a wait that lasts GRID_POLLS polls gives
// up: it marks the arrival word unless the last arrival came in between, so
// every workgroup gives up at the same exchange, and none stores anything. The
// launch then has had no effect and the host goes on by another path.
// Bound by the latency of its six exchanges: N = 2000, M = 8500 takes 20.6 us an
// attempt in FP32 and 24.3 in FP64 (multi-kernel path 65 and 73), N = 12000,
// M = 51120 43 and 58 (68 and 66).
#pragma once

#include <type_traits>

#include "asat_common.h"
#include "asat_small.h"

namespace asat {

constexpr int GRID_BT = 1024;            // threads per workgroup
constexpr int GRID_MAX = 128;            // workgroups
constexpr int GRID_WAVES = GRID_BT / 64; // variable groups a workgroup can own
constexpr int GRID_POLLS = 1 << 21;      // a second or two
constexpr unsigned GRID_GIVE_UP = 1u << 31;    // in the arrival word
constexpr int GRID_ATTEMPT_CAP = 4096;   // attempts per launch

struct GridArgs {
    const uint32_t* code;    // per workgroup, clause and literal: term entry << 16 | rank << 1 | negated
    const int* cpos;         // per workgroup and clause: its position in the aux block
    const int* wg;           // per workgroup: first clause, clauses, clauses it writes (they come first), term entries
    const int* group;        // per group of 64 ranks: base of its term rows, their number
    const int* vmap;         // rank -> variable (0: none)
    void* x;                 // state buffer: read at entry, newest state written at exit
    Ctrl* ctrl;
    SmallSolve* solve;       // null: Step mode
    void* pub;               // [2][64 * ngroups] published spins
    double* err;             // [2][GRID_MAX] error maxima
    int* count;              // [2][GRID_MAX] violated clauses
    unsigned* barrier;       // arrivals of all launches so far, and GRID_GIVE_UP
    unsigned phase;          // exchanges so far
    long long target, max_steps;
    double max_time;
    int time_float, batch;
    int attempt_cap;         // attempts per launch
    int ngroups, aoff;
    double knorm;
};

// the kernel for a precision, clause length and clauses per thread (null: none);
// solo: the one-workgroup form
const void* grid_kernel(int precision, int k, int cpt, bool solo);

template <typename T>
__device__ __forceinline__ T agent_load(const T* p)
{
    return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
template <typename T>
__device__ __forceinline__ void agent_store(T* p, T v)
{
    __hip_atomic_store(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

// v with its sign flipped where bit 0 of c is set
__device__ __forceinline__ float grid_sign(uint32_t c, float v)
{
    return __uint_as_float((c << 31) ^ __float_as_uint(v));
}
__device__ __forceinline__ double grid_sign(uint32_t c, double v)
{
    return __longlong_as_double((long long)(((unsigned long long)(c << 31) << 32) ^
                                            (unsigned long long)__double_as_longlong(v)));
}

struct GridShared {
    double red[GRID_WAVES];
    int redi[GRID_WAVES];
    double errmax, power;
    int count, give_up;
};

template <typename T, int KT, int CPT>
struct GridRegs {
    T xa[CPT], a1[CPT], a2[CPT], a3[CPT], a4[CPT], a5[CPT];
    T xv, v1, v2, v3, v4, v5;
    uint32_t code[CPT][KT];
};

// clause phase of stage J; nclause, nwrite: this workgroup's clauses, and those
// whose error term and violations it accounts for
template <typename T, int KT, int CPT, int J, bool COUNT>
__device__ __forceinline__ void grid_clauses(GridRegs<T, KT, CPT>& R, const T* s, T* con, int nclause, int nwrite,
                                             T knorm, T hs, double h, double hnext, double floor, double& err,
                                             int& viol)
{
    const int tid = (int)threadIdx.x;
    const int w0 = __builtin_amdgcn_readfirstlane(tid & ~63);
#pragma unroll
    for (int u = 0; u < CPT; u++) {
        if (w0 + u * GRID_BT < nclause) {
            uint32_t c[KT];
            T sv[KT], f[KT];
#pragma unroll
            for (int q = 0; q < KT; q++) {
                asm("" : "+v"(R.code[u][q]));    // nothing derived from a code is kept between stages
                c[q] = R.code[u][q];
                sv[q] = s[(c[q] & 0xFFFFu) >> 1];
            }
            T km = knorm;
#pragma unroll
            for (int q = 0; q < KT; q++) {
                f[q] = (T)1.0 - grid_sign(c[q], sv[q]);
                km *= f[q];
            }
            if constexpr (COUNT) {
                bool sat = false;
#pragma unroll
                for (int q = 0; q < KT; q++) {
                    // the padding rank (spin -1, never negated) is false
                    const bool t = sv[q] > (T)0;
                    sat = sat || ((c[q] & 1u) ? !t : t);
                }
                viol += (!sat && tid + u * GRID_BT < nwrite) ? 1 : 0;
            }
            T am;
            if constexpr (J == 1) am = R.xa[u];
            else am = stage_input<T, J>(R.xa[u], R.a1[u], R.a2[u], R.a3[u], R.a4[u], R.a5[u], hs);
            const T kj = am * km * km;
            if constexpr (J == 1) R.a1[u] = kj;
            else if constexpr (J == 2) R.a2[u] = kj;
            else if constexpr (J == 3) R.a3[u] = kj;
            else if constexpr (J == 4) R.a4[u] = kj;
            else if constexpr (J == 5) R.a5[u] = kj;
            else {
                // x_new waits in the k2 register, which the combination does not read
                T xn;
                double e = 0.0;
                if (w0 + u * GRID_BT < nwrite)
                    final_combination<T>(R.xa[u], R.a1[u], R.a3[u], R.a4[u], R.a5[u], kj, hs, h, hnext, floor, xn, e);
                else
                    xn = R.xa[u] + hs * (Tab<T>::c1 * R.a1[u] + Tab<T>::c3 * R.a3[u] + Tab<T>::c4 * R.a4[u] +
                                         Tab<T>::c6 * kj);
                R.a2[u] = xn;
                err = fmax(err, e);
            }
            const T r = km * knorm * am;
#pragma unroll
            for (int q = 0; q < KT; q++) {
                T p = (T)1.0;
                bool first = true;
#pragma unroll
                for (int qq = 0; qq < KT; qq++) {
                    if (qq == q) continue;
                    p = first ? f[qq] : p * f[qq];
                    first = false;
                }
                con[c[q] >> 16] = grid_sign(c[q], (r * p) * (T)2.0);
            }
        }
    }
}

// left-to-right sum of this lane's entries in `depth` rows of 64.  Eight loads in
// flight: 32 at once spilled, 128 registers being what 1024 threads have
// (N = 400 alone, FP64: 13.6 against 9.3 us an attempt).
template <typename T>
__device__ __forceinline__ T grid_sum(const T* e, int depth)
{
    T sum = (T)0;
    int i = 0;
    for (; i + 8 <= depth; i += 8, e += 8 * 64) {
        T t[8];
#pragma unroll
        for (int u = 0; u < 8; u++) t[u] = e[64 * u];
#pragma unroll
        for (int u = 0; u < 8; u++) sum += t[u];
    }
    for (; i + 2 <= depth; i += 2, e += 2 * 64) {
        const T t0 = e[0], t1 = e[64];
        sum += t0;
        sum += t1;
    }
    if (i < depth) sum += e[0];
    return sum;
}

template <typename T, int KT, int CPT, bool SOLO>
__global__ __launch_bounds__(GRID_BT) void k_grid(GridArgs a)
{
    // [spins by rank, then the padding rank] [terms, then one that nothing reads]
    extern __shared__ __attribute__((aligned(16))) unsigned char grid_lds[];
    __shared__ GridShared sh;
    const int tid = (int)threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int w = SOLO ? 0 : (int)blockIdx.x, G = SOLO ? GRID_WAVES : (int)gridDim.x;
    const int nranks = 64 * a.ngroups;
    T* s = (T*)grid_lds;
    T* con = s + nranks + 2;
    const int c0 = a.wg[4 * w], nclause = a.wg[4 * w + 1], nwrite = a.wg[4 * w + 2], ncon = a.wg[4 * w + 3];
    // wave v owns group w + v * G (alone: group v)
    const int grp = SOLO ? wave : w + wave * G;
    const bool own = grp < a.ngroups;
    const int rank = grp * 64 + lane;
    const int var = own ? a.vmap[rank] : 0;
    const int gbase = own ? a.group[2 * grp] : 0, gdepth = own ? a.group[2 * grp + 1] : 0;
    T* x = (T*)a.x;
    const T knorm = (T)a.knorm;

    GridRegs<T, KT, CPT> R;
#pragma unroll
    for (int u = 0; u < CPT; u++) {
        const int j = tid + u * GRID_BT;
        R.xa[u] = j < nclause ? x[a.aoff + a.cpos[c0 + j]] : (T)0;
        R.a1[u] = R.a2[u] = R.a3[u] = R.a4[u] = R.a5[u] = (T)0;
#pragma unroll
        for (int q = 0; q < KT; q++)
            R.code[u][q] = j < nclause ? a.code[(long long)(c0 + j) * KT + q]
                                       : ((uint32_t)ncon << 16) | ((uint32_t)nranks << 1);
    }
    R.xv = var ? x[var] : (T)0;
    R.v1 = R.v2 = R.v3 = R.v4 = R.v5 = (T)0;
    for (int i = tid; i < nranks; i += GRID_BT) s[i] = a.vmap[i] ? x[a.vmap[i]] : (T)0;
    if (tid < 2) s[nranks + tid] = (T)-1.0;
    for (int i = tid; i < ncon; i += GRID_BT) con[i] = (T)-0.0;
    if (tid == 0) sh.give_up = 0;

    const Ctrl* c = a.ctrl;
    double h = c->h, hnext = c->hnext, time = c->time, hdid = c->hdid, errmax = c->errmax;
    const double eps = c->eps, floor = c->floor;
    long long steps = c->steps, attempts = c->attempts, rhscount = c->rhscount;
    int underflow = c->underflow;
    double* hlog = c->hlog;
    const long long hlog_len = c->hlog_len;
    SmallSolve ss = {0, 0, -1, 0, 0};
    if (a.solve) ss = *a.solve;
    __syncthreads();

    unsigned phase = a.phase;
    double ctl_errmax = 0.0, ctl_power = 0.0;     // what an exchange brought
    int ctl_count = 0;
    // Publish this thread's spin (waves that own a group), wait for every
    // workgroup, then take everyone's spins into LDS.  ERR: with the
    // workgroups' error maxima, from which wave 0 forms errmax and its power;
    // CNT: with their violation counts.  False when the wait was given up.
    auto exchange = [&](T val, auto errc, double e, auto cntc, int cnt) -> bool {
        constexpr bool ERR = decltype(errc)::value, CNT = decltype(cntc)::value;
        if constexpr (SOLO) {
            if (own) s[rank] = val;
            if constexpr (ERR) {
                e = wave_max_dpp(e);
                if (lane == 0) sh.red[wave] = e;
            }
            if constexpr (CNT) {
                cnt = wave_sum(cnt);
                if (lane == 0) sh.redi[wave] = cnt;
            }
            __syncthreads();
            if constexpr (ERR) {
                double m = sh.red[0];
#pragma unroll
                for (int i = 1; i < GRID_WAVES; i++) m = fmax(m, sh.red[i]);
                if (wave == 0) {
                    m /= eps;
                    const double pw = m > TabD::ERRCON ? pow_ctrl(m, m <= 1.0 ? 5 : 4) : 0.0;
                    if (lane == 0) { sh.errmax = m; sh.power = pw; }
                }
                __syncthreads();
                ctl_errmax = sh.errmax;
                ctl_power = sh.power;
            }
            if constexpr (CNT) {
                ctl_count = sh.redi[0];
#pragma unroll
                for (int i = 1; i < GRID_WAVES; i++) ctl_count += sh.redi[i];
            }
            return true;
        }
        const int half = (int)(phase & 1u);
        T* pub = (T*)a.pub + (long long)half * nranks;
        if (own) agent_store(pub + rank, val);
        if constexpr (ERR) {
            e = wave_max_dpp(e);
            if (lane == 0) sh.red[wave] = e;
        }
        if constexpr (CNT) {
            cnt = wave_sum(cnt);
            if (lane == 0) sh.redi[wave] = cnt;
        }
        // the stores have reached memory before the arrival counts
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
        __syncthreads();
        phase++;
        if (tid == 0) {
            if constexpr (ERR) {
                double m = sh.red[0];
#pragma unroll
                for (int i = 1; i < GRID_WAVES; i++) m = fmax(m, sh.red[i]);
                agent_store(a.err + half * GRID_MAX + w, m);
            }
            if constexpr (CNT) {
                int m = 0;
#pragma unroll
                for (int i = 0; i < GRID_WAVES; i++) m += sh.redi[i];
                agent_store(a.count + half * GRID_MAX + w, m);
            }
            if constexpr (ERR || CNT) asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
            const unsigned want = phase * (unsigned)G;
            __hip_atomic_fetch_add(a.barrier, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            int polls = 0;
            unsigned v;
            // (a marked word is past every count)
            while ((v = agent_load(a.barrier)) < want) {
                // marked only while an arrival is missing: nobody has passed this
                // exchange, and nobody will
                if (++polls > GRID_POLLS &&
                    __hip_atomic_compare_exchange_strong(a.barrier, &v, v | GRID_GIVE_UP, __ATOMIC_RELAXED,
                                                         __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT)) {
                    v = GRID_GIVE_UP;
                    break;
                }
            }
            if (v & GRID_GIVE_UP) sh.give_up = 1;
        }
        __syncthreads();
        if (sh.give_up) return false;
        for (int i = tid; i < nranks; i += GRID_BT) s[i] = agent_load(pub + i);
        if constexpr (ERR) {
            if (wave == 0) {
                double e2 = 0.0;
                for (int i = lane; i < G; i += 64) e2 = fmax(e2, agent_load(a.err + half * GRID_MAX + i));
                const double m = wave_max_dpp(e2) / eps;
                const double pw = m > TabD::ERRCON ? pow_ctrl(m, m <= 1.0 ? 5 : 4) : 0.0;
                if (lane == 0) { sh.errmax = m; sh.power = pw; }
            }
        }
        if constexpr (CNT) {
            if (wave == 0) {
                int c2 = 0;
                for (int i = lane; i < G; i += 64) c2 += agent_load(a.count + half * GRID_MAX + i);
                const int m = wave_sum(c2);
                if (lane == 0) sh.count = m;
            }
        }
        __syncthreads();
        if constexpr (ERR) { ctl_errmax = sh.errmax; ctl_power = sh.power; }
        if constexpr (CNT) ctl_count = sh.count;
        return true;
    };
    using Yes = std::integral_constant<bool, true>;
    using No = std::integral_constant<bool, false>;

    int launched = 0;
    bool done = underflow || (a.solve ? ss.result >= 0 : steps >= a.target);
    bool alive = true;
    while (!done && alive) {
        // ---- a step: stage 1 at x
        if (launched >= a.attempt_cap) break;         // pause between steps
        double err = 0.0;
        int cnt = 0;
        T hs = (T)h;
        const bool check = a.solve && ss.check;
        if (check) grid_clauses<T, KT, CPT, 1, true>(R, s, con, nclause, nwrite, knorm, hs, h, hnext, floor, err, cnt);
        else grid_clauses<T, KT, CPT, 1, false>(R, s, con, nclause, nwrite, knorm, hs, h, hnext, floor, err, cnt);
        __syncthreads();
        R.v1 = own ? grid_sum(con + gbase + lane, gdepth) : (T)0;
        {
            const T next = stage_input<T, 2>(R.xv, R.v1, 0, 0, 0, 0, hs);
            alive = check ? exchange(next, No{}, 0.0, Yes{}, cnt) : exchange(next, No{}, 0.0, No{}, 0);
            if (!alive) break;
        }
        if (check) {
            ss.check = 0;
            ss.last_viol = ctl_count;
            if (ss.last_viol == 0) {
                ss.result = SMALL_SAT;
                break;
            }
        }
        if (a.solve && ss.bleft == 0) {
            // top of the SatSolver loop: while (time < maxTime && steps < maxSteps)
            const double tc = a.time_float ? (double)(float)time : time;
            if (!(tc < a.max_time && ss.solver_steps < a.max_steps)) {
                ss.result = tc >= a.max_time ? SMALL_MAXTIME : SMALL_MAXITER;
                break;
            }
            ss.bleft = a.batch;
        }
        bool first = true, accepted = false;
        while (true) {
            hs = (T)h;
            err = 0.0;
#define ASAT_GRID_CLAUSES(J) \
    grid_clauses<T, KT, CPT, J, false>(R, s, con, nclause, nwrite, knorm, hs, h, hnext, floor, err, cnt); \
    __syncthreads();
            ASAT_GRID_CLAUSES(2)
            R.v2 = own ? grid_sum(con + gbase + lane, gdepth) : (T)0;
            if (!(alive = exchange(stage_input<T, 3>(R.xv, R.v1, R.v2, 0, 0, 0, hs), No{}, 0.0, No{}, 0))) break;
            ASAT_GRID_CLAUSES(3)
            R.v3 = own ? grid_sum(con + gbase + lane, gdepth) : (T)0;
            if (!(alive = exchange(stage_input<T, 4>(R.xv, R.v1, R.v2, R.v3, 0, 0, hs), No{}, 0.0, No{}, 0))) break;
            ASAT_GRID_CLAUSES(4)
            R.v4 = own ? grid_sum(con + gbase + lane, gdepth) : (T)0;
            if (!(alive = exchange(stage_input<T, 5>(R.xv, R.v1, R.v2, R.v3, R.v4, 0, hs), No{}, 0.0, No{}, 0))) break;
            ASAT_GRID_CLAUSES(5)
            R.v5 = own ? grid_sum(con + gbase + lane, gdepth) : (T)0;
            if (!(alive = exchange(stage_input<T, 6>(R.xv, R.v1, R.v2, R.v3, R.v4, R.v5, hs), No{}, 0.0, No{}, 0)))
                break;
            ASAT_GRID_CLAUSES(6)
#undef ASAT_GRID_CLAUSES
            T xn = (T)0;
            if (own) {
                double e;
                const T k6 = grid_sum(con + gbase + lane, gdepth);
                final_combination<T>(R.xv, R.v1, R.v3, R.v4, R.v5, k6, hs, h, hnext, floor, xn, e);
                err = fmax(err, e);
            }
            if (!(alive = exchange(xn, Yes{}, err, No{}, 0))) break;
            launched++;
            errmax = ctl_errmax;
            attempts += 1;
            rhscount += first ? 6 : 5;
            first = false;
            if (errmax <= 1.0) {
                const double hn = errmax > TabD::ERRCON ? TabD::SAFETY * h * ctl_power : 5.0 * h;
                hdid = h;
                time += h;
                if (hlog && steps < hlog_len && w == 0 && tid == 0) hlog[steps] = h;
                steps += 1;
                R.xv = xn;
#pragma unroll
                for (int u = 0; u < CPT; u++) R.xa[u] = R.a2[u];
                hnext = hn;
                h = hn;
                accepted = true;
                break;
            }
            const double htemp = TabD::SAFETY * h * ctl_power;
            const double hn = h >= 0.0 ? fmax(htemp, TabD::HFACTOR * h) : fmin(htemp, TabD::HFACTOR * h);
            h = hn;
            if (time + hn == time) {
                underflow = 1;
                if (a.solve) ss.result = SMALL_UNDERFLOW;
                break;
            }
            // a retry restarts at stage 2 with the reduced h
            if (!(alive = exchange(stage_input<T, 2>(R.xv, R.v1, 0, 0, 0, 0, (T)h), No{}, 0.0, No{}, 0))) break;
        }
        if (!accepted) break;
        if (a.solve) {
            if (--ss.bleft == 0) {
                ss.solver_steps += a.batch;
                ss.check = 1;
            }
        } else if (steps >= a.target) {
            done = true;
        }
    }
    if (!alive) return;
    // newest state: spins by their owners, each clause by the one that writes it
    if (var) x[var] = R.xv;
#pragma unroll
    for (int u = 0; u < CPT; u++) {
        const int j = tid + u * GRID_BT;
        if (j < nwrite) x[a.aoff + a.cpos[c0 + j]] = R.xa[u];
    }
    if (w == 0 && tid == 0) {
        Ctrl* cw = a.ctrl;
        cw->h = h; cw->hnext = hnext; cw->time = time; cw->hdid = hdid; cw->errmax = errmax;
        cw->steps = steps; cw->attempts = attempts; cw->rhscount = rhscount;
        cw->step_start = 1; cw->underflow = underflow; cw->active = 0;
        if (a.solve) *a.solve = ss;
    }
}

}  // namespace asat
