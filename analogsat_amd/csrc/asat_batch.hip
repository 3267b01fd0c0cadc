// Batched ragged CTDS solver for MI355X: thousands of independent trajectories
// (each with its own instance, N, M, k, step size and early exit) in one
// persistent launch.  No reference counterpart: the reference runs one
// trajectory per process (Frontend/src/bench_runner.cpp:257-348 launches
// CudaSat*+CudaRungeKutta once per sample).
//
// Mapping: one workgroup owns one trajectory at a time and runs the whole
// Cash-Karp loop for it; RK stages are separated by workgroup barriers, not
// kernel launches.  Per stage:
//   clause phase: each thread takes clauses j = tid, tid+BS, ...; gathers the
//     stage spins from LDS, forms K_m, the aux stage input (x_a, k1..k5 from
//     the workgroup's scratch), k_J(a_m) = a K^2, and writes each literal's
//     contribution 2 c a K K_mi straight into var-major order (LDS, or the
//     workgroup's global scratch for instances too big for LDS)
//   var phase:    each thread takes variables i = tid, tid+BS, ...; sums its
//     contiguous run of contributions in slot order (the reference's
//     accumulation order), writes k_J(s_i) and the next stage's spin input
// Instances that fit run in k_batch_reg, which keeps state and stage
// derivatives in registers and contributions in LDS; instances whose
// contributions do not fit in LDS run in k_batch_chunk, which takes the clauses
// in chunks whose contributions do.  k_batch is the general form (contributions
// in LDS or in global scratch).
// Stage 6 forms x_new and |xerr/xscal|, a block FP64 max feeds the step
// controller (thread 0, FP64, correctly rounded pow), which accepts (parity
// flip) or rejects (retry with smaller h).  After each accepted step the
// violated-clause count of the thresholded state is taken; SAT ends the
// trajectory, and the minimum count is tracked (MAXSAT).
//
// Work queue: workgroups pull trajectory ids from an atomic counter (ids are
// ordered largest first); each launch advances every live trajectory by at
// most chunk_steps accepted steps, so a launch is bounded and a sequence of
// launches is captured once in a hipGraph.
//
// Per-slot packing (uint32): bits 19..31 variable (1-based, 0 = padding),
// bit 18 negated, bits 0..17 position of the slot's contribution in the
// instance's var-major order.  Hence N <= 8191 and L = K*M <= 262143 per
// instance; bigger instances belong to the plain solver.
#include "asat_common.h"

#include <algorithm>
#include <atomic>
#include <chrono>
#include <cmath>
#include <cstring>
#include <exception>
#include <memory>
#include <mutex>
#include <numeric>
#include <system_error>
#include <thread>
#include <type_traits>
#include <vector>

namespace asat {

extern thread_local std::string g_last_error;

namespace batch {

constexpr int KMAX = 4;
constexpr int MAXN = 8191;
constexpr int MAXL = 262143;

enum Status { RUNNING = 0, SOLVED = 1, BUDGET = 2, UNDERFLOW_ = 3, MAXTIME = 4 };

struct Desc {                 // one instance / trajectory (device)
    long long code_off;       // into code[]
    long long row_off;        // into rowptr[]
    long long state_off;      // into xa[]/xb[] (N spins then M aux)
    long long rcode_off, rgroup_off, rvmap_off;   // register kernel's layout (-1: not built)
    long long ccode_off, cgroup_off, crec_off, cstart_off;   // chunked kernel's layout (-1: not built)
    int n, m, k, nslots;      // nslots = number of contributions (non-padding slots)
    float knorm;
    int ngroups, ncontrib;    // register kernel: groups of 64 ranks, contribution entries
    int nchunks, chunk;       // chunked kernel: chunks, clauses per chunk
    int pad_;
};

struct TrajCtrl {             // persistent per-trajectory control (device)
    double t, h, hnext, hdid, errmax, sat_time;
    long long steps, attempts, rhscount;
    int parity, status, min_viol, viol, sat_step, pad_;
};

struct Params {
    const Desc* desc;
    const uint32_t* code;
    const int* rowptr;
    float* xa;
    float* xb;
    TrajCtrl* ctrl;
    float* scratch;          // per-workgroup: 5 * stride (k1..k5) [+ maxL contributions]
    long long scratch_stride;  // floats per k vector in scratch (>= max n+m)
    long long scratch_per_wg;  // floats per workgroup
    const int* order;        // trajectory ids, largest first
    int ntraj;
    int* queue;              // atomic work counter (reset by the host before a launch)
    double eps;
    double floor;            // constant term of xscal (1e-20 = reference TINY)
    double max_time;
    long long max_steps;
    int chunk_steps;
    int check_every;         // take the violation count every this many accepted steps
    int sp_stride;           // floats reserved for the stage spins at the start of LDS
    const uint32_t* rcode;   // register kernel: literal codes, base and depth per group, rank -> variable
    const int* rgroup;
    const int* rvmap;
    const uint2* ccode;      // chunked kernel: literal codes of a clause, (base, depth) per group of 64
    const int2* cgroup;      // variables, its variables, their term indices (two per word), first
    const uint16_t* cperm;   // group of each chunk
    const uint32_t* crec;
    const int* cstart;
    int reg_lds;             // register kernel: LDS bytes of one trajectory
    int chunk_terms;         // chunked kernel: term entries in LDS (the one after holds 0)
    int fac_ranks;           // chunked kernel: factor pairs, then sums reserved in LDS
};

// ---------------------------------------------------------------------------
// MODE 0: contributions in the workgroup's global scratch; 1: in LDS.
template <int BS, int MODE>
__global__ __launch_bounds__(BS) void k_batch(Params P)
{
    extern __shared__ float lds[];          // [stage spins: sp_stride] then contributions
    __shared__ double red[BS / 64];
    __shared__ int redi[BS / 64];
    __shared__ int s_traj;

    float* sp = lds;                        // stage spin input, index i-1 for variable i
    float* scratch = P.scratch + (long long)blockIdx.x * P.scratch_per_wg;
    float* kbuf1 = scratch;
    float* kbuf2 = scratch + P.scratch_stride;
    float* kbuf3 = scratch + 2 * P.scratch_stride;
    float* kbuf4 = scratch + 3 * P.scratch_stride;
    float* kbuf5 = scratch + 4 * P.scratch_stride;
    const int tid = threadIdx.x;

    for (;;) {
        if (tid == 0) s_traj = atomicAdd(P.queue, 1);
        __syncthreads();
        // the trajectory id is the same in every lane: reading it as a
        // scalar lets the descriptor and the instance's base pointers live
        // in scalar registers, leaving the vector registers to the state
        const int slot = __builtin_amdgcn_readfirstlane(s_traj);
        __syncthreads();
        if (slot >= P.ntraj) break;
        const int tr = __builtin_amdgcn_readfirstlane(P.order[slot]);
        const Desc d = P.desc[tr];
        TrajCtrl* cp = P.ctrl + tr;
        if (cp->status != RUNNING) continue;    // uniform: every thread reads the same word

        const int n = d.n, m = d.m, k = d.k;
        const uint32_t* code = P.code + d.code_off;
        const int* rowptr = P.rowptr + d.row_off;
        float* contrib = MODE == 1 ? (lds + P.sp_stride) : (scratch + 5 * P.scratch_stride);
        const float knorm = d.knorm;
        // scratch layout per k vector: spins at [0, n), aux at [n, n+m)
        double t = cp->t, h = cp->h, hnext = cp->hnext, hdid = cp->hdid, errmax_last = cp->errmax;
        long long steps = cp->steps, attempts = cp->attempts, rhscount = cp->rhscount;
        int parity = cp->parity, min_viol = cp->min_viol, viol = cp->viol;
        int status = RUNNING;
        int sat_step = cp->sat_step;
        double sat_time = cp->sat_time;
        int done_in_chunk = 0;

        while (status == RUNNING && done_in_chunk < P.chunk_steps) {
            float* x = (parity ? P.xb : P.xa) + d.state_off;
            float* xn = (parity ? P.xa : P.xb) + d.state_off;
            // ---- stage 1 at x: spins into LDS
            for (int i = tid; i < n; i += BS) sp[i] = x[i];
            __syncthreads();
            bool accepted = false;
            bool first_attempt = true;
            while (!accepted) {
                const float hs = (float)h;
                const bool had_stage1 = first_attempt;
                double err_local = 0.0;
#pragma unroll 1
                for (int J = first_attempt ? 1 : 2; J <= 6; J++) {
                    // ---------------- clause phase
                    for (int j = tid; j < m; j += BS) {
                        const uint32_t* cj = code + (long long)j * k;
                        float f[KMAX];
                        uint32_t cc[KMAX];
                        float km = knorm;
#pragma unroll
                        for (int q = 0; q < KMAX; q++) {
                            f[q] = 1.0f;
                            cc[q] = 0;
                            if (q < k) {
                                uint32_t c = cj[q];
                                cc[q] = c;
                                int v = (int)(c >> 19);
                                float s = v ? sp[v - 1] : -1.0f;
                                f[q] = (c >> 18) & 1u ? 1.0f + s : 1.0f - s;
                                km *= f[q];
                            }
                        }
                        const int ai = n + j;
                        const float xa = x[ai];
                        float am, k1 = 0.f, k3 = 0.f, k4 = 0.f, k5 = 0.f;
                        if (J == 1) {
                            am = xa;
                        } else {
                            k1 = kbuf1[ai];
                            float k2 = J > 2 ? kbuf2[ai] : 0.f;
                            k3 = J > 3 ? kbuf3[ai] : 0.f;
                            k4 = J > 4 ? kbuf4[ai] : 0.f;
                            k5 = J > 5 ? kbuf5[ai] : 0.f;
                            switch (J) {
                            case 2: am = stage_input<float, 2>(xa, k1, k2, k3, k4, k5, hs); break;
                            case 3: am = stage_input<float, 3>(xa, k1, k2, k3, k4, k5, hs); break;
                            case 4: am = stage_input<float, 4>(xa, k1, k2, k3, k4, k5, hs); break;
                            case 5: am = stage_input<float, 5>(xa, k1, k2, k3, k4, k5, hs); break;
                            default: am = stage_input<float, 6>(xa, k1, k2, k3, k4, k5, hs); break;
                            }
                        }
                        const float kj = am * km * km;
                        switch (J) {
                        case 1: kbuf1[ai] = kj; break;
                        case 2: kbuf2[ai] = kj; break;
                        case 3: kbuf3[ai] = kj; break;
                        case 4: kbuf4[ai] = kj; break;
                        case 5: kbuf5[ai] = kj; break;
                        default: {
                            float xv;
                            double e;
                            final_combination<float>(xa, k1, k3, k4, k5, kj, hs, h, hnext, P.floor, xv, e);
                            xn[ai] = xv;
                            err_local = fmax(err_local, e);
                        }
                        }
                        const float r = km * knorm * am;
#pragma unroll
                        for (int q = 0; q < KMAX; q++) {
                            if (q < k && (cc[q] >> 19) != 0) {
                                float p = 1.0f;
                                bool first = true;
#pragma unroll
                                for (int qq = 0; qq < KMAX; qq++) {
                                    if (qq == q || qq >= k) continue;
                                    p = first ? f[qq] : p * f[qq];
                                    first = false;
                                }
                                float rr = r * p;
                                rr *= (cc[q] >> 18) & 1u ? -2.0f : 2.0f;
                                contrib[cc[q] & 0x3FFFFu] = rr;
                            }
                        }
                    }
                    __syncthreads();
                    // ---------------- var phase
                    for (int i = tid; i < n; i += BS) {
                        const float kj = sum_run(0.0f, contrib, rowptr[i], rowptr[i + 1]);
                        const float xi = x[i];
                        switch (J) {
                        case 1:
                            kbuf1[i] = kj;
                            sp[i] = stage_input<float, 2>(xi, kj, 0.f, 0.f, 0.f, 0.f, hs);
                            break;
                        case 2:
                            kbuf2[i] = kj;
                            sp[i] = stage_input<float, 3>(xi, kbuf1[i], kj, 0.f, 0.f, 0.f, hs);
                            break;
                        case 3:
                            kbuf3[i] = kj;
                            sp[i] = stage_input<float, 4>(xi, kbuf1[i], kbuf2[i], kj, 0.f, 0.f, hs);
                            break;
                        case 4:
                            kbuf4[i] = kj;
                            sp[i] = stage_input<float, 5>(xi, kbuf1[i], kbuf2[i], kbuf3[i], kj, 0.f, hs);
                            break;
                        case 5:
                            kbuf5[i] = kj;
                            sp[i] = stage_input<float, 6>(xi, kbuf1[i], kbuf2[i], kbuf3[i], kbuf4[i], kj, hs);
                            break;
                        default: {
                            float xv;
                            double e;
                            final_combination<float>(xi, kbuf1[i], kbuf3[i], kbuf4[i], kbuf5[i], kj, hs, h, hnext,
                                                     P.floor, xv, e);
                            xn[i] = xv;
                            err_local = fmax(err_local, e);
                        }
                        }
                    }
                    __syncthreads();
                    if (J == 1) {
                        // a retry restarts at stage 2: its spin input needs the new h
                        first_attempt = false;
                    }
                }
                // ---------------- error norm + control (FP64), evaluated
                // identically by every thread so h, hnext, t stay uniform
                const double errmax = block_max_all<BS>(err_local, red) / P.eps;
                errmax_last = errmax;
                attempts += 1;
                rhscount += had_stage1 ? 6 : 5;
                if (errmax <= 1.0) {
                    double hn = errmax > TabD::ERRCON ? TabD::SAFETY * h * pow_ctrl(errmax, 5) : 5.0 * h;
                    hdid = h;
                    t += h;
                    steps += 1;
                    hnext = hn;
                    h = hn;
                    accepted = true;
                } else {
                    double htemp = TabD::SAFETY * h * pow_ctrl(errmax, 4);
                    double hn = h >= 0.0 ? fmax(htemp, TabD::HFACTOR * h) : fmin(htemp, TabD::HFACTOR * h);
                    if (t + hn == t) {
                        h = hn;
                        status = UNDERFLOW_;
                        break;
                    }
                    h = hn;
                    // retry: stage-2 spin input from x, k1 and the reduced h
                    const float hs2 = (float)h;
                    for (int i = tid; i < n; i += BS)
                        sp[i] = stage_input<float, 2>(x[i], kbuf1[i], 0.f, 0.f, 0.f, 0.f, hs2);
                    __syncthreads();
                }
            }
            if (status != RUNNING) break;
            parity ^= 1;
            done_in_chunk += 1;
            // ---------------- violated-clause count on the accepted state
            if (steps % P.check_every == 0 || steps >= P.max_steps) {
                const float* xs = (parity ? P.xb : P.xa) + d.state_off;
                int cnt = 0;
                for (int j = tid; j < m; j += BS) {
                    const uint32_t* cj = code + (long long)j * k;
                    int sat = 0;
                    for (int q = 0; q < k && !sat; q++) {
                        uint32_t c = cj[q];
                        int v = (int)(c >> 19);
                        if (!v) continue;
                        int tv = xs[v - 1] > 0.0f;
                        sat = (c >> 18) & 1u ? !tv : tv;
                    }
                    cnt += !sat;
                }
                viol = block_sum_all<BS>(cnt, redi);
                if (viol < min_viol) min_viol = viol;
                if (viol == 0) {
                    status = SOLVED;
                    sat_step = (int)steps;
                    sat_time = t;
                }
            }
            if (status == RUNNING && steps >= P.max_steps) status = BUDGET;
            if (status == RUNNING && t >= P.max_time) status = MAXTIME;
            __syncthreads();
        }
        if (tid == 0) {
            cp->t = t; cp->h = h; cp->hnext = hnext; cp->hdid = hdid; cp->errmax = errmax_last;
            cp->steps = steps; cp->attempts = attempts; cp->rhscount = rhscount;
            cp->parity = parity; cp->status = status; cp->min_viol = min_viol; cp->viol = viol;
            cp->sat_step = sat_step; cp->sat_time = sat_time;
        }
        __syncthreads();
    }
}

// ---------------------------------------------------------------------------
// Register-resident variant: TT threads per trajectory, one workgroup of them,
// or (TT = 64) a wave each in a workgroup of 256, which then needs no barriers.
// Thread tid owns clauses j = tid + u*TT (u < CPT)
// and the variables of rank tid + v*TT (v < VPT) for the whole trajectory;
// their state x and the stage derivatives k1..k5 live in registers.  LDS holds
// the stage factors and the contributions; a step touches global memory only
// for the literal codes, and not even for those where they fit the registers
// too.  The arithmetic and its order are those of k_batch; x_new of the final
// stage goes to the k2 registers, which the final combination does not read.
//
// What bounds it is instruction issue and LDS, so the layout (reg_layout)
// serves both:
// - Variables are ranked by falling number of occurrences, so the 64 of one
//   wave have nearly the same number, and a group of 64 keeps its
//   contributions as rows of 64 (entry e of all 64 variables side by side):
//   the sums read LDS without bank conflicts, without a bound per lane and
//   with addresses that are constants past the group's base.  Missing entries
//   hold -0.0, which changes no sum; every other entry is written again in
//   every clause phase.
// - The stage spins are kept as the two factors 1 - s and 1 + s, so a literal's
//   factor is one LDS read at its code's low 16 bits.  Two ranks past the last
//   variable are constants by the same rule: spin -1 (factor 2: a padding
//   literal of a short clause) and spin 0 (factor 1: a literal beyond the
//   instance's k, and the clauses that fill up the last wave).  Such literals
//   store into an entry that nothing reads, so no slot needs a test.
// - A code's low 16 bits are the byte address of its factor (8 rank + 4 if
//   negated), its high 16 bits the index of its contribution.  Up to 2046
//   variables bits 14 and 15 are zero and code >> 14 is that entry's byte
//   address (WIDE = false); more variables shift twice.
// - The violated-clause count of an accepted state is taken by the next step's
//   first clause phase, whose factors already say s > 0 unless one is exactly 1.
// Against the variable-major contribution runs before (a wave as slow as its
// busiest variable, bank conflicts in the sums, 4 instructions to unpack a
// slot), per 100 steps of 1024 trajectories with N = 2000, M = 8500: 26.0 ->
// 13.2 ms; 1000 steps of 1000 with N = 50, M = 213: 10.8 -> 7.3 ms.
constexpr int REG_WAVES = 4;     // TT = 64: trajectories (waves) per workgroup

// a value every lane holds, moved to scalar registers
__device__ __forceinline__ int uni(int v) { return __builtin_amdgcn_readfirstlane(v); }
__device__ __forceinline__ long long uni(long long v)
{
    return (long long)(((unsigned long long)(unsigned)uni((int)(v >> 32)) << 32) | (unsigned)uni((int)v));
}
__device__ __forceinline__ float uni(float v) { return __int_as_float(uni(__float_as_int(v))); }

template <int TT>
__device__ __forceinline__ int traj_tid()
{
    return TT == 64 ? (int)(threadIdx.x & 63) : (int)threadIdx.x;
}
// LDS written before is seen by the trajectory's threads after.  One wave's
// LDS accesses stay in order, so a wave alone only keeps the compiler to it.
template <int TT>
__device__ __forceinline__ void traj_sync()
{
    if constexpr (TT == 64) {
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
        __builtin_amdgcn_wave_barrier();
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
    } else {
        __syncthreads();
    }
}
// Error norm / eps over the trajectory's threads and the power of it that the
// step control needs (errmax^-0.2 on acceptance above ERRCON, errmax^-0.25 on
// rejection), in every thread; with several waves two barriers.  One wave
// computes them: in all of 16 waves the 190 dependent FP64 operations of
// pow_ctrl would take four times as long, a quarter of the SIMDs' issue each.
struct Control { double errmax, power; };
__device__ __forceinline__ Control control_of(double err, double eps)
{
    Control c;
    c.errmax = err / eps;
    c.power = c.errmax > TabD::ERRCON ? pow_ctrl(c.errmax, c.errmax <= 1.0 ? 5 : 4) : 0.0;
    return c;
}
template <int TT>
__device__ __forceinline__ Control traj_control(double v, double eps, double* red, Control* out)
{
    v = wave_max_dpp(v);
    if constexpr (TT == 64) return control_of(v, eps);
    const int lane = (int)(threadIdx.x & 63);
    if (lane == 0) red[threadIdx.x >> 6] = v;
    __syncthreads();
    if (threadIdx.x < 64) {
        const Control c = control_of(wave_max_dpp(lane < TT / 64 ? red[lane] : 0.0), eps);
        if (lane == 0) *out = c;
    }
    __syncthreads();
    return *out;
}
// sum over the trajectory's threads, in every one of them; LDS written before is
// seen after, as with traj_sync
template <int TT>
__device__ __forceinline__ int traj_sum(int v, int* sh)
{
    if constexpr (TT == 64) {
        traj_sync<TT>();
        return wave_sum(v);
    } else {
        return block_sum_all<TT>(v, sh);
    }
}

template <int TT, int CPT, int VPT, int KK>
struct RegState {
    float xa[CPT], a1[CPT], a2[CPT], a3[CPT], a4[CPT], a5[CPT];
    float xv[VPT], v1[VPT], v2[VPT], v3[VPT], v4[VPT], v5[VPT];
    // registers of a thread at this workgroup size, less the state, the
    // literal codes and about 36 for one clause's work
    static constexpr int BUDGET = TT >= 1024 ? 128 : TT >= 768 ? 168 : 256;
    static constexpr bool HOLD = CPT * (6 + KK) + VPT * 8 + 36 <= BUDGET;
    uint32_t code[HOLD ? CPT : 1][KK];
};

template <bool WIDE>
__device__ __forceinline__ float code_factor(const unsigned char* fac, uint32_t c)
{
    return *(const float*)(fac + (c & (WIDE ? 0xFFFFu : 0x3FFFu)));
}
template <bool WIDE>
__device__ __forceinline__ void code_store(unsigned char* con, uint32_t c, float v)
{
    if constexpr (WIDE) *(float*)(con + ((c >> 16) << 2)) = v;
    else *(float*)(con + (c >> 14)) = v;
}
// v with its sign flipped for a negated literal: c << 29 is bit 2 alone (a code's
// bits 0 and 1 are 0), and adding the top bit flips it
__device__ __forceinline__ float code_sign(uint32_t c, float v)
{
    return __uint_as_float((c << 29) + __float_as_uint(v));
}

// the two factors of a spin, written by its variable's thread
__device__ __forceinline__ void put_factors(unsigned char* fac, int rank, float sv)
{
    *(float2*)(fac + 8 * rank) = make_float2(1.0f - sv, 1.0f + sv);
}

// clauses [first, first + 64) of a wave: the codes are stored in whole groups
// of 64 clauses, so a wave with any clause loads all of its lanes'
template <int KK>
__device__ __forceinline__ void load_code(const uint32_t* code, int j, uint32_t (&c)[KK])
{
    unsigned at = (unsigned)j * (4 * KK);
    asm("" : "+v"(at));         // not kept in a register from stage to stage
    const uint32_t* p = (const uint32_t*)((const char*)code + at);
#pragma unroll
    for (int q = 0; q < KK; q++) c[q] = p[q];
}

// Clause phase of stage J; kn2 = 4^-k.  COUNT (J = 1): viol receives the number of this
// thread's clauses violated by the state whose factors are in LDS; pos has a
// bit per rank, s > 0, for the factors that are exactly 1.
template <int TT, int CPT, int VPT, int J, int KK, bool WIDE, bool COUNT>
__device__ __forceinline__ void reg_clauses(RegState<TT, CPT, VPT, KK>& R, const uint32_t* code, int m, float kn2,
                                            const unsigned char* fac, unsigned char* con, float hs,
                                            double h, double hnext, double floor, double& err,
                                            const unsigned long long* pos, int& viol)
{
    constexpr bool HOLD = RegState<TT, CPT, VPT, KK>::HOLD;
    const int tid = traj_tid<TT>();
    const int w0 = __builtin_amdgcn_readfirstlane(tid & ~63);
    uint32_t nx[KK];
    if constexpr (!HOLD) {
        if (w0 < m) load_code<KK>(code, tid, nx);
    }
#pragma unroll
    for (int u = 0; u < CPT; u++) {
        if (w0 + u * TT < m) {
            uint32_t c[KK];
            if constexpr (HOLD) {
#pragma unroll
                for (int q = 0; q < KK; q++) {
                    // an opaque value: what follows from a code is formed
                    // again in every stage, not kept in registers
                    asm("" : "+v"(R.code[u][q]));
                    c[q] = R.code[u][q];
                }
            } else {
                // the next clause's codes are loaded while this one is processed
#pragma unroll
                for (int q = 0; q < KK; q++) c[q] = nx[q];
                // (past the wave's last one: its first again, which keeps
                // the loads free of branches)
                if (u + 1 < CPT) load_code<KK>(code, tid + (w0 + (u + 1) * TT < m ? (u + 1) * TT : 0), nx);
            }
            float f[KK];
#pragma unroll
            for (int q = 0; q < KK; q++) f[q] = code_factor<WIDE>(fac, c[q]);
            // products of the factors of K_m left to right, without 2^-k: the
            // powers of two are exact wherever they are multiplied in
            float km = f[0];
#pragma unroll
            for (int q = 1; q < KK; q++) km *= f[q];
            if constexpr (COUNT) {
                bool sat = false, unsat = true;
#pragma unroll
                for (int q = 0; q < KK; q++) {
                    sat |= f[q] < 1.0f;
                    unsat &= f[q] > 1.0f;
                }
                if (!sat && !unsat) {
                    // a spin too small to move its factor, or NaN: its bit
                    // decides (the constants' bits are 0: false)
#pragma unroll
                    for (int q = 0; q < KK; q++) {
                        const uint32_t a = c[q] & (WIDE ? 0xFFFFu : 0x3FFFu);
                        const int rank = (int)(a >> 3);
                        const bool t = (pos[rank >> 6] >> (rank & 63)) & 1ull;
                        const bool neg = (a >> 2) & 1u;
                        sat |= neg ? !t : t;
                    }
                }
                viol += (!sat && tid + u * TT < m) ? 1 : 0;
            }
            float am;
            if constexpr (J == 1) am = R.xa[u];
            else am = stage_input<float, J>(R.xa[u], R.a1[u], R.a2[u], R.a3[u], R.a4[u], R.a5[u], hs);
            const float am_km = am * km;
            const float kj = am_km * km * kn2;
            if constexpr (J == 1) R.a1[u] = kj;
            else if constexpr (J == 2) R.a2[u] = kj;
            else if constexpr (J == 3) R.a3[u] = kj;
            else if constexpr (J == 4) R.a4[u] = kj;
            else if constexpr (J == 5) R.a5[u] = kj;
            else {
                float xv;
                double e;
                final_combination<float>(R.xa[u], R.a1[u], R.a3[u], R.a4[u], R.a5[u], kj, hs, h, hnext, floor, xv, e);
                R.a2[u] = xv;
                err = fmax(err, e);
            }
            // K_m 2^-k a_m and the factor 2 of every term
            const float r = am_km * (2.0f * kn2);
#pragma unroll
            for (int q = 0; q < KK; q++) {
                float p = 1.0f;
                bool first = true;
#pragma unroll
                for (int qq = 0; qq < KK; qq++) {
                    if (qq == q) continue;
                    p = first ? f[qq] : p * f[qq];
                    first = false;
                }
                code_store<WIDE>(con, c[q], code_sign(c[q], r * p));
            }
        }
        // one clause at a time: keeps the live registers to the state plus
        // one clause's temporaries (a wave alone overlaps its few clauses)
        if constexpr (TT > 64) __builtin_amdgcn_sched_barrier(0);
    }
}

// left-to-right sum of a group's entries for this lane (depth is uniform)
__device__ __forceinline__ float group_sum(const float* e, int depth)
{
    float sum = 0.0f;
    int i = 0;
    for (; i + 8 <= depth; i += 8, e += 8 * 64) {
        float t[8];
#pragma unroll
        for (int u = 0; u < 8; u++) t[u] = e[64 * u];
#pragma unroll
        for (int u = 0; u < 8; u++) sum += t[u];
    }
    if (depth & 4) {
        float t[4];
#pragma unroll
        for (int u = 0; u < 4; u++) t[u] = e[64 * u];
#pragma unroll
        for (int u = 0; u < 4; u++) sum += t[u];
        e += 4 * 64;
    }
    if (depth & 2) {
        const float t0 = e[0], t1 = e[64];
        sum += t0;
        sum += t1;
        e += 2 * 64;
    }
    if (depth & 1) sum += e[0];
    return sum;
}

// Var phase of stage J.  gb, gd: base entry and depth of the wave's groups
// (depth -1: the wave has no such group).
template <int TT, int CPT, int VPT, int J, int KK>
__device__ __forceinline__ void reg_vars(RegState<TT, CPT, VPT, KK>& R, const int (&gb)[VPT], const int (&gd)[VPT],
                                         unsigned char* fac, const unsigned char* con, float hs, double h,
                                         double hnext, double floor, double& err)
{
    const int tid = traj_tid<TT>();
#pragma unroll
    for (int v = 0; v < VPT; v++) {
        if (gd[v] >= 0) {
            const float kj = group_sum((const float*)con + gb[v] + (tid & 63), gd[v]);
            const float xi = R.xv[v];
            const int rank = tid + v * TT;
            if constexpr (J == 1) {
                R.v1[v] = kj;
                put_factors(fac, rank, stage_input<float, 2>(xi, kj, 0.f, 0.f, 0.f, 0.f, hs));
            } else if constexpr (J == 2) {
                R.v2[v] = kj;
                put_factors(fac, rank, stage_input<float, 3>(xi, R.v1[v], kj, 0.f, 0.f, 0.f, hs));
            } else if constexpr (J == 3) {
                R.v3[v] = kj;
                put_factors(fac, rank, stage_input<float, 4>(xi, R.v1[v], R.v2[v], kj, 0.f, 0.f, hs));
            } else if constexpr (J == 4) {
                R.v4[v] = kj;
                put_factors(fac, rank, stage_input<float, 5>(xi, R.v1[v], R.v2[v], R.v3[v], kj, 0.f, hs));
            } else if constexpr (J == 5) {
                R.v5[v] = kj;
                put_factors(fac, rank, stage_input<float, 6>(xi, R.v1[v], R.v2[v], R.v3[v], R.v4[v], kj, hs));
            } else {
                float xn;
                double e;
                final_combination<float>(xi, R.v1[v], R.v3[v], R.v4[v], R.v5[v], kj, hs, h, hnext, floor, xn, e);
                R.v2[v] = xn;
                err = fmax(err, e);
            }
        }
    }
}

// what else a trajectory keeps in LDS
template <int TT, int VPT>
struct alignas(16) RegShared {
    unsigned long long pos[(TT / 64) * VPT];
    double red[TT / 64];
    Control control;
    int redi[TT / 64];
    int traj;
};

template <int TT, int CPT, int VPT, int KK, bool WIDE>
__global__ __launch_bounds__(TT == 64 ? 64 * REG_WAVES : TT) void k_batch_reg(Params P)
{
    // per trajectory [factors: 2 per rank, TT * VPT ranks] [RegShared]
    // [contributions]; no other LDS, so the factors start at address 0
    extern __shared__ __attribute__((aligned(16))) unsigned char rlds[];
    using Shared = RegShared<TT, VPT>;
    const int tid = traj_tid<TT>();
    const int sub = TT == 64 ? uni((int)(threadIdx.x >> 6)) : 0;
    const int wave = TT == 64 ? 0 : uni(tid >> 6);
    unsigned char* fac = rlds + (TT == 64 ? sub * P.reg_lds : 0);
    Shared* sh = (Shared*)(fac + 8 * TT * VPT);
    unsigned char* con = fac + 8 * TT * VPT + sizeof(Shared);
    unsigned long long* pos = sh->pos;

    for (;;) {
        // the trajectory id is the same in every lane: reading it as a
        // scalar lets the descriptor and the instance's base pointers live
        // in scalar registers, leaving the vector registers to the state
        int slot = 0;
        if constexpr (TT == 64) {
            if (tid == 0) slot = atomicAdd(P.queue, 1);
        } else {
            if (tid == 0) sh->traj = atomicAdd(P.queue, 1);
            __syncthreads();
            slot = sh->traj;
            __syncthreads();
        }
        slot = __builtin_amdgcn_readfirstlane(slot);
        if (slot >= P.ntraj) break;
        const int tr = __builtin_amdgcn_readfirstlane(P.order[slot]);
        const Desc d = P.desc[tr];
        TrajCtrl* cp = P.ctrl + tr;
        if (cp->status != RUNNING) continue;    // uniform: every thread reads the same word

        const int n = uni(d.n), m = uni(d.m);
        const uint32_t* code = P.rcode + uni(d.rcode_off);
        const int* group = P.rgroup + uni(d.rgroup_off);     // base and depth per 64 ranks
        const int* vmap = P.rvmap + uni(d.rvmap_off);        // rank -> variable
        const int ngroups = uni(d.ngroups);
        const float kn2 = uni(d.knorm * d.knorm);       // 4^-k
        double t = cp->t, h = cp->h, hnext = cp->hnext, hdid = cp->hdid, errmax_last = cp->errmax;
        long long steps = cp->steps, attempts = cp->attempts, rhscount = cp->rhscount;
        int parity = cp->parity, min_viol = cp->min_viol, viol = cp->viol;
        int status = RUNNING;
        int sat_step = cp->sat_step;
        double sat_time = cp->sat_time;
        int done_in_chunk = 0;

        RegState<TT, CPT, VPT, KK> R;
        int gb[VPT], gd[VPT];
        {
            const float* x = (parity ? P.xb : P.xa) + d.state_off;
#pragma unroll
            for (int u = 0; u < CPT; u++) {
                const int j = tid + u * TT;
                R.xa[u] = j < m ? x[n + j] : 0.f;
                R.a1[u] = R.a2[u] = R.a3[u] = R.a4[u] = R.a5[u] = 0.f;
                if constexpr (RegState<TT, CPT, VPT, KK>::HOLD) {
                    if (wave * 64 + u * TT < m) load_code<KK>(code, j, R.code[u]);
                }
            }
#pragma unroll
            for (int v = 0; v < VPT; v++) {
                const int g = wave + v * (TT / 64), rank = tid + v * TT;
                gb[v] = g < ngroups ? __builtin_amdgcn_readfirstlane(group[2 * g]) : 0;
                gd[v] = g < ngroups ? __builtin_amdgcn_readfirstlane(group[2 * g + 1]) : -1;
                // ranks n and n + 1 are the constants
                R.xv[v] = rank < n ? x[vmap[rank]] : (rank == n ? -1.0f : 0.0f);
                R.v1[v] = R.v2[v] = R.v3[v] = R.v4[v] = R.v5[v] = 0.f;
            }
        }
        for (int i = tid; i < d.ncontrib; i += TT) ((float*)con)[i] = -0.0f;
        bool count = false;       // the state is a newly accepted one whose violations are due

        while (true) {
            // ---- stage 1 at x: its factors, and where they do not tell, s > 0
#pragma unroll
            for (int v = 0; v < VPT; v++) {
                const int rank = tid + v * TT;
                if (gd[v] >= 0) {
                    put_factors(fac, rank, R.xv[v]);
                    // constants: positive literals that read as false
                    const unsigned long long b = __ballot(rank < n && R.xv[v] > 0.0f);
                    if ((tid & 63) == 0) pos[rank >> 6] = b;
                }
            }
            traj_sync<TT>();
            const double h_at1 = h;
            double err_local = 0.0;
            int cnt = 0;
            if (count) {
                reg_clauses<TT, CPT, VPT, 1, KK, WIDE, true>(R, code, m, kn2, fac, con, (float)h_at1, h_at1,
                                                             hnext, P.floor, err_local, pos, cnt);
                viol = traj_sum<TT>(cnt, sh->redi);
                count = false;
                if (viol < min_viol) min_viol = viol;
                if (viol == 0) {
                    status = SOLVED;
                    sat_step = (int)steps;
                    sat_time = t;
                }
                if (status == RUNNING && steps >= P.max_steps) status = BUDGET;
                if (status == RUNNING && t >= P.max_time) status = MAXTIME;
                if (status != RUNNING || done_in_chunk >= P.chunk_steps) break;
            } else {
                reg_clauses<TT, CPT, VPT, 1, KK, WIDE, false>(R, code, m, kn2, fac, con, (float)h_at1, h_at1,
                                                              hnext, P.floor, err_local, pos, cnt);
                traj_sync<TT>();
            }
            reg_vars<TT, CPT, VPT, 1, KK>(R, gb, gd, fac, con, (float)h, h, hnext, P.floor, err_local);
            traj_sync<TT>();
            bool accepted = false;
            bool had_stage1 = true;
            while (true) {
                const float hs = (float)h;
                err_local = 0.0;
#define ASAT_REG_STAGE(J)                                                                                             \
    reg_clauses<TT, CPT, VPT, J, KK, WIDE, false>(R, code, m, kn2, fac, con, hs, h, hnext, P.floor, err_local, \
                                                  pos, cnt);                                                          \
    traj_sync<TT>();                                                                                                  \
    reg_vars<TT, CPT, VPT, J, KK>(R, gb, gd, fac, con, hs, h, hnext, P.floor, err_local);
                ASAT_REG_STAGE(2)
                traj_sync<TT>();
                ASAT_REG_STAGE(3)
                traj_sync<TT>();
                ASAT_REG_STAGE(4)
                traj_sync<TT>();
                ASAT_REG_STAGE(5)
                traj_sync<TT>();
                ASAT_REG_STAGE(6)
#undef ASAT_REG_STAGE
                // ---------------- error norm + control (FP64), uniform in every thread
                const Control ctl = traj_control<TT>(err_local, P.eps, sh->red, &sh->control);
                const double errmax = ctl.errmax;
                errmax_last = errmax;
                attempts += 1;
                rhscount += had_stage1 ? 6 : 5;
                had_stage1 = false;
                if (errmax <= 1.0) {
                    double hn = errmax > TabD::ERRCON ? TabD::SAFETY * h * ctl.power : 5.0 * h;
                    hdid = h;
                    t += h;
                    steps += 1;
                    hnext = hn;
                    h = hn;
                    accepted = true;
                    break;
                }
                double htemp = TabD::SAFETY * h * ctl.power;
                double hn = h >= 0.0 ? fmax(htemp, TabD::HFACTOR * h) : fmin(htemp, TabD::HFACTOR * h);
                h = hn;
                if (t + hn == t) {
                    status = UNDERFLOW_;
                    break;
                }
                // retry: stage-2 spin input from x, k1 and the reduced h
                const float hs2 = (float)h;
#pragma unroll
                for (int v = 0; v < VPT; v++)
                    if (gd[v] >= 0)
                        put_factors(fac, tid + v * TT,
                                    stage_input<float, 2>(R.xv[v], R.v1[v], 0.f, 0.f, 0.f, 0.f, hs2));
                traj_sync<TT>();
            }
            if (!accepted) break;
            // accept: x <- x_new (held in the k2 registers)
#pragma unroll
            for (int u = 0; u < CPT; u++) R.xa[u] = R.a2[u];
#pragma unroll
            for (int v = 0; v < VPT; v++) R.xv[v] = R.v2[v];
            parity ^= 1;
            done_in_chunk += 1;
            count = steps % P.check_every == 0 || steps >= P.max_steps;
            if (!count) {
                if (t >= P.max_time) status = MAXTIME;
                if (status != RUNNING || done_in_chunk >= P.chunk_steps) break;
            }
        }
        // the state after the last accepted step goes to the parity buffer it names
        {
            float* x = (parity ? P.xb : P.xa) + d.state_off;
#pragma unroll
            for (int u = 0; u < CPT; u++) {
                const int j = tid + u * TT;
                if (j < m) x[n + j] = R.xa[u];
            }
#pragma unroll
            for (int v = 0; v < VPT; v++) {
                const int rank = tid + v * TT;
                if (rank < n) x[vmap[rank]] = R.xv[v];
            }
        }
        if (tid == 0) {
            cp->t = t; cp->h = h; cp->hnext = hnext; cp->hdid = hdid; cp->errmax = errmax_last;
            cp->steps = steps; cp->attempts = attempts; cp->rhscount = rhscount;
            cp->parity = parity; cp->status = status; cp->min_viol = min_viol; cp->viol = viol;
            cp->sat_step = sat_step; cp->sat_time = sat_time;
        }
        traj_sync<TT>();
    }
}

// ---------------------------------------------------------------------------
// Clause-chunked variant, for instances whose contributions do not fit in LDS.
// Clauses are taken in chunks whose KK terms per clause do.  Per chunk:
//   clause phase: each thread's clauses leave their terms in LDS, term q of
//     clause jl at q * chunk + jl (lanes side by side: no bank conflicts)
//   var phase: the chunk's variables, 64 at a time and ranked by their number of
//     occurrences in it, add the terms that their index list names to the
//     variable's running sum in LDS
// Chunks follow the clause order, so every variable's terms are added in the
// reference's order.  After the last chunk each variable's stage combination
// (state and derivatives of both kinds in global scratch) puts the next
// stage's factors 1 - s and 1 + s into LDS.
//
// It is bound by memory: per slot and stage a 2-byte code and a 2-byte term
// index, per clause the stage's derivatives (27 floats an attempt), about 60 %
// less than 4-byte codes and 8-byte records, from which each variable formed
// its terms itself (three LDS reads per slot and uncoalesced records).
// 512 ragged instances (N in [50, 5000], 3- and 4-SAT) for 20 steps, their
// smallest quarter in registers: 89 -> 19 ms; the largest quarter (M up to
// 60 000) 21.9 -> 4.8 us per trajectory and attempt, on 128 of 256 CUs.
template <int KK, int J, bool COUNT>
__device__ __forceinline__ void chunk_clauses(const uint2* code, const float* x, float* const (&kb)[5], float* xn,
                                              int c0, int cn, int cs, int n, float knorm, float knorm2,
                                              const float* fac, float* term, float hs, double h, double hnext,
                                              double floor, double& err, int& viol)
{
    constexpr int U = 2;                     // clauses whose loads are in flight together
    const int BS = (int)blockDim.x;
    for (int jb = (int)threadIdx.x; jb < cn; jb += U * BS) {
        uint2 c[U];
        float xa[U], a1[U], a2[U], a3[U], a4[U], a5[U];
#pragma unroll
        for (int u = 0; u < U; u++) {
            const int jl = jb + u * BS;
            xa[u] = a1[u] = a2[u] = a3[u] = a4[u] = a5[u] = 0.f;
            c[u] = make_uint2(0u, 0u);
            if (jl < cn) {
                c[u] = code[c0 + jl];
                const int ai = n + c0 + jl;
                xa[u] = x[ai];
                if constexpr (J > 1) a1[u] = kb[0][ai];
                if constexpr (J > 2) a2[u] = kb[1][ai];
                if constexpr (J > 3) a3[u] = kb[2][ai];
                if constexpr (J > 4) a4[u] = kb[3][ai];
                if constexpr (J > 5) a5[u] = kb[4][ai];
            }
        }
#pragma unroll
        for (int u = 0; u < U; u++) {
            const int jl = jb + u * BS;
            if (jl >= cn) break;
            const uint32_t w[4] = {c[u].x & 0xFFFFu, c[u].x >> 16, c[u].y & 0xFFFFu, c[u].y >> 16};
            float f[KK];
            float km = knorm;
#pragma unroll
            for (int q = 0; q < KK; q++) {
                f[q] = fac[w[q]];
                km *= f[q];
            }
            if constexpr (COUNT) {
                bool sat = false, unsat = true;
#pragma unroll
                for (int q = 0; q < KK; q++) {
                    sat |= f[q] < 1.0f;
                    unsat &= f[q] > 1.0f;
                }
                if (!sat && !unsat) {
                    // a spin too small to move its factor, or NaN; the
                    // constants (variables n and n + 1) are false
#pragma unroll
                    for (int q = 0; q < KK; q++) {
                        const int v = (int)(w[q] >> 1);
                        if (v >= n) continue;
                        const bool t = x[v] > 0.0f;
                        sat |= (w[q] & 1u) ? !t : t;
                    }
                }
                viol += sat ? 0 : 1;
            }
            float am;
            if constexpr (J == 1) am = xa[u];
            else am = stage_input<float, J>(xa[u], a1[u], a2[u], a3[u], a4[u], a5[u], hs);
            const float kj = am * km * km;
            const int ai = n + c0 + jl;
            if constexpr (J < 6) {
                kb[J - 1][ai] = kj;
            } else {
                float xv;
                double e;
                final_combination<float>(xa[u], a1[u], a3[u], a4[u], a5[u], kj, hs, h, hnext, floor, xv, e);
                xn[ai] = xv;
                err = fmax(err, e);
            }
            const float r = km * knorm2 * am;
#pragma unroll
            for (int q = 0; q < KK; q++) {
                float p = 1.0f;
                bool first = true;
#pragma unroll
                for (int qq = 0; qq < KK; qq++) {
                    if (qq == q) continue;
                    p = first ? f[qq] : p * f[qq];
                    first = false;
                }
                term[q * cs + jl] = __uint_as_float((w[q] << 31) ^ __float_as_uint(r * p));
            }
        }
    }
}

// the chunk's variables: groups [g0, g1) of 64, a wave each
__device__ __forceinline__ void chunk_vars(const int2* group, const uint16_t* perm, const uint32_t* rec, int g0,
                                           int g1, const float* term, float* sums)
{
    const int lane = (int)(threadIdx.x & 63);
    const int wave = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6)), nw = (int)(blockDim.x >> 6);
    for (int g = g0 + wave; g < g1; g += nw) {
        const int2 gd = group[g];            // first word, words per lane (two entries each)
        const int v = perm[g * 64 + lane];
        const uint32_t* r = rec + gd.x + lane;
        float sum = sums[v];
        int i = 0;
        for (; i + 4 <= gd.y; i += 4) {
            uint32_t w[4];
            float t[8];
#pragma unroll
            for (int u = 0; u < 4; u++) w[u] = r[64 * (i + u)];
#pragma unroll
            for (int u = 0; u < 4; u++) {
                t[2 * u] = term[w[u] & 0xFFFFu];
                t[2 * u + 1] = term[w[u] >> 16];
            }
#pragma unroll
            for (int u = 0; u < 8; u++) sum += t[u];
        }
        for (; i < gd.y; i++) {
            const uint32_t w = r[64 * i];
            const float t0 = term[w & 0xFFFFu], t1 = term[w >> 16];
            sum += t0;
            sum += t1;
        }
        sums[v] = sum;
    }
}

template <int BS>
__global__ __launch_bounds__(BS) void k_batch_chunk(Params P)
{
    // [factors: fac_ranks pairs] [running sums: fac_ranks] [terms, then 0]
    extern __shared__ __attribute__((aligned(16))) float clds[];
    __shared__ double red[BS / 64];
    __shared__ int redi[BS / 64];
    __shared__ Control s_control;
    __shared__ int s_traj;
    float* fac = clds;
    float* sums = clds + 2 * P.fac_ranks;
    float* term = clds + 3 * P.fac_ranks;
    float* scratch = P.scratch + (long long)blockIdx.x * P.scratch_per_wg;
    float* const kb[5] = {scratch, scratch + P.scratch_stride, scratch + 2 * P.scratch_stride,
                          scratch + 3 * P.scratch_stride, scratch + 4 * P.scratch_stride};
    const int tid = threadIdx.x;

    for (;;) {
        if (tid == 0) s_traj = atomicAdd(P.queue, 1);
        __syncthreads();
        const int slot = __builtin_amdgcn_readfirstlane(s_traj);
        __syncthreads();
        if (slot >= P.ntraj) break;
        const int tr = __builtin_amdgcn_readfirstlane(P.order[slot]);
        const Desc d = P.desc[tr];
        TrajCtrl* cp = P.ctrl + tr;
        if (cp->status != RUNNING) continue;    // uniform: every thread reads the same word

        const int n = uni(d.n), m = uni(d.m), cs = uni(d.chunk), nc = uni(d.nchunks);
        const uint2* code = P.ccode + uni(d.ccode_off);
        const int2* group = P.cgroup + uni(d.cgroup_off);
        const uint16_t* perm = P.cperm + uni(d.cgroup_off) * 64;
        const uint32_t* rec = P.crec + uni(d.crec_off);
        const int* cstart = P.cstart + uni(d.cstart_off);
        const float knorm = uni(d.knorm), knorm2 = 2.0f * knorm;
        const int klen = uni(d.k);
        double t = cp->t, h = cp->h, hnext = cp->hnext, hdid = cp->hdid, errmax_last = cp->errmax;
        long long steps = cp->steps, attempts = cp->attempts, rhscount = cp->rhscount;
        int parity = cp->parity, min_viol = cp->min_viol, viol = cp->viol;
        int status = RUNNING;
        int sat_step = cp->sat_step;
        double sat_time = cp->sat_time;
        int done_in_chunk = 0;
        bool count = false;       // the state is a newly accepted one whose violations are due
        float* x = nullptr;
        float* xn = nullptr;

        auto put = [&](int i, float sv) { *(float2*)(fac + 2 * i) = make_float2(1.0f - sv, 1.0f + sv); };
        if (tid == 0) {
            put(n, -1.0f);        // a padding literal of a short clause: factor 2
            put(n + 1, 0.0f);     // a literal beyond k: factor 1
            term[P.chunk_terms] = 0.0f;   // entries that fill up a list
        }
        // one stage: every chunk's clauses and variables, then the variables'
        // stage combination; with COUNT the violated clauses first
        auto stage = [&](auto jc, auto cc, float hs, double& err, int& cnt) {
            constexpr int J = decltype(jc)::value;
            constexpr bool COUNT = decltype(cc)::value;
            for (int i = tid; i <= n; i += BS) sums[i] = 0.0f;
            for (int c = 0; c < nc; c++) {
                const int c0 = c * cs, cn = min(cs, m - c0);
                if (klen <= 3)
                    chunk_clauses<3, J, COUNT>(code, x, kb, xn, c0, cn, cs, n, knorm, knorm2, fac, term, hs, h, hnext,
                                               P.floor, err, cnt);
                else
                    chunk_clauses<4, J, COUNT>(code, x, kb, xn, c0, cn, cs, n, knorm, knorm2, fac, term, hs, h, hnext,
                                               P.floor, err, cnt);
                __syncthreads();
                chunk_vars(group, perm, rec, cstart[c], cstart[c + 1], term, sums);
                __syncthreads();
            }
            for (int i = tid; i < n; i += BS) {
                const float kj = sums[i], xi = x[i];
                if constexpr (J < 6) kb[J - 1][i] = kj;
                if constexpr (J == 1) put(i, stage_input<float, 2>(xi, kj, 0.f, 0.f, 0.f, 0.f, hs));
                else if constexpr (J == 2) put(i, stage_input<float, 3>(xi, kb[0][i], kj, 0.f, 0.f, 0.f, hs));
                else if constexpr (J == 3) put(i, stage_input<float, 4>(xi, kb[0][i], kb[1][i], kj, 0.f, 0.f, hs));
                else if constexpr (J == 4)
                    put(i, stage_input<float, 5>(xi, kb[0][i], kb[1][i], kb[2][i], kj, 0.f, hs));
                else if constexpr (J == 5)
                    put(i, stage_input<float, 6>(xi, kb[0][i], kb[1][i], kb[2][i], kb[3][i], kj, hs));
                else {
                    float xv;
                    double e;
                    final_combination<float>(xi, kb[0][i], kb[2][i], kb[3][i], kb[4][i], kj, hs, h, hnext, P.floor, xv,
                                             e);
                    xn[i] = xv;
                    err = fmax(err, e);
                }
            }
            __syncthreads();
        };
        using std::integral_constant;
        using NoCount = integral_constant<bool, false>;

        while (true) {
            x = (parity ? P.xb : P.xa) + d.state_off;
            xn = (parity ? P.xa : P.xb) + d.state_off;
            // ---- stage 1 at x
            for (int i = tid; i < n; i += BS) put(i, x[i]);
            __syncthreads();
            double err_local = 0.0;
            int cnt = 0;
            if (count) {
                stage(integral_constant<int, 1>{}, integral_constant<bool, true>{}, (float)h, err_local, cnt);
                viol = block_sum_all<BS>(cnt, redi);
                count = false;
                if (viol < min_viol) min_viol = viol;
                if (viol == 0) {
                    status = SOLVED;
                    sat_step = (int)steps;
                    sat_time = t;
                }
                if (status == RUNNING && steps >= P.max_steps) status = BUDGET;
                if (status == RUNNING && t >= P.max_time) status = MAXTIME;
                if (status != RUNNING || done_in_chunk >= P.chunk_steps) break;
            } else {
                stage(integral_constant<int, 1>{}, NoCount{}, (float)h, err_local, cnt);
            }
            bool accepted = false;
            bool had_stage1 = true;
            while (true) {
                const float hs = (float)h;
                err_local = 0.0;
                stage(integral_constant<int, 2>{}, NoCount{}, hs, err_local, cnt);
                stage(integral_constant<int, 3>{}, NoCount{}, hs, err_local, cnt);
                stage(integral_constant<int, 4>{}, NoCount{}, hs, err_local, cnt);
                stage(integral_constant<int, 5>{}, NoCount{}, hs, err_local, cnt);
                stage(integral_constant<int, 6>{}, NoCount{}, hs, err_local, cnt);
                const Control ctl = traj_control<BS>(err_local, P.eps, red, &s_control);
                const double errmax = ctl.errmax;
                errmax_last = errmax;
                attempts += 1;
                rhscount += had_stage1 ? 6 : 5;
                had_stage1 = false;
                if (errmax <= 1.0) {
                    double hn = errmax > TabD::ERRCON ? TabD::SAFETY * h * ctl.power : 5.0 * h;
                    hdid = h;
                    t += h;
                    steps += 1;
                    hnext = hn;
                    h = hn;
                    accepted = true;
                    break;
                }
                double htemp = TabD::SAFETY * h * ctl.power;
                double hn = h >= 0.0 ? fmax(htemp, TabD::HFACTOR * h) : fmin(htemp, TabD::HFACTOR * h);
                h = hn;
                if (t + hn == t) {
                    status = UNDERFLOW_;
                    break;
                }
                // retry: stage-2 spin input from x, k1 and the reduced h
                const float hs2 = (float)h;
                for (int i = tid; i < n; i += BS)
                    put(i, stage_input<float, 2>(x[i], kb[0][i], 0.f, 0.f, 0.f, 0.f, hs2));
                __syncthreads();
            }
            if (!accepted) break;
            parity ^= 1;
            done_in_chunk += 1;
            count = steps % P.check_every == 0 || steps >= P.max_steps;
            if (!count) {
                if (t >= P.max_time) status = MAXTIME;
                if (status != RUNNING || done_in_chunk >= P.chunk_steps) break;
            }
        }
        if (tid == 0) {
            cp->t = t; cp->h = h; cp->hnext = hnext; cp->hdid = hdid; cp->errmax = errmax_last;
            cp->steps = steps; cp->attempts = attempts; cp->rhscount = rhscount;
            cp->parity = parity; cp->status = status; cp->min_viol = min_viol; cp->viol = viol;
            cp->sat_step = sat_step; cp->sat_time = sat_time;
        }
        __syncthreads();
    }
}

// Current states of trajectories first .. first + gridDim.y - 1, packed as they
// lie in the state buffers (each from the buffer its parity names)
__global__ __launch_bounds__(256) void k_pack_states(const Desc* desc, const TrajCtrl* ctrl, const float* xa,
                                                     const float* xb, int first, float* out)
{
    const int tr = first + (int)blockIdx.y;
    const Desc& d = desc[tr];
    const float* x = (ctrl[tr].parity ? xb : xa) + d.state_off;
    float* o = out + (d.state_off - desc[first].state_off);
    for (int i = (int)(blockIdx.x * 256 + threadIdx.x); i < d.n + d.m; i += (int)gridDim.x * 256) o[i] = x[i];
}

__global__ void k_reset_queue(int* q)
{
    if (threadIdx.x == 0 && blockIdx.x == 0) *q = 0;
}

static inline long long round_up_ll(long long a, long long b) { return (a + b - 1) / b * b; }

// ---------------------------------------------------------------------------
// host side
// ---------------------------------------------------------------------------
struct Instance {
    int n = 0, m = 0, k = 0, nslots = 0;
    std::vector<uint32_t> code;   // m*k
    std::vector<int> rowptr;      // n+1
    std::vector<float> pub0;      // n+m
};

// Layout of the register kernel for one instance: variables ranked by falling
// number of occurrences, contributions in groups of 64 ranks with the entries of
// one index side by side, codes padded to whole groups of 64 clauses and to kk
// literals (see k_batch_reg).
struct RegLayout {
    std::vector<int> rank;      // variable -> rank
    std::vector<int> vmap;      // rank -> variable
    std::vector<int> group;     // base and depth per group of 64 ranks (two constant ranks at the end)
    int ngroups = 0, ncontrib = 0;
};

static void reg_layout(const Instance& I, RegLayout& L)
{
    const int n = I.n;
    int top = 0;
    for (int i = 0; i < n; i++) top = std::max(top, I.rowptr[i + 1] - I.rowptr[i]);
    std::vector<int> at((size_t)top + 2, 0);
    for (int i = 0; i < n; i++) at[(size_t)(top - (I.rowptr[i + 1] - I.rowptr[i])) + 1]++;
    for (int g = 0; g <= top; g++) at[(size_t)g + 1] += at[(size_t)g];
    L.rank.resize((size_t)n);
    L.vmap.resize((size_t)n);
    for (int i = 0; i < n; i++) {
        const int r = at[(size_t)(top - (I.rowptr[i + 1] - I.rowptr[i]))]++;
        L.rank[i] = r;
        L.vmap[r] = i;
    }
    L.ngroups = ceil_div(n + 2, 64);
    L.group.resize((size_t)2 * L.ngroups);
    int base = 0;
    for (int g = 0; g < L.ngroups; g++) {
        const int v = 64 * g < n ? L.vmap[64 * g] : -1;      // the group's first rank occurs most
        const int depth = v >= 0 ? I.rowptr[v + 1] - I.rowptr[v] : 0;
        L.group[2 * g] = base;
        L.group[2 * g + 1] = depth;
        base += 64 * depth;
    }
    L.ncontrib = base;
}

// the codes, rcode_len(I, kk) words; entry L.ncontrib is the one nothing reads
static long long rcode_len(const Instance& I, int kk) { return round_up_ll(I.m, 64) * kk; }
static void reg_codes(const Instance& I, const RegLayout& L, int kk, uint32_t* out)
{
    const uint32_t none = (uint32_t)L.ncontrib << 16;
    const uint32_t pad = none | (8u * (uint32_t)I.n), absent = none | (8u * (uint32_t)(I.n + 1));
    // per variable: the contribution entry of position 0 of the instance's var-major
    // order, of which each position is 64 entries further on, and 8 times its rank
    struct Place { uint32_t entry, rank8; };
    std::vector<Place> place((size_t)I.n);
    for (int v = 0; v < I.n; v++) {
        const int r = L.rank[v];
        place[(size_t)v] = {(uint32_t)(L.group[2 * (r / 64)] + r % 64 - 64 * I.rowptr[v]), 8u * (uint32_t)r};
    }
    for (int j = 0; j < I.m; j++) {
        const uint32_t* c = I.code.data() + (size_t)j * I.k;
        uint32_t* o = out + (size_t)j * kk;
        for (int q = 0; q < I.k; q++) {
            const int v = (int)(c[q] >> 19) - 1;
            o[q] = v < 0 ? pad
                         : (place[(size_t)v].entry + 64 * (c[q] & 0x3FFFFu)) << 16 | place[(size_t)v].rank8 |
                               ((c[q] >> 18) & 1u) << 2;
        }
        for (int q = I.k; q < kk; q++) o[q] = absent;
    }
    for (long long s = (long long)I.m * kk; s < rcode_len(I, kk); s++) out[s] = absent;
}

// Layout of the chunked kernel for one instance (see k_batch_chunk): chunks of
// cs clauses; per chunk its variables with any occurrence, ranked by their number
// and 64 to a group, each with the indices of its terms in clause order, two
// per word; missing entries and lanes name entry `zero` and variable n.
struct ChunkLayout {
    int nchunks = 0, cs = 0;
    std::vector<uint2> code;
    std::vector<int2> group;
    std::vector<uint16_t> perm;
    std::vector<uint32_t> rec;
    std::vector<int> start;
};

static void chunk_layout(const Instance& I, int max_cs, int zero, ChunkLayout& L)
{
    const int n = I.n, m = I.m, k = I.k;
    L.nchunks = ceil_div(m, max_cs);
    L.cs = std::min(max_cs, (int)round_up_ll(ceil_div(m, L.nchunks), 64));
    L.nchunks = ceil_div(m, L.cs);
    L.code.resize((size_t)m);
    std::vector<int> cnt((size_t)n), slot((size_t)n);
    std::vector<int> vars, at;
    for (int c = 0; c < L.nchunks; c++) {
        const int c0 = c * L.cs, c1 = std::min(m, c0 + L.cs);
        std::fill(cnt.begin(), cnt.end(), 0);
        for (int j = c0; j < c1; j++) {
            uint32_t w[4];
            for (int q = 0; q < 4; q++) {
                w[q] = 2u * (uint32_t)(n + 1);
                if (q >= k) continue;
                const uint32_t code = I.code[(size_t)j * k + q];
                const int v = (int)(code >> 19) - 1;
                w[q] = v < 0 ? 2u * (uint32_t)n : 2u * (uint32_t)v + ((code >> 18) & 1u);
                if (v >= 0) cnt[v]++;
            }
            L.code[j] = make_uint2(w[0] | (w[1] << 16), w[2] | (w[3] << 16));
        }
        // variables by falling count, stable
        int top = 0;
        for (int v = 0; v < n; v++) top = std::max(top, cnt[v]);
        at.assign((size_t)top + 2, 0);
        int used = 0;
        for (int v = 0; v < n; v++)
            if (cnt[v]) { at[(size_t)(top - cnt[v]) + 1]++; used++; }
        for (int g = 0; g <= top; g++) at[(size_t)g + 1] += at[(size_t)g];
        vars.resize((size_t)used);
        for (int v = 0; v < n; v++)
            if (cnt[v]) {
                const int r = at[(size_t)(top - cnt[v])]++;
                vars[r] = v;
                slot[v] = r;
            }
        const int g0 = (int)L.group.size(), ng = ceil_div(used, 64);
        L.start.push_back(g0);
        for (int g = 0; g < ng; g++) {
            const int words = (cnt[vars[(size_t)64 * g]] + 1) / 2;
            L.group.push_back(make_int2((int)L.rec.size(), words));
            for (int l = 0; l < 64; l++)
                L.perm.push_back((uint16_t)(64 * g + l < used ? vars[(size_t)(64 * g + l)] : n));
            L.rec.resize(L.rec.size() + (size_t)64 * words, (uint32_t)zero | ((uint32_t)zero << 16));
        }
        std::fill(cnt.begin(), cnt.end(), 0);
        for (int j = c0; j < c1; j++)
            for (int q = 0; q < k; q++) {
                const int v = (int)(I.code[(size_t)j * k + q] >> 19) - 1;
                if (v < 0) continue;
                const int r = slot[v], e = cnt[v]++;
                uint32_t& w = L.rec[(size_t)L.group[(size_t)g0 + r / 64].x + (size_t)64 * (e / 2) + r % 64];
                const uint32_t idx = (uint32_t)(q * L.cs + (j - c0));
                w = (e & 1) ? (w & 0xFFFFu) | (idx << 16) : (w & 0xFFFF0000u) | idx;
            }
    }
    L.start.push_back((int)L.group.size());
}

struct Bucket {
    std::vector<int> ids;          // trajectory ids, largest first
    int block = 0;                 // workgroup size (256/512/1024), 0 = autotune
    int lds = -1;                  // contributions in LDS (1) or global scratch (0); 2: register-
                                   // resident kernel (contributions in LDS); 3: clause-chunked
                                   // (no contribution array); -1 = auto
    bool chunked = false;          // the clause-chunked layout is built for this bucket's instances
    int chunk_terms = 0;           // clause-chunked mode: term entries in LDS
    const struct RegVariant* reg = nullptr;   // register kernel: its variant
    int kk = 0;                    // register kernel: literals per clause (3 or 4)
    int ncontrib = 0;              // register kernel: contribution entries of the largest instance
    int grid = 0;
    int maxn = 0, maxm = 0, maxl = 0;
    int sp_stride = 0;
    long long scratch_stride = 0, scratch_per_wg = 0;
    size_t lds_bytes = 0;
    bool lds_fits = false;         // contributions of k_batch fit in LDS
    int* d_order = nullptr;
    int* d_queue = nullptr;
    float* d_scratch = nullptr;
    double tuned_us = -1.0;        // autotune: microseconds per trajectory-attempt
    void free_dev()
    {
        (void)hipFree(d_order); (void)hipFree(d_queue); (void)hipFree(d_scratch);
        d_order = nullptr; d_queue = nullptr; d_scratch = nullptr;
    }
};

struct Batch {
    std::vector<Instance> inst;
    double eps = 1e-6;
    double floor = 1e-20;
    double max_time = 1e300;
    long long max_steps = 10000;
    int chunk_steps = 256;
    int check_every = 1;
    int force_block = 0;           // 0: autotune per bucket
    int force_lds = -1;            // -1: auto
    int force_chunk = 0;           // clause-chunked mode: clauses per chunk, 0 = as large as LDS allows
    int nbuckets_req = 4;
    bool prepared = false;
    std::vector<Bucket> buckets;
    // device
    Desc* d_desc = nullptr;
    uint32_t* d_code = nullptr;
    uint32_t* d_rcode = nullptr;
    int *d_rgroup = nullptr, *d_rvmap = nullptr;
    uint2* d_ccode = nullptr;
    int2* d_cgroup = nullptr;
    uint16_t* d_cperm = nullptr;
    uint32_t* d_crec = nullptr;
    int* d_cstart = nullptr;
    int* d_rowptr = nullptr;
    float* d_xa = nullptr;
    float* d_xb = nullptr;
    TrajCtrl* d_ctrl = nullptr;
    std::vector<TrajCtrl> h_ctrl, h_ctrl0;
    float* d_x0 = nullptr;          // start states
    long long state_total = 0;      // floats of a state buffer
    std::vector<long long> state_off;
    // states on their way to the host, see get_state.  run() holds the lock over its
    // capture and over each launch with what follows it up to the control
    // blocks' copy, so a state read from another thread is the one of the latest
    // finished launch; readers counts the threads that wait for it
    std::mutex win_lock;
    std::atomic<int> readers{0};
    float *d_win = nullptr, *h_win = nullptr;
    int win_first = 0, win_last = 0;   // trajectories whose current states h_win holds
    int last_state = -1;               // trajectory of the latest get_state since the states changed
    void drop_window() { win_first = win_last = 0; last_state = -1; }
    // the lock for a launch; waiting readers go first (a mutex alone would give it
    // back to the thread that has just released it)
    std::unique_lock<std::mutex> launch_lock()
    {
        while (readers.load() > 0) std::this_thread::yield();
        return std::unique_lock<std::mutex>(win_lock);
    }
    hipStream_t stream = nullptr;
    hipStream_t side[3] = {nullptr, nullptr, nullptr};   // further buckets' launches, see run
    int cus = 0;
    size_t lds_limit = 0;
    // results
    std::vector<double> solved_wall_ms;
    double run_ms = 0.0;
    int chunks_run = 0;

    void free_dev()
    {
        (void)hipFree(d_desc); (void)hipFree(d_code); (void)hipFree(d_rowptr); (void)hipFree(d_xa);
        (void)hipFree(d_xb); (void)hipFree(d_ctrl); (void)hipFree(d_x0);
        d_x0 = nullptr;
        for (void* q : {(void*)d_rcode, (void*)d_rgroup, (void*)d_rvmap, (void*)d_ccode, (void*)d_cgroup,
                        (void*)d_cperm, (void*)d_crec, (void*)d_cstart})
            (void)hipFree(q);
        d_rcode = d_crec = nullptr; d_rgroup = d_rvmap = d_cstart = nullptr;
        d_ccode = nullptr; d_cgroup = nullptr; d_cperm = nullptr;
        d_desc = nullptr; d_code = nullptr; d_rowptr = nullptr; d_xa = d_xb = nullptr; d_ctrl = nullptr;
        for (auto& b : buckets) b.free_dev();
    }
    ~Batch()
    {
        free_dev();
        (void)hipFree(d_win);
        if (h_win) (void)hipHostFree(h_win);
        for (hipStream_t st : side)
            if (st) (void)hipStreamDestroy(st);
        if (stream) (void)hipStreamDestroy(stream);
    }
};

// build one instance: SatProblem::AddClauses semantics, clause matrix padded to
// K, contributions numbered in var-major slot order
static void build_instance(const int* lits, const int* lens, int nclauses, Instance& I)
{
    require(nclauses > 0 && lits && lens, ASAT_ERR_INVALID_ARGUMENT, "empty instance");
    int n = 0, m = 0, k = 0;
    size_t off = 0;
    for (int j = 0; j < nclauses; j++) {
        require(lens[j] >= 0, ASAT_ERR_INVALID_ARGUMENT, "negative clause length");
        int len1 = 0;
        for (int i = 0; i < lens[j]; i++) {
            int l = lits[off + i];
            if (!l) continue;
            require(l != INT32_MIN, ASAT_ERR_INVALID_ARGUMENT, "literal out of range");
            n = std::max(n, std::abs(l));
            len1++;
        }
        if (len1) { m++; k = std::max(k, len1); }
        off += (size_t)lens[j];
    }
    require(m > 0, ASAT_ERR_INVALID_ARGUMENT, "empty instance");
    require(k <= KMAX, ASAT_ERR_UNSUPPORTED, "batched solver supports clauses of up to 4 literals");
    require(n <= MAXN, ASAT_ERR_UNSUPPORTED, "batched solver supports up to 8191 variables per instance");
    require((long long)m * k <= MAXL, ASAT_ERR_UNSUPPORTED, "batched solver supports up to 262143 literal slots");
    I.n = n; I.m = m; I.k = k;
    std::vector<int> C((size_t)m * k, 0);
    off = 0;
    int row = 0;
    for (int j = 0; j < nclauses; j++) {
        int q = 0;
        for (int i = 0; i < lens[j]; i++) {
            int l = lits[off + i];
            if (l) C[(size_t)row * k + q++] = l;
        }
        if (q) row++;
        off += (size_t)lens[j];
    }
    // rowptr[i-1] .. rowptr[i]: contributions of variable i, in slot order
    std::vector<int> cnt((size_t)n + 1, 0);
    for (int l : C)
        if (l) cnt[std::abs(l)]++;
    I.rowptr.assign((size_t)n + 1, 0);
    for (int i = 1; i <= n; i++) I.rowptr[i] = I.rowptr[i - 1] + cnt[i];
    I.nslots = I.rowptr[n];
    std::vector<int> fill(I.rowptr.begin(), I.rowptr.end() - 1);
    I.code.assign((size_t)m * k, 0u);
    for (size_t s = 0; s < C.size(); s++) {
        int l = C[s];
        if (!l) continue;
        int v = std::abs(l);
        uint32_t p = (uint32_t)fill[v - 1]++;
        I.code[s] = ((uint32_t)v << 19) | ((l < 0 ? 1u : 0u) << 18) | p;
    }
}

// f(i) for every i in [0, count), on up to 8 threads while each gets 60 000 of the
// literal slots (about 0.2 ms; a thread costs about 50 us).  Instances are
// independent; building the layouts of 1024 of N = 2000, M = 8500 takes 85 ms on one.
template <typename F>
static void each_instance(int count, long long slots, F f)
{
    const long long most = std::min<long long>(8, std::max(1u, std::thread::hardware_concurrency()));
    const int nt = (int)std::max<long long>(1, std::min<long long>({most, (long long)count, 1 + slots / 60000}));
    std::atomic<int> next{0};
    std::mutex lock;
    std::exception_ptr failed;
    auto work = [&] {
        try {
            for (int i; (i = next++) < count;) f(i);
        } catch (...) {
            std::lock_guard<std::mutex> l(lock);
            failed = std::current_exception();
            next = count;
        }
    };
    std::vector<std::thread> th;
    th.reserve((size_t)nt);
    try {
        for (int t = 1; t < nt; t++) th.emplace_back(work);
    } catch (const std::system_error&) {
        // no more threads: those there are, and this one, do it
    }
    work();
    for (std::thread& t : th) t.join();
    if (failed) std::rethrow_exception(failed);
}

// host memory on its way to the device, not cleared first
template <typename V>
struct Staging {
    std::unique_ptr<unsigned char[]> raw;
    size_t count;
    explicit Staging(size_t n) : raw(new unsigned char[std::max<size_t>(n, 1) * sizeof(V)]), count(n) {}
    V* data() { return (V*)raw.get(); }
    void upload(V*& d)
    {
        HIP_CHECK(hipMalloc((void**)&d, sizeof(V) * std::max<size_t>(count, 1)));
        if (count) HIP_CHECK(hipMemcpy(d, raw.get(), sizeof(V) * count, hipMemcpyHostToDevice));
    }
};

static size_t bucket_lds(const Bucket& b, bool lds)
{
    return sizeof(float) * ((size_t)b.sp_stride + (lds ? (size_t)round_up_ll(b.maxl, 4) : 0));
}

// register-resident variants: threads per trajectory, clauses and variables
// per thread, more than 2046 variables (two shifts per contribution address).
// The smallest that an instance fits comes first; 1024 x (12, 3) and 512 x (24, 6)
// reach as far as the LDS does with 3-literal clauses.
struct RegVariant {
    int tt, cpt, vpt;
    bool wide;
    int block() const { return tt == 64 ? 64 * REG_WAVES : tt; }
    int waves() const { return tt == 64 ? REG_WAVES : 1; }
};
#define ASAT_REG_VARIANTS(X)                                                                             \
    X(64, 4, 1, false) X(64, 8, 2, false) X(256, 1, 1, false) X(256, 4, 2, false) X(512, 8, 4, false)    \
    X(768, 12, 3, true) X(1024, 9, 2, false) X(512, 17, 4, false) X(1024, 12, 3, true) X(512, 24, 6, true)
static const RegVariant REG_VARIANTS[] = {
#define ASAT_REG_ROW(T, C, V, W) {T, C, V, W},
    ASAT_REG_VARIANTS(ASAT_REG_ROW)
#undef ASAT_REG_ROW
};

// LDS of one trajectory: factors of every rank, contributions, the entry
// nothing reads
static size_t reg_lds(const RegVariant& r, const Bucket& b)
{
    const size_t waves = (size_t)r.tt / 64;      // RegShared, rounded up
    const size_t shared = ((size_t)8 * waves * r.vpt + 12 * waves + 20 + 15) / 16 * 16;
    return 8 * (size_t)r.tt * r.vpt + shared + sizeof(float) * (size_t)round_up_ll(b.ncontrib + 1, 4);
}
constexpr size_t LDS_STATIC = 1024;      // the kernels' static shared arrays

static bool reg_fits(const RegVariant& r, const Bucket& b, size_t lds_limit)
{
    return b.maxm <= r.tt * r.cpt && b.maxn + 2 <= r.tt * r.vpt && (r.wide || b.maxn <= 2046) &&
           b.ncontrib + 1 <= 65535 && reg_lds(r, b) * r.waves() <= lds_limit;
}

// first variant the bucket's instances fit (of workgroup size bs, or any)
static const RegVariant* reg_variant(const Bucket& b, size_t lds_limit, int bs = 0)
{
    for (const RegVariant& r : REG_VARIANTS)
        if ((!bs || r.block() == bs) && reg_fits(r, b, lds_limit)) return &r;
    return nullptr;
}

static const void* reg_kernel(const RegVariant& r, int kk)
{
#define ASAT_REG_PTR(T, C, V, W)                                                              \
    if (r.tt == T && r.cpt == C)                                                              \
        return kk == 3 ? (const void*)k_batch_reg<T, C, V, 3, W> : (const void*)k_batch_reg<T, C, V, 4, W>;
    ASAT_REG_VARIANTS(ASAT_REG_PTR)
#undef ASAT_REG_PTR
    throw Error(ASAT_ERR_HIP, "no register-resident kernel for this tiling");
}

static void launch_ptr(const void* f, hipStream_t st, const Params& P, int grid, int bs, size_t shmem)
{
    Params arg = P;
    void* args[] = {&arg};
    HIP_CHECK(hipLaunchKernel(f, dim3(grid), dim3(bs), args, shmem, st));
}

// chunked mode: LDS entries before the terms (factor pairs and sums), and the
// clauses per chunk that an instance may take
static int chunk_ranks(const Bucket& b) { return (int)round_up_ll((long long)b.maxn + 2, 4); }
static int chunk_terms_for(const Bucket& b, size_t lds_limit)
{
    const long long t = (long long)(lds_limit - LDS_STATIC) / (long long)sizeof(float) - 3LL * chunk_ranks(b) - 1;
    return (int)std::min<long long>(t, 65535);
}
static int chunk_max(const Instance& I, int terms, int force)
{
    const int cs = terms / (I.k <= 3 ? 3 : 4) / 64 * 64;
    return force > 0 ? std::min(cs, std::max(force, 1)) : cs;
}

template <int MODE>
static void launch_mode(hipStream_t st, const Params& P, int grid, int bs, size_t shmem)
{
    if (bs == 256) hipLaunchKernelGGL((k_batch<256, MODE>), dim3(grid), dim3(256), shmem, st, P);
    else if (bs == 512) hipLaunchKernelGGL((k_batch<512, MODE>), dim3(grid), dim3(512), shmem, st, P);
    else hipLaunchKernelGGL((k_batch<1024, MODE>), dim3(grid), dim3(1024), shmem, st, P);
}

template <int MODE>
static const void* kernel_of(int bs)
{
    return bs == 256 ? (const void*)k_batch<256, MODE> : bs == 512 ? (const void*)k_batch<512, MODE>
                                                                   : (const void*)k_batch<1024, MODE>;
}

static const void* chunk_kernel(int bs)
{
    return bs == 256 ? (const void*)k_batch_chunk<256> : bs == 512 ? (const void*)k_batch_chunk<512>
                                                                   : (const void*)k_batch_chunk<1024>;
}

static void dispatch(hipStream_t st, const Params& P, const Bucket& b)
{
    const int grid = b.grid, bs = b.block;
    const size_t shmem = b.lds_bytes;
    if (b.lds == 2) launch_ptr(reg_kernel(*b.reg, b.kk), st, P, grid, bs, shmem);
    else if (b.lds == 1) launch_mode<1>(st, P, grid, bs, shmem);
    else if (b.lds == 3) launch_ptr(chunk_kernel(bs), st, P, grid, bs, shmem);
    else launch_mode<0>(st, P, grid, bs, shmem);
}

static Params params_of(const Batch& B, const Bucket& b)
{
    Params P;
    P.desc = B.d_desc; P.code = B.d_code; P.rowptr = B.d_rowptr; P.xa = B.d_xa; P.xb = B.d_xb;
    P.ctrl = B.d_ctrl; P.scratch = b.d_scratch; P.scratch_stride = b.scratch_stride;
    P.scratch_per_wg = b.scratch_per_wg; P.order = b.d_order; P.ntraj = (int)b.ids.size();
    P.queue = b.d_queue; P.eps = B.eps; P.floor = B.floor; P.max_time = B.max_time; P.max_steps = B.max_steps;
    P.chunk_steps = B.chunk_steps; P.check_every = std::max(1, B.check_every);
    P.sp_stride = b.sp_stride;
    P.rcode = B.d_rcode; P.rgroup = B.d_rgroup; P.rvmap = B.d_rvmap;
    P.ccode = B.d_ccode; P.cgroup = B.d_cgroup; P.cperm = B.d_cperm; P.crec = B.d_crec; P.cstart = B.d_cstart;
    P.reg_lds = b.reg ? (int)reg_lds(*b.reg, b) : 0;
    P.chunk_terms = b.chunk_terms;
    P.fac_ranks = chunk_ranks(b);
    return P;
}

// resident workgroups per CU for a configuration with `lds_bytes` of LDS each
static int per_cu(const Batch& B, int bs, size_t lds_bytes)
{
    int by_lds = std::max(1, (int)(B.lds_limit / std::max<size_t>(lds_bytes, 1)));
    int by_threads = std::max(1, 2048 / bs);
    return std::max(1, std::min(by_lds, by_threads));
}

// mode: 0 contributions in global scratch, 1 in LDS, 2 register-resident
// kernel (bs names the workgroup size of its variant, or rv the variant), 3
// clause-chunked.  grid_cap > 0 limits the resident workgroups (global-scratch
// mode: the scattered contribution writes of fewer workgroups stay in the
// Infinity Cache).
static void configure_bucket(Batch& B, Bucket& b, int bs, int mode, int grid_cap = 0, const RegVariant* rv = nullptr)
{
    b.reg = nullptr;
    if (mode == 2) {
        if (!rv) rv = reg_variant(b, B.lds_limit, bs);
        if (!rv) rv = reg_variant(b, B.lds_limit);
        require(rv != nullptr, ASAT_ERR_INVALID_ARGUMENT, "instances too large for the register-resident kernel");
        b.reg = rv;
        bs = rv->block();
    }
    if (mode == 3)
        require(b.chunked, ASAT_ERR_INVALID_ARGUMENT, "the clause-chunked layout was not built for this bucket");
    b.block = bs;
    b.lds = mode;
    const int per_wg = mode == 2 ? b.reg->waves() : 1;      // trajectories of a workgroup
    b.lds_bytes = mode == 2   ? reg_lds(*b.reg, b) * per_wg
                  : mode == 3 ? sizeof(float) * (3 * (size_t)chunk_ranks(b) + (size_t)b.chunk_terms + 1)
                              : bucket_lds(b, mode == 1);
    b.grid = std::max(1, std::min(ceil_div((long long)b.ids.size(), per_wg),
                                  B.cus * per_cu(B, bs, mode == 0 ? 0 : b.lds_bytes)));
    if (grid_cap > 0) b.grid = std::min(b.grid, grid_cap);
    b.scratch_stride = round_up_ll((long long)b.maxn + b.maxm, 64);
    b.scratch_per_wg = mode == 2 ? 0 : 5 * b.scratch_stride + (mode == 0 ? round_up_ll(b.maxl, 64) : 0);
    (void)hipFree(b.d_scratch);
    b.d_scratch = nullptr;
    const size_t sbytes = sizeof(float) * std::max<size_t>((size_t)b.scratch_per_wg * b.grid, 1);
    HIP_CHECK(hipMalloc((void**)&b.d_scratch, sbytes));
    HIP_CHECK(hipMemsetAsync(b.d_scratch, 0, sbytes, B.stream));
    const void* f = mode == 2   ? reg_kernel(*b.reg, b.kk)
                    : mode == 3 ? chunk_kernel(bs)
                    : mode == 1 ? kernel_of<1>(bs)
                                : kernel_of<0>(bs);
    HIP_CHECK(hipFuncSetAttribute(f, hipFuncAttributeMaxDynamicSharedMemorySize, (int)b.lds_bytes));
}

// every trajectory back to its start (the start states stay on the device)
static void reset_state(Batch& B)
{
    const size_t T = B.inst.size(), bytes = sizeof(float) * (size_t)B.state_total;
    std::lock_guard<std::mutex> lock(B.win_lock);
    B.drop_window();
    HIP_CHECK(hipMemcpyAsync(B.d_xa, B.d_x0, bytes, hipMemcpyDeviceToDevice, B.stream));
    HIP_CHECK(hipMemcpyAsync(B.d_xb, B.d_x0, bytes, hipMemcpyDeviceToDevice, B.stream));
    HIP_CHECK(hipMemcpyAsync(B.d_ctrl, B.h_ctrl0.data(), sizeof(TrajCtrl) * T, hipMemcpyHostToDevice, B.stream));
    HIP_CHECK(hipStreamSynchronize(B.stream));
    B.h_ctrl = B.h_ctrl0;
    B.solved_wall_ms.assign(T, -1.0);
}

// State of one trajectory to the host.  A caller that walks through the
// trajectories in order (the second call in a row on) gets them from a window of
// at most WIN_FLOATS, packed on the device and copied at once into pinned memory
// that the batch keeps: one copy per trajectory cost 12 us each (1000 states:
// 14 ms with N = 50; 1024 of 42 KB: 12.7 ms).  Any other order copies
// one state as before, and so do states larger than the window.
constexpr long long WIN_FLOATS = 1 << 20;
static void get_state(Batch& B, int index, float* pub)
{
    const Instance& I = B.inst[(size_t)index];
    const size_t len = (size_t)I.n + I.m;
    std::unique_lock<std::mutex> lock(B.win_lock, std::try_to_lock);
    if (!lock.owns_lock()) {
        B.readers++;
        lock.lock();
        B.readers--;
    }
    HIP_CHECK(hipStreamSynchronize(B.stream));
    const bool in_order = B.last_state >= 0 && index == B.last_state + 1;
    B.last_state = index;
    if (index < B.win_first || index >= B.win_last) {
        const long long off = B.state_off[(size_t)index];
        if (!in_order || (long long)len > WIN_FLOATS) {
            const float* src = (B.h_ctrl[(size_t)index].parity ? B.d_xb : B.d_xa) + off;
            HIP_CHECK(hipMemcpy(pub, src, sizeof(float) * len, hipMemcpyDeviceToHost));
            return;
        }
        if (!B.d_win) HIP_CHECK(hipMalloc((void**)&B.d_win, sizeof(float) * WIN_FLOATS));
        if (!B.h_win) HIP_CHECK(hipHostMalloc((void**)&B.h_win, sizeof(float) * WIN_FLOATS, hipHostMallocDefault));
        int last = index;
        long long used = 0, most = 0;
        while (last < (int)B.inst.size() && last - index < 65535) {
            const Instance& J = B.inst[(size_t)last];
            const long long end = B.state_off[(size_t)last] - off + J.n + J.m;
            if (end > WIN_FLOATS) break;
            used = end;
            most = std::max(most, (long long)J.n + J.m);
            last++;
        }
        B.win_first = B.win_last = 0;
        hipLaunchKernelGGL(k_pack_states, dim3(std::min(64, ceil_div(most, 256)), last - index), dim3(256), 0, B.stream,
                           (const Desc*)B.d_desc, (const TrajCtrl*)B.d_ctrl, (const float*)B.d_xa,
                           (const float*)B.d_xb, index, B.d_win);
        HIP_CHECK(hipGetLastError());
        HIP_CHECK(hipMemcpyAsync(B.h_win, B.d_win, sizeof(float) * (size_t)used, hipMemcpyDeviceToHost, B.stream));
        HIP_CHECK(hipStreamSynchronize(B.stream));
        B.win_first = index;
        B.win_last = last;
    }
    memcpy(pub, B.h_win + (B.state_off[(size_t)index] - B.state_off[(size_t)B.win_first]), sizeof(float) * len);
}

// Autotuner: for each bucket, time one short chunk (2 to 32 accepted steps of
// every trajectory in the bucket, more for small instances, whose launch would
// hide the difference) of each configuration that fits, keep the fastest per
// trajectory-attempt, then restore the start.  Register variants exclude
// the others, and the clause-chunked kernel excludes global scratch (never the
// faster ones where both fit: 1024 trajectories of N = 2000, us per trajectory and
// attempt 0.12 in registers, 0.27 chunked, 0.50 with the terms in LDS, 1.44 in global
// scratch), unless asat_batch_set_tiling asks for one.
static void autotune(Batch& B)
{
    const int saved_chunk = B.chunk_steps;
    hipEvent_t e0, e1;
    HIP_CHECK(hipEventCreate(&e0));
    HIP_CHECK(hipEventCreate(&e1));
    for (auto& b : B.buckets) {
        B.chunk_steps = std::min(32, std::max(2, 60000 / std::max(b.maxl, 1)));
        struct Cand { int bs, mode, cap; const RegVariant* rv; };
        std::vector<Cand> cand;
        // register variants: the first that fits, and those of at most twice as many
        // threads as clauses or variables (run of 200 steps with 256, 512 and
        // 1024 threads, ms, N = 50, M = 213: 1000 trajectories 1.5, 4.5, 5.5, 64 of them
        // 1.1, 1.4, 1.7; N = 100, M = 426: 500 1.6, 2.8, 3.5)
        const int idle = 2 * std::max(b.maxm, b.maxn);
        if (B.force_lds == -1 || B.force_lds == 2)
            for (const RegVariant& r : REG_VARIANTS)
                if ((!B.force_block || r.block() == B.force_block) && reg_fits(r, b, B.lds_limit) &&
                    (r.tt <= idle || cand.empty()))
                    cand.push_back({r.block(), 2, 0, &r});
        const bool reg_only = !cand.empty() && B.force_lds == -1;
        const long long contrib_bytes = 4 * round_up_ll(b.maxl, 64);
        for (int bs : {256, 512, 1024}) {
            if (reg_only) break;
            if (B.force_block && bs != B.force_block) continue;
            if (b.lds_fits && (B.force_lds == -1 || B.force_lds == 1)) cand.push_back({bs, 1, 0, nullptr});
            if (b.chunked && (B.force_lds == -1 || B.force_lds == 3)) cand.push_back({bs, 3, 0, nullptr});
            if (B.force_lds == 0 || (B.force_lds == -1 && !b.chunked && !b.lds_fits)) {
                cand.push_back({bs, 0, 0, nullptr});
                const int full = std::max(1, std::min((int)b.ids.size(), B.cus * per_cu(B, bs, 0)));
                for (long long mb : {256LL, 128LL, 64LL}) {
                    const int cap = (int)std::max<long long>(8, (mb << 20) / std::max<long long>(contrib_bytes, 1));
                    if (cap < full) cand.push_back({bs, 0, cap, nullptr});
                }
            }
        }
        require(!cand.empty(), ASAT_ERR_INVALID_ARGUMENT, "no kernel configuration fits this bucket");
        double best = 1e300;
        Cand pick = cand.front();
        if (cand.size() > 1) {
            for (auto& c : cand) {
                configure_bucket(B, b, c.bs, c.mode, c.cap, c.rv);
                reset_state(B);
                Params P = params_of(B, b);
                hipLaunchKernelGGL(k_reset_queue, dim3(1), dim3(64), 0, B.stream, b.d_queue);
                HIP_CHECK(hipEventRecord(e0, B.stream));
                dispatch(B.stream, P, b);
                HIP_CHECK(hipEventRecord(e1, B.stream));
                HIP_CHECK(hipEventSynchronize(e1));
                HIP_CHECK(hipGetLastError());
                float ms = 0.f;
                HIP_CHECK(hipEventElapsedTime(&ms, e0, e1));
                std::vector<TrajCtrl> hc(B.inst.size());
                HIP_CHECK(hipMemcpy(hc.data(), B.d_ctrl, sizeof(TrajCtrl) * hc.size(), hipMemcpyDeviceToHost));
                long long att = 0;
                for (int id : b.ids) att += hc[id].attempts;
                double us = ms * 1e3 / std::max<long long>(att, 1);
                if (us < best) { best = us; pick = c; }
            }
        }
        configure_bucket(B, b, pick.bs, pick.mode, pick.cap, pick.rv);
        b.tuned_us = best < 1e300 ? best : -1.0;
    }
    (void)hipEventDestroy(e0);
    (void)hipEventDestroy(e1);
    B.chunk_steps = saved_chunk;
    reset_state(B);
}

static void prepare(Batch& B, bool tune)
{
    require(!B.inst.empty(), ASAT_ERR_INVALID_ARGUMENT, "no trajectories added");
    if (!B.stream) HIP_CHECK(hipStreamCreateWithFlags(&B.stream, hipStreamNonBlocking));
    HIP_CHECK(hipStreamSynchronize(B.stream));
    B.free_dev();
    const int T = (int)B.inst.size();
    int dev = 0;
    HIP_CHECK(hipGetDevice(&dev));
    HIP_CHECK(hipDeviceGetAttribute(&B.cus, hipDeviceAttributeMultiprocessorCount, dev));
    {
        int v = 0, v2 = 0;
        HIP_CHECK(hipDeviceGetAttribute(&v, hipDeviceAttributeMaxSharedMemoryPerBlock, dev));
        B.lds_limit = (size_t)v;
        if (hipDeviceGetAttribute(&v2, hipDeviceAttributeSharedMemPerBlockOptin, dev) == hipSuccess && v2 > v)
            B.lds_limit = (size_t)v2;
    }
    std::vector<Desc> desc(T);
    long long state_total = 0;
    B.state_off.assign(T, 0);
    for (int i = 0; i < T; i++) {
        const Instance& I = B.inst[i];
        desc[i].code_off = desc[i].row_off = -1;
        desc[i].state_off = state_total;
        B.state_off[i] = state_total;
        desc[i].n = I.n; desc[i].m = I.m; desc[i].k = I.k; desc[i].nslots = I.nslots;
        desc[i].rcode_off = desc[i].rgroup_off = desc[i].rvmap_off = -1;
        desc[i].ccode_off = desc[i].cgroup_off = desc[i].crec_off = desc[i].cstart_off = -1;
        desc[i].knorm = (float)std::pow(2.0, -I.k);
        state_total += round_up_ll((long long)I.n + I.m, 64);
    }
    std::vector<float> x0((size_t)state_total, 0.f);
    B.state_total = state_total;
    for (int i = 0; i < T; i++) {
        const Instance& I = B.inst[i];
        std::copy(I.pub0.begin(), I.pub0.end(), x0.begin() + desc[i].state_off);
    }
    // size buckets: trajectories sorted by work (slots + clauses), largest
    // first, split into up to nbuckets_req groups of equal count
    std::vector<int> order(T);
    std::iota(order.begin(), order.end(), 0);
    auto work = [&](int i) { return (long long)B.inst[i].nslots + B.inst[i].m; };
    std::stable_sort(order.begin(), order.end(), [&](int a, int b) { return work(a) > work(b); });
    int nb = std::max(1, std::min(B.nbuckets_req, T));
    if (work(order.front()) == work(order.back())) nb = 1;   // uniform batch: one launch
    B.buckets.assign(nb, Bucket());
    for (int q = 0; q < nb; q++) {
        Bucket& b = B.buckets[q];
        int lo = (int)((long long)T * q / nb), hi = (int)((long long)T * (q + 1) / nb);
        b.ids.assign(order.begin() + lo, order.begin() + hi);
        for (int id : b.ids) {
            b.maxn = std::max(b.maxn, B.inst[id].n);
            b.maxm = std::max(b.maxm, B.inst[id].m);
            b.maxl = std::max(b.maxl, B.inst[id].nslots);
            b.kk = std::max(b.kk, B.inst[id].k <= 3 ? 3 : 4);
        }
        b.sp_stride = (int)round_up_ll((long long)b.maxn + 1, 4);
        b.lds_fits = bucket_lds(b, true) <= B.lds_limit;
        HIP_CHECK(hipMalloc((void**)&b.d_order, sizeof(int) * b.ids.size()));
        HIP_CHECK(hipMalloc((void**)&b.d_queue, sizeof(int)));
        HIP_CHECK(hipMemcpy(b.d_order, b.ids.data(), sizeof(int) * b.ids.size(), hipMemcpyHostToDevice));
    }
    auto slots_of = [&](const Bucket& b) {
        long long n = 0;
        for (int id : b.ids) n += B.inst[id].nslots;
        return n;
    };
    // the register kernel's layout for the buckets that fit one of its
    // variants, the clause-chunked layout for the others
    {
        std::vector<RegLayout> reg((size_t)T);
        long long rcode = 0, rgroup = 0, rvmap = 0;
        for (auto& b : B.buckets) {
            bool may = false;
            for (const RegVariant& r : REG_VARIANTS) may = may || reg_fits(r, b, B.lds_limit);
            if (!may || (B.force_lds != -1 && B.force_lds != 2)) { b.ncontrib = 1 << 30; continue; }
            // (the ranking goes through variables, a tenth of the slots)
            each_instance((int)b.ids.size(), slots_of(b) / 10, [&](int i) {
                const int id = b.ids[(size_t)i];
                reg_layout(B.inst[id], reg[(size_t)id]);
            });
            for (int id : b.ids) b.ncontrib = std::max(b.ncontrib, reg[(size_t)id].ncontrib);
            if (!reg_variant(b, B.lds_limit)) continue;
            for (int id : b.ids) {
                const RegLayout& L = reg[(size_t)id];
                desc[id].rcode_off = rcode; desc[id].rgroup_off = rgroup; desc[id].rvmap_off = rvmap;
                desc[id].ngroups = L.ngroups; desc[id].ncontrib = L.ncontrib;
                rcode += rcode_len(B.inst[id], b.kk);
                rgroup += (long long)L.group.size();
                rvmap += (long long)L.vmap.size();
            }
        }
        if (rcode > 0) {
            Staging<uint32_t> hc((size_t)rcode);
            Staging<int> hg((size_t)rgroup), hv((size_t)rvmap);
            for (auto& b : B.buckets)
                each_instance((int)b.ids.size(), slots_of(b), [&](int i) {
                    const int id = b.ids[(size_t)i];
                    if (desc[id].rcode_off < 0) return;
                    RegLayout& L = reg[(size_t)id];
                    reg_codes(B.inst[id], L, b.kk, hc.data() + desc[id].rcode_off);
                    std::copy(L.group.begin(), L.group.end(), hg.data() + desc[id].rgroup_off);
                    std::copy(L.vmap.begin(), L.vmap.end(), hv.data() + desc[id].rvmap_off);
                });
            hc.upload(B.d_rcode);
            hg.upload(B.d_rgroup);
            hv.upload(B.d_rvmap);
        }
    }
    {
        std::vector<ChunkLayout> chunk((size_t)T);
        long long ccode = 0, cgroup = 0, crec = 0, cstart = 0;
        for (auto& b : B.buckets) {
            const bool want = B.force_lds == 3 || (B.force_lds == -1 && !reg_variant(b, B.lds_limit));
            b.chunk_terms = chunk_terms_for(b, B.lds_limit);
            b.chunked = want && b.chunk_terms >= 4 * 64;
            if (!b.chunked) continue;
            each_instance((int)b.ids.size(), slots_of(b), [&](int i) {
                const Instance& I = B.inst[b.ids[(size_t)i]];
                chunk_layout(I, chunk_max(I, b.chunk_terms, B.force_chunk), b.chunk_terms,
                             chunk[(size_t)b.ids[(size_t)i]]);
            });
            for (int id : b.ids) {
                const ChunkLayout& L = chunk[(size_t)id];
                Desc& d = desc[id];
                d.ccode_off = ccode; d.cgroup_off = cgroup; d.crec_off = crec; d.cstart_off = cstart;
                d.nchunks = L.nchunks; d.chunk = L.cs;
                ccode += (long long)L.code.size(); cgroup += (long long)L.group.size();
                crec += (long long)L.rec.size(); cstart += (long long)L.start.size();
            }
        }
        if (ccode > 0) {
            Staging<uint2> hcode((size_t)ccode);
            Staging<int2> hgroup((size_t)cgroup);
            Staging<uint16_t> hperm((size_t)cgroup * 64);
            Staging<uint32_t> hrec((size_t)crec);
            Staging<int> hstart((size_t)cstart);
            for (auto& b : B.buckets)
                each_instance((int)b.ids.size(), slots_of(b), [&](int i) {
                    const Desc& d = desc[(size_t)b.ids[(size_t)i]];
                    if (d.ccode_off < 0) return;
                    ChunkLayout& L = chunk[(size_t)b.ids[(size_t)i]];
                    std::copy(L.code.begin(), L.code.end(), hcode.data() + d.ccode_off);
                    std::copy(L.group.begin(), L.group.end(), hgroup.data() + d.cgroup_off);
                    std::copy(L.perm.begin(), L.perm.end(), hperm.data() + d.cgroup_off * 64);
                    std::copy(L.rec.begin(), L.rec.end(), hrec.data() + d.crec_off);
                    std::copy(L.start.begin(), L.start.end(), hstart.data() + d.cstart_off);
                });
            hcode.upload(B.d_ccode);
            hgroup.upload(B.d_cgroup);
            hperm.upload(B.d_cperm);
            hrec.upload(B.d_crec);
            hstart.upload(B.d_cstart);
        }
    }
    // k_batch's codes and rows, for the buckets that may run it
    {
        long long code = 0, rows = 0;
        for (auto& b : B.buckets) {
            const bool reg_ok = reg_variant(b, B.lds_limit, B.force_block) != nullptr;
            if (B.force_lds != 0 && B.force_lds != 1 && (B.force_lds != -1 || reg_ok || (b.chunked && !b.lds_fits)))
                continue;
            for (int id : b.ids) {
                desc[id].code_off = code;
                desc[id].row_off = rows;
                code += (long long)B.inst[id].code.size();
                rows += (long long)B.inst[id].rowptr.size();
            }
        }
        Staging<uint32_t> hcode((size_t)code);
        Staging<int> hrows((size_t)rows);
        for (auto& b : B.buckets)
            each_instance(code > 0 ? (int)b.ids.size() : 0, slots_of(b), [&](int i) {
                const int id = b.ids[(size_t)i];
                if (desc[id].code_off < 0) return;
                const Instance& I = B.inst[id];
                std::copy(I.code.begin(), I.code.end(), hcode.data() + desc[id].code_off);
                std::copy(I.rowptr.begin(), I.rowptr.end(), hrows.data() + desc[id].row_off);
            });
        hcode.upload(B.d_code);
        hrows.upload(B.d_rowptr);
    }
    HIP_CHECK(hipMalloc((void**)&B.d_desc, sizeof(Desc) * T));
    HIP_CHECK(hipMalloc((void**)&B.d_xa, sizeof(float) * std::max<long long>(state_total, 1)));
    HIP_CHECK(hipMalloc((void**)&B.d_xb, sizeof(float) * std::max<long long>(state_total, 1)));
    HIP_CHECK(hipMalloc((void**)&B.d_x0, sizeof(float) * std::max<long long>(state_total, 1)));
    HIP_CHECK(hipMemcpy(B.d_x0, x0.data(), sizeof(float) * state_total, hipMemcpyHostToDevice));
    HIP_CHECK(hipMalloc((void**)&B.d_ctrl, sizeof(TrajCtrl) * T));
    HIP_CHECK(hipMemcpy(B.d_desc, desc.data(), sizeof(Desc) * T, hipMemcpyHostToDevice));
    B.h_ctrl0.assign(T, TrajCtrl());
    for (int i = 0; i < T; i++) {
        TrajCtrl& c = B.h_ctrl0[i];
        memset(&c, 0, sizeof(c));
        c.h = 1e-9; c.hnext = 1e-9;
        c.min_viol = INT32_MAX; c.viol = -1; c.sat_step = -1; c.sat_time = -1.0;
        c.status = RUNNING;
    }
    for (auto& b : B.buckets) {
        int bs = B.force_block ? B.force_block : 1024;
        const bool reg_any = B.force_lds != 0 && B.force_lds != 1 && reg_variant(b, B.lds_limit);
        const bool reg_ok = reg_any && (!B.force_block || reg_variant(b, B.lds_limit, B.force_block));
        int mode = B.force_lds == -1 ? (reg_ok ? 2 : (b.lds_fits ? 1 : (b.chunked ? 3 : 0))) : B.force_lds;
        require(mode == 0 || mode == 2 || mode == 3 || b.lds_fits, ASAT_ERR_UNSUPPORTED,
                "instances too large for LDS contributions");
        require(mode != 3 || b.chunked, ASAT_ERR_UNSUPPORTED, "instances too large for the clause-chunked kernel");
        require(mode != 2 || reg_any, ASAT_ERR_UNSUPPORTED, "instances too large for the register-resident kernel");
        if (mode == 2 && !B.force_block) bs = 0;
        configure_bucket(B, b, bs, mode);
    }
    reset_state(B);
    if (tune) autotune(B);
    B.prepared = true;
}

// run chunks until every trajectory has finished (or max_chunks chunks)
static void run(Batch& B, int max_chunks, int graph_chunks)
{
    require(B.prepared, ASAT_ERR_NOT_CONFIGURED, "batch has not been prepared");
    require(max_chunks > 0 && graph_chunks > 0, ASAT_ERR_INVALID_ARGUMENT, "chunk counts must be positive");
    const int T = (int)B.inst.size();
    // events, graph and executable are released on every exit, and a capture
    // left open by an error is ended, so the stream stays usable
    struct Owned {
        hipStream_t st;
        hipEvent_t e0 = nullptr, e1 = nullptr;
        hipEvent_t fork = nullptr, join[3] = {nullptr, nullptr, nullptr};
        hipGraph_t graph = nullptr;
        hipGraphExec_t exec = nullptr;
        bool capturing = false;
        ~Owned()
        {
            if (capturing) {
                hipGraph_t g = nullptr;
                if (hipStreamEndCapture(st, &g) == hipSuccess && g) (void)hipGraphDestroy(g);
            }
            if (exec) (void)hipGraphExecDestroy(exec);
            if (graph) (void)hipGraphDestroy(graph);
            if (e0) (void)hipEventDestroy(e0);
            if (e1) (void)hipEventDestroy(e1);
            if (fork) (void)hipEventDestroy(fork);
            for (hipEvent_t e : join)
                if (e) (void)hipEventDestroy(e);
        }
    } o{B.stream};
    HIP_CHECK(hipEventCreate(&o.e0));
    HIP_CHECK(hipEventCreate(&o.e1));
    hipEvent_t e0 = o.e0, e1 = o.e1;
    // one graph = graph_chunks x (per bucket: reset its queue, persistent
    // launch).  Buckets are independent, so their launches go to up to four
    // branches: a bucket with fewer trajectories than resident workgroups leaves
    // CUs to the next one, and so does the end of every launch, when the last
    // trajectories run alone (512 ragged instances, 128 per bucket on 256 CUs:
    // 19.5 -> 13.5 ms for 20 steps)
    const int nb = (int)B.buckets.size(), branches = std::min(nb, 4);
    HIP_CHECK(hipEventCreateWithFlags(&o.fork, hipEventDisableTiming));
    for (int q = 1; q < branches; q++) {
        if (!B.side[q - 1]) HIP_CHECK(hipStreamCreateWithFlags(&B.side[q - 1], hipStreamNonBlocking));
        HIP_CHECK(hipEventCreateWithFlags(&o.join[q - 1], hipEventDisableTiming));
    }
    std::unique_lock<std::mutex> lock = B.launch_lock();   // no reader's work gets into the capture
    HIP_CHECK(hipStreamBeginCapture(B.stream, hipStreamCaptureModeThreadLocal));
    o.capturing = true;
    HIP_CHECK(hipEventRecord(o.fork, B.stream));
    for (int q = 0; q < branches; q++) {
        hipStream_t st = q ? B.side[q - 1] : B.stream;
        if (q) HIP_CHECK(hipStreamWaitEvent(st, o.fork, 0));
        for (int c = 0; c < graph_chunks; c++)
            for (int i = q; i < nb; i += branches) {
                Bucket& b = B.buckets[(size_t)i];
                Params P = params_of(B, b);
                hipLaunchKernelGGL(k_reset_queue, dim3(1), dim3(64), 0, st, b.d_queue);
                dispatch(st, P, b);
            }
        if (q) {
            HIP_CHECK(hipEventRecord(o.join[q - 1], st));
            HIP_CHECK(hipStreamWaitEvent(B.stream, o.join[q - 1], 0));
        }
    }
    o.capturing = false;
    HIP_CHECK(hipStreamEndCapture(B.stream, &o.graph));
    lock.unlock();
    HIP_CHECK(hipGraphInstantiate(&o.exec, o.graph, nullptr, nullptr, 0));
    hipGraphExec_t exec = o.exec;
    auto t0 = std::chrono::steady_clock::now();
    HIP_CHECK(hipEventRecord(e0, B.stream));
    int launched = 0;
    std::vector<TrajCtrl>& hc = B.h_ctrl;
    while (launched < max_chunks) {
        lock = B.launch_lock();
        B.drop_window();
        HIP_CHECK(hipGraphLaunch(exec, B.stream));
        launched += graph_chunks;
        HIP_CHECK(hipMemcpyAsync(hc.data(), B.d_ctrl, sizeof(TrajCtrl) * T, hipMemcpyDeviceToHost, B.stream));
        HIP_CHECK(hipStreamSynchronize(B.stream));
        lock.unlock();
        double now = std::chrono::duration<double, std::milli>(std::chrono::steady_clock::now() - t0).count();
        int live = 0;
        for (int i = 0; i < T; i++) {
            if (hc[i].status == RUNNING) live++;
            else if (hc[i].status == SOLVED && B.solved_wall_ms[i] < 0) B.solved_wall_ms[i] = now;
        }
        if (!live) break;
    }
    HIP_CHECK(hipEventRecord(e1, B.stream));
    HIP_CHECK(hipEventSynchronize(e1));
    float ms = 0.f;
    HIP_CHECK(hipEventElapsedTime(&ms, e0, e1));
    B.run_ms += ms;
    B.chunks_run += launched;
}

}  // namespace batch
}  // namespace asat

// ===========================================================================
// C ABI
// ===========================================================================
using namespace asat;
using namespace asat::batch;

struct asat_batch { Batch b; };

#define BAPI_BEGIN try {
#define BAPI_END                                                 \
    }                                                            \
    catch (const asat::Error& e) {                               \
        asat::g_last_error = e.what();                           \
        return e.code;                                           \
    }                                                            \
    catch (const std::exception& e) {                            \
        asat::g_last_error = e.what();                           \
        return ASAT_ERR_HIP;                                     \
    }                                                            \
    return ASAT_OK;

extern "C" {

int asat_batch_create(asat_batch_t** out)
{
    BAPI_BEGIN
    require(out != nullptr, ASAT_ERR_INVALID_ARGUMENT, "null argument: out");
    *out = new asat_batch();
    BAPI_END
}

int asat_batch_destroy(asat_batch_t* b)
{
    BAPI_BEGIN
    delete b;
    BAPI_END
}

int asat_batch_add(asat_batch_t* b, const int* literals, const int* lengths, int nclauses, const float* pub0,
                   int* index_out)
{
    BAPI_BEGIN
    require(b && pub0, ASAT_ERR_INVALID_ARGUMENT, "null argument");
    Instance I;
    build_instance(literals, lengths, nclauses, I);
    I.pub0.assign(pub0, pub0 + (size_t)I.n + I.m);
    b->b.inst.push_back(std::move(I));
    b->b.prepared = false;
    if (index_out) *index_out = (int)b->b.inst.size() - 1;
    BAPI_END
}

int asat_batch_set_params(asat_batch_t* b, double eps, long long max_steps, double max_time, int chunk_steps,
                          int check_every)
{
    BAPI_BEGIN
    require(b != nullptr, ASAT_ERR_INVALID_ARGUMENT, "null batch");
    require(!(eps < 1e-16 || eps > 1.0), ASAT_ERR_INVALID_ARGUMENT, "epsilon must be between 1e-16 and 1");
    require(max_steps >= 1, ASAT_ERR_INVALID_ARGUMENT, "Max iterations must be positive");
    require(max_time > 0.0, ASAT_ERR_INVALID_ARGUMENT, "Max time must be positive");
    require(chunk_steps >= 1 && check_every >= 1, ASAT_ERR_INVALID_ARGUMENT, "chunk/check sizes must be positive");
    b->b.eps = eps; b->b.max_steps = max_steps; b->b.max_time = max_time;
    b->b.chunk_steps = chunk_steps; b->b.check_every = check_every;
    BAPI_END
}

int asat_batch_set_xscal_floor(asat_batch_t* b, double floor)
{
    BAPI_BEGIN
    require(b != nullptr, ASAT_ERR_INVALID_ARGUMENT, "null batch");
    require(floor > 0.0 && floor <= 1.0, ASAT_ERR_INVALID_ARGUMENT, "xscal floor must be in (0, 1]");
    b->b.floor = floor;
    BAPI_END
}

int asat_batch_set_chunk(asat_batch_t* b, int clauses)
{
    BAPI_BEGIN
    require(b != nullptr, ASAT_ERR_INVALID_ARGUMENT, "null batch");
    require(clauses >= 0, ASAT_ERR_INVALID_ARGUMENT, "chunk size must be >= 0");
    b->b.force_chunk = clauses;
    b->b.prepared = false;
    BAPI_END
}

int asat_batch_set_tiling(asat_batch_t* b, int block, int lds_mode, int nbuckets)
{
    BAPI_BEGIN
    require(b != nullptr, ASAT_ERR_INVALID_ARGUMENT, "null batch");
    require(block == 0 || block == 256 || block == 512 || block == 1024, ASAT_ERR_INVALID_ARGUMENT,
            "block must be 0 (autotune), 256, 512 or 1024");
    require(lds_mode >= -1 && lds_mode <= 3, ASAT_ERR_INVALID_ARGUMENT, "lds_mode must be -1, 0, 1, 2 or 3");
    require(nbuckets >= 1 && nbuckets <= 64, ASAT_ERR_INVALID_ARGUMENT, "nbuckets must be in [1, 64]");
    b->b.force_block = block; b->b.force_lds = lds_mode; b->b.nbuckets_req = nbuckets;
    b->b.prepared = false;
    BAPI_END
}

int asat_batch_prepare(asat_batch_t* b, int autotune)
{
    BAPI_BEGIN
    require(b != nullptr, ASAT_ERR_INVALID_ARGUMENT, "null batch");
    prepare(b->b, autotune != 0);
    BAPI_END
}

int asat_batch_run(asat_batch_t* b, int max_chunks, int graph_chunks)
{
    BAPI_BEGIN
    require(b != nullptr, ASAT_ERR_INVALID_ARGUMENT, "null batch");
    run(b->b, max_chunks, graph_chunks);
    BAPI_END
}

int asat_batch_reset(asat_batch_t* b)
{
    BAPI_BEGIN
    require(b != nullptr && b->b.prepared, ASAT_ERR_NOT_CONFIGURED, "batch has not been prepared");
    reset_state(b->b);
    b->b.run_ms = 0.0;
    b->b.chunks_run = 0;
    BAPI_END
}

int asat_batch_size(const asat_batch_t* b, int* count)
{
    BAPI_BEGIN
    require(b && count, ASAT_ERR_INVALID_ARGUMENT, "null argument");
    *count = (int)b->b.inst.size();
    BAPI_END
}

int asat_batch_result(const asat_batch_t* b, int index, asat_batch_result_t* out)
{
    BAPI_BEGIN
    require(b && out, ASAT_ERR_INVALID_ARGUMENT, "null argument");
    require(b->b.prepared, ASAT_ERR_NOT_CONFIGURED, "batch has not been prepared");
    require(index >= 0 && index < (int)b->b.inst.size(), ASAT_ERR_INVALID_ARGUMENT, "index out of range");
    const TrajCtrl& c = b->b.h_ctrl[index];
    out->status = c.status;
    out->steps = c.steps;
    out->attempts = c.attempts;
    out->rhscount = c.rhscount;
    out->time = c.t;
    out->hdid = c.hdid;
    out->hnext = c.hnext;
    out->min_violations = c.min_viol == INT32_MAX ? -1 : c.min_viol;
    out->violations = c.viol;
    out->sat_step = c.sat_step;
    out->sat_time = c.sat_time;
    out->solved_wall_ms = b->b.solved_wall_ms[index];
    BAPI_END
}

int asat_batch_get_state(const asat_batch_t* b, int index, float* pub)
{
    BAPI_BEGIN
    require(b && pub, ASAT_ERR_INVALID_ARGUMENT, "null argument");
    require(b->b.prepared, ASAT_ERR_NOT_CONFIGURED, "batch has not been prepared");
    require(index >= 0 && index < (int)b->b.inst.size(), ASAT_ERR_INVALID_ARGUMENT, "index out of range");
    get_state(const_cast<Batch&>(b->b), index, pub);
    BAPI_END
}

int asat_batch_stats(const asat_batch_t* b, double* run_ms, int* chunks, int* nbuckets)
{
    BAPI_BEGIN
    require(b != nullptr, ASAT_ERR_INVALID_ARGUMENT, "null batch");
    if (run_ms) *run_ms = b->b.run_ms;
    if (chunks) *chunks = b->b.chunks_run;
    if (nbuckets) *nbuckets = (int)b->b.buckets.size();
    BAPI_END
}

int asat_batch_bucket_info(const asat_batch_t* b, int bucket, asat_batch_bucket_t* out)
{
    BAPI_BEGIN
    require(b && out, ASAT_ERR_INVALID_ARGUMENT, "null argument");
    require(bucket >= 0 && bucket < (int)b->b.buckets.size(), ASAT_ERR_INVALID_ARGUMENT, "bucket out of range");
    const Bucket& k = b->b.buckets[bucket];
    out->trajectories = (int)k.ids.size();
    out->max_n = k.maxn;
    out->max_m = k.maxm;
    out->max_slots = k.maxl;
    out->block = k.block;
    out->lds = k.lds;
    out->grid = k.grid;
    out->lds_bytes = (long long)k.lds_bytes;
    out->tuned_us_per_attempt = k.tuned_us;
    BAPI_END
}

}  // extern "C"
