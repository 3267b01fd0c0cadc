// Plain single-trajectory CTDS solver for MI355X (gfx950): one problem, one
// trajectory, the whole chip.  Replaces CudaSat1/2/3 + CudaRungeKutta
// (AnalogSAT/cuda_sat/CudaSat3.cu:33-430, AnalogSAT/cuda_sat/CudaRungeKutta.cu:56-484).
//
// Data layout in HBM (T = double for ASAT_F64, float for ASAT_F32):
//   lit[m*K + q]      int32 signed literal (+v / -v, 0 = padding), clause-major,
//                     padded to whole tiles of at most TC clauses
//   contrib[p]        per-slot contribution 2 c a K K_mi of the current stage.
//                     Variables are split into groups (at most about 2048 float
//                     / 1024 double variables, halved until the largest region
//                     fits the LDS); a group's contributions form one
//                     region (64-element aligned, at most 144 KB), in slot
//                     (clause) order.  Between a var pass and the next clause
//                     pass the same array holds the slot spins: each slot's
//                     stage spin at the slot's position
//   spos, srank       per tile: the positions of the tile's slots in ascending
//                     order (int32), and each slot's rank in that order (uint16,
//                     the literal's sign in bit 15; literal q of the tile's
//                     clauses at q*TC + clause, so each load is one run)
//   runs              big FP32 tiles (up to 4608 clauses): a word per variable
//                     group in place of spos (the tile's positions in one
//                     region are consecutive: first rank, first offset)
//   pw16, pv0         big FP32 tiles: per clause its primary variable relative
//                     to the tile's first (pv0), the primary literal's position
//                     and sign, in place of pvar and the primary slots' ranks
//   csr_ptr[0..N+1]   var-major CSR row pointers
//   rloc, ploc        uint16 per region entry, and per clause for its direct
//                     primary term: its place in the group's var-major slot
//                     list (variables in order, each one's slots in slot order)
//   state buffer      [ -1, s_1..s_N, pad | a_1..a_M, pad ], aux at aoff
//   k1..k5            same layout as the state (stage derivatives)
//   tmp               spin part of the next stage's input (aux stage inputs are
//                     recomputed inside the clause pass and never stored)
// Problems outside the fast paths use a generic clause pass (K other than 3
// and 4: pos[m*K + q] per slot) and a gather var pass (a group whose region
// exceeds the LDS: csr_pos global positions, ~400 KB groups, or one
// workgroup per variable when rows are long); both gather the stage spins by
// variable from x / tmp.
//
// One RK45 attempt = 6 x (clause pass + var pass) + 1 control kernel:
//   clause pass J: per tile, read the slot spins through the tile's sorted
//                  positions (one run per region), K_m, aux stage input and
//                  k_J(a_m) = a K^2, then store the tile's contributions at
//                  the same positions
//   var pass J:    one workgroup per group reads the group's region into LDS
//                  with coalesced loads, adds each variable's contributions
//                  in slot order (== the reference's accumulation order),
//                  then k_J(s_i), the spin part of stage J+1's input, and
//                  writes the region back as stage J+1's slot spins
//   J = 6 passes also form x_new and |xerr/xscal| and a per-block FP64 max;
//   the control kernel finishes the max-norm and runs the Cash-Karp
//   accept/reject/step-size logic in FP64 on the device.
// Step(count) fills the slot spins of x, enqueues attempts without host
// round trips and reads the control block back once per round of attempts.
#include "asat_common.h"
#include "asat_grid.h"
#include "asat_small.h"

#include <algorithm>
#include <atomic>
#include <climits>
#include <cmath>
#include <cstring>
#include <memory>
#include <mutex>
#include <new>
#include <numeric>
#include <vector>

namespace asat {

thread_local std::string g_last_error;

constexpr int BLK = 256;          // stage-kernel block size (4 waves)
constexpr int CTRL_BLK = 1024;    // control kernel block size

static inline long long round_up(long long a, long long b) { return (a + b - 1) / b * b; }

// ===========================================================================
// problem (host)
// ===========================================================================
constexpr int TC = 2048;                  // clauses per tile of the tiled clause pass (one workgroup), at most
constexpr int TC_BIG = 4608;              // FP32 3-literal systems with direct primary slots: the most
                                          // clauses a tile may have (its size is chosen per problem)
constexpr int TC_MAX = TC_BIG;
constexpr unsigned PW_VMASK = 0x1FFFu;    // big tiles' primary words: relative variable bits,
constexpr int PW_QSHIFT = 13;             // then the primary literal's position, then its sign
constexpr int TILE_BT = 1024;             // threads per tile workgroup (a clause each)
constexpr int VAR_SUM = 8;              // terms of a variable in flight in the var pass
constexpr int VBLK = 1024;                // var-pass workgroup (one variable group)
constexpr int VAR_LDS_BYTES = 147456;     // LDS holding one group's contribution region
constexpr int VAR_LDS_CU = 163840 - 1024; // LDS two var workgroups may share on one CU
constexpr int REGION_ALIGN = 64;          // region starts, in elements
constexpr bool REORDER_CLAUSES = true;    // tiled pass: process clauses sorted by a primary variable

struct HostProblem {
    int n = 0, m = 0, k = 0;
    std::vector<int> lit;          // m*k, zero padded, clause-major, in processing order
    std::vector<int> perm;         // processing position -> clause index (empty: identity)
    // contribution layout: variables split into groups of vg; the
    // contributions of a group's variables form one region, in slot (clause)
    // order; region starts are REGION_ALIGN-element aligned
    int vg = 0, ngroups = 0;
    long long max_region = 0;      // largest region incl. alignment padding
    std::vector<long long> gstart; // ngroups+1
    std::vector<int> pos;          // m*k: the slot's contribution position, -1 for padding
    std::vector<int> csr_ptr;      // n+2
    std::vector<int> csr_pos;      // gather var pass: contribution positions of each variable, in slot order
    // LDS var pass: each region entry's place in its group's var-major slot list
    // (entries of no slot: past the list), and each clause's direct primary term's
    std::vector<uint16_t> rloc, ploc;
    // tiled clause pass: per tile of TC clauses, its slots sorted by position
    std::vector<int> spos;         // ntiles*TC*k positions (-1 past the tile's last slot)
    // big tiles: per tile, a run table in place of spos.
    // Word g of tile t: bits 0-15 the first rank of group g's run in the
    // tile's sorted list, bits 16-31 the run's first position relative to
    // the region start gstart[g]; word ngroups holds the tile's slot count
    // (run_stride words per tile)
    std::vector<uint32_t> runs;
    int run_stride = 0;
    // big tiles: primary words in place of pvar and of the primary slots'
    // ranks.  pw16[j] holds the clause's primary variable relative to its
    // tile's first (pv0[tile]) in bits 0-12, the primary literal's position
    // in bits 13-14 (3: padding clause) and its sign in bit 15; srank then
    // holds K - 1 ranks per clause, the other literals in clause order
    std::vector<uint16_t> pw16;
    std::vector<int> pv0;
    std::vector<uint16_t> srank;   // per slot: its rank in the tile's sorted list, the literal's sign
                                   // in bit 15, 0xFFFF for padding; per tile, literal q of every
                                   // clause first (index tile*TC*K + q*TC + clause in the tile)
    // primary variables (tiled pass): pvar[j] is the primary variable of
    // processing-order clause j and pq[j] the first of its literals on it
    std::vector<int> pvar;
    std::vector<unsigned char> pq;
    // direct primary slots (tiled pass with LDS regions): a clause's primary
    // slot is not in any region; its spin is read from the stage vector by
    // variable and its term stored at the clause's processing position of
    // pcontrib.  Regions hold the other slots.  pc0[g] is the first clause
    // whose primary variable is in group g (ngroups+1 entries).
    bool split = false;
    std::vector<int> pc0;
    int tc = TC;                   // tiled pass: clauses per tile
};

// SatProblem::AddClauses semantics (AnalogSAT/problem/SatProblem.cpp:64-95) +
// CpuSat::InitProblem clause matrix (AnalogSAT/cpu_sat/CpuSat.cpp:352-377).
static void parse_clauses(const int* literals, const int* lengths, int nclauses, HostProblem& P)
{
    require(nclauses >= 0, ASAT_ERR_INVALID_ARGUMENT, "negative clause count");
    require(nclauses == 0 || (literals && lengths), ASAT_ERR_INVALID_ARGUMENT, "null clause arrays");
    int n = 0, m = 0, k = 0;
    size_t off = 0;
    for (int j = 0; j < nclauses; j++) {
        require(lengths[j] >= 0, ASAT_ERR_INVALID_ARGUMENT, "negative clause length");
        int len1 = 0;
        for (int i = 0; i < lengths[j]; i++) {
            int l = literals[off + i];
            if (l == 0) continue;
            require(l != INT32_MIN, ASAT_ERR_INVALID_ARGUMENT, "literal out of range");
            n = std::max(n, std::abs(l));
            len1++;
        }
        if (len1 > 0) { m++; k = std::max(k, len1); }
        off += (size_t)lengths[j];
    }
    require(m > 0 && k > 0, ASAT_ERR_INVALID_ARGUMENT, "empty SAT problem");
    require(k <= GEN_KMAX, ASAT_ERR_UNSUPPORTED, "clauses longer than 32 literals are not supported");
    require((long long)m * k < (1LL << 31) - (long long)TC_MAX * k, ASAT_ERR_UNSUPPORTED, "more than 2^31 literal slots");
    P.n = n; P.m = m; P.k = k;
    P.lit.assign((size_t)m * k, 0);
    off = 0;
    int row = 0;
    for (int j = 0; j < nclauses; j++) {
        int q = 0;
        for (int i = 0; i < lengths[j]; i++) {
            int l = literals[off + i];
            if (l == 0) continue;
            P.lit[(size_t)row * k + q++] = l;
        }
        if (q > 0) row++;
        off += (size_t)lengths[j];
    }
}

// Processing order of the tiled clause pass.  Every clause gets one primary
// variable (greedily its least-loaded variable, so that each variable is
// primary for about M/N clauses) and clauses are processed sorted by it
// (stable).  A wave then reads its clauses' primary spins from a few adjacent
// lines, and a tile stores its primary contributions as one run.  Literal
// order inside a clause is kept, and so is every per-variable sum order.
static void reorder_clauses(HostProblem& P)
{
    const int K = P.k, m = P.m, n = P.n;
    std::vector<int> load((size_t)n + 1, 0), prim((size_t)m, 0);
    for (int j = 0; j < m; j++) {
        int best = 0;
        for (int q = 0; q < K; q++) {
            const int l = P.lit[(size_t)j * K + q];
            if (!l) continue;
            const int v = std::abs(l);
            if (best == 0 || load[v] < load[best]) best = v;
        }
        prim[j] = best;
        load[best]++;
    }
    P.pvar.assign((size_t)m, 0);
    P.pq.assign((size_t)m, 0);
    std::vector<int> start((size_t)n + 2, 0);
    for (int j = 0; j < m; j++) start[(size_t)prim[j] + 1]++;
    for (int v = 0; v <= n; v++) start[v + 1] += start[v];
    P.perm.assign((size_t)m, 0);
    for (int j = 0; j < m; j++) P.perm[(size_t)start[prim[j]]++] = j;
    std::vector<int> lit2(P.lit.size());
    for (int j = 0; j < m; j++)
        std::copy_n(P.lit.begin() + (size_t)P.perm[j] * K, K, lit2.begin() + (size_t)j * K);
    P.lit.swap(lit2);
    for (int j = 0; j < m; j++) {
        const int v = prim[(size_t)P.perm[j]];
        P.pvar[(size_t)j] = v;
        int q = 0;
        while (std::abs(P.lit[(size_t)j * K + q]) != v) q++;
        P.pq[(size_t)j] = (unsigned char)q;
    }
}

// Contribution layout for groups of vg variables, and the transposed
// var-major slot list (role of CudaSat3::InitProblem,
// AnalogSAT/cuda_sat/CudaSat3.cu:266-307, without the pad-to-32).
// pv > 0 (tiled pass with primary variables): direct primary slots.  The
// regions then hold only the other slots, and the LDS var pass reads the
// group's primary terms from pcontrib (from pc0[g] rounded down to a multiple of
// pv elements, its 16-byte load unit).
// cap > 0: for the LDS var pass; false, with nothing but the regions' sizes made,
// when the largest region with its primary terms exceeds cap entries.
static bool build_layout(HostProblem& P, int vg, int pv, long long cap)
{
    const int n = P.n, m = P.m, K = P.k;
    const bool split = pv > 0 && !P.pvar.empty();
    P.split = split;
    P.vg = vg;
    P.ngroups = (n + vg - 1) / vg;
    std::vector<int> grp((size_t)n + 1, 0);
    for (int v = 1; v <= n; v++) grp[(size_t)v] = (v - 1) / vg;
    // f(slot, clause, variable, the clause's primary slot?) over all literals
    auto each = [&](auto f) {
        for (int j = 0; j < m; j++) {
            const int pq = split ? P.pq[(size_t)j] : -1;
            for (int q = 0; q < K; q++) {
                const size_t s = (size_t)j * K + q;
                if (P.lit[s]) f(s, j, std::abs(P.lit[s]), q == pq);
            }
        }
    };
    std::vector<long long> gcount((size_t)P.ngroups, 0);
    each([&](size_t, int, int v, bool prim) { gcount[(size_t)grp[(size_t)v]] += !prim; });
    P.pc0.clear();
    if (split) {
        // clauses are sorted by primary variable: group g's primaries are the
        // processing range [pc0[g], pc0[g+1])
        P.pc0.assign((size_t)P.ngroups + 1, m);
        for (int j = m - 1; j >= 0; j--) P.pc0[(size_t)grp[(size_t)P.pvar[(size_t)j]]] = j;
        for (int g = P.ngroups - 1; g >= 0; g--) P.pc0[g] = std::min(P.pc0[g], P.pc0[(size_t)g + 1]);
    }
    P.gstart.assign((size_t)P.ngroups + 1, 0);
    P.max_region = 0;
    for (int g = 0; g < P.ngroups; g++) {
        const long long sz = round_up(std::max<long long>(gcount[g], 1), REGION_ALIGN);
        P.gstart[g + 1] = P.gstart[g] + sz;
        long long lds = sz;
        if (split) lds += round_up(P.pc0[(size_t)g + 1] - (P.pc0[g] / pv) * pv, pv);
        P.max_region = std::max(P.max_region, lds);
    }
    if (cap > 0 && P.max_region > cap) return false;
    require(P.gstart[P.ngroups] < (1LL << 31), ASAT_ERR_UNSUPPORTED, "contribution array exceeds 2^31 entries");
    P.pos.assign(P.lit.size(), -1);
    P.csr_ptr.assign((size_t)n + 2, 0);
    std::vector<long long> gfill(P.gstart.begin(), P.gstart.end() - 1);
    each([&](size_t s, int, int v, bool prim) {
        if (!prim) P.pos[s] = (int)gfill[(size_t)grp[(size_t)v]]++;
        P.csr_ptr[(size_t)v + 1]++;
    });
    for (int i = 0; i <= n; i++) P.csr_ptr[i + 1] += P.csr_ptr[i];
    // the variables' slot lists; slots visited in the original clause order,
    // which is the reference's accumulation order
    std::vector<int> row((size_t)m);
    for (int j = 0; j < m; j++) row[P.perm.empty() ? j : P.perm[j]] = j;
    P.csr_pos.clear();
    P.rloc.clear();
    P.ploc.clear();
    std::vector<int> fill(P.csr_ptr.begin(), P.csr_ptr.end() - 1);
    if (cap > 0) {
        // cursors relative to the group's list
        P.rloc.resize((size_t)P.gstart[P.ngroups]);
        if (split) P.ploc.resize((size_t)m);
        for (int g = 0; g < P.ngroups; g++) {
            const int i0 = g * vg + 1, i1 = std::min(n, (g + 1) * vg), e0 = P.csr_ptr[i0];
            for (int v = i0; v <= i1; v++) fill[(size_t)v] -= e0;
            std::fill(P.rloc.begin() + P.gstart[g], P.rloc.begin() + P.gstart[(size_t)g + 1],
                      (uint16_t)(P.csr_ptr[i1 + 1] - e0));
        }
    } else {
        P.csr_pos.resize((size_t)P.csr_ptr[n + 1]);
    }
    for (int mo = 0; mo < m; mo++) {
        const int j = row[(size_t)mo], pq = split ? P.pq[(size_t)j] : -1;
        for (int q = 0; q < K; q++) {
            const size_t s = (size_t)j * K + q;
            if (!P.lit[s]) continue;
            const int e = fill[(size_t)std::abs(P.lit[s])]++;
            if (cap == 0) P.csr_pos[(size_t)e] = P.pos[s];
            else if (q == pq) P.ploc[(size_t)j] = (uint16_t)e;
            else P.rloc[(size_t)P.pos[s]] = (uint16_t)e;
        }
    }
    return true;
}

// Per tile of TC clauses: the tile's slots in ascending position order.
// Positions inside a region follow slot order, so this is a stable counting
// sort of the tile's slots by variable group; the clause pass then writes
// each group's run of contributions with neighbouring lanes.  With direct
// primary slots only the other slots are sorted (K - 1 per clause), and a
// primary slot's rank entry is 0x4000 with the sign bit.
static void build_tile_order(HostProblem& P)
{
    const int K = P.k, TCt = P.tc;
    const int NR = P.split ? K - 1 : K;
    const long long ntiles = ceil_div((long long)P.m, TCt);
    const size_t per = (size_t)TCt * K, nper = (size_t)TCt * NR;
    // run tables (big tiles): a tile's positions in one region are
    // consecutive (tiles are ranges of slots, region positions follow slot
    // order), so the sorted list is one run per group
    const bool rt = P.split && TCt > TC;
    require(!rt || (long long)(P.ngroups + 1) * 4 <= (long long)nper, ASAT_ERR_UNSUPPORTED,
            "run tables larger than the positions they replace");
    P.runs.clear();
    P.run_stride = 0;
    if (rt) {
        P.run_stride = (int)round_up((long long)P.ngroups + 1, 16);
        P.runs.assign((size_t)ntiles * P.run_stride, 0);
    } else {
        P.spos.assign((size_t)ntiles * nper, -1);
    }
    // big tiles store K - 1 ranks per clause (the primary one is in pw16)
    const bool cp = P.split && TCt > TC;
    const int KR = cp ? NR : K;
    const size_t rper = (size_t)TCt * KR;
    P.srank.assign((size_t)ntiles * rper, 0xFFFF);
    P.pw16.clear();
    P.pv0.clear();
    if (cp) {
        P.pw16.assign((size_t)ntiles * TCt, (uint16_t)(3u << PW_QSHIFT));
        P.pv0.assign((size_t)ntiles, 0);
        for (long long t = 0; t < ntiles; t++) {
            const long long j0 = t * TCt, j1 = std::min<long long>(P.m, j0 + TCt);
            const int v0 = P.pvar[(size_t)j0];
            P.pv0[(size_t)t] = v0;
            for (long long j = j0; j < j1; j++) {
                const int rel = P.pvar[(size_t)j] - v0;
                require(rel >= 0 && rel <= (int)PW_VMASK, ASAT_ERR_UNSUPPORTED, "tile's primary variables too far apart");
                const int q = P.pq[(size_t)j];
                const unsigned sg = P.lit[(size_t)j * K + q] < 0 ? 0x8000u : 0u;
                P.pw16[(size_t)j] = (uint16_t)(rel | (q << PW_QSHIFT) | sg);
            }
        }
    }
    // a tile's slots of one group hold consecutive positions (in any order):
    // a slot's rank is its run's first rank plus its offset from the run's
    // lowest position
    std::vector<int> cnt((size_t)P.ngroups + 1, 0);
    std::vector<int> rmin((size_t)P.ngroups + 1, INT_MAX);
    std::vector<int> touched;
    touched.reserve(per);
    for (long long t = 0; t < ntiles; t++) {
        const size_t s0 = (size_t)t * per, s1 = std::min(P.lit.size(), s0 + per);
        const size_t r0 = (size_t)t * nper;
        touched.clear();
        for (size_t s = s0; s < s1; s++) {
            int l = P.lit[s];
            if (!l || P.pos[s] < 0) continue;
            int g = (std::abs(l) - 1) / P.vg;
            if (cnt[g]++ == 0) touched.push_back(g);
            rmin[g] = std::min(rmin[g], P.pos[s]);
        }
        std::sort(touched.begin(), touched.end());
        int acc = 0;
        if (rt) {
            // every group's word: its first rank (untouched groups: that of
            // the next run); region offsets are filled from the slots below
            uint32_t* w = P.runs.data() + (size_t)t * P.run_stride;
            size_t i = 0;
            for (int g = 0; g <= P.ngroups; g++) {
                while (i < touched.size() && touched[i] < g) acc += cnt[touched[i++]];
                w[g] = (uint32_t)acc;
            }
            require(acc <= (int)nper, ASAT_ERR_UNSUPPORTED, "run table exceeds the tile");
            acc = 0;
        }
        for (int g : touched) { int c = cnt[g]; cnt[g] = acc; acc += c; }
        for (size_t s = s0; s < s1; s++) {
            int l = P.lit[s];
            if (!l) continue;
            const size_t ls = s - s0;   // tile-local slot: clause ls / K, literal ls % K
            const unsigned sign = l < 0 ? 0x8000u : 0u;
            if (P.pos[s] < 0) {   // a direct primary slot
                if (!cp) P.srank[(size_t)t * rper + (ls % K) * TCt + ls / K] = (uint16_t)(0x4000u | sign);
                continue;
            }
            size_t qs = ls % K;   // the slot's rank row: with primary words, among the other literals
            if (cp && qs > P.pq[(size_t)t * TCt + ls / K]) qs--;
            uint16_t& rk = P.srank[(size_t)t * rper + qs * TCt + ls / K];
            int g = (std::abs(l) - 1) / P.vg;
            const size_t j = (size_t)cnt[g] + (size_t)(P.pos[s] - rmin[g]);
            if (rt) {
                uint32_t& w = P.runs[(size_t)t * P.run_stride + g];
                if (j == (w & 0xFFFFu)) {   // the run's lowest position
                    const long long off = P.pos[s] - P.gstart[g];
                    require(off >= 0 && off < 65536, ASAT_ERR_UNSUPPORTED, "run offset exceeds 16 bits");
                    w |= (uint32_t)off << 16;
                }
            } else {
                P.spos[r0 + j] = P.pos[s];
            }
            rk = (uint16_t)(j | sign);
        }
        for (int g : touched) { cnt[g] = 0; rmin[g] = INT_MAX; }
    }
}

// ===========================================================================
// device kernels
// ===========================================================================
template <typename T>
struct StageArgs {
    const int* lit;
    const int* pos;        // contribution position of each slot (-1: padding); generic-K pass
    const int* spos;       // tiled pass: per tile, positions in ascending order (-1: none)
    const uint16_t* srank; // tiled pass: rank of each slot in its tile's sorted list
    const unsigned* runs;  // big tiles: per tile, run table in place of spos
    int run_stride;        // words per tile of the run tables
    const int* csr_ptr;
    const int* litq;       // generic pass, K <= 10: literals and contribution positions by literal (mq apart)
    const int* posq;
    int mq;
    double* th;            // its tanh table, 2 per variable from 0 (null: not used)
    const int* csr_pos;    // per-variable contribution positions (gather var pass)
    const uint16_t* rloc;      // LDS var pass: list place of each region entry
    const uint16_t* ploc;      // and of each clause's direct primary term
    const long long* gstart;   // region starts, ngroups+1
    const int* pvar;       // direct primary slots: primary variable of each clause (processing order)
    const uint16_t* pw16;  // big tiles: primary word of each clause (in place of pvar)
    const int* pv0;        // big tiles: each tile's first primary variable
    const int* pc0;        // direct primary slots: first clause of each group's primaries, ngroups+1
    T* pcontrib;           // direct primary slots: each clause's primary term (processing order)
    T* contrib;
    T* xa;       // state buffer 0
    T* xb;       // state buffer 1 (x = parity ? xb : xa; x_new is the other)
    T* k1; T* k2; T* k3; T* k4; T* k5;
    T* tmp;      // spin stage input (n+1)
    // slot spins: between a var pass and the next clause pass, contrib holds
    // the next stage's spins in contribution layout (each slot's spin at the
    // slot's contribution position); 0: the clause pass gathers from x / tmp
    int slot_spins;
    double* partial;   // per-block error maxima: clause blocks first, then var blocks
    double* apart;     // bias term: per clause-block sums of the stage aux values
    const Ctrl* ctrl;  // null: standalone RHS (x = xa, output to k1, no tmp)
    int n, m, k, aoff;
    int nblk_clause;   // clause-pass grid (its J = 6 error partials come first)
    int vg;            // variables per group
    int var_stagger;      // LDS var pass: CUs whose second workgroup starts late (0: none)
    int vg_blocks;     // gather var pass: blocks per variable group
    int ngroups;
    int clause_per_xcd;   // clause-pass chunks (BLK clauses, or TC-clause tiles) per XCD
    int ntiles;           // tiled pass: tiles
    int tile_clauses;     // tiled pass: clauses per tile
    int split;            // direct primary slots (tiled pass + LDS var pass)
    int family;           // ASAT_FAMILY_CTDS or ASAT_FAMILY_TANH
    int bias;             // sine bias term on (b > 0)
    T knorm;
    T q;                  // tanh family parameter
    T bb, alpha;          // b knorm^2 and M / N (bias term)
};

// XCD-contiguous clause-pass mapping: XCD x (blocks b with b % 8 == x) walks
// the clause chunks [x*per, (x+1)*per) in order.  Contribution positions are
// assigned in clause order inside each region, so every XCD fills its own
// contiguous stretch of each region and its L2 merges the partial lines
// before they are written back.
__device__ __forceinline__ int clause_of_thread(int per)
{
    const int b = blockIdx.x;
    return ((b & 7) * per + (b >> 3)) * BLK + threadIdx.x;
}

// XCD-affine var-pass mapping for the gather var pass: workgroups are
// dispatched to the 8 XCDs round-robin, so block b runs on XCD b % 8.  All
// vg_blocks blocks of one variable group are given to the same XCD, and each
// XCD walks its groups in order, so a group's contribution region stays in
// that XCD's L2 while its variables gather from it.  Returns the block's
// first variable (1-based) and last variable, or 0 for an idle block.
__device__ __forceinline__ int var_block_range(int vg, int vg_blocks, int ngroups, int n, int& last)
{
    const int b = blockIdx.x;
    const int xcd = b & 7, t = b >> 3;
    const int grp = (t / vg_blocks) * 8 + xcd;
    last = 0;
    if (grp >= ngroups) return 0;
    const long long g0 = (long long)grp * vg + 1;
    const long long i0 = g0 + (long long)(t % vg_blocks) * BLK;
    const long long gl = std::min<long long>(g0 + vg - 1, n);
    if (i0 > gl) return 0;
    last = (int)std::min<long long>(i0 + BLK - 1, gl);
    return (int)i0;
}

// Global loads and stores of the solver kernels: ordinary cached accesses.
// Non-temporal hints on the once-per-pass streams were measured on the
// N = 1e6 instance and cost 4% of the attempt rate: the index arrays and the
// state vectors are read again by the next passes, and the memory-side cache
// keeps part of them between passes.
template <typename V>
__device__ __forceinline__ V ld_g(const V* p)
{
    return *p;
}
template <typename V>
__device__ __forceinline__ void st_g(V* p, V v)
{
    *p = v;
}
// non-temporal accesses of the practical-rate probes (plain streams)
template <typename V>
__device__ __forceinline__ V ld_stream(const V* p)
{
    return __builtin_nontemporal_load(p);
}
template <typename V>
__device__ __forceinline__ void st_stream(V* p, V v)
{
    __builtin_nontemporal_store(v, p);
}

// ---- clause pass, compile-time K (Ex order), tiled -----------------------
// Slot ranks: bits 0-13 the rank in the tile's sorted list, bit 14 a direct
// primary slot (its rank bits 0), bit 15 the literal's sign, 0xFFFF padding.
constexpr unsigned RANK_MASK = 0x3FFFu;
constexpr unsigned RANK_PRIMARY = 0x4000u;

// Slot terms of one clause, written to LDS at the slots' ranks in the tile's
// position order (a direct primary slot's term goes to pt instead).  CTDS:
// r = K_m 2^-k a_m times the product of the other factors in KmiProd order,
// times +-2; tanh: tanh_term with r = 2^-k a_m.  Stops at the first padding
// literal (KmiFunc / KmiFuncTanh).
template <typename T, int K, int Q, bool PS>
__device__ __forceinline__ void slot_terms(const int (&l)[K], const T (&f)[K], T r, bool tanh_family, T q,
                                           const uint16_t* rank, T* s_out, T& pt)
{
    if constexpr (Q < K) {
        if (l[Q] != 0) {
            const T p = kmi_prod<T, K, Q>(f);
            T rr;
            if (tanh_family) {
                rr = tanh_term<T>(r, p, f[Q], q, l[Q] < 0, true);
            } else {
                rr = r * p;
                rr *= l[Q] < 0 ? (T)-2.0 : (T)2.0;
            }
            if (PS && (rank[Q] & RANK_PRIMARY)) pt = rr;
            else s_out[rank[Q] & RANK_MASK] = rr;
            slot_terms<T, K, Q + 1, PS>(l, f, r, tanh_family, q, rank, s_out, pt);
        }
    }
}

// Phase 1 of a tile for G of the thread's clauses (its clauses u0 .. u0+G-1,
// see k_clause_tile): K_m, the aux stage input, k_J(a_m) and the slot terms,
// which go to s_out at their ranks (direct primary terms into pt).  Every
// load that does not depend on another is issued first: the slot ranks
// (padded to whole tiles, read unguarded), the literal rows when the spins
// are gathered by variable, and the aux values.
// SS (slot spins): s_out already holds each rank's stage spin (phase 0), and
// psv the clauses' direct primary spins; the literal signs come from the
// ranks' bit 15.  Otherwise sp is the N-element stage spin vector, gathered
// by variable.
// CP (primary words, big tiles, K = 3): a clause's two stored ranks are its
// other literals' in clause order; its primary word names the primary
// literal's position and sign, from which the three slot ranks are formed.
template <typename T, int K, int J, int BT, bool SS, bool PS, int G, int CPT, bool CP>
__device__ __forceinline__ void tile_group(const StageArgs<T>& a, long long c0, int TS, int u0, const T* x, T* xnew,
                                           const T* sp, const T (&psv)[CPT], T hs, double h, double hnext,
                                           double floor, bool tanh_family, T* s_out, double& err, double& asum)
{
    int l[G][K];
    T sv[G][K];
    T ax[G], a1[G], a2[G], a3[G], a4[G], a5[G];
    uint16_t rk[G][K];
    static_assert(!CP || K == 3, "primary words: 3-literal clauses");
    unsigned pw[G], r2[G][2];
#pragma unroll
    for (int g = 0; g < G; g++) {
        const int lc = (u0 + g) * BT + (int)threadIdx.x;   // the clause in the tile (< TS: a clause of it)
        const long long m = c0 + lc;
        if constexpr (!SS) {
#pragma unroll
            for (int q = 0; q < K; q++) l[g][q] = lc < TS ? ld_g(a.lit + m * K + q) : 0;
        }
        if constexpr (CP) {
            pw[g] = lc < TS ? (unsigned)ld_g(a.pw16 + m) : (3u << PW_QSHIFT);
#pragma unroll
            for (int q = 0; q < 2; q++) r2[g][q] = lc < TS ? (unsigned)ld_g(a.srank + c0 * 2 + (long long)q * TS + lc) : 0xFFFFu;
        } else {
#pragma unroll
            for (int q = 0; q < K; q++) rk[g][q] = lc < TS ? ld_g(a.srank + c0 * K + (long long)q * TS + lc) : 0xFFFF;
        }
    }
#pragma unroll
    for (int g = 0; g < G; g++) {
        const int lc = (u0 + g) * BT + (int)threadIdx.x;
        const long long m = c0 + lc;
        const size_t ai = (size_t)a.aoff + m;
        ax[g] = a1[g] = a2[g] = a3[g] = a4[g] = a5[g] = (T)0;
        if (lc < TS && m < a.m) {
            ax[g] = ld_g(x + ai);
            if constexpr (J > 1) a1[g] = ld_g(a.k1 + ai);
            if constexpr (J > 2) a2[g] = ld_g(a.k2 + ai);
            if constexpr (J > 3) a3[g] = ld_g(a.k3 + ai);
            if constexpr (J > 4) a4[g] = ld_g(a.k4 + ai);
            if constexpr (J > 5) a5[g] = ld_g(a.k5 + ai);
        }
    }
    if constexpr (CP) {
        // primary position 3: a padding clause (its stored ranks are 0xFFFF)
#pragma unroll
        for (int g = 0; g < G; g++) {
            const unsigned pq = (pw[g] >> PW_QSHIFT) & 3u;
            const unsigned pr = RANK_PRIMARY | (pw[g] & 0x8000u);
            rk[g][0] = (uint16_t)(pq == 0 ? pr : r2[g][0]);
            rk[g][1] = (uint16_t)(pq == 1 ? pr : (pq == 0 ? r2[g][0] : r2[g][1]));
            rk[g][2] = (uint16_t)(pq == 2 ? pr : (pq == 3 ? 0xFFFFu : r2[g][1]));
        }
    }
    if constexpr (SS) {
        // each rank is read here and overwritten with its slot term below by
        // the same thread (the owner of the slot), so one buffer serves both
#pragma unroll
        for (int g = 0; g < G; g++) {
#pragma unroll
            for (int q = 0; q < K; q++) {
                const unsigned r = rk[g][q];
                l[g][q] = r == 0xFFFFu ? 0 : ((r & 0x8000u) ? -1 : 1);
                if (r == 0xFFFFu) sv[g][q] = (T)-1.0;
                else if (PS && (r & RANK_PRIMARY)) sv[g][q] = psv[u0 + g];
                else sv[g][q] = s_out[r & RANK_MASK];
            }
        }
    } else {
#pragma unroll
        for (int g = 0; g < G; g++) {
#pragma unroll
            for (int q = 0; q < K; q++) {
                const int v = l[g][q] < 0 ? -l[g][q] : l[g][q];
                sv[g][q] = v != 0 ? sp[v] : (T)-1.0;
            }
        }
    }
#pragma unroll
    for (int g = 0; g < G; g++) {
        const int lc = (u0 + g) * BT + (int)threadIdx.x;
        const long long m = c0 + lc;
        T pt = (T)0;
        if (lc < TS && m < a.m) {
            T f[K];
            T km = a.knorm;
#pragma unroll
            for (int q = 0; q < K; q++) {
                f[q] = l[g][q] < 0 ? (T)1.0 + sv[g][q] : (T)1.0 - sv[g][q];
                km *= f[q];
            }
            const size_t ai = (size_t)a.aoff + m;
            T am;
            if constexpr (J == 1) am = ax[g];
            else am = stage_input<T, J>(ax[g], a1[g], a2[g], a3[g], a4[g], a5[g], hs);
            T kj = am * km * km;
            asum += (double)am;
            if constexpr (J == 1) st_g(a.k1 + ai, kj);
            else if constexpr (J == 2) st_g(a.k2 + ai, kj);
            else if constexpr (J == 3) st_g(a.k3 + ai, kj);
            else if constexpr (J == 4) st_g(a.k4 + ai, kj);
            else if constexpr (J == 5) st_g(a.k5 + ai, kj);
            else {
                T xn;
                double e;
                final_combination<T>(ax[g], a1[g], a3[g], a4[g], a5[g], kj, hs, h, hnext, floor, xn, e);
                err = fmax(err, e);
                st_g(xnew + ai, xn);
            }
            const T r = tanh_family ? a.knorm * am : km * a.knorm * am;
            slot_terms<T, K, 0, PS>(l[g], f, r, tanh_family, a.q, rk[g], s_out, pt);
        }
        // pcontrib is padded to whole tiles: padding clauses store 0
        if constexpr (PS)
            if (lc < TS) st_g(a.pcontrib + m, pt);
    }
}

// One workgroup of BT threads per tile of TCt clauses (XCD-contiguous tile
// ranges), TCt / BT clauses per thread.
// Phase 0, a thread per rank (slot spins only): the tile's sorted positions,
// and the stage spins read through them into s_out (neighbouring lanes,
// neighbouring positions of one region); with direct primary slots also the
// thread's clauses' primary spins, from the stage spin vector.
// Phase 1, a thread per clause, in groups of G clauses (tile_group): the
// clause arithmetic, slot terms into s_out at their ranks; direct primary
// terms (PS) are stored at the clauses' own positions of pcontrib.
// Phase 2, a thread per rank: store the terms through the sorted positions.
// Big tiles (TCt = TC_BIG) hold up to 4608 clauses, a size chosen per
// problem (tile_clauses) so that the tiles fill whole rounds of resident
// workgroups: about 4100-clause tiles give each region runs of about 8
// entries per tile in place of 4, and no nearly empty last round (one
// extra tile running alone cost about 5 us per pass).  Phase 1 takes their
// clauses one at a time, which keeps them at 8 waves per SIMD without
// spills; two at a time spilled at J = 6 and ran 1-4 us slower per pass.
// FP64 3-literal tiles run 8 waves per SIMD too, two workgroups per CU (62-76
// registers and one workgroup otherwise: N = 163 840, M = 696 320 169 us per
// attempt, 157 now, 158.5 with spills instead of one clause at a time from
// J = 4 on); 4-literal ones would spill and lose (109 and 111.5 us).
template <typename T, int K, int J, int BT, int TCt, bool SS, bool PS>
__global__ __launch_bounds__(BT) __attribute__((amdgpu_waves_per_eu(TCt > TC || (sizeof(T) == 8 && K == 3) ? 8 : 1)))
void k_clause_tile(StageArgs<T> a)
{
    constexpr int CPT = (TCt + BT - 1) / BT;
    constexpr int G = TCt > TC || (sizeof(T) == 8 && K == 3 && J >= 4) ? 1 : (CPT < 2 ? CPT : 2);
    constexpr int CPTG = (CPT + G - 1) / G * G;   // clause slots of the groups (past CPT: none of the tile)
    constexpr int NR = PS ? K - 1 : K;
    constexpr int NP = CPT * NR;
    static_assert(TCt * NR <= (int)RANK_MASK + 1, "a tile's ranks must fit the rank field");
    // the sorted positions of big tiles wait in LDS for phase 2
    constexpr bool PL = TCt > TC;
    __shared__ double sh[BT / 64];
    __shared__ T s_out[TCt * NR];
    __shared__ int s_pos[PL ? TCt * NR : 1];
    const Ctrl* c = a.ctrl;
    int parity = 0;
    double h = 0.0, hnext = 0.0, floor = TabD::TINY;
    if (c) {
        if (!c->active) return;
        if (J == 1 && !c->step_start) return;
        parity = c->parity; h = c->h; hnext = c->hnext; floor = c->floor;
    }
    const T hs = (T)h;
    const T* x = parity ? a.xb : a.xa;
    T* xnew = parity ? a.xa : a.xb;
    const T* sp = SS ? a.contrib : ((J == 1) ? x : a.tmp);
    const bool tanh_family = a.family == ASAT_FAMILY_TANH;
    const int b = blockIdx.x;
    double err = 0.0, asum = 0.0;
    const int tile = (b & 7) * a.clause_per_xcd + (b >> 3);
    if (tile < a.ntiles) {
        const int TS = a.tile_clauses;
        const long long c0 = (long long)tile * TS;
        int ps[NP];
        T psv[CPTG];
        int pv[CPTG];
        if constexpr (SS && PS) {
            // padding clauses have primary variable 0 (or the tile's first
            // primary variable): x[0] / tmp[0], unused
            if constexpr (PL) {
                const int v0 = a.pv0[tile];
#pragma unroll
                for (int u = 0; u < CPTG; u++) {
                    const int lc = u * BT + (int)threadIdx.x;
                    pv[u] = lc < TS ? v0 + (int)(ld_g(a.pw16 + c0 + lc) & PW_VMASK) : 0;
                }
            } else {
#pragma unroll
                for (int u = 0; u < CPTG; u++) {
                    const int lc = u * BT + (int)threadIdx.x;
                    pv[u] = lc < TS ? ld_g(a.pvar + c0 + lc) : 0;
                }
            }
        }
        if constexpr (PL) {
            // the sorted positions from the tile's run table: group g's
            // ranks [j0(g), j0(g+1)) sit at consecutive positions from
            // gstart[g] + off(g); ranks past the tile's slots get -1
            const unsigned* rt = a.runs + (long long)tile * a.run_stride;
            for (int g = (int)threadIdx.x; g < a.ngroups; g += BT) {
                const unsigned w0 = ld_g(rt + g), w1 = ld_g(rt + g + 1);
                const int j0 = (int)(w0 & 0xFFFFu), j1 = (int)(w1 & 0xFFFFu);
                const int base = (int)ld_g(a.gstart + g) + (int)(w0 >> 16) - j0;
                for (int j = j0; j < j1; j++) s_pos[j] = base + j;
            }
            const int nsl = (int)(ld_g(rt + a.ngroups) & 0xFFFFu);
#pragma unroll
            for (int i = 0; i < NP; i++) {
                const int lr = i * BT + (int)threadIdx.x;
                if (lr >= nsl && lr < TS * NR) s_pos[lr] = -1;
            }
            if constexpr (SS) __syncthreads();
#pragma unroll
            for (int i = 0; i < NP; i++) {
                const int lr = i * BT + (int)threadIdx.x;
                ps[i] = (SS && lr < TS * NR) ? s_pos[lr] : -1;
            }
        } else {
            const int* sp_t = a.spos + c0 * NR;
#pragma unroll
            for (int i = 0; i < NP; i++) {
                const int lr = i * BT + (int)threadIdx.x;
                ps[i] = lr < TS * NR ? ld_g(sp_t + lr) : -1;
            }
        }
        if constexpr (SS) {
            if constexpr (PS) {
                const T* svec = (J == 1) ? x : a.tmp;
#pragma unroll
                for (int u = 0; u < CPTG; u++) psv[u] = ld_g(svec + pv[u]);
            }
            // LDS holds TCt * NR ranks; NP * BT may be more (TCt not a
            // multiple of BT), and a tile has TS * NR <= TCt * NR of them
            T so[NP];
#pragma unroll
            for (int i = 0; i < NP; i++) so[i] = ps[i] >= 0 ? sp[ps[i]] : (T)0;
#pragma unroll
            for (int i = 0; i < NP; i++) {
                const int lr = i * BT + (int)threadIdx.x;
                if (lr < TS * NR) s_out[lr] = so[i];
            }
        }
        if constexpr (SS) __syncthreads();
#pragma unroll
        for (int u0 = 0; u0 < CPT; u0 += G)
            tile_group<T, K, J, BT, SS, PS, G, CPTG, PL>(a, c0, TS, u0, x, xnew, sp, psv, hs, h, hnext, floor,
                                                          tanh_family, s_out, err, asum);
        __syncthreads();
#pragma unroll
        for (int i = 0; i < NP; i++) {
            const int lr = i * BT + (int)threadIdx.x;
            if (lr < TS * NR) {
                const int p = PL ? s_pos[lr] : ps[i];
                if (p >= 0) a.contrib[p] = s_out[lr];
            }
        }
    }
    if (a.bias) {
        const double bs = block_sum_all<BT>(asum, sh);
        if (threadIdx.x == 0) a.apart[blockIdx.x] = bs;
    }
    if constexpr (J == 6) {
        double bm = block_max<BT>(err, sh);
        if (threadIdx.x == 0) a.partial[blockIdx.x] = bm;
    }
}

// ---- clause pass, runtime K (any K <= 32; K > 10 uses CalculateAll order) --
template <typename T, int J>
__global__ __launch_bounds__(BLK) void k_clause_gen(StageArgs<T> a)
{
    __shared__ double sh[BLK / 64];
    __shared__ T fsh[GEN_KMAX * BLK];
    const Ctrl* c = a.ctrl;
    int parity = 0;
    double h = 0.0, hnext = 0.0, floor = TabD::TINY;
    if (c) {
        if (!c->active) return;
        if (J == 1 && !c->step_start) return;
        parity = c->parity; h = c->h; hnext = c->hnext; floor = c->floor;
    }
    const T hs = (T)h;
    const T* x = parity ? a.xb : a.xa;
    T* xnew = parity ? a.xa : a.xb;
    const T* sp = (J == 1) ? x : a.tmp;
    const int K = a.k;
    const int m = clause_of_thread(a.clause_per_xcd);
    T* f = fsh + threadIdx.x;   // f[q*BLK]
    double err = 0.0, asum = 0.0;
    if (m < a.m) {
        const int* lm = a.lit + (size_t)m * K;
        T km = a.knorm;
        for (int q = 0; q < K; q++) {
            T fq = spin_factor<T>(lm[q], sp);
            km *= fq;
            f[q * BLK] = fq;
        }
        const size_t ai = (size_t)a.aoff + m;
        T am, k1 = 0, k3 = 0, k4 = 0, k5 = 0;
        if constexpr (J == 1) {
            am = x[ai];
        } else {
            k1 = a.k1[ai];
            T k2 = J > 2 ? a.k2[ai] : (T)0;
            k3 = J > 3 ? a.k3[ai] : (T)0;
            k4 = J > 4 ? a.k4[ai] : (T)0;
            k5 = J > 5 ? a.k5[ai] : (T)0;
            am = stage_input<T, J>(x[ai], k1, k2, k3, k4, k5, hs);
        }
        T kj = am * km * km;
        asum = (double)am;
        if constexpr (J == 1) a.k1[ai] = kj;
        else if constexpr (J == 2) a.k2[ai] = kj;
        else if constexpr (J == 3) a.k3[ai] = kj;
        else if constexpr (J == 4) a.k4[ai] = kj;
        else if constexpr (J == 5) a.k5[ai] = kj;
        else {
            T xn;
            final_combination<T>(x[ai], k1, k3, k4, k5, kj, hs, h, hnext, floor, xn, err);
            xnew[ai] = xn;
        }
        T* out = a.contrib;
        const int* pm = a.pos + (size_t)m * K;
        if (a.family == ASAT_FAMILY_TANH) {
            // CpuSatTanh: templated helper for K = 3..10, generic loop otherwise
            const T r = a.knorm * am;
            const bool ex = K >= 3 && K <= 10;
            for (int q = 0; q < K; q++) {
                int l = lm[q];
                if (l == 0) break;
                T p = (T)1.0;
                bool first = true;
                for (int qq = 0; qq < K; qq++) {
                    if (qq == q) continue;
                    p = first ? f[qq * BLK] : p * f[qq * BLK];
                    first = false;
                }
                out[pm[q]] = tanh_term<T>(r, p, f[q * BLK], a.q, l < 0, ex);
            }
        } else if (K <= 10) {
            const T r = km * a.knorm * am;
            for (int q = 0; q < K; q++) {
                int l = lm[q];
                if (l == 0) break;
                T p = (T)1.0;
                bool first = true;
                for (int qq = 0; qq < K; qq++) {
                    if (qq == q) continue;
                    p = first ? f[qq * BLK] : p * f[qq * BLK];
                    first = false;
                }
                T rr = r * p;
                rr *= l < 0 ? (T)-2.0 : (T)2.0;
                out[pm[q]] = rr;
            }
        } else {
            for (int q = 0; q < K; q++) {
                int l = lm[q];
                if (l == 0) continue;
                T temp = km;
                for (int qq = 0; qq < K; qq++) temp *= (qq == q) ? (T)1.0 : f[qq * BLK];
                out[pm[q]] = (T)2.0 * temp * a.knorm * am * (l < 0 ? (T)-1.0 : (T)1.0);
            }
        }
    }
    if (a.bias) {
        const double bs = block_sum_all<BLK>(asum, sh);
        if (threadIdx.x == 0) a.apart[blockIdx.x] = bs;
    }
    if constexpr (J == 6) {
        double bm = block_max<BLK>(err, sh);
        if (threadIdx.x == 0) a.partial[blockIdx.x] = bm;
    }
}

// ---- clause pass, K <= 10 other than the tiled 3 and 4 ---------------------
// KT: the compile-time bound of K (2, 6, 8 or 10), so that a clause's factors
// and their left-to-right products stay in registers: k_clause_gen keeps them
// in LDS, 64 KB per workgroup in FP64, with 2 K^2 LDS reads per clause and two
// waves per SIMD.  Literals and positions lie by literal, so every load is one
// run per wave.  The product without factor q is the running product of the
// factors before it times those after it: the same multiplications in the same
// order, K (K - 1) / 2 of them.  One clause; results as k_clause_gen's.
// TAB (tanh family, with the wide var pass: few variables in many clauses, as in
// Ramsey encodings): a slot's tanh(q f) depends on its literal alone, so the var
// pass leaves tanh of both factors of every variable in a.th, and the 2.85e6 tanh
// of a stage of R(5,5) at N = 30 become 870.
// Bound by the gathers of the spins and the scattered stores of the terms.
// R(5,5) at N = 30 (tanh, FP64, K = 10, M = 285 012): 50 -> 16 us a pass, 21 with
// the table rebuilt by every workgroup; N = 60 013, M = 231 000, clauses of 2 to 6
// literals, FP32: 15 -> 12 us.
template <typename T, int KT, int J, bool TAB>
__device__ __forceinline__ void clause_k(const StageArgs<T>& a, int m, const T* sp, const T* x, T* xnew,
                                          T hs, double h, double hnext, double floor, double& err,
                                         double& asum)
{
    const int K = a.k;
    int l[KT], at[KT];
    T sv[KT], f[KT], pre[KT + 1];
#pragma unroll
    for (int q = 0; q < KT; q++) {
        l[q] = q < K ? a.litq[(size_t)q * a.mq + m] : 0;
        at[q] = q < K ? a.posq[(size_t)q * a.mq + m] : 0;
    }
    const size_t ai = (size_t)a.aoff + m;
    T k1 = 0, k2 = 0, k3 = 0, k4 = 0, k5 = 0;
    const T xa = x[ai];
    if constexpr (J > 1) k1 = a.k1[ai];
    if constexpr (J > 2) k2 = a.k2[ai];
    if constexpr (J > 3) k3 = a.k3[ai];
    if constexpr (J > 4) k4 = a.k4[ai];
    if constexpr (J > 5) k5 = a.k5[ai];
#pragma unroll
    for (int q = 0; q < KT; q++) sv[q] = (q < K && l[q] != 0) ? sp[l[q] < 0 ? -l[q] : l[q]] : (T)-1.0;
    T km = a.knorm;
    pre[0] = (T)1.0;
#pragma unroll
    for (int q = 0; q < KT; q++) {
        // past K: factor 1, which changes no product
        f[q] = q < K ? (l[q] < 0 ? (T)1.0 + sv[q] : (T)1.0 - sv[q]) : (T)1.0;
        km *= f[q];
        pre[q + 1] = q == 0 ? f[0] : pre[q] * f[q];
    }
    T am;
    if constexpr (J == 1) am = xa;
    else am = stage_input<T, J>(xa, k1, k2, k3, k4, k5, hs);
    const T kj = am * km * km;
    asum = (double)am;
    if constexpr (J == 1) a.k1[ai] = kj;
    else if constexpr (J == 2) a.k2[ai] = kj;
    else if constexpr (J == 3) a.k3[ai] = kj;
    else if constexpr (J == 4) a.k4[ai] = kj;
    else if constexpr (J == 5) a.k5[ai] = kj;
    else {
        T xn;
        final_combination<T>(xa, k1, k3, k4, k5, kj, hs, h, hnext, floor, xn, err);
        xnew[ai] = xn;
    }
    const T r = TAB ? a.knorm * am : km * a.knorm * am;
#pragma unroll
    for (int q = 0; q < KT; q++) {
        if (q < K && l[q] != 0) {      // a clause's padding literals are its last ones
            T p = q == 0 ? (T)1.0 : pre[q];
#pragma unroll
            for (int qq = q + 1; qq < KT; qq++) p = (q == 0 && qq == 1) ? f[1] : p * f[qq];
            T rr;
            if constexpr (TAB) {
                const T ap = p < (T)0 ? -p : p;
                const double t = a.th[2 * (l[q] < 0 ? -l[q] : l[q]) + (l[q] < 0 ? 1 : 0)];
                if constexpr (sizeof(T) == 4) rr = (T)((double)(r * ap) * t);
                else rr = r * ap * t;
                rr = l[q] < 0 ? -rr : rr;
            } else {
                rr = r * p;
                rr *= l[q] < 0 ? (T)-2.0 : (T)2.0;
            }
            a.contrib[at[q]] = rr;
        }
    }
}

template <typename T, int KT, int J, bool TAB>
__global__ __launch_bounds__(BLK) void k_clause_k(StageArgs<T> a)
{
    __shared__ double sh[BLK / 64];
    const Ctrl* c = a.ctrl;
    int parity = 0;
    double h = 0.0, hnext = 0.0, floor = TabD::TINY;
    if (c) {
        if (!c->active) return;
        if (J == 1 && !c->step_start) return;
        parity = c->parity; h = c->h; hnext = c->hnext; floor = c->floor;
    }
    const T* x = parity ? a.xb : a.xa;
    T* xnew = parity ? a.xa : a.xb;
    const int m = clause_of_thread(a.clause_per_xcd);
    double err = 0.0, asum = 0.0;
    if (m < a.m)
        clause_k<T, KT, J, TAB>(a, m, (J == 1) ? x : a.tmp, x, xnew, (T)h, h, hnext, floor, err, asum);
    if (a.bias) {
        const double bs = block_sum_all<BLK>(asum, sh);
        if (threadIdx.x == 0) a.apart[blockIdx.x] = bs;
    }
    if constexpr (J == 6) {
        const double bm = block_max<BLK>(err, sh);
        if (threadIdx.x == 0) a.partial[blockIdx.x] = bm;
    }
}

// tanh(q f) of both factors f = 1 -+ s of a spin, as tanh_term forms it for
// clauses of 3 to 10 literals: half 0 or 1 of the variable's entry
template <typename T>
__device__ __forceinline__ double tanh_half(T sv, T q, int half)
{
    const T f = half ? (T)1.0 + sv : (T)1.0 - sv;
    return tanh((double)(q * f));
}

// the table of a state's spins, before the first stage; the wide var pass then
// keeps it (entry 0, the padding literal's, is never read)
template <typename T>
__global__ __launch_bounds__(BLK) void k_tanh_fill(const T* x, int n, T q, double* th)
{
    const int i = (int)(blockIdx.x * BLK + threadIdx.x);
    if (i < 2 * (n + 1)) th[i] = tanh_half<T>(x[i >> 1], q, i & 1);
}

// ---- var pass: deterministic per-variable sums + spin stage combination ---
// The state values the stage combination of variable i reads (x and the
// earlier stage derivatives it needs), loaded ahead of the sums.
template <typename T>
struct VarIn {
    T x, k1, k2, k3, k4, k5;
};
template <typename T, int J>
__device__ __forceinline__ VarIn<T> var_load(const StageArgs<T>& a, int i, const T* x, bool fresh)
{
    VarIn<T> v;
    v.x = ld_g(x + i);
    v.k1 = v.k2 = v.k3 = v.k4 = v.k5 = (T)0;
    if (J > 1 || !fresh) v.k1 = ld_g(a.k1 + i);
    if (J > 2 && J < 6) v.k2 = ld_g(a.k2 + i);
    if (J > 3) v.k3 = ld_g(a.k3 + i);
    if (J > 4) v.k4 = ld_g(a.k4 + i);
    if (J > 5) v.k5 = ld_g(a.k5 + i);
    return v;
}

// Stage combination of one variable, shared by both var passes.  kj is the
// variable's summed derivative (or, on a retry's J = 1, read back from k1).
// Returns the spin the next clause pass reads: stage J+1's input, or x_new.
template <typename T, int J>
__device__ __forceinline__ T var_stage(const StageArgs<T>& a, int i, bool fresh, T kj, const VarIn<T>& v, T* xnew,
                                       T hs, double h, double hnext, double floor, double& err)
{
    const T xi = v.x;
    T out = (T)0;
    if constexpr (J == 1) {
        if (fresh) st_g(a.k1 + i, kj);
        else kj = v.k1;
        out = stage_input<T, 2>(xi, kj, 0, 0, 0, 0, hs);
        if (a.tmp) a.tmp[i] = out;
    } else if constexpr (J == 2) {
        st_g(a.k2 + i, kj);
        out = stage_input<T, 3>(xi, v.k1, kj, 0, 0, 0, hs);
        a.tmp[i] = out;
    } else if constexpr (J == 3) {
        st_g(a.k3 + i, kj);
        out = stage_input<T, 4>(xi, v.k1, v.k2, kj, 0, 0, hs);
        a.tmp[i] = out;
    } else if constexpr (J == 4) {
        st_g(a.k4 + i, kj);
        out = stage_input<T, 5>(xi, v.k1, v.k2, v.k3, kj, 0, hs);
        a.tmp[i] = out;
    } else if constexpr (J == 5) {
        st_g(a.k5 + i, kj);
        out = stage_input<T, 6>(xi, v.k1, v.k2, v.k3, v.k4, kj, hs);
        a.tmp[i] = out;
    } else {
        double e;
        final_combination<T>(xi, v.k1, v.k3, v.k4, v.k5, kj, hs, h, hnext, floor, out, e);
        err = fmax(err, e);
        st_g(xnew + i, out);
    }
    return out;
}

// Bias term (AnalogSAT/cpu_sat/CpuSat.cpp:232-239, CudaSatBase.cu:75-121):
// mean(a) alpha b knorm^2 pi/2, with mean(a) the stage aux mean.  Every var
// workgroup adds the clause blocks' partial sums in the same order, so all of
// them use the same value.
template <typename T, int BLOCK>
__device__ __forceinline__ T bias_prefactor(const StageArgs<T>& a, double* sh)
{
    // eight loads in flight; added in order
    double v = 0.0;
    for (int i = threadIdx.x; i < a.nblk_clause; i += 8 * BLOCK) {
        double t[8];
#pragma unroll
        for (int u = 0; u < 8; u++) t[u] = i + u * BLOCK < a.nblk_clause ? a.apart[i + u * BLOCK] : 0.0;
#pragma unroll
        for (int u = 0; u < 8; u++)
            if (i + u * BLOCK < a.nblk_clause) v += t[u];
    }
    const double tot = block_sum_all<BLOCK>(v, sh);
    const T mean = (T)tot / (T)a.m;
    return mean * a.alpha * a.bb * (T)1.570796326794897;
}

template <typename T>
__device__ __forceinline__ T bias_sine(T s)
{
    if constexpr (sizeof(T) == 4) return sinf(s * (T)3.141592653589793);
    else return sin(s * (T)3.141592653589793);
}

// LDS var pass: one workgroup per variable group.  The group's whole
// contribution region is read with coalesced 16-byte loads, together with each
// entry's place in the group's var-major slot list, and scattered to those places
// in LDS: every variable's terms then lie side by side, and one thread adds them
// left to right (slot order, the reference's accumulation order) without looking
// up where they are.  With slot spins on, the thread then writes its variable's
// output spin (stage J+1's input, or x_new) over its own terms, and the workgroup
// gathers the region back and streams it to contrib as the next clause pass's
// slot spins.  The two permutations are spread over all 1024 threads; a variable
// that looked up its own terms instead did so with the few waves that a group of
// 128 to 1000 variables has, each entry behind a branch: 6 of the pass's 9 us in a
// workgroup for 4-SAT, N = 20 011, M = 196 107, FP64, against 3 now (us per
// attempt: 147 to 121; 3-SAT, N = 163 840, FP64: 185 to 174; N = 1e6, FP32: 448 to
// 430; N = 60 013, clauses of 3 to 6, FP32: 111 to 102).  The positions that a tile's
// slots take within its run are free, but spreading them over the LDS banks
// (0.2 %) is not worth the work.
// FP32: two 1024-thread workgroups per CU (LDS holds two regions) need 8
// waves per SIMD, which caps the scalar registers: at J = 6 the compiler
// otherwise takes 90 of them, only one workgroup fits, and the pass took 44
// instead of 36 us.  FP64 systems fit one var workgroup per CU anyway.
template <typename T, int J>
__global__ __launch_bounds__(VBLK) __attribute__((amdgpu_waves_per_eu(sizeof(T) == 4 ? 8 : 1)))
void k_var_region(StageArgs<T> a)
{
    constexpr int V = 16 / (int)sizeof(T);
    constexpr int R = sizeof(T) == 4 ? 4 : 6;   // 16-byte loads in flight per thread and round
    typedef T vT __attribute__((ext_vector_type(V)));
    typedef unsigned short vL __attribute__((ext_vector_type(V)));
    __shared__ double sh[VBLK / 64];
    // dynamic LDS: the group's slot list, a place for entries of no slot, and
    // room for the last variable's rounded-up reads
    extern __shared__ __attribute__((aligned(16))) unsigned char var_lds[];
    const Ctrl* c = a.ctrl;
    int parity = 0;
    double h = 0.0, hnext = 0.0, floor = TabD::TINY;
    bool fresh = true;
    if (c) {
        if (!c->active) return;
        parity = c->parity; h = c->h; hnext = c->hnext; floor = c->floor;
        fresh = (J != 1) || c->step_start;
    }
    const T hs = (T)h;
    const T* x = parity ? a.xb : a.xa;
    T* xnew = parity ? a.xa : a.xb;
    const int g = blockIdx.x;
    // The dispatcher gives each CU one workgroup before any gets a second, so
    // workgroups var_stagger .. 2 var_stagger - 1 are the second ones of the
    // first round.  Started together, a CU's two workgroups would load, add
    // and write back in lockstep, and HBM would idle while both add from LDS;
    // the second starts about 8000 cycles later, so their phases alternate
    // (N = 1e6: 31-34 -> 28-29 us per pass at J = 1..5, 36 -> 32 us at J = 6).
    if (g >= a.var_stagger && g < 2 * a.var_stagger) __builtin_amdgcn_s_sleep(127);
    const int i0 = g * a.vg + 1, i1 = (int)std::min<long long>((long long)(g + 1) * a.vg, a.n);
    T* reg = (T*)var_lds;
    T* s_next = a.slot_spins ? a.contrib : nullptr;
    const long long r0 = a.gstart[g];
    const int nreg = (int)(a.gstart[g + 1] - r0) / V;
    const int ebase = a.csr_ptr[i0], nlist = a.csr_ptr[i1 + 1] - ebase;
    // each thread's state values, loaded before the region (groups of at most
    // VP * VBLK variables; larger groups load them in the loop)
    constexpr int VP = J == 6 && sizeof(T) == 4 ? 1 : 2;   // (2 would spill)
    const bool pre = i1 - i0 + 1 <= VP * VBLK;
    VarIn<T> vin[VP];
    int row[VP][2];
    if (pre) {
#pragma unroll
        for (int u = 0; u < VP; u++) {
            const int i = i0 + (int)threadIdx.x + u * VBLK;
            if (i <= i1) {
                row[u][0] = a.csr_ptr[i] - ebase;
                row[u][1] = a.csr_ptr[i + 1] - ebase;
                vin[u] = var_load<T, J>(a, i, x, fresh);
            }
        }
    }
    // the places of this thread's first RP region units, for the way back: FP64
    // keeps them; FP32, with half the registers, would spill, and reads them
    // again (from L2) before it adds
    constexpr bool KEEP = sizeof(T) == 8;
    constexpr int RP = KEEP ? R : 3;
    vL place[RP];
    const vL* const places = (const vL*)(a.rloc + r0);
    if (fresh || s_next) {
        // region sizes are multiples of REGION_ALIGN.  A retry's J = 1 pass
        // needs only the places (for the slot spins).
        const vT* src = (const vT*)(a.contrib + r0);
        // direct primary slots: the group's primary terms, read from the
        // 16-byte unit holding its first clause; the first and the last unit
        // may hold other groups' terms
        const vT* psrc = src;
        const vL* plsrc = places;
        int npv = 0, pb = 0, p0 = 0, p1 = 0;
        if (a.split && fresh) {
            p0 = a.pc0[g];
            p1 = a.pc0[g + 1];
            pb = p0 / V * V;
            psrc = (const vT*)(a.pcontrib + pb);
            plsrc = (const vL*)(a.ploc + pb);
            npv = (p1 - pb + V - 1) / V;
        }
        const int nt = nreg + npv;
        for (int base = 0; base < nt; base += R * VBLK) {
            vT rb[R];
            vL lb[R];
#pragma unroll
            for (int r = 0; r < R; r++) {
                const int v = base + r * VBLK + (int)threadIdx.x;
                if (v < nt) {
                    if (fresh) rb[r] = ld_g(v < nreg ? src + v : psrc + (v - nreg));
                    lb[r] = ld_g(v < nreg ? places + v : plsrc + (v - nreg));
                }
            }
#pragma unroll
            for (int r = 0; r < R; r++) {
                const int v = base + r * VBLK + (int)threadIdx.x;
                if (KEEP && base == 0 && r < RP) place[r] = lb[r];
                if (v < nt && fresh)
#pragma unroll
                    for (int q = 0; q < V; q++) {
                        const int j = pb + (v - nreg) * V + q;
                        const bool own = v < nreg || (j >= p0 && j < p1);
                        reg[own ? (int)lb[r][q] : nlist] = rb[r][q];
                    }
            }
        }
        __syncthreads();
        if (!KEEP && s_next) {
#pragma unroll
            for (int r = 0; r < RP; r++)
                if (r * VBLK + (int)threadIdx.x < nreg) place[r] = ld_g(places + r * VBLK + (int)threadIdx.x);
        }
    }
    double err = 0.0;
    const T pref = (a.bias && fresh) ? bias_prefactor<T, VBLK>(a, sh) : (T)0;
    int u = 0;
    for (int i = i0 + (int)threadIdx.x; i <= i1; i += VBLK, u++) {
        T kj = (T)0;
        int e0, e1;
        VarIn<T> in;
        if (pre) {
            e0 = u == 0 ? row[0][0] : row[VP - 1][0];
            e1 = u == 0 ? row[0][1] : row[VP - 1][1];
            in = u == 0 ? vin[0] : vin[VP - 1];
        } else {
            e0 = a.csr_ptr[i] - ebase;
            e1 = a.csr_ptr[i + 1] - ebase;
            in = var_load<T, J>(a, i, x, fresh);
        }
        if (fresh) {
            // VAR_SUM entries in flight, added left to right; past the row's end
            // a -0, which changes no sum
            T sum = (T)0;
            for (int e = e0; e < e1; e += VAR_SUM) {
                T v[VAR_SUM];
#pragma unroll
                for (int q = 0; q < VAR_SUM; q++) v[q] = reg[e + q];
#pragma unroll
                for (int q = 0; q < VAR_SUM; q++) sum += e + q < e1 ? v[q] : (T)-0.0;
            }
            kj = sum;
            if (a.bias) kj += pref * bias_sine<T>(J == 1 ? x[i] : a.tmp[i]);
        }
        const T out = var_stage<T, J>(a, i, fresh, kj, in, xnew, hs, h, hnext, floor, err);
        if (s_next)
            for (int e = e0; e < e1; e++) reg[e] = out;
    }
    if (s_next) {
        // the region's entries of no slot (alignment padding) are written out
        // too, with whatever the LDS holds; no slot reads them
        __syncthreads();
        vT* dst = (vT*)(s_next + r0);
        auto give = [&](int v, vL l) {
            vT o;
#pragma unroll
            for (int q = 0; q < V; q++) o[q] = reg[l[q]];
            // ordinary stores: the next clause pass reads these lines right away
            dst[v] = o;
        };
#pragma unroll
        for (int r = 0; r < RP; r++)
            if (r * VBLK + (int)threadIdx.x < nreg) give(r * VBLK + (int)threadIdx.x, place[r]);
        for (int v = RP * VBLK + (int)threadIdx.x; v < nreg; v += VBLK) give(v, places[v]);
    }
    if constexpr (J == 6) {
        double bm = block_max<VBLK>(err, sh);
        if (threadIdx.x == 0) a.partial[a.nblk_clause + blockIdx.x] = bm;
    }
}

// Gather var pass, for groups whose region does not fit in LDS.  A block
// owns up to BLK consecutive variables of one group.  Their CSR entries form
// one contiguous range; the block first gathers that whole range into LDS
// with coalesced csr_pos reads and many independent contribution loads in
// flight, then every thread adds its own variable's run from LDS left to
// right (slot order, as the reference accumulates).
constexpr int VAR_STAGE = 6144;   // staged contributions per round (LDS)

template <typename T, int J>
__global__ __launch_bounds__(BLK) void k_var(StageArgs<T> a)
{
    __shared__ double sh[BLK / 64];
    __shared__ T vals[VAR_STAGE];
    const Ctrl* c = a.ctrl;
    int parity = 0;
    double h = 0.0, hnext = 0.0, floor = TabD::TINY;
    bool fresh = true;
    if (c) {
        if (!c->active) return;
        parity = c->parity; h = c->h; hnext = c->hnext; floor = c->floor;
        fresh = (J != 1) || c->step_start;
    }
    const T hs = (T)h;
    const T* x = parity ? a.xb : a.xa;
    T* xnew = parity ? a.xa : a.xb;
    int i1 = 0;
    const int i0 = var_block_range(a.vg, a.vg_blocks, a.ngroups, a.n, i1);
    const int i = (i0 != 0 && i0 + (int)threadIdx.x <= i1) ? i0 + (int)threadIdx.x : 0;
    double err = 0.0;
    const T pref = (a.bias && fresh) ? bias_prefactor<T, BLK>(a, sh) : (T)0;
    T kj = (T)0;
    if (fresh && i0 != 0) {
        const int base = a.csr_ptr[i0], end = a.csr_ptr[i1 + 1];
        const int e0 = i ? a.csr_ptr[i] : 0, e1 = i ? a.csr_ptr[i + 1] : 0;
        T sum = (T)0;
        for (int r0 = base; r0 < end; r0 += VAR_STAGE) {
            const int r1 = std::min(end, r0 + VAR_STAGE);
            for (int e = r0 + threadIdx.x; e < r1; e += BLK) vals[e - r0] = a.contrib[a.csr_pos[e]];
            __syncthreads();
            const int lo = std::max(e0, r0), hi = std::min(e1, r1);
            sum = sum_run(sum, vals, lo - r0, hi - r0);
            __syncthreads();
        }
        kj = sum;
    }
    if (a.bias && fresh && i != 0) kj += pref * bias_sine<T>(J == 1 ? x[i] : a.tmp[i]);
    if (i != 0) var_stage<T, J>(a, i, fresh, kj, var_load<T, J>(a, i, x, fresh), xnew, hs, h, hnext, floor, err);
    if constexpr (J == 6) {
        double bm = block_max<BLK>(err, sh);
        if (threadIdx.x == 0) a.partial[a.nblk_clause + blockIdx.x] = bm;
    }
}

// Wide var pass, for the gather layout when variables have long rows (at
// least WIDE_MIN_ROW contributions on average): one workgroup per variable.
// The variable's contributions pass through two LDS buffers of WIDE_STAGE
// values: while thread 0 adds one buffer in slot order (so the sum is the
// gather kernel's, and the reference's, exactly), waves 1..3 stage the next
// chunk into the other.  The generic clause pass stores a variable's terms side
// by side (wide_run); the tiled one leaves them where csr_pos says.  It is bound
// by that chain of additions, so thread 0 reads the next values while it adds:
// reading 16, waiting and adding them made it 51 us at R(5,5), N = 30, FP64 (6551
// values a row), 43 now; the additions alone are 20, at 3.0 ns each.
constexpr int WIDE_BLK = 256;
constexpr int WIDE_STAGE = 2048;
constexpr long long WIDE_MIN_ROW = 64;

template <typename T, int J>
__global__ __launch_bounds__(WIDE_BLK) void k_var_wide(StageArgs<T> a)
{
    __shared__ double sh[WIDE_BLK / 64];
    __shared__ __attribute__((aligned(16))) T vals[2][WIDE_STAGE];
    __shared__ T s_sine;
    const Ctrl* c = a.ctrl;
    int parity = 0;
    double h = 0.0, hnext = 0.0, floor = TabD::TINY;
    bool fresh = true;
    if (c) {
        if (!c->active) return;
        parity = c->parity; h = c->h; hnext = c->hnext; floor = c->floor;
        fresh = (J != 1) || c->step_start;
    }
    const T hs = (T)h;
    const T* x = parity ? a.xb : a.xa;
    T* xnew = parity ? a.xa : a.xb;
    const int i = (int)blockIdx.x + 1;          // grid: one workgroup per variable 1..n
    const int t = (int)threadIdx.x;
    double err = 0.0;
    // the stage combination's inputs, ahead of the sum
    VarIn<T> in = var_load<T, J>(a, i, x, fresh);
    T sum = (T)0, pref = (T)0;
    if (fresh) {
        const int e0 = a.csr_ptr[i], e1 = a.csr_ptr[i + 1];
        auto at = [&](int e) { return a.contrib[a.csr_pos ? a.csr_pos[e] : e]; };
        // chunk 0 through registers, so that the bias term's sums overlap its loads
        constexpr int U0 = WIDE_STAGE / WIDE_BLK;
        T first[U0];
#pragma unroll
        for (int u = 0; u < U0; u++) {
            const int e = e0 + t + u * WIDE_BLK;
            first[u] = e < e1 ? at(e) : (T)-0.0;
        }
        if (a.bias) {
            if (t == 64) s_sine = bias_sine<T>(J == 1 ? x[i] : a.tmp[i]);
            pref = bias_prefactor<T, WIDE_BLK>(a, sh);
        }
#pragma unroll
        for (int u = 0; u < U0; u++) vals[0][t + u * WIDE_BLK] = first[u];
        __syncthreads();
        for (int r0 = e0, ch = 0; r0 < e1; r0 += WIDE_STAGE, ch++) {
            const int r1 = std::min(e1, r0 + WIDE_STAGE);
            if (t >= 64) {
                // stage chunk ch + 1 into the buffer added in round ch - 1,
                // every load of a thread in flight together
                constexpr int NT = WIDE_BLK - 64, U = (WIDE_STAGE + NT - 1) / NT;
                const int n1 = std::min(e1, r1 + WIDE_STAGE);
                T* dst = vals[(ch + 1) & 1];
                T g[U];
#pragma unroll
                for (int u = 0; u < U; u++) {
                    const int e = r1 + (t - 64) + u * NT;
                    g[u] = e < n1 ? at(e) : (T)-0.0;
                }
#pragma unroll
                for (int u = 0; u < U; u++) {
                    const int o = (t - 64) + u * NT;
                    if (o < WIDE_STAGE) dst[o] = g[u];
                }
            } else if (t == 0) {
                // 16-byte LDS reads, one batch of eight ahead of the additions,
                // which stay in slot order
                constexpr int V = 16 / (int)sizeof(T), B = 8 * V;
                typedef T vT __attribute__((ext_vector_type(V)));
                const T* v = vals[ch & 1];
                // whole batches: past the row's end the buffer holds -0.0,
                // which changes no sum
                const int full = (r1 - r0 + 2 * B - 1) / (2 * B) * (2 * B);
                auto get = [&](vT (&q)[8], int e) {
#pragma unroll
                    for (int u = 0; u < 8; u++) q[u] = *(const vT*)(v + e + u * V);
                };
                auto add = [&](const vT (&q)[8]) {
#pragma unroll
                    for (int u = 0; u < 8; u++)
#pragma unroll
                        for (int w = 0; w < V; w++) sum += q[u][w];
                };
                vT qa[8], qb[8];
                get(qa, 0);
                for (int e = 0; e < full; e += 2 * B) {
                    get(qb, e + B);
                    __builtin_amdgcn_sched_barrier(0);
                    add(qa);
                    // past the last batch: the first again, unused
                    get(qa, e + 2 * B < full ? e + 2 * B : 0);
                    __builtin_amdgcn_sched_barrier(0);
                    add(qb);
                }
            }
            __syncthreads();
        }
    }
    if (t < 64) {
        T out = (T)0;
        if (t == 0) {
            T kj = sum;
            if (a.bias && fresh) kj += pref * s_sine;
            out = var_stage<T, J>(a, i, fresh, kj, in, xnew, hs, h, hnext, floor, err);
        }
        if (a.th) {
            // the next stage's entries of the tanh table, a lane each
            out = __shfl(out, 0, 64);
            if (t < 2) a.th[2 * i + t] = tanh_half<T>(out, a.q, t);
        }
    }
    if constexpr (J == 6) {
        double bm = block_max<WIDE_BLK>(err, sh);
        if (threadIdx.x == 0) a.partial[a.nblk_clause + blockIdx.x] = bm;
    }
}

// ---- control: max-norm + Cash-Karp step control (CpuRungeKutta.cpp:217-267)
__global__ __launch_bounds__(CTRL_BLK) void k_control(Ctrl* c, const double* partial, int np)
{
    __shared__ double sh[CTRL_BLK / 64];
    if (!c->active) return;
    double v = 0.0;
    for (int i = threadIdx.x; i < np; i += CTRL_BLK) v = fmax(v, partial[i]);
    v = block_max<CTRL_BLK>(v, sh);
    if (threadIdx.x != 0) return;
    const double errmax = v / c->eps;
    const double h = c->h;
    c->errmax = errmax;
    c->attempts += 1;
    c->rhscount += c->step_start ? 6 : 5;
    if (errmax <= 1.0) {
        double hn = errmax > TabD::ERRCON ? TabD::SAFETY * h * pow_ctrl(errmax, 5) : 5.0 * h;
        c->hdid = h;
        c->time += h;
        if (c->hlog && c->steps < c->hlog_len) c->hlog[c->steps] = h;
        c->steps += 1;
        c->parity ^= 1;
        c->step_start = 1;
        c->hnext = hn;
        c->h = hn;
        if (c->steps >= c->target) c->active = 0;
    } else {
        double htemp = TabD::SAFETY * h * pow_ctrl(errmax, 4);
        double hn = h >= 0.0 ? fmax(htemp, TabD::HFACTOR * h) : fmin(htemp, TabD::HFACTOR * h);
        c->h = hn;
        c->step_start = 0;
        if (c->time + hn == c->time) {
            c->underflow = 1;
            c->active = 0;
        }
    }
}

__global__ void k_ctrl_begin(Ctrl* c, long long count, int parity)
{
    if (threadIdx.x == 0 && blockIdx.x == 0) {
        c->target = c->steps + count;
        c->parity = parity;
        c->active = (c->underflow || count <= 0) ? 0 : 1;
    }
}

__global__ void k_ctrl_set_eps(Ctrl* c, double eps, double floor)
{
    if (threadIdx.x == 0 && blockIdx.x == 0) {
        c->eps = eps;
        c->floor = floor;
    }
}

// ---- violated-clause count (CpuSat::CalculateClauses semantics) ----------
// At most VIOL_BLOCKS workgroups walk the clauses, and each leaves its count
// in a word of its own, which the host adds up.  One atomic per 256 clauses on
// a single word took 12 ns each, one after another: 69 us at M = 1.39e6 and
// 198 us at M = 4.2e6, for 17 and 50 MB of literals; now 17-20 and
// 57 us.  KT: the clause length at compile time, so that a clause's
// literals and then its spins are loaded together (0: the length k, literal
// by literal until one is true).  Bound by the spin gathers.
constexpr int VIOL_BLOCKS = 1024;
template <typename T, int KT>
__global__ __launch_bounds__(BLK) void k_violations(const int* __restrict__ lit, int m, int k,
                                                    const T* __restrict__ x, int* __restrict__ out)
{
    __shared__ int sh[BLK / 64];
    int viol = 0;
    for (long long j = (long long)blockIdx.x * BLK + threadIdx.x; j < m; j += (long long)gridDim.x * BLK) {
        int sat = 0;
        if constexpr (KT > 0) {
            int l[KT];
            T sv[KT];
#pragma unroll
            for (int q = 0; q < KT; q++) l[q] = lit[j * KT + q];
#pragma unroll
            for (int q = 0; q < KT; q++) sv[q] = x[l[q] < 0 ? -l[q] : l[q]];
#pragma unroll
            for (int q = 0; q < KT; q++) {
                const int t = sv[q] > (T)0;
                sat |= (l[q] != 0) & (l[q] < 0 ? !t : t);   // padding literal is constant FALSE
            }
        } else {
            for (int q = 0; q < k && !sat; q++) {
                const int l = lit[j * k + q];
                if (l == 0) continue;
                const int t = x[l < 0 ? -l : l] > (T)0;
                sat = l < 0 ? !t : t;
            }
        }
        viol += !sat;
    }
    const int s = block_sum<BLK>(viol, sh);
    if (threadIdx.x == 0) out[blockIdx.x] = s;
}

// ---- random numbers: Philox4x32-10 (Salmon, Moraes, Dror, Shaw, SC'11) ----
__device__ __forceinline__ void philox4x32_10(uint32_t ctr[4], uint32_t key0, uint32_t key1)
{
    const uint32_t M0 = 0xD2511F53u, M1 = 0xCD9E8D57u, W0 = 0x9E3779B9u, W1 = 0xBB67AE85u;
#pragma unroll
    for (int r = 0; r < 10; r++) {
        uint64_t p0 = (uint64_t)M0 * ctr[0];
        uint64_t p1 = (uint64_t)M1 * ctr[2];
        uint32_t hi0 = (uint32_t)(p0 >> 32), lo0 = (uint32_t)p0;
        uint32_t hi1 = (uint32_t)(p1 >> 32), lo1 = (uint32_t)p1;
        uint32_t n0 = hi1 ^ ctr[1] ^ key0;
        uint32_t n2 = hi0 ^ ctr[3] ^ key1;
        ctr[0] = n0; ctr[1] = lo1; ctr[2] = n2; ctr[3] = lo0;
        key0 += W0; key1 += W1;
    }
}

template <typename T>
__global__ void k_uniform(T* out, int len, unsigned long long seed, unsigned long long offset)
{
    const long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= len) return;
    unsigned long long idx = offset + (unsigned long long)i;
    uint32_t ctr[4] = {(uint32_t)idx, (uint32_t)(idx >> 32), 0x5EEDu, 0u};
    philox4x32_10(ctr, (uint32_t)seed, (uint32_t)(seed >> 32));
    if constexpr (sizeof(T) == 8) {
        uint64_t v = ((uint64_t)ctr[0] << 32) | ctr[1];
        out[i] = (double)(v >> 11) * 0x1.0p-53;
    } else {
        out[i] = (float)(ctr[0] >> 8) * 0x1.0p-24f;
    }
}

// s = 2u - 1 for spins, a = u + 1 for aux (CpuSat.cpp:127-132); input uniforms
// are laid out in the public order [s, a] inside the state buffer's spin area
// Slot spins of a state: each variable's spin at all of its contribution
// positions (the layout the LDS var pass writes after each stage).
template <typename T>
__global__ __launch_bounds__(VBLK) void k_slot_fill(const T* x, const int* csr_ptr, const uint16_t* rloc,
                                                    const long long* gstart, int vg, int n, T* sl)
{
    extern __shared__ __attribute__((aligned(16))) unsigned char var_lds[];
    T* reg = (T*)var_lds;
    const int g = blockIdx.x;
    const int i0 = g * vg + 1, i1 = (int)std::min<long long>((long long)(g + 1) * vg, n);
    const int ebase = csr_ptr[i0];
    for (int i = i0 + (int)threadIdx.x; i <= i1; i += VBLK) {
        const T v = x[i];
        for (int e = csr_ptr[i] - ebase; e < csr_ptr[i + 1] - ebase; e++) reg[e] = v;
    }
    __syncthreads();
    for (long long r = gstart[g] + threadIdx.x; r < gstart[g + 1]; r += VBLK) sl[r] = reg[rloc[r]];
}

template <typename T>
__global__ void k_set_initial(T* x, int n, int m, int aoff, const T* u, const int* perm)
{
    const long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) {
        x[1 + i] = u[i] * (T)2.0 - (T)1.0;
    } else if (i < (long long)n + m) {
        const int j = (int)(i - n);
        x[aoff + j] = u[n + (perm ? perm[j] : j)] + (T)1.0;
    }
}

// A state in its public order [s, a by clause] from the internal layout, and
// back (perm: processing position -> clause; null: identity).  The host then
// copies one contiguous block: permuting 4.2e6 clause weights on the host took
// longer than the 21 MB copy itself (see state_get_public).  Bound by the
// scattered 4- or 8-byte accesses of the public side.
template <typename T>
__global__ __launch_bounds__(BLK) void k_to_public(const T* __restrict__ x, int n, int m, int aoff,
                                                   const int* __restrict__ perm, T* __restrict__ pub)
{
    const long long i = (long long)blockIdx.x * BLK + threadIdx.x;
    if (i < n) {
        pub[i] = x[1 + i];
    } else if (i < (long long)n + m) {
        const int j = (int)(i - n);
        pub[n + (perm ? perm[j] : j)] = x[aoff + j];
    }
}

template <typename T>
__global__ __launch_bounds__(BLK) void k_from_public(T* __restrict__ x, int n, int m, int aoff,
                                                     const int* __restrict__ perm, const T* __restrict__ pub)
{
    const long long i = (long long)blockIdx.x * BLK + threadIdx.x;
    if (i == 0) x[0] = (T)-1.0;
    if (i < n) {
        x[1 + i] = pub[i];
    } else if (i < (long long)n + m) {
        const int j = (int)(i - n);
        x[aoff + j] = pub[n + (perm ? perm[j] : j)];
    }
}

// plain streaming copy (16 B per lane): the reference point for HBM byte counters
// Practical HBM rate probes: 16 bytes per lane, STREAM_U loads in flight per
// thread before the first use, non-temporal.
constexpr int STREAM_U = 4;
typedef int stream_v4 __attribute__((ext_vector_type(4)));
__global__ __launch_bounds__(256) void k_stream_copy(const stream_v4* __restrict__ src, stream_v4* __restrict__ dst,
                                                     long long n16)
{
    const long long stride = (long long)gridDim.x * 256 * STREAM_U;
    for (long long base = (long long)blockIdx.x * 256 * STREAM_U + threadIdx.x; base < n16; base += stride) {
        stream_v4 r[STREAM_U];
#pragma unroll
        for (int u = 0; u < STREAM_U; u++) {
            const long long i = base + u * 256;
            if (i < n16) r[u] = ld_stream(src + i);
        }
#pragma unroll
        for (int u = 0; u < STREAM_U; u++) {
            const long long i = base + u * 256;
            if (i < n16) st_stream(dst + i, r[u]);
        }
    }
}
// read-only pass; `out` is written only if the data hash to a value that a
// zero-filled source never gives, which keeps the loads
__global__ __launch_bounds__(256) void k_stream_read(const stream_v4* __restrict__ src, int* out, long long n16)
{
    const long long stride = (long long)gridDim.x * 256 * STREAM_U;
    int acc = 0;
    for (long long base = (long long)blockIdx.x * 256 * STREAM_U + threadIdx.x; base < n16; base += stride) {
        stream_v4 r[STREAM_U];
#pragma unroll
        for (int u = 0; u < STREAM_U; u++) {
            const long long i = base + u * 256;
            r[u] = i < n16 ? ld_stream(src + i) : stream_v4{0, 0, 0, 0};
        }
#pragma unroll
        for (int u = 0; u < STREAM_U; u++) acc ^= r[u].x ^ r[u].y ^ r[u].z ^ r[u].w;
    }
    if (acc == 0x7fffffff) out[0] = acc;
}

__global__ void k_copy16(const int4* __restrict__ src, int4* __restrict__ dst, long long n16)
{
    for (long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x; i < n16; i += (long long)gridDim.x * blockDim.x)
        dst[i] = src[i];
}

template <typename T>
__global__ void k_fill_const(T* x)
{
    if (threadIdx.x == 0 && blockIdx.x == 0) x[0] = (T)-1.0;
}

// ===========================================================================
// host objects
// ===========================================================================
template <typename T>
static void dfree(T*& p)
{
    if (p) { (void)hipFree((void*)p); p = nullptr; }
}

struct Sys;

struct State {
    Sys* sys = nullptr;
    void* d = nullptr;     // device buffer of the system's precision
    int alloc = 0;
    unsigned long long gen = 0;   // the system's problem generation when the state was made
};

struct Sys {
    int prec = ASAT_F64;
    int esize = 8;
    double b = 0.0;
    int n = 0, m = 0, k = 0, aoff = 0, alloc = 0;
    long long nslots = 0;
    hipStream_t stream = nullptr;
    int* d_lit = nullptr;
    int* d_pos = nullptr;        // generic-K clause pass only
    int *d_litq = nullptr, *d_posq = nullptr;   // the same by literal, K <= 10
    int mq = 0;
    double* d_th = nullptr;      // tanh table (generic pass with the wide var pass)
    bool wide_run = false;       // wide var pass: a variable's contributions lie side by side
    int* d_spos = nullptr;       // tiled clause pass (K = 3, 4)
    uint16_t* d_srank = nullptr;
    unsigned* d_runs = nullptr;  // big tiles: run tables in place of d_spos
    int run_stride = 0;
    int* d_csr_ptr = nullptr;
    int* d_csr_pos = nullptr;    // gather var pass only
    uint16_t* d_rloc = nullptr;      // LDS var pass only
    uint16_t* d_ploc = nullptr;      // and only with direct primary slots
    long long* d_gstart = nullptr;
    int* d_pvar = nullptr;       // direct primary slots: primary variable per clause
    uint16_t* d_pw16 = nullptr;  // big tiles: primary word per clause (in place of d_pvar)
    int* d_pv0 = nullptr;        // big tiles: first primary variable of each tile
    int* d_pc0 = nullptr;        // direct primary slots: first clause of each group's primaries
    void* d_pcontrib = nullptr;  // direct primary slots: primary term per clause
    bool split = false;          // direct primary slots (tiled pass + LDS var pass)
    int* d_perm = nullptr;       // processing position -> clause index (null: identity)
    std::vector<int> perm;       // host copy, for the public <-> internal a-block order
    // one-workgroup path (asat_small.h) for problems whose integrator fits in
    // LDS: each slot's position in var-major order (a variable's terms in the
    // reference's accumulation order) and each variable's range of positions;
    // small_lds = 0 when the problem is too big
    int* d_vptr = nullptr;
    int* d_spos_small = nullptr;
    int nlist = 0;
    int runlen = 0;                // uniform run length of the lists (0: ragged)
    long long small_lds = 0;
    // few-workgroup persistent path (asat_grid.h), laid out when an integrator
    // first asks for it; grid_wgs = 0 when the problem does not use it
    std::mutex grid_lock;
    std::atomic<bool> grid_due{false};   // the problem may use it and has not been laid out
    int* d_grid = nullptr;               // one block: the arrays below
    const uint32_t* d_gcode = nullptr;
    const int *d_gcpos = nullptr, *d_gwg = nullptr, *d_ggroup = nullptr, *d_gvmap = nullptr;
    int grid_wgs = 0, grid_cpt = 0, grid_groups = 0;
    long long grid_lds = 0;
    int vg = 0, ngroups = 0, vg_blocks = 0;
    int family = ASAT_FAMILY_CTDS;
    double q = 1.1;              // tanh family parameter (CpuSatTanh.cpp:39)
    bool tiled = false;          // clause pass: tiled kernel (K = 3, 4) or generic
    int tc = TC;                 // tiled pass: clauses per tile (TC or TC_BIG)
    bool lds_var = false;        // var pass: LDS region kernel or gather kernel
    bool wide_var = false;       // gather path with long rows: one workgroup per variable
    int var_lds = 0;             // LDS region kernel: dynamic LDS bytes (a group's slot list)
    int var_stagger = 0;         // LDS region kernel: CUs whose second workgroup starts late
    void* d_contrib = nullptr;
    double* d_apart = nullptr;   // bias term: per clause-block aux sums
    void* d_public = nullptr;    // a state in public order, on its way to or from the host
    std::mutex public_lock;      // its use
    int* d_count = nullptr;      // violated clauses per workgroup of k_violations
    bool ready = false;
    // bumped by every SetProblem: states and integrators record the value
    // they were made for, and a later problem (even one of the same size)
    // invalidates them
    unsigned long long gen = 0;

    void free_problem()
    {
        dfree(d_lit); dfree(d_pos); dfree(d_litq); dfree(d_posq); dfree(d_th); dfree(d_spos);
        dfree(d_srank); dfree(d_csr_ptr); dfree(d_csr_pos);
        dfree(d_runs);
        run_stride = 0;
        dfree(d_rloc); dfree(d_ploc); dfree(d_gstart); dfree(d_perm); dfree(d_contrib); dfree(d_apart);
        dfree(d_pvar); dfree(d_pc0); dfree(d_pcontrib); dfree(d_pw16); dfree(d_pv0);
        split = false;
        dfree(d_vptr); dfree(d_spos_small); dfree(d_public);
        dfree(d_grid);
        grid_wgs = 0;
        grid_due = false;
        perm.clear();
        nlist = 0;
        runlen = 0;
        small_lds = 0;
    }
    ~Sys()
    {
        free_problem();
        dfree(d_count);
        if (stream) (void)hipStreamDestroy(stream);
    }
    void require_ready() const { require(ready, ASAT_ERR_NOT_CONFIGURED, "SAT problem has not been set"); }
};

// clause-pass and var-pass grid sizes of a configured system
static int clause_grid(const Sys* s) { return 8 * ceil_div(s->tiled ? ceil_div(s->m, s->tc) : ceil_div(s->m, BLK), 8); }
static int var_grid(const Sys* s)
{
    if (s->lds_var) return s->ngroups;
    if (s->wide_var) return s->n;
    return 8 * s->vg_blocks * ceil_div(s->ngroups, 8);
}

struct Rng {
    unsigned long long seed = 0, offset = 0;
};

template <typename V>
static void upload(V*& d, const std::vector<V>& h)
{
    HIP_CHECK(hipMalloc((void**)&d, sizeof(V) * std::max<size_t>(h.size(), 1)));
    if (!h.empty()) HIP_CHECK(hipMemcpy(d, h.data(), sizeof(V) * h.size(), hipMemcpyHostToDevice));
}

// Variable groups for the LDS var pass: about 2048 (float) / 1024 (double)
// variables per group, a multiple of 256 groups once there are more than
// 256 (one workgroup per CU per round), at least 256 groups while groups
// keep 128+ variables (4-SAT, N = 20 011, M = 196 107: 143 us per attempt with
// FP64 and 115 with FP32, against 152 and 120 with 256+; sizes with 256 groups
// either way are the same); halved until the largest region fits in LDS (counted
// with two bytes more per entry, from when the pass kept offsets beside it).  When no
// size fits (a variable with more occurrences than the LDS holds), the gather
// var pass runs with ~400 KB regions.
// LDS of the region var pass: the longest group's slot list, a place for entries
// of no slot, and the rounded-up reads past the last variable's terms
static int var_lds_bytes(int max_list, int esize) { return (int)round_up((max_list + 1 + VAR_SUM) * esize, 16); }

static bool choose_layout(HostProblem& P, int esize)
{
    const long long cap = (VAR_LDS_BYTES - 48) / (esize + 2);
    const long long target = esize == 4 ? 2048 : 1024;
    long long G = std::max(ceil_div((long long)P.n, target), std::min(256, ceil_div((long long)P.n, 128)));
    if (G > 256) G = round_up(G, 256);
    int vg = ceil_div((long long)P.n, G);
    // direct primary slots wherever the tiled pass meets the LDS var pass
    // (primary variables exist only for the tiled pass's clause order)
    const int pv = 16 / esize;
    for (;;) {
        if (build_layout(P, vg, pv, cap)) return true;
        if (vg <= 64) break;
        vg = (vg + 1) / 2;
    }
    build_layout(P, esize == 4 ? 8192 : 4096, 0, 0);
    return false;
}

// Var-major term positions of the one-workgroup path, when its LDS
// footprint fits: variable v's terms occupy positions vptr[v] .. vptr[v+1]-1,
// its slots taken with clauses in input order and literals in clause order
// (the order CpuSat::CalculateAllEx adds them, AnalogSAT/cpu_sat/CpuSat.cpp:
// 206-229); spos[j*K + q] is the position of processing-order slot (j, q).
static void build_small_lists(Sys* s, const HostProblem& P)
{
    const int n = P.n, m = P.m, K = P.k;
    if (small_lds_bytes(n, m, K, s->alloc, 0, s->esize) > SMALL_LDS_MAX) return;    // without any list
    std::vector<int> vptr((size_t)n + 2), spos((size_t)m * K), visit;
    if (!P.perm.empty()) {
        visit.resize((size_t)m);
        for (int p = 0; p < m; p++) visit[(size_t)P.perm[p]] = p;
    }
    long long nl = 0;
    const int runlen = small_build_lists(P.lit.data(), visit.empty() ? nullptr : visit.data(), n, m, K, s->alloc,
                                         s->esize, vptr.data(), spos.data(), &nl);
    const long long bytes = small_lds_bytes(n, m, K, s->alloc, nl, s->esize);
    if (bytes > SMALL_LDS_MAX) return;
    upload(s->d_vptr, vptr);
    upload(s->d_spos_small, spos);
    s->nlist = (int)nl;
    s->runlen = runlen;
    s->small_lds = bytes;
}

// Layout of the few-workgroup path (asat_grid.h).  Variables are ranked by
// falling number of occurrences and dealt out in groups of 64, so workgroups
// get the same work and a group's rows of terms are nearly full.  The workgroup
// count is the smallest of 8, 16, .. whose largest clause list is two per
// thread; from 64 on, as many per thread as the registers hold come before more
// workgroups.  us per attempt with 8 / 16 / 32 / 64 / 128 workgroups:
//   N =  2000, M =  8500, FP32   22.5 / 20.6 / 22.6 / 28.1 / 33.4
//   N =  5000, M = 21250, FP32   36.5 / 31.8 / 30.9 / 32.9 / 39.1
//   N = 12000, M = 51120, FP64      - /    - /    - / 59.9 / 69.5
// The layout ends where the spins of all variables no longer fit in LDS or the
// clauses in registers; grid_gain says which calls take it.
constexpr int GRID_CPT_F64 = 4, GRID_CPT_F32 = 8;
constexpr long long GRID_LDS = 158 * 1024;     // beside the kernel's 0.3 KB of static LDS

// Workgroups of 1024 threads that the device holds at once: one on each CU (the
// kernels use more than half of the registers).  An MI355X has 256 CUs, a partition of it may have fewer than a
// layout has workgroups.  (The runtime's occupancy query is no guide: with a second
// ROCm's libraries loaded before the first GPU call, as PyTorch's are when imported in
// between, it counts half the registers and finds room for none.)
static int grid_resident()
{
    int dev = 0, ncu = 0;
    HIP_CHECK(hipGetDevice(&dev));
    HIP_CHECK(hipDeviceGetAttribute(&ncu, hipDeviceAttributeMultiprocessorCount, dev));
    return ncu;
}

// lit: m K literals in processing order, as SetProblem left them
static void build_grid(Sys* s, const std::vector<int>& lit)
{
    const int n = s->n, m = s->m, K = s->k;
    const int ng = ceil_div(n, 64), nranks = 64 * ng;
    const size_t slots = (size_t)m * K;
    std::vector<int> deg((size_t)n + 1, 0);
    for (size_t sl = 0; sl < slots; sl++)
        if (lit[sl]) deg[(size_t)std::abs(lit[sl])]++;
    int top = 0;
    for (int v = 1; v <= n; v++) top = std::max(top, deg[(size_t)v]);
    std::vector<int> vmap((size_t)nranks, 0), rank((size_t)n + 1, 0), at((size_t)top + 2, 0);
    for (int v = 1; v <= n; v++) at[(size_t)(top - deg[(size_t)v]) + 1]++;
    for (int d = 0; d <= top; d++) at[(size_t)d + 1] += at[(size_t)d];
    for (int v = 1; v <= n; v++) {
        const int r = at[(size_t)(top - deg[(size_t)v])]++;
        rank[(size_t)v] = r;
        vmap[(size_t)r] = v;
    }
    // the rank of every slot's variable, -1 for padding (a clause's last literals)
    std::vector<int> srank(slots);
    for (size_t sl = 0; sl < slots; sl++) srank[sl] = lit[sl] ? rank[(size_t)std::abs(lit[sl])] : -1;
    // the workgroups of a clause, the first literal's first (it writes the clause);
    // g: workgroups, a power of two
    auto owners = [&](int j, int g, int (&w)[4]) {
        const int* r = srank.data() + (size_t)j * K;
        int ns = 0;
        for (int q = 0; q < K && r[q] >= 0; q++) {
            const int x = (r[q] >> 6) & (g - 1);
            bool dup = false;
            for (int i = 0; i < ns; i++) dup |= w[i] == x;
            if (!dup) w[ns++] = x;
        }
        return ns;
    };
    const int cpt_max = s->esize == 8 ? GRID_CPT_F64 : GRID_CPT_F32;
    std::vector<int> nwrite((size_t)GRID_MAX), nother((size_t)GRID_MAX);
    int G = 0, most = 0, w4[4];
    // one workgroup alone while its threads hold the clauses (us per attempt
    // against 8 workgroups: N = 480, FP64 10.5 / 16.4, N = 960, FP32 13.2 / 16.6,
    // 4-SAT N = 200, FP64 14.1 / 21.1)
    const int solo_max = (s->esize == 8 ? 2 : 4) * GRID_BT;
    for (int g = n <= 64 * GRID_WAVES && m <= solo_max ? 1 : 8; g <= GRID_MAX; g = g == 1 ? 8 : 2 * g) {
        if (ceil_div(ng, g) > GRID_WAVES) continue;
        // a random instance's clauses are spread over nearly K workgroups each:
        // skip counts that cannot hold them
        if (g > 1 && g < GRID_MAX && (long long)m * (K - 1) > (long long)g * GRID_BT * cpt_max) continue;
        std::fill(nwrite.begin(), nwrite.end(), 0);
        std::fill(nother.begin(), nother.end(), 0);
        for (int j = 0; j < m; j++) {
            const int ns = owners(j, g, w4);
            nwrite[(size_t)w4[0]]++;
            for (int i = 1; i < ns; i++) nother[(size_t)w4[i]]++;
        }
        most = 0;
        for (int w = 0; w < g; w++) most = std::max(most, nwrite[(size_t)w] + nother[(size_t)w]);
        G = g;
        if (g == 1 || most <= 2 * GRID_BT || (g >= 64 && most <= cpt_max * GRID_BT)) break;
    }
    const int cpt = ceil_div(most, GRID_BT);
    if (G == 0 || cpt > cpt_max) return;
    // rows of terms: base of each group inside its workgroup
    std::vector<int> group((size_t)2 * ng), ncon((size_t)G, 0);
    for (int g = 0; g < ng; g++) {
        const int depth = deg[(size_t)vmap[(size_t)64 * g]];
        group[(size_t)2 * g] = ncon[(size_t)(g % G)];
        group[(size_t)2 * g + 1] = depth;
        ncon[(size_t)(g % G)] += 64 * depth;
    }
    const int most_con = *std::max_element(ncon.begin(), ncon.end());
    const long long lds = (long long)s->esize * (nranks + 2 + most_con + 1);
    if (most_con > 65535 || lds > GRID_LDS) return;
    const int kcpt = cpt <= 1 ? 1 : cpt <= 2 ? 2 : cpt <= 4 ? 4 : 8;
    const void* f = grid_kernel(s->prec, K, kcpt, G == 1);
    require(f != nullptr, ASAT_ERR_HIP, "no few-workgroup kernel for this layout");
    HIP_CHECK(hipFuncSetAttribute(f, hipFuncAttributeMaxDynamicSharedMemorySize, (int)GRID_LDS));
    if (G > 1 && grid_resident() < G) return;
    // term entry of every slot in its variable's workgroup: the variable's clauses
    // in input order, literals in clause order (the reference's accumulation order)
    std::vector<int> visit((size_t)m), fill((size_t)nranks), entry(slots);
    for (int p = 0; p < m; p++) visit[(size_t)(s->perm.empty() ? p : s->perm[(size_t)p])] = p;
    for (int r = 0; r < nranks; r++) fill[(size_t)r] = group[(size_t)2 * (r / 64)] + r % 64;
    for (int c = 0; c < m; c++)
        for (int q = 0; q < K; q++) {
            const size_t sl = (size_t)visit[(size_t)c] * K + q;
            if (srank[sl] < 0) break;
            entry[sl] = fill[(size_t)srank[sl]];
            fill[(size_t)srank[sl]] += 64;
        }
    int total = 0;
    std::vector<int> fw((size_t)G), fo((size_t)G);
    std::vector<int> wg((size_t)4 * G);
    for (int w = 0; w < G; w++) {
        const int nw = nwrite[(size_t)w], nc = nw + nother[(size_t)w];
        wg[(size_t)4 * w] = total;
        wg[(size_t)4 * w + 1] = nc;
        wg[(size_t)4 * w + 2] = nw;
        wg[(size_t)4 * w + 3] = ncon[(size_t)w];
        fw[(size_t)w] = total;
        fo[(size_t)w] = total + nw;
        total += nc;
    }
    // one block: codes, positions, workgroups, groups, rank -> variable
    std::vector<int> blk;
    const size_t ncode = (size_t)total * K;
    blk.reserve(ncode + (size_t)total + wg.size() + group.size() + vmap.size());
    blk.resize(ncode + (size_t)total);
    for (int j = 0; j < m; j++) {
        const int ns = owners(j, G, w4);
        for (int i = 0; i < ns; i++) {
            const int w = w4[i], to = (i ? fo : fw)[(size_t)w]++;
            blk[ncode + (size_t)to] = j;
            for (int q = 0; q < K; q++) {
                const size_t sl = (size_t)j * K + q;
                const int r = srank[sl];
                uint32_t where = (uint32_t)ncon[(size_t)w], rk = (uint32_t)nranks;
                if (r >= 0) {
                    rk = (uint32_t)r;
                    if (((r >> 6) & (G - 1)) == w) where = (uint32_t)entry[sl];
                }
                blk[(size_t)to * K + q] = (int)((where << 16) | (rk << 1) | (lit[sl] < 0 ? 1u : 0u));
            }
        }
    }
    blk.insert(blk.end(), wg.begin(), wg.end());
    blk.insert(blk.end(), group.begin(), group.end());
    blk.insert(blk.end(), vmap.begin(), vmap.end());
    upload(s->d_grid, blk);
    s->d_gcode = (const uint32_t*)s->d_grid;
    s->d_gcpos = s->d_grid + ncode;
    s->d_gwg = s->d_gcpos + total;
    s->d_ggroup = s->d_gwg + wg.size();
    s->d_gvmap = s->d_ggroup + group.size();
    s->grid_cpt = kcpt;
    s->grid_groups = ng;
    s->grid_lds = lds;
    s->grid_wgs = G;
}

// The layout, at the first integrator that can use it: a system that only serves
// GetDerivatives, the tanh family or a bias term never pays for it (N = 2000,
// M = 8500 0.5 ms, N = 24 000, M = 102 000 3 ms).  Integrators of one system may ask from
// several threads.  Without memory for it the problem goes without.
static void ensure_grid(Sys* s)
{
    if (!s->grid_due) return;
    std::lock_guard<std::mutex> lock(s->grid_lock);
    if (!s->grid_due) return;
    const int nranks = 64 * ceil_div(s->n, 64), cpt = s->esize == 8 ? GRID_CPT_F64 : GRID_CPT_F32;
    if (nranks + 2 <= 32766 && (long long)s->esize * nranks <= GRID_LDS && s->m <= (long long)GRID_MAX * GRID_BT * cpt) {
        std::vector<int> lit((size_t)s->m * s->k);
        HIP_CHECK(hipMemcpy(lit.data(), s->d_lit, sizeof(int) * lit.size(), hipMemcpyDeviceToHost));
        try {
            build_grid(s, lit);
        } catch (const Error&) {
            (void)hipGetLastError();
            dfree(s->d_grid);
        }
    }
    s->grid_due = false;
}

static void sys_set_problem(Sys* s, const int* lits, const int* lens, int nclauses)
{
    HostProblem P;
    parse_clauses(lits, lens, nclauses, P);
    const bool tiled = P.k == 3 || P.k == 4;
    if (tiled && REORDER_CLAUSES) reorder_clauses(P);
    const bool lds_var = choose_layout(P, s->esize);
    int ncu = 0;
    {
        int dev = 0;
        HIP_CHECK(hipGetDevice(&dev));
        HIP_CHECK(hipDeviceGetAttribute(&ncu, hipDeviceAttributeMultiprocessorCount, dev));
    }
    // FP32 3-literal clauses with direct primary slots: big tiles (the
    // kernel takes their clauses one at a time, and two workgroups still fit
    // on a CU), sized so that they fill whole rounds of the 2 x CUs resident
    // workgroups: N = 1e6, M = 4.2e6 gets 1010 tiles of 4160 clauses, two rounds.
    // Problems too small to give every resident workgroup 2048 clauses keep
    // 2048-clause tiles: with few waves per CU a thread's clauses taken one
    // after another expose their load latency (N = 2000: 16-18 us per pass
    // against 5-7 us; M = 6e5 in 1216-clause tiles: 11 us against 8 us)
    P.tc = TC;
    if (tiled && P.split && s->esize == 4 && P.k == 3) {
        const long long slots = 2LL * (ncu > 0 ? ncu : 1);
        const long long rounds = std::max<long long>(1, ceil_div((long long)P.m, slots * TC_BIG));
        const long long ts = round_up(ceil_div((long long)P.m, rounds * slots), 64);
        P.tc = ts < TC ? TC : (int)std::min<long long>(ts, TC_BIG);
        // big tiles rebuild their sorted positions from run tables, a word
        // per variable group: worth it while that is at most a quarter of
        // the positions (ngroups + 1 <= tc (K - 1) / 4)
        if (P.tc != TC && (long long)(P.ngroups + 1) * 4 > (long long)P.tc * (P.k - 1)) P.tc = TC;
        // primary words hold a clause's primary variable relative to its
        // tile's first: tiles spanning more variables keep 2048 clauses
        for (long long j0 = 0; P.tc != TC && j0 < P.m; j0 += P.tc) {
            const long long j1 = std::min<long long>(P.m, j0 + P.tc) - 1;
            if (P.pvar[(size_t)j1] - P.pvar[(size_t)j0] > (int)PW_VMASK) P.tc = TC;
        }
    }
    // Other problems of 16 tiles and more, but FP32 3-literal ones: tiles of 512 to
    // 2048 clauses, sized so that they fill whole rounds of one workgroup per CU (us
    // per attempt with 2048-clause tiles and these: FP64, 3-SAT, N = 20 011: 83 and
    // 70, 40 000: 98 and 88, 163 840: 170 and 166, 400 000: 346 and 340, the last
    // two 157 and 322 since two of their workgroups fit on a CU; 4-SAT, N = 20 011:
    // 121 and 109, 60 000: 200 and 187; FP32, 4-SAT, N = 20 011: 95 and 90,
    // 100 000: 190 both; 3-SAT, N = 20 011: 59 both, so 2048 stays there).
    if (tiled && P.tc == TC && P.m >= 16 * TC && (s->esize == 8 || P.k == 4)) {
        const long long cus = ncu > 0 ? ncu : 1;
        const long long rounds = ceil_div((long long)P.m, cus * TC);
        P.tc = (int)std::max<long long>(512, round_up(ceil_div((long long)P.m, rounds * cus), 64));
    }
    if (tiled) build_tile_order(P);
    HIP_CHECK(hipStreamSynchronize(s->stream));
    s->free_problem();
    s->ready = false;
    s->gen++;
    s->n = P.n; s->m = P.m; s->k = P.k;
    s->aoff = (int)round_up((long long)P.n + 1, 64);
    s->alloc = (int)(s->aoff + round_up(P.m, 64));
    s->nslots = (long long)P.m * P.k;
    s->vg = P.vg;
    s->ngroups = P.ngroups;
    s->vg_blocks = ceil_div(P.vg, BLK);
    s->tiled = tiled;
    s->tc = P.tc;
    s->lds_var = lds_var;
    s->split = P.split;
    require(!P.split || (tiled && lds_var), ASAT_ERR_INVALID_ARGUMENT, "direct primary slots without their passes");
    // few variables with long rows (dense problems such as Ramsey encodings):
    // the gather kernel would add a block's rows one after another, so each
    // variable gets a workgroup of its own
    s->wide_var = !lds_var && s->nslots >= WIDE_MIN_ROW * (long long)P.n;
    // the generic clause pass can store anywhere: a variable's terms side by side
    s->wide_run = s->wide_var && !tiled;
    if (s->wide_run) {
        std::vector<int> fill(P.csr_ptr.begin(), P.csr_ptr.end() - 1);
        for (size_t sl = 0; sl < P.lit.size(); sl++)
            if (P.lit[sl]) P.pos[sl] = fill[(size_t)std::abs(P.lit[sl])]++;
    }
    int max_list = 0;
    for (int i = 1; i <= P.n; i += P.vg)
        max_list = std::max(max_list, P.csr_ptr[std::min(P.n + 1, i + P.vg)] - P.csr_ptr[i]);
    s->var_lds = lds_var ? var_lds_bytes(max_list, s->esize) : 0;
    // two FP32 var workgroups per CU (LDS for both; the FP64 kernel's
    // registers allow one) and more groups than CUs: stagger the pairs
    s->var_stagger = 0;
    if (lds_var && s->esize == 4 && 2LL * s->var_lds <= VAR_LDS_CU && ncu > 0 && P.ngroups > ncu)
        s->var_stagger = ncu;
    // clause arrays padded to whole tiles (padding literal 0, position -1)
    const size_t mpad = (size_t)round_up(P.m, P.tc);
    P.lit.resize(mpad * P.k, 0);
    upload(s->d_lit, P.lit);
    if (tiled) {
        if (P.runs.empty()) upload(s->d_spos, P.spos);
        else upload(s->d_runs, P.runs);
        s->run_stride = P.run_stride;
        upload(s->d_srank, P.srank);
        if (P.split) {
            if (P.pw16.empty()) {
                P.pvar.resize(mpad, 0);   // padding clauses: variable 0
                upload(s->d_pvar, P.pvar);
            } else {
                upload(s->d_pw16, P.pw16);
                upload(s->d_pv0, P.pv0);
            }
            upload(s->d_pc0, P.pc0);
            // one term per clause padded to whole tiles, plus a 16-byte unit
            const size_t np = mpad + 16;
            HIP_CHECK(hipMalloc(&s->d_pcontrib, (size_t)s->esize * np));
            HIP_CHECK(hipMemsetAsync(s->d_pcontrib, 0, (size_t)s->esize * np, s->stream));
        }
    } else {
        s->mq = 0;
        if (P.k <= 10) {
            // literals and positions by literal (k_clause_k)
            s->mq = (int)round_up((long long)P.m, BLK);
            std::vector<int> lq((size_t)s->mq * P.k, 0), pq((size_t)s->mq * P.k, 0);
            for (int j = 0; j < P.m; j++)
                for (int q = 0; q < P.k; q++) {
                    lq[(size_t)q * s->mq + j] = P.lit[(size_t)j * P.k + q];
                    pq[(size_t)q * s->mq + j] = P.pos[(size_t)j * P.k + q];
                }
            upload(s->d_litq, lq);
            upload(s->d_posq, pq);
            if (s->wide_var && (s->esize == 8 || P.k >= 3))
                HIP_CHECK(hipMalloc((void**)&s->d_th, sizeof(double) * 2 * ((size_t)P.n + 1)));
        }
        // k_clause_gen's positions: more than 10 literals, or the tanh family
        // without its table
        if (!s->d_th) {
            P.pos.resize(mpad * P.k, -1);
            upload(s->d_pos, P.pos);
        }
    }
    upload(s->d_csr_ptr, P.csr_ptr);
    if (lds_var) {
        upload(s->d_rloc, P.rloc);
        if (P.split) {
            P.ploc.resize(mpad + 16, 0);
            upload(s->d_ploc, P.ploc);
        }
    }
    else if (!s->wide_run) upload(s->d_csr_pos, P.csr_pos);
    upload(s->d_gstart, P.gstart);
    build_small_lists(s, P);
    if (!P.perm.empty()) upload(s->d_perm, P.perm);
    s->perm = std::move(P.perm);
    const size_t ncontrib = (size_t)P.gstart[P.ngroups] + REGION_ALIGN;
    HIP_CHECK(hipMalloc(&s->d_contrib, (size_t)s->esize * ncontrib));
    HIP_CHECK(hipMemsetAsync(s->d_contrib, 0, (size_t)s->esize * ncontrib, s->stream));
    HIP_CHECK(hipMalloc((void**)&s->d_apart, sizeof(double) * clause_grid(s)));
    HIP_CHECK(hipMemsetAsync(s->d_apart, 0, sizeof(double) * clause_grid(s), s->stream));
    // up to 512 clauses and variables asat_small.h is the faster one
    s->grid_due = tiled && (s->small_lds == 0 || std::max(P.m, P.n) > 512);
    s->ready = true;
}

static State* state_new(Sys* s)
{
    s->require_ready();
    std::unique_ptr<State> st(new State());
    st->sys = s;
    st->alloc = s->alloc;
    st->gen = s->gen;
    HIP_CHECK(hipMalloc(&st->d, (size_t)s->esize * s->alloc));
    HIP_CHECK(hipMemsetAsync(st->d, 0, (size_t)s->esize * s->alloc, s->stream));
    if (s->prec == ASAT_F64) hipLaunchKernelGGL(k_fill_const<double>, dim3(1), dim3(64), 0, s->stream, (double*)st->d);
    else hipLaunchKernelGGL(k_fill_const<float>, dim3(1), dim3(64), 0, s->stream, (float*)st->d);
    HIP_CHECK(hipGetLastError());
    HIP_CHECK(hipStreamSynchronize(s->stream));
    return st.release();
}

static void state_check(const State* st)
{
    require(st && st->sys, ASAT_ERR_INVALID_ARGUMENT, "null state");
    require(st->alloc == st->sys->alloc && st->gen == st->sys->gen && st->sys->ready, ASAT_ERR_INVALID_ARGUMENT,
            "state does not belong to the current problem");
}

// Host copies of a state go through one device block in public order
// (k_to_public / k_from_public), allocated at the first such copy of a problem
// and kept with the system; the lock covers states of one system copied from
// several threads.
static void* public_block(Sys* s)
{
    if (!s->d_public) HIP_CHECK(hipMalloc(&s->d_public, (size_t)s->esize * ((size_t)s->n + s->m)));
    return s->d_public;
}

static void state_set_public(State* st, const void* pub)
{
    state_check(st);
    Sys* s = st->sys;
    std::lock_guard<std::mutex> lock(s->public_lock);
    void* blk = public_block(s);
    const size_t len = (size_t)s->n + s->m;
    const dim3 g(ceil_div((long long)len, BLK)), b(BLK);
    HIP_CHECK(hipMemcpyAsync(blk, pub, s->esize * len, hipMemcpyHostToDevice, s->stream));
    if (s->prec == ASAT_F64)
        hipLaunchKernelGGL(k_from_public<double>, g, b, 0, s->stream, (double*)st->d, s->n, s->m, s->aoff,
                           (const int*)s->d_perm, (const double*)blk);
    else
        hipLaunchKernelGGL(k_from_public<float>, g, b, 0, s->stream, (float*)st->d, s->n, s->m, s->aoff,
                           (const int*)s->d_perm, (const float*)blk);
    HIP_CHECK(hipGetLastError());
    HIP_CHECK(hipStreamSynchronize(s->stream));
}

// N = 1e6, M = 4.2e6, FP32: 10.5 ms with the clause weights permuted on
// the host through a second buffer, 1.6 ms now (a 21 MB copy into memory
// the caller has not touched yet).  Weights in clause order are copied as they lie:
// through the block, N = 5000, M = 5000, 2 literals takes 27 us instead of 22.
static void state_get_public(const State* st, void* pub)
{
    state_check(st);
    Sys* s = st->sys;
    if (s->perm.empty()) {
        const size_t e = (size_t)s->esize;
        HIP_CHECK(hipStreamSynchronize(s->stream));
        HIP_CHECK(hipMemcpy(pub, (const char*)st->d + e, e * s->n, hipMemcpyDeviceToHost));
        HIP_CHECK(hipMemcpy((char*)pub + e * s->n, (const char*)st->d + e * s->aoff, e * s->m, hipMemcpyDeviceToHost));
        return;
    }
    std::lock_guard<std::mutex> lock(s->public_lock);
    void* blk = public_block(s);
    const size_t len = (size_t)s->n + s->m;
    const dim3 g(ceil_div((long long)len, BLK)), b(BLK);
    if (s->prec == ASAT_F64)
        hipLaunchKernelGGL(k_to_public<double>, g, b, 0, s->stream, (const double*)st->d, s->n, s->m, s->aoff,
                           (const int*)s->d_perm, (double*)blk);
    else
        hipLaunchKernelGGL(k_to_public<float>, g, b, 0, s->stream, (const float*)st->d, s->n, s->m, s->aoff,
                           (const int*)s->d_perm, (float*)blk);
    HIP_CHECK(hipGetLastError());
    HIP_CHECK(hipMemcpyAsync(pub, blk, s->esize * len, hipMemcpyDeviceToHost, s->stream));
    HIP_CHECK(hipStreamSynchronize(s->stream));
}

// the spins alone, in variable order
static void state_get_spins(const State* st, void* spins)
{
    state_check(st);
    Sys* s = st->sys;
    HIP_CHECK(hipMemcpyAsync(spins, (const char*)st->d + s->esize, (size_t)s->esize * s->n, hipMemcpyDeviceToHost,
                             s->stream));
    HIP_CHECK(hipStreamSynchronize(s->stream));
}

template <typename T>
static StageArgs<T> stage_args(Sys* s, T* xa, T* xb, T* const* kk, T* tmp, double* partial, const Ctrl* c)
{
    StageArgs<T> a;
    memset(&a, 0, sizeof(a));   // padding too: the arguments are compared bytewise (captured attempts)
    a.lit = s->d_lit; a.pos = s->d_pos; a.spos = s->d_spos; a.srank = s->d_srank;
    a.runs = s->d_runs; a.run_stride = s->run_stride;
    a.litq = s->d_litq; a.posq = s->d_posq; a.mq = s->mq;
    a.th = s->family == ASAT_FAMILY_TANH ? s->d_th : nullptr;
    a.csr_ptr = s->d_csr_ptr; a.csr_pos = s->d_csr_pos; a.rloc = s->d_rloc; a.ploc = s->d_ploc; a.gstart = s->d_gstart;
    a.pvar = s->d_pvar; a.pw16 = s->d_pw16; a.pv0 = s->d_pv0; a.pc0 = s->d_pc0; a.pcontrib = (T*)s->d_pcontrib; a.split = s->split ? 1 : 0;
    a.contrib = (T*)s->d_contrib;
    a.xa = xa; a.xb = xb;
    a.k1 = kk[0]; a.k2 = kk[1]; a.k3 = kk[2]; a.k4 = kk[3]; a.k5 = kk[4];
    a.tmp = tmp; a.partial = partial; a.ctrl = c;
    a.slot_spins = 0;
    a.n = s->n; a.m = s->m; a.k = s->k; a.aoff = s->aoff;
    a.ntiles = ceil_div(s->m, s->tc);
    a.tile_clauses = s->tc;
    a.clause_per_xcd = ceil_div(s->tiled ? a.ntiles : ceil_div(s->m, BLK), 8);
    a.nblk_clause = clause_grid(s);
    a.vg = s->vg;
    a.var_stagger = s->var_stagger;
    a.vg_blocks = s->vg_blocks;
    a.ngroups = s->ngroups;
    a.knorm = (T)std::pow(2.0, -s->k);
    a.family = s->family;
    a.q = (T)s->q;
    a.apart = s->d_apart;
    a.bb = (T)s->b * a.knorm * a.knorm;
    a.bias = a.bb > (T)0;
    a.alpha = (T)s->m / (T)s->n;
    return a;
}


// k_clause_k and its tanh-table form by the clause length
template <typename T, int J, int KT>
static void launch_clause_k(const StageArgs<T>& a, hipStream_t st)
{
    if (a.th) hipLaunchKernelGGL((k_clause_k<T, KT, J, true>), dim3(a.nblk_clause), dim3(BLK), 0, st, a);
    else hipLaunchKernelGGL((k_clause_k<T, KT, J, false>), dim3(a.nblk_clause), dim3(BLK), 0, st, a);
}

template <typename T, int J>
static void launch_clause(const StageArgs<T>& a, const Sys* s, hipStream_t st)
{
    if (!s->tiled && a.litq && (a.family != ASAT_FAMILY_TANH || a.th)) {
        if (a.k <= 2) launch_clause_k<T, J, 2>(a, st);
        else if (a.k <= 6) launch_clause_k<T, J, 6>(a, st);
        else if (a.k <= 8) launch_clause_k<T, J, 8>(a, st);
        else launch_clause_k<T, J, 10>(a, st);
        return;
    }
    dim3 g(a.nblk_clause), b(BLK);
    const bool tiled = s->tiled;
    const bool ss = a.slot_spins != 0;
    const bool ps = a.split != 0;   // slot spins come with direct primary slots (both need the LDS var pass)
    require(!ss || ps, ASAT_ERR_INVALID_ARGUMENT, "slot spins without direct primary slots");
    const dim3 tb(TILE_BT);
    constexpr int TB = TC_BIG, TS = TC;
    const bool big = s->tc > TC;
    require(!big || (sizeof(T) == 4 && ps && a.k == 3 && a.pw16 && a.pv0 && a.runs), ASAT_ERR_INVALID_ARGUMENT,
            "big clause tiles without their layout");
    if constexpr (sizeof(T) == 4) {
        if (tiled && big) {
            if (ss) hipLaunchKernelGGL((k_clause_tile<T, 3, J, TILE_BT, TB, true, true>), g, tb, 0, st, a);
            else hipLaunchKernelGGL((k_clause_tile<T, 3, J, TILE_BT, TB, false, true>), g, tb, 0, st, a);
            return;
        }
    }
    if (tiled && a.k == 3 && ss) hipLaunchKernelGGL((k_clause_tile<T, 3, J, TILE_BT, TS, true, true>), g, tb, 0, st, a);
    else if (tiled && a.k == 4 && ss) hipLaunchKernelGGL((k_clause_tile<T, 4, J, TILE_BT, TS, true, true>), g, tb, 0, st, a);
    else if (tiled && a.k == 3 && ps) hipLaunchKernelGGL((k_clause_tile<T, 3, J, TILE_BT, TS, false, true>), g, tb, 0, st, a);
    else if (tiled && a.k == 4 && ps) hipLaunchKernelGGL((k_clause_tile<T, 4, J, TILE_BT, TS, false, true>), g, tb, 0, st, a);
    else if (tiled && a.k == 3) hipLaunchKernelGGL((k_clause_tile<T, 3, J, TILE_BT, TS, false, false>), g, tb, 0, st, a);
    else if (tiled && a.k == 4) hipLaunchKernelGGL((k_clause_tile<T, 4, J, TILE_BT, TS, false, false>), g, tb, 0, st, a);
    else hipLaunchKernelGGL((k_clause_gen<T, J>), g, b, 0, st, a);
}

// allow the LDS var pass dynamic LDS beyond the default 64 KB, once per
// instantiation (before the first launch, and outside any stream capture)
template <typename T, int J>
static void var_lds_attr()
{
    static const hipError_t attr = hipFuncSetAttribute(reinterpret_cast<const void*>(&k_var_region<T, J>),
                                                       hipFuncAttributeMaxDynamicSharedMemorySize, VAR_LDS_BYTES);
    HIP_CHECK(attr);
}

template <typename T>
static void var_lds_attrs()
{
    var_lds_attr<T, 1>(); var_lds_attr<T, 2>(); var_lds_attr<T, 3>();
    var_lds_attr<T, 4>(); var_lds_attr<T, 5>(); var_lds_attr<T, 6>();
}

template <typename T, int J>
static void launch_var(const StageArgs<T>& a, const Sys* s, hipStream_t st)
{
    if (s->lds_var) {
        var_lds_attr<T, J>();
        hipLaunchKernelGGL((k_var_region<T, J>), dim3(var_grid(s)), dim3(VBLK), (size_t)s->var_lds, st, a);
    } else if (s->wide_var) {
        hipLaunchKernelGGL((k_var_wide<T, J>), dim3(var_grid(s)), dim3(WIDE_BLK), 0, st, a);
    } else {
        hipLaunchKernelGGL((k_var<T, J>), dim3(var_grid(s)), dim3(BLK), 0, st, a);
    }
}

// One attempt.  tkind >= 0: events e0 / e1 are recorded just before and
// after the kernel of that kind (clause J = kind + 1 for 0..5, var J =
// kind - 5 for 6..11, control for 12).
template <typename T>
static void launch_attempt(const StageArgs<T>& a, const Sys* s, Ctrl* ctrl, const double* partial, int np,
                           hipStream_t st, int tkind = -1, hipEvent_t e0 = nullptr, hipEvent_t e1 = nullptr)
{
    auto mark = [&](int kind, hipEvent_t e) {
        if (kind == tkind) HIP_CHECK(hipEventRecord(e, st));
    };
    mark(0, e0); launch_clause<T, 1>(a, s, st); mark(0, e1);
    mark(6, e0); launch_var<T, 1>(a, s, st); mark(6, e1);
    mark(1, e0); launch_clause<T, 2>(a, s, st); mark(1, e1);
    mark(7, e0); launch_var<T, 2>(a, s, st); mark(7, e1);
    mark(2, e0); launch_clause<T, 3>(a, s, st); mark(2, e1);
    mark(8, e0); launch_var<T, 3>(a, s, st); mark(8, e1);
    mark(3, e0); launch_clause<T, 4>(a, s, st); mark(3, e1);
    mark(9, e0); launch_var<T, 4>(a, s, st); mark(9, e1);
    mark(4, e0); launch_clause<T, 5>(a, s, st); mark(4, e1);
    mark(10, e0); launch_var<T, 5>(a, s, st); mark(10, e1);
    mark(5, e0); launch_clause<T, 6>(a, s, st); mark(5, e1);
    mark(11, e0); launch_var<T, 6>(a, s, st); mark(11, e1);
    mark(12, e0);
    hipLaunchKernelGGL(k_control, dim3(1), dim3(CTRL_BLK), 0, st, ctrl, partial, np);
    mark(12, e1);
}

template <typename T>
static void sys_rhs(Sys* s, State* dxdt, const State* x)
{
    s->require_ready();
    state_check(dxdt); state_check(x);
    T* kk[5] = {(T*)dxdt->d, nullptr, nullptr, nullptr, nullptr};
    StageArgs<T> a = stage_args<T>(s, (T*)x->d, nullptr, kk, nullptr, nullptr, nullptr);
    // dxdt.SetZero(): padding and the constant slot read as 0
    HIP_CHECK(hipMemsetAsync(dxdt->d, 0, (size_t)s->esize * s->alloc, s->stream));
    fill_tanh<T>(a, (const T*)x->d, s->stream);
    launch_clause<T, 1>(a, s, s->stream);
    launch_var<T, 1>(a, s, s->stream);
    HIP_CHECK(hipGetLastError());
    HIP_CHECK(hipStreamSynchronize(s->stream));
}

template <typename T>
static int sys_violations(Sys* s, const State* x)
{
    s->require_ready();
    state_check(x);
    const int nb = std::min(VIOL_BLOCKS, ceil_div(s->m, BLK));
    auto launch = [&](auto kernel) {
        hipLaunchKernelGGL(kernel, dim3(nb), dim3(BLK), 0, s->stream, s->d_lit, s->m, s->k, (const T*)x->d, s->d_count);
    };
    if (s->k == 3) launch(k_violations<T, 3>);
    else if (s->k == 4) launch(k_violations<T, 4>);
    else launch(k_violations<T, 0>);
    HIP_CHECK(hipGetLastError());
    int part[VIOL_BLOCKS];
    HIP_CHECK(hipMemcpyAsync(part, s->d_count, sizeof(int) * nb, hipMemcpyDeviceToHost, s->stream));
    HIP_CHECK(hipStreamSynchronize(s->stream));
    return std::accumulate(part, part + nb, 0);
}

// ---------------------------------------------------------------------------
// integrator
// ---------------------------------------------------------------------------
// The control block and, in a line of its own, the few-workgroup kernel's arrival
// word, which one copy brings to the host.
struct CtrlBlock {
    Ctrl ctrl;
    alignas(128) unsigned arrived;
};

struct RK {
    Sys* sys = nullptr;
    double eps = 1e-4;      // CudaRungeKutta() default (CudaRungeKutta.cu:175)
    double floor = 1e-20;   // xscal constant term (reference TINY)
    double* hlog = nullptr; // optional device log of accepted step sizes (set before Reset)
    long long hlog_len = 0;
    int alloc = 0, prec = -1;
    unsigned long long gen = 0;   // the system's problem generation at Configure
    void* k[5] = {nullptr, nullptr, nullptr, nullptr, nullptr};
    void* tmp = nullptr;
    int tmp_n = 0;            // tmp holds n+1 values of the problem at Configure
    double* partial = nullptr;
    int npartial = 0;
    Ctrl* d_ctrl = nullptr;   // of a CtrlBlock
    Ctrl* h_ctrl = nullptr;   // pinned mirror
    int small_mode = 1;              // 1: one-workgroup path where the problem fits, 0: never
    SmallSolve* d_solve = nullptr;   // device SatSolver loop state (one-workgroup path)
    SmallSolve* h_solve = nullptr;   // pinned mirror
    void* d_grid = nullptr;          // exchange buffers of the few-workgroup path
    size_t grid_bytes = 0;
    bool grid_plain = false;         // launched without the runtime's cooperation, see grid_launch
    bool grid_off = false;           // its workgroups did not all run, or it had no memory: not tried again for
                                     // this problem
    // test limits (asat_rk_set_grid_limits)
    int grid_workgroups = 0, grid_launches = -1, grid_attempts = 0;
    void* pair[2] = {nullptr, nullptr};
    hipEvent_t ev0 = nullptr, ev1 = nullptr;
    float last_ms = -1.f;
    bool configured = false;
    // kernel timer (measurement hook): one event pair per attempt
    int timer_kind = -1;
    std::vector<hipEvent_t> tev;
    double timer_ms = 0.0;
    long long timer_launches = 0;
    // small problems: GRAPH_ATTEMPTS attempts captured once and replayed; the
    // key is the exact launch arguments the graph was captured with, or without a
    // graph those of the last Step that could have had one
    hipGraphExec_t gexec = nullptr;
    std::vector<unsigned char> gkey;

    void drop_graph()
    {
        if (gexec) (void)hipGraphExecDestroy(gexec);
        gexec = nullptr;
        gkey.clear();
    }
    void free_all()
    {
        drop_graph();
        for (auto& p : k) dfree(p);
        dfree(tmp); dfree(partial); dfree(d_ctrl); dfree(d_solve); dfree(d_grid);
        grid_bytes = 0;
        if (h_ctrl) { (void)hipHostFree(h_ctrl); h_ctrl = nullptr; }
        if (h_solve) { (void)hipHostFree(h_solve); h_solve = nullptr; }
    }
    ~RK()
    {
        free_all();
        if (ev0) (void)hipEventDestroy(ev0);
        if (ev1) (void)hipEventDestroy(ev1);
        for (hipEvent_t e : tev) (void)hipEventDestroy(e);
    }
    unsigned* d_arrived() const { return &((CtrlBlock*)d_ctrl)->arrived; }
    unsigned& h_arrived() const { return ((CtrlBlock*)h_ctrl)->arrived; }
    // no arrivals, for the next launch of the few-workgroup kernel
    void clear_arrived(hipStream_t st)
    {
        if (h_arrived() == 0) return;
        HIP_CHECK(hipMemsetD32Async((hipDeviceptr_t)d_arrived(), 0, 1, st));
        h_arrived() = 0;
    }
    void require_configured() const
    {
        require(configured && sys && sys->ready, ASAT_ERR_NOT_CONFIGURED,
                "the RK4 solver has not been configured with an ODE yet");
        // scratch (k1..k5, tmp, partials) is sized for the problem present at
        // Configure; a new problem needs a new Configure
        require(gen == sys->gen, ASAT_ERR_NOT_CONFIGURED,
                "the SAT problem changed since the RK4 solver was configured");
    }
};

// CudaRungeKutta::Reset (h = 1e-9, clock and counters cleared): the control
// block is set on the host and copied in stream order (pinned memory), so a
// solve that follows waits for no round trip.  Every later host write of
// h_ctrl is a device-to-host copy behind this one on the same stream.
static void rk_reset(RK* r)
{
    r->require_configured();
    Ctrl* c = r->h_ctrl;
    memset(c, 0, sizeof(Ctrl));
    c->h = 1e-9; c->hnext = 1e-9; c->eps = r->eps;
    c->floor = r->floor; c->hlog = r->hlog; c->hlog_len = r->hlog_len;
    c->step_start = 1;
    HIP_CHECK(hipMemcpyAsync(r->d_ctrl, c, sizeof(Ctrl), hipMemcpyHostToDevice, r->sys->stream));
    r->pair[0] = r->pair[1] = nullptr;
}

static bool small_path(const RK* r);
static bool grid_path(RK* r);

static void rk_configure(RK* r, Sys* s)
{
    s->require_ready();
    HIP_CHECK(hipStreamSynchronize(s->stream));
    const int npartial = clause_grid(s) + var_grid(s);
    if (r->sys != s || r->gen != s->gen) r->grid_off = false;
    if (r->configured && r->sys == s && r->alloc == s->alloc && r->prec == s->prec && r->npartial == npartial &&
        r->tmp_n == s->n) {
        // same sizes (SatSolver configures before every Solve): keep the
        // buffers, clear them and reset the control block
        r->drop_graph();
        if (r->gen != s->gen) r->clear_arrived(s->stream);
        r->sys = s;
        r->gen = s->gen;
        // the persistent paths keep everything on the CUs and read none of
        // these buffers (a caller solving start after start)
        if (!small_path(r) && !grid_path(r)) {
            const size_t bytes = (size_t)s->esize * s->alloc;
            for (auto& p : r->k) HIP_CHECK(hipMemsetAsync(p, 0, bytes, s->stream));
            HIP_CHECK(hipMemsetAsync(r->tmp, 0, (size_t)s->esize * (s->n + 1), s->stream));
            HIP_CHECK(hipMemsetAsync(r->partial, 0, sizeof(double) * r->npartial, s->stream));
        }
        (void)grid_path(r);     // its layout, where the problem has one
        rk_reset(r);
        return;
    }
    r->free_all();
    r->configured = false;
    r->sys = s;
    r->alloc = s->alloc;
    r->gen = s->gen;
    r->prec = s->prec;
    const size_t bytes = (size_t)s->esize * s->alloc;
    // clears on the kernels' stream: a plain hipMemset returns before it is done, on a
    // stream that theirs does not wait for
    for (auto& p : r->k) {
        HIP_CHECK(hipMalloc(&p, bytes));
        HIP_CHECK(hipMemsetAsync(p, 0, bytes, s->stream));
    }
    HIP_CHECK(hipMalloc(&r->tmp, (size_t)s->esize * (s->n + 1)));
    r->tmp_n = s->n;
    HIP_CHECK(hipMemsetAsync(r->tmp, 0, (size_t)s->esize * (s->n + 1), s->stream));
    r->npartial = npartial;
    HIP_CHECK(hipMalloc((void**)&r->partial, sizeof(double) * r->npartial));
    HIP_CHECK(hipMemsetAsync(r->partial, 0, sizeof(double) * r->npartial, s->stream));
    HIP_CHECK(hipMalloc((void**)&r->d_ctrl, sizeof(CtrlBlock)));
    HIP_CHECK(hipMemsetAsync(r->d_ctrl, 0, sizeof(CtrlBlock), s->stream));
    HIP_CHECK(hipHostMalloc((void**)&r->h_ctrl, sizeof(CtrlBlock), hipHostMallocDefault));
    memset((void*)r->h_ctrl, 0, sizeof(CtrlBlock));
    HIP_CHECK(hipMalloc((void**)&r->d_solve, sizeof(SmallSolve)));
    HIP_CHECK(hipHostMalloc((void**)&r->h_solve, sizeof(SmallSolve), hipHostMallocDefault));
    memset(r->h_solve, 0, sizeof(SmallSolve));
    if (!r->ev0) HIP_CHECK(hipEventCreate(&r->ev0));
    if (!r->ev1) HIP_CHECK(hipEventCreate(&r->ev1));
    r->configured = true;
    (void)grid_path(r);
    rk_reset(r);
}

// the tanh table of a state, where the passes use one
template <typename T>
static void fill_tanh(const StageArgs<T>& a, const T* x, hipStream_t st)
{
    if (!a.th) return;
    hipLaunchKernelGGL(k_tanh_fill<T>, dim3(ceil_div(2LL * (a.n + 1), BLK)), dim3(BLK), 0, st, x, a.n, a.q, a.th);
    HIP_CHECK(hipGetLastError());
}

// Stage arguments of the integrator.  With slot spins (tiled clause pass and
// LDS var pass), contrib is first filled with the slot spins of the current
// state x, which the caller may have changed since the last Step.  Inside
// Step the var passes keep contrib holding the next clause pass's spins: a
// rejected attempt's J = 1 clause pass is skipped, and its J = 1 var pass
// (which reuses k1 and reads no contributions) writes stage 2's spins.
template <typename T>
static StageArgs<T> rk_stage_args(RK* r, int parity)
{
    Sys* s = r->sys;
    T* kk[5] = {(T*)r->k[0], (T*)r->k[1], (T*)r->k[2], (T*)r->k[3], (T*)r->k[4]};
    StageArgs<T> a = stage_args<T>(s, (T*)r->pair[0], (T*)r->pair[1], kk, (T*)r->tmp, r->partial, r->d_ctrl);
    fill_tanh<T>(a, (const T*)r->pair[parity], s->stream);
    if (s->tiled && s->lds_var) {
        a.slot_spins = 1;
        static const hipError_t attr = hipFuncSetAttribute(reinterpret_cast<const void*>(&k_slot_fill<T>),
                                                           hipFuncAttributeMaxDynamicSharedMemorySize, VAR_LDS_BYTES);
        HIP_CHECK(attr);
        hipLaunchKernelGGL(k_slot_fill<T>, dim3(s->ngroups), dim3(VBLK), (size_t)s->var_lds, s->stream,
                           (const T*)r->pair[parity], s->d_csr_ptr, s->d_rloc, s->d_gstart, s->vg, s->n,
                           (T*)s->d_contrib);
        HIP_CHECK(hipGetLastError());
    }
    return a;
}

// Launch-bound problems (few literal slots) replay a captured graph of
// GRAPH_ATTEMPTS attempts instead of launching 13 kernels per attempt, as
// long as a round still needs that many; the rest are launched one by one.
// Up to GRAPH_FIRST_SLOTS from the first Step on.  From there to GRAPH_MAX_BYTES
// of contributions a graph saves 2 to 4 us per attempt (without and with: FP32, N =
// 40 000, M = 170 000 80.9 and 77.6; N = 70 000, M = 297 500 90.4 and 88.1; FP64, N =
// 30 000, M = 127 500 79.2 and 75.7; 4-SAT, FP32, N = 20 000, M = 198 600 89.2 and
// 87.1), less than the 0.15 to 0.25 ms of its capture in a short Step, so only a Step
// that repeats the last one's arguments, or is of GRAPH_LONG steps, makes one.
// Beyond, the kernels hide their launches (FP64, N = 70 000: 113.7 and 114.5).
constexpr long long GRAPH_FIRST_SLOTS = 1LL << 18, GRAPH_MAX_BYTES = 1LL << 22;
constexpr int GRAPH_ATTEMPTS = 8, GRAPH_LONG = 128;

// makes the graph unless it is there; false where this Step of count goes without
template <typename T>
static bool ensure_graph(RK* r, const StageArgs<T>& a, int count)
{
    Sys* s = r->sys;
    hipStream_t st = s->stream;
    if (r->timer_kind >= 0 || s->nslots * s->esize > GRAPH_MAX_BYTES || count < GRAPH_ATTEMPTS) return false;
    // the key: the arguments and every launch size the attempts depend on
    std::vector<unsigned char> key(sizeof(a) + 4 * sizeof(int));
    memcpy(key.data(), &a, sizeof(a));
    const int dims[4] = {clause_grid(s), var_grid(s), s->var_lds, s->tiled ? 1 : 0};
    memcpy(key.data() + sizeof(a), dims, sizeof(dims));
    const bool repeated = r->gkey == key;
    if (r->gexec && repeated) return true;
    if (s->nslots > GRAPH_FIRST_SLOTS && !repeated && count < GRAPH_LONG) {
        r->drop_graph();
        r->gkey = std::move(key);
        return false;
    }
    r->drop_graph();
    var_lds_attrs<T>();
    hipGraph_t g = nullptr;
    HIP_CHECK(hipStreamBeginCapture(st, hipStreamCaptureModeThreadLocal));
    try {
        for (int i = 0; i < GRAPH_ATTEMPTS; i++) launch_attempt<T>(a, s, r->d_ctrl, r->partial, r->npartial, st);
    } catch (...) {
        (void)hipStreamEndCapture(st, &g);
        if (g) (void)hipGraphDestroy(g);
        throw;
    }
    HIP_CHECK(hipStreamEndCapture(st, &g));
    const hipError_t e = hipGraphInstantiate(&r->gexec, g, nullptr, nullptr, 0);
    (void)hipGraphDestroy(g);
    HIP_CHECK(e);
    r->gkey = std::move(key);
    return true;
}

template <typename T>
static int rk_step_impl(RK* r, State* olds, State* news, int count)
{
    Sys* s = r->sys;
    hipStream_t st = s->stream;
    // canonical ping-pong pair: parity 0 means x lives in pair[0]
    if (!((r->pair[0] == olds->d && r->pair[1] == news->d) || (r->pair[0] == news->d && r->pair[1] == olds->d))) {
        r->pair[0] = olds->d;
        r->pair[1] = news->d;
    }
    const int parity = (r->pair[0] == olds->d) ? 0 : 1;
    HIP_CHECK(hipEventRecord(r->ev0, st));
    StageArgs<T> a = rk_stage_args<T>(r, parity);
    hipLaunchKernelGGL(k_ctrl_begin, dim3(1), dim3(64), 0, st, r->d_ctrl, (long long)count, parity);
    long long remaining = count;
    const long long target = r->h_ctrl->steps + count;
    long long last_attempts = r->h_ctrl->attempts;
    const bool graphed = ensure_graph<T>(r, a, count);
    while (remaining > 0) {
        const int tk = r->timer_kind;
        if (graphed) {
            // whole graphs while they fit, the rest one attempt at a time
            const long long full = remaining / GRAPH_ATTEMPTS;
            for (long long i = 0; i < full; i++) HIP_CHECK(hipGraphLaunch(r->gexec, st));
            for (long long i = full * GRAPH_ATTEMPTS; i < remaining; i++)
                launch_attempt<T>(a, s, r->d_ctrl, r->partial, r->npartial, st);
        } else {
            if (tk >= 0)
                while ((long long)r->tev.size() < 2 * remaining) {
                    // timing-only events, read after the stream synchronises:
                    // no system-scope fence, so recording them does not write
                    // back and invalidate the caches between the kernels
                    hipEvent_t e;
                    HIP_CHECK(hipEventCreateWithFlags(&e, hipEventDisableSystemFence));
                    r->tev.push_back(e);
                }
            for (long long i = 0; i < remaining; i++) {
                if (tk >= 0)
                    launch_attempt<T>(a, s, r->d_ctrl, r->partial, r->npartial, st, tk, r->tev[2 * i],
                                      r->tev[2 * i + 1]);
                else
                    launch_attempt<T>(a, s, r->d_ctrl, r->partial, r->npartial, st);
            }
        }
        HIP_CHECK(hipGetLastError());
        HIP_CHECK(hipMemcpyAsync(r->h_ctrl, r->d_ctrl, sizeof(Ctrl), hipMemcpyDeviceToHost, st));
        HIP_CHECK(hipStreamSynchronize(st));
        if (tk >= 0)
            for (long long i = 0; i < remaining; i++) {
                float ms = 0.f;
                HIP_CHECK(hipEventElapsedTime(&ms, r->tev[2 * i], r->tev[2 * i + 1]));
                r->timer_ms += ms;
                r->timer_launches++;
            }
        if (r->h_ctrl->underflow) break;
        remaining = target - r->h_ctrl->steps;
        // every enqueued attempt either accepts, rejects or underflows; no
        // progress here means the control block was left inactive
        require(r->h_ctrl->attempts > last_attempts || remaining <= 0, ASAT_ERR_HIP,
                "integrator made no progress (control block inactive)");
        last_attempts = r->h_ctrl->attempts;
    }
    HIP_CHECK(hipEventRecord(r->ev1, st));
    HIP_CHECK(hipEventSynchronize(r->ev1));
    HIP_CHECK(hipEventElapsedTime(&r->last_ms, r->ev0, r->ev1));
    // hand the newest state to `olds` (the reference swaps the device pointers)
    const int par = r->h_ctrl->parity;
    void* xcur = r->pair[par];
    void* xother = r->pair[par ^ 1];
    olds->d = xcur;
    news->d = xother;
    return r->h_ctrl->underflow ? ASAT_UNDERFLOW : ASAT_OK;
}

// ---------------------------------------------------------------------------
// one-workgroup path (asat_small.h): problems whose whole integrator fits in
// one workgroup's LDS and that use no bias term.  The kernel timer (a
// per-kernel measurement hook) needs the multi-kernel path.
// ---------------------------------------------------------------------------
static bool small_path(const RK* r)
{
    const Sys* s = r->sys;
    return r->small_mode && s->small_lds > 0 && !(s->b > 0.0) && r->timer_kind < 0;
}

template <typename T, int KT, int BS, int FAM = ASAT_FAMILY_CTDS>
static void small_kernel_launch(const SmallArgs& a, size_t lds, hipStream_t st)
{
    static const hipError_t attr = hipFuncSetAttribute(reinterpret_cast<const void*>(&k_small<T, KT, BS, FAM>),
                                                       hipFuncAttributeMaxDynamicSharedMemorySize, SMALL_LDS_MAX);
    HIP_CHECK(attr);
    hipLaunchKernelGGL((k_small<T, KT, BS, FAM>), dim3(1), dim3(BS), lds, st, a);
    HIP_CHECK(hipGetLastError());
}

// 256 threads (a clause and a variable each) up to 512 clauses and
// variables, 1024 threads above; the tanh family runs the generic kernel
template <typename T>
static void small_launch(const Sys* s, const SmallArgs& a, hipStream_t st)
{
    const size_t lds = (size_t)s->small_lds;
    const bool wide = std::max(s->m, s->n) > 512;
    if (s->family == ASAT_FAMILY_TANH) {
        if (wide) small_kernel_launch<T, 0, 1024, ASAT_FAMILY_TANH>(a, lds, st);
        else small_kernel_launch<T, 0, 256, ASAT_FAMILY_TANH>(a, lds, st);
    } else if (s->k == 3) {
        if (wide) small_kernel_launch<T, 3, 1024>(a, lds, st);
        else small_kernel_launch<T, 3, 256>(a, lds, st);
    } else if (s->k == 4) {
        if (wide) small_kernel_launch<T, 4, 1024>(a, lds, st);
        else small_kernel_launch<T, 4, 256>(a, lds, st);
    } else {
        if (wide) small_kernel_launch<T, 0, 1024>(a, lds, st);
        else small_kernel_launch<T, 0, 256>(a, lds, st);
    }
}

static SmallArgs small_args(const RK* r, void* x)
{
    const Sys* s = r->sys;
    SmallArgs a;
    memset(&a, 0, sizeof(a));
    a.lit = s->d_lit; a.vptr = s->d_vptr; a.spos = s->d_spos_small;
    a.x = x;
    a.ctrl = r->d_ctrl;
    a.n = s->n; a.m = s->m; a.k = s->k; a.aoff = s->aoff; a.alloc = s->alloc; a.nlist = s->nlist;
    a.runlen = s->runlen;
    a.family = s->family;
    a.q = s->q;
    a.knorm = std::pow(2.0, -s->k);
    a.batch = 1;
    return a;
}

// ---------------------------------------------------------------------------
// few-workgroup path (asat_grid.h), for the problems it can be laid out for;
// the same conditions as the one-workgroup path, CTDS family only
// ---------------------------------------------------------------------------
static bool grid_path(RK* r)
{
    Sys* s = r->sys;
    if (!r->small_mode || r->grid_off || s->family != ASAT_FAMILY_CTDS || s->b > 0.0 || r->timer_kind >= 0) return false;
    ensure_grid(s);
    return s->grid_wgs > 0 && !(r->grid_workgroups > 0 && s->grid_wgs > r->grid_workgroups);
}

// What the 8 to 128 workgroups gain over the multi-kernel path in `steps` steps, us:
// about 0.3 per attempt for every KB that the spins, which each of them reads six
// times an attempt, stay below 124.  us per attempt, here and there: FP32, N = 12 000,
// M = 51 000 44 and 67, 20 000, 85 000 62 and 71, 24 000, 102 000 68 and 72, 28 000,
// 119 000 74.4 and 73.9, 32 000, 136 000 82 and 76 (50 000 clauses: 68.2 and 68.3);
// FP64, 8000, 34 000 49 and 63, 12 000, 51 120 58 and 65, 15 000, 63 000 64 and 66,
// 17 000, 40 000 61.1 and 61.0; 4-SAT, FP64, 8000, 79 000 68 and 84.
static double grid_gain(const Sys* s, long long steps)
{
    return 0.3 * (double)steps * (124.0 - s->esize * 64.0 * s->grid_groups / 1024.0);
}
// A call costs 20 us more (a cooperative launch, the layout into registers and LDS):
// a Step has to gain that (Step(1), FP32, N = 24 000 130 and 107 us, N = 2000 68 and
// 100).  A solve saves about 60 us per batch for the Step's end and the count on
// the host, so there a batch may lose them.
constexpr double GRID_CALL_US = 20.0;
static bool grid_step(RK* r, int count)
{
    return grid_path(r) && (r->sys->grid_wgs == 1 || grid_gain(r->sys, count) >= GRID_CALL_US);
}
static bool grid_solve(RK* r, int batch)
{
    return grid_path(r) && (r->sys->grid_wgs == 1 || grid_gain(r->sys, batch) >= -GRID_CALL_US);
}

// workgroups of the persistent kernel that runs the problem (0: the multi-kernel path)
static int persistent_workgroups(RK* r)
{
    return grid_path(r) ? r->sys->grid_wgs : small_path(r) ? 1 : 0;
}

// the kernel's arguments; a holds what small_args gives plus the loop's limits.
// False without memory for the exchange buffers.
static bool grid_args(RK* r, const SmallArgs& a, GridArgs& g)
{
    const Sys* s = r->sys;
    const size_t pub = (size_t)s->esize * 2 * 64 * s->grid_groups;
    const size_t need = 2 * GRID_MAX * (sizeof(double) + sizeof(int)) + pub;
    if (r->grid_bytes < need) {
        dfree(r->d_grid);
        r->grid_bytes = 0;
        if (hipMalloc(&r->d_grid, need) != hipSuccess) {
            (void)hipGetLastError();
            r->d_grid = nullptr;
            return false;
        }
        r->grid_bytes = need;
    }
    memset(&g, 0, sizeof(g));
    g.code = s->d_gcode; g.cpos = s->d_gcpos; g.wg = s->d_gwg; g.group = s->d_ggroup; g.vmap = s->d_gvmap;
    g.x = a.x; g.ctrl = a.ctrl; g.solve = a.solve;
    char* p = (char*)r->d_grid;
    g.barrier = r->d_arrived();
    g.err = (double*)p;
    g.count = (int*)(p + 2 * GRID_MAX * sizeof(double));
    g.pub = p + 2 * GRID_MAX * (sizeof(double) + sizeof(int));
    g.target = a.target; g.max_steps = a.max_steps; g.max_time = a.max_time;
    g.time_float = a.time_float; g.batch = a.batch;
    g.ngroups = s->grid_groups; g.aoff = s->aoff;
    g.knorm = a.knorm;
    g.attempt_cap = r->grid_attempts > 0 ? r->grid_attempts : GRID_ATTEMPT_CAP;
    return true;
}

// One launch of the few-workgroup kernel, cooperative where the runtime grants that:
// it takes one such kernel of a process at a time, and launches of several threads
// then never share the CUs out between them.  It grants it to one process on a GPU
// (the next one's launches fail, with "the operation cannot be performed in the
// present state"); there an ordinary launch does, of one thread at a time (alone,
// held until the kernel has ended), and the bounded wait covers what other processes
// run.  give_up: the workgroups find the arrival word marked.
static std::mutex grid_alone;
static void grid_launch(RK* r, GridArgs& g, bool give_up, std::unique_lock<std::mutex>& alone)
{
    Sys* s = r->sys;
    const bool solo = s->grid_wgs == 1;
    const void* f = grid_kernel(s->prec, s->k, s->grid_cpt, solo);
    const dim3 grid(s->grid_wgs), block(GRID_BT);
    void* args[] = {&g};
    if (!solo) {
        // every launch counts on from the last one
        if (r->h_arrived() >= GRID_GIVE_UP / 2) r->clear_arrived(s->stream);
        g.phase = r->h_arrived() / (unsigned)s->grid_wgs;
        if (give_up) HIP_CHECK(hipMemsetD32Async((hipDeviceptr_t)g.barrier, (int)GRID_GIVE_UP, 1, s->stream));
        if (!r->grid_plain) {
            if (hipLaunchCooperativeKernel(f, grid, block, args, (unsigned)s->grid_lds, s->stream) == hipSuccess) return;
            (void)hipGetLastError();
            r->grid_plain = true;
        }
        alone = std::unique_lock<std::mutex>(grid_alone);
    }
    HIP_CHECK(hipLaunchKernel(f, grid, block, args, (size_t)s->grid_lds, s->stream));
}

// Launches a persistent kernel (grid: the few-workgroup one) until it reports done: each
// launch runs at most SMALL_ATTEMPT_CAP (GRID_ATTEMPT_CAP) attempts and leaves its
// state in the control block (and the solver block), so the next launch resumes
// where it stopped.  False: the workgroups of a launch did not all run, which has
// changed nothing, and no persistent kernel is left for the problem; the
// control and solver blocks say how far the launches before it came.
template <typename T>
static bool small_run(RK* r, const SmallArgs& a, bool grid)
{
    Sys* s = r->sys;
    hipStream_t st = s->stream;
    bool left = true;
    GridArgs g;
    if (grid && !grid_args(r, a, g)) {
        r->grid_off = true;
        grid = false;
        if (!small_path(r)) return false;
    }
    HIP_CHECK(hipEventRecord(r->ev0, st));
    long long last = r->h_ctrl->attempts;
    for (int launch = 0;; launch++) {
        std::unique_lock<std::mutex> alone;
        if (grid) grid_launch(r, g, launch == r->grid_launches, alone);
        else small_launch<T>(s, a, st);
        HIP_CHECK(hipMemcpyAsync(r->h_ctrl, r->d_ctrl, grid ? sizeof(CtrlBlock) : sizeof(Ctrl), hipMemcpyDeviceToHost, st));
        if (a.solve) HIP_CHECK(hipMemcpyAsync(r->h_solve, r->d_solve, sizeof(SmallSolve), hipMemcpyDeviceToHost, st));
        HIP_CHECK(hipStreamSynchronize(st));
        if (alone.owns_lock()) alone.unlock();
        if (grid && (r->h_arrived() & GRID_GIVE_UP)) {
            r->clear_arrived(st);
            r->grid_off = true;
            grid = false;
            left = small_path(r);
            if (left) continue;
            break;
        }
        if (r->h_ctrl->underflow) break;
        if (a.solve ? r->h_solve->result >= 0 : r->h_ctrl->steps >= a.target) break;
        require(r->h_ctrl->attempts > last, ASAT_ERR_HIP, "integrator made no progress");
        last = r->h_ctrl->attempts;
    }
    HIP_CHECK(hipEventRecord(r->ev1, st));
    HIP_CHECK(hipEventSynchronize(r->ev1));
    HIP_CHECK(hipEventElapsedTime(&r->last_ms, r->ev0, r->ev1));
    return left;
}

static void rk_check_states(const RK* r, const State* olds, const State* news)
{
    state_check(olds); state_check(news);
    require(olds != news && olds->d != news->d, ASAT_ERR_INVALID_ARGUMENT, "old and new state must differ");
    require(olds->sys == r->sys && news->sys == r->sys, ASAT_ERR_INVALID_ARGUMENT,
            "states belong to another system");
}

static int rk_step(RK* r, State* olds, State* news, int count)
{
    r->require_configured();
    rk_check_states(r, olds, news);
    require(count >= 0, ASAT_ERR_INVALID_ARGUMENT, "negative step count");
    if (r->h_ctrl->underflow) return ASAT_UNDERFLOW;
    if (count == 0) return ASAT_OK;
    const bool grid = grid_step(r, count);
    if (small_path(r) || grid) {
        // the state stays in olds; news is not touched
        SmallArgs a = small_args(r, olds->d);
        a.target = r->h_ctrl->steps + count;
        if (r->prec == ASAT_F64 ? small_run<double>(r, a, grid) : small_run<float>(r, a, grid))
            return r->h_ctrl->underflow ? ASAT_UNDERFLOW : ASAT_OK;
        count = (int)(a.target - r->h_ctrl->steps);
    }
    return r->prec == ASAT_F64 ? rk_step_impl<double>(r, olds, news, count)
                               : rk_step_impl<float>(r, olds, news, count);
}

// SatSolver::DoSolve without a callback (AnalogSAT/solver/SatSolver.h:313-331):
// batches of `batch` accepted steps, the violated-clause count of `olds`
// after each, ending on SAT, underflow, or when the time (compared as a
// float if time_float) or the solver's step count reaches its limit before a
// batch.  The solver's counters start at zero; the integrator's continue
// from where they are (SatSolver::Solve configures it first).  On the
// one-workgroup path the whole loop runs in the persistent kernel; otherwise
// it runs here on the host over rk_step and the violation kernel.
static void rk_solve(RK* r, State* olds, State* news, int batch, long long max_steps, double max_time,
                     int time_float, asat_solve_result_t* out)
{
    r->require_configured();
    rk_check_states(r, olds, news);
    require(batch >= 1, ASAT_ERR_INVALID_ARGUMENT, "Batch size must be positive");
    require(max_steps >= 1, ASAT_ERR_INVALID_ARGUMENT, "Max iterations must be positive");
    require(max_time > 0.0, ASAT_ERR_INVALID_ARGUMENT, "Max time must be positive");
    memset(out, 0, sizeof(*out));
    // the host loop's state, which starts at the top of the loop or, where the
    // persistent kernel gave up, where its last full launch stopped
    long long steps = 0;
    double time = 0.0;
    int lastv = 0, result = -1, todo = 0;     // todo: steps left of the batch
    bool due = false;                         // a batch has ended and its count is due
    const bool grid = grid_solve(r, batch);
    if ((small_path(r) || grid) && !r->h_ctrl->underflow) {
        SmallSolve init;
        memset(&init, 0, sizeof(init));
        init.result = -1;
        *r->h_solve = init;
        HIP_CHECK(hipMemcpyAsync(r->d_solve, r->h_solve, sizeof(SmallSolve), hipMemcpyHostToDevice, r->sys->stream));
        SmallArgs a = small_args(r, olds->d);
        a.solve = r->d_solve;
        a.batch = batch;
        a.max_steps = max_steps;
        a.max_time = max_time;
        a.time_float = time_float;
        if (r->prec == ASAT_F64 ? small_run<double>(r, a, grid) : small_run<float>(r, a, grid)) {
            out->result = r->h_solve->result;
            out->steps = r->h_solve->solver_steps;
            out->last_violations = r->h_solve->last_viol;
            out->on_device = 1;
            return;
        }
        steps = r->h_solve->solver_steps;
        time = r->h_ctrl->time;
        lastv = r->h_solve->last_viol;
        todo = r->h_solve->bleft;
        due = r->h_solve->check != 0;
    }
    auto tcmp = [&](double t) { return time_float ? (double)(float)t : t; };
    for (;;) {
        if (due) {
            due = false;
            lastv = r->prec == ASAT_F64 ? sys_violations<double>(r->sys, olds) : sys_violations<float>(r->sys, olds);
            if (lastv == 0) {
                result = SMALL_SAT;
                break;
            }
        }
        if (todo == 0) {
            if (!(tcmp(time) < max_time && steps < max_steps)) break;
            todo = batch;
        }
        if (rk_step(r, olds, news, todo) == ASAT_UNDERFLOW) {
            result = SMALL_UNDERFLOW;
            break;
        }
        steps += batch;
        time = r->h_ctrl->time;
        todo = 0;
        due = true;
    }
    if (result < 0) {
        if (tcmp(time) >= max_time) result = SMALL_MAXTIME;
        else if (steps >= max_steps) result = SMALL_MAXITER;
        else result = 5;   // SAT_UNKNOWN
    }
    out->result = result;
    out->steps = steps;
    out->last_violations = lastv;
    out->on_device = 0;
}

// Times each kernel kind of one attempt over `reps` launches with HIP events
// on the integrator's stream (order: clause J=1..6, var J=1..6, control).
// The control block is saved and restored, so the integrator state is unchanged;
// the scratch buffers (k1..k5, tmp, x_new) are overwritten, which is harmless
// because the next attempt starts a fresh step (step_start == 1 after Step).
template <typename T>
static void rk_profile_impl(RK* r, State* olds, State* news, int reps, float* us)
{
    Sys* s = r->sys;
    hipStream_t st = s->stream;
    if (!((r->pair[0] == olds->d && r->pair[1] == news->d) || (r->pair[0] == news->d && r->pair[1] == olds->d))) {
        r->pair[0] = olds->d;
        r->pair[1] = news->d;
    }
    const int parity = (r->pair[0] == olds->d) ? 0 : 1;
    StageArgs<T> a = rk_stage_args<T>(r, parity);
    Ctrl* backup = nullptr;
    HIP_CHECK(hipMalloc((void**)&backup, sizeof(Ctrl)));
    HIP_CHECK(hipMemcpyAsync(backup, r->d_ctrl, sizeof(Ctrl), hipMemcpyDeviceToDevice, st));
    hipLaunchKernelGGL(k_ctrl_begin, dim3(1), dim3(64), 0, st, r->d_ctrl, (long long)1 << 40, parity);
    auto timeit = [&](int slot, auto&& launch) {
        launch();   // warm
        HIP_CHECK(hipEventRecord(r->ev0, st));
        for (int i = 0; i < reps; i++) launch();
        HIP_CHECK(hipEventRecord(r->ev1, st));
        HIP_CHECK(hipEventSynchronize(r->ev1));
        float ms = 0.f;
        HIP_CHECK(hipEventElapsedTime(&ms, r->ev0, r->ev1));
        us[slot] = ms * 1000.f / (float)reps;
    };
    timeit(0, [&] { launch_clause<T, 1>(a, s, st); });
    timeit(1, [&] { launch_clause<T, 2>(a, s, st); });
    timeit(2, [&] { launch_clause<T, 3>(a, s, st); });
    timeit(3, [&] { launch_clause<T, 4>(a, s, st); });
    timeit(4, [&] { launch_clause<T, 5>(a, s, st); });
    timeit(5, [&] { launch_clause<T, 6>(a, s, st); });
    timeit(6, [&] { launch_var<T, 1>(a, s, st); });
    timeit(7, [&] { launch_var<T, 2>(a, s, st); });
    timeit(8, [&] { launch_var<T, 3>(a, s, st); });
    timeit(9, [&] { launch_var<T, 4>(a, s, st); });
    timeit(10, [&] { launch_var<T, 5>(a, s, st); });
    timeit(11, [&] { launch_var<T, 6>(a, s, st); });
    timeit(12, [&] { hipLaunchKernelGGL(k_control, dim3(1), dim3(CTRL_BLK), 0, st, r->d_ctrl, r->partial, r->npartial); });
    HIP_CHECK(hipGetLastError());
    HIP_CHECK(hipMemcpyAsync(r->d_ctrl, backup, sizeof(Ctrl), hipMemcpyDeviceToDevice, st));
    HIP_CHECK(hipStreamSynchronize(st));
    (void)hipFree(backup);
}

}  // namespace asat

// ===========================================================================
// C ABI
// ===========================================================================
using namespace asat;

struct asat_sys { Sys s; };
struct asat_state { State st; };
struct asat_rk { RK r; };
struct asat_rng { Rng g; };

#define API_BEGIN try {
#define API_END                                                  \
    }                                                            \
    catch (const asat::Error& e) {                               \
        asat::g_last_error = e.what();                           \
        return e.code;                                           \
    }                                                            \
    catch (const std::bad_alloc&) {                              \
        asat::g_last_error = "host allocation failed";           \
        return ASAT_ERR_HIP;                                     \
    }                                                            \
    catch (const std::exception& e) {                            \
        asat::g_last_error = e.what();                           \
        return ASAT_ERR_HIP;                                     \
    }                                                            \
    return ASAT_OK;

#define CHECK_PTR(p) require((p) != nullptr, ASAT_ERR_INVALID_ARGUMENT, "null argument: " #p)

extern "C" {

const char* asat_last_error(void) { return asat::g_last_error.c_str(); }

const char* asat_version(void) { return "analogsat-mi355x 0.1 (gfx950)"; }

int asat_device_count(void)
{
    int n = 0;
    if (hipGetDeviceCount(&n) != hipSuccess) return 0;
    return n;
}

int asat_sys_create(int precision, asat_sys_t** out)
{
    API_BEGIN
    CHECK_PTR(out);
    require(precision == ASAT_F64 || precision == ASAT_F32, ASAT_ERR_INVALID_ARGUMENT, "unknown precision");
    std::unique_ptr<asat_sys> p(new asat_sys());
    p->s.prec = precision;
    p->s.esize = precision == ASAT_F64 ? 8 : 4;
    HIP_CHECK(hipStreamCreateWithFlags(&p->s.stream, hipStreamNonBlocking));
    HIP_CHECK(hipMalloc((void**)&p->s.d_count, sizeof(int) * VIOL_BLOCKS));
    *out = p.release();
    API_END
}

int asat_sys_destroy(asat_sys_t* sys)
{
    API_BEGIN
    delete sys;
    API_END
}

int asat_sys_set_problem(asat_sys_t* sys, const int* literals, const int* lengths, int nclauses)
{
    API_BEGIN
    CHECK_PTR(sys);
    sys_set_problem(&sys->s, literals, lengths, nclauses);
    API_END
}

int asat_sys_get_nmk(const asat_sys_t* sys, int* n, int* m, int* k)
{
    API_BEGIN
    CHECK_PTR(sys);
    if (n) *n = sys->s.n;
    if (m) *m = sys->s.m;
    if (k) *k = sys->s.k;
    API_END
}

int asat_sys_set_b(asat_sys_t* sys, double b)
{
    API_BEGIN
    CHECK_PTR(sys);
    sys->s.b = b;
    API_END
}

int asat_sys_get_b(const asat_sys_t* sys, double* b)
{
    API_BEGIN
    CHECK_PTR(sys); CHECK_PTR(b);
    *b = sys->s.b;
    API_END
}

int asat_sys_rhs(asat_sys_t* sys, asat_state_t* dxdt, const asat_state_t* x, double t)
{
    (void)t;   // autonomous system (the reference ignores time too)
    API_BEGIN
    CHECK_PTR(sys); CHECK_PTR(dxdt); CHECK_PTR(x);
    if (sys->s.prec == ASAT_F64) sys_rhs<double>(&sys->s, &dxdt->st, &x->st);
    else sys_rhs<float>(&sys->s, &dxdt->st, &x->st);
    API_END
}

int asat_sys_violations(asat_sys_t* sys, const asat_state_t* x, int* count)
{
    API_BEGIN
    CHECK_PTR(sys); CHECK_PTR(x); CHECK_PTR(count);
    *count = sys->s.prec == ASAT_F64 ? sys_violations<double>(&sys->s, &x->st)
                                     : sys_violations<float>(&sys->s, &x->st);
    API_END
}

int asat_state_create(asat_sys_t* sys, asat_state_t** out)
{
    API_BEGIN
    CHECK_PTR(sys); CHECK_PTR(out);
    std::unique_ptr<State> st(state_new(&sys->s));
    asat_state* w = new asat_state();
    w->st = *st;
    st->d = nullptr;
    *out = w;
    API_END
}

int asat_state_destroy(asat_state_t* st)
{
    API_BEGIN
    if (st) {
        if (st->st.d) (void)hipFree(st->st.d);
        delete st;
    }
    API_END
}

int asat_state_set_public(asat_state_t* st, const void* host_pub)
{
    API_BEGIN
    CHECK_PTR(st); CHECK_PTR(host_pub);
    state_set_public(&st->st, host_pub);
    API_END
}

int asat_state_get_public(const asat_state_t* st, void* host_pub)
{
    API_BEGIN
    CHECK_PTR(st); CHECK_PTR(host_pub);
    state_get_public(&st->st, host_pub);
    API_END
}

int asat_state_get_boolean(const asat_state_t* st, unsigned char* out)
{
    API_BEGIN
    CHECK_PTR(st); CHECK_PTR(out);
    const Sys* s = st->st.sys;
    std::vector<char> buf((size_t)s->esize * s->n);
    state_get_spins(&st->st, buf.data());
    for (int i = 0; i < s->n; i++)
        out[i] = s->prec == ASAT_F64 ? (((double*)buf.data())[i] > 0) : (((float*)buf.data())[i] > 0);
    API_END
}

int asat_state_copy(asat_state_t* dst, const asat_state_t* src)
{
    API_BEGIN
    CHECK_PTR(dst); CHECK_PTR(src);
    state_check(&dst->st); state_check(&src->st);
    require(dst->st.sys == src->st.sys, ASAT_ERR_INVALID_ARGUMENT, "states belong to different systems");
    Sys* s = dst->st.sys;
    HIP_CHECK(hipMemcpyAsync(dst->st.d, src->st.d, (size_t)s->esize * s->alloc, hipMemcpyDeviceToDevice, s->stream));
    HIP_CHECK(hipStreamSynchronize(s->stream));
    API_END
}

int asat_state_set_zero(asat_state_t* st)
{
    API_BEGIN
    CHECK_PTR(st);
    state_check(&st->st);
    Sys* s = st->st.sys;
    HIP_CHECK(hipMemsetAsync(st->st.d, 0, (size_t)s->esize * s->alloc, s->stream));
    HIP_CHECK(hipStreamSynchronize(s->stream));
    API_END
}

int asat_state_alloc_size(const asat_state_t* st, int* size)
{
    API_BEGIN
    CHECK_PTR(st); CHECK_PTR(size);
    *size = st->st.alloc;
    API_END
}

int asat_state_device_ptr(asat_state_t* st, void** dev_ptr, int* aux_offset)
{
    API_BEGIN
    CHECK_PTR(st); CHECK_PTR(dev_ptr);
    *dev_ptr = st->st.d;
    if (aux_offset) *aux_offset = st->st.sys->aoff;
    API_END
}

int asat_sys_set_family(asat_sys_t* sys, int family)
{
    API_BEGIN
    CHECK_PTR(sys);
    require(family == ASAT_FAMILY_CTDS || family == ASAT_FAMILY_TANH, ASAT_ERR_INVALID_ARGUMENT,
            "unknown right-hand-side family");
    HIP_CHECK(hipStreamSynchronize(sys->s.stream));
    sys->s.family = family;
    API_END
}

int asat_sys_get_family(const asat_sys_t* sys, int* family)
{
    API_BEGIN
    CHECK_PTR(sys); CHECK_PTR(family);
    *family = sys->s.family;
    API_END
}

int asat_sys_set_q(asat_sys_t* sys, double q)
{
    API_BEGIN
    CHECK_PTR(sys);
    require(std::isfinite(q), ASAT_ERR_INVALID_ARGUMENT, "q must be finite");
    HIP_CHECK(hipStreamSynchronize(sys->s.stream));
    sys->s.q = q;
    API_END
}

int asat_sys_get_q(const asat_sys_t* sys, double* q)
{
    API_BEGIN
    CHECK_PTR(sys); CHECK_PTR(q);
    *q = sys->s.q;
    API_END
}

int asat_sys_clause_order(const asat_sys_t* sys, int* order)
{
    API_BEGIN
    CHECK_PTR(sys); CHECK_PTR(order);
    const Sys* s = &sys->s;
    s->require_ready();
    for (int j = 0; j < s->m; j++) order[j] = s->perm.empty() ? j : s->perm[j];
    API_END
}

int asat_sys_layout(const asat_sys_t* sys, asat_layout_t* out)
{
    API_BEGIN
    CHECK_PTR(sys); CHECK_PTR(out);
    const Sys* s = &sys->s;
    s->require_ready();
    out->clause_pass = s->tiled ? ASAT_CLAUSE_TILED : ASAT_CLAUSE_GENERIC;
    out->var_pass = s->lds_var ? ASAT_VAR_REGION : (s->wide_var ? ASAT_VAR_WIDE : ASAT_VAR_GATHER);
    out->groups = s->ngroups;
    out->group_vars = s->vg;
    out->tiles = s->tiled ? (int)ceil_div(s->m, s->tc) : 0;
    out->tile_clauses = s->tiled ? s->tc : 0;
    out->clause_grid = clause_grid(s);
    out->var_grid = var_grid(s);
    out->var_lds_bytes = s->var_lds;
    out->slot_spins = (s->tiled && s->lds_var) ? 1 : 0;
    out->direct_primary = s->split ? 1 : 0;
    out->run_tables = s->d_runs ? 1 : 0;
    out->primary_words = s->d_pw16 ? 1 : 0;
    API_END
}

int asat_sys_set_random_state(asat_sys_t* sys, asat_state_t* x, asat_rng_t* rng)
{
    API_BEGIN
    CHECK_PTR(sys); CHECK_PTR(x); CHECK_PTR(rng);
    Sys* s = &sys->s;
    s->require_ready();
    state_check(&x->st);
    const int len = s->n + s->m;
    void* u = nullptr;
    HIP_CHECK(hipMalloc(&u, (size_t)s->esize * len));
    dim3 g(ceil_div(len, 256)), b(256);
    if (s->prec == ASAT_F64) {
        hipLaunchKernelGGL(k_uniform<double>, g, b, 0, s->stream, (double*)u, len, rng->g.seed, rng->g.offset);
        hipLaunchKernelGGL(k_set_initial<double>, g, b, 0, s->stream, (double*)x->st.d, s->n, s->m, s->aoff,
                           (const double*)u, (const int*)s->d_perm);
    } else {
        hipLaunchKernelGGL(k_uniform<float>, g, b, 0, s->stream, (float*)u, len, rng->g.seed, rng->g.offset);
        hipLaunchKernelGGL(k_set_initial<float>, g, b, 0, s->stream, (float*)x->st.d, s->n, s->m, s->aoff,
                           (const float*)u, (const int*)s->d_perm);
    }
    rng->g.offset += (unsigned long long)len;
    hipError_t e = hipGetLastError();
    hipError_t e2 = hipStreamSynchronize(s->stream);
    (void)hipFree(u);
    HIP_CHECK(e);
    HIP_CHECK(e2);
    API_END
}

int asat_rk_create(asat_rk_t** out)
{
    API_BEGIN
    CHECK_PTR(out);
    *out = new asat_rk();
    API_END
}

int asat_rk_destroy(asat_rk_t* rk)
{
    API_BEGIN
    delete rk;
    API_END
}

int asat_rk_set_eps(asat_rk_t* rk, double eps)
{
    API_BEGIN
    CHECK_PTR(rk);
    // CpuRungeKutta::SetEpsilon (AnalogSAT/cpu_sat/CpuRungeKutta.cpp:126-131)
    require(!(eps < 1e-16 || eps > 1.0), ASAT_ERR_INVALID_ARGUMENT, "epsilon must be between 1e-16 and 1");
    rk->r.eps = eps;
    if (rk->r.configured) {
        hipLaunchKernelGGL(k_ctrl_set_eps, dim3(1), dim3(64), 0, rk->r.sys->stream, rk->r.d_ctrl, eps, rk->r.floor);
        HIP_CHECK(hipGetLastError());
        HIP_CHECK(hipStreamSynchronize(rk->r.sys->stream));
    }
    API_END
}

int asat_rk_set_xscal_floor(asat_rk_t* rk, double floor)
{
    API_BEGIN
    CHECK_PTR(rk);
    require(floor > 0.0 && floor <= 1.0, ASAT_ERR_INVALID_ARGUMENT, "xscal floor must be in (0, 1]");
    rk->r.floor = floor;
    if (rk->r.configured) {
        hipLaunchKernelGGL(k_ctrl_set_eps, dim3(1), dim3(64), 0, rk->r.sys->stream, rk->r.d_ctrl, rk->r.eps, floor);
        HIP_CHECK(hipGetLastError());
        HIP_CHECK(hipStreamSynchronize(rk->r.sys->stream));
    }
    API_END
}

__global__ void k_ctrl_set_log(Ctrl* c, double* hlog, long long len)
{
    if (threadIdx.x == 0 && blockIdx.x == 0) {
        c->hlog = hlog;
        c->hlog_len = len;
    }
}

int asat_rk_set_step_log(asat_rk_t* rk, double* dev_hlog, long long len)
{
    API_BEGIN
    CHECK_PTR(rk);
    require(len >= 0 && (len == 0 || dev_hlog != nullptr), ASAT_ERR_INVALID_ARGUMENT, "bad step log");
    rk->r.hlog = len ? dev_hlog : nullptr;
    rk->r.hlog_len = len;
    if (rk->r.configured) {
        hipLaunchKernelGGL(k_ctrl_set_log, dim3(1), dim3(64), 0, rk->r.sys->stream, rk->r.d_ctrl, rk->r.hlog,
                           rk->r.hlog_len);
        HIP_CHECK(hipGetLastError());
        HIP_CHECK(hipStreamSynchronize(rk->r.sys->stream));
    }
    API_END
}

int asat_rk_get_eps(const asat_rk_t* rk, double* eps)
{
    API_BEGIN
    CHECK_PTR(rk); CHECK_PTR(eps);
    *eps = rk->r.eps;
    API_END
}

int asat_rk_configure(asat_rk_t* rk, asat_sys_t* sys)
{
    API_BEGIN
    CHECK_PTR(rk); CHECK_PTR(sys);
    rk_configure(&rk->r, &sys->s);
    API_END
}

int asat_rk_step(asat_rk_t* rk, asat_state_t* old_state, asat_state_t* new_state, int count)
{
    API_BEGIN
    CHECK_PTR(rk); CHECK_PTR(old_state); CHECK_PTR(new_state);
    int rc = rk_step(&rk->r, &old_state->st, &new_state->st, count);
    if (rc == ASAT_UNDERFLOW) {
        asat::g_last_error = "step size underflow";
        return rc;
    }
    API_END
}

int asat_rk_set_one_workgroup(asat_rk_t* rk, int enable)
{
    API_BEGIN
    CHECK_PTR(rk);
    rk->r.small_mode = enable ? 1 : 0;
    API_END
}

int asat_rk_uses_one_workgroup(const asat_rk_t* rk, int* uses)
{
    API_BEGIN
    CHECK_PTR(rk); CHECK_PTR(uses);
    rk->r.require_configured();
    *uses = small_path(&rk->r) && persistent_workgroups(const_cast<RK*>(&rk->r)) == 1 ? 1 : 0;
    API_END
}

int asat_rk_workgroups(const asat_rk_t* rk, int* workgroups)
{
    API_BEGIN
    CHECK_PTR(rk); CHECK_PTR(workgroups);
    rk->r.require_configured();
    *workgroups = persistent_workgroups(const_cast<RK*>(&rk->r));
    API_END
}

int asat_rk_set_grid_limits(asat_rk_t* rk, int workgroups, int attempts, int launches)
{
    API_BEGIN
    CHECK_PTR(rk);
    require(workgroups >= 0 && attempts >= 0, ASAT_ERR_INVALID_ARGUMENT, "limits must be >= 0");
    rk->r.grid_workgroups = workgroups;
    rk->r.grid_attempts = attempts;
    rk->r.grid_launches = launches;
    API_END
}

int asat_rk_solve(asat_rk_t* rk, asat_state_t* old_state, asat_state_t* new_state, int batch, long long max_steps,
                  double max_time, int time_float, asat_solve_result_t* out)
{
    API_BEGIN
    CHECK_PTR(rk); CHECK_PTR(old_state); CHECK_PTR(new_state); CHECK_PTR(out);
    rk_solve(&rk->r, &old_state->st, &new_state->st, batch, max_steps, max_time, time_float, out);
    API_END
}

int asat_rk_reset(asat_rk_t* rk)
{
    API_BEGIN
    CHECK_PTR(rk);
    // no copy into the host control block may be pending when it is rewritten
    if (rk->r.configured) HIP_CHECK(hipStreamSynchronize(rk->r.sys->stream));
    rk_reset(&rk->r);
    API_END
}

int asat_rk_stats(const asat_rk_t* rk, asat_rk_stats_t* out)
{
    API_BEGIN
    CHECK_PTR(rk); CHECK_PTR(out);
    rk->r.require_configured();
    const Ctrl* c = rk->r.h_ctrl;
    out->time = c->time;
    out->hdid = c->hdid;
    out->hnext = c->hnext;
    out->errmax = c->errmax;
    out->steps = c->steps;
    out->attempts = c->attempts;
    out->rhscount = c->rhscount;
    API_END
}

int asat_rk_last_step_ms(const asat_rk_t* rk, float* ms)
{
    API_BEGIN
    CHECK_PTR(rk); CHECK_PTR(ms);
    *ms = rk->r.last_ms;
    API_END
}

int asat_rk_set_kernel_timer(asat_rk_t* rk, int kind)
{
    API_BEGIN
    CHECK_PTR(rk);
    require(kind >= -1 && kind <= 12, ASAT_ERR_INVALID_ARGUMENT, "kernel kind must be -1 (off) or 0..12");
    rk->r.timer_kind = kind;
    rk->r.timer_ms = 0.0;
    rk->r.timer_launches = 0;
    API_END
}

int asat_rk_kernel_timer(const asat_rk_t* rk, double* total_ms, long long* launches)
{
    API_BEGIN
    CHECK_PTR(rk); CHECK_PTR(total_ms); CHECK_PTR(launches);
    *total_ms = rk->r.timer_ms;
    *launches = rk->r.timer_launches;
    API_END
}

int asat_rk_profile(asat_rk_t* rk, asat_state_t* old_state, asat_state_t* new_state, int reps, float* us_out)
{
    API_BEGIN
    CHECK_PTR(rk); CHECK_PTR(old_state); CHECK_PTR(new_state); CHECK_PTR(us_out);
    RK* r = &rk->r;
    r->require_configured();
    state_check(&old_state->st); state_check(&new_state->st);
    require(reps > 0, ASAT_ERR_INVALID_ARGUMENT, "reps must be positive");
    require(old_state->st.d != new_state->st.d, ASAT_ERR_INVALID_ARGUMENT, "old and new state must differ");
    if (r->prec == ASAT_F64) rk_profile_impl<double>(r, &old_state->st, &new_state->st, reps, us_out);
    else rk_profile_impl<float>(r, &old_state->st, &new_state->st, reps, us_out);
    API_END
}

int asat_util_copy_bench(long long bytes, int reps, float* us_per_copy)
{
    API_BEGIN
    CHECK_PTR(us_per_copy);
    require(bytes >= 16 && bytes % 16 == 0 && reps > 0, ASAT_ERR_INVALID_ARGUMENT,
            "bytes must be a positive multiple of 16 and reps positive");
    void *a = nullptr, *b = nullptr;
    HIP_CHECK(hipMalloc(&a, (size_t)bytes));
    HIP_CHECK(hipMalloc(&b, (size_t)bytes));
    HIP_CHECK(hipMemset(a, 1, (size_t)bytes));
    hipEvent_t e0, e1;
    HIP_CHECK(hipEventCreate(&e0));
    HIP_CHECK(hipEventCreate(&e1));
    const long long n16 = bytes / 16;
    hipLaunchKernelGGL(k_copy16, dim3(4096), dim3(256), 0, 0, (const int4*)a, (int4*)b, n16);
    HIP_CHECK(hipEventRecord(e0, 0));
    for (int r = 0; r < reps; r++)
        hipLaunchKernelGGL(k_copy16, dim3(4096), dim3(256), 0, 0, (const int4*)a, (int4*)b, n16);
    HIP_CHECK(hipEventRecord(e1, 0));
    HIP_CHECK(hipEventSynchronize(e1));
    float ms = 0.f;
    HIP_CHECK(hipEventElapsedTime(&ms, e0, e1));
    *us_per_copy = ms * 1000.f / reps;
    (void)hipEventDestroy(e0); (void)hipEventDestroy(e1);
    (void)hipFree(a); (void)hipFree(b);
    API_END
}

int asat_util_stream_bench(long long bytes, int reps, float* us_copy, float* us_read)
{
    API_BEGIN
    CHECK_PTR(us_copy); CHECK_PTR(us_read);
    require(bytes >= 16 && bytes % 16 == 0 && reps > 0, ASAT_ERR_INVALID_ARGUMENT,
            "bytes must be a positive multiple of 16 and reps positive");
    void *a = nullptr, *b = nullptr;
    int* o = nullptr;
    HIP_CHECK(hipMalloc(&a, (size_t)bytes));
    HIP_CHECK(hipMalloc(&b, (size_t)bytes));
    HIP_CHECK(hipMalloc((void**)&o, sizeof(int)));
    HIP_CHECK(hipMemset(a, 0, (size_t)bytes));
    hipEvent_t e0, e1;
    HIP_CHECK(hipEventCreate(&e0));
    HIP_CHECK(hipEventCreate(&e1));
    const long long n16 = bytes / 16;
    const dim3 grid(8192), blk(256);
    float ms = 0.f;
    hipLaunchKernelGGL(k_stream_copy, grid, blk, 0, 0, (const stream_v4*)a, (stream_v4*)b, n16);
    HIP_CHECK(hipEventRecord(e0, 0));
    for (int r = 0; r < reps; r++) hipLaunchKernelGGL(k_stream_copy, grid, blk, 0, 0, (const stream_v4*)a, (stream_v4*)b, n16);
    HIP_CHECK(hipEventRecord(e1, 0));
    HIP_CHECK(hipEventSynchronize(e1));
    HIP_CHECK(hipEventElapsedTime(&ms, e0, e1));
    *us_copy = ms * 1000.f / reps;
    hipLaunchKernelGGL(k_stream_read, grid, blk, 0, 0, (const stream_v4*)a, o, n16);
    HIP_CHECK(hipEventRecord(e0, 0));
    for (int r = 0; r < reps; r++) hipLaunchKernelGGL(k_stream_read, grid, blk, 0, 0, (const stream_v4*)a, o, n16);
    HIP_CHECK(hipEventRecord(e1, 0));
    HIP_CHECK(hipEventSynchronize(e1));
    HIP_CHECK(hipEventElapsedTime(&ms, e0, e1));
    *us_read = ms * 1000.f / reps;
    (void)hipEventDestroy(e0); (void)hipEventDestroy(e1);
    (void)hipFree(a); (void)hipFree(b); (void)hipFree(o);
    API_END
}

int asat_util_gpu_name(char* buf, int len)
{
    API_BEGIN
    CHECK_PTR(buf);
    require(len > 0, ASAT_ERR_INVALID_ARGUMENT, "len must be positive");
    int dev = 0;
    HIP_CHECK(hipGetDevice(&dev));
    hipDeviceProp_t prop;
    HIP_CHECK(hipGetDeviceProperties(&prop, dev));
    if (prop.name[0] != '\0') {
        std::snprintf(buf, (size_t)len, "%s", prop.name);
    } else {
        // some drivers leave the marketing name empty: the architecture then
        // names the device (the part of gcnArchName before its feature flags)
        std::string arch(prop.gcnArchName);
        arch = arch.substr(0, arch.find(':'));
        std::snprintf(buf, (size_t)len, "AMD GPU %s", arch.empty() ? "(unknown)" : arch.c_str());
    }
    API_END
}

int asat_rng_create(unsigned long long seed, asat_rng_t** out)
{
    API_BEGIN
    CHECK_PTR(out);
    asat_rng* r = new asat_rng();
    r->g.seed = seed;
    r->g.offset = 0;
    *out = r;
    API_END
}

int asat_rng_destroy(asat_rng_t* rng)
{
    API_BEGIN
    delete rng;
    API_END
}

int asat_rng_uniform(asat_rng_t* rng, void* dev_ptr, int len, int precision)
{
    API_BEGIN
    CHECK_PTR(rng); CHECK_PTR(dev_ptr);
    require(len >= 0, ASAT_ERR_INVALID_ARGUMENT, "negative length");
    require(precision == ASAT_F64 || precision == ASAT_F32, ASAT_ERR_INVALID_ARGUMENT, "unknown precision");
    if (len == 0) return ASAT_OK;
    dim3 g(ceil_div(len, 256)), b(256);
    if (precision == ASAT_F64)
        hipLaunchKernelGGL(k_uniform<double>, g, b, 0, 0, (double*)dev_ptr, len, rng->g.seed, rng->g.offset);
    else
        hipLaunchKernelGGL(k_uniform<float>, g, b, 0, 0, (float*)dev_ptr, len, rng->g.seed, rng->g.offset);
    HIP_CHECK(hipGetLastError());
    HIP_CHECK(hipDeviceSynchronize());
    rng->g.offset += (unsigned long long)len;
    API_END
}

}  // extern "C"
