// The sequential sweeps of OpenFOAM's preconditioners and smoothers, one launch per sweep.
//
// A sweep in index order is a chain of dependencies, as deep as the mesh's level schedule: on 64^3 cells 190
// levels of 1,400 cells, on a 2-D mesh of 12,000 cells 250 levels of 50. What bounds it is the time from one
// level to the next, not bytes or arithmetic. A launch per level costs 3 us of kernel (four dependent loads:
// cell, run, face and neighbour, value) and about 1 us between kernels. Here:
//   - the addressing is laid out once per mesh in level order (SweepPlan), so that the address of everything
//     but the neighbours' values follows from a cell's place in the order and is loaded steps ahead;
//   - up to kLdsCells cells, one workgroup walks every level with the swept values in its LDS and a
//     workgroup barrier between levels; a small launch before it gathers the coefficients into the order
//     the walk reads them in (one CU's gathers would cost more than the chain);
//   - above that, waves take chunks of one level in order and hand values on through memory, each value
//     tagged so that a reader knows it without any fence or barrier (flow* below).
// Each cell's arithmetic is the host loop's, in its face order, so the results are the launch-per-level
// path's and the host's to the bit.
// Measured, a launch per level before: one DILU application on 64^3 cells (forward and backward, 380 levels)
// 1,280 -> 196 us, 0.5 us a level, the time a value takes between two CUs; OpenFOAM's GAMG with Gauss-Seidel
// on a 2-D mesh of 12,180 cells 486 -> 62.6 ms, and 61 -> 42.7 with successive sweeps overlapped.
#include "handover.hpp"
#include "sweep.hpp"

#include <algorithm>

namespace mfv {

// Plan of one mesh's sweeps. "Place" is a cell's index in the forward level order; values in LDS and in the
// hand-over buffer are kept by place, so a level's reads and writes are mostly contiguous. A step is a run
// of at most `threads` cells of one level. Entry k of its lane i -- a face (-1: none), and where its
// neighbour's value is -- is entry first + k*cells + i; in an LDS plan, whose values are found at byte
// offsets, a lane's entries lie in pairs, for loads of two.
struct Walk
{
    int nSteps = 0, nEntries = 0;
    const int4* steps = nullptr;   // {first lane, cells, first entry, entries per cell}
    const int* cell = nullptr;     // per lane: the cell (the level schedule's list);
    int* self = nullptr;           // its place, or (Gauss-Seidel) its number of lower faces
    int *face = nullptr, *pos = nullptr;   // entries
    int* entryCell = nullptr;      // LDS: the entry's cell
    unsigned* at = nullptr;        // LDS: in place of pos
};

struct SweepPlan
{
    bool usable = false;      // false: the mesh keeps a launch per level
    bool lds = false;
    bool wide = false;        // a cell with more lower or owned faces than the narrow kernels load ahead
    SweepFactor factors = 0;  // the last factorisation
    SweepFactor packed = 0;   // LDS: the one whose products are in aFwd, aBwd and dFwd (0: none)
    int n = 0, threads = 64;
    DBuf<int4> steps, gsSteps;     // the walks' steps
    DBuf<uint8_t> mem, gsMem;      // and the rest of them
    int* place = nullptr;          // per cell
    Walk fwd, bwd;            // lower faces ascending; owned faces descending
    bool gsReady = false, gsUsable = false;
    Walk gs;                  // Gauss-Seidel's forward walk: both runs of faces, ascending
    int gsAhead = 0;          // its entries loaded ahead
    int gsLag = 0;            // LDS: a step's neighbours lie fewer steps than this from it
    // LDS: coefficients and cell values in the walks' orders
    double *aFwd = nullptr, *aBwd = nullptr, *dFwd = nullptr, *aGs = nullptr, *aGsBack = nullptr, *gsIn = nullptr;
    // flow: the hand-over buffer and the launches' state (chunks.hpp)
    Word* hand = nullptr;
    DBuf<unsigned> state;
};
void SweepPlanDeleter::operator()(SweepPlan* p) const { delete p; }

namespace {

// 160,008 of the 163,840 bytes of LDS a workgroup may hold. At the line the LDS walk is the faster: a DILU
// solve takes 1.4 ms on 18,850 cells (77 levels, 0.35 us a level), 2.1 ms on 32^3 by flow (94 levels).
constexpr int kLdsCells = 20000;
constexpr int kLdsThreads = 512;
// Above this a mesh keeps a launch per level: the gain falls as the levels widen and the values' words (16
// bytes) become traffic. A DILU solve of n^3 cells against a launch per level: 6.6x at 64^3, 6.0x at 128^3,
// 3.3x at 200^3, 2.0x at 272^3 (20 M cells, 165 -> 83 ms); the plan takes about 76 bytes a cell of a hex mesh, and
// 52 more with Gauss-Seidel's walk.
constexpr int kFlowMaxCells = 1 << 25;
// A mesh of so few levels keeps a launch per level too: its sweep is a stream over the cells, which a launch a level
// runs with the whole chip, one workgroup or kFlowWaves waves with a part of it. A DIC application, one launch a sweep
// and a launch per level, us: cells in two colours (two levels) 51 and 36 on 16^3 cells, 131 and 38 on 27^3, 213 and
// 110 on 64^3, 636 and 153 on 1 M; numbered at random (16 to 20 levels) 75 and 205, 159 and 316, 236 and 512, 697 and
// 802; at 4.1 M 2,640 and 2,400, two Gauss-Seidel sweeps 2,100 and 2,660. On a few hundred cells, GAMG's coarse grids,
// the launches are the cost whatever the levels: there only a mesh of one level has no plan.
int fewLevels(int n, bool lds) { return lds ? std::min(9, 1 + n / 1700) : 2 + std::min(10, n / 60000); }
// Entries of a step's cell that are loaded ahead, by the most that a cell of the mesh has (a hex mesh's have
// three lower and three owned faces, agglomerated ones more); a cell's entries past these are loaded where
// they are used. Substitution in LDS (in pairs) and by flow, Gauss-Seidel in LDS and by flow:
constexpr int kLdsNarrow = 4, kFlowNarrow = 3, kWide = 8;
constexpr int kGsNarrow = 6, kGsMiddle = 8, kGsWide = 12;

// LDS-only ordering between a step's writes and the next one's reads: a full __syncthreads would also wait
// for the loads in flight for later steps.
__device__ __forceinline__ void ldsBarrier()
{
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup", "local");
    __builtin_amdgcn_s_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup", "local");
}

// ---------------- one workgroup, the values in LDS ----------------

struct LdsWalk
{
    int nSteps, lane;                  // lane: the thread's place among those that walk together
    const int4* __restrict__ steps;
    const int* __restrict__ cell;
    const int* __restrict__ self;
    const unsigned* __restrict__ at;   // the entries' values: byte offsets in LDS
    const double* __restrict__ a;      // the entries' coefficients
};

// A lane's step as loaded ahead: its first W entries (a step holds at least W per cell), two values of the
// cell (v, d0), and where its own value is. One wave's instructions, at four cycles each, are most of a
// step, so: addresses are a uniform base and the lane's offset, and an absent entry needs no test -- its
// coefficient is 0 and its value a 1 kept after the last cell's, and s - 0*1 and s - 0/1 are s.
template <int W>
struct Step
{
    int first, cnt, w, e;   // uniform
    unsigned at[W];
    double a[W], v, d0;
    int c;
    unsigned own;
};

__device__ __forceinline__ double& ldsAt(double* val, unsigned byteOffset)
{
    return *reinterpret_cast<double*>(reinterpret_cast<char*>(val) + byteOffset);
}

// Lanes past the step's cells and steps past the walk's end read the last ones: every load is unconditional
// and in bounds, so they issue together and none waits behind a branch. i: the lane's cell in the step.
template <int W>
__device__ __forceinline__ unsigned stepLoad(const LdsWalk& P, const int4 d, Step<W>& q)
{
    q.first = d.x;
    q.cnt = d.y;
    q.e = d.z;
    q.w = d.w;
    const unsigned i = (unsigned)min(P.lane, d.y - 1);
#pragma unroll
    for (int k = 0; k < W; k += 2)
    {
        const uint2* at = reinterpret_cast<const uint2*>(P.at + (d.z + k * d.y));
        const double2* a = reinterpret_cast<const double2*>(P.a + (d.z + k * d.y));
        const uint2 p = at[i];
        const double2 c = a[i];
        q.at[k] = p.x;
        q.at[k + 1] = p.y;
        q.a[k] = c.x;
        q.a[k + 1] = c.y;
    }
    return i;
}

// A walk with A step buffers that take turns (nothing in flight is copied, a copy would wait for it): while
// step s is computed, step s + A - 1 is loaded, with what the walk adds to it (more(step, i): loads at
// addresses that follow from the descriptor), and for step s + 2 what is found through a loaded index
// (gather). The step's own values are read from LDS first; compute(step, values) is the rest. The walk begins
// `late` barriers after the others of its workgroup.
template <int W, int A, typename More, typename Gather, typename Compute>
__device__ __forceinline__ void ldsWalk(const LdsWalk& P, double* val, More more, Gather gather, Compute compute,
                                        int late = 0)
{
    const int n = P.nSteps;
    Step<W> q[A];
    int4 d[A];
#pragma unroll
    for (int u = 0; u < A; ++u) d[u] = P.steps[min(u, n - 1)];
#pragma unroll
    for (int u = 0; u < A - 1; ++u)
    {
        more(q[u], stepLoad<W>(P, d[u], q[u]));
        d[u] = P.steps[min(u + A, n - 1)];
    }
    gather(q[0]);
    gather(q[1]);
    for (; late > 0; --late) ldsBarrier();
    for (int s = 0; s < n; s += A)
    {
#pragma unroll
        for (int u = 0; u < A; ++u)
        {
            if (s + u >= n) break;
            constexpr int last = A - 1;
            const int v = (u + last) % A;
            double x[W];
#pragma unroll
            for (int k = 0; k < W; ++k) x[k] = ldsAt(val, q[u].at[k]);
            more(q[v], stepLoad<W>(P, d[v], q[v]));
            d[v] = P.steps[min(s + u + last + A, n - 1)];
            gather(q[(u + 2) % A]);
            compute(q[u], x);
            ldsBarrier();
        }
    }
}
// buffers of a walk without and with gathers
constexpr int kAhead = 4, kAheadGather = 6;

// v after the entries of a lane's step: fn(v, coefficient, value, entry) per entry in order (Down: from the
// last). Entries past the W loaded ahead are read where they are used.
template <int W, bool Down, typename Fn>
__device__ __forceinline__ double entries(const LdsWalk& P, const Step<W>& q, double* val, const double (&x)[W],
                                          double v, Fn fn)
{
    auto far = [&](int k) {
        const unsigned e = q.e + (k & ~1) * q.cnt + 2 * P.lane + (k & 1);
        v = fn(v, P.a[e], ldsAt(val, P.at[e]), k);
    };
    const bool on = P.lane < q.cnt;
    if (Down && q.w > W && on)
        for (int k = q.w - 1; k >= W; --k) far(k);
#pragma unroll
    for (int j = 0; j < W; ++j)
    {
        const int k = Down ? W - 1 - j : j;
        v = fn(v, q.a[k], x[k], k);
    }
    if (!Down && q.w > W && on)
        for (int k = W; k < q.w; ++k) far(k);
    return v;
}

// d = diag - sum upper*lower/d[lower neighbour]; P.a holds upper*lower, dFwd the diagonal in and 1/d out
template <int W>
__global__ __launch_bounds__(kLdsThreads) void ldsFactorK(int n, LdsWalk P, double* dFwd, double* __restrict__ rD)
{
    extern __shared__ double val[];
    P.lane = threadIdx.x;
    if (threadIdx.x == 0) val[n] = 1.0;
    ldsBarrier();
    ldsWalk<W, kAhead>(
        P, val,
        [&](Step<W>& q, unsigned i) {
            const double* dg = dFwd + q.first;
            const int* cell = P.cell + q.first;
            q.v = dg[i];
            q.c = cell[i];
        },
        [](Step<W>&) {},
        [&](const Step<W>& q, const double (&x)[W]) {
            const double v = entries<W, false>(P, q, val, x, q.v, [](double s, double a, double y, int) { return s - a / y; });
            if ((int)threadIdx.x >= q.cnt) return;
            val[q.first + threadIdx.x] = v;
            const double inv = 1.0 / v;
            rD[q.c] = inv;
            dFwd[q.first + threadIdx.x] = inv;
        });
}

// y = rD*r, y -= (rD*lower)*y forward, y -= (rD*upper)*y backward; the products are in the walks' a
template <int W>
__global__ __launch_bounds__(kLdsThreads) void ldsSubstK(int n, LdsWalk F, LdsWalk B, const double* __restrict__ dFwd,
                                                         const double* __restrict__ r, double* __restrict__ y,
                                                         const int* __restrict__ stop)
{
    extern __shared__ double val[];
    if (stop && *stop) return;
    F.lane = B.lane = threadIdx.x;
    if (threadIdx.x == 0) val[n] = 1.0;
    ldsBarrier();
    auto sub = [](double s, double a, double x, int) { return s - a * x; };
    ldsWalk<W, kAheadGather>(
        F, val,
        [&](Step<W>& q, unsigned i) {
            const double* rd = dFwd + q.first;
            const int* cell = F.cell + q.first;
            q.d0 = rd[i];
            q.c = cell[i];
        },
        [&](Step<W>& q) { q.v = r[q.c]; },
        [&](const Step<W>& q, const double (&x)[W]) {
            const double v = entries<W, false>(F, q, val, x, q.d0 * q.v, sub);
            if ((int)threadIdx.x < q.cnt) val[q.first + threadIdx.x] = v;
        });
    ldsWalk<W, kAhead>(
        B, val,
        [&](Step<W>& q, unsigned i) {
            const int* cell = B.cell + q.first;
            const int* self = B.self + q.first;
            q.c = cell[i];
            q.own = 8u * (unsigned)self[i];
        },
        [](Step<W>&) {},
        [&](const Step<W>& q, const double (&x)[W]) {
            const double v = entries<W, false>(B, q, val, x, ldsAt(val, q.own), sub);
            if ((int)threadIdx.x >= q.cnt) return;
            ldsAt(val, q.own) = v;
            y[q.c] = v;
        });
}

// Gauss-Seidel: psi in LDS; a cell reads its lower neighbours' new values and its upper neighbours' old ones,
// as the in-place host loop does. in: b, the diagonal and psi by place, then room for bPrime.
// One sweep is bound by its chain of levels, 0.33 us each, with most of a workgroup's room unused. The
// neighbours of a step lie at most lag - 1 steps from it, so sweep s + 1 may take a step once sweep s has taken
// the lag - 1 steps after it: teams of `team` threads walk successive sweeps lag steps apart, in the same
// barriers, and no step reads what another team writes between two of them: two sweeps over 12,180 cells in 250
// levels 164 -> 104 us, four over their agglomerates 70 -> 42. Symmetric sweeps take turns (one team).
template <int W, int WB, bool Sym>
__global__ __launch_bounds__(kLdsThreads) void ldsGsK(int n, LdsWalk F, LdsWalk B, double* in, double* __restrict__ psi,
                                                      int nSweeps, int team, int lag)
{
    extern __shared__ double val[];
    const int teams = blockDim.x / team, mine = (int)__builtin_amdgcn_readfirstlane(threadIdx.x / team);
    const int tid = threadIdx.x - mine * team;
    F.lane = B.lane = tid;
    double* bPrime = in + 3 * (size_t)n;
    for (int i = threadIdx.x; i < n; i += blockDim.x) val[i] = in[2 * (size_t)n + i];
    if (threadIdx.x == 0) val[n] = 1.0;
    __syncthreads();
    for (int sw = 0; sw < nSweeps; sw += teams)
    {
        const int now = min(teams, nSweeps - sw);
        if (mine >= now)   // no sweep left for this team
        {
            for (int i = F.nSteps + (now - 1) * lag; i > 0; --i) ldsBarrier();
            continue;
        }
        ldsWalk<W, kAhead>(
            F, val,
            [&](Step<W>& q, unsigned i) {
                const double* b = in + q.first;
                const double* dg = in + n + q.first;
                q.v = b[i];
                q.d0 = dg[i];
                if (Sym)
                {
                    const int* low = F.self + q.first;
                    q.c = low[i];
                }
            },
            [](Step<W>&) {},
            [&](const Step<W>& q, const double (&x)[W]) {
                double low = q.v;   // b less the lower neighbours' terms
                const double t = entries<W, false>(F, q, val, x, q.v, [&](double s, double a, double y, int k) {
                    const double v = s - a * y;
                    if (Sym) low = k + 1 == q.c ? v : low;
                    return v;
                });
                const double v = t / q.d0;
                if (tid >= q.cnt) return;
                if (Sym) bPrime[q.first + tid] = low;
                val[q.first + tid] = v;
            },
            mine * lag);
        for (int i = (now - 1 - mine) * lag; i > 0; --i) ldsBarrier();
        if (!Sym) continue;
        __syncthreads();   // bPrime, written by the forward walk's lanes, is read by the reverse walk's
        // the reverse walk: the backward entries from the last (owned faces ascending)
        ldsWalk<WB, kAheadGather>(
            B, val,
            [&](Step<WB>& q, unsigned i) {
                const int* self = B.self + q.first;
                q.c = self[i];
            },
            [&](Step<WB>& q) {
                q.v = bPrime[q.c];
                q.d0 = in[n + q.c];
            },
            [&](const Step<WB>& q, const double (&x)[WB]) {
                const double t = entries<WB, true>(B, q, val, x, q.v,
                                                   [](double s, double a, double y, int) { return s - a * y; });
                const double v = t / q.d0;
                if (tid < q.cnt) val[q.c] = v;
            });
        __syncthreads();
    }
    __syncthreads();
    for (int i = threadIdx.x; i < n; i += blockDim.x) psi[F.cell[i]] = val[i];
}

// coefficients and cell values into the walks' orders
constexpr int kTpb = 256;

__global__ __launch_bounds__(kTpb) void packFactorK(int nE, const int* __restrict__ face, int n,
                                                    const int* __restrict__ cell, const double* __restrict__ diag,
                                                    const double* __restrict__ upper, const double* __restrict__ lower,
                                                    double* __restrict__ a, double* __restrict__ dFwd)
{
    const int e = blockIdx.x * kTpb + threadIdx.x;
    if (e < n) dFwd[e] = diag[cell[e]];
    if (e >= nE) return;
    const int f = face[e];
    a[e] = f >= 0 ? upper[f] * lower[f] : 0.0;
}

// rD*lower for the forward walk's entries, then rD*upper for the backward walk's
__global__ __launch_bounds__(kTpb) void packSubstK(int nF, const int* __restrict__ faceF, const int* __restrict__ cellF,
                                                   int nB, const int* __restrict__ faceB, const int* __restrict__ cellB,
                                                   const double* __restrict__ rD, const double* __restrict__ upper,
                                                   const double* __restrict__ lower, double* __restrict__ aF,
                                                   double* __restrict__ aB)
{
    const int e = blockIdx.x * kTpb + threadIdx.x;
    if (e < nF)
    {
        const int f = faceF[e];
        aF[e] = f >= 0 ? rD[cellF[e]] * lower[f] : 0.0;
    }
    if (e < nB)
    {
        const int f = faceB[e];
        aB[e] = f >= 0 ? rD[cellB[e]] * upper[f] : 0.0;
    }
}

__global__ __launch_bounds__(kTpb) void packGsK(int nF, const int* __restrict__ faceF, int nB,
                                                const int* __restrict__ faceB, int n, const int* __restrict__ cell,
                                                const double* __restrict__ diag, const double* __restrict__ upper,
                                                const double* __restrict__ b, const double* __restrict__ psi,
                                                double* __restrict__ aF, double* __restrict__ aB, double* __restrict__ in)
{
    const int e = blockIdx.x * kTpb + threadIdx.x;
    if (e < n)
    {
        const int c = cell[e];
        in[e] = b[c];
        in[n + e] = diag[c];
        in[2 * (size_t)n + e] = psi[c];
    }
    if (e < nF)
    {
        const int f = faceF[e];
        aF[e] = f >= 0 ? upper[f] : 0.0;
    }
    if (e < nB)
    {
        const int f = faceB[e];
        aB[e] = f >= 0 ? upper[f] : 0.0;
    }
}

// ---------------- waves that hand values on ----------------
//
// Workgroups of one wave take chunks (steps of at most 64 cells) in order and compute each as soon as the values
// it needs are there, as handover.hpp describes. (Workgroups of four waves, four chunks at a time: 64^3 cells
// 4.2 ms against 3.9, 128^3 9.8 to 18 depending on their number against 11.0.)

struct PlanView
{
    int nFwd, nBwd;
    const int4* __restrict__ steps[2];
    const int* __restrict__ cell[2];
    const int* __restrict__ self[2];
    const int* __restrict__ face[2];
    const int* __restrict__ pos[2];
};

// The addressing of one lane of a chunk: its first W entries (a chunk holds at least W per cell, the missing
// ones marked); lanes past the chunk's cells read the last one's, so every load is unconditional.
template <int W>
struct Lane
{
    int4 d;
    int c, self;
    int face[W], pos[W];
};

template <int W>
__device__ __forceinline__ void laneLoad(const int4* __restrict__ steps, int s, const int* __restrict__ cell,
                                         const int* __restrict__ self, const int* __restrict__ face,
                                         const int* __restrict__ pos, Lane<W>& L)
{
    L.d = steps[s];
    const int j = min((int)threadIdx.x, L.d.y - 1);
    L.c = cell[L.d.x + j];
    L.self = self[L.d.x + j];
#pragma unroll
    for (int k = 0; k < W; ++k)
    {
        L.face[k] = face[L.d.z + k * L.d.y + j];
        L.pos[k] = pos[L.d.z + k * L.d.y + j];
    }
}

// The entries from k0 on (those past the step's marked missing). A chunk with wide rows takes its entries W at a time:
// one after the other each cost the loads of its face and place, of its coefficient and of its value in a chain (110
// levels of 2,700 cells with up to 25 lower faces: 52 us a level, 22 so, 31 with a launch per level).
template <int W>
__device__ __forceinline__ void laneMore(int k0, const int* __restrict__ face, const int* __restrict__ pos, const int4 d,
                                         int (&f)[W], int (&p)[W])
{
    const int j = min((int)threadIdx.x, d.y - 1);
#pragma unroll
    for (int k = 0; k < W; ++k)
    {
        const int e = d.z + min(k0 + k, d.w - 1) * d.y + j;
        f[k] = face[e];
        p[k] = pos[e];
    }
#pragma unroll
    for (int k = 0; k < W; ++k)
        if (k0 + k >= d.w) f[k] = -1;
}

// The values of a lane's W entries; need: a bit per entry. Each poll reads all of them unconditionally
// (an entry that is not needed names a place in bounds), so it costs one round trip, not one per entry.
template <int W>
__device__ __forceinline__ void awaitAll(const Word* hand, const int (&pos)[W], unsigned need,
                                         unsigned tag, double (&x)[W])
{
    while (need)
    {
        Hand<double>::Raw v[W];
#pragma unroll
        for (int k = 0; k < W; ++k) v[k] = Hand<double>::get(hand, pos[k]);
#pragma unroll
        for (int k = 0; k < W; ++k)
            if ((need >> k & 1u) && v[k].is(tag))
            {
                x[k] = v[k].value();
                need &= ~(1u << k);
            }
    }
}

template <int W, bool Factor>
__global__ __launch_bounds__(64) void flowSubstK(PlanView P, const double* __restrict__ diag,
                                                 const double* __restrict__ upper, const double* __restrict__ lower,
                                                 const double* __restrict__ rD, const double* __restrict__ r,
                                                 double* __restrict__ out, Word* hand, unsigned* state,
                                                 const int* __restrict__ stop)
{
    if (stop && *stop) return;
    const unsigned tag = launchTag(state);
    const int lane = threadIdx.x, total = P.nFwd + (Factor ? 0 : P.nBwd);
    WaveChunks order(state);
    for (int s = order.next(); s < total; s = order.next())
    {
        const int back = s >= P.nFwd ? 1 : 0;   // uniform
        Lane<W> L;
        laneLoad<W>(P.steps[back], back ? s - P.nFwd : s, P.cell[back], P.self[back], P.face[back], P.pos[back], L);
        if (lane < L.d.y)
        {
            const int own = L.self;
            const double rd = Factor ? 0.0 : rD[L.c];
            const double v0 = back ? 0.0 : (Factor ? diag[L.c] : r[L.c]);
            const unsigned want = back ? tag + 1 : tag;
            double v = 0.0;
            for (int k0 = 0; k0 < L.d.w; k0 += W)
            {
                if (k0) laneMore<W>(k0, P.face[back], P.pos[back], L.d, L.face, L.pos);
                double a[W], x[W];
                unsigned need = 0;
#pragma unroll
                for (int k = 0; k < W; ++k)
                {
                    const int f = max(L.face[k], 0);
                    a[k] = Factor ? upper[f] * lower[f] : rd * (back ? upper[f] : lower[f]);
                    need |= (L.face[k] >= 0 ? 1u : 0u) << k;
                }
                const unsigned has = need;
                if (!k0)   // its own is there long before the neighbours'
                    v = back ? awaitValue<double>(hand, own, tag) : (Factor ? v0 : rd * v0);
                awaitAll<W>(hand, L.pos, need, want, x);
#pragma unroll
                for (int k = 0; k < W; ++k)
                    if (has >> k & 1u) v = Factor ? v - a[k] / x[k] : v - a[k] * x[k];
            }
            Hand<double>::put(hand, own, want, v);
            if (Factor)
                out[L.c] = 1.0 / v;
            else if (back)
                out[L.c] = v;
        }
    }
    leave(order, (unsigned)total, tag, 2);
}

// One Gauss-Seidel walk: forward (lower neighbours handed over; upper ones read from psi, where their old
// values stay until this cell's is published, since their walk waits for it), or symGaussSeidel's reverse.
template <int W, bool Back>
__global__ __launch_bounds__(64) void flowGsK(int nSteps, const int4* __restrict__ steps, const int* __restrict__ cell,
                                              const int* __restrict__ self, const int* __restrict__ face,
                                              const int* __restrict__ pos, const double* __restrict__ diag,
                                              const double* __restrict__ upper, const double* __restrict__ b,
                                              double* psi, double* bPrime, Word* hand, unsigned* state)
{
    const unsigned tag = launchTag(state);
    const int lane = threadIdx.x;
    WaveChunks order(state);
    for (int t = order.next(); t < nSteps; t = order.next())
    {
        Lane<W> L;
        laneLoad<W>(steps, t, cell, self, face, pos, L);
        if (lane < L.d.y)
        {
            const int own = Back ? L.self : L.d.x + lane;
            const int nl = Back ? L.d.w : L.self;   // the entries handed over: all, or the lower ones
            double v = Back ? bPrime[L.c] : b[L.c];
            const double dg = diag[L.c];
            if (!Back && bPrime && nl == 0) bPrime[L.c] = v;
            // the reverse walk from its last entries
            const int last = Back ? (L.d.w - 1) / W * W : 0;
            for (int k0 = last; Back ? k0 >= 0 : k0 < L.d.w; k0 += Back ? -W : W)
            {
                if (Back ? last > 0 : k0 > 0) laneMore<W>(k0, face, pos, L.d, L.face, L.pos);
                double a[W], x[W];
                unsigned has = 0, need = 0;
#pragma unroll
                for (int k = 0; k < W; ++k)
                {
                    a[k] = upper[max(L.face[k], 0)];
                    const bool on = L.face[k] >= 0;
                    has |= (on ? 1u : 0u) << k;
                    need |= (on && k0 + k < nl ? 1u : 0u) << k;
                    if (on && k0 + k >= nl) x[k] = psi[L.pos[k]];
                }
                awaitAll<W>(hand, L.pos, need, tag, x);
#pragma unroll
                for (int j = 0; j < W; ++j)
                {
                    const int k = Back ? W - 1 - j : j;
                    if (!(has >> k & 1u)) continue;
                    v -= a[k] * x[k];
                    if (!Back && bPrime && k0 + k + 1 == nl) bPrime[L.c] = v;
                }
            }
            v /= dg;
            psi[L.c] = v;
            Hand<double>::put(hand, own, tag, v);
        }
    }
    leave(order, (unsigned)nSteps, tag, 1);
}

// ---------------- host ----------------

bool capturing(hipStream_t s)
{
    hipStreamCaptureStatus st = hipStreamCaptureStatusNone;
    return hipStreamIsCapturing(s, &st) == hipSuccess && st != hipStreamCaptureStatusNone;
}

// ---------------- the plan, laid out on the device ----------------
//
// The first sweep on a mesh pays for it, so it is made where the addressing is: the steps' widths by a launch, their
// entries' places added up on the host (16 bytes a step), the entries written by another launch. First calls on a
// mesh, level schedule and all, against a launch per level without a plan: one DIC application 0.15 ms and 0.3 at
// 10^3 cells, 2.8 and 5.1 at 64^3, 20 and 24 at 128^3, 212 and 215 at 20 M; two Gauss-Seidel sweeps 0.23 and 0.22,
// 2.8 and 5.0, 20 and 24, 214 and 218. (By one host thread with uploads 128^3 took 151 and 257, 20 M 1,700 and 3,200.)

// the faces a walk's cells have as entries: the lower ones ascending, the owned ones descending, or both ascending
enum WalkKind : int { kLowerFaces, kOwnedFaces, kAllFaces };

struct MeshView
{
    const label* __restrict__ ownerStart;
    const label* __restrict__ neighbour;
    const label* __restrict__ losortStart;
    const label* __restrict__ losort;
    const label* __restrict__ losortOwner;
};
MeshView viewOf(const Mesh& m)
{
    return MeshView{m.ownerStart.p, m.neighbour.p, m.losortStart.p, m.losort.p, m.losortOwner.p};
}

__global__ __launch_bounds__(kTpb) void placeK(int n, const int* __restrict__ order, int* __restrict__ place)
{
    const int i = blockIdx.x * kTpb + threadIdx.x;
    if (i < n) place[order[i]] = i;
}

__global__ __launch_bounds__(kTpb) void zeroWordsK(size_t n, Word* __restrict__ w)
{
    const size_t i = (size_t)blockIdx.x * kTpb + threadIdx.x;
    if (i < n) w[i] = 0ull;
}

// a step's widest cell into its w, a wave to a step; the first nA steps are walk A's, the rest walk B's
__global__ __launch_bounds__(kTpb) void stepWidthK(int nSteps, int nA, MeshView M, WalkKind kindA,
                                                   const int* __restrict__ orderA, WalkKind kindB,
                                                   const int* __restrict__ orderB, int4* __restrict__ steps)
{
    const int s = blockIdx.x * (kTpb / 64) + (int)(threadIdx.x >> 6), lane = threadIdx.x & 63;
    if (s >= nSteps) return;
    const WalkKind kind = s < nA ? kindA : kindB;
    const int* order = s < nA ? orderA : orderB;
    const int4 d = steps[s];
    int k = 0;
    for (int i = lane; i < d.y; i += 64)
    {
        const int q = order[d.x + i];
        const int nl = M.losortStart[q + 1] - M.losortStart[q], no = M.ownerStart[q + 1] - M.ownerStart[q];
        k = max(k, kind == kLowerFaces ? nl : kind == kOwnedFaces ? no : nl + no);
    }
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) k = max(k, __shfl_xor(k, o, 64));
    if (lane == 0) steps[s].w = k;
}

// A walk's entries, a wave to a step: every one that its steps have room for, past a cell's faces those that name
// none. stepOf (may be null): per cell, its step.
template <WalkKind Kind, bool Lds>
__global__ __launch_bounds__(kTpb) void entriesK(int n, Walk W, MeshView M, const int* __restrict__ place,
                                                 int* __restrict__ stepOf)
{
    const int s = blockIdx.x * (kTpb / 64) + (int)(threadIdx.x >> 6), lane = threadIdx.x & 63;
    if (s >= W.nSteps) return;
    const int4 d = W.steps[s];
    for (int i = lane; i < d.y; i += 64)
    {
        const int q = W.cell[d.x + i];
        const int l0 = M.losortStart[q], nl = Kind == kOwnedFaces ? 0 : M.losortStart[q + 1] - l0;
        const int o0 = M.ownerStart[q], no = Kind == kLowerFaces ? 0 : M.ownerStart[q + 1] - o0;
        W.self[d.x + i] = Kind == kAllFaces ? nl : place[q];
        if (stepOf) stepOf[q] = s;
        for (int k = 0; k < d.w; ++k)
        {
            const size_t e = Lds ? (size_t)d.z + (size_t)(k & ~1) * d.y + 2 * i + (k & 1) : (size_t)d.z + (size_t)k * d.y + i;
            int f = -1, p = Lds ? n : 0;
            if (k < nl)
            {
                f = M.losort[l0 + k];
                p = place[M.losortOwner[l0 + k]];
            }
            else if (k < nl + no)
            {
                f = Kind == kOwnedFaces ? o0 + no - 1 - k : o0 + k - nl;
                const int c = M.neighbour[f];
                // Gauss-Seidel reads an upper neighbour's old value, in memory by cell
                p = Kind == kAllFaces && !Lds ? c : place[c];
            }
            W.face[e] = f;
            if (Lds)
            {
                W.entryCell[e] = f >= 0 ? q : 0;
                W.at[e] = 8u * (unsigned)p;
            }
            else
                W.pos[e] = p;
        }
    }
}

// the most steps that lie between a face's two cells
__global__ __launch_bounds__(kTpb) void stepReachK(int nF, const label* __restrict__ owner,
                                                   const label* __restrict__ neighbour,
                                                   const int* __restrict__ stepOf, int* __restrict__ reach)
{
    const int f = blockIdx.x * kTpb + threadIdx.x;
    if (f < nF) atomicMax(reach, abs(stepOf[neighbour[f]] - stepOf[owner[f]]));
}

inline int blocks(int n) { return (n + kTpb - 1) / kTpb; }
inline int waveBlocks(int n) { return (n + kTpb / 64 - 1) / (kTpb / 64); }

// Room for a plan's entries: a hex mesh fills about one per face and run, an agglomerated grid two or three.
// A cell with very many faces in a wide level would pad its whole step; such a mesh keeps a launch per level.
long long entryRoom(const Mesh& m) { return std::min(0x7fffffffLL, 16LL * ((long long)m.nCells + m.nFaces)); }

// `steps` gets the levels cut into steps of at most `threads` cells
void cutSteps(const std::vector<int>& start, int threads, std::vector<int4>& steps)
{
    for (size_t l = 0; l + 1 < start.size(); ++l)
        for (int a = start[l]; a < start[l + 1]; a += threads) steps.push_back(int4{a, std::min(threads, start[l + 1] - a), 0, 0});
}

int widestCell(const std::vector<int4>& steps)
{
    int most = 0;
    for (const int4& d : steps) most = std::max(most, d.w);
    return most;
}

// Room for a walk's steps [a, b): the entries of each from its widest cell's, and at least `least`. False where they
// would not fit.
bool placeEntries(std::vector<int4>& steps, size_t a, size_t b, bool lds, int least, long long room, Walk& w)
{
    long long entries = 0;
    for (size_t s = a; s < b; ++s)
    {
        int k = std::max(least, steps[s].w);
        if (lds) k = (k + 1) & ~1;
        steps[s].z = (int)entries;
        steps[s].w = k;
        entries += (long long)k * steps[s].y;
        if (entries > room) return false;
    }
    w.nSteps = (int)(b - a);
    w.nEntries = (int)entries;
    return true;
}

// arrays in one allocation: first with the base null, for the bytes, then with it
struct Carve
{
    uint8_t* base;
    size_t used = 0;
    template <typename T>
    void operator()(T*& p, size_t n)
    {
        p = reinterpret_cast<T*>(base + used);
        used += (n * sizeof(T) + 255) / 256 * 256;
    }
};
template <typename Fn>
void carve(DBuf<uint8_t>& mem, Fn fn)
{
    Carve size{nullptr};
    fn(size);
    mem.resize(size.used);
    Carve at{mem.p};
    fn(at);
}
void carveWalk(Carve& c, Walk& w, int n, bool lds)
{
    c(w.self, (size_t)n);
    c(w.face, (size_t)w.nEntries);
    if (lds)
    {
        c(w.entryCell, (size_t)w.nEntries);
        c(w.at, (size_t)w.nEntries);
    }
    else
        c(w.pos, (size_t)w.nEntries);
}

template <WalkKind Kind>
void writeEntries(Ctx& c, const Mesh& m, const SweepPlan& p, const Walk& w, int* stepOf = nullptr)
{
    if (p.lds)
        entriesK<Kind, true><<<waveBlocks(w.nSteps), kTpb, 0, c.stream>>>(p.n, w, viewOf(m), p.place, stepOf);
    else
        entriesK<Kind, false><<<waveBlocks(w.nSteps), kTpb, 0, c.stream>>>(p.n, w, viewOf(m), p.place, stepOf);
    hipCheck(hipGetLastError(), "sweep plan");
}

// whether the plan's arrays fit the device; without room the mesh keeps a launch per level
template <typename Build>
bool fits(Build build)
{
    try
    {
        return build();
    }
    catch (const Error& e)
    {
        if (e.code != kErrAlloc) throw;
        (void)hipGetLastError();
        return false;
    }
}

bool planBuild(Ctx& c, Mesh& m, SweepPlan* p)
{
    const LevelSched& S = *m.sched;
    const int n = m.nCells;
    p->n = n;
    p->lds = n <= kLdsCells;
    int widest = 1;
    for (const std::vector<int>* st : {&S.fwdStart, &S.bwdStart})
        for (size_t l = 0; l + 1 < st->size(); ++l) widest = std::max(widest, (*st)[l + 1] - (*st)[l]);
    p->threads = p->lds ? std::min(kLdsThreads, (widest + 63) / 64 * 64) : 64;
    std::vector<int4> steps;
    cutSteps(S.fwdStart, p->threads, steps);
    const size_t nF = steps.size();
    cutSteps(S.bwdStart, p->threads, steps);
    p->steps.upload(steps, c.stream);
    stepWidthK<<<waveBlocks((int)steps.size()), kTpb, 0, c.stream>>>((int)steps.size(), (int)nF, viewOf(m), kLowerFaces,
                                                                      S.fwdCells.p, kOwnedFaces, S.bwdCells.p, p->steps.p);
    hipCheck(hipGetLastError(), "sweep plan");
    steps = p->steps.download(c.stream);
    const int narrow = p->lds ? kLdsNarrow : kFlowNarrow;
    p->wide = widestCell(steps) > narrow;
    const int least = p->wide ? kWide : narrow;
    if (!placeEntries(steps, 0, nF, p->lds, least, entryRoom(m), p->fwd) ||
        !placeEntries(steps, nF, steps.size(), p->lds, least, entryRoom(m), p->bwd))
        return false;
    p->steps.upload(steps, c.stream);
    p->fwd.steps = p->steps.p;
    p->bwd.steps = p->steps.p + nF;
    p->fwd.cell = S.fwdCells.p;
    p->bwd.cell = S.bwdCells.p;
    carve(p->mem, [&](Carve& at) {
        at(p->place, (size_t)n);
        carveWalk(at, p->fwd, n, p->lds);
        carveWalk(at, p->bwd, n, p->lds);
        if (p->lds)
        {
            at(p->aFwd, (size_t)p->fwd.nEntries);
            at(p->aBwd, (size_t)p->bwd.nEntries);
            at(p->dFwd, (size_t)n);
        }
        else
            at(p->hand, 2 * (size_t)n);
    });
    placeK<<<blocks(n), kTpb, 0, c.stream>>>(n, S.fwdCells.p, p->place);
    writeEntries<kLowerFaces>(c, m, *p, p->fwd);
    writeEntries<kOwnedFaces>(c, m, *p, p->bwd);
    if (p->lds) return true;
    zeroWordsK<<<blocks(2 * n), kTpb, 0, c.stream>>>(2 * (size_t)n, p->hand);
    hipCheck(hipGetLastError(), "sweep plan");
    p->state.upload(firstHandState(), c.stream);
    return true;
}

// the mesh's plan, or null: a mesh without faces, above kFlowMaxCells or of few levels, or a plan that would not fit
SweepPlan* planOf(const Mesh& m) { return m.sweep && m.sweep->usable ? m.sweep.get() : nullptr; }

// the forward walk of Gauss-Seidel (both runs of a cell's faces), on the first such sweep outside a capture
bool planGs(Ctx& c, Mesh& m, SweepPlan& p)
{
    if (p.gsReady) return p.gsUsable;
    if (capturing(c.stream)) return false;
    const LevelSched& S = *m.sched;
    p.gsReady = true;
    p.gsUsable = fits([&] {
        std::vector<int4> steps;
        cutSteps(S.fwdStart, p.threads, steps);
        p.gsSteps.upload(steps, c.stream);
        const int nS = (int)steps.size();
        stepWidthK<<<waveBlocks(nS), kTpb, 0, c.stream>>>(nS, nS, viewOf(m), kAllFaces, S.fwdCells.p, kAllFaces, S.fwdCells.p,
                                                          p.gsSteps.p);
        hipCheck(hipGetLastError(), "sweep plan");
        steps = p.gsSteps.download(c.stream);
        const int most = widestCell(steps);
        p.gsAhead = most <= kGsNarrow ? kGsNarrow : most <= kGsMiddle ? kGsMiddle : kGsWide;
        if (!placeEntries(steps, 0, steps.size(), p.lds, p.gsAhead, entryRoom(m), p.gs)) return false;
        p.gsSteps.upload(steps, c.stream);
        p.gs.steps = p.gsSteps.p;
        p.gs.cell = S.fwdCells.p;
        int *stepOf = nullptr, *reach = nullptr;
        carve(p.gsMem, [&](Carve& at) {
            carveWalk(at, p.gs, p.n, p.lds);
            if (!p.lds) return;
            at(p.aGs, (size_t)p.gs.nEntries);
            at(p.aGsBack, (size_t)p.bwd.nEntries);
            at(p.gsIn, 4 * (size_t)p.n);
            at(stepOf, (size_t)p.n);
            at(reach, 2);
        });
        writeEntries<kAllFaces>(c, m, p, p.gs, stepOf);
        if (!p.lds) return true;
        int r = 0;
        zeroWordsK<<<1, kTpb, 0, c.stream>>>(1, reinterpret_cast<Word*>(reach));
        stepReachK<<<blocks(m.nFaces), kTpb, 0, c.stream>>>(m.nFaces, m.owner.p, m.neighbour.p, stepOf, reach);
        hipCheck(hipGetLastError(), "sweep plan");
        hipCheck(hipMemcpyAsync(&r, reach, sizeof(int), hipMemcpyDeviceToHost, c.stream), "sweep plan");
        hipCheck(hipStreamSynchronize(c.stream), "sweep plan");
        p.gsLag = r + 1;
        return true;
    });
    if (!p.gsUsable) p.gsMem.release();
    return p.gsUsable;
}

PlanView flowView(const SweepPlan& p)
{
    return PlanView{p.fwd.nSteps, p.bwd.nSteps, {p.fwd.steps, p.bwd.steps}, {p.fwd.cell, p.bwd.cell},
                    {p.fwd.self, p.bwd.self}, {p.fwd.face, p.bwd.face}, {p.fwd.pos, p.bwd.pos}};
}

LdsWalk ldsView(const Walk& w, const double* a)
{
    return LdsWalk{w.nSteps, 0, w.steps, w.cell, w.self, w.at, a};
}

// Dynamic LDS beyond the default is opted into per kernel; a refusal leaves the launch-per-level path. The
// call is cheap and allowed while a stream is captured.
template <typename K>
bool ldsAllowed(K* kernel, size_t bytes)
{
    if (bytes <= 65536) return true;
    if (hipFuncSetAttribute(reinterpret_cast<const void*>(kernel), hipFuncAttributeMaxDynamicSharedMemorySize,
                            (int)bytes) == hipSuccess)
        return true;
    (void)hipGetLastError();
    return false;
}

size_t ldsBytes(const SweepPlan& p) { return sizeof(double) * ((size_t)p.n + 1); }

// waves of a flow launch, the window of chunks in work: more only poll (64^3: 256 waves 3.87 ms a solve, 1024
// 4.21, 2048 5.22; 200^3: 34.4, 35.1, 36.6)
constexpr int kFlowWaves = 256;

template <int W>
bool factorLds(Ctx& c, SweepPlan& p, const double* diag, const double* upper, const double* lower, double* rD)
{
    const size_t bytes = ldsBytes(p);
    p.packed = 0;
    if (!ldsAllowed(&ldsFactorK<W>, bytes) || !ldsAllowed(&ldsSubstK<W>, bytes)) return false;
    p.packed = p.factors;
    const int nF = p.fwd.nEntries, nB = p.bwd.nEntries;
    packFactorK<<<blocks(std::max(nF, p.n)), kTpb, 0, c.stream>>>(nF, p.fwd.face, p.n, p.fwd.cell, diag, upper, lower,
                                                                 p.aFwd, p.dFwd);
    ldsFactorK<W><<<1, p.threads, bytes, c.stream>>>(p.n, ldsView(p.fwd, p.aFwd), p.dFwd, rD);
    packSubstK<<<blocks(std::max(nF, nB)), kTpb, 0, c.stream>>>(nF, p.fwd.face, p.fwd.entryCell, nB, p.bwd.face,
                                                               p.bwd.entryCell, rD, upper, lower, p.aFwd, p.aBwd);
    return true;
}

template <int W>
void substLds(Ctx& c, SweepPlan& p, const double* r, double* y, const int* stop)
{
    ldsSubstK<W><<<1, p.threads, ldsBytes(p), c.stream>>>(p.n, ldsView(p.fwd, p.aFwd), ldsView(p.bwd, p.aBwd), p.dFwd,
                                                         r, y, stop);
}

template <int W, bool Factor>
void substFlow(Ctx& c, SweepPlan& p, const double* diag, const double* upper, const double* lower, const double* rD,
               const double* r, double* out, const int* stop)
{
    const int steps = p.fwd.nSteps + (Factor ? 0 : p.bwd.nSteps);
    flowSubstK<W, Factor><<<std::min(steps, kFlowWaves), 64, 0, c.stream>>>(flowView(p), diag, upper, lower, rD, r, out,
                                                                           p.hand, p.state.p, stop);
}

template <int W, int WB>
bool gsLds(Ctx& c, SweepPlan& p, const double* diag, const double* upper, const double* b, double* psi, int nSweeps,
           bool sym)
{
    const size_t bytes = ldsBytes(p);
    if (!(sym ? ldsAllowed(&ldsGsK<W, WB, true>, bytes) : ldsAllowed(&ldsGsK<W, WB, false>, bytes))) return false;
    const int nF = p.gs.nEntries, nB = sym ? p.bwd.nEntries : 0;
    packGsK<<<blocks(std::max(std::max(nF, nB), p.n)), kTpb, 0, c.stream>>>(
        nF, p.gs.face, nB, p.bwd.face, p.n, p.gs.cell, diag, upper, b, psi, p.aGs, p.aGsBack, p.gsIn);
    const LdsWalk F = ldsView(p.gs, p.aGs), B = ldsView(p.bwd, p.aGsBack);
    // as many teams as the workgroup's room holds, where they gain anything
    const int teams = sym || p.gsLag >= p.gs.nSteps ? 1 : std::max(1, std::min(nSweeps, kLdsThreads / p.threads));
    if (sym)
        ldsGsK<W, WB, true><<<1, p.threads, bytes, c.stream>>>(p.n, F, B, p.gsIn, psi, nSweeps, p.threads, p.gsLag);
    else
        ldsGsK<W, WB, false><<<1, teams * p.threads, bytes, c.stream>>>(p.n, F, B, p.gsIn, psi, nSweeps, p.threads,
                                                                        p.gsLag);
    return true;
}

template <int W, bool Back>
void gsFlow(Ctx& c, SweepPlan& p, const Walk& w, const double* diag, const double* upper, const double* b, double* psi,
            double* bPrime)
{
    flowGsK<W, Back><<<std::min(w.nSteps, kFlowWaves), 64, 0, c.stream>>>(w.nSteps, w.steps, w.cell, w.self, w.face, w.pos,
                                                                        diag, upper, b, psi, bPrime, p.hand,
                                                                        p.state.p);
}

} // namespace

void sweepPlan(Ctx& c, Mesh& m)
{
    m.sweep.reset(new SweepPlan());
    const size_t levels = std::max(m.sched->fwdStart.size(), m.sched->bwdStart.size()) - 1;
    if (!m.nFaces || m.nCells > kFlowMaxCells || (int)levels <= fewLevels(m.nCells, m.nCells <= kLdsCells)) return;
    if (fits([&] { return planBuild(c, m, m.sweep.get()); }))
        m.sweep->usable = true;
    else
        m.sweep.reset(new SweepPlan());
}

SweepFactor sweepFactor(Ctx& c, Mesh& m, const double* diag, const double* upper, const double* lower, double* rD)
{
    SweepPlan* p = planOf(m);
    if (!p) return 0;
    if (++p->factors == 0) ++p->factors;
    bool done = true;
    if (p->lds)
        done = p->wide ? factorLds<kWide>(c, *p, diag, upper, lower, rD) : factorLds<kLdsNarrow>(c, *p, diag, upper, lower, rD);
    else if (p->wide)
        substFlow<kWide, true>(c, *p, diag, upper, lower, nullptr, nullptr, rD, nullptr);
    else
        substFlow<kFlowNarrow, true>(c, *p, diag, upper, lower, nullptr, nullptr, rD, nullptr);
    hipCheck(hipGetLastError(), "sweep factor");
    return done ? p->factors : 0;
}

bool sweepSubstitute(Ctx& c, Mesh& m, SweepFactor factor, const double* rD, const double* upper, const double* lower,
                     const double* r, double* y, const int* stop)
{
    SweepPlan* p = planOf(m);
    if (!p || (p->lds && (factor == 0 || factor != p->packed))) return false;
    if (p->lds)
    {
        if (p->wide)
            substLds<kWide>(c, *p, r, y, stop);
        else
            substLds<kLdsNarrow>(c, *p, r, y, stop);
    }
    else if (p->wide)
        substFlow<kWide, false>(c, *p, nullptr, upper, lower, rD, r, y, stop);
    else
        substFlow<kFlowNarrow, false>(c, *p, nullptr, upper, lower, rD, r, y, stop);
    hipCheck(hipGetLastError(), "sweep substitution");
    return true;
}

bool sweepGaussSeidel(Ctx& c, Mesh& m, const double* diag, const double* upper, const double* b, double* psi,
                      int nSweeps, double* bPrime)
{
    SweepPlan* p = planOf(m);
    if (!p || nSweeps <= 0 || !planGs(c, m, *p)) return false;
    bool done = true;
    if (p->lds)
    {
        const bool sym = bPrime != nullptr;
        if (p->gsAhead == kGsNarrow)
            done = p->wide ? gsLds<kGsNarrow, kWide>(c, *p, diag, upper, b, psi, nSweeps, sym)
                           : gsLds<kGsNarrow, kLdsNarrow>(c, *p, diag, upper, b, psi, nSweeps, sym);
        else if (p->gsAhead == kGsMiddle)
            done = p->wide ? gsLds<kGsMiddle, kWide>(c, *p, diag, upper, b, psi, nSweeps, sym)
                           : gsLds<kGsMiddle, kLdsNarrow>(c, *p, diag, upper, b, psi, nSweeps, sym);
        else
            done = p->wide ? gsLds<kGsWide, kWide>(c, *p, diag, upper, b, psi, nSweeps, sym)
                           : gsLds<kGsWide, kLdsNarrow>(c, *p, diag, upper, b, psi, nSweeps, sym);
    }
    else
        for (int sw = 0; sw < nSweeps; ++sw)
        {
            if (p->gsAhead == kGsNarrow)
                gsFlow<kGsNarrow, false>(c, *p, p->gs, diag, upper, b, psi, bPrime);
            else if (p->gsAhead == kGsMiddle)
                gsFlow<kGsMiddle, false>(c, *p, p->gs, diag, upper, b, psi, bPrime);
            else
                gsFlow<kGsWide, false>(c, *p, p->gs, diag, upper, b, psi, bPrime);
            if (!bPrime) continue;
            if (p->wide)
                gsFlow<kWide, true>(c, *p, p->bwd, diag, upper, b, psi, bPrime);
            else
                gsFlow<kFlowNarrow, true>(c, *p, p->bwd, diag, upper, b, psi, bPrime);
        }
    hipCheck(hipGetLastError(), "gauss-seidel sweep");
    return done;
}

} // namespace mfv
