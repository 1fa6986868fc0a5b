// The small grids' part of a V-cycle in one launch.
//
// A grid of a few thousand rows is all latency: a kernel per step costs 4-6 us of dependent loads and gaps
// whatever its size, and one workgroup for all such grids has too few waves (at 2,400 rows a residual takes it
// 13 us, a post-sweep 22). Here workgroups take the cycle's steps in chunks of 64 rows (a slice) in order -- every grid's sweeps, residual and restriction down, the coarsest solve, prolongation and sweeps up --
// and hand each row's value on as tagged words (handover.hpp), so a step follows the one before by the time a
// value takes between two CUs, about half a microsecond, and steps overlap: addresses, columns and coefficients
// of later chunks are loaded while earlier ones are awaited. Each row's arithmetic is the per-grid kernels', in
// their order, with the vectors' stored precision, so the unscaled cycle's result is the same bits; the scaled
// correction's two sums are taken per chunk and then over the chunks in a fixed order.
#include "cycle_flow.hpp"

#include "handover.hpp"
#include "reduce.hpp"

#include <algorithm>

namespace mfv {

// One grid as the launch reads it. Words: one array per value a row hands on. x: the iterate on the way down
// (two, the sweeps alternate), y: on the way up; f: the finished value as the finer grid prolongs it.
struct FlowGrid
{
    int n;
    const int* slicePtr;
    const int* cols;      // per entry: its column,
    const int* colsC;     // and that column's coarse cell
    const void* val;
    const void* diag;
    const double* scale;
    const float* xm;      // solution-vector multiplier (FP16 cycle), else null
    const int* map;       // row -> coarse cell
    const int* start;     // coarse cell <- its rows
    const int* list;
    Word *b, *x[2], *r, *y[2], *f, *ae, *sums;
};

namespace {

constexpr int kMaxFlowGrids = 32;
// First grid of at most this many rows (and from it every coarser one) runs here. Above, a kernel per step fills the
// chip and its loads overlap by themselves: grids of 11,520 rows in this launch 3.40 ms a solve against 3.33 with
// their own kernels, of 9,025 to 15,625 4.77 against 4.41. Below, the launches are the cost: 4,096 as the line 6.5
// ms against 6.2 (4,847 rows, FP64), 13.0 against 12.8 (7,793, FP16).
constexpr int kFlowRows = 1 << 13;
// 64, 128 and 256 workgroups: 66, 55 and 48 us at 7,793 rows, but 105, 94 and 96 at 4,584 with the scaled correction
// and 6.2 against 6.3 ms for the solve over 45 k cells with 128 and 256 (as first built; 128 now take 46 and 78)
constexpr int kFlowGroups = 128;
constexpr int kStagedCoarsest = 64;   // the coarsest inverse's rows go through LDS up to this size

// a vector entry as its stored form reads back (FP16: rounded under the multiplier m, saturated)
template <typename Tv, typename Ts>
__device__ __forceinline__ Tv stored(Tv v, Tv, Tv) { return v; }
template <>
__device__ __forceinline__ float stored<float, __half>(float v, float m, float im)
{
    return __half2float(__float2half(fminf(fmaxf(v * m, -65504.0f), 65504.0f))) * im;
}

// Holds a wave until value i is there: one lane asks, now and then. Waves wait here for steps far ahead of the
// one in work; if every lane of them asked for all of its values all the time, the words in work would queue
// behind that (a step of a few hundred rows then took 5-10 us).
template <typename Tv>
__device__ __forceinline__ void gate(const Word* p, int i, unsigned tag)
{
    bool there;
    do
    {
        there = true;
        if ((threadIdx.x & 63) == 0) there = Hand<Tv>::get(p, i).is(tag);
        there = __all(there);
        if (!there) __builtin_amdgcn_s_sleep(4);
    } while (!there);
}

// values of up to B entries, asked for together, then those that are missing until none is; nk is uniform
template <typename Tv, int B>
__device__ __forceinline__ void awaitEntries(const Word* p, const int (&i)[B], int nk, unsigned tag, Tv (&v)[B])
{
    typename Hand<Tv>::Raw r[B];
    unsigned missing = 0;
#pragma unroll
    for (int k = 0; k < B; ++k)
        if (k < nk) r[k] = Hand<Tv>::get(p, i[k]);
#pragma unroll
    for (int k = 0; k < B; ++k)
        if (k < nk)
        {
            v[k] = r[k].value();
            missing |= (r[k].is(tag) ? 0u : 1u) << k;
        }
    while (missing)
    {
#pragma unroll
        for (int k = 0; k < B; ++k)
            if (missing >> k & 1u) r[k] = Hand<Tv>::get(p, i[k]);
#pragma unroll
        for (int k = 0; k < B; ++k)
            if ((missing >> k & 1u) && r[k].is(tag))
            {
                v[k] = r[k].value();
                missing &= ~(1u << k);
            }
    }
}

// two sets of values at once
template <typename Tv, int B>
__device__ __forceinline__ void awaitEntries2(const Word* p, const int (&i)[B], unsigned pTag, Tv (&v)[B], const Word* q,
                                              const int (&j)[B], unsigned qTag, Tv (&u)[B], int nk)
{
    typename Hand<Tv>::Raw r[B], t[B];
#pragma unroll
    for (int k = 0; k < B; ++k)
        if (k < nk)
        {
            r[k] = Hand<Tv>::get(p, i[k]);
            t[k] = Hand<Tv>::get(q, j[k]);
        }
#pragma unroll
    for (int k = 0; k < B; ++k)
        if (k < nk)
        {
            while (!r[k].is(pTag)) r[k] = Hand<Tv>::get(p, i[k]);
            v[k] = r[k].value();
        }
    unsigned missing = 0;
#pragma unroll
    for (int k = 0; k < B; ++k)
        if (k < nk)
        {
            u[k] = t[k].value();
            missing |= (t[k].is(qTag) ? 0u : 1u) << k;
        }
    while (missing)
    {
#pragma unroll
        for (int k = 0; k < B; ++k)
            if (missing >> k & 1u) t[k] = Hand<Tv>::get(q, j[k]);
#pragma unroll
        for (int k = 0; k < B; ++k)
            if ((missing >> k & 1u) && t[k].is(qTag))
            {
                u[k] = t[k].value();
                missing &= ~(1u << k);
            }
    }
}

// The step sequence. Per grid on the way down: the pre-sweeps after the first, the residual, the restriction
// (chunks of the next grid); then the coarsest solve; per grid on the way up: the prolongation with the first
// post-sweep (scaled: A e with its sums, then the update), and the further post-sweeps.
enum StepKind : int { kSweepDown, kResidual, kRestrict, kCoarsest, kProlong, kScaleSums, kScaleUpdate, kSweepUp };

struct Steps
{
    int T, nDown, nUp, nExtra, scaled;   // steps per grid on the two ways; extra post-sweeps
    __device__ __forceinline__ int count() const { return 1 + (T - 1) * (nDown + nUp); }
    // step s: what, on which grid, which sweep; rowsOf: the grid whose rows it runs over
    __device__ __forceinline__ void at(int s, int& kind, int& g, int& sweep, int& rowsOf) const
    {
        sweep = 0;
        if (s < (T - 1) * nDown)
        {
            g = s / nDown;
            const int q = s - g * nDown;
            rowsOf = g;
            kind = q < nDown - 2 ? kSweepDown : q == nDown - 2 ? kResidual : kRestrict;
            if (kind == kSweepDown) sweep = q + 1;
            if (kind == kRestrict) rowsOf = g + 1;
            return;
        }
        s -= (T - 1) * nDown;
        if (s == 0)
        {
            kind = kCoarsest;
            g = rowsOf = T - 1;
            return;
        }
        s -= 1;
        const int h = s / nUp, q = s - h * nUp, first = nUp - nExtra;
        g = rowsOf = T - 2 - h;
        kind = q >= first ? kSweepUp : !scaled ? kProlong : q == 0 ? kScaleSums : kScaleUpdate;
        if (kind == kSweepUp) sweep = q - first + 1;
    }
};

// A wave takes kRows rows at a time, four neighbouring lanes (a quad) to a row: the values of a row's entries are
// scattered words, and a wave asks for one word per lane and instruction, so a row a lane made each step wait for
// tens of such instructions. Lane `sub` of the quad asks for entries sub, sub + 4, ...; the products are then
// added in entry order, every lane reading them from its quad in turn, so all four hold the sum.
constexpr int kLanes = 4, kRows = 64 / kLanes;
constexpr int kThreads = 256;   // a chunk is a slice of 64 rows, a quarter to each of the workgroup's waves
constexpr int kAhead = 6;   // a lane's entries per batch: a batch covers rows of 24 entries

// lane U's value in every lane of its quad
template <int U>
__device__ __forceinline__ float quad(float v)
{
    return __int_as_float(__builtin_amdgcn_mov_dpp(__float_as_int(v), U * 0x55, 0xf, 0xf, true));
}
template <int U>
__device__ __forceinline__ double quad(double v)
{
    const long long b = __double_as_longlong(v);
    const int lo = __builtin_amdgcn_mov_dpp((int)b, U * 0x55, 0xf, 0xf, true);
    const int hi = __builtin_amdgcn_mov_dpp((int)(b >> 32), U * 0x55, 0xf, 0xf, true);
    return __longlong_as_double((long long)(((unsigned long long)(unsigned)hi << 32) | (unsigned)lo));
}
// s plus the first n (0..4) of the quad's values, in lane order; n is uniform or the same in the quad
template <typename T>
__device__ __forceinline__ T addQuad(T s, T v, int n)
{
    s = n > 0 ? s + quad<0>(v) : s;
    s = n > 1 ? s + quad<1>(v) : s;
    s = n > 2 ? s + quad<2>(v) : s;
    return n > 3 ? s + quad<3>(v) : s;
}

// What a row needs that the launch does not compute: its diagonal and its entries' columns (Cols), those
// columns' coarse cells (Coarse) and coefficients. The first batch is loaded before the wave waits for
// values, so that only the values are on the chain from step to step.
template <bool Cols, bool Coarse, typename Tv>
struct RowAhead
{
    int p0, w, nk;
    int cx[kAhead], ce[kAhead];
    Tv a[kAhead], dc;
    // entries k0 + sub, k0 + sub + kLanes, ...; lanes past the row's width read its last entry
    template <typename Tm>
    __device__ __forceinline__ void load(const FlowGrid& G, int c, int k0)
    {
        const Tm* val = static_cast<const Tm*>(G.val);
        nk = (min(kAhead * kLanes, w - k0) + kLanes - 1) / kLanes;
#pragma unroll
        for (int j = 0; j < kAhead; ++j)
            if (j < nk)
            {
                const int at = p0 + (min(k0 + j * kLanes + (int)(threadIdx.x & (kLanes - 1)), w - 1) << 6) + (c & 63);
                if (Cols) cx[j] = G.cols[at];
                if (Coarse) ce[j] = G.colsC[at];
                a[j] = cvt<Tv>(val[at]);
            }
    }
    template <typename Tm>
    __device__ __forceinline__ void first(const FlowGrid& G, int c)
    {
        const int slice = __builtin_amdgcn_readfirstlane(c >> 6);
        p0 = G.slicePtr[slice];
        w = (G.slicePtr[slice + 1] - p0) >> 6;
        dc = static_cast<const Tv*>(G.diag)[c];
        load<Tm>(G, c, 0);
    }
};

// A v at a row, v = x (X), x + e (X and E) or e (E), in rowAx's arithmetic. xPlain: x read from the launch's
// input array instead of words. em, eim: the multiplier e is stored under on this grid.
template <bool X, bool E, typename Tm, typename Tv, typename Ts>
__device__ __forceinline__ Tv flowRow(const FlowGrid& G, RowAhead<X, E, Tv>& R, int c, const Ts* xPlain, const Word* x,
                                      unsigned xTag, const Word* e, unsigned eTag, Tv em, Tv eim, Tv vc)
{
    Tv acc = sizeof(Tm) == 2 ? Tv(0) : R.dc * vc;
    for (int k0 = 0; k0 < R.w; k0 += kAhead * kLanes)
    {
        if (k0) R.template load<Tm>(G, c, k0);
        Tv vx[kAhead], ve[kAhead];
        if (X && xPlain)
        {
            const CycVec<Tv, Ts> P(xPlain, em, eim);
#pragma unroll
            for (int j = 0; j < kAhead; ++j)
                if (j < R.nk) vx[j] = P(R.cx[j]);
        }
        if (X && !xPlain && E)
            awaitEntries2<Tv, kAhead>(x, R.cx, xTag, vx, e, R.ce, eTag, ve, R.nk);
        else if (X && !xPlain)
            awaitEntries<Tv, kAhead>(x, R.cx, R.nk, xTag, vx);
        else if (E)
            awaitEntries<Tv, kAhead>(e, R.ce, R.nk, eTag, ve);
#pragma unroll
        for (int j = 0; j < kAhead; ++j)
            if (j < R.nk)
            {
                const Tv ek = E ? stored<Tv, Ts>(ve[j], em, eim) : Tv(0);
                acc = addQuad(acc, R.a[j] * (X && E ? vx[j] + ek : X ? vx[j] : ek), R.w - k0 - j * kLanes);
            }
    }
    if constexpr (sizeof(Tm) == 2) return R.dc * vc + (Tv)(*G.scale) * acc;
    return acc;
}

// a row's own values, asked for one after the other without waiting in between
template <typename Tv>
struct Own
{
    const Word* p;
    int i;
    unsigned tag;
    typename Hand<Tv>::Raw r;
    Tv known;
    __device__ __forceinline__ void have(Tv v)
    {
        p = nullptr;
        known = v;
    }
    __device__ __forceinline__ void ask(const Word* q, int at, unsigned t)
    {
        p = q;
        i = at;
        tag = t;
        r = Hand<Tv>::get(p, i);
    }
    __device__ __forceinline__ Tv value()
    {
        if (!p) return known;
        while (!r.is(tag)) r = Hand<Tv>::get(p, i);
        return r.value();
    }
};

template <typename Tm, typename Tv, typename Ts>
__global__ __launch_bounds__(kThreads) void flowCycleK(const FlowGrid* __restrict__ grids, Steps st,
                                                 const double* __restrict__ inv, int nPre, int nPost,
                                                 const Ts* __restrict__ b0, const Ts* __restrict__ x0, Ts* __restrict__ out,
                                                 Scatter<Tv, Ts> up, unsigned* state,
                                                 const int* __restrict__ stop)
{
    if (stop && *stop) return;
    __shared__ double sb[kMaxDenseCoarsest];
    __shared__ double sInv[64 * (kStagedCoarsest + 1)];
    __shared__ int slots[2];
    __shared__ int chunksOf[kMaxFlowGrids];
    __shared__ double sums[2 * (kThreads / 64)];
    const int lane = threadIdx.x & 63, quarter = (int)__builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const unsigned tag = launchTag(state);
    GroupChunks order(state, slots);
    if ((int)threadIdx.x < st.T) chunksOf[threadIdx.x] = (grids[threadIdx.x].n + 63) >> 6;
    __syncthreads();
    const int nSteps = st.count(), xs = max(nPre - 1, 0);
    int step = 0, first = 0, kind, g, sweep, rowsOf;
    st.at(0, kind, g, sweep, rowsOf);
    int chunks = __builtin_amdgcn_readfirstlane(chunksOf[rowsOf]);
    const Tv omega = Tv(kOmega);
    for (;;)
    {
        const int t = order.next();
        while (step < nSteps && t >= first + chunks)
        {
            first += chunks;
            if (++step < nSteps)
            {
                st.at(step, kind, g, sweep, rowsOf);
                chunks = __builtin_amdgcn_readfirstlane(chunksOf[rowsOf]);
            }
        }
        if (step >= nSteps) break;
        const int part = 4 * (t - first) + quarter, c0 = part * kRows, c = c0 + lane / kLanes;
        const bool lead = lane % kLanes == 0;   // the lane that writes its row's value
        const FlowGrid& G = grids[g];
        const Tv m = G.xm ? (Tv)*G.xm : Tv(1), im = G.xm ? (Tv)(1.0f / *G.xm) : Tv(1);
        Tv done = Tv(0);         // a finished value, handed on below
        bool finished = false;
        auto finish = [&](Tv v) {
            done = v;
            finished = true;
        };
        // before a step on the way up: what the next grid's last step waited for
        auto gateUp = [&](int mc) {
            const FlowGrid& C = grids[g + 1];
            if (g + 2 == st.T)
                gate<Tv>(C.b, mc, tag);
            else if (st.scaled)
                gate<Tv>(C.ae, mc, tag);
            else
                gate<Tv>(grids[g + 2].f, C.map[mc], tag);
        };
        // grid 0's right-hand side and entry iterate are the launch's inputs
        const CycVec<Tv, Ts> B0(b0, nullptr), X0(x0, m, im);
        auto askB = [&](Own<Tv>& o) {
            if (g == 0)
                o.have(B0(c));
            else
                o.ask(G.b, c, tag);
        };
        auto askX = [&](Own<Tv>& o, const Word* in, int v) {
            if (g == 0 && v == 0)
                o.have(X0(c));
            else
                o.ask(in, c, tag + v);
        };
        if (kind == kSweepDown || kind == kSweepUp || kind == kResidual)
        {
            if (c < G.n)
            {
                const bool up_ = kind == kSweepUp;
                const int v = kind == kResidual ? xs : sweep - 1;   // the version of the iterate read
                const bool plain = g == 0 && v == 0 && !up_;
                const Word* in = up_ ? G.y[v & 1] : G.x[v & 1];
                RowAhead<true, false, Tv> R;
                R.template first<Tm>(G, c);
                // the step before the one that makes these values
                if (v > 0 || up_)
                    gate<Tv>(in, c0, tag + v);
                else if (g > 0)
                    gate<Tv>(grids[g - 1].r, grids[g - 1].list[grids[g - 1].start[c0]], tag);
                Own<Tv> ob, ox;
                askB(ob);
                if (plain)
                    ox.have(X0(c));
                else
                    ox.ask(in, c, tag + v);
                const Tv bc = ob.value(), xc = ox.value();
                const Tv ax = flowRow<true, false, Tm, Tv, Ts>(G, R, c, plain ? x0 : nullptr, in, tag + v, nullptr, 0u, m, im,
                                                               xc);
                if (kind == kResidual)
                {
                    if (lead) Hand<Tv>::put(G.r, c, tag, stored<Tv, Ts>(bc - ax, Tv(1), Tv(1)));
                }
                else
                {
                    const Tv xo = xc + omega * (bc - ax) / safeDiag(R.dc);
                    if (up_ && sweep == st.nExtra)
                        finish(xo);
                    else if (lead)
                        Hand<Tv>::put(up_ ? G.y[sweep & 1] : G.x[sweep & 1], c, tag + sweep, stored<Tv, Ts>(xo, m, im));
                }
            }
        }
        else if (kind == kRestrict)
        {
            // c is a cell of the next grid; its rows' residuals in ascending order, one to a lane
            const FlowGrid& C = grids[g + 1];
            if (c < C.n)
            {
                const bool last = g + 2 == st.T;
                const Tv dC = last ? Tv(1) : static_cast<const Tv*>(C.diag)[c];
                const int k0 = G.start[c], k1 = G.start[c + 1], sub = lane % kLanes;
                int i[1] = {G.list[min(k0 + sub, k1 - 1)]};
                if (g > 0) gate<Tv>(G.b, i[0], tag);
                Tv s = Tv(0);
                for (int k = k0; k < k1; k += kLanes)
                {
                    Tv v[1];
                    if (k > k0) i[0] = G.list[min(k + sub, k1 - 1)];
                    awaitEntries<Tv, 1>(G.r, i, 1, tag, v);
                    s = addQuad(s, v[0], k1 - k);
                }
                if (lead)
                {
                    Hand<Tv>::put(C.b, c, tag, stored<Tv, Ts>(s, Tv(1), Tv(1)));
                    if (!last)
                    {
                        const Tv mc = C.xm ? (Tv)*C.xm : Tv(1), imc = C.xm ? (Tv)(1.0f / *C.xm) : Tv(1);
                        const Tv x = nPre > 0 ? Tv(0) + omega * (s - Tv(0)) / safeDiag(dC) : Tv(0);
                        Hand<Tv>::put(C.x[0], c, tag, stored<Tv, Ts>(x, mc, imc));
                    }
                }
            }
        }
        else if (kind == kCoarsest)
        {
            // x = Ainv b in FP64, ascending column per row; a small inverse staged first
            const bool staged = G.n <= kStagedCoarsest;
            if (staged)
                for (int q = threadIdx.x; q < G.n * G.n; q += kThreads)
                    sInv[q / G.n * (kStagedCoarsest + 1) + q % G.n] = inv[q];
            gate<Tv>(grids[g - 1].r, 0, tag);
            for (int j = threadIdx.x; j < G.n; j += kThreads) sb[j] = (double)awaitValue<Tv>(G.b, j, tag);
            __syncthreads();
            if (lead && c < G.n)
            {
                double s = 0.0;
                if (staged)
                {
                    const double* row = sInv + c * (kStagedCoarsest + 1);
#pragma unroll 8
                    for (int j = 0; j < G.n; ++j) s += row[j] * sb[j];
                }
                else
                {
                    const double* row = inv + (size_t)c * G.n;
#pragma unroll 8
                    for (int j = 0; j < G.n; ++j) s += row[j] * sb[j];
                }
                Hand<Tv>::put(G.f, c, tag, (Tv)s);
            }
        }
        else if (kind == kProlong)
        {
            if (c < G.n)
            {
                const Word* in = G.x[xs & 1];
                const Word* e = grids[g + 1].f;
                const int mc = G.map[c];
                RowAhead<true, true, Tv> R;
                R.template first<Tm>(G, c);
                gateUp(mc);
                Own<Tv> ob, ox, oe;
                askB(ob);
                askX(ox, in, xs);
                oe.ask(e, mc, tag);
                const Tv bc = ob.value(), xc = ox.value();
                const Tv vc = xc + stored<Tv, Ts>(oe.value(), m, im);
                Tv xo = vc;
                if (nPost > 0)
                {
                    const Tv ax = flowRow<true, true, Tm, Tv, Ts>(G, R, c, g == 0 && xs == 0 ? x0 : nullptr, in,
                                                                  tag + xs, e, tag, m, im, vc);
                    xo = vc + omega * (bc - ax) / safeDiag(R.dc);
                }
                if (st.nExtra && lead)
                    Hand<Tv>::put(G.y[0], c, tag, stored<Tv, Ts>(xo, m, im));
                else if (!st.nExtra)
                    finish(xo);
            }
        }
        else if (kind == kScaleSums)
        {
            double num = 0.0, den = 0.0;
            if (c < G.n)
            {
                const Word* e = grids[g + 1].f;
                const int mc = G.map[c];
                RowAhead<false, true, Tv> R;
                R.template first<Tm>(G, c);
                gateUp(mc);
                Own<Tv> orr, oe;
                orr.ask(G.r, c, tag);
                oe.ask(e, mc, tag);
                const Tv rc = orr.value();
                const Tv ec = stored<Tv, Ts>(oe.value(), m, im);
                const Tv ae = flowRow<false, true, Tm, Tv, Ts>(G, R, c, nullptr, nullptr, 0u, e, tag, m, im, ec);
                if (lead)
                {
                    Hand<Tv>::put(G.ae, c, tag, stored<Tv, Ts>(ae, Tv(1), Tv(1)));
                    num = (double)ec * (double)rc;
                    den = (double)ec * (double)ae;
                }
            }
            // the chunk's sums, its waves' in order
            num = waveSum(num);
            den = waveSum(den);
            if (lane == 0)
            {
                sums[2 * quarter] = num;
                sums[2 * quarter + 1] = den;
            }
            __syncthreads();
            if (threadIdx.x < 2)
                Hand<double>::put(G.sums, 2 * (t - first) + (int)threadIdx.x, tag,
                                  ((sums[threadIdx.x] + sums[threadIdx.x + 2]) + sums[threadIdx.x + 4]) + sums[threadIdx.x + 6]);
        }
        else   // kScaleUpdate
        {
            const bool on = c < G.n;
            const int mc = on ? G.map[c] : 0;
            const Tv dc = on ? static_cast<const Tv*>(G.diag)[c] : Tv(1);
            gate<Tv>(grids[g + 1].f, mc, tag);
            Own<Tv> ox, orr, oa, oe;
            if (on)
            {
                askX(ox, G.x[xs & 1], xs);
                orr.ask(G.r, c, tag);
                oa.ask(G.ae, c, tag);
                oe.ask(grids[g + 1].f, mc, tag);
            }
            // the grid's sums over its chunks, taken by the workgroup: were every wave to ask for a pair of every wave's,
            // as many words would cross as the grid has rows, squared
            double num = 0.0, den = 0.0;
            for (int q = threadIdx.x; q < chunks; q += kThreads)
            {
                const int i[2] = {2 * q, 2 * q + 1};
                double v[2];
                awaitEntries<double, 2>(G.sums, i, 2, tag, v);
                num += v[0];
                den += v[1];
            }
            num = waveSum(num);
            den = waveSum(den);
            if (lane == 0)
            {
                sums[2 * quarter] = num;
                sums[2 * quarter + 1] = den;
            }
            __syncthreads();
            num = ((sums[0] + sums[2]) + sums[4]) + sums[6];
            den = ((sums[1] + sums[3]) + sums[5]) + sums[7];
            const Tv al = (Tv)(den > 1e-30 ? num / den : 1.0);
            if (on)
            {
                const Tv xc = ox.value(), rc = orr.value(), ae = oa.value(), ec = stored<Tv, Ts>(oe.value(), m, im);
                const Tv xo = nPost > 0 ? xc + al * ec + omega * (rc - al * ae) / safeDiag(dc) : xc + al * ec;
                if (st.nExtra && lead)
                    Hand<Tv>::put(G.y[0], c, tag, stored<Tv, Ts>(xo, m, im));
                else if (!st.nExtra)
                    finish(xo);
            }
        }
        // to the finer grid of this launch, or out of it (once for every kind of step: the kernel's size costs it)
        if (finished && lead)
        {
            if (g > 0)
                Hand<Tv>::put(G.f, c, tag, done);
            else
            {
                if (out)
                {
                    const CycVec<Tv, Ts> XO(out, G.xm);
                    XO.set(c, done);
                }
                up(c, done);
            }
        }
    }
    leave(order, (unsigned)first, tag, (unsigned)(nPre + nPost + 2));   // first: the chunks of every step
}

// a grid's columns (a patterned grid's written out) and their coarse cells, a row a thread
__global__ __launch_bounds__(kThreads) void columnsK(SellView S, const int* __restrict__ map, int* __restrict__ cols,
                                                     int* __restrict__ coarse)
{
    const int r = blockIdx.x * kThreads + threadIdx.x;
    if (r >= S.n) return;
    const int p0 = S.slicePtr[r >> 6], w = (S.slicePtr[(r >> 6) + 1] - p0) >> 6;
    for (int k = 0; k < w; ++k)
    {
        const int e = p0 + (k << 6) + (r & 63);
        const int col = S.pattern ? r + S.patOff[S.pattern[r] * S.width + k] : S.cols[e];
        cols[e] = col;
        coarse[e] = map[col];
    }
}

__global__ __launch_bounds__(kThreads) void zeroWordsK(size_t n, Word* __restrict__ w)
{
    const size_t i = (size_t)blockIdx.x * kThreads + threadIdx.x;
    if (i < n) w[i] = 0ull;
}

} // namespace

// The launch's arrays for a.prec: descriptors, columns (a patterned grid's written out) and their coarse cells,
// and the words. They are written on the device: by the host they made a new hierarchy's first FP64 set-up 1.6 ms at
// 45 k cells and 1.5 at 8,000; so it is 1.2 and 1.0 (before this launch and the staged inverse 1.2 and 1.3).
// a.flowStart: the first grid of at most kFlowRows rows, or -1 where none has a coarser one (or over kMaxFlowGrids do).
void flowCycleBuild(Ctx& c, Amg& a)
{
    const int nG = (int)a.grids.size();
    a.flowStart = -1;
    for (int g = 0; g + 1 < nG && a.flowStart < 0; ++g)
        if (a.grids[g].n <= kFlowRows) a.flowStart = g;
    if (a.flowStart < 0 || nG - a.flowStart > kMaxFlowGrids)
    {
        a.flowStart = -1;
        return;
    }
    const int T = nG - a.flowStart;
    const size_t per = a.prec == Prec::F64 ? 2 : 1;
    std::vector<size_t> entryAt(T + 1, 0), wordAt(T + 1, 0);
    for (int t = 0; t < T; ++t)
    {
        const Grid& G = a.grids[a.flowStart + t];
        entryAt[t + 1] = entryAt[t] + (t + 1 < T ? (size_t)G.sell.nnz : 0);
        wordAt[t + 1] = wordAt[t] + 8 * per * (size_t)G.n + 4 * (((size_t)G.n + 63) / 64);
    }
    // the columns depend on the structure alone
    if (a.flowCols.n != 2 * entryAt[T])
    {
        a.flowCols.resize(2 * entryAt[T]);
        for (int t = 0; t + 1 < T; ++t)
        {
            const Grid& G = a.grids[a.flowStart + t];
            columnsK<<<(G.n + kThreads - 1) / kThreads, kThreads, 0, c.stream>>>(
                viewOf(G.sell), G.map.p, a.flowCols.p + entryAt[t], a.flowCols.p + entryAt[T] + entryAt[t]);
        }
    }
    if (a.flowWords.n != wordAt[T] || !a.flowState.n)
    {
        a.flowWords.resize(wordAt[T]);
        zeroWordsK<<<(unsigned)((wordAt[T] + kThreads - 1) / kThreads), kThreads, 0, c.stream>>>(wordAt[T], a.flowWords.p);
        a.flowState.upload(firstHandState(), c.stream);
    }
    hipCheck(hipGetLastError(), "small grids' columns");
    std::vector<FlowGrid> d(T);
    for (int t = 0; t < T; ++t)
    {
        Grid& G = a.grids[a.flowStart + t];
        FlowGrid& q = d[t];
        q.n = G.n;
        q.slicePtr = G.sell.slicePtr.p;
        q.cols = a.flowCols.p + entryAt[t];
        q.colsC = a.flowCols.p + entryAt[T] + entryAt[t];
        q.val = a.prec == Prec::F64   ? (const void*)G.off64.p
                : a.prec == Prec::F32 ? (const void*)G.off32.p
                                      : (const void*)G.off16.p;
        q.diag = a.prec == Prec::F64 ? (const void*)G.diagV64.p : (const void*)G.diagV32.p;
        q.scale = a.scales.p + a.flowStart + t;
        q.xm = a.prec == Prec::F16 ? a.xmul.p + a.flowStart + t : nullptr;
        q.map = G.map.p;
        q.start = G.cellStart.p;
        q.list = G.cellList.p;
        Word* w = a.flowWords.p + wordAt[t];
        auto take = [&](size_t n) {
            Word* p = w;
            w += n;
            return p;
        };
        const size_t rows = per * (size_t)G.n;
        q.b = take(rows);
        q.x[0] = take(rows);
        q.x[1] = take(rows);
        q.r = take(rows);
        q.y[0] = take(rows);
        q.y[1] = take(rows);
        q.f = take(rows);
        q.ae = take(rows);
        q.sums = take(4 * (((size_t)G.n + 63) / 64));
    }
    a.flowDesc.upload(reinterpret_cast<const uint8_t*>(d.data()), d.size() * sizeof(FlowGrid), c.stream);
}

// A step here costs the time a value takes between two CUs, in one workgroup a barrier: on a few hundred rows the one
// workgroup's many sweeps are the faster. V(4,3) on 512, 1,600 (2-D) and 1,728 (3-D) cells, here and there, us: FP64
// 61 and 51, 87 and 73, 98 and 99; FP16 62 and 61, 90 and 75, 98 and 89. On 4,096 122 and 148, 119 and 120; V(2,1) on
// 1,600 and 1,728 46 and 45, 52 and 59. The one workgroup's coarsest solve has to be small: 962 cells take it 250.
bool flowCycleRuns(const Amg& a, const VcycleControls& vc)
{
    constexpr int kFewRows = 2048, kManySweeps = 5, kFewCoarsest = 128;
    if (a.flowStart < 0) return false;
    return vc.nPre + vc.nPost < kManySweeps || a.grids[a.flowStart].n > kFewRows || a.nCoarsest > kFewCoarsest;
}

template <typename Tm, typename Tv, typename Ts>
void flowCycle(Ctx& c, Amg& a, const VcycleControls& vc, const Ts* b, const Ts* x, Ts* out, const Scatter<Tv, Ts>& up,
               const int* stop)
{
    const int T = (int)a.grids.size() - a.flowStart;
    Steps st;
    st.T = T;
    st.scaled = vc.scale ? 1 : 0;
    st.nDown = std::max(vc.nPre - 1, 0) + 2;
    st.nExtra = (vc.scale || vc.nPost > 0) ? std::max(vc.nPost - 1, 0) : 0;
    st.nUp = (vc.scale ? 2 : 1) + st.nExtra;
    long long chunks = 0;
    for (int t = 0; t < T; ++t) chunks += (a.grids[a.flowStart + t].n + 63) / 64;
    const int groups = (int)std::min<long long>(kFlowGroups, 2 * chunks);
    flowCycleK<Tm, Tv, Ts><<<groups, kThreads, 0, c.stream>>>(reinterpret_cast<const FlowGrid*>(a.flowDesc.p), st, a.coarseInv.p,
                                                       vc.nPre, vc.nPost, b, x, out, up, a.flowState.p, stop);
    hipCheck(hipGetLastError(), "cycle of the small grids");
}

template void flowCycle<double, double, double>(Ctx&, Amg&, const VcycleControls&, const double*, const double*, double*,
                                                const Scatter<double, double>&, const int*);
template void flowCycle<float, float, float>(Ctx&, Amg&, const VcycleControls&, const float*, const float*, float*,
                                             const Scatter<float, float>&, const int*);
template void flowCycle<__half, float, __half>(Ctx&, Amg&, const VcycleControls&, const __half*, const __half*, __half*,
                                               const Scatter<float, __half>&, const int*);

} // namespace mfv
