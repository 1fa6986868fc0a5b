// The launches' chunk order (brae_amd/csrc/chunks.hpp) on a model of the device memory, for test_chunk_order.py.
//
// Workgroups run one call of next() at a time in a random order, as one thread each. Relaxed operations on different
// words may reach memory in any order, so the model lets every request that nobody waits for -- the one a workgroup
// still has under way when it leaves -- arrive only at the very end of the launch. Each launch must still hand out
// every chunk exactly once.
#include <cstdio>
#include <cstdlib>
#include <memory>
#include <random>
#include <vector>

#define __device__
#define __forceinline__ inline
#define __HIP_MEMORY_SCOPE_AGENT 0
struct Dim
{
    unsigned x;
};
static Dim threadIdx{0}, gridDim{0};
static void __syncthreads() {}
static unsigned __builtin_amdgcn_readfirstlane(unsigned v) { return v; }

static unsigned gMemory[8];
static int gUnanswered = 0;   // per workgroup: the requests that it leaves with
static unsigned gLate = 0;

static unsigned __hip_atomic_load(const unsigned* p, int, int) { return *p; }
static void __hip_atomic_store(unsigned* p, unsigned v, int, int) { *p = v; }
static unsigned __hip_atomic_fetch_add(unsigned* p, unsigned v, int, int);

#include "../../brae_amd/csrc/chunks.hpp"

using namespace mfv;

static unsigned __hip_atomic_fetch_add(unsigned* p, unsigned v, int, int)
{
    if (p == gMemory + kDone)   // a workgroup leaves: what it still has under way has not arrived
    {
        gMemory[kNext] -= (unsigned)gUnanswered;
        gLate += (unsigned)gUnanswered;
    }
    const unsigned old = *p;
    *p += v;
    return old;
}

static void fail(const char* what, long a, long b)
{
    std::printf("%s: %ld, %ld\n", what, a, b);
    std::exit(1);
}

template <typename Order, typename Make>
static void launch(std::mt19937& rng, int total, int groups, int unanswered, Make make)
{
    gridDim.x = (unsigned)groups;
    gUnanswered = unanswered;
    const unsigned tag = launchTag(gMemory);
    struct Group
    {
        std::unique_ptr<Order> order;
        std::vector<int> slots;
        bool gone = false;
    };
    std::vector<Group> g(groups);
    std::vector<int> taken(total, 0);
    int left = 0;
    while (left < groups)
    {
        Group& w = g[rng() % groups];
        if (w.gone) continue;
        if (!w.order)
        {
            w.slots.assign(2, 0);
            w.order.reset(make(w.slots.data()));
        }
        const int t = w.order->next();
        if (t < 0) fail("a chunk before the first", t, total);
        if (t < total)
        {
            ++taken[t];
            continue;
        }
        leave(*w.order, (unsigned)total, tag, 3);
        w.gone = true;
        ++left;
    }
    gMemory[kNext] += gLate;   // the launch's end
    gLate = 0;
    for (int t = 0; t < total; ++t)
        if (taken[t] != 1) fail("chunk, times taken", t, taken[t]);
    if (gMemory[kDone] != 0) fail("workgroups counted after the launch", gMemory[kDone], groups);
    if (gMemory[kTag] != tag + 3) fail("tag", gMemory[kTag], tag);
}

int main()
{
    std::mt19937 rng(1);
    for (unsigned start : {0u, 0xffffff00u})   // also where the counter goes round
    {
        gMemory[kNext] = gMemory[kBase] = start;
        gMemory[kDone] = 0;
        gMemory[kTag] = 1;
        for (int k = 0; k < 200; ++k)
        {
            const int total = 1 + (int)(rng() % 90), groups = 1 + (int)(rng() % 40);
            if (rng() % 2)
                launch<GroupChunks>(rng, total, groups, 1, [](int* lds) { return new GroupChunks(gMemory, lds); });
            else
                launch<WaveChunks>(rng, total, groups, 0, [](int*) { return new WaveChunks(gMemory); });
        }
    }
    std::puts("ok");
    return 0;
}
