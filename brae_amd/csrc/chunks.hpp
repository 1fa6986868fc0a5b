// The order in which the workgroups of a launch take its chunks of work (handover.hpp), and how the launch's state in
// device memory is left for the next launch.
//
// Chunks come from one counter that only ever grows: a launch's chunks are the values from the base that its
// predecessor left. Every workgroup asks until it is given a value past the last chunk, so the requests of a launch
// are as many as its chunks and a fixed number a workgroup, and the last workgroup to leave moves the base on by that
// number. No word is written that a request still under way could write as well, so nothing has to be ordered but
// each word with itself: a request whose answer nobody waits for may arrive at any time before the launch ends.
// (A counter put back to 0 would need every such request to have arrived: one that came after would take the first
// chunk from the next launch, whose waves would then wait for it forever.)
#pragma once

namespace mfv {

// the launch's state: the requests so far, the workgroups that have left, the tag of its values, the base
enum : int { kNext = 0, kDone = 1, kTag = 2, kBase = 3, kHandState = 4 };

__device__ __forceinline__ unsigned launchTag(const unsigned* state)
{
    return __hip_atomic_load(state + kTag, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

// The next chunk, for a workgroup of one wave.
struct WaveChunks
{
    static constexpr unsigned kPastEnd = 1;   // a workgroup's requests that are given no chunk
    unsigned* state;
    unsigned base;
    __device__ __forceinline__ explicit WaveChunks(unsigned* s)
        : state(s), base(__hip_atomic_load(s + kBase, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT))
    {
    }
    __device__ __forceinline__ int next()
    {
        unsigned t = 0;
        if (threadIdx.x == 0) t = __hip_atomic_fetch_add(state + kNext, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        return (int)((unsigned)__builtin_amdgcn_readfirstlane(t) - base);
    }
};

// A larger workgroup's chunks in order: next() is the one to work on (the same in every thread). The request for the
// chunk after it goes out first; the order's promise holds, since the workgroup finishes the one in hand before. (As
// compiled for gfx950 its answer is waited for at once -- the compiler combines a wave's atomics and reads the answer
// back behind the request -- so each chunk still pays the counter's round trip before its work.)
struct GroupChunks
{
    static constexpr unsigned kPastEnd = 2;   // the one that ends its work and the one sent before that
    unsigned* state;
    int* slots;      // two, in LDS
    unsigned base;
    unsigned ahead;  // thread 0: the chunk asked for
    int turn;
    __device__ __forceinline__ GroupChunks(unsigned* s, int* lds)
        : state(s), slots(lds), base(__hip_atomic_load(s + kBase, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT)), ahead(0),
          turn(0)
    {
        ask();
    }
    __device__ __forceinline__ void ask()
    {
        if (threadIdx.x == 0)
            ahead = __hip_atomic_fetch_add(state + kNext, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    }
    __device__ __forceinline__ int next()
    {
        if (threadIdx.x == 0) slots[turn] = (int)(ahead - base);
        __syncthreads();
        const int t = __builtin_amdgcn_readfirstlane(slots[turn]);
        turn ^= 1;
        ask();
        return t;
    }
};

// Every workgroup calls it once its next() was past the launch's `total` chunks. The last one moves the base past the
// launch's requests and the tag past the `by` tags that it used.
template <typename Order>
__device__ __forceinline__ void leave(const Order& order, unsigned total, unsigned tag, unsigned by)
{
    if (threadIdx.x) return;
    unsigned* state = order.state;
    if (__hip_atomic_fetch_add(state + kDone, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) + 1 != gridDim.x) return;
    __hip_atomic_store(state + kDone, 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    __hip_atomic_store(state + kBase, order.base + total + Order::kPastEnd * gridDim.x, __ATOMIC_RELAXED,
                       __HIP_MEMORY_SCOPE_AGENT);
    __hip_atomic_store(state + kTag, tag + by, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

} // namespace mfv
