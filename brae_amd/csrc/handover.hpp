// Values handed from wave to wave within one launch (sweep.hip, cycle_flow.hip).
//
// The workgroups of a launch take chunks of work in order from a counter. A value crosses as one or two 8-byte
// words, each 32 bits of the value under a 32-bit tag, stored and loaded as atomic words at device scope: a
// reader that finds the tag it waits for has the value, whatever order words arrive in, so nothing else has
// to be ordered -- no fence, no barrier. Every wait ends: a chunk needs values of earlier chunks only, those
// were taken earlier, by waves that were running and leave no chunk unfinished; the earliest unfinished chunk
// never waits. Nothing depends on how many waves run at once. The tags grow with every launch (kept in device
// memory and advanced by the last workgroup to leave, so a captured launch replays correctly; chunks.hpp).
#pragma once

#include "mfv_internal.hpp"

#include "chunks.hpp"

namespace mfv {

using Word = unsigned long long;

// the words of a value of type T: put, and a read (Raw) that may or may not be the awaited one yet
template <typename T>
struct Hand;

template <>
struct Hand<double>
{
    static constexpr int words = 2;
    struct Raw
    {
        Word a, b;
        __device__ __forceinline__ bool is(unsigned tag) const
        {
            return (unsigned)(a >> 32) == tag && (unsigned)(b >> 32) == tag;
        }
        __device__ __forceinline__ double value() const
        {
            return __longlong_as_double((long long)((a & 0xffffffffull) | (b << 32)));
        }
    };
    static __device__ __forceinline__ void put(Word* p, int i, unsigned tag, double v)
    {
        const Word b = (Word)__double_as_longlong(v), t = (Word)tag << 32;
        __hip_atomic_store(p + 2 * (size_t)i, t | (b & 0xffffffffull), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        __hip_atomic_store(p + 2 * (size_t)i + 1, t | (b >> 32), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    }
    static __device__ __forceinline__ Raw get(const Word* p, int i)
    {
        const Word* q = p + 2 * (size_t)i;
        return Raw{__hip_atomic_load(q, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT),
                   __hip_atomic_load(q + 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT)};
    }
};

template <>
struct Hand<float>
{
    static constexpr int words = 1;
    struct Raw
    {
        Word a;
        __device__ __forceinline__ bool is(unsigned tag) const { return (unsigned)(a >> 32) == tag; }
        __device__ __forceinline__ float value() const { return __uint_as_float((unsigned)a); }
    };
    static __device__ __forceinline__ void put(Word* p, int i, unsigned tag, float v)
    {
        __hip_atomic_store(p + i, (Word)tag << 32 | __float_as_uint(v), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    }
    static __device__ __forceinline__ Raw get(const Word* p, int i)
    {
        return Raw{__hip_atomic_load(p + i, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT)};
    }
};

// the state a launch's first predecessor would have left: tag 1, so that no word as allocated (0) passes for a value
inline std::vector<unsigned> firstHandState() { return {0u, 0u, 1u, 0u}; }

template <typename T>
__device__ __forceinline__ T awaitValue(const Word* p, int i, unsigned tag)
{
    typename Hand<T>::Raw v = Hand<T>::get(p, i);
    while (!v.is(tag))
    {
        __builtin_amdgcn_s_sleep(1);
        v = Hand<T>::get(p, i);
    }
    return v.value();
}

} // namespace mfv
