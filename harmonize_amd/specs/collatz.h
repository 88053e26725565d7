// Collatz step-count specification.
//
// Same program as the reference's example (examples/cpp/collaz/collaz_hrm.cpp:
// Even :9-32, Odd :36-61, make_work :127-144): two async operations that
// carry (value, step, index); Even halves an even value, Odd maps an odd value
// v to 3v+1, each then re-dispatches on the parity of the new value, and a
// value <= 1 writes its step count. Differences, the first two forced by the
// workloads:
//  - starts come from a device array (configurations draw them at random),
//    with start = index when the array is absent, as in the reference;
//  - 3v+1 is checked for overflow of 64 bits (starts below 2^40 exist whose
//    trajectories pass 2^64); such a start records COLLATZ_OVERFLOW;
//  - only Odd tests for the end of a chain (see CollatzEven).
//
// Written against the spec API only; compiled for gfx950 by the runtime and
// for the host by the oracle's sequential executor.
#pragma once

#include <cstdint>

constexpr unsigned int COLLATZ_OVERFLOW = 0xFFFFFFFFu;

struct CollatzState {
    const unsigned long long* starts;
    unsigned int* steps;
    util::iter::AtomicIter<unsigned int>* iterator;
};

struct CollatzEven;
struct CollatzOdd;

template <typename PROGRAM>
__device__ inline void collatz_dispatch(PROGRAM& prog, unsigned long long val, unsigned int step,
                                        unsigned int index) {
    if ((val & 1ull) == 0) {
        prog.template async<CollatzEven>(val, step, index);
    } else {
        prog.template async<CollatzOdd>(val, step, index);
    }
}

// Both ends of a chain in one test: v <= 1, or 3v + 1 beyond 64 bits
// (3v + 1 <= 2^64 - 1  <=>  v <= (2^64 - 2) / 3).
__device__ inline bool collatz_ends(unsigned long long v) { return v - 2ull > 0x5555555555555554ull - 2ull; }

// 3v + 1 of an odd v as v + (2v | 1): two shift-and-add instructions, where a
// product by 3 becomes two 64-bit multiply-adds and their moves.
__device__ inline unsigned long long collatz_odd_step(unsigned long long v) { return v + ((v << 1) | 1ull); }

// The same condition, as a lane mask of its own: code under it and code under
// the condition's complement stay two separate branches, of which the rare
// one is skipped and the common one needs no second half.
__device__ inline bool collatz_apart(bool condition) {
#if defined(__HIP_DEVICE_COMPILE__)
    return __builtin_amdgcn_inverse_ballot_w64(hz::wave::ballot(condition));
#else
    return condition;
#endif
}

// Even halves any value it is given: a chain ends in Odd. Halving reaches 1,
// which Odd ends, and a start of 0 (the only even value <= 1) is queued as an
// Odd promise, which ends it too. Without an end of its own, Even compiles to
// a few predicated vector instructions and no branch.
struct CollatzEven {
    using Type = void (*)(unsigned long long val, unsigned int step, unsigned int index);

    template <typename PROGRAM>
    __device__ static void eval(PROGRAM prog, unsigned long long val, unsigned int step, unsigned int index) {
        collatz_dispatch(prog, val >> 1, step + 1, index);
    }
};

struct CollatzOdd {
    using Type = void (*)(unsigned long long val, unsigned int step, unsigned int index);

    template <typename PROGRAM>
    __device__ static void eval(PROGRAM prog, unsigned long long val, unsigned int step, unsigned int index) {
        const bool ends = collatz_ends(val);
        if (collatz_apart(ends)) prog.device.steps[index] = val <= 1 ? step : COLLATZ_OVERFLOW;
        if (!ends) collatz_dispatch(prog, collatz_odd_step(val), step + 1, index);
    }
};

// Stash links per group. Seven links is the smallest stash
// that does not spill (two open links plus the three kept free before each
// evaluation); fewer links per wavefront mean more resident wavefronts to
// hide LDS and memory latency: 2^26 starts take 79 ms with 7 links against
// 145 ms with 16, while 6 links spill on nearly every cycle.
#ifndef HZ_COLLATZ_STASH
#define HZ_COLLATZ_STASH 7
#endif
// Most starts a lane claims at once (claim_share).
#ifndef HZ_COLLATZ_CLAIM
#define HZ_COLLATZ_CLAIM 32
#endif
// Wavefront groups per workgroup.
#ifndef HZ_COLLATZ_BLOCK
#define HZ_COLLATZ_BLOCK 1
#endif

template <typename PROGRAM>
__device__ inline void collatz_launch(PROGRAM& prog, unsigned int index) {
    unsigned long long start = prog.device.starts ? prog.device.starts[index] : (unsigned long long)index;
    if (start == 0ull) {
        prog.template async<CollatzOdd>(start, 0u, index);
    } else {
        collatz_dispatch(prog, start, 0u, index);
    }
}

struct CollatzSpec {
    typedef OpUnion<CollatzEven, CollatzOdd> OpSet;
    typedef CollatzState DeviceState;
    typedef util::iter::Share<unsigned int> ThreadState;  // starts claimed and not yet launched

    static const size_t STASH_SIZE = HZ_COLLATZ_STASH;
    static const size_t GROUPS_PER_BLOCK = HZ_COLLATZ_BLOCK;
    static const size_t FRAME_SIZE = 8;
    static const size_t POOL_SIZE = 8;
#ifndef HZ_COLLATZ_PASSES
#define HZ_COLLATZ_PASSES 8
#endif
    static const size_t CHAIN_PASSES = HZ_COLLATZ_PASSES;

    template <typename PROGRAM>
    __device__ static void initialize(PROGRAM prog) {
        prog.thread.clear();
    }

    // Claimed starts not launched yet are queued now, so a pass that ends
    // early loses none of them.
    template <typename PROGRAM>
    __device__ static void finalize(PROGRAM prog) {
        unsigned int index;
        while (prog.thread.step(index)) collatz_launch(prog, index);
    }

    // Launches one start per thread per call, as the reference's make_work
    // does (collaz_hrm.cpp:127-144), from the thread's share of the starts.
    template <typename PROGRAM>
    __device__ static bool make_work(PROGRAM prog) {
        // What a group of one generation has claimed and not launched goes to
        // its output queue when it stops, so it takes less at once.
        constexpr bool stays = PROGRAM::PERSISTENT;
        util::iter::claim_share(prog.thread, *prog.device.iterator, stays ? (unsigned int)HZ_COLLATZ_CLAIM : 8u,
                                stays ? 0u : 1u << 22);
        unsigned int index;
        if (!prog.thread.step(index)) return false;
        collatz_launch(prog, index);
        return true;
    }
};
