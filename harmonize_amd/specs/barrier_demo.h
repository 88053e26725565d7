// Remapping-barrier specification, after the reference's barrier demo
// (examples/cpp/barrier_demo/demo.cpp:26-44, :153-162): make_work evaluates
// Step(id) for ids [0, dep + non_dep) in place; a dependent step (id < dep)
// awaits barrier[id % barriers] with a held Step and then decrements that
// barrier's semaphore, which starts at the number of dependents mapped to it.
// The reference's expected count is dep * 2 + non_dep (demo.cpp:214).
//
// Held steps carry HELD_BASE + id so the run can prove that every held promise
// ran exactly once (hits[id]) and only after its barrier was released
// (violations).
#pragma once

#include <cstdint>

struct BarrierStep;

constexpr unsigned int BARRIER_HELD_BASE = 0x80000000u;

struct BarrierDemoState {
    unsigned int dep_count;
    unsigned int non_dep_count;
    unsigned int barrier_count;
    unsigned int pad;
    util::iter::AtomicIter<unsigned int>* source_id_iter;
    unsigned int* counter;     // Step evaluations
    unsigned int* hits;        // [dep_count] runs of each held step
    unsigned int* violations;  // held steps that ran before their barrier was released
    RemappingBarrier<OpUnion<BarrierStep>>* barrier;
};

// The id a thread has claimed (make_work starts it at once, so none is left
// when a launch ends), and the evaluations it has yet to add to the counter.
struct BarrierDemoThread {
    util::iter::Share<unsigned int> ids;
    unsigned int steps;
};

struct BarrierStep {
    using Type = void (*)(unsigned int);

    template <typename PROGRAM>
    __device__ static void eval(PROGRAM prog, unsigned int arg) {
        const BarrierDemoState& st = prog.device;
        prog.thread.steps += 1u;
        if (arg >= BARRIER_HELD_BASE) {
            unsigned int id = arg - BARRIER_HELD_BASE;
            atomicAdd(&st.hits[id], 1u);
            RemappingBarrier<OpUnion<BarrierStep>>& b = st.barrier[id % st.barrier_count];
            if (hz_load(&b.semaphore.sem) != 0u) atomicAdd(st.violations, 1u);
            return;
        }
        if (arg < st.dep_count) {
            RemappingBarrier<OpUnion<BarrierStep>>& b = st.barrier[arg % st.barrier_count];
            b.await(prog, Promise<BarrierStep>(BARRIER_HELD_BASE + arg));
            b.add_semaphore(prog, (unsigned int)-1);
        }
    }
};

struct BarrierDemoSpec {
    using OpSet = OpUnion<BarrierStep>;
    using DeviceState = BarrierDemoState;
    using ThreadState = BarrierDemoThread;

    static const size_t STASH_SIZE = 8;
    static const size_t FRAME_SIZE = 8;
    static const size_t POOL_SIZE = 8;

    // The source iterator and the counter are one word each for the whole
    // device, which passes an atomic or a load every 30 ns. Each thread
    // counts for itself until the group leaves, and a claim is one load and
    // one atomic: 2^21 awaits and as many ids without take 10.6 ms on 64
    // barriers and 6.9 on 1,024 (11.7 and 7.6 with every evaluation counted
    // as it ran). More ids per claim are faster for few and for very many
    // barriers (8: 9.5 ms at 64, 5.6 at 8,192) and slower between them (14.8
    // at 256 and 512, against 7.5): wavefronts then await in step.
    static const unsigned int CLAIM = 1;

    template <typename PROGRAM>
    __device__ static void initialize(PROGRAM prog) {
        prog.thread.ids.clear();
        prog.thread.steps = 0u;
    }

    template <typename PROGRAM>
    __device__ static void finalize(PROGRAM prog) {
        unsigned int steps = prog.thread.steps;
#if defined(__HIP_DEVICE_COMPILE__)
        for (int d = 32; d >= 1; d >>= 1) steps += __shfl_xor(steps, d, 64);
        if (!hz::wave::leader()) return;
#endif
        atomicAdd(prog.device.counter, steps);
    }

    template <typename PROGRAM>
    __device__ static bool make_work(PROGRAM prog) {
        util::iter::claim_share(prog.thread.ids, *prog.device.source_id_iter, (unsigned int)CLAIM);
        unsigned int id;
        if (!prog.thread.ids.step(id)) return false;
        prog.template sync<BarrierStep>(id);
        return true;
    }
};
