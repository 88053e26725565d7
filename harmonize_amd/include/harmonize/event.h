// EventProgram<Spec>: the level-synchronous program type.
//
// Semantics follow the reference's program/event.h:383-518: one launch
// evaluates one generation. Each group evaluates its share of the
// per-operation input queues, then calls the spec's make_work until
// make_work returns false or an output queue is half full; then every queue
// is flipped (outputs become the next generation's inputs). The host loops
// `exec` until a generation produces no promises.
//
// Layout and mechanism are gfx950-native:
//  - a group is one 64-lane wavefront;
//  - queues hold promises as 32-bit words in structure-of-arrays form
//    ([op][word][capacity]), so a wavefront reads or writes 64 consecutive
//    words per row: fully coalesced 256-byte accesses;
//  - each operation's queue is split into SEGMENTS equal segments, each with
//    its own counter on its own 128-byte line. A group pushes to its home
//    segment (blockIdx % SEGMENTS) and moves on to others only when its own
//    is full. Device-scope atomics on one address serialise across the XCDs
//    at a few tens of ns each, so a single counter per queue would cap a
//    generation at tens of millions of pushes per second;
//  - an async call costs one atomic per wavefront per call site (ballot +
//    mbcnt), not one atomic and two system fences per lane as in the
//    reference (util/iter.h:197-214);
//  - input is not claimed at all: the flip leaves, per operation, the
//    segments' counts and the links (64 promises) before each, and group g of
//    G takes every G-th run of links, finding a link's segment with one
//    ballot. Everything a group reads to find its input was written before
//    the launch, so it comes through the XCD's L2; claim counters read and
//    advanced at the device's coherence point took 8,192 groups 60 us to find
//    that a generation of a thousand promises had nothing for them;
//  - the flip runs in a one-group kernel after each generation (the
//    reference's last group checks out through a counter that every group
//    increments).
#pragma once

#include "host.h"
#include "iter.h"
#include "spec.h"

template <typename PROGRAM_SPEC>
class EventProgram {
   public:
    typedef EventProgram<PROGRAM_SPEC> ProgramType;

    using AdrType = typename hz::spec::AdrTypeOr<PROGRAM_SPEC, unsigned int>::type;
    using OpSet = hz::spec::ProgramOpSet<PROGRAM_SPEC>;
    using DeviceState = typename hz::spec::DeviceStateOr<PROGRAM_SPEC, VoidState>::type;
    using GroupState = typename hz::spec::GroupStateOr<PROGRAM_SPEC, VoidState>::type;
    using ThreadState = typename hz::spec::ThreadStateOr<PROGRAM_SPEC, VoidState>::type;

    typedef PromiseUnion<OpSet> PromiseUnionType;

    template <typename TYPE>
    struct Lookup {
        typedef typename PromiseUnionType::template Lookup<TYPE>::type type;
    };

    static_assert(!hz::spec::GROUP_SIZEOr<PROGRAM_SPEC, 64>::given ||
                      hz::spec::GROUP_SIZEOr<PROGRAM_SPEC, 64>::value == 64,
                  "On gfx950 a group is one 64-lane wavefront; GROUP_SIZE must be 64 if given.");

    static const size_t GROUP_SIZE = 64;
    static const size_t WORK_GROUP_SIZE = 64;
    // Groups live for one generation only.
    static constexpr bool PERSISTENT = false;

    static const unsigned int BAD_FUNC_ID_FLAG = 0x00000001;
    static const unsigned int OVERFLOW_FLAG = 0x00000004;
    static const unsigned int USAGE_FLAG = 0x00000020;
    static const unsigned int EARLY_HALT_FLAG = 0x40000000;
    static const unsigned int COMPLETION_FLAG = 0x80000000;

    static const unsigned char FN_ID_COUNT = PromiseUnionType::Info::COUNT;
    static constexpr uint32_t OPS = PromiseUnionType::Info::COUNT;
    static constexpr uint32_t OPS1 = OPS > 0 ? OPS : 1;
    static constexpr uint32_t WORDS = hz::PromiseWords<OpSet>::value;
    static constexpr uint32_t SEGMENTS = 64;

    static_assert(std::is_trivially_copyable<PromiseUnionType>::value,
                  "promise arguments must be trivially copyable");

    struct ThreadContext {
        unsigned int thread_id;
        unsigned int rand_state;
    };

    struct GroupContext {
        unsigned int toggle;
    };

    // Counters of one segment of one operation's queue (one 128-byte line).
    struct Segment {
        unsigned int out_count;  // output slots claimed (may pass the capacity)
        unsigned int halt;       // operation 0's: set by halt_early for this generation
        unsigned int pad[30];
    };

    // Queue counters and run status, kept in HBM.
    struct Status {
        unsigned int toggle;
        unsigned int flags;
        unsigned int flip_count;
        unsigned int complete_at;  // flip_count when COMPLETION was last set
        unsigned int links[OPS1];  // input links (of 64 promises, per segment) of each operation
        alignas(8) unsigned long long int promises;
        unsigned long long int make_work_calls;
        alignas(128) unsigned int in_count[OPS1][SEGMENTS];  // promises in each input segment
        unsigned int in_start[OPS1][SEGMENTS];               // input links of the operation before the segment
        alignas(128) Segment seg[OPS1][SEGMENTS];
    };

    // The words of Status that a host loop looks at between generations.
    struct Header {
        unsigned int toggle, flags, flip_count, complete_at;
        unsigned int links[OPS1];
    };

    struct DeviceContext {
        typedef ProgramType ParentProgramType;
        Status* status;
        unsigned int* queues[2];  // each [OPS][WORDS][capacity]
        unsigned int capacity;    // per operation, SEGMENTS * seg_capacity
        unsigned int seg_capacity;
        unsigned int most_links;  // a launch leaves a generation of more input links to a later one (0: never)
    };

    // Owns the queues and status of one program instance (reference
    // program/event.h:139-230). `io_size` is the per-operation capacity of
    // each queue, in promises (rounded up to a multiple of SEGMENTS).
    struct Instance {
        unsigned int seg_capacity;
        unsigned int capacity;
        util::host::DevBuf<Status> status;
        util::host::DevBuf<unsigned int> queue_a;
        util::host::DevBuf<unsigned int> queue_b;
        DeviceState device_state;
        Status host_status{};
        // For hosts that launch generations ahead, with groups for what they
        // last saw: a launch that finds more input links than this does
        // nothing, so that a generation that has grown waits for a launch of
        // its size. 0: every launch runs its generation.
        unsigned int most_links = 0;

        static unsigned int seg_cap_for(size_t io_size) {
            if (io_size == 0 || io_size > 0x7FFFFFFFu) {
                throw std::runtime_error("EventProgram::Instance: io_size must be in [1, 2^31)");
            }
            return (unsigned int)((io_size + SEGMENTS - 1) / SEGMENTS);
        }

        Instance(size_t io_size, DeviceState gs)
            : seg_capacity(seg_cap_for(io_size)),
              capacity(seg_capacity * SEGMENTS),
              status((size_t)1),
              queue_a((size_t)OPS1 * WORDS * (size_t)seg_capacity * SEGMENTS),
              queue_b((size_t)OPS1 * WORDS * (size_t)seg_capacity * SEGMENTS),
              device_state(gs) {
            util::host::auto_throw(hipMemset(status.data(), 0, sizeof(Status)));
        }

        DeviceContext to_context() {
            DeviceContext result;
            result.status = status.data();
            result.queues[0] = queue_a.data();
            result.queues[1] = queue_b.data();
            result.capacity = capacity;
            result.seg_capacity = seg_capacity;
            result.most_links = most_links;
            return result;
        }

        Status read_status() {
            util::host::auto_throw(hipMemcpy(&host_status, status.data(), sizeof(Status), hipMemcpyDeviceToHost));
            return host_status;
        }

        // Reads only the flags word (the per-generation completion check).
        unsigned int read_flags() {
            unsigned int flags = 0;
            util::host::auto_throw(
                hipMemcpy(&flags, &status.data()->flags, sizeof(flags), hipMemcpyDeviceToHost));
            host_status.flags = flags;
            return flags;
        }

        // True once a generation has produced no promises. Raises if an
        // output queue overflowed (promises would have been lost).
        bool complete() { return flags_complete(read_flags()); }

        void clear_flags() {
            unsigned int zero = 0;
            util::host::auto_throw(
                hipMemcpy(&status.data()->flags, &zero, sizeof(unsigned int), hipMemcpyHostToDevice));
        }

        // Clears every queue counter, the flags and the statistics with a
        // kernel on `stream`, so that the instance can run a new job without
        // a synchronous copy (queued promises are discarded).
        void reset(hipStream_t stream);

        unsigned long long int promises() { return read_status().promises; }
    };

    // What the flags of a finished generation say (Instance::complete).
    static bool flags_complete(unsigned int flags) {
        if (flags & OVERFLOW_FLAG) {
            throw std::runtime_error(
                "EventProgram: an output queue overflowed; construct the Instance with a larger io_size");
        }
        if (flags & USAGE_FLAG) {
            throw std::runtime_error(
                "EventProgram: a Return forwarded a future that was not ready (EventProgram cannot hold "
                "promises on a barrier)");
        }
        return (flags & COMPLETION_FLAG) != 0;
    }

    DeviceContext& _dev_ctx;
    GroupContext& _grp_ctx;
    ThreadContext& _thd_ctx;

    DeviceState& device;
    GroupState& group;
    ThreadState& thread;

    __device__ EventProgram(DeviceContext& d_c, GroupContext& g_c, ThreadContext& t_c, DeviceState& d,
                            GroupState& g, ThreadState& t)
        : _dev_ctx(d_c), _grp_ctx(g_c), _thd_ctx(t_c), device(d), group(g), thread(t) {}

   protected:
    // (A choice, not an index: indexed by a variable, the context is kept in
    // LDS, a copy per lane.)
    __device__ unsigned int* queue_row(unsigned int which, OpDisc op, unsigned int word) {
        unsigned int* queue = which != 0u ? _dev_ctx.queues[1] : _dev_ctx.queues[0];
        return queue + ((size_t)op * WORDS + word) * _dev_ctx.capacity;
    }

    __device__ Segment& segment(OpDisc op, uint32_t s) { return _dev_ctx.status->seg[op][s]; }

    // Whether the generation, of `links` input links, is too large for this
    // launch (DeviceContext::most_links).
    __device__ static bool left_to_later(const DeviceContext& ctx, unsigned long long links) {
        return ctx.most_links != 0u && links > ctx.most_links;
    }

    __device__ uint32_t home_segment() const { return blockIdx.x % SEGMENTS; }

    __device__ void set_flags(unsigned int bits) { hz::wave::atomic_or(&_dev_ctx.status->flags, bits); }

   public:
    // Appends one promise per active lane to the output queue of TYPE: one
    // atomic per wavefront on the home segment, spilling to the following
    // segments only when it is full. The depth delta is accepted and ignored:
    // a generation runs every queued promise, whatever its depth (as in the
    // reference, program/event.h:326-358).
    template <typename TYPE>
    __device__ void async_call_cast(int /*depth_delta*/, Promise<TYPE> param_value) {
        constexpr OpDisc D = Lookup<TYPE>::type::DISC;
        static_assert(Lookup<TYPE>::type::CONTAINED, "operation is not part of this program's OpSet");
        PromiseUnionType pu;
        pu.template cast<TYPE>() = param_value;
        uint32_t words[WORDS];
        __builtin_memcpy(words, &pu, sizeof(PromiseUnionType));
        const unsigned int out = _grp_ctx.toggle ^ 1u;
        const uint32_t cap = _dev_ctx.seg_capacity;
        bool pending = true;
        uint32_t s = home_segment();
        for (uint32_t attempt = 0; attempt < SEGMENTS; ++attempt) {
            uint64_t want = hz::wave::ballot(pending);
            if (want == 0) break;
            uint32_t r = hz::wave::rank(want);
            uint32_t base = 0;
            if (pending && r == 0) base = hz::wave::atomic_add(&segment(D, s).out_count, hz::wave::popc(want));
            base = hz::wave::first(hz::wave::read_lane(base, (uint32_t)__builtin_ctzll(want)));
            if (pending) {
                uint32_t idx = base + r;
                if (idx < cap) {
                    size_t at = (size_t)s * cap + idx;
#pragma unroll
                    for (uint32_t w = 0; w < WORDS; ++w) queue_row(out, D, w)[at] = words[w];
                    pending = false;
                }
            }
            s = (s + 1 == SEGMENTS) ? 0 : s + 1;
        }
        if (hz::wave::ballot(pending) != 0 && hz::wave::leader()) set_flags(OVERFLOW_FLAG);
    }

    // Queues up to K promises of one operation per active lane, those with
    // want[k], with one atomic for all of them while the home segment has
    // room.
    template <typename TYPE, int K>
    __device__ void async_each(int depth_delta, const Promise<TYPE> (&values)[K], const bool (&want)[K]) {
        constexpr OpDisc D = Lookup<TYPE>::type::DISC;
        static_assert(Lookup<TYPE>::type::CONTAINED, "operation is not part of this program's OpSet");
        uint32_t at[K], total = 0;
#pragma unroll
        for (int k = 0; k < K; ++k) {
            const uint64_t m = hz::wave::ballot(want[k]);
            at[k] = total + hz::wave::rank(m);
            total += hz::wave::popc(m);
        }
        if (total == 0u) return;
        const unsigned int out = _grp_ctx.toggle ^ 1u;
        const uint32_t cap = _dev_ctx.seg_capacity;
        const uint32_t s = home_segment();
        uint32_t base = 0;
        if (hz::wave::leader()) base = hz::wave::atomic_add(&segment(D, s).out_count, total);
        base = hz::wave::first(base);
        bool left = false;
#pragma unroll
        for (int k = 0; k < K; ++k) {
            if (want[k] && base + at[k] < cap) {
                PromiseUnionType pu;
                pu.template cast<TYPE>() = values[k];
                uint32_t words[WORDS];
                __builtin_memcpy(words, &pu, sizeof(PromiseUnionType));
                const size_t i = (size_t)s * cap + base + at[k];
#pragma unroll
                for (uint32_t w = 0; w < WORDS; ++w) queue_row(out, D, w)[i] = words[w];
            } else if (want[k]) {
                left = true;
            }
        }
        if (hz::wave::ballot(left) == 0ull) return;
#pragma unroll
        for (int k = 0; k < K; ++k) {
            if (want[k] && base + at[k] >= cap) async_call_cast(depth_delta, values[k]);
        }
    }

    // Depth level of the promise being evaluated: a level-synchronous
    // program keeps no levels, so always 0.
    __device__ unsigned int depth() { return 0u; }

   protected:
    template <typename TYPE>
    __device__ void immediate_call_cast(Promise<TYPE> param_value) {
        param_value(*this);
    }

    __device__ void eval_words(OpDisc op, const uint32_t* words) {
        PromiseUnionType pu;
        __builtin_memcpy(&pu, words, sizeof(PromiseUnionType));
        pu.template loose_eval<ProgramType>(*this, op);
    }

   public:
    __device__ void init_program() {}

    // One generation (reference program/event.h:383-518).
    __device__ void exec(unsigned int chunk_size) {
        const uint32_t lane = hz::wave::lane();
        _thd_ctx.thread_id = blockIdx.x * 64u + lane;
        _thd_ctx.rand_state = _thd_ctx.thread_id;
        Status* st = _dev_ctx.status;
        const unsigned int in = st->toggle;
        unsigned long long all = 0;
        for (uint32_t op = 0; op < OPS; ++op) all += st->links[op];
        if (left_to_later(_dev_ctx, all)) return;
        _grp_ctx.toggle = in;
        hz::wave::sync();
        const uint32_t home = home_segment();
        unsigned long long made = 0;

        // The spec hooks are inlined: a hook left out of line would take the
        // program object and push the state it refers to into scratch memory.
        [[clang::always_inline]] PROGRAM_SPEC::initialize(*this);

        // This group's links of each operation, up to chunk_size of them in a
        // row (fewer where the generation would leave groups without any).
        // Operations start at different groups, so that small generations of
        // several operations do not all fall to the same ones.
        const uint32_t most = chunk_size == 0 ? 1u : chunk_size;
        for (uint32_t op = 0; op < OPS; ++op) {
            const uint32_t links = st->links[op];
            if (links == 0u) continue;
            const uint32_t start = st->in_start[op][lane];
            const uint32_t count = st->in_count[op][lane];
            uint32_t run = links / gridDim.x;
            run = run < 1u ? 1u : (run > most ? most : run);
            uint32_t g = blockIdx.x + op * (gridDim.x / OPS1);
            if (g >= gridDim.x) g -= gridDim.x;
            for (uint64_t first = (uint64_t)g * run; first < links; first += (uint64_t)gridDim.x * run) {
                const uint32_t last = first + run < links ? (uint32_t)first + run : links;
                for (uint32_t l = (uint32_t)first; l < last; ++l) {
                    // The last segment that starts at or before link l holds
                    // it: an empty segment starts where its successor does.
                    const uint32_t s = hz::wave::popc(hz::wave::ballot(start <= l)) - 1u;
                    const uint32_t at = (l - hz::wave::read_lane(start, s)) * 64u + lane;
                    if (at < hz::wave::read_lane(count, s)) {
                        const size_t i = (size_t)s * _dev_ctx.seg_capacity + at;
                        uint32_t words[WORDS];
#pragma unroll
                        for (uint32_t w = 0; w < WORDS; ++w) words[w] = queue_row(in, op, w)[i];
                        eval_words(op, words);
                    }
                    hz::wave::sync();
                }
            }
        }

        // Make work until the spec says it has none or this group's output
        // segment is half full.
        bool more = hz::wave::first(hz::wave::atomic_load(&segment(0, home).halt)) == 0u;
        while (more) {
            for (uint32_t i = 0; i < OPS; ++i) {
                uint32_t n = hz::wave::first(hz::wave::atomic_load(&segment(i, home).out_count));
                if (n >= _dev_ctx.seg_capacity / 2) more = false;
            }
            if (!more) break;
            bool mine;
            [[clang::always_inline]] mine = PROGRAM_SPEC::make_work(*this);
            more = hz::wave::ballot(mine) != 0;
            if (more) made++;
        }

        [[clang::always_inline]] PROGRAM_SPEC::finalize(*this);
        if (lane == 0 && made) hz::wave::atomic_add(&st->make_work_calls, made);
    }

    // Zeroes the Status struct (grid-stride over its 32-bit words).
    __device__ static void kernel_reset(DeviceContext ctx) {
        unsigned int* w = (unsigned int*)ctx.status;
        const size_t words = sizeof(Status) / sizeof(unsigned int);
        for (size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x; i < words; i += (size_t)gridDim.x * blockDim.x) {
            w[i] = 0u;
        }
    }

    // Flips every queue for the next generation (reference event.h:500-515,
    // util/iter.h:437-445) and records completion when nothing was produced.
    // Launched as one 64-lane group after each generation; lane s handles
    // segment s of every operation.
    static_assert(SEGMENTS == 64, "flip assigns one segment per lane");
    __device__ static void flip(DeviceContext ctx) {
        Status* st = ctx.status;
        const uint32_t lane = hz::wave::lane();
        unsigned long long executed = 0, all = 0;
        uint32_t produced = 0;
        // The counts are read together: a generation of few promises is one
        // trip to memory after another.
        constexpr uint32_t AHEAD = OPS1 < 8u ? OPS1 : 8u;
        uint32_t came[AHEAD], went[AHEAD];
#pragma unroll
        for (uint32_t i = 0; i < AHEAD; ++i) {
            came[i] = st->in_count[i][lane];
            went[i] = st->seg[i][lane].out_count;
        }
        for (uint32_t i = 0; i < OPS; ++i) all += st->links[i];
        if (left_to_later(ctx, all)) return;
#pragma unroll 8
        for (uint32_t i = 0; i < OPS; ++i) {
            Segment& g = st->seg[i][lane];
            executed += i < AHEAD ? came[i < AHEAD ? i : 0u] : st->in_count[i][lane];
            const uint32_t out = i < AHEAD ? went[i < AHEAD ? i : 0u] : g.out_count;
            const uint32_t n = out < ctx.seg_capacity ? out : ctx.seg_capacity;
            g.out_count = 0;
            g.halt = 0;
            // Links before this lane's segment: an inclusive scan, less its own.
            const uint32_t mine = n / 64u + (n % 64u != 0u ? 1u : 0u);
            uint32_t upto = mine;
#pragma unroll
            for (uint32_t d = 1; d < 64u; d <<= 1) {
                const uint32_t below = __shfl_up(upto, d, 64);
                if (lane >= d) upto += below;
            }
            st->in_count[i][lane] = n;
            st->in_start[i][lane] = upto - mine;
            const uint32_t links = hz::wave::read_lane(upto, 63u);
            if (lane == 0) st->links[i] = links;
            produced += links;
        }
#pragma unroll
        for (int d = 32; d >= 1; d >>= 1) executed += __shfl_xor(executed, d, 64);
        if (lane == 0) {
            st->promises += executed;
            st->toggle ^= 1u;
            st->flip_count += 1;
            unsigned int flags = st->flags;
            if (produced == 0 && (flags & EARLY_HALT_FLAG) == 0) {
                if ((flags & COMPLETION_FLAG) == 0) st->complete_at = st->flip_count;
                flags |= COMPLETION_FLAG;
            }
            st->flags = flags & ~EARLY_HALT_FLAG;
        }
    }

    template <typename TYPE, typename... ARGS>
    __device__ void async(ARGS... args) {
        async_call_cast<TYPE>(0, Promise<TYPE>(args...));
    }

    template <typename TYPE>
    __device__ void async_call(Promise<TYPE> promise) {
        async_call_cast<TYPE>(0, promise);
    }

    template <typename TYPE, typename... ARGS>
    __device__ void sync(ARGS... args) {
        immediate_call_cast<TYPE>(Promise<TYPE>(args...));
    }

    template <typename TYPE>
    __device__ void sync_call(Promise<TYPE> promise) {
        immediate_call_cast<TYPE>(promise);
    }

    // Fill fraction of TYPE's output in this group's home segment (reference
    // event.h:540-544 reports the whole queue's).
    template <typename TYPE>
    __device__ float load_fraction() {
        unsigned int n =
            hz::wave::atomic_load(&segment(Lookup<TYPE>::type::DISC, home_segment()).out_count);
        return (float)n / (float)_dev_ctx.seg_capacity;
    }

    // Rare, so it tells every home segment: a group looks only at its own.
    __device__ void halt_early() {
        set_flags(EARLY_HALT_FLAG);
        for (uint32_t s = 0; s < SEGMENTS; ++s) hz::wave::atomic_store(&segment(0, s).halt, 1u);
    }

    // Promises cannot be held on a RemappingBarrier (see barrier_await).
    static constexpr bool REMAPPING_AWAIT = false;
    static constexpr bool RETURN_RELEASE = hz::spec::RETURN_RELEASEOr<PROGRAM_SPEC, 1>::value != 0;
    // Records a misuse of the future API; complete() reports it.
    __device__ void usage_error() { set_flags(USAGE_FLAG); }

    // Queues a promise held as a PromiseEnum (UnitBarrier release).
    __device__ HZ_INLINE void async_call(PromiseEnum<OpSet> promise) { async_enum<0>(promise); }

    // Holding promises on a RemappingBarrier needs the async program's link
    // arena, as in the reference (sync/barrier.h uses AsyncProgram internals
    // throughout), so awaiting is rejected at compile time. Releasing one is
    // allowed and has nothing to run: no promise can have been held. (A
    // future backed by a RemappingBarrier still carries its value and its
    // ready state under EventProgram.)
    template <typename BARRIER, typename OP_TYPE>
    __device__ void barrier_await(BARRIER&, Promise<OP_TYPE>) {
        static_assert(sizeof(OP_TYPE) == 0, "RemappingBarrier::await is supported by AsyncProgram, not EventProgram");
    }
    template <typename BARRIER>
    __device__ void barrier_release(BARRIER&) {}

   protected:
    template <unsigned int I>
    __device__ HZ_INLINE void async_enum(PromiseEnum<OpSet>& pe) {
        if constexpr (I < OPS) {
            using Op = typename hz::OpOf<I, OpSet>::type;
            if (pe.disc == I) {
                async_call_cast<Op>(0, pe.data.template cast<Op>());
            } else {
                async_enum<I + 1>(pe);
            }
        }
    }

   public:

    __device__ static void kernel_exec(DeviceContext ctx, DeviceState state, unsigned int chunk) {
        __shared__ GroupContext gctx;
        __shared__ GroupState group_state;
        ThreadContext tctx;
        ThreadState thread_state;
        ProgramType prog(ctx, gctx, tctx, state, group_state, thread_state);
        prog.exec(chunk);
    }
};
