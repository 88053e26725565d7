// hz_wait_selftest: a program whose promises requeue themselves until another
// promise has run, which the group makes only after the waiting ones. It
// checks that lanes that go on chaining do not keep a group from making work.
#include "workspace.h"

using hz::capi::check;
using hz::capi::guarded;

namespace {

struct WaitState {
    unsigned int* words;   // 0: gate, 1: make_work calls, 2: promises let through
    unsigned int waiting;  // promises that wait, fewer than a wavefront's lanes
};

struct WaitAtGate {
    using Type = void (*)(unsigned int);
    template <typename PROGRAM>
    __device__ static void eval(PROGRAM prog, unsigned int id) {
        if (hz_load(&prog.device.words[0]) == 0u) {
            prog.template async<WaitAtGate>(id);
        } else {
            atomicAdd(&prog.device.words[2], 1u);
        }
    }
};

struct WaitOpen {
    using Type = void (*)(unsigned int);
    template <typename PROGRAM>
    __device__ static void eval(PROGRAM prog, unsigned int) {
        hz::wave::atomic_store(&prog.device.words[0], 1u);
    }
};

template <size_t MIXED>
struct WaitSpec {
    using OpSet = OpUnion<WaitAtGate, WaitOpen>;
    using DeviceState = WaitState;
    static const size_t STASH_SIZE = 8;
    static const size_t FRAME_SIZE = 8;
    static const size_t POOL_SIZE = 8;
    static const size_t CHAIN_MIXED = MIXED;

    template <typename PROGRAM>
    __device__ static void initialize(PROGRAM) {}
    template <typename PROGRAM>
    __device__ static void finalize(PROGRAM) {}

    // The waiting promises first, the one they wait for in the call after.
    template <typename PROGRAM>
    __device__ static bool make_work(PROGRAM prog) {
        const unsigned int lane = hz::wave::lane();
        unsigned int call = 0u;
        if (lane == 0u) call = hz::wave::atomic_add(&prog.device.words[1], 1u);
        call = hz::wave::first(call);
        if (call == 0u && lane < prog.device.waiting) prog.template async<WaitAtGate>(lane);
        if (call == 1u && lane == 0u) prog.template async<WaitOpen>(0u);
        return call <= 1u;
    }
};

template <typename P>
void run_wait(uint32_t waiting, const hz_run_config& cfg, uint32_t* passed, hz_run_stats* stats) {
    hz::capi::Lease<hz::capi::Scratch> words(256, 0);
    check(hipMemset(words->p, 0, 256), "zero words");
    const uint32_t groups = 1;
    hz::capi::Lease<hz::capi::AsyncSpace<P>> ws(1024, 1);
    ws->begin(WaitState{(unsigned int*)words->p, waiting}, cfg, groups);
    ws->run(groups, cfg, stats);
    check(hipMemcpy(passed, (unsigned int*)words->p + 2, sizeof(uint32_t), hipMemcpyDeviceToHost), "passed");
}

}  // namespace

extern "C" int hz_wait_selftest(uint32_t waiting, int mixed, uint32_t cycles, uint32_t max_launches, uint32_t* passed) {
    return guarded([&] {
        if (!passed || waiting > 63u) throw std::invalid_argument("hz_wait_selftest: at most 63 promises wait");
        hz_run_config cfg{};
        cfg.cycles = cycles;
        cfg.max_launches = max_launches;
        if (mixed) {
            run_wait<AsyncProgram<WaitSpec<1>>>(waiting, cfg, passed, nullptr);
        } else {
            run_wait<AsyncProgram<WaitSpec<0>>>(waiting, cfg, passed, nullptr);
        }
    });
}
