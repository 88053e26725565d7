// Shared plumbing of the C-ABI translation units: error capture, the
// per-program entry-point generator, and launch sizing.
#pragma once

#include <harmonize.h>

#include <atomic>
#include <chrono>
#include <cstddef>
#include <cstring>
#include <string>

#include "harmonize_amd.h"

namespace hz {
namespace capi {

void set_error(const std::string& message);
void clear_error();

// Runs `fn`, turning exceptions into a status code and a stored message.
template <typename F>
int guarded(F&& fn) {
    try {
        clear_error();
        fn();
        return HZ_OK;
    } catch (const std::invalid_argument& e) {
        set_error(e.what());
        return HZ_ERR_ARGUMENT;
    } catch (const std::exception& e) {
        set_error(e.what());
        return HZ_ERR_RUNTIME;
    }
}

inline void check(hipError_t e, const char* what) {
    if (e != hipSuccess) {
        throw std::runtime_error(std::string(what) + ": " + hipGetErrorString(e));
    }
}

int compute_units();

// Groups (64-lane wavefronts) that fit on the device at once for `kernel`,
// launched in workgroups of `block_threads` threads.
template <typename K>
int resident_groups(K kernel, int block_threads = 64) {
    int per_cu = 0;
    check(hipOccupancyMaxActiveBlocksPerMultiprocessor(&per_cu, kernel, block_threads, 0), "occupancy query");
    if (per_cu < 1) per_cu = 1;
    return per_cu * compute_units() * (block_threads / 64);
}

// The same for a program type's exec kernel (asked once per device).
template <typename P>
int resident_groups_of() {
    static std::atomic<int> known[64];
    int dev = 0;
    check(hipGetDevice(&dev), "hipGetDevice");
    if (dev < 0 || dev >= 64) return resident_groups(hz::exec_kernel<P>(), (int)P::WORK_GROUP_SIZE);
    int n = known[dev].load(std::memory_order_relaxed);
    if (n == 0) {
        n = resident_groups(hz::exec_kernel<P>(), (int)P::WORK_GROUP_SIZE);
        known[dev].store(n, std::memory_order_relaxed);
    }
    return n;
}

// Groups for a program that starts from `items` items, `per_group` of them in
// a group: no more than are resident, and none that would find no item. (An
// idle group still checks in and out of counters that all groups share: 1,024
// Collatz starts took 0.57 ms with 5,632 groups.)
template <typename P>
uint32_t groups_for(uint64_t items, uint64_t per_group = 64) {
    const uint64_t want = items == 0 ? 1 : (items + per_group - 1) / per_group;
    const uint64_t most = (uint64_t)resident_groups_of<P>();
    return (uint32_t)(want < most ? want : most);
}

// Owns a device AtomicIter<unsigned int> set to [0, limit).
struct DeviceIter {
    util::iter::AtomicIter<unsigned int>* ptr = nullptr;
    explicit DeviceIter(unsigned int limit) {
        util::iter::AtomicIter<unsigned int> host(0u, limit);
        check(util::host::device_malloc((void**)&ptr, sizeof(host)), "hipMalloc(iterator)");
        check(hipMemcpy(ptr, &host, sizeof(host), hipMemcpyHostToDevice), "hipMemcpy(iterator)");
    }
    ~DeviceIter() {
        if (ptr) (void)hipFree(ptr);
    }
    DeviceIter(const DeviceIter&) = delete;
    DeviceIter& operator=(const DeviceIter&) = delete;
};

// Times a span on the null stream with hipEvents.
struct EventTimer {
    hipEvent_t a{}, b{};
    EventTimer() {
        check(hipEventCreate(&a), "hipEventCreate");
        check(hipEventCreate(&b), "hipEventCreate");
    }
    ~EventTimer() {
        (void)hipEventDestroy(a);
        (void)hipEventDestroy(b);
    }
    void start() { check(hipEventRecord(a, nullptr), "hipEventRecord"); }
    // The span's end, if no later mark() moves it.
    void mark() { check(hipEventRecord(b, nullptr), "hipEventRecord"); }
    double elapsed() {
        check(hipEventSynchronize(b), "hipEventSynchronize");
        float ms = 0;
        check(hipEventElapsedTime(&ms, a, b), "hipEventElapsedTime");
        return ms;
    }
    double stop() {
        mark();
        return elapsed();
    }
};

// Runs an EventProgram instance, reset on `stream`, generation by generation
// until it is complete; returns the number of generations. `header` is
// page-locked.
//
// A generation of few promises takes 10 us on the device and one look at its
// flags from the host 20 us more, so generations are launched several at a
// time (one that finds the program complete does nothing): four while the
// program is young, then sixteen, and then, if `adapt`, with no more groups
// than twice the links of the last generation seen have use for. A generation
// that has meanwhile grown beyond four links a group waits (most_links): the
// program is young again, and its generations get all groups. (A path of 40
// vertices into a graph of 2^20 was searched on 66 groups for up to sixteen
// generations: 9.1 ms, now 1.9; into one of 2^22, 32.1 and 3.1.) At most
// `groups` groups and `max_launches` generations run.
template <typename P>
uint64_t run_generations(typename P::Instance& inst, uint32_t groups, bool adapt, uint32_t chunk,
                         uint32_t max_launches, hipStream_t stream, typename P::Header* header) {
    static_assert(offsetof(typename P::Status, links) == offsetof(typename P::Header, links), "status header");
    constexpr uint64_t YOUNG = 16;
    uint64_t done = 0, calm = 0;  // generations in all, and since the start or the last growth
    uint32_t now = groups;
    while (true) {
        if (done >= max_launches) throw std::runtime_error("EventProgram: launch bound reached before completion");
        const uint64_t want = calm < YOUNG ? 4u : 16u;
        const uint64_t batch = want < max_launches - done ? want : max_launches - done;
        inst.most_links = now < groups ? 4u * now : 0u;
        for (uint64_t i = 0; i < batch; ++i) exec<P>(inst, now, chunk, stream);
        check(hipGetLastError(), "exec launch");
        check(hipMemcpyAsync(header, inst.status.data(), sizeof(*header), hipMemcpyDeviceToHost, stream), "status copy");
        check(hipStreamSynchronize(stream), "event exec");
        if (P::flags_complete(header->flags)) {
            inst.most_links = 0u;
            return header->complete_at;
        }
        calm += header->flip_count - done;
        done = header->flip_count;
        uint64_t links = 0;
        for (uint32_t i = 0; i < P::OPS; ++i) links += header->links[i];
        if (inst.most_links != 0u && links > inst.most_links) calm = 0;
        const uint64_t use = 2u * links + 64u;
        now = adapt && calm >= YOUNG && use < groups ? (uint32_t)use : groups;
    }
}

}  // namespace capi
}  // namespace hz

// Generates the reference-shaped per-program C entry points
// (harmonize/python/templates.py:3-184) for program type PROG whose device
// state is a plain struct STATE. The instance keeps a by-value copy of the
// state and refreshes it from the device copy before every launch, so the
// device copy behaves like the reference's state pointer.
#define HZ_DEFINE_PROGRAM_ABI(suffix, PROG, STATE)                                                      \
    namespace {                                                                                         \
    struct suffix##_handle {                                                                            \
        PROG::Instance inst;                                                                            \
        void* dev_state;                                                                                \
        suffix##_handle(STATE s, size_t n, void* d) : inst(n, s), dev_state(d) {}                       \
        void refresh() {                                                                                \
            hz::capi::check(hipMemcpy(&inst.device_state, dev_state, sizeof(STATE), hipMemcpyDeviceToHost), \
                            "state refresh");                                                           \
        }                                                                                               \
    };                                                                                                  \
    }                                                                                                   \
    extern "C" void* alloc_state_##suffix(void) {                                                       \
        void* p = nullptr;                                                                              \
        hz::capi::guarded([&] { hz::capi::check(util::host::device_malloc(&p, sizeof(STATE)), "hipMalloc(state)"); }); \
        return p;                                                                                       \
    }                                                                                                   \
    extern "C" void free_state_##suffix(void* state) {                                                  \
        hz::capi::guarded([&] { hz::capi::check(hipFree(state), "hipFree(state)"); });                  \
    }                                                                                                   \
    extern "C" void load_state_device_##suffix(void* host_ptr, void* dev_ptr) {                         \
        hz::capi::guarded([&] {                                                                         \
            hz::capi::check(hipMemcpy(host_ptr, dev_ptr, sizeof(STATE), hipMemcpyDeviceToHost), "load_state"); \
        });                                                                                             \
    }                                                                                                   \
    extern "C" void store_state_device_##suffix(void* dev_ptr, void* host_ptr) {                        \
        hz::capi::guarded([&] {                                                                         \
            hz::capi::check(hipMemcpy(dev_ptr, host_ptr, sizeof(STATE), hipMemcpyHostToDevice), "store_state"); \
        });                                                                                             \
    }                                                                                                   \
    extern "C" void* alloc_program_##suffix(void* device_arg, size_t size) {                            \
        suffix##_handle* h = nullptr;                                                                   \
        hz::capi::guarded([&] {                                                                         \
            if (device_arg == nullptr) throw std::invalid_argument("alloc_program: null device state");  \
            STATE s;                                                                                    \
            hz::capi::check(hipMemcpy(&s, device_arg, sizeof(STATE), hipMemcpyDeviceToHost), "state read"); \
            h = new suffix##_handle(s, size, device_arg);                                               \
        });                                                                                             \
        return h;                                                                                       \
    }                                                                                                   \
    extern "C" void free_program_##suffix(void* instance_ptr) {                                         \
        hz::capi::guarded([&] { delete (suffix##_handle*)instance_ptr; });                              \
    }                                                                                                   \
    extern "C" void init_program_##suffix(void* instance_ptr, size_t grid_size) {                       \
        hz::capi::guarded([&] {                                                                         \
            auto h = (suffix##_handle*)instance_ptr;                                                    \
            init<PROG>(h->inst, grid_size);                                                             \
            hz::capi::check(hipDeviceSynchronize(), "init_program");                                    \
        });                                                                                             \
    }                                                                                                   \
    extern "C" void exec_program_##suffix(void* instance_ptr, size_t grid_size, size_t cycle_count) {   \
        hz::capi::guarded([&] {                                                                         \
            auto h = (suffix##_handle*)instance_ptr;                                                    \
            h->refresh();                                                                               \
            exec<PROG>(h->inst, grid_size, cycle_count);                                                \
            hz::capi::check(hipGetLastError(), "exec_program launch");                                  \
            hz::capi::check(hipDeviceSynchronize(), "exec_program");                                    \
        });                                                                                             \
    }                                                                                                   \
    extern "C" void init_program_on_##suffix(void* instance_ptr, size_t grid_size, void* stream) {       \
        hz::capi::guarded([&] {                                                                         \
            auto h = (suffix##_handle*)instance_ptr;                                                    \
            h->refresh();                                                                               \
            init<PROG>(h->inst, grid_size, (hipStream_t)stream);                                        \
            hz::capi::check(hipGetLastError(), "init_program launch");                                  \
        });                                                                                             \
    }                                                                                                   \
    extern "C" void exec_program_on_##suffix(void* instance_ptr, size_t grid_size, size_t cycle_count,  \
                                             void* stream) {                                            \
        hz::capi::guarded([&] {                                                                         \
            auto h = (suffix##_handle*)instance_ptr;                                                    \
            exec<PROG>(h->inst, grid_size, cycle_count, (hipStream_t)stream);                           \
            hz::capi::check(hipGetLastError(), "exec_program launch");                                  \
        });                                                                                             \
    }                                                                                                   \
    extern "C" int complete_##suffix(void* instance_ptr) {                                              \
        int result = -1;                                                                                \
        hz::capi::guarded([&] { result = ((suffix##_handle*)instance_ptr)->inst.complete() ? 1 : 0; });  \
        return result;                                                                                  \
    }                                                                                                   \
    extern "C" void clear_flags_##suffix(void* instance_ptr) {                                          \
        hz::capi::guarded([&] { ((suffix##_handle*)instance_ptr)->inst.clear_flags(); });               \
    }                                                                                                   \
    extern "C" void set_device_##suffix(int device) {                                                   \
        hz::capi::guarded([&] { hz::capi::check(hipSetDevice(device), "hipSetDevice"); });              \
    }
