// Workspaces of the run entry points: the program instance, claim iterator,
// events and status buffer that one hz_*_run call needs.
//
// Allocating them cost each call eight to twelve hipMallocs and as many
// hipFrees, 0.35-0.45 ms in all (more than 1,024 Collatz starts take), and now
// and then milliseconds where the driver had mappings to clean up. A call that
// ends well therefore leaves its workspace for the next call of its kind and
// sizes on its device. A call owns its workspace alone while it runs, so
// calls of several threads each have one; it is cleared by kernels before
// use. Idle workspaces hold at most IDLE_BYTES over all devices, the ones
// idle longest are freed first, all of them when a device allocation of this
// library fails (util::host::device_malloc) or on hz_workspace_release(); a
// call that failed frees its own. An object that keeps a workspace for its own
// calls (a BFS batch) leaves it on the same shelf, so that it too is freed
// when memory runs short, but beside the bound.
#pragma once

#include <exception>
#include <memory>

#include "common.h"

namespace hz {
namespace capi {

constexpr uint64_t IDLE_BYTES = 1ull << 30;

struct Workspace {
    virtual ~Workspace() = default;
};

// An idle workspace of this kind and these sizes on the current device, or null.
std::unique_ptr<Workspace> workspace_take(const void* kind, uint64_t a, uint64_t b);
// Keeps a workspace for later calls (or frees it, or others, at the bound).
void workspace_give(const void* kind, uint64_t a, uint64_t b, uint64_t bytes, std::unique_ptr<Workspace> w) noexcept;
// Keeps a workspace for the object that `b` names, beside the bound.
void workspace_keep(const void* kind, uint64_t a, uint64_t b, std::unique_ptr<Workspace> w) noexcept;
// Frees the idle workspaces of a kind that are kept for the object `b`.
void workspace_drop(const void* kind, uint64_t b) noexcept;
// Frees every idle workspace; returns how many there were.
size_t workspace_release();

// A workspace W for the duration of one call. W is built from (a, b), its
// sizes, and says how many device bytes it holds (bytes()).
template <typename W>
class Lease {
   public:
    Lease(uint64_t a, uint64_t b) : a_(a), b_(b), exceptions_(std::uncaught_exceptions()) {
        w_.reset(static_cast<W*>(workspace_take(&KIND, a, b).release()));
        if (w_) return;
        try {
            w_ = std::make_unique<W>(a, b);
        } catch (const std::exception&) {
            // Host memory, events: freeing idle workspaces may help there too.
            (void)hipGetLastError();
            if (workspace_release() == 0) throw;
            w_ = std::make_unique<W>(a, b);
        }
    }
    ~Lease() {
        if (std::uncaught_exceptions() > exceptions_) return;  // the call failed: free it
        const uint64_t bytes = w_->bytes();
        workspace_give(&KIND, a_, b_, bytes, std::move(w_));
    }
    Lease(const Lease&) = delete;
    Lease& operator=(const Lease&) = delete;
    W* operator->() const { return w_.get(); }
    W& operator*() const { return *w_; }

   private:
    static inline const char KIND = 0;  // its address names W
    uint64_t a_, b_;
    int exceptions_;
    std::unique_ptr<W> w_;
};

// Device memory carved by the caller.
struct Scratch : Workspace {
    unsigned char* p = nullptr;
    uint64_t size;
    Scratch(uint64_t bytes, uint64_t) : size(bytes ? bytes : 1) { check(util::host::device_malloc((void**)&p, size), "hipMalloc(scratch)"); }
    ~Scratch() override {
        if (p) (void)hipFree(p);
    }
    uint64_t bytes() const { return size; }
};

// Page-locked host memory of one T.
template <typename T>
struct HostCell {
    T* p = nullptr;
    HostCell() { check(hipHostMalloc((void**)&p, sizeof(T), hipHostMallocDefault), "hipHostMalloc"); }
    ~HostCell() {
        if (p) (void)hipHostFree(p);
    }
    HostCell(const HostCell&) = delete;
    HostCell& operator=(const HostCell&) = delete;
};

// Sets *it to [0, limit) with a kernel on the null stream.
void launch_set_iter(util::iter::AtomicIter<unsigned int>* it, unsigned int limit);

// What both program types need beside their instance.
struct RunParts {
    DeviceIter iter{0u};
    EventTimer timer;

    // Sets the claim iterator to [0, limit), in stream order.
    util::iter::AtomicIter<unsigned int>* set_iter(unsigned int limit) {
        launch_set_iter(iter.ptr, limit);
        return iter.ptr;
    }
};

// An AsyncProgram run: sizes are the arena's links and the queue count.
template <typename P>
struct AsyncSpace : Workspace {
    typename P::Instance inst;
    RunParts parts;
    HostCell<AsyncStatus> status;

    AsyncSpace(uint64_t arena, uint64_t queues) : inst(arena, typename P::DeviceState{}, (unsigned int)queues) {}
    uint64_t bytes() const {
        return 4ull * (inst.arena.size() + inst.queue_slots.size() + inst.free_slots.size() + inst.link_meta.size() +
                       inst.link_aux.size());
    }

    // Prepares the instance for a run of `state`, in stream order.
    void begin(const typename P::DeviceState& state, const hz_run_config& cfg, uint32_t groups) {
        inst.device_state = state;
        const uint32_t coalesce = cfg.coalesce ? cfg.coalesce : 64u;
        inst.coalesce = coalesce > 64u ? 64u : coalesce;
        init<P>(inst, groups);
    }

    // Runs the instance to completion: exec launches until it is complete.
    // With HZ_RUN_AUDIT, its queues and arena are audited after every launch
    // (Instance::audit) and the number of audits is reported.
    void run(uint32_t groups, const hz_run_config& cfg, hz_run_stats* stats, bool barriers = false) {
        const uint32_t cycles = cfg.cycles ? cfg.cycles : (1u << 24);
        uint64_t launches = 0;
        uint64_t last_progress = ~0ull;
        uint32_t audits = 0;
        parts.timer.start();
        while (true) {
            if (cfg.max_launches && launches >= cfg.max_launches) {
                throw std::runtime_error("AsyncProgram: launch bound reached before completion");
            }
            exec<P>(inst, groups, cycles);
            check(hipGetLastError(), "exec launch");
            parts.timer.mark();
            check(hipMemcpyAsync(status.p, inst.status.data(), sizeof(AsyncStatus), hipMemcpyDeviceToHost, nullptr),
                  "status copy");
            check(hipStreamSynchronize(nullptr), "exec");
            launches++;
            const bool done = P::status_complete(*status.p);  // raises on a runtime error first
            if (cfg.flags & HZ_RUN_AUDIT) {
                AsyncCensus c = inst.audit(barriers);
                audits++;
                if (done && (c.queued_links != 0 || c.held_links != 0)) {
                    throw std::runtime_error("AsyncProgram audit: complete with links still queued or held");
                }
            }
            if (done) break;
            // A launch that evaluated no promise signals lost accounting rather
            // than unfinished work: report it instead of looping.
            if (status.p->promises == last_progress) {
                throw std::runtime_error("AsyncProgram: a launch made no progress before completion");
            }
            last_progress = status.p->promises;
        }
        if (stats) {
            const AsyncStatus& s = *status.p;
            stats->promises = s.promises;
            stats->launches = launches;
            stats->spills = s.spills;
            stats->fills = s.fills;
            stats->make_work_calls = s.make_work_calls;
            stats->groups = (uint32_t)(blocks_for<P>(groups) * (P::WORK_GROUP_SIZE / 64));
            stats->elapsed_ms = parts.timer.elapsed();
            for (int i = 0; i < 8; ++i) stats->phase_cycles[i] = s.phase_cycles[i];
            stats->links_run = s.links_run;
            stats->forwarded = s.forwarded;
            stats->audits = audits;
            stats->arena_links = s.claim < inst.arena_size ? s.claim : inst.arena_size;
        }
    }
};

// An EventProgram run: its size is the queue capacity per operation.
template <typename P>
struct EventSpace : Workspace {
    typename P::Instance inst;
    RunParts parts;
    HostCell<typename P::Header> header;

    EventSpace(uint64_t io, uint64_t) : inst(io, typename P::DeviceState{}) {}
    uint64_t bytes() const { return 4ull * (inst.queue_a.size() + inst.queue_b.size()); }

    // Runs the program of `state`, its iterator set, generation by generation,
    // on the caller's number of groups or on up to `groups` of them.
    void run(const typename P::DeviceState& state, uint32_t groups, uint32_t chunk, const hz_run_config& cfg,
             hz_run_stats* stats) {
        inst.device_state = state;
        inst.reset(nullptr);
        parts.timer.start();
        const uint64_t launches =
            run_generations<P>(inst, groups, cfg.groups == 0, chunk, cfg.max_launches ? cfg.max_launches : 1u << 24,
                               nullptr, header.p);
        parts.timer.mark();
        if (stats) {
            auto s = inst.read_status();
            stats->promises = s.promises;
            stats->launches = launches;
            stats->make_work_calls = s.make_work_calls;
            stats->groups = groups;
            stats->elapsed_ms = parts.timer.elapsed();
        }
    }
};

}  // namespace capi
}  // namespace hz
