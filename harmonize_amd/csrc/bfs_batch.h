// A batch of BFS jobs (hz_bfs_batch_*) and the programs that search it: its
// graphs on the device, the AsyncProgram instances and hipGraphs it keeps by
// configuration, and the run of its EventProgram.
#pragma once

#include <map>
#include <memory>
#include <tuple>
#include <vector>

#include "workspace.h"
#include "bfs.h"
#include "graph.h"

namespace hz {
namespace bfs {

using hz::capi::check;
using hz::graph::bfs_reset_kernel;
using hz::graph::grid_for;

struct DeviceBytes {
    void* p = nullptr;
    DeviceBytes() = default;
    explicit DeviceBytes(size_t bytes) { check(util::host::device_malloc(&p, bytes ? bytes : 1), "hipMalloc(bfs)"); }
    ~DeviceBytes() {
        if (p) (void)hipFree(p);
    }
    DeviceBytes(const DeviceBytes&) = delete;
    DeviceBytes& operator=(const DeviceBytes&) = delete;
    DeviceBytes(DeviceBytes&& o) noexcept : p(o.p) { o.p = nullptr; }
    DeviceBytes& operator=(DeviceBytes&& o) noexcept {
        std::swap(p, o.p);
        return *this;
    }
    template <typename T>
    T* as() const {
        return (T*)p;
    }
};

// hipEvent timing on one stream.
struct StreamTimer {
    hipEvent_t a{}, b{};
    hipStream_t s;
    explicit StreamTimer(hipStream_t stream) : s(stream) {
        check(hipEventCreate(&a), "hipEventCreate");
        check(hipEventCreate(&b), "hipEventCreate");
    }
    ~StreamTimer() {
        (void)hipEventDestroy(a);
        (void)hipEventDestroy(b);
    }
    void start() { check(hipEventRecord(a, s), "hipEventRecord"); }
    double stop() {
        check(hipEventRecord(b, s), "hipEventRecord");
        check(hipEventSynchronize(b), "hipEventSynchronize");
        float ms = 0;
        check(hipEventElapsedTime(&ms, a, b), "hipEventElapsedTime");
        return ms;
    }
};

struct Runner {
    virtual ~Runner() = default;
    // audit: check the queues and arena on the host after every launch.
    virtual void run(hz_run_stats* stats, bool audit) = 0;
};

}  // namespace bfs
}  // namespace hz

struct hz_bfs_batch {
    using DeviceBytes = hz::bfs::DeviceBytes;
    uint32_t graphs = 0;
    std::vector<uint32_t> vertices, sources;
    std::vector<uint64_t> edges, vertex_base, edge_base, row_base;
    uint64_t total_vertices = 0, total_edges = 0;
    DeviceBytes row_ptr, col, level, jobs, hints;
    std::unique_ptr<hz::capi::DeviceIter> iter;
    hipStream_t stream = nullptr;
    double build_ms = 0.0;
    std::map<std::vector<uint64_t>, std::unique_ptr<hz::bfs::Runner>> runners;

    ~hz_bfs_batch() {
        runners.clear();
        release_event_space();
        if (stream) (void)hipStreamDestroy(stream);
    }

    void release_event_space() noexcept;

    void layout(const uint32_t* v, const uint64_t* e, const uint32_t* src) {
        vertices.assign(v, v + graphs);
        edges.assign(e, e + graphs);
        sources.resize(graphs);
        vertex_base.resize(graphs);
        edge_base.resize(graphs);
        row_base.resize(graphs);
        uint64_t vb = 0, eb = 0;
        for (uint32_t g = 0; g < graphs; ++g) {
            if (edges[g] > 0x7FFFFFFFull) throw std::invalid_argument("hz_bfs: a graph has 2^31 or more edges");
            if (vertices[g] > 0x7FFFFFFEu) throw std::invalid_argument("hz_bfs: a graph has too many vertices");
            sources[g] = src ? src[g] : 0u;
            vertex_base[g] = vb;
            row_base[g] = vb + g;
            edge_base[g] = eb;
            vb += vertices[g];
            eb += edges[g];
        }
        total_vertices = vb;
        total_edges = eb;
        row_ptr = DeviceBytes((total_vertices + graphs) * sizeof(int32_t));
        col = DeviceBytes(total_edges * sizeof(int32_t));
        level = DeviceBytes(total_vertices * sizeof(int32_t));
        jobs = DeviceBytes(graphs * sizeof(BfsJob));
        iter = std::make_unique<hz::capi::DeviceIter>(graphs);
        hz::capi::check(hipStreamCreate(&stream), "hipStreamCreate");
    }

    void write_jobs() {
        std::vector<BfsJob> host(graphs);
        for (uint32_t g = 0; g < graphs; ++g) {
            host[g].row_ptr = row_ptr.as<int32_t>() + row_base[g];
            host[g].col = col.as<int32_t>() + edge_base[g];
            host[g].level = level.as<int32_t>() + vertex_base[g];
            host[g].vertices = vertices[g];
            host[g].source = sources[g];
        }
        hz::capi::check(hipMemcpy(jobs.p, host.data(), graphs * sizeof(BfsJob), hipMemcpyHostToDevice), "jobs upload");
    }

    // Whether a run of this kind looks levels up through hints. They cost a
    // look of their own at each edge, and pay where the levels are fetched
    // from beyond the caches often enough: where there are many and each is
    // looked at often. Measured with / without, in ms, R-MAT graphs of 2^18 to
    // 2^26 vertices with 4 to 64 edges each: EventProgram below 2^28 edges
    // 0.93..2.11 / 0.84..1.96 (grids, rings, paths: 25.1 / 23.2, 21.1 / 19.2,
    // 17.9 / 17.2), at 2^28 edges 4.96 / 5.23, 5.34 / 5.23, 5.17 / 5.84, above
    // it 9.30 / 12.4, 18.4 / 26.0. AsyncProgram, which has fewer looks in
    // flight, at 2^28 edges 7.86 / 7.48, 6.91 / 6.80, 9.99 / 8.93; above 2^29
    // edges 22.7 / 24.2, 24.2 / 26.6 and on 2^29 12.95 / 13.7, 11.9 / 12.7, but
    // with 2^23 vertices (whose levels fit the caches) 9.47 / 8.59. Grids and
    // the like 15.3 / 13.7, 17.7 / 14.7, 8.90 / 8.14.
    bool through_hints(bool async, uint32_t flags) const {
        if (flags & HZ_RUN_LEVEL_HINTS) return true;
        return async ? total_edges >= (1ull << 29) && total_vertices >= (1ull << 24) : total_edges >= (1ull << 28);
    }

    void need_hints() {
        if (hints.p == nullptr) hints = DeviceBytes((total_vertices + 7) / 8 * 4);
    }

    template <typename STATE>
    STATE state(uint32_t split) const {
        STATE s{};
        if constexpr (STATE::HINTS) {
            s.hints = hints.as<unsigned char>();
            s.level_base = level.as<int32_t>();
        }
        s.jobs = jobs.as<BfsJob>();
        s.job_iter = iter->ptr;
        s.job_count = graphs;
        s.split = split ? split : BFS_DEFAULT_SPLIT;
        return s;
    }

    void enqueue_reset(bool with_hints) {
        hipLaunchKernelGGL(hz::graph::bfs_reset_kernel, dim3(hz::graph::grid_for(total_vertices)), dim3(256), 0,
                           stream, level.as<int32_t>(), total_vertices, iter->ptr, graphs,
                           with_hints ? hints.as<uint32_t>() : nullptr);
    }
};

namespace hz {
namespace bfs {

inline uint32_t default_split(const hz_run_config& c) { return c.spec_param ? c.spec_param : BFS_DEFAULT_SPLIT; }

// Arena links for a batch: room for one visit per vertex and one edge-range
// promise per `split` edges at once, twice over, within [2^16, 2^26] links.
inline uint64_t default_arena(const hz_bfs_batch& b, uint32_t split) {
    uint64_t promises = b.total_vertices + b.total_edges / split + b.graphs;
    uint64_t links = 2 * ((promises + 63) / 64);
    if (links < (1ull << 16)) links = 1ull << 16;
    if (links > (1ull << 26)) links = 1ull << 26;
    return links;
}

template <typename P>
struct AsyncRunner : Runner {
    hz_bfs_batch& b;
    typename P::Instance inst;
    uint32_t groups, cycles, max_launches;
    hipGraphExec_t graph_exec = nullptr;

    AsyncRunner(hz_bfs_batch& batch, const hz_run_config& c)
        : b(batch),
          inst(c.arena ? c.arena : default_arena(batch, default_split(c)), batch.state<typename P::DeviceState>(default_split(c)), c.queues,
               c.coalesce ? c.coalesce : 64u),
          groups(c.groups ? c.groups : (uint32_t)hz::capi::resident_groups_of<P>()),
          cycles(c.cycles ? c.cycles : (1u << 24)),
          max_launches(c.max_launches) {
        if (c.flags & HZ_RUN_GRAPH) {
            hipGraph_t graph = nullptr;
            check(hipStreamBeginCapture(b.stream, hipStreamCaptureModeThreadLocal), "hipStreamBeginCapture");
            enqueue_pass();
            check(hipStreamEndCapture(b.stream, &graph), "hipStreamEndCapture");
            hipError_t e = hipGraphInstantiate(&graph_exec, graph, nullptr, nullptr, 0);
            (void)hipGraphDestroy(graph);
            check(e, "hipGraphInstantiate");
        }
    }
    ~AsyncRunner() override {
        if (graph_exec) (void)hipGraphExecDestroy(graph_exec);
    }

    // Reset of levels, jobs and queues, then the first exec launch.
    void enqueue_pass() {
        b.enqueue_reset(P::DeviceState::HINTS);
        init<P>(inst, groups, b.stream);
        exec<P>(inst, groups, cycles, b.stream);
    }

    void run(hz_run_stats* stats, bool audit) override {
        StreamTimer t(b.stream);
        t.start();
        if (graph_exec) {
            check(hipGraphLaunch(graph_exec, b.stream), "hipGraphLaunch");
        } else {
            enqueue_pass();
        }
        check(hipGetLastError(), "bfs launch");
        check(hipStreamSynchronize(b.stream), "bfs exec");
        uint64_t launches = 1, last = ~0ull;
        uint32_t audits = 0;
        auto audit_now = [&] {
            if (!audit) return;
            const bool done = inst.complete();  // raises on a runtime error first
            hz::AsyncCensus c = inst.audit(false);
            audits++;
            if (done && c.queued_links != 0) {
                throw std::runtime_error("AsyncProgram audit: complete with links still queued");
            }
        };
        audit_now();
        // A pass that ends early (cycle budget) resumes with plain launches.
        while (!inst.complete()) {
            if (max_launches && launches >= max_launches) {
                throw std::runtime_error("AsyncProgram: launch bound reached before completion");
            }
            uint64_t progress = inst.read_status().promises;
            if (progress == last) throw std::runtime_error("AsyncProgram: a launch made no progress");
            last = progress;
            exec<P>(inst, groups, cycles, b.stream);
            check(hipGetLastError(), "bfs relaunch");
            check(hipStreamSynchronize(b.stream), "bfs exec");
            launches++;
            audit_now();
        }
        double ms = t.stop();
        if (stats) {
            hz::AsyncStatus s = inst.read_status();
            std::memset(stats, 0, sizeof(*stats));
            stats->promises = s.promises;
            stats->launches = launches;
            stats->spills = s.spills;
            stats->fills = s.fills;
            stats->make_work_calls = s.make_work_calls;
            stats->groups = (uint32_t)(blocks_for<P>(groups) * (P::WORK_GROUP_SIZE / 64));
            stats->elapsed_ms = ms;
            for (int i = 0; i < 8; ++i) stats->phase_cycles[i] = s.phase_cycles[i];
            stats->links_run = s.links_run;
            stats->forwarded = s.forwarded;
            stats->audits = audits;
            stats->arena_links = s.claim < inst.arena_size ? s.claim : inst.arena_size;
        }
    }
};

// EventProgram's instance and header, kept by the batch between its searches:
// the queues hold gigabytes for a large batch, which cost 1.5 ms or, after an
// idle spell, a hundred to allocate and free on every search. A batch keeps up
// to KEPT_BYTES; idle, they are freed like other workspaces when an allocation
// fails.
constexpr uint64_t KEPT_BYTES = 8ull << 30;
template <typename P>
inline const char EVENT_SPACE = 0;  // its address names the program's kind

template <typename P>
struct EventSpaceHold {
    using Space = hz::capi::EventSpace<P>;
    hz_bfs_batch& b;
    const uint64_t io;
    const int exceptions = std::uncaught_exceptions();
    std::unique_ptr<Space> space;

    EventSpaceHold(hz_bfs_batch& batch, uint64_t size) : b(batch), io(size) {
        space.reset(static_cast<Space*>(hz::capi::workspace_take(&EVENT_SPACE<P>, io, (uint64_t)&b).release()));
        if (space) return;
        b.release_event_space();  // one of another size or program
        try {
            space = std::make_unique<Space>(io, 0);
        } catch (const std::exception&) {
            // Allocations have freed the idle workspaces; the batch's async
            // runners are left.
            if (b.runners.empty()) throw;
            (void)hipGetLastError();
            b.runners.clear();
            space = std::make_unique<Space>(io, 0);
        }
    }
    ~EventSpaceHold() {
        if (std::uncaught_exceptions() > exceptions || space->bytes() > KEPT_BYTES) return;
        hz::capi::workspace_keep(&EVENT_SPACE<P>, io, (uint64_t)&b, std::move(space));
    }
};

template <typename P>
void run_event(hz_bfs_batch& b, const hz_run_config& c, hz_run_stats* stats) {
    uint64_t io = c.arena;
    if (io == 0) {
        uint64_t split = default_split(c);
        io = b.total_vertices + b.total_edges / split + b.graphs;
        if (io < (1ull << 20)) io = 1ull << 20;
        if (io > (1ull << 30)) io = 1ull << 30;
    }
    EventSpaceHold<P> hold(b, io);
    typename P::Instance& inst = hold.space->inst;
    inst.device_state = b.state<typename P::DeviceState>(default_split(c));
    inst.reset(b.stream);
    // 16 groups per CU: measured 22.2 ms on the 64-graph batch against 23.7
    // with 32 per CU and 23.9 with 8 per CU.
    uint32_t groups = c.groups ? c.groups : (uint32_t)(hz::capi::compute_units() * 16);
    uint32_t chunk = c.cycles ? c.cycles : 4u;
    uint32_t max_launches = c.max_launches ? c.max_launches : (1u << 24);
    StreamTimer t(b.stream);
    t.start();
    b.enqueue_reset(P::DeviceState::HINTS);
    const uint64_t launches =
        hz::capi::run_generations<P>(inst, groups, c.groups == 0, chunk, max_launches, b.stream, hold.space->header.p);
    double ms = t.stop();
    if (stats) {
        auto s = inst.read_status();
        std::memset(stats, 0, sizeof(*stats));
        stats->promises = s.promises;
        stats->launches = launches;
        stats->make_work_calls = s.make_work_calls;
        stats->groups = groups;
        stats->elapsed_ms = ms;
    }
}

template <unsigned int STASH, bool HINTS>
std::unique_ptr<Runner> make_async_runner_stash(hz_bfs_batch& b, const hz_run_config& c) {
    switch (c.block_groups) {
        case 0:
        case 1:
            return std::make_unique<AsyncRunner<AsyncProgram<BfsSpecT<1, STASH, HINTS>>>>(b, c);
        case 2:
            return std::make_unique<AsyncRunner<AsyncProgram<BfsSpecT<2, STASH, HINTS>>>>(b, c);
        case 4:
            return std::make_unique<AsyncRunner<AsyncProgram<BfsSpecT<4, STASH, HINTS>>>>(b, c);
        default:
            throw std::invalid_argument("hz_bfs_batch_run: block_groups must be 1, 2 or 4");
    }
}

template <bool HINTS>
std::unique_ptr<Runner> make_async_runner(hz_bfs_batch& b, const hz_run_config& c) {
    switch (c.stash) {
        case 0:
        case 16:
            return make_async_runner_stash<16, HINTS>(b, c);
        case 8:
            return make_async_runner_stash<8, HINTS>(b, c);
        default:
            throw std::invalid_argument("hz_bfs_batch_run: stash must be 8 or 16 links");
    }
}

// A translation unit each: bfs.hip without hints, bfs_hints.hip with them.
template <bool HINTS>
using EventOf = EventProgram<BfsSpecT<1, 16, HINTS>>;
extern template std::unique_ptr<Runner> make_async_runner<false>(hz_bfs_batch&, const hz_run_config&);
extern template std::unique_ptr<Runner> make_async_runner<true>(hz_bfs_batch&, const hz_run_config&);
extern template void run_event<EventOf<false>>(hz_bfs_batch&, const hz_run_config&, hz_run_stats*);
extern template void run_event<EventOf<true>>(hz_bfs_batch&, const hz_run_config&, hz_run_stats*);

}  // namespace bfs
}  // namespace hz
