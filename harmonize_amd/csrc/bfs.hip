// Batched BFS of the C ABI: R-MAT graphs generated and turned into int32 CSR
// on the device, and one AsyncProgram (or EventProgram) that runs the BFS of
// every graph of the batch at once, optionally through a captured hipGraph.
#include <hipcub/hipcub.hpp>

#include <cmath>
#include <memory>
#include <vector>

#include "bfs_batch.h"
#include "rmat.h"

using BfsAsync1 = AsyncProgram<BfsSpecT<1>>;
using BfsEvent = EventProgram<BfsSpecT<1>>;

static_assert(sizeof(BfsJob) == 32, "BfsJob layout");
static_assert(sizeof(hz_bfs_state) == sizeof(BfsState), "C and C++ BFS states must match");
static_assert(HZ_BFS_MAX_SPLIT == BFS_MAX_SPLIT, "C and C++ split limits must match");

HZ_DEFINE_PROGRAM_ABI(bfs_event, BfsEvent, BfsState)
HZ_DEFINE_PROGRAM_ABI(bfs_async, BfsAsync1, BfsState)

using hz::capi::check;
using hz::capi::guarded;

using hz::graph::grid_for;
using hz::graph::row_ptr_kernel;
using hz::graph::rmat_edges_kernel;

using namespace hz::bfs;

template std::unique_ptr<Runner> hz::bfs::make_async_runner<false>(hz_bfs_batch&, const hz_run_config&);
template void hz::bfs::run_event<EventOf<false>>(hz_bfs_batch&, const hz_run_config&, hz_run_stats*);

void hz_bfs_batch::release_event_space() noexcept {
    hz::capi::workspace_drop(&EVENT_SPACE<EventOf<false>>, (uint64_t)this);
    hz::capi::workspace_drop(&EVENT_SPACE<EventOf<true>>, (uint64_t)this);
}

namespace {

std::vector<uint64_t> runner_key(const hz_run_config& c) {
    return {c.groups, c.cycles, c.arena, c.queues, c.coalesce, c.max_launches, c.block_groups, c.flags, c.spec_param,
            c.stash};
}

void check_batch(const hz_bfs_batch* b) {
    if (!b) throw std::invalid_argument("hz_bfs: null batch");
}

}  // namespace

extern "C" int hz_bfs_batch_sizes(uint64_t seed, uint32_t graphs, double min_log2, double max_log2,
                                  uint32_t* vertices) {
    return guarded([&] {
        if (graphs && !vertices) throw std::invalid_argument("hz_bfs_batch_sizes: null output");
        if (!(min_log2 >= 0.0 && max_log2 >= min_log2 && max_log2 <= 30.0)) {
            throw std::invalid_argument("hz_bfs_batch_sizes: need 0 <= min_log2 <= max_log2 <= 30");
        }
        for (uint32_t g = 0; g < graphs; ++g) {
            uint32_t bits = hz::rmat::size_bits(g, (uint32_t)seed, (uint32_t)(seed >> 32));
            double u = (double)bits * (1.0 / 4294967296.0);
            double v = std::nearbyint(std::exp2(min_log2 + (max_log2 - min_log2) * u));
            vertices[g] = v < 1.0 ? 1u : (uint32_t)v;
        }
    });
}

extern "C" int hz_bfs_batch_create(uint64_t seed, uint32_t graphs, const uint32_t* vertices, uint32_t edge_factor,
                                   hz_bfs_batch** out) {
    return guarded([&] {
        if (!out || (graphs && !vertices)) throw std::invalid_argument("hz_bfs_batch_create: null argument");
        *out = nullptr;
        if (graphs == 0) throw std::invalid_argument("hz_bfs_batch_create: no graphs");
        auto b = std::make_unique<hz_bfs_batch>();
        b->graphs = graphs;
        std::vector<uint64_t> edges(graphs);
        for (uint32_t g = 0; g < graphs; ++g) {
            if (vertices[g] == 0) throw std::invalid_argument("hz_bfs_batch_create: a graph has no vertices");
            edges[g] = (uint64_t)edge_factor * vertices[g];
        }
        b->layout(vertices, edges.data(), nullptr);

        uint64_t max_e = 0;
        for (uint64_t e : edges) max_e = e > max_e ? e : max_e;
        DeviceBytes src_in(max_e * 4), dst_in(max_e * 4), src_out(max_e * 4);
        size_t temp_bytes = 0;
        check(hipcub::DeviceRadixSort::SortPairs(nullptr, temp_bytes, src_in.as<uint32_t>(), src_out.as<uint32_t>(),
                                                 dst_in.as<uint32_t>(), b->col.as<uint32_t>(), (int)max_e, 0, 32,
                                                 b->stream),
              "radix sort sizing");
        DeviceBytes temp(temp_bytes);
        StreamTimer t(b->stream);
        t.start();
        for (uint32_t g = 0; g < graphs; ++g) {
            uint32_t V = vertices[g];
            uint32_t E = (uint32_t)edges[g];
            uint32_t scale = hz::rmat::scale_of(V);
            int32_t* rows = b->row_ptr.as<int32_t>() + b->row_base[g];
            if (E > 0) {
                hipLaunchKernelGGL(rmat_edges_kernel, dim3(grid_for(E)), dim3(256), 0, b->stream, g, E, V, scale,
                                   (uint32_t)seed, (uint32_t)(seed >> 32), src_in.as<uint32_t>(),
                                   dst_in.as<uint32_t>());
                check(hipGetLastError(), "rmat launch");
                size_t tb = temp_bytes;
                check(hipcub::DeviceRadixSort::SortPairs(temp.p, tb, src_in.as<uint32_t>(), src_out.as<uint32_t>(),
                                                         dst_in.as<uint32_t>(),
                                                         b->col.as<uint32_t>() + b->edge_base[g], (int)E, 0,
                                                         scale > 0 ? (int)scale : 1, b->stream),
                      "radix sort");
            }
            hipLaunchKernelGGL(row_ptr_kernel, dim3(grid_for((uint64_t)V + 1)), dim3(256), 0, b->stream,
                               src_out.as<uint32_t>(), E, V, rows);
            check(hipGetLastError(), "row_ptr launch");
        }
        b->build_ms = t.stop();
        b->write_jobs();
        *out = b.release();
    });
}

extern "C" int hz_bfs_batch_from_csr(uint32_t graphs, const uint32_t* vertices, const uint64_t* edges,
                                     const int32_t* row_ptr, const int32_t* col, const uint32_t* sources,
                                     hz_bfs_batch** out) {
    return guarded([&] {
        if (!out || !vertices || !edges || !row_ptr) throw std::invalid_argument("hz_bfs_batch_from_csr: null argument");
        *out = nullptr;
        if (graphs == 0) throw std::invalid_argument("hz_bfs_batch_from_csr: no graphs");
        auto b = std::make_unique<hz_bfs_batch>();
        b->graphs = graphs;
        b->layout(vertices, edges, sources);
        if (b->total_edges && !col) throw std::invalid_argument("hz_bfs_batch_from_csr: null col");
        // Validate the CSR on the host before any kernel reads it.
        for (uint32_t g = 0; g < graphs; ++g) {
            const int32_t* rows = row_ptr + b->row_base[g];
            const int32_t* cols = col + b->edge_base[g];
            if (rows[0] != 0 || (uint64_t)rows[vertices[g]] != edges[g]) {
                throw std::invalid_argument("hz_bfs_batch_from_csr: row_ptr does not span the edges");
            }
            for (uint32_t v = 0; v < vertices[g]; ++v) {
                if (rows[v] > rows[v + 1]) throw std::invalid_argument("hz_bfs_batch_from_csr: row_ptr decreases");
            }
            for (uint64_t i = 0; i < edges[g]; ++i) {
                if (cols[i] < 0 || (uint32_t)cols[i] >= vertices[g]) {
                    throw std::invalid_argument("hz_bfs_batch_from_csr: column index out of range");
                }
            }
        }
        check(hipMemcpy(b->row_ptr.p, row_ptr, (b->total_vertices + graphs) * 4, hipMemcpyHostToDevice), "row_ptr");
        if (b->total_edges) check(hipMemcpy(b->col.p, col, b->total_edges * 4, hipMemcpyHostToDevice), "col");
        b->write_jobs();
        *out = b.release();
    });
}

extern "C" int hz_bfs_batch_destroy(hz_bfs_batch* batch) {
    return guarded([&] { delete batch; });
}

extern "C" int hz_bfs_batch_info(const hz_bfs_batch* batch, hz_bfs_info* info) {
    return guarded([&] {
        check_batch(batch);
        if (!info) throw std::invalid_argument("hz_bfs_batch_info: null output");
        std::memset(info, 0, sizeof(*info));
        info->graphs = batch->graphs;
        info->total_vertices = batch->total_vertices;
        info->total_edges = batch->total_edges;
        info->d_row_ptr = batch->row_ptr.as<int32_t>();
        info->d_col = batch->col.as<int32_t>();
        info->d_level = batch->level.as<int32_t>();
        info->build_ms = batch->build_ms;
    });
}

extern "C" int hz_bfs_batch_layout(const hz_bfs_batch* batch, uint32_t* vertices, uint64_t* edges,
                                   uint64_t* vertex_base, uint64_t* edge_base, uint64_t* row_base) {
    return guarded([&] {
        check_batch(batch);
        for (uint32_t g = 0; g < batch->graphs; ++g) {
            if (vertices) vertices[g] = batch->vertices[g];
            if (edges) edges[g] = batch->edges[g];
            if (vertex_base) vertex_base[g] = batch->vertex_base[g];
            if (edge_base) edge_base[g] = batch->edge_base[g];
            if (row_base) row_base[g] = batch->row_base[g];
        }
    });
}

extern "C" int hz_bfs_batch_run(hz_bfs_batch* batch, int kind, const hz_run_config* config, hz_run_stats* stats) {
    return guarded([&] {
        hz_run_config c{};
        if (config) c = *config;
        if (stats) std::memset(stats, 0, sizeof(*stats));
        if (c.spec_param > BFS_MAX_SPLIT) {
            throw std::invalid_argument("hz_bfs_batch_run: the split threshold (spec_param) must be in [1, 2^24] "
                                        "(0 = default 64)");
        }
        check_batch(batch);
        if (kind == HZ_EVENT) {
            if (c.flags & HZ_RUN_GRAPH) throw std::invalid_argument("hz_bfs_batch_run: graph launch is for HZ_ASYNC");
            if (batch->through_hints(false, c.flags)) {
                batch->need_hints();
                run_event<EventOf<true>>(*batch, c, stats);
            } else {
                run_event<EventOf<false>>(*batch, c, stats);
            }
        } else if (kind == HZ_ASYNC) {
            auto key = runner_key(c);
            auto it = batch->runners.find(key);
            if (it == batch->runners.end()) {
                std::unique_ptr<Runner> made;
                auto make = [&] {
                    if (!batch->through_hints(true, c.flags)) return make_async_runner<false>(*batch, c);
                    batch->need_hints();
                    return make_async_runner<true>(*batch, c);
                };
                try {
                    made = make();
                } catch (const std::invalid_argument&) {
                    throw;
                } catch (const std::exception&) {
                    // Room taken by what earlier runs left behind.
                    (void)hipGetLastError();
                    if (hz::capi::workspace_release() == 0) throw;
                    made = make();
                }
                it = batch->runners.emplace(key, std::move(made)).first;
            }
            it->second->run(stats, (c.flags & HZ_RUN_AUDIT) != 0);
        } else {
            throw std::invalid_argument("hz_bfs_batch_run: kind must be HZ_EVENT or HZ_ASYNC");
        }
    });
}

extern "C" int hz_bfs_batch_release(hz_bfs_batch* batch) {
    return guarded([&] {
        check_batch(batch);
        batch->runners.clear();
        batch->release_event_space();
    });
}
