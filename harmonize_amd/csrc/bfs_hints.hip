// The programs of a BFS batch that look levels up through hints
// (hz_bfs_batch::through_hints).
#include "bfs_batch.h"

template std::unique_ptr<hz::bfs::Runner> hz::bfs::make_async_runner<true>(hz_bfs_batch&, const hz_run_config&);
template void hz::bfs::run_event<hz::bfs::EventOf<true>>(hz_bfs_batch&, const hz_run_config&, hz_run_stats*);
