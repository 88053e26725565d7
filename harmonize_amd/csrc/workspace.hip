// The idle workspaces of the run entry points (workspace.h).
#include "workspace.h"

#include <list>
#include <mutex>

namespace hz {
namespace capi {

namespace {

struct Idle {
    const void* kind;
    uint64_t a, b;
    int device;
    uint64_t bytes;  // counted against the bound (0: kept for an object)
    std::unique_ptr<Workspace> w;
};

struct Shelf {
    std::mutex mutex;
    std::list<Idle> idle;  // the one left last first
    uint64_t bytes = 0;
};

// Never destroyed: device memory cannot be freed once the process's static
// objects go, and ends with the process.
Shelf& shelf() {
    static Shelf* s = new Shelf;
    return *s;
}

int current_device() {
    int dev = 0;
    check(hipGetDevice(&dev), "hipGetDevice");
    return dev;
}

}  // namespace

std::unique_ptr<Workspace> workspace_take(const void* kind, uint64_t a, uint64_t b) {
    const int dev = current_device();
    Shelf& s = shelf();
    std::lock_guard<std::mutex> lock(s.mutex);
    for (auto it = s.idle.begin(); it != s.idle.end(); ++it) {
        if (it->kind == kind && it->a == a && it->b == b && it->device == dev) {
            std::unique_ptr<Workspace> w = std::move(it->w);
            s.bytes -= it->bytes;
            s.idle.erase(it);
            return w;
        }
    }
    return nullptr;
}

void workspace_give(const void* kind, uint64_t a, uint64_t b, uint64_t bytes, std::unique_ptr<Workspace> w) noexcept {
    int dev = 0;
    if (bytes > IDLE_BYTES || hipGetDevice(&dev) != hipSuccess) return;
    std::list<Idle> old;  // freed after the lock
    Shelf& s = shelf();
    std::lock_guard<std::mutex> lock(s.mutex);
    try {
        s.idle.push_front(Idle{kind, a, b, dev, bytes, std::move(w)});
    } catch (const std::exception&) {
        return;
    }
    s.bytes += bytes;
    for (auto it = s.idle.end(); s.bytes > IDLE_BYTES && it != s.idle.begin();) {
        auto last = std::prev(it);
        if (last->bytes == 0) {
            it = last;
            continue;
        }
        s.bytes -= last->bytes;
        old.splice(old.begin(), s.idle, last);
    }
}

void workspace_keep(const void* kind, uint64_t a, uint64_t b, std::unique_ptr<Workspace> w) noexcept {
    workspace_give(kind, a, b, 0, std::move(w));
}

void workspace_drop(const void* kind, uint64_t b) noexcept {
    std::list<Idle> old;  // freed after the lock
    Shelf& s = shelf();
    std::lock_guard<std::mutex> lock(s.mutex);
    for (auto it = s.idle.begin(); it != s.idle.end();) {
        auto next = std::next(it);
        if (it->kind == kind && it->b == b) {
            s.bytes -= it->bytes;
            old.splice(old.begin(), s.idle, it);
        }
        it = next;
    }
}

size_t workspace_release() {
    std::list<Idle> old;
    {
        Shelf& s = shelf();
        std::lock_guard<std::mutex> lock(s.mutex);
        old.swap(s.idle);
        s.bytes = 0;
    }
    return old.size();
}

namespace {
// Device allocations that fail free the idle workspaces and try again.
const bool hooked = [] {
    util::host::free_idle_memory = [] { return workspace_release() != 0; };
    return true;
}();

__global__ void __launch_bounds__(64) set_iter_kernel(util::iter::AtomicIter<unsigned int>* it, unsigned int limit) {
    if (blockIdx.x == 0 && threadIdx.x == 0) *it = util::iter::AtomicIter<unsigned int>(0u, limit);
}
}  // namespace

void launch_set_iter(util::iter::AtomicIter<unsigned int>* it, unsigned int limit) {
    hipLaunchKernelGGL(set_iter_kernel, dim3(1), dim3(64), 0, nullptr, it, limit);
    check(hipGetLastError(), "set_iter_kernel launch");
}

}  // namespace capi
}  // namespace hz

extern "C" int hz_workspace_release(void) {
    return hz::capi::guarded([] { (void)hz::capi::workspace_release(); });
}
