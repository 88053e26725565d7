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
    uint64_t bytes;
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
    while (s.bytes > IDLE_BYTES) {
        s.bytes -= s.idle.back().bytes;
        old.splice(old.begin(), s.idle, std::prev(s.idle.end()));
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
