// Index iterators that specifications use to claim work (reference
// util/iter.h: Iter :13-60, AtomicIter :138-223, ArrayIter :228-314,
// IOBuffer :320-474).
//
// Portable: the including platform layer provides hz_fetch_add (a
// fetch-and-add; on gfx950 it is aggregated across the active lanes of a
// wavefront) and hz_load (a relaxed atomic load).
#pragma once

#include "portable.h"

namespace util {
namespace iter {

template <typename INDEX_TYPE>
struct Iter {
    typedef INDEX_TYPE IndexType;
    IndexType value;
    IndexType limit;

    Iter() = default;
    HZ_HD Iter(IndexType v, IndexType l) : value(v), limit(l) {}

    HZ_HD void reset(IndexType start_val, IndexType limit_val) {
        value = start_val;
        limit = limit_val;
    }

    // Yields the next index, or false once the range is exhausted.
    HZ_HD bool step(IndexType& iter_val) {
        if (value >= limit) return false;
        iter_val = value;
        value += 1;
        return true;
    }

    // Splits off the next `length` indices (fewer at the end of the range).
    HZ_HD Iter<IndexType> leap(IndexType length) {
        IndexType old_value = value;
        IndexType sub_limit = (limit - value > length) ? value + length : limit;
        if (value >= limit) sub_limit = value;
        value = sub_limit;
        return Iter<IndexType>(old_value, sub_limit);
    }

    HZ_HD bool done() const { return value >= limit; }
};

// A range shared by every thread of a program; claims are atomic.
template <typename INDEX_TYPE>
struct AtomicIter {
    typedef INDEX_TYPE IndexType;
    IndexType value;
    IndexType limit;

    AtomicIter() = default;
    HZ_HD AtomicIter(IndexType start_val, IndexType limit_val) : value(start_val), limit(limit_val) {}
    HZ_HD AtomicIter(Iter<IndexType> it) : value(it.value), limit(it.limit) {}
    HZ_HD AtomicIter& operator=(Iter<IndexType> it) {
        value = it.value;
        limit = it.limit;
        return *this;
    }

    // Claims the next `leap_size` indices. Claims past the limit come back empty.
    __device__ Iter<IndexType> leap(IndexType leap_size) {
        IndexType start_val = 0;
        IndexType limit_val = 0;
        IndexType lim = limit;
        if (hz_load(&value) < lim) {
            start_val = hz_fetch_add(&value, leap_size);
            limit_val = start_val + leap_size;
            // guard against wrap of the counter past the top of IndexType
            if (limit_val < start_val) limit_val = lim;
            start_val = (start_val < lim) ? start_val : lim;
            limit_val = (limit_val < lim) ? limit_val : lim;
        }
        return Iter<IndexType>(start_val, limit_val);
    }

    // Claims a single index.
    __device__ bool step(IndexType& iter_val) {
        if (hz_load(&value) >= limit) return false;
        IndexType try_val = hz_fetch_add(&value, (IndexType)1);
        if (try_val >= limit) return false;
        iter_val = try_val;
        return true;
    }

    __device__ bool done() const { return hz_load(&value) >= limit; }

    // The reference's barrier demo calls sync_done(); same meaning as done().
    __device__ bool sync_done() const { return done(); }
};

// A lane's share of a claimed range: next, next + stride, ... below end. No
// index beyond end is formed, so that end may be the type's greatest value.
template <typename INDEX_TYPE>
struct Share {
    INDEX_TYPE next;
    INDEX_TYPE end;
    INDEX_TYPE stride;

    HZ_HD void clear() {
        next = 0;
        end = 0;
        stride = 1;
    }

    HZ_HD bool step(INDEX_TYPE& index) {
        if (next >= end) return false;
        index = next;
        next = end - next > stride ? next + stride : end;
        return true;
    }

    // The share of lane r of n in [first, limit).
    HZ_HD void take(INDEX_TYPE first, INDEX_TYPE limit, INDEX_TYPE r, INDEX_TYPE n) {
        next = first < limit && r < limit - first ? first + r : limit;
        end = limit;
        stride = n;
    }
};

// Gives lanes whose share is used up a new one from `range`.
//
// On the GPU one atomic claims for the whole wavefront: per lane, what is left
// over the launch's lanes, 1 to `most` indices (1 once fewer than `from` are
// left). The range's counter is one address for the whole device, where loads
// and atomics take their turn (30 ns each), so a large range is claimed in
// large parts, and its end, or a small range, one index per lane. The parts
// follow the counter as it is: sized from a wavefront's previous claim
// instead, they leave too much to the last few wavefronts. The lanes take the
// claimed indices in turn, so that a step of every lane reads consecutive
// elements.
template <typename INDEX_TYPE>
__device__ inline void claim_share(Share<INDEX_TYPE>& share, AtomicIter<INDEX_TYPE>& range, INDEX_TYPE most,
                                   INDEX_TYPE from = 0) {
    static_assert(sizeof(INDEX_TYPE) == 4, "claims broadcast 32-bit indices");
#if defined(__HIP_DEVICE_COMPILE__)
    const bool need = share.next >= share.end;
    const uint64_t lanes = hz::wave::ballot(need);
    if (lanes == 0ull) return;
    // The counter only grows, so a copy in the XCD's L2 that has passed the
    // end settles it without a turn at the counter.
    const INDEX_TYPE limit = range.limit;
    if (__hip_atomic_load(&range.value, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP) >= limit) return;
    const INDEX_TYPE at = (INDEX_TYPE)hz::wave::first((uint32_t)hz_load(&range.value));
    if (at >= limit) return;
    const INDEX_TYPE n = (INDEX_TYPE)hz::wave::popc(lanes);
    const INDEX_TYPE r = (INDEX_TYPE)hz::wave::rank(lanes);
    const uint64_t all = (uint64_t)gridDim.x * blockDim.x;
    uint64_t per = (uint64_t)(limit - at) / all;
    per = per > most ? most : per;
    if (per < 1 || limit - at < from) per = 1;
    const INDEX_TYPE total = n * (INDEX_TYPE)per;
    // Claims that add their whole size move the counter past the end, each
    // resident wavefront by at most 64 shares of `most` (17 million for 32 and
    // 8,192 wavefronts). Where that could wrap it, claims stop at the end.
    INDEX_TYPE base = 0;
    if (need && r == 0) {
        base = limit > (INDEX_TYPE)0xF0000000u ? hz::wave::claim_below(&range.value, total, limit)
                                               : hz::wave::atomic_add(&range.value, total);
    }
    base = (INDEX_TYPE)hz::wave::read_lane((uint32_t)base, (uint32_t)__builtin_ctzll(lanes));
    INDEX_TYPE end = base + total;
    if (end < base || end > limit) end = limit;
    if (need) share.take(base, end, r, n);
#else
    (void)most;
    (void)from;
    if (share.next >= share.end) {
        Iter<INDEX_TYPE> it = range.leap((INDEX_TYPE)1);
        share.next = it.value;
        share.end = it.limit;
        share.stride = 1;
    }
#endif
}

template <typename T, template <typename> class ITER_TYPE = Iter, typename INDEX_TYPE = unsigned int>
struct ArrayIter {
    typedef INDEX_TYPE IndexType;
    typedef ITER_TYPE<IndexType> IterType;

    T* array;
    IterType iter;

    ArrayIter() = default;
    HZ_HD ArrayIter(T* adr, IterType other_iter) : array(adr), iter(other_iter) {}

    HZ_HD void reset(T* new_array, IterType new_iter) {
        array = new_array;
        iter = new_iter;
    }

    __device__ bool step_val(T& val) {
        IndexType index;
        if (iter.step(index)) {
            val = array[index];
            return true;
        }
        return false;
    }

    __device__ bool step_idx_val(IndexType& idx, T& val) {
        IndexType index;
        if (iter.step(index)) {
            idx = index;
            val = array[index];
            return true;
        }
        return false;
    }

    __device__ bool step_ptr(T*& val) {
        IndexType index;
        if (iter.step(index)) {
            val = &array[index];
            return true;
        }
        return false;
    }

    __device__ ArrayIter<T, Iter, IndexType> leap(IndexType leap_size) {
        return ArrayIter<T, Iter, IndexType>(array, iter.leap(leap_size));
    }

    __device__ bool done() { return iter.done(); }
};

// The reference's EventProgram queue type. The native EventProgram keeps its
// queues in structure-of-arrays form instead; this type is kept so that
// specifications that name it (as a field type) still compile.
template <typename T, typename INDEX_TYPE = unsigned int>
struct IOBuffer {
    typedef INDEX_TYPE IndexType;
    bool toggle;
    T* data_a;
    T* data_b;
    IndexType capacity;
    AtomicIter<IndexType> input_iter;
    AtomicIter<IndexType> output_iter;
};

}  // namespace iter
}  // namespace util
