// Reads a program specification's optional members, falling back to defaults
// when a member is absent. Same contract as the reference's MEMBER_SWITCH /
// CONST_SWITCH (program/async.h:26-36, 101-131; program/event.h:22-32,
// 59-75): OpSet, DeviceState, GroupState, ThreadState, AdrType and the
// *_SIZE constants are all optional. A state declared as a member template
// (as the reference's barrier demo does) is not a type and falls back to
// VoidState, as in the reference.
#pragma once

#include "promise.h"

namespace hz {
namespace spec {

#define HZ_TYPE_OR(NAME)                                                     \
    template <typename S, typename D, typename = void>                       \
    struct NAME##Or {                                                        \
        using type = D;                                                      \
    };                                                                       \
    template <typename S, typename D>                                        \
    struct NAME##Or<S, D, std::void_t<typename S::NAME>> {                   \
        using type = typename S::NAME;                                       \
    };

HZ_TYPE_OR(OpSet)
HZ_TYPE_OR(DeviceState)
HZ_TYPE_OR(GroupState)
HZ_TYPE_OR(ThreadState)
HZ_TYPE_OR(AdrType)
#undef HZ_TYPE_OR

#define HZ_CONST_OR(NAME)                                                    \
    template <typename S, size_t D, typename = void>                         \
    struct NAME##Or {                                                        \
        static constexpr size_t value = D;                                   \
        static constexpr bool given = false;                                 \
    };                                                                       \
    template <typename S, size_t D>                                          \
    struct NAME##Or<S, D, std::void_t<decltype(S::NAME)>> {                  \
        static constexpr size_t value = (size_t)S::NAME;                     \
        static constexpr bool given = true;                                  \
    };

HZ_CONST_OR(STASH_SIZE)
HZ_CONST_OR(FRAME_SIZE)
HZ_CONST_OR(POOL_SIZE)
HZ_CONST_OR(STACK_SIZE)
HZ_CONST_OR(GROUP_SIZE)
// Groups (wavefronts) launched per workgroup by the async program type; they
// share the workgroup's __shared__ memory. Not a reference constant.
HZ_CONST_OR(GROUPS_PER_BLOCK)
// Nonzero: a group that holds several links hands some to groups that have
// none (for work that grows from few seeds). Not a reference constant.
HZ_CONST_OR(SHARE_WORK)
// Zero: a group that takes a queued link acquires nothing besides it. For
// promises that carry all they need, or read the rest with hz_load. Default 1.
// Not a reference constant.
HZ_CONST_OR(LINK_ACQUIRE)
// Zero: resolving a unit future publishes the returned value only, and reads
// the future's barrier and its promise with plain loads. For value-returning
// operations that hand over nothing else, values read with hz_load, and
// barriers built before the launch. Default 1. Not a reference constant.
HZ_CONST_OR(RETURN_RELEASE)
// Nonzero: a group runs its ready links oldest first (the order in which
// they filled), rather than by stash position. Work whose later promises can
// supersede earlier ones (a BFS level lowered again) wastes less. Not a
// reference constant.
HZ_CONST_OR(OLDEST_FIRST)
// Nonzero, with STACK_SIZE depth levels: run and pull the shallowest level
// first instead of the deepest. Not a reference constant.
HZ_CONST_OR(SHALLOW_FIRST)
// Zero: no lane keeps its successor promise in registers (CHAIN_LANES'
// default), and a program that chains all the same does not count the
// promises that run in the pass that queued them. Not a reference constant.
HZ_CONST_OR(FORWARD_LINKS)
// Nonzero: lanes keep their first successor promise in registers and run it
// next (lane chaining, async.h); zero: every promise passes through the
// stash. Defaults to FORWARD_LINKS. Not a reference constant.
HZ_CONST_OR(CHAIN_LANES)
// Nonzero: chaining lanes may hold different operations, which then run one
// after another in one pass. Default for up to two operations. Not a
// reference constant.
HZ_CONST_OR(CHAIN_MIXED)
// Passes over the lanes' promises between two looks at how many lanes still
// hold one (default 1): a specification whose operations are a few
// instructions, and whose chains are long, spares most of the looks. Not a
// reference constant.
HZ_CONST_OR(CHAIN_PASSES)
#undef HZ_CONST_OR

// The operation set a program type executes: the specification's OpSet, plus
// ReturnOp when an operation returns a value (hz::ExecOpSet).
template <typename S>
using ProgramOpSet = typename ExecOpSet<typename OpSetOr<S, OpUnion<>>::type>::type;

}  // namespace spec
}  // namespace hz
