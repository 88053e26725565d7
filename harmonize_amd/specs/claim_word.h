// What groups, housekeeper and host share of a job-table entry
// (specs/resident.h): its claim word and its completion word.
//
// The claim word holds the items claimed so far in its low half and the items
// in all in its high half.
//
// Groups claim from an entry while the housekeeper may be replacing its job,
// so a claim must not combine one job's counter with another's size. It is one
// 64-bit add of what is wanted to the low half: the value before it holds the
// counter and the size that belongs to it, and nothing read later decides. An
// entry is replaced in three steps with a wait after each: the word is closed,
// the other fields are written, the word is opened. A claim that was granted
// items may read the other fields afterwards: it found the word open, so they
// are complete, and the job cannot end before the granted items have.
//
// (A claim that adds to a 32-bit counter and reads the size afterwards is
// wrong however short the time between: with the counter past the old job's
// end, the word closed, the new size written and then read, the claimer takes
// the overshoot for items of the new job, which are handed out again when the
// counter is set back to 0.)
//
// Portable: MEM supplies add (returns the value before), store and wait, so
// that the order of accesses can be enumerated on a host.
#pragma once

#include "harmonize/portable.h"

namespace hz {
namespace resident {

// Counter of a word that grants nothing. Sizes stay below it, and adds to a
// word that grants nothing (at most one per wavefront that saw the job open,
// each below 2^10) stay far from the carry into the high half.
constexpr unsigned int CLOSED = 0x80000000u;

HZ_HD inline unsigned long long claim_word(unsigned int next, unsigned int limit) {
    return (unsigned long long)limit << 32 | next;
}

// Items [base, base + got) of the job that the entry holds.
struct Grant {
    unsigned int base;
    unsigned int got;
};

template <typename MEM>
HZ_HD inline Grant take_items(MEM& mem, unsigned long long* word, unsigned int want) {
    const unsigned long long before = mem.add(word, (unsigned long long)want);
    const unsigned int next = (unsigned int)before, limit = (unsigned int)(before >> 32);
    return Grant{next, next < limit ? (limit - next < want ? limit - next : want) : 0u};
}

// `write_fields` writes the entry's other fields.
template <typename MEM, typename FIELDS>
HZ_HD inline void replace_job(MEM& mem, unsigned long long* word, unsigned int size, FIELDS&& write_fields) {
    mem.store(word, claim_word(CLOSED, size));
    mem.wait();
    write_fields();
    mem.wait();
    mem.store(word, claim_word(0u, size));
}

// The doorbell word in which the kernel reports that ring entry `entry`,
// installed in job-table entry `job`, has completed. The host gives a table
// entry to the next job only when it has seen the completion of the last, so
// the words of jobs in flight are distinct. (Ring positions are not: a large
// job claimed smallest first is overtaken by more entries than the ring has,
// and of two jobs in flight a ring's length apart one completion overwrote
// the other before the host had looked.)
HZ_HD inline unsigned int completion_word(unsigned int entry, unsigned int job) {
    (void)entry;
    return job;
}

}  // namespace resident
}  // namespace hz
