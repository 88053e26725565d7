// ORACLE — test infrastructure only (see host_shim.h).
//
// What groups, housekeeper and host share of the resident program's job table
// (specs/claim_word.h), on the host.
//
// Every order of the memory accesses of two groups that claim from a
// job-table entry of the resident program while the housekeeper replaces the
// entry's job. The accesses are those of specs/claim_word.h, or of the
// protocol that it replaces, planted here as a mistake that must be found:
// the counter and the limit as words of their own, the limit read after the
// add. Actors are coroutines that stop before each access.
#include <ucontext.h>

#include <cstdint>
#include <functional>
#include <memory>
#include <vector>

#include "host_shim.h"
#include "claim_word.h"

namespace {

constexpr unsigned int OLD_SIZE = 10, OLD_SEED = 1, OLD_BASE = 100;
constexpr unsigned int NEW_SIZE = 200, NEW_SEED = 2, NEW_BASE = 5000;
constexpr unsigned int OVERSHOOT = 64;  // added to the old job's counter beyond its size
constexpr size_t STACK = 1 << 16;

struct Actor {
    ucontext_t context;
    std::unique_ptr<char[]> stack{new char[STACK]};
    std::function<void()> body;
    bool ended = false;
};

// Runs the actors to their ends, the next one by a list of choices.
struct Scheduler {
    ucontext_t home;
    std::vector<std::unique_ptr<Actor>> actors;
    Actor* now = nullptr;

    static Scheduler*& current() {
        static thread_local Scheduler* s = nullptr;
        return s;
    }
    static void enter() {
        Scheduler* s = current();
        s->now->body();
        s->now->ended = true;
        swapcontext(&s->now->context, &s->home);
    }
    void add(std::function<void()> body) {
        actors.emplace_back(new Actor);
        Actor& a = *actors.back();
        a.body = std::move(body);
        getcontext(&a.context);
        a.context.uc_stack.ss_sp = a.stack.get();
        a.context.uc_stack.ss_size = STACK;
        a.context.uc_link = nullptr;
        makecontext(&a.context, enter, 0);
    }
    void access() { swapcontext(&now->context, &home); }

    // `choices` holds (taken, of how many) per step; missing ones are 0.
    void run(std::vector<std::pair<int, int>>& choices) {
        current() = this;
        for (size_t step = 0;; ++step) {
            std::vector<Actor*> can;
            for (auto& a : actors) {
                if (!a->ended) can.push_back(a.get());
            }
            if (can.empty()) return;
            if (step == choices.size()) choices.push_back({0, 0});
            choices[step].second = (int)can.size();
            now = can[(size_t)choices[step].first];
            swapcontext(&home, &now->context);
        }
    }
};

// The next list of choices in order; false after the last.
bool advance(std::vector<std::pair<int, int>>& choices) {
    while (!choices.empty()) {
        if (++choices.back().first < choices.back().second) return true;
        choices.pop_back();
    }
    return false;
}

struct Entry {
    unsigned long long claims = hz::resident::claim_word(OLD_SIZE + OVERSHOOT, OLD_SIZE);
    unsigned int seed = OLD_SEED, base = OLD_BASE;
};

struct SteppedMemory {
    Scheduler* s;
    unsigned long long add(unsigned long long* p, unsigned long long v) {
        s->access();
        const unsigned long long before = *p;
        *p += v;
        return before;
    }
    void store(unsigned long long* p, unsigned long long v) {
        s->access();
        *p = v;
    }
    void wait() {}
};

// One order: whether each of the new job's items was granted once, with that
// job's fields, and nothing else was.
bool order_is_right(bool planted, std::vector<std::pair<int, int>>& choices) {
    Scheduler s;
    Entry e;
    SteppedMemory memory{&s};
    bool right = true;
    std::vector<int> granted(NEW_SIZE, 0);
    auto half = [&](int which) -> unsigned int& { return ((unsigned int*)&e.claims)[which]; };  // little-endian
    auto take = [&](unsigned int want) {
        hz::resident::Grant g{0u, 0u};
        if (planted) {
            s.access();
            g.base = half(0);
            half(0) += want;
            s.access();
            const unsigned int limit = half(1);
            g.got = g.base < limit ? (limit - g.base < want ? limit - g.base : want) : 0u;
        } else {
            g = hz::resident::take_items(memory, &e.claims, want);
        }
        if (g.got == 0u) return false;
        s.access();
        const unsigned int seed = e.seed, base = e.base;
        right = right && seed == NEW_SEED && base == NEW_BASE;
        for (unsigned int i = g.base; i < g.base + g.got; ++i) {
            right = right && i < NEW_SIZE;
            if (i < NEW_SIZE) granted[i] += 1;
        }
        return true;
    };
    s.add([&] {
        auto fields = [&] {
            s.access();
            e.seed = NEW_SEED;
            s.access();
            e.base = NEW_BASE;
        };
        if (planted) {
            s.access();
            half(0) = hz::resident::CLOSED;
            s.access();
            half(1) = NEW_SIZE;
            fields();
            s.access();
            half(0) = 0u;
        } else {
            hz::resident::replace_job(memory, &e.claims, NEW_SIZE, fields);
        }
    });
    // Both saw the old job with items left.
    s.add([&] { take(64); });
    s.add([&] { take(37); });
    s.run(choices);
    // What is left goes to a group that comes later.
    for (unsigned int i = half(0); i < half(1); ++i) granted[i] += 1;
    for (int n : granted) right = right && n == 1;
    return right;
}

}  // namespace

// Jobs all there at once, served by a table of `table` entries that the host
// fills in order, smallest installed job first: how many pairs of jobs that
// are in flight together report in the same completion word. `ring` is 0 for
// the runtime's words, or the length of a ring whose positions are the words
// (the planted mistake).
extern "C" uint64_t oracle_shared_completion_words(const uint32_t* sizes, uint32_t jobs, uint32_t table,
                                                   uint32_t ring) {
    struct Flight {
        uint32_t entry, job;
    };
    std::vector<Flight> flying;
    std::vector<uint32_t> free_entries;
    for (uint32_t t = table; t > 0; --t) free_entries.push_back(t - 1u);
    auto word = [&](const Flight& f) { return ring ? f.entry % ring : hz::resident::completion_word(f.entry, f.job); };
    uint64_t shared = 0;
    for (uint32_t next = 0; next < jobs || !flying.empty();) {
        while (next < jobs && !free_entries.empty()) {
            const Flight f{next++, free_entries.back()};
            free_entries.pop_back();
            for (const Flight& o : flying) shared += word(o) == word(f);
            flying.push_back(f);
        }
        size_t least = 0;
        for (size_t i = 1; i < flying.size(); ++i) {
            if (sizes[flying[i].entry] < sizes[flying[least].entry]) least = i;
        }
        free_entries.push_back(flying[least].job);
        flying.erase(flying.begin() + (long)least);
    }
    return shared;
}

// Runs every order; returns how many there are, and in *wrong how many of
// them grant an item twice, not at all, or with another job's fields.
extern "C" uint64_t oracle_claim_orders(int planted, uint64_t* wrong) {
    uint64_t orders = 0;
    *wrong = 0;
    std::vector<std::pair<int, int>> choices;
    do {
        *wrong += order_is_right(planted != 0, choices) ? 0u : 1u;
        orders++;
    } while (advance(choices));
    return orders;
}
