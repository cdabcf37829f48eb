// mpm_recurring.hpp -- which of a program's repeated calls get a captured
// graph (host code only; Graph is a pointer-like handle, null when empty).
#pragma once
#include <stddef.h>
#include <stdint.h>

#include <iterator>
#include <map>

namespace mpm {

// Counts calls by key and holds the graphs.  A handle in a steady state comes
// back to the same key after a cycle of calls: the key holds the substeps
// since the last sort and the current buffers, so an interval of 128 substeps
// and calls of 17 have a cycle of more than 200 keys.  The counts of a cycle
// of up to KEYS / 2 keys are therefore never forgotten, and the first GRAPHS
// of its keys to come back are the ones that get a graph.  A graph of 43
// launches holds 2 MB of device memory and its capture costs about 180 us,
// hence the bound, and hence a graph gives way only when it has been idle for
// longer than any cycle that is counted, and to a key that has come back
// REPLACE_CALLS times: a program that keeps changing its time step stays
// eager unless each lasts.
// A replay saves 10 to 40 us, so a capture pays after some 16 of them.  The
// credit, which outlives clear(), stops captures that do not pay: a program
// that loads particles every 24 frames of 8 substeps (1,000 particles)
// replayed 0.75 times per capture, 164 -> 176 us a frame; 40 frames of 20
// substeps (8,192 particles) never, 446 -> 471 us.
template <class Key, class Graph>
class RecurringCalls {
public:
    static constexpr uint32_t CALLS = 4;  // eager calls of a key before its capture
    static constexpr uint32_t REPLACE_CALLS = 32;
    static constexpr size_t KEYS = 1024;
    static constexpr size_t GRAPHS = 64;
    static constexpr uint32_t CAPTURE_COST = 16;  // in replays
    static constexpr uint32_t CREDIT = uint32_t(GRAPHS) * CAPTURE_COST;  // at the start, and at most

    struct Entry {
        uint32_t calls = 0;
        uint64_t used = 0;  // the last call, by the clock
        Graph graph{};
    };

    // The key's entry, with this call counted.  References stay valid until
    // the next call() or clear().
    Entry& call(const Key& key) {
        if (entries_.size() >= KEYS)
            for (auto it = entries_.begin(); it != entries_.end();)
                it = !it->second.graph && clock_ - it->second.used >= KEYS / 2 ? entries_.erase(it) : std::next(it);
        Entry& e = entries_[key];
        e.used = ++clock_;
        e.calls++;
        if (e.graph && credit_ < CREDIT) credit_++;
        return e;
    }

    // Whether the entry of the present call is to be captured now.  A graph
    // that gives way to it goes through destroy.
    template <class Destroy>
    bool due(Entry& e, Destroy destroy) {
        if (e.graph || e.calls <= CALLS || credit_ < CAPTURE_COST) return false;
        if (graphs_ < GRAPHS) return true;
        if (e.calls <= REPLACE_CALLS) return false;
        Entry* oldest = nullptr;
        for (auto& kv : entries_)
            if (kv.second.graph && (!oldest || kv.second.used < oldest->used)) oldest = &kv.second;
        if (clock_ - oldest->used <= KEYS) {
            e.calls = CALLS;  // ask again later
            return false;
        }
        destroy(oldest->graph);
        *oldest = Entry{0u, oldest->used, Graph{}};
        graphs_--;
        return true;
    }

    void keep(Entry& e, Graph g) {
        e.graph = g;
        graphs_++;
        credit_ -= CAPTURE_COST;
    }

    // A capture failed: the key's counted calls start over.
    void failed(const Key& key) {
        auto it = entries_.find(key);
        if (it != entries_.end()) it->second.calls = 0;
        credit_ -= CAPTURE_COST;
    }

    template <class Destroy>
    void clear(Destroy destroy) {
        for (auto& kv : entries_)
            if (kv.second.graph) destroy(kv.second.graph);
        entries_.clear();
        graphs_ = 0;
    }

    size_t graphs() const { return graphs_; }
    size_t keys() const { return entries_.size(); }

private:
    std::map<Key, Entry> entries_;
    uint64_t clock_ = 0;
    size_t graphs_ = 0;
    uint32_t credit_ = CREDIT;
};

}  // namespace mpm
