// arena.hpp - the device memory arena and the library's scratch block, host
// code without a HIP call: segments come from two functions that the runtime
// supplies, so that a program without a GPU can run both.
#pragma once

#include <algorithm>
#include <cstddef>
#include <cstdint>
#include <map>
#include <vector>

namespace sdh {

constexpr size_t kAlign = 256;

inline size_t round_up(size_t v, size_t a) { return (v + a - 1) / a * a; }

// Arena: segments of device memory; free ranges indexed by address (for
// coalescing) and by size (for best fit). Blocks never span segments.
struct Arena {
    struct Seg {
        uintptr_t base;
        size_t bytes;
    };
    void* (*reserve)(size_t) = nullptr;    // a new segment, null where there is none
    void (*unreserve)(void*) = nullptr;
    std::vector<Seg> segs;
    std::map<uintptr_t, size_t> free_by_addr;          // addr -> size
    std::multimap<size_t, uintptr_t> free_by_size;     // size -> addr
    std::map<uintptr_t, size_t> live;                  // addr -> rounded size
    std::map<uintptr_t, size_t> requested;             // addr -> bytes asked for
    size_t reserved = 0, in_use = 0, limit = 0;        // limit 0 = none

    int seg_of(uintptr_t a) const {
        for (size_t i = 0; i < segs.size(); ++i)
            if (a >= segs[i].base && a < segs[i].base + segs[i].bytes) return (int)i;
        return -1;
    }
    void erase_free(uintptr_t a, size_t sz) {
        free_by_addr.erase(a);
        auto r = free_by_size.equal_range(sz);
        for (auto it = r.first; it != r.second; ++it)
            if (it->second == a) {
                free_by_size.erase(it);
                return;
            }
    }
    void insert_free(uintptr_t a, size_t sz) {
        // coalesce with neighbours inside the same segment
        const int s = seg_of(a);
        auto next = free_by_addr.lower_bound(a);
        if (next != free_by_addr.end() && next->first == a + sz && seg_of(next->first) == s) {
            const uintptr_t na = next->first;
            const size_t nsz = next->second;
            erase_free(na, nsz);
            sz += nsz;
        }
        auto prev = free_by_addr.lower_bound(a);
        if (prev != free_by_addr.begin()) {
            --prev;
            if (prev->first + prev->second == a && seg_of(prev->first) == s) {
                const uintptr_t pa = prev->first;
                const size_t psz = prev->second;
                erase_free(pa, psz);
                a = pa;
                sz += psz;
            }
        }
        free_by_addr[a] = sz;
        free_by_size.emplace(sz, a);
    }
    bool grow(size_t need) {
        size_t bytes = round_up(std::max(need, (size_t)256 << 20), (size_t)2 << 20);
        if (limit && reserved + bytes > limit) {
            if (reserved + round_up(need, (size_t)2 << 20) > limit) return false;
            bytes = round_up(need, (size_t)2 << 20);
        }
        void* p = reserve(bytes);
        if (!p) return false;
        segs.push_back({(uintptr_t)p, bytes});
        reserved += bytes;
        insert_free((uintptr_t)p, bytes);
        return true;
    }
    void* alloc(size_t bytes) {
        const size_t sz = round_up(bytes, kAlign);
        auto it = free_by_size.lower_bound(sz);
        if (it == free_by_size.end()) {
            if (!grow(sz)) return nullptr;
            it = free_by_size.lower_bound(sz);
            if (it == free_by_size.end()) return nullptr;
        }
        const uintptr_t a = it->second;
        const size_t fsz = it->first;
        erase_free(a, fsz);
        if (fsz > sz) insert_free(a + sz, fsz - sz);
        live[a] = sz;
        requested[a] = bytes;
        in_use += sz;
        return (void*)a;
    }
    bool release(void* p) {
        auto it = live.find((uintptr_t)p);
        if (it == live.end()) return false;
        const size_t sz = it->second;
        live.erase(it);
        requested.erase((uintptr_t)p);
        in_use -= sz;
        insert_free((uintptr_t)p, sz);
        return true;
    }
    void clear() {
        for (auto& s : segs) unreserve((void*)s.base);
        segs.clear();
        free_by_addr.clear();
        free_by_size.clear();
        live.clear();
        requested.clear();
        reserved = in_use = 0;
    }
};

// The library's scratch block. One op at a time holds it: from the op's first
// request to the end of its entry point (end_op) a second request is refused,
// since it would be answered with the memory that the op already uses.
struct Scratch {
    Arena& arena;
    void (*sync)();  // waits for the work queued so far
    void* block = nullptr;
    size_t bytes = 0;
    bool held = false;
    // Blocks that grew out of use while captured graphs were alive: a graph
    // keeps the pointers it was captured with, so they are given back only
    // when the last graph is destroyed.
    std::vector<void*> retired;
    int graphs = 0;

    enum Answer { kHave, kHeld, kCapturing, kFull };

    // After kHave `block` holds at least `want` bytes for the op that asks.
    Answer take(size_t want, bool capturing) {
        if (held) return kHeld;
        if (want > bytes) {
            if (capturing) return kCapturing;
            if (!grow(want)) return kFull;
        }
        held = true;
        return kHave;
    }
    void end_op() { held = false; }

    // Returns an idle block to an exhausted arena (the next op that needs
    // scratch asks for it again); false where there is none, an op holds it
    // or a graph may.
    bool give_back(bool capturing) {
        if (!block || held || capturing || graphs > 0) return false;
        sync();
        arena.release(block);
        block = nullptr;
        bytes = 0;
        return true;
    }

    void clear() {
        block = nullptr;
        bytes = 0;
        held = false;
        retired.clear();
    }

    // Replaces the block by one of at least `want` bytes; false when the
    // arena cannot hold it (there is then no block).
    bool grow(size_t want) {
        if (block) {
            if (graphs > 0) {
                retired.push_back(block);
            } else {
                // Work queued earlier may still read the old block.
                sync();
                arena.release(block);
            }
        }
        bytes = round_up(std::max(want, (size_t)1 << 20), kAlign);
        block = arena.alloc(bytes);
        if (!block) bytes = 0;
        return block != nullptr;
    }

    void graph_made() { ++graphs; }
    void graph_gone() {
        if (--graphs > 0) return;
        for (void* p : retired) arena.release(p);
        retired.clear();
    }
};

}  // namespace sdh
