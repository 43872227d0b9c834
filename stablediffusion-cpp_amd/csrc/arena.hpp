// arena.hpp - the device memory arena and the library's scratch block, host
// code without a HIP call: segments come from two functions that the runtime
// supplies, so that a program without a GPU can run both.
#pragma once

#include <algorithm>
#include <cstddef>
#include <cstdint>
#include <iterator>
#include <map>
#include <set>
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
    size_t releases = 0;                               // calls of release that gave a block back

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
        ++releases;
        insert_free((uintptr_t)p, sz);
        return true;
    }
    bool has_free(size_t bytes) const { return free_by_size.lower_bound(round_up(bytes, kAlign)) != free_by_size.end(); }
    // The free range that releasing p would leave.
    size_t room_around(void* p) const {
        const auto it = live.find((uintptr_t)p);
        if (it == live.end()) return 0;
        const uintptr_t a = it->first;
        const int s = seg_of(a);
        size_t n = it->second;
        auto next = free_by_addr.lower_bound(a);
        const auto prev = next;
        if (next != free_by_addr.end() && next->first == a + it->second && seg_of(next->first) == s) n += next->second;
        if (prev != free_by_addr.begin()) {
            const auto b = std::prev(prev);
            if (b->first + b->second == a && seg_of(b->first) == s) n += b->second;
        }
        return n;
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
    // A graph keeps the pointers it was captured with: a block that an op asked
    // for during a capture is replaced, but given back only when the last graph
    // is destroyed.
    bool captured = false;
    std::vector<void*> retired;
    std::set<void*> graphs;
    // The last size that the arena could not hold, and its count of releases
    // then: until one more, a request that has another route is not tried again.
    size_t refused = 0, refused_at = 0;

    enum Answer { kHave, kHeld, kCapturing, kFull };

    // After kHave `block` holds at least `want` bytes for the op that asks;
    // after any other answer the block is what it was. `must`: the op has no
    // route without it.
    Answer take(size_t want, bool capturing, bool must = true) {
        if (held) return kHeld;
        if (want > bytes) {
            if (capturing) return kCapturing;
            if (!must && refused && want >= refused && arena.releases == refused_at) return kFull;
            if (!grow(want)) return kFull;
        }
        held = true;
        captured |= capturing;
        return kHave;
    }
    void end_op() { held = false; }

    // Returns an idle block to an exhausted arena (the next op that needs
    // scratch asks for it again); false where there is none, an op holds it
    // or a graph may.
    bool give_back(bool capturing) {
        if (!block || held || capturing || kept()) return false;
        sync();
        arena.release(block);
        block = nullptr;
        bytes = 0;
        return true;
    }

    void clear() {
        block = nullptr;
        bytes = 0;
        held = captured = false;
        retired.clear();
        graphs.clear();
        refused = 0;
    }

    // Replaces the block by one of at least `want` bytes; false, and the block
    // stays, when the arena cannot hold that much. The old block makes room
    // for the new one only where that is known to be enough, so a refusal
    // costs no wait and moves nothing: an op whose scratch does not fit asks
    // on each call and then takes its other route.
    bool grow(size_t want) {
        const size_t size = round_up(std::max(want, (size_t)1 << 20), kAlign);
        void* old = block;
        if (old && !kept() && !arena.has_free(size) && arena.room_around(old) >= size) {
            // work queued earlier may still read the old block
            sync();
            arena.release(old);
            old = nullptr;
        }
        void* fresh = arena.alloc(size);
        if (!fresh) {
            refused = want;
            refused_at = arena.releases;
            return false;
        }
        if (old && kept()) {
            retired.push_back(old);
        } else if (old) {
            sync();
            arena.release(old);
        }
        block = fresh;
        bytes = size;
        captured = false;
        return true;
    }

    void graph_made(void* g) { graphs.insert(g); }
    void graph_gone(void* g) {
        if (!graphs.erase(g) || !graphs.empty()) return;
        for (void* p : retired) arena.release(p);
        retired.clear();
        captured = false;
    }

    bool kept() const { return captured && !graphs.empty(); }
};

}  // namespace sdh
