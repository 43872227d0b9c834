// The scratch block's rules (csrc/arena.hpp) on host memory: each function
// below is one scenario; main runs the one that its argument names.
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <map>
#include <string>

#include "arena.hpp"

using namespace sdh;

namespace {

constexpr size_t MB = 1 << 20;
int waits = 0;
void* reserve(size_t n) { return std::aligned_alloc(4096, n); }
void unreserve(void* p) { std::free(p); }
void sync() { ++waits; }

#define CHECK(c)                                                  \
    do {                                                          \
        if (!(c)) {                                               \
            std::printf("line %d: %s\n", __LINE__, #c);           \
            return 1;                                             \
        }                                                         \
    } while (0)

struct World {
    Arena arena{reserve, unreserve};
    Scratch s{arena, sync};
    World(size_t limit) {
        arena.limit = limit;
        arena.grow(limit);
    }
    ~World() { arena.clear(); }
};

// An op that holds the block is never answered with it again, nor does the
// block move, whoever asks inside the op: conv2d's patches against the product.
int held() {
    World w(64 * MB);
    CHECK(w.s.take(8 * MB, false) == Scratch::kHave);
    void* cols = w.s.block;
    CHECK(w.s.take(4 * MB, false) == Scratch::kHeld);
    CHECK(w.s.take(16 * MB, false) == Scratch::kHeld);
    CHECK(w.s.take(16 * MB, true) == Scratch::kHeld);
    CHECK(!w.s.give_back(false));
    CHECK(w.s.block == cols && w.s.bytes == 8 * MB && w.arena.live.count((uintptr_t)cols));
    w.s.end_op();
    CHECK(w.s.take(16 * MB, false) == Scratch::kHave);
    w.s.end_op();
    CHECK(w.s.take(16 * MB, true) == Scratch::kHave);  // no growth: also during a capture
    w.s.end_op();
    CHECK(w.s.take(17 * MB, true) == Scratch::kCapturing);
    CHECK(w.s.give_back(false) && w.arena.in_use == 0);
    return 0;
}

// Memory for someone else, inside an op that holds the block: the arena finds
// none rather than the op's own (the GEMM workspace against the packed input).
int exhausted() {
    World w(96 * MB);
    CHECK(w.s.take(32 * MB, false) == Scratch::kHave);
    CHECK(!w.arena.alloc(80 * MB));
    CHECK(!w.s.give_back(false) && !w.arena.alloc(80 * MB));
    w.s.end_op();
    CHECK(w.s.give_back(false));  // between ops it is idle
    void* p = w.arena.alloc(80 * MB);
    CHECK(p && w.s.take(32 * MB, false) == Scratch::kFull);
    w.arena.release(p);
    CHECK(w.s.take(32 * MB, false) == Scratch::kHave);
    return 0;
}

// A request that does not fit leaves the block as it was, without a wait, and
// repeated ones take nothing from the arena, with a graph or without.
int refused() {
    World w(64 * MB);
    for (int graph = 0; graph < 2; ++graph) {
        CHECK(w.s.take(8 * MB, false) == Scratch::kHave);
        w.s.end_op();
        if (graph) {
            CHECK(w.s.take(MB, true) == Scratch::kHave);
            w.s.end_op();
            w.s.graph_made(&w);
        }
        void* b = w.s.block;
        const size_t used = w.arena.in_use, n = w.s.bytes;
        waits = 0;
        for (int i = 0; i < 20; ++i) {
            CHECK(w.s.take(100 * MB, false, false) == Scratch::kFull);
            CHECK(w.s.take(100 * MB, false) == Scratch::kFull);
            CHECK(w.s.take(8 * MB, false) == Scratch::kHave);  // the other route's, smaller
            w.s.end_op();
            CHECK(w.s.block == b && w.s.bytes == n && w.arena.in_use == used);
        }
        CHECK(waits == 0 && w.s.retired.empty());
    }
    // once something is given back, a request that may do without is tried again
    void* p = w.arena.alloc(48 * MB);
    CHECK(p && w.s.take(40 * MB, false, false) == Scratch::kFull);
    w.arena.release(p);
    CHECK(w.s.take(40 * MB, false, false) == Scratch::kHave && w.s.bytes == 40 * MB);
    return 0;
}

// The old block's memory is used for the new one where only both together suffice.
int in_place() {
    World w(64 * MB);
    CHECK(w.s.take(40 * MB, false) == Scratch::kHave);
    w.s.end_op();
    CHECK(w.s.take(60 * MB, false) == Scratch::kHave);
    CHECK(w.s.bytes == 60 * MB && w.arena.in_use == 60 * MB);
    return 0;
}

// A graph keeps the block of its capture and no other, until the last one goes.
int graphs() {
    World w(256 * MB);
    int g1, g2;
    CHECK(w.s.take(8 * MB, false) == Scratch::kHave);
    w.s.end_op();
    w.s.graph_made(&g1);  // a graph without scratch
    CHECK(w.s.take(16 * MB, false) == Scratch::kHave);
    w.s.end_op();
    CHECK(w.s.retired.empty() && w.arena.in_use == 16 * MB);
    CHECK(w.s.take(16 * MB, true) == Scratch::kHave);
    w.s.end_op();
    w.s.graph_made(&g2);
    void* kept = w.s.block;
    CHECK(!w.s.give_back(false));
    CHECK(w.s.take(32 * MB, false) == Scratch::kHave);
    w.s.end_op();
    CHECK(w.s.retired.size() == 1 && w.s.retired[0] == kept && w.arena.in_use == 48 * MB);
    CHECK(w.s.give_back(false));  // the new block is in no graph
    CHECK(w.arena.live.count((uintptr_t)kept));
    w.s.graph_gone(&g1);
    CHECK(w.arena.live.count((uintptr_t)kept));
    w.s.graph_gone(&w);  // not one of them
    CHECK(w.arena.live.count((uintptr_t)kept));
    w.s.graph_gone(&g2);
    CHECK(w.s.retired.empty() && w.arena.in_use == 0);
    // a shutdown with a graph left: the next blocks are free of it, and so is its late end
    w.s.graph_made(&g1);
    w.s.clear();
    CHECK(w.s.take(8 * MB, false) == Scratch::kHave);
    w.s.end_op();
    w.s.graph_gone(&g1);
    CHECK(w.s.take(8 * MB, true) == Scratch::kHave);
    w.s.end_op();
    w.s.graph_made(&g2);
    CHECK(!w.s.give_back(false));
    w.s.graph_gone(&g2);
    CHECK(w.s.give_back(false));
    return 0;
}

}  // namespace

int main(int argc, char** argv) {
    const std::map<std::string, int (*)()> all = {{"held", held}, {"exhausted", exhausted}, {"refused", refused}, {"in_place", in_place},
                                                           {"graphs", graphs}};
    const auto it = all.find(argc > 1 ? argv[1] : "");
    return it == all.end() ? 2 : it->second();
}
