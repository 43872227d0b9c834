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

}  // namespace

int main(int argc, char** argv) {
    const std::map<std::string, int (*)()> all = {{"held", held}, {"exhausted", exhausted}};
    const auto it = all.find(argc > 1 ? argv[1] : "");
    return it == all.end() ? 2 : it->second();
}
