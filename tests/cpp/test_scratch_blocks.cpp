// The blocks behind a context's scratch (fusilli_amd/csrc/scratch_blocks.h), with host
// memory in the place of the device's.
#include "../../fusilli_amd/csrc/scratch_blocks.h"
#include "mini_test.h"

#include <cstdint>
#include <map>

namespace {
struct Memory {
  std::map<void *, size_t> live;
  size_t limit = ~size_t(0), next = 4096;
  size_t used() const {
    size_t n = 0;
    for (const auto &b : live)
      n += b.second;
    return n;
  }
  bool grow(FhipScratchBlocks &s, size_t want) {
    return s.grow(want,
                  [&](size_t size) -> void * {
                    if (used() + size > limit)
                      return nullptr;
                    void *p = reinterpret_cast<void *>(static_cast<uintptr_t>(next));
                    next += size + 4096;
                    live[p] = size;
                    return p;
                  },
                  [&](void *p) { CHECK(live.erase(p) == 1); });
  }
  void release_all(FhipScratchBlocks &s) {
    s.release_all([&](void *p) { CHECK(live.erase(p) == 1); });
  }
};
constexpr size_t kMb = 1 << 20;
} // namespace

TEST("a block that no capture saw goes when it is outgrown") {
  Memory m;
  FhipScratchBlocks s;
  REQUIRE(m.grow(s, 100));
  CHECK(s.bytes == 64 << 10);
  REQUIRE(m.grow(s, kMb));
  CHECK(s.bytes == kMb && m.live.size() == 1 && m.live.count(s.block) == 1);
  m.release_all(s);
  CHECK(m.live.empty() && s.block == nullptr && s.bytes == 0);
}

TEST("a recorded block stays until the context goes") {
  Memory m;
  FhipScratchBlocks s;
  REQUIRE(m.grow(s, kMb));
  void *first = s.block;
  s.recorded = true;
  REQUIRE(m.grow(s, kMb + 1));
  CHECK(s.block != first && !s.recorded && s.bytes == 2 * kMb);
  CHECK(m.live.count(first) == 1);
  // outgrown again without a capture in between: only the recorded one stays
  REQUIRE(m.grow(s, 5 * kMb));
  CHECK(m.live.size() == 2 && m.live.count(first) == 1 && m.live.count(s.block) == 1);
  m.release_all(s);
  CHECK(m.live.empty());
}

TEST("kept blocks together are smaller than the one in use") {
  Memory m;
  FhipScratchBlocks s;
  for (size_t want = 1; want < (size_t)1 << 40; want = s.bytes + 1) {
    REQUIRE(m.grow(s, want));
    s.recorded = true;
    CHECK(m.used() < 2 * s.bytes);
  }
  CHECK(s.kept_count < FhipScratchBlocks::kMaxKept);
  m.release_all(s);
  CHECK(m.live.empty());
}

TEST("without room for twice the size the size asked for is taken") {
  Memory m;
  m.limit = 2500 * kMb;
  FhipScratchBlocks s;
  REQUIRE(m.grow(s, 1000 * kMb));
  void *first = s.block;
  s.recorded = true;
  REQUIRE(m.grow(s, 1200 * kMb));
  CHECK(s.bytes == 1200 * kMb);
  // no memory at all: the recorded ones stay, nothing is handed out
  s.recorded = true;
  void *second = s.block;
  CHECK(!m.grow(s, 1300 * kMb));
  CHECK(s.block == nullptr && s.bytes == 0 && !s.recorded);
  CHECK(m.live.count(first) == 1 && m.live.count(second) == 1);
  CHECK(m.grow(s, kMb));
  m.release_all(s);
  CHECK(m.live.empty());
}

TEST("a full list refuses instead of dropping a block") {
  Memory m;
  FhipScratchBlocks s;
  REQUIRE(m.grow(s, kMb));
  s.recorded = true;
  s.kept_count = FhipScratchBlocks::kMaxKept;
  void *first = s.block;
  CHECK(!m.grow(s, 3 * kMb));
  CHECK(s.block == first && s.recorded && s.bytes == kMb);
}

int main(int argc, char **argv) { return mini::run(argc, argv); }
