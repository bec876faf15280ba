// The device memory behind a context's scratch: one block in use, and the outgrown
// blocks that a recorded graph still names.
//
// A graph recorded while the block was handed out has its address in its kernels'
// arguments, and a replay writes there.  Such a block therefore outlives its
// replacement: it is kept until the context goes.  Blocks that no capture saw are
// released when they are outgrown.  The replacement of a kept block is at least twice
// its size, so the kept ones together are smaller than the one in use (where the device
// still has that much; else the size asked for).
//
// Host code without HIP calls: allocation and release are the caller's.
#ifndef FUSILLI_AMD_CSRC_SCRATCH_BLOCKS_H
#define FUSILLI_AMD_CSRC_SCRATCH_BLOCKS_H

#include <cstddef>

struct FhipScratchBlocks {
  static constexpr int kMaxKept = 64;
  void *block = nullptr;
  size_t bytes = 0;
  bool recorded = false; // a capture has seen `block`
  void *kept[kMaxKept];
  int kept_count = 0;

  // Replaces the block by one of at least `want` > `bytes` bytes.  alloc(size): memory
  // or null; release(p): the device is done with p.  False without memory (no block is
  // left then, except where it could not be kept).
  template <typename Alloc, typename Release> bool grow(size_t want, Alloc &&alloc, Release &&release) {
    constexpr size_t kLeast = 64u << 10;
    want = want < kLeast ? kLeast : want;
    size_t more = want;
    if (block && recorded) {
      if (kept_count == kMaxKept)
        return false;
      kept[kept_count++] = block;
      more = want > 2 * bytes ? want : 2 * bytes;
    } else if (block) {
      release(block);
    }
    block = nullptr;
    bytes = 0;
    recorded = false;
    void *p = alloc(more);
    if (!p && more > want)
      p = alloc(more = want);
    if (!p)
      return false;
    block = p;
    bytes = more;
    return true;
  }

  template <typename Release> void release_all(Release &&release) {
    if (block)
      release(block);
    while (kept_count > 0)
      release(kept[--kept_count]);
    block = nullptr;
    bytes = 0;
    recorded = false;
  }
};

#endif // FUSILLI_AMD_CSRC_SCRATCH_BLOCKS_H
