// chunk_scratch.hpp -- growth of the prompt chunks' scratch (host only, no HIP).
//
// A model keeps one block of scratch for chunks of `tokens` prompt positions.  It
// grows along a few rungs of chunk sizes; the block that it holds is freed before a
// larger one is asked for, so the two never stand beside each other, and where
// memory is short the next smaller rung is taken: the prompt then goes through
// more chunks.  The pair (mem, tokens) always describes a live block or none, and
// nothing else is kept, so a failed growth leaves no address behind.
#pragma once

#include <stdint.h>

namespace pk {

struct ChunkScratch {
    uint8_t* mem = nullptr;
    uint32_t tokens = 0;
};

// Readies scratch for chunks of min(n, rungs[n_rungs - 1]) positions, or as many as
// memory allows; false where not even rungs[0] fits (s is empty then).  rungs
// ascend; bytes(tokens) is a block's size, alloc(bytes) returns null on failure.
template <typename Bytes, typename Alloc, typename Free>
bool chunk_scratch_ready(ChunkScratch& s, const uint32_t* rungs, uint32_t n_rungs, uint32_t n,
                         Bytes bytes, Alloc alloc, Free release) {
    uint32_t r = 0;
    while (r + 1u < n_rungs && rungs[r] < n) ++r;
    if (s.tokens >= rungs[r]) return true;
    if (s.mem) release(s.mem);
    s = ChunkScratch{};
    for (;; --r) {
        if (uint8_t* mem = alloc(bytes(rungs[r]))) {
            s = ChunkScratch{mem, rungs[r]};
            return true;
        }
        if (r == 0u) return false;
    }
}

}  // namespace pk
