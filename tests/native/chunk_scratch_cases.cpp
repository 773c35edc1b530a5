// chunk_scratch_ready against an allocator with a limit: after every call the
// scratch must be a live block of its chunk size, or empty, and nothing may leak or
// be freed twice.  Prints one PASS or FAIL line per case.
#include <stdio.h>
#include <stdlib.h>

#include <map>

#include "../../pokitlms_amd/csrc/chunk_scratch.hpp"

namespace {

struct Heap {
    uint64_t limit = ~0ull, used = 0, peak = 0;
    uint32_t refused = 0;
    bool bad_free = false;
    std::map<uint8_t*, uint64_t> live;
    uint8_t* alloc(uint64_t n) {
        if (used + n > limit) {
            ++refused;
            return nullptr;
        }
        uint8_t* p = static_cast<uint8_t*>(malloc(1));
        live[p] = n;
        used += n;
        peak = used > peak ? used : peak;
        return p;
    }
    void release(uint8_t* p) {
        const auto it = live.find(p);
        if (it == live.end()) {
            bad_free = true;
            return;
        }
        used -= it->second;
        live.erase(it);
        free(p);
    }
};

constexpr uint32_t kRungs[3] = {64, 192, 512};
uint64_t bytes(uint32_t t) { return 1000ull * t; }

bool ready(Heap& h, pk::ChunkScratch& s, uint32_t n) {
    const bool ok = pk::chunk_scratch_ready(s, kRungs, 3, n, bytes, [&](uint64_t b) { return h.alloc(b); },
                                            [&](uint8_t* p) { h.release(p); });
    return ok;
}

// The state a prompt may rely on: a live block of its size, or none.
bool sound(const Heap& h, const pk::ChunkScratch& s, bool ok) {
    if (h.bad_free || ok != (s.mem != nullptr)) return false;
    if (!s.mem) return s.tokens == 0u && h.live.empty();
    const auto it = h.live.find(s.mem);
    return h.live.size() == 1u && it != h.live.end() && it->second >= bytes(s.tokens) && s.tokens != 0u;
}

int failed = 0;
void report(const char* name, bool ok) {
    printf("%s %s\n", ok ? "PASS" : "FAIL", name);
    failed += ok ? 0 : 1;
}

}  // namespace

int main() {
    {  // the rungs, and a block that already serves
        Heap h;
        pk::ChunkScratch s;
        bool ok = true;
        const uint32_t n[] = {1, 64, 65, 192, 40, 193, 5000, 300};
        const uint32_t want[] = {64, 64, 192, 192, 192, 512, 512, 512};
        for (int i = 0; i < 8; ++i) ok = ok && ready(h, s, n[i]) && sound(h, s, true) && s.tokens == want[i];
        report("rungs", ok && h.peak == bytes(512));  // never two blocks at once
    }
    {  // 40 positions, 300 with no memory for them, 40 again
        Heap h;
        pk::ChunkScratch s;
        h.limit = bytes(64);
        bool ok = ready(h, s, 40) && sound(h, s, true) && s.tokens == 64u;
        ok = ok && ready(h, s, 300) && sound(h, s, true) && s.tokens == 64u && h.refused == 2u;
        ok = ok && ready(h, s, 40) && sound(h, s, true) && s.tokens == 64u && h.refused == 2u;
        report("failed_growth_keeps_a_smaller_block", ok);
    }
    {  // memory gone altogether, then back
        Heap h;
        pk::ChunkScratch s;
        bool ok = ready(h, s, 40) && sound(h, s, true);
        h.limit = 0;
        const bool mid = ready(h, s, 300);
        ok = ok && !mid && sound(h, s, mid);
        const bool again = ready(h, s, 40);
        ok = ok && !again && sound(h, s, again);
        h.limit = ~0ull;
        ok = ok && ready(h, s, 600) && sound(h, s, true) && s.tokens == 512u;
        report("nothing_left_then_memory_again", ok);
    }
    return failed ? 1 : 0;
}
