// event_list.hpp -- the plug-in fold's list of one key's events: summed in the
// order of their numbers.
#pragma once
#include <cstdint>

namespace edl {

// One host-pushed event: its weight and the event that reached the key's list
// before it (1 + its number; 0 ends the list).
struct FoldNode {
    uint32_t next;
    float w;
};

// Adds the events listed from `hd` (not 0) to g in the order of their numbers.
// Each walk finds the next four of them, so a list of up to four takes one.
// False when the chain is no list of at most n nodes numbered 1 to n: the
// allocation-free updates of one GPU share their nodes, and a call that
// overlaps another overwrites its lists.  Every loop ends on any contents, and
// no access leaves the n nodes.
template <class Nodes>
__host__ __device__ inline bool event_list_add(Nodes node, uint32_t n, uint32_t hd, float &g) {
    uint32_t last = 0u;
    for (uint32_t done = 4u;; done += 4u) {
        uint32_t b0 = ~0u, b1 = ~0u, b2 = ~0u, b3 = ~0u, m = 0u;
        float w0 = 0.0f, w1 = 0.0f, w2 = 0.0f, w3 = 0.0f;
        for (uint32_t q = hd; q != 0u; m++) {
            if (q > n || m == n) return false;
            const uint32_t next = node[q - 1u].next;
            const float w = node[q - 1u].w;
            if (q > last && q < b3) {
                b3 = q;
                w3 = w;
                if (b3 < b2) { const uint32_t t = b2; b2 = b3; b3 = t; const float u = w2; w2 = w3; w3 = u; }
                if (b2 < b1) { const uint32_t t = b1; b1 = b2; b2 = t; const float u = w1; w1 = w2; w2 = u; }
                if (b1 < b0) { const uint32_t t = b0; b0 = b1; b1 = t; const float u = w0; w0 = w1; w1 = u; }
            }
            q = next;
        }
        if (b0 == ~0u) return false;
        g = g + w0;
        if (b1 != ~0u) g = g + w1;
        if (b2 != ~0u) g = g + w2;
        if (b3 != ~0u) g = g + w3;
        if (m <= done) return true;
        if (b3 == ~0u) return false;
        last = b3;
    }
}

}  // namespace edl
