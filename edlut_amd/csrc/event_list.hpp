// event_list.hpp -- the plug-in fold's list of one key's events: summed in the
// order of their numbers.
#pragma once
#include <cstdint>

namespace edl {

// One host-pushed event: its weight and the event that reached the key's list
// before it (1 + its number; 0 ends the list).
struct alignas(8) FoldNode {
    uint32_t next;
    float w;
};

// Lists of up to this many events are summed by selection, longer ones sorted
// first.  An update of one AdEx cell, of 8 and of 64 cells with 96 events on
// each takes 270, 322 and 482 us by selection, with 97 (sorted) 184, 348 and
// 532 us.
constexpr uint32_t kListShort = 96;

// Sorts the list from `hd` by event number: its runs (a wave's events arrive
// together, in descending order seen from the head) are merged two by two
// through `next`, pass by pass.  Returns the new head, 0 when the chain is no
// list of at most n nodes numbered 1 to n.
template <class Nodes>
__host__ __device__ inline uint32_t event_list_sort(Nodes node, uint32_t n, uint32_t hd) {
    uint32_t m = 0u, prev = 0u;
    for (uint32_t q = hd; q != 0u; m++) {
        if (q > n || m == n) return 0u;
        const uint32_t next = node[q - 1u].next;
        node[q - 1u].next = prev;
        prev = q;
        q = next;
    }
    hd = prev;
    // a pass at least halves the runs
    for (int pass = 0; pass < 32; pass++) {
        uint32_t runs = 0u, left = m, ahead = m, tail = 0u, p = hd;
        while (p != 0u) {
            // x: the run from p to e; y: the one after it
            uint32_t x = p, e = p, y;
            for (;;) {
                y = node[e - 1u].next;
                if (y > n || ahead-- == 0u) return 0u;
                if (y <= e) break;
                e = y;
            }
            bool more_x = true, more_y = y != 0u;
            p = 0u;
            runs++;
            if (!more_y && tail == 0u) return hd;   // one run: sorted
            while (more_x || more_y) {
                const bool take_x = more_x && (!more_y || x < y);
                const uint32_t t = take_x ? x : y;
                const uint32_t next = node[t - 1u].next;
                if (next > n || left-- == 0u) return 0u;
                if (tail != 0u) node[tail - 1u].next = t;
                else hd = t;
                tail = t;
                if (take_x) {
                    more_x = t != e;
                    x = next;
                    if (more_x && x == 0u) return 0u;
                } else {
                    more_y = next > t;
                    if (more_y) y = next;
                    else p = next;
                }
            }
        }
        node[tail - 1u].next = 0u;
        if (runs == 1u) return hd;
    }
    return 0u;
}

// Adds the events listed from `hd` (not 0) to g in the order of their numbers.
// The loads along the chain bound it: each waits for the one before.  A walk
// finds the next four events, so a list of up to four takes one and one of m
// events m / 4.
// kListLong: more than kListShort events, nothing added.  kListBad: the chain is
// no list of at most n nodes numbered 1 to n (the allocation-free updates of
// one GPU share their nodes, and a call that overlaps another overwrites its
// lists).  Every loop ends on any contents, and no access leaves the n nodes.
enum ListEnd : uint32_t { kListDone = 0, kListLong = 1, kListBad = 2 };
template <class Nodes>
__host__ __device__ inline ListEnd event_list_add(Nodes node, uint32_t n, uint32_t hd, float &g) {
    if (hd > n) return kListBad;
    const uint32_t next1 = node[hd - 1u].next;
    const float first = node[hd - 1u].w;
    if (next1 == 0u) {
        g = g + first;
        return kListDone;
    }
    uint32_t last = 0u, q, m = 0u;
    for (uint32_t done = 4u;; done += 4u) {
        uint32_t b0 = ~0u, b1 = ~0u, b2 = ~0u, b3 = ~0u, i = 0u;
        float w0 = 0.0f, w1 = 0.0f, w2 = 0.0f, w3 = 0.0f;
        // the first walk counts the events (0, the end, is past n as well), the
        // others keep to their number
        const uint32_t limit = m == 0u ? kListShort : m;
        for (q = hd; (q - 1u < n) & (i < limit); i++) {
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
        if (q != 0u) return m == 0u && q <= n ? kListLong : kListBad;
        m = i;
        g = g + w0;
        if (b1 != ~0u) g = g + w1;
        if (b2 != ~0u) g = g + w2;
        if (b3 != ~0u) g = g + w3;
        if (done >= m) return b0 != ~0u ? kListDone : kListBad;
        if (b3 == ~0u) return kListBad;
        last = b3;
    }
}

// The same for a list that is longer: sorted, which takes a walk to turn it
// round and about one and a half for each doubling of its runs, and added in one.
// An update of one cell with 1,000 events 3.4 ms, with 3,000 12.6 ms (by
// selection 19.2 and 170 ms), with 100,000 0.65 s.
template <class Nodes>
__host__ __device__ inline ListEnd event_list_add_long(Nodes node, uint32_t n, uint32_t hd, float &g) {
    uint32_t q = event_list_sort(node, n, hd);
    if (q == 0u) return kListBad;
    for (uint32_t left = n; q != 0u; left--) {
        if (q > n || left == 0u) return kListBad;
        g = g + node[q - 1u].w;
        q = node[q - 1u].next;
    }
    return kListDone;
}

}  // namespace edl
