// Which work item a block of a sliced-Q launch takes.  Plain C++, for the host too.
#pragma once
#include <stdint.h>

namespace khm {

// The hardware deals consecutive block ids round-robin to the XCDs.
constexpr uint32_t kNumXcds = 8;

struct WorkItem {
    uint32_t head_group, task;
    bool live;
};

// A launch over `total` templates (of which `active` are live) x `head_groups` head groups has a grid of
// (total, min(head_groups, 8), ceil(head_groups / 8)) blocks; block (x, y, z) -> (head group, template).
// Within a slice z of the grid: head groups fastest, templates last to first.  With 8 KV heads every XCD keeps one head and with 4
// or 2 two or four XCDs take turns with a head's templates: the Q ranges of one sequence share their K/V through an XCD's L2, and
// every XCD gets long and short templates alike.  (A head-major list cut into 8 contiguous runs gave a head's long half
// to one XCD and its short half to another: whole layer of one prompt of 4150 / 8300 tokens at Hq24/Hkv4/D256 318 / 1126 us,
// now 265 / 880 us; two of 4200 at Hq16/Hkv2/D256 512 -> 373 us, one of 8192 at Hq16/Hkv1 407 -> 276 us; 8 KV heads the
// same either way.)  Last to first: within a request the later Q ranges see more keys, so the long blocks start early and the
// short ones fill the end of the launch.
// More than eight head groups go slice by slice, so that an XCD finishes one before it starts the next: with all of them
// fastest it took turns between two or more heads' K/V, which do not fit its L2 together (32 KV heads at Hq32/D128: one prompt
// of 8192 tokens 1587 us, by slices 1136 us, as in the head-major runs; four of 1500..2048 on up to 8000 cached 1824 -> 1382 us; 20 KV
// heads 1174 -> 950 us; 16 at Hq16 736 -> 674 us.  At 16 KV heads the turns win where four Q heads share a KV head, FP8 pages 1925
// against 1976 us, and at Hq16/D256, 1530 against 1574 us; the runs took 2012 and 1578 us).  The groups of a full slice lie
// head_groups / 8 apart, which keeps neighbours on one XCD one after the other (eight neighbours to a slice: up to 1 %
// faster at head dim 128, 1 % slower at 256 on bf16 pages).
// The padding of a slice comes last.
constexpr uint32_t head_groups_per_slice(uint32_t head_groups) { return head_groups < kNumXcds ? head_groups : kNumXcds; }
constexpr uint32_t head_group_slices(uint32_t head_groups) { return (head_groups + kNumXcds - 1) / kNumXcds; }

constexpr WorkItem sliced_q_work_item(uint32_t x, uint32_t y, uint32_t z, uint32_t total, uint32_t active, uint32_t head_groups) {
    const uint32_t full_slices = head_groups / kNumXcds;
    const uint32_t linear = y * total + x;
    uint32_t rank = linear / kNumXcds;
    uint32_t head_group = linear % kNumXcds * full_slices + z;
    if (z >= full_slices) {
        const uint32_t groups = head_groups % kNumXcds;
        rank = linear / groups;
        head_group = full_slices * kNumXcds + linear - rank * groups;
    }
    if (active > total) active = total;
    return WorkItem{head_group, active - 1 - rank, rank < active};
}

// The same for tiles of bf16 pages that are the only readers of their K/V bytes (verify and drafting blocks): nothing to share, so each
// XCD takes a run of the head-major list.  On caches that no pass has read before, against head groups fastest: 25 drafting
// requests on 1200..12000 tokens at Hq24/Hkv4/D256 148.2 -> 143.6 us, 30 verify requests on 1200..24000 at Hq16/Hkv2/D256
// 180.9 -> 178.1 us, 24 on 1000..20000 at Hq64/Hkv4/D128 139 -> 130 us, 15 on 1200..5000 at Hq32/Hkv4 44.4 -> 44.8 us; 33 such
// batches 0.8 % faster on average.  FP8 pages are as fast either way (25 batches 0.1 % slower in runs, 33 requests on 400..1500 tokens at
// Hq24/Hkv4/D256 37.9 -> 40.0 us).  Only where the runs are whole head groups or equal parts of one: with 7 or 9 groups they end
// inside a head (24 requests at Hq36/Hkv9/D128 223 against 228 us in runs).  8 KV heads are the same list.
constexpr bool runs_fit_head_groups(uint32_t head_groups) {
    return head_groups % kNumXcds == 0 || (head_groups < kNumXcds && (head_groups & (head_groups - 1)) == 0);
}

constexpr WorkItem sole_reader_work_item(uint32_t x, uint32_t y, uint32_t z, uint32_t width, uint32_t height, uint32_t active, uint32_t head_groups) {
    if (!runs_fit_head_groups(head_groups)) return sliced_q_work_item(x, y, z, width, active, head_groups);
    if (active > width) active = width;
    const uint32_t items = active * head_groups;
    const uint32_t block = (z * height + y) * width + x;   // the grid has no blocks beyond width * head_groups
    if (block >= items) return WorkItem{0u, 0u, false};
    const uint32_t run = items / kNumXcds;
    const uint32_t item = block < run * kNumXcds ? (block % kNumXcds) * run + block / kNumXcds : block;
    const uint32_t head_group = item / active;
    return WorkItem{head_group, active - 1 - (item - head_group * active), true};
}

}  // namespace khm
