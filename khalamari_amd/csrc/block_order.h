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
    const uint32_t groups = z < full_slices ? kNumXcds : head_groups % kNumXcds;
    const uint32_t linear = y * total + x;
    const uint32_t rank = linear / groups;
    const uint32_t within = linear - rank * groups;
    if (active > total) active = total;
    return WorkItem{z < full_slices ? within * full_slices + z : full_slices * kNumXcds + within, active - 1 - rank, rank < active};
}

}  // namespace khm
