"""Which (head group, template) a block of a sliced-Q launch takes, from the header the kernel uses, built for the host: every item once,
padding last, templates last to first, and no XCD between two head groups' K/V at a time."""
import ctypes
import os
import subprocess

import numpy as np
import pytest

from khalamari_amd.build import CSRC_DIR

XCDS = 8
SOURCE = """
#include "block_order.h"
extern "C" unsigned items(unsigned total, unsigned active, unsigned head_groups, unsigned* out) {
    unsigned n = 0;
    for (unsigned z = 0; z < khm::head_group_slices(head_groups); ++z)
        for (unsigned y = 0; y < khm::head_groups_per_slice(head_groups); ++y)
            for (unsigned x = 0; x < total; ++x, ++n) {
                const khm::WorkItem item = khm::sliced_q_work_item(x, y, z, total, active, head_groups);
                out[3 * n] = item.head_group; out[3 * n + 1] = item.task; out[3 * n + 2] = item.live;
            }
    return n;
}
"""


@pytest.fixture(scope="module")
def order(tmp_path_factory):
    folder = tmp_path_factory.mktemp("block_order")
    source, library = folder / "order.cpp", folder / "order.so"
    source.write_text(SOURCE)
    subprocess.run([os.environ.get("CXX", "g++"), "-std=c++17", "-O1", "-Wall", "-Werror", "-shared", "-fPIC", "-I", CSRC_DIR, str(source), "-o", str(library)], check=True)
    return ctypes.CDLL(str(library))


@pytest.mark.parametrize("head_groups", [1, 2, 3, 4, 8, 9, 12, 16, 20, 32, 64])
@pytest.mark.parametrize("active,total", [(0, 3), (1, 1), (1, 5), (7, 7), (24, 24), (23, 40), (64, 64)])
def test_every_item_once_and_head_groups_one_after_the_other(order, head_groups, active, total):
    out = np.zeros(((head_groups + XCDS) * total, 3), dtype=np.uint32)
    blocks = order.items(total, active, head_groups, out.ctypes.data_as(ctypes.c_void_p))
    assert blocks <= len(out)
    out = out[:blocks]
    live = out[:, 2] == 1
    assert np.count_nonzero(live) == active * head_groups
    if head_groups <= XCDS:
        assert np.all(live[:active * head_groups])   # the padding comes last
    heads, tasks = out[live, 0].astype(int), out[live, 1].astype(int)
    assert sorted(zip(heads, tasks)) == [(h, t) for h in range(head_groups) for t in range(active)]
    for h in range(head_groups):
        assert np.all(np.diff(tasks[heads == h]) == -1)
    if head_groups % XCDS == 0:
        for xcd in range(XCDS):   # blocks are dealt to the XCDs in turn
            mine = out[xcd::XCDS]
            mine = mine[mine[:, 2] == 1, 0].astype(int)
            assert np.count_nonzero(np.diff(mine)) == (head_groups // XCDS - 1) * (active > 0)   # no way back to a head left
