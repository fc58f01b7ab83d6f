"""Which (head group, template) a block of a sliced-Q launch takes, from the header the kernel uses, built for the host: every item once.
Tiles whose Q ranges share K/V: templates last to first, and no XCD between two head groups' K/V at a time."""
import ctypes
import os
import subprocess

import numpy as np
import pytest

from khalamari_amd.build import CSRC_DIR

XCDS = 8
SOURCE = """
#include "block_order.h"
extern "C" unsigned items(unsigned total, unsigned active, unsigned head_groups, int sole_reader, unsigned* out) {
    unsigned n = 0;
    const unsigned height = khm::head_groups_per_slice(head_groups);
    for (unsigned z = 0; z < khm::head_group_slices(head_groups); ++z)
        for (unsigned y = 0; y < height; ++y)
            for (unsigned x = 0; x < total; ++x, ++n) {
                const khm::WorkItem item = sole_reader ? khm::sole_reader_work_item(x, y, z, total, height, active, head_groups)
                                                       : khm::sliced_q_work_item(x, y, z, total, active, head_groups);
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


def items_of(order, total, active, head_groups, sole_reader):
    """Rows (head group, template, live) of the launch's blocks in the order the hardware starts them."""
    out = np.zeros(((head_groups + XCDS) * total, 3), dtype=np.uint32)
    blocks = order.items(total, active, head_groups, sole_reader, out.ctypes.data_as(ctypes.c_void_p))
    assert blocks <= len(out)
    out = out[:blocks].astype(int)
    live = out[out[:, 2] == 1]
    assert sorted(map(tuple, live[:, :2])) == [(h, t) for h in range(head_groups) for t in range(active)]
    return out


HEAD_GROUPS = pytest.mark.parametrize("head_groups", [1, 2, 3, 4, 8, 9, 12, 16, 20, 32, 64])
COUNTS = pytest.mark.parametrize("active,total", [(0, 3), (1, 1), (1, 5), (7, 7), (24, 24), (23, 40), (64, 64), (9, 4)])


@HEAD_GROUPS
@COUNTS
def test_head_groups_one_after_the_other(order, head_groups, active, total):
    active_in_table = min(active, total)   # a replayed count beyond the shape
    out = items_of(order, total, active_in_table, head_groups, 0)
    if active > total:
        beyond = np.zeros(((head_groups + XCDS) * total, 3), dtype=np.uint32)
        blocks = order.items(total, active, head_groups, 0, beyond.ctypes.data_as(ctypes.c_void_p))
        assert np.array_equal(out, beyond[:blocks])
    if head_groups <= XCDS:
        assert np.all(out[:active_in_table * head_groups, 2] == 1)   # the padding comes last
    live = out[out[:, 2] == 1]
    for h in range(head_groups):
        assert np.all(np.diff(live[live[:, 0] == h, 1]) == -1)
    if head_groups % XCDS == 0:
        for xcd in range(XCDS):   # blocks are dealt to the XCDs in turn
            mine = out[xcd::XCDS]
            mine = mine[mine[:, 2] == 1, 0]
            assert np.count_nonzero(np.diff(mine)) == (head_groups // XCDS - 1) * (active > 0)   # no way back to a head left


@pytest.mark.parametrize("head_groups", [3, 7, 9, 12, 20])
def test_sole_readers_of_other_counts_go_head_groups_fastest(order, head_groups):
    assert np.array_equal(items_of(order, 40, 23, head_groups, 1), items_of(order, 40, 23, head_groups, 0))


@pytest.mark.parametrize("head_groups", [1, 2, 4, 8, 16, 32, 64])
@COUNTS
def test_sole_readers_take_runs_of_the_head_major_list(order, head_groups, active, total):
    out = items_of(order, total, min(active, total), head_groups, 1)
    if active > total:
        beyond = np.zeros(((head_groups + XCDS) * total, 3), dtype=np.uint32)
        blocks = order.items(total, active, head_groups, 1, beyond.ctypes.data_as(ctypes.c_void_p))
        assert np.array_equal(out, beyond[:blocks])
        active = total
    items = active * head_groups
    assert np.all(out[:items, 2] == 1)
    for xcd in range(XCDS):
        run = out[xcd:items // XCDS * XCDS:XCDS]
        assert np.all(np.diff(run[:, 0] * active + active - 1 - run[:, 1]) == 1)
