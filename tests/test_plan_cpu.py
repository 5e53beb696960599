"""CPU: the default plan of the tiled decode path keeps the kernel's limits over all its inputs."""

from __future__ import annotations

import math
import os

import pytest
import torch

from flashspec_amd import triton_utils
from flashspec_amd.triton_utils import plan_rows


@pytest.mark.parametrize("head_dim,max_waves,per_channel,group", [  # tile groups: per-channel stores
    (64, 16, False, 1), (64, 8, False, 1), (128, 16, False, 1), (256, 8, False, 1), (128, 8, True, 1),
    (128, 8, True, 2), (64, 8, True, 4), (128, 8, True, 8), (128, 8, True, 64)])
def test_plans_cover_the_row_within_the_limits(head_dim, max_waves, per_channel, group):
    for seq_len in (1, 16, 17, 300, 1024, 4095, 4096, 9000, 65536, 200000):
        for rows in (1, 7, 24, 72, 88, 96, 113, 114, 128, 129, 160, 192, 255, 256, 257, 511, 512, 5000):
            for light, full_rows in ((False, False), (True, False), (False, True), (True, True)):
                split, n, waves = plan_rows(seq_len, rows, head_dim, 256, max_waves=max_waves, tile_group=group,
                                            light=light, per_channel=per_channel, full_rows=full_rows)
                tiles = -(-seq_len // 16)
                assert split >= 1 and n >= 1 and waves in (1, 2, 4, 8, 16) and waves <= max_waves
                assert split * n >= tiles > split * (n - 1)  # whole row, no empty split
                assert split % group == 0
                assert group * math.ceil(split // group / waves) <= 64  # tiles a wave holds


def test_plans_at_the_lines_of_the_rule():
    plan = lambda s, rows, d=128, **kw: plan_rows(s, rows, d, 256, **kw)  # noqa: E731
    assert plan(1008, 64) == (63, 1, 8) and plan(1024, 64) == (16, 4, 8)  # 63 and 64 tiles
    assert plan(4096, 85) == (86, 3, 8) and plan(4096, 86) == (128, 2, 8)  # floor of CUs / rows
    assert plan(16384, 8) == (64, 16, 8)  # sqrt(1024) / 2
    assert plan(4096, 128) == (128, 2, 8) and plan(4080, 129) == (255, 1, 8)
    assert plan(4096, 129) == (86, 3, 4) and plan(4096, 255) == (128, 2, 4)  # two 4-wave workgroups a CU
    assert plan(4096, 256) == (256, 1, 16) and plan(4096, 256, light=True) == (256, 1, 4)
    assert plan(2032, 512) == (127, 1, 8) and plan(2048, 512) == (128, 1, 16)
    assert plan(512, 64, 256, max_waves=8) == (16, 2, 4) and plan(512, 64) == (32, 1, 8)


def test_plans_of_rows_that_leave_cus_idle():
    def plan(tiles, rows, d=128, full_rows=False, **kw):
        return plan_rows(16 * tiles, rows, d, 256, max_waves=8 if d > 128 or kw.get("per_channel") else 16,
                         full_rows=full_rows, **kw)

    for full in (False, True):  # over half of the CUs: three splits, two of short rows, whole long and costly ones
        assert plan(512, 170, full_rows=full) == (171, 3, 4) and plan(511, 171, full_rows=full) == (256, 2, 4)
        assert plan(512, 171, full_rows=full) == (512, 1, 8) and plan(513, 255, full_rows=full) == (513, 1, 16)
        assert plan(256, 192, 256, full_rows=full) == (256, 1, 8)
        assert plan(256, 193, per_channel=True, full_rows=full) == (256, 1, 8)
        assert plan(1024, 128, full_rows=full) == (512, 2, 8)
    assert plan(512, 192, 64) == (256, 2, 8) and plan(512, 192, 64, full_rows=True) == (512, 1, 8)
    # rows of unlike length take more workgroups than CUs where that was measured to gain
    chan = {"per_channel": True}
    assert plan(96, 96, **chan) == (32, 3, 8) and plan(96, 96, full_rows=True, **chan) == (48, 2, 8)
    assert plan(95, 96, **chan) == (48, 2, 8) and plan(256, 80, **chan) == (86, 3, 8)
    assert plan(256, 52, **chan) == (52, 5, 8) and plan(256, 60, **chan) == (64, 4, 8)
    assert plan(256, 48, **chan) == (43, 6, 8) and plan(256, 48, full_rows=True, **chan) == (52, 5, 8)
    assert plan(256, 144, **chan) == (128, 2, 8) and plan(256, 144, full_rows=True, **chan) == (86, 3, 4)
    assert plan(256, 192, **chan) == (128, 2, 8) and plan(256, 192, full_rows=True, **chan) == (256, 1, 8)
    for dim in (64, 128, 256):
        assert plan(96, 88, dim) == (32, 3, 8) and plan(96, 88, dim, full_rows=True) == (48, 2, 8)
        assert plan(256, 96, dim) == (128, 2, 8)
    assert plan(511, 102) == (256, 2, 8) and plan(512, 102) == (103, 5, 4) and plan(512, 103) == (256, 2, 8)
    assert plan(512, 102, full_rows=True) == (256, 2, 8)
    assert plan(768, 113) == (256, 3, 16) and plan(768, 114) == (384, 2, 8) and plan(768, 96, 64) == (154, 5, 8)
    # light tiles on 4 waves: every CU, or nearly every one with full rows
    assert plan(512, 120, light=True) == (256, 2, 8) and plan(510, 120, light=True, full_rows=True) == (255, 2, 4)
    assert plan(512, 120, light=True, full_rows=True) == (256, 2, 8)
    assert plan(16, 256, light=True) == (16, 1, 4) and plan(16, 256) == (16, 1, 8)


@pytest.fixture()
def launch_plan(monkeypatch):
    """triton_utils.launch_plan for a GPU of 256 CUs with no knob set, and a setter of knobs."""

    from flashspec_amd import _lib

    _lib.require()  # the tiled-path rule is a host function of the library
    for key in triton_utils._PLAN_KNOBS:
        monkeypatch.delenv(key, raising=False)
    monkeypatch.setitem(triton_utils._CU_CACHE, 0, 256)
    triton_utils._launch_plan_cached.cache_clear()
    dev = torch.device("cuda", 0)
    yield (lambda seq, rows, dim=128, **kw: triton_utils.launch_plan(seq, rows, dim, 16, 16, dev, **kw),
           monkeypatch.setenv)
    triton_utils._launch_plan_cached.cache_clear()


@pytest.mark.parametrize("knob,value", [
    ("FLASHSPEC_BLOCK_N", "128"), ("FLASHSPEC_BLOCK_N", "16"), ("FLASHSPEC_BLOCK_N", "48"), ("FLASHSPEC_BLOCK_N", ""),
    ("FLASHSPEC_NUM_SPLITS", "0"), ("FLASHSPEC_NUM_SPLITS", "-1"), ("FLASHSPEC_NUM_SPLITS", "many"),
    ("FLASHSPEC_NUM_WARPS", "3"), ("FLASHSPEC_NUM_WARPS", "x")])
def test_knobs_that_force_nothing_leave_the_default_plan(launch_plan, knob, value):
    plan, setenv = launch_plan
    shapes = [(seq, rows, dim, light) for seq in (128, 1024, 4096, 16384) for rows in (8, 96, 128, 160, 256, 512)
              for dim in (64, 128, 256) for light in (False, True)]
    default = [plan(seq, rows, dim, light=light)[:4] for seq, rows, dim, light in shapes]
    setenv(knob, value)
    assert [plan(seq, rows, dim, light=light)[:4] for seq, rows, dim, light in shapes] == default


def test_knobs_that_force_a_plan_still_do(launch_plan):
    plan, setenv = launch_plan
    assert plan(4096, 96)[1:4] == (8, 128, 2)
    setenv("FLASHSPEC_NUM_WARPS", "4")
    assert plan(4096, 96)[1] == 4
    setenv("FLASHSPEC_NUM_SPLITS", "4")
    assert plan(4096, 96)[1:4] == (4, 64, 4)


def test_knobs_are_read_from_the_environ_in_place(launch_plan, monkeypatch):
    plan, _ = launch_plan
    assert plan(4096, 96)[3] == 2
    monkeypatch.setattr(os, "environ", {**os.environ, "FLASHSPEC_NUM_SPLITS": "4"})
    assert plan(4096, 96)[3] == 4
    os.environ["FLASHSPEC_NUM_SPLITS"] = "3"
    assert plan(4096, 96)[3] == 3


def test_caches_built_on_the_host_know_whether_their_rows_are_full():
    from flashspec_amd import PagedKVAllocator, PagedKVCache

    k = torch.zeros((4, 2, 32, 16))
    full = lambda lengths: PagedKVCache.from_dense(k, k, 16, lengths=lengths).full_rows  # noqa: E731
    assert full(None) and full(torch.tensor([32, 32, 32, 0])) and not full(torch.tensor([32, 32, 31, 0]))
    cache = PagedKVCache.from_dense(k, k, 16)
    step = torch.zeros((4, 2, 1, 16))
    assert cache.append(step, step).full_rows
    assert not PagedKVCache.from_dense(k, k, 16, lengths=torch.tensor([32, 1, 1, 1])).append(step, step).full_rows
    pool = PagedKVAllocator(capacity_blocks=16, heads=2, head_dim=16)
    for rid, n in enumerate((32, 30, 2)):
        pool.add_request(rid, k[:1, :, :n], k[:1, :, :n])
    assert pool.to_cache([0, 1]).full_rows and not pool.to_cache([0, 2]).full_rows
    old = PagedKVCache.from_dense(k, k, 16)
    del old.__dict__["full_rows"]  # as unpickled from before the field
    assert not old.full_rows
    assert not PagedKVCache(cache.k_quant, cache.v_quant, cache.block_table, cache.lengths, 16, 32).full_rows
    for bad in ([33, 1, 1, 1], [1, -1, 1, 1], [1, 1, 1]):
        with pytest.raises(ValueError):
            full(torch.tensor(bad))
