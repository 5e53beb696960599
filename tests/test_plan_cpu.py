"""CPU: the default plan of the tiled decode path keeps the kernel's limits over all its inputs."""

from __future__ import annotations

import math

import pytest

from flashspec_amd.triton_utils import plan_rows


@pytest.mark.parametrize("head_dim,max_waves,per_channel,group", [  # tile groups: per-channel stores
    (64, 16, False, 1), (64, 8, False, 1), (128, 16, False, 1), (256, 8, False, 1), (128, 8, True, 1),
    (128, 8, True, 2), (64, 8, True, 4), (128, 8, True, 8), (128, 8, True, 64)])
def test_plans_cover_the_row_within_the_limits(head_dim, max_waves, per_channel, group):
    for seq_len in (1, 16, 17, 300, 1024, 4095, 4096, 9000, 65536, 200000):
        for rows in (1, 7, 24, 96, 128, 129, 160, 192, 255, 256, 257, 511, 512, 5000):
            for light in (False, True):
                split, n, waves = plan_rows(seq_len, rows, head_dim, 256, max_waves=max_waves, tile_group=group,
                                            light=light, per_channel=per_channel)
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
