"""Rules that choose a kernel, as far as they run without a GPU."""
import os
import subprocess
import sys

import pytest
import torch

from dli_amd import ops

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def _moe_rows(env, *args):
    code = f"from dli_amd import ops; print(*[ops.hip().moe_tile_rows(*a) for a in {args!r}])"
    e = {**os.environ, **env}
    return [int(x) for x in subprocess.run([sys.executable, "-c", code], cwd=ROOT, env=e, capture_output=True, text=True, check=True).stdout.split()]


@pytest.mark.parametrize("asked", ["96", "-5", "128"])
def test_expert_row_tiles_are_ones_that_a_kernel_has(asked):
    """The experts' GEMMs align rows to this number and launch the tile of that size: any other value would be tiles past the rows."""
    H = 4096
    calls = (0, 8, H, True), (0, 4000, H, True), (0, 4000, H, False), (32, 4000, H, True), (64, 8, H, True), (256, 8, H, True), (256, 8, H, False)
    assert _moe_rows({"DLI_MOE_TILE": asked}, *calls) == [128, 128, 128, 32, 64, 256, 128]


@pytest.mark.parametrize("hidden", [512, 1920, 2048, 4096])
def test_expert_row_tiles_by_rows_and_by_choice(hidden):
    """Up to 53 rows the streaming tiles, from 128 the 256² ones where they fit; between the two those of 256 rows only for wide layers."""
    rule = ops.hip().moe_tile_rows
    between = 256 if hidden >= 2048 else 128
    for rows, want in ((0, 32), (1, 32), (20, 32), (21, 64), (53, 64), (54, between), (127, between), (128, 256), (10 ** 6, 256)):
        assert rule(0, rows, hidden, True) == want and rule(0, rows, hidden, False) == min(want, 128)
        for given in (32, 64, 128, 48, 7, -1):
            assert rule(given, rows, hidden, True) == (given if given in (32, 64) else 128)
        assert rule(256, rows, hidden, True) == 256 and rule(256, rows, hidden, False) == 128
