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
    calls = (0, 8, True), (0, 4000, True), (0, 4000, False), (32, 4000, True), (64, 8, True), (256, 8, True), (256, 8, False)
    assert _moe_rows({"DLI_MOE_TILE": asked}, *calls) == [128, 128, 128, 32, 64, 256, 128]


def test_expert_row_tiles_by_rows_and_by_choice():
    rule = ops.hip().moe_tile_rows
    for rows in (0, 1, 20, 21, 53, 54, 127, 128, 10 ** 6):
        assert rule(0, rows, True) in (32, 64, 256) and rule(0, rows, False) in (32, 64, 128)
        for given in (32, 64, 128, 48, 7, -1):
            assert rule(given, rows, True) == (given if given in (32, 64) else 128)
        assert rule(256, rows, True) == 256 and rule(256, rows, False) == 128
