"""What a step of the matrix-state scans allocates (sizes only: no GPU)."""
import pytest

from dli_amd import ops


@pytest.mark.parametrize("H,D,Dv", [(32, 128, 128), (4, 256, 256), (3, 17, 33)])
def test_delta_rule_workspace_grows_with_tiles_only(H, D, Dv):
    size = lambda seqs, tiles: ops.hip().gm_scan_workspace_bytes(8192, seqs, tiles, H, D, Dv, True)
    up = lambda n: (n + 15) // 16 * 16
    row = 4 * H * (64 * 64 + 3 * 64 * up(D) + 64 * up(Dv) + up(D))       # scores, queries, keys twice, values, decays
    assert size(512, 130) - size(512, 30) == 100 * row
    assert size(512, 130) - size(2, 130) == 4 * 510                       # a batch row: one entry of the table
    assert ops.hip().gm_scan_workspace_bytes(8192, 512, 640, H, 512, Dv, True) == 0      # past the block kernels: none
