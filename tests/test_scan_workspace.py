"""What a step of the matrix-state scans allocates, and that the cache leaves room for it (sizes only: no GPU)."""
import types

import pytest

from dli_amd import ops
from dli_amd.config import EngineConfig, SchedulerConfig, get_model_config
from dli_amd.models.mixers import scan_workspace_bytes
from dli_amd.runtime.model_runner import ModelRunner


@pytest.mark.parametrize("H,D,Dv", [(32, 128, 128), (4, 256, 256), (3, 17, 33)])
def test_delta_rule_workspace_grows_with_tiles_only(H, D, Dv):
    size = lambda seqs, tiles: ops.hip().gm_scan_workspace_bytes(8192, seqs, tiles, H, D, Dv, True)
    up = lambda n: (n + 15) // 16 * 16
    row = 4 * H * (64 * 64 + 3 * 64 * up(D) + 64 * up(Dv) + up(D))       # scores, queries, keys twice, values, decays
    assert size(512, 130) - size(512, 30) == 100 * row
    assert size(512, 130) - size(2, 130) == 4 * 510                       # a batch row: one entry of the table
    assert ops.hip().gm_scan_workspace_bytes(8192, 512, 640, H, 512, Dv, True) == 0      # past the block kernels: none


def test_cache_leaves_room_for_the_scans():
    reserve = lambda model, stateful: ModelRunner._step_reserve(types.SimpleNamespace(
        cfg=EngineConfig(model=model, sched=SchedulerConfig(max_num_seqs=512, max_num_batched_tokens=8192)), stateful=stateful,
        ctx=types.SimpleNamespace(tp_size=1)))
    for name, kind, delta in (("tiny-nefarax", "delta", True), ("tiny-mozalix", "channel_delta", True)):
        m = get_model_config(name)
        spec = next(p for s in m.layer_specs for p in (s, *s.parts) if p.kind == kind)
        alone = ops.hip().gm_scan_workspace_bytes(8192, 512, 8192 // 64 + 512, spec.heads, spec.dim, spec.vdim, delta)
        want = scan_workspace_bytes(m.layer_specs, 8192, 512)
        assert want >= alone > 0
        assert reserve(m, True) - reserve(m, False) == 2 * want
