"""DLI_DECODE_NT=0: decode rows read the cache with plain loads, by themselves and beside prompt tiles, and give the same bits."""
import os
import subprocess
import sys

import pytest

pytestmark = pytest.mark.gpu

STEPS = """
import hashlib, torch
from torch.profiler import ProfilerActivity, profile
from test_mixed_launch_gpu import _step, ROWS
from dli_amd import ops
ops.attention_in_one_launch = lambda *a: True
for name, listed, dtype, prompts in (("tiles of one group", True, torch.bfloat16, [(2100, 2100)]), ("two groups", True, torch.float8_e4m3fn, [(500, 300)]),
                                     ("uniform ranges", False, torch.bfloat16, [(500, 300)]), ("rows alone", True, torch.bfloat16, [])):
    kc, vc, meta, qkv = _step(32, 8, dtype, ROWS, prompts, listed)
    call = lambda: ops.paged_attention(qkv, kc, vc, meta, 32, 8, 128, 0.088)
    call()
    torch.cuda.synchronize()
    with profile(activities=[ProfilerActivity.CPU, ProfilerActivity.CUDA]) as p:
        out = call()
        torch.cuda.synchronize()
    kernels = [e.name for e in p.events() if "paged_mixed_kernel" in e.name or "paged_decode_kernel" in e.name]
    print("STEP", name, "|", hashlib.sha1(out.view(torch.int16).cpu().numpy().tobytes()).hexdigest(), "|", kernels)
"""


def _run(**env):
    here = os.path.dirname(os.path.abspath(__file__))
    paths = [here, os.path.dirname(here)] + [os.environ[k] for k in ("PYTHONPATH",) if k in os.environ]
    r = subprocess.run([sys.executable, "-c", STEPS], env={**os.environ, "PYTHONPATH": os.pathsep.join(paths), **env}, capture_output=True, text=True, timeout=110)
    assert r.returncode == 0, r.stderr[-2000:]
    return [line.split("|") for line in r.stdout.splitlines() if line.startswith("STEP")]


def test_plain_loads_in_every_form():
    usual, plain = _run(), _run(DLI_DECODE_NT="0")
    assert len(usual) == len(plain) == 4
    for (name, bits, kernels), (_, plain_bits, plain_kernels) in zip(usual, plain):
        assert "true>" in kernels and "false>" not in kernels, (name, kernels)
        assert "false>" in plain_kernels and "true>" not in plain_kernels, (name, plain_kernels)      # (the loads are the last of the kernel's parameters)
        assert bits == plain_bits, name
