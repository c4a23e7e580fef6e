"""Calls under HIP graph capture with no more workspace than their partition
needs: a captured call cannot grow the library's workspace, so one that suffices
for a call's smallest partition has to go on sufficing.  The workspace only ever
grows, so each check runs in a child process of its own, which captures, replays
three times with eager calls between, and compares with the eager result."""
import os
import subprocess
import sys

import pytest

pytestmark = pytest.mark.gpu

CHILD = """
import sys
sys.path[:0] = {path!r}
import torch
from khq import ops, _lib, layer as KL
from khqdata import layer_consts
dev, SCALE = "cuda", 1 / 16
def rnd(*shape):
    return torch.randn(*shape, generator=gen, device=dev).half()
gen = torch.Generator(device=dev).manual_seed(3)
def check(fn, out, tol):
    # fn launches once on static buffers and returns its code
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        rc = fn()
    assert rc == 0, rc
    for _ in range(3):
        out.zero_()
        graph.replay()
        torch.cuda.synchronize()
        got = out.float().clone()
        assert fn() == 0
        torch.cuda.synchronize()
        assert (got - out.float()).abs().max() <= tol and got.abs().max() > 0
{body}
print("ok")
"""


def child(body):
    path = [p for p in sys.path if p]
    r = subprocess.run([sys.executable, "-c", CHILD.format(path=path, body=body)], capture_output=True,
                       text=True, timeout=100)
    assert r.returncode == 0 and r.stdout.strip().endswith("ok"), r.stdout + r.stderr


@pytest.mark.parametrize("H_q,H_kv,length", [(8, 1, 8192), (16, 2, 4096), (64, 8, 1000)])
def test_fp16_attention_smallest_workspace(device, H_q, H_kv, length):
    """8 x 512 or 16 x 256 parts of 258 floats are past the 4 MiB that the
    smallest reserve allocates; 256, 254 and 64 parts are not."""
    child(f"""
H_q, H_kv, n = {H_q}, {H_kv}, {length}
q, k, v = rnd(H_q, 512), rnd(n, H_kv, 256), rnd(n, H_kv, 256)
out, tri = torch.zeros(H_q, 256, device=dev).half(), torch.zeros(H_q, 258, device=dev)
ops.workspace_reserve(1)
check(lambda: ops.window_attn(q, k, v, tri, win_start=5, win_len=n, ring_cap=n, H_q=H_q, H_kv=H_kv,
                              scale=SCALE, check=False), tri, 0)
ops.workspace_reserve(min(256, (n + 7) // 8) * H_q * 258 * 4)
check(lambda: ops.gqa_attn(q, k, v, out, seq_len=n, H_q=H_q, H_kv=H_kv, scale=SCALE, check=False), out, 0)
""")
