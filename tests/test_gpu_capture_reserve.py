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


@pytest.mark.parametrize("n_q,splits", [(700, 1), (400, 3), (16, 28)])
def test_prefill_attn_smallest_workspace(device, n_q, splits):
    """Triples of every row in the splits that one round of the chip holds; a
    faster plan with more of them must not need more under capture."""
    child(f"""
n = {n_q} + 880
q, k, vt = rnd({n_q}, 24, 512), rnd(n, 4, 256), rnd(4, 256, (n + 63) // 64 * 64)
out = torch.zeros({n_q}, 24, 256, device=dev).half()
ops.workspace_reserve({n_q} * 24 * {splits} * 258 * 4)
check(lambda: ops.prefill_attn(q, k, vt, out, ld_vt=vt.shape[2], n_k=n, n_q={n_q}, vis0=881, H_q=24,
                               H_kv=4, scale=SCALE, check=False), out, 1e-3)
""")


@pytest.mark.parametrize("n", [600, 2000])
def test_layer_prefill_smallest_workspace(device, n):
    """A captured prompt with the workspace of a 128-token pass, against an
    eager one (other splits, so to fp16 rounding)."""
    child(f"""
lc, _ = layer_consts(5)
a, b = (KL.NativeKhqLayer(lc, H_q=24, H_kv=4, cap=4096, device=dev,
                          options=KL.KhqOptions(splits=8, fused=True)) for _ in range(2))
q, k, v = rnd({n}, 24, 512), rnd({n}, 4, 256), rnd({n}, 4, 256)
out, want = (torch.zeros({n}, 24, 256, device=dev).half() for _ in range(2))
a.prefill(q[:1], k[:1], v[:1], k[:1], out[:1], SCALE)  # the layer's own buffers
a.reset()
ops.workspace_reserve(128 * 24 * 10 * 258 * 4)
graph = torch.cuda.CUDAGraph()
with torch.cuda.graph(graph):
    a.prefill(q, k, v, k, out, SCALE)
b.prefill(q, k, v, k, want, SCALE)
torch.cuda.synchronize()
for _ in range(3):
    out.zero_()
    graph.replay()
    torch.cuda.synchronize()
    assert (out.float() - want.float()).abs().max() <= 1e-3 and out.abs().max() > 0
assert a.state() == b.state()
""")
