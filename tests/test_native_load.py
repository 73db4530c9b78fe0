"""The native libraries arriving after the package's import (built later in
the same process), in a fresh interpreter that first looks for them elsewhere."""
import os
import subprocess
import sys

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

PRELUDE = """
import sys
sys.path.insert(0, {pkg!r})
import torch
from torch._subclasses.fake_tensor import FakeTensorMode
from gmdn_amd import _native
real = _native.{attr}
_native.{attr} = real + ".missing"
import fast_scan
from gmdn_amd import chunk, mixer, scan, wy
op = torch.ops.gmdn
with FakeTensorMode():
    U, a = torch.empty(1, 2, 3, 64, 64, device="cuda"), torch.empty(1, 2, 3, device="cuda")
    q, g = torch.empty(1, 2, 128, 64, device="cuda", dtype=torch.bfloat16), torch.empty(1, 2, 128, device="cuda")
net, x = mixer.FastWeightMixer(128, 2, "muon"), torch.zeros(1, 128, 128)
"""


def _run(body, attr="LIB_PATH"):
    code = PRELUDE.format(pkg=os.path.join(ROOT, "gmdn-gated-muon-deltanet_amd"), attr=attr) + body
    r = subprocess.run([sys.executable, "-c", code], capture_output=True, text=True, timeout=300)
    assert r.returncode == 0, r.stderr


@pytest.mark.parametrize("attr", ["LIB_PATH", "OPS_PATH"])
def test_every_entry_point_names_the_missing_library(attr):
    _run("""
calls = (lambda: chunk.chunk_scan(q, q, q, g, g, rule="delta"), lambda: wy.wy_scan(q, q, q, g, g),
         lambda: scan.hip_state_scan(U, U, a, a, a, a, 0, 3), lambda: scan.HipScan.apply(U, U, a, a, a, a, 0, 3),
         lambda: net(x), lambda: fast_scan.fast_state_scan(U, U, a, a, a, a, 0, 3))
for i, call in enumerate(calls):
    try:
        call()
    except RuntimeError as e:
        assert ".missing" in str(e) + str(e.__cause__), (i, e)
    else:
        raise AssertionError(i)
""", attr)


def test_late_load_registers_fakes_and_keeps_the_precision():
    _run("""
scan.set_precision("ieee")
assert not _native.available()
_native.LIB_PATH = real
assert wy.ops.ensure() is None and wy.ops.REGISTERED
U = torch.empty(1, 2, 3, 64, 64, device="meta")
a = torch.empty(1, 2, 3, device="meta")
assert op.state_scan(U, U, a, a, a, a, 1, 3, 0, True)[1].shape == U.shape
from torch.fx.experimental.proxy_tensor import make_fx

def step(q, g):
    q = q.detach().requires_grad_()
    return torch.autograd.grad(op.chunk_fwd(q, q, q, g, g, g, None, 1, 3, 1e-6, True)[0].float().sum(), q)

gm = make_fx(step)(torch.empty(1, 2, 128, 64, device="meta", dtype=torch.bfloat16), torch.empty(1, 2, 128, device="meta"))
args = [n.args for n in gm.graph.nodes if "chunk_bwd_muon" in str(n.target)][0]
assert args[-1] == _native.PREC_IEEE, args
with FakeTensorMode():
    U, a = torch.empty(1, 2, 3, 64, 64, device="cuda"), torch.empty(1, 2, 3, device="cuda")
    assert fast_scan.fast_state_scan(U, U, a, a, a, a, 0, 3).shape == U.shape
""")
