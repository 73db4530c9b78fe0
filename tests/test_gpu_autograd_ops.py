"""The C++ operators' autograd (csrc/torch_ops.cpp) under what reaches around
an operator: saved-tensor hooks, another stream, the precision setting, and
the error of a forward that recorded nothing."""
import pytest
import torch

from gmdn_amd import scan
from gmdn_amd.chunk import chunk_scan
from gmdn_amd.wy import wy_scan
from gmdn_amd.workloads import Workload, make_inputs

pytestmark = pytest.mark.gpu


def _dev():
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    return torch.device("cuda:0")


def _case(rule, dev):
    inp = make_inputs(Workload("t", "delta" if rule == "wy" else rule, 1, 2, 192, 64), seed=4, device=dev)
    names = ["q", "k", "v", "beta", "g"] + ["gmu"] * (rule in ("muon", "adam")) + ["gnu"] * (rule == "adam")
    xs = [inp[n].requires_grad_(True) for n in names]
    call = (lambda: wy_scan(*xs)) if rule == "wy" else (lambda: chunk_scan(*xs, rule=rule, ns=3))
    return xs, call, inp["dO"]


@pytest.mark.parametrize("rule", ["delta", "muon", "adam", "wy"])
def test_saved_tensor_hooks_and_side_stream(rule):
    dev = _dev()
    xs, call, dO = _case(rule, dev)
    want = torch.autograd.grad(call(), xs, dO)
    packed = []

    def pack(t):
        packed.append(t.numel())
        return t.cpu()

    with torch.autograd.graph.saved_tensors_hooks(pack, lambda t: t.to(dev)):
        o = call()
    assert len(packed) == len(xs) + 1  # the inputs and the checkpoint
    got = torch.autograd.grad(o, xs, dO)
    s = torch.cuda.Stream()
    s.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(s):
        side = torch.autograd.grad(call(), xs, dO)
    torch.cuda.current_stream().wait_stream(s)
    for a, b, c in zip(want, got, side):
        assert torch.equal(a, b) and torch.equal(a, c)


def test_precision_setting_reaches_the_backward():
    """Setting the precision between the forward and the backward selects the
    muon backward's Newton-Schulz products, as it does per call."""
    dev = _dev()
    xs, call, dO = _case("muon", dev)
    q, k, v, beta, g, gmu = (t.detach() for t in xs)
    with torch.no_grad():
        _, states = torch.ops.gmdn.chunk_fwd(q, k, v, beta, g, gmu, None, 1, 3, 1e-6, True)
    try:
        for name, code in (("ieee", 1), ("tf32", 0)):
            o = call()
            scan.set_precision(name)
            got = torch.autograd.grad(o, xs, dO)
            want = torch.ops.gmdn.chunk_bwd_muon(q, k, v, beta, g, gmu, states, dO, 3, code)
            assert all(torch.equal(a, b) for a, b in zip(got, want)), name
    finally:
        scan.set_precision("tf32")


def test_unrecorded_forward_has_no_backward():
    dev = _dev()
    xs, _, dO = _case("delta", dev)
    o, _ = torch.ops.gmdn.chunk_fwd(*xs, None, None, 0, 3, 1e-6, False)
    with pytest.raises(RuntimeError, match="without recording its state checkpoint"):
        torch.autograd.grad(o, xs, dO)
    with pytest.raises(RuntimeError, match="failed with code"):
        torch.ops.gmdn.chunk_fwd(*[t.detach()[..., :50, :] if t.dim() == 4 else t.detach() for t in xs], None, None, 0,
                                 3, 1e-6, False)


def test_wrong_ranks_are_refused():
    """An operator that takes its sizes from a tensor's leading dimensions
    refuses any other rank before it launches; a head norm of empty rows is an
    error, not a division by zero."""
    dev = _dev()
    op = torch.ops.gmdn
    U, g = torch.zeros(1, 2, 3, 64, 64, device=dev), torch.zeros(1, 2, 3, device=dev)
    for x in (U[0], U[None]):
        with pytest.raises(RuntimeError, match="5 dimensions"):
            op.state_scan(x, x, g, g, g, g, 0, 3, 0, False)
        with pytest.raises(RuntimeError, match="5 dimensions"):
            op.state_scan_bwd(x, x, g, g, g, g, x, x, x, x, 0, 3, 0)
    y, w, b = torch.zeros(2, 70, 384, device=dev), torch.zeros(384, 1, 4, device=dev), torch.zeros(384, device=dev)
    for x in (y[0], y[None]):
        with pytest.raises(RuntimeError, match="3 dimensions"):
            op.front_fwd(x, w, b, 64)
        with pytest.raises(RuntimeError, match="3 dimensions"):
            op.front_bwd(x, w, b, y, y, y, 64)
        with pytest.raises(RuntimeError, match="3 dimensions"):
            op.gates_fwd(x, 128, 3)
        with pytest.raises(RuntimeError, match="3 dimensions"):
            op.gates_bwd(x, x, 128, 3)
    e = torch.zeros(4, 0, device=dev)
    with pytest.raises(RuntimeError, match="empty"):
        op.head_norm_bwd(e, torch.zeros(0, device=dev), torch.zeros(4, device=dev), e)
