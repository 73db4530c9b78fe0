"""CPU checks of the registered operators (torch.ops.gmdn.*): registration,
shape-only fake implementations, and whole-graph capture by torch.compile
(the reference trainer compiles its model, train_ablation.py:420-422) on
fake GPU tensors, so nothing runs on a device."""
import os
import sys

import pytest
import torch
from torch._subclasses.fake_tensor import FakeTensorMode

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
sys.path.insert(0, os.path.join(ROOT, "gmdn-gated-muon-deltanet_amd"))

import fast_scan  # noqa: E402
from gmdn_amd import _native, chunk, ops  # noqa: E402,F401

OPS = ("state_scan", "state_scan_bwd", "chunk_fwd", "chunk_bwd", "chunk_bwd_muon", "front_fwd", "front_bwd", "msign")


def _capture(fn, *args):
    """torch.compile(fullgraph=True) of fn on fake tensors; the captured graph's call targets."""
    graphs = []

    def backend(gm, example_inputs):
        graphs.append(gm)
        return gm.forward

    torch._dynamo.reset()
    out = torch.compile(fn, backend=backend, fullgraph=True)(*args)
    assert len(graphs) == 1
    return out, [str(n.target) for n in graphs[0].graph.nodes if n.op == "call_function"]


def test_ops_registered():
    for name in OPS:
        assert hasattr(torch.ops.gmdn, name), name


@pytest.mark.parametrize("rule", [0, 1, 2])
def test_state_scan_compiles_to_one_graph(rule):
    with FakeTensorMode():
        U, K = (torch.empty(2, 3, 4, 64, 64, device="cuda") for _ in range(2))
        g = [torch.empty(2, 3, 4, device="cuda") for _ in range(4)]
        out, targets = _capture(lambda *x: fast_scan.fast_state_scan(*x, rule, 3) * 2, U, K, *g)
    assert "gmdn.state_scan" in targets
    assert tuple(out.shape) == (2, 3, 4, 64, 64) and out.dtype == torch.float32


@pytest.mark.parametrize("rule,d", [("delta", 128), ("adam", 64), ("muon", 64)])
def test_chunk_scan_compiles_to_one_graph(rule, d):
    with FakeTensorMode():
        q, k, v = (torch.empty(1, 2, 128, d, device="cuda", dtype=torch.bfloat16) for _ in range(3))
        gates = [torch.empty(1, 2, 128, device="cuda") for _ in range(4)]
        out, targets = _capture(lambda *x: chunk.chunk_scan(*x, rule=rule, ns=3), q, k, v, *gates)
    # every rule's forward is the one fused operator
    assert "gmdn.chunk_fwd" in targets
    assert tuple(out.shape) == (1, 2, 128, d) and out.dtype == torch.bfloat16


def test_fake_shapes():
    with FakeTensorMode():
        U, K = (torch.empty(2, 3, 4, 32, 32, device="cuda") for _ in range(2))
        g = [torch.empty(2, 3, 4, device="cuda") for _ in range(4)]
        for rule, moments in ((0, 0), (1, 1), (2, 2)):
            S, M, V = torch.ops.gmdn.state_scan(U, K, *g, rule, 3, 0, True)
            assert S.shape == U.shape
            assert [t.numel() > 0 for t in (M, V)] == [moments >= 1, moments >= 2]
            S, M, V = torch.ops.gmdn.state_scan(U, K, *g, rule, 3, 0, False)
            assert M.numel() == 0 and V.numel() == 0
        grads = torch.ops.gmdn.state_scan_bwd(U, K, *g, U, U, U, U, 2, 3, 0)
        assert [tuple(t.shape) for t in grads] == [tuple(U.shape)] * 2 + [(2, 3, 4)] * 4

        q, k, v = (torch.empty(2, 4, 256, 128, device="cuda", dtype=torch.bfloat16) for _ in range(3))
        beta, gg = (torch.empty(2, 4, 256, device="cuda") for _ in range(2))
        o, states = torch.ops.gmdn.chunk_fwd(q, k, v, beta, gg, None, None, 0, 3, 1e-6, True)
        assert o.shape == q.shape and o.dtype == torch.bfloat16
        # the delta checkpoint holds one d x d fp32 state per (b, h, even chunk)
        assert states.numel() == 2 * 4 * ((256 // 64 + 1) // 2) * 128 * 128
        o, states = torch.ops.gmdn.chunk_fwd(q, k, v, beta, gg, None, None, 0, 3, 1e-6, False)
        assert states.numel() == 0
        dq, dk, dv, db, dg, dgmu, dgnu = torch.ops.gmdn.chunk_bwd(q, k, v, beta, gg, None, None, states, q,
                                                                 0, 3, 1e-6)
        assert dq.shape == q.shape and dq.dtype == torch.bfloat16 and db.shape == beta.shape
        assert dgmu.numel() == 0 and dgnu.numel() == 0
        # a head-interleaved (B, T, H, d) stream keeps its strides in the gradients
        qi = torch.empty(2, 256, 4, 128, device="cuda", dtype=torch.bfloat16).transpose(1, 2)
        dqi = torch.ops.gmdn.chunk_bwd(qi, qi, qi, beta, gg, None, None, states, q, 0, 3, 1e-6)[0]
        assert dqi.stride() == qi.stride()


def test_cpu_tensors_never_reach_the_ops():
    q = torch.zeros(1, 1, 64, 64, dtype=torch.bfloat16)
    gg = torch.zeros(1, 1, 64)
    with pytest.raises(RuntimeError, match="GPU tensors"):
        chunk.chunk_scan(q, q, q, gg, gg, rule="delta")


def test_front_fake_shapes():
    with FakeTensorMode():
        y = torch.empty(2, 100, 768, device="cuda", dtype=torch.bfloat16)
        w, b = torch.empty(768, 1, 4, device="cuda"), torch.empty(768, device="cuda")
        q, k, v = torch.ops.gmdn.front_fwd(y, w, b, 128)
        assert all(tuple(t.shape) == (2, 100, 256) and t.dtype == torch.bfloat16 for t in (q, k, v))
        dy, dw, db = torch.ops.gmdn.front_bwd(y, w, b, q, k, v, 128)
        assert dy.shape == y.shape and dw.shape == w.shape and db.shape == b.shape


def _meta_ops():
    """(name, call, differentiable inputs) of every forward operator, on meta tensors."""
    def t(*shape, dtype=torch.float32):
        return torch.empty(*shape, device="meta", dtype=dtype, requires_grad=True)

    U, K, a, b, m, n = t(1, 2, 3, 64, 64), t(1, 2, 3, 64, 64), *(t(1, 2, 3) for _ in range(4))
    q, k, v = (t(1, 2, 128, 64, dtype=torch.bfloat16) for _ in range(3))
    beta, g, mu, nu = (t(1, 2, 128) for _ in range(4))
    y, w, bias, hw = t(2, 70, 384), t(384, 1, 4), t(384), t(64)
    op = torch.ops.gmdn
    for r in range(3):
        yield f"state_scan-{r}", lambda *x, r=r: op.state_scan(*x, r, 3, 0, True), (U, K, a, b, m, n)
    yield "chunk_fwd-delta", lambda *x: op.chunk_fwd(*x, None, None, 0, 3, 1e-6, True), (q, k, v, beta, g)
    yield "chunk_fwd-muon", lambda *x: op.chunk_fwd(*x, None, 1, 3, 1e-6, True), (q, k, v, beta, g, mu)
    yield "chunk_fwd-adam", lambda *x: op.chunk_fwd(*x, 2, 3, 1e-6, True), (q, k, v, beta, g, mu, nu)
    yield "wy_fwd", lambda *x: op.wy_fwd(*x, True), (q, k, v, beta, g)
    yield "front_fwd", lambda *x: op.front_fwd(*x, 64), (y, w, bias)
    yield "gates_fwd", lambda x: op.gates_fwd(x, 128, 3), (y,)
    yield "head_norm_fwd", lambda *x: op.head_norm_fwd(*x, 1e-6), (q, hw)


@pytest.mark.parametrize("name", [x[0] for x in _meta_ops()])
def test_second_derivative_raises(name):
    """A gradient taken with create_graph=True is usable, and differentiating
    it again raises: the backward operators have no derivative of their own,
    and must not drop out of the graph."""
    _, call, xs = next(x for x in _meta_ops() if x[0] == name)
    out = call(*xs)
    out = out[0] if isinstance(out, tuple) else out
    grads = torch.autograd.grad(out.float().square().sum(), xs, create_graph=True)
    assert all(g.requires_grad for g in grads)
    for g in grads:
        with pytest.raises(RuntimeError, match="not implemented|no autograd formula"):
            torch.autograd.grad(g.float().square().sum(), xs, retain_graph=True, allow_unused=True)


def test_hip_scan_second_derivative_raises(monkeypatch):
    from gmdn_amd import scan
    monkeypatch.setattr(scan, "_check_inputs", lambda *x: None)  # (it wants GPU tensors)
    _, _, xs = next(_meta_ops())
    grads = torch.autograd.grad(scan.HipScan.apply(*xs, 1, 3).square().sum(), xs[:2], create_graph=True)
    with pytest.raises(RuntimeError, match="not implemented|no autograd formula"):
        torch.autograd.grad(grads[0].square().sum(), xs, allow_unused=True)


def test_operator_schemas():
    """Integers are symbolic and every operator is marked safe for torch.compile
    (only_allow_pt2_compliant_ops refuses the others)."""
    for name in OPS + ("wy_fwd", "wy_bwd", "gates_fwd", "gates_bwd", "head_norm_fwd", "head_norm_bwd"):
        op = getattr(torch.ops.gmdn, name).default
        assert torch.Tag.pt2_compliant_tag in op.tags, name
        assert ", int " not in str(op._schema), name


def test_traced_sizes_stay_symbolic():
    """A size of a traced input reaches the operators, and the backward's,
    without being specialised to a number."""
    from torch.fx.experimental.proxy_tensor import make_fx

    def step(y):
        y = y.detach().requires_grad_()
        out = torch.ops.gmdn.gates_fwd(y, y.shape[2] // 3, 3)
        return torch.autograd.grad(out.sum(), y)

    gm = make_fx(step, tracing_mode="symbolic")(torch.empty(2, 70, 24, device="meta"))
    nodes = {str(n.target): n for n in gm.graph.nodes if "gmdn" in str(n.target)}
    assert isinstance(nodes["gmdn.gates_fwd.default"].args[1], torch.fx.Node)
    assert isinstance(nodes["gmdn.gates_bwd.default"].args[2], torch.fx.Node)


@pytest.mark.parametrize("name", [x[0] for x in _meta_ops()])
def test_compiled_autograd_traces_the_backward(name):
    """torch's compiled autograd takes every operator's autograd function, and
    traces again when the product precision has changed."""
    from gmdn_amd import scan
    from torch._dynamo import compiled_autograd

    _, call, xs = next(x for x in _meta_ops() if x[0] == name)
    traces = []

    def compiler(gm):
        traces.append(gm)
        return torch.compile(gm, backend=lambda m, _: m.forward, fullgraph=True)

    def step():
        for t in xs:
            t.grad = None
        out = call(*xs)
        with compiled_autograd._enable(compiler):
            (out[0] if isinstance(out, tuple) else out).float().sum().backward()
        assert all(t.grad.shape == t.shape for t in xs)

    torch._dynamo.reset()
    compiled_autograd.reset()
    step()
    step()
    assert len(traces) == 1
    if name.startswith("chunk_fwd"):
        try:
            scan.set_precision("ieee")
            step()
        finally:
            scan.set_precision("tf32")
        assert len(traces) == 2


def test_operators_by_module_name():
    from gmdn_amd import wy
    for name in ("state_scan", "state_scan_bwd", "chunk_fwd", "chunk_bwd", "chunk_bwd_muon", "front_fwd", "front_bwd",
                 "gates_fwd", "gates_bwd", "head_norm_fwd", "head_norm_bwd", "msign"):
        assert callable(getattr(ops, name)), name
    q, g = torch.empty(1, 2, 128, 64, device="meta", dtype=torch.bfloat16), torch.empty(1, 2, 128, device="meta")
    o, ckpt = wy.wy_fwd(q, q, q, g, g, True)
    assert o.shape == q.shape and len(wy.wy_bwd(q, q, q, g, g, ckpt, o)) == 5
    with pytest.raises(AttributeError):
        ops.no_such_operator
