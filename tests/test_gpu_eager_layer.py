"""The eager layer path (ops._eager_layer: native argument scan, one autograd function) against the torch.library
operator it stands for: bitwise equal results for every form of call, the operator for whatever watches or transforms
operators, the operator path's errors for what it refuses."""
import pytest
import torch
from torch.utils._python_dispatch import TorchDispatchMode

from tests import _cases as CS

pytestmark = pytest.mark.gpu
DEV = torch.device("cuda:0")


def _args(dtype=torch.bfloat16, S=1, T=70, D=128, E=8, I=64, k=2, grad=True, seed=0):
    x, p, dy = CS.make_inputs(CS.Case("e", T, D, E, I, k, S, 96, dtype, "normal"), seed=seed, with_dy=True)
    leaf = lambda t: t.to(DEV).requires_grad_(grad)
    ws = [[leaf(t) for t in ts] for ts in (p.w1, p.w2, p.w3, p.sw1, p.sw2, p.sw3)]
    return leaf(x), leaf(p.gate_w), p.gate_bias.to(DEV), ws, dy.to(DEV)


class _Seen(TorchDispatchMode):
    def __init__(self):
        super().__init__()
        self.names = []

    def __torch_dispatch__(self, func, types, args=(), kwargs=None):
        self.names.append(str(func))
        return func(*args, **(kwargs or {}))


def _step(x, gw, gb, ws, dy, operator, **kw):
    from dsmoe import moe_layer
    leaves = [x, gw, *[t for ts in ws for t in ts]]
    for t in leaves:
        t.grad = None
    if operator:
        with _Seen() as seen:
            out = moe_layer(x, gw, gb, *ws, k=2, **kw)
        assert any("dsmoe.moe_fwd" in n for n in seen.names)
    else:
        out = moe_layer(x, gw, gb, *ws, k=2, **kw)
    if out[0].requires_grad:
        out[0].backward(dy)
    return [t.detach() for t in out], [t.grad for t in leaves]


def _same(a, b):
    return (a is None) == (b is None) and (a is None or (a.dtype == b.dtype and torch.equal(a, b)))


@pytest.mark.parametrize("dtype,S", [(torch.bfloat16, 1), (torch.bfloat16, 0), (torch.float32, 2)])
@pytest.mark.parametrize("frozen", ["none", "x", "weights", "all"])
def test_equals_the_operator(dtype, S, frozen):
    x, gw, gb, ws, dy = _args(dtype, S)
    if frozen in ("x", "all"):
        x.requires_grad_(False)
    if frozen in ("weights", "all"):
        for t in (gw, *[t for ts in ws for t in ts]):
            t.requires_grad_(False)
    a, ga = _step(x, gw, gb, ws, dy, False)
    b, gb_ = _step(x, gw, gb, ws, dy, True)
    assert all(map(_same, a, b)) and all(map(_same, ga, gb_))
    with torch.no_grad():
        c, _ = _step(x, gw, gb, ws, dy, False)
        d, _ = _step(x, gw, gb, ws, dy, True)
    assert all(map(_same, c, d)) and all(map(_same, a[1:], c[1:]))


def test_strided_inputs_and_mixed_strides():
    x, gw, gb, ws, dy = _args()
    xt = x.detach().t().contiguous().t().requires_grad_()
    ws[1][3] = ws[1][3].detach().t().contiguous().t().requires_grad_()     # one weight with other strides
    a, ga = _step(xt, gw, gb, ws, dy, False)
    b, gb_ = _step(xt, gw, gb, ws, dy, True)
    assert all(map(_same, a, b)) and all(map(_same, ga, gb_))


def test_master_weights():
    x, gw, gb, ws, dy = _args()
    flat = [t for ts in ws for t in ts]
    masters = [t.detach().float().requires_grad_() for t in flat]
    for t in flat:
        t.requires_grad_(False)
    _step(x, gw, gb, ws, dy, False, master_weights=masters)
    a = [m.grad.clone() for m in masters]
    for m in masters:
        m.grad = None
    _step(x, gw, gb, ws, dy, True, master_weights=masters)
    assert all(torch.equal(p, m.grad) and p.dtype == torch.float32 for p, m in zip(a, masters))


def test_saved_tensor_hooks_and_backward_under_a_mode():
    x, gw, gb, ws, dy = _args()
    want = _step(x, gw, gb, ws, dy, False)[1]
    packed = []
    with torch.autograd.graph.saved_tensors_hooks(lambda t: packed.append(t.shape) or t.clone(), lambda t: t.clone()):
        got = _step(x, gw, gb, ws, dy, False)[1]
    assert len(packed) == 3 + sum(map(len, ws)) and all(map(_same, want, got))
    with torch.autograd.graph.save_on_cpu():
        got = _step(x, gw, gb, ws, dy, False)[1]
    assert all(map(_same, want, got))
    from dsmoe import moe_layer
    for t in (x, gw, *[t for ts in ws for t in ts]):
        t.grad = None
    y = moe_layer(x, gw, gb, *ws, k=2)[0]
    with _Seen() as seen:
        y.backward(dy)
    assert any("dsmoe.moe_bwd" in n for n in seen.names)
    assert all(map(_same, want, [t.grad for t in (x, gw, *[t for ts in ws for t in ts])]))


def _other_strides(t):
    """An equal tensor, its elements two apart."""
    return torch.stack([t, t], -1)[..., 0]


@pytest.mark.parametrize("path", ["eager", "operator", "seam", "attention"])
def test_saved_tensors_that_come_back_with_other_strides(path):
    """A saved-tensor hook may hand back equal tensors of other strides: the same gradients.  Tensors on another device
    are an error, before any kernel."""
    from dsmoe import grouped_moe_dispatch
    from dsmoe.mla import mla_attention
    from tests.test_gpu_mla import _inputs
    hooks = torch.autograd.graph.saved_tensors_hooks
    g = torch.Generator(device=DEV).manual_seed(1)
    n = lambda *s: torch.randn(*s, generator=g, device=DEV).bfloat16().requires_grad_()
    if path in ("eager", "operator"):
        args = _args()
        run = lambda: _step(*args, path == "operator")[1]
    elif path == "seam":
        ins = (n(40, 64), n(3, 32, 64), n(3, 64, 32), n(3, 32, 64), n(40))
        off = torch.tensor([0, 7, 7, 40], device=DEV)
        run = lambda: torch.autograd.grad(grouped_moe_dispatch(*ins, off).float().square().sum(), ins)
    else:
        ins, sc = _inputs(2, 3, 70, 70, 64, 32, 16, 24, seed=1)
        ins = [t.requires_grad_() for t in ins]
        run = lambda: torch.autograd.grad(mla_attention(*ins, sc, is_causal=True).float().square().sum(), ins)
    want = run()
    with hooks(lambda t: t, _other_strides):
        got = run()
    assert all(map(_same, want, got))
    with hooks(lambda t: t, lambda t: t.cpu() if t.dim() > 1 and t.dtype == torch.bfloat16 else t):
        with pytest.raises(RuntimeError, match="device"):
            run()


def test_no_gradient_of_gradients():
    x, gw, gb, ws, dy = _args()
    from dsmoe import moe_layer
    y = moe_layer(x, gw, gb, *ws, k=2)[0]
    (g,) = torch.autograd.grad(y, x, dy, create_graph=True)
    with pytest.raises(RuntimeError):
        g.float().sum().backward()


def test_training_flag_and_errors():
    from dsmoe import moe_layer
    x, gw, gb, ws, dy = _args()
    y = moe_layer(x, gw, gb, *ws, k=2, training=False)[0]
    with pytest.raises(RuntimeError, match="without saving activations"):
        y.backward(dy)
    with pytest.raises(ValueError, match="same number"):
        moe_layer(x, gw, gb, ws[0][:-1], *ws[1:], k=2)
    with pytest.raises(ValueError, match="weight dtype"):
        moe_layer(x, gw, gb, [t.float() for t in ws[0]], *ws[1:], k=2)
    with pytest.raises(ValueError, match="must be"):
        moe_layer(x, gw, gb, ws[1], *ws[1:], k=2)
    with pytest.raises(ValueError, match="n_activated_experts"):
        moe_layer(x, gw, gb, *ws, k=9)
    with pytest.raises(ValueError, match="gate weight"):
        moe_layer(x, gw.detach().bfloat16(), gb, *ws, k=2)


def test_module_reads_replaced_and_computed_weights():
    """The module's weights are looked up on every call: replaced parameters, data swapped in place, weights that a
    parametrisation computes."""
    import torch.nn.utils.parametrize as P
    from dsmoe import DeepSeekMoE
    m = DeepSeekMoE({"dim": 64, "n_routed_experts": 4, "n_shared_experts": 1, "moe_inter_dim": 32,
                     "n_activated_experts": 2}).to(DEV)
    x = torch.randn(33, 64, device=DEV)
    with torch.no_grad():
        a = m(x)
        m.experts[1].w1.weight = torch.nn.Parameter(m.experts[1].w1.weight * 2)
        m.shared_experts[0].w2.weight.data = m.shared_experts[0].w2.weight.data * 3
        b = m(x)
        again = m(x)
    assert not torch.equal(a, b) and torch.equal(b, again)

    class Twice(torch.nn.Module):
        def forward(self, w):
            return 2 * w

    P.register_parametrization(m.experts[0].w3, "weight", Twice())
    with torch.no_grad():
        c = m(x)
        P.remove_parametrizations(m.experts[0].w3, "weight")
        d = m(x)
    assert torch.equal(c, d) and not torch.equal(b, c)


def test_without_the_host_module(monkeypatch):
    """The layer without dsmoe/_host.so: the same results through the operators."""
    import sys

    import dsmoe._lib as L
    args = _args()
    want = _step(*args, False)
    monkeypatch.setattr(L, "_layer_fns", None)
    monkeypatch.setitem(sys.modules, "dsmoe._host", None)
    monkeypatch.delattr("dsmoe._host", raising=False)
    with pytest.warns(RuntimeWarning, match="_host.so"):
        got = _step(*args, False)
    assert all(map(_same, want[0], got[0])) and all(map(_same, want[1], got[1]))
