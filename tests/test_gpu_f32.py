"""GPU parity of the fp32 layer and seam on the fp32 matrix kernels (csrc/gemm_f32.hip, gate_f32_kernel): tile
edges, K and N remainders, the element-wise loads of unaligned sizes, split and whole weight gradients.

Bar: that of the golden fp32 fixtures, 1e-5 relative to each tensor's scale (sums of at most a few thousand fp32
products in another order than the CPU's differ by a few 1e-6 of the scale)."""
import pytest
import torch

from oracle import moe_ref as R
from tests import _cases as CS
from tests.test_gpu_backward import _close, _run
from tests.test_gpu_forward import _layer_raw

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("T,D,E,I,k,S,I_s", [
    (1, 64, 4, 128, 2, 1, 128),         # one token
    (65, 68, 5, 36, 2, 1, 100),         # K and N remainders, 16-byte chunks
    (130, 100, 8, 64, 3, 2, 72),        # two shared segments that no K slab fits
    (257, 66, 4, 30, 2, 1, 34),         # sizes that take the element-wise loads
    (96, 63, 3, 33, 2, 1, 31),          # odd sizes: the FMA gate too
    (300, 256, 40, 96, 2, 0, 0),        # no shared expert, experts over two gate tiles
    (520, 132, 130, 64, 2, 1, 64),      # experts without rows, eight gate tiles
    (1100, 256, 8, 128, 2, 1, 128),     # split shared weight gradients
], ids=str)
def test_layer_forward_and_backward(T, D, E, I, k, S, I_s):
    case = CS.Case("f32", T, D, E, I, k, S, I_s, torch.float32, "normal", 1.5)
    x, p, dy = CS.make_inputs(case, with_dy=True)
    out = _run(x, p.gate_w, p.gate_bias, p.w1, p.w2, p.w3, p.sw1, p.sw2, p.sw3, k, 1.5, dy)
    ref = R.moe_forward_backward_ref(x, p, k, dy, route_scale=1.5, indices=out["idx"])
    own = R.moe_forward_backward_ref(x, p, k, dy, route_scale=1.5)
    assert torch.equal(out["idx"].sort(1)[0], own["indices"].sort(1)[0])
    for name in ("y", "dx", "dgate_w"):
        _close(out[name], ref[name], 1e-5, 1e-5 * ref[name].abs().max().item(), name)
    for name in ("dw1", "dw2", "dw3", "dsw1", "dsw2", "dsw3"):
        if ref[name]:
            b = torch.stack(ref[name])
            _close(torch.stack(out[name]), b, 1e-5, 1e-5 * b.abs().max().item(), name)


def test_unaligned_weights_take_the_element_loads():
    """Weights that are views four bytes past a 16-byte boundary: same result as aligned ones, to rounding."""
    T, D, E, I, k = 100, 64, 4, 128, 2
    x, p, dy = CS.make_inputs(CS.Case("f32", T, D, E, I, k, 1, 128, torch.float32), with_dy=True)

    def shift(t):
        buf = torch.empty(t.numel() + 1, dtype=t.dtype, device="cuda:0")
        v = buf[1:].view(t.shape)
        v.copy_(t)
        return v

    from dsmoe import moe_layer
    dev = lambda ts: [t.to("cuda:0") for t in ts]
    sh = lambda ts: [shift(t) for t in ts]
    gw, gb = p.gate_w.to("cuda:0"), p.gate_bias.to("cuda:0")
    with torch.no_grad():
        a = moe_layer(x.to("cuda:0"), gw, gb, *map(dev, (p.w1, p.w2, p.w3, p.sw1, p.sw2, p.sw3)), k=k)
        b = moe_layer(shift(x), shift(gw), gb, *map(sh, (p.w1, p.w2, p.w3, p.sw1, p.sw2, p.sw3)), k=k)
    assert torch.equal(a[1], b[1])
    _close(a[0].cpu(), b[0].cpu(), 1e-5, 1e-5 * a[0].abs().max().item(), "y")


@pytest.mark.parametrize("T,D,E,k", [(1, 64, 4, 2), (33, 8, 20, 4), (2048, 768, 20, 4), (300, 256, 40, 2), (65, 68, 97, 3),
                                     (520, 132, 200, 2), (70, 2052, 130, 9), (96, 63, 3, 3)], ids=str)
def test_the_gate_alone_equals_the_layers(T, D, E, k):
    """dsmoe_gate_fwd and the gate inside dsmoe_moe_fwd on fp32 x: the same logits bit for bit, hence the same experts,
    order and weights, near ties included."""
    from dsmoe import ops
    case = CS.Case("gate", T, D, E, 32, k, 0, 0, torch.float32, "normal", 1.5)
    x, p, _ = CS.make_inputs(case)
    dev = lambda t: t.to("cuda:0")
    gate = ops.gate_forward(dev(x), dev(p.gate_w), dev(p.gate_bias), k, 1.5, want_logits=True)
    layer = _layer_raw(case, x, p)
    for name in ("logits", "idx", "weights", "counts"):
        assert (gate[name].cpu().numpy() == layer[name]).all(), name
