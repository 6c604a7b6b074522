"""Which kernels the layer's routed forward GEMMs take (dsmoe_moe_fwd_kernels, host code only), on both sides of each
line of the rules in csrc/api.hip."""
import ctypes

import pytest

OTHER, PERSISTENT, SMALL, FEW = range(4)


def _kernels(T, D, E, I, k, S, I_s, training=0, dtype=None):
    import dsmoe._lib as L
    if not L.LIB_PATH.exists():
        from dsmoe import build
        build.build(verbose=False)
    out = (ctypes.c_int32 * 2)()
    d = L.Dims(T, D, E, k, I, S, I_s, L.DSMOE_BF16 if dtype is None else dtype, 1.0)
    L.check(L.load().dsmoe_moe_fwd_kernels(ctypes.byref(d), training, out), "dsmoe_moe_fwd_kernels")
    return tuple(out)


WIDE = dict(D=2048, E=64, I=1408, k=6, S=2, I_s=1408)
SINGLE = dict(D=1024, E=16, I=512, k=4, S=1, I_s=1024)


@pytest.mark.parametrize("T,shape,training,want", [
    (1, WIDE, 0, (FEW, FEW)),
    (64, WIDE, 0, (FEW, FEW)),
    (333, WIDE, 0, (PERSISTENT, SMALL)),     # a nearly empty last round of 256-row down tiles
    (1150, WIDE, 0, (PERSISTENT, SMALL)),
    (1300, WIDE, 0, (PERSISTENT, PERSISTENT)),
    (8192, WIDE, 0, (PERSISTENT, PERSISTENT)),
    (200, SINGLE, 0, (FEW, FEW)),
    (200, SINGLE, 1, (SMALL, FEW)),          # the few-row kernel does not save the pre-activations
    (256, SINGLE, 0, (FEW, FEW)),            # 64 rows per expert
    (300, SINGLE, 0, (SMALL, SMALL)),
    (8192, SINGLE, 0, (PERSISTENT, PERSISTENT)),
])
def test_bench_shapes(T, shape, training, want):
    assert _kernels(T, training=training, **shape) == want


@pytest.mark.parametrize("T,want", [(256, FEW), (4096, PERSISTENT), (8192, PERSISTENT)])
def test_few_rows_per_expert_beside_many_shared_rows(T, want):
    """Many small experts, one each: few routed rows per expert up to 8192 tokens, all of which the shared expert takes."""
    assert _kernels(T, D=1024, E=128, I=128, k=1, S=1, I_s=1024)[0] == want


def test_few_row_tiles_past_one_round():
    shape = dict(D=2048, E=8, I=1408, k=2, S=1, I_s=1408)
    assert _kernels(128, **shape) == (FEW, FEW)
    assert _kernels(200, **shape) == (SMALL, FEW)
    shape = dict(D=1024, E=32, I=256, k=2, S=0, I_s=0)
    assert _kernels(600, **shape) == (FEW, FEW)
    assert _kernels(1000, **shape) == (FEW, SMALL)


@pytest.mark.parametrize("shape,line", [
    (dict(D=2048, E=64, I=512, k=4, S=1, I_s=512), 40),       # shared down projection of the routed one's depth
    (dict(D=1024, E=128, I=512, k=8, S=1, I_s=512), 40),
    (dict(D=2048, E=64, I=1408, k=6, S=1, I_s=1408), 40),
    (dict(D=2048, E=64, I=1408, k=6, S=1, I_s=2816), 112),    # twice as deep
    (dict(D=1024, E=128, I=128, k=8, S=1, I_s=1024), 112),
])
def test_down_tiles_with_a_nearly_empty_last_round(shape, line):
    """The rows per expert up to which 128-row tiles are taken.  (The dense tiles' share of the last round stays under a
    quarter of the CUs here.)"""
    T = lambda rows: rows * shape["E"] // shape["k"]
    assert _kernels(T(line), **shape)[1] == SMALL
    assert _kernels(T(line + 1), **shape)[1] == PERSISTENT


def test_other_kernels_and_errors():
    import dsmoe._lib as L
    assert _kernels(100, 256, 8, 128, 2, 1, 128, dtype=L.DSMOE_F32) == (OTHER, OTHER)
    assert _kernels(100, 100, 8, 64, 2, 1, 64) == (OTHER, OTHER)          # K = 100
    with pytest.raises(ValueError, match="n_activated_experts"):
        _kernels(16, 64, 4, 32, 5, 0, 0)
