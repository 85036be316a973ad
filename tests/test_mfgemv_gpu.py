"""One to four activation rows on the matrix cores (rlxq_gemv*_mf*) against
the float64 oracle: the smallest K (a unit per wave) and one whose units do not
divide over the waves, weight rows that end inside a tile, the rows of a tile
per launch, and rows of very different size.

Bound per output, f32 rows: the hi + lo f16 split keeps each element to 2^-22
of itself or 2^-39 of B_k, the largest |x| of k's block of 32, and each of the
K / 32 block results is rounded a few times in f32 on its way into the sum, so
|error| <= (2^-21 + (K / 32 + 8) 2^-23) sum_k (|x_k| + 2^-18 B_k) 3 W_k, W_k
the largest weight of the block (scale * code and the min / bias are each at
most three times that in the synthetic rows).  bf16 rows are exact in f16 above
2^-31 of B_k, and 2^-39 of it off below; their sums round alike."""
import numpy as np
import pytest

from conftest import announce
from test_bs_gemm_gpu import MLX4, NAMES, Q4_1, Q4_K, Q6_K, Q8_0, _case, _t

pytestmark = pytest.mark.gpu

SCHEMES = [Q8_0, Q4_1, MLX4, Q4_K, Q6_K]


def _check(ctx, orc, scheme, m, k, n, bf16, y_dtype=None, change=None, group=None, slab="f32"):
    import torch

    rng = np.random.default_rng(m * 11 + k + n * 5 + scheme)
    w, sc, bi, group, wd = _case(orc, scheme, rng, n, k, group, slab)
    x = rng.standard_normal((m, k)).astype(np.float32)
    x[0] *= 1e-6
    x[m // 2] *= 3e4
    x[m - 1, ::3] = 0.0
    if change:
        change(x, w, sc, bi, wd)
    xt = _t(x).to(torch.bfloat16) if bf16 else _t(x)
    x = xt.float().cpu().numpy().astype(np.float64)
    y = ctx.dequant_matmul(xt, w, scheme, n, group=group, scales=sc, biases=bi, y_dtype=y_dtype or torch.float32)
    kern = ctx.last_kernel
    torch.cuda.synchronize()
    want = x @ wd.T
    wmax = np.repeat(np.abs(wd).reshape(n, k // 32, 32).max(2), 32, 1)
    xa = np.abs(x) + 2.0 ** -18 * np.repeat(np.abs(x).reshape(m, k // 32, 32).max(2), 32, 1)
    lim = (2.0 ** -21 + (k / 32 + 8) * 2.0 ** -23) * (xa @ (3 * wmax).T)
    if y_dtype is not None:
        lim = lim + np.abs(want) * 2.0 ** -8   # one rounding to bf16
    got = y.double().cpu().numpy()
    assert np.all(np.abs(got - want) <= lim), (kern, float(np.max(np.abs(got - want) / lim)))
    return kern


@pytest.mark.parametrize("scheme", SCHEMES, ids=lambda s: NAMES[s])
@pytest.mark.parametrize("bf16", [False, True], ids=["f32", "bf16"])
def test_edges(ctx, orc, monkeypatch, scheme, bf16):
    monkeypatch.setenv("RLXQ_GEMV_MF", "1")
    for m in (1, 2, 3, 4):
        for k, n in ((2048, 16), (2048, 17), (4608, 61), (4096, 4130)):
            announce(f"matrix-core decode {NAMES[scheme]} m={m} k={k} n={n} bf16={bf16}")
            assert "_mf" in _check(ctx, orc, scheme, m, k, n, bf16)
    import torch

    _check(ctx, orc, scheme, 3, 2560 if scheme != Q6_K else 3072, 33, bf16, y_dtype=torch.bfloat16)


@pytest.mark.parametrize("scheme", SCHEMES, ids=lambda s: NAMES[s])
def test_rows_in_pairs_and_defaults(ctx, orc, scheme):
    """Four f32 rows whose fragments pass the LDS go two to a launch; what the
    kernel does not take (K not whole units, fewer than eight of them, fewer
    than 16 weight rows, MLX groups that are no power of two) stays where it
    was."""
    announce(f"matrix-core decode in pairs {NAMES[scheme]}")
    for m in (3, 4):
        kern = _check(ctx, orc, scheme, m, 12288, 40, False)
        assert "_mf2_F" in kern, kern
    for m, k, n in ((2, 1536, 64), (2, 4096, 15)) + (((2, 2176, 64),) if scheme in (Q8_0, Q4_1, MLX4) else ()):
        assert "_mf" not in _check(ctx, orc, scheme, m, k, n, True), (m, k, n)


@pytest.mark.parametrize("scheme", SCHEMES, ids=lambda s: NAMES[s])
@pytest.mark.parametrize("bf16", [False, True], ids=["f32", "bf16"])
def test_large_elements_on_zero_weights(ctx, orc, monkeypatch, scheme, bf16):
    """Elements 2^30 times the others, where every weight is zero, take
    nothing from the rest: not from the blocks of their own 256 (but for their
    own block of 32, whose weights are zero in the formats that have a scale
    for it alone) nor from the same wave's next 256."""
    monkeypatch.setenv("RLXQ_GEMV_MF", "1")
    k, n = 6144, 48
    unit = scheme in (Q4_K, Q6_K)   # (a scale, and so zeros, for 256 weights)

    def change(x, w, sc, bi, wd):
        for u in range(0, k // 256, 3):   # every wave has three units
            a, b = 256 * u + 64, 256 * u + (256 if unit else 128)
            a -= 64 if unit else 0
            x[:, a:b] *= 2.0 ** 30
            wd[:, a:b] = 0.0
            if sc is not None:
                sc[:, a // 64:b // 64] = 0.0
                bi[:, a // 64:b // 64] = 0.0
            else:
                rows = w.view(n, -1)
                rows[:, orc.row_bytes(scheme, a) if a else 0:orc.row_bytes(scheme, b)] = 0

    for m in (1, 2, 4):
        announce(f"matrix-core decode, large elements on zero weights {NAMES[scheme]} m={m} bf16={bf16}")
        kern = _check(ctx, orc, scheme, m, k, n, bf16, change=change)
        assert "_mf" in kern, kern


@pytest.mark.parametrize("group", [32, 64, 128])
@pytest.mark.parametrize("slab", ["f32", "bf16"])
@pytest.mark.parametrize("bf16", [False, True], ids=["f32", "bf16"])
def test_mlx_groups_and_slabs(ctx, orc, monkeypatch, group, slab, bf16):
    """A lane's two blocks under one scale and bias or two, from either slab."""
    monkeypatch.setenv("RLXQ_GEMV_MF", "1")
    for m, k, n in ((1, 2048, 17), (2, 4608, 61), (4, 4608, 17)):
        announce(f"matrix-core decode mlx4 group={group} slab={slab} m={m} k={k} n={n} bf16={bf16}")
        kern = _check(ctx, orc, MLX4, m, k, n, bf16, group=group, slab=slab)
        assert "_mf" in kern, kern


def test_mlx_short_rows_stay_on_the_register_kernel(ctx, orc):
    """Three and four bf16 rows of MLX 4-bit at K = 2048: the register kernel,
    past it (and with many weight rows) this one."""
    for m, k, n, want in ((3, 2048, 64, False), (4, 2048, 2048, False), (4, 2304, 64, True), (3, 2048, 8192, True)):
        announce(f"matrix-core decode rule mlx4 m={m} k={k} n={n}")
        kern = _check(ctx, orc, MLX4, m, k, n, True)
        assert ("_mf" in kern) == want, (m, k, n, kern)


def test_a_row_that_is_not_finite_stays_alone(ctx, orc):
    """An infinity or NaN in one row leaves the others' bits as they were."""
    import torch

    announce("matrix-core decode with rows that are not finite")
    rng = np.random.default_rng(5)
    w, *_ = _case(orc, Q8_0, rng, 64, 2048)
    x = rng.standard_normal((4, 2048)).astype(np.float32)
    y0 = ctx.dequant_matmul(_t(x), w, Q8_0, 64)
    x[1, 7], x[2, 9] = np.inf, np.nan
    y1 = ctx.dequant_matmul(_t(x), w, Q8_0, 64)
    torch.cuda.synchronize()
    assert "_mf" in ctx.last_kernel
    assert torch.equal(y0[0], y1[0]) and torch.equal(y0[3], y1[3])
    assert not torch.isfinite(y1[1]).any() and torch.isnan(y1[2]).all()
