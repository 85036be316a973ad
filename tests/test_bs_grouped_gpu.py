"""The grouped (expert) form of the block-scaled MFMA matmul, f32 activations
and at least eight entries per fired expert, against the float64 oracle: every
format of it, plain and (where compiled) with SwiGLU, K that is not whole
256-element units, widths at the edges of its 128-column tiles, experts with
exactly a chunk of 32 entries, one more and none, experts of many chunks, and
invalid ids.

Bound per output of the plain form: that of the dense one, lim = (2^-21 +
(K / 32 + 8) 2^-23) sum_k |x_k| 3 W_k.  SwiGLU, silu(g) u: g and u each off by
their lim, silu's slope at most 1.1, and 2^-20 of the result for its expf,
division and products."""
import numpy as np
import pytest

from conftest import announce
from test_bs_gemm_gpu import MLX4, MLX8, NAMES, Q4_0, Q4_1, Q4_K, Q5_K, Q6_K, Q8_0, _case, _t

pytestmark = pytest.mark.gpu

E = 6


@pytest.fixture(autouse=True)
def _force_bs(monkeypatch):
    """The block-scaled kernel wherever it applies (its rule: test_rule)."""
    monkeypatch.setenv("RLXQ_BS", "1")


def _entries(rng, counts):
    """Experts of the entries in random order; two of them invalid."""
    ids = np.concatenate([np.full(c, e) for e, c in enumerate(counts)])
    ids = np.concatenate([ids, [-1, E]])
    return rng.permutation(ids)


def _want(x, wd, ids, n):
    """Sums in float64 and their bound, [entries, n]; zeros where invalid."""
    k = x.shape[1]
    wmax = np.repeat(np.abs(wd).reshape(-1, k // 32, 32).max(2), 32, 1)
    y, lim = np.zeros((len(ids), n)), np.zeros((len(ids), n))
    for e in range(E):
        r = ids == e
        y[r] = x[r] @ wd[e * n:(e + 1) * n].T
        lim[r] = (2.0 ** -21 + (k / 32 + 8) * 2.0 ** -23) * (np.abs(x[r]) @ (3 * wmax[e * n:(e + 1) * n]).T)
    return y, lim


def _plain(ctx, orc, scheme, counts, k, n, group=64, slab="f32", y_dtype=None):
    import torch

    rng = np.random.default_rng(scheme * 31 + k + n + group)
    w, sc, bi, group, wd = _case(orc, scheme, rng, E * n, k, group, slab)
    ids = _entries(rng, counts)
    x = rng.standard_normal((len(ids), k)).astype(np.float32)
    x[0] *= 1e-6
    x[1] *= 3e4
    idx = ids.astype(np.float32)
    idx[ids == E] = 0.5   # (not whole: invalid too)
    y = ctx.grouped_matmul(_t(x), w.view(-1), _t(idx), scheme, n, E, group=group, scales=sc, biases=bi, y_dtype=y_dtype)
    kern = ctx.last_kernel
    torch.cuda.synchronize()
    want, lim = _want(x.astype(np.float64), wd, ids, n)
    if y_dtype is not None:
        lim = lim + np.abs(want) * 2.0 ** -8   # one rounding to bf16
    got = y.double().cpu().numpy()
    assert np.all(np.abs(got - want) <= lim), (kern, float(np.max(np.abs(got - want) / np.maximum(lim, 1e-300))))
    assert kern == f"rlxq_moesk_{NAMES[scheme]}_bs", kern


@pytest.mark.parametrize("scheme", list(NAMES), ids=lambda s: NAMES[s])
def test_plain(ctx, orc, scheme):
    import torch

    kq = scheme in (Q4_K, Q5_K, Q6_K)
    for k, n in ((256, 1), (512 if kq else 384, 127), (768 if kq else 640, 129)):
        announce(f"block-scaled grouped {NAMES[scheme]} k={k} n={n}")
        _plain(ctx, orc, scheme, (32, 33, 0, 1, 100, 9), k, n)
    announce(f"block-scaled grouped {NAMES[scheme]} bf16 output")
    _plain(ctx, orc, scheme, (31, 64, 0, 0, 65, 2), 512, 40, y_dtype=torch.bfloat16)


@pytest.mark.parametrize("scheme", [MLX4, MLX8], ids=lambda s: NAMES[s])
@pytest.mark.parametrize("group", [32, 64, 128])
@pytest.mark.parametrize("slab", ["f32", "bf16"])
def test_mlx_groups_and_slabs(ctx, orc, scheme, group, slab):
    announce(f"block-scaled grouped {NAMES[scheme]} group={group} slab={slab}")
    _plain(ctx, orc, scheme, (32, 33, 0, 1, 100, 9), 640, 130, group, slab)


@pytest.mark.parametrize("counts", [(8, 400, 0, 33, 0, 64), (0, 0, 3000, 0, 0, 0), (300, 0, 257, 288, 0, 1)], ids=str)
def test_experts_of_many_chunks(ctx, orc, counts):
    announce(f"block-scaled grouped, entries per expert {counts}")
    _plain(ctx, orc, Q4_1, counts, 128, 33)


@pytest.mark.parametrize("scheme", [Q4_1, Q4_0, Q8_0, Q4_K, Q5_K], ids=lambda s: NAMES[s])
def test_swiglu(ctx, orc, scheme):
    import rlxq
    import torch

    kq = scheme in (Q4_K, Q5_K)
    for k, i, div in ((256, 1, 1), (512 if kq else 384, 127, 2), (768 if kq else 640, 129, 2)):
        announce(f"block-scaled grouped SwiGLU {NAMES[scheme]} k={k} width={i}")
        rng = np.random.default_rng(scheme * 17 + k + i)
        w, _, _, _, wd = _case(orc, scheme, rng, E * 2 * i, k)
        ids = _entries(rng, (32, 33, 0, 1, 100, 10 - div))
        ids = ids[:len(ids) // div * div]
        x = (rng.standard_normal((len(ids) // div, k)) * 0.2).astype(np.float32)
        y = ctx.moe_grouped(_t(x), w.view(-1), _t(ids.astype(np.int32).reshape(-1, div)), None, scheme,
                            rlxq.MOE_EXPAND_SWIGLU, 2 * i, E)
        kern = ctx.last_kernel
        torch.cuda.synchronize()
        gu, lim = _want(np.repeat(x.astype(np.float64), div, 0), wd, ids, 2 * i)
        g, u, lg, lu = gu[:, :i], gu[:, i:], lim[:, :i], lim[:, i:]
        s = g / (1.0 + np.exp(-g))
        lim = 1.1 * lg * (np.abs(u) + lu) + np.abs(s) * lu + 2.0 ** -20 * np.abs(s * u)
        got = y.double().cpu().numpy()
        assert np.all(np.abs(got - s * u) <= lim), (kern, float(np.max(np.abs(got - s * u) / np.maximum(lim, 1e-300))))
        assert kern == f"rlxq_moesk_{NAMES[scheme]}_bs_sw", kern


@pytest.mark.parametrize("case", [
    # (scheme, experts, entries of each, k, width, SwiGLU, block-scaled?)
    (Q4_1, 2, 8, 1024, 4096, False, True), (Q4_1, 2, 8, 1280, 4096, False, False), (Q4_1, 2, 16, 1280, 4224, False, True),
    (Q4_1, 2, 8, 1280, 8320, False, True), (Q4_K, 2, 8, 512, 256, True, True), (Q8_0, 2, 8, 512, 256, True, False),
    (Q4_K, 2, 16, 768, 3072, True, False), (Q4_K, 2, 16, 768, 3200, True, True), (Q4_K, 2, 8, 768, 7168, True, False),
    (Q4_K, 2, 8, 768, 7296, True, True)], ids=str)
def test_rule(ctx, orc, monkeypatch, case):
    """Both sides of the lines between this kernel and the row-pair ones."""
    import rlxq
    import torch

    monkeypatch.delenv("RLXQ_BS")
    scheme, experts, each, k, width, sw, want = case
    announce(f"block-scaled grouped rule {case}")
    rng = np.random.default_rng(k + width)
    n = 2 * width if sw else width
    w, _, _, _, wd = _case(orc, scheme, rng, experts * n, k)
    ids = rng.permutation(np.repeat(np.arange(experts), each))
    x = (rng.standard_normal((len(ids), k)) * 0.1).astype(np.float32)
    if sw:
        y = ctx.moe_grouped(_t(x), w.view(-1), _t(ids.astype(np.int32).reshape(-1, 1)), None, scheme,
                            rlxq.MOE_EXPAND_SWIGLU, n, experts)
    else:
        y = ctx.grouped_matmul(_t(x), w.view(-1), _t(ids.astype(np.float32)), scheme, n, experts)
    kern = ctx.last_kernel
    torch.cuda.synchronize()
    assert kern.startswith(f"rlxq_moesk_{NAMES[scheme]}_") and ("_bs" in kern) == want, kern
    gu = np.stack([x[i].astype(np.float64) @ wd[e * n:(e + 1) * n].T for i, e in enumerate(ids)])
    ref = gu[:, :width] / (1.0 + np.exp(-gu[:, :width])) * gu[:, width:] if sw else gu
    assert np.max(np.abs(y.double().cpu().numpy() - ref)) <= 2e-5 * np.max(np.abs(ref)), kern
