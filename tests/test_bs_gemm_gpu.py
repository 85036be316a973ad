"""The block-scaled MFMA matmul (f32 activations, more than 16 rows) against
the float64 oracle: edges of its row, column and K tiles, K that is not whole
256-element units, K splits, and rows of very different size.

Bound per output: the activations' hi + lo split keeps each element to 2^-22,
and each of the K / 32 block results is rounded a few times in f32 on its way
into the sum, so |error| <= (2^-21 + (K / 32 + 8) 2^-23) sum_k |x_k| 3 W_k,
W_k the largest weight of k's block of 32 (scale * code and the min / bias
are each at most three times that in the synthetic rows)."""
import numpy as np
import pytest

from conftest import announce

pytestmark = pytest.mark.gpu


@pytest.fixture(autouse=True)
def _force_bs(monkeypatch):
    """The block-scaled kernel wherever it applies (its rule: test_rule)."""
    monkeypatch.setenv("RLXQ_BS", "1")


Q8_0, Q4_0, Q4_1, MLX4, MLX8, Q4_K, Q6_K, Q5_K = 1, 2, 3, 4, 5, 7, 8, 10
NAMES = {Q8_0: "q8_0", Q4_0: "q4_0", Q4_1: "q4_1", MLX4: "mlx4", MLX8: "mlx8", Q4_K: "q4_k", Q6_K: "q6_k", Q5_K: "q5_k"}


def _t(a):
    import torch

    return torch.from_numpy(np.ascontiguousarray(a)).cuda()


def _case(orc, scheme, rng, n, k, group=None, slab="f32"):
    """(packed, scales, biases, group, dequantized float64 weights)"""
    if scheme in (MLX4, MLX8):
        import torch

        bits, group = (4, group or 64) if scheme == MLX4 else (8, group or 32)
        codes = rng.integers(0, 1 << bits, (n, k)).astype(np.uint32)
        wq = orc.mlx_pack(codes, bits)
        sc = rng.uniform(0.01, 0.1, (n, k // group)).astype(np.float32)
        bi = rng.uniform(-0.5, 0.1, (n, k // group)).astype(np.float32)
        if slab == "bf16":
            ts, tb = _t(sc).to(torch.bfloat16), _t(bi).to(torch.bfloat16)
            sc, bi = ts.float().cpu().numpy(), tb.float().cpu().numpy()
        else:
            ts, tb = _t(sc), _t(bi)
        wd = codes * np.repeat(sc.astype(np.float64), group, 1) + np.repeat(bi.astype(np.float64), group, 1)
        return _t(wq.view(np.uint8)), ts, tb, group, wd
    packed = orc.synth(scheme, rng, n, k)
    return _t(packed), None, None, 32, orc.dequantize(scheme, packed, k).astype(np.float64).reshape(n, k)


def _check(ctx, orc, scheme, m, k, n, y_dtype=None, bs_only=True, group=None, slab="f32"):
    import torch

    rng = np.random.default_rng(m * 7 + k + n * 3 + scheme)
    w, sc, bi, group, wd = _case(orc, scheme, rng, n, k, group, slab)
    x = rng.standard_normal((m, k)).astype(np.float32)
    x[0] *= 1e-6
    x[m // 2] *= 3e4
    x[m - 1, ::3] = 0.0
    y = ctx.dequant_matmul(_t(x), w, scheme, n, group=group, scales=sc, biases=bi, y_dtype=y_dtype)
    kern = ctx.last_kernel
    torch.cuda.synchronize()
    want = x.astype(np.float64) @ wd.T
    wmax = np.repeat(np.abs(wd).reshape(n, k // 32, 32).max(2), 32, 1)
    lim = (2.0 ** -21 + (k / 32 + 8) * 2.0 ** -23) * (np.abs(x).astype(np.float64) @ (3 * wmax).T)
    got = y.double().cpu().numpy()
    if y_dtype is not None:
        lim = lim + np.abs(want) * 2.0 ** -8   # one rounding to bf16
    if not bs_only:   # (the other kernels hold weights as f16 hi + lo: to 2^-22, or 2^-25 of 1)
        lim = lim * 4 + 2.0 ** -24 * np.abs(x).astype(np.float64).sum(1, keepdims=True)
    assert np.all(np.abs(got - want) <= lim), (kern, float(np.max(np.abs(got - want) / lim)))
    return kern


@pytest.mark.parametrize("scheme", list(NAMES), ids=lambda s: NAMES[s])
@pytest.mark.parametrize("mkn", [(17, 256, 1), (32, 512, 127), (33, 1792, 129), (64, 1024, 128), (65, 768, 300),
                                 (200, 2304, 130), (256, 4096, 64)], ids=str)
def test_batched(ctx, orc, scheme, mkn):
    announce(f"block-scaled {NAMES[scheme]} {mkn}")
    kern = _check(ctx, orc, scheme, *mkn)
    assert kern == f"rlxq_bs_{NAMES[scheme]}_rt{2 if mkn[0] > 32 else 1}", kern


@pytest.mark.parametrize("scheme,mkn", [(Q4_1, (300, 64 * 13, 301)), (Q4_0, (257, 64 * 5, 130)), (Q8_0, (259, 64 * 7, 33)),
                                        (MLX4, (258, 64 * 9, 65)), (Q4_1, (18, 384, 5)), (MLX8, (20, 128, 40)),
                                        (Q4_K, (513, 2560, 385)), (Q5_K, (321, 256, 256)),
                                        (Q6_K, (300, 1280, 131)), (Q6_K, (65, 256, 3))], ids=str)
@pytest.mark.parametrize("ydt", ["f32", "bf16"])
def test_partial_units_and_prefill(ctx, orc, scheme, mkn, ydt):
    import torch

    announce(f"block-scaled {NAMES[scheme]} {mkn} y={ydt}")
    if ydt == "bf16" and mkn[0] < 64:
        pytest.skip("bf16 output takes this kernel from 64 rows")
    kern = _check(ctx, orc, scheme, *mkn, y_dtype=torch.bfloat16 if ydt == "bf16" else None)
    assert kern == f"rlxq_bs_{NAMES[scheme]}_rt{2 if mkn[0] > 32 else 1}", kern


@pytest.mark.parametrize("cfg", ["1,1", "1,3", "2,1", "2,5", "2,32"])
def test_row_tiles_and_splits(ctx, orc, monkeypatch, cfg):
    monkeypatch.setenv("RLXQ_BS", cfg)
    for scheme, mkn in ((Q4_1, (70, 1792, 200)), (Q4_K, (40, 2816, 129)), (Q6_K, (70, 1792, 133))):
        announce(f"block-scaled {cfg} {NAMES[scheme]} {mkn}")
        kern = _check(ctx, orc, scheme, *mkn)
        assert kern == f"rlxq_bs_{NAMES[scheme]}_rt{cfg[0]}", kern


@pytest.mark.parametrize("scheme", [MLX4, MLX8], ids=lambda s: NAMES[s])
@pytest.mark.parametrize("group", [32, 64, 128])
@pytest.mark.parametrize("slab", ["f32", "bf16"])
def test_mlx_groups_and_slabs(ctx, orc, scheme, group, slab):
    for mkn in ((17, 640, 17), (70, 1152, 131), (300, 4608, 129)):
        announce(f"block-scaled {NAMES[scheme]} group={group} slab={slab} {mkn}")
        kern = _check(ctx, orc, scheme, *mkn, group=group, slab=slab)
        assert kern.startswith(f"rlxq_bs_{NAMES[scheme]}_rt"), kern


def test_noalloc_is_the_same(ctx, orc):
    """The no-allocation entry point runs the same kernel on its own array."""
    import torch

    rng = np.random.default_rng(4)
    for (m, k, n) in ((64, 4096, 2048), (300, 2048, 1024)):
        announce(f"block-scaled noalloc {(m, k, n)}")
        w = _t(orc.synth_q4_1(rng, n, k))
        x = _t(rng.standard_normal((m, k)).astype(np.float32))
        want = ctx.dequant_matmul(x, w, Q4_1, n)
        y = torch.full((m, n), float("nan"), device="cuda")
        ctx.dequant_matmul_noalloc(x, w, Q4_1, n, y=y)
        torch.cuda.synchronize()
        assert torch.equal(y, want)


@pytest.mark.parametrize("scheme", list(NAMES), ids=lambda s: NAMES[s])
def test_wide_rows_form(ctx, orc, monkeypatch, scheme):
    """The form with 64-bit row offsets, on rows that do not need it."""
    monkeypatch.setenv("RLXQ_BS", "0,0")
    for mkn in ((17, 512, 33), (70, 1792, 200), (300, 1280, 129)):
        announce(f"block-scaled 64-bit row offsets {NAMES[scheme]} {mkn}")
        kern = _check(ctx, orc, scheme, *mkn)
        assert kern == f"rlxq_bs_{NAMES[scheme]}_wide", kern


@pytest.mark.parametrize("scheme", [Q8_0, Q6_K], ids=lambda s: NAMES[s])
def test_rows_past_4_gb(orc, scheme):
    """32 weight rows past 4 GB.  x is zero but for three stretches of K, so
    that the bound above holds with those alone."""
    import rlxq
    import torch

    m, n, k = 17, 32, 21 << 23 if scheme == Q6_K else 1 << 27
    rb = orc.row_bytes(scheme, k)
    assert 31 * rb >= 1 << 32
    announce(f"block-scaled rows of {rb} bytes {NAMES[scheme]} k={k}")
    seg = [(0, 2048), (k // 2 - 1024, k // 2 + 1024), (k - 2048, k)]
    gen = torch.Generator(device="cuda").manual_seed(scheme)
    # (bytes below 60: every f16 and int8 scale finite)
    w = torch.randint(0, 60, (n, rb), device="cuda", dtype=torch.uint8, generator=gen)
    x = torch.zeros((m, k), device="cuda")
    for a, b in seg:
        x[:, a:b] = torch.randn((m, b - a), device="cuda", generator=gen)
    c = rlxq.Context(0)
    try:
        y = c.dequant_matmul(x, w.view(-1), scheme, n)
        kern = c.last_kernel
        torch.cuda.synchronize()
    finally:
        c.close()
    xs = torch.cat([x[:, a:b] for a, b in seg], 1).cpu().numpy().astype(np.float64)
    wd = np.concatenate([orc.dequantize(scheme, w[:, orc.row_bytes(scheme, a) if a else 0:orc.row_bytes(scheme, b)]
                                        .cpu().numpy(), b - a).astype(np.float64) for a, b in seg], 1)
    want = xs @ wd.T
    ks = wd.shape[1]
    wmax = np.repeat(np.abs(wd).reshape(n, ks // 32, 32).max(2), 32, 1)
    lim = (2.0 ** -21 + (ks / 32 + 8) * 2.0 ** -23) * (np.abs(xs) @ (3 * wmax).T)
    got = y.double().cpu().numpy()
    assert np.all(np.abs(got - want) <= lim), (kern, float(np.max(np.abs(got - want) / lim)))
    assert kern == f"rlxq_bs_{NAMES[scheme]}_wide", kern


@pytest.mark.parametrize("case", [
    # 17 to 256 rows: (scheme, m, k, n, bf16 output, block-scaled?)
    (Q4_1, 64, 4096, 4096, False, True), (Q4_1, 17, 256, 64, False, True), (Q4_1, 32, 384, 4096, False, False),
    (Q4_1, 32, 384, 128 * 129, False, True), (Q4_1, 64, 512, 128 * 64, False, False), (Q4_K, 64, 512, 128 * 65, False, True),
    (MLX4, 64, 384, 128 * 128, False, False), (MLX4, 64, 384, 128 * 129, False, True), (Q6_K, 33, 768, 128 * 32, False, True),
    (Q6_K, 33, 768, 128 * 33, False, False), (Q4_1, 64, 1024, 64, False, True), (Q4_1, 64, 8192, 512, False, False),
    (Q4_1, 64, 8192, 513, False, True), (Q8_0, 64, 8192, 128, False, False), (Q8_0, 64, 8192, 256, False, True),
    (Q4_0, 33, 640, 4096, False, False), (Q4_0, 33, 640, 4224, False, True), (Q8_0, 40, 256, 128, False, True),
    (MLX8, 160, 1792, 12288, False, False), (MLX8, 64, 640, 512, False, False), (MLX8, 192, 4096, 4096, False, True),
    # prefill
    (Q4_1, 300, 64, 4096, False, True), (Q4_1, 1024, 64, 4096, False, False), (Q4_1, 128, 128, 512, True, False),
    (Q4_1, 130, 128, 512, True, True), (Q4_0, 512, 256, 300, False, True), (Q8_0, 300, 64, 512, False, False),
    (Q8_0, 1024, 192, 4096, False, False), (Q8_0, 1024, 576, 4096, False, True), (MLX8, 1024, 1024, 4096, False, False),
    (MLX8, 512, 1024, 4096, False, True), (MLX8, 300, 4096, 2048, False, False), (MLX8, 257, 4096, 768, False, True), (MLX4, 1100, 8256, 256, False, False),
    (MLX4, 1100, 8256, 257, False, True), (Q5_K, 300, 256, 64, False, True)], ids=str)
def test_rule(ctx, orc, monkeypatch, case):
    """Both sides of the lines between this kernel and the batched-decode
    kernels and the exact GEMM, each against the oracle."""
    import torch

    monkeypatch.delenv("RLXQ_BS")
    scheme, m, k, n, ybf, want = case
    announce(f"block-scaled rule {NAMES[scheme]} {case[1:]}")
    kern = _check(ctx, orc, scheme, m, k, n, y_dtype=torch.bfloat16 if ybf else None, bs_only=False)
    assert kern.startswith(f"rlxq_bs_{NAMES[scheme]}_rt") == want, kern
    if not want:
        assert kern.startswith("rlxq_gemm_" if ybf or m > 256 else "rlxq_skinny"), kern
