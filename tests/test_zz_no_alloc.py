"""rlxq_dequant_matmul_noalloc against rlxq_dequant_matmul through the C ABI:
the same kernels on the library's static scratch array, so the outputs are
bit-identical.  Two calls in a row, the second smaller (the array keeps the
first call's contents), on paths that use scratch: prefill split-K partial
sums, batched-decode prepared activations, Int8Block split-K; plus the
rejection of a call that needs more than RLXQ_NOALLOC_SCRATCH_BYTES."""
import numpy as np
import pytest

from conftest import announce

pytestmark = pytest.mark.gpu


def _q4_1(orc, rng, n, k):
    import torch

    return torch.from_numpy(orc.synth_q4_1(rng, n, k)).cuda()


def _x(rng, m, k):
    import torch

    return torch.from_numpy(rng.standard_normal((m, k)).astype(np.float32)).cuda().to(torch.bfloat16)


@pytest.mark.parametrize("first,second", [
    ((256, 12288, 4096, "bf16"), (16, 4096, 2048, "f32")),    # split-K GEMM, then batched decode
    ((64, 4096, 6144, "f32"), (8, 4096, 1024, "f32")),        # batched decode, larger then smaller
])
def test_noalloc_matches_dequant_matmul(ctx, orc, first, second):
    import torch
    import rlxq

    rng = np.random.default_rng(77)
    for (m, k, n, yd) in (first, second):
        announce(f"noalloc Q4_1 m={m} k={k} n={n} y={yd}")
        w = _q4_1(orc, rng, n, k)
        x = _x(rng, m, k)
        ydt = torch.bfloat16 if yd == "bf16" else torch.float32
        want = ctx.dequant_matmul(x, w, rlxq.GGUF_Q4_1, n, y_dtype=ydt)
        kern = ctx.last_kernel
        y = torch.full((m, n), float("nan"), dtype=ydt, device="cuda")
        ctx.dequant_matmul_noalloc(x, w, rlxq.GGUF_Q4_1, n, y=y)
        torch.cuda.synchronize()
        assert ctx.last_kernel == kern
        assert torch.equal(y, want), f"m={m} k={k} n={n}: no-allocation result differs"
        ref = orc.matmul_f64(orc.Q4_1, x.float().cpu().numpy(), w.cpu().numpy(), n)
        rel = float(np.max(np.abs(y.float().cpu().numpy() - ref)) / np.max(np.abs(ref)))
        assert rel <= (8e-3 if yd == "bf16" else 1e-3)


def test_noalloc_int8_block_twice(ctx, orc):
    import torch
    import rlxq

    rng = np.random.default_rng(78)
    for (m, k, n) in ((32, 4096, 2048), (3, 2048, 1024)):
        announce(f"noalloc Int8Block m={m} k={k} n={n}")
        wq = torch.from_numpy(rng.integers(-127, 128, (k, n), dtype=np.int8)).cuda()
        sc = torch.from_numpy(rng.uniform(0.001, 0.01, n).astype(np.float32)).cuda()
        x = torch.from_numpy(rng.standard_normal((m, k)).astype(np.float32)).cuda()
        want = ctx.dequant_matmul(x, wq, rlxq.INT8_BLOCK, n, group=k, scales=sc)
        y = torch.full((m, n), float("nan"), device="cuda")
        ctx.dequant_matmul_noalloc(x, wq, rlxq.INT8_BLOCK, n, group=k, scales=sc, y=y)
        torch.cuda.synchronize()
        assert torch.equal(y, want)


def test_noalloc_rejects_oversized_scratch(ctx, orc):
    import torch
    import rlxq

    rng = np.random.default_rng(79)
    m, k, n = 3072, 12288, 4096       # f32 output: the exact GEMM's f16 activations alone are 72 MiB
    w = _q4_1(orc, rng, n, k)
    x = _x(rng, m, k)
    y = torch.zeros((m, n), device="cuda")
    announce("noalloc oversized call is rejected before any launch")
    with pytest.raises(rlxq.RlxqError) as e:
        ctx.dequant_matmul_noalloc(x, w, rlxq.GGUF_Q4_1, n, y=y)
    assert e.value.status == rlxq.E_SCRATCH
    torch.cuda.synchronize()
    assert float(y.abs().max()) == 0.0


def _bytes_q4_1(gen, n, k):
    """Q4_1 rows of finite scales (every byte below 60)."""
    import torch

    return torch.randint(0, 60, (n, k // 32 * 20), device="cuda", dtype=torch.uint8, generator=gen)


@pytest.mark.parametrize("k,m", [(64, 254176), (128, 129024), (320, 52096)], ids=str)
def test_noalloc_f32_prefill_up_to_the_limit(ctx, orc, monkeypatch, k, m):
    """f32 rows at prefill count as the exact GEMM lays them out (a hi and a lo
    f16 row and a factor each): m rows are the most that fit, and one more is
    refused.  The block-scaled matmul, whose fragments take whole 256-element
    units, does them in passes: the same bits."""
    import torch
    import rlxq

    monkeypatch.setenv("RLXQ_BS", "1")
    n = 64
    need = lambda rows: (rows + 31) // 32 * 64 * (2 * k + 4)   # (both parts whole 256 bytes here)
    assert need(m) <= 64 << 20 < need(m + 1)
    announce(f"noalloc f32 prefill limit k={k} m={m}")
    gen = torch.Generator(device="cuda").manual_seed(k)
    w = _bytes_q4_1(gen, n, k).view(-1)
    x = torch.randn((m + 1, k), device="cuda", generator=gen)
    want = ctx.dequant_matmul(x[:m], w, rlxq.GGUF_Q4_1, n)
    kern = ctx.last_kernel
    y = torch.full((m + 1, n), float("nan"), device="cuda")
    ctx.dequant_matmul_noalloc(x[:m], w, rlxq.GGUF_Q4_1, n, y=y[:m])
    torch.cuda.synchronize()
    assert ctx.last_kernel == kern == "rlxq_bs_q4_1_rt2"
    assert torch.equal(y[:m], want) and bool(torch.isnan(y[m]).all())
    rows = np.array([0, 1, m // 2, m - 1])
    wd = orc.dequantize(orc.Q4_1, w.view(n, -1).cpu().numpy(), k).astype(np.float64)
    ref = x[torch.from_numpy(rows).cuda()].cpu().numpy().astype(np.float64) @ wd.T
    assert np.max(np.abs(y[torch.from_numpy(rows).cuda()].cpu().numpy() - ref)) <= 2e-5 * np.max(np.abs(ref))
    with pytest.raises(rlxq.RlxqError) as e:
        ctx.dequant_matmul_noalloc(x, w, rlxq.GGUF_Q4_1, n, y=y)
    assert e.value.status == rlxq.E_SCRATCH


def test_noalloc_f32_batched_near_the_limit(ctx, monkeypatch):
    """f32 rows of a batch count as the batched-decode kernels lay them out.
    Partial sums of more splits than theirs: passes over the rows, or where one
    tile of rows does not fit, those kernels."""
    import torch
    import rlxq

    gen = torch.Generator(device="cuda").manual_seed(5)
    for bs, m, k, n, same in (("2,32", 256, 57344, 256, True), ("1,32", 32, 458752, 4096, False)):
        monkeypatch.setenv("RLXQ_BS", bs)
        announce(f"noalloc f32 batched near the limit {(m, k, n)}")
        w = _bytes_q4_1(gen, n, k).view(-1)
        x = torch.randn((m, k), device="cuda", generator=gen)
        want = ctx.dequant_matmul(x, w, rlxq.GGUF_Q4_1, n)
        assert ctx.last_kernel == f"rlxq_bs_q4_1_rt{bs[0]}"
        y = torch.full((m, n), float("nan"), device="cuda")
        ctx.dequant_matmul_noalloc(x, w, rlxq.GGUF_Q4_1, n, y=y)
        torch.cuda.synchronize()
        if same:
            assert ctx.last_kernel == f"rlxq_bs_q4_1_rt{bs[0]}"
            assert torch.equal(y, want)
        else:
            assert ctx.last_kernel.startswith("rlxq_skinny"), ctx.last_kernel
            assert float((y - want).abs().max()) <= 2e-5 * float(want.abs().max())
        del w, x, y, want
        torch.cuda.empty_cache()
