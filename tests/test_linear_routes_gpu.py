"""tgohip_linear where its routes meet: a K that is no whole number of four-k-step groups,
f32 activations split into a pair ahead of the projection (in one band of rows or
several), and the allocation-free linear over the same bands. Against the f64 product of
the activations and the oracle's dequantized weights, with the budgets of test_gemm_gpu:
AccumF32 (4 sqrt(K) 2^-24), plus 2^-22 for f32 activations and pairs."""
import numpy as np
import pytest

import tgo_amd
from test_gemm_gpu import deq, make_weight

pytestmark = pytest.mark.gpu


def operand(torch, x, xk):
    """(the stored activation, its dtype code)"""
    if xk == "f32":
        return x, tgo_amd.F32
    hi = x.half()
    if xk == "f16":
        return hi, tgo_amd.F16
    return torch.stack([hi, (x - hi.float()).half()]), tgo_amd.F16X2


def check(torch, ctx, form, K, N, M, xk, seed):
    wd, _ = make_weight(form, K, N, np.random.default_rng(seed))
    w = torch.from_numpy(deq(form, K, N, wd)).cuda()
    h = ctx.weight_upload(form, K, N, wd["plane"], wd.get("scales"), wd.get("zeros"))
    try:
        x, xd = operand(torch, torch.randn(M, K, device="cuda"), xk)
        y = torch.full((M, N), float("nan"), device="cuda")
        y16 = torch.full((M, N), float("nan"), device="cuda", dtype=torch.float16)
        n = torch.full((M, N), float("nan"), device="cuda")
        print("linear routes: form %d [%d,%d] M=%d %s" % (form, K, N, M, xk), flush=True)
        ctx.linear(h, x, M, y, x_dtype=xd)
        ctx.linear(h, x, M, y16, x_dtype=xd, y_dtype=tgo_amd.F16)
        if ctx.linear_workspace(h, M, x_dtype=xd) <= 64 << 20:
            ctx.linear_noalloc(h, x, M, n, x_dtype=xd)
            torch.cuda.synchronize()
            assert torch.equal(n, y)
        else:
            with pytest.raises(tgo_amd.TgoError, match="static workspace holds 67108864"):
                ctx.linear_noalloc(h, x, M, n, x_dtype=xd)
        torch.cuda.synchronize()
        assert torch.equal(y16, y.half())
        xu = x[0].double() + x[1].double() if xk == "x2" else x.double()
        wu = w.half().double() if xk == "f16" else w.double()
        rel = 4 * K ** 0.5 * 2.0 ** -24 + (0.0 if xk == "f16" else 2.0 ** -22)
        tol = rel * (xu.abs() @ wu.abs()) + 1e-30
        err = (y.double() - xu @ wu).abs()
        assert bool((err <= tol).all()), float((err / tol).max())
    finally:
        ctx.weight_free(h)


@pytest.mark.parametrize("xk", ["f32", "x2", "f16"])
@pytest.mark.parametrize("form", [0, 1, 2, 3])
@pytest.mark.parametrize("K,N,M", [(64, 256, 40), (320, 384, 65), (576, 2432, 400), (2240, 128, 130),
                                   (1216, 640, 33), (704, 896, 520)])
def test_linear_over_any_whole_k_step(ctx, torch_gpu, form, K, N, M, xk):
    """K = 64, 320, 576, 704, 1216, 2240: 1, 5, 9, 11, 19 and 35 k-steps of 64 (one, two and
    three left after the groups of four; split K at 2240 and 1216), at partial row and
    column tiles of the 64- and 128-row launches."""
    check(torch_gpu, ctx, form, K, N, M, xk, 5 + K + M)


@pytest.mark.parametrize("xk", ["f32", "x2", "f16"])
@pytest.mark.parametrize("form", [0, 1, 2, 3])
@pytest.mark.parametrize("K,N,M", [
    (64, 128, 1), (192, 256, 2), (1024, 384, 8), (576, 640, 9), (2048, 256, 16),   # staged rows, packed
    (256, 16512, 3), (320, 8320, 16),       # more column blocks than workgroups: they go round
    (8192, 256, 5), (12288, 128, 16), (25600, 128, 13),  # K in 2, 8 and 16 shares
    (512, 384, 17), (1600, 128, 31), (704, 256, 32),     # unpacked, one row block
    (1024, 128, 33), (576, 384, 65), (3072, 128, 127), (2048, 256, 129),  # two row blocks a workgroup
])
def test_linear_over_few_rows(ctx, torch_gpu, form, K, N, M, xk):
    """The row kernel at the edges of its launches: 1 to 16 rows staged in LDS (hi and lo
    packed into one MFMA operand), 17 up turned in LDS (up to 32 rows at one k-step a wave: from
    L2), k-steps that do not deal evenly over the waves, shares of K, column blocks past the last
    whole round."""
    check(torch_gpu, ctx, form, K, N, M, xk, 11 + K + M)


@pytest.mark.parametrize("xk", ["f32", "x2", "f16"])
@pytest.mark.parametrize("form", [0, 1, 2, 3])
@pytest.mark.parametrize("K,N,M", [
    (320, 4224, 65),    # two row tiles of 132 column blocks: f16 weights pair the blocks
    (1088, 8192, 128),  # 17 k-steps over 8 waves, the pair of blocks at its largest
    (576, 128, 32), (512, 128, 33),  # just past and at one k-step a wave, one and two row blocks
    (4096, 2048, 48),   # split K, whole lines of every wave
    (4096, 4224, 24),   # eight k-steps a wave through one row block's part of LDS
])
def test_linear_turns_its_rows_in_lds(ctx, torch_gpu, form, K, N, M, xk):
    check(torch_gpu, ctx, form, K, N, M, xk, 11 + K + M)


@pytest.mark.parametrize("form", [0, 1, 2, 3])
@pytest.mark.parametrize("K,N,M", [(4096, 4096, 4200), (4096, 4096, 257)])
def test_f32_activations_in_bands(ctx, torch_gpu, form, K, N, M):
    """4200 f32 rows of K = 4096: a pair of 69 MB, more than one 64 MiB band. 257 rows split
    K, and the allocation-free call's bands hold the planes too. The bands take the whole
    call's splits, so the two entry points agree to the bit."""
    check(torch_gpu, ctx, form, K, N, M, "f32", 7 + M)
