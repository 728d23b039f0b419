"""K-contiguous GEMMs whose outputs need at most one 128-row tile per CU
(k_gemm_deep: four stages of 64 k in flight, split over K where that is
faster) against a plain F32 product.

Sizes: one row, tile edges (63..65, 127..129 rows and columns), ragged
outputs, 1, 2, 4 and 5 stages (fewer and more than the pipeline holds), long
K with ragged splits.  Bound: one rounding to BF16 (half an ulp, 2^-9
relative) of an F32 sum whose order differs from the reference's: an ulp
flips where the two sums straddle a rounding boundary, so at most one ulp, or
2^-20 sum |x y| where cancellation leaves less than that.
"""
import pytest
import torch

from gpu_util import DEV, P, S, call

pytestmark = pytest.mark.gpu


def rand(g, *shape, std=1.0):
    return (torch.randn(*shape, generator=g, device=DEV) * std).bfloat16()


@pytest.mark.parametrize("beta,bias", [(0.0, False), (1.0, False), (0.0, True)])
@pytest.mark.parametrize("M,N,K", [
    (1, 64, 64), (63, 65, 128), (64, 127, 256), (65, 129, 320), (127, 896, 896),
    (129, 200, 1984), (300, 1152, 896), (64, 896, 4864), (128, 72, 9728), (257, 136, 4864),
    (2331, 128, 1536), (512, 1536, 8960),
])
def test_small_gemm(M, N, K, beta, bias):
    g = torch.Generator(device=DEV)
    g.manual_seed(M * 7 + N * 3 + K)
    x, y = rand(g, M, K), rand(g, N, K, std=0.05)
    c0, b = rand(g, M, N), rand(g, N)
    c = c0.clone()
    call("ta_gemm_rm", 1, 1, M, N, K, 1.0, P(x), K, P(y), K, beta, P(c), N,
         P(b) if bias else None, S())
    want = x.float() @ y.float().t() + beta * c0.float()
    mag = x.float().abs() @ y.float().abs().t() + beta * c0.float().abs()
    if bias:
        want = want.bfloat16().float() + b.float()
    got = c.float()
    err = (got - want.bfloat16().float()).abs()
    ulp = 2.0 ** -7 * want.abs()
    if bias:  # the first rounding's ulp too
        ulp = ulp + 2.0 ** -7 * (want - b.float()).abs()
    assert bool((err <= ulp + 2.0 ** -20 * mag).all()), float((err / (ulp + 1e-9)).max())
    exact = float((got == want.bfloat16().float()).float().mean())
    assert exact >= 0.9, exact


@pytest.mark.parametrize("ykm", [0, 1])
@pytest.mark.parametrize("beta", [0.0, 1.0])
@pytest.mark.parametrize("M,N,K,ldx,ldy", [
    # K of a rank: k_gemm_rank (odd ranks and strides load element by element)
    (1, 64, 2, 2, 0), (65, 257, 4, 4, 0), (64, 264, 16, 16, 0), (200, 896, 8, 24, 0),
    (129, 100, 33, 33, 3), (2331, 1536, 64, 64, 0),
    # around its limits: up to 8 rows read back take the 32-wide tiles, a whole
    # 64-k stage of K-contiguous operands the pipelined kernels
    (8, 200, 48, 48, 0), (9, 200, 48, 48, 0), (8, 72, 16, 16, 0), (8, 18944, 64, 64, 0),
    (130, 136, 64, 68, 4), (64, 8960, 64, 64, 0),
    # K-strided Y: one tile, ragged tiles, more waves of tiles, K splits
    (1, 64, 64, 64, 0), (130, 72, 128, 128, 8), (127, 200, 320, 320, 0), (64, 896, 4864, 4864, 0),
    (300, 1536, 1536, 1536, 16), (2100, 4872, 192, 192, 0),
])
def test_rank_and_strided_gemm(M, N, K, ldx, ldy, beta, ykm):
    """K of a LoRA rank, and Y(k, n) in rows of n (y_kmajor 0): the delta
    h B^T, dx += s dh A and dy W of a caller that holds W as [out, in].
    ldy is the padding of Y's rows here.  Same bound as above."""
    g = torch.Generator(device=DEV)
    g.manual_seed(M * 5 + N + K)
    x = rand(g, M, ldx)
    y = rand(g, N, K + ldy, std=0.05) if ykm else rand(g, K, N + ldy, std=0.05)
    c0 = rand(g, M, N)
    c = c0.clone()
    call("ta_gemm_rm", 1, ykm, M, N, K, 2.0, P(x), ldx, P(y), y.shape[1], beta, P(c), N, None, S())
    xf = x[:, :K].float()
    yf = (y[:, :K].t() if ykm else y[:, :N]).float()
    want = 2.0 * (xf @ yf) + beta * c0.float()
    mag = 2.0 * (xf.abs() @ yf.abs()) + beta * c0.float().abs()
    err = (c.float() - want.bfloat16().float()).abs()
    assert bool((err <= 2.0 ** -7 * want.abs() + 2.0 ** -20 * mag).all())
    exact = float((c.float() == want.bfloat16().float()).float().mean())
    assert exact >= 0.9 or M * N < 100, exact


def test_small_gemm_in_a_graph():
    """A captured product, whose K split count may differ from the eager call's
    (here it runs unsplit), is right on every replay."""
    g = torch.Generator(device=DEV)
    g.manual_seed(5)
    M, N, K = 160, 896, 4864
    x, y = rand(g, M, K), rand(g, N, K, std=0.05)
    c, e = torch.empty(M, N, dtype=torch.bfloat16, device=DEV), None
    st = torch.cuda.Stream()
    with torch.cuda.stream(st):
        call("ta_gemm_rm", 1, 1, M, N, K, 1.0, P(x), K, P(y), K, 0.0, P(c), N, None, S())
    st.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph, stream=st):
        call("ta_gemm_rm", 1, 1, M, N, K, 1.0, P(x), K, P(y), K, 0.0, P(c), N, None, S())
    for _ in range(3):
        x.copy_(rand(g, M, K))
        torch.cuda.synchronize()
        graph.replay()
        torch.cuda.synchronize()
        want = x.float() @ y.float().t()
        e = (c.float() - want).norm() / want.norm()
        assert float(e) < 4e-3, float(e)
