"""ta_gemm_f32 at the edges of its tiles (32, 64 and 128 on either side), of
its 64-k stages and of its K splits, in both layouts of both operands, with
strides that allow 16-byte loads and strides that do not, against F64.

Bound: the three BF16 parts of an operand keep 24 bits of it and the six part
products leave out what is below 2^-24 of a product; the F32 sums of K terms
add at most K 2^-24 of sum |a b|, in practice its square root: 1e-6
sum |a b| + one F32 rounding of beta C holds for every K used here.
"""
import pytest
import torch

from gpu_util import DEV, P, S, call

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("pad", [0, 1])
@pytest.mark.parametrize("tA,tB", [(0, 0), (0, 1), (1, 0), (1, 1)])
@pytest.mark.parametrize("M,N,K", [(1, 1, 1), (32, 33, 64), (64, 65, 63), (16, 200, 1000),
                                   (200, 16, 1000), (129, 127, 65), (64, 300, 4097)])
def test_gemm_f32_edges(M, N, K, tA, tB, pad):
    g = torch.Generator(device=DEV)
    g.manual_seed(M + 10 * N + 100 * K + tA + 2 * tB)
    # column-major op(A) [M x K], op(B) [K x N]: rows of the stored arrays
    A = torch.randn(*((M, K + pad) if tA else (K, M + pad)), generator=g, device=DEV)
    B = torch.randn(*((K, N + pad) if tB else (N, K + pad)), generator=g, device=DEV)
    C = torch.randn(N, M + pad, generator=g, device=DEV)
    c0 = C.clone()
    call("ta_gemm_f32", tA, tB, M, N, K, 0.75, P(A), A.shape[1], P(B), B.shape[1], 0.5, P(C),
         M + pad, S())
    a = (A[:, :K] if tA else A[:, :M].t()).double()
    b = (B[:, :N].t() if tB else B[:, :K]).double()
    want = 0.75 * (b @ a.t()) + 0.5 * c0[:, :M].double()
    mag = 0.75 * (b.abs() @ a.abs().t()) + 0.5 * c0[:, :M].double().abs()
    assert bool(((C[:, :M].double() - want).abs() <= 1e-6 * mag).all())
    assert torch.equal(C[:, M:], c0[:, M:])  # nothing past a row's end is written
