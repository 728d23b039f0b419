"""The attention with stored probabilities at the edges of its 64-row tiles,
with rows that start on and off a 16-byte boundary (T a multiple of 4 or
not), and with an infinite value at a key, which must not reach the query
tiles before it.  P against F64 to F32 accuracy; O, dQ, dK and dV to one BF16
rounding of sums whose P or dS factors keep 16 bits (relative L2 4e-3)."""
import math

import pytest
import torch

from gpu_util import DEV, P, S, call

pytestmark = pytest.mark.gpu


def run(B, T, Hq, Hk, hd, q, k, v, do):
    o, dq = torch.empty_like(q), torch.empty_like(q)
    dk, dv = torch.empty_like(k), torch.empty_like(k)
    p = torch.full((B * Hq, T, T), 7.0, device=DEV)
    call("ta_sdpa_fwd", P(q), P(k), P(v), P(o), P(p), B, T, Hq, Hk, hd, S())
    call("ta_sdpa_bwd", P(do), P(q), P(k), P(v), P(p), P(dq), P(dk), P(dv), B, T, Hq, Hk, hd, S())
    torch.cuda.synchronize()
    return o, p, dq, dk, dv


def inputs(B, T, Hq, Hk, hd):
    g = torch.Generator(device=DEV)
    g.manual_seed(T * 3 + hd)
    mk = lambda h: torch.randn(B * T, h * hd, generator=g, device=DEV).bfloat16()
    return mk(Hq), mk(Hk), mk(Hk), mk(Hq)


@pytest.mark.parametrize("hd", [64, 128])
@pytest.mark.parametrize("T", [1, 3, 63, 64, 65, 128, 190, 257])
def test_saved_probabilities(T, hd):
    B, Hq, Hk = 2, 4, 2
    q, k, v, do = inputs(B, T, Hq, Hk, hd)
    o, p, dq, dk, dv = run(B, T, Hq, Hk, hd, q, k, v, do)
    hs = lambda x: x.double().reshape(B, T, -1, hd).permute(0, 2, 1, 3).contiguous().requires_grad_()
    Q, K, V = hs(q), hs(k), hs(v)
    kk, vv = (x.repeat_interleave(Hq // Hk, 1) for x in (K, V))
    s = torch.matmul(Q, kk.transpose(2, 3).contiguous()) / math.sqrt(hd)
    s = s.masked_fill(torch.ones(T, T, dtype=torch.bool, device=DEV).triu(1), float("-inf"))
    pr = torch.softmax(s, -1)
    O = torch.matmul(pr, vv)
    O.backward(do.double().reshape(B, T, Hq, hd).permute(0, 2, 1, 3))
    fl = lambda x: x.permute(0, 2, 1, 3).reshape(B * T, -1)
    assert torch.allclose(p.double(), pr.detach().reshape(B * Hq, T, T), rtol=2e-5, atol=1e-7)
    assert bool((p.triu(1) == 0).all())
    for got, want in ((o, O.detach()), (dq, Q.grad), (dk, K.grad), (dv, V.grad)):
        w = fl(want)
        e = float((got.double() - w).norm() / w.norm().clamp_min(1e-30))
        # (T = 1: dS is exactly zero, so dQ and dK are)
        assert e < 4e-3 or float(got.double().abs().max()) < 1e-6, e


def test_infinite_value_stays_behind_the_mask():
    """Query tiles before an infinite V row see neither it nor a NaN from it in
    O and dQ; P and dV take nothing from V."""
    B, T, Hq, Hk, hd = 1, 190, 2, 1, 64
    q, k, v, do = inputs(B, T, Hq, Hk, hd)
    v[150] = float("inf")
    o, p, dq, dk, dv = run(B, T, Hq, Hk, hd, q, k, v, do)
    assert bool(torch.isfinite(o[:128]).all()) and bool(torch.isfinite(p).all())
    assert bool(torch.isfinite(dv).all()) and bool(torch.isfinite(dq[:128]).all())
