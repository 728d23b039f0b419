"""The choice of kernel forms for K-contiguous GEMMs (ta_gemm_plan: host
arithmetic, no GPU).

A product on 256 x 256 tiles whose last wave is nearly empty runs its last
columns as a second launch.  The LoRA terms of that launch exist only in the
layout the fused epilogues read, so it must not split K: a split leaves them
to a pass of its own, which needs the other layout.
"""
import ctypes

import pytest

import tadapt

TILES, DEEP, MID, BIG = range(4)


def plan(M, N, K, lora=1, beta=0, captured=0):
    out = (ctypes.c_int32 * 10)()
    tadapt.call("ta_gemm_plan", M, N, K, lora, beta, captured, ctypes.addressof(out))
    rows = [tuple(out[:5]), tuple(out[5:])]
    return [r for r in rows if r[0]]


def widths(M):
    """Output widths around every last wave of 256-wide tiles of at most half
    the CUs, up to 20,480 columns."""
    tm = (M + 255) // 256
    for full in range(1, 20480 // 256 * tm // 256 + 1):
        if full * 256 % tm:
            continue
        main = full * 256 // tm * 256
        for over in (64, 72, 120, 128, 136, 256, 448, 1000, 2048, 4096):
            if main + over <= 20480:
                yield main + over


@pytest.mark.parametrize("M", [256, 777, 1024, 2048, 2331, 4096, 6144, 8192, 16384])
def test_tail_never_splits(M):
    tails = 0
    for N in widths(M):
        for K in [64 * k for k in (2, 7, 14, 18, 24, 31, 32, 40, 56, 76, 140, 296)]:
            rows = plan(M, N, K)
            assert sum(r[0] for r in rows) == N, (M, N, K, rows)
            if len(rows) == 2:
                tails += 1
                assert rows[0][1] == BIG and rows[0][3] == 1, (M, N, K, rows)
                # and one of the forms whose epilogue takes the LoRA terms
                assert rows[1][1] in (DEEP, MID) and rows[1][3] == 1, (M, N, K, rows)
    assert tails or M in (256, 777, 2331)


def test_tail_of_a_wide_intermediate():
    """2048 tokens, hidden 1536, intermediate 8320, down_proj adapted: 264
    tiles, of which the last 128 columns run apart."""
    rows = plan(2048, 8320, 1536)
    assert len(rows) == 2 and rows[1] == (128, DEEP, 64, 1, 0), rows


def test_short_k_runs_two_blocks_per_cu():
    """Where both were timed, the 128-row forms' choice: 128-wide tiles of few
    stages, or with C read back, run k_gemm_mid's two blocks per CU."""
    for M, N in ((2048, 2048), (8192, 512), (1024, 3584)):
        for K in (64, 256, 512, 896, 1024):
            assert plan(M, N, K, 0)[0][1] == MID, (M, N, K)
            assert plan(M, N, K, 0, beta=1)[0][1] == MID, (M, N, K)
        assert plan(M, N, 1536, 0)[0][1:4] == (DEEP, 128, 1)
        assert plan(M, N, 1536, 0, beta=1)[0][1] == MID
    assert plan(512, 4864, 1536, 0, beta=1)[0][1:4] == (DEEP, 128, 1)
    assert plan(2048, 896, 896, 0, beta=1)[0][1:4] == (DEEP, 64, 1)


def test_splits_pay_for_their_second_launch():
    """Two launches take 10 us, so K = 1024 over a few tiles runs unsplit."""
    for M, N in ((128, 128), (128, 256), (256, 128)):
        assert plan(M, N, 1024, 0)[0][1:4] == (DEEP, 64, 1)
    assert plan(128, 896, 1536, 0)[0][1:4] == (DEEP, 64, 4)
    assert plan(128, 896, 4864, 0)[0][3] > 4


@pytest.mark.parametrize("M,N,K,order", [
    (4864, 3584, 18944, 1), (5888, 3584, 18944, 1), (9472, 3584, 12288, 1), (16640, 1536, 1536, 1),
    (4864, 18944, 3584, 0), (2331, 151936, 1536, 0), (3328, 8960, 1536, 0), (4864, 3584, 8192, 0),
    (3840, 3584, 18944, 0), (8192, 3584, 18944, 0)])
def test_launch_order(M, N, K, order):
    """The products that ran slower with each XCD on a range of tiles of its own."""
    assert plan(M, N, K, 0)[0][4] == order
