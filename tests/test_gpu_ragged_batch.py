"""Batches whose token count is no multiple of 64: the fused LoRA backward
kernels run over the padded rows (zeros), against the CPU oracle over two
steps from the oracle's state, to the step bars (loss 1e-3, gradients 1e-2
relative L2).  The recompute mode gives the cached step's bits there too,
and the padding holds zeros after the steps (a second engine, fed the same,
repeats them bit for bit)."""
import numpy as np
import pytest

import tadapt
from step_util import base_tensors, make_pair, pairs
from test_gpu_step import (SMALL_ADAPT, SMALL_MODEL, check_adamw_of_own_grads, compare, snapshot,
                           sync_state)

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("B,T,mask", [(1, 33, 0b1111111), (3, 45, 0b1111111), (1, 95, 0b0001111),
                                      (2, 63, 0b0110000), (1, 65, 0b1000000)])
def test_ragged_batch_matches_oracle(B, T, mask):
    mc, ac = SMALL_MODEL, dict(SMALL_ADAPT, inject_mask=mask)
    orc, eng = make_pair(mc, ac, B, T, seed=61)
    rng = np.random.default_rng(B * 100 + T)
    for step in range(2):
        sync_state(orc, eng, mc, ac)
        state = snapshot(orc, mc, ac)
        toks = rng.integers(0, mc["vocab"], B * T + 1).astype(np.int32)
        inp, tgt = toks[:-1].copy(), toks[1:].copy()
        so, sg = orc.step(inp, tgt, B, T), eng.step(inp, tgt)
        assert abs(sg["loss"] - so["loss"]) <= 1e-3 * abs(so["loss"]), (step, sg, so)
        assert abs(sg["gnorm_raw"] - so["gnorm_raw"]) <= 1e-2 * so["gnorm_raw"], (step, sg, so)
        compare(orc, eng, mc, ac, ("gB",) if step == 0 else ("gA", "gB"))
        check_adamw_of_own_grads(eng, mc, ac, state, sg["lr"], step + 1, sg["gnorm_raw"])


def test_ragged_batch_recompute_and_repeat_same_bits():
    mc, ac, B, T = SMALL_MODEL, SMALL_ADAPT, 3, 45
    engs = [tadapt.Engine(mc, ac, B, T, recompute=r) for r in (False, True, False)]
    for name, arr in base_tensors(mc, 7).items():
        for e in engs:
            e.set_weight(name, arr)
    rng = np.random.default_rng(3)
    for _ in range(3):
        toks = rng.integers(0, mc["vocab"], B * T + 1).astype(np.int32)
        m = [e.step(toks[:-1].copy(), toks[1:].copy()) for e in engs]
        assert m[0]["loss"] == m[1]["loss"] == m[2]["loss"]
        for l, t in pairs(mc, ac):
            for w in ("gA", "gB", "A", "B"):
                a = engs[0].adapter(l, t, w)
                assert all(np.array_equal(a, e.adapter(l, t, w)) for e in engs[1:]), (l, t, w)
    # named buffers keep the batch's own size
    assert engs[0].buffer("l0.gate")[1] == B * T * mc["inter"]
    assert engs[0].buffer("dQ")[1] == B * T * mc["n_q"] * mc["head_dim"]
