"""A down projection wide enough that its input gradient (2048 x 8320 x 1536)
runs its last 128 columns as a launch of its own, with the LoRA terms of the
adapted projection: two steps against the CPU oracle.

The first step's update (learning rate 0.1) gives B its size, so that in the
second the LoRA terms are a quarter of the gradient.  The gate projection's gB
has one row per column of that gradient, so the last launch's columns are
compared on their own too.  Bars as in the other steps: loss 1e-3, gradients
1e-2 relative L2.
"""
import numpy as np
import pytest

from step_util import make_pair, rel
from test_gpu_step import SMALL_ADAPT, compare, sync_state

pytestmark = pytest.mark.gpu

MODEL = dict(vocab=512, hidden=1536, layers=1, n_q=12, n_kv=2, head_dim=128, inter=8320,
             rms_eps=1e-6, rope_theta=1e6, tie=1)


def test_adapted_tail_columns_match_oracle():
    mc, ac, B, T = MODEL, dict(SMALL_ADAPT, inject_mask=0b1010000), 2, 1024
    orc, eng = make_pair(mc, ac, B, T, seed=23)
    rng = np.random.default_rng(29)
    for step in range(2):
        sync_state(orc, eng, mc, ac)
        toks = rng.integers(0, mc["vocab"], B * T + 1).astype(np.int32)
        inp, tgt = toks[:-1].copy(), toks[1:].copy()
        so = orc.step(inp, tgt, B, T, lr_override=0.1)
        sg = eng.step(inp, tgt, lr_override=0.1)
        assert abs(sg["loss"] - so["loss"]) <= 1e-3 * abs(so["loss"]), (step, sg, so)
        compare(orc, eng, mc, ac, ("gB",) if step == 0 else ("gA", "gB"))
        go, gg = (np.asarray(e.adapter(0, "gate", "gB")).reshape(mc["inter"], -1)
                  for e in (orc, eng))
        assert rel(gg[8192:], go[8192:]) <= 1e-2, (step, rel(gg[8192:], go[8192:]))
