"""The merge's launches (one block per center and Lloyd pass) at their edges,
bit for bit against the oracle: around 64 snapshots per chunk, past 4096 (the
member bits then leave LDS) and past 1024 (the seeding then forms its chains
per draw), dimensions off and past the 32-element and LDS center sizes, data
that settles at once and data that does not, duplicates (empty centers),
few and many passes, and the one-workgroup loop beyond 128 passes."""
import ctypes

import numpy as np
import pytest
import torch

import oracle as O
from gpu_util import DEV, P, S, call, dev, host

pytestmark = pytest.mark.gpu


def data(N, D, kind):
    r = np.random.default_rng(N * 7 + D)
    if kind == "mixture":
        means = r.standard_normal((5, D))
        X = means[r.integers(0, 5, N)] + 0.3 * r.standard_normal((N, D))
    elif kind == "spread":
        X = r.standard_normal((N, D))
    else:  # three points, repeated: empty centers
        X = r.standard_normal((3, D))[r.integers(0, 3, N)]
    return np.ascontiguousarray(X.astype(np.float32)), r.lognormal(0, 1, N).astype(np.float32)


SHAPES = [(1, 1, 1, 5), (2, 3, 2, 4), (63, 33, 9, 25), (64, 512, 32, 25), (65, 500, 32, 7),
          (130, 31, 40, 25), (1030, 17, 6, 12), (4200, 5, 4, 6), (20, 4100, 5, 6)]
# the stress mode's one-workgroup form: its limits (128 snapshots, 8192 values,
# 4096 distances) and one past each, both sides of its rule, passes that stop
# early and none; centers past what is resident at once; one center
PP_SMALL = [(1, 1, 1, 0), (4, 16, 2, 1000), (128, 64, 2, 25), (129, 63, 2, 25), (8, 1024, 2, 5),
            (8, 1025, 2, 5), (64, 5, 64, 300), (65, 5, 64, 300), (16, 50, 8, 0), (16, 50, 8, 25),
            (100, 12, 40, 200), (1100, 33, 1024, 4), (500, 70, 1, 3)]


@pytest.mark.parametrize("kind", ["mixture", "spread", "dups"])
@pytest.mark.parametrize("N,D,k,iters", SHAPES + PP_SMALL)
def test_pp(N, D, k, iters, kind):
    X, W = data(N, D, kind)
    C = torch.empty(k * D, device=DEV)
    A = torch.empty(N, dtype=torch.int32, device=DEV)
    M = torch.empty(k, dtype=torch.float64, device=DEV)
    Sd = torch.empty(k, dtype=torch.int32, device=DEV)
    call("ta_kmeans_pp", P(dev(X)), P(dev(W)), N, D, k, iters, ctypes.c_uint64(77), P(C), P(A),
         P(M), P(Sd), S())
    rc, ra, rm, rs = O.kmeans_pp(X, W, k, iters, 77)
    assert np.array_equal(host(Sd), rs) and np.array_equal(host(A), ra)
    assert np.array_equal(host(C).reshape(k, D), rc)
    assert np.allclose(host(M), rm, rtol=1e-12)


# (the launches are taken by work per pass against the cap: all of these at 50,
# none at 200; members past 4096 snapshots, a ragged last chunk of 64, more
# centers than are resident at once)
REF_LAUNCHED = [(64, 512, 64, 0), (300, 256, 12, 0), (130, 300, 40, 0), (1030, 33, 6, 0),
                (4200, 64, 16, 0), (4229, 33, 16, 0), (20, 4100, 5, 0), (2050, 40, 2049, 0)]


@pytest.mark.parametrize("kind", ["mixture", "spread", "dups"])
@pytest.mark.parametrize("N,D,k,iters", SHAPES + REF_LAUNCHED)
def test_ref(N, D, k, iters, kind):
    X, _ = data(N, D, kind)
    out = []
    for cap in (50, 200):  # one launch per pass (REF_LAUNCHED); the one-workgroup loop
        C = torch.empty(k * D, device=DEV)
        A = torch.empty(N, dtype=torch.int32, device=DEV)
        it = torch.empty(1, dtype=torch.int32, device=DEV)
        call("ta_kmeans_ref", P(dev(X)), N, D, k, cap, P(C), P(A), P(it), S())
        out.append((host(C).reshape(k, D), host(A), int(host(it)[0])))
    rc, ra, ri = O.kmeans_ref(X, k)
    for c, a, i in out[: 2 if out[1][2] <= 50 else 1]:
        assert np.array_equal(a, ra) and np.array_equal(c, rc) and i == ri


@pytest.mark.parametrize("N,D,k", [(90, 64, 8), (300, 256, 12)])
def test_few_passes_match_the_loop(N, D, k):
    """A cap below the passes the data needs, in the one-workgroup loop and in
    launches: centers after the last update, assignments of the last pass; no
    pass at all leaves the initial centers."""
    X, _ = data(N, D, "spread")
    for cap in (0, 1, 2, 3):
        C = torch.full((k * D,), -1.0, device=DEV)
        A = torch.full((N,), -1, dtype=torch.int32, device=DEV)
        it = torch.full((1,), -1, dtype=torch.int32, device=DEV)
        call("ta_kmeans_ref", P(dev(X)), N, D, k, cap, P(C), P(A), P(it), S())
        want_c = X[[(i * N) // k for i in range(k)]].copy()
        asg, n_it = np.zeros(N, np.int32), 0
        for _ in range(cap):
            d = np.zeros((N, k), np.float32)
            for i in range(D):
                t = (X[:, None, i] - want_c[None, :, i]).astype(np.float32)
                d = (d + (t * t).astype(np.float32)).astype(np.float32)
            a = d.argmin(1).astype(np.int32)
            if np.array_equal(a, asg):
                break
            asg, n_it = a, n_it + 1
            for c in range(k):
                mem = np.nonzero(asg == c)[0]
                s = np.zeros(D, np.float32)
                for n in mem:
                    s = (s + X[n]).astype(np.float32)
                want_c[c] = s / np.float32(len(mem)) if len(mem) else 0
        assert np.array_equal(host(C).reshape(k, D), want_c)
        assert np.array_equal(host(A), asg) and int(host(it)[0]) == n_it


@pytest.mark.parametrize("pp", [True, False])
@pytest.mark.parametrize("N,D,k", [(2, 2_200_000, 2), (64 * 65536 + 10, 1, 2)])
def test_more_blocks_than_a_small_grid_dimension(N, D, k, pp):
    """Dimensions and snapshot counts beyond 65,535 tiles or blocks: the grids
    put them in x."""
    X, W = data(N, D, "dups")
    C = torch.empty(k * D, device=DEV)
    A = torch.empty(N, dtype=torch.int32, device=DEV)
    it = torch.empty(1, dtype=torch.int32, device=DEV)
    if pp:
        call("ta_kmeans_pp", P(dev(X)), P(dev(W)), N, D, k, 2, ctypes.c_uint64(5), P(C), P(A),
             None, None, S())
        rc, ra = O.kmeans_pp(X, W, k, 2, 5)[:2]
    else:
        call("ta_kmeans_ref", P(dev(X)), N, D, k, 50, P(C), P(A), P(it), S())
        rc, ra, ri = O.kmeans_ref(X, k)
        assert int(host(it)[0]) == ri
    assert np.array_equal(host(A), ra)
    assert np.array_equal(host(C).reshape(k, D), rc)
