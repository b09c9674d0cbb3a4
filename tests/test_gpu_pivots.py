"""The cooperative factorisation's pivot choice and the batched trips of small boxes.

Pivots: block-diagonal matrices of 2 x 2 blocks whose first columns tie exactly, rows and
columns permuted over the whole matrix, so that elimination stays in exact arithmetic and
the rule "largest magnitude, ties to the lowest row" fixes the whole permutation.
Entries of 1 and 1 + 2^-40 share the upper 32 bits and zeros have none set: the cases that
the search by upper words must settle on the lower ones.
"""
import numpy as np
import pytest
import torch   # before the unit library: a process takes its HIP runtime from the first of the two

import test_gpu_unit as U
from pelelm_amd import cells, reactor


def _matrix(rng, n1, kind):
    m = np.zeros((n1, n1))
    for k in range(0, n1 - 1, 2):
        s = 2.0 ** rng.integers(-3, 4)
        m[k:k + 2, k:k + 2] = [[s, s], [s if kind != "lower" else s * (1 + 2.0 ** -40), -s]]
    if n1 % 2:
        m[-1, -1] = 1.0
    if kind == "singular":
        m[:, 0] = 0.0
    return m[rng.permutation(n1)][:, rng.permutation(n1)]


def _pivots(m):
    """Row order and first zero-pivot column (0: none) by the rule, unblocked, rows in place."""
    m, n1 = m.copy(), len(m)
    live, perm, sing = np.ones(n1, bool), [], 0
    for k in range(n1):
        mag = np.where(live, np.abs(m[:, k]), -1.0)
        p = int(np.argmax(mag))          # the first of equal ones
        if mag[p] == 0.0 and sing == 0:
            sing = k + 1
        perm.append(p)
        live[p] = False
        if mag[p] > 0.0:
            l = np.where(live, m[:, k] * (1.0 / m[p, k]), 0.0)
            rest = np.outer(l, m[p, k + 1:])
            m[:, k + 1:] -= np.where(l[:, None] != 0.0, rest, 0.0)
    return perm, sing


@pytest.mark.gpu
@pytest.mark.parametrize("kind", ["ties", "lower", "singular"])
@pytest.mark.parametrize("mech,n1", [("LiDryer", 10), ("drm19", 22), ("dodecane53", 54)])
def test_pivot_order_with_ties(mech, n1, kind):
    rng = np.random.default_rng(n1)
    n = 67   # an odd count: the last wave of two cells is half empty
    m = np.stack([_matrix(rng, n1, kind) for _ in range(n)])
    J = np.ascontiguousarray(np.eye(n1)[None] - m)   # gamma = 1: I - gamma J is m
    m = np.eye(n1)[None] - J                          # as the kernel forms it
    pend = np.ones(n, dtype=np.int32)
    b = rng.integers(-8, 9, (n, n1)).astype(float)
    x, sing, lu, perm, _ = U.run_lu(U._load("libunit_gpu.so"), mech, 1, J, np.ones(n), pend, b)
    for c in range(n):
        want, first = _pivots(m[c])
        assert sing[c] == first
        assert list(perm[c]) == want
        if kind in ("ties", "lower"):
            # condition number below 10: a few hundred rounding errors of the solution
            xe = np.linalg.solve(m[c], b[c])
            assert np.max(np.abs(x[c] - xe)) <= 1e-12 * np.max(np.abs(xe))


@pytest.mark.gpu
@pytest.mark.parametrize("mech,n1", [("LiDryer", 10), ("drm19", 22), ("dodecane53", 54)])
def test_factorisation_solves_its_first_system(mech, n1):
    """The solution that the cooperative factorisation forms from its registers: that of the
    solve kernel and of numpy, on the pending cells alone (every fifth is idle, every seventh
    singular: those keep what they held, 0)."""
    rng = np.random.default_rng(100 + n1)
    n = 131   # half a wave left over where two cells share one
    m = np.eye(n1)[None] + rng.uniform(-0.5, 0.5, (n, n1, n1)) / np.sqrt(n1)
    m = np.stack([a[rng.permutation(n1)] for a in m])
    singular = np.arange(n) % 7 == 3
    m[singular, :, n1 // 2] = 0.0
    pend = (np.arange(n) % 5 != 0).astype(np.int32)
    b = rng.normal(size=(n, n1))
    J = np.ascontiguousarray(np.eye(n1)[None] - m)
    m = np.eye(n1)[None] - J
    G = U._load("libunit_gpu.so")
    x, sing, lu, perm, _ = U.run_lu(G, mech, 3, J, np.ones(n), pend, b)
    x1, sing1, lu1, perm1, _ = U.run_lu(G, mech, 1, J, np.ones(n), pend, b)
    ok = (pend == 1) & ~singular
    np.testing.assert_array_equal(sing, sing1)
    np.testing.assert_array_equal(perm, perm1)
    np.testing.assert_array_equal(lu, lu1)
    assert np.all(sing[ok] == 0) and np.all(sing[(pend == 1) & singular] == n1 // 2 + 1)
    assert np.all(x[~ok] == 0.0)
    # condition numbers below 100: 1e4 rounding errors of the solution at most
    xe = np.linalg.solve(m[ok], b[ok][..., None])[..., 0]
    size = np.abs(xe).max(axis=1, keepdims=True)
    assert np.linalg.cond(m[ok]).max() < 100.0
    assert np.max(np.abs(x[ok] - xe) / size) < 1e-12
    assert np.max(np.abs(x[ok] - x1[ok]) / size) < 1e-12


@pytest.mark.gpu
@pytest.mark.parametrize("solve", ["denseAJ_direct", "GMRES"])
@pytest.mark.parametrize("schedule", ["plain", "queue"])
@pytest.mark.parametrize("wl,mech,n", [("lidryer_16", "LiDryer", 4096), ("drm19_64", "drm19", 4096),
                                       ("dodecane53_64_mix", "dodecane53", 2048)])
def test_batched_trips_change_nothing(wl, mech, n, schedule, solve):
    """A box whose trips come in batches (GMRES, and the compacted lists of the smallest
    mechanism) or with each evaluation ahead of the counts (plain), and the same box with its
    kernels timed, where trips come one by one: the same states, counts and trips, with all
    cells done and with a cap on trips that is no multiple of a batch."""
    d = cells.generate_workload(wl, ncell=n)
    for cap in (0, 19):
        got = []
        for profile in (0, 1):
            r = reactor.ReactorBase.create("ReactorCvode")
            for k, v in (("mi.mechanism", mech), ("ode.rtol", 1e-6), ("ode.atol", 1e-10), ("mi.schedule", schedule),
                         ("cvode.solve_type", solve), ("mi.max_trips", cap), ("mi.on_fail", "continue"),
                         ("mi.profile", profile)):
                r.set(k, v)
            r.init(2, n)
            s = [torch.tensor(d[k], device="cuda") for k in ("rY", "T", "rE")]
            FC = torch.zeros(n, dtype=torch.float64, device="cuda")
            r.react(s[0], None, s[1], s[2], None, FC, None, d["dt"])
            torch.cuda.synchronize()
            st = r.stats()
            r.close()
            got.append([t.cpu().numpy() for t in s + [FC]] + [np.array([st[k] for k in ("ntrips", "nfe", "nsteps", "nfail")])])
            assert st["nfail"] == np.count_nonzero(FC.cpu().numpy() < 0)
            # (without a cap, five Krylov vectors leave one cell of the 53-species mix unsolved)
            assert st["nfail"] > 0 or cap == 0
            assert cap == 0 or st["ntrips"] == 19
        for a, b in zip(*got):
            np.testing.assert_array_equal(a, b)
