"""The cooperative factorisation's pivot choice and the batched trips of small boxes.

Pivots: block-diagonal matrices of 2 x 2 blocks whose first columns tie exactly, rows and
columns permuted over the whole matrix, so that elimination stays in exact arithmetic and
the rule "largest magnitude, ties to the lowest row" fixes the whole permutation.
Entries of 1 and 1 + 2^-40 share the upper 32 bits and zeros have none set: the cases that
the search by upper words must settle on the lower ones.
"""
import numpy as np
import pytest

import test_gpu_unit as U


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
