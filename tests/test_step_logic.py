"""A trip's step logic against the algorithm written out operation by operation.

Lane::trip_end decides first and then makes one pass over the Nordsieck array that takes
back or completes a step, weights, changes the order, rescales and predicts.  Here every
path through it starts from a prepared state and must leave what CVODE's separate
operations leave (Cohen & Hindmarsh, CVODE's cvRestore, cvCompleteStep, cvPrepareNextStep,
cvAdjustOrder, cvRescale, cvPredict and cvGetDky): the history, the weights, the step size,
order, counters and the next request.

Tolerance: an entry is the sum of at most 2^q = 32 terms of the column it starts from,
each through a dozen roundings: 400 of them, 1e-13 of the sum of magnitudes.
"""
import ctypes as C
import glob
import os
import subprocess

import numpy as np
import pytest

HERE = os.path.dirname(os.path.abspath(__file__))
EMU = os.path.join(HERE, "cpu_emulation")
CSRC = os.path.join(os.path.dirname(HERE), "pelelm_amd", "csrc")
SRC = [os.path.join(EMU, "emu_step.cpp"), os.path.join(EMU, "hip", "hip_runtime.h")]
SRC += [os.path.join(CSRC, f) for f in ("reactor_bdf.hip", "reactor_internal.h", "mlp_internal.h")]
CLANG = "/opt/rocm/llvm/bin/clang++"
SCAL = ("tn h hprime hscale eta etamax gamma gammap gamrat rl1 crate delp saved_tq5 saved_t a1 a2 teval rtol "
        "tout").split()
INTS = ("q qprime L qwait nst nstlp nstlj nstloc ncf nef nflag m convfail phase status setup_pending jcur "
        "callSetup").split()
NEED_CELL, NEWTON, RESTART_F = 0, 3, 4
FIRST_CALL, PREV_CONV_FAIL, PREV_ERR_FAIL = 0, 1, 2
NO_FAILURES, FAIL_BAD_J, FAIL_OTHER = 0, 1, 2
QMAX, RTOL, TOL = 5, 1e-6, 1e-13


@pytest.fixture(scope="module", params=["LiDryer", "drm19"])
def lib(request):
    m = request.param
    out = os.path.join(EMU, "_build", f"libstep_{m}.so")
    src = SRC + glob.glob(os.path.join(CSRC, "mech", m + ".inc"))
    if not os.path.exists(out) or any(os.path.getmtime(s) > os.path.getmtime(out) for s in src):
        os.makedirs(os.path.dirname(out), exist_ok=True)
        subprocess.run([CLANG, "-O1", "-std=c++17", "-fPIC", "-shared", "-DPELE_TU_MECH",
                        f'-DPELE_TU_MECH_INC="mech/{m}.inc"', f"-DPELE_TU_MECH_TYPE=mech_{m}",
                        f"-DPELE_TU_MECH_FN=mech_table_{m}", "-I" + EMU, "-I" + CSRC, "-o", out, SRC[0]], check=True)
    return C.CDLL(out)


class Cell:
    """A cell in the middle of an integration, its step converging at the first correction."""

    def __init__(self, N1, q, seed):
        rng = np.random.default_rng(seed)
        self.N1 = N1
        h = 1e-7
        self.s = dict(tn=5e-6, h=h, hprime=h, hscale=h, eta=1.0, etamax=10.0, gamma=0.7 * h, gammap=0.7 * h, gamrat=1.0,
                      rl1=0.7, crate=1.0, delp=0.0, saved_tq5=0.0, saved_t=5e-6 - h, a1=0.0, a2=0.0, teval=5e-6,
                      rtol=RTOL, tout=1e-5)
        self.n = dict(q=q, qprime=q, L=q + 1, qwait=3, nst=40, nstlp=39, nstlj=30, nstloc=40, ncf=1, nef=0,
                      nflag=FIRST_CALL, m=0, convfail=NO_FAILURES, phase=NEWTON, status=0, setup_pending=0, jcur=1,
                      callSetup=0)
        self.tq = np.array([0.0, 1e8, 0.5, 1e8, 1e9, 0.3])     # dsm = 0.5 |x|; other orders never pay
        self.l = np.concatenate([rng.uniform(0.2, 1.5, q + 1), np.zeros(5 - q)])
        self.tau = np.concatenate([[0.0], h * rng.uniform(0.5, 2.0, 6)])
        self.zn = rng.normal(size=(6, N1)) * 10.0 ** -np.arange(6)[:, None]
        self.zn[0] += 2.0 * np.sign(self.zn[0])
        self.ewt = 10.0 ** rng.uniform(0, 3, N1)
        self.x = rng.normal(size=N1)
        self.size(0.8)                                          # |x| = 0.8: the step passes
        self.acor = np.full(N1, np.nan)
        self.f = rng.normal(size=N1) * 1e3
        self.atol = np.full(N1, 1e-9)
        self.singular = 0
        self.mag = np.abs(self.zn)                              # of the terms summed so far

    def size(self, norm):
        self.x *= norm / self.wrms(self.x)

    def wrms(self, v):
        return np.sqrt(np.sum((v * self.ewt) ** 2) / self.N1)

    def run(self, lib):
        """The device code's trip; (reached, finite)."""
        d = np.array([self.s[k] for k in SCAL] + list(self.tq) + list(self.l) + list(self.tau))
        n = np.array([self.n[k] for k in INTS] + [QMAX, 20000], dtype=np.int32)
        p = lambda a: a.ctypes.data_as(C.c_void_p)  # noqa: E731
        zn, ewt, acor, fin = self.zn.copy(), self.ewt.copy(), self.acor.copy(), C.c_int(0)
        reached = lib.step_trip(p(d), p(n), p(zn), p(ewt), p(acor), p(self.x), p(self.f), p(self.atol), self.singular,
                                C.byref(fin))
        k = len(SCAL)
        return {"s": dict(zip(SCAL, d)), "n": dict(zip(INTS, n.tolist())), "tq": d[k:k + 6], "tau": d[k + 12:],
                "zn": zn, "ewt": ewt, "acor": acor, "reached": bool(reached), "finite": bool(fin.value)}

    # -- CVODE's operations, one by one ----------------------------------------
    def predict(self):
        self.s["tn"] += self.s["h"]
        for k in range(1, self.n["q"] + 1):
            for j in range(self.n["q"], k - 1, -1):
                self.zn[j - 1] += self.zn[j]
                self.mag[j - 1] += self.mag[j]

    def restore(self):
        self.s["tn"] = self.s["saved_t"]
        for k in range(1, self.n["q"] + 1):
            for j in range(self.n["q"], k - 1, -1):
                self.zn[j - 1] -= self.zn[j]
                self.mag[j - 1] += self.mag[j]

    def rescale(self):
        for j in range(1, self.n["q"] + 1):
            self.zn[j] *= self.s["eta"] ** j
            self.mag[j] *= self.s["eta"] ** j
        self.s["h"] = self.s["hscale"] = self.s["hscale"] * self.s["eta"]

    def order(self, dq):
        """cvAdjustOrder (BDF); the order itself is set by the caller's rules below."""
        q, hscale = self.n["q"], self.s["hscale"]
        l = np.zeros(7)
        l[2] = 1.0
        if dq == 1:
            alpha1 = prod = xiold = 1.0
            alpha0, hsum = -1.0, hscale
            for j in range(1, q):
                hsum += self.tau[j + 1]
                xi = hsum / hscale
                prod *= xi
                alpha0 -= 1.0 / (j + 1)
                alpha1 += 1.0 / xi
                for i in range(j + 2, 1, -1):
                    l[i] = l[i] * xiold + l[i - 1]
                xiold = xi
            A1 = (-alpha0 - alpha1) / prod
            self.zn[q + 1] = A1 * self.acor
            self.mag[q + 1] = np.abs(self.zn[q + 1])
            for j in range(2, q + 1):
                self.zn[j] += l[j] * self.zn[q + 1]
                self.mag[j] += np.abs(l[j] * self.zn[q + 1])
        elif q > 2:
            hsum = 0.0
            for j in range(1, q - 1):
                hsum += self.tau[j]
                xi = hsum / hscale
                for i in range(j + 2, 1, -1):
                    l[i] = l[i] * xi + l[i - 1]
            for j in range(2, q):
                self.zn[j] -= l[j] * self.zn[q]
                self.mag[j] += np.abs(l[j] * self.zn[q])
        self.n["q"] = q + dq
        self.n["L"] = self.n["qwait"] = q + dq + 1

    def attempt(self):
        """cvPredict and what the next trip is asked for."""
        self.predict()
        n = self.n
        n["convfail"] = NO_FAILURES if n["nflag"] in (FIRST_CALL, PREV_ERR_FAIL) else FAIL_OTHER
        n["m"], n["phase"] = 0, NEWTON
        self.s.update(a1=0.0, a2=0.0, teval=self.s["tn"])

    def complete(self, acnrm):
        """cvCompleteStep and cvPrepareNextStep; True when the order is to rise."""
        s, n, q = self.s, self.n, self.n["q"]
        n["nst"] += 1
        n["nstloc"] += 1
        self.tau[2:q + 1] = self.tau[1:q]
        if q == 1:
            self.tau[2] = self.tau[1]
        self.tau[1] = s["h"]
        for j in range(q + 1):
            self.zn[j] += self.l[j] * self.acor
            self.mag[j] += np.abs(self.l[j] * self.acor)
        n["qwait"] -= 1
        if n["qwait"] == 1 and q != QMAX:
            self.zn[QMAX] = self.acor
            s["saved_tq5"] = self.tq[5]
        def eta(bias, d, k):
            return 1.0 / ((bias * d) ** (1.0 / k) + 1e-6)
        etaq = eta(6.0, acnrm * self.tq[2], q + 1)
        n["qprime"] = q
        if s["etamax"] == 1.0:
            n["qwait"] = max(n["qwait"], 2)
            s["eta"] = 1.0
        else:
            s["eta"] = etaq
            if n["qwait"] == 0:
                n["qwait"] = 2
                down = eta(6.0, self.wrms(self.zn[q]) * self.tq[1], q) if q > 1 else 0.0
                up = 0.0
                if q != QMAX and s["saved_tq5"] != 0.0:
                    cq = (self.tq[5] / s["saved_tq5"]) * (s["h"] / self.tau[2]) ** (q + 1)
                    up = eta(10.0, self.wrms(self.acor - cq * self.zn[QMAX]) * self.tq[3], q + 2)
                best = max(down, etaq, up)
                if best >= 1.5 and best != etaq:
                    n["qprime"] = q - 1 if best == down else q + 1
                    if best == up:
                        self.zn[QMAX] = self.acor
                s["eta"] = best
            if s["eta"] < 1.5:
                s["eta"] = 1.0
                n["qprime"] = q
            else:
                s["eta"] = min(s["eta"], s["etamax"])
        s["hprime"] = s["h"] * s["eta"]
        s["etamax"] = 10.0
        return n["qprime"] - q


def _check(got, c, columns=None):
    cols = range(c.n["q"] + 1) if columns is None else columns
    for j in cols:
        assert np.all(np.abs(got["zn"][j] - c.zn[j]) <= TOL * c.mag[j]), j
    np.testing.assert_allclose(got["ewt"], c.ewt, rtol=TOL)
    np.testing.assert_allclose(got["tau"], c.tau, rtol=1e-15)
    for k in ("tn", "h", "hscale", "hprime", "eta", "etamax", "saved_t", "saved_tq5", "teval", "a1", "a2"):
        assert got["s"][k] == pytest.approx(c.s[k], rel=1e-12, abs=0.0), k
    for k in ("q", "L", "qwait", "qprime", "nst", "nstloc", "ncf", "nef", "nflag", "m", "convfail", "phase"):
        assert got["n"][k] == c.n[k], k


def _finish_step(c):
    """A completed step up to the next attempt."""
    c.acor = c.x.copy()
    acnrm = c.wrms(c.x)
    dq = c.complete(acnrm)
    c.ewt = 1.0 / (RTOL * np.abs(c.zn[0]) + c.atol)
    c.s["saved_t"] = c.s["tn"]
    c.n.update(ncf=0, nef=0, nflag=FIRST_CALL)
    if c.s["hprime"] != c.s["h"]:
        if dq:
            c.order(dq)
        c.rescale()
    c.attempt()


@pytest.mark.parametrize("q", [1, 2, 3, 4, 5])
@pytest.mark.parametrize("kind", ["same step", "larger step", "keeps the correction", "order down", "order up",
                                  "no growth allowed", "undecided order"])
def test_completed_step(lib, q, kind):
    if (kind == "order down" and q == 1) or (kind == "order up" and q == QMAX):
        pytest.skip("no such order")
    c = Cell(lib.step_n1(), q, 100 + q)
    if kind == "larger step":
        c.size(1e-4)
    elif kind == "keeps the correction":
        c.n["qwait"] = 2
    elif kind in ("order down", "order up"):
        # the measure of that order such that the step grows about threefold
        c.n["qwait"], c.s["saved_tq5"] = 1, 0.2
        if kind == "order down":
            c.tq[1] = 3.0 ** -q / (6.0 * c.wrms(c.zn[q] + c.l[q] * c.x))
        else:
            cq = c.tq[5] / 0.2 * (c.s["h"] / c.tau[1]) ** (q + 1)
            c.tq[3] = 3.0 ** -(q + 2) / (10.0 * c.wrms(c.x - cq * c.zn[QMAX]))
    elif kind == "no growth allowed":
        c.size(1e-4)
        c.n["qwait"], c.s["etamax"] = 1, 1.0
    elif kind == "undecided order":
        c.n["qwait"], c.s["saved_tq5"] = 1, 0.2
    got = c.run(lib)
    _finish_step(c)
    if kind in ("order down", "order up"):
        assert c.n["q"] == q + (1 if kind == "order up" else -1) and 2.9 < c.s["eta"] < 3.1
    _check(got, c)
    if kind == "keeps the correction" and q < QMAX:
        np.testing.assert_array_equal(got["zn"][QMAX], c.zn[QMAX])
    np.testing.assert_array_equal(got["acor"], c.x)


@pytest.mark.parametrize("q", [1, 2, 4, 5])
def test_later_correction_adds_up(lib, q):
    """The third correction: acor is the sum, and its norm is the error test's."""
    c = Cell(lib.step_n1(), q, 200 + q)
    c.n["m"], c.s["a2"], c.s["delp"], c.s["crate"] = 2, 1.0, 2.0, 0.5
    c.acor = 0.3 * c.x
    got = c.run(lib)
    c.s["crate"] = max(0.3 * 0.5, c.wrms(c.x) / 2.0)
    c.x = c.acor + c.x
    _finish_step(c)
    _check(got, c)
    np.testing.assert_array_equal(got["acor"], c.x)


@pytest.mark.parametrize("q", [1, 2, 3, 4, 5])
@pytest.mark.parametrize("nef", [0, 1, 3])
def test_failed_error_test(lib, q, nef):
    c = Cell(lib.step_n1(), q, 300 + q)
    c.size(5.0)                     # dsm = 2.5
    c.n["nef"] = nef
    got = c.run(lib)
    s, n = c.s, c.n
    n.update(nef=nef + 1, nflag=PREV_ERR_FAIL)
    c.restore()
    s["etamax"] = 1.0
    if nef + 1 <= 3:
        s["eta"] = max(0.1, 1.0 / ((6.0 * 2.5) ** (1.0 / (q + 1)) + 1e-6))
        if nef + 1 >= 2:
            s["eta"] = min(s["eta"], 0.2)
        c.rescale()
        c.attempt()
    elif q > 1:
        s["eta"] = 0.1
        c.order(-1)
        n["qwait"] = q
        c.rescale()
        c.attempt()
    else:
        s["eta"] = 0.1
        s["h"] = s["hscale"] = s["h"] * 0.1
        n.update(qwait=10, phase=RESTART_F)
        s.update(a1=0.0, a2=0.0, teval=s["tn"])
    _check(got, c)


@pytest.mark.parametrize("q", [1, 3, 5])
@pytest.mark.parametrize("cause", ["singular", "diverged with a current Jacobian"])
def test_convergence_failure_takes_the_step_back(lib, q, cause):
    c = Cell(lib.step_n1(), q, 400 + q)
    if cause == "singular":
        c.singular, c.n["setup_pending"] = 1, 1
    else:
        c.n["m"], c.s["a2"], c.s["delp"] = 1, 1.0, 1e-3     # twice the last correction and more
        c.acor = c.x.copy()
        c.tq[4] = 1e-9
    got = c.run(lib)
    c.n.update(ncf=2, nflag=PREV_CONV_FAIL)
    c.restore()
    c.s.update(etamax=1.0, eta=0.25)
    c.rescale()
    c.attempt()
    _check(got, c)
    assert got["n"]["callSetup"] == 1


@pytest.mark.parametrize("q", [1, 2, 5])
@pytest.mark.parametrize("bad", [False, True])
def test_output_is_interpolated_to_tout(lib, q, bad):
    c = Cell(lib.step_n1(), q, 500 + q)
    c.s["tout"] = c.s["tn"] - 0.3 * c.s["h"]
    if bad:
        c.zn[q, 3] = c.mag[q, 3] = np.inf
    got = c.run(lib)
    c.acor = c.x.copy()
    c.complete(c.wrms(c.x))
    want, mag = np.zeros(c.N1), np.zeros(c.N1)
    for j in range(q + 1):
        want += c.zn[j] * (-0.3) ** j
        mag += c.mag[j]
    assert got["reached"] and got["finite"] == (not bad)
    ok = np.isfinite(want)
    # the fraction of the step back to tout is a difference of times of 50 steps' size
    assert np.all(np.abs(got["zn"][0][ok] - want[ok]) <= (TOL + 50 * 2.3e-16) * mag[ok])


def test_restart_from_the_right_hand_side(lib):
    c = Cell(lib.step_n1(), 1, 600)
    c.n.update(phase=RESTART_F, nflag=PREV_ERR_FAIL, qwait=10)
    c.s["tn"] = c.s["saved_t"]
    got = c.run(lib)
    c.zn[1] = c.s["h"] * c.f
    c.mag[1] = np.abs(c.zn[1])
    c.attempt()
    _check(got, c)


def test_unconverged_correction_asks_for_another(lib):
    c = Cell(lib.step_n1(), 3, 700)
    c.tq[4] = 1e-9
    got = c.run(lib)
    assert got["n"]["m"] == 1 and got["s"]["a2"] == 1.0 and got["s"]["teval"] == c.s["tn"]
    assert got["s"]["delp"] == pytest.approx(c.wrms(c.x), rel=1e-14)
    np.testing.assert_array_equal(got["zn"], c.zn)
    np.testing.assert_array_equal(got["acor"], c.x)


def test_divergence_with_an_old_jacobian_starts_the_attempt_again(lib):
    c = Cell(lib.step_n1(), 3, 800)
    c.n.update(m=1, jcur=0)
    c.s["a2"], c.s["delp"] = 1.0, 1e-3
    c.acor = c.x.copy()
    c.tq[4] = 1e-9
    got = c.run(lib)
    n = got["n"]
    assert (n["m"], n["phase"], n["convfail"], n["callSetup"], n["ncf"]) == (0, NEWTON, FAIL_BAD_J, 1, 1)
    assert got["s"]["a2"] == 0.0 and got["s"]["teval"] == c.s["tn"] == got["s"]["tn"]
    np.testing.assert_array_equal(got["zn"], c.zn)
