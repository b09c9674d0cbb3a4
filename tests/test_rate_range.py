"""Rates and Jacobians at temperatures where exponentials of single species' g/RT and their
products leave a double's range (below about 100 to 170 K, by mechanism) though those of a
reaction's own difference do not: the generated forms multiply the former, so outside a
range of temperatures the reactions are evaluated one by one (M::T_LOW, M::T_HIGH).

Every entry has to be a number and right on both sides of the line.  The rates are compared
with 50-digit values; an entry may be off by 1e-11 of the sum of its reactions' forward and
backward rates: an exponent of up to 1200 is known to 1200 roundings of its terms, 1.3e-13,
twice over, and each sum has up to 400 terms.  The Jacobians are compared with the oracle's
where those are numbers, with the same tolerance on the same kind of sums: a row's largest
entry for the derivatives by composition, and for those by temperature the reactions'
forward and backward rates times what their logarithms' derivatives are summed from.
"""
import ctypes as C
import glob
import os
import subprocess
import sys

import numpy as np
import pytest

from oracle import oracle as O
from pelelm_amd.mechanisms import hipgen
from pelelm_amd.mechanisms import mechanism as M

HERE = os.path.dirname(os.path.abspath(__file__))
EMU = os.path.join(HERE, "cpu_emulation")
CSRC = os.path.join(os.path.dirname(HERE), "pelelm_amd", "csrc")
SRC = [os.path.join(EMU, "emu_chem.cpp"), os.path.join(EMU, "hip", "hip_runtime.h")]
SRC += [os.path.join(CSRC, f) for f in ("reactor_bdf.hip", "reactor_internal.h", "mlp_internal.h")]
CLANG = "/opt/rocm/llvm/bin/clang++"
MECHS = ["LiDryer", "drm19", "dodecane53", "dodecane56", "heptane88"]
TOL = 1e-11


def _lib(mech):
    out = os.path.join(EMU, "_build", f"libchem_{mech}.so")
    src = SRC + glob.glob(os.path.join(CSRC, "mech", mech + ".inc"))
    if not os.path.exists(out) or any(os.path.getmtime(s) > os.path.getmtime(out) for s in src):
        os.makedirs(os.path.dirname(out), exist_ok=True)
        subprocess.run([CLANG, "-O1", "-std=c++17", "-fPIC", "-shared", "-DPELE_TU_MECH",
                        f'-DPELE_TU_MECH_INC="mech/{mech}.inc"', f"-DPELE_TU_MECH_TYPE=mech_{mech}",
                        f"-DPELE_TU_MECH_FN=mech_table_{mech}", "-I" + EMU, "-I" + CSRC, "-o", out, SRC[0]], check=True)
    return C.CDLL(out)


def _p(a):
    return a.ctypes.data_as(C.c_void_p)


def _states(mech):
    """Concentrations and temperatures: 80 K up to the fits, the line's two sides among them."""
    lo, hi = hipgen.shared_range(mech)
    rng = np.random.default_rng(7)
    T = np.array([80.0, 90.0, 100.0, 110.0, 120.0, 130.0, 150.0, 170.0, lo - 0.5, lo + 0.5, 260.0, 300.0,
                  1500.0, 3500.0, hi + 100.0])
    Cc = 10.0 ** rng.uniform(-14.0, -5.0, (len(T), mech.nspec))
    return Cc, T


def _golden():
    sys.path.insert(0, os.path.join(HERE, "golden"))
    try:
        import make_wdot_golden as G
    finally:
        sys.path.pop(0)
    return G


def _gross(mech, Cc, T, G):
    """Sums over the reactions that each species takes part in of their forward and backward
    rates, and of these times the terms of d ln k / dT."""
    mp = G.mp
    g, hs = [], []
    for sp in mech.species:
        _, h, s = G.nasa(sp, mp.mpf(T))
        g.append(h - s)
        hs.append(abs(h))
    refC = mp.mpf(M.P_ATM) / (mp.mpf(M.R_CGS) * T)
    out = [[mp.mpf(0)] * mech.nspec for _ in range(2)]
    for r in mech.reactions:
        k = mp.mpf(r.A) * mp.mpf(T) ** r.beta * mp.exp(-mp.mpf(r.Ea) / (mp.mpf(M.R_CAL) * T))
        if r.has_third_body:   # an upper bound: without fall-off
            k *= sum(r.efficiencies.get(i, 1.0) * mp.mpf(c) for i, c in enumerate(Cc))
            if r.kind == "falloff":
                A0, b0, E0 = r.low
                k = mp.mpf(A0) * mp.mpf(T) ** b0 * mp.exp(-mp.mpf(E0) / (mp.mpf(M.R_CAL) * T)) * k / (
                    mp.mpf(r.A) * mp.mpf(T) ** r.beta * mp.exp(-mp.mpf(r.Ea) / (mp.mpf(M.R_CAL) * T)))
        f = k
        for i, nu in r.reactants.items():
            f *= mp.mpf(Cc[i]) ** nu
        if r.reversible:
            b = k
            for i, nu in r.products.items():
                b *= mp.mpf(Cc[i]) ** nu
            dG = sum(nu * g[i] for i, nu in r.products.items()) - sum(nu * g[i] for i, nu in r.reactants.items())
            dnu = sum(r.products.values()) - sum(r.reactants.values())
            f += b * mp.exp(dG) * refC ** (-dnu)
        terms = abs(r.beta) + abs(r.Ea) / (M.R_CAL * T)
        if r.low is not None:
            terms += abs(r.low[1]) + abs(r.low[2]) / (M.R_CAL * T)
        for side in (r.reactants, r.products):
            terms += sum(nu * (hs[i] + 1) for i, nu in side.items())
        for side in (r.reactants, r.products):
            for i, nu in side.items():
                out[0][i] += nu * f
                out[1][i] += nu * f * terms / T
    return out


def _enthalpy(mech, rY, T):
    """rho h [erg/cm^3] of cells rY [nspec, n] at T [n]."""
    return np.array([sum(rY[k, c] / sp.W * M.R_CGS * T[c] * M.h_RT(sp, T[c]) for k, sp in enumerate(mech.species))
                     for c in range(len(T))])


def _check_rates(mech, rY, Tc, out):
    G, W = _golden(), np.array(mech.W)
    for c in range(len(Tc)):
        conc = rY[:, c] / W
        want, gross = G.wdot(mech, conc, Tc[c]), _gross(mech, conc, Tc[c], G)[0]
        for k in range(mech.nspec):
            if gross[k] * W[k] > 1e280:
                continue
            got = out[k, c] / W[k]
            assert np.isfinite(got), (mech.name, Tc[c], mech.names[k])
            # 1e-280: an entry below is as good as zero
            assert abs(G.mp.mpf(got) - want[k]) <= TOL * gross[k] + 1e-280, (mech.name, Tc[c], mech.names[k], got)


@pytest.mark.parametrize("name", MECHS)
def test_rates_are_right_down_to_80_K(name):
    mech, L = M.load(name), _lib(name)
    lo, hi = C.c_double(), C.c_double()
    L.chem_range(C.byref(lo), C.byref(hi))
    assert (lo.value, hi.value) == hipgen.shared_range(mech)
    Cc, T = _states(mech)
    rY = np.ascontiguousarray((Cc * np.array(mech.W)).T)
    rH, Tc, out = _enthalpy(mech, rY, T), T.copy(), np.zeros((mech.nspec, len(T)))
    assert L.chem_rates(C.c_long(len(T)), _p(rY), _p(rH), _p(Tc), _p(out)) == 0
    assert np.abs(Tc - T).max() < 1e-6
    _check_rates(mech, rY, Tc, out)


@pytest.mark.gpu
@pytest.mark.parametrize("name", MECHS)
def test_gpu_rates_are_right_down_to_80_K(name):
    import torch

    from pelelm_amd import reactor
    mech = M.load(name)
    Cc, T = _states(mech)
    rY = np.ascontiguousarray((Cc * np.array(mech.W)).T)
    dev = [torch.tensor(a, device="cuda") for a in (rY, _enthalpy(mech, rY, T), T)]
    out, Tc = torch.zeros_like(dev[0]), torch.zeros_like(dev[2])
    r = reactor.ReactorBase.create("ReactorCvode")
    r.set("mi.mechanism", name)
    r.init(2, len(T))
    r.reaction_rates(*dev, None, out, Tc)
    torch.cuda.synchronize()
    r.close()
    _check_rates(mech, rY, Tc.cpu().numpy(), out.cpu().numpy())


def _jac_inputs(mech, m):
    Cc, T = _states(mech)
    y = np.ascontiguousarray(np.concatenate([Cc * np.array(mech.W), T[:, None]], axis=1))
    return Cc, T, y, np.array([m.rhs_fixedT(y[c])[-1] for c in range(len(T))])


def _check_jacobian(mech, m, Cc, T, y, fT, J):
    G, W, N = _golden(), np.array(mech.W), mech.nspec
    seen = 0
    for c in range(len(T)):
        ref = m.jac(y[c])
        if not (np.isfinite(ref).all() and np.isfinite(fT[c])):
            continue
        seen += 1
        assert np.isfinite(J[c]).all(), (mech.name, T[c])
        d = np.abs(J[c] - ref)[:N]
        scale = np.abs(ref[:N, :N]).max(axis=1)
        assert (d[:, :N] <= TOL * scale[:, None] + 1e-280).all(), (mech.name, T[c])
        for k, t in enumerate(_gross(mech, Cc[c], T[c], G)[1]):
            assert d[k, -1] <= TOL * W[k] * t + 1e-280, (mech.name, T[c], mech.names[k])
    assert seen >= 8


@pytest.mark.parametrize("name", MECHS)
def test_jacobian_is_right_down_to_80_K(name):
    mech, L, m = M.load(name), _lib(name), O.Mech(name)
    Cc, T, y, fT = _jac_inputs(mech, m)
    J = np.zeros((len(T),) + (mech.nspec + 1,) * 2)
    L.chem_jac(C.c_long(len(T)), _p(y), _p(fT), _p(J))
    _check_jacobian(mech, m, Cc, T, y, fT, J)


@pytest.mark.gpu
@pytest.mark.parametrize("name", MECHS[:3])
def test_gpu_jacobian_is_right_down_to_80_K(name):
    import test_gpu_unit as U
    mech, m = M.load(name), O.Mech(name)
    Cc, T, y, fT = _jac_inputs(mech, m)
    # every state in three lanes: the unit kernel leaves each third one idle
    assert 3 * len(T) <= 64
    y3, T3, fT3 = (np.repeat(a, 3, axis=0) for a in (y, T, fT))
    J = U.run_jac_lu(U._load("libunit_gpu.so"), name, y3, T3, fT3, np.full(len(T3), 1e-30), np.zeros_like(y3))[0]
    for lane in (1, 2):
        _check_jacobian(mech, m, Cc, T, y, fT, J[lane::3])


def test_range_follows_the_shift_in_use():
    """A reaction that does not conserve the elements leaves the mechanism without their
    shift: the range in which products of exponentials are used is then that of the others."""
    import copy
    mech = M.load("drm19")
    lumped = copy.deepcopy(mech)
    lumped.reactions.append(M.Reaction("CH4 => CO2", {mech.index("CH4"): 1}, {mech.index("CO2"): 1}, False,
                                       "elementary", 1e10, 0.0, 2e4))
    assert set(hipgen._element_shift(lumped)) == {(0.0, 0.0)}
    for m, below, inside in ((mech, 0.0, True), (mech, 5.0, False), (lumped, 0.0, True), (lumped, 5.0, False)):
        T = hipgen.shared_range(m)[0] - below
        worst = 0.0
        for r in m.reactions:
            for side in (r.reactants, r.products):
                g = sum(c * (M.h_RT(m.species[i], T) - M.s_R(m.species[i], T) + d5 / T - d6)
                        for i, c in side.items() for d5, d6 in [hipgen._element_shift(m)[i]])
                worst = max(worst, abs(g), abs(r.beta * np.log(T) - r.Ea / M.R_CAL / T))
        assert (worst <= hipgen.SHARED_LIMIT) == inside
