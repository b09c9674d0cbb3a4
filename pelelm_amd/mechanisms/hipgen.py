"""Emit HIP device code for one mechanism (one cell per lane).

The generated header defines ``struct mech_<name>`` with static members:

* ``NS``, ``NR``, ``N1`` and the constant tables host code needs (molecular weights,
  species names);
* ``range(T)`` and ``mix(range, w, A)`` -- the NASA-7 range of a temperature, and the
  mixture's coefficients A_j = sum_k w_k a_jk / W_k in it, so that h and cp of a mixture
  are one polynomial each (HY2T, energy equation);
* ``thermo_cph(T, cpR, hRT)``, ``thermo_dcp(T, dcpR)`` -- cp/R, h/RT and d(cp/R)/dT of
  every species (Jacobian);
* ``gibbs(T, logT, gRT)`` -- g/RT, each element's potential shifted by a constant that no
  balanced reaction sees (``_element_shift``);
* ``wdot(C, T, logT, invT, gRT, wd)`` -- net molar production rates [mol/cm^3/s];
* ``jacobian(C, T, logT, invT, gRT, hRT, wd, dwdT, acc)`` -- the analytic derivatives
  d(wdot_i W_i)/d(rhoY_k) accumulated through ``acc(i, k, value)`` plus dwdot/dT.

The NASA-7 coefficients come from tables in constant memory whose address is uniform over
a wave (scalar loads, one scalar operand per FMA): the two ranges are the two trips of a
loop that a wave enters for the lanes on that side, so a wave on one side runs one of
them.  (Coefficients written as selects between two literals cost four moves and two
selects each, three times the polynomial's own arithmetic.)

Every transcendental of a state is evaluated once: exp(g_k/RT) and its reciprocal per
species instead of exp(-dG/RT) per reaction, and exp(b ln T - Ta/T) once per distinct
(b, Ta), the reactions that share it emitted next to each other.  drm19: 199 of them
become 133; the 88-species mechanism: 856 become 278.  Troe terms with T*** = 1e-30 /
T* = 1e30 vanish / become constants; third-body sums start from the total concentration
and add (eff - 1) C_k only for species with non-unit efficiency.

``gen_thermo``, ``gen_wdot`` and ``gen_jacobian(shared=False)`` write the same arithmetic
out species by species and reaction by reaction; the operation counts "functions" are
counted on that form, which says what a mechanism asks for and not how the emitted code
saves on it, and "emitted" on the code that runs.
"""
from __future__ import annotations

import json
import math
import os
import re

import numpy as np

from . import mechanism as M


def _d(x: float) -> str:
    r = repr(float(x))
    if "e" not in r and "." not in r and "inf" not in r and "nan" not in r:
        r += ".0"
    return r


def _cname(name: str) -> str:
    return name.replace("(", "_").replace(")", "_").replace("-", "m").replace("*", "s")


def _prod(terms: list) -> str:
    return " * ".join(terms) if terms else "1.0"


def _power_terms(side: dict) -> list:
    t = []
    for i, c in sorted(side.items()):
        t += [f"C[{i}]"] * c
    return t


def _dpower_terms(side: dict, k: int) -> tuple[float, list]:
    """d/dC_k of prod C^nu: coefficient and remaining factors."""
    c = side[k]
    t = []
    for i, ci in sorted(side.items()):
        n = ci - 1 if i == k else ci
        t += [f"C[{i}]"] * n
    return float(c), t


def _thermo_groups(mech: M.Mechanism) -> dict:
    groups: dict = {}
    for k, s in enumerate(mech.species):
        groups.setdefault(s.T[1], []).append(k)
    return groups


def gen_thermo(mech: M.Mechanism) -> str:
    out = []
    out.append("static __device__ __forceinline__ void thermo_cph(const double T, double* __restrict__ cpR, "
               "double* __restrict__ hRT) {")
    out.append("  const double T2 = T * T, T3 = T2 * T, T4 = T3 * T, iT = 1.0 / T;")
    for tmid, ks in _thermo_groups(mech).items():
        out.append(f"  {{ const bool lo = T < {_d(tmid)};")
        for k in ks:
            s = mech.species[k]
            a = [f"(lo ? {_d(s.low[i])} : {_d(s.high[i])})" for i in range(7)]
            out.append(f"    {{ const double a0 = {a[0]}, a1 = {a[1]}, a2 = {a[2]}, a3 = {a[3]}, a4 = {a[4]}, a5 = {a[5]};")
            out.append(f"      cpR[{k}] = a0 + a1 * T + a2 * T2 + a3 * T3 + a4 * T4;")
            out.append(f"      hRT[{k}] = a0 + 0.5 * a1 * T + (1.0 / 3.0) * a2 * T2 + 0.25 * a3 * T3 + 0.2 * a4 * T4 + a5 * iT; }}")
        out.append("  }")
    out.append("}")
    out.append("")
    out.append("static __device__ __forceinline__ void thermo_dcp(const double T, double* __restrict__ dcpR) {")
    out.append("  const double T2 = T * T, T3 = T2 * T;")
    for tmid, ks in _thermo_groups(mech).items():
        out.append(f"  {{ const bool lo = T < {_d(tmid)};")
        for k in ks:
            s_ = mech.species[k]
            a = [f"(lo ? {_d(s_.low[i])} : {_d(s_.high[i])})" for i in range(5)]
            out.append(f"    dcpR[{k}] = {a[1]} + 2.0 * {a[2]} * T + 3.0 * {a[3]} * T2 + 4.0 * {a[4]} * T3;")
        out.append("  }")
    out.append("}")
    out.append("")
    out.append("static __device__ __forceinline__ void gibbs(const double T, const double logT, double* __restrict__ gRT) {")
    out.append("  const double T2 = T * T, T3 = T2 * T, T4 = T3 * T, iT = 1.0 / T;")
    for tmid, ks in _thermo_groups(mech).items():
        out.append(f"  {{ const bool lo = T < {_d(tmid)};")
        for k in ks:
            s = mech.species[k]
            a = [f"(lo ? {_d(s.low[i])} : {_d(s.high[i])})" for i in range(7)]
            out.append(f"    {{ const double a0 = {a[0]}, a1 = {a[1]}, a2 = {a[2]}, a3 = {a[3]}, a4 = {a[4]}, a5 = {a[5]}, a6 = {a[6]};")
            # g/RT = h/RT - s/R
            out.append(f"      gRT[{k}] = a0 * (1.0 - logT) - 0.5 * a1 * T - (1.0 / 6.0) * a2 * T2 - (1.0 / 12.0) * a3 * T3"
                       f" - 0.05 * a4 * T4 + a5 * iT - a6; }}")
        out.append("  }")
    out.append("}")
    return "\n".join(out)


def _element_shift(mech: M.Mechanism) -> list:
    """(d5, d6) per species: what to add to the NASA coefficients a5 and a6 so that g/RT
    loses sum_e n_ke (alpha_e + beta_e / T).  A reaction that conserves its elements does
    not see it, while exp(g/RT) of every species, and the product over either side of a
    reaction, stays within the range of a double down to the cold end that ``shared_range``
    finds (105 to 210 K).  alpha and beta are the least-squares fit of g/RT over
    200 - 4000 K, rounded (1, and 10 K).  A reaction that does not conserve them (the loader
    refuses such a mechanism) leaves g/RT as it is; ``shared_range`` goes by the shift in use."""
    els = list(mech.elements)
    for r in mech.reactions:
        for e in els:
            n = sum(c * mech.species[i].composition.get(e, 0) for i, c in r.products.items()) - \
                sum(c * mech.species[i].composition.get(e, 0) for i, c in r.reactants.items())
            if n != 0:
                return [(0.0, 0.0)] * mech.nspec
    rows, rhs = [], []
    for s in mech.species:
        for T in (200.0, 250.0, 300.0, 400.0, 600.0, 1000.0, 1500.0, 2500.0, 4000.0):
            a = s.low if T < s.T[1] else s.high
            n = [s.composition.get(e, 0) for e in els]
            rows.append(n + [x * 1000.0 / T for x in n])
            rhs.append(a[0] * (1.0 - math.log(T)) - a[1] * T / 2 - a[2] * T ** 2 / 6 - a[3] * T ** 3 / 12
                       - a[4] * T ** 4 / 20 + a[5] / T - a[6])
    x = np.linalg.lstsq(np.array(rows), np.array(rhs), rcond=None)[0]
    alpha = [float(round(v)) for v in x[:len(els)]]
    beta = [10.0 * round(100.0 * v) for v in x[len(els):]]
    return [(-sum(b * s.composition.get(e, 0) for e, b in zip(els, beta)),
             sum(v * s.composition.get(e, 0) for e, v in zip(els, alpha))) for s in mech.species]


# Up to this many species the coefficients are literals in the code, chosen by selects: a
# launch on a few cells waits for each line of a table in turn (LiDryer's rates of 1,000
# cells 9.4 us with tables, 7.6 with literals), and nine species' selects cost little.
LITERAL_SPECIES = 16


def gen_tables(mech: M.Mechanism) -> str:
    """The constant-memory tables (none up to LITERAL_SPECIES species), [range][species][8]: NASA coefficients over the
    molecular weight (mixture sums), as they are (per species), and g/RT's (a0, a1/2,
    a2/6, a3/12, a4/20, a5, a6, shifted)."""
    cn = _cname(mech.name)
    if mech.nspec <= LITERAL_SPECIES:
        return ""
    out = []
    for name in ("mass", "nasa", "gibbs"):
        out.append(f"static __constant__ double {cn}_{name}[2][{mech.nspec}][8] = {{")
        for side in _table_rows(mech, name):
            out.append(" {")
            out += ["  {" + ", ".join(_d(v) for v in row) + "}," for row in side]
            out.append(" },")
        out.append("};")
    return "\n".join(out)


# The shared form (gen_wdot_shared) multiplies exponentials that a reaction's own difference
# would have cancelled, so it stands only where every product of them, partial ones
# included, is within exp(+-SHARED_LIMIT): what is left of a double's exp(+-709) is for the
# concentrations, whose products may then be as small as 1e-60 (1e-138 at 298 K in the
# mechanism that needs most).  A lower limit moves the line up into temperatures that
# forced cells reach: at 480 (250 K for the 56-species mechanism) a box of 33 x 31 x 29 such
# cells took 29 ms in k_eval against 11, the few cold lanes making their waves take both
# forms.
SHARED_LIMIT = 570.0


def shared_range(mech: M.Mechanism) -> tuple:
    """(low, high): the temperatures between which the shared form's exponentials and
    their products stay within SHARED_LIMIT, on a grid of 5 K below 3500 K and 100 K above,
    at most 20000 K.  Outside, the rates take one exponential per reaction."""
    shift = _element_shift(mech)

    def holds(T):
        logT = math.log(T)
        g = []
        for s, (d5, d6) in zip(mech.species, shift):
            a = s.low if T < s.T[1] else s.high
            g.append(a[0] * (1.0 - logT) - a[1] * T / 2 - a[2] * T ** 2 / 6 - a[3] * T ** 3 / 12 - a[4] * T ** 4 / 20
                     + (a[5] + d5) / T - (a[6] + d6))
        for r in mech.reactions:
            if abs(r.beta * logT - r.Ea / M.R_CAL / T) > SHARED_LIMIT:
                return False
            for side in (r.reactants, r.products):
                t = 0.0
                for i, c in sorted(side.items()):
                    for _ in range(c):
                        t += g[i]
                        if abs(t) > SHARED_LIMIT:
                            return False
        return all(abs(x) <= SHARED_LIMIT for x in g)

    low, high = 3500.0, 3500.0
    while low > 5.0 and holds(low - 5.0):
        low -= 5.0
    while high < 20000.0 and holds(high + 100.0):
        high += 100.0
    return low, high


def gen_reaction_tables(mech: M.Mechanism) -> str:
    """The reactions as tables, for the rates and Jacobian outside the shared form's range.
    Integers: kind (0 elementary, 1 three-body, 2 Lindemann, 3 Troe), reversible, first and
    last + 1 of the efficiencies, then the species of either side, each as often as its
    coefficient, -1 beyond; the species whose coefficients differ between the sides, -1
    beyond, and by how much.  Numbers: f, x, b, Ta of the rate constant f exp(x + b ln T -
    Ta / T) and of the low-pressure one, then Fcent = c3 exp(-T/T3) + c1 exp(-T/T1) + c2
    exp(-T2/T) as (c3, -1/T3, c1, -1/T1, c2, T2).  Efficiencies: species, and e - 1."""
    cn = _cname(mech.name)
    width = max(sum(s.values()) for r in mech.reactions for s in (r.reactants, r.products))
    ints, nums, eff_k, eff_e = [], [], [], []

    def arrhenius(A, b, Ea):   # a constant is kept as it is, as _kf_expr writes it
        return [A, 0.0, 0.0, 0.0] if b == 0.0 and Ea == 0.0 else [1.0, math.log(A), b, Ea / M.R_CAL]

    for r in mech.reactions:
        first = len(eff_k)
        if r.has_third_body:
            for k, e in sorted(r.efficiencies.items()):
                if e != 1.0:
                    eff_k.append(k)
                    eff_e.append(e - 1.0)
        kind = {"elementary": 0, "three-body": 1, "falloff": 2 if r.troe is None else 3}[r.kind]
        row = [kind, int(r.reversible), first, len(eff_k)]
        for side in (r.reactants, r.products):
            ks = [i for i, c in sorted(side.items()) for _ in range(c)]
            row += ks + [-1] * (width - len(ks))
        net = {k: r.products.get(k, 0) - r.reactants.get(k, 0) for k in sorted({**r.reactants, **r.products})}
        net = [(k, v) for k, v in net.items() if v != 0]
        for j in (0, 1):
            row += [kv[j] for kv in net] + [-1] * (2 * width - len(net))
        ints.append(row)
        f = [0.0] * 6
        if r.troe is not None:
            a, T3, T1 = r.troe[:3]
            if T3 > 1e-20:
                f[0], f[1] = 1.0 - a, -1.0 / T3
            f[2], f[3] = a, (0.0 if T1 >= 1e20 else -1.0 / T1)
            if len(r.troe) == 4:
                f[4], f[5] = 1.0, r.troe[3]
        nums.append(arrhenius(r.A, r.beta, r.Ea) + arrhenius(*(r.low or (1.0, 0.0, 0.0))) + f)
    out = [f"static __constant__ int {cn}_rx_int[{mech.nreac}][{4 + 6 * width}] = {{"]
    out += ["  {" + ", ".join(str(v) for v in row) + "}," for row in ints]
    out.append("};")
    out.append(f"static __constant__ double {cn}_rx_num[{mech.nreac}][14] = {{")
    out += ["  {" + ", ".join(_d(v) for v in row) + "}," for row in nums]
    out.append("};")
    out.append(f"static __constant__ int {cn}_eff_k[] = {{" + ", ".join(str(k) for k in eff_k or [0]) + "};")
    out.append(f"static __constant__ double {cn}_eff_e[] = {{" + ", ".join(_d(e) for e in eff_e or [0.0]) + "};")
    return "\n".join(out)


def gen_reaction_access(mech: M.Mechanism) -> str:
    cn = _cname(mech.name)
    width = max(sum(s.values()) for r in mech.reactions for s in (r.reactants, r.products))
    low, high = shared_range(mech)
    return "\n".join([
        "// temperatures between which wdot and jacobian hold; outside, the reaction tables",
        f"static constexpr double T_LOW = {_d(low)}, T_HIGH = {_d(high)};",
        f"static constexpr int RX_SIDE = {width};",
        f"static __device__ __forceinline__ const int* rx_int(int j) {{ return {cn}_rx_int[j]; }}",
        f"static __device__ __forceinline__ const double* rx_num(int j) {{ return {cn}_rx_num[j]; }}",
        f"static __device__ __forceinline__ int eff_k(int e) {{ return {cn}_eff_k[e]; }}",
        f"static __device__ __forceinline__ double eff_e(int e) {{ return {cn}_eff_e[e]; }}"])


def _table_rows(mech: M.Mechanism, name: str) -> list:
    """[range][species] -> 8 values."""
    shift = _element_shift(mech) if name == "gibbs" else None

    def row(k, s, a):
        if name == "mass":
            return [a[i] / mech.W[k] for i in range(6)] + [0.0, 0.0]
        if name == "nasa":
            return [a[i] for i in range(7)] + [0.0]
        return [a[0], a[1] / 2.0, a[2] / 6.0, a[3] / 12.0, a[4] / 20.0, a[5] + shift[k][0], a[6] + shift[k][1], 0.0]

    return [[row(k, s, s.low if side == 0 else s.high) for k, s in enumerate(mech.species)] for side in (0, 1)]


def gen_thermo_tables(mech: M.Mechanism) -> str:
    cn = _cname(mech.name)
    groups = list(_thermo_groups(mech).items())
    literal = mech.nspec <= LITERAL_SPECIES
    out = []

    def sided(table, body):
        # body(k, t) for every species; t(i) is coefficient i of its row
        if literal:
            rows = _table_rows(mech, table)
            out.append("  const bool up[] = {" + ", ".join(f"((range >> {g}) & 1u) != 0u" for g in range(len(groups))) + "};")
            for g, (tmid, ks) in enumerate(groups):
                for k in ks:
                    out.append("  " + body(k, lambda i: f"(up[{g}] ? {_d(rows[1][k][i])} : {_d(rows[0][k][i])})", ""))
            return
        for g, (tmid, ks) in enumerate(groups):
            out.append("#pragma unroll 1")
            out.append(f"  for (int r = 0; r < 2; ++r) if ((int)((range >> {g}) & 1u) == r) {{")
            # inside the branch the compiler knows r to be the lane's own bit: keep it scalar
            out.append("    const int u = PELE_UNIFORM(r);")
            for k in ks:
                out.append("    " + body(k, lambda i: f"t[{i}]", f"const double* t = {cn}_{table}[u][{k}]; "))
            out.append("  }")

    out.append("// one bit per break temperature: T in its upper range")
    out.append("static __device__ __forceinline__ unsigned range(const double T) {")
    out.append("  return " + " | ".join(f"(T < {_d(t)} ? 0u : {1 << g}u)" for g, (t, _) in enumerate(groups)) + ";")
    out.append("}")
    out.append("// A[j] = sum_k w_k a_jk / W_k, j = 0..5")
    out.append("static __device__ __forceinline__ void mix(const unsigned range, const double* __restrict__ w, "
               "double* __restrict__ A) {")
    out.append("  for (int j = 0; j < 6; ++j) A[j] = 0.0;")
    sided("mass", lambda k, t, row: "{ " + row + " ".join(f"A[{j}] += w[{k}] * {t(j)};" for j in range(6)) + " }")
    out.append("}")
    out.append("static __device__ __forceinline__ void thermo_cph(const double T, double* __restrict__ cpR, "
               "double* __restrict__ hRT) {")
    out.append("  const double iT = 1.0 / T;")
    out.append("  const unsigned range = mech_" + cn + "::range(T);")
    sided("nasa", lambda k, t, row: f"{{ {row}"
          f"const double a0 = {t(0)}, a1 = {t(1)}, a2 = {t(2)}, a3 = {t(3)}, a4 = {t(4)};"
          f" cpR[{k}] = a0 + T * (a1 + T * (a2 + T * (a3 + T * a4)));"
          f" hRT[{k}] = a0 + T * (0.5 * a1 + T * ((1.0 / 3.0) * a2 + T * (0.25 * a3 + T * (0.2 * a4)))) + {t(5)} * iT; }}")
    out.append("}")
    out.append("static __device__ __forceinline__ void thermo_dcp(const double T, double* __restrict__ dcpR) {")
    out.append("  const unsigned range = mech_" + cn + "::range(T);")
    sided("nasa", lambda k, t, row: f"{{ {row}"
          f"dcpR[{k}] = {t(1)} + T * (2.0 * {t(2)} + T * (3.0 * {t(3)} + T * (4.0 * {t(4)}))); }}")
    out.append("}")
    out.append("static __device__ __forceinline__ void gibbs(const double T, const double logT, double* __restrict__ gRT) {")
    out.append("  const double iT = 1.0 / T, l1 = 1.0 - logT;")
    out.append("  const unsigned range = mech_" + cn + "::range(T);")
    sided("gibbs", lambda k, t, row: f"{{ {row}"
          f"gRT[{k}] = {t(0)} * l1 - T * ({t(1)} + T * ({t(2)} + T * ({t(3)} + T * {t(4)}))) + {t(5)} * iT - {t(6)}; }}")
    out.append("}")
    return "\n".join(out)


def _kf_expr(A: float, b: float, Ta: float) -> str:
    if b == 0.0 and Ta == 0.0:
        return _d(A)
    parts = [_d(math.log(A))]
    if b != 0.0:
        parts.append(f"{_d(b)} * logT")
    if Ta != 0.0:
        parts.append(f"{_d(-Ta)} * invT")
    return f"exp({' + '.join(parts)})"


def _dlnk_expr(b: float, Ta: float) -> str:
    # d ln(A T^b exp(-Ta/T)) / dT = (b + Ta/T) / T
    if b == 0.0 and Ta == 0.0:
        return "0.0"
    if Ta == 0.0:
        return f"{_d(b)} * invT"
    if b == 0.0:
        return f"{_d(Ta)} * invT * invT"
    return f"({_d(b)} + {_d(Ta)} * invT) * invT"


def _mc_expr(r: M.Reaction, ns: int) -> str:
    terms = ["Ctot"]
    for k in range(ns):
        e = r.efficiencies.get(k, 1.0)
        if e != 1.0:
            terms.append(f"{_d(e - 1.0)} * C[{k}]")
    return " + ".join(terms)


def _troe_fc(r: M.Reaction) -> tuple[str, str]:
    """Fcent and dFcent/dT expressions with constant folding of the 1e-30 / 1e30 forms."""
    a = r.troe[0]
    T3, T1 = r.troe[1], r.troe[2]
    fc, dfc = [], []
    if (1.0 - a) != 0.0 and T3 > 1e-20:
        fc.append(f"{_d(1.0 - a)} * exp({_d(-1.0 / T3)} * T)")
        dfc.append(f"{_d(-(1.0 - a) / T3)} * exp({_d(-1.0 / T3)} * T)")
    if a != 0.0:
        if T1 >= 1e20:
            fc.append(_d(a))
        else:
            fc.append(f"{_d(a)} * exp({_d(-1.0 / T1)} * T)")
            dfc.append(f"{_d(-a / T1)} * exp({_d(-1.0 / T1)} * T)")
    if len(r.troe) == 4:
        T2 = r.troe[3]
        fc.append(f"exp({_d(-T2)} * invT)")
        dfc.append(f"{_d(T2)} * invT * invT * exp({_d(-T2)} * invT)")
    return (" + ".join(fc) or "0.0"), (" + ".join(dfc) or "0.0")


def _kc_exprs(r: M.Reaction) -> tuple[str, str, int]:
    """Sum of nu g/RT (products minus reactants), the same for h/RT, and sum nu."""
    def side(arr: str) -> str:
        out = ""
        for i, c in sorted(r.products.items()):
            t = f"{_d(c)} * {arr}[{i}]" if c != 1 else f"{arr}[{i}]"
            out += t if not out else f" + {t}"
        for i, c in sorted(r.reactants.items()):
            t = f"{_d(c)} * {arr}[{i}]" if c != 1 else f"{arr}[{i}]"
            out += f" - {t}"
        return out
    dnu = sum(r.products.values()) - sum(r.reactants.values())
    return side("gRT"), side("hRT"), dnu


def _refc_factor(dnu: int) -> str:
    # (P_atm / RT)^(-dnu) = (RT/P_atm)^dnu = refCinv^dnu
    if dnu == 0:
        return ""
    if dnu > 0:
        return " * " + " * ".join(["refCinv"] * dnu)
    return " * " + " * ".join(["refC"] * (-dnu))


def gen_wdot(mech: M.Mechanism) -> str:
    ns = mech.nspec
    out = []
    out.append("static __device__ __forceinline__ void wdot(const double* __restrict__ C, const double T, const double logT, "
               "const double invT, const double* __restrict__ gRT, double* __restrict__ wd) {")
    out.append(f"  for (int k = 0; k < {ns}; ++k) wd[k] = 0.0;")
    out.append(f"  const double refC = {_d(M.P_ATM / M.R_CGS)} * invT, refCinv = 1.0 / refC;")
    if any(r.has_third_body for r in mech.reactions):
        out.append("  double Ctot = 0.0;")
        out.append(f"  for (int k = 0; k < {ns}; ++k) Ctot += C[k];")
    for j, r in enumerate(mech.reactions):
        out.append(f"  {{ // {j}: {r.equation}")
        out.append(f"    const double kf = {_kf_expr(r.A, r.beta, r.Ea / M.R_CAL)};")
        if r.kind == "elementary":
            out.append("    const double keff = kf;")
        elif r.kind == "three-body":
            out.append(f"    const double keff = kf * ({_mc_expr(r, ns)});")
        else:
            A0, b0, E0 = r.low
            out.append(f"    const double k0 = {_kf_expr(A0, b0, E0 / M.R_CAL)};")
            out.append(f"    const double Pr = k0 * ({_mc_expr(r, ns)}) / kf;")
            if r.troe is not None:
                fc, _ = _troe_fc(r)
                out.append(f"    const double logFc = log10(fmax({fc}, 1e-300));")
                out.append("    const double cc = -0.4 - 0.67 * logFc, nn = 0.75 - 1.27 * logFc;")
                out.append("    const double u = log10(fmax(Pr, 1e-300)) + cc;")
                out.append("    const double f1 = u / (nn - 0.14 * u);")
                out.append("    const double F = exp(2.302585092994045684 * logFc / (1.0 + f1 * f1));")
                out.append("    const double keff = kf * Pr / (1.0 + Pr) * F;")
            else:
                out.append("    const double keff = kf * Pr / (1.0 + Pr);")
        pf = _prod(_power_terms(r.reactants))
        if r.reversible:
            gs, _, dnu = _kc_exprs(r)
            pr = _prod(_power_terms(r.products))
            out.append(f"    const double q = keff * ({pf} - {pr} * exp({gs}){_refc_factor(dnu)});")
        else:
            out.append(f"    const double q = keff * ({pf});")
        for i, c in sorted(r.reactants.items()):
            out.append(f"    wd[{i}] -= {_d(c) + ' * ' if c != 1 else ''}q;")
        for i, c in sorted(r.products.items()):
            out.append(f"    wd[{i}] += {_d(c) + ' * ' if c != 1 else ''}q;")
        out.append("  }")
    out.append("}")
    return "\n".join(out)


def _exponent(b: float, Ta: float) -> str:
    return " + ".join(([f"{_d(b)} * logT"] if b != 0.0 else []) + ([f"{_d(-Ta)} * invT"] if Ta != 0.0 else []))


def _rate_groups(mech: M.Mechanism) -> list:
    """Reactions grouped by the (b, Ta) of their rate constant, third-body ones first
    (they read the concentrations, the others only C exp(g/RT)); the group (0, 0) needs no
    exponential."""
    groups: dict = {}
    for j, r in enumerate(mech.reactions):
        groups.setdefault((not r.has_third_body, r.beta, r.Ea), []).append(j)
    return sorted(((k[1], k[2], js) for k, js in groups.items()),
                  key=lambda g: (not mech.reactions[g[2][0]].has_third_body, g[2][0]))


def _species_exps(mech: M.Mechanism) -> list:
    return ["  double E[NS], I[NS];   // exp(g/RT) and its reciprocal",
            "#pragma unroll",
            "  for (int k = 0; k < NS; ++k) { E[k] = exp(gRT[k]); I[k] = 1.0 / E[k]; }"]


def gen_wdot_shared(mech: M.Mechanism) -> str:
    """The production rates with every transcendental evaluated once.  With X_k = C_k
    exp(g_k/RT), a reaction's net rate is kf prod_f exp(-g/RT) (prod_f X - prod_r X
    (P_atm/RT)^-dnu)."""
    ns = mech.nspec
    out = []
    out.append("static __device__ __forceinline__ void wdot(const double* __restrict__ C, const double T, const double logT, "
               "const double invT, const double* __restrict__ gRT, double* __restrict__ wd) {")
    out.append(f"  const double refC = {_d(M.P_ATM / M.R_CGS)} * invT, refCinv = 1.0 / refC;")
    out += _species_exps(mech)
    out.append("  double X[NS];")
    out.append("#pragma unroll")
    out.append("  for (int k = 0; k < NS; ++k) { X[k] = C[k] * E[k]; wd[k] = 0.0; }")
    if any(r.has_third_body for r in mech.reactions):
        out.append("  double Ctot = 0.0;")
        out.append("#pragma unroll")
        out.append("  for (int k = 0; k < NS; ++k) Ctot += C[k];")

    def xs(side):
        return _prod([t for i, c in sorted(side.items()) for t in [f"X[{i}]"] * c])

    for b, Ea, js in _rate_groups(mech):
        x = _exponent(b, Ea / M.R_CAL)
        if x:
            out.append(f"  {{ const double x = exp({x});")
        else:
            out.append("  {")
        for j in js:
            r = mech.reactions[j]
            out.append(f"  {{ // {j}: {r.equation}")
            out.append(f"    const double kf = {_d(r.A)}{' * x' if x else ''};")
            if r.kind == "elementary":
                out.append("    const double keff = kf;")
            elif r.kind == "three-body":
                out.append(f"    const double keff = kf * ({_mc_expr(r, ns)});")
            else:
                A0, b0, E0 = r.low
                out.append(f"    const double k0 = {_kf_expr(A0, b0, E0 / M.R_CAL)};")
                out.append(f"    const double Pr = k0 * ({_mc_expr(r, ns)}) / kf;")
                if r.troe is not None:
                    fc, _ = _troe_fc(r)
                    out.append(f"    const double logFc = log10(fmax({fc}, 1e-300));")
                    out.append("    const double cc = -0.4 - 0.67 * logFc, nn = 0.75 - 1.27 * logFc;")
                    out.append("    const double u = log10(fmax(Pr, 1e-300)) + cc;")
                    out.append("    const double f1 = u / (nn - 0.14 * u);")
                    out.append("    const double F = exp(2.302585092994045684 * logFc / (1.0 + f1 * f1));")
                    out.append("    const double keff = kf * Pr / (1.0 + Pr) * F;")
                else:
                    out.append("    const double keff = kf * Pr / (1.0 + Pr);")
            back = ""
            if r.reversible:
                dnu = sum(r.products.values()) - sum(r.reactants.values())
                back = f" - {xs(r.products)}{_refc_factor(dnu)}"
            inv = "".join(f" * I[{i}]" * c for i, c in sorted(r.reactants.items()))
            out.append(f"    const double q = keff{inv} * ({xs(r.reactants)}{back});")
            for i, c in sorted(r.reactants.items()):
                out.append(f"    wd[{i}] -= {_d(c) + ' * ' if c != 1 else ''}q;")
            for i, c in sorted(r.products.items()):
                out.append(f"    wd[{i}] += {_d(c) + ' * ' if c != 1 else ''}q;")
            out.append("  }")
        out.append("  }")
    out.append("}")
    return "\n".join(out)


def gen_jacobian(mech: M.Mechanism, shared: bool = True) -> str:
    """Derivatives of f_i = W_i wdot_i with respect to rhoY_k (=W_k C_k) and T.

    Two phases, so that no Jacobian entry is accumulated in memory (a read-modify-
    write chain whose latency would dominate): per reaction j the rate of progress q_j,
    its T derivative and every distinct dq_j/dC_k go to write-once private arrays; then
    wd and dwdT are formed species by species, and the entries column by column (k
    ascending, rows i ascending, structural zeros included), each sum over reactions in
    reaction order.  acc(i, k, v) receives each entry v = sum_j W_i/W_k nu_ij dq_j/dC_k
    exactly once, and colend(k) follows the last row of column k.  dwdT is the molar
    dwdot/dT and wd the molar production rates at the same state.  shared: with every
    transcendental evaluated once, as in ``gen_wdot_shared``.
    """
    ns = mech.nspec
    nr = mech.nreac
    W = mech.W
    out = []
    body = []
    nu_all = []          # per reaction: {species: net stoichiometric coefficient}
    entries: dict = {}   # (i, k) -> [(coefficient, D index)] in reaction order
    nd = 0
    if any(r.has_third_body for r in mech.reactions):
        body.append("  double Ctot = 0.0;")
        body.append(f"  for (int k = 0; k < {ns}; ++k) Ctot += C[k];")
    blocks = []          # per reaction: its lines
    for j, r in enumerate(mech.reactions):
        head, body = body, []
        blocks.append(body)
        if j == 0:
            first = head
        body.append(f"  {{ // {j}: {r.equation}")
        if shared:
            body.append(f"    const double kf = {_d(r.A)}{' * x' if r.beta != 0.0 or r.Ea != 0.0 else ''};")
        else:
            body.append(f"    const double kf = {_kf_expr(r.A, r.beta, r.Ea / M.R_CAL)};")
        body.append(f"    const double dlnkf = {_dlnk_expr(r.beta, r.Ea / M.R_CAL)};")
        if r.kind == "elementary":
            body.append("    const double keff = kf, dkeffdT = kf * dlnkf;")
        elif r.kind == "three-body":
            body.append(f"    const double Mc = {_mc_expr(r, ns)};")
            body.append("    const double keff = kf * Mc, dkeffdT = keff * dlnkf, dkeffdM = kf;")
        else:
            A0, b0, E0 = r.low
            body.append(f"    const double Mc = {_mc_expr(r, ns)};")
            body.append(f"    const double k0 = {_kf_expr(A0, b0, E0 / M.R_CAL)};")
            body.append(f"    const double dlnk0 = {_dlnk_expr(b0, E0 / M.R_CAL)};")
            body.append("    const double Pr = k0 * Mc / kf, dPrdM = k0 / kf, dPrdT = Pr * (dlnk0 - dlnkf);")
            if r.troe is not None:
                fc, dfc = _troe_fc(r)
                body.append(f"    double Fc = {fc}, dFc = {dfc};")
                body.append("    if (Fc < 1e-300) { Fc = 1e-300; dFc = 0.0; }")
                body.append("    const double logFc = log10(Fc);")
                body.append("    const double cc = -0.4 - 0.67 * logFc, nn = 0.75 - 1.27 * logFc;")
                body.append("    const double PrS = fmax(Pr, 1e-300);")
                body.append("    const double u = log10(PrS) + cc, dd = nn - 0.14 * u, f1 = u / dd, den = 1.0 + f1 * f1;")
                body.append("    const double F = exp(2.302585092994045684 * logFc / den);")
                body.append("    const double df1du = nn / (dd * dd), df1dl = (-0.67 * dd + 1.1762 * u) / (dd * dd);")
                body.append("    const double dlFdlPr = -logFc * 2.0 * f1 / (den * den) * df1du;")
                body.append("    const double dlFdlFc = 1.0 / den - logFc * 2.0 * f1 / (den * den) * df1dl;")
                body.append("    const double dFdPr = F * dlFdlPr / PrS, dFdT = F * dlFdlFc * dFc / Fc;")
            else:
                body.append("    const double F = 1.0, dFdPr = 0.0, dFdT = 0.0;")
            body.append("    const double gg = Pr / (1.0 + Pr), dg = 1.0 / ((1.0 + Pr) * (1.0 + Pr));")
            body.append("    const double keff = kf * gg * F;")
            body.append("    const double dkeffdM = kf * (dg * F + gg * dFdPr) * dPrdM;")
            body.append("    const double dkeffdT = keff * dlnkf + kf * (dg * F + gg * dFdPr) * dPrdT + kf * gg * dFdT;")
        pf = _prod(_power_terms(r.reactants))
        body.append(f"    const double pf = {pf};")
        if r.reversible:
            gs, hs, dnu = _kc_exprs(r)
            pr = _prod(_power_terms(r.products))
            body.append(f"    const double pr = {pr};")
            if shared:
                gs = " * ".join([f"E[{i}]" for i, c in sorted(r.products.items()) for _ in range(c)]
                                + [f"I[{i}]" for i, c in sorted(r.reactants.items()) for _ in range(c)])
                body.append(f"    const double invKc = {gs}{_refc_factor(dnu)};")
            else:
                body.append(f"    const double invKc = exp({gs}){_refc_factor(dnu)};")
            body.append(f"    const double dlnKc = ({hs} - {_d(dnu)}) * invT;")
            body.append("    const double net = pf - pr * invKc;")
            body.append("    const double dqdT = dkeffdT * net + keff * pr * invKc * dlnKc;")
        else:
            body.append("    const double net = pf;")
            body.append("    const double dqdT = dkeffdT * net;")
        body.append(f"    Q[{j}] = keff * net; QT[{j}] = dqdT;")
        nu: dict = {}
        for i, c in r.reactants.items():
            nu[i] = nu.get(i, 0) - c
        for i, c in r.products.items():
            nu[i] = nu.get(i, 0) + c
        nu = {i: v for i, v in nu.items() if v != 0}
        nu_all.append(nu)
        # dq/dC_k from the mass-action products
        dq: dict = {}
        for k in sorted(r.reactants):
            coef, terms = _dpower_terms(r.reactants, k)
            e = f"{_d(coef)} * {_prod(terms)}" if coef != 1.0 else _prod(terms)
            dq.setdefault(k, []).append(f"keff * {e}")
        if r.reversible:
            for k in sorted(r.products):
                coef, terms = _dpower_terms(r.products, k)
                e = f"{_d(coef)} * {_prod(terms)}" if coef != 1.0 else _prod(terms)
                dq.setdefault(k, []).append(f"- keff * invKc * {e}")
        if r.has_third_body:
            body.append("    const double tb = dkeffdM * net;")
            for k in range(ns):
                e = r.efficiencies.get(k, 1.0)
                if e != 0.0:
                    dq.setdefault(k, []).append(f"{_d(e)} * tb" if e != 1.0 else "tb")
        for k in sorted(dq):
            expr = " + ".join(dq[k]).replace("+ -", "-")
            body.append(f"    D[{nd}] = {expr};")
            for i, v in sorted(nu.items()):
                entries.setdefault((i, k), []).append((v * W[i] / W[k], nd))
            nd += 1
        body.append("  }")
    out.append("template <class Acc, class ColEnd>")
    out.append("static __device__ __forceinline__ void jacobian(const double* __restrict__ C, const double T, const double logT, "
               "const double invT, const double* __restrict__ gRT, const double* __restrict__ hRT, "
               "double* __restrict__ wd, double* __restrict__ dwdT, Acc&& acc, ColEnd&& colend) {")
    out.append(f"  const double refC = {_d(M.P_ATM / M.R_CGS)} * invT, refCinv = 1.0 / refC;")
    out.append(f"  double Q[{nr}], QT[{nr}], D[{max(nd, 1)}];")
    if not shared:
        out += first
        for b in blocks:
            out += b
    else:
        out += _species_exps(mech)
        out += first
        for b, Ea, js in _rate_groups(mech):
            x = _exponent(b, Ea / M.R_CAL)
            out.append(f"  {{ const double x = exp({x});" if x else "  {")
            for j in js:
                out += blocks[j]
            out.append("  }")
    # production rates and their T derivatives, species by species
    for i in range(ns):
        terms = [(nu_all[j][i], j) for j in range(nr) if i in nu_all[j]]
        if not terms:
            out.append(f"  wd[{i}] = 0.0; dwdT[{i}] = 0.0;")
            continue
        v, j = terms[0]
        out.append(f"  {{ double s = {_d(v)} * Q[{j}], t = {_d(v)} * QT[{j}];")
        for v, j in terms[1:]:
            out.append(f"    s += {_d(v)} * Q[{j}]; t += {_d(v)} * QT[{j}];")
        out.append(f"    wd[{i}] = s; dwdT[{i}] = t; }}")
    # Jacobian entries, column by column
    for k in range(ns):
        for i in range(ns):
            terms = entries.get((i, k))
            if not terms:
                out.append(f"  acc({i}, {k}, 0.0);")
                continue
            c, m = terms[0]
            out.append(f"  {{ double s = {_d(c)} * D[{m}];")
            for c, m in terms[1:]:
                out.append(f"    s += {_d(c)} * D[{m}];")
            out.append(f"    acc({i}, {k}, s); }}")
        out.append(f"  colend({k});")
    out.append("}")
    return "\n".join(out)


_TRANS = ("exp", "log10", "log", "pow", "sqrt")


def count_ops(code: str) -> dict:
    """Static operation count of generated straight-line code: every binary + - * /
    as written counts one flop (so a fused multiply-add counts two), fmax/fmin one, and
    exp / log / log10 / pow / sqrt are counted separately as transcendentals.  Loops in
    the generated code are the fixed per-species ones ("for (int k = 0; k < NS; ...)"),
    whose single-statement bodies are weighted by NS."""
    flops = 0
    trans = {t: 0 for t in _TRANS}
    ns = None
    for line in code.splitlines():
        line = line.split("//")[0]
        m = re.search(r"for \(int k = 0; k < (\d+); \+\+k\)(.*)", line)
        weight = 1
        if m:
            weight = int(m.group(1))
            line = m.group(2)
        # drop the ternary coefficient selects of the NASA polynomials
        line = re.sub(r"\(lo \? [^:]+ : [^)]+\)", "a", line)
        for t in _TRANS:
            n = len(re.findall(r"\b%s\(" % t, line))
            trans[t] += n * weight
        n = len(re.findall(r"\bfm(ax|in)\(", line))
        # binary operators: + * / anywhere; - when it follows an operand
        ops = len(re.findall(r"(?<=[\w\)\]\s])\s*[\+\*/](?!=)", line))
        ops += len(re.findall(r"(?<=[\w\)\]])\s+-\s+", line))
        ops += len(re.findall(r"[\+\-\*/]=", line))
        flops += (ops + n) * weight
    del ns
    return {"flops": flops, "transcendentals": sum(trans.values()), "by_function": trans}


def emitted_counts(mech: M.Mechanism) -> dict:
    """Operation counts of the emitted code, for one side of the fits' break temperature:
    ``mix`` (the mixture's coefficients), ``gibbs``, ``wdot`` and ``jacobian``."""
    ns = mech.nspec
    loops = re.compile(r"k < NS; \+\+k\) \{ (.*) \}$")

    def flat(code):   # loops over the species as count_ops knows them, a statement a line
        out = []
        for line in code.splitlines():
            m = loops.search(line)
            out += [f"for (int k = 0; k < {ns}; ++k) {t};" for t in m.group(1).split("; ")] if m else \
                [line.replace("k < NS;", f"k < {ns};")]
        return "\n".join(out)

    thermo = {}
    for part in gen_thermo(mech).split("static __device__ __forceinline__ void ")[1:]:
        thermo[part.split("(")[0]] = count_ops(part)
    return {"mix": {"flops": 12 * ns, "transcendentals": 0}, "gibbs": thermo["gibbs"],
            "wdot": count_ops(flat(gen_wdot_shared(mech))), "jacobian": count_ops(flat(gen_jacobian(mech)))}


def write_inc(mech: M.Mechanism, path: str) -> None:
    ns = mech.nspec
    name = mech.name
    cn = _cname(name)
    lines = [f"// GENERATED by pelelm_amd/mechanisms/hipgen.py from {name}.yaml -- do not edit.",
             f"// {ns} species, {mech.nreac} reactions.", "#pragma once", "",
             gen_tables(mech), "", gen_reaction_tables(mech), "",
             f"struct mech_{cn} {{", "",
             f"static constexpr int NS = {ns};", f"static constexpr int NR = {mech.nreac};",
             f"static constexpr int N1 = {ns + 1};",
             f"static constexpr const char* NAME = \"{name}\";",
             f"static constexpr double RU = {_d(M.R_CGS)};", f"static constexpr double PATM = {_d(M.P_ATM)};",
             "static __host__ __device__ __forceinline__ double mw(int k) {",
             "  constexpr double t[NS] = {" + ", ".join(_d(w) for w in mech.W) + "};",
             "  return t[k];", "}",
             "static __host__ __device__ __forceinline__ double imw(int k) {",
             "  constexpr double t[NS] = {" + ", ".join(_d(1.0 / w) for w in mech.W) + "};",
             "  return t[k];", "}",
             "static const char* species(int k) {",
             "  static const char* t[NS] = {" + ", ".join(f'"{s.name}"' for s in mech.species) + "};",
             "  return t[k];", "}",
             ""]
    th = gen_thermo(mech)
    wd = gen_wdot(mech)
    jac = gen_jacobian(mech, shared=False)
    parts = th.split("static __device__ __forceinline__ void ")
    counts = {}
    for part in parts[1:]:
        fname = part.split("(")[0]
        counts[fname] = count_ops(part)
    counts["wdot"] = count_ops(wd)
    counts["jacobian"] = count_ops(jac)
    lines.append(gen_thermo_tables(mech))
    lines.append("")
    lines.append(gen_wdot_shared(mech))
    lines.append("")
    lines.append(gen_reaction_access(mech))
    lines.append("")
    lines.append(gen_jacobian(mech))
    lines.append("")
    lines.append(f"}};  // struct mech_{cn}")
    with open(path, "w") as f:
        f.write("\n".join(lines) + "\n")
    ops_path = os.path.join(os.path.dirname(os.path.dirname(path)), "..", "mechanisms", f"{name}_ops.json")
    with open(os.path.normpath(ops_path), "w") as f:
        # "functions": written out species by species and reaction by reaction, what the model
        # asks for; "emitted": the code that runs, one range of the NASA fits
        json.dump({"mechanism": name, "nspec": ns, "nreac": mech.nreac, "functions": counts,
                   "emitted": emitted_counts(mech)}, f, indent=1)
