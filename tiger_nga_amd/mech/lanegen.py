"""Generates the lane-per-state right-hand side of each compiled mechanism.

For one mechanism, writes ``csrc/lane_rhs_<mech>.h``: a specialisation of
``tgr::LaneRhs<NEQ>`` whose ``rates`` computes PRODRATES / GETLINDRATECOEFF
(e.g. combustion/HYDROGENF.f90:4-316) and ``eval`` finitechem_compute_rhs
(combustion/finitechem.f90:93-175, with COMPTHERMODATA, HYDROGENF.f90:514-673)
for a whole state held by ONE lane: straight-line code in which every species index is a
compile-time constant, so concentrations and production rates stay in
registers and every coefficient is an immediate operand.  The integrator uses
it where it needs many independent right-hand sides at once: the NEQ columns
of the difference-quotient Jacobian, one column per lane.

The arithmetic is that of the wave-per-cell evaluation in chem_device.h
(same coefficient values, same Arrhenius / Troe / NASA-7 forms, third-body
sums as total concentration plus (efficiency - 1) corrections); only the
order of the production-rate sums differs (reaction order instead of the
gather schedule), which changes rounding only.

Input: the mechanism data written by mechc.py (``data/<mech>.json``).
Usage: ``python -m tiger_nga_amd.mech.lanegen``.
"""
from __future__ import annotations

import os
import sys
from decimal import Decimal, localcontext
from fractions import Fraction

from tiger_nga_amd.mech import mechc

HERE = os.path.dirname(os.path.abspath(__file__))
MECHANISMS = ("h2", "gri30", "dme39", "ethyred")
T_UNIT = 512  # kTUnit of chem_device.h


def _c(x) -> str:
    return mechc._c(x)


def _log2e(d, inverse=False):
    """log2(e) d, or log2(e) / d, rounded once."""
    l2e = Fraction("1.442695040888963407359924681001892137426645954153")
    return float(l2e / Fraction(d) if inverse else l2e * Fraction(d))


def _arrh(w, var, k, lt="lt", irt="irt"):
    """k = A T^b exp(e / (R T)) as in chem_device.h arrhenius(), T in units of T_UNIT."""
    with localcontext() as ctx:
        ctx.prec = 40
        A = float(Decimal(k["A"]) * Decimal(T_UNIT) ** Decimal(k["b"]))
    w("    const double %s = %s * fexp2(fma(%s, %s, %s * %s));" % (var, _c(A), _c(k["e"]), irt, _c(k["b"]), lt))


def _prod(base, facs):
    e = base
    for f in facs:
        e = "%s * C%d" % (e, f)
    return e


def emit_lane_rhs(mech: dict) -> str:
    name = mech["name"]
    nsp = len(mech["species"])
    neq = nsp + 1
    W = mech["W"]
    L = []
    w = L.append
    w("/* Generated by tiger_nga_amd/mech/lanegen.py from the compiled mechanism %s" % name)
    w(" * (reference %s).  Do not edit.  Lane-per-state right-hand side of" % mech["source"])
    w(" * finitechem_compute_rhs (combustion/finitechem.f90:93-175). */")
    w("#pragma once")
    w('#include "lane_rhs.h"')
    w("")
    w("namespace tgr {")
    w("")
    w("template <>")
    w("struct LaneRhs<%d> {" % neq)
    w("  // production rates cd (kmol/m3/s) from the concentrations, temperature and pressure of this lane's state")
    w("  static __device__ __forceinline__ void rates(const double (&C)[%d], double T, double P, double (&cd)[%d]) {"
      % (nsp, nsp))
    for k in range(nsp):
        w("    const double C%d = C[%d];" % (k, k))
    w("    const double lt = flog2(T * (1.0 / kTUnit));")
    w("    const double rt = kRgasF4 * T;")
    w("    const double irt = kLog2e / rt;")
    w("    const double invT = 1.0 / T;")
    w("    const double p_rt = P / rt;")
    w("    double ctot = C0;")
    for k in range(1, nsp):
        w("    ctot += C%d;" % k)
    # third-body sums as lambdas evaluated at use
    eff = mech["third_body"]
    for j, row in enumerate(eff):
        terms = "".join(" s_ = fma(%s, C%d, s_);" % (_c(e - 1.0), k) for k, e in enumerate(row) if e != 1.0)
        w("    auto M%d = [&]() { double s_ = ctot;%s return s_; };" % (j, terms))
    for k in range(nsp):
        w("    double cd%d = 0.0;" % k)
    # reactions, grouped by the third-body sum they use so that each sum is
    # formed once and is live only over its group (fewer registers); the
    # order changes the rounding of the production-rate sums only
    def m_of(r):
        return r["m_fo"] if r["type"] == "falloff" else r["m_w"]
    rxs = sorted(mech["reactions"], key=lambda r: m_of(r))
    for r in rxs:
        w("    {  // %s (%s)" % (r["name"], r["type"]))
        rev = r["slot_b"] >= 0
        if r["type"] == "falloff":
            _arrh(w, "kinf_f", r["f_kinf"])
            _arrh(w, "k0_f", r["f_k0"])
            if rev:
                _arrh(w, "kinf_b", r["b_kinf"])
                _arrh(w, "k0_b", r["b_k0"])
            fc = r["fc"]
            lind = len(fc) == 1 and fc[0][0] == 1.0 and fc[0][1] == 1 and fc[0][2] == 0.0
            mi = r["m_fo"]
            if mi >= 0:
                w("    const double m_ = M%d();" % mi)
                w("    const double conc = m_ > 0.0 ? m_ : p_rt;")
            else:
                w("    const double conc = p_rt;")
            if lind:
                # Fc = 1: log10 Fc = 0 and F = 1 exactly
                w("    const double pr_f = k0_f * conc / fmax(kinf_f, 1.0e-60);")
                w("    const double kf = kinf_f * pr_f / (1.0 + pr_f);")
                if rev:
                    w("    const double pr_b = k0_b * conc / fmax(kinf_b, 1.0e-60);")
                    w("    const double kb = kinf_b * pr_b / (1.0 + pr_b);")
            else:
                w("    double fc = 0.0;")
                for c, kind, d in fc:
                    # exp(-d / T) as 2^(-(log2(e) d) (1/T)); exp(-T / d) as 2^(-(log2(e) / d) T)
                    x = "-(%s * %s)" % ((_c(_log2e(d)), "invT") if kind == 1 else (_c(_log2e(d, True)), "T"))
                    w("    fc = fma(%s, fexp2(%s), fc);" % (_c(c), x))
                w("    const double l2fc = flog2(fc);")
                w("    const double lfc = l2fc * kLog10Of2;")
                w("    const double ntmp = fma(-kTroeN1, lfc, kTroeN0);")
                w("    const double cco = fma(-kTroeC1, lfc, -kTroeC0);")
                w("    const double kf = troe(kinf_f, k0_f, conc, l2fc, ntmp, cco);")
                if rev:
                    w("    const double kb = troe(kinf_b, k0_b, conc, l2fc, ntmp, cco);")
        else:
            _arrh(w, "kf", r["f"])
            if rev:
                _arrh(w, "kb", r["b"])
        wf = _prod("kf", r["reac"])
        if rev:
            q = "%s - %s" % (wf, _prod("kb", r["prod"]))
        else:
            q = wf
        if r["type"] == "third_body":
            w("    const double q = (%s) * M%d();" % (q, r["m_w"]))
        else:
            w("    const double q = %s;" % q)
        for sp, nu in r["nu"]:
            if nu == 1.0:
                w("    cd%d += q;" % sp)
            elif nu == -1.0:
                w("    cd%d -= q;" % sp)
            else:
                w("    cd%d = fma(%s, q, cd%d);" % (sp, _c(nu), sp))
        w("    }")
    for k in range(nsp):
        w("    cd[%d] = cd%d;" % (k, k))
    w("  }")
    w("")
    w("  // s: [rho*Y (%d), rho*T] of this lane's state; f: the right-hand side" % nsp)
    w("  static __device__ __forceinline__ void eval(const double (&s)[%d], double P, double (&f)[%d]) {"
      % (neq, neq))
    # density, temperature, concentrations
    w("    double rho = s[0];")
    for k in range(1, nsp):
        w("    rho += s[%d];" % k)
    w("    const double T = s[%d] / rho;" % nsp)
    w("    const double irho = 1.0 / rho;")
    w("    double C[%d], cd[%d];" % (nsp, nsp))
    for k in range(nsp):
        w("    C[%d] = s[%d] * %s;" % (k, k, _c(1.0 / W[k])))
    # mixture heat capacity (COMPTHERMODATA cp, finitechem_Cp)
    w("    const bool hi = T > %s;" % _c(mech["tmid"]))
    w("    double cpm = 0.0;")
    for blk, cond in (("thermo_hi", "if (hi) {"), ("thermo_lo", "} else {")):
        w("    " + cond)
        for k in range(nsp):
            d = mech[blk][k]["cp"]
            w("      cpm = fma(s[%d] * irho, %s * (%s + T * (%s + T * (%s + T * (%s + T * %s)))), cpm);"
              % (k, _c(d[0]), _c(d[1]), _c(d[2]), _c(d[3]), _c(d[4]), _c(d[5])))
    w("    }")
    w("    rates(C, T, P, cd);")
    # rhs: species then temperature
    for k in range(nsp):
        w("    f[%d] = cd[%d] * %s;" % (k, k, _c(W[k])))
    w("    double tmp = 0.0;")
    for blk, cond in (("thermo_hi", "if (hi) {"), ("thermo_lo", "} else {")):
        w("    " + cond)
        for k in range(nsp):
            c = mech[blk][k]["h"]
            w("      tmp = fma(-(%s * (T * (%s + T * (%s + T * (%s + T * (%s + T * %s)))) + %s)), f[%d], tmp);"
              % (_c(c[0]), _c(c[1]), _c(c[2]), _c(c[3]), _c(c[4]), _c(c[5]), _c(c[6]), k))
    w("    }")
    w("    f[%d] = tmp / cpm;" % nsp)
    w("  }")
    w("};")
    w("")
    w("}  // namespace tgr")
    return "\n".join(L) + "\n"


def main(argv=None):
    names = (argv if argv else None) or list(MECHANISMS)
    for name in names:
        mech = mechc.from_json(open(os.path.join(HERE, "data", name + ".json")).read())
        out = os.path.join(HERE, "..", "csrc", "lane_rhs_%s.h" % name)
        with open(out, "w") as f:
            f.write(emit_lane_rhs(mech))
        print("%s -> %s" % (name, os.path.relpath(out)))


if __name__ == "__main__":
    sys.exit(main(sys.argv[1:]))
