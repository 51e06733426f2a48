"""Outputs of the molar-diffusion correction beside walls, bit for bit.

``python -m tests.golden.make_diffusion LIBRARY OUT`` (on a GPU) records what
LIBRARY computes for the cases below into OUT; tests/golden/diffusion.npz holds
the ones of the kernels that round every sum as the reference's text orders it.
The inputs are uniform numbers and sums, products and quotients of them, so
that they are the same bits on every machine.
"""
import sys

import numpy as np

from tiger_nga_amd import metric
from tiger_nga_amd.finitechem import FiniteChem, Grid
from tiger_nga_amd.mech import meta

# mech, order, molar, gas radiation, cv
CASES = [("h2", 2, True, False, True), ("ethyred", 2, True, True, False), ("dme39", 2, False, False, False),
         ("gri30", 4, True, True, False), ("dme39", 4, True, False, True), ("h2", 4, False, False, False)]


def name(case):
    return "_".join(str(int(v)) if isinstance(v, bool) else str(v) for v in case)


def fields(case):
    mech, order = case[:2]
    nover = order - 1
    sh = tuple(n + 2 * nover for n in (5, 6, 4))
    nsp = len(meta.species(mech))
    rng = np.random.default_rng(97 + nsp + order)
    Y = 0.05 + rng.random((nsp,) + sh)
    total = Y[0].copy()
    for k in range(1, nsp):
        total += Y[k]
    SC_ = np.empty(sh + (nsp + 1,), order="F")
    for k in range(nsp):
        SC_[..., k] = Y[k] / total
    SC_[..., nsp] = 400.0 + 1600.0 * rng.random(sh)
    RHO_ = np.asfortranarray(0.2 + rng.random(sh))
    DIFF_ = np.asfortranarray(1e-5 + 9e-5 * rng.random(SC_.shape))
    g = Grid.block(5, 6, 4, nsp + 1, 1, nsp + 1, nover=nover)
    x, y = (np.cumsum(np.concatenate([[0.0], 1e-4 * (1.0 + 0.3 * rng.random(n))])) for n in sh[:2])
    mask = np.zeros(g.mask_shape, dtype=np.int32, order="F")
    mask[:, nover] = mask[nover + 3, nover + 2] = 1  # the row at jmin_ and one cell inside
    return g, metric.cartesian(g, x, y, 1.1e-4, order), RHO_, SC_, DIFF_, mask


def outputs(case, set_options=lambda fc: None):
    """diff_corr and diff_gp of a case, interior cells, and the updated source."""
    import torch

    def dev(a):
        t = torch.empty_strided(a.shape, tuple(int(np.prod(a.shape[:k])) for k in range(a.ndim)),
                                dtype=torch.float64 if a.dtype == np.float64 else torch.int32, device="cuda")
        return t.copy_(torch.from_numpy(np.ascontiguousarray(a)))
    mech, order, molar, gasrad, cv = case
    g, m, RHO_, SC_, DIFF_, mask = fields(case)
    nsp, v = SC_.shape[-1] - 1, slice(order - 1, 1 - order)
    fc = FiniteChem(mech)
    set_options(fc)
    md = {k: (a if k in ("st1", "st2") else dev(np.asfortranarray(a))) for k, a in m.items()}
    corr, gp, src = (dev(np.full(g.shape + (n,), f, order="F")) for n, f in ((nsp + 1, 0.0), (3, 0.0), (nsp + 1, 1e-4)))
    fc.diffusion(1e-6, g, md, dev(RHO_), dev(SC_), dev(DIFF_), mask=dev(mask), diff_corr=corr, diff_gp=gp, src=src,
                 molar=molar, gasrad=gasrad, cv=cv)
    torch.cuda.synchronize()
    fc.close()
    return {k: a.cpu().numpy()[v, v, v].copy(order="F") for k, a in (("corr", corr), ("gp", gp), ("src", src))}


if __name__ == "__main__":
    import torch  # its HIP runtime first
    from tiger_nga_amd import finitechem
    assert torch.cuda.is_available()
    finitechem.load_library(sys.argv[1])
    np.savez_compressed(sys.argv[2], **{"%s_%s" % (name(c), k): a for c in CASES for k, a in outputs(c).items()})
