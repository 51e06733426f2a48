"""finitechem_diffusion on the GPU (tgr_chem_diffusion_device, C ABI) against
the CPU oracle (oracle/diffusion.c, pinned in tests/test_diffusion.py), on
random fields over stretched grids with the reference's metric operators:
second and fourth order, molar diffusion on and off, gas radiation, cv, a
wall row in the mask, and the update of the transport source.  Outputs agree
to 1e-12 of each field's scale (the kernels sum the same terms in the same
order; FMA contraction changes the last bits)."""
import gc
import os

import numpy as np
import pytest

from tests.golden import make_diffusion
from tiger_nga_amd import inputs, metric
from tiger_nga_amd.finitechem import Grid

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def torch_dev():
    import torch
    assert torch.cuda.is_available(), "GPU test without a HIP device"
    return torch


def _dev(torch, a):
    strides = tuple(int(np.prod(a.shape[:k])) for k in range(a.ndim))
    dtype = torch.float64 if a.dtype == np.float64 else torch.int32
    t = torch.empty_strided(a.shape, strides, dtype=dtype, device="cuda:0")
    t.copy_(torch.from_numpy(np.ascontiguousarray(a)).to("cuda:0"))
    return t


@pytest.mark.parametrize("mech,workload,order,molar,gasrad,cv,wall", [
    ("gri30", "gri30_uneven", 2, True, False, False, False), ("gri30", "gri30_uneven", 2, False, True, False, True),
    ("gri30", "gri30_uneven", 4, True, True, True, False), ("h2", "h2", 2, True, False, False, True),
    ("dme39", "dme39", 4, True, True, False, True)])
def test_diffusion_vs_oracle(torch_dev, oracle, mech, workload, order, molar, gasrad, cv, wall):
    torch = torch_dev
    from tiger_nga_amd.finitechem import FiniteChem
    nx, ny, nz = 9, 7, 6
    nover = {2: 1, 4: 3}[order]
    sh = (nx + 2 * nover, ny + 2 * nover, nz + 2 * nover)
    _, Y, T, rho, P, dt = inputs.states(workload, n=int(np.prod(sh)), seed=17)
    nsp = Y.shape[1]
    g = Grid.block(nx, ny, nz, nsp + 2, 1, nsp + 1, nover=nover)  # one extra scalar after T
    SC_ = np.zeros(sh + (nsp + 2,), order="F")
    for k in range(nsp):
        SC_[..., k] = Y[:, k].reshape(sh, order="F")
    SC_[..., nsp] = T.reshape(sh, order="F")
    SC_[..., nsp + 1] = 0.3
    RHO_ = np.asfortranarray(rho.reshape(sh, order="F"))
    rng = np.random.default_rng(5)
    DIFF_ = np.asfortranarray(10.0 ** rng.uniform(-5.0, -4.0, sh + (nsp + 2,)))
    x = np.cumsum(np.concatenate([[0.0], 1e-4 * (1.0 + 0.3 * rng.random(sh[0]))]))
    y = np.cumsum(np.concatenate([[0.0], 1e-4 * (1.0 + 0.3 * rng.random(sh[1]))]))
    m = metric.cartesian(g, x, y, 1.1e-4, order)
    mask = None
    if wall:
        mask = np.zeros(g.mask_shape, dtype=np.int32, order="F")
        mask[:, nover + 2] = 1  # a wall row at j = jmin_ + 2
    dc_o, gp_o = oracle.diffusion(mech, g, m, dt, RHO_, SC_, DIFF_, mask=mask, molar=molar, gasrad=gasrad, cv=cv)
    fc = FiniteChem(mech, 1e-6, 1e-12)
    md = {k: (v if k in ("st1", "st2") else _dev(torch, np.asfortranarray(v))) for k, v in m.items()}
    dc = _dev(torch, np.zeros(sh + (nsp + 1,), order="F"))
    gp = _dev(torch, np.zeros(sh + (3,), order="F"))
    src0 = np.asfortranarray(rng.standard_normal(SC_.shape))
    src = _dev(torch, src0)
    print("diffusion: %s order %d molar %d gasrad %d cv %d wall %d" % (mech, order, molar, gasrad, cv, wall),
          flush=True)
    fc.diffusion(dt, g, md, _dev(torch, RHO_), _dev(torch, SC_), _dev(torch, DIFF_),
                 mask=None if mask is None else _dev(torch, mask), diff_corr=dc, diff_gp=gp, src=src, molar=molar,
                 gasrad=gasrad, cv=cv)
    torch.cuda.synchronize()
    fc.close()
    dc, gp, src = dc.cpu().numpy(), gp.cpu().numpy(), src.cpu().numpy()
    for k in range(nsp + 1):
        scale = max(np.abs(dc_o[..., k]).max(), 1e-300)
        assert np.abs(dc[..., k] - dc_o[..., k]).max() <= 1e-12 * scale + 1e-300, k
    for q in range(3):
        scale = max(np.abs(gp_o[..., q]).max(), 1e-300)
        assert np.abs(gp[..., q] - gp_o[..., q]).max() <= 1e-12 * scale + 1e-300, q
    # finitechem_source_transport: src(species, T) += diff_corr on interior non-wall cells, nothing else
    want = src0.copy(order="F")
    want[..., :nsp + 1] += dc_o
    assert np.allclose(src, want, rtol=1e-12, atol=1e-12 * np.abs(dc_o).max())
    assert np.array_equal(src[..., nsp + 1], src0[..., nsp + 1])
    print("   max |diff_corr| species %.3e, T %.3e" % (np.abs(dc_o[..., :nsp]).max(), np.abs(dc_o[..., nsp]).max()))


@pytest.mark.parametrize("mech,nx,ny,nz,molar", [("h2", 1, 1, 1, True), ("gri30", 16, 16, 2, True),
                                                 ("dme39", 257, 1, 3, False), ("h2", 33, 32, 5, True)])
def test_second_order_workgroup_edges(torch_dev, oracle, mech, nx, ny, nz, molar):
    """One cell, whole workgroups, a few cells over, and planes of several strips
    of workgroups; the row and column past the block are walls that hold NaN
    species and diffusivities, which no flux may read.  Bound: as above, the
    sums differ in their order only."""
    torch = torch_dev
    from tiger_nga_amd.finitechem import FiniteChem
    sh = (nx + 2, ny + 2, nz + 2)
    _, Y, T, rho, P, dt = inputs.states(mech, n=int(np.prod(sh)), seed=23)
    nsp = Y.shape[1]
    g = Grid.block(nx, ny, nz, nsp + 1, 1, nsp + 1, nover=1)
    SC_ = np.zeros(sh + (nsp + 1,), order="F")
    for k in range(nsp):
        SC_[..., k] = Y[:, k].reshape(sh, order="F")
    SC_[..., nsp] = T.reshape(sh, order="F")
    RHO_ = np.asfortranarray(rho.reshape(sh, order="F"))
    rng = np.random.default_rng(6)
    DIFF_ = np.asfortranarray(10.0 ** rng.uniform(-5.0, -4.0, SC_.shape))
    x, y = (np.cumsum(np.concatenate([[0.0], 1e-4 * (1.0 + 0.3 * rng.random(n))])) for n in sh[:2])
    m = metric.cartesian(g, x, y, 1.1e-4, 2)
    mask = np.zeros(g.mask_shape, dtype=np.int32, order="F")
    mask[-1, :] = mask[:, -1] = 1
    dc_o, gp_o = oracle.diffusion(mech, g, m, dt, RHO_, SC_, DIFF_, mask=mask, molar=molar)
    for a in (SC_[..., :nsp], DIFF_):
        a[-1] = a[:, -1] = np.nan
    fc = FiniteChem(mech, 1e-6, 1e-12)
    md = {k: (v if k in ("st1", "st2") else _dev(torch, np.asfortranarray(v))) for k, v in m.items()}
    dc, gp = (_dev(torch, np.zeros(sh + (n,), order="F")) for n in (nsp + 1, 3))
    fc.diffusion(dt, g, md, _dev(torch, RHO_), _dev(torch, SC_), _dev(torch, DIFF_), mask=_dev(torch, mask),
                 diff_corr=dc, diff_gp=gp, molar=molar)
    torch.cuda.synchronize()
    fc.close()
    for got, want in ((dc.cpu().numpy(), dc_o), (gp.cpu().numpy(), gp_o)):
        for k in range(want.shape[-1]):
            scale = max(np.abs(want[..., k]).max(), 1e-300)
            assert np.abs(got[..., k] - want[..., k]).max() <= 1e-12 * scale + 1e-300, k


@pytest.mark.parametrize("mech,nx,ny,nz,molar", [("h2", 1, 1, 1, True), ("gri30", 13, 13, 3, False),
                                                 ("dme39", 254, 1, 2, True), ("ethyred", 10200, 1, 1, True)])
def test_fourth_order_workgroup_edges(torch_dev, oracle, mech, nx, ny, nz, molar):
    """One cell, whole workgroups of faces, a few over, and a block whose
    fluxes need two passes through the workspace, the second of one species;
    the last row and column are walls.  Bound: as above."""
    torch = torch_dev
    from tiger_nga_amd.finitechem import FiniteChem
    sh = (nx + 6, ny + 6, nz + 6)
    _, Y, T, rho, P, dt = inputs.states(mech, n=499, seed=29)
    nsp = Y.shape[1]
    g = Grid.block(nx, ny, nz, nsp + 1, 1, nsp + 1, nover=3)
    pick = np.arange(np.prod(sh)) * 7919 % 499
    SC_ = np.asfortranarray(np.concatenate([Y, T[:, None]], axis=1)[pick].reshape(sh + (nsp + 1,), order="F"))
    RHO_ = np.asfortranarray(rho[pick].reshape(sh, order="F"))
    rng = np.random.default_rng(7)
    DIFF_ = np.asfortranarray(10.0 ** rng.uniform(-5.0, -4.0, SC_.shape))
    x, y = (np.cumsum(np.concatenate([[0.0], 1e-4 * (1.0 + 0.3 * rng.random(n))])) for n in sh[:2])
    m = metric.cartesian(g, x, y, 1.1e-4, 4)
    mask = np.zeros(g.mask_shape, dtype=np.int32, order="F")
    mask[-1, :] = mask[:, -1] = 1
    dc_o, gp_o = oracle.diffusion(mech, g, m, dt, RHO_, SC_, DIFF_, mask=mask, molar=molar)
    fc = FiniteChem(mech, 1e-6, 1e-12)
    md = {k: (v if k in ("st1", "st2") else _dev(torch, np.asfortranarray(v))) for k, v in m.items()}
    dc, gp = (_dev(torch, np.zeros(sh + (n,), order="F")) for n in (nsp + 1, 3))
    fc.diffusion(dt, g, md, _dev(torch, RHO_), _dev(torch, SC_), _dev(torch, DIFF_), mask=_dev(torch, mask),
                 diff_corr=dc, diff_gp=gp, molar=molar)
    torch.cuda.synchronize()
    fc.close()
    for got, want in ((dc.cpu().numpy(), dc_o), (gp.cpu().numpy(), gp_o)):
        for k in range(want.shape[-1]):
            scale = max(np.abs(want[..., k]).max(), 1e-300)
            assert np.abs(got[..., k] - want[..., k]).max() <= 1e-12 * scale + 1e-300, k


@pytest.mark.parametrize("case", make_diffusion.CASES, ids=make_diffusion.name)
def test_walls_round_as_recorded(torch_dev, case):
    """Cells beside walls, where the molar fluxes nearly cancel and another
    order of the sums shows at 1e-12 of the field: the recorded outputs (sums in
    the order of the reference's text) to the last bit."""
    want = np.load(os.path.join(os.path.dirname(make_diffusion.__file__), "diffusion.npz"))
    for k, a in make_diffusion.outputs(case).items():
        w = want["%s_%s" % (make_diffusion.name(case), k)]
        assert np.abs(w).max() > 0.0
        print("%s: largest difference over the rms %.1e" % (k, np.abs(a - w).max() / np.sqrt(np.mean(w * w))))
        assert np.array_equal(a, w), k


@pytest.mark.parametrize("order", [2, 4])
@pytest.mark.parametrize("nx,ny,nz", [(1, 1, 300), (1, 300, 2), (35, 35, 3)])
def test_thin_blocks(torch_dev, oracle, order, nx, ny, nz):
    """Blocks one cell wide, and a plane of several workgroups and a remainder;
    bound as above."""
    torch = torch_dev
    from tiger_nga_amd.finitechem import FiniteChem
    nover = order - 1
    sh = (nx + 2 * nover, ny + 2 * nover, nz + 2 * nover)
    _, Y, T, rho, P, dt = inputs.states("h2", n=499, seed=31)
    nsp = Y.shape[1]
    g = Grid.block(nx, ny, nz, nsp + 1, 1, nsp + 1, nover=nover)
    pick = np.arange(np.prod(sh)) * 7919 % 499
    SC_ = np.asfortranarray(np.concatenate([Y, T[:, None]], axis=1)[pick].reshape(sh + (nsp + 1,), order="F"))
    RHO_ = np.asfortranarray(rho[pick].reshape(sh, order="F"))
    rng = np.random.default_rng(8)
    DIFF_ = np.asfortranarray(10.0 ** rng.uniform(-5.0, -4.0, SC_.shape))
    x, y = (np.cumsum(np.concatenate([[0.0], 1e-4 * (1.0 + 0.3 * rng.random(n))])) for n in sh[:2])
    m = metric.cartesian(g, x, y, 1.1e-4, order)
    dc_o, gp_o = oracle.diffusion("h2", g, m, dt, RHO_, SC_, DIFF_, molar=True)
    fc = FiniteChem("h2")
    md = {k: (v if k in ("st1", "st2") else _dev(torch, np.asfortranarray(v))) for k, v in m.items()}
    dc, gp = (_dev(torch, np.zeros(sh + (n,), order="F")) for n in (nsp + 1, 3))
    fc.diffusion(dt, g, md, _dev(torch, RHO_), _dev(torch, SC_), _dev(torch, DIFF_), diff_corr=dc, diff_gp=gp, molar=True)
    torch.cuda.synchronize()
    fc.close()
    for got, want in ((dc.cpu().numpy(), dc_o), (gp.cpu().numpy(), gp_o)):
        for k in range(want.shape[-1]):
            scale = max(np.abs(want[..., k]).max(), 1e-300)
            assert np.abs(got[..., k] - want[..., k]).max() <= 1e-12 * scale + 1e-300, k


def test_column_of_four_million_cells(torch_dev):
    """1 x 1 x (2^22 + 3) cells: no more workgroups than cells / 256, which a
    launch of whole workgroups per plane exceeds.  Its first and last 500 planes
    equal the same planes as a block of their own."""
    torch = torch_dev
    from tiger_nga_amd.finitechem import FiniteChem
    nz, part = (1 << 22) + 3, 500
    fc = FiniteChem("h2")
    nsp = fc.nsp
    gen = torch.Generator(device="cuda").manual_seed(3)
    face = np.arange(4) * 1e-4

    def run(RHO_, SC_, DIFF_, n):
        g = Grid.block(1, 1, n, nsp + 1, 1, nsp + 1, nover=1)
        md = {k: (v if k in ("st1", "st2") else _dev(torch, np.asfortranarray(v)))
              for k, v in metric.cartesian(g, face, face, 1.1e-4, 2).items()}
        fortran = lambda a: a.permute(*reversed(range(a.ndim)))
        corr = torch.zeros(nsp + 1, n + 2, 3, 3, dtype=torch.float64, device="cuda")
        fc.diffusion(1e-6, g, md, fortran(RHO_.contiguous()), fortran(SC_.contiguous()), fortran(DIFF_.contiguous()),
                     diff_corr=fortran(corr), molar=True)
        return corr
    SC_ = torch.rand(nsp + 1, nz + 2, 3, 3, generator=gen, dtype=torch.float64, device="cuda")
    SC_[:nsp] /= SC_[:nsp].sum(0)
    SC_[nsp] = 400.0 + 1600.0 * SC_[nsp]
    DIFF_ = 1e-5 + 1e-4 * torch.rand(SC_.shape, generator=gen, dtype=torch.float64, device="cuda")
    RHO_ = torch.ones(nz + 2, 3, 3, dtype=torch.float64, device="cuda")
    whole = run(RHO_, SC_, DIFF_, nz)
    assert float(whole[:, 1:-1, 1, 1].abs().min()) > 0.0
    for z in (slice(0, part + 2), slice(nz - part, nz + 2)):
        assert torch.equal(whole[:, z][:, 1:-1], run(RHO_[z], SC_[:, z], DIFF_[:, z], part)[:, 1:-1])
    fc.close()


@pytest.mark.parametrize("case", make_diffusion.CASES[3:], ids=make_diffusion.name)
def test_fourth_order_workspace_sizes(torch_dev, case):
    """Fourth order without a flux workspace (the general kernels), with one
    that holds a part of the species at a time, and with the default: the same
    outputs to the last bit."""
    ref = make_diffusion.outputs(case, lambda fc: fc.set_option("diff_flux_mb", 0))
    for mb in (1, 1024):
        got = make_diffusion.outputs(case, lambda fc: fc.set_option("diff_flux_mb", mb))
        for k in ref:
            assert np.array_equal(got[k], ref[k]), (mb, k)


def _block(torch, mech, nx, ny, nz, order):
    """Fields of a block on the GPU and a call of the correction on them."""
    from tiger_nga_amd.finitechem import FiniteChem
    fc = FiniteChem(mech)
    nsp, nover = fc.nsp, order - 1
    g = Grid.block(nx, ny, nz, nsp + 1, 1, nsp + 1, nover=nover)
    gen = torch.Generator(device="cuda").manual_seed(5)
    fortran = lambda a: a.permute(*reversed(range(a.ndim)))
    shp = tuple(reversed(g.shape))
    SC_ = torch.rand((nsp + 1,) + shp, generator=gen, dtype=torch.float64, device="cuda")
    SC_[:nsp] /= SC_[:nsp].sum(0)
    SC_[nsp] = 400.0 + 1600.0 * SC_[nsp]
    DIFF_ = 1e-5 + 1e-4 * torch.rand(SC_.shape, generator=gen, dtype=torch.float64, device="cuda")
    RHO_ = torch.ones(shp, dtype=torch.float64, device="cuda")
    corr = torch.zeros_like(SC_)

    ops = {o: {k: (v if k in ("st1", "st2") else _dev(torch, np.asfortranarray(v))) for k, v in
               metric.cartesian(g, np.arange(g.shape[0] + 1) * 1e-4, np.arange(g.shape[1] + 1) * 1e-4, 1.1e-4, o).items()}
           for o in {2, order}}

    def call(order=order, stream=None):
        fc.diffusion(1e-6, g, ops[order], fortran(RHO_), fortran(SC_), fortran(DIFF_), diff_corr=fortran(corr),
                     stream=stream)
        return corr
    return fc, call


def test_fourth_order_takes_a_quarter_of_the_memory(torch_dev):
    """With 3 GiB free a block whose fluxes would fill 1 GiB gets a workspace of
    at most a quarter of that, once: the outputs are those of the general
    kernels, which take three times as long."""
    torch = torch_dev
    fc, call = _block(torch, "gri30", 120, 120, 120, 4)

    def timed():
        ev = [torch.cuda.Event(enable_timing=True) for _ in range(2)]
        ev[0].record()
        out = call()
        ev[1].record()
        torch.cuda.synchronize()
        return out, ev[0].elapsed_time(ev[1])
    fc.set_option("diff_flux_mb", 0)
    call()
    want, general = timed()
    want = want.clone()
    fc.set_option("diff_flux_mb", 1024)
    gc.collect()  # what earlier tests left
    torch.cuda.synchronize()
    torch.cuda.empty_cache()
    hog, free0 = [], torch.cuda.mem_get_info()[0]
    while free0 > 3.1 * 2 ** 30 and len(hog) < 8:  # memory freed before may come back late
        hog.append(torch.empty(free0 - (3 << 30), dtype=torch.uint8, device="cuda"))
        torch.cuda.synchronize()
        free0 = torch.cuda.mem_get_info()[0]
    assert torch.equal(call(), want)
    left = torch.cuda.mem_get_info()[0]
    out, fluxes = timed()
    again = torch.cuda.mem_get_info()[0]
    assert torch.equal(out, want) and fluxes < 0.6 * general, (fluxes, general)
    del hog
    torch.cuda.empty_cache()
    fc.close()
    assert free0 - left <= free0 // 4 and again >= left


def test_orders_under_capture(torch_dev):
    """Second order captured in a graph, then fourth order captured on a context
    that has had this block at second order only (nothing may be allocated:
    it runs without a flux workspace), then fourth order called, whose
    workspace leaves the second-order graph's alone: every replay equals the
    eager call."""
    torch = torch_dev
    fc, call = _block(torch, "h2", 13, 11, 9, 4)
    side = torch.cuda.Stream()
    graphs = {}
    with torch.cuda.stream(side):
        call(2, side.cuda_stream)
    torch.cuda.synchronize()
    for order in (2, 4):
        graphs[order] = torch.cuda.CUDAGraph()
        with torch.cuda.graph(graphs[order], stream=side):
            call(order, torch.cuda.current_stream().cuda_stream)
    want = {order: call(order).clone() for order in (4, 2)}
    for _ in range(3):
        for order in (2, 4):
            out = call(6 - order)
            graphs[order].replay()
            torch.cuda.synchronize()
            assert torch.equal(out, want[order])
    fc.close()


def test_second_order_beyond_32_bit_offsets(torch_dev):
    """A block of more than 2^29 cells goes by slabs of planes: the planes at its
    ends and on both sides of the slabs' border equal the same planes as a block
    of their own."""
    torch = torch_dev
    from tiger_nga_amd.finitechem import FiniteChem
    if torch.cuda.mem_get_info()[0] < 200 << 30:
        pytest.skip("needs 200 GB of GPU memory")
    n, nz = 1024, 513
    fc = FiniteChem("h2")
    nsp = fc.nsp
    fortran = lambda a: a.permute(*reversed(range(a.ndim)))

    def run(RHO_, SC_, DIFF_, corr, nz):
        g = Grid.block(n, n, nz, nsp + 1, 1, nsp + 1, nover=1)
        face = np.arange(n + 3) * 1e-4
        md = {k: (v if k in ("st1", "st2") else _dev(torch, np.asfortranarray(v)))
              for k, v in metric.cartesian(g, face, face, 1.1e-4, 2).items()}
        fc.diffusion(1e-6, g, md, fortran(RHO_), fortran(SC_), fortran(DIFF_), diff_corr=fortran(corr), molar=True)
        return corr
    shp = (nsp + 1, nz + 2, n + 2, n + 2)
    assert shp[1] * shp[2] * shp[3] > 1 << 29
    gen = torch.Generator(device="cuda").manual_seed(3)
    SC_, DIFF_ = (torch.empty(shp, dtype=torch.float64, device="cuda") for _ in range(2))
    for k in range(nsp + 1):  # 0.1 <= Y < 0.12, 400 <= T < 2000
        SC_[k].uniform_(0.1, 0.12, generator=gen) if k < nsp else SC_[k].uniform_(400.0, 2000.0, generator=gen)
        DIFF_[k].uniform_(1e-5, 1e-4, generator=gen)
    RHO_ = torch.ones(shp[1:], dtype=torch.float64, device="cuda")
    whole = run(RHO_, SC_, DIFF_, torch.zeros(shp, dtype=torch.float64, device="cuda"), nz)
    for z in (slice(0, 6), slice((1 << 29) // (n + 2) ** 2 - 6, nz + 2)):
        part = [a[..., z, :, :].contiguous() for a in (RHO_, SC_, DIFF_)]
        own = run(*part, torch.zeros_like(part[1]), part[0].shape[0] - 2)
        assert float(own[:, 1:-1, 1:-1, 1:-1].abs().max()) > 0.0
        assert torch.equal(whole[:, z][:, 1:-1], own[:, 1:-1])
    fc.close()


@pytest.mark.parametrize("mech,molar,wall", [("h2", True, True), ("gri30", False, False), ("ethyred", True, False)])
def test_general_stencil_vs_oracle(torch_dev, oracle, mech, molar, wall):
    """Sixth order, the stencil that only the general kernels take; bound as above."""
    torch = torch_dev
    from tiger_nga_amd.finitechem import FiniteChem
    order, nover = 6, 5
    sh = (5 + 2 * nover, 4 + 2 * nover, 3 + 2 * nover)
    _, Y, T, rho, P, dt = inputs.states(mech, n=499, seed=37)
    nsp = Y.shape[1]
    g = Grid.block(5, 4, 3, nsp + 1, 1, nsp + 1, nover=nover)
    pick = np.arange(np.prod(sh)) * 7919 % 499
    SC_ = np.asfortranarray(np.concatenate([Y, T[:, None]], axis=1)[pick].reshape(sh + (nsp + 1,), order="F"))
    RHO_ = np.asfortranarray(rho[pick].reshape(sh, order="F"))
    rng = np.random.default_rng(9)
    DIFF_ = np.asfortranarray(10.0 ** rng.uniform(-5.0, -4.0, SC_.shape))
    x, y = (np.cumsum(np.concatenate([[0.0], 1e-4 * (1.0 + 0.3 * rng.random(n))])) for n in sh[:2])
    m = metric.cartesian(g, x, y, 1.1e-4, order)
    assert (m["st1"], m["st2"]) == (2, 3)
    mask = None
    if wall:
        mask = np.zeros(g.mask_shape, dtype=np.int32, order="F")
        mask[:, nover + 1] = 1
    dc_o, gp_o = oracle.diffusion(mech, g, m, dt, RHO_, SC_, DIFF_, mask=mask, molar=molar, gasrad=True)
    fc = FiniteChem(mech)
    md = {k: (v if k in ("st1", "st2") else _dev(torch, np.asfortranarray(v))) for k, v in m.items()}
    dc, gp = (_dev(torch, np.zeros(sh + (n,), order="F")) for n in (nsp + 1, 3))
    fc.diffusion(dt, g, md, _dev(torch, RHO_), _dev(torch, SC_), _dev(torch, DIFF_),
                 mask=None if mask is None else _dev(torch, mask), diff_corr=dc, diff_gp=gp, molar=molar, gasrad=True)
    torch.cuda.synchronize()
    fc.close()
    for got, want in ((dc.cpu().numpy(), dc_o), (gp.cpu().numpy(), gp_o)):
        for k in range(want.shape[-1]):
            scale = max(np.abs(want[..., k]).max(), 1e-300)
            assert np.abs(got[..., k] - want[..., k]).max() <= 1e-12 * scale + 1e-300, k
