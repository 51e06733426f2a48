"""Python host mirror of the reference's finite-rate chemistry interface.

Wraps the C ABI of ``libtiger_chem.so`` (include/tiger_chem.h) with the names
and argument meaning of the reference Fortran (combustion/finitechem.f90):

* ``FiniteChem(mech, rtol, atol)``          ~ finitechem_init (184-319)
* ``.source_chemistry(RHO_, SC_, ...)``    ~ finitechem_source_chemistry(RHO_, SC_) (962-1071)
* ``.prodrates(C, T, P)``                  ~ PRODRATES (HYDROGENF.f90:4-277), batched
* ``.compute_rhs(sol, p_gp)``              ~ finitechem_compute_rhs (93-175), batched
* ``.species_names`` / ``.molar_mass``     ~ GETSPECIESNAMES / GETMOLARMASS

Arrays are Fortran-ordered 3-D/4-D fields (i fastest).  Host numpy arrays
take the synchronous host entry point; CUDA/HIP torch tensors take the
device-resident entry point.  The HIP library is required: there is no CPU
fallback, and a missing library raises ``RuntimeError``.
"""
from __future__ import annotations

import ctypes
import os
from dataclasses import dataclass

import numpy as np

_HERE = os.path.dirname(os.path.abspath(__file__))
LIB_PATH = os.path.join(_HERE, "libtiger_chem.so")


class _Grid(ctypes.Structure):
    _fields_ = [(n, ctypes.c_int) for n in (
        "imin_", "imax_", "jmin_", "jmax_", "kmin_", "kmax_",
        "imino_", "imaxo_", "jmino_", "jmaxo_", "kmino_", "kmaxo_",
        "imino", "imaxo", "jmino", "jmaxo", "nscalar", "isc_sc", "isc_T")]


class _Stats(ctypes.Structure):
    _fields_ = [(n, ctypes.c_int64) for n in (
        "cells", "nst", "nfe", "nfe_dq", "nje", "nsetups", "nni", "netf", "ncfn", "nlu", "failed")] + [
        ("kernel_ms", ctypes.c_double)]


REAL_OPTIONS = ("surr_tol_y", "surr_tol_t", "surr_newton_tol", "surr_grade", "surr_min_accept", "surr_h0_fac",
                "surr_grow", "surr_keep", "surr_jac_theta", "surr_sa_tol")


class _SurrStats(ctypes.Structure):
    _fields_ = [(n, ctypes.c_int64) for n in (
        "accepted", "rejected", "newton_iters", "rhs_evals", "rej_newton", "rej_error", "rej_enthalpy",
        "substeps", "factorizations", "jacobians")] + [
        ("surrogate_ms", ctypes.c_double), ("fallback_ms", ctypes.c_double), ("guided", ctypes.c_int)]


METRIC_OPERATORS = ("interp_sc_x", "interp_sc_y", "interp_sc_z", "grad_x", "grad_y", "grad_z", "div_u", "div_v",
                    "div_w", "interp_u_xm", "interp_v_ym", "interp_w_zm", "grad_xm", "grad_ym", "grad_zm")


class _Metric(ctypes.Structure):
    _fields_ = [("st1", ctypes.c_int), ("st2", ctypes.c_int)] + [(n, ctypes.c_void_p) for n in METRIC_OPERATORS]


class _Info(ctypes.Structure):
    _fields_ = [(n, ctypes.c_int) for n in (
        "nsp", "nrxn", "nslot", "n_third", "n_falloff", "n_third_body_rxn", "n_reversible", "n_nu", "n_fc_terms",
        "n_conc_factors", "n_eff_corr", "n_rev_falloff")]


@dataclass
class Grid:
    """Block extents (reference geometry/partition.f90:53-90, masks.f90:55);
    scalar indices are 1-based as in the reference."""
    imin_: int
    imax_: int
    jmin_: int
    jmax_: int
    kmin_: int
    kmax_: int
    imino_: int
    imaxo_: int
    jmino_: int
    jmaxo_: int
    kmino_: int
    kmaxo_: int
    nscalar: int
    isc_sc: int
    isc_T: int
    imino: int | None = None
    imaxo: int | None = None
    jmino: int | None = None
    jmaxo: int | None = None

    @staticmethod
    def block(nx, ny, nz, nscalar, isc_sc, isc_T, nover=0):
        """Interior 1..n with ``nover`` ghost layers on each side."""
        return Grid(1, nx, 1, ny, 1, nz, 1 - nover, nx + nover, 1 - nover, ny + nover, 1 - nover, nz + nover,
                    nscalar, isc_sc, isc_T)

    @property
    def shape(self):
        return (self.imaxo_ - self.imino_ + 1, self.jmaxo_ - self.jmino_ + 1, self.kmaxo_ - self.kmino_ + 1)

    @property
    def mask_shape(self):
        return (self.imaxo_m - self.imino_m + 1, self.jmaxo_m - self.jmino_m + 1)

    @property
    def imino_m(self):
        return self.imino_ if self.imino is None else self.imino

    @property
    def imaxo_m(self):
        return self.imaxo_ if self.imaxo is None else self.imaxo

    @property
    def jmino_m(self):
        return self.jmino_ if self.jmino is None else self.jmino

    @property
    def jmaxo_m(self):
        return self.jmaxo_ if self.jmaxo is None else self.jmaxo

    def _c(self):
        return _Grid(self.imin_, self.imax_, self.jmin_, self.jmax_, self.kmin_, self.kmax_,
                     self.imino_, self.imaxo_, self.jmino_, self.jmaxo_, self.kmino_, self.kmaxo_,
                     self.imino_m, self.imaxo_m, self.jmino_m, self.jmaxo_m,
                     self.nscalar, self.isc_sc, self.isc_T)


_lib = None


def load_library(path: str = LIB_PATH):
    """Load the HIP chemistry library; raises if it is not built."""
    global _lib
    if _lib is not None:
        return _lib
    if not os.path.exists(path):
        raise RuntimeError("libtiger_chem.so not built (%s): run __graft_entry__.build()" % path)
    lib = ctypes.CDLL(path)
    vp, dp, ip = ctypes.c_void_p, ctypes.POINTER(ctypes.c_double), ctypes.POINTER(ctypes.c_int)
    lib.tgr_chem_create.argtypes = [ctypes.c_char_p, ctypes.c_double, ctypes.c_double, ctypes.c_int,
                                    ctypes.POINTER(vp)]
    lib.tgr_chem_destroy.argtypes = [vp]
    lib.tgr_chem_mech_info.argtypes = [vp, ctypes.POINTER(_Info)]
    lib.tgr_chem_species_name.argtypes = [vp, ctypes.c_int, ctypes.c_char_p, ctypes.c_int]
    lib.tgr_chem_molar_mass.argtypes = [vp, dp]
    step_args = [vp, ctypes.c_double, ctypes.c_double, ctypes.c_double, ctypes.POINTER(_Grid), vp, vp, vp, vp, vp]
    lib.tgr_chem_source_chemistry.argtypes = step_args + [ctypes.POINTER(_Stats)]
    lib.tgr_chem_source_chemistry_device.argtypes = step_args + [vp, ctypes.POINTER(_Stats)]
    lib.tgr_chem_source_chemistry_device_noalloc.argtypes = step_args + [vp]
    lib.tgr_chem_prodrates_device.argtypes = [vp, ctypes.c_int64, vp, vp, vp, vp, vp]
    lib.tgr_chem_rhs_device.argtypes = [vp, ctypes.c_int64, ctypes.c_double, vp, vp, vp]
    lib.tgr_chem_temperature_device.argtypes = [vp, ctypes.c_int64, vp, vp, vp, vp, vp, vp]
    lib.tgr_chem_properties_device.argtypes = [vp, ctypes.c_double, ctypes.POINTER(_Grid), vp, vp, vp, ctypes.c_int,
                                               vp, vp, vp, vp]
    lib.tgr_chem_diffusion_device.argtypes = [vp, ctypes.c_double, ctypes.POINTER(_Grid), ctypes.POINTER(_Metric),
                                              ctypes.c_int, vp, vp, vp, vp, vp, vp, vp, vp]
    lib.tgr_chem_set_option.argtypes = [vp, ctypes.c_char_p, ctypes.c_int64]
    lib.tgr_chem_set_option_real.argtypes = [vp, ctypes.c_char_p, ctypes.c_double]
    fp = ctypes.POINTER(ctypes.c_float)
    lib.tgr_chem_set_surrogate.argtypes = [vp, vp, fp, fp, dp]
    lib.tgr_chem_surrogate_features_device.argtypes = [vp, ctypes.c_double, ctypes.POINTER(_Grid), vp, vp,
                                                       ctypes.c_int64, vp]
    lib.tgr_chem_source_chemistry_surrogate_device.argtypes = step_args + [vp, ctypes.POINTER(_Stats),
                                                                           ctypes.POINTER(_SurrStats)]
    lib.tgr_chem_source_chemistry_surrogate.argtypes = step_args + [ctypes.POINTER(_Stats),
                                                                    ctypes.POINTER(_SurrStats)]
    lib.tgr_chem_load_surrogate.argtypes = [vp, ctypes.c_char_p]
    lib.tgr_chem_last_error.restype = ctypes.c_char_p
    _lib = lib
    return lib


class ChemError(RuntimeError):
    pass


def _check(lib, rc, what):
    if rc != 0:
        raise ChemError("%s failed (%d): %s" % (what, rc, lib.tgr_chem_last_error().decode()))


def _ptr(a):
    """Raw pointer of a numpy array or torch tensor (None -> NULL)."""
    if a is None:
        return None
    if isinstance(a, np.ndarray):
        return a.ctypes.data
    return a.data_ptr()


def _is_device(a):
    return a is not None and not isinstance(a, np.ndarray) and getattr(a, "is_cuda", False)


class FiniteChem:
    """Finite-rate chemistry on one GPU (mechanism: 'h2' | 'gri30' | 'dme39')."""

    def __init__(self, mech: str, rtol: float = 1e-6, atol: float = 1e-12, max_steps: int = 10000):
        self.lib = load_library()
        self.mech = mech
        self.options = {}  # knobs set through set_option
        self.rtol, self.atol = rtol, atol
        h = ctypes.c_void_p()
        _check(self.lib, self.lib.tgr_chem_create(mech.encode(), rtol, atol, max_steps, ctypes.byref(h)),
               "tgr_chem_create")
        self._h = h
        info = _Info()
        _check(self.lib, self.lib.tgr_chem_mech_info(h, ctypes.byref(info)), "mech_info")
        self.info = {n: getattr(info, n) for n, _ in _Info._fields_}
        self.nsp = info.nsp
        self.neq = info.nsp + 1
        buf = ctypes.create_string_buffer(64)
        names = []
        for k in range(self.nsp):
            _check(self.lib, self.lib.tgr_chem_species_name(h, k, buf, 64), "species_name")
            names.append(buf.value.decode())
        self.species_names = names
        W = np.zeros(self.nsp)
        _check(self.lib, self.lib.tgr_chem_molar_mass(h, W.ctypes.data_as(ctypes.POINTER(ctypes.c_double))),
               "molar_mass")
        self.molar_mass = W

    def close(self):
        if getattr(self, "_h", None):
            self.lib.tgr_chem_destroy(self._h)
            self._h = None

    def __del__(self):
        try:
            self.close()
        except Exception:
            pass

    def set_option(self, key: str, value):
        """Integer knobs ("grid", "rhs_mapping", "step_mapping", "step_waves", "props_mapping",
        "diff_flux_mb", "jacobian",
        "max_order", "max_steps",
        "surr_nsub", "surr_guess", "surr_newton_max", "surr_probe", "surr_adaptive", "surr_max_att", "surr_max_jac",
        "surr_mode", "surr_split_jac") or real ones (REAL_OPTIONS)."""
        if key in REAL_OPTIONS:
            _check(self.lib, self.lib.tgr_chem_set_option_real(self._h, key.encode(), float(value)), "set_option")
        else:
            _check(self.lib, self.lib.tgr_chem_set_option(self._h, key.encode(), int(value)), "set_option")
        self.options[key] = value

    def set_surrogate(self, net, in_shift, in_scale, out_scale):
        """Attach a trained tiger_nga_amd.mlp.MLP (None detaches) with its
        input shift/scale (nsp + 2) and output scale (nsp + 1)."""
        self._net = net
        if net is None:
            _check(self.lib, self.lib.tgr_chem_set_surrogate(self._h, None, None, None, None), "set_surrogate")
            return
        fs = np.ascontiguousarray(in_shift, dtype=np.float32)
        fc = np.ascontiguousarray(in_scale, dtype=np.float32)
        oc = np.ascontiguousarray(out_scale, dtype=np.float64)
        fptr = ctypes.POINTER(ctypes.c_float)
        _check(self.lib, self.lib.tgr_chem_set_surrogate(
            self._h, net._h, fs.ctypes.data_as(fptr), fc.ctypes.data_as(fptr),
            oc.ctypes.data_as(ctypes.POINTER(ctypes.c_double))), "set_surrogate")

    def load_surrogate(self, path: str):
        """Load and attach a network file (the context owns it)."""
        self._net = None
        _check(self.lib, self.lib.tgr_chem_load_surrogate(self._h, path.encode()), "load_surrogate")

    def surrogate_features(self, SC_, grid: Grid, dt: float, X, stream=None):
        """Network inputs of the block's interior cells into X (bfloat16
        [rows, in_pad], rows a multiple of 64 >= cells)."""
        g = grid._c()
        _check(self.lib, self.lib.tgr_chem_surrogate_features_device(self._h, dt, ctypes.byref(g), _ptr(SC_),
                                                                     _ptr(X), X.shape[0], stream), "features")

    def source_chemistry_surrogate(self, RHO_, SC_, grid: Grid, dt: float, p_thermo: float,
                                   p_thermo_old: float | None = None, mask=None, HR_gp=None, chemsrc_gp=None,
                                   stream=None, sync: bool = True):
        """The surrogate-guided step on device tensors or host numpy arrays;
        returns (step stats, guided-solve stats) when sync (always for host
        arrays), else None."""
        if p_thermo_old is None:
            p_thermo_old = p_thermo
        dev = _is_device(SC_)
        self._check_arrays(RHO_, SC_, grid, mask, HR_gp, chemsrc_gp, dev)
        st, ss = _Stats(), _SurrStats()
        g = grid._c()
        if dev:
            rc = self.lib.tgr_chem_source_chemistry_surrogate_device(
                self._h, dt, p_thermo, p_thermo_old, ctypes.byref(g), _ptr(RHO_), _ptr(SC_), _ptr(mask),
                _ptr(HR_gp), _ptr(chemsrc_gp), stream, ctypes.byref(st) if sync else None,
                ctypes.byref(ss) if sync else None)
        else:
            sync = True
            rc = self.lib.tgr_chem_source_chemistry_surrogate(
                self._h, dt, p_thermo, p_thermo_old, ctypes.byref(g), _ptr(RHO_), _ptr(SC_), _ptr(mask),
                _ptr(HR_gp), _ptr(chemsrc_gp), ctypes.byref(st), ctypes.byref(ss))
        _check(self.lib, rc, "source_chemistry_surrogate")
        if not sync:
            return None
        return ({n: getattr(st, n) for n, _ in _Stats._fields_}, {n: getattr(ss, n) for n, _ in _SurrStats._fields_})

    def source_chemistry(self, RHO_, SC_, grid: Grid, dt: float, p_thermo: float, p_thermo_old: float | None = None,
                         mask=None, HR_gp=None, chemsrc_gp=None, stream=None, sync: bool = True):
        """Advance species and T of the interior, non-wall cells by dt in place
        (finitechem.f90:962-1071).  RHO_: (nxo,nyo,nzo) and SC_: (nxo,nyo,nzo,nscalar)
        Fortran-ordered float64; mask: (mx,my) int32 Fortran-ordered (1 = wall)."""
        if p_thermo_old is None:
            p_thermo_old = p_thermo
        dev = _is_device(SC_)
        self._check_arrays(RHO_, SC_, grid, mask, HR_gp, chemsrc_gp, dev)
        st = _Stats()
        g = grid._c()
        if dev:
            rc = self.lib.tgr_chem_source_chemistry_device(
                self._h, dt, p_thermo, p_thermo_old, ctypes.byref(g), _ptr(RHO_), _ptr(SC_), _ptr(mask),
                _ptr(HR_gp), _ptr(chemsrc_gp), stream, ctypes.byref(st) if sync else None)
        else:
            rc = self.lib.tgr_chem_source_chemistry(
                self._h, dt, p_thermo, p_thermo_old, ctypes.byref(g), _ptr(RHO_), _ptr(SC_), _ptr(mask),
                _ptr(HR_gp), _ptr(chemsrc_gp), ctypes.byref(st))
        _check(self.lib, rc, "source_chemistry")
        return {n: getattr(st, n) for n, _ in _Stats._fields_}

    @staticmethod
    def _fortran_ok(a, shape, dtype):
        if isinstance(a, np.ndarray):
            return a.shape == shape and a.dtype == dtype and a.flags.f_contiguous
        # torch tensor: Fortran order means stride[0] == 1 and increasing strides
        st = a.stride()
        exp, acc = [], 1
        for s in shape:
            exp.append(acc)
            acc *= s
        tdt = {np.float64: "torch.float64", np.int32: "torch.int32"}[dtype]
        return tuple(a.shape) == shape and tuple(st) == tuple(exp) and str(a.dtype) == tdt

    def _check_arrays(self, RHO_, SC_, grid, mask, HR_gp, chemsrc_gp, dev):
        sh = grid.shape
        if not self._fortran_ok(RHO_, sh, np.float64):
            raise ValueError("RHO_ must be float64 Fortran-ordered with shape %s" % (sh,))
        if not self._fortran_ok(SC_, sh + (grid.nscalar,), np.float64):
            raise ValueError("SC_ must be float64 Fortran-ordered with shape %s" % (sh + (grid.nscalar,),))
        if mask is not None and not self._fortran_ok(mask, grid.mask_shape, np.int32):
            raise ValueError("mask must be int32 Fortran-ordered with shape %s" % (grid.mask_shape,))
        if HR_gp is not None and not self._fortran_ok(HR_gp, sh, np.float64):
            raise ValueError("HR_gp has the wrong shape/layout")
        if chemsrc_gp is not None and not self._fortran_ok(chemsrc_gp, sh + (3,), np.float64):
            raise ValueError("chemsrc_gp has the wrong shape/layout")
        for a in (RHO_, SC_, mask, HR_gp, chemsrc_gp):
            if a is not None and _is_device(a) != dev:
                raise ValueError("mix of host and device arrays")

    def prodrates(self, C, T, P, stream=None):
        """CDOT[nsp, n] from C[nsp, n] (kmol/m3), T[n], P[n] -- device tensors."""
        import torch
        n = T.shape[0]
        assert C.shape == (self.nsp, n) and C.is_contiguous() and T.is_contiguous() and P.is_contiguous()
        out = torch.empty_like(C)
        _check(self.lib, self.lib.tgr_chem_prodrates_device(self._h, n, _ptr(C), _ptr(T), _ptr(P), _ptr(out),
                                                            stream), "prodrates")
        return out

    def properties(self, SC_, grid: Grid, p_thermo: float, mask=None, Lewis=None, isc_zmix: int = 0, RHO_=None,
                   VISC_=None, DIFF_=None, stream=None):
        """finitechem_density / finitechem_viscosity / finitechem_diffusivity
        (finitechem.f90:324-461) on every cell of the block with mask /= 1, device
        tensors in the step's Fortran layout; outputs that are None are skipped."""
        g = grid._c()
        _check(self.lib, self.lib.tgr_chem_properties_device(
            self._h, p_thermo, ctypes.byref(g), _ptr(SC_), _ptr(mask), _ptr(Lewis), int(isc_zmix), _ptr(RHO_),
            _ptr(VISC_), _ptr(DIFF_), stream), "properties")

    def diffusion(self, dt: float, grid: Grid, metric: dict, RHO_, SC_, DIFF_, mask=None, diff_corr=None,
                  diff_gp=None, src=None, molar: bool = True, gasrad: bool = False, cv: bool = False, stream=None):
        """finitechem_diffusion (finitechem.f90:538-923) on device tensors in
        the step's Fortran layout; metric: st1, st2 and the 15 operator
        tensors of tgr_metric (Fortran-ordered, the reference's extents, see
        tiger_nga_amd.metric).  Writes the interior of diff_corr (..., nsp + 1),
        diff_gp (..., 3) and adds to src (..., nscalar) where given."""
        m = _Metric(int(metric["st1"]), int(metric["st2"]), *[_ptr(metric[n]) for n in METRIC_OPERATORS])
        flags = (1 if molar else 0) | (2 if gasrad else 0) | (4 if cv else 0)
        g = grid._c()
        _check(self.lib, self.lib.tgr_chem_diffusion_device(
            self._h, dt, ctypes.byref(g), ctypes.byref(m), flags, _ptr(RHO_), _ptr(SC_), _ptr(DIFF_), _ptr(mask),
            _ptr(diff_corr), _ptr(diff_gp), _ptr(src), stream), "diffusion")

    def temperature(self, Y, hmix, T0=None, stream=None):
        """(T[n], iters[n]) from mass fractions Y[nsp, n] and mixture enthalpy
        hmix[n] (J/kg) -- device tensors; Newton inversion of the NASA-7 h(T)."""
        import torch
        n = hmix.shape[0]
        assert Y.shape == (self.nsp, n) and Y.is_contiguous() and hmix.is_contiguous()
        T = torch.empty_like(hmix)
        it = torch.empty(n, dtype=torch.int32, device=hmix.device)
        _check(self.lib, self.lib.tgr_chem_temperature_device(self._h, n, _ptr(Y), _ptr(hmix), _ptr(T0), _ptr(T),
                                                               _ptr(it), stream), "temperature")
        return T, it

    def compute_rhs(self, sol, p_gp: float, stream=None):
        """rhs[neq, n] of sol[neq, n] = [rho*Y, rho*T] -- device tensors."""
        import torch
        n = sol.shape[1]
        assert sol.shape == (self.neq, n) and sol.is_contiguous()
        out = torch.empty_like(sol)
        _check(self.lib, self.lib.tgr_chem_rhs_device(self._h, n, p_gp, _ptr(sol), _ptr(out), stream), "rhs")
        return out
