"""Residuals in the forms the library chooses by itself: second-order ones in one launch over
patches of cells, first-order, WENO and limited viscous ones with wave tasks from 20,000 cells on,
in RCM orders, whose groups are grown over neighbouring cells, and in Hilbert order. All forms
evaluate gradients and faces from the same states in the same way and add a cell's slots in the
same order, so the results are bitwise equal to the separate passes in quad-per-cell form."""
import numpy as np
import pytest

from fvens_amd import fvx, meshgen, states

pytestmark = pytest.mark.gpu

INVISCID = [(2, "slipwall"), (4, "farfield")]
VISCOUS = [(4, "inflowoutflow"), (2, "adiabaticwall", (0.0, 0.0))]
FORMS = [("ROE", "NONE", "first"), ("HLLC", "LEASTSQUARES", "VENKATAKRISHNAN"),
         ("ROE", "LEASTSQUARES", "VANALBADA"), ("AUSM", "GREENGAUSS", "NONE"),
         ("LLF", "LEASTSQUARES", "WENO")]


def _num(flux, grad, recon):
    return (fvx.numerics_cfg(flux=flux, gradient="NONE", order2=False) if recon == "first"
            else fvx.numerics_cfg(flux=flux, gradient=grad, recon=recon))


def _phys(viscous, M=0.5, a=1.0):
    extra = dict(Tinf=288.15, Reinf=5000.0, Pr=0.72, viscous=True) if viscous else {}
    return fvx.physics_cfg(Minf=M, aoa_deg=a, bcs=VISCOUS if viscous else INVISCID, **extra)


# triangles outside quadrilaterals, and quadrilaterals only; 24,640 and 20,007 cells
@pytest.mark.parametrize("shape", [(224, 80, 30), (247, 81, 0)])
@pytest.mark.parametrize("viscous", [False, True])
@pytest.mark.parametrize("form", FORMS, ids=lambda f: f[2])
def test_single(torch_cuda, shape, viscous, form):
    import torch
    raw = meshgen.airfoil_omesh(shape[0], shape[1], shape[2])
    raw = raw.permuted(fvx.rcm_permutation(raw))
    assert raw.nelem >= 20000
    d = fvx.FlowFV(fvx.Mesh(raw), _phys(viscous), _num(*form))
    u = torch.tensor(states.perturbed_freestream(raw, Minf=0.5, aoa_deg=1.0), device="cuda")
    out = []
    for quad in (False, True):
        if quad:
            d.set_launch("flux", 256, True)
        for steps in (True, False):
            r = torch.full_like(u, 0.5)
            dt = torch.zeros(raw.nelem, dtype=torch.float64, device="cuda")
            d.compute_residual(u, r, steps, dt if steps else None)
            out.append((r, dt))
    for a, b in zip(out[:2], out[2:]):
        assert torch.isfinite(a[0]).all()
        assert torch.equal(a[0], b[0]) and torch.equal(a[1], b[1])


# a patch with one cell, one that is the whole mesh, one task too many, triangles
@pytest.mark.parametrize("shape", [(1, 1, 0), (10, 10, 0), (11, 11, 0), (45, 21, 2), (40, 33, 33)])
@pytest.mark.parametrize("order", ["rcm", "hilbert"])
@pytest.mark.parametrize("viscous", [False, True])
@pytest.mark.parametrize("form", FORMS[1:4] + [("VANLEER", "GREENGAUSS", "BARTHJESPERSEN")],
                         ids=lambda f: f[2])
def test_patches(torch_cuda, shape, order, viscous, form):
    import torch
    raw = meshgen.gaussian_bump(*shape)
    raw = raw.permuted(fvx.rcm_permutation(raw) if order == "rcm" else fvx.hilbert_permutation(raw))
    extra = dict(Tinf=288.15, Reinf=5000.0, Pr=0.72, viscous=True) if viscous else {}
    bcs = [(2, "adiabaticwall", (0.0, 0.0)) if viscous else (2, "slipwall"),
           (3, "inflowoutflow"), (4, "inflowoutflow")]
    d = fvx.FlowFV(fvx.Mesh(raw), fvx.physics_cfg(Minf=0.5, bcs=bcs, **extra), _num(*form))
    u = torch.tensor(states.perturbed_freestream(raw, Minf=0.5, L=3.0), device="cuda")
    out = []
    for _ in range(2):
        r = torch.full_like(u, 0.5)
        dt = torch.zeros(raw.nelem, dtype=torch.float64, device="cuda")
        d.compute_residual(u, r, True, dt)
        out.append((r, dt))
        d.set_launch("flux", 256, True)
    assert torch.isfinite(out[0][0]).all()
    assert torch.equal(out[0][0], out[1][0]) and torch.equal(out[0][1], out[1][1])


def _same(a, b):
    """The same values, NaN where the other is NaN (its sign and payload are not promised)."""
    return bool(((a == b) | (a.isnan() & b.isnan())).all())


# one patch, several, and enough cells for wave tasks
@pytest.mark.parametrize("shape", [(16, 4, 2), (61, 23, 9), (247, 81, 0)])
@pytest.mark.parametrize("viscous", [False, True])
@pytest.mark.parametrize("form", FORMS + [("HLLC", "GREENGAUSS", "BARTHJESPERSEN")],
                         ids=lambda f: f[2])
def test_non_finite_states(torch_cuda, shape, viscous, form):
    """Cells of NaN, infinities, zero density and negative pressure, inside and at boundaries."""
    import torch
    raw = meshgen.airfoil_omesh(*shape)
    raw = raw.permuted(fvx.rcm_permutation(raw))
    d = fvx.FlowFV(fvx.Mesh(raw), _phys(viscous), _num(*form))
    u = torch.tensor(states.perturbed_freestream(raw, Minf=0.5, aoa_deg=1.0), device="cuda")
    n = raw.nelem
    u[0, 2] = float("nan")
    u[n // 5, 1] = float("inf")
    u[n // 4, 3] = -float("inf")
    u[n // 3, 0] = 0.0
    u[n // 2, 3] = 0.0
    u[2 * n // 3] = float("nan")
    out = []
    for quad in (False, True):
        if quad:
            d.set_launch("flux", 256, True)
        r = torch.full_like(u, 0.5)
        dt = torch.zeros(n, dtype=torch.float64, device="cuda")
        d.compute_residual(u, r, True, dt)
        out.append((r, dt))
    assert not out[0][0].isfinite().all()
    assert _same(out[0][0], out[1][0]) and _same(out[0][1], out[1][1])


# what a batch does by size in wave tasks: first order, WENO weights, limited viscous terms
@pytest.mark.parametrize("viscous,form", [(False, FORMS[0]), (True, FORMS[0]), (False, FORMS[4]),
                                          (True, FORMS[4]), (True, FORMS[1])],
                         ids=lambda v: v if isinstance(v, bool) else v[2])
def test_batch_in_wave_tasks(torch_cuda, viscous, form):
    _batch(viscous, form)


@pytest.mark.parametrize("viscous", [False, True])
def test_batch(torch_cuda, viscous):
    _batch(viscous, FORMS[2 if viscous else 1])


def _batch(viscous, form):
    """Instances of one batch in the form the library chooses for their number against single
    evaluations in the quad form."""
    import torch
    raw = meshgen.airfoil_omesh(61, 23, 9)
    raw = raw.permuted(fvx.rcm_permutation(raw))
    n = 20000 // raw.nelem + 1
    mach, aoa = np.linspace(0.3, 0.6, n), np.linspace(-2.0, 3.0, n)
    gm = fvx.Mesh(raw)
    d = fvx.FlowFV(gm, _phys(viscous), _num(*form))
    b = fvx.Batch(d, mach, aoa)
    u = torch.tensor(np.stack([states.perturbed_freestream(raw, Minf=m, aoa_deg=a, seed=i)
                               for i, (m, a) in enumerate(zip(mach, aoa))]), device="cuda")
    r, dt = torch.zeros_like(u), torch.zeros(u.shape[:2], dtype=torch.float64, device="cuda")
    b.compute_residual(u, r, True, dt)
    for i in range(n):
        di = fvx.FlowFV(gm, _phys(viscous, mach[i], aoa[i]), _num(*form))
        di.set_launch("flux", 256, True)
        ri, dti = torch.zeros_like(u[i]), torch.zeros_like(dt[i])
        di.compute_residual(u[i].contiguous(), ri, True, dti)
        assert torch.equal(r[i], ri) and torch.equal(dt[i], dti), i
