"""The wave-task form of the face-flux pass against the oracle.

Each wave64 owns a group of neighbouring cells whose faces make at most 64 tasks and evaluates
every face touching them once (an internal face for both cells); each cell sums its four face
slots in the quad-per-cell form's order. It applies to inviscid first-order and linear
reconstruction. Checked against the oracle's residual (per cell within 1e-12 of the local flux
scale) and time steps: on the bump for every flux (second order with the Venkatakrishnan limiter
and first order), on the airfoil in RCM, Hilbert and natural order, for a batch of operating
points against single evaluations, and bitwise reproducible run to run. Both forms evaluate each
face flux from the face's left and right states and sum a cell's four slots in the same order,
so their residuals and time steps are bitwise equal. Where a caller may select the wave form and the
cell order packs at least 24 cells per group, a new discretisation reports it as selected (what
the library runs of its own choice is tested in test_gpu_flux_groups.py).
"""
import numpy as np
import pytest

import pyoracle as po
from fvens_amd import fvx, meshgen, states

pytestmark = pytest.mark.gpu

BUMP_BCS = [(2, "slipwall"), (3, "inflowoutflow"), (4, "inflowoutflow")]
AIRFOIL_BCS = [(2, "slipwall"), (4, "farfield")]


def _check(raw, phys, num, u):
    import torch
    od = po.Disc(po.Mesh(raw), po.make_config(**phys, **num))
    r_ref, dt_ref = od.residual(u)
    scale = np.maximum(np.abs(r_ref), od.flux_magnitude(u))
    disc = fvx.FlowFV(fvx.Mesh(raw), fvx.physics_cfg(**phys), fvx.numerics_cfg(**num))
    disc.set_launch("flux_wave", 64, True)
    assert disc.get_launch("flux_wave")[0] == 64
    ut = torch.tensor(u, device="cuda")
    out = []
    for _ in range(2):
        r = torch.full((raw.nelem, 4), 0.25, dtype=torch.float64, device="cuda")
        dt = torch.zeros(raw.nelem, dtype=torch.float64, device="cuda")
        disc.compute_residual(ut, r, True, dt)
        torch.cuda.synchronize()
        out.append((r - 0.25, dt))
    assert torch.equal(out[0][0], out[1][0]) and torch.equal(out[0][1], out[1][1])
    rel = np.abs(out[0][0].cpu().numpy() - r_ref) / scale
    assert rel.max() <= 1e-12, rel.max()
    assert np.allclose(out[0][1].cpu().numpy(), dt_ref, rtol=1e-12, atol=0)


@pytest.mark.parametrize("flux", ["ROE", "HLLC", "HLL", "LLF", "AUSM", "AUSMPLUS", "VANLEER"])
def test_wave_tasks_match_the_oracle_on_the_bump(torch_cuda, flux):
    raw = meshgen.mesh_k1()
    u = states.perturbed_freestream(raw, Minf=0.5, L=3.0)
    phys = dict(Minf=0.5, bcs=BUMP_BCS)
    _check(raw, phys, dict(flux=flux, gradient="LEASTSQUARES", recon="VENKATAKRISHNAN",
                           limiter_param=5.0), u)
    _check(raw, phys, dict(flux=flux, gradient="NONE", order2=False), u)


@pytest.mark.parametrize("order", ["rcm", "hilbert", "natural"])
def test_wave_tasks_match_the_oracle_on_the_airfoil(torch_cuda, order):
    raw = meshgen.mesh_k2()
    if order != "natural":
        raw = raw.permuted(fvx.rcm_permutation(raw) if order == "rcm"
                           else fvx.hilbert_permutation(raw))
    u = states.perturbed_freestream(raw, Minf=0.8, aoa_deg=1.25, L=1.0)
    _check(raw, dict(Minf=0.8, aoa_deg=1.25, bcs=AIRFOIL_BCS),
           dict(flux="HLLC", gradient="LEASTSQUARES", recon="VENKATAKRISHNAN",
                limiter_param=5.0), u)


def test_wave_tasks_for_a_batch_match_single_evaluations(torch_cuda):
    import torch
    raw = meshgen.mesh_k1()
    num = dict(flux="ROE", gradient="GREENGAUSS", recon="NONE")
    disc = fvx.FlowFV(fvx.Mesh(raw), fvx.physics_cfg(Minf=0.5, bcs=BUMP_BCS),
                      fvx.numerics_cfg(**num))
    disc.set_launch("flux_wave", 64, True)
    mach, aoa = np.array([0.3, 0.5, 0.7]), np.array([0.0, 2.0, -1.0])
    b = fvx.Batch(disc, mach, aoa)
    u = np.stack([states.perturbed_freestream(raw, Minf=m, aoa_deg=a, L=3.0, seed=7 + i)
                  for i, (m, a) in enumerate(zip(mach, aoa))])
    ut = torch.tensor(u, device="cuda")
    r = torch.zeros_like(ut)
    dt = torch.zeros((3, raw.nelem), dtype=torch.float64, device="cuda")
    b.compute_residual(ut, r, True, dt)
    torch.cuda.synchronize()
    for i in range(3):
        di = fvx.FlowFV(fvx.Mesh(raw), fvx.physics_cfg(Minf=mach[i], aoa_deg=aoa[i],
                                                       bcs=BUMP_BCS), fvx.numerics_cfg(**num))
        di.set_launch("flux_wave", 64, True)
        ri = torch.zeros_like(ut[i])
        dti = torch.zeros(raw.nelem, dtype=torch.float64, device="cuda")
        di.compute_residual(ut[i].contiguous(), ri, True, dti)
        torch.cuda.synchronize()
        assert torch.equal(r[i], ri) and torch.equal(dt[i], dti), i


def _both_forms(raw, phys, num, u, instances=None):
    import torch
    disc = fvx.FlowFV(fvx.Mesh(raw), fvx.physics_cfg(**phys), fvx.numerics_cfg(**num))
    ut = torch.tensor(u, device="cuda")
    out = []
    for form in ("flux", "flux_wave"):
        disc.set_launch(form, 256 if form == "flux" else 64, True)
        r = torch.full((raw.nelem, 4), 0.5, dtype=torch.float64, device="cuda")
        dt = torch.zeros(raw.nelem, dtype=torch.float64, device="cuda")
        disc.compute_residual(ut, r, True, dt)
        torch.cuda.synchronize()
        out.append((r, dt))
    assert torch.equal(out[0][0], out[1][0]) and torch.equal(out[0][1], out[1][1])


@pytest.mark.parametrize("flux", ["ROE", "HLLC", "AUSM", "VANLEER"])
@pytest.mark.parametrize("recon", ["VENKATAKRISHNAN", "BARTHJESPERSEN", "NONE", "WENO", "first"])
def test_wave_and_quad_forms_are_bitwise_equal_on_the_bump(torch_cuda, flux, recon):
    raw = meshgen.mesh_k1()
    u = states.perturbed_freestream(raw, Minf=0.5, L=3.0)
    num = (dict(flux=flux, gradient="NONE", order2=False) if recon == "first" else
           dict(flux=flux, gradient="LEASTSQUARES", recon=recon, limiter_param=5.0))
    _both_forms(raw, dict(Minf=0.5, bcs=BUMP_BCS), num, u)


def test_wave_and_quad_forms_are_bitwise_equal_on_the_airfoil(torch_cuda):
    raw = meshgen.mesh_k2()
    raw = raw.permuted(fvx.hilbert_permutation(raw))
    u = states.perturbed_freestream(raw, Minf=0.8, aoa_deg=1.25, L=1.0)
    _both_forms(raw, dict(Minf=0.8, aoa_deg=1.25, bcs=AIRFOIL_BCS),
                dict(flux="HLLC", gradient="LEASTSQUARES", recon="VENKATAKRISHNAN",
                     limiter_param=5.0), u)


def test_the_form_is_selected_by_the_cell_order(torch_cuda):
    """What fvx_get_launch reports of the wave form on a new discretisation."""
    raw = meshgen.mesh_k2()
    num = dict(flux="HLLC", gradient="LEASTSQUARES", recon="VENKATAKRISHNAN")
    phys = dict(Minf=0.8, aoa_deg=1.25, bcs=AIRFOIL_BCS)
    for order, wave in (("hilbert", True), ("natural", True), ("rcm", False)):
        r = raw if order == "natural" else raw.permuted(
            fvx.rcm_permutation(raw) if order == "rcm" else fvx.hilbert_permutation(raw))
        d = fvx.FlowFV(fvx.Mesh(r), fvx.physics_cfg(**phys), fvx.numerics_cfg(**num))
        assert (d.get_launch("flux_wave")[0] == 64) == wave, order
    # not for MUSCL-Van Albada or viscous flow, whatever the order
    r = raw.permuted(fvx.hilbert_permutation(raw))
    d = fvx.FlowFV(fvx.Mesh(r), fvx.physics_cfg(**phys),
                   fvx.numerics_cfg(flux="HLLC", gradient="LEASTSQUARES", recon="VANALBADA"))
    assert d.get_launch("flux_wave")[0] == 0
    with pytest.raises(fvx.FvxError):
        d.set_launch("flux_wave", 64, True)
    d = fvx.FlowFV(fvx.Mesh(r), fvx.physics_cfg(Minf=0.5, Tinf=288.15, Reinf=5000.0, Pr=0.72,
                                                 viscous=True,
                                                 bcs=[(2, "adiabaticwall"), (4, "farfield")]),
                   fvx.numerics_cfg(**num))
    assert d.get_launch("flux_wave")[0] == 0
    with pytest.raises(fvx.FvxError):
        d.set_launch("flux_wave", 64, True)
    assert d.get_launch("flux_wave")[0] == 0


def test_full_size_hilbert_workload_matches_the_oracle(torch_cuda):
    """The benchmark's residual workload at its full size: the 2048x512 O-mesh (1,572,864 cells)
    in Hilbert order, HLLC + weighted least squares + Venkatakrishnan K=5 at M0.8, 1.25 deg.
    The library does it in one launch; residual and time steps match the oracle per cell (1e-12
    of the local flux scale), repeat bitwise, and equal the wave-task form's and the quad form's
    bitwise."""
    import torch
    raw = meshgen.mesh_k2l()
    raw = raw.permuted(fvx.hilbert_permutation(raw))
    u = states.perturbed_freestream(raw, Minf=0.8, aoa_deg=1.25, L=1.0)
    phys = dict(Minf=0.8, aoa_deg=1.25, bcs=AIRFOIL_BCS)
    num = dict(flux="HLLC", gradient="LEASTSQUARES", recon="VENKATAKRISHNAN", limiter_param=5.0)
    disc = fvx.FlowFV(fvx.Mesh(raw), fvx.physics_cfg(**phys), fvx.numerics_cfg(**num))
    assert disc.get_launch("flux_wave")[0] == 64 and disc.get_launch("residual")[0] == 256
    ut = torch.tensor(u, device="cuda")

    def evaluate():
        r = torch.zeros((raw.nelem, 4), dtype=torch.float64, device="cuda")
        dt = torch.zeros(raw.nelem, dtype=torch.float64, device="cuda")
        disc.compute_residual(ut, r, True, dt)
        torch.cuda.synchronize()
        return r, dt

    r1, dt1 = evaluate()
    r2, dt2 = evaluate()
    assert torch.equal(r1, r2) and torch.equal(dt1, dt2)
    od = po.Disc(po.Mesh(raw), po.make_config(**phys, **num))
    r_ref, dt_ref = od.residual(u)
    scale = np.maximum(np.abs(r_ref), od.flux_magnitude(u))
    rel = np.abs(r1.cpu().numpy() - r_ref) / scale
    assert rel.max() <= 1e-12, rel.max()
    assert np.allclose(dt1.cpu().numpy(), dt_ref, rtol=1e-12, atol=0)
    disc.set_launch("flux_wave", 64, True)
    assert disc.get_launch("residual")[0] == 0
    rw, dtw = evaluate()
    assert torch.equal(r1, rw) and torch.equal(dt1, dtw)
    disc.set_launch("flux", 256, True)
    assert disc.get_launch("flux_wave")[0] == 0
    rq, dtq = evaluate()
    assert torch.equal(r1, rq) and torch.equal(dt1, dtq)
