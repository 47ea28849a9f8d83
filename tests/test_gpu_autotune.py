"""Autotuner: every launch shape of the cell kernels gives bitwise the same residual, time
steps and Jacobian (each cell is computed independently of how cells are grouped), the tuner
returns its timing table and keeps a shape from it, and the preconditioner tuner returns a
schedule that reaches the tolerance."""
import numpy as np
import pytest

from fvens_amd import fvx, meshgen, states

pytestmark = pytest.mark.gpu

BCS = [(2, "slipwall"), (4, "farfield")]


def _case():
    import torch
    raw = meshgen.airfoil_omesh(128, 32, 16)
    raw = raw.permuted(fvx.rcm_permutation(raw))
    gm = fvx.Mesh(raw)
    d = fvx.FlowFV(gm, fvx.physics_cfg(Minf=0.7, aoa_deg=2.0, bcs=BCS),
                   fvx.numerics_cfg(flux="HLLC", gradient="LEASTSQUARES", recon="VENKATAKRISHNAN"))
    u = torch.tensor(states.perturbed_freestream(raw, Minf=0.7, aoa_deg=2.0), device="cuda")
    return raw, gm, d, u


def _eval(raw, gm, d, u):
    import torch
    r = torch.zeros_like(u)
    dt = torch.zeros(raw.nelem, dtype=torch.float64, device="cuda")
    d.compute_residual(u, r, True, dt)
    A = fvx.Matrix(gm)
    d.assemble_jacobian(u, A)
    return r.clone(), dt.clone(), A.to_bsr()[2]


def test_results_do_not_depend_on_launch_shape(torch_cuda):
    import torch
    raw, gm, d, u = _case()
    r0, dt0, J0 = _eval(raw, gm, d, u)
    for block in (64, 128, 256, 512):
        for xcd in (False, True):
            d.set_launch("gradients", block, xcd)
            d.set_launch("flux", block, xcd)
            d.set_launch("jacobian", min(block, 256), xcd)
            r, dt, J = _eval(raw, gm, d, u)
            assert torch.equal(r, r0) and torch.equal(dt, dt0), (block, xcd)
            assert np.array_equal(J, J0), (block, xcd)
    # the wave-task form of the flux pass
    for xcd in (False, True):
        d.set_launch("flux_wave", 64, xcd)
        r, dt, J = _eval(raw, gm, d, u)
        assert torch.equal(r, r0) and torch.equal(dt, dt0), ("wave", xcd)


def test_autotuner_keeps_the_fastest_shape(torch_cuda):
    raw, gm, d, u = _case()
    table = d.autotune(u, reps=5)
    # 8 shapes each for the gradient and quad-form flux kernels, the wave-task flux form in
    # both block orders, 6 Jacobian shapes
    assert len(table) == 8 + 8 + 2 + 6
    assert all(t[3] > 0 for t in table)
    for k in ("gradients", "jacobian"):
        best = min((t for t in table if t[0] == k), key=lambda t: t[3])
        assert d.get_launch(k) == (best[1], best[2])
    quad = min((t for t in table if t[0] == "flux"), key=lambda t: t[3])
    best = min((t for t in table if t[0] in ("flux", "flux_wave")), key=lambda t: t[3])
    assert d.get_launch("flux")[0] == quad[1]
    if best[0] == "flux_wave":
        assert d.get_launch("flux_wave") == (64, best[2])
    else:
        assert d.get_launch("flux") == (best[1], best[2]) and d.get_launch("flux_wave")[0] == 0


def test_preconditioner_tuner_returns_a_schedule_that_converges(torch_cuda):
    import torch
    raw, gm, d, u = _case()
    (pc, sweeps), table = d.autotune_pc(u, cfl=200.0, rtol=0.1)
    assert len(table) == 10
    ok = [t for t in table if t[3] > 0]
    assert ok and (pc, sweeps) == min(ok, key=lambda t: t[3])[:2]
    # the chosen schedule solves the system to the tolerance
    A = fvx.Matrix(gm)
    r = torch.zeros_like(u)
    dt = torch.zeros(raw.nelem, dtype=torch.float64, device="cuda")
    dtm = torch.zeros_like(dt)
    d.compute_residual(u, r, True, dt)
    d.assemble_jacobian(u, A)
    d.add_pseudotime(A, dt, 200.0, dtm)
    P = fvx.Preconditioner(gm, pc, sweeps=sweeps)
    P.setup(A)
    x = torch.zeros_like(u)
    assert fvx.linear_solve(A, P, r, x, restart=30, rtol=0.1) < 30


def test_preconditioner_tuner_times_what_a_solve_runs(torch_cuda):
    """Symmetric Gauss-Seidel runs several sweeps per launch once it has been applied a few times, up
    to five times as fast as its first applications on this mesh; the tuner's time is that of a
    solve with a preconditioner that has been in use. Each side takes the least of several
    measurements, and a factor of two stays for what they include besides (set-up, launches)."""
    import time
    import torch
    raw = meshgen.mesh_k1()
    raw = raw.permuted(fvx.rcm_permutation(raw))
    gm = fvx.Mesh(raw)
    d = fvx.FlowFV(gm, fvx.physics_cfg(Minf=0.5, bcs=[(2, "slipwall"), (3, "inflowoutflow"),
                                                      (4, "inflowoutflow")]),
                   fvx.numerics_cfg(flux="ROE", gradient="NONE", order2=False))
    u = torch.tensor(states.perturbed_freestream(raw, Minf=0.5), device="cuda")
    rows = [{t[:2]: t for t in d.autotune_pc(u, cfl=100.0)[1]} for _ in range(4)]
    A = fvx.Matrix(gm)
    r, x = torch.zeros_like(u), torch.zeros_like(u)
    dt = torch.zeros(raw.nelem, dtype=torch.float64, device="cuda")
    d.compute_residual(u, r, True, dt)
    d.assemble_jacobian(u, A)
    d.add_pseudotime(A, dt, 100.0, torch.zeros_like(dt))
    for sweeps in (4, 8, 16):
        P = fvx.Preconditioner(gm, "sgs", sweeps=sweeps)
        t = []
        for _ in range(150):
            torch.cuda.synchronize()
            t0 = time.perf_counter()
            P.setup(A)
            fvx.linear_solve(A, P, r, x, rtol=0.1)
            torch.cuda.synchronize()
            t.append(1e3 * (time.perf_counter() - t0))
        assert min(q["sgs", sweeps][3] for q in rows) <= 2 * min(t[100:]), (sweeps, min(t[100:]))


def _launches(d, u):
    """(flux launches, gradient passes, whether the gradients had a pass of their own)"""
    import torch
    r = torch.zeros_like(u)
    d.profile_enable(True)
    d.compute_residual(u, r)
    torch.cuda.synchronize()
    out = d.profile_read("flux")[1], d.profile_read("gradients")[1], d.profile_read("gradients")[0] > 0
    d.profile_enable(False)
    return out, r


@pytest.mark.parametrize("order", ["rcm", "hilbert"])
def test_launch_settings_can_be_read_and_set_again(torch_cuda, order):
    """The residual in one launch, the choice of a new discretisation, given up for a selected form
    and taken again, also on another discretisation from the settings that were read."""
    import torch
    raw = meshgen.airfoil_omesh(128, 32, 16)
    raw = raw.permuted(fvx.rcm_permutation(raw) if order == "rcm" else fvx.hilbert_permutation(raw))
    gm = fvx.Mesh(raw)

    def disc():
        return fvx.FlowFV(gm, fvx.physics_cfg(Minf=0.7, aoa_deg=2.0, bcs=BCS), fvx.numerics_cfg(
            flux="HLLC", gradient="LEASTSQUARES", recon="VENKATAKRISHNAN"))

    def read(d):
        return {k: d.get_launch(k) for k in ("gradients", "jacobian", "flux", "flux_wave", "residual")}

    def restore(d, got):
        for k in ("gradients", "jacobian", "flux"):
            d.set_launch(k, *got[k])
        for k, block in (("flux_wave", 64), ("residual", 256)):
            if got[k][0] == block:
                d.set_launch(k, *got[k])

    u = torch.tensor(states.perturbed_freestream(raw, Minf=0.7, aoa_deg=2.0), device="cuda")
    d = disc()
    new = read(d)
    assert new["residual"] == (256, True)
    assert new["flux_wave"][0] == (64 if order == "hilbert" else 0)
    one, r0 = _launches(d, u)
    assert one == (1, 1, False)
    settings = [new]
    for form, block in (("flux", 128), ("flux_wave", 64)):
        d.set_launch(form, block, False)
        assert d.get_launch("residual")[0] == 0 and d.get_launch(form) == (block, False)
        got, r = _launches(d, u)
        assert got == (1, 1, True) and torch.equal(r, r0)
        settings.append(read(d))
    restore(d, new)
    assert read(d) == new and _launches(d, u)[0] == one
    for s in settings:
        e = disc()
        restore(e, s)
        assert read(e) == s
        got, r = _launches(e, u)
        assert got == (one if s is new else (1, 1, True)) and torch.equal(r, r0)
    with pytest.raises(fvx.FvxError):
        d.set_launch("residual", 64)
    # the tuner keeps the library's choice or a form of its table, and says which
    d.autotune(u, reps=3)
    assert _launches(d, u)[0] == (one if d.get_launch("residual")[0] == 256 else (1, 1, True))
