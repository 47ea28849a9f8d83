"""Residual on the smallest meshes against the oracle.

A single quadrilateral (every face a boundary face, no interior face), two triangles (one
interior face), and small ragged triangle/quadrilateral mixes whose wave-task cell groups are
far from full (fewer tasks than lanes, a last group of a few cells). For the first-order, the
unlimited Green-Gauss and the limited least-squares configurations the residual matches the
oracle per cell (1e-12 of the local flux scale) and the time steps to 1e-12, and the
quad-per-cell and wave-task forms of the flux pass give bitwise equal results
(FlowFV::compute_residual, src/spatial/flow_spatial.cpp:488-816).
"""
import numpy as np
import pytest

import pyoracle as po
from fvens_amd import fvx, meshgen, states

pytestmark = pytest.mark.gpu

BUMP_BCS = [(2, "slipwall"), (3, "inflowoutflow"), (4, "inflowoutflow")]
MESHES = [(1, 1, 0), (1, 1, 1), (3, 2, 1), (5, 3, 2), (7, 5, 0)]
CONFIGS = {
    "first": dict(flux="ROE", gradient="NONE", order2=False),
    "gg": dict(flux="ROE", gradient="GREENGAUSS", recon="NONE"),
    "wls_venkat": dict(flux="HLLC", gradient="LEASTSQUARES", recon="VENKATAKRISHNAN",
                       limiter_param=5.0),
}


@pytest.mark.parametrize("cfg", sorted(CONFIGS))
@pytest.mark.parametrize("shape", MESHES, ids=lambda s: "x".join(map(str, s)))
def test_smallest_meshes_match_the_oracle(torch_cuda, shape, cfg):
    import torch
    raw = meshgen.gaussian_bump(*shape)
    num = CONFIGS[cfg]
    phys = dict(Minf=0.5, bcs=BUMP_BCS)
    u = states.perturbed_freestream(raw, Minf=0.5, L=3.0)
    od = po.Disc(po.Mesh(raw), po.make_config(**phys, **num))
    r_ref, dt_ref = od.residual(u)
    scale = np.maximum(np.abs(r_ref), od.flux_magnitude(u))
    disc = fvx.FlowFV(fvx.Mesh(raw), fvx.physics_cfg(**phys), fvx.numerics_cfg(**num))
    ut = torch.tensor(u, device="cuda")
    out = []
    for form, block in (("flux", 256), ("flux_wave", 64)):
        disc.set_launch(form, block, True)
        r = torch.zeros((raw.nelem, 4), dtype=torch.float64, device="cuda")
        dt = torch.zeros(raw.nelem, dtype=torch.float64, device="cuda")
        disc.compute_residual(ut, r, True, dt)
        torch.cuda.synchronize()
        rel = np.abs(r.cpu().numpy() - r_ref) / scale
        assert rel.max() <= 1e-12, (form, rel.max())
        assert np.allclose(dt.cpu().numpy(), dt_ref, rtol=1e-12, atol=0), form
        out.append((r, dt))
    assert torch.equal(out[0][0], out[1][0]) and torch.equal(out[0][1], out[1][1])


@pytest.mark.parametrize("shape", MESHES, ids=lambda s: "x".join(map(str, s)))
def test_smallest_meshes_jacobian_and_linear_solves(torch_cuda, shape):
    """The assembled Jacobian (src/spatial/flow_spatial.cpp:818-1040) matches the oracle's
    block by block (1e-12 of the row scale) with the same sparsity; with the pseudo-time term
    added, FGMRES(31) with multicolour SGS and ILU(0) (4 sweeps; and block Jacobi on the smallest meshes)
    reaches a relative residual of 1e-10, checked with a dense product (one colour on the
    one-cell mesh)."""
    import torch
    raw = meshgen.gaussian_bump(*shape)
    n = raw.nelem
    phys = dict(Minf=0.5, bcs=BUMP_BCS)
    num = dict(flux="ROE", gradient="LEASTSQUARES", recon="VANALBADA")
    od = po.Disc(po.Mesh(raw), po.make_config(**phys, **num))
    gm = fvx.Mesh(raw)
    gd = fvx.FlowFV(gm, fvx.physics_cfg(**phys), fvx.numerics_cfg(**num))
    u = states.perturbed_freestream(raw, Minf=0.5, L=3.0)
    ut = torch.tensor(u, device="cuda")
    A = fvx.Matrix(gm, "f64")
    gd.assemble_jacobian(ut, A)
    rp, ci, vg = A.to_bsr()
    rpo, cio, vo = od.jacobian(u)
    assert np.array_equal(rp, rpo) and np.array_equal(ci, cio)
    for i in range(n):
        s = slice(rp[i], rp[i + 1])
        assert np.abs(vg[s] - vo[s]).max() <= 1e-12 * np.abs(vo[s]).max(), i
    r = torch.zeros_like(ut)
    dt = torch.zeros(n, dtype=torch.float64, device="cuda")
    dtm = torch.zeros_like(dt)
    gd.compute_residual(ut, r, True, dt)
    gd.add_pseudotime(A, dt, 100.0, dtm)
    rp, ci, v = A.to_bsr()
    D = np.zeros((4 * n, 4 * n))
    for i in range(n):
        for k in range(rp[i], rp[i + 1]):
            D[4 * i:4 * i + 4, 4 * ci[k]:4 * ci[k] + 4] = v[k]
    b = r.cpu().numpy().ravel()
    for kind in ("jacobi", "sgs", "ilu0"):
        P = fvx.Preconditioner(gm, kind, "f64", sweeps=1 if kind == "jacobi" else 4)
        P.setup(A)
        if n == 1:
            assert P.ordering()[1] == 1
        x = torch.zeros_like(r)
        its = fvx.linear_solve(A, P, r, x, restart=31, rtol=1e-10)
        assert 0 < its <= 31, (kind, its)
        res = np.linalg.norm(D @ x.cpu().numpy().ravel() - b) / np.linalg.norm(b)
        # block Jacobi on the larger meshes: 31 iterations fall short of 4 n unknowns
        if res > 1e-9:
            assert kind == "jacobi" and its == 31 and res < 1e-2, (kind, its, res)


def _doublets(nx, ny, cells):
    """A bump mesh with the given quadrilaterals divided in two along a path through a new node in
    their middle: the halves share both faces at that node."""
    raw = meshgen.gaussian_bump(nx, ny, 0)
    inpoel, coords = raw.inpoel.copy(), [raw.coords]
    for i, c in enumerate(cells):
        a, b, cc, d = inpoel[c]
        x = raw.npoin + i
        # off the middle, so that the two shared faces differ in length and normal
        w = np.array([0.4, 0.2, 0.25, 0.15])
        coords.append(w @ raw.coords[[a, b, cc, d]][None])
        inpoel[c] = a, b, cc, x
        inpoel = np.vstack([inpoel, [[a, x, cc, d]]]).astype(np.int32)
    out = meshgen.RawMesh(np.vstack(coords), inpoel,
                          np.concatenate([raw.nnode, np.full(len(cells), 4, np.int32)]).astype(np.int32),
                          raw.bface, raw.btag)
    assert (out.signed_areas() > 0).all()
    return out


@pytest.mark.parametrize("order", ["natural", "rcm", "hilbert"])
@pytest.mark.parametrize("cfg", ["first", "gg", "wls"])
def test_cells_that_share_two_faces(torch_cuda, order, cfg):
    """Residual and time steps in the library's own form against the oracle (to which every face is
    one item of a list), and bitwise in the other forms."""
    import torch
    raw = _doublets(30, 20, [5, 6, 100, 333, 599])
    if order != "natural":
        raw = raw.permuted(fvx.rcm_permutation(raw) if order == "rcm" else fvx.hilbert_permutation(raw))
    num = dict(CONFIGS, wls=dict(flux="HLLC", gradient="LEASTSQUARES", recon="NONE"))[cfg]
    phys = dict(Minf=0.5, bcs=BUMP_BCS)
    u = states.perturbed_freestream(raw, Minf=0.5, L=3.0)
    od = po.Disc(po.Mesh(raw), po.make_config(**phys, **num))
    r_ref, dt_ref = od.residual(u)
    scale = np.maximum(np.abs(r_ref), od.flux_magnitude(u))
    disc = fvx.FlowFV(fvx.Mesh(raw), fvx.physics_cfg(**phys), fvx.numerics_cfg(**num))
    ut = torch.tensor(u, device="cuda")
    out = []
    for form, block in (("residual", 256), ("flux", 256), ("flux_wave", 64)):
        disc.set_launch(form, block, True)
        r = torch.zeros((raw.nelem, 4), dtype=torch.float64, device="cuda")
        dt = torch.zeros(raw.nelem, dtype=torch.float64, device="cuda")
        disc.compute_residual(ut, r, True, dt)
        out.append((r, dt))
    rel = np.abs(out[0][0].cpu().numpy() - r_ref) / scale
    assert rel.max() <= 1e-12, rel.max()
    assert np.allclose(out[0][1].cpu().numpy(), dt_ref, rtol=1e-12, atol=0)
    for r, dt in out[1:]:
        assert torch.equal(r, out[0][0]) and torch.equal(dt, out[0][1])


def test_reverse_slots_of_cells_that_share_two_faces(torch_cuda):
    """The warm start's network finds, for every slot, the neighbour's slot of the same face."""
    raw = _doublets(30, 20, [5, 6, 100, 333, 599])
    f = fvx.MPNN(fvx.Mesh(raw), 2, 1).features()
    c, k = np.nonzero(f["nbr"] >= 0)
    j, kk = f["nbr"][c, k], f["rev"][c, k]
    assert (f["nbr"][j, kk] == c).all() and (f["rev"][j, kk] == k).all()
