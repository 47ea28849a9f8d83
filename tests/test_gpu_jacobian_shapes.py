"""Jacobian assembly at the edges of its workgroups: cell counts that leave a workgroup nearly
empty or just full, every workgroup size, every flux with a Jacobian, boundary faces on both even
and odd local faces. Each shape equals the others bitwise and the oracle to 1e-12 of the row scale
(the parity bound of the other Jacobian tests: the same derivative in another operation order)."""
import numpy as np
import pytest

import pyoracle as po
from fvens_amd import fvx, meshgen, states

pytestmark = pytest.mark.gpu

BCS = [(2, "slipwall"), (3, "inflowoutflow"), (4, "extrapolation")]
VISC = [(2, "isothermalwall", (0.1, 1.05)), (3, "inflowoutflow"), (4, "inflowoutflow")]


@pytest.mark.parametrize("nx,ny,nsplit", [(1, 1, 0), (4, 4, 0), (17, 1, 0), (11, 3, 0), (9, 5, 2)])
@pytest.mark.parametrize("flux", ["ROE", "HLLC", "HLL", "LLF", "AUSM"])
@pytest.mark.parametrize("viscous", [False, True])
def test_jacobian_shapes_match_the_oracle(torch_cuda, nx, ny, nsplit, flux, viscous):
    import torch
    raw = meshgen.gaussian_bump(nx, ny, nsplit)
    phys = dict(Minf=0.5, bcs=VISC if viscous else BCS)
    if viscous:
        phys.update(Reinf=5000.0, Pr=0.72, Tinf=288.15, viscous=True)
    gm = fvx.Mesh(raw)
    d = fvx.FlowFV(gm, fvx.physics_cfg(**phys), fvx.numerics_cfg(flux=flux))
    u = states.perturbed_freestream(raw, Minf=0.5)
    ut = torch.tensor(u, device="cuda")
    A = fvx.Matrix(gm, "f64")
    got = []
    for block in (64, 128, 256):
        d.set_launch("jacobian", block, True)
        d.assemble_jacobian(ut, A)
        got.append(A.to_bsr())
    rp, ci, v = got[0]
    assert all(np.array_equal(v, g[2]) for g in got[1:])
    rpo, cio, vo = po.Disc(po.Mesh(raw), po.make_config(flux=flux, **phys)).jacobian(u)
    assert np.array_equal(rp, rpo) and np.array_equal(ci, cio)
    for i in range(raw.nelem):
        s = slice(rp[i], rp[i + 1])
        assert np.abs(v[s] - vo[s]).max() <= 1e-12 * np.abs(vo[s]).max()
