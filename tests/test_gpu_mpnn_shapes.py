"""Warm-start kernels at the edges of their tiles: rows that do not fill a 16-row tile, a 64-row
chunk or a workgroup, one tile in all, triangles (an unused slot per cell), and tiles that hold
the end of one graph and the start of the next.

A value that lands on the other side of a bf16 rounding boundary moves by one unit, 2^-8 of its
size. If that happened to every entry in each of the four layers, outputs and gradients would be
off by 4 x 2^-8 in relative L2 norm; small meshes have too few entries for the dilution that
tighter bounds rely on.
"""
import numpy as np
import pytest

import mpnn_oracle as mo
import pyoracle as po
from fvens_amd import fvx, meshgen, warmstart

pytestmark = pytest.mark.gpu

WALL = 2
TOL = 4 * 2.0 ** -8


# cells: 9, 16, 33 and 65 quads; 60 and 1,035 with triangles
@pytest.mark.parametrize("nx,ny,nsplit", [(3, 3, 0), (4, 4, 0), (11, 3, 0), (13, 5, 0), (12, 4, 1),
                                          (45, 21, 2)])
@pytest.mark.parametrize("ng", [1, 3])
def test_shapes(torch_cuda, nx, ny, nsplit, ng):
    import torch
    raw = meshgen.gaussian_bump(nx, ny, nsplit)
    net = fvx.MPNN(fvx.Mesh(raw), WALL, 4)
    g = mo.graph(po.Mesh(raw), raw, WALL)
    rng = np.random.default_rng(nx + ng)
    w = warmstart.init_params(3, dec_scale=0.3)
    o = 0
    for name, shape in mo.layout():
        n = int(np.prod(shape))
        if name.startswith("b"):
            w[o:o + n] = rng.standard_normal(n).astype(np.float32) * 0.1
        o += n
    mach, aoa = np.array([0.45, 0.62, 0.74])[:ng], np.array([-3.0, 1.25, 5.5])[:ng]
    net.set_params(w)
    net.set_points(mach, aoa)
    y = torch.full((ng, raw.nelem, 4), np.nan, dtype=torch.float32, device="cuda")
    net.predict(y)
    yo, _ = mo.forward(w, g, mach, aoa, quant=True)
    assert np.linalg.norm(y.cpu().numpy() - yo) <= TOL * np.linalg.norm(yo)

    tgt = (rng.standard_normal((4, raw.nelem, 4)) * 0.2).astype(np.float32)
    ids = np.array([2, 0, 3])[:ng]
    grad = torch.full((mo.nparams(),), np.nan, dtype=torch.float32, device="cuda")
    loss = net.gradient(torch.tensor(tgt, device="cuda"), ids, grad)
    gg = grad.cpu().numpy()
    lo, go = mo.loss_and_grad(w, g, mach, aoa, tgt[ids], quant=True)
    assert abs(loss - lo) <= TOL * lo
    o = 0
    for name, shape in mo.layout():
        n = int(np.prod(shape))
        assert np.linalg.norm(gg[o:o + n] - go[o:o + n]) <= TOL * np.linalg.norm(go[o:o + n]), name
        o += n
