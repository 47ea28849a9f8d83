"""Solves one after the other on one discretisation, with other factor precisions and numbers of
instances: each gives, bit for bit, what a fresh discretisation gives. The solves are long
enough that the preconditioner's patches (several sweeps per launch) serve the first of them, at
sizes where the patches of the precisions hold different numbers of cells."""
import numpy as np
import pytest

from fvens_amd import fvx, meshgen, states, train_warmstart as tw, warmstart as ws

pytestmark = pytest.mark.gpu

BUMP = [(2, "slipwall"), (3, "inflowoutflow"), (4, "inflowoutflow")]
AIRFOIL = [(2, "slipwall"), (4, "farfield")]
FIRST = dict(flux="ROE", gradient="NONE", order2=False)
# tight linear solves: about 40 applications of 16 sweeps in three steps
SOLVE = dict(cflinit=100.0, cflfin=100.0, tol=1e-12, maxiter=3, krylov_rtol=1e-4, pc_sweeps=16)
PRECISIONS = {"f64": dict(pc_precision="f64", jac_precision="f64"),
              "f32": dict(pc_precision="f32", jac_precision="f32"),
              "bf16": dict(pc_precision="bf16", jac_precision="f32")}


def _airfoil(nx, ny):
    raw = meshgen.airfoil_omesh(nx, ny, ny // 2)
    return raw.permuted(fvx.rcm_permutation(raw))


def _disc(gm, bcs):
    return fvx.FlowFV(gm, fvx.physics_cfg(Minf=0.5, aoa_deg=1.0, bcs=bcs), fvx.numerics_cfg(**FIRST))


def _solve(d, prec, ninst):
    """Three steps: of one instance with the single solver, of several as a batch."""
    import torch
    kw = dict(SOLVE, **PRECISIONS[prec])
    if ninst == 1:
        u = torch.tensor(d.freestream(), device="cuda").expand(d.mesh.nelem, 4).contiguous()
        st = [d.steady_solve(u, raise_on_failure=False, **kw)]
    else:
        b = fvx.Batch(d, np.linspace(0.4, 0.6, ninst), np.linspace(-1.0, 2.0, ninst))
        u = ws.freestream_states(b)
        st = b.steady_solve(u, **kw)
    assert all(s["steps"] == 3 for s in st), st
    assert torch.isfinite(u).all()
    return u, [s["lin_iters"] for s in st]


def _sequence(raw, bcs, solves):
    import torch
    gm = fvx.Mesh(raw)
    d = _disc(gm, bcs)
    for prec, ninst in solves:
        u, its = _solve(d, prec, ninst)
        uf, itsf = _solve(_disc(gm, bcs), prec, ninst)
        assert its == itsf and torch.equal(u, uf), (prec, ninst, its, itsf)


@pytest.mark.parametrize("shape", [(300, 75), (512, 128)])       # 33,600 and 98,304 cells
@pytest.mark.parametrize("precs", [("f32", "f64"), ("bf16", "f64"), ("f64", "f32"),
                                   ("f32", "bf16", "f64", "bf16")], ids="-".join)
def test_precisions_in_turn(torch_cuda, shape, precs):
    _sequence(_airfoil(*shape), AIRFOIL, [(p, 1) for p in precs])


@pytest.mark.parametrize("solves", [[("f32", 16), ("f64", 2), ("f64", 1)],
                                    [("f64", 1), ("f32", 16), ("f32", 2), ("f64", 1)],
                                    [("bf16", 16), ("f64", 16), ("f32", 1)]],
                         ids=lambda s: "-".join(f"{n}x{p}" for p, n in s))
def test_batches_in_turn(torch_cuda, solves):
    raw = meshgen.mesh_k1()
    _sequence(raw.permuted(fvx.rcm_permutation(raw)), BUMP, solves)


def test_preconditioner_types_in_turn(torch_cuda):
    import torch
    gm = fvx.Mesh(_airfoil(512, 128))
    d = _disc(gm, AIRFOIL)
    for kw in (dict(PRECISIONS["f32"]), dict(PRECISIONS["f64"], pc="ilu0", pc_sweeps=1),
               dict(PRECISIONS["f64"])):
        out = []
        for dd in (d, _disc(gm, AIRFOIL)):
            u = torch.tensor(dd.freestream(), device="cuda").expand(gm.nelem, 4).contiguous()
            st = dd.steady_solve(u, raise_on_failure=False, **dict(SOLVE, **kw))
            out.append((u, st["lin_iters"]))
        assert torch.isfinite(out[0][0]).all()
        assert out[0][1] == out[1][1] and torch.equal(out[0][0], out[1][0]), kw


def test_fallback_with_no_solve_before_it(torch_cuda):
    """The warm start's fallback: FP32 solves that fail, then the same points in FP64 on the same
    discretisations, without an FP64 solve before; it equals the plain solve on fresh ones."""
    import torch
    raw = meshgen.mesh_k2()
    gm = fvx.Mesh(raw.permuted(fvx.rcm_permutation(raw)))
    mach, aoa = np.array([0.45, 0.55]), np.array([0.5, 1.5])
    pc32, pc64, starter, main = tw.solver_settings(16, 3, 1e-8)
    starter = dict(starter, maxiter=4)
    net = fvx.MPNN(gm, 2, 2)
    net.set_params(np.zeros(fvx.MPNN.nparams(), np.float32))      # predicts the free stream
    d1, d2 = tw.discretisations(gm)
    b = fvx.Batch(d2, mach, aoa)
    norms = b.residual_norms(ws.freestream_states(b))
    u, res = tw.solve_with_fallback(net, d1, d2, mach, aoa, pc32, pc64, starter, main, norms)
    assert all(r["path"] == "fallback" for r in res)
    f1, f2 = tw.discretisations(gm)
    up, _ = ws.solve_batch(f2, mach, aoa, starter=f1, starter_cfg=dict(starter, **pc64),
                           main_cfg=dict(main, **pc64), norms=norms)
    assert torch.isfinite(u).all() and torch.equal(u, up)
