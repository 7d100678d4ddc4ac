"""The vector-Jacobian product of fe() at the edges of its kernels: lines of three and four
cells (every ghost row adds to an end row, periodic stencils wrap onto themselves), columns
that do not fill a wave, several segments per column, each tracer count and each pair of
boundary kinds, against the CPU oracle (1e-10 of a component's norm, the bound of the other
tests of this product); and tracers of wbar in the same memory as an input's, which gives the
same bits as separate arrays."""
import importlib.util
import os

import numpy as np
import pytest

import orc
from conftest import PKG, normwise_err

spec = importlib.util.spec_from_file_location("mvd_problems", os.path.join(PKG, "problems.py"))
problems = importlib.util.module_from_spec(spec)
spec.loader.exec_module(problems)

pytestmark = pytest.mark.gpu
TOL = 1e-10
PER = (0,) * 6


def states(dims, nchem, seed=3):
    nx, ny, nz = dims
    w = problems.smooth_state(nx, ny, nz, nchem, seed=seed)
    rng = np.random.default_rng(seed + 1)
    ncell = nx * ny * nz
    v = [rng.standard_normal(ncell) for _ in range(5)] + \
        [rng.standard_normal(max(nchem, 1) * ncell)]
    return w, v


@pytest.mark.parametrize("dims,nchem,bc", [
    ((3, 3, 3), 10, PER), ((3, 3, 3), 1, (1, 3, 3, 1, 1, 1)), ((4, 3, 5), 6, (3, 3, 0, 0, 1, 3)),
    ((3, 40, 4), 2, (0, 0, 3, 1, 1, 3)), ((4, 5, 50), 10, (1, 1, 3, 3, 0, 0)),
    ((130, 3, 3), 4, (3, 1, 1, 1, 3, 3)), ((67, 4, 3), 1, PER), ((65, 18, 4), 0, (3, 1, 0, 0, 1, 3)),
    ((33, 17, 19), 10, (1, 3, 3, 1, 0, 0)), ((5, 66, 3), 0, PER), ((31, 3, 34), 6, (0, 0, 1, 1, 3, 1)),
    ((200, 4, 4), 10, (0, 0, 3, 3, 1, 1))])
def test_edges(mvd, torch_gpu, dims, nchem, bc):
    torch = torch_gpu
    print(f"[fe vjp edges] dims={dims} nchem={nchem} bc={bc}", flush=True)
    w, v = states(dims, nchem)
    ref = orc.fe_vjp(orc.make_grid(*dims, nchem, bc), w, v)
    ctx = mvd.Context(mvd.make_params(*dims, nchem, bc))
    wd = [torch.from_numpy(a).to("cuda") for a in w]
    vd = [torch.from_numpy(a).to("cuda") for a in v]
    if nchem == 0:
        wd[5] = vd[5] = None
    wb = [torch.full_like(a, float("nan")) for a in wd[:5]] + \
         [torch.full_like(wd[5], float("nan")) if nchem else None]
    ctx.fe_vjp(wd, vd, wb)
    for q in range(5):
        assert normwise_err(wb[q].cpu().numpy(), ref[q]) <= TOL, q
    if nchem:
        got, r = wb[5].cpu().numpy().reshape(-1, nchem), ref[5].reshape(-1, nchem)
        for s in range(nchem):
            assert normwise_err(got[:, s], r[:, s]) <= TOL, ("chem", s)
    ctx.close()


@pytest.mark.parametrize("which", ["w", "v"])
def test_tracers_in_place(mvd, torch_gpu, which):
    torch = torch_gpu
    dims, nchem, bc = (9, 20, 7), 6, (0, 0, 1, 3, 3, 1)
    print(f"[fe vjp in place] {which}", flush=True)
    w, v = states(dims, nchem)
    ctx = mvd.Context(mvd.make_params(*dims, nchem, bc))
    wd = [torch.from_numpy(a).to("cuda") for a in w]
    vd = [torch.from_numpy(a).to("cuda") for a in v]
    ref = [torch.empty_like(a) for a in wd]
    ctx.fe_vjp(wd, vd, ref)
    out = [torch.empty_like(a) for a in wd[:5]] + [wd[5] if which == "w" else vd[5]]
    ctx.fe_vjp(wd, vd, out)
    assert all(torch.equal(a, b) for a, b in zip(out, ref))
    ctx.close()
