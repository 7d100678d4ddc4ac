"""fe() on grids that exercise the z kernel's walk up the columns: one chunk of 16 faces, its
edges (15 and 16 cells), several segments per column, and whole columns of several chunks
(grids wide enough to fill the device without cutting columns), with every tracer count's
passes. Against the oracle; tolerance 1e-12 of the field norm, the bound of the other fe()
tests (re-associated FP64 sums of a few hundred terms)."""
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
TOL = 1e-12


@pytest.mark.parametrize("dims,nchem,bc", [
    ((5, 4, 3), 0, (0,) * 6),
    ((17, 3, 14), 0, (1,) * 6),
    ((16, 5, 15), 0, (3,) * 6),
    ((15, 4, 16), 1, (0, 0, 1, 3, 3, 1)),
    ((18, 7, 31), 2, (0,) * 6),
    ((33, 17, 32), 4, (3,) * 6),
    ((20, 16, 47), 6, (1, 3, 0, 0, 3, 1)),
    ((33, 350, 33), 0, (0,) * 6),
    ((17, 520, 16), 10, (3,) * 6),
])
def test_fe_columns(mvd, torch_gpu, dims, nchem, bc):
    torch = torch_gpu
    print(f"[fe columns] dims={dims} nchem={nchem} bc={bc}", flush=True)
    w = problems.smooth_state(*dims, nchem=nchem, seed=23, noise=0.02)
    flag, ref = orc.fe(orc.make_grid(*dims, nchem, bc), w)
    assert flag == 0
    ctx = mvd.Context(mvd.make_params(*dims, nchem, bc))
    wd = [torch.from_numpy(a).to("cuda") for a in w[:5]]
    wd.append(torch.from_numpy(w[5]).to("cuda") if nchem else None)
    out = [torch.full_like(a, float("nan")) if a is not None else None for a in wd]
    ctx.fe(wd, out)
    for q in range(5):
        assert normwise_err(out[q].cpu().numpy(), ref[q]) <= TOL, q
    if nchem:
        got, want = out[5].cpu().numpy().reshape(-1, nchem), ref[5].reshape(-1, nchem)
        for s in range(nchem):
            assert normwise_err(got[:, s], want[:, s]) <= TOL, s
    ctx.close()
