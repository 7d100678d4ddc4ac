"""The one-launch fe() with tracers (boxes of 8 x 4 x 4 cells): grids at, below and past the
edges of its boxes and of the number of boxes up to which it is taken (512), every boundary rule,
every tracer count, against the oracle to 1e-12 of the field norm (as the other fe() tests). The
same grids with profiling on, which takes the three kernels."""
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
MIXED = (0, 0, 1, 3, 3, 1)


@pytest.mark.parametrize("dims,nchem,bc", [
    ((3, 3, 3), 1, (1,) * 6), ((8, 4, 4), 2, (0,) * 6), ((9, 5, 5), 10, (3,) * 6),
    ((7, 3, 9), 6, MIXED), ((17, 12, 8), 4, (3, 3, 0, 0, 1, 1)), ((3, 4, 65), 10, MIXED),
    ((64, 32, 32), 4, MIXED), ((65, 32, 32), 10, (0,) * 6),
])
@pytest.mark.parametrize("three", [False, True])
def test_fe_box_tracers(mvd, torch_gpu, dims, nchem, bc, three):
    torch = torch_gpu
    print(f"[fe box tracers] dims={dims} nchem={nchem} bc={bc} three={three}", flush=True)
    w = problems.smooth_state(*dims, nchem=nchem, seed=31, noise=0.02)
    flag, ref = orc.fe(orc.make_grid(*dims, nchem, bc), w)
    assert flag == 0
    ctx = mvd.Context(mvd.make_params(*dims, nchem, bc))
    if three:
        ctx.profile()
    wd = [torch.from_numpy(a).to("cuda") for a in w]
    out = [torch.full_like(a, float("nan")) for a in wd]
    ctx.fe(wd, out)
    for q in range(6):
        assert normwise_err(out[q].cpu().numpy(), ref[q]) <= 1e-12, q
    ctx.close()
