"""Kernel timing: the kernels timed are those an ordinary call runs (the same bits, and their
launches in their slots), on both sides of the limits of the one-launch fe(); on = 2 takes the face
kernels on small grids too, within the 1e-12 of the field norm of the other fe() tests."""
import importlib.util
import os

import pytest

import orc
from conftest import PKG, normwise_err

spec = importlib.util.spec_from_file_location("mvd_problems", os.path.join(PKG, "problems.py"))
problems = importlib.util.module_from_spec(spec)
spec.loader.exec_module(problems)

pytestmark = pytest.mark.gpu
MIXED = (0, 0, 1, 3, 3, 1)


@pytest.mark.parametrize("dims,nchem,box", [
    ((3, 3, 3), 0, True), ((17, 12, 8), 0, True), ((50, 50, 50), 0, True), ((51, 50, 50), 0, False),
    ((3, 3, 3), 1, True), ((8, 4, 4), 2, True), ((9, 5, 5), 10, True), ((7, 3, 9), 6, True),
    ((17, 12, 8), 4, True), ((3, 4, 65), 10, True), ((64, 32, 32), 4, True),
    ((65, 32, 32), 10, False),
])
def test_profile_times_what_runs(mvd, torch_gpu, dims, nchem, box):
    torch = torch_gpu
    print(f"[profile] dims={dims} nchem={nchem}", flush=True)
    w = problems.smooth_state(*dims, nchem=nchem, seed=31, noise=0.02)
    nf = 6 if nchem else 5
    flag, ref = orc.fe(orc.make_grid(*dims, nchem, MIXED), w)
    assert flag == 0
    ctx = mvd.Context(mvd.make_params(*dims, nchem, MIXED))
    wd = [torch.from_numpy(a).to("cuda") for a in w]
    got = []
    for on in (0, 1, 2):
        assert mvd.lib().mvd_profile(ctx.h, on) == 0
        out = [torch.full_like(a, float("nan")) for a in wd]
        for _ in range(2):
            ctx.fe(wd, out)
        got.append(out)
        count = {k: v[1] for k, v in ctx.profile_read().items()}
        boxes = 2 if on == 1 and box else 0
        faces = 2 if on and not boxes else 0
        assert count["fe_box"] == boxes, (on, count)
        assert count["fe_xyface_div"] == count["fe_zface_div"] == faces, (on, count)
        for q in range(nf):
            assert normwise_err(out[q].cpu().numpy(), ref[q]) <= 1e-12, (on, q)
    for q in range(nf):
        assert torch.equal(got[0][q], got[1][q]), q
    ctx.close()
