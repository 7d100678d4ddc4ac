"""The one-launch fe() of small grids (boxes of 8 x 4 x 4 cells) and the explicit evolution
over it: grids at, below and past the edges of its boxes and of the size up to which it is
taken, every boundary rule, against the oracle. fe() to 1e-12 of the field norm (as the other
fe() tests); evolutions to 1e-10 after a few steps, with tables whose last stage is the new
state (no rate evaluated twice) and others (one, three and six stages), below and above that
size; a run in one call equals the same steps in two bitwise."""
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


@pytest.mark.parametrize("dims,bc", [
    ((3, 3, 3), (1,) * 6), ((8, 4, 4), (0,) * 6), ((9, 5, 5), (3,) * 6), ((7, 3, 9), MIXED),
    ((17, 12, 8), MIXED), ((128, 3, 3), (1,) * 6), ((3, 4, 65), (3, 1, 0, 0, 1, 3)),
    ((50, 50, 50), (0,) * 6), ((51, 50, 50), (3,) * 6),
])
def test_fe_box(mvd, torch_gpu, dims, bc):
    torch = torch_gpu
    print(f"[fe box] dims={dims} bc={bc}", flush=True)
    w = problems.smooth_state(*dims, seed=29, noise=0.02)
    flag, ref = orc.fe(orc.make_grid(*dims, 0, bc), w)
    assert flag == 0
    ctx = mvd.Context(mvd.make_params(*dims, 0, bc))
    wd = [torch.from_numpy(a).to("cuda") for a in w[:5]] + [None]
    out = [torch.full_like(a, float("nan")) for a in wd[:5]] + [None]
    ctx.fe(wd, out)
    for q in range(5):
        assert normwise_err(out[q].cpu().numpy(), ref[q]) <= 1e-12, q
    ctx.close()


def table(name):
    """(A, b, c): Euler, Shu-Osher's SSPRK3, Bogacki-Shampine 3 and a six-stage table of
    order one with every entry used."""
    if name == "bs3":
        return orc.bs3_table()
    if name == "euler":
        return np.zeros((1, 1)), np.array([1.0]), np.zeros(1)
    if name == "ssprk3":
        A = np.zeros((3, 3))
        A[1, 0] = 1.0
        A[2, :2] = 0.25
        return A, np.array([1 / 6, 1 / 6, 2 / 3]), A.sum(1)
    A = np.tril(np.linspace(0.05, 0.2, 36).reshape(6, 6), -1)
    b = np.array([0.1, 0.15, 0.2, 0.25, 0.2, 0.1])
    return A, b, A.sum(1)


@pytest.mark.parametrize("name", ["euler", "ssprk3", "bs3", "six"])
@pytest.mark.parametrize("dims,nchem", [((13, 6, 5), 0), ((12, 7, 6), 2), ((56, 50, 48), 0)])
def test_erk_tables(mvd, torch_gpu, name, dims, nchem):
    torch = torch_gpu
    nsteps, h, bc = 5, 5e-4, (3, 3, 1, 1, 0, 0)
    print(f"[erk tables] {name} dims={dims} nchem={nchem}", flush=True)
    A, b, c = table(name)
    t = mvd.ErkTable()
    t.stages = len(b)
    for i in range(len(b)):
        t.b[i], t.c[i] = b[i], c[i]
        for j in range(len(b)):
            t.A[6 * i + j] = A[i, j]
    w0 = problems.smooth_state(*dims, nchem, seed=31)
    ref = [np.ascontiguousarray(a).reshape(-1).copy() for a in w0]
    assert orc.erk_evolve(orc.make_grid(*dims, nchem, bc), orc.erk(A, b, c), h, nsteps, ref) == 0
    ctx = mvd.Context(mvd.make_params(*dims, nchem, bc))

    def dev():
        return [torch.from_numpy(np.ascontiguousarray(a).copy()).to("cuda") for a in w0[:5]] + \
            [torch.from_numpy(w0[5].copy()).to("cuda") if nchem else None]

    one, two = dev(), dev()
    assert ctx.erk_evolve(one, h, nsteps, table=t) == 0
    assert ctx.erk_evolve(two, h, 2, table=t) == 0
    assert ctx.erk_evolve(two, h, nsteps - 2, table=t) == 0
    for q in range(5 + (nchem > 0)):
        assert normwise_err(one[q].cpu().numpy(), ref[q]) <= 1e-10, q
        assert torch.equal(one[q], two[q]), q
    ctx.close()
