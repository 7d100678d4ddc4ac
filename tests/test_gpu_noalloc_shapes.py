"""The allocation-free batched step with launch shapes of more waves than full chunks of 64 cells:
it has room for 4096 blocks, and a shape is refused only where full chunks need more. Bitwise the
allocating step's states, temperatures and Newton work."""
import importlib.util
import os

import numpy as np
import pytest

import orc
from conftest import PKG

spec = importlib.util.spec_from_file_location("mvd_problems", os.path.join(PKG, "problems.py"))
problems = importlib.util.module_from_spec(spec)
spec.loader.exec_module(problems)

pytestmark = pytest.mark.gpu


# full chunks: 4096 blocks (the limit), one more than that, and 4096 blocks of two waves
@pytest.mark.parametrize("n,block,waves,ok", [(1 << 18, 64, 8192, True),
                                              ((1 << 18) + 1, 64, 8192, False),
                                              (1 << 19, 128, 16384, True)])
def test_noalloc_shapes(mvd, torch_gpu, n, block, waves, ok):
    torch = torch_gpu
    print(f"[noalloc shapes] n={n} block={block} waves={waves}", flush=True)
    y, _ = problems.chem_cells(n, seed=45)
    got = []
    for noalloc in (False, True):
        ctx = mvd.Context(mvd.make_params(4, 4, 4, 10))
        ctx.chem_setup(orc.load_tables(), n)
        yd = torch.from_numpy(y.copy()).to("cuda")
        ctx.chem_prepare(yd)
        ctx.dirk_set_shape(block, waves)
        if noalloc and not ok:
            with pytest.raises(Exception) as e:
                ctx.dirk_step_noalloc(yd, 1e3)
            assert str(mvd.MVD_BAD_ARGUMENT) in str(e.value)
            ctx.close()
            return
        failed, st = (ctx.dirk_step_noalloc if noalloc else ctx.dirk_step)(yd, 1e3)
        got.append((failed, st["newton_iters"], st["setups"], st["hist"], yd.cpu().numpy(),
                    ctx.chem_state("Ts", torch).cpu().numpy()))
        ctx.close()
    assert got[0][:4] == got[1][:4]
    assert np.array_equal(got[0][4], got[1][4]) and np.array_equal(got[0][5], got[1][5])
