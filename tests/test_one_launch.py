"""Stages in one launch against stages in two: the same sums in the same
order, so the same bits."""
import numpy as np
import pytest

from adfvm_amd import meshgen
from tests import casefactory as cf
from tests.test_gpu_primal import CASES

torch = pytest.importorskip('torch')
pytestmark = pytest.mark.gpu

BOXES = [(1, 1, 1), (4, 4, 4), (13, 5, 1), (7, 9, 11), (16, 8, 24)]


def _box(n):
    case = cf.CaseDef(meshgen.permute_and_rcm(meshgen.periodic_box(n), seed=5), {}, 1e-3)
    return case, cf.smooth_state(case, 4)


@pytest.mark.parametrize('name', sorted(CASES) + BOXES)
@pytest.mark.parametrize('prec', [np.float32, np.float64])
def test_residual_into_its_input(name, prec):
    """The residual written over the state it is taken of (two launches) and
    elsewhere (one)."""
    case, u = CASES[name]() if name in CASES else _box(name)
    ctx = case.context(prec)
    u = torch.as_tensor(u.astype(prec), device='cuda').contiguous()
    dtc = [torch.zeros(ctx.nIC, dtype=ctx.tdtype, device='cuda') for _ in range(2)]
    one, two = ctx.residual(u, dtc_cell=dtc[0]), u.clone()
    ctx.residual(two, out=two, dtc_cell=dtc[1])
    assert torch.equal(one, two) and torch.equal(*dtc)


@pytest.mark.parametrize('n', [(38, 43, 47), (41, 37, 31)])
@pytest.mark.parametrize('prec', [np.float32, np.float64])
def test_step_with_and_without_records(n, prec):
    """76798 and 47027 cells: more and fewer tiles than a stage that keeps its
    records takes in one launch."""
    case, u = _box(n)
    ctx = case.context(prec)
    out = []
    for tape in (None, ctx.new_tapes(1)[0]):
        v = torch.as_tensor(u.astype(prec), device='cuda').contiguous()
        dtc = torch.zeros(1, dtype=torch.float64, device='cuda')
        ctx.primal_step(v, 1e-6, dtc_out=dtc, tape=tape)
        out.append((v, dtc))
    assert torch.equal(out[0][0], out[1][0]) and torch.equal(out[0][1], out[1][1])
