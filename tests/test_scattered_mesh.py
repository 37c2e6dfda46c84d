"""Tiles whose surroundings do not fit the one-launch stage's tables: meshes
with neighbours anywhere."""
import numpy as np
import pytest

from adfvm_amd import meshgen
from tests import casefactory as cf
from tests.test_tiles import CELLS, HALO, shim, slot_tables  # noqa: F401

RING = 320


def scattered(n, seed=3):
    """n cells in a row, whose y and z faces are paired at random: all cyclic
    neighbours but the row's are anywhere."""
    cyclic = {a + e: (a + e, 'cyclic', a + '10'[int(e)]) for a in 'xyz' for e in '01'}
    md = meshgen.box((n, 1, 1), (n, 1., 1.), patches=cyclic)
    rng = np.random.default_rng(seed)
    for name, b in md.boundary.items():
        if b['nFaces'] == n and b['startFace'] < md.boundary[b['neighbourPatch']]['startFace']:
            rows = slice(b['startFace'], b['startFace'] + n)
            order = rng.permutation(n)
            md.faces[rows], md.owner[rows] = md.faces[rows][order], md.owner[rows][order]
    return cf.CaseDef(md, {}, 1e-3, objective=('kinetic_energy',))


def outer_ring(shim, m):  # noqa: F811
    """The largest number of cells beside a tile's halo, over the tiles."""
    import ctypes as C
    nIC = m.nInternalCells
    tables = slot_tables(m)
    p = lambda a: a.ctypes.data_as(C.c_void_p)
    n = shim.tiles_build(nIC, m.nInternalFaces, m.nFaces, *[p(a) for a in tables], C.c_uint(4))
    toUser, toTile, halo = np.zeros(n * CELLS, np.int32), np.zeros(nIC, np.int32), np.zeros((n, HALO), np.int32)
    rest = [np.zeros(n * k, t) for k, t in ((256, np.int32), (256, np.uint32), (CELLS, np.uint64),
                                            (CELLS, np.uint64), (CELLS, np.uint64))]
    shim.tiles_get(p(toUser), p(toTile), p(halo), *[p(a) for a in rest])
    most = 0
    for t in range(n):
        own = toUser[t * CELLS:(t + 1) * CELLS]
        own = set(own[own >= 0])
        ring1 = set(toUser[halo[t]]) - own
        ring2 = set(tables[1][:, sorted(ring1)].ravel()) - own - ring1
        most = max(most, len(ring2))
    return most


@pytest.mark.parametrize('n,fits', [(300, True), (1500, False)])
def test_outer_ring(shim, n, fits):  # noqa: F811
    """What the two meshes of the next test are for."""
    assert (outer_ring(shim, scattered(n).mesh) <= RING) == fits


@pytest.mark.gpu
@pytest.mark.parametrize('n', [300, 1500])
@pytest.mark.parametrize('with_tape', [False, True])
def test_step_and_adjoint(n, with_tape):
    """FP64 step and adjoint step against the oracle and its autograd, with the
    bounds of the tile edges' test (1e-12, 1e-10), and which kernels ran."""
    import torch
    case = scattered(n)
    rng = np.random.default_rng(4)
    u = cf.smooth_state(case, 4, amp=1e-5)       # extrapolated over up to n cells
    dt = 1e-4
    oc = case.oracle()
    t = torch.as_tensor(u, dtype=torch.float64).requires_grad_(True)
    ua = rng.normal(size=u.shape) * np.abs(1 / u).mean(1, keepdims=True)
    r, rU, rE, _, J = oc.step(t[0:1].T, t[1:4].T, t[4:5].T, dt)
    out = torch.cat([r.T, rU.T, rE.T])
    ref, = torch.autograd.grad((out * torch.as_tensor(ua)).sum() + J.sum(), t)
    ctx = case.context(np.float64)
    d = torch.as_tensor(u, device='cuda').contiguous()
    v, g = d.clone(), torch.as_tensor(ua, device='cuda').contiguous()
    tape = ctx.new_tapes(1)[0] if with_tape else None
    ctx.profile_start()
    ctx.primal_step(v, dt, tape=tape)
    kernels = set(ctx.profile_stop())
    assert ('tile_stage_kernel' in kernels) == (n == 300) and ('flux_stage_kernel' in kernels) == (n == 1500)
    ctx.adjoint_step(d, dt, g, obja=1.0, tape=tape)
    err = lambda a, b: float(np.linalg.norm(a - b) / np.linalg.norm(b))
    assert err(v.cpu().numpy(), out.detach().numpy()) < 1e-12
    assert err(g.cpu().numpy(), ref.numpy()) < 1e-10
