"""Cell tiles: the tables the tile kernels read (tiles.hpp, on the host), and
the kernels at the edges of tiles against the oracle."""
import ctypes as C
import os
import subprocess

import numpy as np
import pytest

from adfvm_amd import meshgen
from adfvm_amd.mesh import Mesh
from tests import casefactory as cf

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
CELLS, FACES, HALO = 64, 256, 128
COPY = 4

MESHES = {
    'one_cell': lambda: meshgen.periodic_box((1, 1, 1)),
    'two_cells': lambda: meshgen.periodic_box((2, 1, 1)),
    'one_tile': lambda: meshgen.periodic_box((3, 3, 3)),
    'random_order': lambda: meshgen.permute_and_rcm(meshgen.periodic_box((9, 10, 11)), seed=3),
    'walls': lambda: meshgen.box((13, 9, 7)),
    'tube': lambda: meshgen.shock_tube(131),
    'o_grid': lambda: meshgen.o_grid(48, 24),
    'two_regions': lambda: meshgen.concatenate([meshgen.periodic_box((5, 4, 3)), meshgen.periodic_box((7, 5, 4))])[0],
}


@pytest.fixture(scope='module')
def shim():
    out = os.path.join(ROOT, '_build', 'tiles_shim.so')
    os.makedirs(os.path.dirname(out), exist_ok=True)
    subprocess.check_call(['g++', '-O1', '-std=c++17', '-shared', '-fPIC', '-pthread', '-I',
                           os.path.join(ROOT, 'adfvm_amd', 'csrc'),
                           os.path.join(ROOT, 'tests', 'shim', 'tiles_shim.cpp'), '-o', out])
    return C.CDLL(out)


def slot_tables(m):
    """The context's slot tables of a built mesh ([6][nIC] rows) and face kinds."""
    nIF, nF = m.nInternalFaces, m.nFaces
    own = m.cellOwner != 0
    kind = np.zeros(nF, np.uint8)
    other, pair = np.empty(nF, np.int64), np.full(nF, -1)
    other[:nIF], other[nIF:] = m.neighbour[:nIF], -1 - np.arange(nF - nIF)
    kind[nIF:] = 2 | COPY
    for b in m.boundary.values():
        if 'neighbourPatch' in b:
            r = b['startFace'] + np.arange(b['nFaces'])
            g = m.boundary[b['neighbourPatch']]['startFace'] + np.arange(b['nFaces'])
            other[r], pair[r], kind[r] = m.owner[g], g, 0
    i32 = lambda a: np.ascontiguousarray(a.T, np.int32)
    f = m.cellFaces
    return (i32(f), i32(np.where(own, other[f], m.owner[f])), i32(pair[f]),
            np.ascontiguousarray(own.T.astype(np.uint8)), kind)


@pytest.mark.parametrize('name', sorted(MESHES))
def test_tile_tables(shim, name):
    """Every cell in one tile; every slot's face, other cell, side and pair
    found again through the words; unused entries harmless."""
    m = Mesh.from_data(MESHES[name]())
    nIC = m.nInternalCells
    sFace, sOther, sPair, sOwn, kind = slot_tables(m)
    p = lambda a: a.ctypes.data_as(C.c_void_p)
    n = shim.tiles_build(nIC, m.nInternalFaces, m.nFaces, p(sFace), p(sOther), p(sPair), p(sOwn), p(kind),
                         C.c_uint(COPY))
    toUser, toTile = np.zeros(n * CELLS, np.int32), np.zeros(nIC, np.int32)
    halo, faceId = np.zeros((n, HALO), np.int32), np.zeros((n, FACES), np.int32)
    face = np.zeros((n, FACES), np.uint32)
    slots, pairs, nbr = [np.zeros(n * CELLS, np.uint64) for _ in range(3)]
    shim.tiles_get(*[p(a) for a in (toUser, toTile, halo, faceId, face, slots, pairs, nbr)])
    used = toUser >= 0
    assert used.sum() == nIC and np.array_equal(np.sort(toUser[used]), np.arange(nIC))
    assert np.array_equal(toUser[toTile], np.arange(nIC))
    real = np.where(used, toUser, ~toUser)
    assert (0 <= real).all() and (real < nIC).all()
    assert (0 <= halo).all() and (halo < n * CELLS).all() and used[halo].all()
    assert (0 <= faceId).all() and (faceId < m.nFaces).all()
    pos = np.nonzero(used)[0]
    cells, tile = toUser[pos], pos // CELLS

    def cell(t, local):          # a tile's local cell -> the mesh's cell
        at = np.where(local < CELLS, t * CELLS + local, halo[t, np.maximum(local - CELLS, 0)])
        return toUser[at]

    byte = lambda w, j: ((w >> np.uint64(8 * j)) & np.uint64(255)).astype(np.int64)
    bit = lambda w, b: ((w >> np.uint64(b)) & np.uint64(1)).astype(bool)
    for j in range(6):
        f, o, g = sFace[j][cells], sOther[j][cells], sPair[j][cells]
        lf = byte(slots[pos], j)
        assert np.array_equal(faceId[tile, lf], f)
        own = bit(slots[pos], 48 + j)
        assert np.array_equal(own, sOwn[j][cells] != 0)
        assert np.array_equal(bit(slots[pos], 54 + j), g >= 0)
        assert np.array_equal(bit(nbr[pos], 48 + j), o < 0)
        assert np.array_equal(bit(nbr[pos], 54 + j), o < 0)
        inner = o >= 0
        assert np.array_equal(cell(tile, byte(nbr[pos], j))[inner], o[inner])
        w = face[tile, lf]
        lP, lN = (w & 255).astype(np.int64), ((w >> 8) & 255).astype(np.int64)
        assert np.array_equal(cell(tile, lP), np.where(own, cells, o))
        assert np.array_equal(cell(tile, lN)[inner], np.where(own, o, cells)[inner])
        assert np.array_equal((w >> 16) & 255, kind[f]) and np.array_equal((w >> 24) & 1, f < m.nInternalFaces)
        c = g >= 0
        lg = byte(pairs[pos], j)[c]
        assert np.array_equal(faceId[tile[c], lg], g[c])
        w = face[tile[c], lg]
        assert np.array_equal(cell(tile[c], (w & 255).astype(np.int64)), o[c])
        assert np.array_equal(cell(tile[c], ((w >> 8) & 255).astype(np.int64)), cells[c])
    assert (((face & 255) < CELLS + HALO) & (((face >> 8) & 255) < CELLS + HALO)).all()


@pytest.mark.gpu
@pytest.mark.parametrize('n', [(3, 3, 3), (4, 4, 4), (13, 5, 1), (8, 8, 8), (7, 9, 11)])
@pytest.mark.parametrize('rcm', [True, False])
def test_step_and_adjoint_at_tile_edges(n, rcm):
    """27, 64, 65, 512 and 693 cells, in reverse Cuthill-McKee and generated
    order: FP64 step and adjoint step against the oracle and its autograd,
    within the rounding of sums of a few hundred terms (1e-12, 1e-10)."""
    import torch
    md = meshgen.periodic_box(n)
    if rcm:
        md = meshgen.permute_and_rcm(md, seed=5)
    case = cf.CaseDef(md, {}, 1e-3, objective=('kinetic_energy',))
    u = cf.smooth_state(case, 4)
    dt = 1e-5
    oc = case.oracle()
    t = torch.as_tensor(u, dtype=torch.float64).requires_grad_(True)
    ua = np.random.default_rng(6).normal(size=u.shape) * np.abs(1 / u).mean(1, keepdims=True)
    r, rU, rE, _, J = oc.step(t[0:1].T, t[1:4].T, t[4:5].T, dt)
    out = torch.cat([r.T, rU.T, rE.T])
    ref, = torch.autograd.grad((out * torch.as_tensor(ua)).sum() + J.sum(), t)
    ctx = case.context(np.float64)
    d = torch.as_tensor(u, device='cuda').contiguous()
    v, g = d.clone(), torch.as_tensor(ua, device='cuda').contiguous()
    tape = ctx.new_tapes(1)[0]
    ctx.primal_step(v, dt, tape=tape)
    ctx.adjoint_step(d, dt, g, obja=1.0, tape=tape)
    err = lambda a, b: float(np.linalg.norm(a - b) / np.linalg.norm(b))
    assert err(v.cpu().numpy(), out.detach().numpy()) < 1e-12
    assert err(g.cpu().numpy(), ref.numpy()) < 1e-10
