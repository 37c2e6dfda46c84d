"""The adjoint viscosity's two ways to sweep, one sweep a launch and several
over patches, on the same context: the same bits."""
import numpy as np
import pytest

from adfvm_amd import meshgen
from tests import casefactory as cf


def _inputs(case, ctx):
    import torch
    u = cf.smooth_state(case, 4)
    ua = np.random.default_rng(6).normal(size=u.shape) * np.abs(1 / u).mean(1, keepdims=True)
    dt = 2e-5
    scaling = 0.1 * case.mesh.volumes.min() ** (2. / 3) / dt
    t = lambda a: torch.as_tensor(a.astype(ctx.precision), device='cuda').contiguous()
    return t(u), t(ua), dt, scaling


def _sweep_kernels(ctx, f):
    ctx.profile_start()
    f()
    return {k: n for k, (_, n) in ctx.profile_stop().items() if k in ('visc_rings_kernel', 'visc_jacobi_kernel')}


@pytest.mark.gpu
@pytest.mark.parametrize('prec', [np.float32, np.float64])
def test_first_call_captured(prec):
    """A context whose first call is captured sweeps one at a time in the
    graph, and over patches in calls outside it."""
    import torch
    case = cf.CaseDef(meshgen.permute_and_rcm(meshgen.periodic_box((40, 30, 1)), seed=5), {}, 1e-3)
    ctx = case.context(prec)
    u, ua, dt, scaling = _inputs(case, ctx)
    a = ua.clone()
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph, capture_error_mode='relaxed'):
        ctx.adjoint_viscosity(u, a, dt, 'abarbanel', scaling, iterations=20)
    eager = ua.clone()
    kernels = _sweep_kernels(ctx, lambda: ctx.adjoint_viscosity(u, eager, dt, 'abarbanel', scaling, iterations=20))
    assert list(kernels) == ['visc_rings_kernel'] and kernels['visc_rings_kernel'] < 20
    for _ in range(3):
        a.copy_(ua)
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(a, eager)
        eager.copy_(ua)
        ctx.adjoint_viscosity(u, eager, dt, 'abarbanel', scaling, iterations=20)


@pytest.mark.gpu
@pytest.mark.parametrize('n', [(40, 30, 1), (61, 60, 59)])
@pytest.mark.parametrize('prec', [np.float32, np.float64])
def test_alongside_steps_that_keep_tapes(n, prec):
    """Sweeps on one stream while steps that keep their tapes run on another,
    as in a reverse sweep that smooths the adjoint during a segment's re-run
    (1200 cells, and 215940, whose steps convert rows): the bits of both in
    turn."""
    import torch
    case = cf.CaseDef(meshgen.permute_and_rcm(meshgen.periodic_box(n), seed=5), {}, 1e-3)
    ctx = case.context(prec)
    u, ua, dt, scaling = _inputs(case, ctx)
    steps = 8
    tapes = ctx.new_tapes(steps)

    def run_steps(v):
        for k in range(steps):
            ctx.primal_step(v, 1e-7, tape=tapes[k])

    def smooth(a):
        for _ in range(2):
            ctx.adjoint_viscosity(u, a, dt, 'abarbanel', scaling, iterations=40)

    v, a = u.clone(), ua.clone()
    run_steps(v)
    smooth(a)
    kept = tapes.clone()
    side = torch.cuda.Stream()
    for _ in range(3):
        v2, a2 = u.clone(), ua.clone()
        tapes.zero_()
        torch.cuda.synchronize()
        with torch.cuda.stream(side):
            run_steps(v2)
        smooth(a2)
        torch.cuda.synchronize()
        assert torch.equal(v2, v) and torch.equal(a2, a)
        rows = 5 * ctx.nIC
        assert torch.equal(tapes[:, :rows], kept[:, :rows])


# tiles a patch, and whether several sweeps a launch pay
PATCHES = {
    'o_grid_2_tiles': (lambda: meshgen.o_grid(160, 130), True),
    'o_grid_5_tiles': (lambda: meshgen.o_grid(301, 261), True),
    'walls_2_tiles': (lambda: meshgen.permute_and_rcm(meshgen.box((31, 30, 29)), seed=5), True),
    'box_above_limit': (lambda: meshgen.permute_and_rcm(meshgen.periodic_box((64, 63, 62)), seed=5), False),
}


@pytest.mark.gpu
@pytest.mark.parametrize('name', sorted(PATCHES))
@pytest.mark.parametrize('prec', [np.float32, np.float64])
@pytest.mark.parametrize('iterations', [2, 37])
def test_patches_of_several_tiles(name, prec, iterations):
    """Patches of 2 and 5 tiles, the last one smaller than the others, with and
    without ghosts, and a mesh whose rings do not fit: the sweeps of a captured
    first call, one at a time, against those of a call outside a capture."""
    import torch
    make, several = PATCHES[name]
    case = cf.CaseDef(make(), {}, 1e-3)
    ctx = case.context(prec)
    u, ua, dt, scaling = _inputs(case, ctx)
    one = ua.clone()
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph, capture_error_mode='relaxed'):
        ctx.adjoint_viscosity(u, one, dt, 'abarbanel', scaling, iterations=iterations)
    graph.replay()
    many = ua.clone()
    kernels = _sweep_kernels(ctx, lambda: ctx.adjoint_viscosity(u, many, dt, 'abarbanel', scaling,
                                                                iterations=iterations))
    assert list(kernels) == (['visc_rings_kernel'] if several else ['visc_jacobi_kernel'])
    assert torch.isfinite(many).all() and not torch.equal(many, ua)
    assert torch.equal(one, many)
