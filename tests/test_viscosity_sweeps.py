"""The adjoint viscosity's Jacobi sweeps, several to a launch, against the
oracle."""
import numpy as np
import pytest

from adfvm_amd import meshgen
from tests import casefactory as cf


@pytest.mark.gpu
@pytest.mark.parametrize('n', [(2, 1, 1), (13, 5, 1), (131, 1, 1), (70, 61, 1), (19, 17, 12)])
@pytest.mark.parametrize('iterations', [1, 2, 33, 70])
def test_sweeps_match_oracle(n, iterations):
    """2 to 4270 cells in one, two and three directions, fewer and more sweeps
    than a launch takes: FP64 against the oracle (1e-10, the bound of the
    eigenvalues), FP32 (1e-4)."""
    import torch
    from oracle import viscosity_oracle as vo
    case = cf.CaseDef(meshgen.permute_and_rcm(meshgen.periodic_box(n), seed=5), {}, 1e-3)
    u = cf.smooth_state(case, 4)
    ua = np.random.default_rng(6).normal(size=u.shape) * np.abs(1 / u).mean(1, keepdims=True)
    dt = 2e-5
    scaling = 0.1 * case.mesh.volumes.min() ** (2. / 3) / dt
    for prec, tol in ((np.float64, 1e-10), (np.float32, 1e-4)):
        r = lambda a: a.astype(prec).astype(np.float64)
        ref, _ = vo.adjoint_viscosity(case.oracle(), 'abarbanel', r(u), r(ua), dt, scaling, iterations,
                                      ghostInit=[torch.as_tensor(a, dtype=torch.float64) for a in cf.ghost_init(case)])
        ctx = case.context(prec)
        g = torch.as_tensor(ua.astype(prec), device='cuda').contiguous()
        ctx.adjoint_viscosity(torch.as_tensor(u.astype(prec), device='cuda').contiguous(), g, dt, 'abarbanel', scaling,
                              iterations=iterations)
        got = g.cpu().numpy().astype(np.float64)
        assert np.linalg.norm(got - ref) <= tol * np.linalg.norm(ref)
