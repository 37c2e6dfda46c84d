"""The work that programs built on this framework have it do, as cases that can
be timed and compared: time steps, adjoint steps, residuals and their
transposes, checkpointed sweeps and the adjoint viscosity, from meshes of a
thousand cells to the 128^3 box of bench.py.

  listed()            the named cases
  draw(rng)           one more case of the same ranges
  prepare(case, seed) context and device arrays, from the seed
  run(state)          one pass through the public entry points; its outputs
  work(case)          bytes and operations that one pass cannot do without
  exact(case, seed)   run's outputs from a plain torch FP64 evaluation

A mesh is built once per shape and kept (a program builds its mesh once); the
context and every array are made anew by each prepare().
"""
import functools
import math

import numpy as np
import torch

from adfvm_amd import BCs, _lib, cases, config, meshgen
from adfvm_amd.context import Context
from adfvm_amd.graphs import GraphSweep
from adfvm_amd.mesh import Mesh

GAMMA, CP, PR = 1.4, 1004.5, 0.7
CV = CP / GAMMA
R = CP - CV
VISC_ITERATIONS = 1000          # the default of Context.adjoint_viscosity


def listed():
    return [
        # a shock-tube program's step: one launch-bound call per time step, limited reconstruction, FP64
        dict(name='sod_1000_step_f64', mesh='sod', nx=1000, ny=1, nz=1, op='step', precision=64),
        # a small ensemble member or a debugging run: step and adjoint step where launches are all that counts
        dict(name='tgv_16_pa_f32', mesh='tgv', nx=16, ny=16, nz=16, op='pa', precision=32),
        # the operator pieces, as tests and matrix-free solvers call them, on an odd-sized O-grid
        dict(name='cyl_129x67_residual_f32', mesh='cyl', nx=129, ny=67, nz=1, op='residual', precision=32),
        # walls, inlet, outlet and a source term in blockMesh's cell order, every parameter gradient on
        dict(name='duct_37x29x23_pa_f64', mesh='duct', nx=37, ny=29, nz=23, op='pa', precision=64),
        # a whole checkpointed sweep (10 steps forward, re-run, 10 adjoint steps, twice) in HIP graphs
        dict(name='tgv_48_sweep_f32', mesh='tgv', nx=48, ny=48, nz=48, op='sweep', precision=32),
        # the 64^3 adjoint workload's step, in both precisions
        dict(name='tgv_64_pa_f32', mesh='tgv', nx=64, ny=64, nz=64, op='pa', precision=32),
        dict(name='tgv_64_pa_f64', mesh='tgv', nx=64, ny=64, nz=64, op='pa', precision=64),
        # the cylinder wake's step: drag objective, wall and far-field value gradients
        dict(name='cyl_512x256_pa_f32', mesh='cyl', nx=512, ny=256, nz=1, op='pa', precision=32),
        # its adjoint-viscosity smoothing, 1000 Jacobi sweeps
        dict(name='cyl_512x256_visc_f32', mesh='cyl', nx=512, ny=256, nz=1, op='visc', precision=32),
        # a forward run's step on a box of odd sides, time-step control and objective on
        dict(name='tgv_101x83x67_step_f32', mesh='tgv', nx=101, ny=83, nz=67, op='step', precision=32),
        # the headline box: a forward run's step, and the step with its adjoint step
        dict(name='tgv_128_step_f32', mesh='tgv', nx=128, ny=128, nz=128, op='step', precision=32),
        dict(name='tgv_128_pa_f32', mesh='tgv', nx=128, ny=128, nz=128, op='pa', precision=32),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    mesh = rng.choice(['tgv', 'tgv', 'tgv', 'cyl', 'cyl', 'duct', 'sod'])
    precision = rng.choice([32, 32, 64])
    if mesh == 'sod':
        return dict(mesh=mesh, nx=_log(rng, 100, 20000), ny=1, nz=1, op='step', precision=precision)
    if mesh == 'cyl':
        op = rng.choice(['pa', 'pa', 'residual', 'step', 'visc'])
        return dict(mesh=mesh, nx=_log(rng, 48, 512), ny=_log(rng, 24, 256), nz=1, op=op, precision=precision)
    if mesh == 'duct':
        op = rng.choice(['pa', 'pa', 'step', 'residual'])
        return dict(mesh=mesh, nx=_log(rng, 6, 60), ny=_log(rng, 5, 60), nz=_log(rng, 4, 60), op=op,
                    precision=precision)
    op = rng.choice(['pa', 'pa', 'step', 'sweep', 'residual'])
    top = 48 if op == 'sweep' else 100 if precision == 64 else 125
    n = _log(rng, 8, top)                   # sides within a quarter of one another
    nx, ny, nz = [max(6, min(top, int(round(n * rng.uniform(0.8, 1.25))))) for _ in range(3)]
    return dict(mesh=mesh, nx=nx, ny=ny, nz=nz, op=op, precision=precision)


# ------------------------------------------------------------------- cases --

@functools.lru_cache(maxsize=None)
def _setup(kind, nx, ny, nz):
    """The generated case (mesh, initial fields, boundary conditions)."""
    if kind == 'tgv':
        return cases.taylor_green((nx, ny, nz))
    if kind == 'cyl':
        return cases.cylinder(nx, ny)
    if kind == 'sod':
        return cases.shock_tube(nx)
    patches = {'x0': ('inlet', 'patch'), 'x1': ('outlet', 'patch'), 'y0': ('bottom', 'symmetryPlane'),
               'y1': ('top', 'patch'), 'z0': ('sides', 'empty'), 'z1': ('sides', 'empty')}
    md = meshgen.box((nx, ny, nz), (0.02 * nx, 0.02 * ny, 0.02 * nz), patches=patches)
    mesh = Mesh.from_data(md)
    nIC, n_in, n_out, n_top = mesh.nInternalCells, ny * nz, ny * nz, nx * nz
    U0 = np.array([30., 2., 0.])
    bnd = {'U': {'inlet': {'type': 'fixedValue', 'value': np.tile(U0, (n_in, 1))},
                 'top': {'type': 'fixedValue', 'value': np.zeros((n_top, 3))}, 'bottom': {'type': 'slip'},
                 'outlet': {'type': 'CBC_UPT'}},
           'T': {'inlet': {'type': 'fixedValue', 'value': np.full((n_in, 1), 300.)},
                 'top': {'type': 'zeroGradient'}, 'bottom': {'type': 'symmetryPlane'},
                 'outlet': {'type': 'CBC_UPT'}},
           'p': {'inlet': {'type': 'zeroGradient'}, 'top': {'type': 'zeroGradient'},
                 'bottom': {'type': 'symmetryPlane'},
                 'outlet': {'type': 'CBC_UPT', 'U0': U0, 'T0': np.full((n_out, 1), 300.),
                            'p0': np.full((n_out, 1), 1e5)}}}
    return cases.CaseSetup(md, np.tile(U0, (nIC, 1)), np.full((nIC, 1), 300.), np.full((nIC, 1), 1e5), bnd, 1.8e-5,
                           mesh)


def _case_setup(case):
    return _setup(case['mesh'], case['nx'], case['ny'], case['nz'])


def _options(case):
    """(limiter, boundary flux, objective) of the case's kind."""
    if case['mesh'] == 'cyl':
        return 0, _lib.RIEMANN_LF, ('drag', 'cylinder')
    if case['mesh'] == 'duct':
        return 0, _lib.RIEMANN_ROE, ('kinetic_energy', None)
    return int(case['mesh'] == 'sod'), _lib.RIEMANN_ROE, ('kinetic_energy', None)


def _context(case, setup):
    precision = np.float32 if case['precision'] == 32 else np.float64
    limiter, bflux, (obj, patch) = _options(case)
    ph = dict(gamma=GAMMA, Cp=CP, Pr=PR, mu=(_lib.MU_CONSTANT, float(setup.mu), 0., 0.),
              riemann=_lib.RIEMANN_ROE, boundaryRiemann=bflux, small=config.small_for(precision),
              integrator=_lib.RK_SSPRK3, limiter=limiter,
              objective=_lib.OBJ_DRAG if obj == 'drag' else _lib.OBJ_KINETIC_ENERGY)
    if patch is not None:
        ph['objectivePatch'] = patch
    return Context(setup.mesh, BCs.validate(setup.mesh, setup.boundary), ph, precision)


def _device():
    return 'cuda' if torch.cuda.is_available() else 'cpu'


def _dt(case, setup):
    """CFL about 0.5 on the smallest cell spacing."""
    h = float(setup.mesh.deltas[:setup.mesh.nInternalFaces].min())
    U = float(np.abs(setup.U).max())
    return 0.4 * h / (U + math.sqrt(GAMMA * R * float(setup.T.max())))


def _arrays(case, seed, setup):
    """The pass's fields in the case's precision: state, adjoint state and
    source.  Primitive fields with 1% noise per cell; adjoint fields of the
    size a kinetic-energy or drag sensitivity has; a source of the size of
    one percent of the flow through a cell per second."""
    dtype = torch.float32 if case['precision'] == 32 else torch.float64
    dev = _device()
    g = torch.Generator(device='cpu').manual_seed(int(seed))
    nIC = setup.mesh.nInternalCells
    f64 = lambda a: torch.as_tensor(a, dtype=torch.float64).to(dev)
    noise = (2 * torch.rand((5, nIC), generator=g, dtype=torch.float64) - 1).to(dev)
    U, T, p = f64(setup.U).T, f64(setup.T)[:, 0], f64(setup.p)[:, 0]
    scale = float(np.abs(setup.U).max()) or 1.0
    U = U * (1 + 0.01 * noise[:3]) + 0.002 * scale * noise[[1, 2, 0]]
    T, p = T * (1 + 0.001 * noise[3]), p * (1 + 0.001 * noise[4])
    rho = p / (R * T)
    u = torch.cat([rho[None], rho * U, (rho * (CV * T + 0.5 * (U * U).sum(0)))[None]])
    V = f64(setup.mesh.volumes)[:, 0]
    size = f64([[scale * scale], [scale], [scale], [scale], [1.0]])
    ua = torch.randn((5, nIC), generator=g, dtype=torch.float64).to(dev) * size * V
    S = torch.randn((5, nIC), generator=g, dtype=torch.float64).to(dev) * 0.01 * u.abs().mean(1, keepdim=True)
    return [a.to(dtype).contiguous() for a in (u, ua, S)]


def prepare(case, seed):
    setup = _case_setup(case)
    ctx = _context(case, setup)
    u0, ua0, S = _arrays(case, seed, setup)
    s = dict(case=case, ctx=ctx, u0=u0, ua0=ua0, S=S if case['mesh'] == 'duct' else None, dt=_dt(case, setup))
    new = lambda n: torch.zeros(n, dtype=torch.float64, device=u0.device)
    op = case['op']
    if op in ('step', 'pa'):
        s.update(u=torch.empty_like(u0), obj=new(1), dtc=new(1))
    if op == 'pa':
        s.update(tape=ctx.new_tapes(1)[0], ua=torch.empty_like(u0),
                 Sbar=torch.empty_like(u0) if s['S'] is not None else None,
                 bcg=ctx.bc_state() if case['mesh'] in ('cyl', 'duct') else None)
    elif op == 'residual':
        s.update(R=torch.empty_like(u0), ubar=torch.empty_like(u0))
    elif op == 'visc':
        s.update(ua=torch.empty_like(u0), m2=torch.empty(ctx.nIC, dtype=u0.dtype, device=u0.device))
    elif op == 'sweep':
        s['sweep'] = GraphSweep(ctx, s['dt'], 10)
        s['sweep'].run(u0, 20)                 # captures its graphs
    return s


def run(s):
    ctx, op = s['ctx'], s['case']['op']
    if op == 'step':
        s['u'].copy_(s['u0'])
        ctx.primal_step(s['u'], s['dt'], source=s['S'], dtc_out=s['dtc'], obj_out=s['obj'])
        return s['u'], s['obj'], s['dtc']
    if op == 'pa':
        s['u'].copy_(s['u0'])
        ctx.primal_step(s['u'], s['dt'], source=s['S'], obj_out=s['obj'], tape=s['tape'])
        s['ua'].copy_(s['ua0'])
        for a in (s['Sbar'], s['bcg']):
            if a is not None:
                a.zero_()
        ctx.adjoint_step(s['u0'], s['dt'], s['ua'], obja=1.0, source=s['S'], source_grad=s['Sbar'],
                         bc_grad=s['bcg'], tape=s['tape'])
        return [a for a in (s['u'], s['obj'], s['ua'], s['Sbar'], s['bcg']) if a is not None]
    if op == 'residual':
        ctx.residual(s['u0'], out=s['R'])
        ctx.residual_vjp(s['u0'], s['ua0'], out=s['ubar'])
        return s['R'], s['ubar']
    if op == 'visc':
        s['ua'].copy_(s['ua0'])
        ctx.adjoint_viscosity(s['u0'], s['ua'], s['dt'], 'abarbanel', 1.0, VISC_ITERATIONS, m2norm_out=s['m2'])
        return s['ua'], s['m2']
    J, ua = s['sweep'].run(s['u0'], 20)
    return J, ua


def _counts(case):
    """(cells, faces, boundary faces) of the case's mesh."""
    x, y, z = case['nx'], case['ny'], case['nz']
    if case['mesh'] == 'cyl':
        inner, outer = x * y + x * (y - 1), 2 * x + 2 * x * y
    else:
        inner = (x - 1) * y * z + x * (y - 1) * z + x * y * (z - 1)
        outer = 2 * (x * y + y * z + z * x)
    return x * y * z, inner + outer, outer


def work(case):
    """State, adjoint and source rows read and written once per call, face
    and cell geometry and connectivity read once per call; operations as the
    formulas count them per face and stage (gradient, reconstruction, Roe
    and viscous flux: about 700; their transposes with the re-evaluated
    forward: about 1900)."""
    nC, nF, nB = _counts(case)
    s = case['precision'] // 8
    geometry = s * (17 * nF + nC) + 8 * nF
    row = 5 * s * nC
    source = 2 * row if case['mesh'] == 'duct' else 0
    op = case['op']
    if op == 'step':
        return {'bytes': geometry + 2 * row + source / 2, 'flops': 3 * 700. * nF}
    if op == 'pa':
        return {'bytes': 2 * geometry + 5 * row + 2 * source + 5 * s * nB, 'flops': 3 * 2600. * nF}
    if op == 'residual':
        return {'bytes': 2 * geometry + 5 * row, 'flops': 2600. * nF + 700. * nF}
    if op == 'visc':
        return {'bytes': geometry + 3 * row + s * nC, 'flops': VISC_ITERATIONS * 70. * nC}
    # forward, re-run and reverse of 20 steps, each step a call
    return {'bytes': 20 * (3 * geometry + 7 * row), 'flops': 20 * 3 * 3300. * nF}


# ------------------------------------------------------- FP64 evaluation --

class _Fp64(object):
    """The discretisation in plain torch, FP64, on the mesh's arrays."""

    def __init__(self, case, setup):
        m = setup.mesh
        dev = _device()
        f = lambda a: torch.as_tensor(np.asarray(a), dtype=torch.float64).to(dev)
        i = lambda a: torch.as_tensor(np.asarray(a), dtype=torch.int64).to(dev)
        self.limiter, bflux, (self.objective, self.objPatch) = _options(case)
        self.lf = bflux == _lib.RIEMANN_LF
        self.small = config.small_for(np.float32 if case['precision'] == 32 else np.float64)
        self.mu = float(setup.mu)
        self.nIC, self.nIF, self.nF = m.nInternalCells, m.nInternalFaces, m.nFaces
        self.P = i(m.owner)
        self.A, self.w, self.delta = f(m.areas)[:, 0], f(m.weights)[:, 0], f(m.deltas)[:, 0]
        self.n, self.D = f(m.normals).T.contiguous(), f(m.deltasUnit).T.contiguous()
        self.lw = f(m.linearWeights)
        self.qw = f(m.quadraticWeights)
        self.V = f(m.volumes)[:, 0]
        self.slots = i(m.cellFaces)                                 # [cells][6]
        nB = self.nF - self.nIF
        other = np.array(m.owner[self.nIF:], np.int64)             # the cell a ghost's values start from
        kind = np.full(nB, 2)                                       # 0 coupled, 1 characteristic, 2 other
        fixed = np.zeros((5, nB), bool)
        value = np.zeros((5, nB))
        slip = np.zeros(nB, bool)
        spec = BCs.validate(m, setup.boundary)
        for name, b in m.boundary.items():
            sl = slice(b['startFace'] - self.nIF, b['startFace'] - self.nIF + b['nFaces'])
            if b['type'] == 'cyclic':
                other[sl] = b['loc_neighbourIndices']
                kind[sl] = 0
                continue
            p = spec[name]['p']
            if p['type'] == 'CBC_UPT':
                kind[sl] = 1
                fixed[:, sl] = True
                value[:, sl] = np.concatenate([np.broadcast_to(p[k], (b['nFaces'], c)) for k, c in
                                               (('U0', 3), ('T0', 1), ('p0', 1))], 1).T
                continue
            for field, rows in (('U', slice(0, 3)), ('T', slice(3, 4)), ('p', slice(4, 5))):
                e = spec[name][field]
                if e['type'] == 'fixedValue':
                    fixed[rows, sl] = True
                    value[rows, sl] = e['value'].T
            slip[sl] = spec[name]['U']['type'] in ('slip', 'symmetryPlane')
        self.from_cell, self.fixed, self.value = i(other), torch.as_tensor(fixed).to(dev), f(value)
        self.slip = torch.as_tensor(slip).to(dev)
        kind = torch.as_tensor(kind).to(dev)
        inner = torch.arange(self.nIF, device=dev)
        self.flux_faces = torch.cat([inner, self.nIF + torch.nonzero(kind == 0)[:, 0]])
        self.char_faces = self.nIF + torch.nonzero(kind == 1)[:, 0]
        self.ghost_faces = self.nIF + torch.nonzero(kind == 2)[:, 0]
        self.coupled = kind == 0
        self.N = torch.cat([i(m.neighbour[:self.nIF]), self.nIC + torch.arange(nB, device=dev)])
        if self.objective == 'drag':
            b = m.boundary[self.objPatch]
            self.drag_faces = torch.arange(b['startFace'], b['startFace'] + b['nFaces'], device=dev)

    def primitive(self, u):
        U = u[1:4] / u[0]
        e = u[4] / u[0] - 0.5 * (U * U).sum(0)
        return torch.cat([U, (e / CV)[None], ((GAMMA - 1) * u[0] * e)[None]])

    def with_ghosts(self, w, value):
        g = w[:, self.from_cell]
        n = self.n[:, self.nIF:]
        un = (g[:3] * n).sum(0) * self.slip
        g = torch.cat([g[:3] - un * n, g[3:]])
        return torch.cat([w, torch.where(self.fixed, value, g)], 1)

    def gradient(self, wa):
        """[5][3][cells and ghosts]: a ghost's is its owner's, a cyclic one's
        the paired cell's"""
        f = wa[:, self.P] * self.w + wa[:, self.N] * (1 - self.w)
        S = self.A * self.n
        out = []
        for c in range(5):
            flow = f[c] * S
            g = torch.zeros((3, self.nIC), dtype=torch.float64, device=wa.device)
            g = g.index_add(1, self.P, flow).index_add(1, self.N[:self.nIF], -flow[:, :self.nIF]) / self.V
            out.append(torch.cat([g, g[:, self.from_cell]], 1))
        return torch.stack(out)

    @staticmethod
    def conservative(w):
        rho = w[4] / (R * w[3])
        return torch.cat([rho[None], rho * w[:3], (rho * (CV * w[3] + 0.5 * (w[:3] * w[:3]).sum(0)))[None]])

    def reconstruct(self, wc, gc, wd, f, side):
        v = wc + (wd - wc) * self.lw[f, side] + (gc * self.qw[f, side].T).sum(1)
        if self.limiter:
            v = torch.minimum(torch.maximum(v, torch.minimum(wc, wd)), torch.maximum(wc, wd))
        return v

    def euler(self, q, w, n):
        Un = (w[:3] * n).sum(0)
        return torch.cat([(q[0] * Un)[None], q[1:4] * Un + w[4] * n, ((q[4] + w[4]) * Un)[None]])

    def lax_friedrichs(self, wL, wR, n):
        qL, qR = self.conservative(wL), self.conservative(wR)
        speed = lambda w, q: (w[:3] * n).sum(0).abs() + torch.sqrt(GAMMA * w[4] / q[0])
        a = torch.maximum(speed(wL, qL), speed(wR, qR))
        return 0.5 * (self.euler(qL, wL, n) + self.euler(qR, wR, n) - a * (qR - qL))

    def roe(self, wL, wR, n):
        qL, qR = self.conservative(wL), self.conservative(wR)
        hL, hR = (qL[4] + wL[4]) / qL[0], (qR[4] + wR[4]) / qR[0]
        sL, sR = torch.sqrt(qL[0]), torch.sqrt(qR[0])
        U = (wL[:3] * sL + wR[:3] * sR) / (sL + sR)
        h = (hL * sL + hR * sR) / (sL + sR)
        k = 0.5 * (U * U).sum(0)
        a2 = (GAMMA - 1) * (h - k)
        a = torch.sqrt(a2)
        Un = (U * n).sum(0)
        d = qR - qL
        sound = lambda w, q: torch.sqrt(GAMMA * w[4] / q[0])
        eps = 0.5 * ((wL[:3] * n).sum(0) - (wR[:3] * n).sum(0)).abs() + \
            0.5 * (sound(wL, qL) - sound(wR, qR)).abs() + self.small
        fix = lambda lam: torch.where(lam < 2 * eps, 0.25 * lam * lam / eps + eps, lam)
        l1, l2, l3 = fix(Un.abs()), fix((Un + a).abs()), fix((Un - a).abs())
        c3, c2 = 0.5 * (l2 + l3) - l1, 0.5 * (l2 - l3)
        x = (GAMMA - 1) * (k * d[0] - (U * d[1:4]).sum(0) + d[4])
        y = Un * d[0] - (d[1:4] * n).sum(0)
        s = c3 * x / a2 - c2 * y / a
        t = c3 * y - c2 * x / a
        D = torch.cat([(l1 * d[0] + s)[None], l1 * d[1:4] + U * s - n * t, (l1 * d[4] + h * s - Un * t)[None]])
        return 0.5 * (self.euler(qL, wL, n) + self.euler(qR, wR, n) - D)

    def viscous(self, wP, wN, wF, g, f):
        """g: face gradients [4][3][f] of U, T; the viscous part of the flux."""
        n, D = self.n[:, f], self.D[:, f]
        sn = (wN[:4] - wP[:4]) / self.delta[f]
        g = g + (sn - (g * D).sum(1))[:, None] * D
        tr = g[0, 0] + g[1, 1] + g[2, 2]
        sigma = self.mu * (((g[:3] + g[:3].transpose(0, 1)) * n).sum(1) - 2. / 3 * tr * n)
        q = self.mu * CP / PR * (g[3] * n).sum(0)
        return torch.cat([torch.zeros_like(q)[None], sigma, (q + (sigma * wF[:3]).sum(0))[None]])

    def flux(self, wa, ga):
        """(flux, spectral radius) per face"""
        F = torch.zeros((5, self.nF), dtype=torch.float64, device=wa.device)
        lam = torch.zeros(self.nF, dtype=torch.float64, device=wa.device)
        for faces, kind in ((self.flux_faces, 0), (self.char_faces, 1), (self.ghost_faces, 2)):
            if not len(faces):
                continue
            P, N, n = self.P[faces], self.N[faces], self.n[:, faces]
            wP, wN, gP = wa[:, P], wa[:, N], ga[:, :, P]
            if kind == 0:
                gN = ga[:, :, N]
                wL = self.reconstruct(wP, gP, wN, faces, 0)
                wR = self.reconstruct(wN, gN, wP, faces, 1)
                conv, wF, gF = self.roe(wL, wR, n), 0.5 * (wL + wR), 0.5 * (gP[:4] + gN[:4])
            elif kind == 1:
                wL = self.reconstruct(wP, gP, wN, faces, 0)
                conv = (self.lax_friedrichs if self.lf else self.roe)(wL, wN, n)
                wF, gF = wN, gP[:4]
            else:
                conv, wF, gF = self.euler(self.conservative(wN), wN, n), wN, gP[:4]
            F = F.index_add(1, faces, conv - self.viscous(wP, wN, wF, gF, faces))
            lam = lam.index_add(0, faces, (wF[:3] * n).sum(0).abs() + torch.sqrt(CP * wF[3] * (GAMMA - 1)))
        return F, lam

    def residual(self, u, value):
        wa = self.with_ghosts(self.primitive(u), value)
        ga = self.gradient(wa)
        F, lam = self.flux(wa, ga)
        FA = F * self.A
        Rr = torch.zeros_like(u).index_add(1, self.P, FA).index_add(1, self.N[:self.nIF], -FA[:, :self.nIF])
        lA = lam * self.A
        rate = torch.zeros_like(self.V).index_add(0, self.P, lA).index_add(0, self.N[:self.nIF], lA[:self.nIF])
        return Rr / self.V, rate / self.V

    def J(self, u, value):
        if self.objective == 'kinetic_energy':
            return (0.5 * (u[1:4] * u[1:4]).sum(0) / u[0] * self.V).sum()
        wa = self.with_ghosts(self.primitive(u), value)
        f = self.drag_faces
        wi, wg = wa[:, self.P[f]], wa[:, self.N[f]]
        return ((wg[4] * self.n[0, f] - self.mu * (wg[0] - wi[0]) / self.delta[f]) * self.A[f]).sum()

    STAGES = ((1., 1.), (1. / 4, 1. / 4), (2. / 3, 2. / 3))       # weight of u_i, of dt*(L - S); u_0 has the rest

    @torch.no_grad()
    def step(self, u0, dt, S=None):
        """(u after the step, stage states, objective, dtc)"""
        us, u, J, dtc = [], u0, None, None
        for k, (a, b) in enumerate(self.STAGES):
            us.append(u)
            L, rate = self.residual(u, self.value)
            if k == 1:
                J, dtc = self.J(u, self.value), rate.max()
            u = (1 - a) * u0 + a * u - b * dt * (L if S is None else L - S)
        return u, us, J, dtc

    def transpose(self, fn, u, weight):
        """weight . d fn / d (u, boundary values)"""
        u = u.detach().requires_grad_(True)
        value = self.value.clone().requires_grad_(True)
        gu, gv = torch.autograd.grad((fn(u, value) * weight).sum(), (u, value), allow_unused=True)
        return gu, torch.zeros_like(value) if gv is None else gv * self.fixed

    def adjoint_step(self, us, dt, ua):
        """(adjoint at the step's start, source and boundary-value gradients)"""
        acc, Sbar, vbar = torch.zeros_like(ua), torch.zeros_like(ua), torch.zeros_like(self.value)
        for k in (2, 1, 0):
            a, b = self.STAGES[k]
            g, v = self.transpose(lambda x, y: self.residual(x, y)[0], us[k], -b * dt * ua)
            vbar = vbar + v
            if k == 1:
                gj, v = self.transpose(self.J, us[1], 1.0)
                g, vbar = g + gj, vbar + v
            Sbar = Sbar + b * dt * ua
            acc = acc + (1 - a) * ua
            ua = a * ua + g
        return ua + acc, Sbar, vbar

    @torch.no_grad()
    def viscosity(self, u, ua, dt, scaling, iterations):
        w = self.primitive(u)
        wa = self.with_ghosts(w, self.value)
        c = torch.sqrt(GAMMA * R * wa[3])
        fields = torch.cat([wa[:3], wa[4:5], c[None]])
        f = fields[:, self.P] * self.w + fields[:, self.N] * (1 - self.w)
        keep = torch.cat([torch.ones(self.nIF, dtype=torch.bool, device=u.device), self.coupled])
        f = torch.where(keep, f, fields[:, self.N])
        grads = []
        for k in range(5):
            flow = f[k] * self.A * self.n
            g = torch.zeros((3, self.nIC), dtype=torch.float64, device=u.device)
            grads.append(g.index_add(1, self.P, flow).index_add(1, self.N[:self.nIF], -flow[:, :self.nIF]) / self.V)
        gU, gp, gc = torch.stack(grads[:3]), grads[3], grads[4]
        div, p, c, rho = gU[0, 0] + gU[1, 1] + gU[2, 2], w[4], c[:self.nIC], u[0]
        grho = GAMMA * (gp - c * p) / (c * c)
        sg, g1 = math.sqrt(GAMMA), GAMMA - 1
        gb, ga = gc / sg, gc * math.sqrt(g1) / sg
        t1, t2, t3 = c / sg * grho / rho, math.sqrt(g1) * c / sg * gp / (2 * p), 2 * ga / g1
        M = torch.zeros((self.nIC, 5, 5), dtype=torch.float64, device=u.device)
        for k in range(5):
            M[:, k, k] = 0.5 * div
        for k in range(3):
            M[:, 0, 1 + k] = 0.5 * gb[k] - t1[k]
            M[:, 1 + k, 0] = 0.5 * gb[k]
            M[:, 1 + k, 4] = 0.5 * ga[k] - t2[k]
            M[:, 4, 1 + k] = 0.5 * ga[k] - t3[k]
            for j in range(3):
                M[:, 1 + k, 1 + j] -= gU[k, j]
        M[:, 0, 4] = -math.sqrt(g1) * div / 2
        M[:, 4, 4] -= g1 * div / 2
        eig = torch.linalg.eigvalsh((0.5 * (M + M.transpose(1, 2))).cpu())[:, -1].to(u.device)
        m2 = eig * scaling / torch.sqrt((eig * eig * self.V).sum() / self.V.sum())
        P, N = self.P[:self.nIF], self.N[:self.nIF]
        DT = m2[P] * self.w[:self.nIF] + m2[N] * (1 - self.w[:self.nIF])
        k = self.A[:self.nIF] * DT / self.delta[:self.nIF] * dt
        faces = self.slots.clamp(max=self.nIF - 1)
        nb = torch.where(P[faces] == torch.arange(self.nIC, device=u.device)[:, None], N[faces], P[faces])
        k = torch.where(self.slots < self.nIF, k[faces], 0.) / self.V[:, None]          # [cells][6]
        diag, b = 1 + k.sum(1), ua / self.V
        phi = b
        for _ in range(iterations):
            phi = (b + (phi[:, nb] * k).sum(2)) / diag
        return phi * self.V, m2


def exact(case, seed):
    setup = _case_setup(case)
    u, ua, S = [a.double() for a in _arrays(case, seed, setup)]
    f, dt, op = _Fp64(case, setup), _dt(case, setup), case['op']
    S = S if case['mesh'] == 'duct' else None
    if op == 'step':
        out, _, J, dtc = f.step(u, dt, S)
        return out, J.reshape(1), dtc.reshape(1)
    if op == 'pa':
        out, us, J, _ = f.step(u, dt, S)
        g, Sbar, vbar = f.adjoint_step(us, dt, ua)
        return [out, J.reshape(1), g] + ([Sbar] if S is not None else []) + \
            ([vbar] if case['mesh'] in ('cyl', 'duct') else [])
    if op == 'residual':
        with torch.no_grad():
            L, _ = f.residual(u, f.value)
        return L, f.transpose(lambda x, y: f.residual(x, y)[0], u, ua)[0]
    if op == 'visc':
        return f.viscosity(u, ua, dt, 1.0, VISC_ITERATIONS)
    stages, J = [], 0.
    for _ in range(20):
        u, us, j, _ = f.step(u, dt)
        stages.append(us)
        J = J + j
    g = torch.zeros_like(u)
    for us in reversed(stages):
        g, _, _ = f.adjoint_step(us, dt, g)
    return J.reshape(1), g
