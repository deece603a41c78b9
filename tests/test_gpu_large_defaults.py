"""What a handle runs by default on large grids (a single last step on the single-step kernel, the marching
kernel for averaged material) against the single-step kernel, bit for bit, from a random state."""
import numpy as np
import pytest

from poe2d_amd import _abi
from poe2d_amd.configs import BRINE, biot_fields
from poe2d_amd.material import material_biot
from poe2d_amd.solver import Batch, Problem, ReceiverSpec, Solver, SourceSpec

from .test_gpu_tiles import STATE, _run, _same

pytestmark = pytest.mark.gpu


def problem(nx, nz, entries, **opts):
    """A 211 x 211 block of random materials repeated over the grid."""
    n, rng = 211, np.random.default_rng(nx)
    p = biot_fields(n - 1, n - 1)
    if entries:
        p["phi"] = 0.2 + 0.1 * rng.integers(0, entries, p["phi"].shape) / entries
    else:
        p["phi"] = rng.uniform(0.2, 0.3, p["phi"].shape)
        p["mu_fr"] = BRINE["mu_fr"] * rng.uniform(0.9, 1.1, p["phi"].shape)
    reps = (nz // n + 1, nx // n + 1)
    coeffs = {k: np.tile(v.astype(np.float32), reps)[:nz + 1, :nx + 1] for k, v in material_biot(**p).items()}
    ix = np.unique(np.linspace(0, nx, 40).astype(np.int32))
    gx, gz = (a.ravel() for a in np.meshgrid(ix, np.array([0, 35, 36, nz // 2, nz], np.int32)))
    return Problem(nx=nx, nz=nz, dx=0.5, dz=0.5, dt=5e-5, nt=4, coeffs=coeffs,
                   source=SourceSpec(kind=_abi.SRC_PRESSURE_DGAUSS, ix=nx // 2, iz=nz // 2, amp=1e6),
                   receivers=ReceiverSpec(ix=gx, iz=gz), npml=20, f0=80.0, **opts)


@pytest.mark.parametrize("nx,nz,entries,precision", [(2449, 2449, 2, 64), (599, 10007, 0, 64), (9000, 700, 2, 64),
                                                     (5003, 4001, 0, 32)])
@pytest.mark.parametrize("steps", [(1, 3), (4,)])
def test_single_last_steps_of_large_grids(nx, nz, entries, precision, steps):
    prob = problem(nx, nz, entries)
    _same(_run(prob, precision, None, steps), _run(prob, precision, (0, 256, 14), [4]), f"{nx}x{nz} {precision} {steps}")


def test_single_last_steps_of_a_large_batch():
    probs = [problem(1731, 1733, 2), problem(2100, 1480, 2)]  # 6.1 M points together
    alone = [_run(p, 64, (0, 256, 14), [4]) for p in probs]
    solvers = [Solver(p, precision=64) for p in probs]
    for s in solvers:
        g = np.random.default_rng(11)
        for f in STATE:
            s.set_field(f, g.standard_normal((s.problem.nz + 1, s.problem.nx + 1)) * (1e-9 if f[0] in "ez" else 1e-6))
    with Batch(solvers) as b:
        b.run(1)
        b.run(3)
        for s, ref in zip(solvers, alone):
            _same((s.seismograms(), {f: s.snapshot(f) for f in STATE + ("p",)}, s.checkpoint()), ref, "batch")
    for s in solvers:
        s.close()


@pytest.mark.parametrize("steps", [(1, 2, 1), (4,)])
def test_averaged_material_on_a_large_grid(steps):
    prob = problem(5200, 3900, 0, staggered_material=_abi.MATERIAL_AVERAGED)
    _same(_run(prob, 32, None, steps), _run(prob, 32, (0, 256, 14), [4]), f"averaged {steps}")
