"""The tile kernel (schedule 3, block width 64, and what a handle runs until a shape is chosen)
against the single-step kernel it must reproduce bit for bit: from a random state, on grids at the
remainders of its 52-column tiles and 12-, 20- and 36-row tiles, with a material palette, one beyond the
marching kernel's limit and none, in both precisions, over odd and even step counts."""
import numpy as np
import pytest

from poe2d_amd import _abi
from poe2d_amd.configs import BRINE, biot_fields
from poe2d_amd.material import material_biot
from poe2d_amd.solver import Batch, Problem, ReceiverSpec, Solver, SourceSpec

from .helpers import device_memory_free

pytestmark = pytest.mark.gpu

STATE = ("vx", "vy", "wx", "wy", "exx", "eyy", "zeta", "sxy")


def _problem(nx, nz, npml, entries, seed=3, **opts):
    rng = np.random.default_rng(seed)
    p = biot_fields(nx, nz)
    if entries:  # `entries` materials in random places; 0: every point its own
        p["phi"] = 0.2 + 0.1 * rng.integers(0, entries, p["phi"].shape) / entries
    else:
        p["phi"] = rng.uniform(0.2, 0.3, p["phi"].shape)
        p["mu_fr"] = BRINE["mu_fr"] * rng.uniform(0.9, 1.1, p["phi"].shape)
    ix = np.unique(np.clip([0, 5, 51, 52, 53, nx // 2, nx - 1, nx], 0, nx)).astype(np.int32)
    iz = np.unique(np.clip([0, 11, 12, 35, 36, nz // 2, nz], 0, nz)).astype(np.int32)
    gx, gz = (a.ravel() for a in np.meshgrid(ix, iz))
    return Problem(nx=nx, nz=nz, dx=0.5, dz=0.5, dt=5e-5, nt=9, coeffs=material_biot(**p),
                   source=SourceSpec(kind=_abi.SRC_PRESSURE_DGAUSS, ix=nx // 2, iz=nz // 2, amp=1e6),
                   receivers=ReceiverSpec(ix=gx, iz=gz, decimate=2), npml=npml, f0=80.0, **opts)


def _run(prob, precision, shape, steps):
    with Solver(prob, precision=precision) as s:
        rng = np.random.default_rng(11)
        if shape:
            s.set_schedule(*shape)
        for f in STATE:
            s.set_field(f, rng.standard_normal((prob.nz + 1, prob.nx + 1)) * (1e-9 if f[0] in "ez" else 1e-6))
        for n in steps:
            s.run(n)
        return s.seismograms(), {f: s.snapshot(f) for f in STATE + ("p",)}, s.checkpoint()


def _same(a, b, label):
    assert np.isfinite(a[0]).all() and np.abs(a[0]).max() > 0
    assert np.array_equal(a[0], b[0]), f"{label}: traces differ"
    for f in a[1]:
        assert np.array_equal(a[1][f], b[1][f]), f"{label}: field {f} differs"
    assert np.array_equal(a[2], b[2]), f"{label}: checkpoint differs"


@pytest.mark.parametrize("nx,nz,npml", [(10, 10, 1), (51, 47, 4), (103, 107, 20), (104, 131, 10), (230, 171, 20)])
@pytest.mark.parametrize("entries", [2, 40, 0])
@pytest.mark.parametrize("precision", [32, 64])
def test_tiles_equal_the_single_step_kernel(nx, nz, npml, entries, precision):
    prob = _problem(nx, nz, npml, entries)
    ref = _run(prob, precision, (0, 256, 14), [9])
    for shape, steps in (((3, 64, 12), [4, 5]), ((3, 64, 36), [9]), ((3, 64, 6), [8, 1]), ((3, 64, 30), [2, 7]),
                         (None, [1, 2, 6])):
        _same(_run(prob, precision, shape, steps), ref, f"{nx}x{nz} npml {npml} {entries} entries shape {shape}")


@pytest.mark.parametrize("nz", [40, 41, 42, 57, 58])
@pytest.mark.parametrize("entries", [2, 0])
@pytest.mark.parametrize("precision", [32, 64])
def test_tile_bands_at_the_heights_of_their_tiles(nz, entries, precision):
    """Edge and tall bands of 19 to 37 rows (13 to 31 with three steps): one row less, as many and one
    more than a tile of 20 or 36 (14 or 30) takes."""
    prob = _problem(150, nz, 4, entries)
    ref = _run(prob, precision, (0, 256, 14), [6])
    for shape in ((3, 64, 36), (3, 64, 30), (3, 64, 12)):
        _same(_run(prob, precision, shape, [6]), ref, f"{nz} rows {entries} entries shape {shape}")


@pytest.mark.parametrize("opts", [dict(stress_law=1), dict(staggered_material=1)])
@pytest.mark.parametrize("entries", [2, 0])
@pytest.mark.parametrize("precision", [32, 64])
def test_tiles_physics_variants(opts, entries, precision):
    prob = _problem(230, 171, 20, entries, **opts)
    _same(_run(prob, precision, (3, 64, 36), [9]), _run(prob, precision, (0, 256, 14), [9]), f"{opts} {entries}")


def test_ragged_fp64_batch_on_tiles():
    probs = [_problem(130, 90, 10, 2, seed=1), _problem(61, 200, 10, 2, seed=2)]
    alone = [_run(p, 64, (0, 256, 14), [9])[0] for p in probs]
    solvers = [Solver(p, precision=64) for p in probs]
    rng = [np.random.default_rng(11) for _ in probs]
    for s, g in zip(solvers, rng):
        for f in STATE:
            s.set_field(f, g.standard_normal((s.problem.nz + 1, s.problem.nx + 1)) * (1e-9 if f[0] in "ez" else 1e-6))
    with Batch(solvers) as b:
        b.run(9)
        for s, ref in zip(solvers, alone):
            assert np.array_equal(s.seismograms(), ref)
    for s in solvers:
        s.close()


@pytest.mark.parametrize("precision", [32, 64])
def test_reset_after_a_run_starts_from_zero(precision):
    # reset clears the buffer the next step reads; a run after it equals a new handle's, whichever
    # buffer the earlier run ended in and whichever kernel ran before
    prob = _problem(104, 131, 10, 2)
    ref = None
    for before in (None, (3, 64, 36), (0, 256, 14), (1, 256, 14)):
        with Solver(prob, precision=precision) as s:
            if before:
                s.set_schedule(*before)
                s.set_field("vx", np.ones((prob.nz + 1, prob.nx + 1)) * 1e-6)
                s.run(5)
                s.reset()
                s.set_schedule(3, 64, 36)
            s.run(9)
            got = s.seismograms(), {f: s.snapshot(f) for f in STATE}, s.checkpoint()
        if ref is None:
            ref = got
        _same(got, ref, f"after {before}")


@pytest.mark.parametrize("shape", [(1, 1), (3, 2), (33, 31), (64, 65), (5, 1000)])
def test_traces_keep_their_order(shape):
    # (samples, receivers) around the transposing kernel's 32 x 32 tiles: trace k of receiver r is
    # what a snapshot holds at its point
    nt, nrec = shape
    rng = np.random.default_rng(nt)
    prob = _problem(104, 131, 10, 2)
    prob.receivers = ReceiverSpec(ix=rng.integers(0, 105, nrec), iz=rng.integers(0, 132, nrec), comp_mask=_abi.VX | _abi.P)
    prob.nt = nt
    with Solver(prob) as s:
        s.set_field("vx", rng.standard_normal((132, 105)) * 1e-6)
        snaps = []
        for _ in range(nt):
            snaps.append(s.snapshot("vx")[prob.receivers.iz, prob.receivers.ix])
            s.run(1)
        g = s.seismograms()
    assert g.shape == (2, nrec, nt)
    assert np.array_equal(g[0], np.stack(snaps, axis=1))


@pytest.mark.parametrize("precision", [32, 64])
def test_long_traces_are_read_in_parts(precision):
    # 600 traces of a million samples (2.4 GB in FP32): reading them takes less than 128 MB more, 16 (8 in
    # FP64) of them at a time, and every one holds what a short record of the same points holds
    rng = np.random.default_rng(2)
    prob = _problem(104, 131, 10, 2)
    prob.receivers = ReceiverSpec(ix=rng.integers(0, 105, 200), iz=rng.integers(0, 132, 200))
    got = []
    for nsamp in (7, 1000000):
        prob.receivers.nsamp = nsamp
        with Solver(prob, precision=precision) as s:
            s.set_field("vx", rng.standard_normal((132, 105)) * 1e-6 if not got else vx)
            vx = s.snapshot("vx")
            s.run(7)
            before = device_memory_free()
            g = s.seismograms()
            assert before - device_memory_free() < 128 << 20
            got.append(g[..., :7])
            assert not g[..., 7:].any()
    assert np.abs(got[0]).max() > 0 and np.array_equal(got[0], got[1])


@pytest.mark.parametrize("opts", [dict(), dict(staggered_material=1)])
@pytest.mark.parametrize("entries", [2, 40, 0])
@pytest.mark.parametrize("precision", [32, 64])
def test_launches_of_more_tiles_than_compute_units(opts, entries, precision):
    """Over 256 tiles, an FP32 launch runs two blocks to a CU: half the registers, profiles of the columns in
    LDS, coefficients read where they are used.  46 to 92 MB of state are also stored through the caches
    (smaller launches store past them).  Receivers stand on the edges of 46- and 52-column tiles."""
    prob = _problem(900, 800, 20, entries, **opts)
    ix = np.unique([0, 1, 45, 46, 47, 51, 52, 53, 91, 92, 103, 104, 459, 460, 467, 468, 850, 899, 900]).astype(np.int32)
    iz = np.unique([0, 1, 26, 29, 30, 35, 36, 61, 62, 400, 401, 772, 799, 800]).astype(np.int32)
    gx, gz = (a.ravel() for a in np.meshgrid(ix, iz))
    prob.receivers = ReceiverSpec(ix=gx, iz=gz)
    ref = _run(prob, precision, (0, 256, 14), [7])
    for shape, steps in (((3, 64, 36), [7]), ((3, 64, 30), [5, 2]), ((3, 64, 12), [7]), ((3, 64, 6), [7]), (None, [4, 3])):
        _same(_run(prob, precision, shape, steps), ref, f"{opts} {entries} entries shape {shape}")


@pytest.mark.parametrize("precision", [32, 64])
def test_batch_of_palette_and_continuous_members_on_tiles(precision):
    # the whole batch reads the coefficient groups; large enough for more tiles than compute units
    probs = [_problem(520, 610, 10, 2, seed=1), _problem(430, 500, 10, 0, seed=2), _problem(61, 200, 10, 40, seed=3)]
    alone = [_run(p, precision, (0, 256, 14), [9]) for p in probs]
    solvers = [Solver(p, precision=precision) for p in probs]
    for s in solvers:
        g = np.random.default_rng(11)
        for f in STATE:
            s.set_field(f, g.standard_normal((s.problem.nz + 1, s.problem.nx + 1)) * (1e-9 if f[0] in "ez" else 1e-6))
    with Batch(solvers) as b:
        b.run(4)
        b.run(5)
        for s, ref in zip(solvers, alone):
            _same((s.seismograms(), {f: s.snapshot(f) for f in STATE + ("p",)}, s.checkpoint()), ref, "batch")
    for s in solvers:
        s.close()


@pytest.mark.parametrize("after", [(0, 256, 14), (1, 256, 14), (2, 256, 14), (3, 256, 24), (3, 64, 36), None])
@pytest.mark.parametrize("before", [(0, 256, 14), (1, 256, 14), (3, 256, 24), (3, 64, 30), None])
def test_reset_clears_what_any_kernel_reads(before, after):
    # every field set at every point (the border's too), or infinite somewhere, whichever buffer and kernel
    # it ran on: after a reset every kernel starts from zero
    prob = _problem(104, 131, 10, 2)
    rng = np.random.default_rng(1)
    noise = {f: rng.standard_normal((132, 105)) * (1e-9 if f[0] in "ez" else 1e-6) for f in STATE}
    with Solver(prob) as s:
        if after:
            s.set_schedule(*after)
        s.run(9)
        ref = s.seismograms(), {f: s.snapshot(f) for f in STATE}, s.checkpoint()
    for broken in (False, True):
        with Solver(prob) as s:
            if before:
                s.set_schedule(*before)
            for f in STATE:
                s.set_field(f, noise[f])
            if broken:
                s.set_field("vy", np.where(rng.random((132, 105)) < 0.01, np.inf, noise["vy"]))
                with pytest.raises(_abi.Poe2dError):
                    s.run(4)
            else:
                s.run(5)
            s.reset()
            if after or before:
                s.set_schedule(*(after or (3, 64, 30)))
            s.run(9)
            _same((s.seismograms(), {f: s.snapshot(f) for f in STATE}, s.checkpoint()), ref, f"{before} then {after}")
