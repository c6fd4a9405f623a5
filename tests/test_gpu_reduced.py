"""GPU parity of the reduced-basis GL step (AUTO on grids whose N1 and N3 have
fused kernels): against the FP64 oracle and against the field-major kernels,
for every number of components, at every fused length of either axis, with
each option of the update.

Tolerances: FP64 as in the other parity tests (1e-12 against the oracle after
12 steps); the FP32 modes differ from their field-major runs by the FP32
rounding of the transforms (a few 2^-24 of values of order 1 a step): 2e-6."""
import sys

import numpy as np
import pytest

import oraclepy as O
import pfdd_amd as pa
from pfdd_amd import configs as C
from pfdd_amd import hip

pytestmark = pytest.mark.gpu
PRECS = [pa.FP64, pa.MIXED, pa.MIXED_LEAN]
FUSED = (32, 48, 64, 96, 128, 192, 256, 384, 512)


@pytest.fixture(scope="module", autouse=True)
def need_gpu():
    if hip.device_count() < 1:
        pytest.skip("no GPU visible")


def options(w, masked, tau_pp):
    rng = np.random.default_rng(17)
    bc = None
    if masked:
        bc = (rng.random((w.ns,) + w.shape) < 0.1).astype(np.complex128)
    tau = rng.uniform(-0.02, 0.02, (w.P, w.ns)) if tau_pp else w.tau
    return bc, tau


def gpu(w, plan, prec, steps=12, bc=None, tau=None, quirk=True, bmode=pa.B_RECOMPUTE, eps=None, chunks=()):
    p = w.params(prec, bmode, plan)
    with pa.Context(p) as c:
        c.set_tau(w.tau if tau is None else tau, per_point=tau is not None and np.ndim(tau) == 2)
        c.upload_xi(w.xi, bc)
        c.begin_outer(quirk)
        out = [c.gl_steps(n)[1] for n in (chunks or (steps,))]
        return c.download_xi(), np.concatenate(out)


def oracle(w, steps=12, bc=None, tau=None, quirk=True):
    o = O.Oracle(O.make_params(w.shape, w.eps, C.C11, C.C12, C.C44, [0.1] * w.ns, C.asf2_reference(w.ns),
                               [1.0] * w.ns))
    o.set_xi(w.xi, bc)
    o.set_tau(w.tau if tau is None else tau, per_point=tau is not None and np.ndim(tau) == 2)
    o.prologue(quirk)
    _, ga = o.gl_steps(steps)
    x = o.get_xi()
    o.close()
    return x, ga


def check(w, prec, bc=None, tau=None, quirk=True, bmode=pa.B_RECOMPUTE):
    tau_arg = tau if tau is not None and np.ndim(tau) == 2 else None
    x1, g1 = gpu(w, pa.PLAN_AUTO, prec, bc=bc, tau=tau_arg, quirk=quirk, bmode=bmode)
    if prec == pa.FP64:
        xo, go = oracle(w, bc=bc, tau=tau_arg, quirk=quirk)
        assert np.abs(x1 - xo).max() <= 1e-12
        assert np.abs(g1 - go).max() <= 1e-12
    else:
        x0, g0 = gpu(w, pa.PLAN_FIELD_MAJOR | pa.PLAN_NO_PLANE, prec, bc=bc, tau=tau_arg, quirk=quirk, bmode=bmode)
        assert np.abs(x1 - x0).max() <= 2e-6
        assert np.abs(g1 - g0).max() <= 2e-6


@pytest.mark.parametrize("prec", PRECS)
@pytest.mark.parametrize("ns", range(1, 13))
def test_component_counts(ns, prec):
    """ns = 1..12 of the FCC systems: 1, 2, 2, 3, 4, 4, 5 ... 5 components."""
    check(C.small_fcc((32, 4, 32), ns=ns), prec)


def test_six_components():
    """Strains with a trace (no slip systems) span all six dimensions."""
    w = C.small_fcc((32, 2, 32), ns=7)
    rng = np.random.default_rng(3)
    w.eps = w.eps + 0.3 * rng.standard_normal(w.eps.shape)
    check(w, pa.FP64)


@pytest.mark.parametrize("prec", PRECS)
@pytest.mark.parametrize("n", FUSED)
def test_lengths_of_the_row_and_column_kernels(n, prec):
    """Each length along N1 and along N3, five components and two; N2 = 3 and 6."""
    for shape, ns in (((n, 3, 32), 12), ((32, 6, n), 12), ((n, 2, 48), 3), ((48, 3, n), 3)):
        check(C.small_fcc(shape, ns=ns, nloops=3), prec)


@pytest.mark.parametrize("prec", PRECS)
@pytest.mark.parametrize("masked,tau_pp", [(True, False), (False, True), (True, True)])
def test_frozen_points_and_per_point_shear(masked, tau_pp, prec):
    w = C.small_fcc((48, 6, 64), ns=5)
    bc, tau = options(w, masked, tau_pp)
    check(w, prec, bc=bc, tau=tau)
    if masked:
        x, _ = gpu(w, pa.PLAN_AUTO, pa.FP64, bc=bc)
        assert np.array_equal(x[bc != 0], w.xi[bc != 0])


@pytest.mark.parametrize("quirk", [True, False])
def test_prologue_term_and_first_step(quirk):
    """The prologue's per-field term enters the first update only, however the
    steps are split over calls (eager first step, graph replays, eager rest)."""
    w = C.small_fcc((32, 8, 32), ns=6)
    check(w, pa.FP64, quirk=quirk)
    x1, g1 = gpu(w, pa.PLAN_AUTO, pa.FP64, quirk=quirk, chunks=(21,))
    x2, g2 = gpu(w, pa.PLAN_AUTO, pa.FP64, quirk=quirk, chunks=(1, 8, 9, 3))
    assert np.array_equal(x1, x2) and np.array_equal(g1, g2)


@pytest.mark.parametrize("prec", PRECS)
def test_ensemble_class_equals_single(prec):
    """Instances of a batched class get the bits of their own contexts."""
    members = [C.small_fcc((32, 4, 48), ns=3, seed=C.BASE_SEED + 500 + i) for i in range(3)]
    with pa.Ensemble([m.params(prec) for m in members]) as e:
        for i, m in enumerate(members):
            e.set_tau(i, m.tau)
            e.upload_xi(i, m.xi)
        e.begin_outer(True)
        g = e.gl_steps(19)
        for i, m in enumerate(members):
            x, ga = gpu(m, pa.PLAN_AUTO, prec, steps=19)
            assert np.array_equal(e.download_xi(i), x)
            assert np.abs(g[:, i] - ga.sum(1)).max() <= 1e-14


SHORT = (2, 3, 4, 6, 8, 12, 16, 24)


@pytest.mark.parametrize("prec", PRECS)
@pytest.mark.parametrize("n", SHORT)
def test_short_axes(n, prec):
    """Lengths below 32 along N1 or N3, where blocks hold several rows or many
    columns and N1 N2 rows (or N2 N3 columns) are no multiple of a block's."""
    for shape, ns in (((n, 3, 32), 1), ((3, 6, n), 6), ((n, 2, 2), 12), ((48, 3, n), 3), ((2, 3, n), 4)):
        w = C.small_fcc(shape, ns=ns, nloops=2, rmin=1.0, rmax=2.0)
        bc, tau = options(w, ns == 6, ns == 4)
        check(w, prec, bc=bc, tau=tau)


@pytest.mark.parametrize("sizes", [(16, 32), (16, 24, 32, 48, 12, 8)])
def test_classes_on_parallel_branches(sizes):
    """Fewer and more classes than a graph has branches, in different
    precisions; replays, eager steps between them and a new prologue:
    bit-identical to each instance alone."""
    ws = [C.small_fcc((n, n, n), ns=1 + k % 4, seed=C.BASE_SEED + 700 + k) for k, n in enumerate(sizes)]
    precs = [PRECS[k % 3] for k in range(len(ws))]
    calls = (19, 8, 3, 17)
    with pa.Ensemble([w.params(p) for w, p in zip(ws, precs)]) as e:
        for i, w in enumerate(ws):
            e.set_tau(i, w.tau)
            e.upload_xi(i, w.xi)
        g = []
        for n in calls:
            e.begin_outer(True)
            g.append(e.gl_steps(n))
        got = [e.download_xi(i) for i in range(len(ws))]
    for i, (w, p) in enumerate(zip(ws, precs)):
        with pa.Context(w.params(p)) as c:
            c.set_tau(w.tau)
            c.upload_xi(w.xi)
            gs = []
            for n in calls:
                c.begin_outer(True)
                gs.append(c.gl_steps(n)[0])
            assert np.array_equal(c.download_xi(), got[i]), i
        assert np.array_equal(np.concatenate(gs), np.concatenate(g)[:, i]), i


@pytest.mark.parametrize("prec", PRECS)
@pytest.mark.parametrize("n1", sorted(SHORT + FUSED))
def test_both_sides_of_the_plane_kernel(n1, prec):
    """The largest N2 whose N1 x N2 plane is transformed in one launch, and
    the smallest that takes the N2 passes and the column kernel."""
    for ns, n3 in ((3, 8), (12, 3)):
        last = None
        for n2 in sorted(SHORT + FUSED):
            w = C.small_fcc((n1, n2, n3), ns=ns, nloops=3)
            with pa.Context(w.params(prec)) as c:
                plane = c.step_plan()[pa.STAGE_FFT_AXIS2] == 0
            if not plane:
                break
            last = w
        assert not plane
        check(w, prec)
        if last is not None:
            check(last, prec)
        check(w, prec, bmode=pa.B_STORED)
        if last is not None:
            check(last, prec, bmode=pa.B_STORED)


@pytest.mark.parametrize("prec", PRECS)
@pytest.mark.parametrize("n1,n2,ns", [(32, 32, 4), (24, 32, 5), (8, 96, 5), (48, 16, 4), (16, 32, 12)])
def test_large_planes(n1, n2, ns, prec):
    """Planes that take one launch only when there are many of them."""
    w = C.small_fcc((n1, n2, 128), ns=ns, nloops=3)
    with pa.Context(w.params(prec)) as c:
        assert c.step_plan()[pa.STAGE_FFT_AXIS2] == 0
    check(w, prec)


@pytest.mark.parametrize("prec", PRECS)
@pytest.mark.parametrize("n1", [384, 512])
@pytest.mark.parametrize("ns", [1, 3, 4, 5, 6])
def test_wide_column_tiles(n1, ns, prec):
    """Column counts that are no multiple of the tiles at the longest N1."""
    check(C.small_fcc((n1, 3, 6), ns=ns, nloops=2), prec)
    check(C.small_fcc((n1, 3, 6), ns=ns, nloops=2), prec, bmode=pa.B_STORED)
