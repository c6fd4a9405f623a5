"""GPU: large read-backs (staged through pinned slots by several threads) and
the gamma history that the steps write straight to the host."""
import numpy as np
import pytest

import pfdd_amd as pa
from pfdd_amd import configs as C
from pfdd_amd import hip

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module", autouse=True)
def need_gpu():
    if hip.device_count() < 1:
        pytest.skip("no GPU visible")


@pytest.mark.parametrize("prec", [pa.FP64, pa.MIXED, pa.MIXED_LEAN])
@pytest.mark.parametrize("shape,ns", [((8, 8, 8), 3), ((64, 64, 64), 2), ((48, 96, 128), 5)])
def test_read_back_of_every_size(shape, ns, prec):
    """What was uploaded comes back: FP64 bit for bit, the mixed forms as the
    stored halves make it up (hi + lo, or FP32); below and above the size at
    which the read is staged, and with a last stretch shorter than a slot."""
    w = C.small_fcc(shape, ns=ns, nloops=1)
    rng = np.random.default_rng(7)
    z = rng.standard_normal((ns,) + shape) + 1j * rng.standard_normal((ns,) + shape)
    with pa.Context(w.params(prec)) as c:
        c.upload_xi(z)
        got = c.download_xi(ns + 2)
    f = lambda v: v.astype(np.float32).astype(np.float64)  # noqa: E731
    if prec == pa.FP64:
        want = z
    elif prec == pa.MIXED:
        want = f(z.real) + f(z.real - f(z.real)) + 1j * f(z.imag)
    else:
        want = f(z.real) + 1j * f(z.imag)
    assert np.array_equal(got[:ns], want) and np.all(got[ns:] == 0)


def test_gamma_history_over_many_calls():
    """Calls of any length, whose rows run through the history's end more than
    once and are read or not, return the rows of one long call."""
    w = C.small_fcc((16, 16, 32), ns=3)

    def run(chunks):
        with pa.Context(w.params()) as c:
            c.set_tau(w.tau)
            c.upload_xi(w.xi)
            c.begin_outer(True)
            out = []
            for n, record in chunks:
                g, ga = c.gl_steps(n, record)
                if record:
                    out.append(np.column_stack([g, ga]))
                else:
                    out.append(np.full((n, 4), np.nan))
            return np.concatenate(out), c.download_xi()

    g0, x0 = run([(2400, True)])
    chunks = [(1, True), (7, True), (700, True), (300, False), (400, True), (1, True), (983, True), (8, True)]
    g1, x1 = run(chunks)
    assert len(g1) == 2400 and np.array_equal(x0, x1)
    seen = ~np.isnan(g1[:, 0])
    assert seen.sum() == 2100 and np.array_equal(g1[seen], g0[seen])
