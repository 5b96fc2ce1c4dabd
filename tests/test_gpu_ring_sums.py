"""The ring sums of a workgroup (ring_seq_sum) against the left-to-right sum that
they stand for, bit for bit: the shortest rings that are added up so (640 cells)
and one cell less, remainders of the lanes' shares, the longest rings; sums of
one sign, of both, through zero, in ties at every addition, that hit powers of
two, over many magnitudes; infinities and NaN."""
import numpy as np
import pytest

from cudaprotoplanetarydisks_amd import Simulation
from cudaprotoplanetarydisks_amd.native import call

pytestmark = pytest.mark.gpu

NRAD = 16


def rows(ns, seed):
    rng = np.random.default_rng(seed)
    odd = lambda scale: (2 * rng.integers(0, 1 << 20, ns) + 1) * scale  # noqa: E731
    out = [rng.uniform(0.9, 1.1, ns), -rng.uniform(0.01, 1.9, ns), rng.normal(0.0, 1.0, ns),
           1.0 + odd(2.0**-42), 1.0 + odd(2.0**-43), -1.0 - odd(2.0**-44), np.ones(ns), np.zeros(ns),
           np.where(np.arange(ns) % 2, 1.0, -1.0), 10.0**rng.uniform(-12, 0.4, ns),
           np.where(np.arange(ns) == ns // 2, -float(ns) / 4, 1.0) / 64, np.full(ns, -0.0),
           np.cos(np.arange(ns) * 2 * np.pi / ns), np.full(ns, 1.0 + 2.0**-30), np.full(ns, 2.0 - 2.0**-52),
           np.sort(rng.uniform(0, 1, ns))]
    return np.array(out)


def means(a):
    return np.cumsum(a, axis=1)[:, -1] / a.shape[1]  # (cumsum adds left to right)


@pytest.mark.parametrize("ns", [3, 512, 639, 640, 641, 768, 1000, 1025, 1536, 2047, 3072, 4096, 8192])
def test_ring_means(deck, ns):
    with Simulation(deck(Nrad=NRAD, Nsec=ns, InnerBoundary="OPEN", Viscosity=None, AlphaViscosity=1e-3)) as s:
        c = s.ctx
        for seed in range(3):
            a = np.zeros((NRAD + 1, ns))
            a[:-1] = rows(ns, seed)
            want = means(a[:-1])
            # (-0.0 / ns of a ring of -0.0 is 0.0: the sum starts at 0.0)
            want = np.where(want == 0.0, 0.0, want)
            c.set_field("SOUNDSPEED", a)
            call("fg_ring_mean_cs", c.h)
            assert np.array_equal(c.rings()["cs_mean"], want)
            c.set_field("VTHETA", a)
            call("fg_transport", c.h, 1e-4, 1.0, None)
            assert np.array_equal(c.rings()["vmed"], want)
        a[:-1] = rows(ns, 9)
        a[0, ns // 3] = np.nan
        a[1, ns - 1] = np.inf
        a[2, 0], a[2, ns // 2] = np.inf, -np.inf
        a[3, :] *= 1e305
        a[4, :] *= 1e-308
        with np.errstate(all="ignore"):
            want = means(a[:-1])
        want = np.where(want == 0.0, 0.0, want)
        c.set_field("SOUNDSPEED", a)
        call("fg_ring_mean_cs", c.h)
        assert np.array_equal(c.rings()["cs_mean"], want, equal_nan=True)


@pytest.mark.parametrize("nrad, ns", [(8, 200), (6, 1153), (5, 3072), (4, 3073), (4, 4096)])
def test_ring_means_of_a_substep(deck, nrad, ns):
    with Simulation(deck(Nrad=nrad, Nsec=ns, DT=0.01), fused=True) as s:
        for _ in range(3):
            s.substep()
            vt = s.state()[2][:-1]
            assert np.array_equal(s.ctx.rings()["vmoy"], means(vt))
