"""k_src32's column strips and ring bands at their edges: rings of one strip at
its widest (59 cells) and one cell more, rings narrower than a wave, disks of a
few rings, bands that end with the ghost ring.  Against the FP64 path within
the FP32 bulk mode's bounds, and bit for bit for every band (a cell's result
does not depend on the strip and band that evaluate it), alone and batched,
with planets beyond the first."""
import ctypes

import numpy as np
import pytest

from conftest import write_planets
from cudaprotoplanetarydisks_amd import Simulation
from cudaprotoplanetarydisks_amd.ensemble import Ensemble
from cudaprotoplanetarydisks_amd.native import call, lib
from test_gpu_fp32 import DENS_LINF, VEL_LINF

pytestmark = pytest.mark.gpu

STEPS = 5
PD = ctypes.POINTER(ctypes.c_double)


def run(path, precision, tiles=None):
    with Simulation(path, precision=precision, fused=True) as s:
        if tiles:
            call("fg_set_tiles", lib().fg_sim_ctx(s.h), *tiles)
        for _ in range(STEPS):
            s.substep()
        return [a[:-1].copy() for a in s.state()]


@pytest.mark.parametrize("nrad, nsec", [(9, 5), (12, 59), (12, 60), (7, 118), (7, 119), (3, 64), (4, 177), (131, 700)])
def test_strips_and_bands(deck, tmp_path, nrad, nsec):
    cfg = write_planets(tmp_path / "p.cfg", [("A", 1.0, 1e-3, 0.0, "NO", "NO"), ("B", 1.7, 5e-4, 0.0, "NO", "NO"),
                                             ("C", 2.1, 1e-4, 0.0, "NO", "NO")])
    path = deck(Nrad=nrad, Nsec=nsec, PlanetConfig=cfg)
    ref = run(path, "fp64")
    base = run(path, "fp32")
    for a, b, bound in zip(base, ref, (DENS_LINF, VEL_LINF, VEL_LINF)):
        assert np.abs(a - b).max() <= bound * np.abs(b).max()
    for tiles in ((8, 8), (16, 5), (32, 64)):
        for a, b in zip(run(path, "fp32", tiles), base):
            assert np.array_equal(a, b), tiles
    with Ensemble([path, path], tiles={}) as ens:
        ens.set_tiles(1, 8, 3)
        for _ in range(STEPS):
            ens.substep(1e30)
        for k in range(2):
            got = [np.empty((nrad + 1, nsec)) for _ in range(3)]
            call("fg_sim_get_state", ens.sim_handle(k), *[a.ctypes.data_as(PD) for a in got], None)
            for a, b in zip(got, base):
                assert np.array_equal(a[:-1], b), k
