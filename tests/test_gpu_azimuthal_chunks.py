"""k_tazw's chunks of two cells a lane (119 cells) and of three (183 cells, from
2^20 cells on) at their edges: rings of one chunk, of one cell more and of two
chunks, on both paths bit for bit against the oracle; in the FP32 bulk mode bit
for bit against a batch, whose chunks are always of two cells a lane, and
Sigma within the mode's bound of FP64."""
import ctypes

import numpy as np
import pytest

from cudaprotoplanetarydisks_amd import Simulation
from cudaprotoplanetarydisks_amd.ensemble import Ensemble
from cudaprotoplanetarydisks_amd.native import call
from test_gpu_fp32 import DENS_LINF
from test_gpu_fused import run_fused
from test_gpu_parity import run_pair

pytestmark = pytest.mark.gpu

GRIDS = [(6, 118), (6, 119), (6, 120), (6, 238), (6, 239), (5731, 183), (5700, 184), (2866, 366), (2866, 367)]
PD = ctypes.POINTER(ctypes.c_double)


@pytest.mark.parametrize("nrad, nsec", GRIDS)
def test_chunks(deck, nrad, nsec):
    path = deck(Nrad=nrad, Nsec=nsec, DT=0.001)
    _, orc = run_fused(path, 2)
    run_pair(path, 1, 0.0)
    with Simulation(path, precision="fp32") as s, Ensemble([path], tiles={}) as ens:
        for _ in range(2):
            s.substep()
            ens.substep(1e30)
        single = s.state()[:3]
        batch = [np.empty((nrad + 1, nsec)) for _ in single]
        call("fg_sim_get_state", ens.sim_handle(0), *[a.ctypes.data_as(PD) for a in batch], None)
    for a, b in zip(single, batch):
        assert np.array_equal(a[:-1], b[:-1])
    want = orc.field("Dens")[:-1]
    assert np.abs(single[0][:-1] - want).max() <= DENS_LINF * np.abs(want).max()
