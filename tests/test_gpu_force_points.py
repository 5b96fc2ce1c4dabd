"""The disk force on several planets summed at once: planets that feel the disk
between ones that do not, none, one and as many as a system can have, on both
paths bit for bit against the oracle, in the FP32 bulk mode against FP64."""
import numpy as np
import pytest

from conftest import write_planets
from cudaprotoplanetarydisks_amd import Simulation
from test_gpu_fused import run_fused
from test_gpu_parity import run_pair

pytestmark = pytest.mark.gpu

FEEL = {"none": "NN", "one": "Y", "mixed": "NYNYYN", "sixteen": "Y" * 16}


def planets(tmp_path, feel):
    return write_planets(tmp_path / "p.cfg", [(f"P{k}", 0.6 + 0.11 * k, 1e-4 * (1 + k % 3), 0.0,
                                               "YES" if c == "Y" else "NO", "YES") for k, c in enumerate(feel)])


@pytest.mark.parametrize("feel", sorted(FEEL))
def test_force_points(deck, tmp_path, feel):
    cfg = planets(tmp_path, FEEL[feel])
    run_pair(deck(Nrad=20, Nsec=70, PlanetConfig=cfg), 4, 0.0)
    run_pair(deck(Nrad=20, Nsec=70, PlanetConfig=cfg, InnerBoundary="OPEN"), 4, 0.0)
    path = deck(Nrad=20, Nsec=70, PlanetConfig=cfg)
    run_fused(path, 4)
    out = {}
    for precision in ("fp64", "fp32"):
        with Simulation(path, precision=precision, fused=True) as s:
            for _ in range(4):
                s.substep()
            out[precision] = s.planets()
    # a force is a sum of Sigma, within 1e-5 (the mode's bound) of its magnitude
    # per substep; the disk's pull is below 1e-2 of the star's and dt below 0.1
    assert np.abs(out["fp32"] - out["fp64"]).max() <= 4 * 1e-5 * 1e-2 * 0.1
