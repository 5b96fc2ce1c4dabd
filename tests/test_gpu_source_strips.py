"""k_src's column strips and ring bands at their edges, bit for bit against
the FP64 oracle: rings of one strip at its widest (59 cells) and one cell
more, rings narrower than a wave, disks of a few rings (every ring an edge
case), bands that end with the ghost ring, and the planet potential with
operands near the end of the exponent range (its general form)."""
import pytest

from conftest import write_planets
from test_gpu_fused import run_fused
from test_gpu_fused_adsg import ADI, SG, run_fused_vs_routine

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nrad, nsec", [(9, 5), (12, 59), (12, 60), (7, 118), (7, 119), (3, 64), (4, 177), (131, 700)])
def test_strip_edges(deck, nrad, nsec):
    run_fused(deck(Nrad=nrad, Nsec=nsec), 6)


@pytest.mark.parametrize("smoothing", [1e-60, 0.6])
def test_planet_potential_forms(deck, tmp_path, smoothing):
    cfg = write_planets(tmp_path / "p.cfg", [("A", 1.0, 1e-3, 0.0, "NO", "NO"), ("B", 1.7, 5e-4, 0.0, "NO", "YES"),
                                             ("C", 2.1, 0.0, 0.0, "NO", "NO")])
    run_fused(deck(Nrad=24, Nsec=90, ThicknessSmoothing=smoothing, PlanetConfig=cfg), 6)


@pytest.mark.parametrize("kw", [ADI, SG, dict(ADI, **SG)], ids=["adiabatic", "gravity", "both"])
@pytest.mark.parametrize("nrad, nsec", [(4, 60), (40, 236)])
def test_strip_edges_energy_and_gravity(deck, kw, nrad, nsec):
    run_fused_vs_routine(deck(Nrad=nrad, Nsec=nsec, DT=0.01, **kw), 5, "Adiabatic" in kw, sg="SelfGravity" in kw)
