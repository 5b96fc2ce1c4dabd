"""k_fft_pow2's ways through the levels, bit for bit against the oracle: a deepest
factor of 2 with an even and an odd number of levels (rows and columns of 2 to
2048 elements), a deepest 3, 5 or prime with an even and an odd number of radix-2
levels above it, workgroups that the groups of four do not fill."""
import pytest

from test_gpu_parity import run_pair
from test_gpu_selfgravity import SG

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nrad, nsec", [(4, 2), (4, 4), (8, 8), (16, 64), (32, 128), (6, 2048), (3, 1024), (5, 24),
                                        (10, 48), (12, 80), (7, 160), (14, 14), (20, 28), (96, 1536)])
def test_levels(deck, nrad, nsec):
    run_pair(deck(Nrad=nrad, Nsec=nsec, DT=0.01, **SG), 2, 0.0)
