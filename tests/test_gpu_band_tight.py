"""The banded LU factorisation where the LDS holds the window of a step but not the next row and column
beside it: bit for bit against the oracle at the edges of that range, and as fast as next to it."""
import pytest

from tests.test_gpu_band_window import test_factors_match_the_oracle as factors_match
from tests.test_gpu_neighbours import micros, ra  # noqa: F401

pytestmark = pytest.mark.gpu


# (kl + 2)(kl + ku + 2) doubles above 160 KB, (kl + 1)(kl + ku + 1) below or at it; the last one
# above it; matrices larger than the window and smaller
@pytest.mark.parametrize("n,kl,ku", [(700, 30, 612), (60, 30, 612), (1060, 18, 1005), (240, 100, 101), (300, 142, 0),
                                     (143, 142, 0), (400, 63, 255), (330, 63, 256), (500, 30, 630), (500, 30, 631)])
def test_factors(n, kl, ku):
    factors_match(n, kl, ku)


def test_time_next_to_the_wider_window(ra):  # noqa: F811
    """n = 640, kl = 30: ku = 612 took 2.4 times as long as ku = 560 in the global-memory kernel"""
    import torch
    t = []
    for ku in (612, 560):
        n, kl, nb = 640, 30, 32
        g = torch.Generator(device="cuda").manual_seed(ku)
        ab = torch.zeros((nb, n, 2 * kl + ku + 1), dtype=torch.float64, device="cuda")
        ab[:, :, kl:] = torch.randn((nb, n, kl + ku + 1), dtype=torch.float64, device="cuda", generator=g)
        ab[:, :, kl + ku] += 100.0
        piv = torch.empty(nb * n, dtype=torch.int32, device="cuda")
        info = torch.empty(nb, dtype=torch.int32, device="cuda")
        a = ab.view(-1).clone()

        def call():
            a.copy_(ab.view(-1))
            ra.lu_decompose_band(a, piv, info, n, kl, ku)

        t.append(micros(call, reps=3, tries=3))
    assert t[0] <= 1.7 * t[1], t
