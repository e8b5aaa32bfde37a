"""phi FFTs and the fused reforms over the lengths their kernels are chosen by: 2^k and 3 * 2^k (compiled
for the length), every radix of the run-time schedule, one to five stages, lines of one and of
several hundred threads, last workgroups with missing lines, plans whose l_max fills or does not
fill 2/3 of the modes, and plans without some m."""
import numpy as np
import pytest

from oracle import oracle as O
from tests.gpu_helpers import dev, empty, host, rel_max

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def ra():
    import torch
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    import rayleigh_amd
    return rayleigh_amd


# N_phi / 2: the compiled lengths, then the others by their radices
COMPILED = [16, 32, 64, 128, 256, 512, 1024, 2048, 4096, 24, 48, 96, 192, 384, 768, 1536, 3072]
OTHERS = [1, 2, 3, 4, 5, 6, 7, 8, 9, 10, 12, 14, 15, 18, 25, 27, 49, 63, 80, 150, 210, 225, 240, 245, 343, 625, 720, 1000,
          1215, 1875, 2187, 2401, 3125, 3675, 3750, 4000]


@pytest.mark.parametrize("n2", COMPILED + OTHERS)
def test_both_directions(ra, n2):
    nphi = 2 * n2
    lines = max(3, min(301, 200000 // nphi)) | 1
    rng = np.random.default_rng(n2)
    x = rng.standard_normal((lines, nphi + 2))
    tol = 1e-14 * max(1.0, np.log2(nphi))  # the repository's bound for the FFTs
    d = dev(x.ravel())
    ra.fft_to_physical(d, nphi)
    assert rel_max(host(d), O.fft_c2r(nphi, x).ravel()) <= tol
    for rsc in (False, True):
        d = dev(x.ravel())
        (ra.fft_to_spectral_rsc if rsc else ra.fft_to_spectral)(d, nphi)
        assert rel_max(host(d), O.fft_r2c(nphi, x, rsc).ravel()) <= tol


# (N_phi / 2, N_theta, l_max, N_r, N_f, m dropped): theta blocks that end early, l_max below, at and
# above 2/3 of the modes, lines of more than 128 threads (two kernels)
REFORMS = [(24, 6, 15, 3, 2, []), (48, 70, 47, 2, 1, [3]), (96, 34, 63, 3, 1, []), (192, 18, 150, 2, 2, [0, 150]),
           (384, 10, 255, 2, 1, []), (768, 6, 511, 1, 2, [7]), (1536, 10, 1100, 1, 1, []), (3072, 4, 2000, 1, 1, []),
           (16, 66, 9, 2, 1, []), (32, 22, 31, 3, 1, []), (128, 20, 84, 2, 2, [1]), (256, 10, 169, 3, 1, []),
           (512, 6, 400, 1, 2, []), (1024, 10, 681, 1, 1, []), (4096, 4, 2700, 1, 1, []),
           (1, 4, 0, 2, 1, []), (5, 66, 3, 3, 2, []), (15, 34, 14, 2, 1, [4]), (100, 22, 65, 3, 2, []),
           (240, 36, 159, 2, 2, [0]), (360, 14, 359, 1, 2, []), (1000, 6, 665, 1, 1, []), (1215, 4, 809, 1, 1, []),
           (2187, 4, 1457, 1, 1, [])]


@pytest.mark.parametrize("n2,nt,lmax,nr,nf,drop", REFORMS)
def test_reforms_are_the_separate_calls(ra, n2, nt, lmax, nr, nf, drop):
    """Bit for bit, whatever the grid held before (NaN here)."""
    nphi = 2 * n2
    ms = np.array([m for m in O.m_order_balanced(lmax) if m not in drop], dtype=np.int32)
    plan = ra.LegendrePlan(nt, lmax, ms, nr, nf)
    rng = np.random.default_rng(n2 + nt)
    p2 = dev(rng.standard_normal(plan.hybrid_size))
    n = (nphi + 2) * nr * nt * nf
    a, b = empty(n), empty(n)
    plan.reform_2a3a(p2, a, nphi)
    ra.fft_to_physical(a, nphi)
    plan.reform_to_physical(p2, b, nphi)
    assert np.array_equal(host(a), host(b))
    grid = rng.standard_normal(n)
    c, d = dev(grid), dev(grid)
    q, w = empty(plan.hybrid_size), empty(plan.hybrid_size)
    ra.fft_to_spectral(c, nphi)
    plan.reform_3b2b(c, q, nphi)
    plan.reform_to_spectral(d, w, nphi)
    assert np.array_equal(host(q), host(w))
    # the grid: left alone for 3 * 2^k (24 .. 3072), transformed in place otherwise
    k = n2
    while k % 2 == 0:
        k //= 2
    assert np.array_equal(host(d), grid if k == 3 and n2 >= 24 else host(c))
