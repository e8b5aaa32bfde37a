"""Calls of so many lines or matrices that one launch of their kernel cannot hold them: a launch has fewer
than 2^32 threads."""
import pytest

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def ra():
    import torch
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    import rayleigh_amd
    return rayleigh_amd


def test_more_lines_than_a_launch_holds(ra):
    """2^32 + 1001 lines of N_phi = 2, one thread each: both directions, every line (137 GB)"""
    import torch
    lines = 2 ** 32 + 1001
    if torch.cuda.mem_get_info()[0] < 32 * lines + 8e9:
        pytest.skip("too little device memory")
    x = torch.ones(4 * lines, dtype=torch.float64, device="cuda")
    piece = 1 << 28

    def expect(line):
        want = torch.tensor(line, dtype=torch.float64, device="cuda")
        for at in range(0, lines, piece):
            assert bool((x[4 * at: 4 * min(at + piece, lines)].view(-1, 4) == want).all()), at

    ra.fft_to_physical(x, 2)  # x_j = X_0 + (-1)^j X_1
    expect([2.0, 0.0, 0.0, 0.0])
    ra.fft_to_spectral(x, 2)  # X_0 = x_0 + x_1, X_1 = x_0 - x_1
    expect([2.0, 0.0, 2.0, 0.0])
    del x
    torch.cuda.empty_cache()


@pytest.mark.parametrize("nb,kl", [(2 ** 22 + 3, 81), (2 ** 23 + 3, 25)])
def test_band_matrices_by_the_million(ra, nb, kl):
    """as many matrices of one row as 1024 (kl > 80) and 512 (kl > 24) threads each would pass the limit"""
    import torch
    ldab = 2 * kl + 1
    if torch.cuda.mem_get_info()[0] < 8 * nb * ldab + 4e9:
        pytest.skip("too little device memory")
    ab = torch.full((nb, ldab), 7.0, dtype=torch.float64, device="cuda")
    ab[::3, kl] = 0.0  # the diagonal
    want = ab.clone()
    piv = torch.full((nb,), -5, dtype=torch.int32, device="cuda")
    info = torch.full((nb,), -5, dtype=torch.int32, device="cuda")
    ra.lu_decompose_band(ab.view(-1), piv, info, 1, kl, 0)
    assert torch.equal(ab, want)
    assert bool((piv == 1).all())
    assert int(info[::3].min()) == 1 and int(info.sum()) == (nb + 2) // 3
