"""The banded LU factorisation with its window in LDS, and the solve, bit for bit against the oracle: window
sizes around a wave and around the largest that fits (kl = ku = 99 is the last), matrices
smaller than their window, unequal bands, and columns that the pivot search and the updates
treat specially (equal candidates, zero columns, zeros in the pivot row, NaN, infinities)."""
import numpy as np
import pytest

from oracle import oracle as O

pytestmark = pytest.mark.gpu


def matrices(n, kl, ku):
    rng = np.random.default_rng(1000 * n + 10 * kl + ku)
    i, j = np.indices((n, n))
    out = (i - j > kl) | (j - i > ku)
    generic = rng.standard_normal((n, n))
    ties = rng.integers(-2, 3, (n, n)).astype(float)
    holes = rng.standard_normal((n, n))
    holes[:, n // 2] = 0.0
    holes[n // 3, :] = -0.0
    special = rng.standard_normal((n, n))
    special[min(n - 1, n // 3 + kl // 2), n // 3] = np.nan
    special[n // 2, n // 2] = np.inf
    special[(4 * n) // 5, (4 * n) // 5] = np.nan
    mats = [generic, ties, holes, special]
    for m in mats:
        m[out] = 0.0
    return mats


@pytest.mark.parametrize("n,kl,ku", [(1, 0, 0), (2, 1, 1), (9, 0, 3), (9, 3, 0), (20, 31, 31), (64, 1, 1), (90, 16, 16),
                                     (90, 17, 17), (130, 40, 40), (130, 41, 41), (150, 62, 62), (150, 63, 63),
                                     (150, 64, 64), (200, 72, 72), (230, 98, 98), (230, 99, 99), (230, 100, 100),
                                     (170, 139, 1), (300, 5, 290), (300, 40, 200), (300, 2, 600)])
def test_factors_match_the_oracle(n, kl, ku):
    import torch
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    import rayleigh_amd as ra
    abs_ = [ra.band_storage(m, kl, ku) for m in matrices(n, kl, ku)]
    for ab in abs_:
        ab[:kl, :] = np.nan
    nb, ldab = len(abs_), abs_[0].shape[0]
    d = torch.from_numpy(np.concatenate([ab.ravel(order="F") for ab in abs_])).cuda()
    piv = torch.zeros(nb * n, dtype=torch.int32, device="cuda")
    info = torch.full((nb,), -7, dtype=torch.int32, device="cuda")
    ra.lu_decompose_band(d, piv, info, n, kl, ku)
    got, piv_g, info_g = d.cpu().numpy().reshape(nb, n, ldab), piv.cpu().numpy().reshape(nb, n), info.cpu().numpy()
    for b, ab in enumerate(abs_):
        with np.errstate(all="ignore"):
            f, p, inf = O.band_lu_decompose(ab, kl, ku)
        assert np.array_equal(piv_g[b], p) and info_g[b] == inf, (n, kl, ku, b)
        assert np.array_equal(got[b].T, f, equal_nan=True), (n, kl, ku, b)
        assert np.array_equal(np.signbit(got[b].T[f == 0.0]), np.signbit(f[f == 0.0])), (n, kl, ku, b)


@pytest.mark.parametrize("n,kl,ku", [(1, 0, 0), (2, 1, 1), (63, 62, 62), (64, 3, 3), (65, 64, 64), (128, 70, 70),
                                     (129, 5, 9), (192, 72, 72), (255, 130, 2), (257, 96, 96), (512, 8, 8),
                                     (513, 70, 3), (1000, 65, 65), (1024, 2, 130)])
def test_solutions_match_the_oracle(n, kl, ku):
    """column counts around a wave's columns, zeros of both signs, whole zero columns, an infinity"""
    import torch
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    import rayleigh_amd as ra
    rng = np.random.default_rng(n + kl)
    facs, pivs, counts = [], [], [11, 4, 1]
    for m in matrices(n, kl, ku)[:2] + matrices(n, kl, ku)[:1]:
        with np.errstate(all="ignore"):
            f, p, _ = O.band_lu_decompose(ra.band_storage(m, kl, ku), kl, ku)
        facs.append(f)
        pivs.append(p)
    offs = np.concatenate([[0], np.cumsum([c * n + 3 for c in counts])]).astype(np.int64)
    rhs_np = rng.standard_normal(int(offs[-1]))
    rhs_np[: n] = 0.0
    rhs_np[n: 2 * n: 2] = -0.0
    rhs_np[2 * n + n // 2] = np.inf
    rhs_np[offs[2]: offs[2] + n: 3] = 0.0
    rhs = torch.from_numpy(rhs_np.copy()).cuda()
    ra.lu_solve_band(torch.from_numpy(np.concatenate([f.ravel(order="F") for f in facs])).cuda(),
                     torch.from_numpy(np.concatenate(pivs)).cuda(), rhs, torch.from_numpy(offs[:-1]).cuda(),
                     torch.tensor(counts, dtype=torch.int32).cuda(), n, kl, max(counts), ku=ku)
    got, want = rhs.cpu().numpy(), rhs_np.copy()
    for b, c in enumerate(counts):
        bb = rhs_np[offs[b]: offs[b] + c * n].reshape(c, n).T
        with np.errstate(all="ignore"):
            want[offs[b]: offs[b] + c * n] = O.band_lu_solve(facs[b], kl, ku, pivs[b], bb).T.ravel()
    assert np.array_equal(got, want, equal_nan=True), (n, kl, ku)
    assert np.array_equal(np.signbit(got[got == 0.0]), np.signbit(want[want == 0.0])), (n, kl, ku)
