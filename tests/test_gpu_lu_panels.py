"""The panelled LU factorisation and the solve bit for bit against the oracle at the edges of its panels (16
columns), waves, workgroups and trailing tiles, on matrices whose columns hold what the pivot
search and the updates treat specially: equal candidates, zero rows of U, zero columns, NaNs and
infinities."""
import numpy as np
import pytest

from oracle import oracle as O

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def ra():
    import torch
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    import rayleigh_amd
    return rayleigh_amd


def matrices(n):
    """generic; small whole numbers (many equal candidates, exact zeros in U); a zero column and
    a zero row; NaN and infinities"""
    rng = np.random.default_rng(n)
    generic = rng.standard_normal((n, n))
    ties = rng.integers(-2, 3, (n, n)).astype(float)
    holes = rng.standard_normal((n, n))
    holes[:, n // 2] = 0.0
    holes[n // 3, :] = 0.0
    special = rng.standard_normal((n, n))
    special[(3 * n) // 4, n // 3] = np.nan
    special[n - 1, n // 2] = np.inf
    special[n // 5, n // 5] = np.nan
    return [generic, ties, holes, special]


@pytest.mark.parametrize("n", [1, 3, 15, 16, 17, 31, 32, 33, 63, 64, 65, 96, 127, 128, 129, 255, 256, 257, 271, 289,
                               511, 512, 513, 767, 1024])
def test_factors_match_the_oracle(ra, n):
    import torch
    mats = matrices(n) if n <= 513 else matrices(n)[:2]
    nb = len(mats)
    d = torch.from_numpy(np.concatenate([m.ravel(order="F") for m in mats])).cuda()
    piv = torch.zeros(nb * n, dtype=torch.int32, device="cuda")
    info = torch.full((nb,), -7, dtype=torch.int32, device="cuda")
    ra.lu_decompose_full(d, piv, info, n)
    got, piv_g, info_g = d.cpu().numpy().reshape(nb, n, n), piv.cpu().numpy().reshape(nb, n), info.cpu().numpy()
    for b, m in enumerate(mats):
        with np.errstate(all="ignore"):
            lu, p, inf = O.lu_decompose(m)
        assert np.array_equal(piv_g[b], p) and info_g[b] == inf, (n, b)
        assert np.array_equal(got[b].T, lu, equal_nan=True), (n, b)


@pytest.mark.parametrize("n", [1, 3, 7, 8, 9, 15, 16, 17, 31, 33, 63, 64, 65, 127, 128, 129, 255, 256, 257, 259, 300,
                               511, 512, 513, 515, 700, 1024])
def test_solutions_match_the_oracle(ra, n):
    """right-hand-side counts around a workgroup's columns, zeros of both signs and zero columns,
    factors with entries that a row past the matrix must not see (infinities, NaN)"""
    import torch
    rng = np.random.default_rng(n)
    nb = 3 if n <= 300 else 2
    facs, pivs = [], []
    for b in range(nb):
        f = rng.standard_normal((n, n)) / n + np.eye(n)
        if b == 1:
            f[n // 2, n // 3] = np.inf
            f[n // 4, (2 * n) // 3] = np.nan
        facs.append(f)
        pivs.append(np.array([rng.integers(k, n) + 1 for k in range(n)], dtype=np.int32))
    counts = [33, 17, 1][:nb]
    offs = np.concatenate([[0], np.cumsum([c * n + 3 for c in counts])]).astype(np.int64)
    rhs_np = rng.standard_normal(int(offs[-1]))
    rhs_np[: n] = 0.0
    rhs_np[n: 2 * n: 2] = -0.0
    rhs_np[offs[1]: offs[1] + n: 3] = 0.0
    d = torch.from_numpy(np.concatenate([f.ravel(order="F") for f in facs])).cuda()
    rhs = torch.from_numpy(rhs_np.copy()).cuda()
    ra.lu_solve_full(d, torch.from_numpy(np.concatenate(pivs)).cuda(), rhs, torch.from_numpy(offs[:-1]).cuda(),
                     torch.tensor(counts, dtype=torch.int32).cuda(), n, max(counts))
    want = rhs_np.copy()
    for b in range(nb):
        bb = rhs_np[offs[b]: offs[b] + counts[b] * n].reshape(counts[b], n).T
        with np.errstate(all="ignore"):
            want[offs[b]: offs[b] + counts[b] * n] = O.lu_solve(facs[b], pivs[b], bb).T.ravel()
    got = rhs.cpu().numpy()
    assert np.array_equal(got, want, equal_nan=True), n
    assert np.array_equal(np.signbit(got[got == 0.0]), np.signbit(want[want == 0.0]))
