"""FP64 Legendre kernels at the edges of their tiles: 16-row blocks and K chunks of 16 that are
partly filled, odd node counts per hemisphere, blocks dealt unevenly to row tiles, and column
counts that leave waves of a tile empty -- against the oracle; and the isolation of columns,
whose operand loads reach into the next column at the end of a contraction."""
import numpy as np
import pytest

from oracle import oracle as O
from tests.gpu_helpers import dev, empty, host, rel_max

pytestmark = pytest.mark.gpu

# (N_theta, l_max, m values, columns): nt2 = 1 .. 129; nl = 1 (m = l_max) and around 2, 30 .. 34
# and 64 (chunks of 16 parity-l values), 129 (nine blocks: 3 + 3 + 3 rows)
SHAPES = [
    (2, 0, [0], 1),
    (6, 3, [3, 0, 1, 2], 5),
    (30, 19, [0, 19, 18, 4], 17),
    (32, 31, [0, 1, 2, 15], 16),
    (34, 33, [0, 1, 2, 3], 127),
    (66, 43, [0, 11, 12, 13, 43], 129),
    (98, 64, [0, 1, 33], 48),
    (130, 85, [0, 21, 84], 144),
    (258, 257, [0, 129, 1], 33),
]


@pytest.fixture(scope="module")
def ra():
    import torch
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    import rayleigh_amd
    return rayleigh_amd


def problem(nt, lmax, ms, ncols, seed=11):
    ms = np.array(ms, dtype=np.int32)
    rng = np.random.default_rng(seed)
    s = rng.standard_normal(int(sum(lmax - int(m) + 1 for m in ms)) * ncols)
    p = rng.standard_normal(len(ms) * ncols * nt)
    return ms, O.legendre_tables(nt, lmax, ms), s, p


@pytest.mark.parametrize("nt,lmax,ms,ncols", SHAPES)
def test_tile_edges_against_oracle(ra, nt, lmax, ms, ncols):
    ms, tabs, s, p = problem(nt, lmax, ms, ncols)
    plan = ra.LegendrePlan(nt, lmax, ms, 0, 0, n_cols=ncols)
    out, back = empty(plan.hybrid_size), empty(plan.spectral_size)
    plan.stp(dev(s), out)
    plan.pts(dev(p), back)
    # 1e-13: the repository's bound for FP64 transforms; the sums here have at most 129 terms
    assert rel_max(host(out), O.stp_cols(nt, lmax, ms, ncols, tabs, s)) <= 1e-13
    assert rel_max(host(back), O.pts_cols(nt, lmax, ms, ncols, tabs, p)) <= 1e-13


@pytest.mark.parametrize("nt,lmax,ms,ncols", SHAPES[1:])
def test_columns_stay_apart(ra, nt, lmax, ms, ncols):
    """NaN and infinities in one column leave every other column's bits alone."""
    ms, _, s, p = problem(nt, lmax, ms, ncols)
    plan = ra.LegendrePlan(nt, lmax, ms, 0, 0, n_cols=ncols)
    bad = ncols // 2
    off_s = 0
    s2, p2 = s.copy(), p.reshape(len(ms), ncols, nt).copy()
    p2[:, bad] = np.nan
    keep = []
    for m in ms:
        nl = lmax - int(m) + 1
        blk = s2[off_s: off_s + nl * ncols].reshape(ncols, nl)
        blk[bad] = np.where(np.arange(nl) % 2 == 0, np.nan, np.inf)
        k = np.ones((ncols, nl), bool)
        k[bad] = False
        keep.append(k.ravel())
        off_s += nl * ncols
    keep = np.concatenate(keep)
    got = []
    for a, b in ((s, p), (s2, p2.ravel())):
        out, back = empty(plan.hybrid_size), empty(plan.spectral_size)
        plan.stp(dev(a), out)
        plan.pts(dev(b), back)
        got.append((host(out).reshape(len(ms), ncols, nt), host(back)))
    others = np.arange(ncols) != bad
    assert np.array_equal(got[0][0][:, others], got[1][0][:, others])
    assert np.array_equal(got[0][1][keep], got[1][1][keep])
    assert np.isnan(got[1][0][:, bad]).all() and np.isnan(got[1][1][~keep]).all()
