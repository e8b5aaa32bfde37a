"""The argument check of the FFT calls, which every call goes through first: which lengths it takes (no lines,
so nothing is launched), and that it costs no more host time for one length than for another."""
import time

from rayleigh_amd import _lib

OK, EINVAL, EUNSUPPORTED = 0, 1, 4


def smooth(n):
    for p in (2, 3, 5, 7):
        while n % p == 0:
            n //= p
    return n == 1


def test_lengths_taken_and_refused():
    f = _lib.lib().raysht_fft_to_physical
    for n2 in range(1, 4200):
        assert f(2 * n2, 0, None, None) == (OK if n2 <= 4096 and smooth(n2) else EUNSUPPORTED), n2
    for nphi in (0, -2, 1, 7):
        assert f(nphi, 0, None, None) == EINVAL


def test_check_costs_no_search():
    """N_phi / 2 = 4032 took 3.5 us more than 16, once more for each entry point that a call went through"""
    f = _lib.lib().raysht_fft_to_physical

    def micros(nphi):
        best = float("inf")
        for _ in range(20):
            t = time.perf_counter()
            for _ in range(500):
                f(nphi, 0, None, None)
            best = min(best, (time.perf_counter() - t) / 500 * 1e6)
        return best

    assert micros(2 * 4032) <= micros(2 * 16) + 1.5
