"""Multihistogram kernels at the sizes where their cut changes: bins below, at
and above a block of 128, runs cut over several workgroups (above 512 bins, or
a slice beyond LDS), more temperatures than threads, more runs than one launch
holds; against the oracle's plain loops."""
import numpy as np
import pytest

from conftest import gpu_available
from oracle.multihist import KB, K_MULTIHIST, multihistogram_npt, multihistogram_nvt

pytestmark = pytest.mark.gpu

if not gpu_available():
    pytest.skip("no GPU visible", allow_module_level=True)

import paralleltemperingmontecarlo as pt  # noqa: E402


def _hists(rng, t, nb, npt):
    """Counts of a harmonic system on the bins of its range."""
    k = 6.0
    e0, e1 = 0.2 * k * KB * t[0], 2.5 * k * KB * t[-1]
    e = e0 + (np.arange(nb) + 0.5) * (e1 - e0) / nb
    p = np.exp((k - 1) * np.log(e) - e / (KB * t[:, None]))
    p /= p.sum(1, keepdims=True)
    if not npt:
        h = np.zeros((len(t), nb + 2))
        h[:, 1:-1] = rng.multinomial(20_000, p)
        return h, e0, e1
    v = np.exp(-0.5 * ((np.arange(nb) + 0.5) / nb * 6 - 3) ** 2)
    h = np.zeros((len(t), nb + 2, nb + 2))
    h[:, 1:-1, 1:-1] = [rng.multinomial(20_000, np.outer(q, v / v.sum()).ravel()).reshape(nb, nb) for q in p]
    return h, e0, e1


# Rounding: exponents of at most a few hundred carry 1e-13, the free energies
# add it per iteration, and <h^2> - <h>^2 loses up to two digits more.
TOL = dict(rtol=1e-10, atol=0)


@pytest.mark.parametrize("n_runs,R,nb,iters", [(1, 2, 1, 3), (3, 5, 127, 50), (2, 5, 128, 50), (2, 7, 129, 50),
                                               (1, 3, 512, 20), (2, 3, 513, 20), (1, 24, 512, 2), (1, 300, 3, 3),
                                               (300, 2, 30, 10)])
def test_nvt(n_runs, R, nb, iters):
    rng = np.random.default_rng(100 * R + nb)
    t = 5.0 * 2.0 ** (np.arange(R) / max(R - 1, 1))
    hs = [_hists(rng, t, nb, False) for _ in range(min(n_runs, 3))]
    pick = [hs[r % len(hs)] for r in range(n_runs)]
    cv, _, fe, it = pt.multihistogram_nvt_batch([t] * n_runs, np.tile(1.0 / (KB * t), (n_runs, 1)),
                                                np.array([h[0] for h in pick]), [h[1] for h in pick],
                                                [h[2] for h in pick], nb, 1e-6, max_iter=iters)
    for r, (h, e0, e1) in enumerate(hs):
        ref, _, rfe, rit = multihistogram_nvt(t.tolist(), (1.0 / (KB * t)).tolist(), h.tolist(), e0, e1, nb, 1e-6,
                                              max_iter=iters)
        assert it[r] == rit
        # one bin has no fluctuation; around zero only the cancelled digits are left
        np.testing.assert_allclose(cv[r], ref, rtol=TOL["rtol"], atol=0 if nb > 1 else 1e-12)
        np.testing.assert_allclose(fe[r], rfe, rtol=1e-11, atol=1e-11)
    for r in range(len(hs), n_runs):  # equal inputs, equal bits
        assert np.array_equal(cv[r], cv[r % len(hs)])


@pytest.mark.parametrize("n_runs,R,nb,iters", [(1, 3, 11, 20), (2, 3, 22, 20), (2, 3, 23, 20), (260, 2, 23, 5),
                                               (1, 90, 23, 1), (1, 160, 23, 1), (1, 48, 182, 1)])
def test_npt(n_runs, R, nb, iters):
    rng = np.random.default_rng(100 * R + nb)
    t = 10.0 * 2.0 ** (np.arange(R) / (R - 1))
    beta = 1.0 / (KB * t)
    hs = [_hists(rng, t, nb, True) for _ in range(min(n_runs, 2))]
    pick = [hs[r % len(hs)] for r in range(n_runs)]
    p = 3e-9
    cp, _, mom, fe, it = pt.multihistogram_npt_batch([t] * n_runs, np.tile(beta, (n_runs, 1)),
                                                     np.array([h[0] for h in pick]), [h[1] for h in pick],
                                                     [h[2] for h in pick], [900.0] * n_runs, [1500.0] * n_runs,
                                                     [p] * n_runs, nb, 1e-6, max_iter=iters)
    for r, (h, e0, e1) in enumerate(hs):
        ref, _, rfe, rit, rmom = multihistogram_npt(t.tolist(), beta.tolist(), h, e0, e1, 900.0, 1500.0, nb, p, 1e-6,
                                                    max_iter=iters)
        assert it[r] == rit
        np.testing.assert_allclose(cp[r], ref, **TOL)
        np.testing.assert_allclose(mom[r], np.array(rmom), rtol=1e-11)
        np.testing.assert_allclose(fe[r], rfe, rtol=1e-11, atol=1e-11)
    for r in range(len(hs), n_runs):
        assert np.array_equal(cp[r], cp[r % len(hs)])


# 8 ((R + 3) (nb + 3) + 247) bytes of LDS for the slice and the temperatures'
# terms are 24 short of the 160 KiB of a workgroup: with those the kernel declares
# itself they do not fit, and the slice is not kept
@pytest.mark.parametrize("R,nb", [(2887, 4), (167, 116)])
def test_nvt_slice_at_the_lds_limit(R, nb):
    rng = np.random.default_rng(R)
    t = 5.0 * 2.0 ** (np.arange(R) / (R - 1))
    h, e0, e1 = _hists(rng, t, nb, False)
    beta = 1.0 / (KB * t)
    cv, t_res, fe, it = pt.multihistogram_nvt_batch([t], beta[None], h[None], [e0], [e1], nb, 0.0, max_iter=3)
    e = e0 + (np.arange(nb) + 0.5) * (e1 - e0) / nb
    f, n, hs = np.zeros(R), h[:, 1:-1].sum(1), h[:, 1:-1].sum(0)

    def terms():
        x = -beta[:, None] * e - f[:, None]
        off = x.max(0) + np.log(1000.0)
        return off, hs / (n[:, None] * np.exp(x - off)).sum(0)

    for _ in range(3):
        off, ratio = terms()
        f = np.log((ratio * np.exp(-beta[:, None] * e - off)).sum(1))
    off, ratio = terms()
    tr = t[0] * (t[-1] / t[0]) ** (np.arange(10 * R) / (10 * R - 1))
    q = ratio * np.exp(-e / (KB * tr)[:, None] - off)
    q /= q.sum(1, keepdims=True)
    d = e - (q * e).sum(1, keepdims=True)
    assert it[0] == 3
    np.testing.assert_allclose(fe[0], f, rtol=1e-11, atol=1e-11)
    np.testing.assert_allclose(cv[0], (q * d * d).sum(1) / (K_MULTIHIST * tr**2), **TOL)
