"""Binned power spectrum at the sizes where its walk can go wrong: boxes of a few
modes, columns that do not fill a wavefront, one bin and the most bins, and a
table that rises and falls along the walk."""
import numpy as np
import pytest
import torch

from conftest import pkg
from oracle import deltat

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("D,nbins", [(2, 1), (4, 3), (6, 512), (34, 40), (66, 1), (130, 40)])
def test_power_spectrum_sizes(gpu, D, nbins):
    g, dt = pkg("gpu"), pkg("Programs.delta_T")
    L = 1.7 * D
    edges = dt.log_edges(L, D, nbins) if nbins > 1 else np.array([2.5 * np.pi * D / L])
    lut = g._device_bin_lut(D, L, edges)
    assert np.array_equal(lut.cpu().numpy(), g.bin_lut(D, L, edges))
    f = (1.0 + 0.3 * np.random.default_rng(D).standard_normal((D, D, D))).astype(np.float32)
    box = torch.from_numpy(f).cuda()
    ps, ks, cnt = g.power_spectrum(box, L, edges)
    _, _, n, (ps_want, ks_want) = deltat.power_spectrum(f.astype(np.float64), L, edges)
    assert np.array_equal(cnt.cpu().numpy(), n)
    # whole-number weights and FP64 sums of at most D^3 terms; the transform is float32
    np.testing.assert_allclose(ks.cpu().numpy(), ks_want, rtol=1e-12)
    np.testing.assert_allclose(ps.cpu().numpy(), ps_want, rtol=2e-5, atol=1e-12 * max(ps_want.max(), 1e-300))
    again = g.power_spectrum(box, L, edges)
    assert torch.equal(ps, again[0]) and torch.equal(ks, again[1])


def test_power_spectrum_any_table(gpu):
    """Bins in no order, some dropped: counts and sums of k are those of the table."""
    g = pkg("gpu")
    D, L, nb = 34, 50.0, 7
    m = np.arange(3 * (D // 2) ** 2 + 1)
    lut = ((m * 2654435761) % 9 - 1).astype(np.int32)  # -1 and 7 are dropped
    f = torch.from_numpy((1.0 + np.random.default_rng(1).random((D, D, D))).astype(np.float32)).cuda()
    _, ks, cnt = g.power_spectrum(f, L, np.ones(nb), lut=torch.from_numpy(lut).cuda())
    n = np.fft.fftfreq(D, 1.0 / D)
    m2 = (n[:, None, None] ** 2 + n[None, :, None] ** 2 + n[None, None, :] ** 2).astype(int)
    b = lut[m2]
    k = 2 * np.pi / L * np.sqrt(m2)
    assert np.array_equal(cnt.cpu().numpy(), [np.sum(b == q) for q in range(nb)])
    np.testing.assert_allclose(ks.cpu().numpy(), [k[b == q].sum() for q in range(nb)], rtol=1e-12)
