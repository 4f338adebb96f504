"""Batches large enough to run rows and lines of a plane together against the same
boxes two at a time, which run them apart: the same transforms in the same order,
so the ionized boxes are equal bit for bit.  Among them a box that stays
neutral, one that is ionized throughout and one that holds a NaN."""
import pytest
import torch

from conftest import pkg
from oracle import sigma

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("D,nbox,fil", [(64, 12, 1), (64, 13, 2), (96, 8, 1), (96, 9, 2), (128, 4, 1), (128, 5, 2),
                                        (160, 12, 1)])
def test_planes_equal_rows_and_lines(gpu, D, nbox, fil):
    g, bm = pkg("gpu"), pkg("Programs.find_HII_bubbles_batched")
    sig = pkg("cosmo_files.sigmas")
    L = 1.5625 * D
    spectrum = sig.PowerLawSpectrum(D, L)
    zeta = [2.0, 1e4, 25.0] + [10.0 + 3.0 * i for i in range(nbox - 3)]
    specs = [{"D": D, "box_len": L, "zeta": zeta[i], "deltac": 1.686, "sigma_min2": 0.5 + 0.01 * i, 
              "sig0": lambda R: sigma.sig0_discrete(R, D, L)}
             for i in range(nbox)]
    deltas = [g.c2r(g.grf_init(D, L, spectrum.amp, i)) for i in range(nbox)]
    deltas[2].view(-1)[7] = float("nan")

    def run(lo, hi):
        bb = bm.BatchedBubbles(specs[lo:hi], fil=fil, LE=True, graph=False, tiles=None)
        bb.set_deltas(deltas[lo:hi])
        bb.run()
        return [bb.ionized(i).clone() for i in range(hi - lo)]

    together = run(0, nbox)
    apart = [x for lo in range(0, nbox, 2) for x in run(lo, min(lo + 2, nbox))]
    for i, (a, b) in enumerate(zip(together, apart)):
        assert torch.equal(torch.isnan(a), torch.isnan(b)) and torch.equal(torch.nan_to_num(a), torch.nan_to_num(b)), i
    ion = [float((x == 1).double().mean()) for x in together]
    assert ion[0] < 0.05 and ion[1] > 0.95 and all(0.02 < x < 0.98 for x in ion[3:])
