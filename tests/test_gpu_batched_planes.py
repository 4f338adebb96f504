"""Batches large enough to run rows and lines of a plane together against the same
boxes two at a time, which run them apart: the same transforms in the same order,
so the ionized boxes are equal bit for bit.  Among them a box that stays
neutral, one that is ionized throughout and one that holds a NaN."""
import math

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


def _batch(D, nbox, linear=True, **kw):
    g, bm = pkg("gpu"), pkg("Programs.find_HII_bubbles_batched")
    L = 1.5625 * D
    spectrum = pkg("cosmo_files.sigmas").PowerLawSpectrum(D, L)
    specs = [{"D": D, "box_len": L, "zeta": 12.0 + i, "deltac": 1.686 if linear else 14.05, "sigma_min2": 0.5 if linear else 40.0,
              "sig0": lambda R: sigma.sig0_discrete(R, D, L)} for i in range(nbox)]
    bb = bm.BatchedBubbles(specs, fil=1, LE=linear, graph=False, tiles=None, **kw)
    bb.set_deltas([g.c2r(g.grf_init(D, L, spectrum.amp, i)) * (1.0 if linear else 0.12) for i in range(nbox)])
    return bb


def _stage_calls(bb):
    """Launches of (rows, lines) passes of one run."""
    lib = pkg("_lib")
    lib.profile_enable(True)
    try:
        bb.run()
        torch.cuda.synchronize()
        counts = lib.profile_collect()
    finally:
        lib.profile_enable(False)
    return counts.get("fused_rows", (0, 0))[1], counts["fused_lines"][1]


@pytest.mark.parametrize("D,nbox", [(64, 16), (128, 2)])
def test_a_choice_of_lines_is_kept(gpu, D, nbox):
    """A tile that is asked for runs rows and lines apart, "planes" runs them
    together, whatever the number of boxes would choose by itself; a tuned
    group runs what was written into it."""
    bb = _batch(D, nbox)
    lib = pkg("_lib").load()
    key, = bb.tiles()
    n = lib.cm21_batch_tile_count(D, 1)
    assert lib.cm21_batch_tile_name(D, 1, n - 1) == b"planes" and lib.cm21_batch_tile_name(D, 1, n) is None
    assert _stage_calls(bb)[0] == (0 if nbox == 16 else 1)
    for l in range(n):
        bb.set_tiles({key: (0, l)})
        assert _stage_calls(bb) == ((0, 1) if l == n - 1 else (1, 1)), l
        if l < n - 1:  # the same tile with the choice left open
            bb.set_tiles({key: (0, -2 - l)})
            assert _stage_calls(bb) == ((0, 1) if nbox == 16 else (1, 1)), l
    bb.stream = torch.cuda.Stream()
    res = bb.autotune(reps=2)[key]
    assert res["chosen"][1] == res["names"][-n:][res["lines"]]
    assert _stage_calls(bb)[0] == (0 if res["chosen"][1] == "planes" else 1)


def test_planes_are_for_linear_input(gpu):
    lib = pkg("_lib")
    bb = _batch(64, 12, linear=False)
    key, = bb.tiles()
    assert _stage_calls(bb)[0] == 1
    bb.set_tiles({key: (0, lib.load().cm21_batch_tile_count(64, 1) - 1)})
    with pytest.raises(lib.CM21Error):
        bb.run()
    bb.set_tiles({key: (-1, -1)})
    bb.stream = torch.cuda.Stream()
    assert bb.autotune(reps=1)[key]["chosen"][1] != "planes"


@pytest.mark.parametrize("D,nbox,late", [(64, 12, True), (64, 16, False), (96, 8, True), (128, 4, False), (160, 12, True)])
def test_planes_where_boxes_are_ionized_late(gpu, D, nbox, late):
    """Without a choice: planes for boxes that stay neutral, and for boxes that are
    ionized late only where the planes do not lose on them."""
    lib = pkg("_lib")
    bb = _batch(D, nbox)
    g = bb._garr[0]
    for j in range(nbox):
        # zeta erfc(deltac / denom) of 0.1, then of 0.9 in every box
        g.boxes[j].zeta = 0.1 / math.erfc(g.boxes[j].deltac / g.denoms[j * g.n_radii])
    assert _stage_calls(bb)[0] == 0
    for j in range(nbox):
        g.boxes[j].zeta *= 9.0
    assert _stage_calls(bb)[0] == (1 if late else 0)
    n = lib.load().cm21_batch_tile_count(D, 1)
    bb.set_tiles({list(bb.tiles())[0]: (-1, -1 - n)})  # past the last tile
    with pytest.raises(lib.CM21Error):
        bb.run()


@pytest.mark.parametrize("D,nbox", [(64, 3), (96, 2), (128, 2), (160, 3)])
def test_forced_planes_equal_rows_and_lines(gpu, D, nbox):
    """Both ways on the same boxes, with tiles of the same factors: equal bit for bit."""
    bb = _batch(D, nbox)
    key, = bb.tiles()
    out = []
    for l in (0, pkg("_lib").load().cm21_batch_tile_count(D, 1) - 1):
        bb.set_tiles({key: (0, l)})
        bb.run()
        out.append([bb.ionized(i).clone() for i in range(nbox)])
    for a, b in zip(*out):
        assert torch.equal(a, b) and 0.01 < float((a == 1).double().mean()) < 0.99
