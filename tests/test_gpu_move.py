"""The mass move at the edges of its patches and tiles: sides that do not fill
a patch, every ratio class DIM/sw, boxes smaller than a tile and displacements
that leave it.  Against the oracle with its bars (NGP cells exact, sums 1e-5)."""
import numpy as np
import pytest
import torch

from conftest import pkg
from oracle import perturb

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("DIM,sw", [(8, 8), (8, 1), (16, 1), (16, 2), (24, 24), (32, 32), (40, 20), (48, 48), (48, 16),
                                    (56, 28), (64, 32), (72, 24), (80, 16), (80, 8), (96, 12), (112, 56), (128, 32), (144, 144), (176, 88)])
@pytest.mark.parametrize("amp", [0.0, 3.0, 60.0, 400.0])
def test_move_mass_edges(gpu, DIM, sw, amp):
    g = pkg("gpu")
    L = 60.0
    rng = np.random.default_rng(DIM * 1000 + sw)
    delta = rng.standard_normal((DIM,) * 3).astype(np.float32)
    v = [(amp * rng.standard_normal((sw,) * 3)).astype(np.float32) for _ in range(3)]
    growth, ginit = 0.12, 0.0036
    s = pkg("Programs.perturb_field").displacement_scale(growth, ginit, L)
    dev = lambda a: torch.from_numpy(a).cuda()  # noqa: E731
    dv = [dev(a) for a in v]
    got = g.move_mass(dev(np.zeros_like(delta)), *dv, s, ginit, "ngp").cpu().numpy()
    assert np.array_equal(got, perturb.move_mass_ngp(np.zeros_like(delta), *v, growth, ginit, L))
    got = g.move_mass(dev(delta), *dv, s, ginit, "ngp").cpu().numpy()
    assert np.allclose(got, perturb.move_mass_ngp(delta, *v, growth, ginit, L), rtol=1e-5, atol=2e-6)
    if DIM % 16 == 0:
        got = g.move_mass(dev(delta), *dv, s, ginit, "cic").cpu().numpy()
        assert np.allclose(got, perturb.move_mass_cic(delta, *v, growth, ginit, L), rtol=1e-5, atol=2e-6)
    else:
        with pytest.raises(pkg("_lib").CM21Error):
            g.move_mass(dev(delta), *dv, s, ginit, "cic")


def test_move_mass_keeps_bad_particles_apart(gpu):
    """A non-finite mass reaches only the cells of its own particle, and a
    non-finite displacement drops the particles of its cell, as the move
    particle by particle does."""
    g = pkg("gpu")
    DIM, sw, L = 64, 32, 60.0
    rng = np.random.default_rng(5)
    delta = np.zeros((DIM,) * 3, np.float32)
    v = [(3.0 * rng.standard_normal((sw,) * 3)).astype(np.float32) for _ in range(3)]
    s = pkg("Programs.perturb_field").displacement_scale(0.12, 0.0036, L)
    dev = lambda a: torch.from_numpy(a).cuda()  # noqa: E731
    delta[10, 20, 31] = np.nan
    delta[40, 41, 42] = np.inf
    for scheme, most in (("ngp", 1), ("cic", 8)):
        got = g.move_mass(dev(delta), *[dev(a) for a in v], s, 0.0036, scheme).cpu().numpy()
        assert 1 <= np.isnan(got).sum() <= most and 1 <= np.isinf(got).sum() <= most
    delta[:] = 0.0
    v[1][4, 5, 6] = np.nan
    v[2][7, 8, 9] = np.inf
    for scheme in ("ngp", "cic"):
        got = g.move_mass(dev(delta), *[dev(a) for a in v], s, 0.0036, scheme).cpu().numpy()
        assert np.isfinite(got).all()
        # 16 particles of 64^3 are gone; cells hold (mass / 8) - 1
        assert abs((got.astype(np.float64) + 1.0).sum() * 8 - (DIM ** 3 - 16)) < 0.05


@pytest.mark.parametrize("DIM,sw", [(48, 3), (96, 2), (128, 1), (128, 2), (160, 10), (176, 16), (208, 26), (272, 34)])
@pytest.mark.parametrize("amp", [0.0, 3.0, 200.0])
def test_move_mass_large_ratios(gpu, DIM, sw, amp):
    """A wavefront per displacement cell: shares of one cell, of its planes and
    columns, patches of 1, 2 and 4 cells that the side does not fill, and cells
    that leave their patch's tile."""
    test_move_mass_edges(gpu, DIM, sw, amp)


def test_move_mass_large_ratio_keeps_bad_particles_apart(gpu):
    g = pkg("gpu")
    DIM, sw, L = 96, 6, 60.0
    rng = np.random.default_rng(6)
    delta = np.zeros((DIM,) * 3, np.float32)
    v = [(3.0 * rng.standard_normal((sw,) * 3)).astype(np.float32) for _ in range(3)]
    s = pkg("Programs.perturb_field").displacement_scale(0.12, 0.0036, L)
    dev = lambda a: torch.from_numpy(a).cuda()  # noqa: E731
    delta[10, 20, 31] = np.nan
    delta[40, 41, 42] = np.inf
    for scheme, most in (("ngp", 1), ("cic", 8)):
        got = g.move_mass(dev(delta), *[dev(a) for a in v], s, 0.0036, scheme).cpu().numpy()
        assert 1 <= np.isnan(got).sum() <= most and 1 <= np.isinf(got).sum() <= most
    delta[:] = 0.0
    v[0][0, 0, 0] = np.nan  # a patch's first cell
    v[2][4, 5, 3] = np.inf
    for scheme in ("ngp", "cic"):
        got = g.move_mass(dev(delta), *[dev(a) for a in v], s, 0.0036, scheme).cpu().numpy()
        assert np.isfinite(got).all()
        assert abs((got.astype(np.float64) + 1.0).sum() * 16 ** 3 - (DIM ** 3 - 2 * 16 ** 3)) < 2.0


def test_move_mass_time_does_not_grow_with_the_ratio(gpu):
    """The same 256^3 particles on fewer cells: nowhere near the 31 times of a
    thread per cell between 32^3 and 8^3 cells (both take about 50 us)."""
    g = pkg("gpu")
    delta = torch.zeros((256,) * 3, device="cuda")

    def best(sw):
        v = [torch.zeros((sw,) * 3, device="cuda") for _ in range(3)]
        times = []
        for _ in range(6):
            e = [torch.cuda.Event(enable_timing=True) for _ in range(2)]
            e[0].record()
            g.move_mass(delta, *v, 1e-4, 0.0036, "cic")
            e[1].record()
            torch.cuda.synchronize()
            times.append(e[0].elapsed_time(e[1]))
        return min(times)

    assert best(8) < 6.0 * best(32)


@pytest.mark.parametrize("DIM,sw", [(64, 64), (64, 32), (48, 16), (64, 16), (160, 32), (64, 8)])
@pytest.mark.parametrize("offset", [1, 2, 3])
def test_move_mass_of_an_unaligned_view(gpu, DIM, sw, offset):
    """Density and displacements that start in the middle of an allocation."""
    g = pkg("gpu")
    L = 60.0
    rng = np.random.default_rng(DIM + sw)
    delta = rng.standard_normal((DIM,) * 3).astype(np.float32)
    v = [(3.0 * rng.standard_normal((sw,) * 3)).astype(np.float32) for _ in range(3)]
    s = pkg("Programs.perturb_field").displacement_scale(0.12, 0.0036, L)

    def view(a):
        t = torch.empty(a.size + offset, device="cuda")[offset:].view(a.shape)
        return t.copy_(torch.from_numpy(a))

    got = g.move_mass(view(delta), *[view(a) for a in v], s, 0.0036, "cic").cpu().numpy()
    assert np.allclose(got, perturb.move_mass_cic(delta, *v, 0.12, 0.0036, L), rtol=1e-5, atol=2e-6)
    got = g.move_mass(view(delta), *[view(a) for a in v], s, 0.0036, "ngp").cpu().numpy()
    assert np.allclose(got, perturb.move_mass_ngp(delta, *v, 0.12, 0.0036, L), rtol=1e-5, atol=2e-6)


def _coherent(sw, cells, rng, L, s):
    """Displacement boxes of `cells` cells along each axis and a wave of the box's length
    half as high, with a tenth of a cell of noise."""
    x = np.sin(2.0 * np.pi * np.arange(sw) / sw)
    wave = np.stack(np.broadcast_arrays(x[:, None, None], x[None, :, None], x[None, None, :]))
    d = np.array(cells)[:, None, None, None] + 0.5 * abs(max(cells, key=abs)) * wave
    return [(a / (s * sw) + 0.1 / (s * sw) * rng.standard_normal((sw,) * 3)).astype(np.float32) for a in d]


@pytest.mark.parametrize("DIM,sw", [(48, 48), (80, 40), (96, 32), (128, 32), (160, 32), (144, 144)])
@pytest.mark.parametrize("cells", [(5.0, -7.0, 11.0), (-23.4, 30.6, -0.5), (400.0, -1000.0, 70.0)])
def test_move_mass_of_a_patch_that_goes_far_together(gpu, DIM, sw, cells):
    """The block's tile lies where its patch goes, across the box's faces and
    several box lengths away too."""
    g = pkg("gpu")
    L, growth, ginit = 60.0, 0.12, 0.0036
    rng = np.random.default_rng(DIM + sw)
    delta = rng.standard_normal((DIM,) * 3).astype(np.float32)
    s = pkg("Programs.perturb_field").displacement_scale(growth, ginit, L)
    v = _coherent(sw, cells, rng, L, s)
    dev = lambda a: torch.from_numpy(a).cuda()  # noqa: E731
    for scheme, ref in (("ngp", perturb.move_mass_ngp), ("cic", perturb.move_mass_cic)):
        got = g.move_mass(dev(delta), *[dev(a) for a in v], s, ginit, scheme).cpu().numpy()
        assert np.allclose(got, ref(delta, *v, growth, ginit, L), rtol=1e-5, atol=2e-6)


def test_move_mass_time_does_not_grow_with_a_common_displacement(gpu):
    """256^3 particles on as many cells, moved by 40 cells together: the 0.22 ms of no
    displacement, where deposits outside the tile take four times that."""
    g = pkg("gpu")
    n = 256
    delta = torch.zeros((n,) * 3, device="cuda")

    def best(cells):
        v = [torch.full((n,) * 3, cells / (1e-3 * n), device="cuda") for _ in range(3)]
        times = []
        for _ in range(6):
            e = [torch.cuda.Event(enable_timing=True) for _ in range(2)]
            e[0].record()
            g.move_mass(delta, *v, 1e-3, 0.0036, "cic")
            e[1].record()
            torch.cuda.synchronize()
            times.append(e[0].elapsed_time(e[1]))
        return min(times)

    assert best(40.3) < 2.0 * best(0.3)
