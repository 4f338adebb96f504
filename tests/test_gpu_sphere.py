"""Sphere paint and threshold of the generic path at the sizes where their
tiles end: sides around the 64-cell tile and the 64-bit word, reaches of zero,
of a fraction of a cell, across the box and past the 16-bit form's limit.  All
of it is whole-number or decided away from the threshold, so the results are
equal to the oracle's."""
import numpy as np
import pytest
import torch

from conftest import pkg
from oracle import bubbles

pytestmark = pytest.mark.gpu

DELTAC, DENOM, ZETA = 1.686, np.float32(1.0), 1.6  # centres where delta >~ 1.34


def _paint(D, n, R, periodic, seed):
    rng = np.random.default_rng(seed)
    centers = np.zeros(D ** 3, bool)
    centers[rng.choice(D ** 3, n, replace=False)] = True
    centers = centers.reshape(D, D, D)
    sm = np.where(centers, 2.0, -1.0).astype(np.float32)
    start = rng.choice(np.array([0.0, 0.25, 1.0], np.float32), (D, D, D), p=[0.8, 0.1, 0.1])
    start[: D // 2] = 1.0 if seed % 2 else start[: D // 2]  # tiles that are painted already
    ion = torch.from_numpy(start.copy()).cuda()
    pkg("gpu").update_sphere(ion, torch.from_numpy(sm).cuda(), DELTAC, DENOM, ZETA, R, periodic)
    assert np.array_equal(ion.cpu().numpy(), bubbles.paint_spheres(start, centers, np.float32(R), periodic))


@pytest.mark.parametrize("periodic", [False, True])
@pytest.mark.parametrize("D,n,R", [(2, 1, 1.0), (12, 0, 3.0), (12, 3, 0.0), (12, 3, 0.5), (12, 1, 40.0), (62, 9, 5.0),
                                   (64, 7, 8.7), (66, 5, 33.1), (66, 2, 65.0), (130, 40, 11.9), (130, 3, 70.5),
                                   (130, 2, 190.0)])
def test_sphere_paint_tiles(gpu, D, n, R, periodic):
    _paint(D, n, R, periodic, D + n)


@pytest.mark.parametrize("D,n,R,periodic", [(194, 1, 191.4, False), (194, 1, 192.0, True), (40, 2, 1024.0, True)])
def test_sphere_paint_far(gpu, D, n, R, periodic):
    _paint(D, n, R, periodic, D + n)


@pytest.mark.parametrize("D,denom", [(2, 1.3), (14, 1.3), (14, -1.3), (14, 0.0), (34, 0.02)])
@pytest.mark.parametrize("final", [False, True])
def test_threshold_forms(gpu, D, denom, final):
    """Remainders of a threshold block, NaN, infinities, and denominators for
    which no density threshold exists."""
    rng = np.random.default_rng(D)
    sm = (rng.standard_normal((D, D, D)) * 0.8 + 1.0).astype(np.float32)
    sm.reshape(-1)[:3] = [np.nan, np.inf, -np.inf]
    start = rng.choice(np.array([0.0, 1.0], np.float32), (D, D, D))
    with np.errstate(all="ignore"):
        f = bubbles.fcoll_f32(sm, DELTAC, np.float32(denom)).astype(np.float64)
    near = np.abs(f * ZETA - 1.0) < 1e-5
    want = np.where(f >= 1 / ZETA, 1.0, f * ZETA if final else start).astype(np.float32)
    want = np.where(start == 1.0, np.float32(1.0), want)
    ion = torch.from_numpy(start).cuda()
    pkg("gpu").fcoll_threshold(ion, torch.from_numpy(sm).cuda(), DELTAC, np.float32(denom), ZETA, final_step=final)
    got = ion.cpu().numpy()
    assert np.array_equal((got == 1)[~near], (want == 1)[~near])
    assert np.allclose(got[~near], want[~near], rtol=1e-5, atol=1e-7, equal_nan=True)


@pytest.mark.parametrize("D,R", [(150, 256.0), (150, 257.0), (160, 270.0), (180, 256.5), (180, 300.0), (190, 327.0),
                                 (190, 1024.0)])
def test_sphere_paint_radius_past_the_box(gpu, D, R):
    """A clipped sphere of more cells than the side: the reach along an axis ends
    at the box, the squared radius does not, and past 65535 it is beyond what 16
    bits hold."""
    centers = np.zeros((D, D, D), bool)
    centers[0, 0, D - 1] = True
    sm = np.where(centers, 2.0, -1.0).astype(np.float32)
    ion = torch.zeros((D, D, D), device="cuda")
    pkg("gpu").update_sphere(ion, torch.from_numpy(sm).cuda(), DELTAC, DENOM, ZETA, R, False)
    assert np.array_equal(ion.cpu().numpy(), bubbles.paint_spheres(np.zeros_like(sm), centers, np.float32(R), False))


@pytest.mark.parametrize("D,R,centre,periodic", [(128, 300.0, True, True), (128, 300.0, False, True), (130, 257.0, True, True),
                                                 (380, 381.0, True, True), (190, 327.5, True, False), (190, 1024.0, False, False),
                                                 (148, 256.0, True, False)])
def test_sphere_paint_radius_past_every_cell(gpu, D, R, centre, periodic):
    """No cell as far as R, R^2 past 16 bits: one centre paints the whole box, none paints nothing."""
    sm = torch.full((D, D, D), -1.0, device="cuda")
    if centre:
        sm[0, D - 1, D - 1] = 2.0
    ion = torch.zeros_like(sm)
    pkg("gpu").update_sphere(ion, sm, DELTAC, DENOM, ZETA, R, periodic)
    assert bool((ion == (1.0 if centre else 0.0)).all())


@pytest.mark.parametrize("scale", [-0.1, -1.0, -30.0])
def test_sphere_paint_negative_scale_paints_nothing(gpu, scale):
    """A negative sphere radius has no offset inside it: every radius but the
    last (threshold and partial values) leaves the box as it is, so the list of
    radii and its last one alone give the same."""
    lib = pkg("_lib")
    D, L = 32, 48.0
    delta = torch.randn((D,) * 3, generator=torch.Generator().manual_seed(1)).cuda()
    radii = np.array([9.0, 5.0, 1.2], np.float32)
    den = np.full(3, 1.0, np.float32)
    prm = lib.BubbleParams(box_len=L, deltac=1.686, zeta=30.0, growth_inv=1.0, fc_mean=0.1, linear_input=1, filter_type=1,
                           ref_fallthrough=1, update=1, sphere_periodic=0, sphere_r_scale=scale, fused=0)
    work = torch.empty(lib.query("cm21_find_bubbles_workspace_bytes", D, 3, 1), dtype=torch.uint8, device="cuda")

    def run(r, d):
        out = torch.empty_like(delta)
        lib.call("cm21_find_bubbles", lib.plan(D, 1).handle, lib.ptr(delta), lib.ptr(out),
                 r.ctypes.data_as(lib.c_float_p), d.ctypes.data_as(lib.c_float_p), len(r), prm, lib.ptr(work),
                 work.numel(), lib.stream_handle())
        return out

    assert torch.equal(run(radii, den), run(radii[2:], den[2:]))
