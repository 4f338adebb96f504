"""Smoothed and displacement boxes picked on every q-th cell: the folded
spectrum (cm21_fold_fields) against the full-size filter, displacement and
inverse transforms followed by the pick.  Both run in float32 from the same
windowed modes, so they differ by the rounding of two transforms: a few 1e-7
of the field's maximum; the bar is 2e-6."""
import numpy as np
import pytest
import torch

from conftest import pkg

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("D,sw", [(2, 2), (16, 16), (32, 16), (30, 10), (60, 20), (64, 16), (40, 4), (30, 15), (48, 3),
                                  (128, 64), (126, 42)])
@pytest.mark.parametrize("R", [None, 0.3])
def test_folded_fields_equal_full_size_pick(gpu, D, sw, R):
    g = pkg("gpu")
    L = 50.0
    gen = torch.Generator(device="cuda").manual_seed(D * 100 + sw)
    x = torch.randn((D, D, D), generator=gen, device="cuda")
    spec = g.r2c(x)
    keep = spec.clone()
    # R: the initial conditions' smoothing, and a window wider than the whole grid (every alias counts)
    R = float(pkg("Programs.initialize").smoothing_radius(L, sw)) if R is None else R * L / D
    scale = 1.0 / D ** 3
    got = g.smoothed_fields(spec, L, sw, R, scale=scale)
    assert torch.equal(spec, keep) and len(got) == 4
    want = [g.subsample(g.c2r(g.hii_filter(spec, L, R, filter_type=0, korder=1, scale=scale)), sw)]
    want += [g.subsample(g.c2r(g.velocity(spec, L, k, filter_type=0, R=R)), sw) * scale for k in range(3)]
    for a, b in zip(got, want):
        assert a.shape == (sw, sw, sw) and a.dtype == torch.float32
        assert float((a - b).abs().max()) <= 2e-6 * max(float(b.abs().max()), 1e-30)
    for a, b in zip(g.smoothed_fields(spec, L, sw, R, displacements=False, scale=scale) +
                    g.smoothed_fields(spec, L, sw, R, smoothed=False, scale=scale), got):
        assert torch.equal(a, b)


def test_fold_rejects_sides_that_do_not_divide(gpu):
    g = pkg("gpu")
    lib = pkg("_lib")
    spec = g.empty_spec(16).zero_()
    with pytest.raises(ValueError):
        g.smoothed_fields(spec, 10.0, 5, 1.0)
    out = torch.zeros(64, dtype=torch.complex64, device="cuda")
    for sw in (0, 3, 6, 32):
        with pytest.raises(lib.CM21Error):
            lib.call("cm21_fold_fields", lib.ptr(out), lib.ptr(spec), 16, sw, 0.6, 1.0, 1.0, 1, 0, lib.stream_handle())
