"""The framework's own whole inverse transform, and the fields taken from a real
box through its own pruned forward transform, against the library transforms.
Both run in float32, so they differ by the rounding of two transforms: a
few 1e-7 of the field's maximum; the bar is 2e-6."""
import pytest
import torch

from conftest import pkg

pytestmark = pytest.mark.gpu


def _close(a, b):
    return a.shape == b.shape and float((a - b).abs().max()) <= 2e-6 * max(float(b.abs().max()), 1e-30)


def _box(D, offset=0):
    gen = torch.Generator(device="cuda").manual_seed(D)
    return torch.randn(D ** 3 + offset, generator=gen, device="cuda")[offset:].view(D, D, D)


@pytest.mark.parametrize("D", [2, 64, 90, 96, 128, 160, 256, 512])
def test_inverse_equals_library(gpu, D):
    g = pkg("gpu")
    spec = g.r2c(_box(D))
    keep = spec.clone()
    got = g.inverse(spec)
    assert torch.equal(spec, keep)
    assert _close(got, g.c2r(spec))


@pytest.mark.parametrize("D,sw", [(64, 64), (64, 16), (96, 48), (128, 64), (160, 20), (256, 128), (512, 256),
                                  (64, 1), (40, 20), (96, 3)])
@pytest.mark.parametrize("R", [None, 0.3])
def test_box_fields(gpu, D, sw, R):
    g = pkg("gpu")
    L = 50.0
    box = _box(D)
    keep = box.clone()
    # the initial conditions' smoothing, and a window that keeps every mode
    R = float(pkg("Programs.initialize").smoothing_radius(L, sw)) if R is None else R * L / D
    got = g.box_fields(box, L, sw, R, scale=1.0 / D ** 3)
    assert torch.equal(box, keep)
    want = g.smoothed_fields(g.r2c(box), L, sw, R, scale=1.0 / D ** 3)
    assert len(got) == len(want) == 4 and all(_close(a, b) for a, b in zip(got, want))


def test_box_at_an_odd_address(gpu):
    """A box aligned to 4 bytes only takes the library's transform."""
    g = pkg("gpu")
    box = _box(64, offset=1)
    assert box.data_ptr() % 8
    got = g.box_fields(box, 50.0, 32, 1.0, displacements=False)
    assert _close(got[0], g.box_fields(box.clone(), 50.0, 32, 1.0, displacements=False)[0])
