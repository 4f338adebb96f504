"""Kinds of numbers that the radius schedule and the barrier take."""
import numpy as np
import pytest
import torch

from conftest import pkg


@pytest.mark.parametrize("kind", [float, np.float64, np.array, lambda v: torch.tensor(v, dtype=torch.float64)])
def test_radius_schedule_takes_any_scalar(kind):
    fb = pkg("Programs.find_HII_bubbles")
    want = fb.radius_schedule(100.0, 64, r_min=0.7, delta_r_factor=1.3)[0]
    got = fb.radius_schedule(100.0, 64, r_min=kind(0.7), delta_r_factor=kind(1.3))[0]
    assert got.dtype == np.float32 and np.array_equal(got, want)


def test_radius_schedule_follows_its_arguments():
    """A tensor changed in place, and a float32 that equals a float64 (whose
    quotients are taken in float32), are not taken for what came before."""
    fb = pkg("Programs.find_HII_bubbles")
    f = torch.tensor(1.1, dtype=torch.float64)
    assert len(fb.radius_schedule(100.0, 64, delta_r_factor=f)[0]) == 37
    f.fill_(1.5)
    assert len(fb.radius_schedule(100.0, 64, delta_r_factor=f)[0]) == 9
    wide = fb.radius_schedule(100.0, 64, r_max=1e9, delta_r_factor=1.125)[0]
    narrow = fb.radius_schedule(100.0, 64, r_max=1e9, delta_r_factor=np.float32(1.125))[0]
    R, want = 1e9, []
    while True:
        final = (R / np.float32(1.125)) <= float(np.float32(0.620350491)) * 100.0 / 64 or (R / np.float32(1.125)) <= 0.5
        want.append(np.float32(R))
        if final:
            break
        R = float(np.float32(R)) / np.float32(1.125)
    assert np.array_equal(narrow, np.array(want, np.float32)) and len(wide) == len(narrow)
