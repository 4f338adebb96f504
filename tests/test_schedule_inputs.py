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


@pytest.mark.parametrize("kind", [float, np.float32, np.array, lambda v: torch.tensor(v, dtype=torch.float64)])
def test_barrier_takes_any_scalar_of_sigma(kind):
    fb = pkg("Programs.find_HII_bubbles")
    radii = np.array([5.0, 2.0], np.float32)
    got = fb.barrier_denominators(radii, 2.0, lambda R: kind(0.5 / R))
    assert got.shape == (2,) and got.dtype == np.float32
    assert np.array_equal(got, np.sqrt([2.0 * (2.0 - float(np.float32(0.5 / R))) for R in (5.0, 2.0)]).astype(np.float32))


@pytest.mark.filterwarnings("ignore::DeprecationWarning")
def test_barrier_of_one_element_arrays_and_the_first_radius_without_one():
    """S(R) as an array of one element, and the first radius that has no
    barrier named also where S fails at a smaller one."""
    fb = pkg("Programs.find_HII_bubbles")
    radii = np.array([5.0, 2.0], np.float32)
    assert fb.barrier_denominators(radii, 2.0, lambda R: np.array([0.5 / R])).shape == (2,)

    def sigma(R):
        if R < 3.0:
            raise KeyError(R)
        return 5.0

    with pytest.raises(ValueError, match=r"S\(R=5.0\)=5.0"):
        fb.barrier_denominators(radii, 2.0, sigma)
    with pytest.raises(KeyError):
        fb.barrier_denominators(radii, 20.0, sigma)
