"""The loop of sides from 256 on asks, for its leading radii, whether the box stays
neutral, runs those radii a launch further ahead through a ring of six
intermediates and passes their box sums or thresholds over.  Against the same
radii three at a time (a list of four never asks): a cell is ionized by the list
when it is by one of its parts, and what the last radius paints is the same in each,
bit for bit."""
import numpy as np
import pytest
import torch

from conftest import pkg

pytestmark = pytest.mark.gpu

ZETA, GROWTH = 30.0, 0.12


class Loop:
    def __init__(self, D, L, linear, mean, amp, seed=3):
        from scipy.special import erfc, erfcinv
        self.lib, fb, g = pkg("_lib"), pkg("Programs.find_HII_bubbles"), pkg("gpu")
        sp = pkg("cosmo_files.sigmas").PowerLawSpectrum(D, L)
        self.D, self.linear = D, linear
        self.delta = (g.c2r(g.grf_init(D, L, sp.amp, seed)) * ((1.0 if linear else GROWTH) * amp)).contiguous()
        dc = 1.686 / GROWTH
        smin = (dc / float(erfcinv(mean / ZETA))) ** 2 / 2.0
        self.radii = fb.radius_schedule(L, D)[0]
        self.denoms = fb.barrier_denominators(self.radii, smin, sp.sig0_discrete)
        self.prm = self.lib.BubbleParams(
            box_len=L, deltac=float(np.float32(dc)), zeta=ZETA, growth_inv=float(np.float32(1.0 / GROWTH)),
            fc_mean=float(np.float32(erfc(dc / np.sqrt(2 * smin)))), linear_input=1 if linear else 0, filter_type=1,
            ref_fallthrough=1, update=0, sphere_periodic=0, sphere_r_scale=1.0, fused=1, graph=0)

    def run(self, which):
        """Ionized box, launches and verdicts of the radii `which`."""
        lib = self.lib
        r = np.ascontiguousarray(self.radii[which], np.float32)
        d = np.ascontiguousarray(self.denoms[which], np.float32)
        nbytes = lib.query("cm21_find_bubbles_workspace_bytes", self.D, len(r), 0)
        work = torch.full((nbytes,), 255, dtype=torch.uint8, device="cuda")
        # scale, threshold, band and verdict per radius are the workspace's last region
        last = work[nbytes - (16 * len(r) + 255) // 256 * 256:].view(torch.int32)
        out = torch.full_like(self.delta, -7.0)
        lib.profile_enable(["fused_radius"])
        lib.call("cm21_find_bubbles", lib.plan(self.D, 1).handle, lib.ptr(self.delta), lib.ptr(out),
                 r.ctypes.data_as(lib.c_float_p), d.ctypes.data_as(lib.c_float_p), len(r), self.prm, lib.ptr(work), nbytes,
                 lib.stream_handle())
        torch.cuda.synchronize()
        launches = lib.profile_collect()["fused_radius"][1]
        lib.profile_enable(False)
        return out, launches, last[3::4][:len(r)].cpu().numpy()

    def check(self, n):
        """The first n - 1 radii and the last; returns how many were passed over."""
        end = len(self.radii) - 1
        which = list(range(n - 1)) + [end]
        got, launches, verdicts = self.run(which)
        plain = 1 if self.linear else 3
        assert launches == len(which) + plain + 1, "no radius ran ahead"
        want = None
        for k in range(0, n - 1, 3):
            part, launches, _ = self.run(which[:-1][k:k + 3] + [end])
            assert launches == min(3, n - 1 - k) + 1 + plain
            want = part if want is None else torch.where((want == 1) | (part == 1), torch.ones_like(part), want)
        assert torch.equal(got, want)
        return int((verdicts == 1).sum()), float((want == 1).double().mean())


@pytest.mark.parametrize("D,L,linear", [(256, 300.0, True), (256, 300.0, False), (512, 500.0, True), (512, 500.0, False)])
@pytest.mark.parametrize("mean", [0.1, 0.5])
def test_verdicts_change_nothing(gpu, D, L, linear, mean):
    """Fields at the barrier's own variance and far above it, where the rule that
    asks is wrong and the verdict has to say no."""
    passed, ionized = [], []
    for amp in (1.0, 4.0):
        loop = Loop(D, L, linear, mean, amp)
        for n in (5, 6, 7, 8, 11, len(loop.radii)):
            p, x = loop.check(n)
            print(f"D={D} linear={linear} mean={mean} amp={amp} radii={n}: {p} passed over, ionized {x:.4f}", flush=True)
            passed.append(p)
            ionized.append(x)
    assert max(passed) >= 4 and max(ionized) > 1e-3  # radii passed over, and cells ionized at radii that were asked
