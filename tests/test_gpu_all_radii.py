"""The loop with every radius in one launch per pass (a workspace of
cm21_find_bubbles_full_workspace_bytes) against the loop with one launch per
radius (the smallest workspace): the same device code on the same tiles, so the
boxes are equal bit for bit."""
import numpy as np
import pytest
import torch

from conftest import pkg

pytestmark = pytest.mark.gpu


def _run(D, L, LE, fil, mean, radii, extra, seed=3, graph=0):
    lib = pkg("_lib")
    fb = pkg("Programs.find_HII_bubbles")
    g = pkg("gpu")
    sp = pkg("cosmo_files.sigmas").PowerLawSpectrum(D, L)
    from scipy.special import erfc, erfcinv
    growth, zeta = (1.0 if LE else 0.12), 30.0
    delta = (g.c2r(g.grf_init(D, L, sp.amp, seed)) * growth).contiguous()
    dc = 1.686 / 0.12
    smin = (dc / float(erfcinv(mean / zeta))) ** 2 / 2.0
    den = fb.barrier_denominators(radii, smin, sp.sig0_discrete)
    prm = lib.BubbleParams(box_len=L, deltac=float(np.float32(dc)), zeta=zeta, growth_inv=float(np.float32(1 / 0.12)),
                           fc_mean=float(np.float32(erfc(dc / np.sqrt(2 * smin)))), linear_input=1 if LE else 0,
                           filter_type=fil, ref_fallthrough=1, update=0, sphere_periodic=0, sphere_r_scale=1.0, fused=1,
                           graph=graph)
    r = np.ascontiguousarray(radii, np.float32)
    rp, dp = r.ctypes.data_as(lib.c_float_p), den.ctypes.data_as(lib.c_float_p)
    least = lib.query("cm21_find_bubbles_workspace_bytes", D, len(r), 0)
    nbytes = max(least, lib.query("cm21_find_bubbles_full_workspace_bytes", D, rp, len(r), prm)) if extra else least
    work = torch.full((nbytes,), 255, dtype=torch.uint8, device="cuda")
    out = torch.full_like(delta, -7.0)
    stream = torch.cuda.Stream()
    stream.wait_stream(torch.cuda.current_stream())
    for _ in range(3 if graph else 1):
        out.fill_(-7.0)
        stream.wait_stream(torch.cuda.current_stream())
        lib.call("cm21_find_bubbles", lib.plan(D, 1).handle, lib.ptr(delta), lib.ptr(out), rp, dp, len(r), prm,
                 lib.ptr(work), nbytes, lib.stream_handle(stream))
        stream.synchronize()
    return out.cpu().numpy(), nbytes, least


@pytest.mark.parametrize("D,L", [(64, 100.0), (64, 40.0), (96, 150.0), (128, 128.0), (128, 300.0), (160, 200.0)])
@pytest.mark.parametrize("LE", [True, False])
@pytest.mark.parametrize("fil,mean", [(1, 0.5), (1, 0.95), (1, 0.01), (2, 0.5)])
def test_all_radii_equal_one_launch_per_radius(gpu, D, L, LE, fil, mean):
    radii = pkg("Programs.find_HII_bubbles").radius_schedule(L, D)[0]
    want, _, _ = _run(D, L, LE, fil, mean, radii, False)
    got, nbytes, least = _run(D, L, LE, fil, mean, radii, True)
    print(f"D={D} ionized {np.mean(want == 1):.3f} workspace {nbytes >> 20} MiB (least {least >> 20})", flush=True)
    assert nbytes >= least and np.array_equal(got, want)


@pytest.mark.parametrize("n", [1, 2, 48, 49])
@pytest.mark.parametrize("LE", [True, False])
def test_all_radii_counts(gpu, n, LE):
    """One radius, two, the most that the table holds, and one more (which
    takes the launch per radius)."""
    radii = np.geomspace(30.0, 1.6, n).astype(np.float32)
    want, _, _ = _run(64, 100.0, LE, 1, 0.5, radii, False)
    got, _, _ = _run(64, 100.0, LE, 1, 0.5, radii, True)
    assert np.array_equal(got, want)


def test_all_radii_graph_replay(gpu):
    radii = pkg("Programs.find_HII_bubbles").radius_schedule(100.0, 64)[0]
    for LE in (True, False):
        want, _, _ = _run(64, 100.0, LE, 1, 0.5, radii, True)
        got, _, _ = _run(64, 100.0, LE, 1, 0.5, radii, True, graph=1)
        assert np.array_equal(got, want)


def test_sides_without_the_form_ask_for_the_least(gpu):
    lib = pkg("_lib")
    radii = np.array([3.0, 2.0], np.float32)
    rp = radii.ctypes.data_as(lib.c_float_p)
    for D, upd, fused in ((256, 0, 1), (100, 0, 1), (64, 1, 1), (64, 0, 0)):
        prm = lib.BubbleParams(box_len=100.0, zeta=30.0, growth_inv=1.0, filter_type=1, ref_fallthrough=1, update=upd,
                               fused=fused)
        assert lib.query("cm21_find_bubbles_full_workspace_bytes", D, rp, 2, prm) == \
            lib.query("cm21_find_bubbles_workspace_bytes", D, 2, upd)


@pytest.mark.parametrize("graph", [False, True])
def test_conv_bubbles_without_room_for_every_radius(gpu, graph):
    """Where the memory holds the workspace of the launch per radius but not that
    of every radius at once, the call still runs, with the same box."""
    fb, g = pkg("Programs.find_HII_bubbles"), pkg("gpu")
    D, L = 160, 160.0
    sp = pkg("cosmo_files.sigmas").PowerLawSpectrum(D, L)
    delta = g.c2r(g.grf_init(D, L, sp.amp, 5)).contiguous()
    from scipy.special import erfcinv
    dc = 1.686 / 0.12
    kw = dict(fil=2, LE=True, quiet=True, deltac=dc, sigma_min2=(dc / float(erfcinv(0.5 / 30.0))) ** 2 / 2.0, zeta=30.0,
              sig0=sp.sig0_discrete)
    want = fb.conv_bubbles(delta, {"BoxSize": L, "HIIdim": D}, **kw)
    fb._graph_cache.clear()
    stream = torch.cuda.Stream() if graph else None
    torch.cuda.synchronize()
    torch.cuda.empty_cache()
    room = torch.cuda.memory_reserved() + (400 << 20)
    torch.cuda.set_per_process_memory_fraction(room / torch.cuda.get_device_properties(0).total_memory)
    try:
        for _ in range(2):
            got = fb.conv_bubbles(delta, {"BoxSize": L, "HIIdim": D}, graph=graph, stream=stream, **kw)
            torch.cuda.synchronize()
            assert torch.equal(got, want)
    finally:
        torch.cuda.set_per_process_memory_fraction(1.0)
        fb._graph_cache.clear()
    assert (want == 1).any() and want.unique().numel() > 1000  # ionized cells and partial values


@pytest.mark.parametrize("LE", [True, False])
def test_gaussian_window_on_a_box_ionized_at_once(gpu, LE):
    """160^3 with filter 2: a box that is all ionized at the largest radius takes the
    launch per radius, which ends early there (0.82 times the time); the form with
    every radius at once asks for its workspace elsewhere, and the boxes are the same."""
    radii = pkg("Programs.find_HII_bubbles").radius_schedule(250.0, 160)[0]
    for mean, per_radius in ((1.0, False), (3.0, True)):
        want, _, _ = _run(160, 250.0, LE, 2, mean, radii, False)
        got, nbytes, least = _run(160, 250.0, LE, 2, mean, radii, True)
        assert (nbytes == least) == per_radius and np.array_equal(got, want)
    assert np.all(want == 1)
    for D, fil in ((160, 1), (128, 2)):
        assert _run(D, 250.0, LE, fil, 3.0, radii, True)[1] > _run(D, 250.0, LE, fil, 3.0, radii, False)[1]
