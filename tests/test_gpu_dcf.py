"""Pipe DCF on the GPU (mrn_dcf_calc) against the oracle's restatement of
RECON::dcf_calc (recon_lib.cpp:854-917) and DCFgridFFT (DCFgridFFT.cpp).

The GPU's general form adds with float atomics, its tile form along matrix
products, so the order of the additions into a grid cell differs from the
oracle's sample order: results agree to FP32 rounding of those sums, carried through the ratio iteration.  Bars: relative
L2 <= 1e-5 after one iteration, <= 1e-4 after 20 (the default), against the
FP32 oracle; the FP64 oracle within 1e-4.  The gather, the update, the table
and scale_kw have no ordering freedom.
"""
import numpy as np
import pytest
import torch

from oracle import oracle as orc
from mri_recon_amd import MrnError, dcf_calc, dcf_params, synth
from mri_recon_amd.dcf import dcf_grid_size, dcf_last_atomics
from tests.helpers import rel

pytestmark = pytest.mark.gpu


def dev(a):
    return torch.from_numpy(np.ascontiguousarray(a, np.float32)).cuda()


def radial(nspokes=300, npts=24, N=32):
    kx, ky, kz, _ = [t.numpy() for t in synth.radial_traj(nspokes, npts, N)]
    return kx, ky, kz


@pytest.mark.parametrize("iters,tol", [(1, 1e-5), (5, 3e-5), (20, 1e-4)])
def test_dcf_matches_oracle(iters, tol):
    kx, ky, kz = radial()
    kw, sums = dcf_calc(dev(kx), dev(ky), dev(kz), N=32, iters=iters, return_sums=True)
    p = orc.dcf_params(32, iters=iters)
    ref, rsums = orc.dcf_calc(p, kx, ky, kz, "f32")
    ref64, _ = orc.dcf_calc(p, kx, ky, kz, "f64")
    got = kw.cpu().numpy()
    e32, e64 = rel(got, ref), rel(got, ref64)
    print("dcf iters=%d: vs f32 %.2e vs f64 %.2e" % (iters, e32, e64))
    assert e32 <= tol and e64 <= 1e-4
    assert np.allclose(sums, rsums, rtol=1e-4)
    assert np.array_equal(got == 0, ref == 0)


@pytest.mark.parametrize("N,acc,kernel,dwin,os_", [((24, 16, 12), 1.0, "poly", 2.1, 2.1),
                                                  (32, 2.0, "poly", 2.1, 2.1),
                                                  (32, 1.0, "poly2", 1.5, 1.5),
                                                  (20, 1.5, "poly", 3.0, 2.5),
                                                  (16, 3.0, "poly", 4.0, 2.1)])
def test_dcf_settings_match_oracle(N, acc, kernel, dwin, os_):
    """Non-cubic sizes (the x extent follows Nz), kernel widening with |k|,
    the second polynomial, other widths and oversampling; the last case has
    rows of up to 10 taps (more than the scatter's 8 lanes per sample)."""
    n = N if isinstance(N, tuple) else (N, N, N)
    kx, ky, kz = radial(200, 16, min(n))
    kw = dcf_calc(dev(kx), dev(ky), dev(kz), N=n, iters=8, acc=acc, kernel=kernel, dwin=dwin, overgrid=os_)
    p = orc.dcf_params(n, iters=8, acc=acc, kernel=1 if kernel == "poly2" else 0, dwin=dwin, overgrid=os_)
    assert dcf_grid_size(dcf_params(n, dwin=dwin, overgrid=os_)) == orc.dcf_grid_size(p)
    ref, _ = orc.dcf_calc(p, kx, ky, kz, "f32")
    assert rel(kw.cpu().numpy(), ref) <= 5e-5


def test_dcf_single_sample_closed_form():
    t = orc.dcf_table(2.1, 0, "f64")
    want = 1.0 / (t[0] ** 2 + 2 * t[600] ** 2 + 2 * t[1200] ** 2) ** 3
    z = torch.zeros(1, dtype=torch.float32, device="cuda")
    kw = dcf_calc(z, z, z, N=32, iters=3).item()
    assert abs(kw / want - 1) < 2e-6


def test_dcf_duplicates_halve_and_edges():
    kx, ky, kz = radial(150, 20)
    # samples off the grid (beyond trunc(os*N+16)/2 cells) get weight 0
    kx = np.r_[kx, [400.0, -400.0]].astype(np.float32)
    ky = np.r_[ky, [0.0, 0.0]].astype(np.float32)
    kz = np.r_[kz, [0.0, 0.0]].astype(np.float32)
    a = dcf_calc(dev(kx), dev(ky), dev(kz), N=32, iters=6).cpu().numpy()
    b = dcf_calc(dev(np.r_[kx, kx]), dev(np.r_[ky, ky]), dev(np.r_[kz, kz]), N=32, iters=6).cpu().numpy()
    M = kx.size
    assert a[-1] == 0 and a[-2] == 0
    assert rel(b[:M], a / 2) < 1e-5 and rel(b[M:], a / 2) < 1e-5
    # no samples: nothing to do
    e = torch.zeros(0, dtype=torch.float32, device="cuda")
    assert dcf_calc(e, e, e, N=32).numel() == 0


def test_dcf_bad_arguments_raise():
    z = torch.zeros(4, dtype=torch.float32, device="cuda")
    with pytest.raises(MrnError, match="dcf_dwin"):
        dcf_calc(z, z, z, N=32, dwin=-1.0)
    with pytest.raises(MrnError, match="dcf_iter"):
        dcf_calc(z, z, z, N=32, iters=-2)
    with pytest.raises(MrnError, match="too large"):
        dcf_calc(z, z, z, N=32, dwin=40.0)


def test_dcf_parse_args():
    p = dcf_params(64, args=["-dcf_iter", "7", "-dcf_dwin", "3.0", "-dcf_overgrid", "1.8", "-dcf_acc", "2",
                             "-dcf_scale", "0.5", "-other"])
    assert (p.iters, p.dwin, p.overgrid, p.acc, p.scale) == (7, 3.0, np.float32(1.8), 2.0, 0.5)


def test_dcf_full_size_duplicate_property():
    """The 256^3 radial workload (5.12 M samples), where the oracle would take
    minutes: duplicating every sample doubles A^T A, so every weight halves."""
    kx, ky, kz, _ = synth.radial_traj(20000, 256, 256, device="cuda")
    a = dcf_calc(kx, ky, kz, N=256, iters=4)
    b = dcf_calc(torch.cat([kx, kx]), torch.cat([ky, ky]), torch.cat([kz, kz]), N=256, iters=4)
    M = kx.numel()
    assert torch.count_nonzero(a).item() > 0.99 * M
    assert rel(b[:M].cpu().numpy(), a.cpu().numpy() / 2) < 1e-4


@pytest.mark.parametrize("N,spokes,npts,dwin,os_", [(7, 3, 5, 2.1, 2.1), ((9, 21, 33), 40, 30, 1.0, 1.3),
                                                   (24, 400, 60, 2.5, 2.1), (31, 50, 40, 2.9, 1.7),
                                                   (20, 9000, 24, 2.0, 2.1)])
def test_dcf_tiles_match_oracle(N, spokes, npts, dwin, os_):
    """The one-width form at its edges: a grid of a few tiles with partly
    filled last ones, narrow and wide kernels (3 to 6 taps), tiles whose visits
    fill several work items (9000 spokes through the centre), samples off the
    grid and at infinity; the same weights on every call."""
    n = N if isinstance(N, tuple) else (N, N, N)
    kx, ky, kz = radial(spokes, npts, min(n))
    kx, ky, kz = [np.r_[k, e].astype(np.float32) for k, e in
                  ((kx, [300.0, 0.0, 0.0, 1e30]), (ky, [0.0, -300.0, 0.0, 0.0]), (kz, [0.0, 0.0, n[0] / 2.0, 0.0]))]
    d = [dev(k) for k in (kx, ky, kz)]
    got = dcf_calc(*d, N=n, iters=4, dwin=dwin, overgrid=os_).cpu().numpy()
    again = dcf_calc(*d, N=n, iters=4, dwin=dwin, overgrid=os_).cpu().numpy()
    assert np.array_equal(got, again, equal_nan=True)
    p = orc.dcf_params(n, iters=4, dwin=dwin, overgrid=os_)
    ref, _ = orc.dcf_calc(p, kx[:-1], ky[:-1], kz[:-1], "f32")
    assert not got[-1] > 0  # the sample at infinity has no taps
    assert rel(got[:-1], ref) <= 3e-5


def general(kx, ky, kz, **kw):
    """The general form of the same calculation: a kernel scale that grows by
    one part in 10^7 over |k| = 128."""
    return dcf_calc(kx, ky, kz, acc=float(np.nextafter(np.float32(1), np.float32(2))), **kw)


def best_ms(fn, reps=6):
    ev = [torch.cuda.Event(enable_timing=True) for _ in range(2)]
    best = 1e9
    for _ in range(reps):
        ev[0].record()
        fn()
        ev[1].record()
        torch.cuda.synchronize()
        best = min(best, ev[0].elapsed_time(ev[1]))
    return best


@pytest.mark.parametrize("N,spokes", [(32, 1500), (64, 800)])
def test_dcf_dense_centre_is_not_slower_by_tiles(N, spokes):
    """A small trajectory whose centre tiles hold thousands of visits: the tiles'
    walks are short enough that the call is not slower than the general form
    (with up to 2048 visits per walk it took 1.5 times as long)."""
    k = [dev(v) for v in radial(spokes, N, N)]
    t = best_ms(lambda: dcf_calc(*k, N=N, iters=20))
    assert dcf_last_atomics() == 0
    tg = best_ms(lambda: general(*k, N=N, iters=20))
    assert dcf_last_atomics() > 0
    print("dcf %d^3, %d spokes: %.2f ms, general %.2f" % (N, spokes, t, tg))
    assert t <= 1.1 * tg


@pytest.mark.parametrize("M", [100, 8191, 52000])
def test_dcf_item_lengths_match_oracle(M):
    """128 visits per work item up to 104857 samples, more beyond; here the tiles
    hold fewer, about as many, and several times that."""
    kx, ky, kz = [v[:M] for v in radial(M // 20 + 1, 20, 16)]
    got = dcf_calc(dev(kx), dev(ky), dev(kz), N=16, iters=4).cpu().numpy()
    assert dcf_last_atomics() == 0
    ref, _ = orc.dcf_calc(orc.dcf_params(16, iters=4), kx, ky, kz, "f32")
    assert rel(got, ref) <= 3e-5


@pytest.mark.parametrize("N,M,kind,iters,tiles", [
    (24, 5000, "radial", 0, False), (24, 5000, "radial", 2, False), (24, 5000, "radial", 3, True),
    (24, 524288, "radial", 1, False), (24, 524288, "radial", 2, True),   # iters * M at 2^20
    (256, 200000, "random", 5, False), (256, 200000, "random", 3, True), (256, 200000, "radial", 20, True),
    (128, 200000, "random", 20, True)])
def test_dcf_form_rule(N, M, kind, iters, tiles):
    """Which calls go by tiles: from 3 iterations or 2^20 sample visits on, and
    not with samples so scattered that the tiles' items are nearly empty.  Both
    forms' weights agree (to their summation order)."""
    if kind == "radial":
        kx, ky, kz = radial(-(-M // N), N, N)
    else:
        kx, ky, kz = np.random.default_rng(5).uniform(-N / 2, N / 2, (3, M)).astype(np.float32)
    k = [dev(v[:M]) for v in (kx, ky, kz)]
    got = dcf_calc(*k, N=N, iters=iters).cpu().numpy()
    if iters > 0:
        assert (dcf_last_atomics() == 0) == tiles
    ref = general(*k, N=N, iters=iters).cpu().numpy()
    assert rel(got, ref) <= 1e-4


def test_dcf_without_memory_for_the_tiles(monkeypatch):
    """The tiles' lists take memory the general form does not: without it the
    call is the general form's, not an error."""
    kx, ky, kz = radial(400, 60, 24)
    monkeypatch.setenv("MRN_ALLOC_MAX", "100000")
    got = dcf_calc(dev(kx), dev(ky), dev(kz), N=24, iters=4).cpu().numpy()
    assert dcf_last_atomics() > 0
    ref, _ = orc.dcf_calc(orc.dcf_params(24, iters=4), kx, ky, kz, "f32")
    assert rel(got, ref) <= 3e-5
