"""GPU L1 wavelet step and L1 FISTA against the oracle (oracle/gridfft_oracle.c).

* the device wavelet matches the FP64 oracle's transform (FP32 rounding) and
  inverts itself;
* the device threshold equals, bit for bit, the FP32 oracle's fraction
  threshold evaluated on the device's own coefficients (same |c| rounding, same
  float recurrence);
* the full cycle-spun L1 step and L1 FISTA (graph and no graph) match the
  oracle with the same shifts / seed.
"""
import math

import numpy as np
import pytest

from oracle import oracle as orc
from tests.helpers import crandn, radial_problem, rel, to_dev, traj_dev

N = 32


def _op(F=1, C=1, N_=N):
    from mri_recon_amd import GridFFT
    return GridFFT(N_, ncoils=C, nframes=F, overgrid=1.5)


@pytest.mark.gpu
@pytest.mark.parametrize("levels,shift", [((4, 4, 4), (0, 0, 0)), ((4, 4, 4), (1, 3, 2)), ((2, 1, 3), (3, 0, 1))])
def test_wavelet_matches_oracle_and_inverts(levels, shift):
    import torch
    op = _op(F=2)
    x = crandn((2, N, N, N), 5)
    X = to_dev(x)
    op.wavelet(X, levels, shift)
    got = X.cpu().numpy()
    for f in range(2):
        ref = orc.wavelet3d(x[f], levels, shift)
        assert rel(got[f], ref) < 2e-6
    op.wavelet(X, levels, shift, inverse=True)
    assert rel(X.cpu().numpy(), x) < 2e-6


@pytest.mark.gpu
@pytest.mark.parametrize("fraction", [0.3, 0.5, 0.8])
def test_threshold_bitwise_on_device_coefficients(fraction):
    import torch
    op = _op(F=2)
    x = crandn((2, N, N, N), 6)
    X = to_dev(x)
    sh = ((2, 1, 0),)
    thr = op.l1_wavelet(X.clone(), fraction, (4, 4, 4), shifts=sh)
    W = to_dev(x)
    op.wavelet(W, (4, 4, 4), sh[0])
    coef = W.cpu().numpy()
    ref = orc.fraction_threshold(coef, fraction, precision="f32")
    assert np.float32(thr) == np.float32(ref)


@pytest.mark.gpu
@pytest.mark.parametrize("spins", [1, 4])
def test_l1_step_matches_oracle(spins):
    op = _op(F=2)
    x = crandn((2, N, N, N), 7)
    shifts = orc.spin_shifts(11, 3 * spins).reshape(spins, 3)
    X = to_dev(x)
    thr = op.l1_wavelet(X, 0.6, (4, 4, 4), shifts=shifts.tolist())
    ref, rthr = orc.l1_wavelet(x, 0.6, (4, 4, 4), shifts, precision="f64")
    assert abs(thr - rthr) < 1e-4 * rthr
    assert rel(X.cpu().numpy(), ref) < 1e-4


@pytest.mark.gpu
def test_bad_l1_arguments_raise():
    from mri_recon_amd import MrnError
    op = _op()
    X = to_dev(crandn((1, N, N, N), 1))
    with pytest.raises(MrnError):
        op.l1_wavelet(X, 1.5)
    with pytest.raises(MrnError):
        op.l1_wavelet(X, 0.5, shifts=((0, 4, 0),))
    with pytest.raises(MrnError):
        op.set_fista_l1(0.5, spins=0)


@pytest.mark.gpu
@pytest.mark.parametrize("graph", [True, False])
def test_l1_fista_matches_oracle(graph):
    import torch
    Nf = 16
    traj, X, smaps, d = radial_problem(Nf, 2, 120, 16, seed=31)
    from mri_recon_amd import GridFFT
    op = GridFFT(Nf, ncoils=2, overgrid=1.5)
    op.set_traj(*traj_dev(traj))
    op.set_smaps(to_dev(smaps))
    op.set_kdata(to_dev(d))
    o = orc.OracleOp(Nf, overgrid=1.5, precision="f64")
    step, _ = o.power_method(smaps, traj, iters=15)
    iters, spins, seed = 5, 2, 9
    op.set_fista_l1(0.5, (4, 4, 4), spins, seed)
    Xg, res = op.fista(iters, step, graph=graph)
    thr = op.fista_thresholds(iters).numpy()
    Xr, rres, rthr = o.fista_l1(smaps, d, traj, iters, step, 0.5, (4, 4, 4), spins, seed)
    assert np.allclose(thr, rthr, rtol=2e-3)
    assert rel(Xg[0].cpu().numpy(), Xr) < 2e-3
    assert np.allclose(res.numpy(), rres, rtol=1e-3)
    # turning the step off gives plain FISTA again
    op.set_fista_l1(0.0)
    X0, _ = op.fista(iters, step, graph=graph)
    Xp, _ = o.fista(smaps, d, traj, iters, step)
    assert rel(X0[0].cpu().numpy(), Xp) < 1e-4


@pytest.mark.gpu
@pytest.mark.parametrize("n,levels", [((20, 34, 12), 4), ((4, 4, 6), 1), ((64, 32, 16), 1), ((84, 18, 10), 3),
                                      ((15, 32, 16), 2), ((2, 8, 8), 3)])
def test_l1_step_on_uneven_volumes(n, levels):
    """The step at partly filled tiles of the three-axis first level, lines
    shorter than the filter, one level only, and an odd axis (no level there:
    in place), two frames, against the FP64 oracle; and one forward and inverse
    transform of the same shifts in place, whose coefficients it thresholds."""
    op = _op(F=2, N_=n)
    x = crandn((2, n[2], n[1], n[0]), 17)
    shifts = orc.spin_shifts(3, 6).reshape(2, 3)
    X = to_dev(x)
    thr = op.l1_wavelet(X, 0.5, (levels,) * 3, shifts=shifts.tolist())
    ref, rthr = orc.l1_wavelet(x, 0.5, (levels,) * 3, shifts, precision="f64")
    assert abs(thr - rthr) <= 1e-4 * rthr
    assert rel(X.cpu().numpy(), ref) < 1e-4
    W = to_dev(x)
    op.wavelet(W, (levels,) * 3, [int(v) for v in shifts[0]])
    c = W.cpu().numpy()
    assert np.float32(op.l1_wavelet(to_dev(x), 0.5, (levels,) * 3, shifts=shifts[:1].tolist())) == \
        np.float32(orc.fraction_threshold(c, 0.5, precision="f32"))


def _bisect(c, fraction):
    """The fraction threshold by plain counting, one float32 step at a time; a
    NaN is below nothing and no extreme."""
    with np.errstate(all="ignore"):
        a = np.sqrt(c.real.astype(np.float64) ** 2 + c.imag.astype(np.float64) ** 2).astype(np.float32).ravel()
        h, n = np.float32(0.5), a.size
        mn, mx = np.nanmin(a), np.nanmax(a)
        target, acc = int(np.float64(np.float32(fraction)) * n), int(0.001 * n)
        v, hi, lo = h * (mx - mn), np.float32(fraction) * mx, mn
        if target < 2:
            return np.float32(0)
        for it in range(1, 65):
            found = int(np.count_nonzero(a < v))
            if abs(found - target) <= acc or it == 64:
                break
            if found > target:
                hi = v
            else:
                lo = v
            v = h * (hi + lo)
    return v


@pytest.mark.gpu
@pytest.mark.parametrize("levels", [(3, 3, 3), (3, 1, 2), (2, 3, 2)])
@pytest.mark.parametrize("fraction,scale,bad", [(0.02, 1.0, None), (0.4, 1e-25, None), (0.9, 1e25, None),
                                                (0.97, 1.0, np.nan), (0.5, 1.0, np.inf), (0.5, 0.0, None)])
def test_threshold_counts_all_values(levels, fraction, scale, bad):
    """The histogram over sorted candidates counts what a comparison per candidate
    counts: fractions that put the first value above the bracket, magnitudes
    whose squares leave float32, a NaN, an infinity, equal values; axes with
    levels that others do not have (finished in place).  The same bits as one
    float32 step at a time on the device's coefficients."""
    x = crandn((2, N, N, N), 9) * np.float32(scale)
    if bad is not None:
        x[1, 3, 4, 5] = bad
    sh = ((1, 2, 3),)
    op = _op(F=2)
    X = to_dev(x)
    thr = op.l1_wavelet(X, fraction, levels, shifts=sh)
    W = to_dev(x)
    op.wavelet(W, levels, sh[0])
    c = W.cpu().numpy()
    ref = _bisect(c, fraction)
    assert np.float32(thr) == ref or (np.isnan(thr) and np.isnan(ref))
    if bad is None:  # and the step: threshold on those coefficients, transformed back
        a = np.sqrt(c.real.astype(np.float64) ** 2 + c.imag.astype(np.float64) ** 2).astype(np.float32)
        with np.errstate(all="ignore"):
            f = np.where(a <= ref, np.float32(0), np.float32(1) - ref / a)
        W = to_dev((c * f).astype(np.complex64))
        op.wavelet(W, levels, sh[0], inverse=True)
        got, want = X.cpu().numpy().astype(np.complex128), W.cpu().numpy().astype(np.complex128)
        assert rel(got, want) <= 1e-6


@pytest.mark.gpu
def test_l1_step_without_levels_on_many_frames():
    """Odd axes have no level: the step is the threshold alone, of more frames
    than a launch grid has rows."""
    F = 66000
    op = _op(F=1, N_=(3, 5, 3))
    x = crandn((F, 3, 5, 3), 5)
    X = to_dev(x)
    thr = np.float32(op.l1_wavelet(X, 0.5, (2, 2, 2), shifts=((0, 1, 2),)))
    a = np.sqrt(x.real.astype(np.float64) ** 2 + x.imag.astype(np.float64) ** 2).astype(np.float32)
    assert abs(np.count_nonzero(a < thr) / a.size - 0.5) <= 2e-3
    assert rel(X.cpu().numpy(), np.where(a <= thr, 0, x * (np.float32(1) - thr / a))) <= 1e-6
