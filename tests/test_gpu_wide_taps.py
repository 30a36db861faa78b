"""Samples exactly on the kernel window's edge have one more tap per axis
than the rest (taps ceil(dk - dwin) .. floor(dk + dwin) with dk - dwin an
integer, gridFFT.cpp:1061-1094).  The tile scatter sizes each tile's bin
reach for the usual count and scatters those samples separately; the gather
takes them tap by tap.  Trajectories with many such samples (half-integer dk
for dwin 2.5, integer dk for dwin 2.0, at os 2 where dk = 2 k + S/2 is exact)
against the FP32 oracle, for every accumulate form."""
import numpy as np
import pytest

from oracle import oracle as orc
from mri_recon_amd import GridFFT
from tests.helpers import crandn, rel, to_dev, traj_dev
from mri_recon_amd import synth

pytestmark = pytest.mark.gpu


def _edge_traj(N, dwin, n_edge, seed):
    rng = np.random.default_rng(seed)
    kx, ky, kz, kw = [t.numpy() for t in synth.radial_traj(300, 24, N)]
    # k = j / 2 + off: dk = 2 k + S/2 = j + 2 off + S/2, on the window edge for off = dwin % 1 / 2
    off = (dwin % 1.0) / 2.0
    j = rng.integers(-N + 4, N - 4, size=(n_edge, 3))
    e = (j / 2.0 + off).astype(np.float32)
    axes = rng.integers(0, 3, size=n_edge)  # one axis on the edge, the others anywhere
    other = rng.uniform(-N / 2 + 2, N / 2 - 2, size=(n_edge, 3)).astype(np.float32)
    pts = np.where(np.arange(3)[None, :] == axes[:, None], e, other)
    pts[: n_edge // 4] = e[: n_edge // 4]  # all three axes on the edge
    kx = np.concatenate([kx, pts[:, 0]]).astype(np.float32)
    ky = np.concatenate([ky, pts[:, 1]]).astype(np.float32)
    kz = np.concatenate([kz, pts[:, 2]]).astype(np.float32)
    kw = np.concatenate([kw, rng.uniform(0.5, 2.0, n_edge)]).astype(np.float32)
    return kx, ky, kz, kw


@pytest.mark.parametrize("dwin", [2.5, 2.0])
@pytest.mark.parametrize("C,kw", [(16, {}), (8, {}), (4, {}), (16, {"scatter_valu": True}),
                                  (16, {"bin_edge": 2})])
def test_window_edge_samples(dwin, C, kw):
    N = 32
    traj = _edge_traj(N, dwin, 500, seed=int(dwin * 10) + C)
    smaps = synth.coil_maps(C, N, seed=5).numpy()
    X = crandn((N, N, N), 6)
    d = crandn((C, traj[0].size), 7)
    op = GridFFT(N, ncoils=C, overgrid=2.0, dwin=dwin, **kw)
    op.set_traj(*traj_dev(traj))
    op.set_smaps(to_dev(smaps))
    o32 = orc.OracleOp(N, overgrid=2.0, dwin=dwin, precision="f32")
    h = op.forward(to_dev(d), accumulate=False).cpu().numpy()
    a = op.backward(to_dev(X)).cpu().numpy()
    eh = rel(h, o32.kspace_to_image(d, smaps, traj))
    ea = rel(a, o32.image_to_kspace(X, smaps, traj))
    print("dwin %.1f C=%d %s: A^H %.2e A %.2e" % (dwin, C, kw, eh, ea))
    assert eh <= 1e-5 and ea <= 1e-5


@pytest.mark.parametrize("C,spokes", [(1, 300), (5, 480), (16, 40), (16, 480), (8, 513), (2, 1300)])
def test_centre_of_many_readouts(C, spokes):
    """Every readout starts at k = 0, a window edge at dwin = 2: most listed
    samples are one point, summed before they are added, in chunks of 512; the
    first readout runs along kz, an edge on x and y whose cells are the centre's
    too.  Against the oracle, and the same bits on every call where the list fits
    one chunk."""
    N = 32
    traj = [t.numpy() for t in synth.radial_traj(spokes, 24, N)]
    traj[3] = np.maximum(traj[3], 0.5).astype(np.float32)  # the centre takes part
    smaps = synth.coil_maps(C, N, seed=5).numpy()
    d = crandn((C, traj[0].size), 7)
    op = GridFFT(N, ncoils=C, overgrid=1.5, dwin=2.0)
    op.set_traj(*traj_dev(traj))
    op.set_smaps(to_dev(smaps))
    h = [op.forward(to_dev(d), accumulate=False).cpu().numpy() for _ in range(5)]
    if spokes + 23 <= 512:
        assert all(np.array_equal(h[0], x) for x in h[1:])
    o32 = orc.OracleOp(N, overgrid=1.5, dwin=2.0, precision="f32")
    assert rel(h[0], o32.kspace_to_image(d, smaps, traj)) <= 1e-5


@pytest.mark.parametrize("C,n,repeat,by_sample", [(1, 32767, 1, 0), (1, 32768, 1, 1), (2, 8192, 1, 1), (4, 2047, 1, 0),
                                                  (4, 2048, 1, 1), (8, 512, 1, 0), (8, 513, 1, 1), (16, 512, 1, 0),
                                                  (16, 513, 1, 1), (24, 3000, 3, 1), (16, 4000, 5, 0)])
def test_long_lists_of_grid_positions(C, n, repeat, by_sample):
    """Samples on grid positions (Cartesian lines, partitions of a stack): the
    list's taps are added sample by sample where that costs less than every
    class of cells looking at every sample, on both sides of each line of the
    rule, and where several samples share a position.  Against the oracle."""
    N = 48 if C > 1 else 64
    rng = np.random.default_rng(n + C)
    ax = np.arange(-N // 2 + 4, N // 2 - 4)  # dk = 2 k + S / 2: an integer, the edge at dwin = 2
    pick = rng.permutation(ax.size ** 3)[: -(-n // repeat)]
    pts = np.stack([ax[pick % ax.size], ax[pick // ax.size % ax.size], ax[pick // ax.size ** 2]], 1)
    k = [np.repeat(pts[:, a], repeat)[:n].astype(np.float32) for a in range(3)]
    traj = k + [rng.uniform(0.5, 2.0, n).astype(np.float32)]
    smaps = synth.coil_maps(C, N, seed=5).numpy()
    d = crandn((C, n), 7)
    op = GridFFT(N, ncoils=C, overgrid=2.0, dwin=2.0)
    op.set_traj(*traj_dev(traj))
    op.set_smaps(to_dev(smaps))
    st = op.frame_stats()
    assert st["wide"] == n and st["wide_by_sample"] == by_sample
    o32 = orc.OracleOp(N, overgrid=2.0, dwin=2.0, precision="f32")
    assert rel(op.forward(to_dev(d), accumulate=False).cpu().numpy(), o32.kspace_to_image(d, smaps, traj)) <= 1e-5


def test_frames_of_either_form_in_one_launch():
    """Fused frames: one whose list is the centre of its readouts, one on grid
    positions, one without a list.  E'E of all frames against frame by frame."""
    N, C = 32, 8
    rng = np.random.default_rng(3)
    centre = [t.numpy() for t in synth.radial_traj(600, 24, N)]
    centre[3] = np.maximum(centre[3], 0.5).astype(np.float32)
    grid = [rng.integers(-10, 10, 2000).astype(np.float32) for _ in range(3)] + [np.ones(2000, np.float32)]
    off = [g + np.float32(0.3) for g in grid[:3]] + grid[3:]
    smaps = synth.coil_maps(C, N, seed=5)
    out = []
    for fuse in (1, 0):
        op = GridFFT(N, ncoils=C, nframes=3, overgrid=2.0, dwin=2.0, fuse_frames=fuse)
        op.set_smaps(smaps.cuda())
        for f, t in enumerate((centre, grid, off)):
            op.set_traj(*traj_dev(t), frame=f)
            op.set_kdata(to_dev(crandn((C, t[0].size), 11 + f)), frame=f)
        assert [op.frame_stats(f)["wide_by_sample"] for f in range(3)] == [0, 1, 0]
        out.append(op.cg(2, trace=False)[0].cpu().numpy())
        op.close()
    # two iterations over sums whose atomics differ in order: FP32 rounding, grown by the steps
    assert rel(out[0], out[1]) <= 1e-5
