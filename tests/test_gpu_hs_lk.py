"""GPU parity of the Horn-Schunck and Lucas-Kanade paths against the CPU
oracle: every stage and every full solve must match bit for bit (the kernels
use the oracle's operation order, no FMA contraction, IEEE division)."""
import numpy as np
import pytest

import oracle as O
from amdflow import HornSchunck, LucasKanade, lk_pyramidal, synth
from amdflow import debug as D

pytestmark = pytest.mark.gpu


def _rand(rng, h, w, scale=1.0):
    return (rng.standard_normal((h, w)) * scale).astype(np.float32)


@pytest.mark.parametrize("K,R", [(1, 2), (2, 2), (1, 4), (2, 4), (4, 4), (1, 8), (2, 8), (4, 8),
                                 (8, 8)])
@pytest.mark.parametrize("h,w,iters", [(37, 70, 5), (130, 257, 13), (480, 640, 3)])
def test_hs_jacobi_bitexact(K, R, h, w, iters):
    rng = np.random.default_rng(K * 10 + R + h)
    du, dv = _rand(rng, h, w, 0.2), _rand(rng, h, w, 0.2)
    Ix, Iy, Iz = _rand(rng, h, w, 5.0), _rand(rng, h, w, 5.0), _rand(rng, h, w, 3.0)
    gu, gv = D.hs_jacobi(du, dv, Ix, Iy, Iz, 15.0, iters, K, R)
    ou, ov = du, dv
    for _ in range(iters):
        ou, ov = O.hs_jacobi(ou, ov, Ix, Iy, Iz, 15.0)
    assert np.array_equal(gu, ou) and np.array_equal(gv, ov)


@pytest.mark.parametrize("scale", [0.0, 0.7, 4.0])
def test_hs_warp_derivatives_bitexact(scale):
    rng = np.random.default_rng(int(scale * 10) + 1)
    h, w = 61, 95
    I0 = (rng.random((h, w)) * 255).astype(np.float32)
    I1 = (rng.random((h, w)) * 255).astype(np.float32)
    u, v = _rand(rng, h, w, scale), _rand(rng, h, w, scale)
    I1w, Ix, Iy, Iz = D.hs_warp_derivatives(I0, I1, u, v)
    ow = np.empty_like(I0)
    O._lib.orc_hs_warp(O._p(I1), w, h, w, O._p(u), O._p(v), O._p(ow))
    ox, oy, oz = O.hs_derivatives(I0, ow)
    assert np.array_equal(I1w, ow)
    if scale == 0.0:
        assert np.array_equal(I1w, I1)          # zero flow warps to the identity
    for g, o in zip((Ix, Iy, Iz), (ox, oy, oz)):
        assert np.array_equal(g, o)


def test_hs_640x480_single_scale_matches_oracle():
    """The HS workload: 640x480, |flow| <= 2 px, alpha 15, 100 Jacobi sweeps."""
    cfg = synth.CONFIGS["hs_640x480"]
    I0, I1, fu, fv = synth.make_pair(cfg["width"], cfg["height"], cfg["cap"], 7)
    w, h = cfg["width"], cfg["height"]
    with HornSchunck(1, w, w, h) as hs:
        u, v = hs.ComputeFlow(I0, I1, w, h, w, 15.0, 1, 1, 100)
    ou, ov = O.hs_compute(I0, I1, alpha=15.0, nLevels=1, nWarpIters=1, nSolverIters=100)
    assert np.array_equal(u, ou) and np.array_equal(v, ov)


@pytest.mark.parametrize("levels", [1, 2, 3, 4])
def test_hs_every_level_count_matches_oracle(levels):
    """Every level but the last swaps the solver's flow buffers, so the host
    entry point must return the final flow after an odd and an even number
    of swaps; 96x80 also pads the coarse levels' rows (48 -> stride 64)."""
    import torch
    w, h = 96, 80
    I0, I1, _, _ = synth.make_pair(w, h, 3.0, 7, bumps=True)
    ou, ov = O.hs_compute(I0, I1, 15.0, levels, 2, 30)
    with HornSchunck(levels, w, w, h) as hs:
        u, v = hs.ComputeFlow(I0, I1, w, h, w, 15.0, levels, 2, 30)
        assert np.array_equal(u, ou) and np.array_equal(v, ov)
        d0 = torch.from_numpy(np.ascontiguousarray(I0, np.float32)).cuda()
        d1 = torch.from_numpy(np.ascontiguousarray(I1, np.float32)).cuda()
        du = torch.empty(w * h, dtype=torch.float32, device="cuda")
        dv = torch.empty(w * h, dtype=torch.float32, device="cuda")
        hs.compute_device(d0.data_ptr(), d1.data_ptr(), du.data_ptr(), dv.data_ptr(), 15.0, levels,
                          2, 30)
        assert np.array_equal(du.cpu().numpy().reshape(h, w), ou)
        assert np.array_equal(dv.cpu().numpy().reshape(h, w), ov)


@pytest.mark.parametrize("shape", [(1, 8), (4, 4), (8, 8)])
def test_hs_multilevel_strided_matches_oracle(shape):
    w, h = 300, 200
    stride = 320
    I0, I1, _, _ = synth.make_pair(w, h, 4.0, 8)
    P0 = np.zeros((h, stride), np.float32); P0[:, :w] = I0
    P1 = np.zeros((h, stride), np.float32); P1[:, :w] = I1
    with HornSchunck(3, stride, w, h) as hs:
        hs.set_jacobi_shape(*shape)
        u, v = hs.ComputeFlow(P0, P1, w, h, stride, 0.2, 3, 2, 23)
    ou, ov = O.hs_compute(P0[:, :w], P1[:, :w], alpha=0.2, nLevels=3, nWarpIters=2,
                          nSolverIters=23, stride=stride)
    assert np.array_equal(u[:, :w], ou[:, :w]) and np.array_equal(v[:, :w], ov[:, :w])


@pytest.mark.parametrize("w,h,sweeps", [(1, 1, 5), (2, 3, 14), (5, 200, 15), (36, 4, 29), (63, 31, 1),
                                        (65, 49, 16), (129, 97, 3), (641, 359, 43), (900, 701, 13)])
def test_hs_shape_by_size_matches_oracle(w, h, sweeps):
    """The launch shape follows the level's size and the sweep count: frames
    narrower than a halo (mirrored columns wrap around), one tile, ragged
    tiles, both tile heights, a short last launch."""
    rng = np.random.default_rng(w + h)
    I0 = (rng.random((h, w)) * 255).astype(np.float32)
    I1 = (rng.random((h, w)) * 255).astype(np.float32)
    with HornSchunck(1, w, w, h) as hs:
        u, v = hs.ComputeFlow(I0, I1, w, h, w, 15.0, 1, 2, sweeps)
    ou, ov = O.hs_compute(I0, I1, alpha=15.0, nLevels=1, nWarpIters=2, nSolverIters=sweeps)
    assert np.array_equal(u, ou) and np.array_equal(v, ov)


@pytest.mark.parametrize("w,stride,h,levels", [(8, 8, 4096, 2), (12, 12, 2000, 2), (8, 15, 1000, 3),
                                               (15, 16, 700, 3), (31, 33, 400, 4)])
def test_hs_narrow_levels_match_oracle(w, stride, h, levels):
    """Coarse levels have pitches of whole 32 columns: on narrow frames their
    planes are larger than the finest level's, and so are the buffers that all
    levels share.  Two calls, as the second finds the first one's values."""
    rng = np.random.default_rng(w + h)
    I0 = (rng.random((h, stride)) * 255).astype(np.float32)
    I1 = (rng.random((h, stride)) * 255).astype(np.float32)
    ou, ov = O.hs_compute(np.ascontiguousarray(I0[:, :w]), np.ascontiguousarray(I1[:, :w]), alpha=15.0,
                          nLevels=levels, nWarpIters=2, nSolverIters=9)
    with HornSchunck(levels, stride, w, h) as hs:
        for _ in range(2):
            u, v = hs.ComputeFlow(I0, I1, w, h, stride, 15.0, levels, 2, 9)
            assert np.array_equal(u[:, :w], ou) and np.array_equal(v[:, :w], ov)


@pytest.mark.parametrize("scale", [1e-37, 1e-41, 3e-45])
def test_hs_jacobi_subnormal_increments_bitexact(scale):
    """Quotients that land on and between subnormal floats (a diffusion front
    in a static region), with divisors that have short mantissas: the exact
    quotient is often halfway between two subnormals."""
    rng = np.random.default_rng(9)
    h, w = 40, 70
    du = (rng.integers(-9, 10, (h, w)) * scale).astype(np.float32)
    dv = (rng.integers(-9, 10, (h, w)) * scale).astype(np.float32)
    Ix = rng.integers(-6, 7, (h, w)).astype(np.float32)
    Iy = rng.integers(-6, 7, (h, w)).astype(np.float32)
    Iz = np.zeros((h, w), np.float32)
    gu, gv = D.hs_jacobi(du, dv, Ix, Iy, Iz, 1.0, 2, 2, 2)
    ou, ov = du, dv
    for _ in range(2):
        ou, ov = O.hs_jacobi(ou, ov, Ix, Iy, Iz, 1.0)
    assert np.array_equal(gu, ou) and np.array_equal(gv, ov)


@pytest.mark.parametrize("spac,temp,win", [(3, 2, 5), (5, 2, 7), (7, 3, 3), (9, 5, 9), (1, 2, 5)])
def test_lk_single_scale_matches_oracle(spac, temp, win):
    rng = np.random.default_rng(spac * 10 + temp)
    h, w = 90, 130
    frames = [synth.quantize(synth.make_pair(w, h, 1.0, 40 + k)[0]) for k in range(temp + 2)]
    Vx = np.zeros(h * w, np.float32)
    Vy = np.zeros(h * w, np.float32)
    ring = np.zeros((temp, h, w), np.uint8)
    with LucasKanade(spac, temp, win, w, h) as lk:
        for fr, f in enumerate(frames):
            lk.copy_frames_circularbuffer_GPU_wrapper(f, temp, fr, w * h)
            ring[fr % temp] = f
            if fr >= temp - 1:
                lk.lucas_kanade(Vx, Vy, fr)
                ox, oy = O.lk_single(ring, fr, spac, win)
                assert np.array_equal(Vx.reshape(h, w), ox)
                assert np.array_equal(Vy.reshape(h, w), oy)


@pytest.mark.parametrize("w,h,win,iters", [(320, 240, 3, 1), (320, 240, 5, 5), (320, 240, 7, 5),
                                           (333, 211, 7, 11), (333, 211, 9, 6), (97, 61, 3, 17),
                                           (640, 360, 7, 5), (801, 401, 3, 10), (721, 433, 9, 5),
                                           (700, 451, 5, 9)])
def test_lk_pyramidal_blocked_levels_match_oracle(w, h, win, iters):
    """Windows up to 9 x 9 run blocks of iterations per launch: levels of at
    most 300,000 pixels the deepest blocks, larger levels blocks with a halo
    of at most 9 pixels (9, 4 and 2 iterations at windows 3, 5 and 9); a
    count beyond one block's takes several; ragged tile edges; window 11
    runs the three-kernel iteration."""
    I0, I1, _, _ = synth.make_pair(w, h, 4.0, 31 + win + iters)
    u, v = lk_pyramidal(I0, I1, levels=3, zf=0.5, sigma=1.0, window=win, iters=iters, det_eps=1e-6)
    ou, ov = O.lk_pyr(I0, I1, levels=3, zf=0.5, sigma=1.0, win=win, iters=iters, det_eps=1e-6)
    assert np.array_equal(u, ou) and np.array_equal(v, ov)


# Rows per thread and iterations per launch follow the level's size and window:
# 1, 2 and 4 rows with a shorter last launch, levels one pixel beyond a tile's
# centre, frames lower or narrower than one tile.  Zoom factors 1/2 and 0.6
# sample in pairs of lanes in part of the waves or none; at 0.8 the levels'
# tensors do not fit one buffer and are formed level by level.  The arithmetic
# is the oracle's: no difference.
@pytest.mark.parametrize("w,h,win,iters,levels,zf", [(40, 30, 5, 4, 1, 0.5), (53, 13, 3, 3, 1, 0.5),
                                                     (105, 65, 3, 8, 2, 0.5), (161, 121, 9, 4, 2, 0.5),
                                                     (333, 251, 7, 5, 3, 0.5), (643, 361, 5, 4, 2, 0.5),
                                                     (1283, 701, 3, 3, 2, 0.5), (901, 701, 9, 3, 1, 0.5),
                                                     (200, 150, 5, 2, 3, 0.8), (211, 157, 3, 4, 3, 0.6)])
def test_lk_pyramidal_shapes_by_size_match_oracle(w, h, win, iters, levels, zf):
    I0, I1, _, _ = synth.make_pair(w, h, 3.0, 51 + w + win)
    u, v = lk_pyramidal(I0, I1, levels=levels, zf=zf, sigma=1.0, window=win, iters=iters, det_eps=1e-6)
    ou, ov = O.lk_pyr(I0, I1, levels=levels, zf=zf, sigma=1.0, win=win, iters=iters, det_eps=1e-6)
    assert np.array_equal(u, ou) and np.array_equal(v, ov)


@pytest.fixture
def unblocked():
    D.lk_force_unblocked(True)
    yield
    D.lk_force_unblocked(False)


@pytest.mark.parametrize("w,h,win,iters,levels,zf", [(64, 48, 3, 3, 1, 0.5), (161, 121, 5, 3, 2, 0.5),
                                                     (333, 251, 9, 4, 3, 0.5), (105, 165, 7, 2, 2, 0.8),
                                                     (120, 90, 11, 3, 2, 0.5), (120, 90, 1, 3, 2, 0.5)])
def test_lk_pyramidal_unblocked_matches_oracle(w, h, win, iters, levels, zf, unblocked):
    """Frames beyond the blocked kernel's limits (a side of 2^24, more than 2^30
    pixels) iterate with one launch per step: here at small sizes, windows of
    the fused tensor (3 to 9) and others."""
    I0, I1, _, _ = synth.make_pair(w, h, 3.0, 57 + w + win)
    u, v = lk_pyramidal(I0, I1, levels=levels, zf=zf, sigma=1.0, window=win, iters=iters, det_eps=1e-6)
    ou, ov = O.lk_pyr(I0, I1, levels=levels, zf=zf, sigma=1.0, win=win, iters=iters, det_eps=1e-6)
    assert np.array_equal(u, ou) and np.array_equal(v, ov)


def test_lk_pyramidal_many_rows_of_two_columns():
    """2^27 rows make 2^24 tensor tiles, more than one grid dimension takes.
    The flow of the first rows does not see the others: it has the bits of a
    frame that ends earlier."""
    import torch
    from amdflow.lk import lk_pyramidal_device
    H, N, K = 1 << 27, 4096, 1024
    y = np.arange(N, dtype=np.float32)[:, None] + np.float32([0.0, 0.3])
    I0 = (127 + 90 * np.sin(0.4 * y)).astype(np.float32)
    I1 = (127 + 90 * np.sin(0.4 * (y - 0.7))).astype(np.float32)
    d0, d1 = (torch.from_numpy(a).cuda().reshape(-1).repeat(H // N) for a in (I0, I1))
    u, v = (torch.full((2 * H,), np.nan, dtype=torch.float32, device="cuda") for _ in range(2))
    lk_pyramidal_device(d0.data_ptr(), d1.data_ptr(), 2, H, u.data_ptr(), v.data_ptr(), levels=1, zf=0.5,
                        sigma=1.0, window=3, iters=1, det_eps=1e-6)
    ou, ov = O.lk_pyr(I0, I1, levels=1, zf=0.5, sigma=1.0, win=3, iters=1, det_eps=1e-6)
    for got, want in ((u, ou), (v, ov)):
        assert np.array_equal(got[:2 * K].cpu().numpy().reshape(K, 2), want[:K])
        assert bool(torch.isfinite(got).all())


@pytest.mark.parametrize("bad", [np.nan, np.inf, 3e38])
def test_lk_pyramidal_non_finite_frames_match_oracle(bad):
    """A frame value that makes flows non-finite or huge: such waves take the
    clamped taps, the others the paired ones."""
    I0, I1, _, _ = synth.make_pair(150, 120, 3.0, 53)
    I1 = I1.copy()
    I1[60, 70] = bad
    u, v = lk_pyramidal(I0, I1, levels=1, zf=0.5, sigma=1.0, window=5, iters=4, det_eps=1e-6)
    ou, ov = O.lk_pyr(I0, I1, levels=1, zf=0.5, sigma=1.0, win=5, iters=4, det_eps=1e-6)
    assert np.array_equal(u, ou, equal_nan=True) and np.array_equal(v, ov, equal_nan=True)


def test_lk_pyramidal_1280x720_matches_oracle():
    """The LK workload: 1280x720, |flow| <= 8 px, 3 levels, 7x7, 5 iterations/level."""
    cfg = synth.CONFIGS["lk_1280x720"]
    I0, I1, _, _ = synth.make_pair(cfg["width"], cfg["height"], cfg["cap"], 21)
    u, v = lk_pyramidal(I0, I1, levels=3, zf=0.5, sigma=1.0, window=7, iters=5, det_eps=1e-6)
    ou, ov = O.lk_pyr(I0, I1, levels=3, zf=0.5, sigma=1.0, win=7, iters=5, det_eps=1e-6)
    assert np.array_equal(u, ou) and np.array_equal(v, ov)


@pytest.mark.parametrize("levels,win,iters", [(1, 5, 3), (2, 9, 4), (4, 7, 2), (2, 3, 3), (2, 11, 2),
                                               (1, 1, 2)])
def test_lk_pyramidal_variants_match_oracle(levels, win, iters):
    """Windows 3-9 run the blocked iteration kernel, 1 and 11 the three-kernel
    path; both match the oracle bit for bit."""
    I0, I1, _, _ = synth.make_pair(257, 190, 3.0, 22 + levels)
    u, v = lk_pyramidal(I0, I1, levels=levels, window=win, iters=iters)
    ou, ov = O.lk_pyr(I0, I1, levels=levels, win=win, iters=iters)
    assert np.array_equal(u, ou) and np.array_equal(v, ov)


@pytest.mark.parametrize("zf,sigma", [(0.6, 1.0), (0.5, 2.5), (0.5, 3.5)])
def test_lk_pyramidal_zoom_and_blur_variants_match_oracle(zf, sigma):
    """Zoom 1/2 with taps up to 16 runs the tiled pyramid kernel; another
    zoom factor or wider taps (sigma 3.5: 18 taps) the two-pass form."""
    I0, I1, _, _ = synth.make_pair(211, 157, 3.0, 41)
    u, v = lk_pyramidal(I0, I1, levels=3, zf=zf, sigma=sigma, window=5, iters=3)
    ou, ov = O.lk_pyr(I0, I1, levels=3, zf=zf, sigma=sigma, win=5, iters=3)
    assert np.array_equal(u, ou) and np.array_equal(v, ov)


@pytest.mark.parametrize("out", ["separate", "over_I0", "over_I1"])
def test_lk_pyramidal_device_output_placement(out):
    """The device entry point reads level 0 from the caller's frames and its
    last iteration writes the caller's flow buffers directly; flow buffers that
    overlap the frames take the copying path.  Both match the oracle."""
    import torch
    from amdflow import lk_pyramidal_device
    w, h = 301, 173
    I0, I1, _, _ = synth.make_pair(w, h, 4.0, 31)
    ou, ov = O.lk_pyr(I0, I1, levels=3, win=7, iters=3)
    d0 = torch.from_numpy(I0.reshape(-1).copy()).cuda()
    d1 = torch.from_numpy(I1.reshape(-1).copy()).cuda()
    du = torch.empty(w * h, device="cuda")
    dv = torch.empty(w * h, device="cuda")
    if out == "over_I0":
        du = d0
    elif out == "over_I1":
        dv = d1
    lk_pyramidal_device(d0.data_ptr(), d1.data_ptr(), w, h, du.data_ptr(), dv.data_ptr(),
                        levels=3, window=7, iters=3)
    torch.cuda.synchronize()
    assert np.array_equal(du.cpu().numpy(), ou.reshape(-1))
    assert np.array_equal(dv.cpu().numpy(), ov.reshape(-1))
