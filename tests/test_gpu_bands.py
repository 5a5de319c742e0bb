"""Band renderer (plan kernel + one-shot band writer) against the splat renderer (GPU).

dsx_render_fast_bands must give dsx_render_fast's output bit for bit: the plan
reproduces the splat kernel's fixed-point scale and exact maximum, and the band
writer adds the same fixed-point terms.  Both are called through the C ABI on
the same seeded spot lists; the outputs start as NaN so that every pixel must
be written.  The spot lists mix in-frame and out-of-frame spots, spots on the
same pixel (last write wins), spots within the tap radius of the edges
(reflected taps) and the shapes whose last band is partial.  The library
parity tests (test_gpu_parity.py) check the same path against the FP64
oracle through engine.render_spots.
"""

import ctypes

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _lib():
    from diffsims_amd import _lib as lib
    return lib, lib.load(require_gpu=True)


def _spot_lists(n, cap, H, W, mean, seed, edge=0.0, dup=0.0, margin=2.0, R=4):
    """Spot lists in pixel units around the default centre (calibration 1)."""
    import torch
    rng = np.random.default_rng(seed)
    cnt = np.minimum(rng.poisson(mean, n), cap).astype(np.int32)
    X = rng.uniform(-margin, W + margin, (n, cap))
    Y = rng.uniform(-margin, H + margin, (n, cap))
    if edge > 0:
        e = rng.random((n, cap)) < edge
        side = rng.integers(0, 4, (n, cap))
        near = rng.uniform(0.0, R + 1.0, (n, cap))
        X = np.where(e & (side == 0), near, X)
        X = np.where(e & (side == 1), W - near, X)
        Y = np.where(e & (side == 2), near, Y)
        Y = np.where(e & (side == 3), H - near, Y)
    if dup > 0:
        # a later spot on the pixel of an earlier one (other sub-pixel offset)
        for i in range(n):
            for j in range(1, int(cnt[i])):
                if rng.random() < dup:
                    k = int(rng.integers(0, j))
                    X[i, j] = np.floor(X[i, k]) + rng.uniform(0.05, 0.95)
                    Y[i, j] = np.floor(Y[i, k]) + rng.uniform(0.05, 0.95)
    I = rng.lognormal(0.0, 1.5, (n, cap))
    sp = np.zeros((n, cap, 4), np.float32)
    sp[..., 0] = X - W // 2
    sp[..., 1] = Y - H // 2
    sp[..., 3] = I
    return torch.from_numpy(sp).cuda(), torch.from_numpy(cnt).cuda()


def _render_both(spots, cnt, cap, shape, sigma, normalize=True, angle=0.0, mirrored=False):
    """(splat output, band output, splat status, band status, patterns the
    last round listed for the splat kernel)."""
    import torch
    from diffsims_amd import engine
    lib, L = _lib()
    n = int(cnt.shape[0])
    H, W = shape
    p = engine.render_params(shape, sigma, 1.0, None, angle, mirrored, normalize, True)
    ref = torch.full((n, H, W), float("nan"), dtype=torch.float32, device="cuda")
    out = torch.full((n, H, W), float("nan"), dtype=torch.float32, device="cuda")
    st_ref = torch.full((n,), -1, dtype=torch.int32, device="cuda")
    st = torch.full((n,), -1, dtype=torch.int32, device="cuda")
    stream = lib.stream_handle(spots.device)
    lib.check(L.dsx_render_fast(lib.ptr(spots), lib.ptr(cnt), cap, n, ctypes.byref(p), lib.ptr(ref),
                                lib.ptr(st_ref), stream), "dsx_render_fast")
    ws = int(L.dsx_render_fast_bands_workspace_ints(n, H, W))
    work = torch.full((ws,), -7, dtype=torch.int32, device="cuda")
    lib.check(L.dsx_render_fast_bands(lib.ptr(spots), lib.ptr(cnt), cap, n, ctypes.byref(p),
                                      lib.ptr(work), ws, lib.ptr(out), lib.ptr(st), stream),
              "dsx_render_fast_bands")
    torch.cuda.synchronize()
    return ref, out, st_ref, st, int(work[0].item())


def _assert_same(ref, out, st_ref, st):
    import torch
    assert not torch.isnan(out).any()
    bad = (ref != out).flatten(1).any(1)
    assert not bool(bad.any()), f"patterns differ: {torch.nonzero(bad).flatten()[:8].tolist()}"
    assert torch.equal(st_ref, st)


def test_library_like_patterns_bit_identical():
    print("bands: 3000 x 256x256, sigma 1, ~260 spots", flush=True)
    spots, cnt = _spot_lists(3000, 400, 256, 256, 260, seed=1, edge=0.05, dup=0.02)
    ref, out, st_ref, st, listed = _render_both(spots, cnt, 400, (256, 256), 1.0)
    _assert_same(ref, out, st_ref, st)
    assert listed < 300, listed  # the band path renders most patterns itself


@pytest.mark.parametrize("sigma", [0.3, 0.6, 1.0, 1.4, 2.0])
@pytest.mark.parametrize("normalize", [True, False])
def test_tap_radii_partial_bands_and_edges(sigma, normalize):
    R = int(4 * sigma + 0.5)
    print(f"bands: 400 x 144x144, sigma {sigma} (R={R}), normalize {normalize}", flush=True)
    spots, cnt = _spot_lists(400, 256, 144, 144, 120, seed=10 + R, edge=0.2, dup=0.05, R=R)
    ref, out, st_ref, st, listed = _render_both(spots, cnt, 256, (144, 144), sigma, normalize)
    _assert_same(ref, out, st_ref, st)
    assert listed < 400


def test_in_plane_angle_and_mirror():
    print("bands: 500 x 256x192, angle 23, mirrored", flush=True)
    spots, cnt = _spot_lists(500, 320, 256, 192, 200, seed=3, edge=0.05, dup=0.03)
    for angle, mirrored in ((23.0, False), (23.0, True), (0.0, True)):
        ref, out, st_ref, st, _ = _render_both(spots, cnt, 320, (256, 192), 1.0, angle=angle,
                                               mirrored=mirrored)
        _assert_same(ref, out, st_ref, st)


def test_large_patterns_and_long_lists():
    # lists above the plan's 512 spots go to the splat kernel; the rest stay
    print("bands: 300 x 512x512, ~480 spots, cap 700", flush=True)
    spots, cnt = _spot_lists(300, 700, 512, 512, 480, seed=4, edge=0.02, dup=0.01)
    ref, out, st_ref, st, listed = _render_both(spots, cnt, 700, (512, 512), 1.0)
    _assert_same(ref, out, st_ref, st)
    n_long = int((cnt > 512).sum().item())
    assert n_long > 0 and listed >= n_long


def test_degenerate_lists():
    import torch
    print("bands: empty, out-of-frame, zero-intensity and single-spot lists", flush=True)
    spots, cnt = _spot_lists(64, 32, 128, 128, 20, seed=5)
    cnt[0:8] = 0                          # no spot
    spots[8:16, :, 0] += 1000.0           # every spot out of frame
    spots[16:24, :, 3] = 0.0              # only zero intensities (maximum 0)
    cnt[24:32] = 1                        # one spot
    spots[32:40, :, 3] = 2.5              # equal intensities
    ref, out, st_ref, st, _ = _render_both(spots, cnt, 32, (128, 128), 1.0)
    _assert_same(ref, out, st_ref, st)
    assert torch.equal(out[0:16], torch.zeros_like(out[0:16]))


@pytest.mark.parametrize("shape", [(100, 132), (250, 36), (17, 1020)])
def test_partial_tiles_and_counts_above_capacity(shape):
    # sides that are not multiples of the 16-pixel tile (partial tiles in the
    # bounds and in the candidate evaluation), and counts above the list
    # capacity (only the first cap spots exist)
    import torch
    H, W = shape
    print(f"bands: 300 x {H}x{W}, partial tiles", flush=True)
    spots, cnt = _spot_lists(300, 96, H, W, 60, seed=20 + W, edge=0.2, dup=0.05)
    cnt[::7] = 96 + 40
    ref, out, st_ref, st, listed = _render_both(spots, cnt, 96, shape, 1.0)
    _assert_same(ref, out, st_ref, st)
    assert listed < 300


def test_dense_rows_read_the_row_sorted_list():
    # most spots in a 12-row stripe: bands with more spots than their slot
    # holds take the band's window of the row-sorted list instead
    print("bands: 200 x 256x256, 400 spots, most in 12 rows", flush=True)
    spots, cnt = _spot_lists(200, 400, 256, 256, 380, seed=12, dup=0.02)
    rng = np.random.default_rng(13)
    stripe = rng.random((200, 400)) < 0.8
    y = rng.uniform(120.0, 132.0, (200, 400)).astype(np.float32) - 128.0
    import torch
    spots[:, :, 1] = torch.where(torch.from_numpy(stripe).cuda(), torch.from_numpy(y).cuda(),
                                 spots[:, :, 1])
    ref, out, st_ref, st, listed = _render_both(spots, cnt, 400, (256, 256), 1.0)
    _assert_same(ref, out, st_ref, st)
    assert listed < 200


def test_rounds_of_patterns():
    # five plan/writer rounds of at most 16,384 patterns (the last partial),
    # each reusing the workspace after the previous round's bands are written
    print("bands: 70000 x 32x32", flush=True)
    spots, cnt = _spot_lists(70000, 8, 32, 32, 4, seed=6, dup=0.05)
    ref, out, st_ref, st, _ = _render_both(spots, cnt, 8, (32, 32), 1.0)
    _assert_same(ref, out, st_ref, st)


@pytest.mark.parametrize("shape,sigma", [((128, 128), 3.0), ((128, 130), 1.0)])
def test_shapes_outside_the_band_path(shape, sigma):
    # tap radius 12: the splat kernel alone; a width that is not a multiple of 4
    print(f"bands: 50 x {shape}, sigma {sigma}", flush=True)
    spots, cnt = _spot_lists(50, 64, shape[0], shape[1], 40, seed=7)
    ref, out, st_ref, st, _ = _render_both(spots, cnt, 64, shape, sigma)
    _assert_same(ref, out, st_ref, st)


@pytest.mark.parametrize("shape,sigma", [((37, 33), 0.3), ((61, 101), 1.25), ((231, 201), 1.7),
                                         ((19, 1021), 2.0), ((300, 1023), 1.0), ((64, 513), 1.0)])
@pytest.mark.parametrize("offset", [0, 1])
def test_odd_widths_and_unaligned_output(shape, sigma, offset):
    # rows that are not whole 16-byte vectors, and an output that starts
    # between two of them: every pixel of the output and nothing beside it
    import torch
    from diffsims_amd import engine
    H, W = shape
    n, R = 41, int(4 * sigma + 0.5)
    print(f"bands: {n} x {H}x{W}, sigma {sigma}, output offset {offset}", flush=True)
    spots, cnt = _spot_lists(n, 96, H, W, 60, seed=W, edge=0.2, dup=0.05, R=R)
    ref, out, st_ref, st, _ = _render_both(spots, cnt, 96, shape, sigma)
    _assert_same(ref, out, st_ref, st)
    lib, L = _lib()
    p = engine.render_params(shape, sigma, 1.0)
    buf = torch.full((n * H * W + 8,), -3.0, dtype=torch.float32, device="cuda")
    view = buf[offset:offset + n * H * W]
    ws = int(L.dsx_render_fast_bands_workspace_ints(n, H, W))
    work = torch.empty(ws, dtype=torch.int32, device="cuda")
    lib.check(L.dsx_render_fast_bands(lib.ptr(spots), lib.ptr(cnt), 96, n, ctypes.byref(p),
                                      lib.ptr(work), ws, lib.ptr(view), lib.ptr(st),
                                      lib.stream_handle(spots.device)), "dsx_render_fast_bands")
    assert torch.equal(view.view(n, H, W), ref)
    assert bool((buf[:offset] == -3.0).all()) and bool((buf[offset + n * H * W:] == -3.0).all())


def test_odd_width_without_workspace():
    # such widths need no workspace (the splat kernel alone renders them then)
    import torch
    from diffsims_amd import engine
    lib, L = _lib()
    spots, cnt = _spot_lists(20, 64, 60, 61, 40, seed=9)
    p = engine.render_params((60, 61), 1.0, 1.0)
    ref, _, _, st, _ = _render_both(spots, cnt, 64, (60, 61), 1.0)
    out = torch.full_like(ref, float("nan"))
    lib.check(L.dsx_render_fast_bands(lib.ptr(spots), lib.ptr(cnt), 64, 20, ctypes.byref(p), None,
                                      0, lib.ptr(out), lib.ptr(st),
                                      lib.stream_handle(spots.device)), "dsx_render_fast_bands")
    assert torch.equal(out, ref)


def test_workspace_query_and_rejection():
    import torch
    lib, L = _lib()
    from diffsims_amd import engine
    assert L.dsx_render_fast_bands_workspace_ints(-1, 8, 8) == -1
    assert L.dsx_render_fast_bands_workspace_ints(10, 256, 256) > 0
    spots, cnt = _spot_lists(4, 8, 64, 64, 4, seed=8)
    p = engine.render_params((64, 64), 1.0, 1.0)
    out = torch.empty((4, 64, 64), dtype=torch.float32, device="cuda")
    work = torch.empty(16, dtype=torch.int32, device="cuda")
    rc = L.dsx_render_fast_bands(lib.ptr(spots), lib.ptr(cnt), 8, 4, ctypes.byref(p), lib.ptr(work),
                                 16, lib.ptr(out), None, lib.stream_handle(spots.device))
    assert rc == lib.DSX_EINVAL
    assert b"workspace" in L.dsx_last_error()


def test_render_spots_same_bits_across_the_small_batch_threshold():
    # render_spots takes the splat kernel alone below 768 patterns and the
    # band renderer above: a batch and its leading part give the same pixels
    import torch
    from diffsims_amd import engine
    print("render_spots: 800 and 700 x 256x256 across the dispatch threshold", flush=True)
    spots, cnt = _spot_lists(800, 400, 256, 256, 260, seed=30, edge=0.05, dup=0.02)
    assert engine.fast_renderer(800, 256, 256) == "dsx_render_fast_bands"
    assert engine.fast_renderer(700, 256, 256) == "dsx_render_fast"
    big = engine.render_spots(spots, cnt, 400, (256, 256), 1.0, 1.0)
    small = engine.render_spots(spots[:700].contiguous(), cnt[:700].contiguous(), 400, (256, 256),
                                1.0, 1.0)
    torch.cuda.synchronize()
    assert torch.equal(big[:700], small)


# -- long lists (dsx_render_fast_long) ------------------------------------------


def _render_long(spots, cnt, cap, shape, sigma, normalize=True):
    import torch
    out = _render_long_any(spots, cnt, cap, shape, sigma, normalize)
    assert not torch.isnan(out).any()
    return out


def _render_long_any(spots, cnt, cap, shape, sigma, normalize=True):
    import torch
    from diffsims_amd import engine
    lib, L = _lib()
    n = int(cnt.shape[0])
    H, W = shape
    p = engine.render_params(shape, sigma, 1.0, normalize=normalize)
    assert L.dsx_render_fast_long_fits(cap, p.radius, H, W) == 1
    out = torch.full((n, H, W), float("nan"), dtype=torch.float32, device="cuda")
    st = torch.full((n,), -1, dtype=torch.int32, device="cuda")
    ws = int(L.dsx_render_fast_long_workspace_ints(cap, n, H, W))
    work = torch.empty(ws, dtype=torch.int32, device="cuda")
    lib.check(L.dsx_render_fast_long(lib.ptr(spots), lib.ptr(cnt), cap, n, ctypes.byref(p),
                                     lib.ptr(work), ws, lib.ptr(out), lib.ptr(st),
                                     lib.stream_handle(spots.device)), "dsx_render_fast_long")
    assert not st.any()
    return out


def _fp64_patterns(spots, cnt, shape, sigma, normalize, which):
    """scipy's filter of the last-write-wins image, FP64, patterns ``which``."""
    from scipy.ndimage import gaussian_filter
    H, W = shape
    sp, c = spots.cpu().numpy(), np.minimum(cnt.cpu().numpy(), spots.shape[1])
    out = []
    for i in which:
        img = np.zeros(shape)
        X = sp[i, :c[i], 0] + np.float32(W // 2)
        Y = sp[i, :c[i], 1] + np.float32(H // 2)
        for x, y, v in zip(X, Y, sp[i, :c[i], 3]):
            if 0 <= x < W and 0 <= y < H:
                img[int(y), int(x)] = v
        img = gaussian_filter(img, sigma)
        out.append(img / img.max() if normalize and img.max() > 0 else img)
    return np.stack(out)


# A term has four roundings of 2^-24 (two products, two taps), the output two
# more, and every term half a unit of U / 2.04e9: with at most ~60 spots in a
# pixel's reach and U below 60 maxima 60 * 60 / 2 / 2.04e9 = 9e-7.
LONG_TOL = 6 * 2.0 ** -24 + 9e-7


@pytest.mark.parametrize("shape,sigma,cap,mean", [
    ((129, 128), 1.0, 1100, 1000), ((256, 256), 1.0, 3000, 2300), ((251, 203), 2.0, 2500, 2300),
    ((512, 512), 0.3, 9000, 8000), ((300, 147), 1.25, 1500, 1400), ((256, 256), 1.0, 14000, 12000)])
@pytest.mark.parametrize("normalize", [True, False])
def test_long_lists_against_fp64(shape, sigma, cap, mean, normalize):
    n, R = 9, int(4 * sigma + 0.5)
    print(f"long lists: {n} x {shape}, sigma {sigma}, {mean} spots", flush=True)
    spots, cnt = _spot_lists(n, cap, shape[0], shape[1], mean, seed=mean, edge=0.1, R=R)
    cnt[3] = cap + 50  # more than the list holds
    # later spots on the pixels of earlier ones
    spots[:, cap // 2:cap // 2 + 40, :2] = spots[:, 10:50, :2]
    out = _render_long(spots, cnt, cap, shape, sigma, normalize).cpu().numpy()
    which = [0, 3, n - 1]
    ref = _fp64_patterns(spots, cnt, shape, sigma, normalize, which)
    for o, r in zip(out[which], ref):
        assert np.abs(o - r).max() <= LONG_TOL * r.max()


def test_long_lists_degenerate_and_several_rounds():
    import torch
    print("long lists: 300 x 130x131 in two rounds, empty and zero lists", flush=True)
    cap, shape = 14000, (130, 131)
    spots, cnt = _spot_lists(300, cap, *shape, 30, seed=3)
    cnt[0:4] = 0
    spots[4:8, :, 0] += 1000.0   # out of frame
    spots[8:12, :, 3] = 0.0      # maximum 0
    cnt[12:16] = 1
    spots[16:20, :, 3] = 2.5     # equal intensities
    out = _render_long(spots, cnt, cap, shape, 1.0)
    assert torch.equal(out[:12], torch.zeros_like(out[:12]))
    which = [12, 16, 255, 256, 299]
    ref = _fp64_patterns(spots, cnt, shape, 1.0, True, which)
    assert np.abs(out[which].cpu().numpy() - ref).max() <= LONG_TOL


def test_long_lists_dispatch_and_limits():
    import torch
    from diffsims_amd import engine
    lib, L = _lib()
    fits = L.dsx_render_fast_long_fits
    assert fits(2000, 4, 256, 256) and not fits(17000, 4, 256, 256)
    assert not fits(2000, 0, 256, 256) and not fits(2000, 9, 256, 256)
    assert not fits(2000, 4, 1025, 64) and not fits(2000, 4, 256, 4)
    assert engine.long_renderer(2000, 256, 256, 4)
    assert not engine.long_renderer(2000, 128, 128, 4)   # the dense renderers
    assert not engine.long_renderer(30000, 256, 256, 4)  # dsx_render_fast_large
    # dense lists stay with it: a spot per 4.5 pixels, per 5 of small patterns
    assert engine.long_renderer(7288, 200, 164, 4) and not engine.long_renderer(7289, 200, 164, 4)
    assert engine.long_renderer(3302, 129, 128, 8) and not engine.long_renderer(3303, 129, 128, 8)
    # render_spots on both sides of the lists it takes: the same pixels
    spots, cnt = _spot_lists(6, 1500, 200, 160, 1400, seed=2)
    a = engine.render_spots(spots, cnt, 1500, (200, 160), 1.0, 1.0)
    wide = torch.zeros((6, 16500, 4), dtype=torch.float32, device="cuda")
    wide[:, :1500] = spots
    b = engine.render_spots(wide, cnt, 16500, (200, 160), 1.0, 1.0)
    assert float((a - b).abs().max()) <= 2 * LONG_TOL
    p = engine.render_params((256, 256), 1.0, 1.0)
    work = torch.empty(64, dtype=torch.int32, device="cuda")
    out = torch.empty((6, 256, 256), dtype=torch.float32, device="cuda")
    for c, ws in ((1500, 64), (16500, 64)):
        rc = L.dsx_render_fast_long(lib.ptr(wide), lib.ptr(cnt), c, 6, ctypes.byref(p),
                                    lib.ptr(work), ws, lib.ptr(out), None,
                                    lib.stream_handle(spots.device))
        assert rc == lib.DSX_EINVAL


def _render_windowed(spots, cnt, cap, shape, sigma, normalize):
    """dsx_render_fast_large: the spot image filtered in FP32."""
    import torch
    from diffsims_amd import engine
    lib, L = _lib()
    n = int(cnt.shape[0])
    p = engine.render_params(shape, sigma, 1.0, normalize=normalize)
    out = torch.full((n, *shape), float("inf"), dtype=torch.float32, device="cuda")
    ws = int(L.dsx_render_fast_large_workspace_ints(cap))
    work = torch.empty(ws, dtype=torch.int32, device="cuda")
    lib.check(L.dsx_render_fast_large(lib.ptr(spots), lib.ptr(cnt), cap, n, ctypes.byref(p),
                                      lib.ptr(work), ws, lib.ptr(out), None,
                                      lib.stream_handle(spots.device)), "dsx_render_fast_large")
    return out


@pytest.mark.parametrize("shape,sigma", [((256, 256), 1.0), ((231, 201), 1.75)])
@pytest.mark.parametrize("normalize", [True, False])
def test_long_lists_of_intensities_beyond_fixed_point(shape, sigma, normalize):
    """NaN, infinities, negative and very small or large intensities: NaN and
    infinities where the FP32 filter has them, every other pixel within its
    tolerance of the largest (LONG_TOL, and the filter's own 2 R + 1 roundings
    along both axes)."""
    import torch
    print(f"long lists beyond fixed point: {shape}, sigma {sigma}, normalize {normalize}", flush=True)
    n, cap = 12, 1400
    spots, cnt = _spot_lists(n, cap, *shape, 1300, seed=21, edge=0.1, R=7)
    inf, nan = float("inf"), float("nan")
    spots[0, 5, 3] = nan
    spots[1, 7, 3] = inf
    spots[2, 9, 3] = -inf
    spots[3, 11, 3], spots[3, 12, 3] = nan, inf
    spots[4, 3, 3] = nan                      # under a later spot: not seen
    spots[4, 900, :2] = spots[4, 3, :2]
    spots[5, :, 3] = nan
    spots[6, ::3, 3] *= -1.0
    spots[7, :, 3] *= -1.0                    # no positive pixel: not normalised
    spots[8, :, 3] *= 1e-31
    spots[9, :, 3] *= 1e34
    spots[10, 0:2, :2] = torch.tensor([[-shape[1] // 2 + 1.5, 0.0], [0.0, -shape[0] // 2 + 0.5]])
    spots[10, 0:2, 3] = torch.tensor([nan, inf])   # reflected at the edges
    cnt[11] = 2
    spots[11, 0:2, 3] = torch.tensor([nan, 1.0])
    got = _render_long_any(spots, cnt, cap, shape, sigma, normalize)
    ref = _render_windowed(spots, cnt, cap, shape, sigma, normalize)
    for i in range(n):
        a, r = got[i], ref[i]
        assert torch.equal(torch.isnan(a), torch.isnan(r)), i
        assert torch.equal(torch.isinf(a), torch.isinf(r)), i
        ok = torch.isfinite(r)
        assert torch.equal(a[~ok].sign().nan_to_num(2.0), r[~ok].sign().nan_to_num(2.0)), i
        top = float(r[ok].double().abs().max()) if ok.any() else 0.0
        tol = LONG_TOL + 2 * 15 * 2.0 ** -24
        assert float((a[ok].double() - r[ok].double()).abs().max() if ok.any() else 0.0) <= tol * top, i
    # patterns of ordinary lists do not notice their neighbours
    plain = _render_long(spots[6:8].contiguous(), cnt[6:8].contiguous(), cap, shape, sigma, normalize)
    assert torch.equal(plain, got[6:8])
    which = [4, 6]
    clean = spots.clone()
    clean[4, 3, 3] = 1.0
    for i, r in zip(which, _fp64_patterns(clean, cnt, shape, sigma, normalize, which)):
        assert np.abs(got[i].cpu().numpy() - r).max() <= LONG_TOL * np.abs(r).max()


@pytest.mark.parametrize("shape", [(96, 101), (96, 100)])
def test_short_lists_of_any_intensity_equal_the_splat_renderer(shape):
    # the same bits, NaN included, as the renderer whose calls they take over
    import torch
    print(f"bands: intensities of any kind, {shape}", flush=True)
    spots, cnt = _spot_lists(8, 96, *shape, 60, seed=4)
    inf, nan = float("inf"), float("nan")
    spots[0, 5, 3] = nan
    spots[1, 7, 3] = inf
    spots[2, :, 3] = nan
    spots[3, ::3, 3] *= -1.0
    spots[4, :, 3] *= -1.0
    spots[5, :, 3] = 0.0
    spots[6, 9, 3] = -inf
    ref, out, st_ref, st, _ = _render_both(spots, cnt, 96, shape, 1.0)
    assert torch.equal(st_ref, st)
    assert torch.equal(out.view(torch.int32), ref.view(torch.int32))


@pytest.mark.parametrize("shape", [(130, 600), (200, 255)])
@pytest.mark.parametrize("length", [63, 64, 65, 128, 700])
def test_long_lists_gathered_in_a_few_rows(shape, length):
    """Rows of `length` spots, many of them on the same pixels, either side of the
    length from which a row's pixels are mapped (64) and over several parts of the
    map (256 pixels): the latest spot of a pixel is the one that is seen, a zero
    too.  At most 9 x 1 spots reach a pixel, well inside LONG_TOL's count."""
    import torch
    print(f"long lists in rows: {shape}, {length} spots each", flush=True)
    H, W = shape
    rng = np.random.default_rng(length)
    ys = np.arange(4, H, 12)
    m = len(ys) * length
    sp = np.zeros((3, max(m, 1100), 4), np.float32)
    for i in range(3):
        order = rng.permutation(m)
        y = np.repeat(ys, length)[order]
        # the second pattern's rows take few columns, the third's lie at the end
        x = rng.integers(0, W, m) if i == 0 else rng.integers(0, 20, m) if i == 1 else rng.integers(W - 9, W, m)
        sp[i, :m, 0] = x + 0.5 - W // 2
        sp[i, :m, 1] = y + 0.5 - H // 2
        sp[i, :m, 3] = rng.lognormal(0.0, 1.5, m)
        sp[i, :m:7, 3] = 0.0
    spots = torch.from_numpy(sp).cuda()
    cnt = torch.full((3,), m, dtype=torch.int32, device="cuda")
    out = _render_long(spots, cnt, spots.shape[1], shape, 1.0).cpu().numpy()
    for o, r in zip(out, _fp64_patterns(spots, cnt, shape, 1.0, True, range(3))):
        assert np.abs(o - r).max() <= LONG_TOL


@pytest.mark.parametrize("shape,cap", [((129, 128), 3302), ((200, 164), 7288)])
def test_both_sides_of_the_density_line_give_the_same_pixels(shape, cap):
    # one list either side of the capacity from which the windowed renderer takes it
    import torch
    from diffsims_amd import engine
    print(f"long lists: {shape}, capacity {cap}", flush=True)
    spots, cnt = _spot_lists(4, cap, *shape, 1300, seed=cap)
    assert engine.long_renderer(cap, *shape, 4) and not engine.long_renderer(cap + 1, *shape, 4)
    a = engine.render_spots(spots, cnt, cap, shape, 1.0, 1.0)
    wide = torch.zeros((4, cap + 1, 4), dtype=torch.float32, device="cuda")
    wide[:, :cap] = spots
    b = engine.render_spots(wide, cnt, cap + 1, shape, 1.0, 1.0)
    assert float((a - b).abs().max()) <= 2 * LONG_TOL


@pytest.mark.parametrize("shape,sigma,cap", [
    ((101, 100), 1.75, 75), ((101, 100), 1.75, 76), ((101, 99), 2.0, 75), ((101, 99), 1.5, 76),
    ((64, 128), 1.5, 96), ((82, 100), 1.5, 96), ((300, 257), 1.75, 579), ((300, 257), 1.75, 580)])
def test_narrow_and_wide_bands_give_the_same_bits(shape, sigma, cap):
    # either side of one spot per 133 pixels and of two wide bands, from radius 6 on
    print(f"bands: {shape}, sigma {sigma}, capacity {cap}", flush=True)
    spots, cnt = _spot_lists(50, cap, *shape, 0.7 * cap, seed=cap, edge=0.2, dup=0.05, R=8)
    ref, out, st_ref, st, _ = _render_both(spots, cnt, cap, shape, sigma)
    _assert_same(ref, out, st_ref, st)
