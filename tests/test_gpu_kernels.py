"""Edges of single kernels on the GPU: sizes around their tiles, transform
lengths and remainders, each against the CPU oracle or an FP64 numpy form of
the same stage, with the tolerances of the stage's own tests."""
import numpy as np
import pytest

import ctbangbang_amd as cb

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")


def dev(a):
    return torch.from_numpy(np.ascontiguousarray(a)).cuda()


def host(t):
    torch.cuda.synchronize()
    return t.cpu().numpy()


@pytest.mark.parametrize("n,rows", [(1, 1), (33, 2), (735, 3), (1535, 5), (1536, 4), (1537, 1), (2047, 3), (2048, 6)])
def test_fft_filter_spectrum_sizes(ctx, n, rows):
    """The device spectrum at the edges of both transform lengths (3072 up to
    n = 1536, 4096 up to 2048), odd lengths and row counts: tolerance of the
    FFT form, 2e-6 of the FP64 maximum."""
    import oracle
    rng = np.random.default_rng(n)
    x = rng.standard_normal((rows, n)).astype(np.float32) * 3.0 + 1.0
    taps = (rng.standard_normal(2 * n) / np.sqrt(n)).astype(np.float32)
    want = oracle.filter_fft(x, taps)
    ctx.set_options(filter_mode=cb.FILTER_FFT32, proj_dtype=cb.PROJ_F32)
    out = torch.empty(rows * n, dtype=torch.float32, device="cuda")
    taps_d, x_d = dev(taps), dev(x)
    ctx.filter_rows_dev(taps_d, n, rows, x_d, out)
    got = host(out).reshape(rows, n)
    ctx.set_options(filter_mode=cb.FILTER_F32)
    assert np.abs(got - want).max() <= 2e-6 * np.abs(want).max()


@pytest.mark.parametrize("n,rows", [(1, 3), (256, 2), (257, 1), (1279, 3), (1281, 2), (1472, 5), (1536, 1), (1537, 3),
                                    (1792, 2), (2047, 1), (2048, 3)])
def test_fft_filter_row_ends(ctx, n, rows):
    """Row ends and the last, single row of the FFT form: nothing is written past
    the result, and bfloat16 results are the rounded FP32 ones (the arithmetic
    before the store is the same)."""
    rng = np.random.default_rng(n)
    x_d = dev(rng.standard_normal(rows * n).astype(np.float32))
    taps_d = dev((rng.standard_normal(2 * n) / np.sqrt(n)).astype(np.float32))
    out = {}
    for dtype, tt in ((cb.PROJ_F32, torch.float32), (cb.PROJ_BF16, torch.bfloat16)):
        ctx.set_options(filter_mode=cb.FILTER_FFT32, proj_dtype=dtype)
        o = torch.full((rows * n + 64,), 7.0, dtype=tt, device="cuda")
        ctx.filter_rows_dev(taps_d, n, rows, x_d, o)
        torch.cuda.synchronize()
        assert (o[rows * n:] == 7.0).all()
        out[dtype] = o[:rows * n]
    ctx.set_options(filter_mode=cb.FILTER_F32, proj_dtype=cb.PROJ_F32)
    assert torch.equal(out[cb.PROJ_F32].to(torch.bfloat16), out[cb.PROJ_BF16])


@pytest.mark.parametrize("mode", [cb.FILTER_F32, cb.FILTER_BF16X3, cb.FILTER_F16X3])
@pytest.mark.parametrize("n,rows", [(4, 3), (60, 65), (64, 33000), (66, 2), (68, 64), (128, 127), (188, 130), (192, 128),
                                    (256, 129), (1472, 131), (1472, 1409), (1472, 2700), (1840, 63), (5460, 5), (5888, 2), (7040, 3), (10112, 2)])
def test_toeplitz_edges(ctx, n, rows, mode):
    """Toeplitz products at the edges of the tiles, with a guard past the last
    row.  Samples and taps are small whole numbers, so every product and sum is
    exact in each form and the result has to be equal."""
    rng = np.random.default_rng(10 * n + mode)
    x = rng.integers(-8, 9, (rows, n))
    taps = rng.integers(-8, 9, 2 * n)
    want = np.stack([np.convolve(r, taps)[n:2 * n] for r in x])
    out = torch.full((rows * n + 64,), 7.0, dtype=torch.float32, device="cuda")
    x_d, taps_d = dev(x.astype(np.float32)), dev(taps.astype(np.float32))
    ctx.set_options(filter_mode=mode, proj_dtype=cb.PROJ_F32)
    if mode == cb.FILTER_F32 and n > 7040:
        with pytest.raises(cb.CTBBError):
            ctx.filter_rows_dev(taps_d, n, rows, x_d, out)
        return
    ctx.filter_rows_dev(taps_d, n, rows, x_d, out)
    got = host(out)
    ctx.set_options(filter_mode=cb.FILTER_F32)
    np.testing.assert_array_equal(got[:rows * n].reshape(rows, n), want)
    assert (got[rows * n:] == 7.0).all()


def _mini(tmp_path, channels, nrows, ffs="none", turn=192, centre=None, **scanner):
    """Planned small scan on a scanner of `channels` channels and `turn`
    projections per turn."""
    from ctbangbang_amd import scans
    d = str(tmp_path)
    scans.mini_install(d, dict(scans.MINI_SCANNER, NChannels=channels, NProjTurn=turn,
                               CentralChannel=channels / 2 - 0.25 if centre is None else centre, **scanner))
    prm = str(tmp_path / "m.prm")
    tok = scans.mini_tokens(ffs, nrows=nrows, rotations=max(12, 96 // nrows))
    tok["Readings"] = tok["Readings"] // 192 * turn
    cb.write_prm(prm, tok)
    mr = cb.metadata_from_prm(prm, install_dir=d)
    cb.plan_block(mr, 0)
    return mr


@pytest.mark.parametrize("channels,nrows", [(4, 1), (60, 6), (64, 8), (68, 9), (132, 17)])
def test_adaptive_smoothing_edges(ctx, tmp_path, channels, nrows):
    """5x5x5 smoothing bit for bit at the edges of the 64-channel x 8-row wave
    tile, in the first and last views, and around infinite and NaN samples."""
    import oracle
    mr = _mini(tmp_path, channels, nrows)
    n = int(mr.ri.n_proj_pull)
    rng = np.random.default_rng(channels + nrows)
    raw = rng.random((n, nrows, channels)).astype(np.float32)
    raw[n // 2, nrows // 2, channels // 2] = np.inf
    raw[n // 2 + 9, 0, channels - 1] = np.nan
    T = np.float32(0.6)
    raw_d = dev(raw.ravel())
    out = torch.empty_like(raw_d)
    ctx.set_options(adaptive_threshold=float(T))
    ctx.adaptive_filter_dev(mr, raw_d, out)
    ctx.synchronize()
    ctx.set_options(adaptive_threshold=0.0)
    want = oracle.adaptive_apply(mr, raw.reshape(n, -1), np.full(n, T, dtype=np.float32))
    assert np.count_nonzero(want != raw.reshape(n, -1)) > 0.2 * raw.size
    assert np.array_equal(host(out).reshape(n, -1), want, equal_nan=True)
    cb.free_metadata(mr)


@pytest.mark.parametrize("ffs,channels,nrows,centre,reverse", [
    ("none", 28, 1, None, 0), ("none", 33, 3, 20.0, 0), ("phi", 66, 2, None, 0), ("z", 97, 4, 30.0, 1),
    ("both", 129, 4, None, 1), ("both", 130, 6, 100.0, 0)])
def test_rebin_edges(ctx, tmp_path, ffs, channels, nrows, centre, reverse):
    """Rebinning where a row ends inside a wave or a workgroup, with a number
    of views that is no multiple of a thread's, swapped row interleave, and a
    detector so far off centre that readings before and after the pull are
    clamped.  Tolerance: the stage's 2e-5 of the largest raw sample, and the
    azimuthal index's FP32 rounding (half a unit in the last place of the
    number of readings, for each of the two taps) times the largest step
    between two readings (1)."""
    import oracle
    mr = _mini(tmp_path, channels, nrows, ffs, turn=190, centre=centre, ReverseRowInterleave=reverse)
    s = cb.block_sizes(mr)
    rng = np.random.default_rng(channels)
    raw = rng.random(s.raw_pull).astype(np.float32)
    out = torch.empty(s.rebin, dtype=torch.float32, device="cuda")
    raw_d = dev(raw)
    ctx.rebin_dev(mr, raw_d, out)
    ctx.synchronize()
    want = oracle.rebin(mr, raw, double=True)
    got = host(out).reshape(want.shape)
    assert np.abs(got - want).max() <= 2e-5 + np.spacing(np.float32(mr.ri.n_proj_pull // mr.ri.n_ffs))
    cb.free_metadata(mr)


@pytest.mark.parametrize("ffs,channels,nrows,turn", [("none", 66, 1, 440), ("none", 66, 1, 800), ("z", 97, 2, 460),
                                                     ("phi", 66, 2, 460), ("both", 130, 4, 440), ("both", 130, 4, 480)])
def test_rebin_readings_per_wave(ctx, tmp_path, ffs, channels, nrows, turn):
    """Rebinning where the 64 channels of a wave lie just within, on both sides
    of and beyond the 16 readings up to which it keeps them in LDS.  Tolerance as
    in test_rebin_edges."""
    import oracle
    mr = _mini(tmp_path, channels, nrows, ffs, turn=turn)
    s = cb.block_sizes(mr)
    rng = np.random.default_rng(turn)
    raw = rng.random(s.raw_pull).astype(np.float32)
    out = torch.empty(s.rebin, dtype=torch.float32, device="cuda")
    raw_d = dev(raw)
    ctx.rebin_dev(mr, raw_d, out)
    ctx.synchronize()
    want = oracle.rebin(mr, raw, double=True)
    got = host(out).reshape(want.shape)
    assert np.abs(got - want).max() <= 2e-5 + np.spacing(np.float32(mr.ri.n_proj_pull // mr.ri.n_ffs))
    cb.free_metadata(mr)


@pytest.mark.parametrize("turn", [126, 2040, 2052, 5626, 5636])
def test_adaptive_threshold_windows(ctx, tmp_path, turn):
    """Per-view threshold bit for bit around the window sizes that change the
    bisection's form (1024 and 2816 values) and for a window that does not
    fill one wave, with view maxima that vary over the turn; out of place on
    16-byte aligned buffers and on buffers one sample off."""
    import oracle
    mr = _mini(tmp_path, 4, 16, turn=turn)
    n = int(mr.ri.n_proj_pull)
    rng = np.random.default_rng(turn)
    size = 1.0 + 0.8 * np.sin(np.arange(n) * (4 * np.pi / turn))
    raw = (rng.random((n, 64)) * size[:, None]).astype(np.float32)
    want, thr = oracle.adaptive_filter(mr, raw)
    assert 0 < np.count_nonzero(want != raw) and np.unique(thr).size > 16
    for off in (0, 1):
        buf = dev(np.concatenate([np.zeros(off, np.float32), raw.ravel()]))
        out = torch.zeros(raw.size + off, dtype=torch.float32, device="cuda")
        torch.cuda.synchronize()
        ctx.adaptive_filter_dev(mr, buf[off:], out[off:])
        ctx.synchronize()
        assert np.array_equal(host(out)[off:].reshape(n, 64), want.reshape(n, 64)), off
    cb.free_metadata(mr)


@pytest.mark.parametrize("nx,ny", [(16, 16), (48, 32), (128, 80), (272, 256)])
def test_backproject_parts(ctx, tmp_path, nx, ny):
    """A block whose angles are summed in parts (few tiles for the device),
    against the FP64 oracle on sampled columns with the random-sinogram
    tolerance (2e-4 of the maximum, a voxel at the |q| = 1 step excepted), and
    bit for bit against the entry point that never splits a tile."""
    import oracle
    from ctbangbang_amd import scans
    d = str(tmp_path)
    scans.mini_install(d)
    tok = scans.mini_tokens("none", nrows=8)
    tok.update(Nx=nx, Ny=ny, AcqFOV=240.0)
    prm = str(tmp_path / "p.prm")
    cb.write_prm(prm, tok)
    mr = cb.metadata_from_prm(prm, install_dir=d)
    cb.plan_block(mr, 0)
    s = cb.block_sizes(mr)
    reb = np.random.default_rng(nx).random(s.rebin).astype(np.float32)
    reb_d = dev(reb)
    img = [torch.full((s.image_block,), np.nan, dtype=torch.float32, device="cuda") for _ in range(3)]
    torch.cuda.synchronize()
    ctx.set_options(proj_dtype=cb.PROJ_F32, bp_tile=0)
    ctx.backproject_dev(mr, reb_d, img[0])
    ctx.backproject_dev_noalloc(mr, reb_d, img[1])
    ctx.set_options(bp_tile=32)
    ctx.backproject_dev(mr, reb_d, img[2])
    ctx.set_options(bp_tile=0)
    ctx.synchronize()
    got = host(img[0]).reshape(32, nx, ny)
    assert np.array_equal(got, host(img[1]).reshape(got.shape))
    rng = np.random.default_rng(1)
    cx, cy = rng.integers(0, nx, 64), rng.integers(0, ny, 64)
    want = oracle.backproject(mr, reb, oracle.BP_GPU, cols=(cx, cy))[:, cx, cy]
    for g in (got, host(img[2]).reshape(got.shape)):
        err = np.abs(g[:, cx, cy] - want)
        assert np.count_nonzero(err > 2e-4 * np.abs(want).max()) <= 1e-3 * err.size
    cb.free_metadata(mr)


@pytest.mark.parametrize("nx,ny,thickness,offset", [(32, 32, 2.4, 0), (16, 20, 0.7, 0), (15, 7, 9.6, 0), (32, 16, 8.4, 1),
                                                    (48, 32, 19.2, 0)])
def test_finalize_edges(ctx, tmp_path, nx, ny, thickness, offset):
    """Thickening bit for bit with tap lists of one to more than two batches,
    slice sizes that are no multiple of four and a stack one sample off
    16-byte alignment, in both table directions."""
    import oracle
    from ctbangbang_amd import scans
    scans.mini_install(str(tmp_path))
    for table_dir in ("out", "in"):
        tok = scans.mini_tokens("none", nrows=8, rotations=30, table_dir=table_dir)
        tok.update(Nx=nx, Ny=ny, SliceThickness=thickness, NSlices=3, EndPos=tok["StartPos"] + 2 * thickness)
        prm = str(tmp_path / "f.prm")
        cb.write_prm(prm, tok)
        mr = cb.metadata_from_prm(prm, install_dir=str(tmp_path))
        s = cb.block_sizes(mr)
        img = np.random.default_rng(nx + ny).random(s.image_stack).astype(np.float32) * 0.04
        for mu in (0.0, 0.02):
            ctx.set_options(mu_water=mu)
            buf = dev(np.concatenate([np.zeros(offset, np.float32), img]))
            out = torch.empty(s.final_stack + offset, dtype=torch.float32, device="cuda")
            ctx.finalize_dev(mr, buf[offset:], out[offset:])
            ctx.synchronize()
            got = host(out)[offset:].reshape(-1, nx, ny)
            assert np.array_equal(got, oracle.finalize(mr, img, mu, double=False))
        cb.free_metadata(mr)
    ctx.set_options(mu_water=0.0)


def test_backproject_sixteen_parts(ctx, tmp_path):
    """The most parts a block's angles are summed in, against the form that never
    splits a tile bit for bit and against the oracle (tolerance of
    test_backproject_parts)."""
    import ctypes as C

    import oracle
    from ctbangbang_amd import scans
    d = str(tmp_path)
    scans.mini_install(d, dict(scans.MINI_SCANNER, NProjTurn=1152))
    nx, ny = 64, 128
    tok = scans.mini_tokens("none", nrows=8)
    tok.update(Nx=nx, Ny=ny, AcqFOV=240.0, Readings=tok["Readings"] * 6)
    prm = str(tmp_path / "p.prm")
    cb.write_prm(prm, tok)
    mr = cb.metadata_from_prm(prm, install_dir=d)
    cb.plan_block(mr, 0)
    s = cb.block_sizes(mr)
    rule = cb.lib()._ZN4ctbb17backproject_partsEiii
    rule.restype, rule.argtypes = C.c_int, [C.c_int] * 3
    cus = torch.cuda.get_device_properties(0).multi_processor_count
    assert rule(nx * ny // 256, int(mr.cg.n_proj_turn) // 2, cus) == 16
    reb = np.random.default_rng(nx).random(s.rebin).astype(np.float32)
    reb_d = dev(reb)
    img = [torch.full((s.image_block,), np.nan, dtype=torch.float32, device="cuda") for _ in range(2)]
    torch.cuda.synchronize()
    ctx.set_options(proj_dtype=cb.PROJ_F32, bp_tile=0)
    ctx.backproject_dev(mr, reb_d, img[0])
    ctx.backproject_dev_noalloc(mr, reb_d, img[1])
    ctx.synchronize()
    got = host(img[0]).reshape(32, nx, ny)
    assert np.array_equal(got, host(img[1]).reshape(got.shape))
    rng = np.random.default_rng(1)
    cx, cy = rng.integers(0, nx, 64), rng.integers(0, ny, 64)
    want = oracle.backproject(mr, reb, oracle.BP_GPU, cols=(cx, cy))[:, cx, cy]
    err = np.abs(got[:, cx, cy] - want)
    assert np.count_nonzero(err > 2e-4 * np.abs(want).max()) <= 1e-3 * err.size
    cb.free_metadata(mr)


@pytest.mark.parametrize("mode", [cb.FILTER_F32, cb.FILTER_BF16X3, cb.FILTER_F16X3])
@pytest.mark.parametrize("n", [4, 36, 66, 100, 128, 1840])
def test_toeplitz_first_tap_unused(ctx, n, mode):
    """No sample of the result contains taps[0] (n + l - k is at least 1): its
    value, infinite or NaN, does not reach the rows.  Whole numbers, exact."""
    rng = np.random.default_rng(n)
    rows = 3
    x = rng.integers(-8, 9, (rows, n))
    taps = rng.integers(-8, 9, 2 * n).astype(np.float32)
    want = np.stack([np.convolve(r, taps)[n:2 * n] for r in x])
    ctx.set_options(filter_mode=mode, proj_dtype=cb.PROJ_F32)
    x_d = dev(x.astype(np.float32))
    for first in (np.nan, np.inf):
        taps[0] = first
        taps_d = dev(taps)
        out = torch.empty(rows * n, dtype=torch.float32, device="cuda")
        torch.cuda.synchronize()
        ctx.filter_rows_dev(taps_d, n, rows, x_d, out)
        ctx.synchronize()
        got = host(out).reshape(rows, n)
        np.testing.assert_array_equal(got, want)
    ctx.set_options(filter_mode=cb.FILTER_F32)


@pytest.mark.parametrize("n_ffs", [20460, 20480, 40960, 330000])
def test_adaptive_long_smoothing_windows(ctx, tmp_path, n_ffs):
    """Per-view threshold bit for bit with 18-degree windows around one and two
    parts of a view's sum (1023, 1025 and 2049 maxima; odd numbers only) and of
    many (16501), which no 64 KB of LDS hold."""
    import oracle
    mr = _mini(tmp_path, 4, 16, turn=2040)
    n = int(mr.ri.n_proj_pull)
    mr.cg.n_proj_ffs = n_ffs
    rng = np.random.default_rng(n_ffs)
    size = 1.0 + 0.8 * np.sin(np.arange(n) * (4 * np.pi / 2040))
    raw = (rng.random((n, 64)) * size[:, None]).astype(np.float32)
    want, _ = oracle.adaptive_filter(mr, raw)
    raw_d = dev(raw.ravel())
    out = torch.zeros_like(raw_d)
    torch.cuda.synchronize()
    ctx.adaptive_filter_dev(mr, raw_d, out)
    ctx.synchronize()
    assert np.array_equal(host(out).reshape(n, 64), want.reshape(n, 64))
    cb.free_metadata(mr)


@pytest.mark.parametrize("ffs", ["none", "z", "phi", "both"])
def test_rebin_channels_beyond_the_fan(ctx, tmp_path, ffs):
    """A fan so wide that the outermost parallel channels are parallel to no ray
    (an arcsine beyond 1, NaN coordinates): they clamp to the first reading and
    channel, whole numbers here, and are not taken for non-finite samples."""
    mr = _mini(tmp_path, 300, 4, ffs, turn=1000)
    s = cb.block_sizes(mr)
    raw = np.random.default_rng(3).integers(1, 99, s.raw_pull).astype(np.float32)
    out = torch.full((s.rebin,), np.nan, dtype=torch.float32, device="cuda")
    raw_d = dev(raw)
    torch.cuda.synchronize()
    ctx.rebin_dev(mr, raw_d, out)
    ctx.synchronize()
    got = host(out).reshape(s.n_proj_out, mr.cg.n_rows, mr.cg.n_channels_oversampled)
    assert np.isfinite(got).all()
    sine = (np.arange(600) - 2.0 * mr.cg.central_channel) * (mr.cg.fan_angle_increment / 2)
    beyond = np.flatnonzero(np.abs(sine) > 1.01)
    assert beyond.size > 0
    if ffs in ("none", "z"):
        pull = raw.reshape(-1, mr.cg.n_rows_raw, mr.cg.n_channels)
        for r in range(int(mr.cg.n_rows)):
            spot, row = (r & 1, r >> 1) if ffs == "z" else (0, r)
            assert (got[:, r, beyond] == pull[spot, row, 0]).all()
    cb.free_metadata(mr)


@pytest.mark.parametrize("channels,nrows", [(4, 1), (68, 1), (128, 2), (130, 2), (60, 3), (68, 4), (64, 5)])
@pytest.mark.parametrize("share", [0.002, 0.5])
def test_adaptive_few_rows(ctx, tmp_path, channels, nrows, share):
    """5x5x5 smoothing bit for bit where a wave takes several views of few rows,
    numbers of views and channels that leave some of it over, with few and many
    samples above the threshold, in the first and last views too."""
    import oracle
    mr = _mini(tmp_path, channels, nrows, turn=190)
    n = int(mr.ri.n_proj_pull) // int(mr.ri.n_ffs)
    n -= 1 - n % 2                              # an odd number of views
    mr.ri.n_proj_pull = n
    rng = np.random.default_rng(channels + nrows)
    raw = rng.random((n, nrows, channels)).astype(np.float32)
    raw[[0, n - 1], nrows - 1, channels - 1] = 2.0
    T = np.float32(1.0 - share)
    raw_d = dev(raw.ravel())
    out = torch.full_like(raw_d, float("nan"))
    torch.cuda.synchronize()
    ctx.set_options(adaptive_threshold=float(T))
    ctx.adaptive_filter_dev(mr, raw_d, out)
    ctx.synchronize()
    ctx.set_options(adaptive_threshold=0.0)
    want = oracle.adaptive_apply(mr, raw.reshape(n, -1), np.full(n, T, dtype=np.float32))
    assert 0 < np.count_nonzero(want != raw.reshape(n, -1)) <= 1.2 * share * raw.size
    assert np.array_equal(host(out).reshape(n, -1), want)
    cb.free_metadata(mr)
