"""Calls that follow each other on one context: what one of them leaves in the
context's workspaces must not reach the results of the next."""
import numpy as np
import pytest

import ctbangbang_amd as cb
from ctbangbang_amd import scans

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")


def host(t):
    torch.cuda.synchronize()
    return t.cpu().numpy()


def _scan(ctx, tmp_path, mini_dir, name, n_slices, thickness):
    tok = scans.mini_tokens("none", nrows=8, nx=32, rotations=24, n_slices=n_slices)
    tok.update(SliceThickness=thickness, EndPos=tok["StartPos"] + (n_slices - 1) * thickness)
    prm = str(tmp_path / name)
    cb.write_prm(prm, tok)
    mr = cb.metadata_from_prm(prm, install_dir=mini_dir)
    frame = mr.cg.n_rows_raw * mr.cg.n_channels
    raw = torch.empty(tok["Readings"] * frame, dtype=torch.float32, device="cuda")
    ctx.synth_scan_dev(mr, scans.phantom_for(tok, 5), 0, tok["Readings"], raw)
    out = torch.empty(cb.block_sizes(mr).final_stack, dtype=torch.float32, device="cuda")
    return mr, raw, tok["Readings"], out


@pytest.mark.parametrize("mode", [cb.BATCH_PERSISTENT, cb.BATCH_PIPELINE])
def test_volume_after_batch(ctx, tmp_path, mini_dir, mode):
    """A volume, a batch of scans of other thicknesses and slice numbers (other
    tap lists), the same volume again: equal images, and the same for the
    finalize stage alone."""
    ctx.set_options(mu_water=0.02, adaptive_filter=1, filter_mode=cb.FILTER_FFT32, proj_dtype=cb.PROJ_F32)
    a = _scan(ctx, tmp_path, mini_dir, "a.prm", 12, 2.4)
    b = [_scan(ctx, tmp_path, mini_dir, "b.prm", 5, 6.0), _scan(ctx, tmp_path, mini_dir, "c.prm", 30, 1.3)]
    stack = torch.rand(cb.block_sizes(a[0]).image_stack, device="cuda") * 0.04
    torch.cuda.synchronize()
    want = []
    for again in (False, True):
        for call in (lambda: ctx.reconstruct_dev(*a), lambda: ctx.finalize_dev(a[0], stack, a[3])):
            if again:
                ctx.set_options(batch_mode=mode)
                ctx.reconstruct_batch_dev(*([s[i] for s in b] for i in range(4)))
                ctx.set_options(batch_mode=cb.BATCH_PERSISTENT)
            call()
            ctx.synchronize()
            got = host(a[3]).copy()
            if again:
                assert np.array_equal(got, want.pop(0))
            else:
                want.append(got)
    assert np.abs(got).max() > 0
    for s in [a] + b:
        cb.free_metadata(s[0])
    ctx.set_options(mu_water=0.0)


def test_backproject_without_memory_for_parts(tmp_path):
    """A block whose angles are summed in parts, with less free device memory
    than its partial images take: the same image, and the calls that follow
    work."""
    tok = scans.base_tokens()
    tok.update(Scanner="definitionas.scanner", Nrows=16, CollSlicewidth=1.2, Zffs=0, Phiffs=0, PitchValue=19.2,
               Readings=12 * 1152, Nx=816, Ny=816, ReconFOV=300.0, SliceThickness=2.0, StartPos=80.0, NSlices=10,
               EndPos=98.0)
    prm = str(tmp_path / "p.prm")
    cb.write_prm(prm, tok)
    mr = cb.metadata_from_prm(prm)
    cb.plan_block(mr, 0)
    s = cb.block_sizes(mr)
    reb = torch.rand(s.rebin, device="cuda")
    img = [torch.full((s.image_block,), float("nan"), device="cuda") for _ in range(2)]
    stack = torch.rand(s.image_stack, device="cuda")
    final = torch.empty(s.final_stack, device="cuda")
    torch.cuda.synchronize()
    c = cb.Context(0)
    free = torch.cuda.mem_get_info()[0]
    c.backproject_dev(mr, reb, img[0])
    c.synchronize()
    assert free - torch.cuda.mem_get_info()[0] >= 2 * 4 * s.image_block         # the partial images of two parts or more
    c.close()
    c = cb.Context(0)
    keep, room = [], 2 * 4 * s.image_block + (64 << 20)
    try:
        chunk = 32 << 30
        while chunk >= 1 << 24 and len(keep) < 64:
            n = min(chunk, torch.cuda.mem_get_info()[0] - room)
            try:
                if n >= 1 << 24:
                    keep.append(torch.empty(n, dtype=torch.uint8, device="cuda"))
                    continue
            except torch.OutOfMemoryError:
                pass
            chunk //= 2
        assert torch.cuda.mem_get_info()[0] < 3 * 4 * s.image_block
        c.backproject_dev(mr, reb, img[1])
        c.finalize_dev(mr, stack, final)
        c.synchronize()
    finally:
        keep.clear()
        torch.cuda.empty_cache()
        c.close()
    assert np.array_equal(host(img[0]), host(img[1]))
    cb.free_metadata(mr)


def test_filter_rows_taps_dropped(ctx):
    """Taps overwritten as soon as filter_rows_dev has returned, with work on
    the context's stream ahead of it: the result is the one of the taps that
    were passed."""
    n, rows = 1472, 64
    rng = np.random.default_rng(4)
    taps = torch.from_numpy((rng.standard_normal(2 * n) / np.sqrt(n)).astype(np.float32)).cuda()
    x = torch.from_numpy(rng.standard_normal(rows * n).astype(np.float32)).cuda()
    ahead = torch.zeros(20000 * n, device="cuda")
    ahead_out = torch.empty_like(ahead)
    ahead_taps = torch.ones(2 * n, device="cuda")
    out = [torch.empty(rows * n, device="cuda") for _ in range(2)]
    torch.cuda.synchronize()
    ctx.set_options(filter_mode=cb.FILTER_FFT32, proj_dtype=cb.PROJ_F32)
    ctx.filter_rows_dev(taps, n, rows, x, out[0])
    ctx.synchronize()
    ctx.set_options(filter_mode=cb.FILTER_F32)
    for _ in range(10):
        ctx.filter_rows_dev(ahead_taps, n, 20000, ahead, ahead_out)
    ctx.set_options(filter_mode=cb.FILTER_FFT32)
    ctx.filter_rows_dev(taps, n, rows, x, out[1])
    taps.zero_()
    torch.cuda.synchronize()
    ctx.synchronize()
    ctx.set_options(filter_mode=cb.FILTER_F32)
    assert float(out[0].abs().max()) > 0
    assert torch.equal(out[0], out[1])
