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
