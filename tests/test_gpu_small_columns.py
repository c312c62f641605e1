"""Column transforms of 2 to 30 points in registers, and record rows at every pixel remainder and address."""
import numpy as np
import pytest
import torch

import pyoracle as po
from asarf import _lib as L
from asarf import configs, focus, scene

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n1", [2, 3, 4, 5, 6, 7, 8, 9, 10, 12, 14, 15])
@pytest.mark.parametrize("cols", [1, 255, 257])
def test_short_first_pass(n1, cols, tmp_path):
    """n1 x 105 column transforms with the split forced through the tuner cache file, against numpy in FP64; an FP32
    transform of at most 1575 points stays within 2^-24 * sqrt(2 log2 n) * 4 < 1.2e-6 of it."""
    ctx = focus.Context(0)
    path = str(tmp_path / "tune.txt")
    focus.tune_save(ctx, path)
    n = n1 * 105
    with open(path, "a") as f:
        f.write(f"col {n} {n1}\n")
    focus.tune_load(ctx, path)
    x = (np.random.default_rng(n).standard_normal((n, cols, 2)) @ [1, 1j]).astype(np.complex64)
    t = torch.from_numpy(x).cuda()
    focus.fft(ctx, t, L.FFT_COLUMNS)
    ref = np.fft.fft(x.astype(np.complex128), axis=0)
    assert np.linalg.norm(t.cpu().numpy() - ref) < 1.2e-6 * np.linalg.norm(ref)
    focus.fft(ctx, t, L.FFT_COLUMNS, inverse=True, scale=1.0 / n)
    assert np.linalg.norm(t.cpu().numpy() - x) < 2.4e-6 * np.linalg.norm(x)
    ctx.close()


@pytest.mark.parametrize("n1,n2", [(n, 49) for n in (16, 18, 20, 21, 24, 25, 27, 28, 30)] +
                         [(98, n) for n in (16, 21, 25, 30)] + [(32, 35)])
def test_register_lengths_in_both_passes(n1, n2, tmp_path):
    """16 to 30 points as the strided first pass and as the contiguous second one, in launches too small for the register
    kernel, and the first lengths past them: against numpy in FP64 with the bound of test_short_first_pass (at most 2940
    points)."""
    ctx = focus.Context(0)
    path = str(tmp_path / "tune.txt")
    focus.tune_save(ctx, path)
    n = n1 * n2
    with open(path, "a") as f:
        f.write(f"col {n} {n1}\n")
    focus.tune_load(ctx, path)
    x = (np.random.default_rng(n).standard_normal((n, 257, 2)) @ [1, 1j]).astype(np.complex64)
    t = torch.from_numpy(x).cuda()
    focus.fft(ctx, t, L.FFT_COLUMNS)
    ref = np.fft.fft(x.astype(np.complex128), axis=0)
    assert np.linalg.norm(t.cpu().numpy() - ref) < 1.2e-6 * np.linalg.norm(ref)
    focus.fft(ctx, t, L.FFT_COLUMNS, inverse=True, scale=1.0 / n)
    assert np.linalg.norm(t.cpu().numpy() - x) < 2.4e-6 * np.linalg.norm(x)
    ctx.close()


@pytest.mark.parametrize("n1,n2", [(n, 49) for n in (16, 18, 20, 21, 24, 25, 27, 28, 30)] +
                         [(98, n) for n in (16, 21, 25, 30)])
def test_register_kernel_takes_launches_that_fill_the_chip(n1, n2, tmp_path):
    """16 to 30 points as either pass on 2817 columns (12 workgroups for each of 49 or 98 groups: registers) and on the
    first 257 of them alone (2 for each: LDS): both within the bound of test_short_first_pass of numpy in FP64, and not
    the same sums in the same order."""
    ctx = focus.Context(0)
    path = str(tmp_path / "tune.txt")
    focus.tune_save(ctx, path)
    n = n1 * n2
    with open(path, "a") as f:
        f.write(f"col {n} {n1}\n")
    focus.tune_load(ctx, path)
    x = (np.random.default_rng(n).standard_normal((n, 2817, 2)) @ [1, 1j]).astype(np.complex64)
    wide, narrow = torch.from_numpy(x).cuda(), torch.from_numpy(x[:, :257].copy()).cuda()
    focus.fft(ctx, wide, L.FFT_COLUMNS)
    focus.fft(ctx, narrow, L.FFT_COLUMNS)
    ref = np.fft.fft(x.astype(np.complex128), axis=0)
    got, few = wide.cpu().numpy(), narrow.cpu().numpy()
    assert np.linalg.norm(got - ref) < 1.2e-6 * np.linalg.norm(ref)
    assert np.linalg.norm(few - ref[:, :257]) < 1.2e-6 * np.linalg.norm(ref[:, :257])
    assert not np.array_equal(got[:, :257], few)
    focus.fft(ctx, wide, L.FFT_COLUMNS, inverse=True, scale=1.0 / n)
    assert np.linalg.norm(wide.cpu().numpy() - x) < 2.4e-6 * np.linalg.norm(x)
    ctx.close()


@pytest.mark.parametrize("na,nap", [(1220, 1225), (1310, 1323), (1708, 1715)])
def test_core_of_49_and_63(ctx, na, nap, monkeypatch):
    """Azimuth lengths that only 49 or 63 divides take the fused core: against the separate kernels (FP32 rounding of
    two orders of the same transforms, 2^-24 * sqrt(2 log2 n) * 4 < 1.2e-6 each) and the oracle's interpolation bound."""
    cfg = configs.ers_block().scaled(na=na, nr=1500, n_targets_az=2, n_targets_rg=2, tgt_az=(0.4, 0.6))
    assert focus.padding_size(na) == nap
    raw, _ = scene.generate(cfg)
    out = []
    for fused in ("1", "0"):
        monkeypatch.setenv("ASARF_AZ_FUSED", fused)
        plan = focus.Plan(ctx, cfg)
        plan.execute(torch.from_numpy(raw).cuda())
        assert bool(plan.results()["azimuth_core_fused"]) == (fused == "1")
        out.append(plan.slc_tensor().cpu().numpy())
        plan.close()
    assert np.linalg.norm(out[0] - out[1]) < 1.2e-6 * np.linalg.norm(out[1])
    ref, _ = po.focus_slc(scene.raw_to_complex(raw), cfg)
    assert np.linalg.norm(out[0] - ref) < 1e-4 * np.linalg.norm(ref)


@pytest.mark.parametrize("cols", [17, 18, 19, 20, 23, 24, 25, 1023, 1024, 1025])
@pytest.mark.parametrize("header", [0, 1, 16, 17])
def test_record_rows(ctx, cols, header):
    """Whole 16-byte groups and every remainder, equal to the oracle's records byte for byte (detected values away from
    whole decibels, where single-precision logarithms may differ by an ulp)."""
    rng = np.random.default_rng(cols + header)
    v = (rng.standard_normal((5, cols, 2)) @ [2e4, 2e4j]).astype(np.complex64)
    v[0, :3] = [np.nan, 1e9 - 1e9j, -1e9 + 1j * np.inf]
    got = focus.condition_slc(ctx, torch.from_numpy(v).cuda(), cols, 5, 0.9, header).cpu().numpy()
    assert np.array_equal(got, po.condition_slc(v, cols, 5, 0.9, header))
    d = (10 ** ((rng.integers(-5, 60, (5, cols)) + 0.5) / 10)).astype(np.float32)
    d[1, :3] = [np.nan, 0.0, np.inf]
    got = focus.condition_detected(ctx, torch.from_numpy(d).cuda(), 1.0, header).cpu().numpy()
    assert np.array_equal(got, po.condition_detected(d, 1.0, header))
    m = np.array(focus.image_statistics(ctx, torch.from_numpy(v[1:].copy()).cuda(), cols, 4))
    ref = np.array([v[1:].real.mean(dtype=np.float64), v[1:].imag.mean(dtype=np.float64),
                    v[1:].real.std(dtype=np.float64), v[1:].imag.std(dtype=np.float64)])
    assert np.allclose(m, ref, rtol=1e-9, atol=1e-6)
