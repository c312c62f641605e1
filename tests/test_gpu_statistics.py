"""Statistics of the fused plan: short strips (few lines), the equispaced Doppler fit and the bound that lets a plan
leave out the kernels for shifts beyond the fused core's halo."""
import numpy as np
import pytest
import torch

import pyoracle as po
from asarf import _lib as L
from asarf import configs, focus, scene

pytestmark = pytest.mark.gpu


def _blocks(v, nr, nrp, prf, quirks):
    """Block estimates and their polynomial, as the oracle forms them, of the corrected image v in FP64."""
    step, xs, fs = nr // 32, [], []
    for xb in range(0, nr, step):
        if not quirks & L.Q4_DC_EXTRA_BLOCK and xb + step > nr:
            break
        b = v[:, xb:min(xb + step, nrp)]
        c = np.sum(np.conj(b[:-1]) * b[1:])
        xs.append((2 * xb + step) // 2)
        fs.append(prf * np.angle(c) / (2 * np.pi))
    return np.polyfit(np.array(xs, float), np.array(fs), 2)


@pytest.mark.parametrize("na", [2, 15, 16, 17, 129, 700])
@pytest.mark.parametrize("nr,nc", [(264, 40), (1204, 300), (1201, 300), (4100, 420)])
@pytest.mark.parametrize("quirks", [L.QUIRKS_REFERENCE, 0])
def test_strips_and_fit_against_numpy(ctx, na, nr, nc, quirks):
    """Strips of 16 to 128 rows and every column width of the raw pass: the sums are exact integers, so the I/Q
    estimates match FP64 to 1e-9 and the polynomial, whose fit is well conditioned, to 1e-7 Hz over the swath."""
    rng = np.random.default_rng(na * nr)
    cfg = configs.asar_scene().scaled(na=na, nr=nr, pulse_len=nc / 19.208e6)
    raw = rng.integers(-100, 100, (na, nr, 2)).astype(np.int8)
    plan = focus.Plan(ctx, cfg, quirks=quirks)
    plan.execute(torch.from_numpy(raw).cuda())
    res = plan.results()
    nrp = plan.params.nrp
    plan.close()
    img = np.zeros((na, nrp), np.complex128)
    img[:, :nr] = raw[..., 0] + 1j * raw[..., 1].astype(np.float64)
    iq = po.iq_correction(img, nr, na, quirks=quirks)
    iq = iq[1] if isinstance(iq, tuple) else iq
    for k in ("dc_i", "dc_q", "iq_gain", "phase_error"):
        ref = iq[k] if isinstance(iq, dict) else getattr(iq, k)
        assert abs(res["iq"][k] - ref) <= 1e-9 * max(1.0, abs(ref)), k
    got, ref = np.array(res["dc_poly"]), _blocks(img, nr, nrp, cfg.prf, quirks)
    x = np.arange(0, nr - nc)
    assert np.max(np.abs(np.polyval(got, x) - np.polyval(ref, x))) < 1e-7


@pytest.mark.parametrize("na", [2, 16, 33])
@pytest.mark.parametrize("nr", [298, 300, 367, 959])
@pytest.mark.parametrize("fmt", ["i8", "u8"])
def test_blocks_that_end_on_an_odd_column_inside_the_row(ctx, na, nr, fmt):
    """Without the extra block the last one can end on an odd column before the row's end (300 columns: 33 blocks of 9
    end at 297), whose neighbour must not enter its lag sums. The sums are exact integers, so every estimate is the
    oracle's to FP64 rounding (1e-7 of a PRF of 1.7e3 Hz; one column too many in 9 to 29 moves it by whole Hz)."""
    step = nr // 32
    assert (nr // step * step) % 2 == 1 and nr // step * step < nr and step >= 8
    rng = np.random.default_rng(na * nr)
    base = configs.asar_scene() if fmt == "i8" else configs.ers_block()
    cfg = base.scaled(na=na, nr=nr, pulse_len=40.2 / base.fs)
    v = rng.integers(-100, 100, (na, nr, 2)) if fmt == "i8" else rng.integers(0, 32, (na, nr, 2))
    raw = v.astype(np.int8 if fmt == "i8" else np.uint8)
    plan = focus.Plan(ctx, cfg, quirks=0)
    plan.execute(torch.from_numpy(raw).cuda())
    res = plan.results()
    nrp = plan.params.nrp
    plan.close()
    img = np.zeros((na, nrp), np.complex128)
    img[:, :nr] = scene.raw_to_complex(raw)
    po.iq_correction(img, nr, na, quirks=0)
    _, _, ref = po.doppler_centroid(img, nr, na, cfg.prf, quirks=0)
    assert len(ref) == nr // step and np.max(np.abs(np.array(res["block_freq"]) - ref)) < 1e-7


@pytest.mark.parametrize("sign", [1, -1])
def test_worst_doppler_estimates_stay_in_the_core(ctx, sign):
    """Block estimates of +-0.49 PRF in the pattern that drives the fitted polynomial furthest out at the near end:
    the shift stays within the fused core's halo, and the SLC is the oracle's."""
    cfg = configs.ers_block().scaled(na=600, nr=1600, n_targets_az=1, n_targets_rg=1)
    n, step = 32, cfg.nr // 32
    u = np.arange(n) - (n - 1) / 2
    q, u0 = u * u - np.mean(u * u), -(step // 2) / step - (n - 1) / 2
    w = 1 / n + u0 * u / np.sum(u * u) + (u0 * u0 - np.mean(u * u)) * q / np.sum(q * q)
    f = np.repeat(np.where(w >= 0, 0.49, -0.49) * sign, step)
    ph = 2 * np.pi * f[None, :] * np.arange(cfg.na)[:, None] + np.random.default_rng(3).uniform(0, 6.28, cfg.nr)[None, :]
    raw = np.stack([np.cos(ph), np.sin(ph)], axis=-1) * 12 + 15.5
    raw = np.clip(np.round(raw), 0, 31).astype(np.uint8)
    plan = focus.Plan(ctx, cfg)
    plan.execute(torch.from_numpy(raw).cuda())
    slc, res = plan.slc_tensor().cpu().numpy(), plan.results()
    plan.set_timing(True)
    plan.execute(torch.from_numpy(raw).cuda())
    names = set(plan.kernel_times())
    plan.close()
    assert res["azimuth_core_fused"] and 4 <= res["rcmc_shift_bound"] <= 8
    assert "azimuth_core_wide" not in names and "azimuth_fft_b" not in names
    ref, _ = po.focus_slc(scene.raw_to_complex(raw), cfg)
    assert float(np.sqrt(np.sum(np.abs(slc - ref) ** 2) / np.sum(np.abs(ref) ** 2))) < 1e-4


@pytest.mark.parametrize("what", ["zeros", "constant", "constant Q"])
@pytest.mark.parametrize("fmt", ["i8", "u8"])
def test_undefined_statistics_give_the_same_with_and_without_the_core(ctx, what, fmt, monkeypatch):
    """A channel without variance leaves the I/Q gain and the centroid undefined (a constant Q alone does so without the
    reference's padding columns in the sums): NaN in every pixel of the SLC, whether the radar's bound on the shift
    admits the fused core alone or the separate kernels run."""
    base = configs.asar_scene() if fmt == "i8" else configs.ers_block()
    cfg = base.scaled(na=600, nr=1300, pulse_len=200.2 / base.fs)
    raw = np.zeros((cfg.na, cfg.nr, 2), np.int8 if fmt == "i8" else np.uint8)
    if what != "zeros":
        raw[...] = 15
    if what == "constant Q":
        raw[..., 0] = np.random.default_rng(1).integers(0, 32, (cfg.na, cfg.nr))
    for fused in ("1", "0"):
        monkeypatch.setenv("ASARF_AZ_FUSED", fused)
        plan = focus.Plan(ctx, cfg, quirks=0 if what == "constant Q" else L.QUIRKS_REFERENCE)
        plan.set_timing(True)
        plan.execute(torch.from_numpy(raw).cuda())
        names = set(plan.kernel_times())
        slc, res = plan.slc_tensor().cpu().numpy(), plan.results()
        plan.close()
        assert ("azimuth_core_fused" in names and "azimuth_core_wide" not in names) == (fused == "1")
        assert np.isnan(res["dc_poly"]).all() and np.isnan(slc.real).all() and np.isnan(slc.imag).all(), fused
