"""Range compression in blocks of a line (csrc/rc_block.h): every compiled block length and every raw format, at line
and chirp lengths on both sides of each block boundary, against numpy in FP64 (stage entry point) and against the
transforms of the padded line (plan)."""
import os

import numpy as np
import pytest
import torch

import pyoracle as po
from asarf import configs, focus, scene

pytestmark = pytest.mark.gpu

# Two FP32 transforms of at most 2^13 points, each product and sum rounded to 2^-24: the relative RMS error grows like
# 2^-24 * sqrt(2 * 13) ~ 3e-7 per transform pair; two paths of it and twiddles of their own stay below 1e-6.
TOL = 1e-6


def rel_rms(a, b):
    return float(np.sqrt(np.sum(np.abs(a - b) ** 2) / np.sum(np.abs(b) ** 2)))


@pytest.mark.parametrize("nr", [60, 1024, 1025, 1536, 1537, 2048, 2049, 2560, 2561, 3072, 3073, 4096, 4097,
                                5617, 6144])
@pytest.mark.parametrize("tail", [False, True])
def test_lines_in_place_against_numpy(ctx, nr, tail):
    """Whole lines of every block length, in place; a chirp with a sample past nc takes the padded transform."""
    rng = np.random.default_rng(nr)
    nc = min(521, nr // 2)
    rows, stride = 5, focus.padding_size(nr + nc)
    chirp = np.zeros(stride, np.complex64)
    chirp[:nc] = rng.standard_normal(nc) + 1j * rng.standard_normal(nc)
    if tail:
        chirp[nc] = 2.0
    x = np.zeros((rows + 1, stride), np.complex64)
    x[:rows, :nr] = rng.standard_normal((rows, nr)) + 1j * rng.standard_normal((rows, nr))
    x[:rows, nr:] = 0.25 - 0.5j  # what the I/Q correction leaves in the padding
    t = torch.from_numpy(x).cuda()
    got_nr = focus.range_compression(ctx, t, nr, rows, chirp, nc)
    got = t.cpu().numpy()
    h = np.conj(np.fft.fft(chirp.astype(np.complex128)))
    ref = np.fft.ifft(np.fft.fft(x[:rows].astype(np.complex128), axis=1) * h, axis=1)[:, :nr - nc]
    assert got_nr == nr - nc
    assert rel_rms(got[:rows, :nr - nc], ref) < TOL
    assert not got[:rows, nr - nc:].any() and np.array_equal(got[rows], x[rows])
    # a chirp sample past nc too small to count sends the same lines through the padded transform, which lines of 60
    # samples, far shorter than any block, take anyway
    if not tail:
        chirp[nc] = 1e-30
        padded = torch.from_numpy(x).cuda()
        focus.range_compression(ctx, padded, nr, rows, chirp, nc)
        assert np.array_equal(padded.cpu().numpy()[:rows, :nr - nc], got[:rows, :nr - nc]) == (nr == 60)


def _slc(ctx, cfg, block, run, **kw):
    old = os.environ.get("ASARF_RC_BLOCK")
    os.environ["ASARF_RC_BLOCK"] = str(block)
    try:
        plan = focus.Plan(ctx, cfg, **kw)
    finally:
        if old is None:
            del os.environ["ASARF_RC_BLOCK"]
        else:
            os.environ["ASARF_RC_BLOCK"] = old
    run(plan)
    slc = plan.slc_tensor().cpu().numpy().astype(np.complex128)
    plan.close()
    return slc


@pytest.mark.parametrize("nr,nc", [(1200, 704), (1999, 463), (4937, 497), (5616, 521), (5617, 704), (7001, 300)])
@pytest.mark.parametrize("fmt", ["u8", "i8", "lines", "fbaq4"])
def test_plan_blocks_against_padded_lines(ctx, nr, nc, fmt):
    """Raw lines in one to several blocks, odd pitches, SWST shifts beyond a block's end, short FBAQ records."""
    rng = np.random.default_rng(nr + nc)
    na, fs = 96, 19.208e6
    base = configs.ers_block() if fmt in ("u8", "lines") else configs.asar_scene()
    cfg = base.scaled(na=na, nr=nr, pulse_len=nc / fs, fs=fs, nrp=8192 if nr > 6000 else 0)
    swst = torch.from_numpy((700 + rng.integers(0, 9, na)).astype(np.int16)).cuda()
    if fmt in ("u8", "i8"):
        v = rng.integers(0, 32, (na, nr, 2)) if fmt == "u8" else rng.integers(-100, 100, (na, nr, 2))
        raw = torch.from_numpy(v.astype(np.uint8 if fmt == "u8" else np.int8)).cuda()
        kw, run = {}, lambda p: p.execute(raw)
    elif fmt == "lines":
        spl = nr - 32
        lines = torch.from_numpy(rng.integers(0, 32, (na, 2 * spl)).astype(np.uint8)).cuda()
        kw, run = {"lines": (spl, 2 * spl, 4)}, lambda p: p.execute_lines(lines, swst, 700)
    else:
        nblk = (nr - 8 + 62) // 63
        rec = rng.integers(0, 256, (na, 2 + 64 * nblk)).astype(np.uint8)
        length = np.full(na, 64 * nblk)
        length[::7] = 64 * (nblk // 2) + 9
        rec[:, 0], rec[:, 1] = length & 255, length >> 8
        rec = torch.from_numpy(rec).cuda()
        lut = [torch.from_numpy(rng.standard_normal(4096).astype(np.float32)).cuda() for _ in range(2)]
        kw, run = {"fbaq": (rec.shape[1], 1)}, lambda p: p.execute_fbaq4(rec, swst, 700, lut[0], lut[1])
    padded = _slc(ctx, cfg, 0, run, **kw)
    lengths = [n for n in (1024, 1536, 2048, 2560, 3072, 4096, 6144) if n >= nc + 200]
    for block in [""] + lengths:
        err = rel_rms(_slc(ctx, cfg, block, run, **kw), padded)
        assert 0 < err < TOL, (block, err)  # 0: the padded lines ran again


@pytest.mark.parametrize("mean", [(15.5, 15.5), (60.1, 117.7), (117.3, 60.6), (200.3, 201.9)])
@pytest.mark.parametrize("fmt", ["u8", "lines", "i8"])
def test_correction_rounds_the_signal_and_not_its_mean(ctx, mean, fmt):
    """Weak samples on a large offset, which the affine I/Q correction takes out: the SLC stays within the transforms'
    rounding of the FP64 oracle (TOL: two transform pairs). A coefficient that rounds on the mean leaves a constant of
    up to 2^-24 * 200 / 2 = 6e-6 of the signal."""
    rng = np.random.default_rng(int(mean[0] * 10))
    na, nr, nc, std = 256, 1500, 300, 2.0
    base = configs.asar_scene() if fmt == "i8" else configs.ers_block()
    cfg = base.scaled(na=na, nr=nr, pulse_len=(nc + 0.2) / base.fs)
    v = np.round(rng.standard_normal((na, nr, 2)) * std + np.array(mean) - (128 if fmt == "i8" else 0))
    raw = v.astype(np.int8 if fmt == "i8" else np.uint8)
    plan = focus.Plan(ctx, cfg, lines=(nr, 2 * nr, 1) if fmt == "lines" else None)
    if fmt == "lines":
        plan.execute_lines(torch.from_numpy(raw.reshape(na, 2 * nr)).cuda(), torch.full((na,), 7, dtype=torch.int16).cuda(), 7)
    else:
        plan.execute(torch.from_numpy(raw).cuda())
    slc = plan.slc_tensor().cpu().numpy()
    plan.close()
    ref, _ = po.focus_slc(scene.raw_to_complex(raw), cfg)
    assert rel_rms(slc, ref) < TOL


@pytest.mark.parametrize("nr", [1024, 1536, 2048, 2560, 3072, 4096, 6144])
def test_lines_keep_their_amplitude(ctx, nr):
    """Least-squares gain of the compressed lines against FP64, every block length: rounding errors of about 1.8e-7 per
    sample average to below 1e-9 over 256 lines, so what is left is a common scale, bounded by a third of an FP32
    rounding (2e-8)."""
    rng = np.random.default_rng(nr)
    rows, nc = 256, 400
    stride = focus.padding_size(nr + nc)
    t = np.arange(nc) / nc - 0.5
    chirp = np.zeros(stride, np.complex64)
    chirp[:nc] = np.exp(1j * np.pi * 0.8 * nc * t * t)
    x = np.zeros((rows, stride), np.complex64)
    x[:, :nr] = rng.standard_normal((rows, nr)) + 1j * rng.standard_normal((rows, nr))
    d = torch.from_numpy(x).cuda()
    focus.range_compression(ctx, d, nr, rows, chirp, nc)
    got = d.cpu().numpy()[:, :nr - nc].astype(np.complex128)
    h = np.conj(np.fft.fft(chirp.astype(np.complex128)))
    ref = np.fft.ifft(np.fft.fft(x.astype(np.complex128), axis=1) * h, axis=1)[:, :nr - nc]
    assert abs(np.vdot(ref, got) / np.vdot(ref, ref) - 1) < 2e-8
