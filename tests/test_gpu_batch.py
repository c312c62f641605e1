"""Autotuner and batched focusing on the GPU: tuned schedules keep the results, a heterogeneous batch gives the
same SLCs sequentially and as one captured graph, and repeated graph replays (with eager work between them)
reproduce the eager result every time."""
import numpy as np
import pytest
import torch

import pyoracle as po
from asarf import _lib as L
from asarf import configs, focus, scene

pytestmark = pytest.mark.gpu


def rel_rms(a, b):
    a = np.asarray(a, np.complex128)
    b = np.asarray(b, np.complex128)
    return float(np.sqrt(np.sum(np.abs(a - b) ** 2) / np.sum(np.abs(b) ** 2)))


def test_autotuned_schedules_keep_parity():
    ctx = focus.Context(0)
    cfg = configs.asar_scene().scaled(na=700, nr=1400, n_targets_random=4)
    nrp = focus.padding_size(cfg.nr + cfg.nc)
    nap = focus.padding_size(cfg.na)
    rows = focus.autotune(ctx, nrp, columns=False, batch=256)
    cols = focus.autotune(ctx, nap, columns=True, batch=512)
    print(f"rows {nrp}: {rows}; columns {nap}: {cols}")
    assert rows["candidates"] >= 1 and rows["ms"] > 0
    assert cols["candidates"] >= 1 and cols["ms"] > 0 and nap % cols["choice"] == 0
    raw, _ = scene.generate(cfg)
    plan = focus.Plan(ctx, cfg)
    plan.execute(torch.from_numpy(raw).cuda())
    slc = plan.slc_tensor().cpu().numpy()
    plan.close()
    ref, _ = po.focus_slc(scene.raw_to_complex(raw), cfg)
    assert rel_rms(slc, ref) < 1e-4
    # a length with a compile-time kernel: the tuner weighs it against runtime radix orders
    r6400 = focus.autotune(ctx, 6400, columns=False, batch=128)
    assert r6400["candidates"] >= 2
    ctx.close()


def test_tuner_cache_file_round_trip(tmp_path):
    """Choices saved from one context load into another and drive its plans; the file names the device
    architecture and every choice of the first context."""
    ctx = focus.Context(0)
    cfg = configs.asar_scene().scaled(na=700, nr=1400, n_targets_random=4)
    nrp = focus.padding_size(cfg.nr + cfg.nc)
    nap = focus.padding_size(cfg.na)
    rows = focus.autotune(ctx, nrp, columns=False, batch=256)
    cols = focus.autotune(ctx, nap, columns=True, batch=512)
    path = tmp_path / "tune.txt"
    focus.tune_save(ctx, str(path))
    text = path.read_text().splitlines()
    assert text[0].startswith("asarf-tune 1 gfx950")
    assert f"col {nap} {cols['choice']}" in text
    assert any(t.startswith(f"row {nrp} ") for t in text)
    ctx.close()
    ctx2 = focus.Context(0)
    assert focus.tune_load(ctx2, str(path)) == 2
    # saving the loaded context reproduces the file
    path2 = tmp_path / "tune2.txt"
    focus.tune_save(ctx2, str(path2))
    assert path2.read_text() == path.read_text()
    raw, _ = scene.generate(cfg)
    plan = focus.Plan(ctx2, cfg)
    plan.execute(torch.from_numpy(raw).cuda())
    slc = plan.slc_tensor().cpu().numpy()
    plan.close()
    ref, _ = po.focus_slc(scene.raw_to_complex(raw), cfg)
    assert rel_rms(slc, ref) < 1e-4
    # another architecture's file is refused and changes nothing
    other = tmp_path / "other.txt"
    other.write_text("asarf-tune 1 gfx942\ncol 30240 168\n")
    with pytest.raises(RuntimeError, match="tuned on gfx942"):
        focus.tune_load(ctx2, str(other))
    ctx2.close()


def _slc_with(monkeypatch, cfg, traw, rows="", **env):
    """SLC of a plan in a new context with the given tuner file entries, under the given environment."""
    ctx = focus.Context(0)
    for k, v in env.items():
        monkeypatch.setenv(k, v)
    if rows:
        path = rows["dir"] / "tune.txt"
        focus.tune_save(ctx, str(path))
        path.write_text(path.read_text() + rows["text"] + "\n")
        focus.tune_load(ctx, str(path))
        again = rows["dir"] / "again.txt"
        focus.tune_save(ctx, str(again))
        assert rows["text"] in again.read_text().splitlines()
    plan = focus.Plan(ctx, cfg)
    plan.execute(traw)
    slc = plan.slc_tensor().cpu().numpy()
    plan.close()
    ctx.close()
    for k in env:
        monkeypatch.delenv(k)
    return slc


@pytest.mark.parametrize("choice,env", [("static 3", {"ASARF_RC_VARIANT": "3"}), ("radix 8 8 4 5 5", None)])
def test_padded_row_choices_displace_blocks_only_when_measured_faster(monkeypatch, tmp_path, choice, env):
    """A row choice without the mark leaves the blocks their lines and is taken where blocks are off; a marked one
    replaces them. The same kernels give the same bits."""
    cfg = configs.ers_block().scaled(na=64, n_targets_az=1, n_targets_rg=1)
    assert focus.padding_size(cfg.nr + cfg.nc) == 6400
    traw = torch.from_numpy(scene.generate(cfg)[0]).cuda()
    blocks = _slc_with(monkeypatch, cfg, traw)
    plain = {"dir": tmp_path, "text": f"row 6400 {choice}"}
    marked = {"dir": tmp_path, "text": f"row 6400 padded {choice}"}
    assert np.array_equal(_slc_with(monkeypatch, cfg, traw, plain), blocks)
    padded = _slc_with(monkeypatch, cfg, traw, plain, ASARF_RC_BLOCK="0")
    assert not np.array_equal(padded, blocks) and rel_rms(padded, blocks) < 2e-6
    assert np.array_equal(_slc_with(monkeypatch, cfg, traw, marked), padded)
    if env:
        assert np.array_equal(_slc_with(monkeypatch, cfg, traw, **env), padded)


def test_a_choice_made_after_creation_is_captured(monkeypatch, tmp_path):
    """A plan whose lines run in blocks, captured right after a padded choice was loaded (or forced): every replay gives
    that choice's bits, with eager work between the replays."""
    cfg = configs.ers_block().scaled(na=64, n_targets_az=1, n_targets_rg=1)
    traw = torch.from_numpy(scene.generate(cfg)[0]).cuda()
    want = _slc_with(monkeypatch, cfg, traw, ASARF_RC_VARIANT="3")
    for how in ("file", "environment"):
        stream = torch.cuda.Stream()
        ctx = focus.Context(0, stream=stream)
        plan = focus.Plan(ctx, cfg)
        torch.cuda.synchronize()
        with torch.cuda.stream(stream):
            plan.execute(traw)
            blocks = plan.slc_tensor()
        torch.cuda.synchronize()
        assert not np.array_equal(blocks.cpu().numpy(), want)
        if how == "file":
            path = tmp_path / "tune.txt"
            focus.tune_save(ctx, str(path))
            path.write_text(path.read_text() + "row 6400 padded static 3\n")
            focus.tune_load(ctx, str(path))
        else:
            monkeypatch.setenv("ASARF_RC_VARIANT", "3")
        graph = torch.cuda.CUDAGraph()
        out = torch.zeros_like(blocks)
        with torch.cuda.graph(graph, stream=stream):
            img = plan.execute(traw)
            focus.subset_copy(ctx, img, 0, 0, img.x_size, img.y_size, out)
        for _ in range(3):
            out.zero_()
            torch.cuda.synchronize()
            graph.replay()
            torch.cuda.synchronize()
            assert np.array_equal(out.cpu().numpy(), want), how
            with torch.cuda.stream(stream):
                plan.execute(traw)
            torch.cuda.synchronize()
        monkeypatch.delenv("ASARF_RC_VARIANT", raising=False)
        del graph
        plan.close()
        ctx.close()


def test_row_tuner_measures_the_padded_default_beside_the_blocks(tmp_path):
    """The recorded choice is one of the padded candidates, whichever way the blocks compare, and the file says which."""
    ctx = focus.Context(0)
    r = focus.autotune(ctx, 6400, columns=False, batch=512)
    focus.tune_save(ctx, str(tmp_path / "tune.txt"))
    ctx.close()
    row = [t for t in (tmp_path / "tune.txt").read_text().splitlines() if t.startswith("row 6400 ")]
    want = f"static {-1 - r['choice']}" if r["choice"] < 0 else "radix "
    assert len(row) == 1 and row[0].replace("padded ", "").startswith(f"row 6400 {want}")
    # six compile-time variants and the blocks, beside at least one radix order
    assert r["choice"] >= -6 and r["candidates"] >= 8


def test_batch_graph_equals_sequential_and_replays(ctx):
    cfgs = configs.batch_blocks(6, na_range=(300, 900))
    cfgs = [c.scaled(nr=min(c.nr, 1500)) for c in cfgs]
    raws = [torch.from_numpy(scene.generate(c)[0]).cuda() for c in cfgs]
    b = focus.Batch(ctx, n_streams=3)
    for c, r in zip(cfgs, raws):
        b.add(c, r)
    b.execute(focus.BATCH_SEQUENTIAL)
    seq = [b.slc_tensor(i).cpu().numpy() for i in range(len(cfgs))]
    for rep in range(3):
        b.execute(focus.BATCH_GRAPH)
        b.sync()
        got = [b.slc_tensor(i).cpu().numpy() for i in range(len(cfgs))]
        for i in range(len(cfgs)):
            assert np.array_equal(got[i], seq[i]), (rep, i)
        # eager work on the same buffers between replays
        b.execute(focus.BATCH_SEQUENTIAL)
        torch.cuda.synchronize()
    ref, _ = po.focus_slc(scene.raw_to_complex(scene.generate(cfgs[1])[0]), cfgs[1])
    err = rel_rms(seq[1], ref)
    print(f"batch block 1 ({cfgs[1].name}) slc rel rms {err:.2e}")
    assert err < 1e-4
    b.close()


@pytest.mark.parametrize("which,nvar", [("asar", 10), ("ers", 6), ("ers8192", 7)])
def test_range_compression_variants_match_oracle(ctx, which, nvar):
    """Every compile-time range-compression variant the autotuner may pick gives the oracle's SLC."""
    import os
    if which == "asar":
        cfg = configs.asar_scene().scaled(na=256, n_targets_random=3)
    elif which == "ers":
        cfg = configs.ers_block().scaled(na=256, n_targets_az=1, n_targets_rg=3, tgt_az=(0.5, 0.5))
    else:
        cfg = configs.ers_block().scaled(na=256, n_targets_az=1, n_targets_rg=3, tgt_az=(0.5, 0.5), nrp=8192)
    raw, _ = scene.generate(cfg)
    traw = torch.from_numpy(raw).cuda()
    ref, _ = po.focus_slc(scene.raw_to_complex(raw), cfg)
    for v in range(nvar):
        os.environ["ASARF_RC_VARIANT"] = str(v)
        try:
            plan = focus.Plan(ctx, cfg)
            plan.execute(traw)
            slc = plan.slc_tensor().cpu().numpy()
            plan.close()
        finally:
            del os.environ["ASARF_RC_VARIANT"]
        err = rel_rms(slc, ref)
        print(f"{which} variant {v}: slc rel rms {err:.2e}")
        assert err < 1e-4, v
