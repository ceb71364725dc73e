"""Autotuning (baorec_autotune): the tuned scatter tiles and strided-pass
kernels must leave every result bitwise unchanged, and tuned tables must
survive a save / load round trip."""
import ctypes
import json

import numpy as np
import pytest

import baorec_hip as bh
from baorec_hip import synth

pytestmark = pytest.mark.gpu

F32 = np.float32


def box_kw(ctx, los=(0.0, 0.0, 1.0)):
    return dict(bias=2.0, f=0.8, smoothing_radius=15.0, box_size=[1000.0] * 3, box_min=[0.0] * 3,
                los=None if los is None else list(los), ctx=ctx)


@pytest.mark.parametrize("g,los", [((128, 128, 128), (0.0, 0.0, 1.0)), ((64, 256, 256), None)])
def test_tuned_results_are_bitwise_unchanged(g, los):
    x, y, z, w = synth.box_catalog(300000, L=1000.0, mesh=64, seed=41)
    plain, tuned = bh.Context(0), bh.Context(0)
    rep = bh.autotune(bh.IterativeRecon(**box_kw(tuned, los)), g, x, y, z, w)
    print(json.dumps(rep))
    assert len(rep["scatter"]) == 1
    e = rep["scatter"][0]
    assert e["grid"] == list(g) and e["log2n"] == int(np.floor(np.log2(len(x))))
    tx, ty, tz = e["tile"]
    assert tx * ty * tz <= 32 * 16 * 16
    assert {(s["axis"], s["n"]) for s in rep["strided"]} == {(a, n) for a, n in ((1, g[1]), (2, g[2])) if n >= 256}
    out = []
    for ctx in (plain, tuned):
        rec = bh.IterativeRecon(**box_kw(ctx, los))
        cx, cy, cz = x.copy(), y.copy(), z.copy()
        d = bh.run_(rec, g, cx, cy, cz, w)
        p = bh.reconstructed_positions(rec, cx, cy, cz, field="sum")
        out.append((d, p))
    np.testing.assert_array_equal(out[0][0], out[1][0])
    for a, b in zip(out[0][1], out[1][1]):
        np.testing.assert_array_equal(a, b)


def test_tune_save_load_roundtrip(tmp_path):
    x, y, z, w = synth.box_catalog(100000, L=1000.0, mesh=64, seed=42)
    a, b = bh.Context(0), bh.Context(0)
    rep = bh.autotune(bh.IterativeRecon(**box_kw(a)), (64, 64, 256), x, y, z, w)
    path = tmp_path / "tune.json"
    bh.tune_save(path, a)
    assert json.loads(path.read_text()) == rep
    bh.tune_load(path, b)
    assert bh.tune_report(b) == rep


def test_tune_load_rejects_unusable_entries(tmp_path):
    ctx = bh.Context(0)
    bad = tmp_path / "bad.json"
    bad.write_text('{"scatter": [\n  {"grid": [64, 64, 64], "tsc": 0, "log2n": 10, "tile": [64, 64, 64]}],\n'
                   ' "strided": []}\n')
    with pytest.raises(bh.BaorecError):
        bh.tune_load(bad, ctx)
    assert bh.tune_report(ctx) == {"scatter": [], "strided": []}


def test_failed_tuning_leaves_no_forced_choice():
    """A catalog outside the box: BoundsError, nothing tuned, and later calls
    use the library's own choices."""
    x, y, z, w = synth.box_catalog(50000, L=1000.0, mesh=64, seed=43)
    ctx = bh.Context(0)
    bad = x.copy()
    bad[:100] = -50.0      # below box_min: outside the grid
    with pytest.raises(bh.BoundsError):
        bh.autotune(bh.IterativeRecon(**box_kw(ctx)), (64, 64, 64), bad, y, z, w)
    assert bh.tune_report(ctx) == {"scatter": [], "strided": []}
    plain = bh.Context(0)
    out = []
    for c in (plain, ctx):
        rec = bh.IterativeRecon(**box_kw(c))
        out.append(bh.run_(rec, (64, 64, 64), x.copy(), y.copy(), z.copy(), w))
    np.testing.assert_array_equal(out[0], out[1])


@pytest.mark.parametrize("los", [(0.0, 0.0, 1.0), None])
@pytest.mark.parametrize("g", [(16, 256, 512), (1024, 16, 256), (32, 512, 16), (64, 256, 32)])
def test_staying_passes_match_the_general_ones(tmp_path, g, los):
    """y and z passes of several outputs at 256 and 512 by workgroups that walk
    over tiles, against the general kernel (a table that asks for one column
    per thread), single catalogs and batches, with columns past the last one
    and fewer tiles than workgroups.  The table also changes the passes of one
    output, whose two kernels round differently: about 30 FP32 transforms of
    rms error eps sqrt(log2 n) each, five times that at the largest of 10^6
    cells is 1e-5 of the field, twice that is allowed (a position: 2e-5 of the
    largest displacement of its catalog's field, read at all positions, and two
    roundings)."""
    path = tmp_path / "general.json"
    path.write_text('{"scatter": [],\n "strided": [\n' +
                    ",\n".join(f'  {{"axis": {a}, "n": {n}, "pair": 0}}' for a in (1, 2) for n in (256, 512)) + "]}\n")
    plain, general = bh.Context(0), bh.Context(0)
    bh.tune_load(path, general)
    x, y, z, w = synth.box_catalog(60000, L=1000.0, mesh=64, seed=44)
    off = np.array([0, 20000, 20001, 60000])
    out = []
    for ctx in (plain, general):
        rec = bh.IterativeRecon(**box_kw(ctx, los))
        d = bh.run_(rec, g, x.copy(), y.copy(), z.copy(), w)
        p = bh.reconstructed_positions(rec, x, y, z, field="sum")
        b = bh.run_batch(rec, g, x, y, z, w, off)
        out.append([d, *p, *b])
    (d0, *p0), (d1, *p1) = out
    assert np.max(np.abs(d0 - d1)) <= 2e-5 * np.max(np.abs(d1))
    rec = bh.IterativeRecon(**box_kw(plain, los))
    for k, (b0, b1) in enumerate([(0, 60000), *zip(off[:-1], off[1:])]):
        bh.run_(rec, g, *(v[b0:b1].copy() for v in (x, y, z, w)))
        at = bh.reconstructed_positions(rec, x, y, z, field="sum")
        size = max(np.max(np.abs(q - v)) for q, v in zip(at, (x, y, z)))
        for a, b in zip(p0[:3] if k == 0 else p0[3:], p1[:3] if k == 0 else p1[3:]):
            assert np.max(np.abs(a - b)[b0:b1]) <= 2e-5 * size + 2 * np.spacing(F32(1000.0))


def strided_table(path, **choice):
    """A table with the given choice for both axes at 256 and 512."""
    lines = [f'  {{"axis": {a}, "n": {n}, "{k}": {v}}}' for k, v in choice.items() for a in (1, 2) for n in (256, 512)]
    path.write_text('{"scatter": [],\n "strided": [\n' + ",\n".join(lines) + "]}\n")
    return path


def launches(ctx, fn):
    """Launches per profiler label during fn()."""
    ctx.lib.baorec_profile(ctx.handle, 1)
    fn()
    buf = ctypes.create_string_buffer(1 << 16)
    ctx.lib.baorec_profile_report(ctx.handle, buf, len(buf))
    ctx.lib.baorec_profile(ctx.handle, 0)
    return {k: v["count"] for k, v in json.loads(buf.value.decode()).items()}


def test_pair_choice_leaves_the_passes_of_several_outputs(tmp_path):
    """A tuned or loaded "pair" picks the kernel of the passes of one output
    alone, which is all that the tuner times; the local-LOS iteration's and
    the displacement's passes keep theirs unless the table says "staying": 0."""
    x, y, z, w = synth.box_catalog(60000, L=1000.0, mesh=64, seed=47)
    seen = []
    for choice in ({}, {"pair": 1}, {"pair": 0}, {"pair": 1, "staying": 0}):
        ctx = bh.Context(0)
        if choice:
            bh.tune_load(strided_table(tmp_path / "t.json", **choice), ctx)
            assert [s for s in bh.tune_report(ctx)["strided"] if "staying" in s] == \
                [{"axis": a, "n": n, "staying": 0} for a in (1, 2) for n in (256, 512) if "staying" in choice]
        rec = bh.IterativeRecon(**box_kw(ctx, None))

        def run():
            bh.run_(rec, (16, 512, 256), x.copy(), y.copy(), z.copy(), w)
            bh.reconstructed_positions(rec, x, y, z, field="sum")
        seen.append(launches(ctx, run))
    plain, pair1, pair0, general = seen
    staying = {k: v for k, v in plain.items() if k.endswith("_staying")}
    assert set(staying) == {"fft_y_staying", "fft_z_staying"} and staying["fft_z_staying"] >= 3
    assert plain["fft_z_pair"] > 0 and "fft_z_pair" not in pair0
    for s in (pair1, pair0):
        assert {k: v for k, v in s.items() if k.endswith("_staying")} == staying
    assert not any(k.endswith("_staying") for k in general)


@pytest.mark.parametrize("los", [(0.0, 0.0, 1.0), None])
@pytest.mark.parametrize("g", [(16, 256, 512), (1024, 16, 256), (32, 512, 16), (64, 256, 32)])
def test_staying_passes_match_k_strided(tmp_path, g, los):
    """The same comparison as above with a table that changes the passes of
    several outputs alone, and its tolerance."""
    plain, general = bh.Context(0), bh.Context(0)
    bh.tune_load(strided_table(tmp_path / "t.json", staying=0), general)
    x, y, z, w = synth.box_catalog(60000, L=1000.0, mesh=64, seed=44)
    off = np.array([0, 20000, 20001, 60000])
    out = []
    for ctx in (plain, general):
        rec = bh.IterativeRecon(**box_kw(ctx, los))
        d = bh.run_(rec, g, x.copy(), y.copy(), z.copy(), w)
        p = bh.reconstructed_positions(rec, x, y, z, field="sum")
        out.append([d, *p, *bh.run_batch(rec, g, x, y, z, w, off)])
    (d0, *p0), (d1, *p1) = out
    print(f"{g} los {los}: {sum(int(np.sum(a != b)) for a, b in zip(out[0], out[1]))} values differ")
    assert np.max(np.abs(d0 - d1)) <= 2e-5 * np.max(np.abs(d1))
    rec = bh.IterativeRecon(**box_kw(general, los))
    for k, (b0, b1) in enumerate([(0, 60000), *zip(off[:-1], off[1:])]):
        bh.run_(rec, g, *(v[b0:b1].copy() for v in (x, y, z, w)))
        at = bh.reconstructed_positions(rec, x, y, z, field="sum")
        size = max(np.max(np.abs(q - v)) for q, v in zip(at, (x, y, z)))
        for a, b in zip(p0[:3] if k == 0 else p0[3:], p1[:3] if k == 0 else p1[3:]):
            assert np.max(np.abs(a - b)[b0:b1]) <= 2e-5 * size + 2 * np.spacing(F32(1000.0))
