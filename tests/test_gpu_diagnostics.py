"""The engine's diagnostic modes, the reference HIP backend's E2_HIP_PROFILE and E2_HIP_DUMP
(src/gpu/hip/hip.c:51-108,138-139, forward.c:715-759): E2MI_PROFILE reports per-stage kernel times
of the first call without changing its results; E2MI_DUMP writes the workspace after a call, and the
dumped residual after layer 0 is the oracle's layer-0 output on the dumped rows (per-row cosine
median >= 0.9999, every row >= 0.999)."""
import os

import numpy as np
import pytest

from model_util import oracle_model, random_batch, small_config

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def model(gpu):
    import e2mi
    return e2mi, e2mi.Model.synthetic(small_config(e2mi, n_layers=2), 91)


def test_profile_reports_stages(model, rng, monkeypatch):
    e2mi, m = model
    ids, valid = random_batch(rng, 4, 128, 1000, min_len=40)
    want = e2mi.Engine(m, max_rows=1024).embed_batch(ids, valid)
    monkeypatch.setenv("E2MI_PROFILE", "1")
    eng = e2mi.Engine(m, max_rows=1024)
    monkeypatch.delenv("E2MI_PROFILE")
    lib = e2mi.load()
    assert lib.e2mi_profile_text(eng.h).decode() == ""
    got = eng.embed_batch(ids, valid)
    assert np.array_equal(got, want)
    text = lib.e2mi_profile_text(eng.h).decode()
    stages = {}
    for line in text.splitlines()[1:]:
        f = line.split()
        stages[f[1]] = (float(f[2]), int(f[4]))
    # the O and down projections run their norm_add in the GEMM's epilogue (768-wide model)
    for s in ("embed", "qkv_norm_rope_gemm", "attention", "o_proj+add_norm", "gate_up_geglu", "down+add_norm", "pool"):
        assert s in stages and stages[s][0] > 0, (s, text)
    assert stages["o_proj+add_norm"][1] == 2 and stages["down+add_norm"][1] == 2   # per layer, 2 layers
    assert stages["attention"][1] == 2
    # later calls run the graph and add nothing
    assert np.array_equal(eng.embed_batch(ids, valid), want)
    assert lib.e2mi_profile_text(eng.h).decode() == text


def test_profile_names_the_norm_add_of_few_rows(model, rng, monkeypatch):
    """Up to 256 rows a norm_add runs in the GEMM that reads it: its time is in that GEMM's line, and the
    projections' lines are theirs alone but for the last, which norms in its epilogue."""
    e2mi, m = model
    monkeypatch.setenv("E2MI_PROFILE", "1")
    eng = e2mi.Engine(m, max_rows=1024)
    monkeypatch.delenv("E2MI_PROFILE")
    eng.embed_batch(rng.integers(0, 1000, (1, 19)).astype(np.int32), None)
    lines = [l.split() for l in e2mi.load().e2mi_profile_text(eng.h).decode().splitlines()[1:]]
    calls = {f[1]: int(f[4]) for f in lines}
    assert calls == {"embed": 1, "qkv_norm_rope_gemm": 1, "add_norm+qkv_norm_rope_gemm": 1, "attention": 2, "o_proj": 2,
                     "add_norm+gate_up_geglu": 2, "down": 1, "down+add_norm": 1, "pool": 1}, calls


def test_dump_after_layer_zero(model, oracle, rng, monkeypatch, tmp_path):
    e2mi, m = model
    ids, valid = random_batch(rng, 3, 100, 1000, min_len=30)
    monkeypatch.setenv("E2MI_DUMP", str(tmp_path))
    eng = e2mi.Engine(m, max_rows=1024)
    monkeypatch.delenv("E2MI_DUMP")
    eng.set_layer_limit(1)
    out = eng.embed_batch(ids, valid)
    names = sorted(os.listdir(tmp_path))
    for n in ("e2mi_x.f32", "e2mi_xn.f32", "e2mi_q16.f16", "e2mi_k16.f16", "e2mi_vt16.f16", "e2mi_ctx_q.i8",
              "e2mi_ctx_s.f32", "e2mi_tmp.f32", "e2mi_out.f32", "e2mi_pos.i32", "e2mi_rowmap.i32"):
        assert n in names, names
    assert np.array_equal(np.fromfile(tmp_path / "e2mi_out.f32", np.float32).reshape(3, 768), out)
    rowmap = np.fromfile(tmp_path / "e2mi_rowmap.i32", np.int32)
    pos = np.fromfile(tmp_path / "e2mi_pos.i32", np.int32)
    x = np.fromfile(tmp_path / "e2mi_x.f32", np.float32).reshape(len(rowmap), 768)
    live = rowmap >= 0
    assert np.array_equal(pos[live], rowmap[live] % 100)
    # the oracle's residual after layer 0, on the padded rows the packed rows come from
    om = oracle_model(oracle, m, n_layers=1)
    table = np.ascontiguousarray(m.tensor("language_model.embed_tokens.weight"), np.float32)
    x0 = table[ids.reshape(-1)] * np.float32(m.config.embed_scale)
    want = om.layer(0, x0, valid, 3, 100)
    a, b = x[live].astype(np.float64), want[rowmap[live]].astype(np.float64)
    cos = (a * b).sum(1) / (np.linalg.norm(a, axis=1) * np.linalg.norm(b, axis=1))
    # per row (before pooling) the f16 attention at logit scale 1.0 leaves a few rows near 0.9998
    assert cos.min() >= 0.999 and np.median(cos) >= 0.9999, (cos.min(), np.median(cos))
    # a second call does not dump again
    before = {n: os.path.getmtime(tmp_path / n) for n in names}
    eng.embed_batch(ids, valid)
    assert all(os.path.getmtime(tmp_path / n) == t for n, t in before.items())
