"""The projection with the norm_add in its epilogue (e2mi_i8_gemm_add_norm_quant and
e2mi_i8_gemm_add_norm_scale_quant, gemm_an.hip) against the two launches each replaces,
e2mi_i8_gemm then e2mi_add_norm_quant / e2mi_add_norm_scale_quant (the encoder's O and down
projections and the norm_add after each, text.c:944-953; the reference checkpoint's 512-wide
projections and its PLE layers' scaled norm_add, text.c:955-961).

Up to a row count that follows K the entry points run the two launches themselves, through y or x_out
(gemm_an_split); the cases below that line with y test those, test_one_launch_at_few_rows the kernel there.

Bars: every output bit-identical with the two launches (the same per-128 fold, the same row
arithmetic), which test_gpu_gemm.py and test_gpu_rowops.py pin to the oracle; the projection y also
bit-exact with the oracle's GEMM directly on a small case. Row counts cover one 16-row unit, ragged
last units, fewer units than CUs, one to five units per workgroup and several chunks per workgroup;
K = 768 (O) and 1152 (down); 512-wide rows at K = 512 to 2048, plain and scaled."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu
EPS = 1e-6
D = 768


def _t(a, dev):
    import torch
    return torch.from_numpy(np.ascontiguousarray(a)).to(dev)


def _np(t):
    return t.cpu().numpy()


def _case(rng, M, K, N=D):
    qa = rng.integers(-127, 128, (M, K), dtype=np.int8)
    as_ = rng.uniform(0.001, 0.05, (M, K // 128)).astype(np.float32)
    w = rng.integers(-127, 128, (N, K), dtype=np.int8)
    ws = rng.uniform(0.001, 0.02, N).astype(np.float32)
    res = rng.standard_normal((M, N)).astype(np.float32)
    ga = (1 + 0.05 * rng.standard_normal(N)).astype(np.float32)
    gn = (1 + 0.05 * rng.standard_normal(N)).astype(np.float32)
    return qa, as_, w, ws, res, ga, gn


def _same(a, b, what):
    a, b = _np(a), _np(b)
    assert a.shape == b.shape, what
    bad = np.flatnonzero(a.reshape(-1).view(np.uint8 if a.dtype == np.int8 else np.uint32) !=
                         b.reshape(-1).view(np.uint8 if b.dtype == np.int8 else np.uint32))
    assert bad.size == 0, f"{what}: {bad.size} elements differ, first at {np.unravel_index(bad[0], a.shape)}"


def _both(gpu, rng, M, K, gamma_next=True, want_xn=True, quant=True, inplace=False, N=D, post_scale=None):
    """post_scale None: the plain norm_add; else the scaled one (x itself quantized without gamma_next)"""
    import e2mi
    qa, as_, w, ws, res, ga, gn = _case(rng, M, K, N)
    W = e2mi.DeviceWeight.from_rowmajor(w, ws)
    tqa, tas, tga = _t(qa, gpu), _t(as_, gpu), _t(ga, gpu)
    tgn = _t(gn, gpu) if gamma_next else None
    # the two launches
    y0 = e2mi.i8_gemm(tqa, tas, W)
    r0 = _t(res, gpu)
    if post_scale is None:
        x0, xn0, q0, qs0 = e2mi.add_norm_quant(y0, r0, tga, tgn, EPS, x_out=r0 if inplace else None,
                                               want_xn=want_xn, quant=quant)
    else:
        x0, xn0, q0, qs0 = e2mi.add_norm_scale_quant(y0, r0, tga, post_scale, tgn, EPS,
                                                     x_out=r0 if inplace else None, want_xn=want_xn, quant=quant)
    # the fused one
    r1 = _t(res, gpu)
    if post_scale is None:
        x1, xn1, q1, qs1, y1 = e2mi.i8_gemm_add_norm_quant(tqa, tas, W, r1, tga, tgn, EPS,
                                                           x_out=r1 if inplace else None, want_xn=want_xn,
                                                           quant=quant, want_y=True)
    else:
        x1, xn1, q1, qs1, y1 = e2mi.i8_gemm_add_norm_scale_quant(tqa, tas, W, r1, tga, post_scale, tgn, EPS,
                                                                 x_out=r1 if inplace else None, want_xn=want_xn,
                                                                 quant=quant, want_y=True)
    _same(y1, y0, "y")
    _same(x1, x0, "x")
    if gamma_next and want_xn:
        _same(xn1, xn0, "xn")
    if quant and (gamma_next or post_scale is not None):
        _same(q1, q0, "q")
        _same(qs1, qs0, "qs")
    return qa, as_, w, ws, y1


@pytest.mark.parametrize("M,K", [(1, 768), (16, 768), (50, 1152), (333, 768), (1000, 1152), (4100, 768),
                                 (17408, 768), (17408, 1152), (17264, 768), (44000, 768)])
def test_fused_equals_two_launches(gpu, rng, M, K):
    _both(gpu, rng, M, K)


@pytest.mark.parametrize("variant", ["x_only", "no_xn", "no_q", "inplace"])
def test_fused_output_variants(gpu, rng, variant):
    kw = {"x_only": dict(gamma_next=False), "no_xn": dict(want_xn=False), "no_q": dict(quant=False),
          "inplace": dict(inplace=True)}[variant]
    _both(gpu, rng, 2100, 768, **kw)


@pytest.mark.parametrize("M,K", [(1, 512), (50, 1024), (2100, 2048), (17408, 1024), (17408, 2048)])
def test_fused_512_equals_two_launches(gpu, rng, M, K):
    _both(gpu, rng, M, K, N=512)


@pytest.mark.parametrize("M,K,gamma_next", [(333, 2048, False), (17408, 2048, False), (17408, 512, True),
                                            (5, 512, True)])
def test_fused_scaled_equals_two_launches(gpu, rng, M, K, gamma_next):
    """the PLE layers' norm_adds: after the down projection x itself quantized (scale 1), after the
    PLE projection scaled by the layer scalar and normed for the next layer"""
    _both(gpu, rng, M, K, N=512, gamma_next=gamma_next, post_scale=1.0 if not gamma_next else 0.7373)
    _both(gpu, rng, 300, K, N=512, gamma_next=gamma_next, post_scale=0.2, inplace=True)


def _raw(gpu, case, **over):
    """The entry point on buffers of the caller's choice: the outputs that were asked for, by name."""
    import torch
    import e2mi
    qa, as_, w, ws, res, ga, gn = case
    M, K, N = *qa.shape, w.shape[0]
    W = over.pop("W", None) or e2mi.DeviceWeight.from_rowmajor(w, ws)
    b = dict(qa=_t(qa, gpu), as_=_t(as_, gpu), res=_t(res, gpu), x=torch.empty((M, N), device=gpu), xn=None, y=None,
             q=torch.empty((M, N), dtype=torch.int8, device=gpu), qs=torch.empty((M, N // 128), device=gpu))
    for k, v in over.items():
        b[k] = v(b)
    p = lambda t: None if t is None else t.data_ptr()
    tga, tgn = _t(ga, gpu), _t(gn, gpu)
    e2mi.check(e2mi.load().e2mi_i8_gemm_add_norm_quant(
        torch.cuda.current_stream().cuda_stream, p(b["qa"]), p(b["as_"]), W.ref, M, p(b["res"]), p(tga), p(tgn),
        EPS, p(b["x"]), p(b["xn"]), p(b["q"]), p(b["qs"]), p(b["y"])))
    torch.cuda.synchronize()
    return b


def _split(M, N, K):
    import ctypes as C
    import e2mi
    f = e2mi.load()._ZN4e2mi13gemm_an_splitEiii
    f.argtypes, f.restype = [C.c_int] * 3, C.c_bool
    return f(M, N, K)


@pytest.mark.parametrize("M,K,N,scale,kw", [
    (1, 768, 768, None, {}), (16, 768, 768, None, {}), (17, 1152, 768, None, {}), (333, 768, 768, None, {}),
    (1000, 1152, 768, None, {}), (50, 768, 768, None, dict(gamma_next=False)), (50, 768, 768, None, dict(want_xn=False)),
    (50, 768, 768, None, dict(quant=False)), (1, 512, 512, None, {}), (50, 1024, 512, None, {}), (2100, 2048, 512, None, {}),
    (5, 512, 512, 0.7373, {}), (333, 2048, 512, 1.0, dict(gamma_next=False)), (300, 512, 512, 0.2, dict(want_xn=False))])
def test_one_launch_at_few_rows(gpu, rng, M, K, N, scale, kw):
    """k_gemm_an where a call with y runs as two launches: x updated in the residual's place and no y leaves the
    entry point no scratch. Every output against the GEMM and the row kernel called one after the other."""
    import e2mi
    assert _split(M, N, K)
    kw = dict(kw)
    qa, as_, w, ws, res, ga, gn = _case(rng, M, K, N)
    W = e2mi.DeviceWeight.from_rowmajor(w, ws)
    tqa, tas, tga = _t(qa, gpu), _t(as_, gpu), _t(ga, gpu)
    tgn = _t(gn, gpu) if kw.pop("gamma_next", True) else None
    kw = dict(dict(want_xn=True, quant=True), **kw)
    r0, r1 = _t(res, gpu), _t(res, gpu)
    y = e2mi.i8_gemm(tqa, tas, W)
    if scale is None:
        want = e2mi.add_norm_quant(y, r0, tga, tgn, EPS, x_out=r0, **kw)
        got = e2mi.i8_gemm_add_norm_quant(tqa, tas, W, r1, tga, tgn, EPS, x_out=r1, **kw)
    else:
        want = e2mi.add_norm_scale_quant(y, r0, tga, scale, tgn, EPS, x_out=r0, **kw)
        got = e2mi.i8_gemm_add_norm_scale_quant(tqa, tas, W, r1, tga, scale, tgn, EPS, x_out=r1, **kw)
    for name, a, b in zip(("x", "xn", "q", "qs"), got, want):
        assert (a is None) == (b is None), name
        if a is not None:
            _same(a, b, name)


@pytest.mark.parametrize("M", [7, 333, 2100])  # two launches, then one
def test_normed_rows_over_the_residual(gpu, rng, M):
    """xn_out in the residual's place (the engine's last norm_add at few rows): a row's residual is read before
    its normed row is written."""
    import torch
    import e2mi
    case = _case(rng, M, 768)
    want = _raw(gpu, case, xn=lambda b: torch.empty_like(b["res"]))
    for over in (dict(xn=lambda b: b["res"]), dict(x=lambda b: torch.empty_like(b["res"]), y=lambda b: torch.empty_like(b["res"]),
                                                   xn=lambda b: b["res"])):
        got = _raw(gpu, case, **over)
        for k in ("x", "xn", "q", "qs"):
            _same(got[k], want[k], k)


@pytest.mark.parametrize("M", [7, 333])
def test_fused_over_its_inputs(gpu, rng, M):
    """Outputs on the inputs' own memory at row counts that take two launches: y in the residual's place
    (with x apart from it) is still the projection, and a call whose x lies in the activations' memory
    (one workgroup's rows) is still computed from them."""
    import torch
    case = _case(rng, M, 768)
    want = _raw(gpu, case, y=lambda b: torch.empty_like(b["res"]))
    got = _raw(gpu, case, y=lambda b: b["res"])
    for k in ("x", "y", "q", "qs"):
        _same(got[k], want[k], f"y over res: {k}")
    if M <= 16:
        got = _raw(gpu, case, qa=lambda b: torch.cat([b["qa"].view(-1), torch.zeros(3 * M * D, dtype=torch.int8,
                                                                                   device=gpu)]).view(4 * M, D),
                   x=lambda b: b["qa"].view(torch.float32).view(M, D))
        for k in ("x", "q", "qs"):
            _same(got[k], want[k], f"x over qa: {k}")


@pytest.mark.parametrize("M", [7, 333, 2100])
def test_fused_weight_on_4_bytes(gpu, rng, M):
    """k_gemm_an loads 16 bytes from any 4-byte address; the GEMM of the two launches asks for 16-byte
    ones, so such a weight (a caller's own e2mi_q8w) keeps the one launch at every row count."""
    import ctypes as C
    import torch
    import e2mi
    case = _case(rng, M, 768)
    want = _raw(gpu, case)
    w, ws = case[2], case[3]
    buf = torch.zeros(w.size + 16, dtype=torch.int8, device=gpu)
    buf[4:4 + w.size] = _t(w, gpu).view(-1)
    tws = _t(ws, gpu)

    class Own:
        q = e2mi.Q8W(w=buf.data_ptr() + 4, scale=tws.data_ptr(), N=D, K=768, ld=768, out_min=-1e31, out_max=1e31)
        ref = C.byref(q)
    got = _raw(gpu, case, W=Own)
    for k in ("x", "q", "qs"):
        _same(got[k], want[k], k)


def test_fused_fast_fold(gpu, rng):
    import e2mi
    prev = e2mi.load().e2mi_gemm_set_fold(1)
    try:
        _both(gpu, rng, 3000, 1152)
    finally:
        e2mi.load().e2mi_gemm_set_fold(prev)


def test_fused_projection_vs_oracle(gpu, oracle, rng):
    qa, as_, w, ws, y = _both(gpu, rng, 96, 1152)
    yo = oracle.i8_gemm(qa, as_, w, ws)
    assert np.array_equal(_np(y).view(np.uint32), np.asarray(yo, np.float32).view(np.uint32))


def test_fused_refuses(gpu, rng):
    import e2mi
    qa, as_, w, ws, res, ga, gn = _case(rng, 64, 768)
    Wb = e2mi.DeviceWeight.from_rowmajor(w, ws, bias=np.zeros(D, np.float32))
    with pytest.raises(RuntimeError, match="bias"):
        e2mi.i8_gemm_add_norm_quant(_t(qa, gpu), _t(as_, gpu), Wb, _t(res, gpu), _t(ga, gpu), _t(gn, gpu))
    W2 = e2mi.DeviceWeight.from_rowmajor(np.zeros((256, 768), np.int8), np.ones(256, np.float32))
    with pytest.raises(RuntimeError, match="N = 512 or 768"):
        e2mi.i8_gemm_add_norm_quant(_t(qa, gpu), _t(as_, gpu), W2, _t(res[:, :256], gpu), _t(ga[:256], gpu),
                                    _t(gn[:256], gpu))
    W7 = e2mi.DeviceWeight.from_rowmajor(w, ws)
    with pytest.raises(RuntimeError, match="512-wide"):
        e2mi.i8_gemm_add_norm_scale_quant(_t(qa, gpu), _t(as_, gpu), W7, _t(res, gpu), _t(ga, gpu), 1.0, None)


def test_engine_fused_equals_unfused(gpu, rng, monkeypatch):
    """The engine with the fused O/down + norm_add launches (default) against E2MI_NOFUSE_AN=1 (the
    GEMM, then the row kernel): the same embeddings bit for bit, through the host entry (packed and
    padded rows) and the device entry (planned on the device: the kernel reads the device row
    count and its row ranges follow it, over batches of several row counts)."""
    import sys
    import torch
    sys.path.insert(0, __file__.rsplit("/", 1)[0])
    from model_util import random_batch, small_config
    import e2mi
    m = e2mi.Model.synthetic(small_config(e2mi, n_layers=2), 77)
    fused = e2mi.Engine(m, max_rows=32768)
    monkeypatch.setenv("E2MI_NOFUSE_AN", "1")
    plain = e2mi.Engine(m, max_rows=32768)
    monkeypatch.delenv("E2MI_NOFUSE_AN")
    # the last batch has more rows than one round of the CUs covers: the engine runs the separate
    # kernels there (both entries)
    for B, S, lo in [(4, 128, 40), (9, 300, 1), (16, 256, 200), (2, 512, 500), (50, 512, 480)]:
        ids, valid = random_batch(rng, B, S, 1000, min_len=lo)
        a, b = fused.embed_batch(ids, valid), plain.embed_batch(ids, valid)
        assert np.array_equal(a.view(np.uint32), b.view(np.uint32)), (B, S)
        tid, tv = torch.from_numpy(ids).to(gpu), torch.from_numpy(valid).to(gpu)
        oa = torch.empty((B, 768), device=gpu)
        ob = torch.empty((B, 768), device=gpu)
        fused.embed_batch_device(tid, tv, oa)
        plain.embed_batch_device(tid, tv, ob)
        torch.cuda.synchronize()
        assert np.array_equal(_np(oa).view(np.uint32), a.view(np.uint32)), (B, S, "device entry")
        assert np.array_equal(_np(ob).view(np.uint32), a.view(np.uint32)), (B, S, "device entry, unfused")
    for e in (fused, plain):
        e.set_packing(False)
    ids, valid = random_batch(rng, 5, 200, 1000, min_len=20)
    a, b = fused.embed_batch(ids, valid), plain.embed_batch(ids, valid)
    assert np.array_equal(a.view(np.uint32), b.view(np.uint32)), "padded rows"


def test_engine_fused_equals_unfused_reference_geometry(gpu, rng, monkeypatch):
    """The reference checkpoint's geometry (hidden 512, PLE, window, a head_dim-512 layer): the O,
    down and PLE projections with their norm_adds fused (the down's quantizing x itself, the PLE
    projection's scaled by the layer scalar) give the same embeddings bit for bit as
    E2MI_NOFUSE_AN=1, through the host and the device entry."""
    import sys
    import torch
    sys.path.insert(0, __file__.rsplit("/", 1)[0])
    from model_util import random_batch, reference_small_config
    import e2mi
    m = e2mi.Model.synthetic(reference_small_config(e2mi, n_layers=6), 78)
    fused = e2mi.Engine(m, max_rows=4096)
    monkeypatch.setenv("E2MI_NOFUSE_AN", "1")
    plain = e2mi.Engine(m, max_rows=4096)
    monkeypatch.delenv("E2MI_NOFUSE_AN")
    for B, S, lo in [(4, 256, 60), (3, 1024, 600), (16, 128, 1)]:
        ids, valid = random_batch(rng, B, S, 1000, min_len=lo)
        a, b = fused.embed_batch(ids, valid), plain.embed_batch(ids, valid)
        assert a.shape == (B, 768)
        assert np.array_equal(a.view(np.uint32), b.view(np.uint32)), (B, S)
        tid, tv = torch.from_numpy(ids).to(gpu), torch.from_numpy(valid).to(gpu)
        oa = torch.empty((B, 768), device=gpu)
        fused.embed_batch_device(tid, tv, oa)
        torch.cuda.synchronize()
        assert np.array_equal(_np(oa).view(np.uint32), a.view(np.uint32)), (B, S, "device entry")


@pytest.mark.parametrize("geom", ["base", "ref"])
@pytest.mark.parametrize("fold", ["exact", "fast"])
def test_engine_at_few_rows_equals_unfused(gpu, rng, monkeypatch, geom, fold):
    """Up to 256 rows the engine runs each norm_add in the GEMM that reads it, x moving between two buffers: the
    same embeddings bit for bit as E2MI_NOFUSE_AN=1, through the host and the device entry, at the edges of
    the 32-row tiles and of the form, with both folds and with every layer as the last."""
    import sys
    import torch
    sys.path.insert(0, __file__.rsplit("/", 1)[0])
    from model_util import random_batch, reference_small_config, small_config
    import e2mi
    layers = 3 if geom == "base" else 7
    cfg = small_config(e2mi, n_layers=layers) if geom == "base" else reference_small_config(e2mi, n_layers=layers)
    m = e2mi.Model.synthetic(cfg, 80)
    prev = e2mi.set_gemm_fold(fold)
    try:
        ahead = e2mi.Engine(m, max_rows=2048)
        monkeypatch.setenv("E2MI_NOFUSE_AN", "1")
        plain = e2mi.Engine(m, max_rows=2048)
        monkeypatch.delenv("E2MI_NOFUSE_AN")
        for B, S in [(1, 1), (1, 8), (1, 19), (1, 33), (1, 100), (3, 64), (1, 256), (1, 257), (8, 32)]:
            ids, valid = random_batch(rng, B, S, 1000, min_len=S if B == 1 else 1)
            a, b = ahead.embed_batch(ids, valid), plain.embed_batch(ids, valid)
            assert np.array_equal(a.view(np.uint32), b.view(np.uint32)), (B, S)
            out = torch.empty((B, 768), device=gpu)
            ahead.embed_batch_device(torch.from_numpy(ids).to(gpu), torch.from_numpy(valid).to(gpu), out)
            torch.cuda.synchronize()
            assert np.array_equal(_np(out).view(np.uint32), a.view(np.uint32)), (B, S, "device entry")
        ids = rng.integers(0, 1000, (1, 50)).astype(np.int32)
        for n in range(1, layers + 1):
            ahead.set_layer_limit(n)
            plain.set_layer_limit(n)
            assert np.array_equal(ahead.embed_batch(ids, None), plain.embed_batch(ids, None)), n
    finally:
        e2mi.set_gemm_fold(prev)
