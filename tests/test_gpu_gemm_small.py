"""The GEMM kernels for few rows (gemm_s.hip): every epilogue at row counts on the edges of its 32- and
64-row tiles and of the rounds where one kernel hands over to the next, against the first rows of a
call large enough for the 128- and 256-row tiles. All these GEMMs are row-local, so the bar is equal
bits; the plain one is also held to the oracle's GEMM bit for bit, and rows past the count stay as
they were."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu
BIG = 17408  # rows the large tiles take at every width here but (K, N) = (128, 40), which the oracle covers


def _t(a, dev):
    import torch
    return torch.from_numpy(np.ascontiguousarray(a)).to(dev)


def _ops(rng, gpu, K, N, bias=False):
    import e2mi
    w = rng.integers(-127, 128, (N, K), dtype=np.int8)
    ws = rng.uniform(0.001, 0.02, N).astype(np.float32)
    b = (0.1 * rng.standard_normal(N)).astype(np.float32) if bias else None
    import torch
    g = torch.Generator(device=gpu).manual_seed(7)
    qa = torch.randint(-127, 128, (BIG, K), generator=g, device=gpu, dtype=torch.int8)
    as_ = torch.rand((BIG, K // 128), generator=g, device=gpu) * 0.05 + 0.001
    return qa, as_, w, ws, b, e2mi.DeviceWeight.from_rowmajor(w, ws, bias=b)


def _same(got, want, what):
    import torch
    for i, (a, b) in enumerate(zip(got, want)):
        if b is None:
            continue
        v = {1: torch.int8, 2: torch.int16, 4: torch.int32}[a.element_size()]
        assert torch.equal(a.contiguous().view(v), b.contiguous().view(v)), f"{what}: output {i}"


# (K, N): K-split tiles up to 19 blocks, one and two workgroups a CU, an N that ends inside a tile
@pytest.mark.parametrize("K,N,bias", [(128, 40, True), (768, 768, False), (768, 1156, True), (1152, 800, True),
                                      (2048, 512, False), (3072, 256, False)])
def test_small_f32(gpu, oracle, rng, K, N, bias):
    import e2mi
    import torch
    qa, as_, w, ws, b, W = _ops(rng, gpu, K, N, bias)
    full = e2mi.i8_gemm(qa, as_, W)
    for M in (1, 31, 33, 64, 65, 513, 1030, 2050, 4100):
        y = torch.full((M + 1, N), 7.0, device=gpu)
        e2mi.i8_gemm(qa[:M], as_[:M], W, y=y)
        _same([y[:M]], [full[:M]], f"M={M}")
        assert bool((y[M] == 7.0).all()), f"M={M}: a row past the count was written"
    n = qa[:65].cpu().numpy(), as_[:65].cpu().numpy()
    want = oracle.i8_gemm(n[0], n[1], w, ws, bias=b)
    assert np.array_equal(full[:65].cpu().numpy().view(np.uint32), want.view(np.uint32))


def test_small_f32_column_range_clamp_and_fast_fold(gpu, rng):
    import e2mi
    import torch
    qa, as_, w, ws, b, W = _ops(rng, gpu, 768, 520, True)
    W.set_clamp(-1.5, 2.0)
    for mode in ("exact", "fast"):
        prev = e2mi.set_gemm_fold(mode)
        try:
            full = e2mi.i8_gemm(qa, as_, W, n0=33, n1=501)
            for M in (5, 129, 1500):
                y = e2mi.i8_gemm(qa[:M], as_[:M], W, n0=33, n1=501)
                _same([y], [full[:M]], f"{mode} M={M}")
                assert bool((y[:, :33] == 0).all() and (y[:, 501:] == 0).all())
        finally:
            e2mi.set_gemm_fold(prev)


@pytest.mark.parametrize("K,N", [(512, 512), (768, 1152), (1152, 768)])
def test_small_requant_and_per_token(gpu, rng, K, N):
    import e2mi
    qa, as_, w, ws, b, W = _ops(rng, gpu, K, N)
    at = as_[:, 0].contiguous()
    q, t, tq = e2mi.i8_gemm_q(qa, as_, W), e2mi.i8_gemm_tok(qa, at, W), e2mi.i8_gemm_tok_q(qa, at, W)
    for M in (1, 33, 250, 1030, 2050, 4100):
        _same(e2mi.i8_gemm_q(qa[:M], as_[:M], W), [o[:M] for o in q], f"q M={M}")
        _same([e2mi.i8_gemm_tok(qa[:M], at[:M], W)], [t[:M]], f"tok M={M}")
        _same(e2mi.i8_gemm_tok_q(qa[:M], at[:M], W), [o[:M] for o in tq], f"tok_q M={M}")


@pytest.mark.parametrize("hidden,ffn", [(768, 1152), (512, 2048), (128, 128)])
def test_small_geglu_and_gelu_mul(gpu, rng, hidden, ffn):
    import e2mi
    import torch
    qa, as_, w, ws, b, W = _ops(rng, gpu, hidden, 2 * ffn)
    _, _, _, _, _, Wg = _ops(rng, gpu, hidden, hidden)
    mul = torch.randn((BIG, 3 * hidden), generator=torch.Generator(device=gpu).manual_seed(9), device=gpu)[:, hidden:2 * hidden]
    full, gate = e2mi.i8_gemm_geglu(qa, as_, W), e2mi.i8_gemm_gelu_mul(qa, as_, Wg, mul)
    for M in (1, 32, 33, 65, 513, 897, 1793, 2049, 4100):
        for g in (True, False):
            _same(e2mi.i8_gemm_geglu(qa[:M], as_[:M], W, want_g=g)[:3 if g else 2], [o[:M] for o in full], f"geglu M={M}")
        _same(e2mi.i8_gemm_gelu_mul(qa[:M], as_[:M], Wg, mul[:M]), [o[:M] for o in gate], f"gelu_mul M={M}")


@pytest.mark.parametrize("K,H,KV", [(768, 3, 1), (512, 4, 2)])
def test_small_qkv(gpu, rng, K, H, KV):
    import e2mi
    import torch
    qa, as_, w, ws, b, W = _ops(rng, gpu, K, (H + 2 * KV) * 256)
    g = torch.Generator(device=gpu).manual_seed(11)
    qg, kg = (torch.rand(256, generator=g, device=gpu) + 0.5 for _ in range(2))
    cs, sn = (torch.rand((2048, 256), generator=g, device=gpu) for _ in range(2))
    pos = torch.randint(0, 2048, (BIG,), generator=g, device=gpu, dtype=torch.int32)
    full = e2mi.i8_gemm_qkv(qa, as_, W, H, KV, qg, kg, cs, sn, pos=pos, want_f32=True)
    for M in (1, 33, 64, 520, 1632, 1664, 2200):  # V^T rows of odd, even and 16-byte pitch
        got = e2mi.i8_gemm_qkv(qa[:M], as_[:M], W, H, KV, qg, kg, cs, sn, pos=pos[:M].contiguous(), want_f32=True)
        want = [o[:M] for o in full]
        want[2] = full[2][..., :M]
        _same(got, want, f"packed M={M}")
    S = 34  # padded: positions m % S, V^T per sequence
    big = e2mi.i8_gemm_qkv(qa[:S * 512], as_[:S * 512], W, H, KV, qg, kg, cs, sn, S=S, want_f32=True)
    got = e2mi.i8_gemm_qkv(qa[:S * 3], as_[:S * 3], W, H, KV, qg, kg, cs, sn, S=S, want_f32=True)
    _same(got, [o[:3] if i == 2 else o[:3 * S] for i, o in enumerate(big)], "padded")


@pytest.mark.parametrize("K,N,scale", [(768, 768, None), (1152, 768, None), (2048, 512, None), (512, 512, 0.7)])
def test_small_add_norm(gpu, rng, K, N, scale):
    """Two launches at few rows (the residual beside x_out), k_gemm_an with x updated in place."""
    import e2mi
    import torch
    qa, as_, w, ws, b, W = _ops(rng, gpu, K, N)
    g = torch.Generator(device=gpu).manual_seed(13)
    res = torch.randn((2100, N), generator=g, device=gpu)
    ga, gn = (torch.rand(N, generator=g, device=gpu) + 0.5 for _ in range(2))

    def call(M, **kw):
        if scale is None:
            return e2mi.i8_gemm_add_norm_quant(qa[:M], as_[:M], W, kw.pop("res"), ga, gn, **kw)
        return e2mi.i8_gemm_add_norm_scale_quant(qa[:M], as_[:M], W, kw.pop("res"), ga, scale, kw.pop("gn", gn), **kw)

    for M in (1, 33, 1365, 2050):
        r = res[:M].clone()
        want = call(M, res=r, x_out=r)
        _same(call(M, res=res[:M])[:4], want[:4], f"M={M}")
        y = e2mi.i8_gemm(qa[:M], as_[:M], W)
        _same(call(M, res=res[:M], want_y=True), [*want[:4], y], f"with y, M={M}")
    if scale is not None:  # without the next norm: x itself quantized
        r = res[:200].clone()
        want = call(200, res=r, x_out=r, gn=None)
        _same([o for o in call(200, res=res[:200], gn=None) if o is not None], [o for o in want if o is not None], "x")
    qa2 = as_.clone()
    qa2[3] = float("nan")  # a row of NaN scales: the same bytes on both forms
    r = res[:8].clone()
    f = e2mi.i8_gemm_add_norm_quant
    want = f(qa[:8], qa2[:8].contiguous(), W, r, ga, gn, x_out=r)
    got = f(qa[:8], qa2[:8].contiguous(), W, res[:8], ga, gn)
    _same(got[2:4], want[2:4], "NaN row")


# k_gemm_ring (64 x 128 tiles): odd and even block counts, rows at its tiles' edges
# and at one and two workgroups a CU, an N inside a tile, bias, clamp, column range and both folds; the large call of
# each shape is gemm.hip's
@pytest.mark.parametrize("K,N,rows", [(3072, 256, (1, 63, 64, 65, 300)), (2944, 520, (257, 1000)), (3072, 768, (2520, 2731, 4096)),
                                      (2048, 512, (2520, 4096, 8192)), (1152, 768, (2048, 2730, 2731)),
                                      (896, 768, (2500, 2520))])
def test_ring_f32(gpu, oracle, rng, K, N, rows):
    import e2mi
    import torch
    qa, as_, w, ws, b, W = _ops(rng, gpu, K, N, True)
    for mode in ("exact", "fast"):
        prev = e2mi.set_gemm_fold(mode)
        try:
            W.set_clamp(-3e38, 3e38)
            full = e2mi.i8_gemm(qa, as_, W)
            for M in rows:
                y = torch.full((M + 1, N), 7.0, device=gpu)
                e2mi.i8_gemm(qa[:M], as_[:M], W, y=y)
                _same([y[:M]], [full[:M]], f"{mode} M={M}")
                assert bool((y[M] == 7.0).all()), f"{mode} M={M}: a row past the count was written"
            if mode == "exact":
                want = oracle.i8_gemm(qa[:65].cpu().numpy(), as_[:65].cpu().numpy(), w, ws, bias=b)
                assert np.array_equal(full[:65].cpu().numpy().view(np.uint32), want.view(np.uint32))
            W.set_clamp(-1.5, 2.0)
            full = e2mi.i8_gemm(qa, as_, W, n0=33, n1=N - 19)
            for M in rows:
                y = e2mi.i8_gemm(qa[:M], as_[:M], W, n0=33, n1=N - 19)
                _same([y], [full[:M]], f"{mode} M={M}, clamped columns")
        finally:
            e2mi.set_gemm_fold(prev)


def _route(M, N, K, epi=0, tok=False):
    import ctypes as C
    import e2mi
    f = e2mi.load()._ZN4e2mi16gemm_small_routeEiiiib
    f.argtypes, f.restype = [C.c_int] * 4 + [C.c_bool], C.c_int
    return f(M, N, K, epi, tok)


# every f32 kernel by the rule's own word (0: gemm.hip's tiles; K-split, 32 rows, 64 rows, ring), all rows against
# the oracle bit for bit; the 64-row ones under the fast fold against the large tiles too
@pytest.mark.parametrize("route,K,N,M", [(1, 128, 40, 513), (1, 128, 40, 4100), (1, 768, 768, 1030), (2, 2560, 512, 257),
                                         (2, 2048, 256, 2048), (3, 384, 768, 2400), (3, 384, 256, 8149), (3, 512, 1024, 1921),
                                         (5, 2048, 512, 4096), (0, 384, 768, 6000)])
def test_f32_routes_against_the_oracle(gpu, oracle, rng, route, K, N, M):
    import e2mi
    assert _route(M, N, K) == route
    qa, as_, w, ws, b, W = _ops(rng, gpu, K, N, True)
    y = e2mi.i8_gemm(qa[:M], as_[:M], W)
    want = oracle.i8_gemm(qa[:M].cpu().numpy(), as_[:M].cpu().numpy(), w, ws, bias=b)
    assert np.array_equal(y.cpu().numpy().view(np.uint32), want.view(np.uint32))
    if route == 3:
        assert _route(BIG, N, K) == 0
        prev = e2mi.set_gemm_fold("fast")
        try:
            _same([e2mi.i8_gemm(qa[:M], as_[:M], W)], [e2mi.i8_gemm(qa, as_, W)[:M]], "fast fold")
        finally:
            e2mi.set_gemm_fold(prev)


@pytest.mark.parametrize("M", [33, 1664])  # 32- and 64-row tiles
def test_small_epilogues_under_the_fast_fold(gpu, rng, M):
    import e2mi
    import torch
    K, H, KV = 768, 4, 2
    N = (H + 2 * KV) * 256
    qa, as_, w, ws, b, W = _ops(rng, gpu, K, N)
    _, _, _, _, _, Wk = _ops(rng, gpu, K, K)
    g = torch.Generator(device=gpu).manual_seed(17)
    mul = torch.randn((BIG, K), generator=g, device=gpu)
    qg, kg = (torch.rand(256, generator=g, device=gpu) + 0.5 for _ in range(2))
    cs, sn = (torch.rand((64, 256), generator=g, device=gpu) for _ in range(2))
    pos = torch.randint(0, 64, (BIG,), generator=g, device=gpu, dtype=torch.int32)
    for epi, n in ((1, K), (2, N), (3, K), (4, N)):
        assert _route(M, n, K, epi) != 0 and _route(BIG, n, K, epi) == 0, epi

    def run(m):
        qkv = e2mi.i8_gemm_qkv(qa[:m], as_[:m], W, H, KV, qg, kg, cs, sn, pos=pos[:m].contiguous(), want_f32=True)
        return [*e2mi.i8_gemm_q(qa[:m], as_[:m], Wk), *e2mi.i8_gemm_geglu(qa[:m], as_[:m], W),
                *e2mi.i8_gemm_gelu_mul(qa[:m], as_[:m], Wk, mul[:m]), *qkv]

    exact = run(M)
    prev = e2mi.set_gemm_fold("fast")
    try:
        few, big = run(M), run(BIG)
    finally:
        e2mi.set_gemm_fold(prev)
    _same(few, [o[..., :M] if o.dim() == 4 else o[:M] for o in big], "fast fold")  # (V^T: [1][KV][D][M])
    assert any(not torch.equal(a, b) for a, b in zip(few, exact))  # (the mode was on)


@pytest.mark.parametrize("K", [44800, 44928])  # the last K whose scales fit k_gemm_ring's LDS, and the next
def test_long_k(gpu, oracle, rng, K):
    import e2mi
    M, N = 67, 72
    qa = rng.integers(-127, 128, (M, K), dtype=np.int8)
    as_ = rng.uniform(0.001, 0.05, (M, K // 128)).astype(np.float32)
    w = rng.integers(-127, 128, (N, K), dtype=np.int8)
    ws = rng.uniform(0.001, 0.02, N).astype(np.float32)
    y = e2mi.i8_gemm(_t(qa, gpu), _t(as_, gpu), e2mi.DeviceWeight.from_rowmajor(w, ws))
    assert np.array_equal(y.cpu().numpy().view(np.uint32), oracle.i8_gemm(qa, as_, w, ws).view(np.uint32))
