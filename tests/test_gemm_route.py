"""Which GEMM kernel a call takes (gemm_small_route, gemm_s.hip) and whether a projection and its norm_add
run as two launches (gemm_an_split, gemm_an.hip): host functions, so no GPU is needed. A kernel is offered only
where its LDS holds the K of the call, and no form where it was measured slower than another."""
import ctypes as C

import pytest

NONE, SK, S32, S64, RING = 0, 1, 2, 3, 5  # gemm_args.h
F32, I8Q, GEGLU, GELUMUL, QKV = range(5)
KLDS = 160 * 1024


@pytest.fixture(scope="module")
def route():
    import e2mi
    f = e2mi.load()._ZN4e2mi16gemm_small_routeEiiiib
    f.argtypes, f.restype = [C.c_int] * 4 + [C.c_bool], C.c_int
    return lambda M, N, K, epi=F32, tok=False: f(M, N, K, epi, tok)


@pytest.fixture(scope="module")
def split():
    """Whether a projection of N columns and its norm_add run as two launches (gemm_an.hip)."""
    import e2mi
    f = e2mi.load()._ZN4e2mi13gemm_an_splitEiii
    f.argtypes, f.restype = [C.c_int] * 3, C.c_bool
    return f


def _lds(r, epi, nb):
    """A route's LDS at nb blocks of K, from the kernels' own layouts."""
    if r == SK:
        return 8448 * nb
    if r == RING:
        return 72 * 1024 + 256 * nb + 512
    wide = epi in (GEGLU, QKV)  # 256-column tiles: 16 waves of 16 columns, or 8 of 32 in 64 rows
    nw, ru, cu = (16, 2, 1) if wide and r == S32 else (8, 4, 2) if wide else (8, 2, 1) if r == S32 else (8, 4, 1)
    ring = 4 if ru == 2 else 3
    return nb * ru * 2048 + nw * ring * cu * 2048 + nb * 256 + 64 * nw * cu + 64 * ru


@pytest.mark.parametrize("epi,tok", [(F32, False), (F32, True), (I8Q, False), (I8Q, True), (GEGLU, False),
                                     (GELUMUL, False), (QKV, False)])
def test_a_route_fits_the_lds(route, epi, tok):
    for K in (128, 768, 896, 1024, 1920, 2048, 2432, 2560, 4096, 4480, 4608, 16384, 44800, 44928, 65536):
        for M in (1, 33, 64, 300, 2048, 4096, 17408):
            for N in (256, 768, 2304):
                r = route(M, N, K, epi, tok)
                assert r == NONE or _lds(r, epi, K // 128) <= KLDS, (M, N, K, r)


def test_ring_ends_where_its_scales_fill_the_lds(route):
    assert route(64, 768, 44800) == RING  # 350 blocks: all of the 163,840 bytes
    assert route(64, 768, 44928) == NONE


# shapes at which the K-split tiles take longer than the large ones (short K over many rows), and calls
# of the same widths at which they are the fastest
@pytest.mark.parametrize("M,N,K", [(17408, 768, 128), (65536, 256, 128), (2000, 4608, 128), (262144, 40, 128),
                                   (5000, 1024, 256), (262144, 40, 384), (65536, 40, 512)])
def test_short_k_over_many_rows_takes_the_large_tiles(route, M, N, K):
    assert route(M, N, K) == NONE
    assert route(32, N, K) == SK


# both sides of the line, 512 and 768 columns, and the ends of K
@pytest.mark.parametrize("N,K,two,one", [(768, 768, (1, 768), (769, 17408)), (768, 1152, (1, 1152), (1153,)),
                                         (512, 512, (33, 512), (513,)), (512, 2048, (1, 2944), (2945, 17408)),
                                         (512, 4096, (1, 4096), (4200, 5000, 7000)), (512, 8192, (4096,), (5000,)),
                                         (768, 3840, (5000,), (6000,)), (768, 256, (100,), (257,)),
                                         (768, 128, (), (1, 64, 128)), (512, 256, (), (1, 100, 256))])
def test_two_launches_only_where_they_are_faster(split, N, K, two, one):
    assert all(split(r, N, K) for r in two)
    assert not any(split(r, N, K) for r in one)
