"""Which kernels a device-planned forward takes at an expected row count and a capacity (forward_signature,
forward.cpp, the key of its recording; a host function, so no GPU is needed). An octal digit leads (1-5: the
norm_add fused, in how many row units; 6: in the GEMM that reads it; 7: separate), then one for each distinct GEMM
(0, 4: gemm.hip's tiles; 1, 2, 3, 5: the kernels for few rows) and for the attention at each head_dim (32-, 64- or
128-query blocks as 1, 2, 0), then 8 bits for the fused projections that run as two launches."""
import ctypes as C

import pytest


@pytest.fixture(scope="module")
def kernels():
    import e2mi
    f = e2mi.load()._ZN4e2mi17forward_signatureERK9e2_configbbiiii
    f.argtypes, f.restype = [C.c_void_p, C.c_bool, C.c_bool] + [C.c_int] * 4, C.c_long
    cfg = {"base": e2mi.baseline_config(), "ref": e2mi.reference_config()}

    def of(geom, capacity, est, B=64, S=512):
        """norm_add and GEMMs, attention, two launches"""
        s = f(C.addressof(cfg[geom]), True, True, B, S, capacity, est)
        digits, n = oct(s >> 8)[2:], 1 if geom == "base" else 2
        return digits[:-n], digits[-n:], s & 255
    return of


@pytest.mark.parametrize("geom", ["base", "ref"])
def test_a_small_batch_far_below_capacity_takes_the_large_tiles(kernels, geom):
    """64 x 512 of capacity: the kernels for few rows would start 100 times the workgroups that find a row."""
    for est in (32, 256, 2048, 8192):
        gemms, attention, two = kernels(geom, 32768, est)
        assert gemms[0] in "1234" and set(gemms[1:]) <= {"0", "4"} and two == 0, (est, gemms)
        assert set(attention) == {"0"}


@pytest.mark.parametrize("geom", ["base", "ref"])
def test_near_capacity_the_choice_is_the_estimates(kernels, geom):
    for m in (256, 512, 1024, 2304, 4096):
        # (the row units and gemm.hip's tiles follow the estimate at any capacity)
        assert kernels(geom, m, m) == kernels(geom, min(2 * m, 32768), m), m
    assert kernels(geom, 512, 40)[0][0] == "6" and kernels(geom, 512, 300)[0][0] == "1"


def test_the_attentions_block_size_is_in_the_key(kernels):
    """16 x 512, BASELINE geometry: at the capacity and at a planned 4352 rows the GEMMs are the same, the attention
    runs in 128- and in 64-query blocks, so one recording cannot serve both; 8 x 512 likewise at 2048 and 2304."""
    full, planned = kernels("base", 8192, 8192, 16, 512), kernels("base", 8192, 4352, 16, 512)
    assert full[0] == planned[0] and (full[1], planned[1]) == ("0", "2")
    few, more = kernels("base", 4096, 2048, 8, 512), kernels("base", 4096, 2304, 8, 512)
    assert few[0] == more[0] and (few[1], more[1]) == ("1", "2")
    assert kernels("ref", 3072, 3072, 2, 1500)[1] == "22"
