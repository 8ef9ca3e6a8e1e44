"""The query block size of the packed attention (attn_group_blocks, attn.hip; a host function, so no GPU is
needed): 32 (1), 64 (2) or 128 (0) queries by the blocks that the call has."""
import ctypes as C

import pytest


@pytest.fixture(scope="module")
def blocks():
    import e2mi
    f = e2mi.load()._ZN4e2mi17attn_group_blocksEiiiiib
    f.argtypes, f.restype = [C.c_int] * 5 + [C.c_bool], C.c_int
    return f


# rows, sequences, longest, heads, head_dim -> with a work list, without one (every sequence's grid is the
# longest one's)
@pytest.mark.parametrize("shape,listed,grid", [((768, 2, 300, 3, 256), 1, 1), ((2304, 8, 512, 3, 256), 2, 2),
                                               ((4352, 12, 512, 3, 256), 2, 0), ((4352, 16, 512, 3, 256), 2, 0),
                                               ((10496, 40, 512, 1, 256), 2, 0), ((10240, 32, 512, 3, 256), 0, 0),
                                               ((256, 1, 64, 3, 256), 0, 0), ((2048, 1, 2048, 4, 512), 2, 1),
                                               # measured slower in 64-query blocks, then in 32-query ones
                                               ((4352, 32, 142, 3, 256), 0, 0), ((3584, 48, 77, 3, 256), 0, 0),
                                               ((4864, 16, 319, 3, 256), 0, 2), ((1280, 24, 77, 8, 256), 0, 0),
                                               ((1280, 20, 66, 4, 256), 2, 1)])
def test_block_size(blocks, shape, listed, grid):
    assert blocks(*shape, True) == listed
    assert blocks(*shape, False) == grid
