"""Which prefill passes go through their layers in the few-row form (no GPU needed: the rule is arithmetic on estimates)."""
import ctypes as C

import pytest

from llama_cu_awq_amd._lib import lib

takes_few = lib["_Z21awq_prefill_takes_fewP7awq_ctxiiii"]
takes_few.argtypes, takes_few.restype = [C.c_void_p] + [C.c_int] * 4, C.c_bool

# (dim, key and value columns, hidden): rows at which each side measured 1 % faster or more
FEW = {(1024, 1024, 4096): (1, 16, 32, 33, 64, 65, 96), (1536, 256, 4096): (1, 32, 33, 64), (2048, 256, 5632): (1, 10, 32, 33, 64, 65, 96, 97, 128),
       (4096, 4096, 11008): (1, 32, 33, 64, 65, 96, 97), (4096, 1024, 14336): (1, 32, 33, 64, 65, 96), (5120, 5120, 13824): (1, 32, 33, 64, 65, 96, 97, 128),
       (5120, 1024, 13824): (1, 32, 33, 64, 65, 96, 97), (6656, 6656, 17920): (1, 4, 10, 11, 32, 33, 64, 65, 96), (6656, 512, 17920): (1, 32, 33, 64, 65, 96),
       (7168, 1024, 20480): (1, 32, 33, 64, 65, 96, 97, 128), (8192, 8192, 22016): (32, 33, 64, 65, 96), (8192, 1024, 28672): (1, 4, 16),
       (8192, 8192, 28672): (1, 32, 65, 80)}
ROWS = {(4096, 1024, 14336): (97, 128), (6656, 6656, 17920): (128,), (8192, 1024, 28672): (33, 48, 64, 96, 97, 128), (8192, 8192, 28672): (33, 48, 64, 97, 128)}


def _takes(M, dim, kv_dim, hidden):
    device = (C.c_int * 16)(0, 256)  # a context begins with its device's ordinal and compute units
    return takes_few(device, M, dim, kv_dim, hidden)


@pytest.mark.parametrize("shape", FEW, ids=str)
def test_few_row_form(shape):
    assert [M for M in FEW[shape] if not _takes(M, *shape)] == []


@pytest.mark.parametrize("shape", ROWS, ids=str)
def test_row_forms(shape):
    assert [M for M in ROWS[shape] if _takes(M, *shape)] == []
    assert not _takes(129, *shape)


@pytest.mark.parametrize("shape", [(4096, 4096, 11072), (4160, 4160, 11008)], ids=str)
def test_sizes_that_the_few_row_form_does_not_have(shape):
    """Quantisation groups of 128 have to be whole."""
    assert not any(_takes(M, *shape) for M in (1, 32, 33, 64, 65, 96, 97, 128))
