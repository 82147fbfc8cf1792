"""Which of its two forms the fused schedule's long-context attention takes (no GPU needed: the rule is arithmetic)."""
import ctypes as C

import pytest

from llama_cu_awq_amd._lib import lib

takes_ranges = lib["_Z26awq_attention_takes_rangesiiiii"]
takes_ranges.argtypes, takes_ranges.restype = [C.c_int] * 5, C.c_bool


# (heads, head size, query heads per key head, launch size) on 256 compute units, each on the side that measured faster
@pytest.mark.parametrize("shape", [(8, 128, 8, 1279), (16, 128, 1, 2048), (32, 128, 1, 4096), (32, 128, 4, 32768), (40, 128, 1, 8192), (52, 128, 1, 32768),
                                   (64, 128, 8, 32768), (8, 64, 1, 32768), (2, 256, 2, 1024), (32, 256, 8, 16384)], ids=str)
def test_one_launch_of_ranges(shape):
    assert takes_ranges(256, *shape)


@pytest.mark.parametrize("shape", [(4, 128, 1, 1280), (8, 128, 1, 4096), (8, 128, 4, 2048), (8, 128, 8, 131071), (16, 128, 1, 8192), (16, 128, 8, 8192), (24, 128, 1, 8192),
                                   (32, 128, 1, 8192), (40, 128, 1, 32768), (4, 256, 1, 2048), (16, 256, 1, 4096), (32, 256, 1, 16384)], ids=str)
def test_few_workgroups_with_long_ranges_go_in_two_launches(shape):
    assert not takes_ranges(256, *shape)
