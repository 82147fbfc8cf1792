"""How the batched GEMM says it runs a product (awq_gemm_int4_form: host arithmetic, no device)."""
import pytest

import llama_cu_awq_amd as A


def test_forms_refuse_what_the_products_refuse():
    for M, K, N in ((4, 48, 128), (4, 64, 64), (0, 64, 128), (4, 0, 128)):
        with pytest.raises(A.AwqError) as e:
            A.gemm_form(M, K, N)
        assert e.value.code == -2


def test_split_products_fit_the_workspace():
    """256 tiles, and partial tiles of 32 MiB: what the workspace holds."""
    split = set()
    for M in (1, 33, 77, 150, 300, 512, 700, 1100, 2048):
        for K in (512, 1056, 4096, 11008, 28672):
            for N in (128, 384, 1152, 4096, 8192, 13824):
                rows, cols, slices, parts = A.gemm_form(M, K, N)
                assert (rows, cols) in {(32, 64), (64, 64), (64, 128), (64, 256), (96, 256), (128, 256), (128, 128)}
                assert N % cols == 0 and -(-K // 128) >= parts
                if parts > 1:
                    tiles = -(-M // rows) * (N // cols)
                    assert tiles <= 256 and tiles * parts * rows * cols * 4 <= 32 << 20
                    split.add((rows, cols))
    assert len(split) >= 5
