"""Which route a call takes, as far as the host alone decides it (CPU only)."""
import pytest

from llm_infer_rust_amd import ops


@pytest.mark.parametrize("n,k,rows", [(151936, 1024, 64), (151936, 2560, 64), (151936, 3072, 64),
                                      (151936, 4096, 64), (262144, 8192, 64), (152064, 3584, 32),
                                      (151936, 5120, 32), (262144, 2560, 32), (200000, 2560, 64)])
def test_head_rows_on_the_projection_kernel(n, k, rows):
    """Long rows whose length is no power of two, and the largest heads of shorter ones, stay with
    the library from 33 rows on."""
    assert ops._head_rows(n, k) == rows
