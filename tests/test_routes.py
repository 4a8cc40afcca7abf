"""Which route a call takes, as far as the host alone decides it (CPU only)."""
import pytest

from llm_infer_rust_amd import ops


@pytest.mark.parametrize("k,rows", [(1024, 64), (2560, 64), (3072, 64), (4096, 64), (8192, 64),
                                    (3584, 32), (5120, 32)])
def test_head_rows_on_the_projection_kernel(k, rows):
    """Rows of a wide head whose length is no power of two stay with the library from 33 on."""
    assert ops._head_rows(k) == rows
