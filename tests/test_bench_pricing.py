"""bench.py prices a row kernel's traffic by the form that the library reads."""
import bench
import bootcmatchg_amd as bc


def test_bytes_follow_the_form():
    n, nnz = 96 ** 3, 7 * 96 ** 3 - 6 * 96 ** 2
    # a constant stencil of a size without a narrow column copy (cb = 4)
    assert bench.streamed_bytes(n, nnz, bc.FORM_STENCIL, 4, 3) == 25 * n
    assert bench.streamed_bytes(n, nnz, bc.FORM_CLASSES, 4, 2) == 17 * n
    assert bench.streamed_bytes(n, nnz, bc.FORM_COLUMNS, 4, 4) == 12 * nnz + 4 * (n + 1) + 32 * n
    assert bench.streamed_bytes(n, nnz, bc.FORM_COLUMNS, 0, 2) == 8 * nnz + n + 8 * (n // 256) + 16 * n
    assert bench.streamed_bytes(n, nnz, bc.FORM_SYMMETRIC, 4, 0) == n + 8 * (n + (nnz - n) // 2)
    assert [bench.sweep_vectors(f) for f in (bc.FORM_COLUMNS, bc.FORM_STENCIL)] == [4, 3]
