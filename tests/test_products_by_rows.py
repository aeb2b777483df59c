"""Products of a model's own layers on the host: which kernel a step's rows go to, with recording stand-ins for the compiled libraries."""
from __future__ import annotations

import pytest
import torch

from test_product_routes import host_ops


def zeros(rows, columns):
    return torch.zeros(rows, columns, dtype=torch.bfloat16)


@pytest.mark.parametrize("rows", [129, 300, 513])
@pytest.mark.parametrize("N,K", [(1536, 1536), (1000, 640)])
def test_residuals_that_the_library_does_not_read(rows, N, K):
    """Rows that start on 8 bytes, or in steps of 8, go to the tiles, which read them, at the library's widths as at others; on 2 bytes to the few-row
    kernel."""
    wide = zeros(rows, N + 12)
    for residual, kernel in ((wide[:, 4:N + 4], "tis_gemm_tiles"), (zeros(rows, N), "tis_gemm_tiles"), (wide[:, :N], "tis_gemm_tiles"),
                             (wide[:, 1:N + 1], "tis_gemm_skinny"), (zeros(rows, N + 2)[:, :N], "tis_gemm_skinny")):
        ops = host_ops()
        ops.linear_by_rows(zeros(rows, K), zeros(N, K), residual=residual)
        assert [fn for fn, _ in ops.calls] == [kernel], (residual.stride(), residual.storage_offset())
