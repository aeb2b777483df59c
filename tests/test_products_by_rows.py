"""Products of a model's own layers on the host: which kernel a step's rows go to, with recording stand-ins for the compiled libraries."""
from __future__ import annotations

import pytest
import torch

from test_product_routes import host_ops
from tiny_inference_server_amd.ops.hip_ops import KernelError


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


# (rows, columns, inner columns, gate): sizes at which the tiles are the faster, or so small that the host's time decides; at which the library's product is
# the faster by 4 % and more
ON_TILES = [(140, 2304, 1536, 0), (640, 2304, 1536, 0), (1537, 2304, 1536, 0), (2048, 2304, 1536, 0), (257, 1536, 4096, 0), (640, 1536, 4096, 0), (513, 2048, 5632, 0),
            (900, 2048, 5632, 0), (192, 3072, 2048, 0), (900, 3072, 2048, 0), (140, 8192, 1536, 1), (1024, 8192, 1536, 1), (512, 11264, 2048, 1), (1000, 11264, 2048, 1),
            (2048, 2816, 2048, 1), (384, 2048, 5632, 0), (768, 1536, 4096, 0), (640, 2048, 2048, 0)]
ON_LIBRARY = [(640, 2048, 5632, 0), (768, 2048, 5632, 0), (2048, 3072, 2048, 0), (1400, 1536, 1536, 0), (1532, 1536, 1536, 0), (1152, 2048, 1408, 0),
              (768, 11264, 2048, 1), (1025, 8192, 1536, 1), (1025, 1536, 4096, 0), (2049, 2304, 1536, 0)]


@pytest.mark.parametrize("sizes,kernel", [(ON_TILES, "tis_gemm_tiles"), (ON_LIBRARY, "tis_gemm_library")])
def test_the_faster_of_tiles_and_library(sizes, kernel):
    for rows, N, K, gate in sizes:
        ops = host_ops()
        assert (N, K) in ops.library_widths
        x, w = zeros(rows, K), zeros(N, K)
        ops.linear_swiglu(x, w) if gate else ops.linear_by_rows(x, w, residual=zeros(rows, N))
        assert [fn for fn, _ in ops.calls if fn != "tis_swiglu"] == [kernel], (rows, N, K)


# (rows, columns, inner columns, gate) beyond 1,024 rows: tiles of 128 x 64, 128 x 96 and 128 x 128 that fill the chip, and what lies beside them
@pytest.mark.parametrize("sizes,kernel", [
    ([(1153, 1536, 4096, 0), (1318, 1536, 4096, 0), (2048, 1536, 4096, 0), (1280, 2048, 5632, 0), (1537, 2048, 5632, 0), (2048, 2048, 5632, 0)], "tis_gemm_tiles"),
    ([(1152, 1536, 4096, 0), (1537, 1536, 4096, 0), (1408, 2048, 5632, 0), (1536, 2048, 5632, 0), (2049, 1536, 4096, 0), (1281, 11264, 2048, 1), (2048, 8192, 1536, 1)],
     "tis_gemm_library")])
def test_beyond_a_thousand_rows(sizes, kernel):
    test_the_faster_of_tiles_and_library(sizes, kernel)


def test_what_a_layers_products_refuse():
    """Operands that do not fit together, whichever kernel the sizes go to."""
    ops, x = host_ops(), zeros(300, 1536)
    gain = torch.ones(1536)
    for w in (zeros(1536, 1540), zeros(1536, 3072)[:, ::2], torch.zeros(1536, dtype=torch.bfloat16), zeros(1536, 1536).float()):
        for call in (ops.linear_by_rows, ops.linear_swiglu):
            with pytest.raises(KernelError):
                call(x, w)
    with pytest.raises(KernelError):
        ops.linear_by_rows(x, zeros(1536, 1536), residual=zeros(300, 1535))
    with pytest.raises(KernelError):
        ops.linear_by_rows(x.t(), zeros(1536, 300))
    for rms in ((gain[:-1], 1e-5), (gain.bfloat16(), 1e-5), (torch.ones(3072)[::2], 1e-5)):
        for call in (ops.linear_by_rows, ops.linear_swiglu):
            for rows in (300, 2048):
                with pytest.raises(KernelError):
                    call(zeros(rows, 1536), zeros(1536, 1536), rms=rms)
    assert not ops.calls
