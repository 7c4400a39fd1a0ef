"""fp32 storage at 33 to 63 features: launches that the full-tile kernels leave go to the LDS-panel kernels, whose products are the same, and
those that have fp32 products keep them."""
import numpy as np
import pytest

from test_spmm_gpu import convert, torch_cuda  # noqa: F401
from test_tile_gpu import _random_operand, _sampled_csr
from util import decode

pytestmark = pytest.mark.gpu


# (bounds as for the three products of bf16 parts, 2^-14 of the sum of the sizes, and for fp32 sums, n 2^-24)
@pytest.mark.parametrize("rows,cols,per_row,N,kernel", [(4096, 11008, 1100, 32, "tile"), (4096, 11008, 1100, 36, "panel"), (4096, 4096, 1200, 44, "panel"),
                                                        (4096, 4096, 200, 36, "entries"), (4096, 4096, 130, 60, "entries")])
def test_kernels_by_width(torch_cuda, hs, rows, cols, per_row, N, kernel):
    torch = torch_cuda
    rng = np.random.default_rng(N)
    A = _sampled_csr(rng, rows, cols, per_row, 1, lambda n: rng.normal(size=n))
    plan = hs.Plan(convert(hs, A))
    B, dB = _random_operand(torch, rng, cols, N, 1)
    dC = torch.full((rows, N), 7, dtype=dB.dtype, device="cuda")
    plan.run(dB.data_ptr(), dC.data_ptr(), N, torch.cuda.current_stream().cuda_stream)
    torch.cuda.synchronize()
    assert plan.last_kernel() == "spmm_%s_kernel" % kernel
    D = np.zeros((rows, cols))
    D[np.repeat(np.arange(rows), per_row), A["col_idx"]] = decode(A["values"], 1)
    off = abs(dC.cpu().numpy().astype(np.float64) - D @ B.astype(np.float64))
    assert (off <= (per_row * 2.0**-24 + (0.0 if kernel == "entries" else 2.0**-14)) * (abs(D) @ abs(B.astype(np.float64)))).all()
    plan.close()
