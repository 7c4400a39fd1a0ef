"""Error of fp32 storage against fp64 over the feature dimensions of a large pruned matrix: fp32 products wherever the
kernels that multiply bf16 parts do not say so, and those parts' own bound where they do."""
import os

import numpy as np
import pytest

from test_spmm_gpu import convert, gpu_spmm, torch_cuda  # noqa: F401
from test_tile_gpu import _sampled_csr

pytestmark = pytest.mark.gpu


def _errors(torch, hs, plan, A, N, rng, adversarial=False):
    """Largest error in units of the sum of |a| |b|."""
    rows, cols = A["rows"], A["cols"]
    if adversarial:
        ones = np.frombuffer(np.uint32(0x3FFFFFFF).tobytes(), np.float32)[0]       # 1.9999999: every low mantissa bit set
        B = (ones * np.exp2(rng.integers(-3, 4, (cols, N)))).astype(np.float32)
    else:
        B = rng.normal(size=(cols, N)).astype(np.float32)
    got = gpu_spmm(torch, hs, dict(dtype=1, rows=rows), B, N, plan=plan).astype(np.float64)
    D = torch.zeros((rows, cols), dtype=torch.float64, device="cuda")
    per_row = A["nnzs"] // rows
    at = torch.from_numpy(A["col_idx"].astype(np.int64).reshape(rows, per_row)).cuda()
    D.scatter_(1, at, torch.from_numpy(A["values"].astype(np.float64).reshape(rows, per_row)).cuda())
    dB = torch.from_numpy(B.astype(np.float64)).cuda()
    ref, mag = (D @ dB).cpu().numpy(), (D.abs() @ dB.abs()).cpu().numpy()
    return float((np.abs(got - ref) / mag).max())


def test_narrow_feature_dimensions_are_multiplied_in_fp32(torch_cuda, hs):
    """Rows of B that are no whole 16-byte pieces, and those under 16 features: fp32 products, whose sums of some 800 terms
    are off by rounding only (2^-20 of the sum of |a| |b| is 16 roundings of a whole sum; bf16 parts are at 2^-17.3)."""
    rng = np.random.default_rng(50)
    A = _sampled_csr(rng, 11008, 4096, 800, 1, lambda n: rng.normal(size=n))
    plan = hs.Plan(convert(hs, A))
    for N in (8, 9, 12, 15, 17, 21, 30, 39, 47):
        worst = _errors(torch_cuda, hs, plan, A, N, rng)
        assert worst <= 2.0 ** -20, "N=%d: 2^%.1f" % (N, np.log2(worst))
    plan.close()


@pytest.mark.parametrize("rows,cols,per_row", [(1000, 520, 60), (300, 2048, 200), (130, 65, 5)])
def test_both_parts_of_every_factor_are_multiplied_by_the_full_tile_kernels(torch_cuda, hs, rows, cols, per_row):
    """The bounds of the three-product arithmetic: the product left out is at most 2^-14 of |a| |b|, and over many normal
    entries 2^-16 of their sum.  (A low part that is lost or misplaced costs 2^-8.)"""
    rng = np.random.default_rng(rows)
    ones = np.frombuffer(np.uint32(0x3FFFFFFF).tobytes(), np.float32)[0]
    os.environ["HSPMM_TILE"] = "1"
    try:
        for adversarial, bound in ((False, 2.0 ** -16 if per_row >= 60 else 2.0 ** -14), (True, 2.0 ** -14)):
            A = _sampled_csr(rng, rows, cols, per_row, 1,
                             (lambda n: ones * np.exp2(rng.integers(-3, 4, n))) if adversarial else (lambda n: rng.normal(size=n)))
            plan = hs.Plan(convert(hs, A))
            for N in (4, 16, 17, 32, 44, 64, 100):
                worst = _errors(torch_cuda, hs, plan, A, N, rng, adversarial)
                assert plan.info()["last_kernel_family"] == 3
                assert worst <= bound, "N=%d: 2^%.1f" % (N, np.log2(worst))
            plan.close()
    finally:
        os.environ.pop("HSPMM_TILE", None)
