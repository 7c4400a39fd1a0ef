"""Device memory of a plan: what hspmm_create takes is what hspmm_plan_info says."""
import numpy as np
import pytest

from test_spmm_gpu import convert, torch_cuda  # noqa: F401
from util import random_csr

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("density", [0.02, 0.4])
def test_what_a_plan_takes_is_what_it_says(torch_cuda, hs, density):
    """Tiles of few entries, kept as bitmaps, and dense ones of 33 MB, which make no use of room for a bitmap's elements."""
    torch = torch_cuda
    tiles = convert(hs, random_csr(np.random.default_rng(3), 4096, 4096, density, 0))
    hs.set_kernel_mode(3)                                   # (the gather kernels alone: no later stream that the room would do for)
    try:
        hs.Plan(tiles).close()
        torch.cuda.synchronize()
        before = torch.cuda.mem_get_info()[0]
        plan = hs.Plan(tiles)
        taken = before - torch.cuda.mem_get_info()[0]
    finally:
        hs.set_kernel_mode(0)
    says, step = plan.info()["device_bytes"], 2 << 20       # (the allocator gives whole pages of 2 MB)
    needs = tiles["data"].nbytes + 2 * tiles["tcA2B"].nbytes
    assert needs <= says <= (1.1 if density > 0.3 else 1.7) * needs + (2 << 20)
    assert says - 8 * step <= taken <= says + 8 * step
    plan.close()
