"""The partials' sums at decode sizes (one thread per column) and beyond, and add_rmsnorm on both of its paths (one launch with the row in registers, or the partials' sum first): rows of one to
four float4 per thread and a remainder, partials of every batch size, decode and streaming token counts, at the bound
between the paths. The residual is bit-exact against the oracle's order, the bf16 output within one bf16 rounding of the
f64 norm."""

import numpy as np
import pytest

import oracle
from qwenny_amd import add_rmsnorm, sum_parts
from tests.helpers import bf16_out_err

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("splits,n,hidden", [(1, 1, 4), (2, 3, 20), (3, 2, 1152), (4, 65, 2560), (5, 3, 5120), (9, 2, 5120),
                                             (10, 2, 5120), (12, 5, 4096), (13, 5, 4096), (17, 2, 1152), (19, 1, 2560),
                                             (20, 64, 2560), (8, 100, 5120), (2, 300, 2560), (1, 1030, 1024),
                                             (2, 3, 16384), (1, 257, 8200), (3, 2, 16388)])
def test_add_rmsnorm_paths(splits, n, hidden):
    import torch

    print(f"row norm {splits}x{n}x{hidden}", flush=True)
    rng = np.random.default_rng(hidden + splits + n)
    h = rng.standard_normal((n, hidden)).astype(np.float32)
    x = (rng.standard_normal((splits, n, hidden)) * 0.3).astype(np.float32)
    w = rng.uniform(0.5, 1.5, hidden).astype(np.float32)
    hd, xd, wd = (torch.from_numpy(a).cuda() for a in (h, x, w))
    y = torch.full((n, hidden), float("nan"), dtype=torch.bfloat16, device="cuda")
    add_rmsnorm(None, hd, xd, splits, n, hidden, wd, y, 1e-6)
    torch.cuda.synchronize()
    want_h, want_y = oracle.add_rmsnorm(h, x, splits, w, 1e-6)
    assert np.array_equal(hd.cpu().numpy(), want_h)
    assert bf16_out_err(y.float().cpu().numpy(), want_y) <= 1e-5


@pytest.mark.parametrize("splits,n,ld", [(1, 1, 4), (16, 1, 36), (17, 3, 20), (24, 1, 4096), (49, 2, 2560), (5, 64, 4092),
                                         (5, 64, 4096), (17, 65, 4096), (2, 3, 2560), (3, 16, 4096), (3, 16, 4100),
                                         (4, 16, 4096), (4, 16, 4100), (5, 16, 4100)])
def test_sum_parts_sizes(splits, n, ld):
    import torch

    print(f"sum_parts {splits}x{n}x{ld}", flush=True)
    x = np.random.default_rng(splits + n).standard_normal((splits, n, ld)).astype(np.float32)
    y = torch.full((n, ld), float("nan"), device="cuda")
    sum_parts(None, torch.from_numpy(x).cuda(), splits, n, ld, y)
    torch.cuda.synchronize()
    assert np.array_equal(y.cpu().numpy(), oracle.sum_parts(x, splits))


@pytest.mark.parametrize("splits,n,hidden", [(8, 3, 2560), (9, 2, 2560), (4, 2, 5120), (5, 2, 5120), (16, 2, 1280),
                                             (16, 2, 1284), (2, 3, 10240), (3, 3, 10240), (17, 70, 1024), (17, 70, 2560),
                                             (9, 300, 5120), (9, 70, 8196), (16, 400, 1024), (8, 385, 2560), (3, 255, 5120),
                                             (3, 256, 5120), (3, 1030, 128), (2, 1024, 2048), (2, 66, 16388), (1, 2, 16388),
                                             (1, 512, 5120), (17, 17, 16388)])
def test_add_rmsnorm_bounds(splits, n, hidden):
    """The bounds between its paths: partials of a row in one launch, wide and narrow rows with many of them, streaming
    token counts."""
    test_add_rmsnorm_paths(splits, n, hidden)


@pytest.mark.parametrize("splits,n,ld", [(4, 1, 16384), (4, 1, 16388), (5, 1, 40956), (5, 1, 40960), (16, 1, 40964),
                                         (17, 1, 16380), (17, 1, 16384), (24, 2, 8196), (25, 3, 5464), (8, 3, 2048), (8, 2, 32764),
                                         (8, 2, 32768), (17, 3, 5460), (5, 128, 4092),
                                         (5, 128, 4096), (17, 128, 4096), (64, 46, 1280), (65, 46, 1280), (65, 7, 37444),
                                         (65, 7, 37452), (8, 20, 3276), (8, 20, 3280), (12, 20, 5120)])
def test_sum_parts_bounds(splits, n, ld):
    test_sum_parts_sizes(splits, n, ld)
