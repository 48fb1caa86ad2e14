"""Plain products of more than 48 tokens on dense bf16 matrices of few rows (mid_kernel over blocks of 32 tokens, K split
over the grid, the partials added by a second launch): one partial to the caller, exact products of the stored weights
(1e-4 against the f64 oracle, measured 1e-6)."""

import numpy as np
import pytest

import oracle
from qwenny_amd import Epi, Mat
from qwenny_amd.synth import activations, f32_to_bf16
from tests.helpers import rel_err, to_dev

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("rows,cols", [(16, 128), (16, 17408), (32, 5120), (48, 384), (96, 5120), (256, 2432)])
def test_narrow(gemm, rows, cols):
    import torch

    w = f32_to_bf16(np.random.default_rng(rows + cols).standard_normal((rows, cols)).astype(np.float32) * 0.05)
    mat = Mat.new(gemm, w, cols, int8=False)
    for m in (49, 64, 65, 333, 2049):
        x = activations(m, "x", m, cols)
        want = oracle.dense_f64(w, x)
        assert mat.split(m) == 1 and mat.kernel(m) == "prefill"
        for whole in (False, True):
            for shift in (0, 1):  # y at any 4-byte alignment
                print(f"narrow {rows}x{cols} m={m} whole={whole} shift={shift}", flush=True)
                buf = torch.full((m * rows + 64,), float("nan"), device="cuda")
                y = buf[shift:shift + m * rows]
                assert gemm.run_split(None, m, mat, to_dev(x), y, Epi.Plain, whole) == 1
                torch.cuda.synchronize()
                assert rel_err(y.view(m, rows).cpu().numpy(), want) <= 1e-4
                assert torch.isnan(buf[:shift]).all() and torch.isnan(buf[shift + m * rows:]).all()
