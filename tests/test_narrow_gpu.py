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


@pytest.mark.parametrize("rank", [8, 16, 64])
@pytest.mark.parametrize("rows,cols", [(16, 1024), (48, 5120), (96, 17408), (256, 2432)])
def test_narrow_adapter(gemm, rows, cols, rank):
    """An adapter on such a product (a DeltaNet in_ba projection): outputs whose delta is exactly zero (tokens of slot
    scale 0, rows of an unadapted module) are the plain product's bit for bit, the others the oracle's."""
    import torch

    w = f32_to_bf16(np.random.default_rng(rows + cols).standard_normal((rows, cols)).astype(np.float32) * 0.05)
    mat = Mat.new(gemm, w, cols, int8=False)
    end = rows // 2 + 3  # rows of the second module, from inside a tile, have no adapter
    tab = [end] + [2**31 - 1] * 3 + [rank // 2, -1, -1, -1]
    for m in (49, 333, 1100):
        print(f"narrow adapter {rows}x{cols} m={m} rank={rank}", flush=True)
        rng = np.random.default_rng(m)
        split, m_cols = 2, 2 * rank
        xa = rng.standard_normal((split, m, m_cols)).astype(np.float32)
        b = (rng.standard_normal((rows, rank)) * 0.1).astype(np.float16)
        slot, scale = rng.integers(0, 3, m).astype(np.int32), np.array([0.0, 0.5, 2.0], np.float32)
        dev = [torch.from_numpy(np.ascontiguousarray(v)).cuda()
               for v in (xa, b.view(np.int16), np.asarray(tab, np.int32), slot, scale)]
        lora = (dev[0], split, m_cols, dev[1], rank, dev[2], dev[3], dev[4])
        x = activations(m, "x", m, cols)
        xd = to_dev(x)
        n = mat.split(m)
        plain, y = (torch.full((n, m, rows), float("nan"), device="cuda") for _ in range(2))
        assert gemm.run(None, m, mat, xd, plain) == n
        assert gemm.run_lora(None, m, mat, xd, y, Epi.Plain, lora) == n
        torch.cuda.synchronize()
        plain, y = plain.cpu().numpy(), y.cpu().numpy()
        assert np.array_equal(y[:, scale[slot] == 0].view(np.int32), plain[:, scale[slot] == 0].view(np.int32))
        assert np.array_equal(y[:, :, end:].view(np.int32), plain[:, :, end:].view(np.int32))
        want = oracle.lora_add(oracle.dense_f64(w, x), xa, split, b.view(np.uint16), rank, tab, slot, scale, m)
        assert rel_err(y.astype(np.float64).sum(0), want) <= 1e-4
