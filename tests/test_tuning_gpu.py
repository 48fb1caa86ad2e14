"""The tuning overrides of the decode partition, read once per context at qh_open, give the products of the default
partition: K-wave rows within a workgroup (QH_SKINNY_PLAIN_WK, plain partials reduced through LDS before the staged
16-byte stores) and forced tile waves (QH_SKINNY_TILE_WAVES). Token counts cover one and two 16-token blocks (the
two-block kernel takes at most 512 threads per workgroup, so K-wave rows beyond that bound fall back to the default
partition). Sums of the partials are checked against the default context's to f32 rounding of the different split
(the split itself changes), and against the oracle at the product bar."""

import numpy as np
import pytest

from qwenny_amd import Epi, Gemm, Mat
from qwenny_amd.synth import activations, f32_to_bf16
from tests.helpers import bf16_out_err, make_quant, oracle_y, rel_err, to_dev

pytestmark = pytest.mark.gpu


def _sum(gemm, mat, x, m):
    import torch

    split = mat.split(m)
    y = torch.full((split, m, mat.rows), float("nan"), dtype=torch.float32, device="cuda")
    assert gemm.run(None, m, mat, to_dev(x), y, Epi.Plain) == split
    torch.cuda.synchronize()
    got = y.cpu().numpy().astype(np.float64)
    assert not np.isnan(got).any()
    return got.sum(0), split


@pytest.mark.parametrize("env", [{"QH_SKINNY_PLAIN_WK": "2"}, {"QH_SKINNY_PLAIN_WK": "4"},
                                 {"QH_SKINNY_TILE_WAVES": "4"}, {"QH_SKINNY_TILE_WAVES": "8"}])
@pytest.mark.parametrize("m", [1, 5, 17, 33])
def test_tuned_partition_matches_default(gemm, monkeypatch, env, m):
    print(f"tuned partition {env} m={m}", flush=True)
    for k_, v in env.items():
        monkeypatch.setenv(k_, v)
    tuned = Gemm.load(0)  # reads the overrides
    try:
        q = make_quant(900 + m, "i4", 1024, 4096)
        x = activations(901 + m, "x", m, 4096)
        want_sum, _ = _sum(gemm, Mat.stack(gemm, [q]), x, m)
        got_sum, _ = _sum(tuned, Mat.stack(tuned, [q]), x, m)
        assert rel_err(got_sum, want_sum) <= 1e-5
        assert rel_err(got_sum, oracle_y(q, x)) <= 1e-4
    finally:
        tuned.close()


@pytest.mark.parametrize("pk", ["2", "4"])
def test_part_len_covers_tuned_split(monkeypatch, pk):
    """Under QH_SKINNY_PLAIN_WK the skinny split depends on the token count; part_len must cover the largest
    split x tokens over every count (a product into a part_len-sized buffer writes no further)."""
    import torch

    print(f"part_len QH_SKINNY_PLAIN_WK={pk}", flush=True)
    monkeypatch.setenv("QH_SKINNY_PLAIN_WK", pk)
    tuned = Gemm.load(0)
    try:
        q = make_quant(950, "i4", 1024, 4096)
        mat = Mat.stack(tuned, [q])
        max_tok = 48
        need = max(mat.split(m) * m * mat.rows for m in range(1, max_tok + 1))
        n = tuned.part_len([mat], max_tok)
        assert n >= need
        # a product of every token count into a buffer of exactly part_len floats, guarded by a canary after it
        y = torch.full((n + 4096,), float("nan"), dtype=torch.float32, device="cuda")
        for m in (1, 2, 3, 4, 16, 17, 33, 48):
            x = activations(951 + m, "x", m, 4096)
            split = tuned.run(None, m, mat, to_dev(x), y, Epi.Plain)
            assert split * m * mat.rows <= n
        torch.cuda.synchronize()
        assert torch.isnan(y[n:]).all()
    finally:
        tuned.close()


@pytest.mark.parametrize("epi,whole", [(Epi.Plain, True), (Epi.Silu, False)])
@pytest.mark.parametrize("kind,m", [("i8", 1), ("i8", 5), ("i4", 5), ("i4", 12)])
def test_overrides_reach_whole_sums(monkeypatch, kind, m, epi, whole):
    """The overrides hold for products of whole sums too: one wave per workgroup (QH_SKINNY_MAX_W=1) sums K in one order,
    16 waves and a fill no launch reaches in another, so that some last bits differ; both are within the bar."""
    import torch

    q = make_quant(970 + m, kind, 1024, 4096)
    x = activations(971 + m, "x", m, 4096)
    got = []
    for env in ({"QH_SKINNY_MAX_W": "1"}, {"QH_SKINNY_MAX_W": "16", "QH_SKINNY_FILL": "64"}):
        print(f"overrides {kind} m={m} {epi.name} {env}", flush=True)
        for k_, v in env.items():
            monkeypatch.setenv(k_, v)
        tuned = Gemm.load(0)
        try:
            mat = Mat.stack(tuned, [q], silu=epi == Epi.Silu)
            y = torch.full((m, 1024 if whole else 512), float("nan"), dtype=torch.float32 if whole else torch.bfloat16,
                           device="cuda")
            tuned.run_split(None, m, mat, to_dev(x), y, epi, whole)
            torch.cuda.synchronize()
            got.append(y.float().cpu().numpy())
            del mat
        finally:
            tuned.close()
    want = oracle_y(q, x)
    if not whole:
        g, u = want[:, :512], want[:, 512:]
        want = g / (1 + np.exp(-g)) * u
    for y in got:  # (SwiGLU: beyond one bf16 rounding of the output)
        assert (rel_err if whole else bf16_out_err)(y, want) <= 1e-4
    if whole:
        assert not np.array_equal(got[0], got[1])


@pytest.mark.parametrize("kind", ["i4", "i8g"])
@pytest.mark.parametrize("rows,cols", [(16, 128), (16, 17024), (2064, 1280), (4096, 2560), (5136, 1152)])
def test_split_range(gemm, kind, rows, cols):
    """qh_mat_split over the decode token counts: between 1 and a partial per group of K, and what part_len holds."""
    print(f"split range {kind} {rows}x{cols}", flush=True)
    mat = Mat.stack(gemm, [make_quant(980, kind, rows, cols)])
    for m in range(1, 49):
        assert 1 <= mat.split(m) <= cols // 128
        assert mat.split(m) * m * rows <= gemm.part_len([mat], 48)


@pytest.mark.parametrize("rows,cols", [(16, 1152), (32, 5120), (64, 17408), (128, 2176), (128, 3840), (256, 1024)])
def test_adapter_partials(gemm, rows, cols):
    """An adapter's stacked A (dense bf16, few rows) keeps few partials, which each workgroup of the adapted product reads:
    up to 3 at 1-8 tokens, from 9 at most one per 4 groups of K (mid_kernel's wave rows)."""
    print(f"adapter partials {rows}x{cols}", flush=True)
    w = np.random.default_rng(rows).standard_normal((rows, cols)).astype(np.float32)
    mat = Mat.new(gemm, f32_to_bf16(w), cols, int8=False)
    for m in range(1, 49):
        assert mat.split(m) <= (3 if m <= 8 else (cols // 128 + 3) // 4), m
