"""Products of 9-48 tokens on mid_kernel (whose partition depends on the matrix's tiles, groups and storage, and on the
token count) and whole sums of 1-16 tokens and few-split products of 1-8 on skinny_mw_kernel: odd tile counts and group counts, one tile, one group, both token blocks and their last rows, every
storage and epilogue, gathered logit rows. Products are exact products of the dequantized weights, so the bar is the
decode kernels' 1e-4 against the f64 oracle (measured 1e-6: f32 sums of up to 2432 terms), one bf16 ulp beyond it for
SwiGLU outputs."""

import numpy as np
import pytest

import oracle
from qwenny_amd import Epi, Mat, row_order
from qwenny_amd.synth import activations, bf16_to_f32, f32_to_bf16
from tests.helpers import bf16_out_err, make_quant, oracle_y, rel_err, to_dev

pytestmark = pytest.mark.gpu


def _matrix(gemm, kind, n, k, silu=False):
    if kind == "bf16":
        w = f32_to_bf16(np.random.default_rng(n + k).standard_normal((n, k)).astype(np.float32) * 0.05)
        return Mat.new(gemm, w, k, silu=silu, int8=False), lambda x: bf16_to_f32(x).astype(np.float64) @ bf16_to_f32(w).T
    q = make_quant(n + k, kind[:2] if kind == "i4s32" else kind, n, k)
    if kind == "i4s32":  # scales that bf16 does not hold
        q.scales *= np.float32(1.001)
        q.offsets[:] = -8 * q.scales
    return Mat.stack(gemm, [q], silu=silu), lambda x: oracle_y(q, x)


SHAPES = [(16, 128), (48, 2432), (528, 384), (2064, 1280), (4112, 640), (8208, 256), (24592, 128), (32800, 128),
          (336, 12672), (2560, 6272)]


@pytest.mark.parametrize("kind", ["i4", "i4z", "i4s32", "i8", "i8g", "bf16"])
@pytest.mark.parametrize("n,k", SHAPES)
def test_plain_and_whole(gemm, kind, n, k):
    import torch

    mat, want_of = _matrix(gemm, kind, n, k)
    for m in (1, 2, 4, 5, 8, 9, 13, 16, 17, 25, 32, 33, 48):
        x = activations(m, "x", m, k)
        want = want_of(x)
        split = mat.split(m)
        for whole in (False, True):
            print(f"mid {kind} {n}x{k} m={m} whole={whole}", flush=True)
            s = 1 if whole else split
            y = torch.full((s, m, n), float("nan"), dtype=torch.float32, device="cuda")
            assert gemm.run_split(None, m, mat, to_dev(x), y, Epi.Plain, whole) == s
            torch.cuda.synchronize()
            assert rel_err(y.double().sum(0).cpu().numpy(), want) <= 1e-4, (m, whole)


@pytest.mark.parametrize("kind", ["i4", "i4z", "i4s32", "i8g", "bf16"])
@pytest.mark.parametrize("n,k", [(16, 384), (528, 1280), (8224, 384), (24608, 128), (33024, 256)])
def test_silu(gemm, kind, n, k):
    import torch

    mat, want_of = _matrix(gemm, kind, n, k, silu=True)
    for m in (1, 3, 8, 9, 12, 16, 20, 32, 48):
        print(f"mid silu {kind} {n}x{k} m={m}", flush=True)
        x = activations(m, "x", m, k)
        y = want_of(x)
        g, u = y[:, :n // 2], y[:, n // 2:]
        out = torch.full((m, n // 2), float("nan"), dtype=torch.bfloat16, device="cuda")
        gemm.run(None, m, mat, to_dev(x), out, Epi.Silu)
        torch.cuda.synchronize()
        assert bf16_out_err(out.float().cpu().numpy(), g / (1 + np.exp(-g)) * u) <= 1e-4, m


@pytest.mark.parametrize("kind", ["i4", "i4z", "i4s32", "i8g"])
@pytest.mark.parametrize("n,k", [(528, 512), (528, 640), (528, 1024), (48, 5120), (48, 4992)])
def test_whole_chunks(gemm, kind, n, k):
    """Whole sums of 2-16 tokens with the groups of K whole chunks of a wave and with a shorter last one."""
    import torch

    plain, want_of = _matrix(gemm, kind, n, k)
    gated, _ = _matrix(gemm, kind, n, k, silu=True)
    for m in (2, 4, 5, 8, 9, 16):
        print(f"whole chunks {kind} {n}x{k} m={m}", flush=True)
        x = activations(m, "x", m, k)
        want = want_of(x)
        g, u = want[:, :n // 2], want[:, n // 2:]
        y = torch.full((1, m, n), float("nan"), dtype=torch.float32, device="cuda")
        assert gemm.run_split(None, m, plain, to_dev(x), y, Epi.Plain, True) == 1
        out = torch.full((m, n // 2), float("nan"), dtype=torch.bfloat16, device="cuda")
        gemm.run(None, m, gated, to_dev(x), out, Epi.Silu)
        torch.cuda.synchronize()
        assert rel_err(y[0].double().cpu().numpy(), want) <= 1e-4, m
        assert bf16_out_err(out.float().cpu().numpy(), g / (1 + np.exp(-g)) * u) <= 1e-4, m


@pytest.mark.parametrize("kind", ["i4", "i8g", "bf16"])
@pytest.mark.parametrize("n,k", [(528, 384), (24592, 256), (65552, 128)])
def test_argmax_gathered_rows(gemm, kind, n, k):
    import torch

    mat, want_of = _matrix(gemm, kind, n, k)
    for m in (9, 24, 32, 40):
        print(f"mid argmax {kind} {n}x{k} n_out={m}", flush=True)
        x = activations(m, "x", 2 * m, k)
        rows = np.random.default_rng(m).permutation(2 * m)[:m].astype(np.int32)
        y = torch.full((m, n), float("nan"), dtype=torch.float32, device="cuda")
        keys = torch.zeros(m, dtype=torch.int64, device="cuda")
        gemm.run(None, 2 * m, mat, to_dev(x), y, Epi.Argmax, torch.from_numpy(rows).cuda(), m, keys)
        torch.cuda.synchronize()
        got = y.cpu().numpy()
        assert rel_err(got, want_of(x[rows])) <= 1e-4
        tok = 0xFFFFFFFF - (keys.cpu().numpy().view(np.uint64) & np.uint64(0xFFFFFFFF))
        assert np.array_equal(tok.astype(np.int64), got.argmax(1))


def test_adapter(gemm):
    """The fused adapter delta on mid_kernel: SwiGLU and plain, against the oracle's f64 delta."""
    import torch

    n, k, rank = 1056, 1280, 16
    for m in (1, 4, 7, 12, 33):
        rng = np.random.default_rng(m)
        xa = rng.standard_normal((2, m, 2 * rank)).astype(np.float32)
        b = (rng.standard_normal((n, rank)) * 0.1).astype(np.float16)
        slot, scale = rng.integers(0, 3, m).astype(np.int32), np.array([0.0, 0.5, 2.0], np.float32)
        x = activations(m, "x", m, k)
        for silu in (False, True):
            print(f"mid adapter silu={silu} m={m}", flush=True)
            mat, want_of = _matrix(gemm, "i8g", n, k, silu=silu)
            tab = [2**31 - 1] * 4 + [0, rank if silu else -1, -1, -1]
            dev = [torch.from_numpy(np.ascontiguousarray(v)).cuda()
                   for v in (xa, b.view(np.int16), np.asarray(tab, np.int32), slot, scale)]
            lora = (dev[0], 2, 2 * rank, dev[1], rank, dev[2], dev[3], dev[4])
            if not silu:
                want = oracle.lora_add(want_of(x), xa, 2, b.view(np.uint16), rank, tab, slot, scale, m)
                for whole in (False, True):
                    y = torch.full((1 if whole else mat.split(m), m, n), float("nan"), device="cuda")
                    gemm.run_lora(None, m, mat, to_dev(x), y, Epi.Plain, lora, whole)
                    assert rel_err(y.double().sum(0).cpu().numpy(), want) <= 1e-4, whole
                continue
            out = torch.full((m, n // 2), float("nan"), dtype=torch.bfloat16, device="cuda")
            gemm.run_lora(None, m, mat, to_dev(x), out, Epi.Silu, lora)
            want = oracle.lora_silu(want_of(x)[:, row_order(n, True)], xa, 2, b.view(np.uint16), rank, tab, slot, scale, m)
            assert bf16_out_err(out.float().cpu().numpy(), want) <= 1e-3


@pytest.mark.parametrize("kind", ["i4", "i4z", "i4s32", "i8", "i8g", "bf16"])
@pytest.mark.parametrize("n,k,rank,split", [(528, 1280, 8, 1), (528, 640, 16, 3), (1072, 384, 64, 2), (528, 4096, 64, 4),
                                            (6160, 512, 16, 2)])
def test_adapter_forms(gemm, kind, n, k, rank, split):
    """Every storage's adapter forms at decode sizes: odd tile counts, whole and shorter last chunks of K, each rank, xa
    staged in LDS or read from memory (64 columns twice of 4 partials). Outputs whose delta is exactly zero (tokens of
    slot scale 0; plain products: rows of an unadapted module) are the product's without adapter bit for bit."""
    import torch

    plain, want_of = _matrix(gemm, kind, n, k)
    gated, _ = _matrix(gemm, kind, n, k, silu=True)
    end = n // 2 + 3  # plain: the second module's rows, from inside a tile, have no adapter
    tabs = {False: [end] + [2**31 - 1] * 3 + [rank, -1, -1, -1], True: [2**31 - 1] * 4 + [0, rank, -1, -1]}
    for m in (1, 2, 4, 5, 8, 12, 16, 33, 48):
        rng = np.random.default_rng(m)
        xa = rng.standard_normal((split, m, 2 * rank)).astype(np.float32)
        b = (rng.standard_normal((n, rank)) * 0.1).astype(np.float16)
        slot, scale = rng.integers(0, 3, m).astype(np.int32), np.array([0.0, 0.5, 2.0], np.float32)
        off = torch.from_numpy(scale[slot] == 0).cuda()
        dev = [torch.from_numpy(np.ascontiguousarray(v)).cuda() for v in (xa, b.view(np.int16), slot, scale)]
        x = activations(m, "x", m, k)
        xd, base = to_dev(x), want_of(x)
        for mat, silu, whole in ((plain, False, False), (plain, False, True), (gated, True, False)):
            print(f"adapter {kind} {n}x{k} rank={rank} m={m} silu={silu} whole={whole}", flush=True)
            tab = tabs[silu]
            lora = (dev[0], split, 2 * rank, dev[1], rank, torch.tensor(tab, dtype=torch.int32, device="cuda"), dev[2],
                    dev[3])
            if silu:
                y, ref = (torch.full((m, n // 2), float("nan"), dtype=torch.bfloat16, device="cuda") for _ in range(2))
                gemm.run(None, m, mat, xd, ref, Epi.Silu)
                gemm.run_lora(None, m, mat, xd, y, Epi.Silu, lora)
                torch.cuda.synchronize()
                want = oracle.lora_silu(base[:, row_order(n, True)], xa, split, b.view(np.uint16), rank, tab, slot, scale, m)
                assert bf16_out_err(y.float().cpu().numpy(), want) <= 1e-3, m
                assert torch.equal(y.view(torch.int16)[off], ref.view(torch.int16)[off]), m
                continue
            s = 1 if whole else mat.split(m)
            y, ref = (torch.full((s, m, n), float("nan"), device="cuda") for _ in range(2))
            assert gemm.run_split(None, m, mat, xd, ref, Epi.Plain, whole) == s
            assert gemm.run_lora(None, m, mat, xd, y, Epi.Plain, lora, whole) == s
            torch.cuda.synchronize()
            want = oracle.lora_add(base, xa, split, b.view(np.uint16), rank, tab, slot, scale, m)
            assert rel_err(y.double().sum(0).cpu().numpy(), want) <= 1e-4, (m, whole)
            y, ref = y.view(torch.int32), ref.view(torch.int32)
            assert torch.equal(y[:, off], ref[:, off]) and torch.equal(y[:, :, end:], ref[:, :, end:]), (m, whole)
