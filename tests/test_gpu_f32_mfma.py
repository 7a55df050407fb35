"""The fp32 MFMA kernels at the edges of their tiles (GPU only): the GEMM's
32 x 32 and ring tiles on integer operands (exact), and the flash prefill
against the float64 softmax, with values that are not finite where no query may
see them.

Attention tolerance: scores are fp32 chains of D products of N(0, 1) values
(error about sqrt(D) 2^-24 of their size), each probability one expf (1 ulp) of
a score at most ~8 and sums of positive terms: 2e-6 of the largest output covers
them with a factor of four to spare.
"""
from __future__ import annotations

import ctypes

import numpy as np
import pytest

from schedforge_amd import _abi
from schedforge_amd._abi import BF16, EPI_GLU_SILU_UP, EPI_NONE, EPI_RESIDUAL, EPI_SWIGLU, F32

from _helpers import KEEP_ALIVE, bf16_host, dev, host, stream
from test_gpu_gemm_random import _args, _check, _epilogue, _weights

pytestmark = pytest.mark.gpu
torch = pytest.importorskip("torch")


# 32 x 32 tiles and their edges, fewer slabs than waves, K not a whole slab or
# 16-byte chunk (the VALU kernel), then products large enough for the ring tiles
@pytest.mark.parametrize("m,n,k", [(1, 1, 4), (1, 33, 36), (31, 64, 32), (33, 65, 160), (128, 688, 256), (128, 256, 688),
                                   (40, 24, 30), (700, 1000, 100), (1025, 1030, 68), (1500, 2064, 36)])
def test_f32_gemm_is_exact(m, n, k):
    lib = _abi.load()
    rng = np.random.default_rng(m + n * 3 + k * 7)
    a = rng.integers(-3, 4, size=(m, k)).astype(np.float32)
    res = rng.integers(-5, 6, size=(m, n)).astype(np.float32)
    ad, rd = dev(a), dev(res)
    for epi, c_dtype in ((EPI_NONE, BF16), (EPI_RESIDUAL, F32), (EPI_SWIGLU, F32), (EPI_GLU_SILU_UP, F32)):
        glu = epi in (EPI_SWIGLU, EPI_GLU_SILU_UP)
        bd, b_dtype, _, bm = _weights(rng, "f32", (2 * n if glu else n,), k, 0)
        out = torch.full((m, n), 77, dtype=torch.float32 if c_dtype == F32 else torch.int16, device="cuda")
        KEEP_ALIVE.append(out)
        args = _args(ad, F32, bd, b_dtype, None, out, c_dtype, rd if epi == EPI_RESIDUAL else None, m, n, k, epi, 0, 0)
        _abi.check(lib.sfg_hip_gemm_v1(ctypes.byref(args), None, 0, stream()))
        torch.cuda.synchronize()
        ref = _epilogue(a.astype(np.float64) @ bm.T, epi, n, res).astype(np.float32)
        _check(out, c_dtype, ref, glu, f"{m}x{n}x{k} epi {epi}")


@pytest.mark.parametrize("counts,n,k", [((0, 1, 33, 7), 40, 100), ((700, 0, 3, 300), 1000, 64)])
def test_f32_grouped_gemm_is_exact(counts, n, k):
    lib = _abi.load()
    rng = np.random.default_rng(n + k)
    groups, m, t = len(counts), sum(counts), 90
    offsets = np.concatenate([[0], np.cumsum(counts)]).astype(np.int32)
    a = rng.integers(-3, 4, size=(t, k)).astype(np.float32)
    rows = rng.integers(0, t, size=m).astype(np.int32)
    rows[::13] = t + 1
    arow = np.where((rows < t)[:, None], a[np.clip(rows, 0, t - 1)], 0).astype(np.float64)
    for epi in (EPI_NONE, EPI_GLU_SILU_UP):
        nb = 2 * n if epi != EPI_NONE else n
        bd, b_dtype, _, bm = _weights(rng, "f32", (groups, nb), k, 0)
        out = torch.full((m, n), 77, dtype=torch.float32, device="cuda")
        KEEP_ALIVE.append(out)
        args = _args(dev(a), F32, bd, b_dtype, None, out, F32, None, m, n, k, epi, 0, 0)
        _abi.check(lib.sfg_hip_gemm_grouped_v1(ctypes.byref(args), dev(rows).data_ptr(), t, dev(offsets).data_ptr(),
                                               groups, nb * k, 0, None, 0, stream()))
        torch.cuda.synchronize()
        acc = np.concatenate([arow[offsets[g]:offsets[g + 1]] @ bm[g].T for g in range(groups)])
        _check(out, F32, _epilogue(acc, epi, n).astype(np.float32), epi != EPI_NONE, f"{counts} epi {epi}")


# (batch, q heads, kv heads, queries, keys, D, causal): block and tile edges, the
# causal offset, both key-split forms (64-row blocks under and over 256), GQA
@pytest.mark.parametrize("b,hq,hkv,sq,skv,d,causal", [
    (1, 1, 1, 1, 1, 64, 1), (1, 2, 1, 33, 33, 64, 1), (2, 4, 2, 128, 128, 64, 1), (1, 4, 4, 5, 300, 64, 1),
    (1, 2, 1, 130, 97, 64, 0), (3, 16, 4, 390, 390, 64, 1), (1, 2, 2, 65, 65, 128, 1), (2, 4, 1, 200, 260, 128, 1),
    (1, 3, 3, 70, 31, 128, 0)])
@pytest.mark.parametrize("poison", [False, True])
def test_f32_flash_prefill(b, hq, hkv, sq, skv, d, causal, poison):
    if poison and not causal:
        pytest.skip("every query sees every key")
    lib = _abi.load()
    rng = np.random.default_rng(sq * 31 + skv + d)
    q, k, v = (rng.standard_normal(s).astype(np.float32) for s in ((b, hq, sq, d), (b, hkv, skv, d), (b, hkv, skv, d)))
    if poison:  # the last key: only the last query sees it
        v[:, :, -1, ::3] = np.inf
        v[:, :, -1, 1::3] = np.nan
        k[:, :, -1, 0] = -np.inf
    qd, kd, vd = dev(q), dev(k), dev(v)
    rows = sq - 1 if poison else sq
    ref = np.empty((b, sq, hq, d))
    hide = np.arange(skv)[None, :] > (skv - sq + np.arange(sq))[:, None] if causal else np.zeros((sq, skv), bool)
    for n in range(b):
        for h in range(hq):
            with np.errstate(invalid="ignore", over="ignore"):
                s = q[n, h].astype(np.float64) @ k[n, h * hkv // hq].astype(np.float64).T / np.sqrt(d)
            s[hide] = -np.inf
            p = np.exp(s[:rows] - s[:rows].max(axis=1, keepdims=True))
            ref[n, :rows, h] = (p / p.sum(axis=1, keepdims=True)) @ np.where(np.isfinite(v[n, h * hkv // hq]), v[n, h * hkv // hq], 0)
    for out_dtype in (F32, BF16):
        out = torch.zeros((b, sq, hq, d), dtype=torch.float32 if out_dtype == F32 else torch.int16, device="cuda")
        KEEP_ALIVE.append(out)
        _abi.check(lib.sfg_hip_attn_prefill_v1(qd.data_ptr(), kd.data_ptr(), vd.data_ptr(), out.data_ptr(), F32, out_dtype,
                                               b, hq, hkv, sq, skv, d, causal, ctypes.c_float(0.0), stream()))
        torch.cuda.synchronize()
        got = (host(out) if out_dtype == F32 else bf16_host(out))[:, :rows]
        err = np.abs(got - ref[:, :rows]).max(initial=0.0) / max(np.abs(ref[:, :rows]).max(initial=0.0), 1e-6)
        assert err < (2e-6 if out_dtype == F32 else 4e-3), (err, out_dtype)


# either side of the line to the row kernel: keys of one round of workgroups (60 and
# 150), one round and two (blocks of four rows over 256), short keys in many rounds
@pytest.mark.parametrize("b,hq,hkv,sq,skv,d,causal", [
    (1, 2, 1, 60, 60, 64, 1), (1, 2, 1, 61, 61, 64, 1), (2, 2, 2, 150, 150, 128, 1), (2, 2, 1, 151, 151, 128, 0),
    (8, 8, 4, 16, 16, 64, 1), (8, 8, 2, 17, 33, 64, 1), (16, 8, 8, 22, 22, 128, 1), (16, 8, 2, 9, 23, 128, 1),
    (40, 16, 4, 1, 1, 64, 1), (40, 16, 4, 5, 7, 128, 0)])
def test_f32_prefill_at_the_row_kernels_line(b, hq, hkv, sq, skv, d, causal):
    test_f32_flash_prefill(b, hq, hkv, sq, skv, d, causal, False)
    if causal:
        test_f32_flash_prefill(b, hq, hkv, sq, skv, d, causal, True)
