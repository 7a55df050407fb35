"""Paged attention of several query rows per sequence on the matrix cores (GPU
only): column-block edges (1 .. 70 rows per kv head), GQA groups the one-row
kernel does not take, both head dims, ragged lengths with an empty sequence and
rows that see no key, an unaligned query (the row kernel), 1 split to more than
there are pages, and pool contents that no row may see: stale tokens past the
end and hidden tokens that are not finite.

Q and the probabilities keep fp32 precision, so the tolerance is the fp32 one:
scores of D products (error sqrt(D) 2^-24 of their size), expf at 1 ulp, sums of
positive terms -- 3e-6 of the largest output, four times what those add up to.
"""
from __future__ import annotations

import ctypes

import numpy as np
import pytest

import oracle
from schedforge_amd import _abi
from schedforge_amd._abi import BF16, F32

from _helpers import KEEP_ALIVE, bf16_dev, dev, host, stream

pytestmark = pytest.mark.gpu
torch = pytest.importorskip("torch")
PT = 16

# (q heads, kv heads, rows, D, longest, causal, splits, unaligned, poison)
CASES = [(4, 4, 2, 128, 33, 1, 0, False, False), (16, 4, 4, 128, 1000, 1, 0, False, True),
         (16, 4, 5, 128, 300, 1, 3, False, True), (6, 2, 1, 64, 200, 1, 0, False, False),
         (12, 2, 7, 64, 120, 1, 40, False, True), (35, 5, 10, 128, 90, 1, 2, False, True),
         (4, 1, 3, 64, 50, 0, 1, False, False), (8, 2, 6, 128, 64, 1, 0, True, True),
         (32, 1, 2, 128, 500, 1, 0, False, True)]


@pytest.mark.parametrize("pool", ["bf16", "f32"])
@pytest.mark.parametrize("hq,hkv,sq,d,longest,causal,splits,unaligned,poison", CASES)
def test_paged_rows_on_the_matrix_cores(hq, hkv, sq, d, longest, causal, splits, unaligned, poison, pool):
    lib = _abi.load()
    rng = np.random.default_rng(hq * 7 + sq * 3 + longest)
    lens = np.array([longest, 0, 1, max(1, sq - 1), rng.integers(1, longest + 1)], np.int32)
    b, pps = len(lens), (longest + PT - 1) // PT
    pages = b * pps + 3
    table = rng.permutation(pages)[: b * pps].reshape(b, pps).astype(np.int32)
    kp, vp = (rng.standard_normal(s).astype(np.float32) for s in ((pages, hkv, PT, d), (pages, hkv, d, PT)))
    if pool == "bf16":
        kp, vp = oracle.round_bf16(kp), oracle.round_bf16(vp)
    q = rng.standard_normal((b, hq, sq, d)).astype(np.float32)
    rows_seen = np.full(b, sq)  # rows compared
    if poison:
        for n in range(b):
            for t in range(lens[n], pps * PT):  # past the end: anything
                kp[table[n, t // PT], :, t % PT] = np.nan
                vp[table[n, t // PT], :, :, t % PT] = np.inf if t % 2 else np.nan
            if lens[n] > sq > 1:  # the last key: only the last row sees it
                t = lens[n] - 1
                vp[table[n, t // PT], :, ::2, t % PT] = -np.inf
                vp[table[n, t // PT], :, 1::2, t % PT] = np.nan
                rows_seen[n] = sq - 1
    ref = np.full((b, hq, sq, d), np.nan)
    for n in range(b):
        L = int(lens[n])
        k = kp[table[n]].transpose(1, 0, 2, 3).reshape(hkv, -1, d)[:, :L].astype(np.float64)
        v = vp[table[n]].transpose(1, 0, 3, 2).reshape(hkv, -1, d)[:, :L].astype(np.float64)
        for h in range(hq):
            for i in range(rows_seen[n]):
                end = min(L, L - sq + i + 1) if causal else L
                if end <= 0:
                    continue
                j = h * hkv // hq
                s = (k[j, :end] @ q[n, h, i].astype(np.float64)) / np.sqrt(d)
                p = np.exp(s - s.max())
                ref[n, h, i] = (p / p.sum()) @ v[j, :end]
    buf = torch.zeros(q.size + 4, device="cuda")
    qd = buf[1:1 + q.size] if unaligned else buf[:q.size]
    qd.copy_(dev(q).reshape(-1))
    kv_dtype, to = (F32, dev) if pool == "f32" else (BF16, bf16_dev)
    kd, vd, td, ld = to(kp), to(vp), dev(table), dev(lens)
    out = torch.zeros((b, hq, sq, d), device="cuda")
    ws = torch.full((max(1, lib.sfg_hip_attn_paged_workspace_v1(b, hq, hkv, sq, d, kv_dtype, longest, PT, splits)),), 255,
                    dtype=torch.uint8, device="cuda")
    KEEP_ALIVE.extend([buf, out, ws])
    _abi.check(lib.sfg_hip_attn_paged_v1(
        qd.data_ptr(), kd.data_ptr(), vd.data_ptr(), kv_dtype, td.data_ptr(), ld.data_ptr(), out.data_ptr(), F32, b, hq, hkv,
        sq, d, PT, pps, pages, longest, int(causal and sq <= longest), splits, ctypes.c_float(0.0), 0, ws.data_ptr(),
        ws.numel(), stream()))
    torch.cuda.synchronize()
    got = host(out)
    for n in range(b):
        g, r = got[n, :, :rows_seen[n]], ref[n, :, :rows_seen[n]]
        np.testing.assert_array_equal(np.isnan(g), np.isnan(r), err_msg=f"sequence {n}")
        if np.isfinite(r).any():
            err = np.nanmax(np.abs(g - r)) / max(np.nanmax(np.abs(r)), 1e-6)
            assert err < 3e-6, (n, err)


def _reference(q, kp, vp, table, lens, causal):
    """softmax(q k / sqrt(d)) v in float64, infinities and NaN as they come."""
    b, hq, sq, d = q.shape
    hkv = kp.shape[1]
    ref = np.full(q.shape, np.nan)
    with np.errstate(invalid="ignore", over="ignore"):
        for n in range(b):
            L = int(lens[n])
            k = kp[table[n]].transpose(1, 0, 2, 3).reshape(hkv, -1, d)[:, :L].astype(np.float64)
            v = vp[table[n]].transpose(1, 0, 3, 2).reshape(hkv, -1, d)[:, :L].astype(np.float64)
            for h in range(hq):
                j = h * hkv // hq
                for i in range(sq):
                    end = min(L, L - sq + i + 1) if causal else L
                    s = (k[j, :end] * q[n, h, i].astype(np.float64)).sum(axis=1) / np.sqrt(d)
                    p = np.exp(s - s.max())
                    ref[n, h, i] = ((p / p.sum())[:, None] * v[j, :end]).sum(axis=0)
    return ref


def _run_paged(q, kp, vp, table, lens, causal, splits, pool):
    lib = _abi.load()
    b, hq, sq, d = q.shape
    pages, hkv = kp.shape[:2]
    longest, pps = int(lens.max()), table.shape[1]
    kv_dtype, to = (F32, dev) if pool == "f32" else (BF16, bf16_dev)
    qd, kd, vd, td, ld = dev(q), to(kp), to(vp), dev(table), dev(lens)
    out = torch.zeros(q.shape, device="cuda")
    n = lib.sfg_hip_attn_paged_workspace_v1(b, hq, hkv, sq, d, kv_dtype, longest, PT, splits)
    ws = torch.full((max(1, n),), 255, dtype=torch.uint8, device="cuda")
    KEEP_ALIVE.extend([out, ws])
    _abi.check(lib.sfg_hip_attn_paged_v1(
        qd.data_ptr(), kd.data_ptr(), vd.data_ptr(), kv_dtype, td.data_ptr(), ld.data_ptr(), out.data_ptr(), F32, b, hq, hkv,
        sq, d, PT, pps, pages, longest, causal, splits, ctypes.c_float(0.0), 0, ws.data_ptr(), ws.numel(), stream()))
    torch.cuda.synchronize()
    return host(out)


def _check_non_finite(got, ref):
    np.testing.assert_array_equal(np.isnan(got), np.isnan(ref))
    inf = np.isinf(ref)
    np.testing.assert_array_equal(got[inf], ref[inf])
    fin = np.isfinite(ref)
    assert np.isfinite(got[fin]).all()
    assert np.abs(got[fin] - ref[fin]).max() < 3e-6 * np.abs(ref[fin]).max()


def _random_pools(rng, b, hq, hkv, sq, d, longest, pool):
    pps = (longest + PT - 1) // PT
    table = rng.permutation(b * pps).reshape(b, pps).astype(np.int32)
    kp, vp = (rng.standard_normal(s).astype(np.float32) for s in ((b * pps, hkv, PT, d), (b * pps, hkv, d, PT)))
    if pool == "bf16":
        kp, vp = oracle.round_bf16(kp), oracle.round_bf16(vp)
    return table, kp, vp, rng.standard_normal((b, hq, sq, d)).astype(np.float32)


# sequence 0: keys of -inf against positive query elements (exact in bf16 and not),
# weight 0; 1: infinite values; 2: both, on every page; 3: a key of +inf, so NaN;
# 4: a query element above the largest bf16 against tiny key elements
@pytest.mark.parametrize("pool", ["bf16", "f32"])
@pytest.mark.parametrize("hq,hkv,sq,d,longest,causal,splits", [(16, 4, 2, 128, 300, 1, 0), (8, 2, 5, 64, 70, 1, 1),
                                                               (12, 2, 3, 128, 130, 0, 3), (34, 2, 1, 64, 200, 1, 0)])
def test_visible_infinities_give_the_reference_result(hq, hkv, sq, d, longest, causal, splits, pool):
    rng = np.random.default_rng(d + longest)
    b = 5
    table, kp, vp, q = _random_pools(rng, b, hq, hkv, sq, d, longest, pool)
    lens = np.array([longest, longest - 1, longest, longest - 3, longest], np.int32)
    q[..., 3] = 1.0
    q[..., 9] = np.abs(q[..., 9]) + 0.1
    q[4, ..., 5] = 3.4e38
    for n, keys, values in ((0, 0, None), (1, None, 0), (2, 0, 3)):
        for t in range(0, lens[n] - sq - 3, 7):  # tokens that every row sees
            if keys is not None:
                kp[table[n, t // PT], :, t % PT, 3 if t % 2 else 9] = -np.inf
            if values is not None:
                pg, at = table[n, (t + values) // PT], (t + values) % PT
                vp[pg, :, 1::5, at] = np.inf
                vp[pg, :, 2::5, at] = -np.inf
    kp[table[3, 1], :, 4, 9] = np.inf
    kp[table[4], ..., 5] = np.copysign(np.float32(2.0 ** -125), kp[table[4], ..., 5])
    ref = _reference(q, kp, vp, table, lens, causal)
    assert np.isfinite(ref[0]).all() and np.isinf(ref[1]).any() and np.isnan(ref[3]).all() and np.isfinite(ref[4]).all()
    _check_non_finite(_run_paged(q, kp, vp, table, lens, causal, splits, pool), ref)


def test_decode_workspace_covers_every_kv_head_count():
    """The one-row workspace query, which is not told the kv head count."""
    lib = _abi.load()
    for b, hq, ctx in ((1, 6, 5000), (4, 24, 900), (16, 48, 4096)):
        top = lib.sfg_hip_attn_decode_workspace_v1(b, hq, 128, ctx, PT, 0)
        for hkv in range(1, hq + 1):
            if hq % hkv == 0:
                need = lib.sfg_hip_attn_paged_workspace_v1(b, hq, hkv, 1, 128, BF16, ctx, PT, 0)
                assert need <= top, (b, hq, hkv, need, top)


@pytest.mark.parametrize("b,hkv,longest", [(1, 8, 127), (1, 8, 129), (1, 8, 4096), (8, 8, 2000), (3, 2, 700)])
def test_automatic_split_counts_match_one_split(b, hkv, longest):
    """One-row steps of small batches, whose automatic split count keeps as few
    as 8 pages a split: the same result as one split, within the rounding of the
    probabilities to bf16 (2^-9 of a sum of positive weights)."""
    lib = _abi.load()
    rng = np.random.default_rng(longest)
    hq, d, pps = 4 * hkv, 128, (longest + PT - 1) // PT
    table = rng.permutation(b * pps).reshape(b, pps).astype(np.int32)
    k, v = (bf16_dev(rng.standard_normal(s).astype(np.float32)) for s in ((b * pps, hkv, PT, d), (b * pps, hkv, d, PT)))
    lens = np.full(b, longest, np.int32)
    lens[-1] = max(1, longest // 9)
    q, td, ld = dev(rng.standard_normal((b, hq, 1, d)).astype(np.float32)), dev(table), dev(lens)
    outs = []
    for splits in (0, 1):
        n = lib.sfg_hip_attn_paged_workspace_v1(b, hq, hkv, 1, d, BF16, longest, PT, splits)
        out = torch.zeros((b, hq, d), device="cuda")
        ws = torch.full((max(1, n),), 255, dtype=torch.uint8, device="cuda")
        KEEP_ALIVE.extend([out, ws])
        _abi.check(lib.sfg_hip_attn_paged_v1(
            q.data_ptr(), k.data_ptr(), v.data_ptr(), BF16, td.data_ptr(), ld.data_ptr(), out.data_ptr(), F32, b, hq, hkv,
            1, d, PT, pps, b * pps, longest, 1, splits, ctypes.c_float(0.0), 0, ws.data_ptr(), ws.numel(), stream()))
        torch.cuda.synchronize()
        outs.append(host(out))
    np.testing.assert_allclose(outs[0], outs[1], atol=2.0 ** -8 * np.abs(outs[1]).max())


# batches whose last doubling of the splits would start a second round of workgroups:
# without lengths of their own they take as many splits as fit, powers of two or not
@pytest.mark.parametrize("b,hkv,longest,d", [(6, 16, 2206, 128), (24, 16, 276, 128), (3, 8, 4096, 128), (6, 16, 2206, 64),
                                             (40, 2, 1500, 128)])
def test_split_counts_of_equal_sequences_match_one_split(b, hkv, longest, d):
    lib = _abi.load()
    rng = np.random.default_rng(longest + b)
    hq, pps = hkv, (longest + PT - 1) // PT
    table = rng.permutation(b * pps).reshape(b, pps).astype(np.int32)
    k, v = (bf16_dev(rng.standard_normal(s).astype(np.float32)) for s in ((b * pps, hkv, PT, d), (b * pps, hkv, d, PT)))
    q, td, ld = dev(rng.standard_normal((b, hq, 1, d)).astype(np.float32)), dev(table), dev(np.full(b, longest, np.int32))
    outs = []
    for splits, lens in ((0, None), (0, ld.data_ptr()), (1, None)):
        n = lib.sfg_hip_attn_paged_workspace_v1(b, hq, hkv, 1, d, BF16, longest, PT, splits)
        out = torch.zeros((b, hq, d), device="cuda")
        ws = torch.full((max(1, n),), 255, dtype=torch.uint8, device="cuda")
        KEEP_ALIVE.extend([out, ws])
        _abi.check(lib.sfg_hip_attn_paged_v1(
            q.data_ptr(), k.data_ptr(), v.data_ptr(), BF16, td.data_ptr(), lens, out.data_ptr(), F32, b, hq, hkv,
            1, d, PT, pps, b * pps, longest, 1, splits, ctypes.c_float(0.0), 0, ws.data_ptr(), ws.numel(), stream()))
        torch.cuda.synchronize()
        outs.append(host(out))
    for got in outs[:2]:
        np.testing.assert_allclose(got, outs[2], atol=2.0 ** -8 * np.abs(outs[2]).max())
