"""The middle-size GEMM (65 rows up, bf16 or int8 weights) at the edges of its
tiles and slabs (GPU only): rows and columns one past a tile, a K of one slab,
of half a slab more, of fewer slabs than the LDS ring holds, with the split-K
workspace, one too small for the split it would take, and none.  Integer
operands, so every value is exact whatever the tile, split or order.
"""
from __future__ import annotations

import ctypes

import numpy as np
import pytest

from schedforge_amd import _abi
from schedforge_amd._abi import BF16, EPI_GLU_SILU_UP, EPI_NONE, EPI_RESIDUAL, EPI_SWIGLU, F32

from _helpers import KEEP_ALIVE, bf16_dev, dev, host, stream, tile_nk
from test_gpu_gemm_random import _args, _check, _epilogue, _weights

pytestmark = pytest.mark.gpu
torch = pytest.importorskip("torch")

# (m, n, k): tile edges of 64 / 128 / 256 rows and 64 / 128 columns, one slab, a
# half slab, ring depths 3 .. 6, splits (short and wide, long K), 1024 rows up
DENSE = [(65, 64, 32), (65, 68, 64), (128, 132, 96), (129, 1, 160), (257, 65, 352), (100, 512, 1376),
         (200, 516, 2816), (512, 256, 4096), (1023, 130, 416), (1025, 1028, 224), (1300, 2052, 96)]


@pytest.mark.parametrize("kind", ["bf16", "i8"])
@pytest.mark.parametrize("m,n,k", DENSE)
def test_ring_dense_is_exact(m, n, k, kind):
    lib = _abi.load()
    rng = np.random.default_rng(m * 7 + n * 3 + k)
    a = rng.integers(-3, 4, size=(m, k)).astype(np.float32)
    res = rng.integers(-5, 6, size=(m, n)).astype(np.float32)
    ad, rd = bf16_dev(a), dev(res)
    full = lib.sfg_hip_gemm_workspace_v1(m, n, k)
    for epi, c_dtype in ((EPI_NONE, F32), (EPI_RESIDUAL, F32), (EPI_SWIGLU, BF16), (EPI_GLU_SILU_UP, F32)):
        glu = epi in (EPI_SWIGLU, EPI_GLU_SILU_UP)
        bd, b_dtype, sd, bm = _weights(rng, kind, (2 * n if glu else n,), k, 0)
        ref = _epilogue(a.astype(np.float64) @ bm.T, epi, n, res).astype(np.float32)
        for ws_bytes in sorted({0, full // 3, full}):
            label = f"{kind} {m}x{n}x{k} epi {epi} workspace {ws_bytes}"
            print(label, flush=True)
            out = torch.full((m, n), 77, dtype=torch.float32 if c_dtype == F32 else torch.int16, device="cuda")
            ws = torch.empty(max(ws_bytes, 1), dtype=torch.uint8, device="cuda")
            KEEP_ALIVE.extend([out, ws])
            args = _args(ad, BF16, bd, b_dtype, sd, out, c_dtype, rd if epi == EPI_RESIDUAL else None, m, n, k, epi, 0, 0)
            _abi.check(lib.sfg_hip_gemm_v1(ctypes.byref(args), ws.data_ptr() if ws_bytes else None, ws_bytes, stream()))
            torch.cuda.synchronize()
            _check(out, c_dtype, ref, glu, label)


# groups of no row, one row and one past a tile; ids outside A read zero rows
# (layout 1: fragment-tiled weights, up to 512 rows in all)
@pytest.mark.parametrize("kind", ["bf16", "i8"])
@pytest.mark.parametrize("counts,n,k,layout", [((0, 65, 1, 500), 64, 96, 0), ((600, 0, 0, 129, 3), 192, 1376, 0),
                                               ((257, 300, 255, 1, 0, 64, 200), 1408, 160, 0), ((0, 65, 1, 200), 64, 128, 1),
                                               ((300, 0, 129, 3), 208, 384, 1), ((100, 412), 16, 1408, 1)])
def test_ring_grouped_is_exact(counts, n, k, layout, kind):
    lib = _abi.load()
    rng = np.random.default_rng(n + k)
    groups, m, t = len(counts), sum(counts), 300
    offsets = np.concatenate([[0], np.cumsum(counts)]).astype(np.int32)
    a = rng.integers(-3, 4, size=(t, k)).astype(np.float32)
    rows = rng.integers(0, t, size=m).astype(np.int32)
    rows[::17] = -1
    rows[5::31] = t
    valid = (rows >= 0) & (rows < t)
    arow = np.where(valid[:, None], a[np.clip(rows, 0, t - 1)], 0).astype(np.float64)
    for epi in (EPI_NONE, EPI_GLU_SILU_UP):
        nb = 2 * n if epi != EPI_NONE else n
        bd, b_dtype, sd, bm = _weights(rng, kind, (groups, nb), k, 0)
        if layout:
            w = host(bd).reshape(groups, nb, k)
            bd = dev(np.stack([tile_nk(w[g], "int8" if kind == "i8" else "bf16") for g in range(groups)]))
        out = torch.full((m, n), 77, dtype=torch.float32, device="cuda")
        KEEP_ALIVE.append(out)
        args = _args(bf16_dev(a), BF16, bd, b_dtype, sd, out, F32, None, m, n, k, epi, layout, 0)
        _abi.check(lib.sfg_hip_gemm_grouped_v1(ctypes.byref(args), dev(rows).data_ptr(), t, dev(offsets).data_ptr(),
                                               groups, nb * k, nb if sd is not None else 0, None, 0, stream()))
        torch.cuda.synchronize()
        acc = np.concatenate([arow[offsets[g]:offsets[g + 1]] @ bm[g].T for g in range(groups)])
        _check(out, F32, _epilogue(acc, epi, n).astype(np.float32), epi != EPI_NONE, f"{kind} {counts} epi {epi}")


# the fused split + RoPE epilogue where sequences end inside a lane's run of four
# rows: shortest sequences, one row past a tile, rows under and over 1024 (where a
# named tile, or the 256 x 256 tile, takes the separate pass), int8
@pytest.mark.parametrize("dtype,batch,seq", [("bf16", 40, 5), ("bf16", 3, 43), ("w8", 9, 29), ("w8", 2, 777),
                                             ("bf16", 1, 1031), ("bf16", 5, 257), ("w8", 16, 4), ("bf16", 30, 3)])
def test_qkv_epilogue_on_ragged_sequences(dtype, batch, seq):
    import oracle
    from schedforge_amd import CONFIGS
    from schedforge_amd.layer import compile_decoder, execute_decoder_layer
    from _helpers import TOL, decoder_data
    cfg = CONFIGS["c4"].replace(batch=batch, sequence=seq, hidden=512, intermediate=1024, query_heads=4, kv_heads=2,
                                dtype=dtype)
    d = oracle.make_layer_data(cfg, 4100 + seq)
    plan = compile_decoder(cfg, decoder_data(d), "cuda")
    out = execute_decoder_layer(plan, d.input, warmup=0, repetitions=1).output
    assert oracle.rel_error(out, oracle.decoder_layer(cfg, d)) < TOL[dtype]
    if dtype == "bf16":  # the same bits as a tile named by the plan
        plan.desc.gemm_tile = _abi.TILE_128x128
        assert np.array_equal(execute_decoder_layer(plan, d.input, warmup=0, repetitions=1).output, out)


# weights that do not start on 16 bytes: the fused epilogue's tiles read whole
# 16-byte vectors, so such a layer takes the separate split + RoPE pass
@pytest.mark.parametrize("dtype,batch,seq", [("bf16", 2, 40), ("bf16", 4, 257), ("w8", 2, 40)])
def test_prefill_layer_with_unaligned_qkv_weights(dtype, batch, seq):
    import oracle
    from schedforge_amd import CONFIGS
    from schedforge_amd.layer import compile_decoder, execute_decoder_layer
    from _helpers import TOL, decoder_data
    cfg = CONFIGS["c4"].replace(batch=batch, sequence=seq, hidden=512, intermediate=512, query_heads=4, kv_heads=2,
                                dtype=dtype)
    d = oracle.make_layer_data(cfg, 4300 + seq)
    plan = compile_decoder(cfg, decoder_data(d), "cuda")
    w = plan.t["w_qkv"].reshape(-1)
    off = 1 if dtype == "bf16" else 2  # elements: 2 bytes either way
    moved = torch.empty(w.numel() + 16, dtype=w.dtype, device="cuda")
    moved[off:off + w.numel()] = w
    KEEP_ALIVE.append(moved)
    plan.weights.w_qkv = moved.data_ptr() + 2
    out = execute_decoder_layer(plan, d.input, warmup=0, repetitions=1).output
    assert oracle.rel_error(out, oracle.decoder_layer(cfg, d)) < TOL[dtype]
