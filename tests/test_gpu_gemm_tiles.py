"""Every tile that the launcher's estimate can choose for a tiled product (GPU
only), at ragged rows and columns and at depths of one slab, one and a half and
more than its LDS ring holds.  Each case first asks the estimate itself (compiled
from its header by the host compiler), so that a changed table shows here instead
of quietly moving a case to another tile.  Integer operands: every value exact.

Also the products whose operands end past 4 GiB, which run on the register-staged
kernels with 64-bit addresses, beside one that ends just under.
"""
from __future__ import annotations

import ctypes
import subprocess
from pathlib import Path

import numpy as np
import pytest

from schedforge_amd import _abi
from schedforge_amd._abi import BF16, EPI_GLU_SILU_UP, EPI_NONE, EPI_RESIDUAL, EPI_SWIGLU, F32, I8

from _helpers import KEEP_ALIVE, bf16_dev, dev, host, stream
from test_gpu_gemm_random import _args, _check, _epilogue, _weights

torch = pytest.importorskip("torch")

CSRC = Path(__file__).resolve().parents[1] / "schedforge_amd" / "csrc"
V, T256x128, T128x128, T64x128, T128x64, T64x64, SMALL, DMA = range(1, 9)
DT = {"f32": F32, "bf16": BF16, "i8": I8}

# (weights, tile, m, n, epilogue), each at the depths of DEPTHS
TILES = [
    ("i8", V, 861, 8257, EPI_RESIDUAL), ("i8", V, 810, 8401, EPI_NONE), ("i8", V, 300, 8423, EPI_SWIGLU),
    ("i8", T256x128, 399, 8574, EPI_RESIDUAL), ("i8", T256x128, 131, 8513, EPI_GLU_SILU_UP),
    ("i8", T128x128, 199, 8389, EPI_RESIDUAL), ("i8", T128x128, 72, 8284, EPI_SWIGLU),
    ("i8", T128x64, 70, 67, EPI_NONE), ("i8", T64x128, 70, 65, EPI_SWIGLU), ("i8", T64x64, 1043, 67, EPI_RESIDUAL),
    ("bf16", T256x128, 396, 8304, EPI_NONE), ("bf16", T256x128, 135, 8512, EPI_SWIGLU),
    ("bf16", T128x128, 5450, 266, EPI_RESIDUAL), ("bf16", T128x128, 71, 8246, EPI_GLU_SILU_UP),
    ("bf16", T64x128, 67, 66, EPI_RESIDUAL), ("bf16", T128x64, 343, 5419, EPI_NONE), ("bf16", T64x64, 1113, 70, EPI_RESIDUAL),
    ("f32", T256x128, 835, 7020, EPI_RESIDUAL), ("f32", T256x128, 208, 8197, EPI_SWIGLU),
    ("f32", T128x128, 321, 8238, EPI_RESIDUAL), ("f32", T128x128, 73, 8446, EPI_GLU_SILU_UP),
    ("f32", T64x128, 69, 8302, EPI_NONE), ("f32", T64x128, 5628, 65, EPI_SWIGLU), ("f32", T64x64, 67, 2793, EPI_RESIDUAL),
    ("f32", SMALL, 68, 69, EPI_RESIDUAL), ("f32", SMALL, 67, 66, EPI_SWIGLU),
]
DEPTHS = {"i8": (64, 96, 416), "bf16": (64, 96, 416), "f32": (68, 100, 260)}
# the direct-to-LDS tiles take whole 64-k slabs
WHOLE = [("bf16", V, 790, 8339, EPI_RESIDUAL, 192), ("bf16", V, 1026, 3613, EPI_SWIGLU, 704), ("bf16", V, 1031, 7196, EPI_NONE, 704),
         ("bf16", DMA, 1291, 5901, EPI_NONE, 64), ("bf16", DMA, 5898, 1321, EPI_RESIDUAL, 64),
         ("bf16", DMA, 2194, 1795, EPI_GLU_SILU_UP, 64)]
CASES = [(k, t, m, n, e, d) for k, t, m, n, e in TILES for d in DEPTHS[k]] + WHOLE


@pytest.fixture(scope="module")
def estimate(tmp_path_factory):
    d = tmp_path_factory.mktemp("plan")
    (d / "plan.cpp").write_text(
        f'#include "{CSRC / "sfg_gemm_plan.hpp"}"\n'
        'extern "C" int tile(int dt, int64_t m, int64_t n, int64_t k, int epi, int c, int groups, int qkv) {\n'
        '    const bool v = dt == SFG_BF16 || (dt == SFG_I8 && !qkv), dma = dt == SFG_BF16 && !qkv;\n'
        '    return sfg::ring_plan(sfg::RingAsk{dt, m, n, k, epi, c, groups, false, v, dma, 0}).tile; }\n')
    subprocess.run(["g++", "-std=c++20", "-O1", "-shared", "-fPIC", str(d / "plan.cpp"), "-o", str(d / "plan.so")], check=True)
    fn = ctypes.CDLL(str(d / "plan.so")).tile
    fn.argtypes = [ctypes.c_int, ctypes.c_int64, ctypes.c_int64, ctypes.c_int64, *[ctypes.c_int] * 4]
    return lambda *a, qkv=0: fn(*a, qkv)


@pytest.mark.parametrize("kind,tile,m,n,epi,k", CASES)
def test_the_estimate_chooses_the_tile(estimate, kind, tile, m, n, epi, k):
    assert estimate(DT[kind], m, n, k, epi, F32, 1) == tile


def test_the_estimate_chooses_a_tile_for_any_product(estimate):
    """From 65 rows up (fp32: any), whatever the sizes, groups and output type."""
    rng = np.random.default_rng(7)
    for _ in range(4000):
        dt = int(rng.choice([F32, BF16, I8]))
        m, n = (int(np.exp(rng.uniform(0, 17))) for _ in range(2))
        k = int(np.exp(rng.uniform(0, 10))) * (4 if dt == F32 else 32)
        t = estimate(dt, m if dt == F32 else m + 64, n, k, int(rng.integers(0, 4)), int(rng.choice([F32, BF16])),
                     int(rng.choice([1, 1, 2, 8, 64])))
        assert V <= t <= DMA, (dt, m, n, k)


@pytest.mark.gpu
@pytest.mark.parametrize("kind,tile,m,n,epi,k", CASES)
def test_tile_is_exact(estimate, kind, tile, m, n, epi, k):
    assert estimate(DT[kind], m, n, k, epi, F32, 1) == tile
    lib = _abi.load()
    rng = np.random.default_rng(m + 3 * n + k)
    a = rng.integers(-3, 4, size=(m, k)).astype(np.float32)
    res = rng.integers(-5, 6, size=(m, n)).astype(np.float32) if epi == EPI_RESIDUAL else None
    glu = epi in (EPI_SWIGLU, EPI_GLU_SILU_UP)
    bd, b_dtype, sd, bm = _weights(rng, kind, (2 * n if glu else n,), k, 0)
    ad = dev(a) if kind == "f32" else bf16_dev(a)
    ref = _epilogue((torch.from_numpy(a).cuda().double() @ torch.from_numpy(bm).cuda().double().T).cpu().numpy(), epi, n, res)
    out = torch.full((m, n), 77, dtype=torch.float32, device="cuda")
    KEEP_ALIVE.append(out)
    args = _args(ad, F32 if kind == "f32" else BF16, bd, b_dtype, sd, out, F32, dev(res) if res is not None else None, m, n, k,
                 epi, 0, 0)
    _abi.check(lib.sfg_hip_gemm_v1(ctypes.byref(args), None, 0, stream()))
    torch.cuda.synchronize()
    _check(out, F32, ref.astype(np.float32), glu, f"{kind} {m}x{n}x{k} epi {epi}")


# the 256 x 256 tile's bf16 stores: GLU rows through the stages that held the last
# slab (odd widths: rows that start off 16 bytes), residual in pairs of half blocks
@pytest.mark.gpu
@pytest.mark.parametrize("kind,m,n,epi,k", [("i8", 300, 8423, EPI_SWIGLU, 64), ("i8", 300, 8424, EPI_GLU_SILU_UP, 416),
                                            ("i8", 861, 8257, EPI_RESIDUAL, 96), ("bf16", 1300, 3613, EPI_SWIGLU, 704)])
def test_256x256_bf16_stores(estimate, kind, m, n, epi, k):
    assert estimate(DT[kind], m, n, k, epi, BF16, 1) == V
    lib = _abi.load()
    rng = np.random.default_rng(m + 5 * n + k)
    a = rng.integers(-3, 4, size=(m, k)).astype(np.float32)
    res = rng.integers(-5, 6, size=(m, n)).astype(np.float32)
    glu = epi != EPI_RESIDUAL
    bd, b_dtype, sd, bm = _weights(rng, kind, (2 * n if glu else n,), k, 0)
    ref = _epilogue((torch.from_numpy(a).cuda().double() @ torch.from_numpy(bm).cuda().double().T).cpu().numpy(), epi, n, res)
    out = torch.full((m, n), 77, dtype=torch.int16, device="cuda")
    KEEP_ALIVE.append(out)
    args = _args(bf16_dev(a), BF16, bd, b_dtype, sd, out, BF16, dev(res) if not glu else None, m, n, k, epi, 0, 0)
    _abi.check(lib.sfg_hip_gemm_v1(ctypes.byref(args), None, 0, stream()))
    torch.cuda.synchronize()
    _check(out, BF16, ref.astype(np.float32), glu, f"{kind} {m}x{n}x{k} epi {epi}")


# int8 experts whose products take the 256 x 256 tile
@pytest.mark.gpu
@pytest.mark.parametrize("epi", [EPI_NONE, EPI_GLU_SILU_UP])
def test_grouped_int8_256x256_is_exact(estimate, epi):
    lib = _abi.load()
    counts, n, k = (700, 0, 1300, 257), 4224, 416
    assert estimate(I8, sum(counts), n, k, epi, F32, len(counts)) == V
    rng = np.random.default_rng(n + k + epi)
    groups, m, t = len(counts), sum(counts), 300
    offsets = np.concatenate([[0], np.cumsum(counts)]).astype(np.int32)
    a = rng.integers(-3, 4, size=(t, k)).astype(np.float32)
    rows = rng.integers(0, t, size=m).astype(np.int32)
    rows[::29] = t
    arow = np.where((rows < t)[:, None], a[np.clip(rows, 0, t - 1)], 0).astype(np.float64)
    nb = 2 * n if epi != EPI_NONE else n
    bd, b_dtype, sd, bm = _weights(rng, "i8", (groups, nb), k, 0)
    out = torch.full((m, n), 77, dtype=torch.float32, device="cuda")
    KEEP_ALIVE.append(out)
    args = _args(bf16_dev(a), BF16, bd, b_dtype, sd, out, F32, None, m, n, k, epi, 0, 0)
    _abi.check(lib.sfg_hip_gemm_grouped_v1(ctypes.byref(args), dev(rows).data_ptr(), t, dev(offsets).data_ptr(),
                                           groups, nb * k, nb, None, 0, stream()))
    torch.cuda.synchronize()
    acc = np.concatenate([arow[offsets[g]:offsets[g + 1]] @ bm[g].T for g in range(groups)])
    _check(out, F32, _epilogue(acc, epi, n).astype(np.float32), epi != EPI_NONE, f"grouped int8 epi {epi}")


# A rows lda elements apart: the operand ends past 2^32 bytes (lda 2^21 at 1030 rows
# of bf16, 1031 of fp32 at 2^20), or just under; fp32 then runs on the VALU kernel
@pytest.mark.gpu
@pytest.mark.parametrize("kind,m,lda,epi,n", [
    ("bf16", 1030, 1 << 21, EPI_RESIDUAL, 384), ("bf16", 1030, 1 << 21, EPI_SWIGLU, 192), ("i8", 1030, 1 << 21, EPI_NONE, 256),
    ("i8", 1030, 1 << 21, EPI_GLU_SILU_UP, 130), ("bf16", 300, 1 << 23, EPI_SWIGLU, 100), ("i8", 300, 1 << 23, EPI_RESIDUAL, 130),
    ("f32", 1031, 1 << 20, EPI_RESIDUAL, 130), ("bf16", 1023, 1 << 21, EPI_NONE, 130), ("f32", 1023, 1 << 20, EPI_NONE, 130)])
def test_operands_around_4_gib(kind, m, lda, epi, n):
    lib = _abi.load()
    k = 128
    rng = np.random.default_rng(m + n)
    a = rng.integers(-3, 4, size=(m, k)).astype(np.float32)
    res = rng.integers(-5, 6, size=(m, n)).astype(np.float32) if epi == EPI_RESIDUAL else None
    glu = epi in (EPI_SWIGLU, EPI_GLU_SILU_UP)
    bd, b_dtype, sd, bm = _weights(rng, kind, (2 * n if glu else n,), k, 0)
    big = torch.empty(((m - 1) * lda + k,), dtype=torch.float32 if kind == "f32" else torch.int16, device="cuda")
    big.as_strided((m, k), (lda, 1)).copy_(dev(a) if kind == "f32" else bf16_dev(a))
    out = torch.full((m, n), 77, dtype=torch.float32, device="cuda")
    args = _args(big, F32 if kind == "f32" else BF16, bd, b_dtype, sd, out, F32, dev(res) if res is not None else None, m, n, k,
                 epi, 0, 0)
    args.lda = lda
    _abi.check(lib.sfg_hip_gemm_v1(ctypes.byref(args), None, 0, stream()))
    torch.cuda.synchronize()
    _check(out, F32, _epilogue(a.astype(np.float64) @ bm.T, epi, n, res).astype(np.float32), glu, f"{kind} {m}x{n} lda {lda}")


# grouped, past 4 GiB: the register-staged kernels' group walk
@pytest.mark.gpu
@pytest.mark.parametrize("kind,counts,epi,n", [("bf16", (700, 0, 429), EPI_GLU_SILU_UP, 192), ("i8", (900, 3, 200), EPI_NONE, 256),
                                               ("bf16", (500, 0, 77), EPI_NONE, 130)])
def test_grouped_operands_past_4_gib(kind, counts, epi, n):
    lib = _abi.load()
    k, groups, m = 128, len(counts), sum(counts)
    lda = (1 << 32) // 2 // m // 8 * 8 + 16384  # the rows end past 2^32 bytes
    assert (m - 1) * lda * 2 > 1 << 32
    rng = np.random.default_rng(m + n)
    offsets = np.concatenate([[0], np.cumsum(counts)]).astype(np.int32)
    a = rng.integers(-3, 4, size=(m, k)).astype(np.float32)
    nb = 2 * n if epi != EPI_NONE else n
    bd, b_dtype, sd, bm = _weights(rng, kind, (groups, nb), k, 0)
    big = torch.empty(((m - 1) * lda + k,), dtype=torch.int16, device="cuda")
    big.as_strided((m, k), (lda, 1)).copy_(bf16_dev(a))
    out = torch.full((m, n), 77, dtype=torch.float32, device="cuda")
    args = _args(big, BF16, bd, b_dtype, sd, out, F32, None, m, n, k, epi, 0, 0)
    args.lda = lda
    _abi.check(lib.sfg_hip_gemm_grouped_v1(ctypes.byref(args), None, 0, dev(offsets).data_ptr(), groups, nb * k,
                                           nb if sd is not None else 0, None, 0, stream()))
    torch.cuda.synchronize()
    acc = np.concatenate([a[offsets[g]:offsets[g + 1]].astype(np.float64) @ bm[g].T for g in range(groups)])
    _check(out, F32, _epilogue(acc, epi, n).astype(np.float32), epi != EPI_NONE, f"grouped {kind} {counts}")


# prefill layers whose QKV product (1536 columns of hidden 512) takes the tiles whose
# wave blocks of 64 x 64 go through LDS in the RoPE epilogue: odd sequences, ones
# that end inside a lane's run of four or eight rows, shorter than a step of the read-back
@pytest.mark.gpu
@pytest.mark.parametrize("dtype,tile,batch,seq", [
    ("w8", T128x128, 2, 777), ("w8", T128x128, 300, 5), ("w8", T128x128, 4, 340), ("w8", T128x128, 350, 4),
    ("w8", T256x128, 4, 777), ("w8", T256x128, 11, 257), ("w8", T256x128, 9, 300), ("w8", T256x128, 600, 5),
    ("w8", T64x64, 4, 257), ("bf16", T256x128, 4, 777), ("bf16", T256x128, 11, 257), ("bf16", T256x128, 9, 300),
    ("bf16", T256x128, 600, 5), ("bf16", T128x128, 2, 777), ("bf16", T128x128, 300, 5)])
def test_qkv_epilogue_through_lds(estimate, dtype, tile, batch, seq):
    import oracle
    from schedforge_amd import CONFIGS
    from schedforge_amd.layer import compile_decoder, execute_decoder_layer
    from _helpers import TOL, decoder_data
    cfg = CONFIGS["c4"].replace(batch=batch, sequence=seq, hidden=512, intermediate=256, query_heads=4, kv_heads=4,
                                dtype=dtype)
    assert estimate(I8 if dtype == "w8" else BF16, batch * seq, 1536, 512, EPI_NONE, BF16, 1, qkv=1) == tile
    d = oracle.make_layer_data(cfg, 4400 + seq)
    plan = compile_decoder(cfg, decoder_data(d), "cuda")
    out = execute_decoder_layer(plan, d.input, warmup=0, repetitions=1).output
    assert oracle.rel_error(out, oracle.decoder_layer(cfg, d)) < TOL[dtype]
