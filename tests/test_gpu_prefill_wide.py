"""The 128-row prefill kernel (shapes whose 128 x 256 tiles fill the GPU, unsplit or split through a
workspace) against the oracle, at the prefill bar: 1e-3 normwise, fp16 operands with fp32 sums."""
import numpy as np
import pytest
import torch

import cretif_amd as cri
from conftest import normwise_rel_err
from test_gpu_decode_step import load_cache, make_decoder, make_model, random_cache
from test_gpu_parity import FMTS, PREFILL_TOL, dev, host, weights

pytestmark = pytest.mark.gpu


def tiled(fmt, N, K, seed, rows=640):
    """[N, K] weights of `rows` distinct rows repeated, and the distinct rows."""
    w = weights(fmt, rows, K, seed).reshape(rows, -1)
    return np.ascontiguousarray(np.resize(np.arange(rows), N)), w


def tile_rows(fmt, M, N, K, ws_bytes=0, swiglu=False):
    """The rows of the prefill GEMM's tiles for this call: 128 is the kernel of this file."""
    import ctypes

    f = cri.lib().cri_internal_prefill_tile_rows
    f.argtypes = [ctypes.c_int] * 4 + [ctypes.c_longlong, ctypes.c_int]
    return f(cri.FORMAT_IDS[fmt], M, N, K, ws_bytes, swiglu)


def product(fmt, A, w, order, N, K, ws=None, rows=128):
    M = A.shape[0]
    assert tile_rows(fmt, M, N, K, 0 if ws is None else 4 * ws.numel()) == rows
    C = torch.full((M, N), float("nan"), device="cuda")
    B = dev(w)[torch.from_numpy(order).cuda()].contiguous()
    if ws is None:
        cri.matmul(fmt, dev(A), B, C, M, N, K)
    else:
        cri.matmul_ws(fmt, dev(A), B, C, M, N, K, ws)
    return host(C)


# one to five groups of four steps; one and three row tiles with ragged last ones; a ragged last column tile
@pytest.mark.parametrize("fmt", FMTS)
@pytest.mark.parametrize("M,N,K", [(65, 65533, 256), (128, 65536, 768), (300, 21755, 512), (129, 32768, 1280)])
def test_matches_oracle(orc, fmt, M, N, K):
    rng = np.random.default_rng(M + K)
    A = rng.standard_normal((M, K)).astype(np.float32)
    order, w = tiled(fmt, N, K, M)
    got = product(fmt, A, w, order, N, K)
    ref = orc.matmul_quant(fmt, A, w.reshape(-1), w.shape[0], K)
    # every tile on its own: 64 rows x 256 columns
    for m in range(0, M, 64):
        for n in range(0, N, 256):
            assert normwise_rel_err(got[m:m + 64, n:n + 256], ref[m:m + 64, order[n:n + 256]]) <= PREFILL_TOL, (m, n)


@pytest.mark.parametrize("fmt", ["q4_k", "q6_k", "fp16"])
def test_exact_integers(orc, fmt):
    """Small integer activations, power-of-two weights: every sum is exact, so the bits are the oracle's."""
    M, N, K = 128, 65536, 256
    rng = np.random.default_rng(5)
    A = rng.integers(-4, 5, (M, K)).astype(np.float32)
    order, w = tiled("fp16", N, K, 7)
    w = (rng.integers(-8, 9, (w.shape[0], K)).astype(np.float16)).view(np.uint8)
    if fmt != "fp16":
        from cretif_amd import quant
        w = quant.quantize_q4_k(w.view(np.float16).astype(np.float32)) if fmt == "q4_k" else \
            quant.quantize_q6_k(w.view(np.float16).astype(np.float32))
        w = w.reshape(640, -1)
    ref = orc.matmul_quant(fmt, A, w.reshape(-1), w.shape[0], K)
    got = product(fmt, A, w, order, N, K)
    if fmt == "fp16":
        assert np.array_equal(got, ref[:, order])
    else:
        assert normwise_rel_err(got, ref[:, order]) <= PREFILL_TOL


@pytest.mark.parametrize("fmt", ["q4_k", "q8_0", "q4_0", "q5_0", "fp16"])
def test_workspace_split(orc, fmt):
    """A long prompt's down projection: K in two splits through the workspace (the same bits on every
    call); without a workspace, or with one too small, or unaligned, the unsplit 64-row kernel."""
    M, N, K = 2048, 2048, 8192
    rng = np.random.default_rng(9)
    A = rng.standard_normal((M, K)).astype(np.float32)
    order, w = tiled(fmt, N, K, 11)
    need = cri.matmul_workspace_bytes(fmt, M, N, K)
    assert need == 2 * M * N * 4
    ws = torch.full((need // 4,), float("nan"), device="cuda")
    a = product(fmt, A, w, order, N, K, ws)
    assert np.array_equal(a, product(fmt, A, w, order, N, K, ws))
    rows = [0, 63, 64, 127, 128, 1000, 2047]
    ref = orc.matmul_quant(fmt, A[rows], w.reshape(-1), w.shape[0], K)[:, order]
    assert normwise_rel_err(a[rows], ref) <= PREFILL_TOL
    b = product(fmt, A, w, order, N, K, rows=64)
    assert normwise_rel_err(a, b) <= 1e-5  # the order of fp32 sums
    C = torch.full((M, N), float("nan"), device="cuda")
    B = dev(w)[torch.from_numpy(order).cuda()].contiguous()
    for args in ((None, 0), (ws, need - 16), (ws.view(torch.uint8)[4:], need - 4)):
        C.fill_(float("nan"))
        cri.matmul_ws(fmt, dev(A), B, C, M, N, K, *args)
        assert np.array_equal(host(C), b)


def test_activation_range(orc):
    """Rows past fp16's range or below it, in either half of a 128-row tile, are recomputed in fp32."""
    for fmt in FMTS:
        M, N, K = 128, 65536, 256
        rng = np.random.default_rng(13)
        A = rng.standard_normal((M, K)).astype(np.float32)
        A[3] *= 1e5
        A[70] *= 3e-8
        A[127, 100] = 7e4
        order, w = tiled(fmt, N, K, 15)
        got = product(fmt, A, w, order, N, K)
        ref = orc.matmul_quant(fmt, A, w.reshape(-1), w.shape[0], K)[:, order]
        assert np.isfinite(got).all()
        for r in range(M):
            assert normwise_rel_err(got[r], ref[r]) <= PREFILL_TOL, (fmt, r)


@pytest.mark.parametrize("norm", [1.0, 1e5])
def test_prompt_swiglu(orc, norm):
    """The SiLU(gate) * up epilogue of 128-row tiles in a prompt's step, and its fp32 rows (an FFN norm
    weight of 1e5 takes every row past fp16's range)."""
    m = make_model(1, dim=256, n_heads=4, n_kv_heads=2, head_dim=64, ffn=32768, vocab=900, seed=91,
                   fmts={n: "fp16" for n in ("q", "k", "v", "o", "gate", "up", "down")}, tok="q8_0", lm="fp16",
                   big_tables=False)
    m["layers"][0]["ffn_norm"] = (m["layers"][0]["ffn_norm"] * norm).astype(np.float32)
    M, pos, max_seq = 100, 5, 256
    dec = make_decoder(m, max_seq=max_seq, max_batch=M)
    kc, vc = random_cache(m, max_seq, 92)
    load_cache(dec, kc, vc)
    ids = torch.from_numpy(np.random.default_rng(93).integers(0, m["vocab"], M).astype(np.int32)).cuda()
    a = torch.empty(M, m["vocab"], device="cuda")
    dec.set_position(pos)
    dec.forward(ids, M, a)
    got = a.cpu().numpy()
    assert tile_rows("fp16", M, 32768, 256, swiglu=True) == 128
    ref, _ = orc.decode_step(m, list(ids.cpu().numpy()), pos, [k.copy() for k in kc], [v.copy() for v in vc])
    assert np.isfinite(got).all() and normwise_rel_err(got, ref) <= PREFILL_TOL
