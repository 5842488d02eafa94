"""Split decode attention: the heads per workgroup, the tiles per wave and the edges of both."""
from __future__ import annotations

import numpy as np
import pytest
import torch

import cretif_amd as cri

pytestmark = pytest.mark.gpu


def _f64(q, k, v, H, Hkv, D, T, scale):
    """Attention of one query in float64: q [H * D], k and v [T, Hkv, D]."""
    q, k, v = q.astype(np.float64).reshape(H, D), k.astype(np.float64), v.astype(np.float64)
    out = np.empty((H, D))
    for h in range(H):
        g = h // (H // Hkv)
        s = k[:, g] @ q[h] * scale
        p = np.exp(s - s.max())
        out[h] = (p / p.sum()) @ v[:, g]
    return out


def _run(q, k, v, H, Hkv, D, T, scale, chunks=None):
    need = cri.decode_attention_workspace_size(H, Hkv, D, T)
    nbytes = need if chunks is None else chunks * H * (D + 4) * 4
    ws = torch.full((nbytes // 4 + 4,), float("nan"), device="cuda")
    out = torch.full((H * D,), float("nan"), device="cuda")
    dq, dk, dv = (torch.from_numpy(a).cuda() for a in (q, k, v))
    cri.fused_decode_attention_ws(dq, dk, dv, out, H, Hkv, D, T, scale, ws.data_ptr(), nbytes)
    return out.cpu().numpy().reshape(H, D)


# Heads per KV head: 1, 2 and 3 of them in a workgroup, quads with a shorter last one (5, 7) and two quads
# (8).  One chunk: lengths around a wave's tile (16 positions at 4 lanes each, 8 at 8), the four waves'
# round (64, 32) and two, three and more rounds, so that waves end on either of their two tiles.
@pytest.mark.parametrize("D", [64, 128, 20, 100])
@pytest.mark.parametrize("G", [1, 2, 3, 4, 5, 7, 8])
def test_heads_and_lengths(G, D):
    rng = np.random.default_rng(100 * G + D)
    Hkv = 2
    H = G * Hkv
    for T, chunks in [(1, 1), (7, 1), (8, 1), (9, 1), (17, 1), (33, 1), (63, 1), (64, 1), (65, 1), (97, 1), (129, 1),
                      (193, 1), (200, 1), (333, 1), (1000, 1), (333, 3), (1000, 7), (1000, None), (33, None)]:
        q = rng.standard_normal(H * D).astype(np.float32)
        k, v = (rng.standard_normal((T, Hkv, D)).astype(np.float32) for _ in range(2))
        got = _run(q, k, v, H, Hkv, D, T, D ** -0.5, chunks)
        ref = _f64(q, k, v, H, Hkv, D, T, D ** -0.5)
        # scores of magnitude up to ~5 from D fp32 products: |error| <= D * 2^-24 * sum |q k| scale ~ 2e-5 at
        # worst, usually its square root over D; the softmax passes a score's error on as a relative one
        err = np.linalg.norm(got - ref) / np.linalg.norm(ref)
        assert err <= 5e-6, (G, D, T, chunks, err)


@pytest.mark.parametrize("D", [64, 128])
def test_positions_of_weight_zero(D):
    # keys that give a score of -infinity for whole tiles, first, middle and last, have no weight
    H, Hkv, T = 8, 2, 600
    rng = np.random.default_rng(D)
    q = np.abs(rng.standard_normal(H * D)).astype(np.float32) + 0.1
    k, v = (rng.standard_normal((T, Hkv, D)).astype(np.float32) for _ in range(2))
    off = np.zeros(T, bool)
    off[:70] = off[200:264] = off[500:] = True
    k[off, :, 3] = -np.inf
    for chunks in (1, 4):  # the kernel of long chunks
        got = _run(q, k, v, H, Hkv, D, T, 0.05, chunks)
        ref = _f64(q, k[~off], v[~off], H, Hkv, D, int((~off).sum()), 0.05)
        assert np.linalg.norm(got - ref) <= 5e-6 * np.linalg.norm(ref), chunks


def test_nan_key_reaches_only_its_heads():
    H, Hkv, D, T = 8, 2, 64, 300
    rng = np.random.default_rng(3)
    q = rng.standard_normal(H * D).astype(np.float32)
    k, v = (rng.standard_normal((T, Hkv, D)).astype(np.float32) for _ in range(2))
    k[130, 1, 5] = np.nan
    got = _run(q, k, v, H, Hkv, D, T, 0.125)
    assert np.isfinite(got[:4]).all() and np.isnan(got[4:]).all()
