"""The prompt attention kernel (cri_prefill_attention at head_dim 64 and 128 from 32 rows) at the
edges of its tiles, query groups and chunks, against the oracle's decode attention row by row.

Bar: 1e-5 normwise, the bar of every fp32 path.  The kernel's own error is the fp16 parts' (at most 2^-23
of each operand and 2^-22 of a product for the one dropped, a tenth of that in a sum of many) plus fp32
sums over the positions, a few 1e-7 in all.
"""
import numpy as np
import pytest
import torch

import cretif_amd as cri
from conftest import normwise_rel_err

pytestmark = pytest.mark.gpu


def run(q, ldq, kc, vc, M, H, Hkv, D, pos, scale):
    out = torch.full((M, H * D), float("nan"), device="cuda")
    cri.prefill_attention(torch.from_numpy(q).cuda(), ldq, torch.from_numpy(kc).cuda(), torch.from_numpy(vc).cuda(),
                          out, M, H, Hkv, D, pos, scale)
    return out.cpu().numpy()


def inputs(M, H, Hkv, D, pos, past=9):
    rng = np.random.default_rng(1000 * M + pos + D + H)
    ldq = (H + 2 * Hkv) * D
    q = rng.standard_normal((M, ldq)).astype(np.float32)
    kc = rng.standard_normal((pos + M + past, Hkv, D)).astype(np.float32)
    vc = rng.standard_normal((pos + M + past, Hkv, D)).astype(np.float32)
    kc[pos + M:] = np.nan  # rows past the prompt are never read into the products
    vc[pos + M:] = np.nan
    return q, ldq, kc, vc


def rows_of(M):
    return sorted({0, 1, M // 3, M // 2, M - 2, M - 1, *(r for r in (31, 32, 63, 64, 127, 128) if r < M)})


# one query group and its remainder, groups that straddle rows (G = 3, 7), one head per KV head, tile
# remainders, every chunk count from 16 down to one, two- and four-block workgroups, paired ones with an
# even and an odd group count
@pytest.mark.parametrize("H,Hkv,D,M,pos", [
    (1, 1, 64, 32, 0), (7, 1, 64, 33, 31), (3, 1, 128, 37, 3), (8, 8, 128, 65, 0), (32, 8, 64, 64, 959),
    (4, 1, 128, 300, 700), (32, 8, 64, 513, 0), (8, 8, 64, 1000, 24), (32, 8, 64, 1025, 0), (32, 8, 64, 2050, 0),
    (32, 8, 128, 1030, 5), (32, 8, 128, 2049, 0),
])
def test_matches_oracle(orc, H, Hkv, D, M, pos):
    q, ldq, kc, vc = inputs(M, H, Hkv, D, pos)
    scale = np.float32(1.0 / np.sqrt(D))
    got = run(q, ldq, kc, vc, M, H, Hkv, D, pos, scale)
    assert np.isfinite(got).all()
    for m in rows_of(M):
        ref = orc.decode_attention(q[m, :H * D], kc, vc, H, Hkv, D, pos + m + 1, scale)
        assert normwise_rel_err(got[m], ref) <= 1e-5, m


@pytest.mark.parametrize("D", [64, 128])
@pytest.mark.parametrize("what", ["wide", "spread", "tiny_k", "big_q", "zero_v", "peak"])
def test_ranges(orc, D, what):
    """Operands near the ends of the range, and tiles (that every row sees) of magnitudes far apart."""
    H, Hkv, M, pos = 4, 2, 70, 90
    q, ldq, kc, vc = inputs(M, H, Hkv, D, pos)
    if what == "wide":  # V tiles 2^40 apart, K tiles 2^20 apart (scores stay moderate)
        vc[32:64] *= np.float32(2.0 ** -40)
        kc[96:128] *= np.float32(2.0 ** -20)
    elif what == "spread":
        vc[:32] *= np.float32(2.0 ** -60)
        vc[64:96] *= np.float32(2.0 ** 60)
    elif what == "tiny_k":
        kc *= np.float32(2.0 ** -104)
        q *= np.float32(2.0 ** 100)
    elif what == "big_q":
        q[:] = np.float32(2.0 ** 126) * np.sign(q)
        kc *= np.float32(2.0 ** -125)
    elif what == "zero_v":
        vc[:64] = 0
    else:  # one score far above the rest, then a later higher one: the running maximum is raised late
        kc[40] = 30 * q[0, :D]
        kc[120] = 60 * q[0, :D]
    scale = np.float32(1.0 / np.sqrt(D))
    got = run(q, ldq, kc, vc, M, H, Hkv, D, pos, scale)
    for m in rows_of(M):
        ref = orc.decode_attention(q[m, :H * D], kc, vc, H, Hkv, D, pos + m + 1, scale)
        assert normwise_rel_err(got[m], ref) <= 1e-5, m


def test_nonfinite_keys_and_values():
    """A NaN key or an infinite value reaches exactly the rows and heads that see it."""
    H, Hkv, D, M = 4, 2, 64, 100
    q, ldq, kc, vc = inputs(M, H, Hkv, D, 0)
    clean = run(q, ldq, kc, vc, M, H, Hkv, D, 0, 0.125)
    kc[50, 0, 3] = np.nan
    vc[70, 1, 5] = np.inf
    got = run(q, ldq, kc, vc, M, H, Hkv, D, 0, 0.125).reshape(M, H, D)
    clean = clean.reshape(M, H, D)
    assert np.isnan(got[50:, :2]).all()
    assert normwise_rel_err(got[:50, :2], clean[:50, :2]) <= 1e-5
    assert normwise_rel_err(got[:70, 2:], clean[:70, 2:]) <= 1e-5
    assert np.isposinf(got[70:, 2:, 5]).all()
    keep = [d for d in range(D) if d != 5]
    assert normwise_rel_err(got[70:, 2:][..., keep], clean[70:, 2:][..., keep]) <= 1e-5


def f64(q, kc, vc, rows, H, Hkv, D, pos, scale):
    """The rows' outputs in float64 and the sums of their terms' magnitudes, [len(rows), H, D] each."""
    out, mag = np.empty((2, len(rows), H, D))
    for n, m in enumerate(rows):
        T = pos + m + 1
        for h in range(H):
            g = h // (H // Hkv)
            v = vc[:T, g].astype(np.float64)
            s = kc[:T, g].astype(np.float64) @ q[m, h * D:(h + 1) * D].astype(np.float64) * np.float64(scale)
            p = np.exp(s - s.max())
            p /= p.sum()
            out[n, h] = p @ v
            mag[n, h] = p @ np.abs(v)
    return out, mag


def times(x, at, e):
    x[at] = (x[at].astype(np.float64) * 2.0 ** e).astype(np.float32)


# Magnitudes that differ between positions, or between dims: a row before the first changed position must not
# notice it, a dim is as good as if it were alone.  Bar: 5e-6 of the sum of an output's terms.  A score is an fp32
# sum of D products, good to D 2^-24 = 4 to 8e-6 of their magnitudes' sum (about 4) at worst and usually to the root
# of D in place of D; the softmax passes the error of a score on as a relative one.
@pytest.mark.parametrize("e", [8, 11, 13, 16, 20, 24, 30, 40, -8, -11, -13, -16, -20, -24, -30, -40])
@pytest.mark.parametrize("D", [64, 128])
@pytest.mark.parametrize("what", ["v_tile", "v_row", "k_tile", "k_row", "v_dim", "k_dim", "q_dim", "v_one_key"])
def test_uneven_magnitudes(what, D, e):
    H, Hkv, M, pos = 2, 2, 96, 0
    q, ldq, kc, vc = inputs(M, H, Hkv, D, pos)
    qh = q.reshape(M, -1, D)
    scale = np.float32(1.0 / np.sqrt(D))
    every, first = (slice(None), slice(None), 0), 31
    if what == "v_tile":
        times(vc, slice(32, 64), e)
    elif what == "v_row":
        times(vc, 31, e)
    elif what == "k_tile":
        first = 32
        times(kc, slice(32, 64), e)
    elif what == "k_row":
        times(kc, 31, e)
    elif what == "v_dim":
        times(vc, every, e)
    elif what == "k_dim":  # a score is the sum of a product of a large and a small operand and of the others
        times(kc, every, e)
        times(qh, every, -e)
    elif what == "q_dim":  # the queries' large dim meets keys that are zero there
        times(qh, every, e)
        kc[:, :, 0] = 0
    else:  # value 40 is as large as its weight in row 50 is small
        for h in range(H):
            a = qh[50, h].astype(np.float64)
            kc[40, h] = -abs(e) * np.log(2.0) * np.sqrt(D) * np.sign(a) / np.abs(a).sum()
        times(vc, 40, abs(e))
    got = run(q, ldq, kc, vc, M, H, Hkv, D, pos, scale).reshape(M, H, D)
    assert np.isfinite(got).all()
    rows = rows_of(M) + [50]
    if what in ("k_tile", "k_row") and e > 0:  # scores 2^e larger, and the errors of fp32 products with them
        rows = [m for m in rows if m < first]
    ref, mag = f64(q, kc, vc, rows, H, Hkv, D, pos, scale)
    for n, m in enumerate(rows):
        assert (np.abs(got[m] - ref[n]) <= 5e-6 * mag[n]).all(), (m, np.max(np.abs(got[m] - ref[n]) / mag[n]))


# Both operands of the scores small or large together, either side of the range the parts are used in; scores of
# exactly 0 from large operands; a tile that a query group reads but does not see (rows 0..63 share one at head_dim
# 64), far from those it sees.  Bar as above.
@pytest.mark.parametrize("D", [64, 128])
@pytest.mark.parametrize("what,a,b", [
    ("qk", -62, -62), ("qk", -75, -75), ("qk", -49, -49), ("qk", -48, -53), ("qk", -45, -99), ("qk", 58, -58),
    ("qk", -61, 61), ("zero", 70, 70), ("zero", 50, 50), ("zero", 3, 3), ("later_v", 116, 0), ("later_v", -99, 41),
    ("later_v", -60, 50), ("later_v", 59, -47), ("later_k", -99, -60), ("later_k", -49, -46)])
def test_exponents(what, a, b, D):
    H, Hkv, M, pos = 2, 2, 160, 0
    q, ldq, kc, vc = inputs(M, H, Hkv, D, pos)
    qh = q.reshape(M, -1, D)
    every = slice(None)
    rows = [m for m in rows_of(M)]
    if what == "qk":
        times(qh, every, a)
        times(kc, every, b)
    elif what == "zero":
        times(qh, every, a)
        times(kc, every, b)
        qh[:, :, D // 2:] = 0
        kc[:, :, :D // 2] = 0
    elif what == "later_v":
        times(vc, slice(64, None), a)
        times(vc, slice(64), b)
    else:
        times(kc, slice(64, None), a)
        times(qh, every, b)
    scale = np.float32(1.0 / np.sqrt(D))
    got = run(q, ldq, kc, vc, M, H, Hkv, D, pos, scale).reshape(M, H, D)
    ref, mag = f64(q, kc, vc, rows, H, Hkv, D, pos, scale)
    for n, m in enumerate(rows):
        assert (np.abs(got[m] - ref[n]) <= 5e-6 * mag[n]).all(), m


# Values too small for the parts: every workgroup takes the fp32 products, in all the forms of test_matches_oracle.  A
# NaN key and an infinite value reach exactly the rows that see them.
@pytest.mark.parametrize("H,Hkv,D,M,pos", [
    (1, 1, 64, 32, 0), (7, 1, 64, 33, 31), (3, 1, 128, 37, 3), (8, 8, 128, 65, 0), (32, 8, 64, 64, 959),
    (4, 1, 128, 300, 700), (32, 8, 64, 513, 0), (8, 8, 64, 1000, 24), (32, 8, 64, 1025, 0), (32, 8, 128, 1030, 5)])
def test_fp32_products(H, Hkv, D, M, pos):
    q, ldq, kc, vc = inputs(M, H, Hkv, D, pos)
    times(vc, slice(None), -60)
    t_inf, t_nan = pos + M // 2, pos + M - 5
    vc[t_inf, 0, 5] = np.inf
    kc[t_nan, Hkv - 1, 3] = np.nan
    scale = np.float32(1.0 / np.sqrt(D))
    got = run(q, ldq, kc, vc, M, H, Hkv, D, pos, scale).reshape(M, H, D)
    rows = sorted({*rows_of(M), M // 2 - 1, M - 6, M - 5})
    vc[t_inf, 0, 5] = 0
    kc[t_nan, Hkv - 1, 3] = 0
    ref, mag = f64(q, kc, vc, rows, H, Hkv, D, pos, scale)
    G = H // Hkv
    for n, m in enumerate(rows):
        for h in range(H):
            if pos + m >= t_nan and h // G == Hkv - 1:
                assert np.isnan(got[m, h]).all(), (m, h)
                continue
            dims = np.ones(D, bool)
            if pos + m >= t_inf and h // G == 0:
                dims[5] = False
                assert not np.isfinite(got[m, h, 5]), (m, h)  # NaN where the records of chunks are merged
            assert (np.abs(got[m, h] - ref[n, h]) <= 5e-6 * mag[n, h])[dims].all(), (m, h)
