"""Attention where its inputs leave the ordinary range: norms that are not finite past a query's
length, centroid tables far from 1, weights far below the largest, NaN scores."""
import numpy as np
import pytest
import torch

import oracle
from fracture_amd import kernels as K
from test_gpu_attention import build_pool, dev_t, run_prefill
from test_gpu_paged_attention import run_decode

pytestmark = pytest.mark.gpu

WIDTHS = [(8, 8), (4, 2), (4, 4), (3, 3), (2, 2)]


def tq_want(pool, q, n, kbits, vbits, kvh, rows=None):
    rows = pool["table"][0] if rows is None else rows
    return oracle.tq_attention(q, rows, n, pool["KP"], pool["KN"], pool["VP"], pool["VN"], pool["krot"],
                               pool["vrot"], pool["kc"], pool["vc"], kbits, vbits, kvh).astype(np.float32)


def assert_rel(got, want, rel, what=""):
    """|got - want| <= rel * the row's largest magnitude."""
    err = np.abs(got - want).max(-1) / np.abs(want).max(-1)
    assert np.isfinite(got).all() and err.max() <= rel, f"{what}: {err.max()}"


def run_tq_decode(dev, pool, q, lens, kbits, vbits, kvh):
    out = torch.empty(q.shape, dtype=torch.float16, device=dev)
    K.attention_tq_decode(out, dev_t(q, dev), dev_t(pool["table"], dev), dev_t(np.array(lens, np.int32), dev),
                          *(dev_t(pool[n], dev) for n in ("KP", "KN", "VP", "VN", "krot", "vrot", "kc", "vc")),
                          kbits, vbits, kvh)
    torch.cuda.synchronize()
    return out.cpu().numpy().astype(np.float32)


@pytest.mark.parametrize("kbits,vbits", WIDTHS)
@pytest.mark.parametrize("qh,kvh,T,kv_len", [(8, 2, 6, 90), (8, 4, 8, 131), (8, 8, 9, 300)])
def test_short_prefill_hides_later_norms(dev, kbits, vbits, qh, kvh, T, kv_len):
    """Queries that share MFMA columns (8 / G of them): a value norm of infinity and a key norm of NaN at
    the last two positions reach the queries that see them and no earlier one."""
    rng = np.random.default_rng(kbits * 10 + T)
    pool = build_pool(rng, [kv_len], kvh, 128, kbits, vbits)
    table = pool["table"][0]
    pool["VN"][table[(kv_len - 2) // 16], (kv_len - 2) % 16] = np.inf
    pool["KN"][table[(kv_len - 1) // 16], (kv_len - 1) % 16] = np.nan
    q = rng.standard_normal((T, qh, 128)).astype(np.float16)
    got = run_prefill(dev, pool, q, kvh, kv_len, kv_len - T, kbits, vbits)
    for t in range(T - 2):
        # fp16 rounding of the output (2^-11) and of the oracle's, plus fp32 sums
        assert_rel(got[t], tq_want(pool, q[t], kv_len - T + t + 1, kbits, vbits, kvh), 2e-3, f"token {t}")
    assert not np.isfinite(got[T - 2]).any()


@pytest.mark.parametrize("kbits,vbits", WIDTHS)
@pytest.mark.parametrize("exp", [18, -18])
@pytest.mark.parametrize("G,T", [(4, 1), (8, 1), (2, 5), (4, 200)])
def test_centroid_tables_of_any_scale(dev, kbits, vbits, exp, G, T):
    """Centroids times 2^exp, with norms and queries that bring scores and outputs back: past fp16's
    range on either side, inside fp32's. Decode and the two prefill kernels."""
    rng = np.random.default_rng(kbits + G)
    kvh, kv_len = (8, 700) if T > 100 else (2, 300)
    pool = build_pool(rng, [kv_len], kvh, 128, kbits, vbits)
    pool["kc"], pool["vc"] = (pool[n] * np.float32(2.0 ** exp) for n in ("kc", "vc"))
    back = np.float16(2.0 ** (-exp // 2))
    pool["KN"], pool["VN"] = pool["KN"] * back, pool["VN"] * back
    q = (rng.standard_normal((T, kvh * G, 128)) * float(back)).astype(np.float16)
    if T == 1:
        got = run_tq_decode(dev, pool, q, [kv_len], kbits, vbits, kvh)
    else:
        got = run_prefill(dev, pool, q, kvh, kv_len, kv_len - T, kbits, vbits)
    for t in range(0, T, max(1, T // 10)):
        assert_rel(got[t], tq_want(pool, q[t], kv_len - T + t + 1, kbits, vbits, kvh), 2e-3, f"token {t}")


@pytest.mark.parametrize("kbits,vbits", WIDTHS)
@pytest.mark.parametrize("G,T", [(4, 1), (8, 1), (2, 5), (4, 200)])
def test_value_norms_up_to_the_largest(dev, kbits, vbits, G, T):
    """Value norms of 2^15 and more: the low parts of the weights stay finite."""
    rng = np.random.default_rng(kbits + G)
    kvh, kv_len = (8, 700) if T > 100 else (2, 300)
    pool = build_pool(rng, [kv_len], kvh, 128, kbits, vbits)
    pool["VN"] = rng.uniform(3e4, 65504, pool["VN"].shape).astype(np.float16)
    q = rng.standard_normal((T, kvh * G, 128)).astype(np.float16)
    if T == 1:
        got = run_tq_decode(dev, pool, q, [kv_len], kbits, vbits, kvh)
    else:
        got = run_prefill(dev, pool, q, kvh, kv_len, kv_len - T, kbits, vbits)
    for t in range(0, T, max(1, T // 10)):
        assert_rel(got[t], tq_want(pool, q[t], kv_len - T + t + 1, kbits, vbits, kvh), 2e-3, f"token {t}")


@pytest.mark.parametrize("hd", [32, 64, 128])
@pytest.mark.parametrize("kv_len", [200, 5000])
def test_fp16_prefill_small_weights(dev, hd, kv_len):
    """One position holds nearly all the weight and no value; the output is what the others, at about
    2^-24 of it, add up to. 2^-11 is the rounding of the output; a weight is right to 2^-37 of the largest,
    2^-13 of itself here."""
    T, qh, kvh = 64, 8, 2
    P = (kv_len + 15) // 16
    kp = np.zeros((P, 16, kvh, hd), np.float16)
    vp = np.zeros((P, 16, kvh, hd), np.float16)
    rng = np.random.default_rng(hd)
    vp[:] = rng.uniform(4e4, 6e4, (kvh, hd)).astype(np.float16)
    vp[0, 0] = 0
    top = 16.6  # nats: 2^-24 = exp(-16.6)
    kp[0, 0] = np.float16(top / np.sqrt(hd))
    q = (np.ones((T, qh, hd)) * rng.uniform(0.93, 1.0, (T, qh, 1))).astype(np.float16)
    tk, tv = dev_t(kp, dev), dev_t(vp, dev)
    ptr = [torch.tensor([x.data_ptr() for x in t], dtype=torch.int64, device=dev) for t in (tk, tv)]
    out = torch.empty(q.shape, dtype=torch.float16, device=dev)
    K.paged_attention(out, dev_t(q, dev), torch.arange(P, dtype=torch.int32, device=dev), *ptr, kvh, kv_len,
                      kv_len - T)
    torch.cuda.synchronize()
    got = out.cpu().numpy().astype(np.float64)
    s = q.astype(np.float64)[:, :, 0] * float(kp[0, 0, 0, 0]) * hd / np.sqrt(hd)
    n = kv_len - T + 1 + np.arange(T)
    w = (n[:, None] - 1) * np.exp(-s) / (1 + (n[:, None] - 1) * np.exp(-s))
    want = w[:, :, None] * np.repeat(vp[1, 1].astype(np.float64), qh // kvh, 0)
    assert np.abs(got / want - 1).max() <= 2.0 ** -11 + 2.0 ** -12


@pytest.mark.parametrize("kbits,vbits", WIDTHS)
@pytest.mark.parametrize("late", [np.inf, 6e4])
def test_tq_prefill_late_norm_costs_no_precision(dev, kbits, vbits, late):
    """The first position holds nearly all the weight and a value norm of 0; what the others add, at
    about 2^-18 of it, is the output. A large value norm at position 40, in the first tile of all the
    first block's queries, changes none before it."""
    rng = np.random.default_rng(kbits)
    T, qh, kvh = 400, 32, 8
    pool = build_pool(rng, [T], kvh, 128, kbits, vbits)
    rows = pool["table"][0]
    pos = lambda n, t: pool[n][rows[t // 16], t % 16]
    for t in range(1, T):
        pos("KP", t)[:] = pos("KP", 0)
        pos("VP", t)[:] = pos("VP", 1)
        pos("KN", t)[:] = np.float16(0.125)
        pos("VN", t)[:] = np.float16(1024)
    pos("KN", 0)[:] = np.float16(8)
    pos("VN", 0)[:] = 0
    pos("VN", 40)[:] = late
    # q along the first key: a score of about 12.5 nats (2^-18) against a sixty-fourth of it
    codes = oracle.tq_unpack_rows(pos("KP", 0).reshape(kvh, -1), 128, kbits)
    k = pool["kc"][codes] @ pool["krot"]
    a = 12.5 * np.sqrt(128) / 8 / (k * k).sum(-1, keepdims=True)
    q = ((a * k)[None, :, None] * rng.uniform(0.97, 1.0, (T, kvh, qh // kvh, 1))).reshape(T, qh, 128).astype(np.float16)
    got = run_prefill(dev, pool, q, kvh, T, 0, kbits, vbits)
    for t in range(2, 40, 3):
        # the rounding of the output and of the oracle's, 2^-11 each of the larger elements
        assert_rel(got[t], tq_want(pool, q[t], t + 1, kbits, vbits, kvh), 1.2e-3, f"token {t}")


@pytest.mark.parametrize("n,bad", [(1000, (0, 64)), (1000, (128, 256)), (1000, (256, 512)), (3000, (1024, 2048)),
                                   (40000, (2048, 2304))])
def test_nan_scores_of_a_whole_piece(dev, n, bad):
    """Key rows of NaN over positions that make up a whole wave's piece, a 256-position part or a split:
    the result is what one such row gives anywhere: NaN over TurboQuant pages, zeros over FP16 pages."""
    rng = np.random.default_rng(n)
    qh, kvh = 8, 2
    pool = build_pool(rng, [n], kvh, 128, 4, 4)
    rows = pool["table"][0]
    for t in range(*bad):
        pool["KN"][rows[t // 16], t % 16] = np.nan
    q = rng.standard_normal((1, qh, 128)).astype(np.float16)
    assert np.isnan(run_tq_decode(dev, pool, q, [n], 4, 4, kvh)).all()
    kp = rng.standard_normal((len(rows), 16, kvh, 128)).astype(np.float16)
    vp = rng.standard_normal(kp.shape).astype(np.float16)
    for t in range(*bad):
        kp[t // 16, t % 16] = np.nan
    table = np.arange(len(rows), dtype=np.int32)[None]
    assert not run_decode(dev, q, table, [n], kp, vp, kvh).any()


@pytest.mark.parametrize("kbits,vbits", [(4, 4), (8, 8), (8, 2)])
@pytest.mark.parametrize("T", [1, 5, 200])
def test_nan_query_gives_nan(dev, kbits, vbits, T):
    """A query with NaN among its elements gives NaN, as the reference's sums do
    (attention_paged_tq.cu:56-257), and disturbs no other one."""
    rng = np.random.default_rng(T)
    qh, kvh, n = 32, 8, 700
    pool = build_pool(rng, [n], kvh, 128, kbits, vbits)
    q = rng.standard_normal((T, qh, 128)).astype(np.float16)
    clean = run_prefill(dev, pool, q, kvh, n, n - T, kbits, vbits)
    q[T // 2, 3, 7] = np.nan
    got = run_prefill(dev, pool, q, kvh, n, n - T, kbits, vbits)
    assert np.isnan(got[T // 2, 3]).all()
    got[T // 2, 3] = clean[T // 2, 3]
    np.testing.assert_array_equal(got, clean)
