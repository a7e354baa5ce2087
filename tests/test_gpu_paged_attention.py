"""GPU parity of FP16 paged attention against the oracle's restatement of attention_paged.cu
(fp16 output, |a - e| <= 1e-3 + 1e-3|e|).

Covers the batched decode entry over contiguous page pools (one query per sequence,
per-sequence lengths around page and 1024-position split edges, permuted block tables, GQA
groups of 1 to 12 q heads, head_dim 32 / 64 / 128 / 256 on the MFMA kernels and 16 / 20 / 80 /
96 on the generic kernel, masked pages, empty sequences) and the reference-interface entry with
per-block pointer arrays and causal prefill queries.
"""
import numpy as np
import pytest
import torch

import oracle
import rules
from conftest import assert_close
from fracture_amd import kernels as K

pytestmark = pytest.mark.gpu


def dev_t(a, dev):
    return torch.from_numpy(np.ascontiguousarray(a)).to(dev)


def build_pool(rng, lens, kvh, hd, extra_pages=3):
    """Random fp16 K/V pages for each sequence in a shared, permuted pool; unused rows hold
    garbage (large values and NaN) that must never reach the output."""
    nbs = [(n + 15) // 16 for n in lens]
    P = sum(nbs) + extra_pages
    perm = rng.permutation(P).astype(np.int32)
    kp = rng.standard_normal((P, 16, kvh, hd)).astype(np.float16)
    vp = rng.standard_normal((P, 16, kvh, hd)).astype(np.float16)
    maxb = max(max(nbs), 1)
    table = np.full((len(lens), maxb), -7, np.int32)
    at = 0
    for b, n in enumerate(lens):
        pages = perm[at:at + nbs[b]]
        at += nbs[b]
        table[b, :nbs[b]] = pages
        if n % 16:  # rows past the sequence end in its last page
            kp[pages[-1], n % 16:] = np.float16(6e4)
            vp[pages[-1], n % 16:] = np.float16(np.nan)
    return kp, vp, table


def run_decode(dev, q, table, lens, kp, vp, kvh):
    out = torch.empty(q.shape, dtype=torch.float16, device=dev)
    K.attention_paged_decode(out, dev_t(q, dev), dev_t(table, dev),
                             dev_t(np.asarray(lens, np.int32), dev), dev_t(kp, dev),
                             dev_t(vp, dev), kvh)
    torch.cuda.synchronize()
    return out.cpu().numpy()


@pytest.mark.parametrize("hd", [32, 64, 128, 256, 16, 20, 96])
@pytest.mark.parametrize("qh,kvh", [(32, 8), (8, 8), (16, 1), (24, 2)])
def test_decode_small_contexts(dev, hd, qh, kvh):
    rng = np.random.default_rng(hd * 100 + qh + kvh)
    lens = [1, 15, 16, 17, 33, 100]
    kp, vp, table = build_pool(rng, lens, kvh, hd)
    q = (rng.standard_normal((len(lens), qh, hd)) * 2).astype(np.float16)
    got = run_decode(dev, q, table, lens, kp, vp, kvh)
    for b, n in enumerate(lens):
        want = oracle.paged_attention(q[b], table[b], n, kp, vp, kvh)
        assert_close(got[b].astype(np.float32), want.astype(np.float32), 1e-3, 1e-3,
                     f"seq {b} len {n}")


@pytest.mark.parametrize("nseq,qh,kvh,hd,waves", [
    (32, 8, 8, 64, 8), (33, 8, 8, 64, 4), (33, 32, 8, 128, 4), (64, 16, 8, 32, 4), (65, 16, 8, 128, 2),
    (65, 16, 8, 64, 2), (65, 16, 8, 256, 2), (65, 8, 8, 32, 2), (65, 16, 16, 128, 4), (65, 16, 16, 64, 2),
    (65, 64, 64, 32, 1)])
def test_decode_waves_per_split(dev, nseq, qh, kvh, hd, waves):
    """8, 4, 2 and 1 waves per split: lengths that leave waves empty, end inside each wave's piece and on
    its edges, and a masked page that is a wave's whole piece of one chunk."""
    assert rules.paged_waves(nseq, qh, kvh, hd, 1024) == waves
    rng = np.random.default_rng(nseq + hd)
    edges = [0, 1, 127, 128, 129, 255, 257, 511, 512, 513, 640, 897, 1000, 1023, 1024]
    lens = (edges * 5)[:nseq]
    kp, vp, table = build_pool(rng, lens, kvh, hd)
    for b, n in enumerate(lens):
        if n == 640:
            table[b, 32:40] = -1  # positions 512..639
    q = (rng.standard_normal((len(lens), qh, hd)) * 2).astype(np.float16)
    got = run_decode(dev, q, table, lens, kp, vp, kvh)
    for b, n in enumerate(lens):
        if b >= 20 and b < nseq - 5:
            continue  # repeats of the same lengths
        rows = table[b]
        if n == 640:
            rows, n = rows[:32], 512
        want = oracle.paged_attention(q[b], rows, n, kp, vp, kvh) if n else np.zeros_like(q[b])
        assert_close(got[b].astype(np.float32), want.astype(np.float32), 1e-3, 1e-3,
                     f"seq {b} len {n}")


@pytest.mark.parametrize("nseq,qh,kvh,hd,widest", [
    (513, 4, 1, 128, 2100),   # 1539 splits: the last workgroup's second wave has none
    (513, 8, 1, 128, 2100), (257, 16, 2, 128, 2100), (257, 8, 2, 64, 3000), (515, 4, 2, 256, 20),
    (257, 8, 2, 256, 1100), (1025, 1, 1, 32, 100)])
def test_decode_one_wave_per_split(dev, nseq, qh, kvh, hd, widest):
    """Two splits of neighbouring kv heads to a workgroup, each a wave's own: odd counts of splits, pairs
    across a split and a sequence, a wave whose split lies past its sequence beside one that goes on,
    a masked page, empty sequences."""
    assert rules.paged_waves(nseq, qh, kvh, hd, -(-widest // 16) * 16) == 1
    rng = np.random.default_rng(nseq + hd)
    some = [n for n in (0, 1, 15, 17, 33, 640, 1000, 1023, 1024, 1025, 2048, widest) if n <= widest]
    lens = [some[b] if b < len(some) else (b * 7) % 40 for b in range(nseq)]
    lens[-1] = widest
    kp, vp, table = build_pool(rng, lens, kvh, hd)
    masked = {}
    for b in (5, nseq - 1):
        if lens[b] >= 48:
            table[b, 1] = -1  # positions 16..31
            masked[b] = np.delete(table[b], 1)
    q = (rng.standard_normal((nseq, qh, hd)) * 2).astype(np.float16)
    got = run_decode(dev, q, table, lens, kp, vp, kvh)
    for b in sorted(set(range(len(some) + 4)) | {nseq // 2, nseq - 2, nseq - 1}):
        n = lens[b] - 16 if b in masked else lens[b]
        want = oracle.paged_attention(q[b], masked.get(b, table[b]), n, kp, vp, kvh) if n else np.zeros_like(q[b])
        assert_close(got[b].astype(np.float32), want.astype(np.float32), 1e-3, 1e-3, f"seq {b} len {lens[b]}")


@pytest.mark.parametrize("hd", [128, 64, 80])
def test_decode_split_edges(dev, hd):
    """Lengths around the 1024-position splits: the combine merges 1 to 3 splits."""
    rng = np.random.default_rng(7 + hd)
    qh, kvh = 16, 4
    lens = [1023, 1024, 1025, 2048, 2100, 3001]
    kp, vp, table = build_pool(rng, lens, kvh, hd)
    q = (rng.standard_normal((len(lens), qh, hd)) * 3).astype(np.float16)
    got = run_decode(dev, q, table, lens, kp, vp, kvh)
    for b, n in enumerate(lens):
        want = oracle.paged_attention(q[b], table[b], n, kp, vp, kvh)
        assert_close(got[b].astype(np.float32), want.astype(np.float32), 1e-3, 1e-3,
                     f"seq {b} len {n}")


def test_decode_long_contexts(dev):
    """Llama-3.1-8B heads (32 q / 8 kv, hd 128) at contexts up to 32768 positions."""
    rng = np.random.default_rng(11)
    qh, kvh, hd = 32, 8, 128
    lens = [32768, 20000, 5000, 1]
    kp, vp, table = build_pool(rng, lens, kvh, hd, extra_pages=1)
    q = (rng.standard_normal((len(lens), qh, hd)) * 3).astype(np.float16)
    got = run_decode(dev, q, table, lens, kp, vp, kvh)
    for b, n in enumerate(lens):
        want = oracle.paged_attention(q[b], table[b], n, kp, vp, kvh)
        assert_close(got[b].astype(np.float32), want.astype(np.float32), 1e-3, 1e-3,
                     f"seq {b} len {n}")


def test_decode_empty_sequence_and_masked_pages(dev):
    """Length 0 gives zeros; a page id outside the pool masks its 16 positions, which equals
    attending to the sequence without that page."""
    rng = np.random.default_rng(12)
    qh, kvh, hd = 8, 2, 128
    lens = [0, 80, 1100]
    kp, vp, table = build_pool(rng, lens, kvh, hd)
    P = kp.shape[0]
    table[1, 2] = P + 5          # page 2 of sequence 1 (positions 32..47)
    table[2, 10] = -3            # page 10 of sequence 2 (positions 160..175)
    q = (rng.standard_normal((len(lens), qh, hd)) * 2).astype(np.float16)
    got = run_decode(dev, q, table, lens, kp, vp, kvh)
    assert not got[0].any()
    keep1 = np.delete(table[1], 2)
    want1 = oracle.paged_attention(q[1], keep1, 80 - 16, kp, vp, kvh)
    assert_close(got[1].astype(np.float32), want1.astype(np.float32), 1e-3, 1e-3, "seq 1")
    keep2 = np.delete(table[2], 10)
    want2 = oracle.paged_attention(q[2], keep2, 1100 - 16, kp, vp, kvh)
    assert_close(got[2].astype(np.float32), want2.astype(np.float32), 1e-3, 1e-3, "seq 2")


@pytest.mark.parametrize("kv_len,T,start_pos,qh,kvh,hd", [
    (90, 6, 84, 8, 2, 64), (40, 5, 38, 8, 2, 64), (1030, 3, 1027, 8, 2, 64),
    (16, 1, 15, 8, 2, 64),
    # 8 / G queries per wave: ragged last groups, groups whose lengths straddle a page or
    # the 1024-position split edge, whole prefills from position 0
    (1050, 19, 1020, 4, 4, 128), (300, 13, 0, 8, 4, 32), (1100, 11, 1019, 6, 2, 256),
    (70, 70, 0, 8, 2, 128), (2100, 9, 2040, 16, 16, 64), (50, 7, 43, 16, 2, 64),
    # 16 / G queries per wave on the MFMA prefill kernel: G = 8 (2 queries), G = 1 (16)
    (2100, 33, 2067, 32, 4, 128), (600, 37, 563, 4, 4, 64), (1030, 21, 1010, 24, 3, 32),
    # the generic kernel (other head_dims): one query per wave
    (5, 5, 0, 4, 2, 16), (1040, 9, 1031, 8, 2, 96), (40, 17, 23, 6, 3, 20)])
def test_reference_interface_prefill_causal(dev, kv_len, T, start_pos, qh, kvh, hd):
    """fhip_launch_paged_attention: T queries at start_pos.. over per-block pointer arrays;
    query i attends to min(start_pos + i + 1, kv_len) positions."""
    rng = np.random.default_rng(kv_len + T)
    kp, vp, table = build_pool(rng, [kv_len], kvh, hd, extra_pages=2)
    P = kp.shape[0]
    tk, tv = dev_t(kp, dev), dev_t(vp, dev)
    kptr = torch.tensor([tk[i].data_ptr() for i in range(P)], dtype=torch.int64, device=dev)
    vptr = torch.tensor([tv[i].data_ptr() for i in range(P)], dtype=torch.int64, device=dev)
    q = (rng.standard_normal((T, qh, hd)) * 2).astype(np.float16)
    tq_ = dev_t(q, dev)
    out = torch.empty_like(tq_)
    tb = dev_t(table[0], dev)
    K.paged_attention(out, tq_, tb, kptr, vptr, kvh, kv_len, start_pos)
    torch.cuda.synchronize()
    got = out.cpu().numpy()
    # the caller-workspace form launches the same kernels
    ws = K.attention_paged_workspace(T, qh, hd, table.shape[1], dev)
    out2 = torch.empty_like(tq_)
    K.paged_attention(out2, tq_, tb, kptr, vptr, kvh, kv_len, start_pos, ws)
    torch.cuda.synchronize()
    np.testing.assert_array_equal(out2.cpu().numpy().view(np.uint16), got.view(np.uint16))
    for t in range(T):
        clen = min(start_pos + t + 1, kv_len)
        want = oracle.paged_attention(q[t], table[0], clen, kp, vp, kvh)
        assert_close(got[t].astype(np.float32), want.astype(np.float32), 1e-3, 1e-3,
                     f"token {t}")


@pytest.mark.parametrize("kv_len,T,hd", [(300, 40, 128), (70, 70, 64), (3000, 9, 128), (5000, 3, 32)])
def test_prefill_into_an_output_of_any_alignment(dev, kv_len, T, hd):
    """Outputs that start at an odd element: one split goes through the merge, which stores single
    elements, instead of storing 8 bytes itself."""
    rng = np.random.default_rng(kv_len)
    qh, kvh = 8, 2
    kp, vp, table = build_pool(rng, [kv_len], kvh, hd)
    tk, tv = dev_t(kp, dev), dev_t(vp, dev)
    ptr = [torch.tensor([x.data_ptr() for x in t], dtype=torch.int64, device=dev) for t in (tk, tv)]
    q = dev_t((rng.standard_normal((T, qh, hd)) * 2).astype(np.float16), dev)
    want = torch.empty_like(q)
    K.paged_attention(want, q, dev_t(table[0], dev), *ptr, kvh, kv_len, kv_len - T)
    held = torch.full((q.numel() + 4,), 7.0, dtype=torch.float16, device=dev)
    K.paged_attention(held[1:-3].view(q.shape), q, dev_t(table[0], dev), *ptr, kvh, kv_len, kv_len - T)
    torch.cuda.synchronize()
    assert (held[[0, -3, -2, -1]] == 7.0).all()
    # the merge divides the same sums
    assert_close(held[1:-3].view(q.shape).cpu().numpy().astype(np.float32), want.cpu().numpy().astype(np.float32),
                 1e-3, 1e-3)


def test_reference_interface_rejects_unsupported_head_dim(dev):
    q = torch.zeros((1, 4, 264), dtype=torch.float16, device=dev)
    out = torch.empty_like(q)
    bt = torch.zeros(1, dtype=torch.int32, device=dev)
    ptr = torch.zeros(1, dtype=torch.int64, device=dev)
    with pytest.raises(RuntimeError):
        K.paged_attention(out, q, bt, ptr, ptr, 4, 1, 0)


@pytest.mark.parametrize("qh,kvh,hd", [(32, 8, 128), (8, 8, 64), (12, 2, 256), (4, 2, 16)])
def test_reference_interface_prefill_masked_page_and_no_blocks(dev, qh, kvh, hd):
    """Causal prefill with a negative page id in the block table: its 16 positions are masked
    for every query whose causal length covers them, which equals attending without that page
    (queries whose length ends inside it see the positions before it). With no blocks at all,
    every query returns zeros."""
    rng = np.random.default_rng(qh + hd)
    kv_len, T, start_pos = 1090, 40, 1050
    kp, vp, table = build_pool(rng, [kv_len], kvh, hd, extra_pages=2)
    P = kp.shape[0]
    tk, tv = dev_t(kp, dev), dev_t(vp, dev)
    kptr = torch.tensor([tk[i].data_ptr() for i in range(P)], dtype=torch.int64, device=dev)
    vptr = torch.tensor([vp_.data_ptr() for vp_ in tv], dtype=torch.int64, device=dev)
    tab = table[0].copy()
    tab[3] = -1  # positions 48..63
    q = (rng.standard_normal((T, qh, hd)) * 2).astype(np.float16)
    tq_ = dev_t(q, dev)
    out = torch.empty_like(tq_)
    K.paged_attention(out, tq_, dev_t(tab, dev), kptr, vptr, kvh, kv_len, start_pos)
    torch.cuda.synchronize()
    got = out.cpu().numpy()
    keep = np.delete(tab, 3)
    for t in range(T):
        clen = min(start_pos + t + 1, kv_len)
        want = oracle.paged_attention(q[t], keep, clen - 16, kp, vp, kvh)
        assert_close(got[t].astype(np.float32), want.astype(np.float32), 1e-3, 1e-3,
                     f"token {t}")
    empty = torch.full_like(tq_, 7.0)
    K.paged_attention(empty, tq_, dev_t(tab[:0], dev), kptr, vptr, kvh, 0, 0)
    torch.cuda.synchronize()
    assert not empty.cpu().numpy().any()


@pytest.mark.parametrize("kv_len,T,start_pos,qh,kvh,hd", [
    # two splits of 1056 positions: a split outlives the 64 pages a wave keeps at hand
    (2100, 129, 1971, 128, 128, 32),
    # full, partial and empty waves of columns; lengths on both sides of a 64-position tile
    (64, 32, 32, 4, 1, 64), (129, 34, 95, 8, 2, 128), (65, 3, 62, 3, 1, 128), (193, 65, 128, 5, 1, 32)])
def test_prefill_tiles(dev, kv_len, T, start_pos, qh, kvh, hd):
    rng = np.random.default_rng(kv_len + qh)
    kp, vp, table = build_pool(rng, [kv_len], kvh, hd, extra_pages=1)
    q = (rng.standard_normal((T, qh, hd)) * 2).astype(np.float16)
    got = prefill(dev, q, kp, vp, table[0], kvh, kv_len, start_pos)
    for t in range(T):
        want = oracle.paged_attention(q[t], table[0], start_pos + t + 1, kp, vp, kvh)
        assert_close(got[t].astype(np.float32), want.astype(np.float32), 1e-3, 1e-3, f"token {t}")


def prefill(dev, q, kp, vp, table, kvh, kv_len, start_pos):
    tk, tv = dev_t(kp, dev), dev_t(vp, dev)
    kptr = torch.tensor([x.data_ptr() for x in tk], dtype=torch.int64, device=dev)
    vptr = torch.tensor([x.data_ptr() for x in tv], dtype=torch.int64, device=dev)
    tq_ = dev_t(q, dev)
    out = torch.empty_like(tq_)
    K.paged_attention(out, tq_, dev_t(table, dev), kptr, vptr, kvh, kv_len, start_pos)
    torch.cuda.synchronize()
    return out.cpu().numpy()


@pytest.mark.parametrize("T,start_pos,hd", [(40, 30, 128), (20, 1100, 64)])
def test_prefill_non_finite_values_stay_with_their_queries(dev, T, start_pos, hd):
    """An infinity and a NaN among the V rows of the queries' own positions reach the queries that
    attend to them and none before, and a K row of NaN likewise (its score makes the sum NaN,
    which the merge writes as 0)."""
    rng = np.random.default_rng(T)
    qh, kvh = 8, 2
    kv_len = start_pos + T
    kp, vp, table = build_pool(rng, [kv_len], kvh, hd, extra_pages=1)
    q = (rng.standard_normal((T, qh, hd)) * 2).astype(np.float16)
    clean = [oracle.paged_attention(q[t], table[0], start_pos + t + 1, kp, vp, kvh) for t in range(T)]

    def at(pages, pos):
        return pages[table[0][pos // 16], pos % 16]

    inf_t, nan_t, k_t = T // 3, T // 2, T - 5
    at(vp, start_pos + inf_t)[1, 3] = np.inf
    at(vp, start_pos + nan_t)[0, 5] = np.nan
    at(kp, start_pos + k_t)[1, :] = np.nan
    got = prefill(dev, q, kp, vp, table[0], kvh, kv_len, start_pos).astype(np.float32)
    for t in range(T):
        want = clean[t].astype(np.float32)
        keep = np.ones((qh, hd), bool)
        if t >= inf_t:
            keep[4:, 3] = False
            assert np.all(np.isposinf(got[t][4:, 3])) or t >= k_t
        if t >= nan_t:
            keep[:4, 5] = False
            assert np.all(np.isnan(got[t][:4, 5]))
        if t >= k_t:
            keep[4:] = False
            assert not got[t][4:].any()
        assert_close(got[t][keep], want[keep], 1e-3, 1e-3, f"token {t}")
