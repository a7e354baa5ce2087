"""CPU models of the work split of the FP16 paged-attention kernels: which query rows each wave of
paged_attn_split_kernel reads and which split partials it writes, checked against the combine kernel's
reads, and the tiled prefill kernels' blocks and splits (FP16 and TurboQuant), through the functions
that the launchers and kernels call.

A workgroup item of the split kernel is (query group, kv head g, head block hb, split). In causal
prefill over one shared block table at head_dim 256, a group is tok = 8 / G consecutive queries
(G = qh / kvh < 8); MFMA column c is head g G + c % G of query tq0 + c / G. Otherwise tok = 1 and
column c is head g G + 8 hb + c. Each column scores positions below min(split end, its own causal
length). The combine reads partial (vector, split) for every split below the vector's causal length;
the model asserts that each of those is written by exactly one item, with the causal length of
that vector, and that nothing else is read. No GPU is used.
"""
import numpy as np
import pytest

import rules

PAGE = 16
SPLIT = 1024
HEADS_MAX = 8


def causal_len(qi, kv_len, start_pos, max_blocks, seq_lens=None):
    c = int(seq_lens[qi]) if seq_lens is not None else min(start_pos + qi + 1, kv_len)
    return max(0, min(c, max_blocks * PAGE))


def model_split_kernel(nq, qh, kvh, kv_len, start_pos, shared_table=True, seq_lens=None,
                       wrap=None):
    G = qh // kvh
    wrap = G if wrap is None else wrap  # head count at which the acc loop's counter wraps
    nhb = (G + HEADS_MAX - 1) // HEADS_MAX
    max_blocks = (max(kv_len, int(max(seq_lens)) if seq_lens is not None else 0) + 15) // 16
    nsplit = max(1, (max_blocks * PAGE + SPLIT - 1) // SPLIT)
    prefill = seq_lens is None and shared_table and nq > 1
    tok = HEADS_MAX // G if prefill and G < HEADS_MAX else 1
    NH = 4 if G * tok <= 4 else 8
    per_q = kvh * nhb * nsplit
    items = []  # (tq0, ntok, g, hb, split, t_begin, t_end) of each item that runs the loop
    for item in range(-(-nq // tok) * per_q):
        tq0 = (item // per_q) * tok
        if tq0 >= nq:
            continue
        ntok = min(tok, nq - tq0)
        g = item % kvh
        hb = (item // kvh) % nhb
        split = (item // (kvh * nhb)) % nsplit
        clen = causal_len(tq0 + ntok - 1, kv_len, start_pos, max_blocks, seq_lens)
        t_begin = split * SPLIT
        if t_begin >= clen:
            continue
        items.append((tq0, ntok, g, hb, split, t_begin, min(clen, t_begin + SPLIT)))
    written = {}
    q_rows = set()
    for tq0, ntok, g, hb, split, t_begin, t_end in items:
        h0 = g * G + hb * HEADS_MAX
        ncols = ntok * G if tok > 1 else min(HEADS_MAX, G - hb * HEADS_MAX)
        assert ncols <= NH
        # per lane column n (0..15): the Q row and the masking limit
        for n in range(16):
            col_ok = n < ncols
            ct = n // G if col_ok else 0
            hn = n - ct * G if col_ok else 0
            # a column past the queries reads the group's first query row (unused)
            row = (tq0 + ct) * qh + h0 + hn
            assert 0 <= row < nq * qh
            if not col_ok:
                continue
            assert tok > 1 or ct == 0
            col_len = causal_len(tq0 + ct, kv_len, start_pos, max_blocks, seq_lens) \
                if tok > 1 else t_end
            lim = min(t_end, col_len)
            q_rows.add(row)
            # the partial write of lane n (== column n) and of the acc loop's column n
            hc, hh = 0, 0
            for h in range(NH):
                if h == n:
                    assert (tq0 + hc) * qh + h0 + hh == row
                hh += 1
                if hh == wrap:
                    hh, hc = 0, hc + 1
            key = (row, split)
            assert key not in written, f"partial {key} written twice"
            written[key] = (lim, t_begin)
    # every partial the combine reads is written once, with that vector's own length
    for qi in range(nq):
        c = causal_len(qi, kv_len, start_pos, max_blocks, seq_lens)
        ns = (c + SPLIT - 1) // SPLIT
        for h in range(qh):
            for s in range(ns):
                lim, t_begin = written.pop((qi * qh + h, s))
                assert lim == min(c, t_begin + SPLIT), (qi, h, s, lim)
                assert lim > t_begin or c == 0
    # what is left was written past a vector's causal length and is never read
    for (row, s), (lim, t_begin) in written.items():
        assert lim <= t_begin
    assert len(q_rows) == sum(qh for qi in range(nq)
                              if causal_len(qi, kv_len, start_pos, max_blocks, seq_lens) > 0)
    return tok


@pytest.mark.parametrize("nq,qh,kvh,kv_len,start_pos,tok", [
    (19, 4, 4, 1050, 1020, 8), (13, 8, 4, 300, 0, 4), (11, 6, 2, 1100, 1019, 2), (70, 8, 2, 70, 0, 2),
    (9, 16, 16, 2100, 2040, 8), (7, 16, 2, 50, 43, 1), (37, 32, 8, 3000, 2963, 2), (5, 24, 2, 1030, 1025, 1),
    (1, 8, 8, 40, 39, 1), (33, 32, 4, 2100, 2067, 1), (21, 8, 8, 600, 579, 8)])
def test_prefill_groups_cover_every_partial(nq, qh, kvh, kv_len, start_pos, tok):
    assert model_split_kernel(nq, qh, kvh, kv_len, start_pos) == tok


def test_decode_rows_keep_one_query_per_wave():
    lens = np.array([5, 1030, 0, 2048, 17], np.int32)
    assert model_split_kernel(len(lens), 32, 8, 0, 0, shared_table=False, seq_lens=lens) == 1


def test_column_mapping_error_is_caught():
    """The model fails when the acc loop's column counter wraps at the wrong head count."""
    with pytest.raises(AssertionError):
        model_split_kernel(13, 8, 4, 300, 0, wrap=3)


@pytest.mark.parametrize("nq,qh,kvh,kv_len,start_pos", [
    (2, 8, 8, 40, 38), (130, 32, 8, 1130, 1000), (129, 128, 128, 2100, 1971), (37, 24, 3, 1200, 1163),
    (1000, 32, 8, 4001, 3001), (70, 7, 1, 70, 0), (65, 16, 2, 5000, 4000)])
@pytest.mark.parametrize("part", [SPLIT, 256])
@pytest.mark.parametrize("cus", [0, 8, 64, 256])
def test_tiled_prefill_covers_every_partial(nq, qh, kvh, kv_len, start_pos, part, cus):
    """Workgroups of the tiled prefill kernels (128 columns of one kv head, one split), as the launchers'
    functions split them over a workspace of `part`-position partials: each (vector, split) below the
    vector's causal length is written once, no split count exceeds the workspace's, tiles start inside a
    64-page window with their four pages, and the order of blocks (from the last down, folded where
    they fit `cus` CUs twice) is a permutation."""
    G = qh // kvh
    ws = max(1, -(-(-(-kv_len // PAGE) * PAGE) // part))
    nqb, nblk, nsplit, pos, wgs = rules.prefill_split(nq, G, kvh, kv_len, ws)
    assert nsplit <= ws and pos % 64 == 0 and wgs == nblk * kvh * nsplit
    assert nqb * G <= 128 and (nblk - 1) * nqb < nq <= nblk * nqb and (nsplit - 1) * pos < kv_len <= nsplit * pos
    fold = rules.lib().fhip_rule_prefill_fold(nsplit, wgs, kvh, cus)
    assert 0 <= fold < max(nblk, 1)
    order = [rules.lib().fhip_idx_prefill_block(bi, nblk, fold) for bi in range(nblk)]
    assert sorted(order) == list(range(nblk))
    written = {}
    for blk in order:
        q0 = blk * nqb
        n = min(nqb, nq - q0)
        clen = min(start_pos + q0 + n, kv_len)
        for split in range(nsplit):
            t_begin = split * pos
            if nsplit > 1 and t_begin >= clen:
                continue
            win = t_begin
            for t0 in range(t_begin, min(clen, t_begin + pos), 64):
                if t0 >= win + 64 * PAGE:
                    win = t0
                assert 0 <= (t0 - win) // PAGE <= 60 and (t0 - win) % PAGE == 0
            for col in range(n * G):
                for g in range(kvh):
                    key = ((q0 + col // G) * qh + g * G + col % G, split)
                    assert key not in written
                    written[key] = min(clen, t_begin + pos)
    for qi in range(nq):
        c = min(start_pos + qi + 1, kv_len)
        for s in range(-(-c // pos)):
            for h in range(qh):
                assert written[(qi * qh + h, s)] >= min(c, (s + 1) * pos)


def test_prefill_folds_a_single_split():
    """2048 queries of 32 / 8 heads: 512 workgroups on 256 CUs, the second half from the first block up."""
    nqb, nblk, nsplit, pos, wgs = rules.prefill_split(2048, 4, 8, 2048, 8)
    assert (nqb, nblk, nsplit, wgs) == (32, 64, 1, 512)
    fold = rules.lib().fhip_rule_prefill_fold(nsplit, wgs, 8, 256)
    assert fold == 32
    order = [rules.lib().fhip_idx_prefill_block(bi, nblk, fold) for bi in range(nblk)]
    assert order == list(range(63, 31, -1)) + list(range(32))


@pytest.mark.parametrize("bits", [2, 3, 4, 8])
@pytest.mark.parametrize("kvh", [1, 3, 8])
def test_prefill_code_loads_cover_each_row_once(bits, kvh):
    """A tile's 64 rows of four quarters: each byte of kv head g's codes on the tile's four pages once."""
    for g in range(kvh):
        seen = np.zeros((4, PAGE * kvh * 16 * bits), np.int32)
        for row in range(64):
            for quarter in range(4):
                off = rules.lib().fhip_idx_prefill_code_offset(row, quarter, kvh, g, bits)
                seen[row // PAGE, off:off + 4 * bits] += 1
        rows = seen.reshape(4, PAGE, kvh, 16 * bits)
        assert (rows[:, :, g] == 1).all() and rows.sum() == 64 * 16 * bits
