"""Which kernel and split the attention and matmul launchers choose (fracture_amd/csrc/launch_rules.h)."""
import pytest

import rules


@pytest.mark.parametrize("queries,qh,kvh,hd,tokens,waves", [
    # up to 256, 512, 1024 splits and more, tables of whole splits
    (1, 32, 8, 128, 4000, 8), (32, 32, 8, 128, 1024, 8), (33, 32, 8, 128, 1024, 4), (64, 32, 8, 128, 1000, 4),
    (65, 32, 8, 128, 1024, 2), (128, 32, 8, 128, 1024, 2), (193, 32, 8, 128, 1024, 1),
    (64, 32, 8, 128, 4000, 1), (256, 32, 8, 128, 1100, 1), (64, 32, 32, 128, 1000, 1),
    (16, 64, 8, 64, 8000, 2), (16, 8, 8, 32, 8000, 1), (257, 16, 4, 256, 1000, 1), (128, 16, 4, 256, 1000, 4),
    # between 512 and 1536 splits, by head_dim
    (129, 32, 8, 128, 1024, 4), (192, 32, 8, 128, 1024, 4), (129, 32, 8, 128, 528, 4), (129, 32, 8, 128, 512, 1),
    (96, 16, 8, 64, 2000, 2), (97, 16, 8, 64, 2000, 1), (192, 32, 8, 64, 512, 1), (128, 16, 8, 64, 300, 2),
    (128, 16, 8, 64, 128, 1), (256, 16, 4, 256, 1000, 2), (32, 8, 8, 32, 3000, 2), (33, 8, 8, 32, 3000, 1),
    # short tables: no waves past their end, at head_dim 128 not below two
    (1, 32, 8, 128, 128, 2), (1, 32, 8, 128, 144, 8), (64, 32, 8, 128, 256, 2), (64, 32, 8, 128, 272, 4),
    (128, 32, 8, 128, 100, 2), (256, 32, 8, 128, 16, 1), (8, 16, 8, 64, 64, 1), (8, 16, 8, 64, 208, 8),
    (64, 16, 8, 64, 368, 1), (64, 16, 8, 64, 400, 4), (64, 8, 8, 32, 16, 1), (8, 16, 4, 256, 100, 1)])
def test_waves_of_a_paged_decode(queries, qh, kvh, hd, tokens, waves):
    assert rules.paged_waves(queries, qh, kvh, hd, tokens) == waves


@pytest.mark.parametrize("queries,qh,kvh,kbits,vbits,kv_len,part,waves", [
    # 256-position parts: at most 768 of their workgroups and 48 parts
    (1, 32, 8, 4, 2, 4001, 256, 4), (32, 32, 8, 4, 2, 700, 256, 4), (64, 32, 8, 4, 4, 16, 256, 4),
    (1, 32, 8, 4, 2, 12288, 256, 4), (1, 32, 8, 4, 2, 12289, 1024, 4), (1, 32, 8, 8, 8, 32000, 1024, 4),
    (64, 32, 8, 3, 3, 1000, 1024, 4), (8, 32, 8, 8, 8, 8000, 1024, 4), (32, 32, 8, 4, 2, 1000, 1024, 4),
    # up to 1536 where 1024-position parts would be a second turn: 257 .. 384 workgroups, 512 of several parts
    (40, 32, 8, 4, 2, 700, 256, 4), (48, 32, 8, 4, 2, 1024, 256, 4), (49, 32, 8, 4, 2, 700, 1024, 4),
    (24, 32, 8, 8, 8, 1400, 256, 4), (32, 32, 8, 4, 4, 1400, 256, 4), (32, 32, 8, 4, 4, 1600, 1024, 4),
    # above 512 workgroups two waves
    (65, 32, 8, 4, 2, 1024, 1024, 2), (64, 32, 8, 4, 2, 32768, 1024, 2), (256, 32, 8, 2, 2, 16, 1024, 2)])
def test_route_of_a_tq_decode(queries, qh, kvh, kbits, vbits, kv_len, part, waves):
    r = rules.TqRoute(queries, qh, kvh, kbits, vbits, kv_len)
    assert (r.kind, r.part, r.waves, r.tok) == (rules.DECODE, part, waves, 1)
    assert r.nsplit == -(-(-(-kv_len // 16) * 16) // part)


@pytest.mark.parametrize("qh,kvh,hd,kbits,vbits", [(8, 2, 64, 4, 4), (8, 2, 256, 4, 2), (8, 2, 128, 8, 2), (8, 2, 128, 3, 4),
                                                  (8, 2, 128, 5, 5)])
def test_other_widths_and_head_dims_stay_on_the_valu_kernel(qh, kvh, hd, kbits, vbits):
    for causal in (False, True):
        r = rules.TqRoute(300, qh, kvh, kbits, vbits, 3000, causal, hd=hd)
        assert (r.kind, r.part, r.nsplit) == (rules.VALU, 1024, 3)


@pytest.mark.parametrize("queries,qh,kvh,kbits,vbits,kv_len,kind,part,nsplit,split_pos", [
    # few columns or short: the decode kernel, in the parts a decode would take
    (2, 32, 8, 4, 2, 8000, rules.DECODE, 256, 32, 256), (16, 32, 8, 4, 2, 100, rules.DECODE, 256, 1, 256),
    (8, 32, 8, 4, 2, 8000, rules.DECODE, 1024, 8, 1024), (32, 32, 8, 4, 2, 3000, rules.DECODE, 1024, 3, 1024),
    # many
    (2048, 32, 8, 4, 2, 2048, rules.PREFILL, 1024, 1, 2048), (130, 32, 8, 4, 4, 1000, rules.PREFILL, 256, 4, 256),
    # the codes' expansion is dearer at 8 and 3 bits
    (32, 32, 8, 8, 8, 3000, rules.PREFILL, 256, 12, 256), (32, 32, 8, 3, 3, 3000, rules.PREFILL, 256, 12, 256),
    # from 4096 vectors on 128 workgroups at 4 and 2 bits, and the 8 splits that a wave merges or, of long
    # contexts, as many as fit at once
    (130, 32, 8, 4, 2, 2560, rules.PREFILL, 256, 8, 320), (600, 8, 8, 4, 4, 600, rules.DECODE, 1024, 1, 1024),
    (64, 64, 8, 4, 4, 30000, rules.PREFILL, 1024, 16, 1920), (130, 32, 8, 4, 4, 30000, rules.PREFILL, 1024, 12, 2560),
    (200, 32, 8, 4, 4, 30000, rules.PREFILL, 1024, 9, 3392), (130, 64, 8, 4, 4, 30000, rules.PREFILL, 1024, 7, 4288),
    (130, 32, 8, 4, 4, 3000, rules.DECODE, 1024, 3, 1024), (600, 8, 8, 8, 8, 3000, rules.PREFILL, 1024, 3, 1024),
    # long tiles on a part of the chip lose to the decode kernel
    (200, 64, 8, 4, 2, 1000, rules.DECODE, 1024, 1, 1024), (8, 32, 8, 4, 2, 30000, rules.DECODE, 1024, 30, 1024)])
def test_route_of_a_tq_prefill(queries, qh, kvh, kbits, vbits, kv_len, kind, part, nsplit, split_pos):
    r = rules.TqRoute(queries, qh, kvh, kbits, vbits, kv_len, causal=True)
    assert (r.kind, r.part, r.nsplit, r.split_pos) == (kind, part, nsplit, split_pos)


@pytest.mark.parametrize("m,n,k,streamed", [
    (1, 4096, 4096, True), (16, 1024, 4096, True), (17, 1024, 4096, False), (8, 14336, 4096, False),
    # a workgroup's waves share K: 8192 of it with up to 4 rows, 4096 with up to 16
    (4, 1024, 8192, True), (5, 1024, 8192, False), (16, 2048, 14336, False), (1, 16, 1 << 20, False),
    (1, 512, 1 << 18, False),
    # one or two rows on up to 2^27 elements of a wide B
    (2, 14336, 4096, True), (2, 4096, 14336, True), (3, 14336, 4096, False), (2, 2048, 14336, False),
    (1, 32000, 4096, True), (1, 128256, 4096, False),
    # many short rows; K that is no multiple of 8
    (1, 65536, 64, True), (16, 1 << 19, 64, False), (1, 4096, 4, False), (1, 4096, 4100, False), (0, 8, 8, False)])
def test_route_of_a_matmul(m, n, k, streamed):
    assert bool(rules.lib().fhip_rule_matmul_skinny(m, n, k)) == streamed


@pytest.mark.parametrize("queries,qh,hd", [(1, 32, 128), (1, 8, 128), (7, 24, 128), (64, 32, 128), (300, 64, 128), (5, 8, 64)])
def test_workspace_serves_every_table_of_its_splits(queries, qh, hd):
    """A workspace sized for one table serves, in every layout that a launch may choose, each table of as many
    1024-position splits, and every smaller call; the size never falls as an argument grows."""
    G = 8 if qh % 8 == 0 else 1
    last = 0
    for split in (1, 2, 3, 9, 12, 13, 48, 64):
        sizes = set()
        for blocks in (64 * split - 63, 64 * split - 40, 64 * split - 15, 64 * split):
            n = 16 * blocks
            size = rules.tq_workspace(queries, qh, hd, n)
            sizes.add(size)
            for causal in (False, True):
                for bits in (4, 8):
                    smallest = rules.tq_workspace(queries, qh, hd, 16 * (64 * split - 63))
                    r = rules.TqRoute(queries, qh, qh // G, bits, bits, n, causal, hd=hd, ws_bytes=size)
                    assert r.bytes <= smallest, (blocks, causal, r.part)
        assert len(sizes) == 1
        assert last <= size and size <= rules.tq_workspace(queries + 1, qh, hd, n)
        assert size <= rules.tq_workspace(queries, qh + G, hd, n)
        last = size
