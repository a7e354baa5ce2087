"""GPU parity of TurboQuant paged decode attention against the oracle's restatement of
attention_paged_tq.cu (fp16 output, |a - e| <= 1e-3 + 1e-3|e|).

Covers the batched decode entry over contiguous page pools (one query per sequence,
per-sequence lengths, permuted block tables, split-K merging across 1024-position splits),
the reference-interface entry with per-block pointer arrays and causal prefill queries, and
several bit-width pairs.
"""
import numpy as np
import pytest
import torch

import oracle
import rules
from conftest import assert_close
from fracture_amd import kernels as K
from fracture_amd import turboquant as tq

pytestmark = pytest.mark.gpu


def dev_t(a, dev):
    return torch.from_numpy(np.ascontiguousarray(a)).to(dev)


def build_pool(rng, lens, kvh, hd, kbits, vbits, extra_pages=3):
    """Compress random K/V for each sequence into a shared, permuted page pool."""
    pdk, pdv = oracle.packed_dim(hd, kbits), oracle.packed_dim(hd, vbits)
    nbs = [(n + 15) // 16 for n in lens]
    P = sum(nbs) + extra_pages
    perm = rng.permutation(P).astype(np.int32)
    krot, vrot = tq.rotation_matrix(hd, 42), tq.rotation_matrix(hd, 542)
    kc, vc = tq.codebook(hd, kbits)[0], tq.codebook(hd, vbits)[0]
    KP = rng.integers(0, 256, (P, 16, kvh * pdk)).astype(np.uint8)  # garbage in unused slots
    VP = rng.integers(0, 256, (P, 16, kvh * pdv)).astype(np.uint8)
    KN = np.full((P, 16, kvh), np.float16(3.0))
    VN = np.full((P, 16, kvh), np.float16(3.0))
    maxb = max(nbs)
    table = np.full((len(lens), maxb), -7, np.int32)
    at = 0
    for b, n in enumerate(lens):
        pages = perm[at:at + nbs[b]]
        at += nbs[b]
        table[b, :nbs[b]] = pages
        if n == 0:
            continue
        k = (rng.standard_normal((n, kvh, hd)) * np.exp(rng.normal(0, 0.5, (n, 1, 1)))).astype(np.float16)
        v = (rng.standard_normal((n, kvh, hd)) * np.exp(rng.normal(0, 0.5, (n, 1, 1)))).astype(np.float16)
        kp, kn, _ = oracle.tq_compress(k, krot, kc, kbits)
        vp, vn, _ = oracle.tq_compress(v, vrot, vc, vbits)
        for t in range(n):
            p, s = pages[t // 16], t % 16
            KP[p, s] = kp.reshape(n, -1)[t]
            KN[p, s] = kn.reshape(n, kvh)[t]
            VP[p, s] = vp.reshape(n, -1)[t]
            VN[p, s] = vn.reshape(n, kvh)[t]
    return dict(KP=KP, KN=KN, VP=VP, VN=VN, table=table, krot=krot, vrot=vrot, kc=kc, vc=vc)


@pytest.mark.parametrize("kbits,vbits", [(4, 4), (4, 2), (3, 3), (8, 2)])
@pytest.mark.parametrize("lens", [[1, 15, 16, 17], [300, 1024, 1025, 2100]])
def test_decode_attention_vs_oracle(dev, kbits, vbits, lens):
    rng = np.random.default_rng(sum(lens) + kbits * 10 + vbits)
    qh, kvh, hd = 8, 2, 128
    pool = build_pool(rng, lens, kvh, hd, kbits, vbits)
    B = len(lens)
    q = rng.standard_normal((B, qh, hd)).astype(np.float16)
    out = torch.empty((B, qh, hd), dtype=torch.float16, device=dev)
    K.attention_tq_decode(out, dev_t(q, dev), dev_t(pool["table"], dev),
                          dev_t(np.array(lens, np.int32), dev), dev_t(pool["KP"], dev),
                          dev_t(pool["KN"], dev), dev_t(pool["VP"], dev), dev_t(pool["VN"], dev),
                          dev_t(pool["krot"], dev), dev_t(pool["vrot"], dev),
                          dev_t(pool["kc"], dev), dev_t(pool["vc"], dev), kbits, vbits, kvh)
    torch.cuda.synchronize()
    got = out.cpu().numpy()
    for b in range(B):
        want = oracle.tq_attention(q[b], pool["table"][b], lens[b], pool["KP"], pool["KN"],
                                   pool["VP"], pool["VN"], pool["krot"], pool["vrot"],
                                   pool["kc"], pool["vc"], kbits, vbits, kvh)
        assert_close(got[b].astype(np.float32), want.astype(np.float32), 1e-3, 1e-3,
                     f"sequence {b} (len {lens[b]})")


def test_decode_attention_llama_heads(dev):
    # Llama-3.1-8B head layout: 32 q heads over 8 kv heads, K4/V4
    rng = np.random.default_rng(8)
    lens = [37, 1500, 3000, 16]
    qh, kvh, hd = 32, 8, 128
    pool = build_pool(rng, lens, kvh, hd, 4, 4)
    q = rng.standard_normal((len(lens), qh, hd)).astype(np.float16)
    out = torch.empty((len(lens), qh, hd), dtype=torch.float16, device=dev)
    K.attention_tq_decode(out, dev_t(q, dev), dev_t(pool["table"], dev),
                          dev_t(np.array(lens, np.int32), dev), dev_t(pool["KP"], dev),
                          dev_t(pool["KN"], dev), dev_t(pool["VP"], dev), dev_t(pool["VN"], dev),
                          dev_t(pool["krot"], dev), dev_t(pool["vrot"], dev),
                          dev_t(pool["kc"], dev), dev_t(pool["vc"], dev), 4, 4, kvh)
    torch.cuda.synchronize()
    got = out.cpu().numpy()
    for b in range(len(lens)):
        want = oracle.tq_attention(q[b], pool["table"][b], lens[b], pool["KP"], pool["KN"],
                                   pool["VP"], pool["VN"], pool["krot"], pool["vrot"],
                                   pool["kc"], pool["vc"], 4, 4, kvh)
        assert_close(got[b].astype(np.float32), want.astype(np.float32), 1e-3, 1e-3, f"seq {b}")


def test_reference_interface_prefill_causal(dev):
    """fhip_launch_attention_paged_tq: T queries at start_pos.., per-block pointer arrays."""
    rng = np.random.default_rng(21)
    qh, kvh, hd, kbits, vbits = 4, 2, 128, 4, 2
    kv_len, T = 90, 6
    start_pos = kv_len - T
    pool = build_pool(rng, [kv_len], kvh, hd, kbits, vbits, extra_pages=2)
    P = pool["KP"].shape[0]
    tKP, tKN, tVP, tVN = (dev_t(pool[n], dev) for n in ("KP", "KN", "VP", "VN"))
    ptrs = [torch.tensor([t[i].data_ptr() for i in range(P)], dtype=torch.int64, device=dev)
            for t in (tKP, tKN, tVP, tVN)]
    q = rng.standard_normal((T, qh, hd)).astype(np.float16)
    tq_ = dev_t(q, dev)
    out = torch.empty_like(tq_)
    table = dev_t(pool["table"][0], dev)
    lib = K._L()
    krot, vrot = dev_t(pool["krot"], dev), dev_t(pool["vrot"], dev)
    kc, vc = dev_t(pool["kc"], dev), dev_t(pool["vc"], dev)
    code = lib.fhip_launch_attention_paged_tq(
        out.data_ptr(), tq_.data_ptr(), table.data_ptr(), ptrs[0].data_ptr(), ptrs[1].data_ptr(),
        ptrs[2].data_ptr(), ptrs[3].data_ptr(), krot.data_ptr(), vrot.data_ptr(), kc.data_ptr(),
        vc.data_ptr(), T, qh, kvh, hd, kv_len, start_pos, kbits, vbits,
        oracle.packed_dim(hd, kbits), oracle.packed_dim(hd, vbits),
        torch.cuda.current_stream().cuda_stream)
    assert code == 0
    torch.cuda.synchronize()
    got = out.cpu().numpy()
    for t in range(T):
        clen = min(start_pos + t + 1, kv_len)
        want = oracle.tq_attention(q[t], pool["table"][0], clen, pool["KP"], pool["KN"],
                                   pool["VP"], pool["VN"], pool["krot"], pool["vrot"],
                                   pool["kc"], pool["vc"], kbits, vbits, kvh)
        assert_close(got[t].astype(np.float32), want.astype(np.float32), 1e-3, 1e-3, f"token {t}")


@pytest.mark.parametrize("kbits,vbits", [(8, 8), (3, 3), (2, 2), (4, 2), (4, 4)])
@pytest.mark.parametrize("qh,kvh,reps,part,waves", [
    (8, 2, 1, 256, 4), (8, 1, 1, 256, 4), (16, 8, 13, 1024, 2), (64, 8, 13, 1024, 2), (16, 4, 4, 1024, 4),
    (32, 4, 4, 1024, 4)])
def test_decode_widths_and_waves(dev, kbits, vbits, qh, kvh, reps, part, waves):
    """Every width pair of the MFMA kernel, at up to 4 and up to 8 q heads per kv head, in 256-position
    parts, in 1024-position blocks of four waves and of two: lengths on the edges of chunks, of the
    waves' splits and of pages, a masked page, an empty sequence."""
    rng = np.random.default_rng(kbits * 10 + vbits + qh)
    hd = 128
    lens = ([1, 65, 128, 0, 300] if waves == 2 else
            [1, 63, 64, 65, 127, 129, 255, 257, 511, 513, 0, 1023, 1025 if part == 256 else 1800])
    route = rules.TqRoute(len(lens) * reps, qh, kvh, kbits, vbits, max(lens))
    assert (route.kind, route.part, route.waves) == (rules.DECODE, part, waves)
    pool = build_pool(rng, lens, kvh, hd, kbits, vbits)
    pool["table"][2, 1] = -1  # the third sequence (of 128 or 64): positions 16..31 masked
    table, lens = np.tile(pool["table"], (reps, 1)), lens * reps
    q = rng.standard_normal((len(lens), qh, hd)).astype(np.float16)
    out = torch.empty(q.shape, dtype=torch.float16, device=dev)
    K.attention_tq_decode(out, dev_t(q, dev), dev_t(table, dev), dev_t(np.array(lens, np.int32), dev),
                          *(dev_t(pool[n], dev) for n in ("KP", "KN", "VP", "VN", "krot", "vrot", "kc", "vc")),
                          kbits, vbits, kvh)
    torch.cuda.synchronize()
    got = out.cpu().numpy()
    for b, n in enumerate(lens):
        rows = table[b]
        if n == 0:
            assert not got[b].any()
            continue
        if rows[1] == -1 and n > 32:
            rows, n = np.delete(rows, 1), n - 16
        want = oracle.tq_attention(q[b], rows, n, pool["KP"], pool["KN"], pool["VP"], pool["VN"],
                                   pool["krot"], pool["vrot"], pool["kc"], pool["vc"], kbits, vbits, kvh)
        assert_close(got[b].astype(np.float32), want.astype(np.float32), 1e-3, 1e-3, f"seq {b} len {n}")


@pytest.mark.parametrize("bits", [8, 3, 2])
def test_code_pages_at_odd_addresses(dev, bits):
    """Code pages that start at any byte (the widths other than 4 assume no alignment), through the
    per-block pointer arrays."""
    rng = np.random.default_rng(bits)
    qh, kvh, hd, n = 4, 2, 128, 100
    pool = build_pool(rng, [n], kvh, hd, bits, bits)
    P = pool["KP"].shape[0]
    held, ptrs = [], []
    for name in ("KP", "KN", "VP", "VN"):
        t = []
        for i in range(P):
            raw = np.ascontiguousarray(pool[name][i]).view(np.uint8).ravel()
            buf = torch.zeros(raw.size + 16, dtype=torch.uint8, device=dev)
            off = (2 * i + 1) % 16 if name in ("KP", "VP") else 0
            buf[off:off + raw.size] = torch.from_numpy(raw.copy()).to(dev)
            held.append(buf)
            t.append(buf.data_ptr() + off)
        ptrs.append(torch.tensor(t, dtype=torch.int64, device=dev))
    q = rng.standard_normal((1, qh, hd)).astype(np.float16)
    tq_, table = dev_t(q, dev), dev_t(pool["table"][0], dev)
    tabs = [dev_t(pool[x], dev) for x in ("krot", "vrot", "kc", "vc")]
    out = torch.empty_like(tq_)
    pd = oracle.packed_dim(hd, bits)
    code = K._L().fhip_launch_attention_paged_tq(
        out.data_ptr(), tq_.data_ptr(), table.data_ptr(), *(p.data_ptr() for p in ptrs),
        *(t.data_ptr() for t in tabs), 1, qh, kvh, hd, n, n - 1, bits, bits, pd, pd,
        torch.cuda.current_stream().cuda_stream)
    assert code == 0
    torch.cuda.synchronize()
    want = oracle.tq_attention(q[0], pool["table"][0], n, pool["KP"], pool["KN"], pool["VP"], pool["VN"],
                               pool["krot"], pool["vrot"], pool["kc"], pool["vc"], bits, bits, kvh)
    assert_close(out.cpu().numpy()[0].astype(np.float32), want.astype(np.float32), 1e-3, 1e-3)


@pytest.mark.parametrize("splits", [1, 3, 4, 5, 16, 17, 33])
def test_merge_of_splits(dev, splits):
    """The head_dim 128 merge at the edges of its chunks of 4 and of 16 splits, beside sequences that end in
    an earlier split and an empty one."""
    rng = np.random.default_rng(splits)
    qh, kvh = 8, 2
    lens = [256 * splits, 256 * splits - 255, 1, 0, max(1, 256 * (splits - 2)), 256 * splits - 16]
    route = rules.TqRoute(len(lens), qh, kvh, 4, 4, lens[0])
    assert (route.kind, route.part, route.nsplit) == (rules.DECODE, 256, splits)
    pool = build_pool(rng, lens, kvh, 128, 4, 4)
    q = rng.standard_normal((len(lens), qh, 128)).astype(np.float16)
    out = torch.empty(q.shape, dtype=torch.float16, device=dev)
    K.attention_tq_decode(out, dev_t(q, dev), dev_t(pool["table"], dev), dev_t(np.array(lens, np.int32), dev),
                          *(dev_t(pool[n], dev) for n in ("KP", "KN", "VP", "VN", "krot", "vrot", "kc", "vc")),
                          4, 4, kvh)
    got = out.cpu().numpy().astype(np.float32)
    for b, n in enumerate(lens):
        want = oracle.tq_attention(q[b], pool["table"][b], n, pool["KP"], pool["KN"], pool["VP"], pool["VN"],
                                   pool["krot"], pool["vrot"], pool["kc"], pool["vc"], 4, 4, kvh)
        assert_close(got[b], want.astype(np.float32), 1e-3, 1e-3, f"sequence {b}")


@pytest.mark.parametrize("kbits,vbits,qh,kvh", [(4, 2, 32, 8), (8, 8, 8, 2)])
def test_workspace_of_a_shorter_table(dev, kbits, vbits, qh, kvh):
    """A workspace sized for one block serves a table of 60, which launches in 256-position parts, in decode
    and through the entry that is told its size; nothing is written past it."""
    rng = np.random.default_rng(kbits)
    n, guard = 960, 1 << 20
    pool = build_pool(rng, [n], kvh, 128, kbits, vbits)
    route = rules.TqRoute(1, qh, kvh, kbits, vbits, n)
    assert (route.kind, route.part, route.nsplit) == (rules.DECODE, 256, 4)
    size = K._L().fhip_attention_tq_workspace_bytes(1, qh, 128, 1)
    assert size == rules.tq_workspace(1, qh, 128, n) and route.bytes <= size
    parts = [dev_t(pool[x], dev) for x in ("KP", "KN", "VP", "VN")]
    tabs = [dev_t(pool[x], dev) for x in ("krot", "vrot", "kc", "vc")]
    q = rng.standard_normal((1, qh, 128)).astype(np.float16)
    tq_, table, lens = dev_t(q, dev), dev_t(pool["table"], dev), dev_t(np.array([n], np.int32), dev)
    ptrs = [torch.tensor([x.data_ptr() for x in t], dtype=torch.int64, device=dev) for t in parts]
    pd = [oracle.packed_dim(128, b) for b in (kbits, vbits)]
    s = torch.cuda.current_stream().cuda_stream
    want = oracle.tq_attention(q[0], pool["table"][0], n, pool["KP"], pool["KN"], pool["VP"], pool["VN"],
                               pool["krot"], pool["vrot"], pool["kc"], pool["vc"], kbits, vbits, kvh)
    for told in (False, True):
        ws = torch.full((size + guard,), 0x5A, dtype=torch.uint8, device=dev)
        out = torch.empty_like(tq_)
        if told:
            code = K._L().fhip_launch_attention_paged_tq_ws(
                out.data_ptr(), tq_.data_ptr(), table.data_ptr(), *(p.data_ptr() for p in ptrs),
                *(t.data_ptr() for t in tabs), 1, qh, kvh, 128, n, n - 1, kbits, vbits, *pd, ws.data_ptr(), size, s)
        else:
            code = K._L().fhip_launch_attention_tq_decode(
                out.data_ptr(), tq_.data_ptr(), table.data_ptr(), lens.data_ptr(), 1, table.shape[1],
                parts[0].shape[0], *(p.data_ptr() for p in parts), *(p[0].nbytes for p in parts),
                *(t.data_ptr() for t in tabs), qh, kvh, 128, kbits, vbits, ws.data_ptr(), s)
        assert code == 0
        torch.cuda.synchronize()
        assert (ws[size:] == 0x5A).all()
        assert_close(out.cpu().numpy()[0].astype(np.float32), want.astype(np.float32), 1e-3, 1e-3, f"told {told}")


def run_prefill(dev, pool, q, kvh, kv_len, start_pos, kbits, vbits):
    P, T, qh, hd = pool["KP"].shape[0], *q.shape
    parts = [dev_t(pool[n], dev) for n in ("KP", "KN", "VP", "VN")]
    ptrs = [torch.tensor([x.data_ptr() for x in t], dtype=torch.int64, device=dev) for t in parts]
    tq_, table = dev_t(q, dev), dev_t(pool["table"][0], dev)
    tabs = [dev_t(pool[x], dev) for x in ("krot", "vrot", "kc", "vc")]
    out = torch.empty_like(tq_)
    code = K._L().fhip_launch_attention_paged_tq(
        out.data_ptr(), tq_.data_ptr(), table.data_ptr(), *(p.data_ptr() for p in ptrs),
        *(t.data_ptr() for t in tabs), T, qh, kvh, hd, kv_len, start_pos, kbits, vbits,
        oracle.packed_dim(hd, kbits), oracle.packed_dim(hd, vbits), torch.cuda.current_stream().cuda_stream)
    assert code == 0
    torch.cuda.synchronize()
    return out.cpu().numpy().astype(np.float32)


@pytest.mark.parametrize("kbits,vbits,qh,kvh,T,kv_len,tiled", [
    # several splits, ragged columns: G = 2, 4, 8, 3, 1 (5 splits of the positions or more)
    (4, 2, 16, 8, 130, 1100, True), (4, 4, 16, 4, 300, 1800, True), (8, 8, 16, 2, 60, 3000, True),
    (3, 3, 24, 8, 45, 1301, True), (2, 2, 8, 8, 260, 1537, True),
    # the same with too few columns for it, on the decode kernel
    (4, 4, 16, 4, 65, 1800, False), (2, 2, 8, 8, 130, 1537, False),
    # one split and a batch of vectors that skips the merge, blocks going up after those going down
    (4, 2, 32, 8, 2048, 2048, True),
    # a batch of vectors whose splits the wave merge takes
    (4, 2, 32, 8, 130, 2560, True),
    # a batch in fewer and longer splits, and in 16 that the merge in LDS takes
    (3, 3, 32, 8, 130, 3000, True), (4, 4, 16, 2, 256, 20000, True)])
def test_prefill_tiles(dev, kbits, vbits, qh, kvh, T, kv_len, tiled):
    """The causal prefill kernel against the oracle, with a masked page and with a value norm of
    infinity and a key norm of NaN at late positions, which no earlier query may see; the value norms
    span 2^-10 .. 2^10."""
    route = rules.TqRoute(T, qh, kvh, kbits, vbits, kv_len, causal=True)
    assert (route.kind == rules.PREFILL) == tiled
    rng = np.random.default_rng(kbits * 100 + T)
    hd, start = 128, kv_len - T
    pool = build_pool(rng, [kv_len], kvh, hd, kbits, vbits)
    table = pool["table"][0]
    pool["VN"] *= np.exp2(rng.uniform(-10, 10, pool["VN"].shape[:2]))[..., None].astype(np.float16)
    table[2] = -5  # positions 32..47 masked
    pool["VN"][table[(kv_len - 3) // 16], (kv_len - 3) % 16] = np.inf
    pool["KN"][table[(kv_len - 2) // 16], (kv_len - 2) % 16] = np.nan
    q = rng.standard_normal((T, qh, hd)).astype(np.float16)
    got = run_prefill(dev, pool, q, kvh, kv_len, start, kbits, vbits)
    for t in sorted({0, 1, T // 3, T // 2, T - 5, T - 4} | set(range(0, T - 4, max(1, T // 12)))):
        n = start + t + 1
        if n <= 48:
            n = min(n, 32)
            rows = table
        else:
            rows, n = np.delete(table, 2), n - 16
        want = oracle.tq_attention(q[t], rows, n, pool["KP"], pool["KN"], pool["VP"], pool["VN"],
                                   pool["krot"], pool["vrot"], pool["kc"], pool["vc"], kbits, vbits, kvh)
        scale = max(1.0, float(np.abs(want.astype(np.float32)).max()))  # norms up to 2^10
        assert_close(got[t] / scale, want.astype(np.float32) / scale, 1e-3, 1e-3, f"token {t}")
