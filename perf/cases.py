"""The work a user of this backend has it do, as timed cases: the kernels between the GEMMs of
a decode step and of a prefill, the sampler's reductions, the TurboQuant cache's writer and
reader, attention over TurboQuant and FP16 pages (one sequence, a batch, a causal prefill) and
a whole decode step through the handle runtime.

Sizes are Llama-3.1-8B's (hidden 4096, FFN 14336, 32 query / 8 kv heads of 128, vocabulary
128256), the model of this repository's benchmark, with other head counts, widths and ragged
lengths among the drawn cases. Inputs come from the seed alone. TurboQuant pages hold codes of
Gaussian coordinates, which is what a rotated unit vector has.
"""
from __future__ import annotations

import functools
import math

import numpy as np
import torch

from fracture_amd import DType, HipBackend
from fracture_amd import kernels as K
from fracture_amd import turboquant as tq

PAGE = tq.BLOCK_SIZE
EPS = 1e-5
THETA = 500000.0
DTYPES = {"fp16": torch.float16, "bf16": torch.bfloat16, "fp32": torch.float32}


def listed():
    return [
        # the launches between the GEMMs of one decode step of a batch, captured as a graph
        {"name": "step-chain-b64", "kind": "step_chain", "tokens": 64, "hidden": 4096, "ffn": 14336},
        # the same ops over the rows of a prefill batch, where memory bounds them
        {"name": "prefill-chain-8192", "kind": "rows_chain", "tokens": 8192, "hidden": 4096,
         "ffn": 14336, "dtype": "fp16"},
        # sampling probabilities and greedy tokens of a batch's logits
        {"name": "sample-64", "kind": "sample", "rows": 64, "vocab": 128256},
        # a layer's keys and values compressed after a prefill, default cache widths
        {"name": "compress-32k", "kind": "compress", "tokens": 32768, "kvh": 8, "kb": 4, "vb": 2},
        # and read back to fp16 at 4 bits each
        {"name": "dequant-32k", "kind": "dequant", "tokens": 32768, "kvh": 8, "kb": 4, "vb": 4},
        # decode of a full serving batch with ragged contexts, default cache
        {"name": "tq-decode-b64", "kind": "tq_decode", "batch": 64, "lo": 1024, "hi": 32768,
         "qh": 32, "kvh": 8, "kb": 4, "vb": 2},
        # decode of a small batch in a protected layer (8-bit keys and values)
        {"name": "tq-decode-b8-k8v8", "kind": "tq_decode", "batch": 8, "lo": 1000, "hi": 8000,
         "qh": 32, "kvh": 8, "kb": 8, "vb": 8},
        # one interactive sequence: one token over a registered page pool
        {"name": "tq-pool-decode-4k", "kind": "tq_pool", "tokens": 1, "start": 4001, "qh": 32,
         "kvh": 8, "kb": 4, "vb": 2},
        # a prompt's causal prefill over its own TurboQuant pages
        {"name": "tq-pool-prefill-2k", "kind": "tq_pool", "tokens": 2048, "start": 0, "qh": 32,
         "kvh": 8, "kb": 4, "vb": 2},
        # decode of a medium batch over an FP16 cache
        {"name": "f16-decode-b16", "kind": "f16_decode", "batch": 16, "lo": 500, "hi": 8192,
         "qh": 32, "kvh": 8, "hd": 128},
        # a chunk of a chunked prefill over an FP16 cache, ragged sizes
        {"name": "f16-prefill-1000", "kind": "f16_prefill", "tokens": 1000, "start": 3001,
         "qh": 32, "kvh": 8, "hd": 128},
        # a whole decode step (two layers and the output head) of one sequence
        {"name": "step-b1", "kind": "step", "batch": 1, "ctx": 1000, "layers": 2,
         "vocab": 128256, "kb": 4, "vb": 2},
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["step_chain", "rows_chain", "sample", "compress", "dequant", "tq_decode",
                       "tq_decode", "tq_pool", "tq_pool", "f16_decode", "f16_prefill", "step"])
    heads = rng.choice([(32, 8), (32, 8), (16, 8), (8, 8), (32, 4)])
    bits = rng.choice([(4, 2), (4, 2), (4, 4), (3, 3), (2, 2), (8, 8)])
    if kind == "step_chain":
        return {"kind": kind, "tokens": _log_int(rng, 1, 256),
                "hidden": rng.choice([2048, 4096]), "ffn": rng.choice([5632, 14336])}
    if kind == "rows_chain":
        return {"kind": kind, "tokens": _log_int(rng, 256, 4096),
                "hidden": rng.choice([2048, 4096]), "ffn": rng.choice([5632, 14336]),
                "dtype": rng.choice(["fp16", "bf16", "fp32"])}
    if kind == "sample":
        return {"kind": kind, "rows": _log_int(rng, 1, 64), "vocab": _log_int(rng, 32000, 128256)}
    if kind in ("compress", "dequant"):
        return {"kind": kind, "tokens": _log_int(rng, 16, 32768),
                "kvh": rng.choice([2, 4, 8]), "kb": bits[0], "vb": bits[1]}
    if kind == "tq_decode":
        batch = _log_int(rng, 1, 64)
        most = 1 << 20 if bits[0] == 4 else 1 << 16  # positions of the batch
        hi = _log_int(rng, 128, min(32768, most // batch))
        return {"kind": kind, "batch": batch, "lo": max(1, hi // rng.choice([1, 4, 16])),
                "hi": hi, "qh": heads[0], "kvh": heads[1], "kb": bits[0], "vb": bits[1]}
    if kind == "tq_pool":
        tokens = 1 if rng.random() < 0.5 else _log_int(rng, 16, 1500)
        start = _log_int(rng, 16, 16384 if tokens == 1 else 2000)
        if bits[0] != 4:
            tokens = min(tokens, 256)
        return {"kind": kind, "tokens": tokens, "start": start, "qh": heads[0], "kvh": heads[1],
                "kb": bits[0], "vb": bits[1]}
    if kind == "f16_decode":
        batch = _log_int(rng, 1, 64)
        hi = _log_int(rng, 128, min(16384, (1 << 17) // batch))
        return {"kind": kind, "batch": batch, "lo": max(1, hi // rng.choice([1, 4, 16])),
                "hi": hi, "qh": heads[0], "kvh": heads[1], "hd": rng.choice([64, 128, 128])}
    if kind == "f16_prefill":
        return {"kind": kind, "tokens": _log_int(rng, 16, 1500), "start": _log_int(rng, 1, 2500) - 1,
                "qh": heads[0], "kvh": heads[1], "hd": rng.choice([64, 128, 128])}
    return {"kind": "step", "batch": _log_int(rng, 1, 8), "ctx": _log_int(rng, 16, 1500),
            "layers": 1, "vocab": _log_int(rng, 32000, 128256), "kb": bits[0], "vb": bits[1]}


# --- inputs ----------------------------------------------------------------------------
def _gen(seed):
    return torch.Generator(device="cuda").manual_seed(int(seed) + 1)


def _randn(g, *shape, dtype=torch.float16, scale=1.0):
    """Gaussian values; made in pieces, so that large tensors cost no fp32 copy of themselves."""
    out = torch.empty(shape, dtype=dtype, device="cuda")
    flat = out.view(-1)
    for i in range(0, flat.numel(), 1 << 26):
        n = min(1 << 26, flat.numel() - i)
        flat[i:i + n] = torch.randn(n, generator=g, device="cuda") * scale
    return out


def _randint(g, lo, hi, n, dtype=torch.int32):
    return torch.randint(lo, hi, (n,), generator=g, device="cuda").to(dtype)


@functools.lru_cache(maxsize=None)
def _tables(hd, bits, seed):
    """Rotation, centroids and boundaries of a TurboQuant layer, as host arrays."""
    c, b = tq.codebook(hd, bits)
    return tq.rotation_matrix(hd, seed), c, b


def _dev_tables(hd, bits, seed):
    rot, cent, bound = _tables(hd, bits, seed)
    return torch.from_numpy(rot).cuda(), torch.from_numpy(cent).cuda(), torch.from_numpy(bound).cuda()


def _pack(codes, bits):
    """codes u8 [..., hd] to the MSB-first bitstream u8 [..., hd * bits / 8]."""
    if bits == 8:
        return codes.contiguous()
    lead, hd = codes.shape[:-1], codes.shape[-1]
    if bits == 3:
        c = codes.view(*lead, hd // 8, 8).int()
        word = sum(c[..., i] << (21 - 3 * i) for i in range(8))
        return torch.stack([(word >> s) & 255 for s in (16, 8, 0)], -1).to(torch.uint8).view(*lead, -1)
    per = 8 // bits
    c = codes.view(*lead, hd // per, per)
    out = torch.zeros(*lead, hd // per, dtype=torch.uint8, device=codes.device)
    for i in range(per):
        out |= c[..., i] << (8 - bits * (i + 1))
    return out


def _codes(g, rows, hd, bits, bound):
    """Packed codes [rows, pd] of Gaussian coordinates and fp16 norms [rows]."""
    packed = torch.empty((rows, hd * bits // 8), dtype=torch.uint8, device="cuda")
    for i in range(0, rows, 1 << 19):
        n = min(1 << 19, rows - i)
        y = torch.randn((n, hd), generator=g, device="cuda") / math.sqrt(hd)
        packed[i:i + n] = _pack(torch.bucketize(y, bound).to(torch.uint8), bits)
    norms = (math.sqrt(hd) * torch.exp(0.2 * torch.randn(rows, generator=g, device="cuda"))).half()
    return packed, norms


def _lengths(g, case):
    return _randint(g, case["lo"], case["hi"] + 1, case["batch"])


def _block_table(g, lens):
    """[B, widest] physical pages in scattered order (-1 past a sequence's end), pages in all."""
    blocks = (lens + PAGE - 1) // PAGE
    total, widest = int(blocks.sum()), int(blocks.max())
    pages = torch.randperm(total, generator=g, device="cuda").int()
    table = torch.full((lens.numel(), widest), -1, dtype=torch.int32, device="cuda")
    table[torch.arange(widest, device="cuda")[None] < blocks[:, None]] = pages
    return table, total


def _inputs(case, seed):
    g, k = _gen(seed), case["kind"]
    s = {}
    if k in ("step_chain", "rows_chain"):
        T, H, F = case["tokens"], case["hidden"], case["ffn"]
        dt = DTYPES[case.get("dtype", "fp16")]
        s = {"table": _randn(g, 32000, H, dtype=dt), "ids": _randint(g, 0, 32000, T),
             "attn": _randn(g, T, H, dtype=dt), "mlp": _randn(g, T, H, dtype=dt),
             "w1": _randn(g, H, dtype=dt, scale=0.1) + 1, "w2": _randn(g, H, dtype=dt, scale=0.1) + 1,
             "gate": _randn(g, T, F, dtype=dt), "up": _randn(g, T, F, dtype=dt)}
    elif k == "sample":
        s = {"logits": _randn(g, case["rows"], case["vocab"], dtype=torch.float32, scale=3.0)}
    elif k == "compress":
        N, H = case["tokens"], case["kvh"]
        for n in "kv":
            s[n] = _randn(g, N, H, 128) * torch.exp(0.3 * torch.randn(128, generator=g, device="cuda")).half()
    elif k == "dequant":
        for n, bits in (("k", case["kb"]), ("v", case["vb"])):
            s[n] = _codes(g, case["tokens"] * case["kvh"], 128, bits, _dev_tables(128, bits, 1)[2])
    elif k in ("tq_decode", "f16_decode"):
        s["lens"] = _lengths(g, case)
        s["table"], pages = _block_table(g, s["lens"])
        hd = case.get("hd", 128)
        s["q"] = _randn(g, case["batch"], case["qh"], hd)
        for n in "kv":
            if k == "f16_decode":
                s[n] = _randn(g, pages, PAGE, case["kvh"], hd)
            else:
                bits = case[n + "b"]
                p, nn = _codes(g, pages * PAGE * case["kvh"], hd, bits, _dev_tables(hd, bits, 1)[2])
                s[n] = (p.view(pages, PAGE, -1), nn.view(pages, PAGE, -1))
    elif k in ("tq_pool", "f16_prefill"):
        n_pos = case["start"] + case["tokens"]
        s["table"], pages = _block_table(g, torch.tensor([n_pos], device="cuda"))
        s["table"] = s["table"].view(-1)
        hd = case.get("hd", 128)
        s["q"] = _randn(g, case["tokens"], case["qh"], hd)
        for n in "kv":
            if k == "f16_prefill":
                s[n] = _randn(g, pages, PAGE, case["kvh"], hd)
            else:
                bits = case[n + "b"]
                p, nn = _codes(g, pages * PAGE * case["kvh"], hd, bits, _dev_tables(hd, bits, 1)[2])
                s[n] = (p.view(pages, PAGE, -1), nn.view(pages, PAGE, -1))
    else:
        B, H, F, V, ctx = case["batch"], 4096, 14336, case["vocab"], case["ctx"]
        lens = torch.full((B,), ctx + 1, device="cuda")
        s["table"], pages = _block_table(g, lens)
        s["ids"] = _randint(g, 0, V, B)
        s["embed"] = _randn(g, V, H)  # the output head too (tied)
        s["norm"] = _randn(g, H, scale=0.1) + 1
        s["layers"] = []
        for _ in range(case["layers"]):
            w = {"n1": _randn(g, H, scale=0.1) + 1, "n2": _randn(g, H, scale=0.1) + 1}
            for n, o, i in (("q", H, H), ("k", 1024, H), ("v", 1024, H), ("o", H, H),
                            ("gate", F, H), ("up", F, H), ("down", H, F)):
                w[n] = _randn(g, o, i, scale=1 / math.sqrt(i))
            for n in "kv":
                bits = case[n + "b"]
                p, nn = _codes(g, pages * PAGE * 8, 128, bits, _dev_tables(128, bits, 1)[2])
                w[n + "pages"] = (p.view(pages, PAGE, -1), nn.view(pages, PAGE, -1))
            s["layers"].append(w)
    return s


# --- states ----------------------------------------------------------------------------
@functools.lru_cache(maxsize=None)
def _backend():
    b = HipBackend(0)
    b.precompute_rope_freqs(128, THETA)
    return b


class _Alias:
    """A backend tensor's memory as torch sees it; holds the tensor's owner."""

    def __init__(self, owner, ptr, shape, kind):
        self.owner = owner
        self.__cuda_array_interface__ = {"shape": tuple(shape), "typestr": kind, "data": (ptr, False),
                                         "version": 3, "strides": None}


class _Held:
    """Backend tensors, page pools and graphs of one state, given back with it."""

    def __init__(self):
        self.b, self.tensors, self.pools, self.graphs = _backend(), [], [], []

    def new(self, shape, dtype=DType.FP16):
        t = self.b.alloc(shape, dtype)
        self.tensors.append(t)
        return t

    def view(self, t):
        kind = {DType.FP16: "<f2", DType.FP32: "<f4", DType.INT8: "|u1"}[t.dtype]
        return torch.as_tensor(_Alias(self, self.b.get_ptr(t.id), t.shape, kind), device="cuda")

    def put(self, x, dtype=None):
        """A backend tensor holding torch tensor x."""
        t = self.new(x.shape, dtype or {torch.float16: DType.FP16, torch.float32: DType.FP32,
                                        torch.uint8: DType.INT8}[x.dtype])
        self.view(t).copy_(x)
        return t

    def pool(self, k, v):
        """A registered pool of per-block tensors, as a cache manager allocates them."""
        lists = [[self.new(part.shape[1:], DType.INT8 if part.dtype == torch.uint8 else DType.FP16)
                  for _ in range(part.shape[0])] for part in (*k, *v)]
        for part, tensors in zip((*k, *v), lists):
            rows = part.reshape(part.shape[0], -1).cpu().numpy().view(np.uint8)
            for t, row in zip(tensors, rows):
                self.b.copy_to_device(t, row)
        p = self.b.page_pool_create(*lists)
        self.pools.append(p)
        return p

    def __del__(self):
        for x in self.graphs:
            self.b.graph_destroy(x)
        for x in self.pools:
            self.b.page_pool_destroy(x)
        for t in self.tensors:
            self.b.free(t)


def _backend_tables(h, kb, vb):
    out = []
    for bits, seed in ((kb, 1), (vb, 2)):
        rot, cent, _ = _dev_tables(128, bits, seed)
        out.append((h.put(rot), h.put(cent)))
    return out[0][0], out[1][0], out[0][1], out[1][1]


def prepare(case, seed):
    s, k = _inputs(case, seed), case["kind"]
    s["case"] = case
    if k == "step_chain":
        h = s["h"] = _Held()
        T = case["tokens"]
        ids = h.new([T], DType.FP32)  # uint32 bytes
        h.b.copy_to_device(ids, s["ids"].cpu().numpy().view(np.uint32))
        t = {n: h.put(s[n]) for n in ("table", "attn", "mlp", "w1", "w2", "gate", "up")}
        x, n1, n2 = (h.new([T, case["hidden"]]) for _ in range(3))
        mid = h.new([T, case["ffn"]])

        def record():
            h.b.embedding_dev(ids, T, t["table"], x)
            h.b.add_rmsnorm(x, t["attn"], t["w1"], EPS, n1)
            h.b.silu_mul(t["gate"], t["up"], mid)
            h.b.add_rmsnorm(x, t["mlp"], t["w2"], EPS, n2)

        torch.cuda.synchronize()
        s["graph"] = h.b.capture(record)
        h.graphs.append(s["graph"])
        s["out"] = {"x": h.view(x), "n1": h.view(n1), "mid": h.view(mid), "n2": h.view(n2)}
    elif k == "rows_chain":
        s["out"] = {"x": torch.empty_like(s["attn"]), "n1": torch.empty_like(s["attn"]),
                    "mid": torch.empty_like(s["gate"]), "n2": torch.empty_like(s["attn"])}
    elif k == "sample":
        r, v = case["rows"], case["vocab"]
        s["out"] = {"probs": torch.empty_like(s["logits"]),
                    "index": torch.empty(r, dtype=torch.int32, device="cuda"),
                    "flags": torch.empty(r, dtype=torch.int32, device="cuda")}
        s["ws"] = K.rows_workspace(r, v)
    elif k in ("compress", "dequant"):
        N, H = case["tokens"], case["kvh"]
        s["plans"] = [K.TqPlan(*_dev_tables(128, bits, seed)[:2], bits)
                      for bits, seed in ((case["kb"], 1), (case["vb"], 2))]
        if k == "compress":
            s["out"] = [torch.empty(sh, dtype=dt, device="cuda") for bits in (case["kb"], case["vb"])
                        for sh, dt in (((N, H * 16 * bits), torch.uint8), ((N, H), torch.float16))]
        else:
            s["out"] = [torch.empty((N, H, 128), dtype=torch.float16, device="cuda") for _ in "kv"]
    elif k == "tq_decode":
        s["tables"] = [_dev_tables(128, bits, seed) for bits, seed in ((case["kb"], 1), (case["vb"], 2))]
        s["out"] = torch.empty_like(s["q"])
        s["ws"] = K.attention_workspace(case["batch"], case["qh"], 128, s["table"].shape[1])
    elif k == "f16_decode":
        s["out"] = torch.empty_like(s["q"])
        s["ws"] = K.attention_paged_workspace(case["batch"], case["qh"], case["hd"], s["table"].shape[1])
    elif k == "f16_prefill":
        s["out"] = torch.empty_like(s["q"])
        s["ws"] = K.attention_paged_workspace(case["tokens"], case["qh"], case["hd"], s["table"].numel())
        for n in "kv":
            s[n + "ptrs"] = (s[n].data_ptr() + s[n][0].nbytes
                             * torch.arange(s[n].shape[0], dtype=torch.int64, device="cuda"))
    elif k == "tq_pool":
        h = s["h"] = _Held()
        s["pool"] = h.pool(s["k"], s["v"])
        s["tables"] = _backend_tables(h, case["kb"], case["vb"])
        s["qt"] = h.put(s["q"])
        s["ot"] = h.new(s["q"].shape)
        s["out"] = h.view(s["ot"])
        s["blocks"] = s["table"].cpu().numpy()
    else:
        h = s["h"] = _Held()
        B, H, F = case["batch"], 4096, 14336
        s["blocks"] = s["table"].cpu().numpy()
        s["host_ids"] = s["ids"].cpu().numpy().view(np.uint32)
        s["lens"] = np.full(B, case["ctx"] + 1, np.uint32)
        s["tables"] = _backend_tables(h, case["kb"], case["vb"])
        s["w"] = {"embed": h.put(s.pop("embed")), "norm": h.put(s.pop("norm"))}
        s["l"] = []
        for w in s.pop("layers"):
            d = {"pool": h.pool(w.pop("kpages"), w.pop("vpages"))}
            while w:
                n, x = w.popitem()
                d[n] = h.put(x)
            s["l"].append(d)
        s["t"] = {n: h.new([B, d]) for n, d in (("x", H), ("n", H), ("q", H), ("k", 1024), ("v", 1024),
                                               ("a", H), ("p", H), ("gate", F), ("up", F), ("mid", F),
                                               ("logits", case["vocab"]))}
        # one sequence's row of the projections, for the cache writer's call per sequence
        s["row"] = {n: [h.new([1, 8, 128]) for _ in range(B)] for n in "kv"} if B > 1 else None
        s["out"] = h.view(s["t"]["logits"])
    torch.cuda.synchronize()
    return s


# --- passes ----------------------------------------------------------------------------
def _step(s):
    c, b, t, B = s["case"], s["h"].b, s["t"], s["case"]["batch"]
    kb, vb, ctx = c["kb"], c["vb"], c["ctx"]
    q3, a3 = t["q"].reshape([B, 32, 128]), t["a"].reshape([B, 32, 128])
    k3, v3 = t["k"].reshape([B, 8, 128]), t["v"].reshape([B, 8, 128])
    b.embedding(s["host_ids"], s["w"]["embed"], t["x"])
    b.rmsnorm(t["x"], s["l"][0]["n1"], EPS, t["n"])
    for i, w in enumerate(s["l"]):
        b.matmul(t["n"], w["q"], t["q"])
        b.matmul(t["n"], w["k"], t["k"])
        b.matmul(t["n"], w["v"], t["v"])
        b.rope(q3, k3, [ctx] * B, THETA, 128)
        if B == 1:
            b.tq_append_kv(w["pool"], k3, v3, *s["tables"], kb, vb, s["blocks"][0], ctx)
            b.attention_paged_tq_pool(q3, s["blocks"][0], w["pool"], *s["tables"], kb, vb, 8, ctx + 1,
                                      ctx, a3)
        else:
            for j in range(B):
                b.copy_rows(k3, s["row"]["k"][j], j, 0, 1)
                b.copy_rows(v3, s["row"]["v"][j], j, 0, 1)
                b.tq_append_kv(w["pool"], s["row"]["k"][j], s["row"]["v"][j], *s["tables"], kb, vb,
                               s["blocks"][j], ctx)
            b.attention_paged_tq_batched(q3, s["blocks"], s["lens"], w["pool"], *s["tables"], kb, vb,
                                         8, a3)
        b.matmul(t["a"], w["o"], t["p"])
        b.add_rmsnorm(t["x"], t["p"], w["n2"], EPS, t["n"])
        b.matmul(t["n"], w["gate"], t["gate"])
        b.matmul(t["n"], w["up"], t["up"])
        b.silu_mul(t["gate"], t["up"], t["mid"])
        b.matmul(t["mid"], w["down"], t["p"])
        nxt = s["l"][i + 1]["n1"] if i + 1 < len(s["l"]) else s["w"]["norm"]
        b.add_rmsnorm(t["x"], t["p"], nxt, EPS, t["n"])
    b.matmul(t["n"], s["w"]["embed"], t["logits"])


def run(s):
    case, k, out = s["case"], s["case"]["kind"], s["out"]
    if k == "step_chain":
        s["h"].b.graph_launch(s["graph"])
    elif k == "rows_chain":
        K.embedding(out["x"], s["table"], s["ids"])
        K.add_rmsnorm(out["x"], s["attn"], s["w1"], EPS, out["n1"])
        K.silu_mul(out["mid"], s["gate"], s["up"])
        K.add_rmsnorm(out["x"], s["mlp"], s["w2"], EPS, out["n2"])
    elif k == "sample":
        K.softmax_argmax_rows(s["logits"], out["probs"], out["index"], out["flags"], 0.8, s["ws"])
    elif k == "compress":
        K.tq_compress_kv_planned(*s["plans"], s["k"], s["v"], *out)
    elif k == "dequant":
        K.tq_dequant_kv_planned(*s["plans"], *s["k"], *s["v"], *out)
    elif k == "tq_decode":
        (kr, kc, _), (vr, vc, _) = s["tables"]
        K.attention_tq_decode(out, s["q"], s["table"], s["lens"], *s["k"], *s["v"], kr, vr, kc, vc,
                              case["kb"], case["vb"], case["kvh"], s["ws"])
    elif k == "f16_decode":
        K.attention_paged_decode(out, s["q"], s["table"], s["lens"], s["k"], s["v"], case["kvh"], s["ws"])
    elif k == "f16_prefill":
        K.paged_attention(out, s["q"], s["table"], s["kptrs"], s["vptrs"], case["kvh"],
                          case["start"] + case["tokens"], case["start"], s["ws"])
    elif k == "tq_pool":
        s["h"].b.attention_paged_tq_pool(s["qt"], s["blocks"], s["pool"], *s["tables"], case["kb"],
                                         case["vb"], case["kvh"], case["start"] + case["tokens"],
                                         case["start"], s["ot"])
    else:
        _step(s)
    return out


# --- what a pass cannot do without -------------------------------------------------------
def _attention_work(case, cached, scored, queries, row_bytes):
    """`cached` positions read once, `scored` (query, position) pairs."""
    hd = case.get("hd", 128)
    return {"bytes": cached * case["kvh"] * row_bytes + 4 * queries * case["qh"] * hd,
            "flops": 4.0 * scored * case["qh"] * hd}


def work(case):
    k = case["kind"]
    if k in ("step_chain", "rows_chain"):
        T, H, F = case["tokens"], case["hidden"], case["ffn"]
        e = 4 if case.get("dtype") == "fp32" else 2
        # the residual is read and written by the two norms, the embedding row read once
        return {"bytes": e * T * (6 * H + 3 * F), "flops": T * (12 * H + 5 * F)}
    if k == "sample":
        return {"bytes": 8 * case["rows"] * case["vocab"], "flops": 4 * case["rows"] * case["vocab"]}
    if k in ("compress", "dequant"):
        n = case["tokens"] * case["kvh"]
        return {"bytes": n * (2 * 258 + 16 * (case["kb"] + case["vb"])), "flops": 2.0 * n * 2 * 128 * 128}
    hd = case.get("hd", 128)
    if k in ("tq_decode", "f16_decode"):
        row = 4 * hd if k == "f16_decode" else 16 * (case["kb"] + case["vb"]) + 4
        n = case["batch"] * (case["lo"] + case["hi"]) / 2
        return _attention_work(case, n, n, case["batch"], row)
    if k in ("tq_pool", "f16_prefill"):
        row = 4 * hd if k == "f16_prefill" else 16 * (case["kb"] + case["vb"]) + 4
        T, st = case["tokens"], case["start"]
        return _attention_work(case, st + T, T * st + T * (T + 1) / 2, T, row)
    B, L, V, n = case["batch"], case["layers"], case["vocab"], case["batch"] * (case["ctx"] + 1)
    w = L * 4096 * (2 * 4096 + 2 * 1024 + 3 * 14336) + V * 4096
    return {"bytes": 2 * w + L * n * 8 * (16 * (case["kb"] + case["vb"]) + 4) + 2 * B * V,
            "flops": 2.0 * B * w + L * 4.0 * n * 32 * 128}


def tolerance(case):
    """About four times the distance from 64 bits that the kernels had when this was written."""
    k = case["kind"]
    if k == "sample":
        return {"rel": 4e-7, "max": 4e-6, "differ": 0.0}  # fp32 sums
    if k == "compress":
        # fp16 norms; a code whose coordinate lies within fp32 rounding of a threshold may differ
        return {"rel": 8e-4, "max": 2e-3, "differ": 1e-5}
    if k == "step":
        return {"rel": 3e-3, "max": 1.2e-2}  # fp16 roundings of every op in turn
    if k in ("step_chain", "rows_chain"):  # the second norm reads the rounded residual
        return {"fp16": {"rel": 1.4e-3, "max": 7e-3}, "bf16": {"rel": 1.1e-2, "max": 5e-2},
                "fp32": {"rel": 3e-7, "max": 1.5e-6}}[case.get("dtype", "fp16")]
    return {"rel": 8e-4, "max": 2e-3}  # fp16 outputs of fp32 sums


# --- the same in 64 bits -----------------------------------------------------------------
def _unpack(packed, bits, hd):
    p = packed.long()
    if bits == 8:
        return p
    if bits == 3:
        p = p.view(*p.shape[:-1], hd // 8, 3)
        word = (p[..., 0] << 16) | (p[..., 1] << 8) | p[..., 2]
        return torch.stack([(word >> (21 - 3 * i)) & 7 for i in range(8)], -1).flatten(-2)
    per = 8 // bits
    return torch.stack([(p >> (8 - bits * (i + 1))) & ((1 << bits) - 1) for i in range(per)],
                       -1).flatten(-2)


def _restore(packed, norms, bits, seed, hd=128):
    """Vectors [rows, hd] in fp64 of packed codes [rows, pd] and norms [rows]."""
    rot, cent, _ = _dev_tables(hd, bits, seed)
    return norms.double()[:, None] * (cent.double()[_unpack(packed, bits, hd)] @ rot.double())


def _attend(q, kk, vv, first):
    """Causal attention of q [T, qh, hd] over kk, vv [n, kvh, hd]; query i sees first + i + 1."""
    T, qh, hd = q.shape
    group = qh // kk.shape[1]
    mask = torch.arange(kk.shape[0], device="cuda")[None] > first + torch.arange(T, device="cuda")[:, None]
    out = torch.empty(q.shape, dtype=torch.float64, device="cuda")
    for h in range(qh):
        sc = q[:, h].double() @ kk[:, h // group].t().contiguous() / math.sqrt(hd)
        out[:, h] = sc.masked_fill_(mask, -math.inf).softmax(-1) @ vv[:, h // group].contiguous()
    return out


def _gathered(s, case, ids, n):
    """K and V rows [n, kvh, hd] in fp64 of one sequence's pages."""
    got, ids = [], ids[: (n + PAGE - 1) // PAGE].long()
    for name, seed in (("k", 1), ("v", 2)):
        if isinstance(s[name], tuple):
            bits = case[name + "b"]
            p, nn = (x[ids].reshape(-1, PAGE * case["kvh"]).reshape(-1) for x in s[name])
            x = _restore(p.view(-1, 16 * bits), nn, bits, seed).view(-1, case["kvh"], 128)
        else:
            x = s[name][ids].flatten(0, 1).double()
        got.append(x[:n])
    return got


def _rms(x, w):
    return x * torch.rsqrt((x * x).mean(-1, keepdim=True) + EPS) * w.double()


def _mm(a, w):
    return torch.cat([a @ w[i:i + 8192].double().t().contiguous() for i in range(0, w.shape[0], 8192)], -1)


def _quantized(x, bits, seed):
    """What x [rows, hd] is after a pass through the cache."""
    rot, cent, bound = _dev_tables(128, bits, seed)
    norm = x.norm(dim=-1, keepdim=True)
    code = torch.bucketize((x / norm) @ rot.double().t().contiguous(), bound.double())
    return norm * (cent.double()[code] @ rot.double())


def _exact_step(case, s):
    B, ctx = case["batch"], case["ctx"]
    x = s["embed"][s["ids"].long()].double()
    inv = THETA ** (-torch.arange(64, dtype=torch.float64, device="cuda") / 64)
    cos, sin = torch.cos(ctx * inv), torch.sin(ctx * inv)

    def rope(y):
        a, b = y[..., :64], y[..., 64:]
        return torch.cat([a * cos - b * sin, b * cos + a * sin], -1)

    for w in s["layers"]:
        n = _rms(x, w["n1"])
        q = rope(_mm(n, w["q"]).view(B, 32, 128))
        k = _quantized(rope(_mm(n, w["k"]).view(B, 8, 128)).reshape(-1, 128), case["kb"], 1).view(B, 8, 128)
        v = _quantized(_mm(n, w["v"]).view(-1, 128), case["vb"], 2).view(B, 8, 128)
        att = []
        for j in range(B):
            kk, vv = _gathered({"k": w["kpages"], "v": w["vpages"]}, {**case, "kvh": 8}, s["table"][j], ctx + 1)
            kk[ctx], vv[ctx] = k[j], v[j]
            att.append(_attend(q[j:j + 1], kk, vv, ctx))
        x = x + _mm(torch.cat(att).view(B, -1), w["o"])
        n = _rms(x, w["n2"])
        x = x + _mm(torch.nn.functional.silu(_mm(n, w["gate"])) * _mm(n, w["up"]), w["down"])
    return _mm(_rms(x, s["norm"]), s["embed"])


def exact(case, seed):
    s, k = _inputs(case, seed), case["kind"]
    if k in ("step_chain", "rows_chain"):
        x = s["table"][s["ids"].long()].double() + s["attn"].double()
        n1 = _rms(x, s["w1"])
        mid = torch.nn.functional.silu(s["gate"].double()) * s["up"].double()
        x = x + s["mlp"].double()
        return {"x": x, "n1": n1, "mid": mid, "n2": _rms(x, s["w2"])}
    if k == "sample":
        return {"probs": (s["logits"].double() / 0.8).softmax(-1), "index": None, "flags": None}
    if k == "compress":
        return [o for n in "kv" for o in (None, s[n].double().norm(dim=-1))]
    if k == "dequant":
        return [_restore(*s[n], case[n + "b"], seed).view(case["tokens"], -1, 128)
                for n, seed in (("k", 1), ("v", 2))]
    if k in ("tq_decode", "f16_decode"):
        return torch.cat([_attend(s["q"][j:j + 1], *_gathered(s, case, s["table"][j], int(n)), int(n) - 1)
                          for j, n in enumerate(s["lens"])])
    if k in ("tq_pool", "f16_prefill"):
        n = case["start"] + case["tokens"]
        return _attend(s["q"], *_gathered(s, case, s["table"], n), case["start"])
    return _exact_step(case, s)
