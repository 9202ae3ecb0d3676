"""Timing cases of the KV-cache path: what an inference server has this package do.

A serving step writes its new keys and values into the packed cache ("store"),
reads the cache back for its single-token decodes ("decode", "step"), for drafts
that it verifies a few tokens at a time ("verify") and for prompts and prompt
chunks ("prefill"), or does all of it in one call of the attention backend
("forward").  "codec" and "pages" are the codec by itself: rows packed and unpacked,
and the pages of a batch unpacked for an attention that reads plain K and V.

Shapes are those of bench.py and the tests: head_dim 128, blocks of 16 tokens, 1 to 8
kv heads (8: a whole layer, 1 or 2: a tensor-parallel rank's share), 1 to 8 query heads
per kv head, 3- and 4-bit codebooks, contexts of 1 to 32768 tokens.  Keys carry strong
channels, as keys do (a scale of 1 + |N(0, 3)| per head and channel); values and queries are
N(0, 1).  The physical blocks of a batch are in random order, as after some hours of serving.
"""
import math
import os
import sys
import types

import numpy as np
import torch

sys.path.insert(0, os.path.join(os.getcwd(), "rotorquant-vllm_amd"))

from rotorquant_vllm import kernels  # noqa: E402
from rotorquant_vllm.quantization import IsoQuantMSE, PlanarQuantMSE  # noqa: E402
from rotorquant_vllm.vllm.rq_backend import RQAttentionImpl, _build_rotation_matrix  # noqa: E402

D = 128       # head_dim
BS = 16       # tokens per block
DTYPES = {"float16": torch.float16, "bfloat16": torch.bfloat16}


def listed():
    common = {"mode": "iso", "k_bits": 3, "v_bits": 3, "dense": False, "dtype": "bfloat16", "heads": 8, "group": 4}
    return [
        # the K and V of one decode step of 16 sequences: the smallest write
        dict(common, name="store_step", kind="store", tokens=16, skipped=0),
        # the K and V of a full batch of prompts
        dict(common, name="store_prompts", kind="store", tokens=32768, skipped=0, dtype="float16"),
        # the codec on 2048 tokens' keys and back, as a user checks a codebook or moves a cache
        dict(common, name="codec", kind="codec", tokens=2048, dtype="float16"),
        # the pages of a small batch unpacked for an attention that takes plain K and V
        dict(common, name="pages", kind="pages", seqs=8, shortest=300, longest=4000),
        # one user's decode step: latency and launches
        dict(common, name="decode_one", kind="decode", seqs=1, shortest=777, longest=777),
        # a serving batch of decodes (32 query / 8 kv heads)
        dict(common, name="decode_batch", kind="decode", seqs=64, shortest=1024, longest=8192),
        # long contexts, 4-bit keys, 2x2 rotations
        dict(common, name="decode_long", kind="decode", seqs=64, shortest=2048, longest=32768, mode="planar", k_bits=4),
        # a decode step of a tensor-parallel rank (one kv head) through the backend, replayed as the HIP
        # graph that the server captures for it
        dict(common, name="step_rank", kind="step", heads=1, seqs=48, shortest=512, longest=8192),
        # drafts of up to 8 tokens verified over their contexts
        dict(common, name="verify", kind="verify", seqs=32, shortest=600, longest=8000, queries=8),
        # one prompt of ordinary length
        dict(common, name="prefill_one", kind="prefill", entry="int8", seqs=1, prefix=0, queries=700, k_bits=4, v_bits=4),
        # a full batch of prompts
        dict(common, name="prefill_batch", kind="prefill", entry="int8", seqs=8, prefix=0, queries=4096, k_bits=4, v_bits=4),
        # a continuous batch in one call of the backend (28 query / 4 kv heads): decodes, and prompt
        # chunks after their prefixes, with the new K and V written first
        dict(common, name="forward_mixed", kind="forward", fused=False, mode="iso_full", heads=4, group=7, seqs=40,
             shortest=512, longest=8192, chunks=3, prefix=5000, queries=1500),
    ]


def draw(rng):
    def log(lo, hi):
        return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))

    heads, group = rng.choice([(8, 4), (8, 4), (4, 7), (4, 8), (2, 4), (1, 4), (8, 1), (2, 7), (1, 8), (4, 2)])
    dense = rng.random() < 0.15
    c = {"mode": rng.choice(["iso", "iso", "iso_full", "planar"]), "k_bits": 3 if dense else rng.choice([3, 4]),
         "v_bits": 3 if dense else rng.choice([3, 4]), "dense": dense, "dtype": rng.choice(["bfloat16", "bfloat16", "float16"]),
         "heads": heads, "group": group}
    kind = rng.choice(["store", "store", "codec", "pages", "decode", "decode", "decode", "step", "verify", "verify",
                       "prefill", "prefill", "prefill", "forward"])
    c["kind"] = kind
    if kind == "store":
        c["tokens"] = log(1, 32768 * 8 // heads if heads > 2 else 65536)
        c["skipped"] = rng.choice([0, 0, c["tokens"] // 5])
    elif kind == "codec":
        c["tokens"] = log(1, 4096)
        c["dense"] = False
    elif kind in ("pages", "decode", "step", "verify"):
        longest = log(40, 4096 if kind == "pages" else 32768)
        c["longest"], c["shortest"] = longest, max(1, int(longest * rng.choice([0.1, 0.5, 0.9])))
        # tokens of context in the batch
        budget = {"pages": 24000, "decode": 400000, "step": 200000, "verify": 150000}[kind]
        c["seqs"] = max(1, min(log(1, 128), budget // longest))
        if kind == "verify":
            c["queries"] = rng.randint(2, 12)
            c["shortest"] = max(c["shortest"], 16)
    elif kind == "prefill":
        c["entry"] = rng.choice(["int8", "int8", "paged"])
        c["queries"] = log(20, 4096)
        c["prefix"] = rng.choice([0, 0, log(1, 16000)])
        # pairs of a query and a key: at most a quarter of the largest listed case's
        pairs = c["queries"] * (c["prefix"] + c["queries"] / 2) * heads * group
        c["seqs"] = max(1, min(rng.randint(1, 8), int(5.0e8 / pairs)))
    else:
        c.update(fused=rng.random() < 0.5, seqs=log(1, 64), shortest=100, longest=log(200, 8192), chunks=rng.randint(1, 3),
                 prefix=log(1, 6000), queries=log(30, 1500))
    return c


# ---------------------------------------------------------------------------
# Inputs
# ---------------------------------------------------------------------------

def _dev():
    return torch.device("cuda")


def _gen(seed, stream):
    return torch.Generator(device=_dev()).manual_seed(1000 * int(seed) + stream)


class _Codec:
    """Codebooks and rotation as the backend sets them up, on the GPU."""

    def __init__(self, case):
        mode = case["mode"]

        def quantizer(bits):
            if mode == "planar":
                return PlanarQuantMSE(D, bits, seed=42)
            return IsoQuantMSE(D, bits, seed=42, mode="full" if mode == "iso_full" else "fast")

        kq, vq = quantizer(case["k_bits"]), quantizer(case["v_bits"])
        R = _build_rotation_matrix(kq, D, "cpu")
        RT = R.T.contiguous()
        self.kc, self.kb, self.vc, self.vb, self.R, self.even, self.odd = (
            t.to(_dev(), torch.float32).contiguous()
            for t in (kq.centroids, kq.boundaries, vq.centroids, vq.boundaries, R, RT[:, 0::2], RT[:, 1::2]))
        self.block = 2 if mode == "planar" else 4


_codecs = {}


def _codec(case):
    key = (case["mode"], case["k_bits"], case["v_bits"])
    if key not in _codecs:
        _codecs[key] = _Codec(case)
    return _codecs[key]


def _channel_scale(case, seed):
    return 1 + (torch.randn(case["heads"], D, generator=_gen(seed, 2), device=_dev()) * 3).abs()


def _quantize(x, R, boundaries):
    """(index per dim, norm per row) of K or V rows, in plain torch."""
    x = x.float()
    norm = x.norm(dim=-1)
    return torch.bucketize((x / (norm[..., None] + 1e-10)) @ R.T, boundaries).to(torch.uint8), norm


def _pack(idx, dense):
    """Index bytes of rows of 128 indices: two per byte, or the dense 3-bit groups."""
    if not dense:
        return (idx[..., 0::2] << 4) | idx[..., 1::2]
    i = idx.view(*idx.shape[:-1], D // 32, 4, 4, 2)  # [group][A, B, C or the rest][byte][even, odd]
    lo, rest = i[..., :3, :, 0] | (i[..., :3, :, 1] << 3), i[..., 3, :, :]
    e, o = rest[..., 0], rest[..., 1]
    top = torch.stack([(e & 3) << 6, (o & 3) << 6, ((e >> 2) << 6) | ((o >> 2) << 7)], dim=-2)
    return (lo | top).reshape(*idx.shape[:-1], D * 3 // 8)


def _slot_bytes(case):
    return case["heads"] * (128 if case["dense"] else 256)


def _layout(lens, seed, spare=7):
    """Random physical blocks for sequences of these lengths: (block table, number of blocks, slots of each sequence)."""
    rng = np.random.RandomState(1000 * int(seed) % (1 << 31) + 5)
    need = [-(-n // BS) for n in lens]
    blocks = sum(need) + spare
    order = rng.permutation(blocks).astype(np.int32)
    table, slots, at = np.zeros((len(lens), max(need)), np.int32), [], 0
    for b, n in enumerate(lens):
        table[b, :need[b]] = order[at:at + need[b]]
        at += need[b]
        pos = np.arange(n)
        slots.append(table[b, pos // BS].astype(np.int64) * BS + pos % BS)
    return table, blocks, slots


def _fill(case, slots, blocks, seed, want=False):
    """A cache whose given slots hold quantized K and V; want: also (K, V) as the cache gives them, in 64 bits
    and rotated space, by slot."""
    p, H, dev = _codec(case), case["heads"], _dev()
    dtype = DTYPES[case["dtype"]]
    cache = torch.zeros(blocks * BS, _slot_bytes(case), dtype=torch.uint8, device=dev)
    plain = [torch.zeros(blocks * BS, H, D, dtype=dtype, device=dev) for _ in range(2)] if want else None
    scale, gk, gv = _channel_scale(case, seed), _gen(seed, 0), _gen(seed, 1)
    slots = torch.from_numpy(slots).to(dev)
    for s in range(0, slots.numel(), 16384):
        at = slots[s:s + 16384]
        parts = []
        for j, (g, c, b) in enumerate(((gk, p.kc, p.kb), (gv, p.vc, p.vb))):
            x = torch.randn(at.numel(), H, D, generator=g, device=dev)
            idx, norm = _quantize((x * scale if j == 0 else x).to(dtype), p.R, b)
            parts += [_pack(idx, case["dense"]).flatten(1), norm.contiguous().view(torch.uint8).flatten(1)]
            if want:
                plain[j][at] = (c[idx.long()] * norm[..., None]).to(dtype)
        row = torch.cat(parts, dim=1)
        cache[at, :row.shape[1]] = row
    return cache.view(blocks, BS, -1), plain


def _lens(case):
    rng = np.random.RandomState(4)  # lengths are part of the case: they do not change with its data
    lens = rng.randint(case["shortest"], case["longest"] + 1, case["seqs"])
    lens[0] = case["longest"]
    return [int(n) for n in lens]


def _batch(case):
    """(context lengths, query lengths) of the batch's sequences, decodes first."""
    kind = case["kind"]
    if kind in ("decode", "step", "pages"):
        lens = _lens(case)
        return lens, [1] * len(lens)
    rng = np.random.RandomState(8)
    if kind == "verify":
        lens = _lens(case)
        queries = rng.randint(1, case["queries"] + 1, len(lens))
        queries[-1] = case["queries"]
        return lens, [int(n) for n in queries]
    chunks = case["seqs"] if kind == "prefill" else case["chunks"]
    # chunks are mostly of the full size; every other one ends earlier, and prefixes differ
    queries = [case["queries"] if j % 2 == 0 else int(rng.randint(max(1, case["queries"] // 2), case["queries"] + 1)) for j in range(chunks)]
    if kind == "prefill" and case["prefix"] == 0:
        queries = [case["queries"]] * chunks
    prefix = [case["prefix"] if j == 0 else int(rng.randint(case["prefix"] // 2, case["prefix"] + 1)) for j in range(chunks)]
    lens = [a + b for a, b in zip(prefix, queries)]
    if kind == "forward":
        decodes = _lens(case)
        return decodes + lens, [1] * len(decodes) + queries
    return lens, queries


def _i32(values):
    return torch.tensor(np.asarray(values), dtype=torch.int32, device=_dev())


def _attention_state(case, seed, want=False):
    lens, queries = _batch(case)
    table, blocks, slots = _layout(lens, seed)
    cache, plain = _fill(case, np.concatenate(slots), blocks, seed, want)
    HQ = case["heads"] * case["group"]
    q = torch.randn(sum(queries), HQ, D, generator=_gen(seed, 6), device=_dev()).to(DTYPES[case["dtype"]])
    return {"case": case, "codec": _codec(case), "lens": lens, "queries": queries, "slots": slots, "cache": cache, "plain": plain, "q": q,
            "table": _i32(table), "seq_lens": _i32(lens), "starts": _i32(np.concatenate([[0], np.cumsum(queries)])), "out": torch.zeros_like(q)}


def _new_kv(case, n, seed):
    scale = _channel_scale(case, seed)
    k, v = (torch.randn(n, case["heads"], D, generator=_gen(seed, j), device=_dev()) for j in (10, 11))
    return (k * scale).to(DTYPES[case["dtype"]]), v.to(DTYPES[case["dtype"]])


def _impl(case, fused):
    """The backend's attention layer, as the server sets it up from the environment."""
    env = {"RQ_MODE": "planar" if case["mode"] == "planar" else "iso", "RQ_ISO_MODE": "full" if case["mode"] == "iso_full" else "fast",
           "RQ_BITS": str(case["k_bits"]), "RQ_K_BITS": str(case["k_bits"]), "RQ_V_BITS": str(case["v_bits"]),
           "RQ_DENSE_3BIT": "1" if case["dense"] else "", "RQ_USE_FUSED_PAGED": "1" if fused else ""}
    before = {k: os.environ.get(k) for k in env}
    os.environ.update(env)
    try:
        return RQAttentionImpl(case["heads"] * case["group"], D, 1.0 / math.sqrt(D), num_kv_heads=case["heads"])
    finally:
        for k, v in before.items():
            if v is None:
                os.environ.pop(k, None)
            else:
                os.environ[k] = v


def prepare(case, seed):
    kind, p = case["kind"], _codec(case)
    if kind == "store":
        n = case["tokens"]
        k, v = _new_kv(case, n, seed)
        blocks = -(-n // BS) + 7
        rng = np.random.RandomState((1000 * int(seed) + 5) % (1 << 31))
        slots = rng.permutation(blocks)[:-(-n // BS)].repeat(BS)[:n] * BS + np.arange(n) % BS
        if case["skipped"]:
            slots[n - case["skipped"]:] = -1  # the padding of a captured batch
        cache = torch.zeros(blocks, BS, _slot_bytes(case), dtype=torch.uint8, device=_dev())
        return {"case": case, "codec": p, "k": k, "v": v, "slots": torch.from_numpy(slots.astype(np.int64)).to(_dev()), "cache": cache}
    if kind == "codec":
        return {"case": case, "codec": p, "k": _new_kv(case, case["tokens"], seed)[0]}
    s = _attention_state(case, seed)
    if kind == "pages":
        used = sum(-(-n // BS) for n in s["lens"])
        s["out"] = [torch.empty(used, BS, case["heads"], D, dtype=DTYPES[case["dtype"]], device=_dev()) for _ in range(2)]
        s["workspace"] = torch.empty(8 * s["cache"].shape[0] + 4096, dtype=torch.uint8, device=_dev())
    if kind in ("step", "forward"):
        fused = kind == "step" or case["fused"]
        s["k"], s["v"] = _new_kv(case, s["q"].shape[0], seed)
        new = np.concatenate([sl[len(sl) - n:] for sl, n in zip(s["slots"], s["queries"])])
        s["meta"] = types.SimpleNamespace(
            num_actual_tokens=s["q"].shape[0], max_query_len=max(s["queries"]), max_seq_len=max(s["lens"]), use_cascade=False,
            slot_mapping=torch.from_numpy(new).to(_dev()), block_table=s["table"], seq_lens=s["seq_lens"], query_start_loc=s["starts"],
            rq_query_start_loc_cpu=s["starts"].cpu(), rq_seq_lens_cpu=s["seq_lens"].cpu())
        s["impl"] = _impl(case, fused)
    if kind == "step":
        side, graph = torch.cuda.Stream(), torch.cuda.CUDAGraph()
        side.wait_stream(torch.cuda.current_stream())
        with torch.cuda.stream(side):
            _forward(s)
            with torch.cuda.graph(graph, stream=side):
                _forward(s)
        torch.cuda.current_stream().wait_stream(side)
        s["graph"] = graph
    return s


def _forward(s):
    return s["impl"].forward(None, s["q"], s["k"], s["v"], s["cache"], s["meta"], output=s["out"])


def run(s):
    case, p = s["case"], s["codec"]
    kind, H = case["kind"], case["heads"]
    if kind == "store":
        kernels.compress_store(s["k"], s["v"], s["cache"], s["slots"], p.even, p.odd, p.kb, p.vb, rot_block=p.block, dense3=case["dense"])
        return s["cache"]
    if kind == "codec":
        planar = case["mode"] == "planar"
        packed, norms = (kernels.planar_compress if planar else kernels.iso_compress)(s["k"], p.even, p.odd, p.kb)
        back = (kernels.planar_decompress if planar else kernels.iso_decompress)(packed, norms, p.kc, s["k"].dtype)
        return {"packed": packed, "norms": norms, "back": back}
    if kind == "pages":
        k, v, table, count = kernels.paged_decompress(s["cache"], s["table"], s["seq_lens"], H, D, p.kc, p.vc, s["q"].dtype, out_k=s["out"][0],
                                                      out_v=s["out"][1], workspace=s["workspace"], dense3=case["dense"])
        return {"k": k, "v": v, "table": table, "count": count}
    if kind == "decode":
        return kernels.fused_paged_rq_decode(s["q"], s["cache"], s["table"], s["seq_lens"], p.kc, p.vc, p.R, H, D, BS, out=s["out"],
                                             dense3=case["dense"])
    if kind == "step":
        s["graph"].replay()
        return {"out": s["out"], "cache": s["cache"]}
    if kind == "forward":
        return {"out": _forward(s), "cache": s["cache"]}
    longest, most = max(s["lens"]), max(s["queries"])
    if kind == "verify":
        return kernels.paged_attention(s["q"], s["cache"], s["table"], s["seq_lens"], s["starts"], most, p.kc, p.vc, p.R, H, D, BS,
                                       out=s["out"], dense3=case["dense"])
    if case["entry"] == "int8":
        return kernels.fused_paged_rq_int8_prefill(s["q"], s["cache"], s["table"], s["seq_lens"], p.kc, p.vc, p.R, H, D, BS, out=s["out"],
                                                   cu_seqlens_q=s["starts"], max_q_len=most, max_seq_len=longest, dense3=case["dense"])
    return kernels.paged_prefill(s["q"], s["cache"], s["table"], s["seq_lens"], s["starts"], most, p.kc, p.vc, p.R, H, D, BS, out=s["out"],
                                 max_seq_len=longest, dense3=case["dense"])


# ---------------------------------------------------------------------------
# Work, tolerance, 64-bit results
# ---------------------------------------------------------------------------

def work(case):
    """Bytes: inputs once (the packed K and V of every context token, with its share of the block table) and outputs
    once; operations: two per product of Q K^T and P V, and for the codec about 20 per value."""
    H, HQ = case["heads"], case["heads"] * case["group"]
    payload = H * 2 * ((D * 3 // 8 if case["dense"] else D // 2) + 4)
    if case["kind"] == "store":
        n = case["tokens"]
        return {"bytes": n * (2 * H * D * 2 + 8) + (n - case["skipped"]) * _slot_bytes(case), "flops": n * 2 * H * D * 20}
    if case["kind"] == "codec":
        n = case["tokens"] * H
        return {"bytes": n * (D * 2 + D // 2 + 4) * 2, "flops": n * D * 21}
    lens, queries = _batch(case)
    tokens = sum(lens)
    blocks = sum(-(-n // BS) for n in lens)
    if case["kind"] == "pages":
        return {"bytes": tokens * payload + blocks * (BS * 2 * H * D * 2 + 8), "flops": tokens * 2 * H * D}
    pairs = sum(n * L - n * (n - 1) // 2 for n, L in zip(queries, lens))
    total = {"bytes": tokens * payload + blocks * 4 + sum(queries) * HQ * D * 4, "flops": pairs * HQ * D * 4}
    if case["kind"] in ("step", "forward"):  # the new K and V, and their slots written
        total["bytes"] += sum(queries) * (2 * H * D * 2 + 8 + _slot_bytes(case) - payload)
        total["flops"] += sum(queries) * 2 * H * D * 20
    return total


def tolerance(case):
    """The codec is exact by contract.  Attention outputs are rounded to the q dtype twice, before and after the rotation
    back, so two correct results differ by about a unit in the last place of the largest value of a rotation block (two
    implementations on a batch of prompts: 1.1e-3, and 0.03 at most)."""
    if case["kind"] in ("store", "codec", "pages"):
        return "exact"
    return {"rel": 0.005, "max": 0.12} if case["dtype"] == "bfloat16" else {"rel": 0.0025, "max": 0.03}


def exact(case, seed):
    kind, p = case["kind"], _codec(case)
    if kind == "store":
        return None
    if kind == "codec":
        x = _new_kv(case, case["tokens"], seed)[0].double()
        norm = x.norm(dim=-1, keepdim=True)
        idx = torch.bucketize((x / (norm + 1e-10)) @ p.R.double().T, p.kb.double())
        return {"packed": None, "norms": norm, "back": p.kc.double()[idx] * norm}
    s = _attention_state(case, seed, want=True)
    if kind == "pages":
        order = torch.unique(torch.cat([s["table"][b, :-(-n // BS)] for b, n in enumerate(s["lens"])])).long()
        k, v = (x.double().view(-1, BS, case["heads"], D)[order] for x in s["plain"])
        return {"k": k, "v": v, "table": None, "count": None}
    if kind in ("step", "forward"):  # the new tokens' K and V replace what their slots held
        new = torch.from_numpy(np.concatenate([sl[len(sl) - n:] for sl, n in zip(s["slots"], s["queries"])])).to(_dev())
        for x, plain, c, b in zip(_new_kv(case, s["q"].shape[0], seed), s["plain"], (p.kc, p.vc), (p.kb, p.vb)):
            idx, norm = _quantize(x, p.R, b)
            plain[new] = (c[idx.long()] * norm[..., None]).to(plain.dtype)
    G, R = case["group"], p.R.double()
    out, at = torch.zeros(s["q"].shape, dtype=torch.float64, device=_dev()), 0
    for sl, n in zip(s["slots"], s["queries"]):
        slots = torch.from_numpy(sl).to(_dev())
        q = s["q"][at:at + n].double() @ R.T
        hidden = torch.arange(len(sl), device=_dev())[None, :] > len(sl) - n + torch.arange(n, device=_dev())[:, None]
        for h in range(case["heads"]):
            k, v = (x[slots, h].double() for x in s["plain"])
            for j in range(h * G, h * G + G):
                w = (q[:, j].contiguous() @ k.T.contiguous() / math.sqrt(D)).masked_fill_(hidden, -math.inf).softmax(dim=-1)
                out[at:at + n, j] = w @ v @ R
        at += n
    return {"out": out, "cache": None} if kind in ("step", "forward") else out
