"""Launches and scratch of the calls with a few query tokens per sequence, on the CPU.

The op wrappers (rotorquant_vllm.kernels) run with CPU tensors and a stand-in for the
library that answers the size queries with the real functions and records the launches
instead of making them.
"""
from types import SimpleNamespace

import pytest
import torch

from rotorquant_vllm import _lib
from rotorquant_vllm import kernels as K

D, BS = 128, 16


@pytest.fixture
def launches(monkeypatch):
    """The launches of the calls made so far: (function, scratch bytes or None, max_seq_len or None)."""
    real, seen = _lib.load(), []

    def record(name):
        def launch(*args):
            if name == "rq_paged_attention":
                seen.append(SimpleNamespace(name=name, scratch=None, max_seq_len=None))
            else:
                seen.append(SimpleNamespace(name=name, scratch=args[-2], max_seq_len=args[21 if name == "rq_int8_prefill" else 22]))
            return 0
        return launch

    lib = {n: getattr(real, n) for n in _lib.EXPORTED if n.endswith("_bytes") or n.endswith("_launches")}
    lib.update({n: record(n) for n in ("rq_paged_attention", "rq_short_attention", "rq_int8_prefill", "rq_paged_prefill")})
    monkeypatch.setattr(_lib, "load", lambda: SimpleNamespace(**lib))
    monkeypatch.setattr(_lib, "stream_ptr", lambda device: 0)
    monkeypatch.setattr(K, "_require_device", lambda *t: torch.device("cpu"))
    monkeypatch.setattr(K, "_ws_cache", {})
    monkeypatch.setattr(K, "_ws_retired", [])
    return seen


def call(entry, seqs, H, HQ, max_q_len, keys, table_keys=None, **kw):
    """One call of an entry point: seqs sequences of max_q_len tokens and up to `keys` keys."""
    q = torch.zeros(seqs * max_q_len, HQ, D, dtype=torch.bfloat16)
    cache = torch.zeros(4, BS, 256 * H, dtype=torch.uint8)
    bt = torch.zeros(seqs, -(-(table_keys or keys) // BS), dtype=torch.int32)
    lens = torch.full((seqs,), keys, dtype=torch.int32)
    cu = torch.arange(0, seqs * max_q_len + 1, max_q_len, dtype=torch.int32)
    c, R = torch.linspace(-1, 1, 8), torch.eye(D)
    if entry == "fused_paged_rq_int8_prefill":
        return K.fused_paged_rq_int8_prefill(q, cache, bt, lens, c, c, R, H, D, BS, cu_seqlens_q=cu, max_q_len=max_q_len, **kw)
    return getattr(K, entry)(q, cache, bt, lens, cu, max_q_len, c, c, R, H, D, BS, **kw)


PREFILLS = ["fused_paged_rq_int8_prefill", "paged_prefill"]


@pytest.mark.parametrize("entry", PREFILLS)
def test_drafts_do_not_grow_the_shared_prefill_buffer(launches, entry):
    """A server reserves the shared prefill buffer once, for the tile images of one longest sequence and the partials
    of key chunks.  Batches of drafts of every size up to 128 sequences then leave it as it is: what they need
    beyond it is scratch of the call, which the allocator gets back."""
    H, HQ, longest = 8, 32, 4096
    L = _lib.load()
    buf = K.shared_workspace("cpu", "prefill", L.rq_int8_prefill_workspace_bytes(1, H, longest) + K.PREFILL_SPLIT_BYTES)
    for seqs in range(1, 129, 9):
        call(entry, seqs, H, HQ, 8, 200, longest, max_seq_len=3000)
    assert K.shared_workspace("cpu", "prefill", 0) is buf and not K._ws_retired
    assert {x.name for x in launches} == {"rq_short_attention"}
    assert max(x.scratch for x in launches) > buf.numel(), "some batch needs more than the buffer"


# (sequences, kv heads, query heads, tokens, keys) -> kernels of paged_attention and of the prefill wrappers; both sides measured
# (us, one launch / short / prefill kernels) at the points of the sweep that the estimates were fitted to.
ROUTES = [
    ((4, 8, 32, 8, 64), "rq_paged_attention", "rq_paged_attention"),      # 9 / 18 / 13
    ((4, 8, 32, 8, 512), "rq_short_attention", "rq_short_attention"),     # 33 / 23 / 24
    ((16, 8, 32, 8, 256), "rq_paged_attention", "rq_paged_attention"),    # 19 / 33 / 25
    ((64, 8, 32, 8, 64), "rq_paged_attention", "rq_paged_attention"),     # 12 / 45 / 20
    ((64, 8, 32, 8, 512), "rq_paged_attention", "rq_paged_attention"),    # 44 / 61 / 58
    ((64, 8, 32, 2, 512), "rq_short_attention", "rq_short_attention"),    # 44 / 33 / 59
    ((128, 8, 32, 8, 256), "rq_paged_attention", "rq_paged_attention"),   # 49 / 81 / 70
    ((128, 8, 8, 4, 128), "rq_short_attention", "rq_short_attention"),    # 31 / 24 / 44
    ((64, 4, 28, 4, 64), "rq_paged_attention", "rq_paged_attention"),     # 10 / 28 / 24
    ((4, 8, 32, 16, 512), "rq_short_attention", "prefill"),               # 33 / 32 / 24
    ((32, 8, 32, 8, 8000), "rq_short_attention", "rq_short_attention"),   # 431 / 83
    ((1, 8, 32, 16, 100000), "rq_short_attention", "rq_short_attention"),
    ((1, 1, 1, 1, 1), "rq_paged_attention", "rq_paged_attention"),
]


@pytest.mark.parametrize("shape,attention,prefill", ROUTES)
def test_short_queries_take_the_faster_kernels(launches, shape, attention, prefill):
    """By sequences, heads, tokens and the bound on the lengths: the block table's capacity, or max_seq_len where it is
    given, whatever the table's width."""
    keys = shape[-1]
    own = {"fused_paged_rq_int8_prefill": "rq_int8_prefill", "paged_prefill": "rq_paged_prefill"}
    call("paged_attention", *shape)
    call("paged_attention", *shape, table_keys=131072, max_seq_len=keys)
    assert [x.name for x in launches] == [attention] * 2
    for entry in PREFILLS:
        launches.clear()
        call(entry, *shape)
        call(entry, *shape, table_keys=131072, max_seq_len=keys)
        assert [x.name for x in launches] == [own[entry] if prefill == "prefill" else prefill] * 2
    for x in launches:
        assert x.max_seq_len is None or keys <= x.max_seq_len < keys + 2 * BS


@pytest.mark.parametrize("entry", ["paged_attention"] + PREFILLS)
def test_calls_outside_the_short_kernels_keep_their_own(launches, entry):
    """Longer queries, more groups of columns than the kernels take, no sequences."""
    own = {"paged_attention": "rq_paged_attention", "fused_paged_rq_int8_prefill": "rq_int8_prefill", "paged_prefill": "rq_paged_prefill"}[entry]
    for shape in ((4, 8, 32, 17, 4000), (4, 1, 9, 5, 4000), (4, 8, 64, 9, 4000), (0, 8, 32, 4, 4000)):
        call(entry, *shape)
    assert [x.name for x in launches] == [own] * 4


@pytest.mark.parametrize("entry", ["paged_attention"] + PREFILLS)
def test_scratch_of_short_calls_over_the_limit(launches, monkeypatch, entry):
    """Calls that need more scratch than the limit keep kernels that need none or less."""
    own = {"paged_attention": "rq_paged_attention", "fused_paged_rq_int8_prefill": "rq_int8_prefill", "paged_prefill": "rq_paged_prefill"}[entry]
    need = _lib.load().rq_short_attention_workspace_bytes(4, 32, 8, 8, 4000)
    for limit, name in ((need, "rq_short_attention"), (need - 1, own)):
        monkeypatch.setattr(K, "_SHORT_WORKSPACE_LIMIT", limit)
        call(entry, 4, 8, 32, 8, 4000)
        assert launches[-1].name == name


def test_scratch_of_short_calls_given_by_the_caller(launches):
    """paged_attention on the caller's scratch: large enough it is what the kernels get, else the one launch runs."""
    need = _lib.load().rq_short_attention_workspace_bytes(4, 32, 8, 8, 4000)
    for given, name, scratch in ((need, "rq_short_attention", need), (need + 64, "rq_short_attention", need + 64),
                                 (need - 1, "rq_paged_attention", None), (0, "rq_paged_attention", None)):
        call("paged_attention", 4, 8, 32, 8, 4000, workspace=torch.empty(given, dtype=torch.uint8))
        assert (launches[-1].name, launches[-1].scratch) == (name, scratch)


def test_scratch_of_short_calls_is_what_they_write():
    """32 sequences of 8 tokens at 32 / 8 heads: 64 groups of 128 columns.  Query operands are 4 KB per group and kv head
    (2 MB), beside the partials (520 bytes per column and slot, at most 4 slots per CU and one per group) and the
    descriptors (272 bytes per 32 keys and group)."""
    need = _lib.load().rq_short_attention_workspace_bytes(32, 32, 8, 8, 8000)
    parts = [64 * 8 * 4096, (4 * 256 + 64) * 128 * 520, 64 * 250 * 272]
    assert sum(parts) <= need <= sum(parts) + 16384


@pytest.mark.parametrize("host_copies", [True, False])
def test_backend_bounds_short_calls_by_the_host_lengths(monkeypatch, host_copies):
    """The non-fused path gives paged_attention the longest context of its sequences where the metadata holds it on the
    host: all sequences of a batch of short queries, or the short ones of a mixed batch."""
    from rotorquant_vllm.vllm import rq_backend as B
    from test_dispatch import _bare_impl, _mixed_metadata
    seen = []

    def attention(q, kv_cache, block_table, seq_lens, cu, max_q_len, *a, out=None, max_seq_len=None, **k):
        seen.append((seq_lens.tolist(), max_seq_len))
        return out

    monkeypatch.setattr(B, "_paged_attention_fn", attention)
    monkeypatch.setattr(B, "_paged_prefill_fn", lambda *a, out=None, **k: out)
    monkeypatch.setattr(B, "_unfused_decode_fn", lambda *a, out=None, **k: out)
    monkeypatch.setattr(K, "_ws_cache", {})
    impl, cache = _bare_impl(False, False), torch.zeros(40, 16, 2048, dtype=torch.uint8)
    for q_lens, lens in (([2, 1, 16], [500, 30, 900]), ([1, 3, 40], [500, 30, 300])):
        md = _mixed_metadata(q_lens, lens, host_copies=host_copies)
        query = torch.zeros(sum(q_lens), 32, 128, dtype=torch.bfloat16)
        impl.forward(None, query, None, None, cache, md, output=torch.zeros_like(query))
    assert seen == [([500, 30, 900], 900 if host_copies else None), ([30], 30)]
