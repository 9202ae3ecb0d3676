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
        call(entry, seqs, H, HQ, 8, 200, longest, max_seq_len=1200)
    assert K.shared_workspace("cpu", "prefill", 0) is buf and not K._ws_retired
    assert {x.name for x in launches} == {"rq_short_attention"}
    assert max(x.scratch for x in launches) > buf.numel(), "some batch needs more than the buffer"
