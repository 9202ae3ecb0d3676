"""GPU parity of the kernels that take a few query tokens per sequence, each by itself: rq_short_attention (the decode
kernels' column groups) and the one-launch rq_paged_attention over many tiles, called through the C ABI so that the
op wrappers' choice between them does not matter.  Oracle and tolerance as in test_gpu_attention.py.
"""
import numpy as np
import pytest
import torch

from rq_testlib import Params
from test_gpu_attention import _dev, attn_case

pytestmark = pytest.mark.gpu


def run(fn, case, causal=True, dense3=False, q=None, out=None):
    """rq_short_attention or rq_paged_attention on a case; q, out: device tensors to use instead of plain ones."""
    from rotorquant_vllm import _lib
    L, p = _lib.load(), case["p"]
    q = _dev(case["q"]) if q is None else q
    out = torch.full_like(q, float("nan")) if out is None else out
    cache, bt, lens, cu = (_dev(case[k]) for k in ("cache", "bt", "lens", "cu"))
    kc, vc, R = (_dev(x.float().contiguous()) for x in (p.kc, p.vc, p.R))
    n, longest, cap = len(case["q_lens"]), max(case["q_lens"]), bt.shape[1] * case["BS"]
    head = (q.data_ptr(), _lib.dtype_code(q.dtype), q.shape[0], case["HQ"], q.stride(0), q.stride(1), cu.data_ptr(), n, longest,
            int(causal), cache.data_ptr(), cache.shape[0], case["BS"], cache.stride(0), cache.stride(1), case["H"], 128, int(dense3),
            bt.data_ptr(), bt.shape[1], bt.stride(0), lens.data_ptr())
    tail = (kc.data_ptr(), kc.numel(), vc.data_ptr(), vc.numel(), R.data_ptr(), p.blk, 128 ** -0.5, out.data_ptr(), out.stride(0),
            out.stride(1))
    stream = _lib.stream_ptr(q.device)
    if fn == "rq_paged_attention":
        _lib.check(L.rq_paged_attention(*head, *tail, stream), fn)
    else:
        need = L.rq_short_attention_workspace_bytes(n, case["HQ"], case["H"], longest, cap)
        assert need > 0, "the shape is one that the call takes"
        ws = torch.empty(need, dtype=torch.uint8, device=q.device)
        _lib.check(L.rq_short_attention(*head, cap, *tail, ws.data_ptr(), need, stream), fn)
    torch.cuda.synchronize()
    return out.float().cpu().numpy()


@pytest.mark.parametrize("H,HQ,longest", [(1, 4, 16), (2, 2, 8)])
@pytest.mark.parametrize("fn", ["rq_short_attention", "rq_paged_attention"])
def test_weights_cancel_where_values_agree(fn, H, HQ, longest):
    """Every key of a sequence holds the same V: whatever the weights, the output is that V.  One key's norm is larger than the
    others', so that most of a row's weight shares one rounding to fp16, of up to 2^-11: divided by the sum of unrounded
    weights, outputs would leave V by an fp16 ulp.  A sequence of one key (weight 1) gives the expected bits."""
    p = Params("iso", 3, 3)
    case = attn_case(88, [longest, longest], [32, 1], H, HQ, p, dtype=torch.float16)
    cache, blocks, other = case["cache"], case["bt"][0][:2], case["bt"][1][0]
    slot = cache[blocks[0], 0].copy()
    norm, v = slice(64 * H, 68 * H), slice(68 * H, 136 * H)  # bytes of the K norms, and of V, in a slot
    cache[blocks] = slot
    cache[blocks[0], 0, norm] = (1.25 * slot[norm].copy().view(np.float32)).view(np.uint8)
    cache[other, 0, v] = slot[v]
    got = run(fn, case, causal=False)
    assert np.isfinite(got).all() and np.abs(got[:longest]).max() > 0
    # the rows of the one-key sequence are equal to one another per query head's kv head
    assert np.array_equal(got[:longest], got[longest:])
