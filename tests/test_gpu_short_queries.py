"""GPU parity of the kernels that take a few query tokens per sequence, each by itself: rq_short_attention (the decode
kernels' column groups) and the one-launch rq_paged_attention over many tiles, called through the C ABI so that the
op wrappers' choice between them does not matter.  Oracle and tolerance as in test_gpu_attention.py.
"""
import numpy as np
import pytest
import torch

from rq_testlib import Params, build_cache_oracle, check_tolerance, kv_config0, paged_layout
from test_gpu_attention import _dev, attn_case, ref

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
    assert np.array_equal(got[:longest], got[longest:])


def drafts(cfg, H, HQ, longest, p, BS=16, dtype=torch.bfloat16):
    """Queries of 1 to `longest` tokens: contexts at the query's own length (the first token sees one key), around the edges
    of the 32- and 64-key tiles, ending a token into a tile, and long; sequences without tokens or keys."""
    q_lens = [longest, 1, 0, max(1, longest - 1), longest, min(2, longest), longest, 0]
    ctx = [longest, 1, 40, 33, 64, 31 + min(2, longest), 1500, 0]
    return attn_case(cfg, q_lens, ctx, H, HQ, p, BS=BS, dtype=dtype)


def check(got, case, tag, causal=True):
    exp = ref(case, causal)
    err, excess, cs = check_tolerance(got, exp, str(case["q"].dtype).replace("torch.", ""), rot_block=case["p"].blk)
    print(f"{tag}: max_abs={err:.3e} excess_over_bound={excess:.3e} cos={cs:.7f}", flush=True)
    assert np.isfinite(got).all() and excess <= 0 and cs >= 0.999, (tag, err, excess, cs)


# 8, 4, 2, 1 and a run-time number of kv heads per workgroup of the decode kernels, on up to 8 columns and on more
HEADS = [(8, 8, 8), (4, 8, 4), (2, 4, 4), (1, 4, 2), (3, 6, 4), (8, 32, 4), (4, 28, 8), (2, 16, 2), (1, 8, 2), (3, 24, 2)]


@pytest.mark.parametrize("H,HQ,longest", HEADS)
def test_short_attention_heads_and_layouts(H, HQ, longest):
    """Each form against the oracle, and on a dense 3-bit cache of the same tokens bit for bit."""
    p = Params("iso", 3, 3)
    case = drafts(130 + HQ, H, HQ, longest, p)
    got = run("rq_short_attention", case)
    check(got, case, f"short-{H}-{HQ}-{longest}")
    ctx = case["lens"].tolist()
    bt, NB, slots = paged_layout(ctx, 16, 130 + HQ)
    k, v = kv_config0(sum(ctx), H, 128, 130 + HQ)
    dense = build_cache_oracle(k, v, np.concatenate(slots), NB, 16, p, dense3=True)
    assert np.array_equal(bt, case["bt"])
    assert np.array_equal(run("rq_short_attention", dict(case, cache=dense), dense3=True), got)


@pytest.mark.parametrize("BS", [1, 12, 32])
@pytest.mark.parametrize("H,HQ,longest,bits,dtype,causal", [(2, 8, 5, (4, 3), torch.float16, True), (8, 16, 4, (3, 4), torch.bfloat16, False)])
def test_short_attention_block_sizes(BS, H, HQ, longest, bits, dtype, causal):
    case = drafts(140 + BS, H, HQ, longest, Params("planar", *bits), BS=BS, dtype=dtype)
    check(run("rq_short_attention", case, causal), case, f"short-blocks-{BS}", causal)


def test_short_attention_strided_rows():
    """Query and output rows at other strides than their widths give the bits of plain ones, and nothing else is written."""
    case = drafts(150, 4, 16, 6, Params("iso", 3, 3))
    plain = run("rq_short_attention", case)
    n, HQ = case["q"].shape[:2]
    q = torch.full((n, HQ + 1, 136), float("nan"), dtype=torch.bfloat16, device="cuda")
    out = torch.full((n, HQ, 132), 7.0, dtype=torch.bfloat16, device="cuda")
    q[:, :HQ, :128] = case["q"].cuda()
    got = run("rq_short_attention", case, q=q[:, :HQ, :128], out=out[..., :128])
    assert np.array_equal(got, plain) and (out[..., 128:] == 7.0).all()


@pytest.mark.parametrize("fn", ["rq_short_attention", "rq_paged_attention"])
def test_more_tokens_than_keys(fn):
    """The tokens before the first key see none and give zeros."""
    case = attn_case(89, [5, 3], [2, 40], 2, 8, Params("iso", 3, 3))
    got = run(fn, case)
    assert (got[:3] == 0).all() and (got[3:] != 0).any(axis=(1, 2)).all()
    case["q_lens"], case["cu"], case["q"] = [2, 3], np.asarray([0, 2, 5], np.int32), case["q"][3:]
    check(got[3:], case, fn)


@pytest.mark.parametrize("H,HQ,longest,bits,dtype,causal", [
    (8, 32, 16, (3, 3), torch.bfloat16, True),
    (8, 32, 1, (4, 4), torch.float16, True),
    (4, 28, 16, (3, 4), torch.bfloat16, False),
    (2, 24, 9, (4, 3), torch.float16, True),      # 12 heads: two workgroups per kv head, more groups than the decode kernels take
    (1, 9, 16, (3, 3), torch.bfloat16, True),     # 9 heads: three
    (1, 1, 16, (3, 3), torch.bfloat16, False),
])
def test_one_launch_over_many_tiles(H, HQ, longest, bits, dtype, causal):
    """rq_paged_attention on queries of at most 16 tokens: both tile buffers, the running maximum and V exponent over up to 24
    tiles, the split of wide groups, waves that only decode tiles."""
    case = drafts(160 + HQ, H, HQ, longest, Params("iso", *bits), dtype=dtype)
    check(run("rq_paged_attention", case, causal), case, f"one-launch-{HQ}-{longest}", causal)


@pytest.mark.parametrize("H,HQ,q_lens,ctx", [
    (2, 16, [17, 40, 1], [1100, 64, 900]),         # groups of 16: 8 heads, one group a workgroup
    (1, 3, [33, 97, 16], [1500, 97, 40]),          # 3 heads, two groups
    (2, 2, [129, 20], [1024 + 129, 20]),           # 1 head, eight
    (2, 12, [50, 17], [300, 17]),                  # groups of 32, two waves that only decode tiles
    (1, 2, [65, 200], [365, 200]),                 # two groups, four such waves
    (8, 32, [260, 30, 257, 200], [260, 90, 300, 200]),   # two groups of four heads
    (8, 32, [17, 3] * 20, [40, 5] * 20),                 # one, four waves
    (8, 8, [33] * 36, [64] * 36),                        # four groups of one head, four waves
])
@pytest.mark.parametrize("dtype,causal", [(torch.bfloat16, True), (torch.float16, False)])
def test_one_launch_longer_queries(H, HQ, q_lens, ctx, dtype, causal):
    """rq_paged_attention's workgroup shapes for queries of more than 16 tokens."""
    case = attn_case(170 + HQ, q_lens, ctx, H, HQ, Params("iso", 3, 4), dtype=dtype)
    check(run("rq_paged_attention", case, causal), case, f"one-launch-longer-{HQ}", causal)


@pytest.mark.parametrize("fused", [True, False], ids=["fused", "unfused"])
@pytest.mark.parametrize("ctx,q_lens", [([2000, 3000, 700, 40], [1, 4, 8, 2]), ([60, 90, 8, 33], [1, 16, 8, 3])], ids=["long", "short"])
def test_backend_drafts(monkeypatch, fused, ctx, q_lens):
    """Drafts after a decode in one forward of the backend, over contexts that take the decode kernels and over short ones:
    the cache bytes and every row, and the shared workspaces as they were reserved."""
    import oracle as O
    from rotorquant_vllm import kernels as K
    from test_gpu_backend import _mixed_setup
    impl, p, c = _mixed_setup(monkeypatch, 8, 32, "iso", 3, "fast", ctx, q_lens, 180, fused=fused)
    cache = _dev(c["cache0"])
    impl._init_cg_buffers(cache, torch.bfloat16)
    retired = len(K._ws_retired)
    out = torch.full(c["q"].shape, float("nan"), dtype=torch.bfloat16, device="cuda")
    impl.forward(None, _dev(c["q"]), _dev(c["k_new"]), _dev(c["v_new"]), cache, c["md"], output=out)
    torch.cuda.synchronize()
    assert len(K._ws_retired) == retired and np.array_equal(cache.cpu().numpy(), c["full_cache"])
    exp = O.unfused_attention(c["q"].float().numpy(), np.concatenate([[0], np.cumsum(q_lens)]).astype(np.int32), c["full_cache"], c["bt"],
                              np.asarray(ctx, np.int32), 8, 128, p.kc.numpy(), p.vc.numpy(), p.R.numpy(), 128 ** -0.5, "bfloat16")
    got = out.float().cpu().numpy()
    err, excess, cs = check_tolerance(got, exp, "bfloat16", rot_block=p.blk)
    assert np.isfinite(got).all() and excess <= 0 and cs >= 0.999, (err, excess, cs)
