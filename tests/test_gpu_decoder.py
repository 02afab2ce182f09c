"""Decoder (the caller of the hot path) on a small configuration: the library
BitLinear inside the full layer stack against a torch emulation of the same
arithmetic, prefill/decode consistency, and the graph-replayed decode loop."""
import numpy as np
import pytest
import torch

from bitnet_amd import _lib, decoder, pack_weight
from bitnet_amd.bitlinear import BitLinearKernel
from tests.gpu_util import host_bits
from oracle import bitlinear_oracle as o

pytestmark = pytest.mark.gpu

SMALL = decoder.ModelArgs(dim=256, n_layers=3, n_heads=4, n_kv_heads=2, vocab_size=512, ffn_dim=512)


class RefBitLinear(torch.nn.Module):
    """gpu/model.py:68-75 + bitnet_kernels.h:79-82 in plain torch: compiled-mode
    quantizer (reciprocal, multiply, bf16 scale, exact fp32 product), exact
    integer product in float64, fp32 divide / multiply / RNE epilogue with the
    equal-slot scale rule."""

    def __init__(self, mod: BitLinearKernel, ws_num: int):
        super().__init__()
        self.w = pack_weight.convert_weight_int2_to_int8(mod.weight.data, mod.out_features, mod.in_features).double()
        self.ws = mod.weight_scale.data.float()
        self.slot = torch.arange(mod.out_features, device=self.w.device) // (mod.out_features // ws_num)

    def forward(self, x):
        xf = x.float()
        amax = xf.abs().amax(dim=-1, keepdim=True).clamp(min=1e-5)
        s = ((1.0 / amax) * 127.0).to(torch.bfloat16).float()
        q = (xf * s).round().clamp(-128, 127)
        acc = (q.double() @ self.w.T).float()
        return (acc / s * self.ws[self.slot]).to(torch.bfloat16)


def _build(args, seed=0):
    torch.manual_seed(seed)
    with torch.device("cuda"):
        prev = torch.get_default_dtype()
        torch.set_default_dtype(torch.bfloat16)
        try:
            model = decoder.Transformer(args)
        finally:
            torch.set_default_dtype(prev)
    return decoder.random_init_(model, seed)


def _reference_copy(model):
    import copy

    ref = copy.deepcopy(model)
    for lr in ref.layers:
        lr.attention.wqkv = RefBitLinear(lr.attention.wqkv, 1)  # shapes outside the reference's table: one slot
        lr.attention.wo = RefBitLinear(lr.attention.wo, 1)
        lr.feed_forward.w13 = RefBitLinear(lr.feed_forward.w13, 1)
        lr.feed_forward.w2 = RefBitLinear(lr.feed_forward.w2, 1)
    return ref


def test_state_dict_names_match_the_reference_checkpoint_layout():
    model = _build(SMALL)
    keys = set(model.state_dict().keys())
    for k in ["tok_embeddings.weight", "norm.weight", "output.weight", "layers.0.attention.wqkv.weight",
              "layers.0.attention.wqkv.weight_scale", "layers.0.attention.wo.weight", "layers.0.attention.attn_sub_norm.weight",
              "layers.0.feed_forward.w13.weight", "layers.0.feed_forward.w2.weight_scale",
              "layers.0.feed_forward.ffn_sub_norm.weight", "layers.0.attention_norm.weight", "layers.0.ffn_norm.weight"]:
        assert k in keys, k
    assert model.layers[0].attention.wqkv.weight.shape == (512, 64) and model.layers[0].attention.wqkv.weight.dtype == torch.int8


def test_logits_equal_torch_emulation_prefill_and_decode():
    model = _build(SMALL, seed=1)
    ref = _reference_copy(model)
    B, P, S = 2, 24, 40
    dev = torch.device("cuda")
    cos, sin = decoder.rope_tables(SMALL.dim // SMALL.n_heads, S, SMALL.rope_theta, dev)
    g = torch.Generator(device="cuda").manual_seed(5)
    prompt = torch.randint(0, SMALL.vocab_size, (B, P), generator=g, device=dev)
    pos = torch.arange(P, device=dev)[None].expand(B, P).contiguous()
    c1, c2 = model.make_cache(B, S, dev), ref.make_cache(B, S, dev)
    l1 = model.forward_tokens(prompt, pos, c1, cos, sin)   # M = 48: quantizer kernel + MFMA GEMM
    l2 = ref.forward_tokens(prompt, pos, c2, cos, sin)
    assert torch.equal(l1, l2)
    tok = torch.argmax(l1[:, -1], dim=-1).view(B, 1)
    p1 = torch.full((B, 1), P, device=dev)
    d1 = model.forward_tokens(tok, p1, c1, cos, sin)        # M = 2: fused one-kernel forward
    d2 = ref.forward_tokens(tok, p1, c2, cos, sin)
    assert torch.equal(d1, d2)
    for (k1, v1), (k2, v2) in zip(c1, c2):
        assert torch.equal(k1, k2) and torch.equal(v1, v2)


def test_decode_step_equals_prefill_of_the_longer_prompt():
    model = _build(SMALL, seed=2)
    B, P, S = 1, 17, 32
    dev = torch.device("cuda")
    cos, sin = decoder.rope_tables(SMALL.dim // SMALL.n_heads, S, SMALL.rope_theta, dev)
    g = torch.Generator(device="cuda").manual_seed(6)
    ids = torch.randint(0, SMALL.vocab_size, (B, P + 1), generator=g, device=dev)
    pos = torch.arange(P + 1, device=dev)[None]
    full = model.forward_tokens(ids, pos, model.make_cache(B, S, dev), cos, sin)[:, -1]
    cache = model.make_cache(B, S, dev)
    model.forward_tokens(ids[:, :P], pos[:, :P], cache, cos, sin)
    step = model.forward_tokens(ids[:, P:], pos[:, P:], cache, cos, sin)[:, -1]
    # every op is per token except attention, whose cache holds the same keys/values
    assert torch.equal(full, step)


def test_graph_decode_loop_equals_eager_loop():
    model = _build(SMALL, seed=3)
    B, P, G = 2, 16, 12
    dev = torch.device("cuda")
    g = torch.Generator(device="cuda").manual_seed(7)
    prompt = torch.randint(0, SMALL.vocab_size, (B, P), generator=g, device=dev)
    outs = []
    for use_graph in (False, True):
        gen = decoder.Generator(model, B, P + G + 1, use_graph=use_graph)
        first = gen.prefill(prompt)
        toks = gen.decode(first, P, G)
        torch.cuda.synchronize()
        outs.append(torch.cat([first[None], toks]).cpu())
    assert torch.equal(outs[0], outs[1])
    assert outs[0].shape == (G + 1, B)


BIG_HEADS = decoder.ModelArgs(dim=512, n_layers=2, n_heads=4, n_kv_heads=1, vocab_size=256, ffn_dim=768)  # head_dim 128


def _ulp(a: torch.Tensor, b: torch.Tensor) -> torch.Tensor:
    def mono(t):
        v = t.view(torch.int16).to(torch.int32)
        return torch.where(v < 0, -(v & 0x7FFF), v)
    return (mono(a) - mono(b)).abs()


@pytest.mark.parametrize("n_splits", [1, 3, 8])
@pytest.mark.parametrize("B,S,nh,nkv", [(1, 641, 20, 5), (8, 200, 20, 5), (2, 64, 4, 1), (3, 1500, 8, 8), (2, 33, 16, 2)])
def test_attention_decode_kernel_against_torch_fp32(B, S, nh, nkv, n_splits):
    """A floating-point kernel: compared with the fp32 torch restatement (rope,
    cache write, softmax(QK^T/sqrt(d))V).  Its probabilities are rounded to
    bf16 for the matrix pipe and its fp32 sums run in another order: 3 bf16 ulp
    or 4e-3 absolute on the bf16 outputs."""
    hd = 128
    dev = torch.device("cuda")
    g = torch.Generator(device="cuda").manual_seed(B * 1000 + S)
    args = decoder.ModelArgs(dim=nh * hd, n_heads=nh, n_kv_heads=nkv, n_layers=1, vocab_size=16, ffn_dim=256)
    att = decoder.Attention.__new__(decoder.Attention)
    torch.nn.Module.__init__(att)
    att.head_dim, att.n_heads, att.n_kv_heads = hd, nh, nkv
    xqkv = torch.randn(B, (nh + 2 * nkv) * hd, generator=g, device=dev).to(torch.bfloat16)
    ck = torch.randn(B, S, nkv, hd, generator=g, device=dev).to(torch.bfloat16)
    cv = torch.randn(B, S, nkv, hd, generator=g, device=dev).to(torch.bfloat16)
    pos = torch.randint(0, S, (B,), generator=g, device=dev)
    pos[0] = S - 1
    if B > 1:
        pos[1] = 0
    cos, sin = decoder.rope_tables(hd, S, 500000.0, dev)
    # reference
    q, k, v = att.split_qkv(xqkv[:, None, :])
    c, s_ = cos[pos][:, None, None, :], sin[pos][:, None, None, :]
    q, k = decoder.apply_rope(q, c, s_), decoder.apply_rope(k, c, s_)
    rk, rv = ck.clone(), cv.clone()
    bidx = torch.arange(B, device=dev)
    rk[bidx, pos] = k[:, 0]
    rv[bidx, pos] = v[:, 0]
    mask = torch.arange(S, device=dev)[None, None, :] <= pos[:, None, None]
    want = att.attend(q, rk, rv, mask)[:, 0]
    ws = decoder.AttnWorkspace(B, nh, nkv, n_splits, dev) if n_splits > 1 else None
    got = decoder.attn_decode(xqkv, ck, cv, pos, cos, sin, nh, nkv, ws)
    torch.cuda.synchronize()
    assert torch.equal(ck, rk) and torch.equal(cv, rv)  # cache rows written exactly
    if ws is not None:
        again = decoder.attn_decode(xqkv, ck, cv, pos, cos, sin, nh, nkv, ws)  # same cache row rewritten
        assert torch.equal(again, got)
    # the same call with the positions' cos | sin rows handed over: identical bits
    emb = torch.randn(16, 64, generator=g, device=dev).to(torch.bfloat16)
    toks = torch.randint(0, 16, (B,), generator=g, device=dev)
    h0, rows = decoder.decode_step_begin(toks, pos, emb, cos, sin)
    assert torch.equal(h0, emb[toks]) and torch.equal(rows, torch.cat([cos[pos], sin[pos]], dim=1))
    ck2, cv2 = ck.clone(), cv.clone()
    with_rows = decoder.attn_decode(xqkv, ck2, cv2, pos, cos, sin, nh, nkv, ws, rope_rows=rows)
    torch.cuda.synchronize()
    assert torch.equal(with_rows, got) and torch.equal(ck2, rk) and torch.equal(cv2, rv)
    ulps, tol = 3, 4e-3
    bad = (_ulp(got, want) > ulps) & ((got.float() - want.float()).abs() > tol)
    assert not bad.any(), f"{int(bad.sum())} of {bad.numel()} outside tolerance"


@pytest.mark.parametrize("n_splits", [5, 16])
@pytest.mark.parametrize("p", [0, 31, 32, 511, 600, 2047, 4099])
def test_attention_decode_long_cache_any_position(p, n_splits):
    """Cache capacity far beyond the position (4100 rows, up to 16 splits, eight
    waves per workgroup): the rows are dealt to splits and waves in blocks of
    32, so positions at block edges, inside the first round and in later rounds
    are covered.  Same comparison and tolerance as above (matrix-pipe kernel)."""
    B, S, nh, nkv, hd = 2, 4100, 8, 2, 128
    dev = torch.device("cuda")
    g = torch.Generator(device="cuda").manual_seed(77 + p)
    att = decoder.Attention.__new__(decoder.Attention)
    torch.nn.Module.__init__(att)
    att.head_dim, att.n_heads, att.n_kv_heads = hd, nh, nkv
    xqkv = torch.randn(B, (nh + 2 * nkv) * hd, generator=g, device=dev).to(torch.bfloat16)
    ck = torch.randn(B, S, nkv, hd, generator=g, device=dev).to(torch.bfloat16)
    cv = torch.randn(B, S, nkv, hd, generator=g, device=dev).to(torch.bfloat16)
    pos = torch.tensor([p, max(0, p - 17)], device=dev)
    cos, sin = decoder.rope_tables(hd, S, 500000.0, dev)
    q, k, v = att.split_qkv(xqkv[:, None, :])
    c, s_ = cos[pos][:, None, None, :], sin[pos][:, None, None, :]
    q, k = decoder.apply_rope(q, c, s_), decoder.apply_rope(k, c, s_)
    rk, rv = ck.clone(), cv.clone()
    bidx = torch.arange(B, device=dev)
    rk[bidx, pos] = k[:, 0]
    rv[bidx, pos] = v[:, 0]
    mask = torch.arange(S, device=dev)[None, None, :] <= pos[:, None, None]
    want = att.attend(q, rk, rv, mask)[:, 0]
    ws = decoder.AttnWorkspace(B, nh, nkv, n_splits, dev)
    got = decoder.attn_decode(xqkv, ck, cv, pos, cos, sin, nh, nkv, ws)
    again = decoder.attn_decode(xqkv, ck, cv, pos, cos, sin, nh, nkv, ws)
    torch.cuda.synchronize()
    assert torch.equal(ck, rk) and torch.equal(cv, rv) and torch.equal(again, got)
    bad = (_ulp(got, want) > 3) & ((got.float() - want.float()).abs() > 4e-3)
    assert not bad.any(), f"{int(bad.sum())} of {bad.numel()} outside tolerance"


@pytest.mark.parametrize("n_splits", [1, 3])
@pytest.mark.parametrize("nh,nkv", [(1, 1), (4, 1), (16, 2)])
def test_attention_decode_takes_the_new_row_at_every_place_of_a_block(nh, nkv, n_splits):
    """The new token's k and v are put into a block's registers at a place that depends on the position: all 32 of them, with
    keys along the queries, so that the new row has most of the weight.  Comparison and tolerance as above."""
    B, S, hd = 32, 70, 128
    dev = torch.device("cuda")
    g = torch.Generator(device="cuda").manual_seed(nh)
    att = decoder.Attention.__new__(decoder.Attention)
    torch.nn.Module.__init__(att)
    att.head_dim, att.n_heads, att.n_kv_heads = hd, nh, nkv
    xqkv = torch.randn(B, nh + 2 * nkv, hd, generator=g, device=dev)
    xqkv[:, nh : nh + nkv] = xqkv[:, :nh].reshape(B, nkv, nh // nkv, hd).mean(2)
    xqkv = xqkv.reshape(B, -1).to(torch.bfloat16)
    ck, cv = (torch.randn(B, S, nkv, hd, generator=g, device=dev).to(torch.bfloat16) for _ in range(2))
    pos = torch.arange(32, 64, device=dev)
    cos, sin = decoder.rope_tables(hd, S, 500000.0, dev)
    q, k, v = att.split_qkv(xqkv[:, None, :])
    c, s_ = cos[pos][:, None, None, :], sin[pos][:, None, None, :]
    q, k = decoder.apply_rope(q, c, s_), decoder.apply_rope(k, c, s_)
    rk, rv = ck.clone(), cv.clone()
    bidx = torch.arange(B, device=dev)
    rk[bidx, pos], rv[bidx, pos] = k[:, 0], v[:, 0]
    want = att.attend(q, rk, rv, torch.arange(S, device=dev)[None, None, :] <= pos[:, None, None])[:, 0]
    got = decoder.attn_decode(xqkv, ck, cv, pos, cos, sin, nh, nkv, decoder.AttnWorkspace(B, nh, nkv, n_splits, dev) if n_splits > 1 else None)
    torch.cuda.synchronize()
    assert torch.equal(ck, rk) and torch.equal(cv, rv)
    bad = (_ulp(got, want) > 3) & ((got.float() - want.float()).abs() > 4e-3)
    assert not bad.any(), f"{int(bad.sum())} of {bad.numel()} outside tolerance"


@pytest.mark.parametrize("n_splits", [1, 8])
def test_attention_decode_ignores_rows_behind_the_position(n_splits):
    """Cache rows behind a sequence's position may never have been written:
    with NaNs there the output has the bits it has with finite values there."""
    B, S, nh, nkv, hd = 3, 300, 8, 2, 128
    dev = torch.device("cuda")
    g = torch.Generator(device="cuda").manual_seed(4242)
    xqkv = torch.randn(B, (nh + 2 * nkv) * hd, generator=g, device=dev).to(torch.bfloat16)
    ck = torch.randn(B, S, nkv, hd, generator=g, device=dev).to(torch.bfloat16)
    cv = torch.randn(B, S, nkv, hd, generator=g, device=dev).to(torch.bfloat16)
    pos = torch.tensor([0, 37, 255], device=dev)
    cos, sin = decoder.rope_tables(hd, S, 500000.0, dev)
    ws = decoder.AttnWorkspace(B, nh, nkv, n_splits, dev) if n_splits > 1 else None
    want = decoder.attn_decode(xqkv, ck.clone(), cv.clone(), pos, cos, sin, nh, nkv, ws)
    behind = torch.arange(S, device=dev)[None, :] > pos[:, None]
    ck[behind] = float("nan")
    cv[behind] = float("nan")
    got = decoder.attn_decode(xqkv, ck, cv, pos, cos, sin, nh, nkv, ws)
    torch.cuda.synchronize()
    assert not torch.isnan(got.float()).any()
    assert torch.equal(got, want)
    assert torch.isnan(ck[behind].float()).all() and torch.isnan(cv[behind].float()).all()


def test_fused_decode_path_against_unfused():
    """Five-kernels-per-layer decode step vs the torch-glue step on a small model
    with 128-wide heads: every sub-step on identical inputs (bit-level bounds, see
    _decode_step_substeps_against_glue), and over a short generation the same
    greedy tokens most of the time (each path's quantizers amplify the other's
    rounding differences, so the token streams may part at a near tie)."""
    model = _build(BIG_HEADS, seed=4)
    assert model.fused_decode_ok(2)
    B, P, G = 2, 20, 8
    dev = torch.device("cuda")
    g = torch.Generator(device="cuda").manual_seed(9)
    prompt = torch.randint(0, BIG_HEADS.vocab_size, (B, P), generator=g, device=dev)
    outs = []
    for fused in (False, True):
        gen = decoder.Generator(model, B, P + G + 1, use_graph=fused, fused=fused)
        first = gen.prefill(prompt)
        outs.append(torch.cat([first[None], gen.decode(first, P, G)]).cpu())
    torch.cuda.synchronize()
    assert (outs[0] == outs[1]).float().mean() > 0.8
    gen = decoder.Generator(model, B, P + G + 1)
    first = gen.prefill(prompt)
    h, hc, worst = _decode_step_substeps_against_glue(model, gen, first.view(B, 1), P)
    cosine = torch.nn.functional.cosine_similarity(model.output(model.norm(h)).float(), model.output(model.norm(hc)).float(), dim=-1)
    assert float(cosine.min()) > 0.99, (float(cosine.min()), worst)


@pytest.mark.parametrize("which", [0, 1])
@pytest.mark.parametrize("B,V,K", [(1, 128256, 2560), (8, 128256, 2560), (3, 1000, 256), (16, 4111, 512), (2, 48, 64),
                                   (2, 4111, 512), (4, 77, 1024), (5, 32000, 2048)])
def test_lm_head_greedy_kernel(B, V, K, which):
    """Final norm + bf16 LM head + greedy token: the normalised rows bit-exact
    against the oracle's RMSNorm, the logits within one bf16 ulp (or 1e-3 of
    the largest logit, where sums cancel) of an fp32 torch evaluation (fp32
    sums in another order), the token equal to the first maximum of the
    kernel's own logits."""
    dev = torch.device("cuda")
    g = torch.Generator(device="cuda").manual_seed(B * 7 + V)
    h = (torch.randn(B, K, generator=g, device=dev) * 3).to(torch.bfloat16)
    emb = (torch.randn(V, K, generator=g, device=dev) * 0.02).to(torch.bfloat16)
    norm = decoder.RMSNorm(K, 1e-5).to(dev)
    norm.weight.data = (1 + 0.1 * torch.randn(K, generator=g, device=dev)).to(torch.bfloat16)
    ws = decoder.LmHeadWorkspace(B, V, K, dev)
    logits = torch.full((B, V), float("nan"), dtype=torch.float32, device=dev)
    lib = _lib.load_library()
    assert lib.bitnet_lm_head_set_kernel(which) == 0  # 0: built-in choice (streaming kernel where it applies), 1: MFMA kernel
    try:
        tok = decoder.lm_head_greedy(h, norm, emb, ws, logits_out=logits)
        torch.cuda.synchronize()
    finally:
        lib.bitnet_lm_head_set_kernel(0)
    want_y = o.rmsnorm_bf16(host_bits(h), host_bits(norm.weight.data), 1e-5)
    assert np.array_equal(host_bits(ws.y), want_y)
    ref = (ws.y.float() @ emb.float().T).to(torch.bfloat16)
    got = logits.to(torch.bfloat16)
    assert torch.equal(got.float(), logits)  # the kernel's logits are bf16 values
    bad = (_ulp(got, ref) > 1) & ((got.float() - ref.float()).abs() > 1e-3 * float(ref.float().abs().max()))
    assert not bad.any(), f"{int(bad.sum())} of {bad.numel()} logits outside tolerance"
    assert torch.equal(tok, torch.argmax(logits, dim=-1))
    # without the logits buffer, and a second call on the same scratch
    tok2 = decoder.lm_head_greedy(h, norm, emb, ws)
    assert torch.equal(tok2, tok)


@pytest.mark.parametrize("logits", ["normal", "flat", "peaked", "masked", "tiny", "huge"])
@pytest.mark.parametrize("B,V", [(1, 128256), (4, 128256), (3, 1024), (16, 4111), (2, 17), (1, 1)])
def test_top_p_sampler_draws_what_torch_draws(B, V, logits):
    gen = torch.Generator(device="cuda").manual_seed(V + B)
    x = torch.randn(B, V, generator=gen, device="cuda")
    if logits == "flat":
        x = torch.zeros_like(x)
    elif logits == "peaked":
        x = x * 8.0
    elif logits == "masked":
        x = torch.where(torch.rand(B, V, generator=gen, device="cuda") < 0.5, float("-inf"), x)
        x[:, 0] = 0.5
    elif logits == "tiny":  # values that share a bucket, in which their order counts
        x = x * 2.0**-21
    elif logits == "huge":
        x = x * 2.0**40
    x = x.to(torch.bfloat16).float()
    sampler = decoder.TopPSampler(B, V, "cuda")
    tok = torch.zeros(B, dtype=torch.int64, device="cpu", pin_memory=True)
    nxt, pos, row = (torch.full((B,), i, dtype=torch.int64, device="cuda") for i in range(3))
    for draw, (t, p) in enumerate([(0.7, 0.95), (0.7, 0.95), (1.3, 0.5), (1.0, 1.0), (1.0, 0.0), (0.1, 0.9)]):
        # (float64: where probabilities differ by less than a float32 resolves, torch's own order is one by index)
        probs = torch.softmax(x.double() / t, dim=-1)
        if logits == "tiny":  # ranked by the logits: their probabilities differ in the last bits only
            order = torch.sort(x, dim=-1, descending=True, stable=True)[1]
        else:
            order = torch.sort(probs, dim=-1, descending=True, stable=True)[1]
        ranked = torch.gather(probs, -1, order)
        kept = torch.where(torch.cumsum(ranked, -1) - ranked > p + 1e-12, 0.0, ranked)
        q = torch.empty(B, V, device="cuda").exponential_(1.0, generator=torch.Generator(device="cuda").manual_seed(draw))
        want = torch.gather(order, -1, torch.argmax(kept / q, dim=-1, keepdim=True)).view(-1)
        sampler(x, t, p, torch.Generator(device="cuda").manual_seed(draw), tok, nxt, pos, row)
        torch.cuda.synchronize()
        sampler.check()
        assert tok.tolist() == want.tolist(), (draw, t, p)
        assert nxt.tolist() == want.tolist() and row.tolist() == want.tolist() and pos.tolist() == [draw + 2] * B
        if logits in ("normal", "peaked", "flat") and V >= 1024:
            ref = decoder.top_p_sample(torch.softmax(x / t, dim=-1), p, torch.Generator(device="cuda").manual_seed(draw))
            assert tok.tolist() == ref.view(-1).tolist(), (draw, t, p)
    for bad in (float("nan"), float("inf")):
        x[B - 1, V - 1] = bad
        sampler(x, 1.0, 0.9, gen, tok)
        torch.cuda.synchronize()
        with pytest.raises(RuntimeError, match="inf or nan"):
            sampler.check()


@pytest.mark.parametrize("sign", ["any", "negative", "masked"])
@pytest.mark.parametrize("scale,temperature", [
    (2.0**-21, 1e-8), (2.0**-21, 2.0**-21), (2.0**-60, 2.0**-61), (2.0**-90, 2e-27),  # small values at small temperatures
    (2.0**20, 2.0**-22), (2.0**50, 0.7), (2.0**44, 2.0**44), (2.0**60, 1.0),          # large ones: the largest alone, or not
    (2.0**95, 3e28), (1.0, 9e29), (2.0**-10, 1e6),                                    # large temperatures
])
def test_top_p_sampler_tells_values_apart_at_every_temperature(scale, temperature, sign):
    B, V = 3, 2048
    gen = torch.Generator(device="cuda").manual_seed(11)
    x = torch.randn(B, V, generator=gen, device="cuda") * scale
    if sign != "any":
        x = -x.abs() - scale
    if sign == "masked":
        x[:, ::3] = float("-inf")
    x = x.to(torch.bfloat16).float()
    x[1, :700] = x[1, x[1].argmax()]  # (many tokens of the largest value)
    assert decoder.TopPSampler.applies(B, V, temperature, 0.9)
    sampler = decoder.TopPSampler(B, V, "cuda")
    tok = torch.zeros(B, dtype=torch.int64, device="cuda")
    probs = torch.softmax(x.double() / float(np.float32(temperature)), dim=-1)
    order = torch.sort(x, dim=-1, descending=True, stable=True)[1]
    ranked = torch.gather(probs, -1, order)
    for draw, p in enumerate((0.95, 0.5, 1.0, 0.0)):
        kept = torch.where(torch.cumsum(ranked, -1) - ranked > p + 1e-12, 0.0, ranked)
        q = torch.empty(B, V, device="cuda").exponential_(1.0, generator=torch.Generator(device="cuda").manual_seed(draw))
        want = torch.gather(order, -1, torch.argmax(kept / q, dim=-1, keepdim=True)).view(-1)
        sampler(x, temperature, p, torch.Generator(device="cuda").manual_seed(draw), tok)
        torch.cuda.synchronize()
        sampler.check()
        assert tok.tolist() == want.tolist(), p
    # what softmax(logits / temperature) cannot express is refused, as it was by torch
    for bad in (x.new_full((), 3e38), x.new_full((), float("-inf"))):
        y = torch.full_like(x, float(bad))
        sampler(y, min(temperature, 0.5), 0.9, gen, tok)
        torch.cuda.synchronize()
        with pytest.raises(RuntimeError, match="inf or nan"):
            sampler.check()


def test_generator_with_and_without_the_lm_head_kernel_agree():
    args = decoder.ModelArgs(dim=256, n_layers=2, n_heads=2, n_kv_heads=1, vocab_size=512, ffn_dim=512)
    model = _build(args, seed=3)
    prompt = torch.randint(0, args.vocab_size, (2, 9), generator=torch.Generator().manual_seed(5)).cuda()
    outs = []
    for fused_head in (True, False):
        gen = decoder.Generator(model, 2, 40, use_graph=True, fused_head=fused_head)
        assert gen.lm_head == fused_head
        first = gen.prefill(prompt)
        outs.append(gen.decode(first, 9, 12).cpu())
    # greedy tokens can only differ where two logits tie within fp32 summation order; with random weights they do not
    assert torch.equal(outs[0], outs[1])


@pytest.mark.parametrize("B,T,S,nh,nkv,start", [(1, 512, 640, 20, 5, 0), (3, 37, 64, 4, 1, 5), (2, 1, 16, 8, 8, 15)])
def test_rope_cache_tokens_kernel_equals_torch(B, T, S, nh, nkv, start):
    """Rope + cache write for a block of tokens: the rotated q and the cache
    rows equal the torch restatement bit for bit (fp32 products, one fp32
    add, one rounding to bf16), other cache rows untouched."""
    hd = 128
    dev = torch.device("cuda")
    g = torch.Generator(device="cuda").manual_seed(B * 100 + T)
    xqkv = torch.randn(B * T, (nh + 2 * nkv) * hd, generator=g, device=dev).to(torch.bfloat16)
    ck = torch.randn(B, S, nkv, hd, generator=g, device=dev).to(torch.bfloat16)
    cv = torch.randn(B, S, nkv, hd, generator=g, device=dev).to(torch.bfloat16)
    pos = (start + torch.arange(T, device=dev))[None, :].expand(B, T).contiguous()
    cos, sin = decoder.rope_tables(hd, S, 500000.0, dev)
    att = decoder.Attention.__new__(decoder.Attention)
    torch.nn.Module.__init__(att)
    att.head_dim, att.n_heads, att.n_kv_heads = hd, nh, nkv
    q, k, v = att.split_qkv(xqkv.view(B, T, -1))
    c, s_ = cos[pos][:, :, None, :], sin[pos][:, :, None, :]
    want_q, want_k = decoder.apply_rope(q, c, s_), decoder.apply_rope(k, c, s_)
    rk, rv = ck.clone(), cv.clone()
    rk[:, start:start + T] = want_k
    rv[:, start:start + T] = v
    got_q = decoder.rope_cache_tokens(xqkv, ck, cv, pos, cos, sin, nh, nkv)
    torch.cuda.synchronize()
    assert torch.equal(got_q, want_q)
    assert torch.equal(ck, rk) and torch.equal(cv, rv)


def test_prompt_through_the_library_kernels_against_the_torch_glue():
    """Generator.prefill with the prompt-sized layer stack (norm / gate /
    residual folded into the BitLinear calls, rope + cache kernel, the prompt
    attention kernel) against forward_tokens (every op in torch around the same
    BitLinear kernels, fp32 attention): the first layer's cache rows and the
    last token's logits within bf16 noise (the norm's and the attention's sums
    run in another order and precision), and each path's first token equal to
    the argmax of its own logits."""
    model = _build(BIG_HEADS, seed=11)
    B, P, S = 2, 70, 96
    dev = torch.device("cuda")
    g = torch.Generator(device="cuda").manual_seed(12)
    prompt = torch.randint(0, BIG_HEADS.vocab_size, (B, P), generator=g, device=dev)
    cos, sin = decoder.rope_tables(128, S, BIG_HEADS.rope_theta, dev)
    c1, c2 = model.make_cache(B, S, dev), model.make_cache(B, S, dev)
    h1 = model.prefill_hidden_fused(prompt, c1, cos, sin)
    pos = torch.arange(P, device=dev)[None].expand(B, P).contiguous()
    logits2 = model.forward_tokens(prompt, pos, c2, cos, sin)
    torch.cuda.synchronize()
    for a_, b_ in zip(c1[0], c2[0]):  # the two RMSNorm evaluations differ in the last bf16 bit of a few elements
        assert torch.allclose(a_.float(), b_.float(), rtol=2e-2, atol=2e-2)
        assert torch.equal(a_[:, P:], b_[:, P:])  # rows behind the prompt untouched
    logits1 = model.output(model.norm(h1[:, -1])).float()
    assert torch.allclose(logits1, logits2[:, -1], rtol=5e-2, atol=5e-2)
    gen = decoder.Generator(model, B, S)
    assert gen.lm_head
    first = gen.prefill(prompt)
    assert torch.equal(first, torch.argmax(logits1, dim=-1))
    gen2 = decoder.Generator(model, B, S, fused_head=False)
    assert torch.equal(gen2.prefill(prompt), torch.argmax(logits2[:, -1], dim=-1))


@pytest.mark.parametrize("B,T,S,nh,nkv,start", [(1, 512, 640, 20, 5, 0), (2, 70, 96, 4, 1, 0), (3, 33, 80, 8, 8, 40),
                                               (1, 1, 16, 16, 2, 9), (2, 200, 256, 8, 4, 17), (1, 16, 16, 2, 2, 0)])
def test_attention_prefill_kernel_against_torch_fp32(B, T, S, nh, nkv, start):
    """Floating-point kernel: compared with the fp32 torch restatement
    softmax(QK^T/sqrt(d))V over cache rows 0..start+t.  The kernel rounds the
    probabilities to bf16 for the matrix pipe (relative error 2^-9 each), so
    the tolerance is 3 bf16 ulp or 4e-3 absolute on the bf16 outputs.  Cache
    rows behind the last position hold NaNs: they must not be touched."""
    hd = 128
    dev = torch.device("cuda")
    g = torch.Generator(device="cuda").manual_seed(B * 1000 + T + start)
    q = torch.randn(B, T, nh, hd, generator=g, device=dev).to(torch.bfloat16)
    ck = torch.randn(B, S, nkv, hd, generator=g, device=dev).to(torch.bfloat16)
    cv = torch.randn(B, S, nkv, hd, generator=g, device=dev).to(torch.bfloat16)
    ck[:, start + T:] = float("nan")
    cv[:, start + T:] = float("nan")
    att = decoder.Attention.__new__(decoder.Attention)
    torch.nn.Module.__init__(att)
    att.head_dim, att.n_heads, att.n_kv_heads = hd, nh, nkv
    pos = start + torch.arange(T, device=dev)
    mask = (torch.arange(start + T, device=dev)[None, None, :] <= pos[None, :, None]).expand(B, T, start + T)
    want = att.attend(q, ck[:, :start + T], cv[:, :start + T], mask).reshape(B * T, nh * hd)
    got = decoder.attn_prefill(q, ck, cv, start)
    torch.cuda.synchronize()
    assert not torch.isnan(got.float()).any()
    bad = (_ulp(got, want) > 3) & ((got.float() - want.float()).abs() > 4e-3)
    assert not bad.any(), f"{int(bad.sum())} of {bad.numel()} outside tolerance, max abs {float((got.float() - want.float()).abs().max())}"


def test_attention_merge_that_gives_up_is_reported():
    """The bounded poll of the merging workgroup, forced to run out from the
    host (a bound of zero polls: every kernel still runs to its end): the
    affected output rows are NaN, the workspace's error word is set and stays
    set, AttnWorkspace.check() raises; with the built-in bound restored and a
    fresh workspace the same call is healthy again."""
    B, S, nh, nkv, hd, n_splits = 2, 400, 8, 2, 128, 4
    dev = torch.device("cuda")
    g = torch.Generator(device="cuda").manual_seed(99)
    xqkv = torch.randn(B, (nh + 2 * nkv) * hd, generator=g, device=dev).to(torch.bfloat16)
    ck = torch.randn(B, S, nkv, hd, generator=g, device=dev).to(torch.bfloat16)
    cv = torch.randn(B, S, nkv, hd, generator=g, device=dev).to(torch.bfloat16)
    pos = torch.tensor([399, 5], device=dev)  # sequence 1 sees one block of rows only: a single active split, nothing to merge
    cos, sin = decoder.rope_tables(hd, S, 500000.0, dev)
    lib = _lib.load_library()
    ws = decoder.AttnWorkspace(B, nh, nkv, n_splits, dev)
    assert ws.error() == 0
    good = decoder.attn_decode(xqkv, ck.clone(), cv.clone(), pos, cos, sin, nh, nkv, ws)
    torch.cuda.synchronize()
    assert ws.error() == 0 and not torch.isnan(good.float()).any()
    try:
        assert lib.bitnet_attn_decode_set_spin_limit(0) == 0
        bad = decoder.attn_decode(xqkv, ck.clone(), cv.clone(), pos, cos, sin, nh, nkv, ws)
        torch.cuda.synchronize()
    finally:
        lib.bitnet_attn_decode_set_spin_limit(-1)
    assert torch.isnan(bad[0].float()).all()           # every head of the sequence whose splits had to be merged
    assert torch.equal(bad[1], good[1])                # the single-split sequence is not affected
    assert ws.error() == 1
    again = decoder.attn_decode(xqkv, ck.clone(), cv.clone(), pos, cos, sin, nh, nkv, ws)
    torch.cuda.synchronize()
    assert torch.equal(again, good) and ws.error() == 1  # results recover; the word stays until someone looks
    with pytest.raises(_lib.BitLinearLibraryError):
        ws.check()
    assert ws.error() == 0                              # reported once: check() put the workspace back to its fresh state
    ws.check()
    once_more = decoder.attn_decode(xqkv, ck.clone(), cv.clone(), pos, cos, sin, nh, nkv, ws)
    torch.cuda.synchronize()
    assert torch.equal(once_more, good) and ws.error() == 0
    ws2 = decoder.AttnWorkspace(B, nh, nkv, n_splits, dev)
    fresh = decoder.attn_decode(xqkv, ck.clone(), cv.clone(), pos, cos, sin, nh, nkv, ws2)
    assert torch.equal(fresh, good) and ws2.error() == 0


def test_attention_decode_clamps_positions_outside_the_cache():
    """A position outside [0, S) must not take any access outside the buffers:
    the kernel clamps it.  Checked on outputs and buffers only: a position of
    S + 1000 (or 2^40) behaves exactly like S - 1, a negative one like 0, and
    guard rows allocated around the cache keep their bytes."""
    B, S, nh, nkv, hd = 3, 96, 8, 2, 128
    dev = torch.device("cuda")
    g = torch.Generator(device="cuda").manual_seed(31337)
    xqkv = torch.randn(B, (nh + 2 * nkv) * hd, generator=g, device=dev).to(torch.bfloat16)
    guard = 8
    big_k = torch.randn(B + 2, S + 2 * guard, nkv, hd, generator=g, device=dev).to(torch.bfloat16)
    big_v = torch.randn(B + 2, S + 2 * guard, nkv, hd, generator=g, device=dev).to(torch.bfloat16)

    def caches():
        # a contiguous [B, S, ...] cache cut out of the middle of a larger allocation
        k = big_k.clone()
        v = big_v.clone()
        flat_k = k.view(-1)[(S + 2 * guard) * nkv * hd:][: B * S * nkv * hd].view(B, S, nkv, hd)
        flat_v = v.view(-1)[(S + 2 * guard) * nkv * hd:][: B * S * nkv * hd].view(B, S, nkv, hd)
        return k, v, flat_k, flat_v

    cos, sin = decoder.rope_tables(hd, S, 500000.0, dev)
    outs = []
    for pos_list in ([S + 1000, -7, 1 << 40], [S - 1, 0, S - 1]):
        k, v, ck, cv = caches()
        pos = torch.tensor(pos_list, device=dev, dtype=torch.int64)
        ws = decoder.AttnWorkspace(B, nh, nkv, 4, dev)
        out = decoder.attn_decode(xqkv, ck, cv, pos, cos, sin, nh, nkv, ws)
        torch.cuda.synchronize()
        outs.append((out, k, v))
    (o_bad, k_bad, v_bad), (o_ok, k_ok, v_ok) = outs
    assert not torch.isnan(o_bad.float()).any()
    assert torch.equal(o_bad, o_ok)
    assert torch.equal(k_bad, k_ok) and torch.equal(v_bad, v_ok)  # same rows written, nothing outside
    # everything outside the [B, S] window is untouched
    n_front = (S + 2 * guard) * nkv * hd
    n_win = B * S * nkv * hd
    for got, src in ((k_bad, big_k), (v_bad, big_v)):
        assert torch.equal(got.view(-1)[:n_front], src.view(-1)[:n_front])
        assert torch.equal(got.view(-1)[n_front + n_win:], src.view(-1)[n_front + n_win:])


def test_host_checks_refuse_mismatched_buffers_before_any_launch():
    dev = torch.device("cuda")
    B, S, nh, nkv, hd = 2, 32, 4, 1, 128
    xqkv = torch.zeros(B, (nh + 2 * nkv) * hd, dtype=torch.bfloat16, device=dev)
    ck = torch.zeros(B, S, nkv, hd, dtype=torch.bfloat16, device=dev)
    cv = torch.zeros_like(ck)
    pos = torch.zeros(B, dtype=torch.int64, device=dev)
    cos, sin = decoder.rope_tables(hd, S, 500000.0, dev)
    ws3 = decoder.AttnWorkspace(3, nh, nkv, 2, dev)
    with pytest.raises(ValueError):
        decoder.attn_decode(xqkv, ck, cv, pos, cos, sin, nh, nkv, ws3)          # workspace of another batch
    with pytest.raises(ValueError):
        decoder.attn_decode(xqkv, ck[:1], cv[:1], pos, cos, sin, nh, nkv)       # cache of another batch
    with pytest.raises(ValueError):
        decoder.attn_decode(xqkv[:, :-128].contiguous(), ck, cv, pos, cos, sin, nh, nkv)
    mod = BitLinearKernel(256, 64).cuda()
    with pytest.raises(ValueError):
        mod(torch.zeros(2, 192, dtype=torch.bfloat16, device=dev))               # short last dimension
    with pytest.raises(TypeError):
        mod(torch.zeros(2, 256, dtype=torch.float16, device=dev))
    model = _build(SMALL, seed=5)
    gen = decoder.Generator(model, 1, 16)
    first = torch.zeros(1, dtype=torch.int64, device=dev)
    with pytest.raises(ValueError):
        gen.decode(first, 10, 8)                                                 # positions 10..17 in a cache of 16 rows


@pytest.mark.parametrize("M", [1, 2, 4, 5, 8, 40])  # every kernel that holds the norm
@pytest.mark.parametrize("K,N", [(128, 48), (1152, 128), (2560, 256), (6912, 64)])
def test_norm_bitlinear_of_rows_that_are_not_finite(M, K, N):
    """A row whose norm gives NaNs: their code is -128, whatever the number of tokens and however K falls into slices."""
    gen = torch.Generator(device="cuda").manual_seed(M + K)
    x = torch.randn(M, K, generator=gen, device="cuda").to(torch.bfloat16)
    x[0, K // 3] = float("nan")                      # every value of the row becomes NaN
    if M > 1:
        x[1, 5] = float("inf")                       # this one does, the others become zeros
        x[1, K - 1] = float("-inf")
    if M > 2:
        x[2] = 0.0
    norm = decoder.RMSNorm(K, 1e-5).cuda().to(torch.bfloat16)
    norm.weight.data = torch.rand(K, generator=gen, device="cuda").add(0.5).to(torch.bfloat16)
    lin = BitLinearKernel(K, N).cuda()
    w = torch.randint(-1, 2, (N, K), generator=gen, device="cuda", dtype=torch.int8)
    lin.weight.data = pack_weight.convert_weight_int8_to_int2(w, keep_device=True)
    lin.weight_scale.data = torch.full((4,), 0.0156, device="cuda").to(torch.bfloat16)
    got = decoder.norm_bitlinear(x, norm, lin)
    xf = x.float()
    mean = xf.double().pow(2).sum(-1, keepdim=True).float() / K
    y = (xf * (1.0 / torch.sqrt(mean + 1e-5)) * norm.weight.float()).to(torch.bfloat16).float()
    # (the row's maximum is one of bit patterns, so a NaN is the largest; the lower bound takes its place)
    amax = torch.where(torch.isnan(y).any(-1, keepdim=True), 0.0, y.nan_to_num().abs().amax(-1, keepdim=True)).clamp(min=1e-5)
    s = ((1.0 / amax) * 127.0).to(torch.bfloat16).float()
    q = torch.where(torch.isnan(y), -128.0, (y * s).nan_to_num().round().clamp(-128, 127)).double()
    want = ((q.cpu() @ w.cpu().double().T).float() / s.cpu() * lin.weight_scale[0].float().cpu()).to(torch.bfloat16)
    assert np.array_equal(host_bits(got), host_bits(want))


# ---------------------------------------------------------------------------
# The end-to-end workload at its real size: 30 layers, dim 2560, ffn 6912, 20 / 5 heads, vocabulary
# 128256 (gpu/model.py:39-49), a 512-token seeded prompt, greedy decode (gpu/generate.py:264-288)
# ---------------------------------------------------------------------------
@pytest.mark.parametrize("T", [1, 31, 33, 64, 65, 97, 129, 161])
@pytest.mark.parametrize("nh,nkv", [(1, 1), (4, 2), (20, 5), (16, 2)])
def test_prompt_attention_of_many_sequences_equals_each_alone(nh, nkv, T):
    """Rows of one to six steps through attn_prefill_kernel (many sequences: more workgroups than two per CU) and, alone, through
    attn_prefill_split_kernel; the cache rows behind the prompt, which the rings' requests reach, hold NaNs."""
    groups = (T + 15) // 16 * nkv
    B, S = 512 // groups + 2, T + 40
    gen = torch.Generator(device="cuda").manual_seed(T)
    q = torch.randn(B, T, nh, 128, generator=gen, device="cuda").to(torch.bfloat16)
    k, v = (torch.randn(B, S, nkv, 128, generator=gen, device="cuda").to(torch.bfloat16) for _ in range(2))
    k[:, T:] = v[:, T:] = float("nan")
    many = decoder.attn_prefill(q, k, v).view(B, T, -1)
    for b in (0, B // 2, B - 1):
        alone = decoder.attn_prefill(q[b : b + 1].contiguous(), k[b : b + 1].contiguous(), v[b : b + 1].contiguous())
        assert not torch.isnan(alone).any() and torch.equal(alone, many[b])


@pytest.mark.parametrize("nh,nkv,start", [(64, 16, 0), (64, 16, 21), (32, 32, 3), (64, 8, 16)])
def test_prompt_attention_at_the_edge_between_its_two_kernels(nh, nkv, start):
    """The longest prompt with two workgroups per CU and one of a block more, which goes through the other kernel: the rows that
    both have are the same bits, also where a key's infinities make scores infinite and NaN for the tokens that see it."""
    heads = min(nh // nkv, 4)
    blocks = 512 // (nh // heads)
    T, S = 16 * blocks, start + 16 * blocks + 40
    gen = torch.Generator(device="cuda").manual_seed(nh + start)
    q = torch.randn(1, T + 16, nh, 128, generator=gen, device="cuda").to(torch.bfloat16)
    k, v = (torch.randn(1, S, nkv, 128, generator=gen, device="cuda").to(torch.bfloat16) for _ in range(2))
    k[0, start + T - 70, 0, :5] = float("inf")
    k[0, start + T - 40, nkv - 1, 7] = float("-inf")
    longer = decoder.attn_prefill(q, k, v, start).view(T + 16, nh, 128)[:T]
    edge = decoder.attn_prefill(q[:, :T].contiguous(), k, v, start).view(T, nh, 128)
    assert torch.isnan(edge).any() and not torch.isnan(edge[: T - 70]).any()
    assert torch.equal(torch.isnan(edge), torch.isnan(longer))
    assert torch.equal(edge.nan_to_num(), longer.nan_to_num())


def _norm_and_linear(K, N, gen, segments=None):
    norm = decoder.RMSNorm(K, 1e-5).cuda().to(torch.bfloat16)
    norm.weight.data = torch.rand(K, generator=gen, device="cuda").add(0.5).to(torch.bfloat16)
    lin = BitLinearKernel(K, N, seg_ends=segments).cuda()
    w = torch.randint(-1, 2, (N, K), generator=gen, device="cuda", dtype=torch.int8)
    lin.weight.data = pack_weight.convert_weight_int8_to_int2(w, keep_device=True)
    lin.weight_scale.data = (0.0156 * (1.0 + 0.3 * torch.arange(4, device="cuda"))).to(torch.bfloat16)
    return norm, lin


@pytest.mark.parametrize("tile", [0, 9, 10, 11, 12])  # the instance chosen, and each of them
@pytest.mark.parametrize("B,T,nh,nkv,K,ffn,S", [(1, 17, 1, 1, 640, 16, 17), (3, 11, 2, 1, 768, 48, 70), (2, 33, 4, 2, 1280, 336, 40),
                                                (1, 129, 5, 5, 896, 1040, 200), (2, 150, 20, 5, 2560, 6912, 512)])
def test_prompt_products_with_rope_and_gate_in_the_epilogue_equal_the_separate_calls(B, T, nh, nkv, K, ffn, S, tile):
    gen = torch.Generator(device="cuda").manual_seed(B * T + ffn)
    x = torch.randn(B * T, K, generator=gen, device="cuda").to(torch.bfloat16)
    qkv_rows = [nh * 128, (nh + nkv) * 128, (nh + 2 * nkv) * 128]
    norm, wqkv = _norm_and_linear(K, qkv_rows[-1], gen, qkv_rows)
    norm2, w13 = _norm_and_linear(K, 2 * ffn, gen, [ffn, 2 * ffn])
    cos, sin = decoder.rope_tables(128, S, 500000.0, "cuda")
    # any order of positions, some of them outside the cache (clamped)
    pos = torch.stack([torch.randperm(S + 2, generator=gen, device="cuda")[:T] - 1 for _ in range(B)])
    pos[:, 1:] = torch.where((pos[:, 1:] <= 0) | (pos[:, 1:] >= S - 1), S // 2, pos[:, 1:])  # (two tokens of one row would race)
    for b in range(B):
        seen = set()
        for i, p in enumerate(pos[b].tolist()):
            while min(max(p, 0), S - 1) in seen:
                p = (p + 1) % S
            seen.add(min(max(p, 0), S - 1))
            pos[b, i] = p
    caches = [torch.randn(B, S, nkv, 128, generator=gen, device="cuda").to(torch.bfloat16) for _ in range(2)]
    got_c, want_c = [c.clone() for c in caches], [c.clone() for c in caches]
    xqkv = decoder.norm_bitlinear(x, norm, wqkv)
    want_q = decoder.rope_cache_tokens(xqkv, *want_c, pos, cos, sin, nh, nkv)
    x13 = decoder.norm_bitlinear(x, norm2, w13)
    want_h = o.squared_relu_glu_bf16(host_bits(x13))
    lib = _lib.load_library()
    try:
        if tile:
            assert lib.bitlinear_set_tuning(5, tile, 0, 0) == 0
        got_q = decoder.norm_rope_bitlinear(x, norm, wqkv, *got_c, pos, cos, sin, nh, nkv)
        got_h = decoder.norm_gate_bitlinear(x, norm2, w13)
        torch.cuda.synchronize()
    finally:
        lib.bitlinear_set_tuning(0, 0, 0, 0)
    assert (got_q is not None and got_h is not None) or tile == 0
    if got_q is not None:
        assert torch.equal(got_q.view(torch.int16), want_q.view(torch.int16))
        assert all(torch.equal(a.view(torch.int16), b.view(torch.int16)) for a, b in zip(got_c, want_c))
    if got_h is not None:
        assert np.array_equal(host_bits(got_h), want_h)


@pytest.mark.parametrize("B,T,K", [(3, 224, 2560), (3, 90, 4096)])  # 64 x 192 and 64 x 96 tiles, which have rope and not the gate
def test_prompt_products_with_rope_in_the_epilogue_of_tiles_of_three_column_tiles_a_wave(B, T, K):
    name = _lib.plan_name(0, B * T, 3840, K)
    assert "<2, 3, 1, 2, 2, 128" in name or "<2, 3, 1, 1, 4, 256" in name, name
    test_prompt_products_with_rope_and_gate_in_the_epilogue_equal_the_separate_calls(B, T, 20, 5, K, 1040, 300, 0)


@pytest.mark.parametrize("B,T,nh,nkv,K,ffn,S", [(1, 17, 1, 1, 640, 16, 17), (1, 33, 20, 5, 2560, 6912, 40), (3, 65, 20, 5, 1280, 1040, 200)])
def test_prompt_products_with_epilogues_in_64_x_64_tiles_equal_the_separate_calls(B, T, nh, nkv, K, ffn, S):
    test_prompt_products_with_rope_and_gate_in_the_epilogue_equal_the_separate_calls(B, T, nh, nkv, K, ffn, S, 13)


def test_prompt_products_that_the_epilogues_do_not_take_are_left_to_the_separate_calls():
    gen = torch.Generator(device="cuda").manual_seed(3)
    for M, K, ffn, ends in ((16, 2560, 6912, None), (512, 2496, 6912, None), (512, 2560, 6912, (6900, 13824)), (4096, 2560, 6912, None),
                            (512, 256, 64, None)):
        norm, w13 = _norm_and_linear(K, 2 * ffn, gen, ends)
        assert decoder.norm_gate_bitlinear(torch.zeros(M, K, dtype=torch.bfloat16, device="cuda"), norm, w13) is None, (M, K, ffn, ends)


@pytest.mark.parametrize("B", [1, 2])
@pytest.mark.parametrize("V,K", [(70, 512), (1000, 2560), (333, 4096), (333, 4608)])
def test_lm_head_that_normalises_its_rows_equals_the_norm_by_itself(B, V, K):
    """One and two rows of up to 4096 values are normalised inside the LM head's kernel: the logits are those of a call of
    three rows, for which the norm is a kernel of its own."""
    gen = torch.Generator(device="cuda").manual_seed(V + K)
    norm = decoder.RMSNorm(K, 1e-5).cuda().to(torch.bfloat16)
    norm.weight.data = torch.rand(K, generator=gen, device="cuda").add(0.5).to(torch.bfloat16)
    h = torch.randn(3, K, generator=gen, device="cuda").to(torch.bfloat16)
    emb = torch.randn(V, K, generator=gen, device="cuda").mul(0.05).to(torch.bfloat16)
    logits = [torch.empty(n, V, device="cuda") for n in (3, B)]
    for out in logits:
        n = out.shape[0]
        tok = decoder.lm_head_greedy(h[:n], norm, emb, decoder.LmHeadWorkspace(n, V, K, "cuda"), logits_out=out)
        assert torch.equal(tok, out.argmax(-1))
    assert torch.equal(logits[0][:B], logits[1])


@pytest.mark.parametrize("workgroups", [0, 1, 7, 600])  # 600: more than can be resident, tasks by ticket
@pytest.mark.parametrize("B,dim,ffn,nh,nkv,S,n_splits,segments", [
    (1, 128, 64, 1, 1, 33, 1, False), (2, 128, 64, 1, 1, 40, 16, False), (1, 1152, 2112, 9, 9, 70, 3, False),
    (2, 1024, 1984, 8, 1, 700, 5, False), (1, 2560, 6912, 20, 5, 545, 8, False), (2, 2560, 6912, 20, 5, 300, 8, False),
    # beyond two tokens the input rows are quantized by tasks of their own
    (3, 128, 64, 1, 1, 40, 16, False), (5, 1152, 2112, 9, 9, 70, 3, False), (8, 1024, 1984, 8, 1, 700, 5, False),
    (8, 2560, 6912, 20, 5, 545, 6, False),
    # a weight scale per sub-tensor, as a converted checkpoint has: up to eight runs of rows (here 6 and 3 of wqkv, 2 of
    # w13, whose halves meet in one task)
    (1, 2560, 6912, 20, 5, 70, 3, True), (2, 512, 2112, 4, 1, 40, 2, True), (4, 384, 64, 3, 3, 40, 2, True),
    (8, 2560, 6912, 20, 5, 70, 6, True),
])
def test_decode_stack_kernel_equals_the_kernels_per_layer(B, dim, ffn, nh, nkv, S, n_splits, workgroups, segments):
    args = decoder.ModelArgs(dim=dim, n_layers=2, n_heads=nh, n_kv_heads=nkv, vocab_size=256, ffn_dim=ffn, segment_scales=segments)
    model = _build(args, seed=dim + B)
    caches = [model.make_cache(B, S, "cuda") for _ in range(2)]
    for (k, v), (k2, v2) in zip(*caches):
        k2.copy_(k.normal_())
        v2.copy_(v.normal_())
    cos, sin = decoder.rope_tables(128, S, args.rope_theta, "cuda")
    ws = decoder.AttnWorkspace(B, nh, nkv, n_splits, "cuda")
    assert decoder.DecodeStack.applies(model, B, caches[1], n_splits)
    stack = decoder.DecodeStack(model, B, caches[1], n_splits)

    def step(i, p):
        pos = torch.full((B, 1), p, dtype=torch.int64, device="cuda")
        pos[0, 0] = min(p + 1, S - 1)
        tok = torch.arange(B, device="cuda").reshape(B, 1) + 5 * i
        want = model.decode_hidden_fused(tok, pos, caches[0], cos, sin, ws)
        h, rows = decoder.decode_step_begin(tok.reshape(B), pos.reshape(B), model.tok_embeddings.weight, cos, sin)
        got = stack(h, pos.reshape(B), rows, workgroups)
        stack.check()
        assert np.array_equal(host_bits(got), host_bits(want)), (i, p)
        for (k, v), (k2, v2) in zip(*caches):
            assert torch.equal(k, k2) and torch.equal(v, v2), (i, p)
        return h, pos.reshape(B), rows

    for i, p in enumerate([0, 30, 31, 32, S // 2, S - 1, 3]):
        operands = step(i, p)
    # a wait that runs out is reported, and the next check clears it
    if workgroups == 0:
        stack(*operands, 0, 1)
        with pytest.raises(_lib.BitLinearLibraryError, match="gave up"):
            stack.check()
        for (k, v), (k2, v2) in zip(*caches):  # that step wrote rows of its own
            k2.copy_(k)
            v2.copy_(v)
        step(9, min(33, S - 1))


@pytest.mark.parametrize("workgroups", [0, 7])
@pytest.mark.parametrize("B,dim,ffn,nh,nkv,S,V", [(1, 128, 64, 1, 1, 33, 3), (2, 1152, 2112, 9, 9, 40, 70), (3, 128, 64, 1, 1, 40, 1),
                                                  (8, 2560, 6912, 20, 5, 70, 256)])
def test_decode_stack_kernel_looks_tokens_and_positions_up_as_the_kernel_in_front_of_it(B, dim, ffn, nh, nkv, S, V, workgroups):
    """Tokens that repeat and that lie outside the embedding, positions outside the cache, a 0xffff in the embedding (which a
    published row cannot hold); tables longer than the cache take the two launches."""
    args = decoder.ModelArgs(dim=dim, n_layers=2, n_heads=nh, n_kv_heads=nkv, vocab_size=256, ffn_dim=ffn)
    model = _build(args, seed=dim + B)
    caches = [model.make_cache(B, S, "cuda") for _ in range(2)]
    for (k, v), (k2, v2) in zip(*caches):
        k2.copy_(k.normal_())
        v2.copy_(v.normal_())
    emb = torch.randn(V, dim, device="cuda").to(torch.bfloat16)
    emb.view(torch.int16)[V - 1, dim - 1] = -1
    stacks = [decoder.DecodeStack(model, B, c, 3) for c in caches]
    for rows in (S, S + 5):
        cos, sin = decoder.rope_tables(128, rows, args.rope_theta, "cuda")
        for tok, pos in (([0] * B, range(B)), (range(V - B, V), [S - 1] * B), (range(-1, B - 1), range(S - 2, S - 2 + B)),
                         ([V // 2, V, 0, V - 1, 1, V + 9, -(1 << 40), 1 << 40][:B], [-3, 31, 32, S + 4, 0, 1, 1 << 40, 5][:B])):
            tok, pos = (torch.tensor(list(t), dtype=torch.int64, device="cuda") for t in (tok, pos))
            h, factors = decoder.decode_step_begin(tok, pos, emb, cos, sin)
            want = stacks[0](h, pos, factors, workgroups)
            got = stacks[1].step(tok, pos, emb, cos, sin, workgroups)
            for stack in stacks:
                stack.check()
            assert torch.equal(torch.isnan(got), torch.isnan(want))
            same = (got.view(torch.int16) == want.view(torch.int16)) | torch.isnan(want)
            assert bool(same.all())
            for (k, v), (k2, v2) in zip(*caches):
                assert torch.equal(k.view(torch.int16), k2.view(torch.int16)) and torch.equal(v.view(torch.int16), v2.view(torch.int16))


@pytest.mark.parametrize("B,dim,ffn,nh,nkv,S,n_splits", [(1, 128, 64, 1, 1, 70, 1), (2, 1024, 1984, 8, 1, 70, 2), (8, 512, 64, 4, 1, 70, 3)])
def test_decode_stack_kernel_takes_the_new_row_at_every_place_of_a_block(B, dim, ffn, nh, nkv, S, n_splits):
    """As test_decode_stack_kernel_equals_the_kernels_per_layer, sequence after sequence over the 32 positions of a block."""
    args = decoder.ModelArgs(dim=dim, n_layers=1, n_heads=nh, n_kv_heads=nkv, vocab_size=256, ffn_dim=ffn)
    model = _build(args, seed=dim + B)
    caches = [model.make_cache(B, S, "cuda") for _ in range(2)]
    for (k, v), (k2, v2) in zip(*caches):
        k2.copy_(k.normal_())
        v2.copy_(v.normal_())
    cos, sin = decoder.rope_tables(128, S, args.rope_theta, "cuda")
    ws, stack = decoder.AttnWorkspace(B, nh, nkv, n_splits, "cuda"), decoder.DecodeStack(model, B, caches[1], n_splits)
    for p in range(32, 64):
        pos = 32 + (torch.arange(B, device="cuda") * 5 + p) % 32
        tok = torch.arange(B, device="cuda").reshape(B, 1) + 3 * p
        want = model.decode_hidden_fused(tok, pos.reshape(B, 1), caches[0], cos, sin, ws)
        h, rows = decoder.decode_step_begin(tok.reshape(B), pos, model.tok_embeddings.weight, cos, sin)
        got = stack(h, pos, rows, 0)
        stack.check()
        assert np.array_equal(host_bits(got), host_bits(want)), p
        assert all(torch.equal(x, y) for pair in zip(*caches) for x, y in zip(*pair)), p


def test_short_divisions_of_the_decode_stack_kernel_equal_the_ieee_operations():
    """Every argument in the ranges that the kernel's callers leave it (where the bits of a float end: inf and the NaNs)."""
    lib = _lib.load_library()
    found = torch.empty(3, dtype=torch.int32, device="cuda")
    stream = torch.cuda.current_stream().cuda_stream

    def bits(x):
        return int(np.float32(x).view(np.uint32))

    def compare(what, calls):
        found.copy_(torch.tensor([0, -1, 0], dtype=torch.int32))
        for by, first, n in calls:
            assert lib.bitlinear_probe_stack_math(what, by, first & 0xFFFFFFFF, n, found.data_ptr(), stream) == 0
        wrong, low, high = (v & 0xFFFFFFFF for v in found.tolist())
        assert wrong == 0, (what, wrong, hex(low), hex(high))

    def floats(low, end=1 << 31):
        return 1.0, bits(low), end - bits(low)

    compare(0, [floats(2.0**-126, bits(2.0**126) + 1), floats(float("inf"))])
    compare(1, [floats(2.0**-102)])
    compare(2, [(float(k), *floats(2.0**-115)[1:]) for k in range(64, 6912 + 1, 64)])
    # a sum of products over the scale of a row: bf16 from 127 / 2^115 to 127 / 1e-5
    largest = 128 * 6912
    lo, hi = bits(2.0**-108) >> 16, bits(127 / 1e-5) >> 16
    scales = (np.arange(lo, hi + 2, dtype=np.uint32) << 16).view(np.float32)
    compare(3, [(float(v), -largest, 2 * largest + 1) for v in scales])
    # and the comparison finds differences where there are some: reciprocals that are no normal numbers
    assert lib.bitlinear_probe_stack_math(0, 1.0, bits(2.0**126) + 1, 1000, found.data_ptr(), stream) == 0
    assert found.tolist() == [1000, bits(2.0**126) + 1, bits(2.0**126) + 1000]


def _equal_or_both_nan(a, b):
    """(Which of the NaNs is not part of a result.)"""
    return bool(torch.equal(torch.isnan(a), torch.isnan(b)) and torch.equal(a.nan_to_num(7.0), b.nan_to_num(7.0)))


@pytest.mark.parametrize("where", ["row", "value", "infinity", "last of four", "large", "all bits set"])
@pytest.mark.parametrize("B,dim,ffn,nh,nkv", [
    (1, 128, 64, 1, 1), (2, 1152, 2112, 9, 9), (1, 2560, 6912, 20, 5),
    # quantized rows between the workgroups; "last of four": the codes 0, 0, 0 and a NaN's, the word that one not yet written holds
    (3, 128, 64, 1, 1), (4, 2560, 6912, 20, 5), (5, 1152, 2112, 9, 9), (8, 2560, 6912, 20, 5),
])
def test_decode_stack_kernel_carries_values_that_are_not_finite_like_the_kernels_per_layer(B, dim, ffn, nh, nkv, where):
    S, n_splits = 70, 3
    args = decoder.ModelArgs(dim=dim, n_layers=3, n_heads=nh, n_kv_heads=nkv, vocab_size=16, ffn_dim=ffn)
    model = _build(args, seed=dim + B)
    emb = model.tok_embeddings.weight.data
    b = B - 1  # the sequence whose embedding row holds them
    if where == "row":
        emb[b] = float("nan")
    elif where == "value":
        emb[b, dim // 2 + 3] = float("nan")
    elif where == "infinity":  # the norm makes zeros of the finite values, a NaN of this one
        emb[b, 5] = float("-inf")
        emb[b, 64:72] = float("inf")
    elif where == "last of four":
        emb[b, dim // 2 + 11] = float("inf")
    elif where == "all bits set":  # the NaN that a value of the hand-over buffers holds before it is written
        emb.view(torch.int16)[b, dim // 2 : dim // 2 + 2] = -1
    else:  # the sum of squares is infinite, the values are not
        emb[b] = emb[b] * 2.0**70
    caches = [model.make_cache(B, S, "cuda") for _ in range(2)]
    for (k, v), (k2, v2) in zip(*caches):
        k2.copy_(k.normal_())
        v2.copy_(v.normal_())
    cos, sin = decoder.rope_tables(128, S, args.rope_theta, "cuda")
    ws = decoder.AttnWorkspace(B, nh, nkv, n_splits, "cuda")
    stack = decoder.DecodeStack(model, B, caches[1], n_splits)
    tok = torch.arange(B, device="cuda").reshape(B, 1)
    for p in (0, 40):
        pos = torch.full((B, 1), p, dtype=torch.int64, device="cuda")
        want = model.decode_hidden_fused(tok, pos, caches[0], cos, sin, ws)
        h, rows = decoder.decode_step_begin(tok.reshape(B), pos.reshape(B), model.tok_embeddings.weight, cos, sin)
        got = stack(h, pos.reshape(B), rows)
        stack.check()
        assert _equal_or_both_nan(got, want), p
        for (k, v), (k2, v2) in zip(*caches):
            assert _equal_or_both_nan(k, k2) and _equal_or_both_nan(v, v2), p


def _rows_whose_largest_value_is_near_a_tie(dim, norm_weight, count, eps=1e-5):
    """Rows h for which max |h g| / rms(h) lies within 2^-21 of the middle between two bf16 numbers."""
    rng = np.random.default_rng(dim)
    g = norm_weight.float().cpu().numpy()
    rows = []
    while len(rows) < count:
        h = torch.from_numpy(rng.standard_normal((20000, dim)).astype(np.float32)).to(torch.bfloat16).float().numpy()
        mean = (h.astype(np.float64) ** 2).sum(-1).astype(np.float32) / np.float32(dim)
        top = np.abs(h * g).max(-1) * (np.float32(1) / np.sqrt(mean + np.float32(eps)))
        bits = lambda x: torch.from_numpy(x.astype(np.float32)).to(torch.bfloat16).view(torch.int16).numpy()
        rows += list(h[bits(top * (1 - 2.0**-21)) != bits(top * (1 + 2.0**-21))])
    return torch.from_numpy(np.stack(rows[:count])).to(torch.bfloat16)


@pytest.mark.parametrize("where", ["tie", "large weight", "small weights", "nan weight", "zero row", "infinite weight", "overflow"])
@pytest.mark.parametrize("B,dim,ffn,nh,nkv", [(1, 128, 64, 1, 1), (2, 128, 64, 1, 1), (2, 1152, 2112, 9, 9), (3, 128, 64, 1, 1), (8, 1152, 2112, 9, 9)])
def test_decode_stack_kernel_exchanges_maxima_that_it_cannot_tell_beforehand(B, dim, ffn, nh, nkv, where):
    """Rows whose largest normalised value does not follow from max |h g| and the sum of squares alone."""
    S, n_splits = 40, 2
    args = decoder.ModelArgs(dim=dim, n_layers=2, n_heads=nh, n_kv_heads=nkv, vocab_size=16, ffn_dim=ffn)
    model = _build(args, seed=dim + B)
    emb = model.tok_embeddings.weight.data
    norms = [l.attention_norm.weight.data for l in model.layers] + [l.ffn_norm.weight.data for l in model.layers]
    if where == "tie":
        emb[:16] = _rows_whose_largest_value_is_near_a_tie(dim, norms[0], 16).cuda()
    for w in norms:
        if where == "large weight":
            w[dim // 3] = 2.0**20
            w[dim // 2] = 2.0**90
        elif where == "small weights":
            w.mul_(2.0**-75)
        elif where == "nan weight":
            w[dim // 2 + 1] = float("nan")
    if where == "zero row":
        emb[B - 1] = 0.0
    if where in ("infinite weight", "overflow"):
        # an infinite maximum: scale 0, codes 0 but for the infinity's -128, here the last of four, which beyond two tokens
        # is the word of a row not yet written.  (In front of the gate, where the quotients by a scale of 0 end as NaNs.)
        emb[:, dim // 2 + 3] = 16.0
        for layer in model.layers:
            layer.ffn_norm.weight.data[dim // 2 + 3] = float("inf") if where == "infinite weight" else 2.0**127
    caches = [model.make_cache(B, S, "cuda") for _ in range(2)]
    cos, sin = decoder.rope_tables(128, S, args.rope_theta, "cuda")
    ws = decoder.AttnWorkspace(B, nh, nkv, n_splits, "cuda")
    stack = decoder.DecodeStack(model, B, caches[1], n_splits)
    for p in range(16 // B if where == "tie" else 2):
        tok = (torch.arange(B, device="cuda") + (p * B if where == "tie" else 0)).reshape(B, 1)
        pos = torch.full((B, 1), p, dtype=torch.int64, device="cuda")
        want = model.decode_hidden_fused(tok, pos, caches[0], cos, sin, ws)
        h, rows = decoder.decode_step_begin(tok.reshape(B), pos.reshape(B), model.tok_embeddings.weight, cos, sin)
        for workgroups in (0, 3):
            got = stack(h, pos.reshape(B), rows, workgroups)
            stack.check()
            assert _equal_or_both_nan(got, want), (p, workgroups)
        for (k, v), (k2, v2) in zip(*caches):
            assert _equal_or_both_nan(k, k2) and _equal_or_both_nan(v, v2), p


@pytest.fixture(scope="module")
def model_2b():
    model = _build(decoder.ModelArgs(), seed=0)
    yield model
    del model
    torch.cuda.empty_cache()


def _rel_l2(a, b):
    return float((a.float() - b.float()).norm() / b.float().norm())


@pytest.mark.parametrize("B", [1, 8])
def test_full_size_decoder_graph_loop_equals_eager_loop(model_2b, B):
    """512-token prompt, then 128 generated tokens as the end-to-end workload names them (the first from the
    prompt pass, 127 greedy steps): the graph-replayed loop and the eager loop run the same kernels on the same
    data, so the tokens must be identical; so must a second generation from the same prompt."""
    P, G = 512, 127
    dev = torch.device("cuda")
    g = torch.Generator(device="cuda").manual_seed(1234 + B)
    prompt = torch.randint(0, model_2b.args.vocab_size, (B, P), generator=g, device=dev)
    outs = []
    for use_graph in (False, True, True):
        gen = decoder.Generator(model_2b, B, P + G + 1, use_graph=use_graph)
        assert gen.fused and gen.lm_head
        first = gen.prefill(prompt)
        toks = gen.decode(first, P, G)
        torch.cuda.synchronize()
        outs.append(torch.cat([first[None], toks]).cpu())
        del gen
    assert outs[0].shape == (G + 1, B)
    assert torch.equal(outs[0], outs[1]) and torch.equal(outs[1], outs[2])
    assert int(outs[0].min()) >= 0 and int(outs[0].max()) < model_2b.args.vocab_size
    assert torch.unique(outs[0]).numel() > 4  # not a constant stream


def _decode_step_substeps_against_glue(model, gen, tok, P):
    """One decode step at position P along the fused path (five library kernels
    per layer).  Every sub-step of every layer is also evaluated the torch-glue
    way (torch RMSNorm / gate / residual around the same BitLinear kernels; torch
    rope + fp32 attention) ON THE FUSED PATH'S INPUT of that sub-step, so that
    differences cannot travel.  Returns the fused hidden state, the glue path's
    own chained hidden state, and the worst distances seen.

    What may differ within a sub-step:
      * norm -> quantizer -> product -> epilogue [-> residual]: the same
        arithmetic on both sides except the RMSNorm's sum of squares (fp64 in the
        library, fp32 in torch's order).  The fp32 mean then differs by a few
        units in the last place, which flips the bf16 rounding of a normalised
        element with probability of about 1e-4 per element; a flipped element
        moves one int8 code by one step, an accumulator by 1 in about 1500, and
        with it roughly every sixth output of that row by one bf16 ulp.
        Asserted: relative L2 distance of the sub-step's output at most 2^-8
        (one or two flipped elements stay below half of that).
      * attention: the library kernel rounds probabilities to bf16 for the matrix
        pipe (2^-9 relative each); the glue keeps fp32.  Asserted: the bound of
        the kernel's own test, 3 bf16 ulp or 4e-3 absolute per element.
    Over a whole layer the attention's 1e-3 relative difference does NOT stay
    that small: each absmax quantizer behind it rounds to a grid of 1/127 of the
    row maximum (about 3 % of a typical element), so a perturbation far below the
    grid step flips the rounding of a share of the elements by a whole step, and
    the relu^2 gate doubles relative changes.  Measured at the 2B size: 1-3 % per
    layer.  That is the conditioning of int8 activation quantization (the same
    would separate the reference's own fp prefill from its int8 decode), not a
    property of either implementation, which is why the sub-steps are compared on
    identical inputs."""
    a = model.args
    B = tok.shape[0]
    dev = tok.device
    pos = torch.full((B, 1), P, device=dev, dtype=torch.int64)
    cos, sin = gen.cos, gen.sin
    c = cos[pos][:, :, None, :]
    s_ = sin[pos][:, :, None, :]
    mask = torch.arange(gen.max_seq, device=dev)[None, None, :] <= pos[:, :, None]
    bidx = torch.arange(B, device=dev)[:, None]
    h, rows = decoder.decode_step_begin(tok.reshape(B), pos.reshape(B), model.tok_embeddings.weight, cos, sin)
    assert torch.equal(h, model.tok_embeddings(tok.reshape(B)))
    hc = h.clone()  # the glue path's own chain
    worst = {"bitlinear": 0.0, "attention_abs": 0.0, "layer": 0.0}

    def sub(name, li, got, want):
        r = _rel_l2(got, want)
        worst["bitlinear"] = max(worst["bitlinear"], r)
        assert r <= 2.0 ** -8, f"layer {li} {name}: relative L2 distance {r}"

    def glue_attention(att, x, ck, cv):
        gk, gv = ck.clone(), cv.clone()
        q, k, v = att.split_qkv(x[:, None, :])
        q, k = decoder.apply_rope(q, c, s_), decoder.apply_rope(k, c, s_)
        gk.index_put_((bidx, pos), k)
        gv.index_put_((bidx, pos), v)
        return att.attend(q, gk, gv, mask)[:, 0], gk, gv

    for li, (layer, (ck, cv)) in enumerate(zip(model.layers, gen.cache)):
        att, ffn = layer.attention, layer.feed_forward
        # the glue path's own chain first (cache copies)
        o_c, _, _ = glue_attention(att, att.wqkv(layer.attention_norm(hc)), ck, cv)
        hc1 = hc + att.wo(att.attn_sub_norm(o_c))
        hc = hc1 + ffn(layer.ffn_norm(hc1))
        # fused sub-steps, each against the glue evaluation of the same input
        h_in = h
        xqkv = decoder.norm_bitlinear(h, layer.attention_norm, att.wqkv)
        sub("wqkv", li, xqkv, att.wqkv(layer.attention_norm(h)))
        o_g, gk, gv = glue_attention(att, xqkv, ck, cv)
        o_f = decoder.attn_decode(xqkv, ck, cv, pos.reshape(B), cos, sin, a.n_heads, a.n_kv_heads, gen.attn_ws, rope_rows=rows)
        assert torch.equal(ck, gk) and torch.equal(cv, gv), f"layer {li}: cache rows"
        bad = (_ulp(o_f, o_g) > 3) & ((o_f.float() - o_g.float()).abs() > 4e-3)
        worst["attention_abs"] = max(worst["attention_abs"], float((o_f.float() - o_g.float()).abs().max()))
        assert not bad.any(), f"layer {li} attention: {int(bad.sum())} of {bad.numel()} outside tolerance"
        h1 = decoder.norm_bitlinear(o_f, att.attn_sub_norm, att.wo, residual=h)
        sub("wo + residual", li, h1, h + att.wo(att.attn_sub_norm(o_f)))
        x13 = decoder.norm_bitlinear(h1, layer.ffn_norm, ffn.w13)
        sub("w13", li, x13, ffn.w13(layer.ffn_norm(h1)))
        h = decoder.norm_bitlinear(x13, ffn.ffn_sub_norm, ffn.w2, glu=True, residual=h1)
        x1, x3 = x13.chunk(2, -1)
        sub("w2 + residual", li, h, h1 + ffn.w2(ffn.ffn_sub_norm(torch.relu(x1) ** 2 * x3)))
        # the whole glue layer on the fused layer's input, for the record
        o_l, _, _ = glue_attention(att, att.wqkv(layer.attention_norm(h_in)), ck, cv)
        hl = h_in + att.wo(att.attn_sub_norm(o_l))
        hl = hl + ffn(layer.ffn_norm(hl))
        worst["layer"] = max(worst["layer"], _rel_l2(h, hl))
    gen.attn_ws.check()
    return h, hc, worst


@pytest.mark.parametrize("B", [1, 8])
def test_full_size_decode_step_substeps_against_the_torch_glue(model_2b, B):
    """Position 512 of the full-size model after the 512-token prompt: all 30 x 5
    sub-steps of the fused decode step against the torch glue on identical
    inputs (bounds: see _decode_step_substeps_against_glue), the library's LM head
    against the argmax of torch logits, and, end to end over the 30 layers, the
    two paths' logits still pointing the same way (cosine above 0.9: per layer the
    quantizers amplify the attention's rounding to 1-3 %, see above)."""
    P = 512
    dev = torch.device("cuda")
    g = torch.Generator(device="cuda").manual_seed(4321 + B)
    prompt = torch.randint(0, model_2b.args.vocab_size, (B, P), generator=g, device=dev)
    gen = decoder.Generator(model_2b, B, P + 8)
    first = gen.prefill(prompt)
    h, hc, worst = _decode_step_substeps_against_glue(model_2b, gen, first.view(B, 1), P)
    logits_f = model_2b.output(model_2b.norm(h)).float()
    logits_g = model_2b.output(model_2b.norm(hc)).float()
    cosine = torch.nn.functional.cosine_similarity(logits_f, logits_g, dim=-1)
    print(f"full-size step, batch {B}: worst BitLinear sub-step relative L2 {worst['bitlinear']:.2e}, worst attention "
          f"|diff| {worst['attention_abs']:.2e}, worst whole-layer relative L2 {worst['layer']:.2e}, logits cosine "
          f"{float(cosine.min()):.4f}, relative L2 {_rel_l2(logits_f, logits_g):.3f}")
    assert float(cosine.min()) > 0.9
    # the library's LM head on the fused hidden state: its greedy token is the argmax of these logits
    tok_lib = decoder.lm_head_greedy(h, model_2b.norm, model_2b.output.weight, gen.lm_ws)
    top2 = torch.topk(logits_f, 2, dim=-1).values
    clear = (top2[:, 0] - top2[:, 1]) > 2e-2  # rows whose best logit is not a near tie
    assert torch.equal(tok_lib[clear], torch.argmax(logits_f, dim=-1)[clear])


def test_decoder_loaded_from_a_gguf_file_gives_the_same_logits(tmp_path):
    """A decoder written out as a GGUF file with I2_S projections (the CPU stack's format) and read back
    through the transcoder computes, prompt and decode step, what the original computes: the packed bytes,
    the scale slots and the norms survive the trip bit for bit, so the logits are equal."""
    from bitnet_amd import gguf

    model = _build(SMALL, seed=4)
    state = {k: v.detach().cpu() for k, v in model.state_dict().items()}
    path = str(tmp_path / "small.gguf")
    gguf.int2_state_to_gguf(state, SMALL, path, embed_dtype=torch.bfloat16)
    with gguf.GGUFReader(path) as r:
        args = gguf.model_args_from_gguf(r)
        back = gguf.gguf_to_int2_state(r)
    assert args == SMALL
    for k, v in state.items():
        assert torch.equal(back[k], v), k
    clone = _build(args, seed=9)  # other weights, then overwritten by the file's
    clone.load_state_dict(back, strict=True)
    B, P, S = 2, 20, 32
    dev = torch.device("cuda")
    cos, sin = decoder.rope_tables(SMALL.dim // SMALL.n_heads, S, SMALL.rope_theta, dev)
    g = torch.Generator(device="cuda").manual_seed(8)
    prompt = torch.randint(0, SMALL.vocab_size, (B, P), generator=g, device=dev)
    pos = torch.arange(P, device=dev)[None].expand(B, P).contiguous()
    c1, c2 = model.make_cache(B, S, dev), clone.make_cache(B, S, dev)
    l1 = model.forward_tokens(prompt, pos, c1, cos, sin)
    l2 = clone.forward_tokens(prompt, pos, c2, cos, sin)
    assert torch.equal(l1, l2) and bool(torch.isfinite(l1).all())
    tok = torch.argmax(l1[:, -1], dim=-1).view(B, 1)
    p1 = torch.full((B, 1), P, device=dev)
    assert torch.equal(model.forward_tokens(tok, p1, c1, cos, sin), clone.forward_tokens(tok, p1, c2, cos, sin))


def test_generate_all_with_ragged_prompts_equals_one_sequence_at_a_time():
    """FastGen.generate_all semantics (gpu/generate.py:217-304): prompts of different lengths in one batch,
    padded on the right.  Every per-token operation is independent of the other rows and the attention of a
    sequence only sees its own cache rows up to its own position, so each answer equals what the same prompt
    generates alone -- on the fused path (graph replays) and on the torch-glue path."""
    model = _build(BIG_HEADS, seed=5)
    assert decoder.Generator(model, batch=3, max_seq=64).lm_head  # head_dim 128: the folded calls and the library's LM head
    g = torch.Generator().manual_seed(3)
    prompts = [torch.randint(2, BIG_HEADS.vocab_size, (n,), generator=g).tolist() for n in (19, 7, 33)]
    gen = 12
    for fused in (True, False):
        batch = decoder.Generator(model, batch=3, max_seq=64, use_graph=fused, fused=fused)
        answers = batch.generate_all(prompts, gen)
        assert [len(a) for a in answers] == [gen] * 3
        for b, q in enumerate(prompts):
            alone = decoder.Generator(model, batch=1, max_seq=64, use_graph=fused, fused=fused)
            assert alone.generate_all([q], gen) == [answers[b]], (fused, b)
    with pytest.raises(ValueError):
        batch.generate_all(prompts[:2], gen)
    with pytest.raises(ValueError):
        batch.generate_all(prompts, 64)
    with pytest.raises(ValueError):
        batch.generate_all([[BIG_HEADS.vocab_size], [1], [1]], 4)


def test_generate_all_stops_at_the_end_token_and_trims_the_answers():
    model = _build(BIG_HEADS, seed=6)
    g = torch.Generator().manual_seed(4)
    prompts = [torch.randint(2, BIG_HEADS.vocab_size, (n,), generator=g).tolist() for n in (9, 14)]
    gen = decoder.Generator(model, batch=2, max_seq=48)
    full = gen.generate_all(prompts, 16)
    # take a token that sequence 1 produces at step 5 as the end token
    eos = full[1][5]
    # the loop ends after the first DECODE step (index >= 1) in which any sequence produced it: a hit in the
    # prompt pass's own token does not end the batch (gpu/generate.py:262-284)
    first_hit = min([a.index(eos, 1) for a in full if eos in a[1:]] + [15])
    timings = {}
    cut = gen.generate_all(prompts, 16, eos_id=eos, timings=timings)
    assert timings["decode_tokens"] == 2 * (len(max(cut, key=len)) - 1) or timings["decode_tokens"] == 2 * first_hit
    assert timings["prefill_s"] > 0 and timings["decode_s"] > 0 and timings["decode_tokens_per_s"] > 0
    for a, f in zip(cut, full):
        want = f[: first_hit + 1]           # the loop ends after the first step in which any sequence hit it
        if eos in want:
            want = want[: want.index(eos) + 1]
        assert a == want
    assert cut[1][-1] == eos or eos in cut[0]
    # the end token as the very first token of sequence 0 (out of the prompt pass): that sequence's answer is the end
    # token alone, the other sequence goes on as if nothing had happened, until a decode step produces the token
    eos0 = full[0][0]
    cut0 = gen.generate_all(prompts, 16, eos_id=eos0)
    assert cut0[0] == [eos0]
    hit = min([a.index(eos0, 1) for a in full if eos0 in a[1:]] + [15])
    want1 = full[1][: hit + 1]
    if eos0 in want1:
        want1 = want1[: want1.index(eos0) + 1]
    assert cut0[1] == want1 and len(cut0[1]) > 1


@pytest.mark.parametrize("use_graph", [True, False])
@pytest.mark.parametrize("sample", [False, True])
def test_steps_awaited_by_their_tokens_end_where_steps_awaited_by_the_stream_do(sample, use_graph):
    """With an end token the host waits for a step's tokens in host memory: directly behind steps that nobody waited for,
    with waits that run out at once (from then on the stream is waited for), and for end tokens of the first, a middle and no step."""
    model = _build(BIG_HEADS, seed=16)
    gen = decoder.Generator(model, batch=2, max_seq=64, use_graph=use_graph)
    prompts = [[5, 9, 2, 44, 7], [3, 1, 8]]
    first, lens = torch.tensor([4, 9], device="cuda"), torch.tensor([5, 3], device="cuda")

    def answers(**kw):
        gen.decode(first, lens, 20)  # still under way when the next call starts
        return gen.generate_all(prompts, 20, use_sampling=sample, rng=torch.Generator(device="cuda").manual_seed(3), **kw)

    full = answers()
    for eos in (full[0][1], full[1][9], 10**6):
        gen._await = True
        got = answers(eos_id=eos)
        assert gen._await
        gen.kAwaitUs = 0  # a wait that is not over at once gives up
        assert answers(eos_id=eos) == got
        del gen.kAwaitUs
        gen._await = False
        assert answers(eos_id=eos) == got
        steps = next((t for t in range(1, 20) if any(f[t] == eos for f in full)), 19)
        assert max(len(a) for a in got) <= steps + 1


@pytest.mark.parametrize("sample", [False, True])
def test_a_late_step_costs_the_call_it_is_in_its_waits_for_tokens_and_no_later_call(sample, monkeypatch):
    model = _build(BIG_HEADS, seed=16)
    gen = decoder.Generator(model, batch=1, max_seq=64)
    calls, late, host = [], [], _lib.host_calls()
    real = host.await_words
    monkeypatch.setattr(host, "await_words", lambda *args: calls.append(1) or (real(*args) and len(calls) not in late))

    def answer():
        calls.clear()
        rng = torch.Generator(device="cuda").manual_seed(3)
        return gen.generate_all([[5, 9, 2]], 10, use_sampling=sample, eos_id=10**6, rng=rng), len(calls)

    want = answer()
    assert want[1] == 8  # every step of nine but the first
    late.append(3)
    assert answer() == (want[0], 3)
    late.clear()
    assert answer() == want


def test_generate_all_sampling_is_reproducible_and_greedy_for_a_tiny_nucleus():
    model = _build(BIG_HEADS, seed=7)
    g = torch.Generator().manual_seed(5)
    prompts = [torch.randint(2, BIG_HEADS.vocab_size, (n,), generator=g).tolist() for n in (11, 6)]
    gen = decoder.Generator(model, batch=2, max_seq=40)
    a = gen.generate_all(prompts, 10, use_sampling=True, rng=torch.Generator(device="cuda").manual_seed(11))
    b = gen.generate_all(prompts, 10, use_sampling=True, rng=torch.Generator(device="cuda").manual_seed(11))
    c = gen.generate_all(prompts, 10, use_sampling=True, rng=torch.Generator(device="cuda").manual_seed(12))
    assert a == b and all(0 <= t < BIG_HEADS.vocab_size for ans in a for t in ans)
    assert a != c  # 20 draws at temperature 0.7 from a 512-token vocabulary
    # a nucleus that only holds the most likely token: the greedy answer (the draw is from the bf16-rounded
    # logits the LM head returns, the greedy token from the same values)
    greedy = gen.generate_all(prompts, 10)
    tiny = gen.generate_all(prompts, 10, use_sampling=True, top_p=1e-9, rng=torch.Generator(device="cuda").manual_seed(1))
    assert tiny == greedy


def test_captured_prompt_pass_equals_the_launch_by_launch_one():
    """Generator.prefill replays one captured graph per bucket of prompt lengths (multiples of 32 tokens, the
    prompt padded up to the bucket); every replay, with other work of the program in between (decode steps,
    prompts of other lengths), gives the tokens, and leaves the cache rows, of the unpadded pass issued launch by
    launch.  Beyond kMaxPrefillGraphs captured passes the least recently used one is dropped."""
    model = _build(BIG_HEADS, seed=8)
    dev = torch.device("cuda")
    g = torch.Generator(device="cuda").manual_seed(21)
    graphed = decoder.Generator(model, batch=2, max_seq=96, use_graph=True)
    eager = decoder.Generator(model, batch=2, max_seq=96, use_graph=False)
    assert graphed.lm_head and eager.lm_head
    for rnd, P in enumerate((24, 40, 24, 24, 7, 40)):
        prompt = torch.randint(0, BIG_HEADS.vocab_size, (2, P), generator=g, device=dev)
        t1 = graphed.prefill(prompt)
        t2 = eager.prefill(prompt)
        assert torch.equal(t1, t2), (rnd, P)
        for (k1, v1), (k2, v2) in zip(graphed.cache, eager.cache):
            assert torch.equal(k1[:, :P], k2[:, :P]) and torch.equal(v1[:, :P], v2[:, :P])
        # the program's own work between two replays
        d1 = graphed.decode(t1, P, 5)
        d2 = eager.decode(t2, P, 5)
        assert torch.equal(d1, d2)
    assert sorted(k[0] for k in graphed._pf_graphs) == [32, 64]  # 7 and 24 share a pass, 40 has the other
    # a bucket cut short by the cache's capacity, and the bound on the passes kept
    graphed.kMaxPrefillGraphs = 2
    prompt = torch.randint(0, BIG_HEADS.vocab_size, (2, 70), generator=g, device=dev)
    assert torch.equal(graphed.prefill(prompt), eager.prefill(prompt))
    assert [k[0] for k in graphed._pf_graphs] == [64, 96]  # 32, replayed longest ago, made room
    prompt = torch.randint(0, BIG_HEADS.vocab_size, (2, 9), generator=g, device=dev)
    assert torch.equal(graphed.prefill(prompt), eager.prefill(prompt))
    assert [k[0] for k in graphed._pf_graphs] == [96, 32]
    graphed.kMaxPrefillGraphs = 12
    # ragged prompts go through the same captured pass with their own lengths
    prompts = [torch.randint(2, BIG_HEADS.vocab_size, (n,), generator=torch.Generator().manual_seed(n)).tolist() for n in (40, 13)]
    assert graphed.generate_all(prompts, 6) == eager.generate_all(prompts, 6)
    prompts = [prompts[1], prompts[0]]
    assert graphed.generate_all(prompts, 6) == eager.generate_all(prompts, 6)


# ---------------------------------------------------------------------------
# A converted Hugging Face checkpoint through the decoder (gpu/convert_safetensors.py:43-93,
# gpu/convert_checkpoint.py:29-32, 42-77)
# ---------------------------------------------------------------------------
HF_ARGS = decoder.ModelArgs(dim=512, n_layers=2, n_heads=4, n_kv_heads=2, vocab_size=320, ffn_dim=768, segment_scales=True)


def _hf_checkpoint(args, seed):
    """Synthetic tensors under the Hugging Face names, bf16 like the published master weights; q, k and v
    projections of clearly different magnitude, so that their three weight scales differ by factors."""
    g = torch.Generator().manual_seed(seed)
    hd = args.dim // args.n_heads
    r = lambda std, *shape: (torch.randn(*shape, generator=g) * std).to(torch.bfloat16)
    st = {}
    for layer in range(args.n_layers):
        b = f"model.layers.{layer}."
        st[b + "self_attn.q_proj.weight"] = r(0.02, args.n_heads * hd, args.dim)
        st[b + "self_attn.k_proj.weight"] = r(0.06, args.n_kv_heads * hd, args.dim)
        st[b + "self_attn.v_proj.weight"] = r(0.009, args.n_kv_heads * hd, args.dim)
        st[b + "self_attn.o_proj.weight"] = r(0.02, args.dim, args.n_heads * hd)
        st[b + "input_layernorm.weight"] = 1 + r(0.1, args.dim)
        st[b + "post_attention_layernorm.weight"] = 1 + r(0.1, args.dim)
        st[b + "self_attn.attn_sub_norm.weight"] = 1 + r(0.1, args.dim)
        st[b + "mlp.ffn_sub_norm.weight"] = 1 + r(0.1, args.ffn_dim)
        st[b + "mlp.gate_proj.weight"] = r(0.03, args.ffn_dim, args.dim)
        st[b + "mlp.up_proj.weight"] = r(0.015, args.ffn_dim, args.dim)
        st[b + "mlp.down_proj.weight"] = r(0.02, args.dim, args.ffn_dim)
    st["model.embed_tokens.weight"] = r(0.5, args.vocab_size, args.dim)
    st["model.norm.weight"] = 1 + r(0.1, args.dim)
    return st


def _hf_convention_logits(st, args, ids):
    """The model the checkpoint describes, evaluated the way the Hugging Face side of the reference's converter
    sees it, in plain torch: projections kept apart and in their original row order, rotary embedding on the two
    halves of a head (rotate_half), every BitLinear as the reference's fp module (activations snapped to the int8
    grid, gpu/model.py:77-85, times weights ternarised and dequantised per tensor, gpu/convert_checkpoint.py:29-32),
    sub-norms and squared-ReLU gate as gpu/model.py:159-160, 195-196.  fp32 arithmetic, rounded to bf16 where the
    decoder's tensors are bf16.  ids [B, T] -> logits fp32 [B, T, vocab]."""
    dev = ids.device
    bf = torch.bfloat16
    hd = args.dim // args.n_heads
    rep = args.n_heads // args.n_kv_heads
    B, T = ids.shape
    w = {k: v.to(dev) for k, v in st.items()}

    def rms(x, g):
        xf = x.float()
        return (xf * torch.rsqrt(xf.pow(2).mean(-1, keepdim=True) + args.norm_eps) * g.float()).to(bf)

    def deq(t):  # convert_checkpoint.py:29-32, in the checkpoint's dtype
        s = 1.0 / t.abs().mean().clamp_(min=1e-5)
        return ((t * s).round().clamp(-1, 1) / s).float()

    def bitlinear_fp(x, t):  # gpu/model.py:77-85
        xf = x.float()
        s = 127 / xf.abs().max(dim=-1, keepdim=True).values.clamp_(min=1e-5)
        return (((xf * s).round().clamp(-128, 127) / s) @ deq(t).T).to(bf)

    inv = 1.0 / (args.rope_theta ** (torch.arange(0, hd, 2, device=dev, dtype=torch.float32) / hd))
    ang = torch.outer(torch.arange(T, device=dev, dtype=torch.float32), inv)
    cos = torch.cat([ang.cos(), ang.cos()], dim=-1)[None, :, None, :]  # [1, T, 1, hd]: frequency i at i and i + hd/2
    sin = torch.cat([ang.sin(), ang.sin()], dim=-1)[None, :, None, :]

    def rope_half(x):  # x [B, T, heads, hd]
        xf = x.float()
        x1, x2 = xf[..., : hd // 2], xf[..., hd // 2 :]
        return (xf * cos + torch.cat([-x2, x1], dim=-1) * sin).to(bf)

    h = w["model.embed_tokens.weight"][ids]  # [B, T, dim] bf16
    causal = torch.ones(T, T, dtype=torch.bool, device=dev).tril()
    for layer in range(args.n_layers):
        b = f"model.layers.{layer}."
        x = rms(h, w[b + "input_layernorm.weight"])
        q = rope_half(bitlinear_fp(x, w[b + "self_attn.q_proj.weight"]).view(B, T, args.n_heads, hd))
        k = rope_half(bitlinear_fp(x, w[b + "self_attn.k_proj.weight"]).view(B, T, args.n_kv_heads, hd))
        v = bitlinear_fp(x, w[b + "self_attn.v_proj.weight"]).view(B, T, args.n_kv_heads, hd)
        k = k.repeat_interleave(rep, dim=2).float()  # query head j reads kv head j // rep
        v = v.repeat_interleave(rep, dim=2).float()
        sc = torch.einsum("bthd,bshd->bhts", q.float(), k) * hd ** -0.5
        sc = sc.masked_fill(~causal[None, None], float("-inf"))
        o = torch.einsum("bhts,bshd->bthd", torch.softmax(sc, dim=-1), v).reshape(B, T, args.dim).to(bf)
        h = (h.float() + bitlinear_fp(rms(o, w[b + "self_attn.attn_sub_norm.weight"]), w[b + "self_attn.o_proj.weight"]).float()).to(bf)
        x = rms(h, w[b + "post_attention_layernorm.weight"])
        gate = bitlinear_fp(x, w[b + "mlp.gate_proj.weight"])
        up = bitlinear_fp(x, w[b + "mlp.up_proj.weight"])
        inner = ((torch.relu(gate.float()) ** 2).to(bf).float() * up.float()).to(bf)
        h = (h.float() + bitlinear_fp(rms(inner, w[b + "mlp.ffn_sub_norm.weight"]), w[b + "mlp.down_proj.weight"]).float()).to(bf)
    return rms(h, w["model.norm.weight"]).float() @ w["model.embed_tokens.weight"].float().T


def _load_converted(path, args):
    with torch.device("cuda"):
        prev = torch.get_default_dtype()
        torch.set_default_dtype(torch.bfloat16)
        try:
            model = decoder.Transformer(args)
        finally:
            torch.set_default_dtype(prev)
    model.load_state_dict(torch.load(path, weights_only=True), strict=True)
    return model


def test_converted_hf_checkpoint_runs_through_the_decoder_like_the_hf_convention_model(tmp_path):
    """Row (f3) on the device: synthetic Hugging Face tensors -> convert_hf_checkpoint (rotary row permutation,
    q|k|v and gate|up fusing, per-sub-tensor ternarisation, four-slot scales, packing) -> strict load into the
    decoder -> prompt pass and decode step through the library's int8 kernels with the segment scale rule.  The
    yardstick never sees a fused, permuted or packed tensor: it evaluates the unfused projections with half-split
    rotary embedding and the reference's fp BitLinear.  Attention scores are invariant under the permutation
    (q and k are permuted alike within a head), and the int8 path differs from the fp module only in where
    roundings fall (same integer products; tests/test_gpu_bitlinear.py::test_fp_path_agrees_with_the_int8_path
    derives the per-call bound), so the logits agree up to the amplification of those roundings by the later
    quantizers: a few percent of the logits' norm.  A wrong row order, segment boundary or scale slot moves them
    by tens of percent -- the control at the end runs the same file with the reference kernel's slot rule
    n // (N // ws_num) (bitnet_kernels.h:80; one slot for a shape outside its table, so k and v rows are scaled
    by s_q) and must land far outside the bound."""
    from safetensors.torch import save_file

    from bitnet_amd import checkpoint

    args = HF_ARGS
    st = _hf_checkpoint(args, seed=11)
    src = str(tmp_path / "model.safetensors")
    save_file(st, src)
    path = checkpoint.convert_hf_checkpoint(src, str(tmp_path / "out"), args)
    model = _load_converted(path, args)
    for lr in model.layers:  # the three scales of a fused wqkv really differ, else the control below proves nothing
        s3 = lr.attention.wqkv.weight_scale.float()
        assert float(s3[1] / s3[0]) > 2.0 and float(s3[0] / s3[2]) > 1.5 and float(s3[3]) == 0.0

    dev = torch.device("cuda")
    B, T, S = 2, 48, 64
    g = torch.Generator(device="cuda").manual_seed(12)
    ids = torch.randint(0, args.vocab_size, (B, T + 1), generator=g, device=dev)
    want = _hf_convention_logits(st, args, ids)  # [B, T + 1, V]

    @torch.no_grad()
    def run(m):
        cos, sin = decoder.rope_tables(args.dim // args.n_heads, S, args.rope_theta, dev)
        cache = m.make_cache(B, S, dev)
        hid = m.prefill_hidden_fused(ids[:, :T].contiguous(), cache, cos, sin)  # quantizer kernels + int8 MFMA GEMM
        prompt_logits = m.output(m.norm(hid)).float()
        ws = decoder.AttnWorkspace(B, args.n_heads, args.n_kv_heads, 8, dev)
        pos = torch.full((B, 1), T, device=dev)
        step_logits = m.forward_decode_fused(ids[:, T:].contiguous(), pos, cache, cos, sin, ws)  # one-kernel forwards
        ws.check()
        # the unfused glue (BitLinearKernel.forward per projection) on the same prompt
        glue = m.forward_tokens(ids[:, :T].contiguous(), torch.arange(T, device=dev)[None].expand(B, T).contiguous(),
                                m.make_cache(B, S, dev), cos, sin)
        torch.cuda.synchronize()
        return torch.cat([prompt_logits, step_logits], dim=1), glue

    rel = lambda a, b: float((a - b).norm() / b.norm())
    got, glue = run(model)
    assert bool(torch.isfinite(got).all())
    err_prompt, err_step, err_glue = rel(got[:, :T], want[:, :T]), rel(got[:, T:], want[:, T:]), rel(glue, want[:, :T])
    bound = 0.035  # measured 0.017-0.020 over three seeds
    assert err_prompt < bound and err_step < bound and err_glue < bound, (err_prompt, err_step, err_glue)
    top = want.topk(2, dim=-1).values
    clear = (top[..., 0] - top[..., 1]) > 0.15 * want.std()
    assert int(clear.sum()) > 10
    assert torch.equal(got.argmax(-1)[clear], want.argmax(-1)[clear])

    # control: the same file through the reference kernel's slot rule
    import dataclasses

    thirds = _load_converted(path, dataclasses.replace(args, segment_scales=False))
    got3, _ = run(thirds)
    assert rel(got3, want) > 2 * bound, rel(got3, want)  # measured 0.094-0.112

    # control: a converter that forgot the rotary row permutation of q and k (convert_safetensors.py:43-47)
    state = checkpoint.hf_to_model_state(st, args)
    hd = args.dim // args.n_heads
    for layer in range(args.n_layers):
        b = f"model.layers.{layer}.self_attn."
        state[f"layers.{layer}.attention.wqkv.weight"] = torch.cat(
            [st[b + "q_proj.weight"], st[b + "k_proj.weight"], st[b + "v_proj.weight"]], dim=0)
    bad = str(tmp_path / "unpermuted.pt")
    torch.save(checkpoint.model_state_to_int2(state, args), bad)
    got_bad, _ = run(_load_converted(bad, args))
    assert rel(got_bad, want) > 2 * bound, rel(got_bad, want)
