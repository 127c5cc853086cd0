"""Attention for head sizes other than 128 (attn<T>, src/csrc/llm/attn.cpp:781-955, is generic in the head size):
the kernels behind tppx_attn_decode / tppx_attn_prefill for those sizes, against the oracle (tolerance as for the 128-wide
kernels: rel-L2 5e-3, max-abs 2^-7 of the largest output) and plain PyTorch fp32 softmax attention (1e-2), and a
decoder layer with 64-wide heads against the oracle composition."""
import numpy as np
import pytest
import torch

import oracle as O
from util import t2bits, randn_bf16, block_bf16, bits2f, assert_close_bf16
from test_gpu_decoder import _attn, _attn_prefill, _llm

pytestmark = pytest.mark.gpu


def _close(got, ref, torch_ref):
    g, r = bits2f(t2bits(got)).astype(np.float64), bits2f(ref).astype(np.float64)
    assert np.isfinite(g).all()
    assert np.sqrt(((g - r) ** 2).sum() / (r ** 2).sum()) <= 5e-3
    assert np.abs(g - r).max() <= 2.0 ** -7 * np.abs(r).max()
    assert np.sqrt(((g - torch_ref) ** 2).sum() / (torch_ref ** 2).sum()) <= 1e-2


@pytest.mark.parametrize("H", [64, 96, 256, 8, 200])
@pytest.mark.parametrize("B,Nq,Nkv,L,Smax", [(3, 8, 2, 77, 128), (2, 4, 4, 1, 64), (1, 8, 8, 300, 320), (2, 2, 1, 64, 64)])
def test_attn_decode_other_head_sizes(H, B, Nq, Nkv, L, Smax):
    F = _llm()
    q = randn_bf16((B, Nq, H), 1.0, 31 + H)
    k = randn_bf16((B, Nkv, Smax, H), 1.0, 32 + H)
    v = randn_bf16((B, Nkv, Smax, H), 1.0, 33 + H)
    k[:, :, L:] = float("nan")  # rows past the valid length must not reach the output
    v[:, :, L:] = float("nan")
    got = _attn(F, q.cuda(), k.cuda(), v.cuda(), L)
    ref = O.attn_decode(t2bits(q), t2bits(k[:, :, :L]), t2bits(v[:, :, :L]))
    kk = k[:, :, :L].float().repeat_interleave(Nq // Nkv, dim=1)
    vv = v[:, :, :L].float().repeat_interleave(Nq // Nkv, dim=1)
    s = torch.einsum("bnh,bnlh->bnl", q.float(), kk) / np.sqrt(float(H))
    t = torch.einsum("bnl,bnlh->bnh", torch.softmax(s, -1), vv).numpy().astype(np.float64)
    _close(got, ref, t)


def test_attn_decode_other_head_size_with_mask():
    F = _llm()
    B, Nq, L, Smax, H = 2, 4, 100, 128, 64
    q = randn_bf16((B, Nq, H), 1.0, 41)
    k = randn_bf16((B, Nq, Smax, H), 1.0, 42)
    v = randn_bf16((B, Nq, Smax, H), 1.0, 43)
    keep = torch.ones(B, L, dtype=torch.int64)
    keep[0, :17] = 0  # left padding of sequence 0
    mask = F.TppCache(Smax).align_and_invert_mask(keep.to(torch.bfloat16))
    got = _attn(F, q.cuda(), k.cuda(), v.cuda(), L, mask=mask.cuda())
    ref = O.attn_decode(t2bits(q), t2bits(k[:, :, :L]), t2bits(v[:, :, :L]), mask.float().numpy())
    g, r = bits2f(t2bits(got)).astype(np.float64), bits2f(ref).astype(np.float64)
    assert np.isfinite(g).all()
    assert np.sqrt(((g - r) ** 2).sum() / (r ** 2).sum()) <= 5e-3


@pytest.mark.parametrize("H", [64, 80, 256, 8, 200])
@pytest.mark.parametrize("B,Nq,Nkv,L,Smax", [(1, 4, 2, 700, 1024), (2, 8, 8, 100, 1024), (1, 2, 1, 1000, 1000)])
def test_attn_decode_other_head_sizes_split_key_range(H, B, Nq, Nkv, L, Smax, monkeypatch):
    """Caches of 512 keys and more: the key range is dealt to several workgroups per query (some of them past the
    valid length, leaving empty states) and merged by a second launch; one split gives the same answer up to the
    order of the sums."""
    F = _llm()
    q = randn_bf16((B, Nq, H), 1.0, 131 + H)
    k = randn_bf16((B, Nkv, Smax, H), 1.0, 132 + H)
    v = randn_bf16((B, Nkv, Smax, H), 1.0, 133 + H)
    k[:, :, L:] = float("nan")
    v[:, :, L:] = float("nan")
    got = _attn(F, q.cuda(), k.cuda(), v.cuda(), L)
    ref = O.attn_decode(t2bits(q), t2bits(k[:, :, :L]), t2bits(v[:, :, :L]))
    kk = k[:, :, :L].float().repeat_interleave(Nq // Nkv, dim=1)
    vv = v[:, :, :L].float().repeat_interleave(Nq // Nkv, dim=1)
    s = torch.einsum("bnh,bnlh->bnl", q.float(), kk) / np.sqrt(float(H))
    t = torch.einsum("bnl,bnlh->bnh", torch.softmax(s, -1), vv).numpy().astype(np.float64)
    _close(got, ref, t)
    monkeypatch.setenv("TPPX_ATTN_GENERIC_SPLITS", "1")
    one = _attn(F, q.cuda(), k.cuda(), v.cuda(), L)
    _close(one, ref, t)
    monkeypatch.setenv("TPPX_ATTN_GENERIC_SPLITS", "5")
    five = _attn(F, q.cuda(), k.cuda(), v.cuda(), L)
    _close(five, ref, t)
    none = _attn(F, q.cuda(), k.cuda(), v.cuda(), L, ws=False)  # no workspace: one split
    assert torch.equal(none, one)


@pytest.mark.parametrize("H", [64, 80, 96, 256, 8, 200])
@pytest.mark.parametrize("B,S,Nq,Nkv,past,Smax", [(1, 130, 4, 4, 0, 256), (2, 77, 8, 2, 0, 128), (2, 5, 4, 4, 100, 128), (3, 1, 4, 2, 40, 64)])
def test_attn_prefill_other_head_sizes(H, B, S, Nq, Nkv, past, Smax):
    _llm()
    L = past + S
    q = randn_bf16((B, S, Nq, H), 1.0, 51 + H)
    k = randn_bf16((B, Nkv, Smax, H), 1.0, 52 + H)
    v = randn_bf16((B, Nkv, Smax, H), 1.0, 53 + H)
    got = _attn_prefill(q.cuda(), k.cuda(), v.cuda(), past)
    ref = O.attn_prefill(t2bits(q), t2bits(k[:, :, :L]), t2bits(v[:, :, :L]))
    kk = k[:, :, :L].float().repeat_interleave(Nq // Nkv, dim=1)
    vv = v[:, :, :L].float().repeat_interleave(Nq // Nkv, dim=1)
    s = torch.einsum("bsnh,bnlh->bnsl", q.float(), kk) / np.sqrt(float(H))
    causal = torch.arange(L)[None, :] > (past + torch.arange(S))[:, None]
    s = s.masked_fill(causal[None, None], float("-inf"))
    t = torch.einsum("bnsl,bnlh->bsnh", torch.softmax(s, -1), vv).numpy().astype(np.float64)
    _close(got, ref, t)


def test_unsupported_head_sizes_are_rejected():
    from tpp_pytorch_extension import _lib
    _llm()
    L = _lib.lib()
    A = 1 << 20
    for H in (4, 12, 264, 512):
        assert L.tppx_attn_decode(A, A, A, None, 0, A, 0, A, 1, 4, 4, H, 64, None, 0, None) == _lib.EUNSUPPORTED
        assert L.tppx_attn_prefill(A, A, A, None, 0, 0, A, 1, 8, 4, 4, H, 64, None) == _lib.EUNSUPPORTED


@pytest.mark.parametrize("H", [64, 96])
@pytest.mark.parametrize("S,past", [(1, 21), (40, 0), (7, 30)])
def test_decoder_layer_with_64_wide_heads(S, past, H):
    """LlamaDecoderLayer (src/csrc/llm/fused_llm_infer.cpp:1229-1275) with head size 64, and 96 (no power of two: the
    rotate-half pairs of a head can straddle two waves of the rotary launch): rotary + cache append as their own
    launch, attention on the kernels for other head sizes, MXFP4 linears; against the composition of the oracle
    functions (rel-L2 <= 2e-2 for the layer output, cached keys / values within 1 bf16 ulp)."""
    import tpp_pytorch_extension  # noqa: F401
    from tpp_pytorch_extension import _ops
    F = _llm()
    HID, INTER, NQ, NKV, MP = 256, 512, 4, 2, 256
    shapes = [(NQ * H, HID), (NKV * H, HID), (NKV * H, HID), (HID, NQ * H), (INTER, HID), (INTER, HID), (HID, INTER)]
    Ws = [randn_bf16(s, 0.05, 910 + i) for i, s in enumerate(shapes)]
    rng = torch.Generator().manual_seed(91)
    g1, g2 = torch.rand(HID, generator=rng) + 0.5, torch.rand(HID, generator=rng) + 0.5
    EP = F.llama_rotary_table(MP, H, device="cpu")
    qws = [_ops.remap_and_quantize_mxfp4(block_bf16(W).cuda()) for W in Ws]
    layer = F.LlamaDecoderLayer([g1.cuda()] + qws[:4] + [g2.cuda()] + qws[4:] + [EP.cuda()], 0, 1e-5, H, MP, H)
    assert (layer.Nq, layer.Nkv, layer.H) == (NQ, NKV, H)
    B, cap = 2, 128
    cache = F.TppCache(cap)
    k0, v0 = randn_bf16((B, NKV, past, H), 1.0, 961), randn_bf16((B, NKV, past, H), 1.0, 962)
    if past:
        cache.fill_(0, k0.cuda(), v0.cuda())
    x = randn_bf16((B, S, HID), 1.0, 963 + S)
    pos = torch.arange(past, past + S, dtype=torch.int64).unsqueeze(0).repeat(B, 1)
    out = layer.forward([x.cuda(), None, pos.cuda()], cache, True)[0]
    cache.advance(S)
    qo = [O.remap_quantize_mxfp4(W.float().numpy()) for W in Ws]
    mm = [(lambda a, post=O.POST_NONE, pin=None, q=q, s=s: O.linear_mxfp4(a, q, s, None, post, pin, None, 1.0, O.MODE_IDEAL)) for q, s in qo]
    xb = t2bits(x).reshape(B * S, HID)
    h = O.rms_norm(xb, g1.numpy(), 1e-5)
    q, k, v = mm[0](h), mm[1](h), mm[2](h)
    q = O.rotary_llama(q.reshape(B, S, -1), EP.numpy(), pos.numpy(), NQ, H).reshape(B, S, NQ, H)
    k = O.rotary_llama(k.reshape(B, S, -1), EP.numpy(), pos.numpy(), NKV, H).reshape(B, S, NKV, H).transpose(0, 2, 1, 3)
    v = v.reshape(B, S, NKV, H).transpose(0, 2, 1, 3)
    kall = np.concatenate([t2bits(k0), k], axis=2)
    vall = np.concatenate([t2bits(v0), v], axis=2)
    if S == 1:
        ctx = O.attn_decode(q.reshape(B, NQ, H), kall, vall).reshape(B, NQ * H)
    else:
        ctx = O.attn_prefill(q, kall, vall).reshape(B * S, NQ * H)
    so = mm[3](ctx, O.POST_ADD_SCALE, xb)
    h2 = O.rms_norm(so, g2.numpy(), 1e-5)
    gate = mm[4](h2, O.POST_SILU)
    ref = mm[6](mm[5](h2, O.POST_MUL, gate), O.POST_ADD_SCALE, so)
    g, r = bits2f(t2bits(out)).reshape(B * S, HID).astype(np.float64), bits2f(ref).astype(np.float64)
    rel = np.sqrt(((g - r) ** 2).sum() / (r ** 2).sum())
    assert rel <= 2e-2, rel
    kc, vc = cache.get(0)
    assert_close_bf16(t2bits(kc[:, :, past:]), np.ascontiguousarray(k), what="cached keys")
    assert_close_bf16(t2bits(vc[:, :, past:]), np.ascontiguousarray(v), what="cached values")


@pytest.mark.parametrize("H", [64, 256])
def test_attn_prefill_other_head_sizes_full_prompt_and_plain_kernel(H, monkeypatch):
    """A prompt long enough for many key tiles and for more than 256 workgroups (the ones past 256 walk their query
    blocks in the other order): sampled rows against the oracle's single-query function, and the MFMA kernel
    against the plain one-wave-per-query kernel it replaced, over every row."""
    _llm()
    B, S, Nq = 2, 600, 16
    q = randn_bf16((B, S, Nq, H), 1.0, 171 + H)
    k = randn_bf16((B, Nq, S, H), 1.0, 172 + H)
    v = randn_bf16((B, Nq, S, H), 1.0, 173 + H)
    got = _attn_prefill(q.cuda(), k.cuda(), v.cuda(), 0).cpu()
    for i in (0, 1, 63, 64, 65, 511, 599):
        ref = O.attn_decode(t2bits(q[:, i]), t2bits(k[:, :, :i + 1]), t2bits(v[:, :, :i + 1]))
        g, r = bits2f(t2bits(got[:, i])).astype(np.float64), bits2f(ref).astype(np.float64)
        assert np.sqrt(((g - r) ** 2).sum() / (r ** 2).sum()) <= 5e-3, i
        assert np.abs(g - r).max() <= 2.0 ** -7 * np.abs(r).max(), i
    monkeypatch.setenv("TPPX_ATTN_PREFILL_MFMA", "0")
    plain = _attn_prefill(q.cuda(), k.cuda(), v.cuda(), 0).cpu()
    d = (plain.float() - got.float()).double()
    assert float(d.norm() / plain.double().norm()) <= 5e-3


@pytest.mark.parametrize("H", [64, 200])
def test_attn_prefill_other_head_size_with_mask(H):
    F = _llm()
    B, S, Nq, Smax = 2, 70, 4, 128
    q = randn_bf16((B, S, Nq, H), 1.0, 181 + H)
    k = randn_bf16((B, Nq, Smax, H), 1.0, 182 + H)
    v = randn_bf16((B, Nq, Smax, H), 1.0, 183 + H)
    keep = torch.ones(B, S, dtype=torch.int64)
    keep[0, :9] = 0  # left padding of sequence 0
    mask = F.TppCache(Smax).align_and_invert_mask(keep.to(torch.bfloat16))
    got = _attn_prefill(q.cuda(), k.cuda(), v.cuda(), 0, mask=mask.cuda())
    ref = O.attn_prefill(t2bits(q), t2bits(k[:, :, :S]), t2bits(v[:, :, :S]), mask.float().numpy())
    g, r = bits2f(t2bits(got)).astype(np.float64), bits2f(ref).astype(np.float64)
    assert np.isfinite(g).all()
    assert np.sqrt(((g - r) ** 2).sum() / (r ** 2).sum()) <= 5e-3


# five and six tiles of 64 keys (one team has one more, or as many), a last tile of one key and a full one, one query block
# whose last tile lies past its own last key; sequence 0 masked over its first tiles (both teams' first ones), or over all
# keys of its first queries
@pytest.mark.parametrize("H", [64, 8, 72, 120])
@pytest.mark.parametrize("B,S,Nq,Nkv,past,hidden", [(1, 257, 4, 4, 0, 0), (2, 70, 4, 2, 314, 0), (2, 5, 8, 8, 252, 130), (2, 300, 4, 4, 0, 70)])
def test_attn_prefill_in_two_teams(H, B, S, Nq, Nkv, past, hidden, monkeypatch):
    """Prompt attention of few workgroups over many keys: two teams of waves take every other key tile.  Equal to the oracle
    within the bounds of the other tests here, and to one team within the rounding of the probabilities: each is rounded to
    bf16 against its own team's maximum (2^-8 relative, independent errors)."""
    F = _llm()
    L, Smax = past + S, 448
    q = randn_bf16((B, S, Nq, H), 1.0, 281 + H)
    k = randn_bf16((B, Nkv, Smax, H), 1.0, 282 + H)
    v = randn_bf16((B, Nkv, Smax, H), 1.0, 283 + H)
    k[:, :, L:] = float("nan")
    v[:, :, L:] = float("nan")
    mask = None
    if hidden:
        keep = torch.ones(B, L, dtype=torch.int64)
        keep[0, :hidden] = 0
        mask = F.TppCache(Smax).align_and_invert_mask(keep.to(torch.bfloat16))
    got = _attn_prefill(q.cuda(), k.cuda(), v.cuda(), past, mask=None if mask is None else mask.cuda())
    monkeypatch.setenv("TPPX_ATTN_TEAMS", "1")
    one = _attn_prefill(q.cuda(), k.cuda(), v.cuda(), past, mask=None if mask is None else mask.cuda())
    ref = O.attn_prefill(t2bits(q), t2bits(k[:, :, :L]), t2bits(v[:, :, :L]), None if mask is None else mask.float().numpy())
    g, r, o = (bits2f(a).astype(np.float64) for a in (t2bits(got), ref, t2bits(one)))
    assert np.isfinite(g).all()
    rows = slice(hidden if past == 0 else 0, None)  # (queries that see no key at all: whatever the mask's finite values leave)
    g, r, o = g[:, rows], r[:, rows], o[:, rows]
    assert np.sqrt(((g - r) ** 2).sum() / (r ** 2).sum()) <= 5e-3
    assert np.sqrt(((g - o) ** 2).sum() / (o ** 2).sum()) <= 2.0 ** -8


# around the edges of a trip (128 or 64 keys) and of a wave's keys (32 or 16), an empty and a full cache, one split and
# several, query heads sharing a K/V head, no mask / mask
@pytest.mark.parametrize("H,HR,style", [(256, 64, "gptj"), (80, 0, None), (64, 64, "llama"), (96, 96, "llama"), (200, 80, "llama"),
                                        (16, 16, "gptj"), (8, 0, None), (72, 48, "gptj"), (136, 136 - 8, "llama")])
@pytest.mark.parametrize("B,Nq,Nkv,past,Smax", [(1, 4, 4, 0, 700), (2, 8, 2, 31, 64), (1, 2, 2, 63, 64), (3, 4, 4, 128, 1024),
                                                (1, 6, 3, 700, 1100), (2, 4, 4, 64, 64), (40, 16, 16, 97, 130)])
def test_decode_step_with_rotary_and_append_in_the_launch(H, HR, style, B, Nq, Nkv, past, Smax):
    """tppx_attn_decode_append against the two launches it stands for: the same cache (positions it must not touch
    included), rotated values within one rounding, the context to the tolerance of the two orders of sums; every replay of a
    captured step the same."""
    from tpp_pytorch_extension import _lib
    F = _llm()
    L = _lib.lib()
    g = torch.Generator(device="cuda").manual_seed(7 * H + past)

    def rnd(*shape):
        return torch.randn(shape, generator=g, device="cuda").to(torch.bfloat16)

    q, k, v, kc, vc = rnd(B, Nq, H), rnd(B, Nkv, H), rnd(B, Nkv, H), rnd(B, Nkv, Smax, H), rnd(B, Nkv, Smax, H)
    kc[:, :, past + 1:] = vc[:, :, past + 1:] = float("nan")
    MP = 512
    pos = torch.randint(0, MP + 20, (B, 1), generator=g, device="cuda")  # some past the table: not rotated
    emb = None
    if style == "llama":
        emb = F.llama_rotary_table(MP, HR)
    elif style == "gptj":
        emb = torch.randn((MP, HR), generator=g, device="cuda")
    mask = torch.where(torch.rand((B, past + 1), generator=g, device="cuda") < 0.2, -10000.0, 0.0).to(torch.bfloat16) if past > 40 else None
    n = torch.tensor([past], dtype=torch.int32, device="cuda")
    ws = _lib.workspace(q)
    st = _lib.stream_of(q)
    P = lambda t: None if t is None else t.data_ptr()  # noqa: E731
    mld = mask.shape[1] if mask is not None else 0
    q2, k2, kc2, vc2 = q.clone(), k.clone(), kc.clone(), vc.clone()
    out, ref = torch.empty_like(q), torch.empty_like(q)

    def step(stream):
        _lib.check(L.tppx_attn_decode_append(q.data_ptr(), k.data_ptr(), v.data_ptr(), P(emb), style == "gptj", pos.data_ptr(), B,
                                             MP, HR, kc.data_ptr(), vc.data_ptr(), P(mask), mld, n.data_ptr(), out.data_ptr(),
                                             B, Nq, Nkv, H, Smax, ws.data_ptr(), ws.numel(), stream))

    q0, k0 = q.clone(), k.clone()
    step(st)
    fn = L.tppx_rotary_kv_append_gptj if style == "gptj" else L.tppx_rotary_kv_append_llama
    _lib.check(fn(q2.data_ptr(), k2.data_ptr(), v.data_ptr(), P(emb), pos.data_ptr(), kc2.data_ptr(), vc2.data_ptr(), n.data_ptr(),
                  B, 1, Nq, Nkv, H, MP, HR if emb is not None else H, B, Smax, st))
    _lib.check(L.tppx_attn_decode(q2.data_ptr(), kc2.data_ptr(), vc2.data_ptr(), P(mask), mld, n.data_ptr(), 1, ref.data_ptr(),
                                  B, Nq, Nkv, H, Smax, ws.data_ptr(), ws.numel(), st))
    assert torch.equal(q, q0) and torch.equal(k, k0)
    a, b = kc.float(), kc2.float()
    assert torch.equal(a.isnan(), b.isnan()) and torch.equal(vc.view(torch.int16), vc2.view(torch.int16))
    a, b = a.nan_to_num(0.0), b.nan_to_num(0.0)
    assert ((a - b).abs() <= 2.0 ** -7 * b.abs()).all() and (a != b).float().mean() < 1e-3
    assert out.isfinite().all()
    assert (out.float() - ref.float()).norm() <= 5e-3 * ref.float().norm()
    first = out.clone()
    s2 = torch.cuda.Stream()
    s2.wait_stream(torch.cuda.current_stream())
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph, stream=s2):
        step(torch.cuda.current_stream().cuda_stream)
    for _ in range(3):
        out.zero_()
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(out, first)


# 128-wide heads: the kernel of long loops, the wide one, the one of grouped heads
@pytest.mark.parametrize("H,HR,style,Nq,wide", [(128, 128, "llama", 4, "0"), (128, 128, "llama", 4, "1"), (128, 128, "llama", 32, "1"),
                                                (64, 64, "llama", 4, "1"), (80, 32, "gptj", 4, "1"), (256, 64, "gptj", 4, "1"), (200, 80, "llama", 8, "1")])
def test_every_rotation_leaves_the_same_key(H, HR, style, Nq, wide, monkeypatch):
    """The launches that rotate a new key agree in every bit: the sine's product rounded, the cosine's fused into it.  The table is
    made so that each pair's first (even pairs) or second (odd pairs) value nearly cancels and what is left is the products'
    rounding; the keys are one row scaled by powers of two."""
    from tpp_pytorch_extension import _lib
    _llm()
    monkeypatch.setenv("TPPX_ATTN_WIDE", wide)
    L = _lib.lib()
    B, Nkv, Smax, past, MP, pairs = 3, 4 if Nq < 32 else 2, 64, 17, 8, HR // 2
    g = torch.Generator().manual_seed(HR + H)
    base = (1.0 + torch.rand(H, generator=g)).to(torch.bfloat16)  # 1 .. 2: all products within a few binades
    k = base * 2.0 ** torch.randint(-3, 4, (B, Nkv, 1), generator=g).to(torch.bfloat16)
    i1 = torch.arange(pairs) * 2 if style == "gptj" else torch.arange(pairs)
    i2 = i1 + (1 if style == "gptj" else pairs)
    x1, x2 = base[i1].double(), base[i2].double()
    t = (0.5 + 0.5 * torch.rand(pairs, generator=g)).double().float()
    even = torch.arange(pairs) % 2 == 0
    cos = torch.where(even, (x2 * t.double() / x1).float(), t)      # x1 cos - x2 sin ~ 0
    sin = torch.where(even, t, (-x2 * t.double() / x1).float())     # x2 cos + x1 sin ~ 0
    table = torch.zeros((MP, HR) if style == "gptj" else (2, MP, HR))
    if style == "gptj":
        table[5] = torch.cat([sin, cos])
    else:
        table[0, 5], table[1, 5] = torch.cat([cos, cos]), torch.cat([sin, sin])
    want = k.clone()
    k1, k2 = k[..., i1].double(), k[..., i2].double()  # (24 + 8 bits: products exact, and so are the sums, in float64)
    want[..., i1] = (k1 * cos.double() - (k2 * sin.double()).float().double()).float().to(torch.bfloat16)
    want[..., i2] = (k2 * cos.double() + (k1 * sin.double()).float().double()).float().to(torch.bfloat16)
    own = (k1 * sin.double() + (k2 * cos.double()).float().double()).float().to(torch.bfloat16)
    assert (own != want[..., i2]).float().mean() > 0.2  # (the other order is told apart)

    dev = lambda a: a.cuda().contiguous()  # noqa: E731
    k, v, q, table = dev(k), torch.zeros((B, Nkv, H), dtype=torch.bfloat16, device="cuda"), dev(base.expand(B, Nq, H)), dev(table)
    kc, vc = (torch.zeros((B, Nkv, Smax, H), dtype=torch.bfloat16, device="cuda") for _ in range(2))
    n, pos = torch.tensor([past], dtype=torch.int32, device="cuda"), torch.full((B, 1), 5, dtype=torch.int64, device="cuda")
    st, out = _lib.stream_of(k), torch.empty_like(q)
    cache = (kc.data_ptr(), vc.data_ptr())
    head = (q.data_ptr(), k.data_ptr(), v.data_ptr(), table.data_ptr())
    tail = (None, 0, n.data_ptr(), out.data_ptr(), B, Nq, Nkv, H, Smax, None, 0, st)
    if H == 128:
        _lib.check(L.tppx_attn_decode_rotary(*head, pos.data_ptr(), B, MP, HR, *cache, *tail))
    else:
        _lib.check(L.tppx_attn_decode_append(*head, style == "gptj", pos.data_ptr(), B, MP, HR, *cache, *tail))
    assert torch.equal(kc[:, :, past].cpu(), want)
    q2, k2 = q.clone(), k.clone()
    fn = L.tppx_rotary_kv_append_gptj if style == "gptj" else L.tppx_rotary_kv_append_llama
    kc.zero_()
    _lib.check(fn(q2.data_ptr(), k2.data_ptr(), v.data_ptr(), table.data_ptr(), pos.data_ptr(), *cache, n.data_ptr(), B, 1, Nq, Nkv, H,
                  MP, HR, B, Smax, st))
    assert torch.equal(kc[:, :, past].cpu(), want) and torch.equal(k2.cpu(), want)


@pytest.mark.parametrize("H,Nq,Nkv", [(64, 8, 2), (80, 4, 4), (256, 2, 2), (8, 2, 1), (200, 4, 2)])
@pytest.mark.parametrize("B,L,Smax", [(2, 77, 128), (1, 1000, 1100)])
def test_decode_step_rounds_the_output_only(H, Nq, Nkv, B, L, Smax):
    """The probabilities keep 16 bits on their way into p . v: against float64 the output is off by its own rounding to bf16,
    half an ulp, and what fp32 scores and sums leave -- 2^-16 of a probability, an exponential good to about 2^-20 of scores up
    to 2^3, so 2^-14 of sum p |v| is far above it.  (With bf16 probabilities the second part would be up to 2^-9.)"""
    F = _llm()
    q, k, v = randn_bf16((B, Nq, H), 1.0, 331 + H), randn_bf16((B, Nkv, Smax, H), 1.0, 332 + H), randn_bf16((B, Nkv, Smax, H), 1.0, 333 + H)
    got = _attn(F, q.cuda(), k.cuda(), v.cuda(), L).cpu().double()
    kk, vv = (t[:, :, :L].double().repeat_interleave(Nq // Nkv, dim=1) for t in (k, v))
    p = torch.softmax((q.double().unsqueeze(2) * kk).sum(-1) / H ** 0.5, -1).unsqueeze(-1)
    ref, mag = (p * vv).sum(2), (p * vv.abs()).sum(2)
    half_ulp = torch.exp2(torch.floor(torch.log2(ref.abs().clamp_min(1e-30))) - 8)
    assert ((got.view_as(ref) - ref).abs() <= half_ulp * (1 + 2.0 ** -8) + 2.0 ** -14 * mag).all()


@pytest.mark.parametrize("H,Nq,Nkv,B", [(80, 32, 32, 4), (256, 16, 16, 4), (128, 28, 4, 2), (128, 32, 32, 2)])
def test_steps_on_two_streams_and_in_a_replayed_graph(H, Nq, Nkv, B):
    """Decode attention with split keys, from two threads on streams of their own beside a replayed graph: launches that
    share arrival counters are the ones that share a workspace, which are ordered, so every output has the bits of the same
    call alone, and the counters are zero again.  96 launches a thread: 4096 counters in rotation, one per (sequence, head),
    would have come round several times.  Without counters: the same bits."""
    import threading
    from tpp_pytorch_extension import _lib
    L = _lib.lib()
    Smax, past = 1600, 1500
    g = torch.Generator(device="cuda").manual_seed(H + Nq)
    rnd = lambda *s: torch.randn(s, generator=g, device="cuda").to(torch.bfloat16)  # noqa: E731
    kc, vc = rnd(B, Nkv, Smax, H), rnd(B, Nkv, Smax, H)
    qs = [rnd(B, Nq, H) for _ in range(3)]
    n = torch.tensor([past], dtype=torch.int32, device="cuda")

    def step(q, counted=True):
        ws, st, out = _lib.workspace(q), _lib.stream_of(q), torch.empty_like(q)
        args = (q.data_ptr(), kc.data_ptr(), vc.data_ptr(), None, 0, n.data_ptr(), 0, out.data_ptr(), B, Nq, Nkv, H, Smax)
        scratch = _lib.with_counters(ws)
        _lib.check(L.tppx_attn_decode_counted(*args, *scratch, st) if counted else L.tppx_attn_decode(*args, *scratch[:2], st))
        return out

    alone = [step(q) for q in qs]
    assert all(torch.equal(step(q, False), a) for q, a in zip(qs, alone))
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        captured = step(qs[2])
    torch.cuda.synchronize()
    outs, errors, buffers = [[], []], [], [None, None]
    streams = [torch.cuda.Stream(), torch.cuda.Stream()]

    def worker(i):
        try:
            with torch.cuda.stream(streams[i]):
                for _ in range(96):
                    outs[i].append(step(qs[i]))
                buffers[i] = _lib.workspace(qs[i])
        except Exception as e:  # reported by the main thread
            errors.append(repr(e))

    threads = [threading.Thread(target=worker, args=(i,)) for i in range(2)]
    replays = []
    for t in threads:
        t.start()
    for _ in range(48):
        graph.replay()
        replays.append(captured.clone())
    for t in threads:
        t.join()
    torch.cuda.synchronize()
    assert not errors, errors
    for i in range(2):
        assert all(torch.equal(y, alone[i]) for y in outs[i]), i
    assert all(torch.equal(y, alone[2]) for y in replays)
    assert buffers[0].data_ptr() != buffers[1].data_ptr()
    for ws in buffers:
        at = _lib.with_counters(ws)[2] - ws.untyped_storage().data_ptr()
        whole = torch.empty(0, dtype=torch.uint8, device="cuda").set_(ws.untyped_storage())
        assert whole.numel() >= at + _lib.COUNTER_BYTES and not whole[at:at + _lib.COUNTER_BYTES].any()


def test_decoder_blocks_count_arrivals_in_their_own_workspace(monkeypatch):
    """The Python layer calls no form of decode attention that shares counters between streams."""
    from tpp_pytorch_extension import _lib
    F = _llm()
    lib, seen = _lib.lib(), []

    class Watch:
        def __getattr__(self, name):
            if name.startswith("tppx_attn_decode"):
                assert name.endswith("_counted"), name
                seen.append(name)
            return getattr(lib, name)

    monkeypatch.setattr(_lib, "lib", lambda: Watch())
    for H, N, style in ((80, 4, None), (256, 2, "gptj"), (128, 4, "gptj")):
        cache = F.TppCache(64)
        table = None if style is None else torch.zeros((64, 64), device="cuda")
        qkv = [torch.randn((1, 1, N * H), device="cuda").to(torch.bfloat16) for _ in range(3)]
        F.rotate_append_attend(*qkv, None, torch.zeros((1, 1), dtype=torch.int64, device="cuda"), cache, 0, 1, 1, N, N, H, table, style)
    torch.cuda.synchronize()
    assert seen == ["tppx_attn_decode_append_counted"] * 2 + ["tppx_attn_decode_counted"]


@pytest.mark.parametrize("H,Nq,Nkv", [(128, 28, 4), (128, 4, 4), (80, 8, 2)])
def test_a_mask_of_no_keys_masks_nothing(H, Nq, Nkv):
    """A mask pointer with mask_ld 0 is as good as none: nothing is read there, by tppx_attn_decode and by the forms that
    append the new token (all of them read the pointer's surroundings here: valid memory that would mask every key)."""
    from tpp_pytorch_extension import _lib
    L = _lib.lib()
    q, k, v = (randn_bf16(s, 1.0, 341 + i).cuda() for i, s in enumerate(((2, Nq, H), (2, Nkv, 128, H), (2, Nkv, 128, H))))
    k0, v0 = k[:, :, 0].contiguous(), v[:, :, 0].contiguous()
    low = torch.full((4096,), -1e30, dtype=torch.bfloat16, device="cuda")
    n, pos = torch.tensor([76], dtype=torch.int32, device="cuda"), torch.zeros(1, dtype=torch.int64, device="cuda")
    ws, st = _lib.workspace(q), _lib.stream_of(q)
    for append in (False, True):
        outs = []
        for mask in (None, low[2048:].data_ptr()):
            kc, vc, out = k.clone(), v.clone(), torch.empty_like(q)
            end = (n.data_ptr(),) + ((out.data_ptr(),) if append else (1, out.data_ptr())) + (2, Nq, Nkv, H, 128, ws.data_ptr(), ws.numel(), st)
            new = (q.data_ptr(), k0.data_ptr(), v0.data_ptr(), None)
            at = (pos.data_ptr(), 1, 1, H, kc.data_ptr(), vc.data_ptr(), mask, 0)
            if not append:
                _lib.check(L.tppx_attn_decode(q.data_ptr(), kc.data_ptr(), vc.data_ptr(), mask, 0, *end))
            elif H == 128:
                _lib.check(L.tppx_attn_decode_rotary(*new, *at, *end))
            else:
                _lib.check(L.tppx_attn_decode_append(*new, 0, *at, *end))
            outs.append(out)
        torch.cuda.synchronize()
        assert torch.equal(*outs)
