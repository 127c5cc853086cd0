"""Parity of the HIP linears against the CPU oracle (ideal mode: fp32
accumulate, one bf16 rounding, reference rounding points in the post-ops).

Stated tolerance: every output within 1 bf16 ulp of the oracle (2 ulp where a
sigmoid is involved, because libm's and the GPU's expf differ in the last
bit), relative L2 error <= 4e-3; against the reference's own bf16 re-rounding
schedule (faithful mode) rel-L2 <= 2^-9 * sqrt(#K-groups) for QINT8.
"""
import numpy as np
import pytest
import torch

import oracle as O
from util import t2bits, randn_bf16, block_bf16, assert_close_bf16, err_stats, qint8_scratch

pytestmark = pytest.mark.gpu

POSTS = {"none": O.POST_NONE, "silu": O.POST_SILU, "mul": O.POST_MUL, "add": O.POST_ADD_SCALE,
         "add2": O.POST_ADD2_SCALE, "gelu": O.POST_GELU, "relu": O.POST_RELU}


def _lib_mod():
    import tpp_pytorch_extension  # noqa: F401
    from tpp_pytorch_extension import _lib
    return _lib


def _ops():
    import tpp_pytorch_extension  # noqa: F401
    from tpp_pytorch_extension import _ops
    return _ops


def _make(fmt, N, K, seed):
    ops = _ops()
    W = randn_bf16((N, K), 0.02, seed)
    Wb = block_bf16(W).cuda()
    if fmt == "mxfp4":
        qw = ops.remap_and_quantize_mxfp4(Wb)
        q_or, s_or = O.remap_quantize_mxfp4(W.float().numpy())
    else:
        qw = ops.remap_and_quantize_qint8(Wb)
        q_or, s_or, _ = O.remap_quantize_qint8(W.float().numpy())
    # the quantized bytes must be identical before the GEMM is compared
    assert np.array_equal(qw.qdata.cpu().numpy(), q_or), "quantized values differ from the oracle"
    assert np.array_equal(qw.scales.cpu().numpy().reshape(s_or.shape), s_or), "scales differ from the oracle"
    return qw, q_or, s_or


def _run(fmt, M, N, K, post, with_bias, seed, ulps=1, flags=0):
    ops = _ops()
    qw, q_or, s_or = _make(fmt, N, K, seed)
    x = randn_bf16((M, K), 1.0, seed + 1)
    bias = randn_bf16((N,), 0.01, seed + 2) if with_bias else None
    in1 = randn_bf16((M, N), 1.0, seed + 3)
    in2 = randn_bf16((M, N), 1.0, seed + 4)
    scale = 0.5 if post in ("add", "add2") else 1.0
    y = ops.linear(x.cuda(), qw, None if bias is None else bias.cuda(), POSTS[post],
                   in1.cuda(), in2.cuda(), scale, flags=flags)
    torch.cuda.synchronize()
    lin = O.linear_mxfp4 if fmt == "mxfp4" else O.linear_qint8
    ref = lin(t2bits(x), q_or, s_or, None if bias is None else t2bits(bias), POSTS[post],
              t2bits(in1), t2bits(in2), scale, O.MODE_IDEAL)
    s = assert_close_bf16(t2bits(y), ref, ulps=ulps, what=f"{fmt} M={M} N={N} K={K} post={post}")
    return y, ref, s, (qw, q_or, s_or, x, bias, in1, in2, scale)


@pytest.mark.parametrize("fmt", ["mxfp4", "qint8"])
@pytest.mark.parametrize("M", [1, 3, 16, 17, 33, 64])
def test_fc_plain_small(fmt, M):
    _run(fmt, M, 256, 512, "none", True, 100 + M)


@pytest.mark.parametrize("fmt", ["mxfp4", "qint8"])
@pytest.mark.parametrize("post", ["silu", "mul", "add", "add2", "gelu", "relu"])
def test_post_ops(fmt, post):
    _run(fmt, 5, 128, 768, post, post != "mul", 200, ulps=2 if post in ("silu", "gelu") else 1)


@pytest.mark.parametrize("fmt", ["mxfp4", "qint8"])
def test_no_bias_ragged_k(fmt):
    # K = 11008 = 86*128 = 43*256: an odd number of K units, waves get uneven ranges
    _run(fmt, 8, 64, 11008, "none", False, 300)


@pytest.mark.parametrize("M,N,K", [(12, 64, 11008), (13, 64, 11008), (9, 64, 14336), (4, 32, 16384), (1, 64, 4096)])
def test_qint8_few_rows_quantised_in_the_gemm_ring_forms(M, N, K):
    """QINT8 with the activation quantisation inside the GEMM kernel, one channel tile per workgroup: up to three
    K blocks per wave run a ring of four weight tiles (six quantisation passes in flight once a wave has more than 16
    (row, block) items: 36 and 39 items here, two rounds), four blocks per wave (K >= 14336) the ring of eight."""
    _run("qint8", M, N, K, "add", True, 9100 + M + K)


# one to eight channel tiles per workgroup (256, 512, .. tiles and one more; two rounds), ragged last groups, one run of K,
# fewer runs than waves, one per wave; rows around the eight of two quantization passes
@pytest.mark.parametrize("M,N,K", [(1, 16, 256), (8, 4096, 512), (9, 4112, 256), (16, 8192, 256), (3, 8208, 768), (8, 12304, 256),
                                   (16, 16400, 256), (9, 20496, 256), (4, 24592, 256), (16, 32784, 256), (1, 1024, 4096),
                                   (16, 272, 4096), (7, 8208, 3584), (2, 528, 4352)])
def test_qint8_few_rows_tile_by_tile(M, N, K):
    """Up to 16 rows and 4096 input channels: the channel tiles of a workgroup one after the other (and 4352 channels, which
    are not)."""
    _run("qint8", M, N, K, "add" if M % 2 else "none", True, 230 + M)


def test_qint8_group_of_few_rows_counts_its_workgroups_by_weight():
    """q/k/v and the first MLP projection as one launch: each weight's last workgroup may be short of tiles."""
    ops = _ops()
    ws = [_make("qint8", N, 512, 240 + i)[0] for i, N in enumerate((4096, 272, 272, 16384))]
    x = randn_bf16((5, 512), 1.0, 250).cuda()
    for y, w, post in zip(ops.qkv_gemm(x, ws, [None] * 4), ws, (O.POST_NONE,) * 3 + (O.POST_GELU,)):
        assert torch.equal(y, ops.linear(x, w, None, post))


# waves with one or two K tiles of 128 (17, 20, 28, 31 in all), one to four channel tiles per workgroup, ragged last groups
@pytest.mark.parametrize("M,N,K", [(1, 96, 2176), (4, 4128, 2560), (3, 8224, 3584), (2, 12320, 3968), (4, 32, 3584), (5, 96, 3584)])
def test_mxfp4_few_rows_of_uneven_wave_slices(M, N, K):
    """Up to 4 rows and K between 2048 and 4096 on the LDS-staged kernel (5 rows: the tile-by-tile one), single, grouped and
    as the gate/up pair."""
    ops = _ops()
    y, _, _, ctx = _run("mxfp4", M, N, K, "add" if M % 2 else "none", True, 260 + M)
    if N > 4200:
        return
    x = ctx[3].cuda()
    ws = [ctx[0], _make("mxfp4", N, K, 270)[0], _make("mxfp4", 32, K, 271)[0]]
    for o, w in zip(ops.qkv_gemm(x, ws, [None] * 3), ws):
        assert torch.equal(o, ops.linear(x, w, None))
    assert torch.equal(ops.swiglu_gate_up(x, ws[0], ws[1]), ops.fc_mul(x, ws[1], None, ops.fc_silu(x, ws[0], None)))


# 17 rows and more behind the operand-order quantizer, 128 and more behind the row-major one; between them, from 65 rows, and
# for K above 8192 the two launches; one to four chunks of 8 values per thread and their edges; gamma in both types
@pytest.mark.parametrize("M,K,gdt", [(17, 256, torch.float32), (64, 2304, torch.bfloat16), (40, 4096, torch.float32),
                                     (100, 1024, torch.float32), (128, 2048, torch.float32), (300, 6144, torch.bfloat16),
                                     (1100, 512, torch.float32), (130, 8192, torch.float32), (130, 8448, torch.float32),
                                     (3, 512, torch.float32)])
def test_qint8_norm_in_the_quantizer(M, K, gdt):
    """q/k/v and gate/up projections with RMSNorm in front equal rms_norm followed by them: ordinary rows, a row of zeros,
    rows with an infinity and with a NaN."""
    ops = _ops()
    ws = [_make("qint8", N, K, 280 + i)[0] for i, N in enumerate((256, 128, 256))]
    assert all(w.block_size == 256 for w in ws)
    g = (torch.randn(K, generator=torch.Generator().manual_seed(283)) * 0.3 + 1.0).to(gdt).cuda()
    x = randn_bf16((M, K), 2.0, 284)
    x[1] = 0.0
    for special in (False, True):
        if special:
            x[0, 3], x[2, K - 1] = float("inf"), float("nan")
        xg = x.cuda()
        n = ops.rms_norm(xg, g, 1e-5)
        for y, w in zip(ops.qkv_gemm(xg, ws, [None] * 3, norm=(g, 1e-5)), ops.qkv_gemm(n, ws, [None] * 3)):
            assert torch.equal(y.view(torch.int16), w.view(torch.int16))
        y, w = ops.swiglu_gate_up(xg, ws[0], ws[2], norm=(g, 1e-5)), ops.swiglu_gate_up(n, ws[0], ws[2])
        assert torch.equal(y.view(torch.int16), w.view(torch.int16))


@pytest.mark.parametrize("M,K", [(3, 512), (17, 512), (64, 1024), (65, 512), (100, 2048), (127, 1024), (128, 512), (300, 1024), (130, 8448)])
def test_qint8_norm_in_the_quantizer_is_one_launch_where_it_is_built(M, K, monkeypatch):
    """From 17 rows on (the pair: from 65, as one launch) and up to 8192 input channels the normalisation is part of the
    quantizer's launch; the library refuses none of those calls, and rms_norm runs once in front of the others.  The bits of
    the two launches, for rows of zeros, with an infinity and with a NaN too."""
    import ctypes
    from tpp_pytorch_extension import _lib
    ops = _ops()
    ws = [_make("qint8", 2048, K, 286 + i)[0] for i in range(2)]
    x, g = randn_bf16((M, K), 2.0, 288), torch.ones(K, device="cuda")
    x[0], x[1, 3], x[2, K - 1] = 0.0, float("inf"), float("nan")
    x = x.cuda()
    n = ops.rms_norm(x, g, 1e-5)
    want = [list(ops.qkv_gemm(n, ws, [None] * 2)), [ops.swiglu_gate_up(n, *ws)]]
    answers, norms, lib, rms = [], [], _lib.lib(), ops.rms_norm

    class Watch:
        def __getattr__(self, name):
            f = getattr(lib, name)
            if "_norm_" not in name:
                return f

            def call(*args):
                rc = f(*args)
                answers.append(rc)
                return rc
            return call

    monkeypatch.setattr(_lib, "lib", lambda: Watch())
    monkeypatch.setattr(ops, "rms_norm", lambda *a: norms.append(1) or rms(*a))
    pair = M > 64 and lib.tppx_group_is_one_launch((ctypes.c_int64 * 2)(2048, 2048), 2, M, K, 1)
    for call, fused, ref in ((lambda n: list(ops.qkv_gemm(x, ws, [None] * 2, norm=n)), M > 16 and K <= 8192, want[0]),
                             (lambda n: [ops.swiglu_gate_up(x, *ws, norm=n)], pair and K <= 8192, want[1])):
        answers.clear(), norms.clear()
        for y, w in zip(call((g, 1e-5)), ref):
            assert torch.equal(y.view(torch.int16), w.view(torch.int16))
        assert answers == [0] * fused and len(norms) == 1 - fused, (answers, norms)


def test_cfg1_mxfp4_fc_plain():
    """M=16, K=N=4096, MXFP4, bias."""
    _run("mxfp4", 16, 4096, 4096, "none", True, 1235)


@pytest.mark.parametrize("M", [1, 8, 32, 64])
def test_cfg2_qint8_fc_add(M):
    """BASELINE config 2 (down-projection shape scaled in N to keep the CPU oracle fast)."""
    y, ref, s, ctx = _run("qint8", M, 512, 11008, "add", False, 1236 + M)
    qw, q_or, s_or, x, bias, in1, in2, scale = ctx
    faithful = O.linear_qint8(t2bits(x), q_or, s_or, None, O.POST_ADD_SCALE, t2bits(in1), None, scale,
                              O.MODE_FAITHFUL)
    st = err_stats(t2bits(y), faithful)
    groups = 11008 // (256 if M == 64 else 64)
    assert st["rel_l2"] <= 2.0 ** -9 * np.sqrt(groups), st["rel_l2"]


def test_qint8_block_64_and_128():
    ops = _ops()
    for K in (192, 384):  # -> QBS 64 and 128 by the reference's rule
        W = randn_bf16((64, K), 0.02, 7)
        qw = ops.remap_and_quantize_qint8(block_bf16(W).cuda())
        q_or, s_or, qbs = O.remap_quantize_qint8(W.float().numpy())
        assert qw.block_size == qbs
        assert np.array_equal(qw.qdata.cpu().numpy(), q_or)
        x = randn_bf16((4, K), 1.0, 8)
        y = ops.fc_plain(x.cuda(), qw, torch.Tensor())
        ref = O.linear_qint8(t2bits(x), q_or, s_or)
        assert_close_bf16(t2bits(y), ref, what=f"qbs={qbs}")


@pytest.mark.parametrize("fmt", ["mxfp4", "qint8"])
def test_qkv_gemm_equals_separate(fmt):
    ops = _ops()
    K, M = 1024, 7
    ws = [_make(fmt, n, K, 40 + i)[0] for i, n in enumerate((512, 128, 128))]
    bs = [randn_bf16((n,), 0.01, 50 + i).cuda() for i, n in enumerate((512, 128, 128))]
    x = randn_bf16((2, M, K), 1.0, 60).cuda()
    outs = torch.ops.tpp_llm.qkv_gemm(x, ws, bs)
    for w, b, o in zip(ws, bs, outs):
        sep = torch.ops.tpp_llm.fc_plain(x, w, b, -1, [])
        assert o.shape == sep.shape == (2, M, w.weight_nk()[0])
        assert torch.equal(o, sep)


def test_swiglu_fused_equals_composition():
    ops = _ops()
    K, N, M = 512, 1024, 9
    wg, wu = _make("mxfp4", N, K, 70)[0], _make("mxfp4", N, K, 71)[0]
    wd = _make("mxfp4", K, N, 72)[0]
    x = randn_bf16((M, K), 1.0, 73).cuda()
    fused = ops.swiglu_gate_up(x, wg, wu)
    g = ops.fc_silu(x, wg, None)
    u = ops.fc_mul(x, wu, None, g)
    assert torch.equal(fused, u)
    out = torch.ops.tpp_llm.swiglu_mlp(x, wg, wu, wd, x, 1.0)
    assert torch.equal(out, ops.fc_add(u, wd, None, x, 1.0))


def test_module_api_and_errors():
    import tpp_pytorch_extension  # noqa: F401
    from tpp_pytorch_extension.llm.llm_common import FixLinear, BlockedLinear
    from tpp_pytorch_extension._lib import TppxError

    torch.manual_seed(0)
    lin = torch.nn.Linear(256, 128, bias=True)
    W, b = lin.weight.data.clone(), lin.bias.data.clone()
    FixLinear(lin, 16, 64, torch.bfloat16, weight_dtype="mxfp4")
    assert isinstance(lin, BlockedLinear) and lin.weight.is_quantized
    assert lin.weight.dtype == torch.quint4x2 and lin.weight.size(-1) == 2
    x = torch.randn(3, 5, 256).cuda()
    y = lin(x)  # fp32 input is cast to bf16 by the module, as in the reference
    q_or, s_or = O.remap_quantize_mxfp4(W.to(torch.bfloat16).float().numpy())
    ref = O.linear_mxfp4(t2bits(x.to(torch.bfloat16).view(15, 256)), q_or, s_or, t2bits(b.to(torch.bfloat16)))
    assert y.shape == (3, 5, 128) and y.dtype == torch.bfloat16
    assert_close_bf16(t2bits(y).reshape(15, 128), ref, what="BlockedLinear")
    with pytest.raises(TppxError):
        torch.ops.tpp_llm.fc_plain(x.to(torch.bfloat16)[..., :128].contiguous(), lin.weight, torch.Tensor(), -1, [])
    yf = torch.ops.tpp_llm.fc_plain(x, lin.weight, torch.Tensor(), -1, [])  # fp32 activations: fp32 result
    assert yf.dtype == torch.float32 and yf.shape == (3, 5, 128)
    with pytest.raises(TppxError):
        torch.ops.tpp_llm.fc_plain(x.to(torch.float64), lin.weight, torch.Tensor(), -1, [])
    e = torch.ops.tpp_llm.fc_plain(torch.empty(0, 256, dtype=torch.bfloat16).cuda(), lin.weight, torch.Tensor(), -1, [])
    assert e.shape == (0, 128)


@pytest.mark.parametrize("fmt", ["mxfp4", "qint8"])
@pytest.mark.parametrize("M", [65, 200, 256])
@pytest.mark.parametrize("family", ["tiled", "skinny", "auto"])
def test_prefill_tiled_small(fmt, M, family):
    """More than 64 rows: the LDS-tiled kernels (N = 384 leaves the last 128-wide block half empty, M = 65 / 200
    leave the last row block ragged) or the decode kernels over several block rows of 64 (the library picks by a
    cost estimate; both families forced here)."""
    from tpp_pytorch_extension import _lib
    flags = {"tiled": _lib.FLAG_FORCE_TILED, "skinny": _lib.FLAG_FORCE_SKINNY, "auto": 0}[family]
    _run(fmt, M, 384, 1024, "add", True, 500 + M, flags=flags)


@pytest.mark.parametrize("fmt", ["mxfp4", "qint8"])
@pytest.mark.parametrize("M,N,K", [(128, 11008, 1024), (192, 4096, 2048), (130, 512, 11008)])
def test_mid_size_m_block_rows(fmt, M, N, K):
    """65..256 rows at 7B-like widths: few output tiles, so the decode kernels run block rows of 64 over the full
    grid (ragged last block row, three channel tiles per workgroup, K split over the waves)."""
    _run(fmt, M, N, K, "add", True, 8800 + M)


@pytest.mark.parametrize("post", ["none", "silu", "mul", "add2", "gelu"])
def test_prefill_mxfp4_ragged_blocks_and_post_ops(post):
    """Large-M MXFP4 kernel (256 x 256 workgroup tiles): two row blocks with a
    ragged second one, three channel blocks with two tiles in the last, an odd
    number of K steps, every fused epilogue through the coalesced store path."""
    _run("mxfp4", 300, 544, 384, post, post != "mul", 700, ulps=2 if post in ("silu", "gelu") else 1)


# (on MXFP4 weights 128 x 256 has one form, of four waves: TPPX_TILED_W8 is the bf16 kernel's and makes no difference here)
@pytest.mark.parametrize("tile,w8", [(1, 1), (2, 1), (2, 0), (3, 1)])
@pytest.mark.parametrize("post", ["none", "silu", "add2"])
def test_prefill_mxfp4_every_workgroup_tile_ragged(tile, w8, post, monkeypatch):
    """The workgroup tiles of the large-M MXFP4 kernel from 128 x 256 on (256 x 256, 128 x 256 with eight waves and with
    four, two per CU, 128 x 512), each forced, on the ragged case above (rows, channel blocks and K steps all uneven)
    against the oracle."""
    monkeypatch.setenv("TPPX_TILED_BIG_TILE", str(tile))
    monkeypatch.setenv("TPPX_TILED_W8", str(w8))
    _run("mxfp4", 300, 544, 384, post, True, 705, ulps=2 if post == "silu" else 1)


@pytest.mark.parametrize("tile", [4, 7, 8, 10, 12, 13, 14, 15, 16, 17])
@pytest.mark.parametrize("post", ["none", "silu", "add2"])
def test_prefill_mxfp4_every_wave_tile_ragged(tile, post, monkeypatch):
    """The same on 64 x 128 and the other wave tiles, each forced."""
    monkeypatch.setenv("TPPX_TILED_MIN_M", "0")
    monkeypatch.setenv("TPPX_TILED_BIG_TILE", str(tile))
    _run("mxfp4", 300, 544, 384, post, True, 705, ulps=2 if post == "silu" else 1)


@pytest.mark.parametrize("fmt", ["mxfp4", "qint8"])
@pytest.mark.parametrize("M,post", [(65, "add"), (130, "add"), (130, "mul"), (300, "silu"), (300, "relu"), (300, "none"), (130, "add2"), (130, "gelu")])
def test_prefill_epilogue_of_every_post_op(fmt, M, post):
    """The epilogue of the large-M kernels is instantiated per post-op (none, SiLU, mul, add) or takes it from the launch
    (the others), and reads the post-op's input ahead, also for rows past the end: ragged rows and channel blocks."""
    from tpp_pytorch_extension import _lib
    _run(fmt, M, 544, 768, post, post != "mul", 740 + M, ulps=2 if post in ("silu", "gelu") else 1, flags=_lib.FLAG_FORCE_TILED)


def test_prefill_mxfp4_workgroup_tiles_and_xcd_splits_agree(monkeypatch):
    """Every workgroup tile and every split of the tile space over the XCDs computes the same sums in the same order:
    identical bits, single GEMM, fused q/k/v and the gate/up pair."""
    ops = _ops()
    M, K = 1024, 512
    w = _make("mxfp4", 4096, K, 710)[0]
    ws = [_make("mxfp4", n, K, 711 + i)[0] for i, n in enumerate((2048, 1024, 1024))]
    wg, wu = _make("mxfp4", 4096, K, 715)[0], _make("mxfp4", 4096, K, 716)[0]
    x = randn_bf16((M, K), 1.0, 717).cuda()

    def run():
        return [ops.fc_plain(x, w, None)] + list(ops.qkv_gemm(x, ws, [None] * 3)) + [ops.swiglu_gate_up(x, wg, wu)]

    monkeypatch.setenv("TPPX_TILED_BIG_TILE", "1")
    monkeypatch.setenv("TPPX_TILED_XCD_M", "1")
    want = run()
    assert torch.equal(want[4], ops.fc_mul(x, wu, None, ops.fc_silu(x, wg, None)))
    for tile in (1, 2, 3):
        for xm in (1, 2, 4):
            monkeypatch.setenv("TPPX_TILED_BIG_TILE", str(tile))
            monkeypatch.setenv("TPPX_TILED_XCD_M", str(xm))
            for i, (a, b) in enumerate(zip(run(), want)):
                assert torch.equal(a, b), (tile, xm, i)


# (64 x 128, 64 x 256 and eight waves: bf16 weights; MXFP4: the wave tiles)
@pytest.mark.parametrize("M", [70, 150, 200, 500])
def test_prefill_forms_for_small_launches_agree(M, monkeypatch):
    """Launches that leave CUs empty run other forms of the large-M kernels -- 64 x 128 workgroups of four waves, eight
    waves per 128 x 256 workgroup up to 256 of those -- with the same sums in the same order: identical bits to the
    four-wave 128 x 256 form, for a single GEMM (ragged rows and channel blocks),
    fused q/k/v, the gate/up pair and unquantized bf16 weights; the same for the QINT8 kernel's 64 x 256 form (single
    GEMM and fused q/k/v); and the single MXFP4 GEMM against the oracle."""
    ops = _ops()
    K = 640
    w, q_or, s_or = _make("mxfp4", 1056, K, 720)[:3]
    ws = [_make("mxfp4", n, K, 721 + i)[0] for i, n in enumerate((1024, 256, 256))]
    wg, wu = _make("mxfp4", 1120, K, 725)[0], _make("mxfp4", 1120, K, 726)[0]
    Wb = randn_bf16((1056, K), 0.05, 727)
    wb = block_bf16(Wb).cuda()
    w8 = _make("qint8", 1056, 768, 729)[0]
    w8s = [_make("qint8", n, 768, 730 + i)[0] for i, n in enumerate((1024, 256, 256))]
    x8 = randn_bf16((M, 768), 1.0, 733).cuda()
    x = randn_bf16((M, K), 1.0, 728)
    xg = x.cuda()

    def run():
        return [ops.fc_plain(xg, w, None)] + list(ops.qkv_gemm(xg, ws, [None] * 3)) + [ops.swiglu_gate_up(xg, wg, wu)] + \
            [ops.linear(xg, wb, None, O.POST_NONE, None, None, 1.0, flags=_lib_mod().FLAG_FORCE_TILED)] + \
            [ops.fc_plain(x8, w8, None)] + list(ops.qkv_gemm(x8, w8s, [None] * 3))

    monkeypatch.setenv("TPPX_TILED_MIN_M", "0")  # the LDS-tiled family whatever the cost estimate says
    got = run()
    ref = O.linear_mxfp4(t2bits(x), q_or, s_or, None, O.POST_NONE, None, None, 1.0, O.MODE_IDEAL)
    assert_close_bf16(t2bits(got[0]), ref, ulps=1, what=f"64 x 128 workgroups M={M}")
    monkeypatch.setenv("TPPX_TILED_SMALL", "0")
    mid = run()
    monkeypatch.setenv("TPPX_TILED_W8", "0")
    base = run()
    for i, (a, b, c) in enumerate(zip(got, mid, base)):
        assert torch.equal(a, c) and torch.equal(b, c), i


@pytest.mark.parametrize("fmt", ["mxfp4", "qint8"])
def test_prefill_tiled_m2048(fmt):
    """Prefill row count of BASELINE config 4 (M = 2048) on a layer slice the
    CPU oracle finishes in seconds; also compared with the reference's chunked
    bf16 re-rounding schedule (K = 8192 > 4096 -> two chunks for MXFP4)."""
    y, ref, s, ctx = _run(fmt, 2048, 256, 8192, "none", True, 600)
    qw, q_or, s_or, x, bias, in1, in2, scale = ctx
    lin = O.linear_mxfp4 if fmt == "mxfp4" else O.linear_qint8
    faithful = lin(t2bits(x), q_or, s_or, t2bits(bias), O.POST_NONE, None, None, 1.0, O.MODE_FAITHFUL)
    st = err_stats(t2bits(y), faithful)
    bound = 2.0 ** -9 * np.sqrt(2 if fmt == "mxfp4" else 8192 // 256)
    assert st["rel_l2"] <= bound, st["rel_l2"]


def test_prefill_qkv_and_swiglu_equal_composition():
    ops = _ops()
    K, M = 1024, 130
    ws = [_make("mxfp4", n, K, 80 + i)[0] for i, n in enumerate((256, 128, 128))]
    x = randn_bf16((M, K), 1.0, 90).cuda()
    outs = torch.ops.tpp_llm.qkv_gemm(x, ws, [torch.Tensor()] * 3)
    for w, o in zip(ws, outs):
        assert torch.equal(o, ops.fc_plain(x, w, None))
    wg, wu = _make("mxfp4", 512, K, 91)[0], _make("mxfp4", 512, K, 92)[0]
    fused = ops.swiglu_gate_up(x, wg, wu)
    assert torch.equal(fused, ops.fc_mul(x, wu, None, ops.fc_silu(x, wg, None)))


@pytest.mark.parametrize("fused", [True, False])
@pytest.mark.parametrize("bias", [False, True])
def test_prefill_swiglu_one_grid_equals_composition(bias, fused, monkeypatch):
    """Prefill rows: gate and up run as ONE launch of the large-M kernel.  fused: every workgroup computes both
    projections of its 128 output channels and forms silu(gate) * up in its epilogue; otherwise (TPPX_TILED_DUAL_FUSED=0)
    the gate tile is parked in the workspace and an elementwise pass forms the product.  Either way the bits of
    fc_silu followed by fc_mul, ragged last row block and ragged last channel block included."""
    monkeypatch.setenv("TPPX_TILED_DUAL_FUSED", "1" if fused else "0")
    ops = _ops()
    K, M, N = 512, 300, 1056
    wg, qg, sg_ = _make("mxfp4", N, K, 191)
    wu, qu, su = _make("mxfp4", N, K, 192)
    x = randn_bf16((M, K), 1.0, 193).cuda()
    bg = randn_bf16((N,), 0.05, 194).cuda() if bias else None
    bu = randn_bf16((N,), 0.05, 195).cuda() if bias else None
    fused = ops.swiglu_gate_up(x, wg, wu, bg, bu)
    assert torch.equal(fused, ops.fc_mul(x, wu, bu, ops.fc_silu(x, wg, bg)))
    gate = O.linear_mxfp4(t2bits(x.cpu()), qg, sg_, None if bg is None else t2bits(bg.cpu()), O.POST_SILU)
    ref = O.linear_mxfp4(t2bits(x.cpu()), qu, su, None if bu is None else t2bits(bu.cpu()), O.POST_MUL, gate)
    assert_close_bf16(t2bits(fused), ref, ulps=2, what="prefill swiglu gate/up")


@pytest.mark.parametrize("M", [2, 12])
def test_swiglu_long_k_few_rows(M):
    """Gate/up pair with K = 8192 (beyond the 16-row LDS image): the 4-row staged kernel (M = 2) and the tile-by-tile
    kernel with one row group (M = 12) with two accumulator sets; bits of silu-then-mul, and the oracle."""
    ops = _ops()
    K, N = 8192, 1056
    wg, qg, sg_ = _make("mxfp4", N, K, 311)
    wu, qu, su = _make("mxfp4", N, K, 312)
    x = randn_bf16((M, K), 1.0, 313)
    fused = ops.swiglu_gate_up(x.cuda(), wg, wu)
    assert torch.equal(fused, ops.fc_mul(x.cuda(), wu, None, ops.fc_silu(x.cuda(), wg, None)))
    gate = O.linear_mxfp4(t2bits(x), qg, sg_, None, O.POST_SILU)
    ref = O.linear_mxfp4(t2bits(x), qu, su, None, O.POST_MUL, gate)
    assert_close_bf16(t2bits(fused), ref, ulps=2, what=f"swiglu gate/up K=8192 M={M}")


@pytest.mark.parametrize("M", [2, 12])
def test_swiglu_full_size_gate_up_equals_composition(M):
    """Llama-7B gate/up shape (688 channel tiles): the fused kernel takes one
    (M <= 4) or two channel tiles of each GEMM per workgroup; both must give the
    bits of silu-then-mul through the single-GEMM kernels, and match the oracle."""
    ops = _ops()
    wg, qg, sg_ = _make("mxfp4", 11008, 512, 301)
    wu, qu, su = _make("mxfp4", 11008, 512, 302)
    x = randn_bf16((M, 512), 1.0, 303)
    fused = ops.swiglu_gate_up(x.cuda(), wg, wu)
    assert torch.equal(fused, ops.fc_mul(x.cuda(), wu, None, ops.fc_silu(x.cuda(), wg, None)))
    gate = O.linear_mxfp4(t2bits(x), qg, sg_, None, O.POST_SILU)
    ref = O.linear_mxfp4(t2bits(x), qu, su, None, O.POST_MUL, gate)
    assert_close_bf16(t2bits(fused), ref, ulps=2, what=f"swiglu gate/up M={M}")


@pytest.mark.parametrize("M", [17, 32, 40, 64])
def test_mxfp4_row_group_kernel_full_size(M):
    """17..64 rows at the Llama-7B up-projection shape (688 channel tiles: three per workgroup, ragged last group,
    M = 40: a partly filled row group) with bias and the residual post-op."""
    y, ref, s, ctx = _run("mxfp4", M, 11008, 1024, "add", True, 7100 + M)


@pytest.mark.parametrize("M", [24, 64])
def test_mxfp4_row_group_kernel_uneven_k_split_and_swiglu(M):
    """K = 11008 (86 K tiles over 8 waves: 10 or 11 each); q/k/v segments in one launch; the gate/up pair as
    silu(gate) then up * gate in place: all equal to the single-GEMM calls bit for bit, which match the oracle."""
    ops = _ops()
    y, ref, s, ctx = _run("mxfp4", M, 256, 11008, "none", False, 7200 + M)
    K = 1024
    ws = [_make("mxfp4", n, K, 7300 + i)[0] for i, n in enumerate((4096, 512, 512))]
    x = randn_bf16((M, K), 1.0, 7310).cuda()
    outs = torch.ops.tpp_llm.qkv_gemm(x, ws, [torch.Tensor()] * 3)
    for w, o in zip(ws, outs):
        assert torch.equal(o, ops.fc_plain(x, w, None))
    wg, qg, sg_ = _make("mxfp4", 11008, K, 7320)
    wu, qu, su = _make("mxfp4", 11008, K, 7321)
    fused = ops.swiglu_gate_up(x, wg, wu)
    assert torch.equal(fused, ops.fc_mul(x, wu, None, ops.fc_silu(x, wg, None)))
    gate = O.linear_mxfp4(t2bits(x.cpu()), qg, sg_, None, O.POST_SILU)
    ref2 = O.linear_mxfp4(t2bits(x.cpu()), qu, su, None, O.POST_MUL, gate)
    assert_close_bf16(t2bits(fused), ref2, ulps=2, what=f"swiglu gate/up M={M}")


@pytest.mark.parametrize("fmt,M,N", [("mxfp4", 40, 4096), ("mxfp4", 64, 4064), ("qint8", 40, 4096), ("qint8", 64, 4080)])
def test_k_split_across_workgroups(fmt, M, N):
    """33..64 rows, at most 256 channel tiles and K = 11008: K is split across workgroups (4 parts of 21/22/21/22
    K tiles for MXFP4, 2 parts of 21/22 blocks for QINT8), the partial sums go through the workspace and the
    workgroup that finishes last adds them.  N = 4064 (254 tiles) or 4080 (255): a ragged last group; M = 40: a partly filled row
    group.  Forty launches in a row must give the same bits (the arrival counters return to zero, no launch sees
    another's partial sums)."""
    ops = _ops()
    y, ref, s, ctx = _run(fmt, M, N, 11008, "add", True, 7400 + M)
    qw, q_or, s_or, x, bias, in1, in2, scale = ctx
    xs, b, r = x.cuda(), bias.cuda(), in1.cuda()
    first = torch.ops.tpp_llm.fc_add(xs, qw, b, r, scale)
    outs = [torch.ops.tpp_llm.fc_add(xs, qw, b, r, scale) for _ in range(40)]
    torch.cuda.synchronize()
    assert torch.equal(first, y)
    for o in outs:
        assert torch.equal(o, first)


@pytest.mark.parametrize("M,N,K,post", [(64, 4096, 8192, "add"), (33, 4080, 14336, "add2"), (50, 2048, 16384, "none"),
                                        (17, 4096, 11008, "mul"), (32, 4064, 14336, "silu"), (64, 1600, 32768, "add"),
                                        (20, 4096, 12288, "gelu")])
def test_qint8_tile_by_k_part_kernel(M, N, K, post, monkeypatch):
    """QINT8, 17..64 rows, up to 256 channel tiles and a long K: four channel tiles x four K parts per workgroup with
    the activation operands shared through LDS, K in four slices across workgroups, partial tiles exchanged as
    128-bit device-scope stores / loads (2..8 steps per wave, ragged last channel group, partly filled row groups,
    every post-op).  Against the oracle; twenty launches give the same bits; the kernel it replaces
    (TPPX_QINT8_NK=0) is within one ulp of it as well (another summation order, so not bit-identical)."""
    import ctypes
    from tpp_pytorch_extension import _lib
    buf = ctypes.create_string_buffer(2048)
    _lib.check(_lib.lib().tppx_plan_linear_qint8(M, N, K, 256, 1, 0, _lib.WORKSPACE_BYTES, buf, len(buf)))
    assert "skinny_qint8_nk_kernel" in buf.value.decode(), buf.value.decode()
    y, ref, st, ctx = _run("qint8", M, N, K, post, True, 7700 + M, ulps=2 if post in ("silu", "gelu") else 1)
    qw, q_or, s_or, x, bias, in1, in2, scale = ctx
    ops = _ops()
    again = [ops.linear(x.cuda(), qw, bias.cuda(), POSTS[post], in1.cuda(), in2.cuda(), scale) for _ in range(20)]
    torch.cuda.synchronize()
    for o in again:
        assert torch.equal(o, y)
    monkeypatch.setenv("TPPX_QINT8_NK", "0")
    old = ops.linear(x.cuda(), qw, bias.cuda(), POSTS[post], in1.cuda(), in2.cuda(), scale)
    assert_close_bf16(t2bits(old), ref, ulps=2 if post in ("silu", "gelu") else 1, what="kernel without the tile x K-part grid")


@pytest.mark.parametrize("form", [0, 1])
@pytest.mark.parametrize("M,N,K,post", [(64, 4096, 8192, "add"), (33, 4064, 14336, "add2"), (50, 2048, 16384, "none"),
                                        (64, 1632, 12288, "silu"), (47, 4096, 11008, "mul")])
def test_mxfp4_tile_by_k_part_kernel(M, N, K, post, form, monkeypatch):
    """MXFP4, 33..64 rows, up to 256 channel tiles and a long K: four channel tiles x four K parts per workgroup (two
    tiles per wave and eight waves, or one and sixteen: TPPX_MXFP4_NK_FORM), a K tile's activations staged once per
    workgroup, K in four slices across workgroups, workgroups walking their K part from rotated starting tiles.
    Against the oracle; twenty launches give the same bits; the kernel it replaces (TPPX_MXFP4_NK=0) meets the oracle
    too."""
    import ctypes
    from tpp_pytorch_extension import _lib
    monkeypatch.setenv("TPPX_MXFP4_NK_FORM", str(form))
    buf = ctypes.create_string_buffer(2048)
    _lib.check(_lib.lib().tppx_plan_linear_mxfp4(M, N, K, 0, _lib.WORKSPACE_BYTES, buf, len(buf)))
    assert "skinny_mxfp4_nk_kernel<4, 4, %d," % (2 - form) in buf.value.decode(), buf.value.decode()
    y, ref, st, ctx = _run("mxfp4", M, N, K, post, True, 7800 + M, ulps=2 if post == "silu" else 1)
    qw, q_or, s_or, x, bias, in1, in2, scale = ctx
    ops = _ops()
    again = [ops.linear(x.cuda(), qw, bias.cuda(), POSTS[post], in1.cuda(), in2.cuda(), scale) for _ in range(20)]
    torch.cuda.synchronize()
    for o in again:
        assert torch.equal(o, y)
    if form == 0:
        monkeypatch.setenv("TPPX_MXFP4_NK", "0")
        old = ops.linear(x.cuda(), qw, bias.cuda(), POSTS[post], in1.cuda(), in2.cuda(), scale)
        assert_close_bf16(t2bits(old), ref, ulps=2 if post == "silu" else 1, what="kernel without the tile x K-part grid")


@pytest.mark.parametrize("split", [True, False])
@pytest.mark.parametrize("M,N,K", [(5, 4096, 11008), (16, 4096, 11008), (9, 2048, 16384), (16, 4096, 8192)])
def test_mxfp4_few_rows_long_k_split_across_workgroups(M, N, K, split, monkeypatch):
    """5..16 rows, at most 256 channel tiles and a K too long for one workgroup's staging: the LDS-staged kernel with
    K in 4 parts across workgroups of 4 channel tiles (21/22 K tiles per part at K = 11008, 1 or 2 per wave), partial
    sums through the workspace, the last workgroup to arrive finishes -- or (TPPX_MXFP4_XL_SPLIT=0) the tile-by-tile
    kernel.  Against the oracle; the row sums of squares the finishing workgroup leaves equal the sums over the output
    bits; repeated launches give the same bits."""
    monkeypatch.setenv("TPPX_MXFP4_XL_SPLIT", "1" if split else "0")
    ops = _ops()
    y, ref, s, ctx = _run("mxfp4", M, N, K, "add", True, 7500 + M)
    qw, q_or, s_or, x, bias, in1, in2, scale = ctx
    xs, b, r = x.cuda(), bias.cuda(), in1.cuda()
    tab = torch.full((16, 256), 3.0, dtype=torch.float32, device="cuda")  # stale contents must not survive
    outs = [ops.fc_add(xs, qw, b, r, scale, row_sumsq=tab) for _ in range(20)]
    torch.cuda.synchronize()
    for o in outs:
        assert torch.equal(o, y)
    want = (y.double() ** 2).sum(-1).cpu().numpy()
    got = tab[:M].double().sum(-1).cpu().numpy()
    assert np.allclose(got, want, rtol=1e-5), (got, want)


def test_prefill_qint8_qkv_one_launch_equals_separate():
    """QINT8, enough rows for the large-M kernel: fused q/k/v share one launch (ragged channel blocks: 544, 128 and
    256 channels) and give the bits of the single-GEMM calls, which match the oracle."""
    ops = _ops()
    K, M = 1024, 300
    made = [_make("qint8", n, K, 280 + i) for i, n in enumerate((544, 128, 256))]
    ws = [m[0] for m in made]
    x = randn_bf16((M, K), 1.0, 290)
    bs = [randn_bf16((n,), 0.01, 295 + i).cuda() for i, n in enumerate((544, 128, 256))]
    outs = torch.ops.tpp_llm.qkv_gemm(x.cuda(), ws, bs)
    for (w, q_or, s_or), b, o in zip(made, bs, outs):
        assert torch.equal(o, ops.fc_plain(x.cuda(), w, b))
        ref = O.linear_qint8(t2bits(x), q_or, s_or, t2bits(b.cpu()))
        assert_close_bf16(t2bits(o), ref, what="qint8 fused qkv, large M")


def test_prefill_qkv_one_launch_equals_separate():
    """With enough rows the fused q/k/v GEMMs share one launch of the large-M
    kernel (one grid over the channel blocks of all three)."""
    ops = _ops()
    K, M = 512, 300
    ws = [_make("mxfp4", n, K, 180 + i)[0] for i, n in enumerate((544, 128, 256))]
    x = randn_bf16((M, K), 1.0, 190).cuda()
    bs = [randn_bf16((n,), 0.01, 195 + i).cuda() for i, n in enumerate((544, 128, 256))]
    outs = torch.ops.tpp_llm.qkv_gemm(x, ws, bs)
    for w, b, o in zip(ws, bs, outs):
        assert torch.equal(o, ops.fc_plain(x, w, b))


_FULL_UP = {}


def _full_up():
    """One Llama-7B up-projection weight (N=11008, K=4096), quantized once."""
    if not _FULL_UP:
        _FULL_UP["w"] = _make("qint8", 11008, 4096, 4242)
    return _FULL_UP["w"]


@pytest.mark.parametrize("M", [1, 4, 8, 16, 32, 40, 64])
def test_cfg2_qint8_up_projection_full_size(M):
    """The kernel variants that only large N selects (two and three channel
    tiles per wave, ragged last workgroup: 688 tiles), at BASELINE's real shape."""
    ops = _ops()
    qw, q_or, s_or = _full_up()
    x = randn_bf16((M, 4096), 1.0, 500 + M)
    r = randn_bf16((M, 11008), 1.0, 600 + M)
    y = torch.ops.tpp_llm.fc_add(x.cuda(), qw, torch.Tensor(), r.cuda(), 1.0)
    ref = O.linear_qint8(t2bits(x), q_or, s_or, None, O.POST_ADD_SCALE, t2bits(r), None, 1.0, O.MODE_IDEAL)
    pre = O.linear_qint8(t2bits(x), q_or, s_or)
    assert_close_bf16(t2bits(y), ref, what=f"qint8 up-projection M={M}", pre_bits=pre)


def test_qint8_fused_quant_shared_lds():
    """16 rows x K=8192 with three channel tiles per workgroup: the quantised activations and the cross-wave
    reduction do not fit the LDS side by side, so the reduction reuses the activations' region."""
    y, ref, s, ctx = _run("qint8", 16, 8448, 8192, "add", True, 4242)
    assert_close_bf16(t2bits(y), ref, what="qint8 M=16 K=8192 N=8448")


@pytest.mark.parametrize("M,K", [(128, 512), (200, 11008), (2048, 4096)])
def test_qint8_activation_quantizer_many_rows_bit_exact(M, K):
    """From 128 rows on, 256-wide blocks take the quantizer that gives 16 lanes to a (row, block); with zero rows, a
    row of one value and a huge value in the input, bytes and scales must equal the oracle's."""
    from tpp_pytorch_extension import _lib
    L = _lib.lib()
    x = randn_bf16((M, K), 1.0, 41)
    x[5] = 0.0
    x[7] = -0.375
    x[9, 300] = 3.0e38
    x = x.cuda()
    xq = torch.empty((M, K), dtype=torch.int8, device="cuda")
    sa = torch.empty((M, K // 256), dtype=torch.float32, device="cuda")
    _lib.check(L.tppx_quant_act_int8(x.data_ptr(), M, K, 256, xq.data_ptr(), sa.data_ptr(), _lib.stream_of(x)))
    xq_or, sa_or = O.quant_act_int8(t2bits(x.cpu()), 256)
    assert np.array_equal(sa.cpu().numpy(), sa_or)
    assert np.array_equal(xq.cpu().numpy(), xq_or)


@pytest.mark.parametrize("M", [3, 24, 64])
def test_qint8_prequantized_and_reused_activations(M):
    """x == NULL takes row-major int8 activations + scales (the reference's
    pre-quantized input); TPPX_FLAG_XQ_REUSE skips the re-quantization when a
    second GEMM runs on the same input.  Both must give the bits of the plain
    call, and the activation quantization itself must match the oracle."""
    from tpp_pytorch_extension import _lib
    L = _lib.lib()
    N, K, qbs = 512, 1024, 256
    qw, q_or, s_or = _make("qint8", N, K, 31)
    qw2, q_or2, s_or2 = _make("qint8", N, K, 32)
    x = randn_bf16((M, K), 1.0, 33).cuda()
    st = _lib.stream_of(x)
    ws = _lib.workspace(x)
    xq_rm = torch.empty((M, K), dtype=torch.int8, device="cuda")
    sa_rm = torch.empty((M, K // qbs), dtype=torch.float32, device="cuda")
    _lib.check(L.tppx_quant_act_int8(x.data_ptr(), M, K, qbs, xq_rm.data_ptr(), sa_rm.data_ptr(), st))
    xq_or, sa_or = O.quant_act_int8(t2bits(x.cpu()), qbs)
    assert np.array_equal(xq_rm.cpu().numpy(), xq_or) and np.array_equal(sa_rm.cpu().numpy(), sa_or)

    def call(xptr, xq, sa, w, flags):
        qn, sn = w.native()
        y = torch.empty((M, N), dtype=torch.bfloat16, device="cuda")
        _lib.check(L.tppx_linear_qint8(xptr, xq.data_ptr(), sa.data_ptr(), qn.data_ptr(), sn.data_ptr(), None, None,
                                       None, y.data_ptr(), M, N, K, qbs, 0, 1.0, flags, ws.data_ptr(), ws.numel(), st))
        return y

    xq = torch.empty(((M + 63) // 64 * 64, K), dtype=torch.int8, device="cuda")
    sa = torch.empty(((M + 63) // 64 * 64, K // qbs), dtype=torch.float32, device="cuda")
    y_plain = call(x.data_ptr(), xq, sa, qw, 0)
    y2_reuse = call(x.data_ptr(), xq, sa, qw2, _lib.FLAG_XQ_REUSE)
    y2_plain = call(x.data_ptr(), xq.clone().zero_(), sa.clone().zero_(), qw2, 0)
    y_pre = call(None, xq_rm, sa_rm, qw, 0)
    torch.cuda.synchronize()
    ref = O.linear_qint8(t2bits(x.cpu()), q_or, s_or)
    assert_close_bf16(t2bits(y_plain), ref, what=f"plain M={M}")
    assert torch.equal(y_pre, y_plain), "pre-quantized input gives different bits"
    assert torch.equal(y2_reuse, y2_plain), "reused activation quantization gives different bits"


def _shape_sweep():
    """48 seeded (format, M, N, K, post-op, bias) cases across the kernel selection boundaries: 1..64 rows, channel
    counts that leave ragged workgroups, K from one native tile to the Llama intermediate size."""
    import random
    rnd = random.Random(20240)
    cases = []
    for i in range(48):
        fmt = rnd.choice(["mxfp4", "qint8"])
        M = rnd.choice([1, 2, 3, 4, 5, 7, 8, 9, 15, 16, 17, 20, 31, 32, 33, 47, 48, 63, 64])
        N = rnd.choice([32, 64, 96, 160, 512, 1056, 4128, 8224])
        K = rnd.choice([128, 256, 384, 512, 1024, 2048, 2304, 4096, 5120, 8192, 11008])
        if fmt == "qint8" and K % 256:
            K = (K // 256 + 1) * 256
        cases.append((fmt, M, N, K, rnd.choice(["none", "silu", "mul", "add", "add2", "gelu", "relu"]), rnd.random() < 0.5, 9100 + i))
    return cases


@pytest.mark.parametrize("fmt,M,N,K,post,bias,seed", _shape_sweep())
def test_shape_sweep(fmt, M, N, K, post, bias, seed):
    ops = _ops()
    qw, q_or, s_or = _make(fmt, N, K, seed)
    x = randn_bf16((M, K), 1.0, seed + 1)
    b = randn_bf16((N,), 0.01, seed + 2) if bias else None
    in1, in2 = randn_bf16((M, N), 1.0, seed + 3), randn_bf16((M, N), 1.0, seed + 4)
    scale = 0.5 if post in ("add", "add2") else 1.0
    y = ops.linear(x.cuda(), qw, None if b is None else b.cuda(), POSTS[post], in1.cuda(), in2.cuda(), scale)
    lin = O.linear_mxfp4 if fmt == "mxfp4" else O.linear_qint8
    bb = None if b is None else t2bits(b)
    ref = lin(t2bits(x), q_or, s_or, bb, POSTS[post], t2bits(in1), t2bits(in2), scale, O.MODE_IDEAL)
    pre = lin(t2bits(x), q_or, s_or, bb) if post in ("add", "add2") else None  # the tile a residual can cancel
    assert_close_bf16(t2bits(y), ref, ulps=2 if post in ("silu", "gelu") else 1,
                      what=f"{fmt} M={M} N={N} K={K} post={post}", pre_bits=pre)


def test_launch_plan_names_the_kernels():
    import ctypes
    from tpp_pytorch_extension import _lib
    L = _lib.lib()
    buf = ctypes.create_string_buffer(2048)
    _lib.check(L.tppx_plan_linear_qint8(64, 11008, 4096, 256, 1, 0, 1 << 25, buf, len(buf)))
    lines = buf.value.decode().strip().splitlines()
    assert len(lines) == 2 and "quant_act_int8_rows_kernel" in lines[0] and "skinny_qint8_kernel<" in lines[1]
    _lib.check(L.tppx_plan_linear_qint8(1, 11008, 4096, 256, 1, 0, 1 << 25, buf, len(buf)))
    assert buf.value.decode().count("\n") == 1 and "skinny_qint8_fq_kernel<" in buf.value.decode()
    _lib.check(L.tppx_plan_linear_mxfp4(2048, 8192, 8192, 0, 0, buf, len(buf)))
    assert "big_mxfp4_kernel" in buf.value.decode()
    _lib.check(L.tppx_plan_linear_mxfp4(100, 8192, 8192, _lib.FLAG_FORCE_TILED, 0, buf, len(buf)))
    assert "wide_kernel<2, 1, 8, false, false, false>" in buf.value.decode()  # small wave tiles from 65 rows on
    _lib.check(L.tppx_plan_linear_mxfp4(128, 1024, 4096, 0, 0, buf, len(buf)))  # few tiles: block rows of 64
    assert "skinny_mxfp4_mg_kernel" in buf.value.decode() and "x2x" in buf.value.decode()


@pytest.mark.parametrize("M,N,K,post,layout", [
    (1, 2000, 512, "none", "vnni2"), (5, 272, 1024, "add", "vnni2"), (16, 4096, 4096, "none", "vnni2"),
    (17, 1008, 384, "silu", "plain"), (33, 528, 640, "mul", "vnni2"), (64, 1024, 11008, "add", "vnni2"),
    (100, 304, 256, "add2", "plain"), (200, 1040, 512, "none", "blocked100")])
def test_bf16_weight_linear(M, N, K, post, layout):
    """Unquantized bf16 weights (the reference's default lm_head class, TppBlockedLinearW<bf16,bf16>) through
    fc_plain / the post-op GEMMs: 1 ulp of the oracle's single-rounding result, for the blocked VNNI2 layout
    BlockedLinear makes, a plain [N][K] matrix, and the lm_head's own blocking (bk = N/10-style odd block
    heights: here 104 = 1040/10 rows per block)."""
    ops = _ops()
    W = randn_bf16((N, K), 0.02, 81)
    x = randn_bf16((M, K), 1.0, 82)
    bias = randn_bf16((N,), 0.01, 83)
    in1, in2 = randn_bf16((M, N), 1.0, 84), randn_bf16((M, N), 1.0, 85)
    scale = 0.5 if post in ("add", "add2") else 1.0
    if layout == "vnni2":
        Wg = block_bf16(W).cuda()
    elif layout == "plain":
        Wg = W.cuda()
    else:
        Wg = block_bf16(W, bk=104, bc=64).cuda()
    y = ops.linear(x.cuda(), Wg, bias.cuda(), POSTS[post], in1.cuda(), in2.cuda(), scale)
    ref = O.linear_bf16(t2bits(x), t2bits(W), t2bits(bias), POSTS[post], t2bits(in1), t2bits(in2), scale)
    assert_close_bf16(t2bits(y), ref, ulps=1, what=f"bf16 weight M={M} N={N} K={K} post={post} {layout}",
                      pre_bits=O.linear_bf16(t2bits(x), t2bits(W), t2bits(bias)) if post in ("add", "add2") else None)
    y2 = ops.linear(x.cuda(), Wg, bias.cuda(), POSTS[post], in1.cuda(), in2.cuda(), scale)  # cached native tiles
    assert torch.equal(y, y2)


@pytest.mark.parametrize("fmt", ["bf16", "mxfp4"])
@pytest.mark.parametrize("M", [16, 40, 200])
def test_outputs_round_to_nearest_even(fmt, M):
    """The fp32 sum of a GEMM becomes bf16 by round to nearest, ties to even, in the epilogues of the decode kernels, the row
    groups and the tiles: sums built from three bf16 parts (all 24 bits, in different MFMA steps, weights of 1) around every
    tie, with carries into the exponent and past the largest value, infinities and NaN, against torch's conversion."""
    from tpp_pytorch_extension import _lib
    ops = _ops()
    K, N = 256, 64
    low = torch.tensor([0x0000, 0x0001, 0x7fff, 0x8000, 0x8001, 0xffff])
    high = torch.tensor([0x3f80, 0x3f81, 0x3fff, 0x4000, 0x1234, 0x7f7e, 0x7f7f, 0x0c01])
    bits = ((high[:, None] << 16) | low[None, :]).flatten()
    bits = torch.cat([bits, bits | 0x80000000, torch.tensor([0x7f800000, 0xff800000, 0x7fc00000, 0])])
    values = torch.from_numpy(bits.numpy().astype(np.uint32).view(np.float32))
    w = block_bf16(torch.ones((N, K), dtype=torch.bfloat16)).cuda()
    if fmt == "mxfp4":
        w = ops.remap_and_quantize_mxfp4(w)
        assert bool((w.dequantize() == 1).all())
    for start in range(0, values.numel(), M):
        v = values[torch.arange(start, start + M) % values.numel()]
        x, rest = torch.zeros((M, K)), v.double()
        for k in (0, 96, 224):
            x[:, k] = torch.from_numpy((rest.float().numpy().view(np.uint32) & np.uint32(0xffff0000)).view(np.float32))
            rest = torch.where(torch.isfinite(v), rest - x[:, k].double(), torch.zeros_like(rest))
        y = ops.linear(x.to(torch.bfloat16).cuda(), w, None, flags=_lib.FLAG_FORCE_TILED if M > 64 else 0).cpu()
        want = v.to(torch.bfloat16)[:, None].expand(M, N).contiguous()
        nan = torch.isnan(want)
        assert torch.equal(torch.isnan(y), nan)
        assert torch.equal(y.masked_fill(nan, 0).view(torch.int16), want.masked_fill(nan, 0).view(torch.int16)), start


def test_bf16_weight_module_and_errors():
    import tpp_pytorch_extension  # noqa: F401
    from tpp_pytorch_extension.llm.llm_common import FixLinear, BlockedLinear
    from tpp_pytorch_extension._lib import TppxError
    torch.manual_seed(3)
    lin = torch.nn.Linear(256, 1000, bias=False)  # lm_head-like: FixLinear(m, 100, 64, bf16) keeps bf16 weights
    W = lin.weight.data.clone().to(torch.bfloat16)
    FixLinear(lin, 100, 64, torch.bfloat16)
    assert isinstance(lin, BlockedLinear) and not lin.weight.is_quantized and lin.weight.dim() == 5
    lin = lin.cuda()
    x = randn_bf16((2, 3, 256), 1.0, 86)
    with pytest.raises(TppxError):  # N = 1000 is not a multiple of 16
        lin(x.cuda())
    lin = torch.nn.Linear(256, 1600, bias=True)
    W, b = lin.weight.data.clone().to(torch.bfloat16), lin.bias.data.clone().to(torch.bfloat16)
    FixLinear(lin, 100, 64, torch.bfloat16)
    lin = lin.cuda()
    y = lin(x.cuda())
    ref = O.linear_bf16(t2bits(x.view(6, 256)), t2bits(W), t2bits(b))
    assert y.shape == (2, 3, 1600)
    assert_close_bf16(t2bits(y).reshape(6, 1600), ref, what="bf16 BlockedLinear")
    with pytest.raises(TppxError):
        _ops().linear(x.cuda()[..., :128].contiguous(), lin.weight, None)


def _mxfp8_from_operand_order(xq, xs, M, K):
    """GPU layout [Mp/16][K/128][2][64][16] / [Mp/64][K/128][64][4] (Mp = M rounded up to 64) -> codes [Mp][K],
    scale bytes [Mp][K/32]."""
    Mt, Kt = (M + 63) // 64 * 4, K // 128
    q = xq.view(Mt, Kt, 2, 4, 16, 16).permute(0, 4, 1, 2, 3, 5).reshape(Mt * 16, K)  # [mt][m][kt][h][g][16]
    s = xs.view(Mt // 4, Kt, 4, 16, 4).permute(0, 4, 3, 1, 2).reshape(Mt * 16, K // 32)  # [q][t][m][kt][b]
    return q.cpu().numpy(), s.cpu().numpy()


@pytest.mark.parametrize("M,K", [(1, 128), (37, 384), (128, 4096)])
def test_mxfp8_activation_quantizer_bit_exact(M, K):
    from tpp_pytorch_extension import _lib
    _ops()
    x = randn_bf16((M, K), 1.0, 91)
    x[0, :32] = 0.0                      # an all-zero block
    x.view(-1)[5::97] *= 37.0            # outliers that set block maxima
    Mp = (M + 63) // 64 * 64
    xq = torch.empty(Mp * K, dtype=torch.uint8, device="cuda")
    xs = torch.empty(Mp * K // 32, dtype=torch.uint8, device="cuda")
    xg = x.cuda()
    _lib.check(_lib.lib().tppx_quant_act_mxfp8(xg.data_ptr(), M, K, xq.data_ptr(), xs.data_ptr(), _lib.stream_of(xg)))
    q, s = _mxfp8_from_operand_order(xq, xs, M, K)
    q_or, s_or = O.quant_act_mxfp8(t2bits(x))
    assert np.array_equal(q[:M], q_or) and np.array_equal(s[:M], s_or)
    assert not q[M:].any() and not s[M:].any()  # padded rows are zeros


@pytest.mark.parametrize("M,N,K,post", [(128, 256, 256, "none"), (1, 32, 128, "none"), (200, 544, 384, "add"),
                                         (333, 4096, 1024, "silu"), (2048, 512, 4096, "none")])
def test_mxfp4_linear_on_fp8_activations(M, N, K, post):
    """TPPX_FLAG_ACT_FP8: MXFP4 weights on the block-scaled MFMA with MXFP8 activations.  Against the oracle of the
    same arithmetic (exact products, fp32 sums: 1 ulp, 2 through SiLU as for the other kernels), and against the reference-arithmetic oracle (bf16
    activations) within the rounding of E4M3: rel-L2 <= 5e-2."""
    from tpp_pytorch_extension import _lib
    ops = _ops()
    qw, q_or, s_or = _make("mxfp4", N, K, 95)
    x = randn_bf16((M, K), 1.0, 96)
    bias = randn_bf16((N,), 0.01, 97)
    in1 = randn_bf16((M, N), 1.0, 98)
    scale = 0.5 if post == "add" else 1.0
    y = ops.linear(x.cuda(), qw, bias.cuda(), POSTS[post], in1.cuda(), None, scale, flags=_lib.FLAG_ACT_FP8)
    ref = O.linear_mxfp4_fp8act(t2bits(x), q_or, s_or, t2bits(bias), POSTS[post], t2bits(in1), None, scale)
    pre = O.linear_mxfp4_fp8act(t2bits(x), q_or, s_or, t2bits(bias)) if post == "add" else None
    # the block-scaled MFMA adds the 128 products of an instruction with the hardware's own internal alignment, not
    # as exact fp64 sums: more elements land one ulp off than with another fp32 order (2-3 per thousand seen)
    assert_close_bf16(t2bits(y), ref, ulps=2 if post == "silu" else 1, what=f"fp8-act M={M} N={N} K={K} {post}",
                      pre_bits=pre, max_mismatch=None if post == "silu" else 1e-2)
    exact = O.linear_mxfp4(t2bits(x), q_or, s_or, t2bits(bias), POSTS[post], t2bits(in1), None, scale, O.MODE_IDEAL)
    assert err_stats(t2bits(y), exact)["rel_l2"] <= 5e-2


@pytest.mark.parametrize("fused", [True, False])
@pytest.mark.parametrize("M,K,widths", [(160, 512, (512, 256, 256)), (300, 384, (544, 288, 288))])
def test_fp8_activation_qkv_and_swiglu_equal_separate_calls(M, K, widths, fused, monkeypatch):
    """fused: the gate/up pair with both projections per workgroup and silu(gate) * up in the epilogue; otherwise
    (TPPX_TILED_DUAL_FUSED=0) the parked gate tile and the elementwise pass.  The second shape has ragged row, channel
    and K blocks."""
    from tpp_pytorch_extension import _lib, _ops as ops
    _ops()
    monkeypatch.setenv("TPPX_TILED_DUAL_FUSED", "1" if fused else "0")
    x = randn_bf16((M, K), 1.0, 99).cuda()
    ws = [_make("mxfp4", n, K, 100 + i)[0] for i, n in enumerate(widths)]
    old = ops.ACT_FP8
    ops.ACT_FP8 = True
    try:
        q, k, v = ops.qkv_gemm(x, ws, [None, None, None])
        sw = ops.swiglu_gate_up(x, ws[1], ws[2])
    finally:
        ops.ACT_FP8 = old
    for got, w in zip((q, k, v), ws):
        assert torch.equal(got, ops.linear(x, w, None, flags=_lib.FLAG_ACT_FP8))
    g = ops.linear(x, ws[1], None, POSTS["silu"], flags=_lib.FLAG_ACT_FP8)
    assert torch.equal(sw, ops.linear(x, ws[2], None, POSTS["mul"], g, flags=_lib.FLAG_ACT_FP8))
    from tpp_pytorch_extension._lib import TppxError
    Lb = _lib.lib()
    y = torch.empty(M, widths[0], dtype=torch.bfloat16, device="cuda")
    qn, sn = ws[0].native()
    with pytest.raises(TppxError):  # no workspace for the quantised activations
        _lib.check(Lb.tppx_linear_mxfp4(x.data_ptr(), qn.data_ptr(), sn.data_ptr(), None, None, None, y.data_ptr(),
                                        M, widths[0], K, 0, 1.0, _lib.FLAG_ACT_FP8, None, 0, _lib.stream_of(x)))


def test_split_launches_from_two_threads_on_two_streams():
    """Launches that split K over workgroups (partial sums in the workspace, an arrival counter per output group, the
    last arrival merges) and split-KV attention launches, issued by two Python threads, each on a stream of its own, so
    that they overlap on the card.  The ops take their workspace per (device, stream) and the library hands the
    arrival counters out in rotation, so the threads need no ordering between them.  Every output must carry the bits
    of the same call made alone on one stream; the comparison stops at the first mismatch."""
    import threading
    from tpp_pytorch_extension import _lib, _ops as ops
    _ops()
    Lb = _lib.lib()
    dev = torch.device("cuda:0")
    cases = []
    for fmt, M, N, K, seed in (("qint8", 64, 4096, 11008, 701), ("mxfp4", 64, 512, 4096, 702), ("mxfp4", 33, 256, 8192, 703)):
        qw = _make(fmt, N, K, seed)[0]
        x = randn_bf16((M, K), 1.0, seed + 1).cuda()
        r = randn_bf16((M, N), 1.0, seed + 2).cuda()
        cases.append(("linear", qw, x, r))
    B, Nq, Smax, Lk = 1, 32, 2304, 2000
    q = randn_bf16((B, Nq, 128), 1.0, 711).cuda()
    kc = randn_bf16((B, Nq, Smax, 128), 1.0, 712).cuda()
    vc = randn_bf16((B, Nq, Smax, 128), 1.0, 713).cuda()
    ln = torch.tensor([Lk - 1], dtype=torch.int32, device=dev)
    cases.append(("attn", q, kc, vc))

    def call(case):
        if case[0] == "linear":
            _, qw, x, r = case
            return ops.linear(x, qw, None, POSTS["add"], r, None, 0.5)
        _, q, kc, vc = case
        ws = _lib.workspace(q)
        out = torch.empty_like(q)
        _lib.check(Lb.tppx_attn_decode(q.data_ptr(), kc.data_ptr(), vc.data_ptr(), None, 0, ln.data_ptr(), 1,
                                       out.data_ptr(), B, Nq, Nq, 128, Smax, ws.data_ptr(), ws.numel(), _lib.stream_of(q)))
        return out

    alone = [call(c) for c in cases]
    torch.cuda.synchronize()
    streams = [torch.cuda.Stream(), torch.cuda.Stream()]
    outs = [[], []]
    seen_ws = [None, None]
    errors = []

    def worker(si):
        try:
            with torch.cuda.stream(streams[si]):
                seen_ws[si] = _lib.workspace(q).data_ptr()
                for it in range(24):
                    ci = (it + 2 * si) % len(cases)  # the two threads run different cases side by side
                    outs[si].append((ci, call(cases[ci])))
        except Exception as e:  # reported by the main thread
            errors.append((si, repr(e)))

    threads = [threading.Thread(target=worker, args=(si,)) for si in (0, 1)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    torch.cuda.synchronize()
    assert not errors, errors
    assert len({seen_ws[0], seen_ws[1], _lib.workspace(q).data_ptr()}) == 3, "each stream works in a workspace of its own"
    for si in (0, 1):
        assert len(outs[si]) == 24
        for it, (ci, y) in enumerate(outs[si]):
            assert torch.equal(y, alone[ci]), f"thread {si}, launch {it}, case {ci}: differs from the single-stream result"


@pytest.mark.parametrize("M", [1, 5, 16])
@pytest.mark.parametrize("widths", [(512, 512, 512), (768, 256, 256), (512, 128)])
def test_qkv_one_gemm_over_concatenated_weights(M, widths, monkeypatch):
    """Decode steps run q/k/v as ONE GEMM over the concatenated native weights with three output matrices
    (tppx_qkv_linear_mxfp4): the same bits as the segment-table launch and as separate calls, with and without the
    RMSNorm in the launch (from handed row sums, or formed in the launch), with some biases missing; the projections'
    own native copies become views into the concatenation and keep working on their own."""
    from tpp_pytorch_extension import _ops as ops
    _ops()
    K = 2048
    ws = [_make("mxfp4", n, K, 140 + i)[0] for i, n in enumerate(widths)]
    bs = [randn_bf16((widths[0],), 0.01, 150).cuda()] + [None] * (len(widths) - 1)
    x = randn_bf16((M, K), 1.0, 160 + M).cuda()
    gamma = (torch.rand(K) + 0.5).cuda()
    monkeypatch.setattr(ops, "QKV_ONE_GEMM", False)
    seg = ops.qkv_gemm(x, ws, bs)
    monkeypatch.setattr(ops, "QKV_ONE_GEMM", True)
    one = ops.qkv_gemm(x, ws, bs)
    assert getattr(ws[0], "_tppx_qkv_cat", None) is not None  # the one-GEMM path ran
    for a, b, w, bias in zip(one, seg, ws, bs):
        assert a.shape == b.shape and a.is_contiguous() and torch.equal(a, b)
        assert torch.equal(a, ops.fc_plain(x, w, bias))  # native views into the concatenation
    # RMSNorm inside the launch, sums formed there
    monkeypatch.setattr(ops, "FUSE_NORM", True)
    monkeypatch.setattr(ops, "QKV_ONE_GEMM", False)
    seg_n = ops.qkv_gemm(x, ws, bs, norm=(gamma, 1e-5))
    monkeypatch.setattr(ops, "QKV_ONE_GEMM", True)
    one_n = ops.qkv_gemm(x, ws, bs, norm=(gamma, 1e-5))
    for a, b in zip(one_n, seg_n):
        assert torch.equal(a, b)
    # RMSNorm from the row sums a producing GEMM left (here: formed by hand in the table's layout, slot 0 of 256)
    table = ops.sums_table(x.device)
    table[:M, 0] = (x.float() ** 2).sum(-1)
    monkeypatch.setattr(ops, "QKV_ONE_GEMM", False)
    seg_s = ops.qkv_gemm(x, ws, bs, norm=(gamma, 1e-5, table))
    monkeypatch.setattr(ops, "QKV_ONE_GEMM", True)
    one_s = ops.qkv_gemm(x, ws, bs, norm=(gamma, 1e-5, table))
    for a, b in zip(one_s, seg_s):
        assert torch.equal(a, b)


@pytest.mark.parametrize("tile", [4, 5])
@pytest.mark.parametrize("M,N,K", [(65, 160, 128), (129, 544, 256), (300, 544, 384), (200, 1056, 640), (70, 2080, 2048)])
def test_prefill_mxfp4_ring_tiles(tile, M, N, K, monkeypatch):
    """The 64 x 128 and 128 x 128 workgroup tiles (operands in a ring of three LDS stages), forced: fewer K steps than
    stages, as many and more, ragged rows and channel blocks.  Same sums in the same order as the 256 x 256 tile: the
    same bits, for a single GEMM, fused q/k/v and the gate/up pair; the single GEMM against the oracle."""
    ops = _ops()
    w, q_or, s_or = _make("mxfp4", N, K, 740)[:3]
    ws = [_make("mxfp4", n, K, 741 + i)[0] for i, n in enumerate((N, 64, 96))]
    wu = _make("mxfp4", N, K, 745)[0]
    x = randn_bf16((M, K), 1.0, 746)
    xg = x.cuda()

    def run():
        return [ops.fc_plain(xg, w, None)] + list(ops.qkv_gemm(xg, ws, [None] * 3)) + [ops.swiglu_gate_up(xg, w, wu)]

    monkeypatch.setenv("TPPX_TILED_MIN_M", "0")  # the LDS-tiled family whatever the cost estimate says
    monkeypatch.setenv("TPPX_TILED_BIG_TILE", "1")
    want = run()
    monkeypatch.setenv("TPPX_TILED_BIG_TILE", str(tile))
    got = run()
    ref = O.linear_mxfp4(t2bits(x), q_or, s_or, None, O.POST_NONE, None, None, 1.0, O.MODE_IDEAL)
    assert_close_bf16(t2bits(got[0]), ref, ulps=1, what=f"tile {tile}")
    for i, (a, b) in enumerate(zip(got, want)):
        assert torch.equal(a, b), i


@pytest.mark.parametrize("M", [65, 150, 333, 1000])
@pytest.mark.parametrize("shape", [((1056, 64, 96), 640), ((4096, 1024, 1024), 256), ((2080, 2080), 128)])
def test_prefill_bf16_groups_agree_with_single_launches(M, shape, monkeypatch):
    """q/k/v and the gate/up pair on unquantized bf16 weights as one launch: the same sums in the same order as one
    launch per weight (ragged rows and channel blocks, one K step and several, biases on some), hence the same bits;
    every projection against a float64 product (bf16 rounding of the sum and of the result)."""
    ops = _ops()
    widths, K = shape
    ws = [block_bf16(randn_bf16((n, K), 0.05, 750 + i)).cuda() for i, n in enumerate(widths)]
    bs = [randn_bf16((widths[0],), 0.5, 755).cuda()] + [None] * (len(widths) - 1)
    wu = block_bf16(randn_bf16((widths[0], K), 0.05, 756)).cuda()
    x = randn_bf16((M, K), 1.0, 757).cuda()
    monkeypatch.setenv("TPPX_TILED_MIN_M", "0")  # the LDS-tiled family whatever the cost estimate says
    got = ops._bf16_group(x, ws, bs)
    pair = ops._bf16_group(x, [ws[0], wu], [bs[0], None], pair=True)
    assert got is not None and pair is not None
    for i, (w, b) in enumerate(zip(ws, bs)):
        assert torch.equal(got[i], ops.linear(x, w, b)), i
        flat = randn_bf16((widths[i], K), 0.05, 750 + i).cuda().double()
        want = x.double() @ flat.t() + (b.double() if b is not None else 0.0)
        assert ((got[i].double() - want).norm() / want.norm()).item() < 2.0 ** -8, i
    assert torch.equal(pair, ops.fc_mul(x, wu, None, ops.fc_silu(x, ws[0], bs[0])))
    assert all(torch.equal(a, b) for a, b in zip(ops.qkv_gemm(x, ws, bs), got))


# rows around the row groups (16, 32, 64), one K tile and fewer than a workgroup has waves, widths that take one, two and three
# channel tiles per workgroup, the last of a GEMM ragged
@pytest.mark.parametrize("M", [1, 16, 17, 32, 33, 64])
@pytest.mark.parametrize("shape", [((4112, 16, 48, 80), 128), ((4096, 4096, 4096), 256), ((5136, 5120), 640), ((1056, 64, 96), 2176)])
def test_decode_bf16_groups_agree_with_single_launches(M, shape):
    """q/k/v (a fourth with its GELU) and the gate/up pair on unquantized bf16 weights as one launch of the decode kernel:
    the bits of one launch per weight, which other tests hold against the oracle."""
    ops = _ops()
    widths, K = shape
    ws = [block_bf16(randn_bf16((n, K), 0.05, 1750 + i)).cuda() for i, n in enumerate(widths)]
    bs = [randn_bf16((widths[0],), 0.5, 1755).cuda()] + [None] * (len(widths) - 1)
    wu = block_bf16(randn_bf16((widths[0], K), 0.05, 1756)).cuda()
    x = randn_bf16((M, K), 1.0, 1757).cuda()
    got = ops._bf16_group(x, ws, bs)
    pair = ops._bf16_group(x, [ws[0], wu], [bs[0], None], pair=True)
    assert got is not None and pair is not None
    for i, (w, b) in enumerate(zip(ws, bs)):
        assert torch.equal(got[i], ops.linear(x, w, b, O.POST_GELU if i == 3 else O.POST_NONE)), i
    assert torch.equal(pair, ops.fc_mul(x, wu, None, ops.fc_silu(x, ws[0], bs[0])))
    want = x.double() @ randn_bf16((widths[1], K), 0.05, 1751).cuda().double().t()
    assert ((got[1].double() - want).norm() / want.norm()).item() < 2.0 ** -8


@pytest.mark.parametrize("tile,w8", [(1, 1), (2, 1), (2, 0), (3, 1), (4, 1)])
@pytest.mark.parametrize("M,N,K", [(65, 160, 128), (129, 544, 256), (300, 544, 384), (200, 1056, 640)])
def test_prefill_bf16_every_workgroup_tile_ragged(tile, w8, M, N, K, monkeypatch):
    """Every workgroup tile for unquantized bf16 weights (256 x 256, 128 x 256 with eight and with four waves, 128 x 512,
    64 x 128), forced: a single GEMM, q/k/v with the fourth GEMM's GELU, and the gate/up pair, over one, an even and an
    odd number of K steps, rows and channel blocks ragged.  Same sums in the same order in every tile, hence the bits of
    the 64 x 128 one, which are checked against a float64 product (bf16 rounding of the result)."""
    ops = _ops()
    widths = (N, 64, 96, 160)
    flat = [randn_bf16((n, K), 0.05, 780 + i) for i, n in enumerate(widths + (N,))]
    ws = [block_bf16(w).cuda() for w in flat]
    bs = [randn_bf16((N,), 0.5, 786).cuda(), None, None, randn_bf16((160,), 0.5, 787).cuda()]
    x = randn_bf16((M, K), 1.0, 788).cuda()

    def run():
        group = ops._bf16_group(x, ws[:4], bs)
        pair = ops._bf16_group(x, [ws[0], ws[4]], [bs[0], None], pair=True)
        assert group is not None and pair is not None
        return [ops.linear(x, ws[0], bs[0]), pair] + list(group)

    monkeypatch.setenv("TPPX_TILED_MIN_M", "0")  # the LDS-tiled family whatever the cost estimate says
    monkeypatch.setenv("TPPX_TILED_W8", str(w8))
    monkeypatch.setenv("TPPX_TILED_BIG_TILE", str(tile))
    got = run()
    monkeypatch.setenv("TPPX_TILED_BIG_TILE", "4")
    want = run()
    for i, (a, b) in enumerate(zip(got, want)):
        assert torch.equal(a, b), i
    for i, (w, b) in enumerate(zip(flat[:3], bs[:3])):
        ref = x.double() @ w.cuda().double().t() + (b.double() if b is not None else 0.0)
        assert ((got[2 + i].double() - ref).norm() / ref.norm()).item() < 2.0 ** -8, i
    assert torch.equal(got[0], got[2])
    assert torch.equal(got[1], ops.fc_mul(x, ws[4], None, ops.fc_silu(x, ws[0], bs[0])))
    assert torch.equal(got[5], ops.linear(x, ws[3], bs[3], O.POST_GELU))
    assert all(torch.equal(a, b) for a, b in zip(ops.qkv_gemm(x, ws[:4], bs), got[2:]))


@pytest.mark.parametrize("M", [5, 200])
def test_bf16_entry_points_without_a_workspace(M):
    """tppx_linear_bf16, tppx_multi_linear_bf16 and tppx_swiglu_bf16: the bits of the forms with a workspace, given none."""
    from tpp_pytorch_extension import _lib
    ops = _ops()
    L, N, K = _lib.lib(), 4096, 3072
    nat = [ops._bf16_native(block_bf16(randn_bf16((N, K), 0.05, 1870 + i)).cuda()) for i in range(2)]
    x, st = randn_bf16((M, K), 1.0, 1872).cuda(), torch.cuda.current_stream().cuda_stream

    def run(ws):
        y = [torch.empty((M, N), dtype=torch.bfloat16, device="cuda") for _ in range(4)]
        segs = (_lib.Seg * 2)()
        for s, w, o in zip(segs, nat, y[1:]):
            s.qw = s.sw = w.data_ptr()
            s.y, s.N, s.post_op, s.post_scale = o.data_ptr(), N, O.POST_NONE, 1.0
        end = (None, 0, st) if ws else (st,)
        f = [getattr(L, f"tppx_{name}_bf16{'_ws' if ws else ''}") for name in ("linear", "multi_linear", "swiglu")]
        _lib.check(f[0](x.data_ptr(), nat[0].data_ptr(), None, None, None, y[0].data_ptr(), M, N, K, O.POST_SILU, 1.0, 0, *end))
        _lib.check(f[1](x.data_ptr(), segs, 2, M, K, 0, *end))
        _lib.check(f[2](x.data_ptr(), nat[0].data_ptr(), None, nat[1].data_ptr(), None, y[3].data_ptr(), M, N, K, 0, *end))
        return y

    assert all(torch.equal(a, b) for a, b in zip(run(False), run(True)))


# ragged rows and channel blocks, slices of unequal and of the fewest steps (four), each number of slices
@pytest.mark.parametrize("fmt", ["mxfp4", "bf16"])
@pytest.mark.parametrize("S,M,N,K", [(2, 65, 160, 1152), (3, 200, 288, 1792), (4, 129, 2080, 2048), (6, 100, 32, 3072), (6, 333, 416, 4224)])
def test_prompt_gemms_with_k_in_slices(fmt, S, M, N, K, monkeypatch):
    """K in S slices whose fp32 sums a second launch adds, in slice order: linear with its residual and bias, a post-op that
    goes through the general epilogue, and q/k/v with a fourth GELU GEMM, against the launch with K whole (another order of
    the fp32 sums: one bf16 ulp here and there) and a float64 product; every replay of a captured call the same."""
    from tpp_pytorch_extension import _lib
    ops = _ops()
    flat = [randn_bf16((n, K), 0.05, 1800 + i) for i, n in enumerate((N, 64, 96, 160))]
    ws = [block_bf16(w).cuda() for w in flat]
    if fmt == "mxfp4":
        ws = [ops.remap_and_quantize_mxfp4(w) for w in ws]
    x, res, b = randn_bf16((M, K), 1.0, 1805).cuda(), randn_bf16((M, N), 1.0, 1806).cuda(), randn_bf16((N,), 0.5, 1807).cuda()

    def run():
        return [ops.fc_add(x, ws[0], b, res, 0.5), ops.fc_add2(x, ws[0], b, res, res, 0.5)] + list(ops.qkv_gemm(x, ws, [b, None, None, None]))

    def left_sums():  # the slices' sums are what these launches write to the workspace
        return bool(_lib.workspace(x).any())

    monkeypatch.setenv("TPPX_TILED_MIN_M", "0")  # the LDS-tiled family whatever the cost estimate says
    monkeypatch.setenv("TPPX_TILED_SPLIT", "0")
    _lib.workspace(x).zero_()
    want = run()
    assert not left_sums()
    monkeypatch.setenv("TPPX_TILED_SPLIT", str(S))
    for call in (lambda: ops.fc_add(x, ws[0], b, res, 0.5), lambda: ops.qkv_gemm(x, ws, [b, None, None, None])):
        _lib.workspace(x).zero_()
        call()
        assert left_sums()
    got = run()
    for i, (a, w) in enumerate(zip(got, want)):
        a, w = a.double(), w.double()
        assert (a - w).norm() <= 2.0 ** -9 * w.norm(), i
        # the bf16 GEMM tile differs by one ulp, 2^-7 of it at most, and is at most |out| + 1.5 |residual|; one more ulp for
        # each of the two roundings behind it; sums near zero by the fp32 sums' own error
        near = w.abs() + (1.5 * res.double().abs() if i < 2 else 0.0)
        assert ((a - w).abs() <= 3 * 2.0 ** -7 * near + 2.0 ** -12 * w.abs().max()).all(), i
    if fmt == "mxfp4":
        import ctypes
        buf = ctypes.create_string_buffer(4096)
        _lib.check(_lib.lib().tppx_plan_linear_mxfp4(M, N, K, 0, 1 << 25, buf, len(buf)))
        assert "false, true> grid=" in buf.value.decode() and f"x{S}x1" in buf.value.decode()
    if fmt == "bf16":
        ref = x.double() @ flat[1].cuda().double().t()
        assert ((got[3].double() - ref).norm() / ref.norm()).item() < 2.0 ** -8
    y = torch.empty(0)
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g):
        y = ops.fc_add(x, ws[0], b, res, 0.5)
    for _ in range(3):
        y.zero_()
        g.replay()
        torch.cuda.synchronize()
        assert torch.equal(y, got[0])


@pytest.mark.parametrize("fmt", ["mxfp4", "qint8", "bf16"])
def test_captured_prompt_gemms_keep_their_slices_in_the_graphs_own_memory(fmt, monkeypatch):
    """K slices of a captured prompt leave their sums in a buffer of the graph's own, so that replays of two graphs on two
    streams need no order; decode steps use the device's capture buffer.  Every replay has the eager call's bits."""
    from tpp_pytorch_extension import _lib
    ops = _ops()
    K, N = 6144, 256
    ws = [block_bf16(randn_bf16((N, K), 0.05, 1850 + i)).cuda() for i in range(2)]
    if fmt != "bf16":
        ws = [{"mxfp4": ops.remap_and_quantize_mxfp4, "qint8": ops.remap_and_quantize_qint8}[fmt](w) for w in ws]
    lib, seen = _lib.lib(), []

    class Watch:
        def __getattr__(self, name):
            f = getattr(lib, name)
            if "linear" not in name:
                return f

            def call(*args):  # (every one of them ends in ws, ws_bytes, stream)
                seen.append((args[-3], args[-2]))
                return f(*args)
            return call

    for M, prompt in ((200, True), (64, False)):
        x = randn_bf16((M, K), 1.0, 1860).cuda()

        def run():
            return [ops.linear(x, ws[0], None)] + list(ops.qkv_gemm(x, ws, [None, None]))

        want = run()
        _lib.workspace(x)
        shared = _lib._workspaces[(x.device.index, "capture")]
        g, seen[:] = torch.cuda.CUDAGraph(), []
        with monkeypatch.context() as m:
            m.setattr(_lib, "lib", lambda: Watch())
            with torch.cuda.graph(g):
                got = run()
        assert seen
        if prompt:
            assert all(at != shared.data_ptr() and n == _lib.WORKSPACE_BYTES for at, n in seen)
        elif fmt != "bf16":
            assert all(at == shared.data_ptr() for at, n in seen)
        for _ in range(3):
            for y in got:
                y.zero_()
            g.replay()
            torch.cuda.synchronize()
            assert all(torch.equal(a, b) for a, b in zip(got, want))


@pytest.mark.parametrize("S,M,N,K", [(2, 65, 160, 512), (2, 200, 288, 1792), (3, 129, 2080, 1792), (4, 100, 32, 2304), (6, 333, 416, 3328)])
def test_prompt_qint8_gemms_with_k_in_slices(S, M, N, K, monkeypatch):
    """QINT8 the same: K in S slices of whole scale blocks (one block a slice, an odd and an even number), against the oracle
    to the tolerance of the launch with K whole."""
    import ctypes
    from tpp_pytorch_extension import _lib
    ops = _ops()
    monkeypatch.setenv("TPPX_TILED_MIN_M", "0")
    monkeypatch.setenv("TPPX_TILED_SPLIT", str(S))
    buf = ctypes.create_string_buffer(4096)
    _lib.check(_lib.lib().tppx_plan_linear_qint8(M, N, K, 256, 1, 0, 1 << 25, buf, len(buf)))
    assert f"big_qint8_split_kernel grid={(M + 63) // 64 * ((N + 127) // 128)}x{S}x1" in buf.value.decode()
    y, _, _, ctx = _run("qint8", M, N, K, "add", True, 1900 + M)  # (checks against the oracle)
    qw, _, _, x, bias, in1, in2, scale = ctx
    other = _make("qint8", 64, K, 1901)[0]
    q, k2 = ops.qkv_gemm(x.cuda(), [qw, other], [bias.cuda(), None])
    monkeypatch.setenv("TPPX_TILED_SPLIT", "0")
    for got, want in ((y, ops.linear(x.cuda(), qw, bias.cuda(), O.POST_ADD_SCALE, in1.cuda(), None, scale)),
                      (q, ops.fc_plain(x.cuda(), qw, bias.cuda())), (k2, ops.fc_plain(x.cuda(), other, None))):
        assert (got.double() - want.double()).norm() <= 2.0 ** -9 * want.double().norm()


@pytest.mark.parametrize("fmt", ["mxfp4", "bf16"])
@pytest.mark.parametrize("steps", [1, 2, 3, 4, 5, 7])
def test_prefill_side_by_side_forms_at_every_loop_remainder(fmt, steps, monkeypatch):
    """The forms whose waves keep the weights in registers (64 x 128; bf16: 64 x 256 and 128 x 256 as well) run their K steps
    of 128 by threes with a tail: one step up to two rounds and a remainder, rows and channel blocks ragged, against the
    256 x 256 form (the same sums in the same order, hence the same bits): linear, q/k/v, pair."""
    ops = _ops()
    M, N, K = 201, 288, 128 * steps
    if fmt == "mxfp4":
        ws = [_make("mxfp4", n, K, 940 + i)[0] for i, n in enumerate((N, 32, 160, N))]
        tiles = ("4",)
    else:
        ws = [block_bf16(randn_bf16((n, K), 0.05, 940 + i)).cuda() for i, n in enumerate((N, 32, 160, N))]
        tiles = ("4", "6", "2")
    x, b = randn_bf16((M, K), 1.0, 945).cuda(), randn_bf16((N,), 0.5, 946).cuda()

    def run():
        return [ops.fc_plain(x, ws[0], b), ops.swiglu_gate_up(x, ws[0], ws[3])] + list(ops.qkv_gemm(x, ws[:3], [b, None, None]))

    monkeypatch.setenv("TPPX_TILED_MIN_M", "0")  # the LDS-tiled family whatever the cost estimate says
    monkeypatch.setenv("TPPX_TILED_BIG_TILE", "1")
    want = run()
    for tile in tiles:
        monkeypatch.setenv("TPPX_TILED_BIG_TILE", tile)
        for i, (a, w) in enumerate(zip(run(), want)):
            assert torch.equal(a, w), (tile, i)


@pytest.mark.parametrize("fmt,tile", [("mxfp4", "17"), ("bf16", "11"), ("bf16", "15")])
@pytest.mark.parametrize("steps", [1, 2, 3, 4, 5, 7])
def test_prefill_wave_tiles_at_every_loop_remainder(fmt, tile, steps, monkeypatch):
    """The same for wave tiles with a ring of three stages (those of up to 64 rows, 64 x 128 above among them, have four)."""
    ops = _ops()
    M, N, K = 201, 288, 128 * steps
    if fmt == "mxfp4":
        ws = [_make("mxfp4", n, K, 940 + i)[0] for i, n in enumerate((N, 32, 160, N))]
    else:
        ws = [block_bf16(randn_bf16((n, K), 0.05, 940 + i)).cuda() for i, n in enumerate((N, 32, 160, N))]
    x, b = randn_bf16((M, K), 1.0, 945).cuda(), randn_bf16((N,), 0.5, 946).cuda()

    def run():
        return [ops.fc_plain(x, ws[0], b), ops.swiglu_gate_up(x, ws[0], ws[3])] + list(ops.qkv_gemm(x, ws[:3], [b, None, None]))

    monkeypatch.setenv("TPPX_TILED_MIN_M", "0")  # the LDS-tiled family whatever the cost estimate says
    monkeypatch.setenv("TPPX_TILED_BIG_TILE", "1")
    want = run()
    monkeypatch.setenv("TPPX_TILED_BIG_TILE", tile)
    for i, (a, w) in enumerate(zip(run(), want)):
        assert torch.equal(a, w), i


@pytest.mark.parametrize("fmt,forms", [("mxfp4", range(7, 18)), ("bf16", (11, 15))])
@pytest.mark.parametrize("M,N,K", [(65, 1056, 128), (70, 288, 640), (97, 1568, 896), (201, 352, 1152), (333, 800, 512)])
def test_prefill_wave_tiles_agree(fmt, forms, M, N, K, monkeypatch):
    """Every wave tile of the launches of up to a few workgroups per CU: 1 .. 9 K steps (rings of three and four stages), rows and
    channel blocks ragged (row tiles of a block past the end, one live channel tile of a wave's three), a pair dealt out over
    the waves, the residual's read-ahead, against the 256 x 256 form: the same sums in the same order, hence the same bits."""
    from tpp_pytorch_extension import _lib
    ops = _ops()
    if fmt == "mxfp4":
        ws = [_make("mxfp4", n, K, 950 + i)[0] for i, n in enumerate((N, 32, 160, N))]
    else:
        ws = [block_bf16(randn_bf16((n, K), 0.05, 950 + i)).cuda() for i, n in enumerate((N, 32, 160, N))]
    x, res, b = randn_bf16((M, K), 1.0, 955).cuda(), randn_bf16((M, N), 1.0, 956).cuda(), randn_bf16((N,), 0.5, 957).cuda()

    def run():
        return [ops.fc_add(x, ws[0], b, res, 0.5), ops.fc_gelu(x, ws[0], b), ops.swiglu_gate_up(x, ws[0], ws[3], b, None)] + \
            list(ops.qkv_gemm(x, ws[:3], [b, None, None]))

    monkeypatch.setenv("TPPX_TILED_MIN_M", "0")  # the LDS-tiled family whatever the cost estimate says
    monkeypatch.setenv("TPPX_TILED_SPLIT", "0")
    monkeypatch.setenv("TPPX_TILED_BIG_TILE", "1")
    want = run()
    for form in forms:
        monkeypatch.setenv("TPPX_TILED_BIG_TILE", str(form))
        for i, (a, w) in enumerate(zip(run(), want)):
            assert torch.equal(a, w), (form, i)


@pytest.mark.parametrize("S", [2, 3, 4, 6])
@pytest.mark.parametrize("form", [7, 8, 9])
def test_prefill_wave_tiles_with_k_in_slices(form, S, monkeypatch):
    """Slices of unequal steps on each wave tile that has them, and without room for their sums (K whole, the same call)."""
    import ctypes
    from tpp_pytorch_extension import _lib
    ops = _ops()
    M, N, K = 77, 288, 128 * (4 * S + 3)
    w = _make("mxfp4", N, K, 960 + S)[0]
    x, res = randn_bf16((M, K), 1.0, 961).cuda(), randn_bf16((M, N), 1.0, 962).cuda()
    monkeypatch.setenv("TPPX_TILED_MIN_M", "0")
    monkeypatch.setenv("TPPX_TILED_BIG_TILE", str(form))
    monkeypatch.setenv("TPPX_TILED_SPLIT", "0")
    want = ops.fc_add(x, w, None, res, 1.0).double()
    monkeypatch.setenv("TPPX_TILED_SPLIT", str(S))
    got = ops.fc_add(x, w, None, res, 1.0).double()
    assert (got - want).norm() <= 2.0 ** -9 * want.norm()
    buf = ctypes.create_string_buffer(4096)
    for ws_bytes, slices in ((1 << 25, True), (1 << 12, False)):
        _lib.check(_lib.lib().tppx_plan_linear_mxfp4(M, N, K, 0, ws_bytes, buf, len(buf)))
        assert ("wide_sum_kernel" in buf.value.decode()) == slices, ws_bytes


@pytest.mark.parametrize("M,N,K", [(65, 16, 256), (64 * 3, 272, 512), (129, 4080, 768), (300, 8208, 1024), (1000, 1040, 1280)])
def test_prefill_qint8_forms_agree_with_the_oracle(M, N, K, monkeypatch):
    """The large-M QINT8 kernel from one K step to five (odd and even: its loop goes by two), a single channel tile, ragged
    rows and channel blocks: 64 x 128, 64 x 256 and 128 x 256 workgroups as the launch picks them against the oracle, and the
    bits of the 128 x 256 form, for the GEMM with its residual and for the gate/up pair."""
    from tpp_pytorch_extension import _lib
    ops = _ops()
    y, _, _, ctx = _run("qint8", M, N, K, "add", True, 900 + M, flags=_lib.FLAG_FORCE_TILED)
    qw, _, _, x, bias, in1, in2, scale = ctx
    monkeypatch.setenv("TPPX_TILED_MIN_M", "0")
    wu = _make("qint8", N, K, 901 + M)[0]
    pair = ops.swiglu_gate_up(x.cuda(), qw, wu, bias.cuda(), None)
    assert torch.equal(pair, ops.fc_mul(x.cuda(), wu, None, ops.fc_silu(x.cuda(), qw, bias.cuda())))
    monkeypatch.setenv("TPPX_TILED_SMALL", "0")
    assert torch.equal(y, ops.linear(x.cuda(), qw, bias.cuda(), O.POST_ADD_SCALE, in1.cuda(), None, scale))
    assert torch.equal(pair, ops.swiglu_gate_up(x.cuda(), qw, wu, bias.cuda(), None))


@pytest.mark.parametrize("fmt", ["qint8", "qint4"])
@pytest.mark.parametrize("M,N,K", [(65, 160, 256), (129, 544, 512), (300, 96, 768), (200, 2080, 1280), (1000, 4160, 512)])
def test_prefill_qint8_pair_agrees_with_two_launches(fmt, M, N, K, monkeypatch):
    """The gate/up pair of QINT8-family weights as one launch: the same sums in the same order and the same rounding
    points as fc_silu followed by fc_mul, hence the same bits (one scale block and several, ragged rows and channel
    blocks, the 64-row and the 128-row workgroups, a bias on one of the two)."""
    ops = _ops()
    monkeypatch.setenv("TPPX_TILED_MIN_M", "0")  # the LDS-tiled family whatever the cost estimate says
    quant = {"qint8": ops.remap_and_quantize_qint8, "qint4": lambda t: ops.quantize_int4sym(t, 256, 2, True)}[fmt]
    ws = [quant(block_bf16(randn_bf16((N, K), 0.05, 760 + i), bc=256).cuda()) for i in range(2)]
    b = randn_bf16((N,), 0.5, 762).cuda()
    x = randn_bf16((M, K), 1.0, 763).cuda()
    with monkeypatch.context() as m:
        m.setattr(ops, "linear", None)  # (the two launches would call it)
        got = ops.swiglu_gate_up(x, ws[0], ws[1], b, None)
    assert torch.equal(got, ops.fc_mul(x, ws[1], None, ops.fc_silu(x, ws[0], b)))


@pytest.mark.parametrize("fmt,M,N,K", [("qint8", 66, 5120, 2048), ("qint8", 128, 1536, 1024), ("bf16", 65, 64, 2048), ("bf16", 100, 32, 4096)])
def test_groups_that_run_per_weight_are_asked_about_first(fmt, M, N, K, monkeypatch):
    """Where the library would answer TPPX_EUNSUPPORTED to a gate/up pair or a q/k/v group (few rows on small weights;
    QINT8: by the row threshold, its estimate takes every pair), the call is not made and nothing is prepared for it:
    the outputs are those of one call per weight."""
    from tpp_pytorch_extension import _lib
    ops = _ops()
    if fmt == "qint8":
        monkeypatch.setenv("TPPX_TILED_MIN_M", "512")
    ws = [block_bf16(randn_bf16((N, K), 0.05, 775 + i), bc=256).cuda() for i in range(2)]
    if fmt == "qint8":
        ws = [ops.remap_and_quantize_qint8(w) for w in ws]
    x = randn_bf16((M, K), 1.0, 777).cuda()
    want = ops.fc_mul(x, ws[1], None, ops.fc_silu(x, ws[0], None))
    qkv = [ops.fc_plain(x, w, None) for w in ws]
    lib = _lib.lib()

    class Without:
        def __getattr__(self, name):
            assert not name.startswith(("tppx_swiglu_qint8", "tppx_swiglu_bf16", "tppx_multi_linear_bf16")), name
            return getattr(lib, name)

    monkeypatch.setattr(_lib, "lib", lambda: Without())
    assert torch.equal(ops.swiglu_gate_up(x, ws[0], ws[1]), want)
    if fmt == "bf16":
        assert all(torch.equal(a, b) for a, b in zip(ops.qkv_gemm(x, ws, [None] * 2), qkv))


@pytest.mark.parametrize("M", [1, 17, 64, 65, 128, 129, 300])
@pytest.mark.parametrize("N,K", [(64, 2048), (1536, 1024), (5120, 2048)])
def test_group_is_one_launch_answers_as_the_calls_do(M, N, K):
    """tppx_group_is_one_launch against what tppx_swiglu_bf16 and tppx_swiglu_qint8 do with the same shape."""
    import ctypes
    from tpp_pytorch_extension import _lib
    ops = _ops()
    L = _lib.lib()
    w = block_bf16(randn_bf16((N, K), 0.05, 778), bc=256).cuda()
    nat, (q, s) = ops._bf16_native(w), ops.remap_and_quantize_qint8(w).native()
    x = randn_bf16((M, K), 1.0, 779).cuda()
    y = torch.empty((M, N), dtype=torch.bfloat16, device="cuda")
    xq, sa = qint8_scratch(x, M, K, 256)
    st, ns = _lib.stream_of(x), (ctypes.c_int64 * 2)(N, N)
    rc = L.tppx_swiglu_bf16(x.data_ptr(), nat.data_ptr(), None, nat.data_ptr(), None, y.data_ptr(), M, N, K, 0, st)
    assert rc in (_lib.OK, _lib.EUNSUPPORTED) and (rc == _lib.OK) == bool(L.tppx_group_is_one_launch(ns, 2, M, K, 2))
    rc = L.tppx_swiglu_qint8(x.data_ptr(), xq.data_ptr(), sa.data_ptr(), q.data_ptr(), s.data_ptr(), None, q.data_ptr(),
                             s.data_ptr(), None, y.data_ptr(), M, N, K, 256, 0, st)
    assert rc in (_lib.OK, _lib.EUNSUPPORTED) and (rc == _lib.OK) == bool(L.tppx_group_is_one_launch(ns, 2, M, K, 1))


def test_prefill_qint8_pair_of_2_31_outputs():
    """The QINT8 gate/up pair with more than 2^31 outputs (64-bit output offsets in the large-M kernels): one launch as
    for fewer, the bits of fc_silu followed by fc_mul."""
    ops = _ops()
    M, N, K = 32800, 65536, 256
    assert M * N >= 1 << 31
    ws = [ops.remap_and_quantize_qint8(block_bf16(randn_bf16((N, K), 0.05, 770 + i)).cuda()) for i in range(2)]
    x = randn_bf16((M, K), 1.0, 772).cuda()
    got = ops.swiglu_gate_up(x, ws[0], ws[1])
    assert torch.equal(got, ops.fc_mul(x, ws[1], None, ops.fc_silu(x, ws[0], None)))


@pytest.mark.parametrize("off", [1, 2])
@pytest.mark.parametrize("M,N,K", [(70, 544, 256), (200, 1056, 640), (300, 96, 1280)])
def test_prefill_mxfp4_takes_scales_at_any_address(off, M, N, K, monkeypatch):
    """Native scale bytes off a 4-byte address (a view into a packed buffer): the bits of aligned ones, for a linear,
    fused q/k/v and the gate/up pair, whichever workgroup tile is asked for."""
    ops = _ops()
    ws = [_make("mxfp4", N, K, 780 + i)[0] for i in range(3)]
    x = randn_bf16((M, K), 1.0, 785).cuda()

    def run():
        return [ops.fc_plain(x, ws[0], None)] + list(ops.qkv_gemm(x, ws, [None] * 3)) + [ops.swiglu_gate_up(x, ws[0], ws[1])]

    monkeypatch.setenv("TPPX_TILED_MIN_M", "0")  # the LDS-tiled family whatever the cost estimate says
    want = run()
    for w in ws:
        qn, sn = w.native()
        buf = torch.empty(sn.numel() + 16, dtype=sn.dtype, device=sn.device)
        buf[off:off + sn.numel()] = sn.reshape(-1)
        w._native = (qn, buf[off:off + sn.numel()].view(sn.shape))
        assert w._native[1].data_ptr() % 4 == off
    for tile in ("0", "2", "4", "5"):
        monkeypatch.setenv("TPPX_TILED_BIG_TILE", tile)
        for a, b in zip(run(), want):
            assert torch.equal(a, b), tile


@pytest.mark.parametrize("off", [1, 2])
@pytest.mark.parametrize("tile", ["7", "8", "10", "12", "13", "14", "15", "16", "17"])
def test_prefill_mxfp4_wave_tiles_take_scales_at_any_address(off, tile, monkeypatch):
    """The same for every wave tile: 200 ragged rows, a last channel block of two tiles, five K steps."""
    ops = _ops()
    N, K = 1056, 640
    ws = [_make("mxfp4", N, K, 780 + i)[0] for i in range(3)]
    x = randn_bf16((200, K), 1.0, 785).cuda()

    def run():
        return [ops.fc_plain(x, ws[0], None)] + list(ops.qkv_gemm(x, ws, [None] * 3)) + [ops.swiglu_gate_up(x, ws[0], ws[1])]

    monkeypatch.setenv("TPPX_TILED_MIN_M", "0")  # the LDS-tiled family whatever the cost estimate says
    want = run()
    for w in ws:
        qn, sn = w.native()
        buf = torch.empty(sn.numel() + 16, dtype=sn.dtype, device=sn.device)
        buf[off:off + sn.numel()] = sn.reshape(-1)
        w._native = (qn, buf[off:off + sn.numel()].view(sn.shape))
    monkeypatch.setenv("TPPX_TILED_BIG_TILE", tile)
    for a, b in zip(run(), want):
        assert torch.equal(a, b)


@pytest.mark.parametrize("M", [1, 9, 16, 17, 31, 33, 50, 64, 70])
@pytest.mark.parametrize("tiles", [1, 8, 13, 24, 33, 47])
def test_row_groups_at_every_number_of_k_tiles_per_wave(M, tiles):
    """The row-group kernel (MXFP4 at 17..64 rows and where K does not suit the LDS-staged kernels; bf16 weights): waves
    without K tiles, with one, two, three and more, odd and even counts in one workgroup, rows past M.  MXFP4: the GEMM
    against the oracle, the gate/up pair against its two GEMMs one after the other (the same three roundings to bf16, of
    sums in another order); bf16 against the product in float64 (one rounding)."""
    from tpp_pytorch_extension import _lib
    ops = _ops()
    K = 128 * tiles
    _, _, _, ctx = _run("mxfp4", M, 96, K, "add", True, 700 + tiles, flags=_lib.FLAG_FORCE_SKINNY)
    wg, x = ctx[0], ctx[3].cuda()
    wu = _make("mxfp4", 96, K, 770 + tiles)[0]
    want = ops.fc_mul(x, wu, None, ops.fc_silu(x, wg, None)).float()
    got = ops.swiglu_gate_up(x, wg, wu).float()
    assert ((got - want).norm() / want.norm()).item() < 3 * 2.0 ** -9
    w = randn_bf16((96, K), 0.05, 790 + tiles)
    got = ops.linear(x, block_bf16(w).cuda(), None, flags=_lib.FLAG_FORCE_SKINNY).double()
    want = x.double() @ w.cuda().double().t()
    assert ((got - want).norm() / want.norm()).item() < 2.0 ** -8
