"""Host-side checks that need no GPU: the C-ABI library loads and exports every
entry point include/tppx.h declares, arguments are validated before any HIP
call (error codes, never a crash or exit), and the Python drop-in layer
(blocked layouts, module classes, helper names) behaves like the reference's.
"""
import ctypes
import os
import re

import pytest
import torch

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def _lib():
    import tpp_pytorch_extension  # noqa: F401
    from tpp_pytorch_extension import _lib
    return _lib


def test_header_symbols_are_exported_and_bound():
    L = _lib()
    hdr = open(os.path.join(ROOT, "include", "tppx.h")).read()
    hdr = re.sub(r"/\*.*?\*/", "", hdr, flags=re.S)
    declared = set(re.findall(r"\b(tppx_[a-z0-9_]+)\s*\(", hdr))
    assert len(declared) >= 14
    lib = L.lib()
    for name in declared:
        assert hasattr(lib, name), f"{name} is declared in tppx.h but not exported"
    assert declared == set(L.SIGNATURES), "ctypes signatures and tppx.h disagree"
    assert lib.tppx_version() == 100


def test_seg_struct_matches_header_layout():
    L = _lib()
    # 6 pointers, int64, int32, float
    assert ctypes.sizeof(L.Seg) == 6 * 8 + 8 + 4 + 4
    assert L.Seg.N.offset == 48 and L.Seg.post_op.offset == 56 and L.Seg.post_scale.offset == 60


def test_argument_validation_without_gpu():
    L = _lib()
    lib = L.lib()
    A = 1 << 20  # a fake, 16-byte aligned "device pointer": validation must reject before touching it

    def err():
        return lib.tppx_last_error().decode()

    # null pointers
    assert lib.tppx_linear_mxfp4(None, A, A, None, None, None, A, 1, 32, 128, 0, 1.0, 0, None, 0, None) == L.EINVAL
    assert "null" in err()
    assert lib.tppx_linear_qint8(A, None, A, A, A, None, None, None, A, 1, 16, 256, 256, 0, 1.0, 0, None, 0, None) == L.EINVAL
    # misaligned
    assert lib.tppx_linear_mxfp4(A + 2, A, A, None, None, None, A, 1, 32, 128, 0, 1.0, 0, None, 0, None) == L.EINVAL
    assert "aligned" in err()
    # shapes: M = 0, K not a multiple of 64, N not a multiple of 32 / 16, block size mismatch
    assert lib.tppx_linear_mxfp4(A, A, A, None, None, None, A, 0, 32, 128, 0, 1.0, 0, None, 0, None) == L.ESHAPE
    assert lib.tppx_linear_mxfp4(A, A, A, None, None, None, A, 1, 32, 100, 0, 1.0, 0, None, 0, None) == L.ESHAPE
    assert lib.tppx_linear_mxfp4(A, A, A, None, None, None, A, 1, 48, 128, 0, 1.0, 0, None, 0, None) == L.ESHAPE
    assert lib.tppx_linear_mxfp4(A, A, A, None, None, None, A, 1, 32, 192, 0, 1.0, 0, None, 0, None) == L.EUNSUPPORTED
    assert lib.tppx_linear_qint8(A, A, A, A, A, None, None, None, A, 1, 24, 256, 256, 0, 1.0, 0, None, 0, None) == L.ESHAPE
    assert lib.tppx_linear_qint8(A, A, A, A, A, None, None, None, A, 1, 16, 256, 192, 0, 1.0, 0, None, 0, None) == L.ESHAPE
    assert "block size" in err()
    # unquantized bf16 weights: K in whole 128-channel tiles, N in 16s, blocking must divide the matrix
    assert lib.tppx_linear_bf16(A, A, None, None, None, A, 1, 16, 192, 0, 1.0, 0, None) == L.ESHAPE
    assert lib.tppx_linear_bf16(A, A, None, None, None, A, 1, 24, 128, 0, 1.0, 0, None) == L.ESHAPE
    assert lib.tppx_linear_bf16(A, None, None, None, None, A, 1, 16, 128, 0, 1.0, 0, None) == L.EINVAL
    assert lib.tppx_prepack_bf16(A, 32, 256, 16, 48, 2, A, None) == L.ESHAPE
    assert lib.tppx_prepack_bf16(A, 32, 256, 16, 64, 3, A, None) == L.ESHAPE
    # W4A8 row groups: scales are read 16 bytes at a time; what does not fit the kernel's offsets is left to others
    mid = lambda s, M=32, N=32, K=128: lib.tppx_linear_mxfp4_int8_mid(A, A, A, A, s, None, None, None, A, M, N, K, 0, 1.0, 0, None)  # noqa: E731
    assert mid(A + 4) == L.EINVAL and "aligned" in err()
    assert mid(A, M=64, N=1 << 25) == L.EUNSUPPORTED and mid(A, K=65536 * 128) == L.EUNSUPPORTED
    assert mid(A, M=0) == L.ESHAPE and mid(A, K=192) == L.ESHAPE
    # post-op id and its inputs
    assert lib.tppx_linear_mxfp4(A, A, A, None, None, None, A, 1, 32, 128, 9, 1.0, 0, None, 0, None) == L.EINVAL
    assert lib.tppx_linear_mxfp4(A, A, A, None, None, None, A, 1, 32, 128, L.POST_MUL, 1.0, 0, None, 0, None) == L.EINVAL
    assert "post_in" in err()
    assert lib.tppx_linear_mxfp4(A, A, A, None, A, None, A, 1, 32, 128, L.POST_ADD2_SCALE, 1.0, 0, None, 0, None) == L.EINVAL
    # flags and workspace
    assert lib.tppx_linear_mxfp4(A, A, A, None, None, None, A, 1, 32, 128, 0, 1.0, 64, None, 0, None) == L.EINVAL
    assert lib.tppx_linear_mxfp4(A, A, A, None, None, None, A, 1, 32, 128, 0, 1.0, 3, None, 0, None) == L.EINVAL
    assert lib.tppx_linear_mxfp4(A, A, A, None, None, None, A, 1, 32, 128, 0, 1.0, 0, None, 4096, None) == L.EINVAL
    # fused groups
    segs = (L.Seg * 5)()
    assert lib.tppx_multi_linear_mxfp4(A, segs, 5, 1, 128, 0, None, 0, None) == L.EINVAL
    assert lib.tppx_multi_linear_mxfp4(A, segs, 0, 1, 128, 0, None, 0, None) == L.EINVAL
    # quantizers
    assert lib.tppx_quantize_mxfp4(A, 0, 48, 128, 16, 64, 2, A, A, None) == L.ESHAPE
    assert lib.tppx_quantize_mxfp4(A, 7, 64, 128, 16, 64, 2, A, A, None) == L.EINVAL
    assert lib.tppx_quantize_qint8(A, 1, 64, 128, 16, 64, 2, 96, A, A, None) == L.ESHAPE
    assert lib.tppx_quant_act_int8(A, 1, 100, 256, A, A, None) == L.ESHAPE
    assert lib.tppx_prepack_mxfp4(A, A, 64, 192, A, A, None) == L.ESHAPE
    assert lib.tppx_dequantize_qint8(None, A, 16, 256, 256, A, None) == L.EINVAL


def test_python_layer_fails_loudly_without_gpu():
    L = _lib()
    from tpp_pytorch_extension._C import _qtype
    if torch.cuda.is_available():
        pytest.skip("checks the no-GPU behaviour")
    w = torch.randn(64, 128).to(torch.bfloat16).view(4, 16, 2, 32, 2).permute(0, 2, 3, 1, 4).contiguous()
    with pytest.raises(L.TppxError):
        _qtype.remap_and_quantize_mxfp4(w)
    with pytest.raises(L.TppxError):
        torch.ops.tpp_llm.fc_plain(torch.randn(2, 128), torch.randn(64, 128), torch.Tensor(), -1, [])


def test_reference_names_are_importable():
    import tpp_pytorch_extension as tpx
    from tpp_pytorch_extension import qtypes, nn
    from tpp_pytorch_extension._C import _qtype, _fused_llm_infer
    from tpp_pytorch_extension.llm import llm_common
    from tpp_pytorch_extension.utils import blocked_layout
    for n in ("quantize_mxfp", "quantize_mxfp4", "quantize_int8sym", "quantize_int4sym", "create_qtensor_int8sym",
              "create_qtensor_int2sym", "q_per_block_scales", "q_per_block_pack_size", "q_per_block_block_size",
              "q_per_block_axis", "remap_and_quantize_mxfp4", "remap_and_quantize_qint8",
              "remap_and_quantize_qint2_intlv", "fix_vnni"):
        assert callable(getattr(_qtype, n)), n
    for n in ("get_qval", "get_scales", "get_axis", "get_block_size", "q_per_block_qval"):
        assert callable(getattr(qtypes, n)), n
    assert callable(_fused_llm_infer.fc_plain) and callable(nn.fc_plain) and callable(llm_common.fc_plain)
    for n in ("BlockedLinear", "FixLinear"):
        assert hasattr(llm_common, n)
    for n in ("TppLinear", "BlockedWeight", "FixLinear", "OptimizeForLinear"):
        assert hasattr(nn, n)
    for n in ("BlockingManager", "BlockedParameter", "BlockedModule"):
        assert hasattr(blocked_layout, n)
    assert tpx.get_vnni_blocking(torch.bfloat16) == 2 and tpx.get_vnni_blocking(torch.float32) == 1
    for op in ("fc_plain", "fc_add", "fc_silu", "fc_mul", "qkv_gemm", "swiglu_mlp"):
        assert hasattr(torch.ops.tpp_llm, op)


def test_blocking_manager_matches_index_formula():
    from tpp_pytorch_extension.utils.blocked_layout import BlockingManager
    from tpp_pytorch_extension.nn import BlockedWeight
    N, K = 48, 128
    W = torch.arange(N * K, dtype=torch.float32).view(N, K)
    bm = BlockingManager(W.shape, blocking_factors=[16, [32, 2]], permute=[0, 2, 3, 1, 4])
    Wb = bm.block(W)
    assert list(Wb.shape) == [3, 2, 32, 16, 2] == bm.blocked_shape
    for (n1, c1, c2, k2, c3) in [(0, 0, 0, 0, 0), (2, 1, 31, 15, 1), (1, 0, 7, 3, 1)]:
        assert Wb[n1, c1, c2, k2, c3] == W[n1 * 16 + k2, c1 * 64 + c2 * 2 + c3]
    assert torch.equal(bm.unblock(Wb), W)
    assert torch.equal(BlockedWeight(W, 16, 64, torch.bfloat16), Wb.to(torch.bfloat16))
    assert torch.equal(BlockedWeight(W, 16, 64, torch.float32), W.view(3, 16, 2, 64).permute(0, 2, 3, 1))
    with pytest.raises(AssertionError):
        BlockingManager((50, 128), blocking_factors=[16, 64], permute=[0, 2, 3, 1])


def test_blocked_module_state_dict_round_trip():
    """BlockedModule saves BlockedParameters in the plain layout and re-blocks
    them on load (reference: blocked_layout.py:309-364)."""
    from tpp_pytorch_extension.utils.blocked_layout import BlockedModule, BlockedParameter

    class Mod(BlockedModule):
        def __init__(self):
            super().__init__()
            self.w = BlockedParameter(torch.arange(64 * 128, dtype=torch.float32).view(64, 128))
            self.w.set_blocking_param(([16, 64], [0, 2, 3, 1]))

    m = Mod()
    plain = m.w.data.clone()
    m.w.block()
    assert list(m.w.shape) == [4, 2, 64, 16] and m.w.is_blocked()
    sd = m.state_dict()
    assert list(sd["w"].shape) == [64, 128] and torch.equal(sd["w"], plain)
    assert m.w.is_blocked()
    m2 = Mod()
    m2.w.block()
    m2.load_state_dict({"w": plain * 2})
    assert m2.w.is_blocked() and list(m2.w.shape) == [4, 2, 64, 16]
    m2.w.unblock()
    assert torch.equal(m2.w.data, plain * 2)


def test_fix_linear_unquantized_keeps_blocked_weight():
    from tpp_pytorch_extension.llm.llm_common import FixLinear, BlockedLinear
    torch.manual_seed(1)
    lin = torch.nn.Linear(128, 64, bias=True)
    W = lin.weight.data.clone()
    FixLinear(lin, 16, 64, torch.float32)
    assert isinstance(lin, BlockedLinear) and list(lin.weight.shape) == [4, 2, 64, 16]
    assert torch.equal(lin.weight.data, W.view(4, 16, 2, 64).permute(0, 2, 3, 1))
    with pytest.raises(ValueError):
        FixLinear(torch.nn.Linear(64, 64), 16, 64, torch.bfloat16, weight_dtype="nf4")


def test_fix_vnni_and_block_size_rule():
    from tpp_pytorch_extension import _ops
    t = torch.arange(2 * 2 * 8 * 4 * 4, dtype=torch.float32).view(2, 2, 8, 4, 4).to(torch.bfloat16)
    v2 = _ops.fix_vnni(t)
    assert list(v2.shape) == [2, 2, 16, 4, 2]
    assert v2[1, 0, 5, 2, 1] == t[1, 0, 2, 2, 3]  # c2'=5 -> c2=2, half 1 -> c3 = 2 + 1
    assert _ops.qint8_block_size_for(4096) == 256 and _ops.qint8_block_size_for(11008) == 256
    assert _ops.qint8_block_size_for(192) == 64 and _ops.qint8_block_size_for(384) == 128


def test_a_quantized_tensor_finds_its_layout_when_asked(monkeypatch):
    """Making a quantized tensor (loading a model, quantizing activations) does not ask for its weight layout, a microsecond of
    a short call; the first question does, the later ones are answered from it."""
    from tpp_pytorch_extension import _qtensor as Q

    asked, find = [], Q.QTensor._find_layout
    monkeypatch.setattr(Q.QTensor, "_find_layout", lambda self: asked.append(1) or find(self))
    w = Q.QTensor(torch.zeros(4, 2, 32, 32, 2, dtype=torch.uint8), torch.zeros(1), (4, 2, 32, 32, 2), torch.quint4x2, Q.QSCHEME_MXFP, 32, 2, True, 2)
    x = Q.QTensor(torch.zeros(3, 256, dtype=torch.int8), torch.zeros(3, 1), (3, 256), torch.qint8, Q.QSCHEME_AFFINE, 256, 1, False, 1)
    assert not asked
    for _ in range(3):
        assert w.weight_layout() == ("mxfp4", 128, 128) and x.weight_layout() == (None, 0, 0)
    assert len(asked) == 2


def test_launch_plans_of_the_baseline_shapes():
    """Host-side planning (no GPU work): which kernel and grid the library would launch for the BASELINE shapes --
    decode GEMMs fill one round of 256 workgroups, the prefill GEMMs get the workgroup tile whose rounds are full, the
    q/k/v GEMM the half-size workgroups that shorten its last round."""
    import ctypes
    from tpp_pytorch_extension import _lib
    L = _lib.lib()
    buf = ctypes.create_string_buffer(4096)

    def plan(fn, *args):
        _lib.check(fn(*args, buf, len(buf)))
        return buf.value.decode().strip().splitlines()

    ws = 1 << 25
    # config 2: QINT8 MLP linears
    assert "skinny_qint8_fq_kernel<3," in plan(L.tppx_plan_linear_qint8, 1, 11008, 4096, 256, 1, 0, ws)[0]
    lines = plan(L.tppx_plan_linear_qint8, 64, 4096, 11008, 256, 1, 0, ws)
    assert len(lines) == 2 and "quant_act_int8_rows_kernel" in lines[0]
    # four channel tiles x four K parts per workgroup, K in four slices across workgroups (64 groups x 4)
    assert "skinny_qint8_nk_kernel<4, 4, 4, 3, 1, 8> grid=256x1x1 block=1024" in lines[1], lines
    lines = plan(L.tppx_plan_linear_qint8, 32, 4096, 11008, 256, 1, 0, ws)
    assert "skinny_qint8_nk_kernel<2, 4, 4, 3, 1, 8> grid=256x1x1" in lines[1], lines
    lines = plan(L.tppx_plan_linear_qint8, 64, 4096, 11008, 256, 1, 0, 0)  # no workspace: no K split
    assert "skinny_qint8_kernel<4, 1, 4, 8, 8, true> grid=256x1x1" in lines[1], lines
    assert len(plan(L.tppx_plan_linear_qint8, 64, 4096, 11008, 256, 0, 0, ws)) == 1             # pre-quantized input
    # config 3 / 5: MXFP4 decode
    assert "skinny_mxfp4_x4_kernel<1, 4, false> grid=256x1x1" in plan(L.tppx_plan_linear_mxfp4, 1, 4096, 11008, 0, ws)[0]
    assert "skinny_mxfp4_xl_kernel<4, 2, false, 0, 8> grid=64x1x4" in plan(L.tppx_plan_linear_mxfp4, 16, 4096, 11008, 0, ws)[0]
    assert "skinny_mxfp4_mg_kernel<1, 1, false> grid=256x1x1 block=1024" in plan(L.tppx_plan_linear_mxfp4, 16, 4096, 11008, 0, 0)[0]  # no workspace
    assert "skinny_mxfp4_xl_kernel<1, 2, false, 0, 8> grid=256x1x1" in plan(L.tppx_plan_linear_mxfp4, 16, 4096, 4096, 0, ws)[0]
    gate_up = (ctypes.c_int64 * 2)(11008, 11008)
    assert "skinny_mxfp4_xl_kernel<3, 2, true, 0, 2> grid=230x1x1" in plan(L.tppx_plan_multi_linear_mxfp4, gate_up, 2, 1, 4096, 1, 0, ws)[0]
    assert "skinny_mxfp4_mg_kernel<4, 3, true> grid=230x1x1 block=512" in plan(L.tppx_plan_multi_linear_mxfp4, gate_up, 2, 64, 4096, 1, 0, ws)[0]
    # config 4: prefill at 2048 rows
    assert "big_mxfp4_kernel<8, false, 1, 8> grid=256x1x1 block=512" in plan(L.tppx_plan_linear_mxfp4, 2048, 8192, 8192, 0, 0)[0]
    assert "big_mxfp4_kernel<8, false, 1, 8> grid=256x1x1" in plan(L.tppx_plan_linear_mxfp4, 2048, 8192, 28672, 0, 0)[0]
    qkv = (ctypes.c_int64 * 3)(8192, 1024, 1024)
    assert "big_mxfp4_kernel<8, false, 1, 4> grid=640x1x1 block=256" in plan(L.tppx_plan_multi_linear_mxfp4, qkv, 3, 2048, 8192, 0, 0, 0)[0]
    pair = (ctypes.c_int64 * 2)(28672, 28672)
    lines = plan(L.tppx_plan_multi_linear_mxfp4, pair, 2, 2048, 8192, 1, 0, 0)
    assert len(lines) == 1 and "big_mxfp4_kernel<8, true, 1, 8> grid=1792x1x1" in lines[0]       # silu*mul in the epilogue
    lines = plan(L.tppx_plan_multi_linear_mxfp4, pair, 2, 2048, 8192, 1, _lib.FLAG_ACT_FP8, 1 << 28)
    assert any("big_fp8_kernel<8, true> grid=1792x1x1" in l for l in lines), lines
    # prompts of a few hundred tokens: the wave tile whose workgroups fill one round of the CUs best
    assert "wide_kernel<4, 2, 4, false, false, false> grid=256x1x1 block=256" in plan(L.tppx_plan_linear_mxfp4, 512, 4096, 4096,
                                                                                      _lib.FLAG_FORCE_TILED, 0)[0]
    assert "wide_kernel<4, 2, 4, false, false, false>" in plan(L.tppx_plan_linear_mxfp4, 512, 4096, 4096, 0, 0)[0]   # and it is the choice
    assert "wide_kernel<4, 3, 8, false, false, false> grid=232x1x1 block=512" in plan(L.tppx_plan_linear_mxfp4, 512, 11008, 4096,
                                                                                      _lib.FLAG_FORCE_TILED, 0)[0]
    assert "wide_kernel<6, 3, 8, false, false, false> grid=242x1x1 block=512" in plan(L.tppx_plan_linear_mxfp4, 2048, 4096, 4096,
                                                                                      _lib.FLAG_FORCE_TILED, 0)[0]
    pair7 = (ctypes.c_int64 * 2)(11008, 11008)
    assert "wide_kernel<4, 3, 8, true, false, false> grid=232x1x1 block=512" in plan(L.tppx_plan_multi_linear_mxfp4, pair7, 2, 256, 4096, 1,
                                                                                     _lib.FLAG_FORCE_TILED, 0)[0]
    pair2 = (ctypes.c_int64 * 2)(2048, 2048)
    assert "wide_kernel<6, 3, 8, true, false, false> grid=242x1x1 block=512" in plan(L.tppx_plan_multi_linear_mxfp4, pair2, 2, 2048, 4096, 1,
                                                                                     _lib.FLAG_FORCE_TILED, 0)[0]
    assert "big_qint8_narrow_kernel grid=256x1x1 block=256" in plan(L.tppx_plan_linear_qint8, 512, 4096, 4096, 256, 1,
                                                                     _lib.FLAG_FORCE_TILED, 1 << 25)[-1]     # 22 us (128 of 64 x 256: 30)
    assert "big_qint8_kernel grid=172x1x1 block=512" in plan(L.tppx_plan_linear_qint8, 512, 11008, 4096, 256, 1,
                                                              _lib.FLAG_FORCE_TILED, 1 << 25)[-1]
    pair1 = (ctypes.c_int64 * 2)(4096, 4096)
    assert "wide_kernel<4, 2, 4, true, false, false> grid=256x1x1 block=256" in plan(L.tppx_plan_multi_linear_mxfp4, pair1, 2, 256, 4096, 1,
                                                                                     _lib.FLAG_FORCE_TILED, 0)[0]
    assert "wide_kernel<6, 2, 8, false, false, false> grid=473x1x1 block=512" in plan(L.tppx_plan_linear_mxfp4, 1024, 11008, 4096,
                                                                                      _lib.FLAG_FORCE_TILED, 0)[0]
    for M, other in ((511, 512), (1000, 1024)):  # whole 128-row blocks make no difference
        assert plan(L.tppx_plan_linear_mxfp4, M, 11008, 4096, 0, 0) == plan(L.tppx_plan_linear_mxfp4, other, 11008, 4096, 0, 0)
    # from 65 rows on the small wave tiles take what the planner hands to a tiled kernel
    assert "wide_kernel<2, 1, 8, false, false, false> grid=160x1x1 block=512" in plan(L.tppx_plan_linear_mxfp4, 160, 4096, 4096, 0, 0)[0]
    assert "wide_kernel<2, 1, 8, false, false, false> grid=128x1x1" in plan(L.tppx_plan_linear_mxfp4, 128, 4096, 4096, 0, ws)[0]  # 12 us (rows 17.9)
    assert "big_qint8_small_kernel grid=129x1x1 block=512" in plan(L.tppx_plan_linear_qint8, 160, 11008, 4096, 256, 1, 0, ws)[-1]
    assert "wide_kernel<2, 1, 8, false, false, false>" in plan(L.tppx_plan_linear_mxfp4, 100, 4096, 4096, _lib.FLAG_FORCE_TILED, 0)[0]


def test_launch_plans_of_per_output_channel_qint8():
    """QINT8 with one scale block = all of K (and other multiples of 256): up to 16 rows the quantisation stays inside
    the GEMM launch (maxima exchanged between the waves), above that the big-block quantizer runs in front; all 8 or
    16 waves of a workgroup get a share of K (the grid and block are those of the 256-wide default)."""
    import ctypes
    from tpp_pytorch_extension import _lib
    L = _lib.lib()
    buf = ctypes.create_string_buffer(4096)

    def plan(*args):
        _lib.check(L.tppx_plan_linear_qint8(*args, buf, len(buf)))
        return buf.value.decode().strip().splitlines()

    ws = 1 << 25
    for M in (1, 8):
        one = plan(M, 11008, 4096, 4096, 1, 0, ws)
        assert len(one) == 1 and "skinny_qint8_fq_kernel<3, 4, 16, 16, 4, true, 8> grid=230x1x1 block=1024" in one[0], one
        one = plan(M, 4096, 11008, 11008, 1, 0, ws)
        assert len(one) == 1 and "skinny_qint8_fq_kernel<1, 4, 16, 16, 6, true, 8> grid=256x1x1 block=1024" in one[0], one
    two = plan(64, 11008, 4096, 4096, 1, 0, ws)
    assert len(two) == 2 and "quant_act_int8_bigblk_kernel grid=64x1x1 block=256" in two[0], two
    assert "skinny_qint8_kernel<4, 3, 2, 8, 8, true> grid=230x1x1 block=512" in two[1], two
    two = plan(64, 4096, 11008, 11008, 1, 0, ws)
    assert "quant_act_int8_bigblk_kernel grid=64x1x1 block=704" in two[0] and "skinny_qint8_nk_kernel<4," in two[1], two
    # a block that is not a whole number of 256-wide runs is dealt tile by tile: still one GEMM launch, quantizer in front
    odd = plan(5, 512, 1280, 320, 1, 0, ws)
    assert len(odd) == 2 and "quant_act_int8_kernel" in odd[0] and "skinny_qint8_kernel<1, 1, 4, 16, 4, true>" in odd[1], odd


def test_kernel_family_of_short_prompts():
    """65 and more rows on the family and tile that measured fastest, where one figure per block row was far off: the
    decode kernels where the block rows share rounds (few channels), tiles where they do not (many), and the small
    tiles' extra cost where an odd number of row blocks leaves no rectangles for the XCDs."""
    import ctypes
    from tpp_pytorch_extension import _lib
    L = _lib.lib()
    buf = ctypes.create_string_buffer(4096)

    def one(M, N, K):
        _lib.check(L.tppx_plan_linear_mxfp4(M, N, K, 0, 1 << 25, buf, len(buf)))
        return buf.value.decode()

    def pair(M, N, K):
        _lib.check(L.tppx_plan_multi_linear_mxfp4((ctypes.c_int64 * 2)(N, N), 2, M, K, 1, 0, 1 << 25, buf, len(buf)))
        return buf.value.decode()

    for M in (65, 128):
        assert "skinny_mxfp4" in pair(M, 1024, 4096) and "skinny_mxfp4" in pair(M, 1536, 18944), M  # 11 us (tiles 22), 38 (79)
        assert "wide_kernel" in one(M, 28672, 2560) and "wide_kernel" in one(M, 18944, 1024), M     # (rows 52 us, 26)
        assert "wide_kernel" in pair(M, 11008, 4096), M                                            # (rows 42 us)
    assert "skinny_mxfp4" in pair(160, 1024, 8192)                                                  # 19 us (tiles 38)
    assert "wide_kernel" in one(192, 14336, 5120)                                                   # (rows 65 us)
    assert "<5, 2, 8," in one(1800, 2560, 11008) and "<5, 2, 4," in one(1500, 1536, 18944)
    assert "<8, true, 1, 8>" in pair(2048, 28672, 8192)                                             # 1254 us (128 x 256: 1283)

    def qkv(M, N, K):
        _lib.check(L.tppx_plan_multi_linear_mxfp4((ctypes.c_int64 * 3)(N, N, N), 3, M, K, 0, 0, 1 << 25, buf, len(buf)))
        return buf.value.decode()

    for M in (96, 127, 128, 129):  # nothing changes at whole block rows of 64
        assert "wide_kernel" in qkv(M, 4096, 4096), M                                               # 17 us (rows 35)
        assert "wide_kernel" in one(M, 12288, 4096) and "wide_kernel" in one(M, 11008, 4096), M     # 17 us (26)
        assert "skinny_mxfp4" in one(M, 1024, 4096), M                                              # 8 us (tiles 16)

    # long prompts: not the small wave tiles, whose workgroups drift apart in K where the XCDs get whole columns
    for shape in ((2048, 9088, 8704), (1744, 6528, 10496), (1421, 4096, 11008), (1421, 4096, 4096), (2048, 4800, 4096)):
        assert not any(small in one(*shape) for small in ("<2, 1, 8,", "<3, 2, 4,", "<4, 2, 4,")), shape
    assert "<3, 2, 4," not in qkv(2048, 1856, 13312) and "<4, 2, 4," not in pair(2048, 2880, 7168)

    def per_weight(M, N, K, weight_bytes):
        return not L.tppx_group_is_one_launch((ctypes.c_int64 * 2)(N, N), 2, M, K, weight_bytes)

    # QINT8 pairs: one launch from 65 rows on, 18 us (per weight 24), 20 (26), 13 (21), 62 (96 on rows, 123 on tiles), 9 (17)
    for M, N, K in ((200, 1024, 3584), (256, 1024, 4096), (212, 1024, 2304), (128, 2432, 16128), (65, 1024, 1024)):
        assert not per_weight(M, N, K, 1), (M, N, K)
    assert per_weight(64, 1024, 4096, 1)
    assert per_weight(160, 1024, 5120, 2) and not per_weight(160, 4096, 5120, 2)  # 25 us (one launch 29)

    def qint8(M, N, K):
        _lib.check(L.tppx_plan_linear_qint8(M, N, K, 256, 1, 0, 1 << 25, buf, len(buf)))
        return buf.value.decode().strip().splitlines()[-1]

    # single QINT8 weights that come from memory: the decode kernels where they are few, also for short K
    assert "skinny_qint8" in qint8(192, 1408, 8448) and "skinny_qint8" in qint8(251, 1152, 11776)    # 28 us (35), 39 (47)
    assert "skinny_qint8" in qint8(128, 2368, 12032) and "skinny_qint8" in qint8(96, 1024, 1024)      # 41 us (48), 8.1 (8.8)
    assert "big_qint8" in qint8(300, 1024, 1024) and "big_qint8" in qint8(128, 11008, 4096)

    def bf16_tiles(M, N, K):
        return L.tppx_group_is_one_launch((ctypes.c_int64 * 1)(N), 1, M, K, 2)

    # single bf16 weights that come from memory: the decode kernels where they are few and K is long
    assert not bf16_tiles(82, 2304, 10496) and not bf16_tiles(128, 2432, 11776) and not bf16_tiles(100, 3584, 18944)  # 39 us (55), 54 (70), 85 (106)
    assert not bf16_tiles(160, 1536, 18944) and not bf16_tiles(105, 2304, 5376)                      # 70 us (91), 24 (32)
    assert bf16_tiles(128, 11008, 4096) and bf16_tiles(300, 4096, 4096) and bf16_tiles(1000, 1024, 4096)


def test_group_is_one_launch():
    """Which groups run as one launch, by sizes alone: rows, blocks of whole tiles, operands below 4 GiB."""
    import ctypes
    from tpp_pytorch_extension import _lib
    L = _lib.lib()

    def one(Ns, M, K, weight_bytes):
        return L.tppx_group_is_one_launch((ctypes.c_int64 * len(Ns))(*Ns), len(Ns), M, K, weight_bytes)

    for bytes_per in (1, 2):
        assert one([11008] * 2, 333, 4096, bytes_per) == 1 and one([11008] * 2, 2048, 4096, bytes_per) == 1
        assert one([11008] * 2, 64, 4096, bytes_per) == bytes_per - 1  # the decode kernels' rows: bf16 weights in one launch
        assert one([11000] * 2, 333, 4096, bytes_per) == 0  # no whole tiles
        assert one([11008] * 2, 0, 4096, bytes_per) == 0 and one([], 333, 4096, bytes_per) == 0
        assert one([1 << 20] * 2, 333, 4096 // bytes_per, bytes_per) == 0  # weights of 4 GiB
    assert one([5120] * 2, 64, 2048, 1) == 0 and one([5120] * 2, 66, 2048, 1) == 1  # per weight, then one launch (14 us, per weight 26)
    assert one([11008] * 2, 333, 4096, 3) == 0
    assert one([4096, 1024, 1024], 2048, 4096, 2) == 1 and one([4096, 1024, 1024], 2048, 4096, 1) == 0  # bf16 only
    for M in (1, 17, 64):
        assert one([4096, 1024, 1024], M, 4096, 2) == 1 and one([1 << 20] * 2, M, 2048, 2) == 1  # (weights of 4 GiB too)
        assert one([4096, 1024], M, 4032, 2) == 0  # K in no whole tiles


def test_prompt_plans_by_tile_and_grid(monkeypatch):
    """What the tests above leave open of MXFP4 prompts: the family of few channels at a long K, which of the small wave tiles,
    whole K where slices measured slower or as fast, and the launches of a forced number of slices."""
    import ctypes
    from tpp_pytorch_extension import _lib
    L = _lib.lib()
    buf = ctypes.create_string_buffer(4096)

    def one(M, N, K):
        _lib.check(L.tppx_plan_linear_mxfp4(M, N, K, 0, 1 << 25, buf, len(buf)))
        return buf.value.decode()

    def group(M, ns, K, dual):
        _lib.check(L.tppx_plan_multi_linear_mxfp4((ctypes.c_int64 * len(ns))(*ns), len(ns), M, K, dual, 0, 1 << 25, buf, len(buf)))
        return buf.value.decode()

    assert "skinny_mxfp4" in one(160, 1024, 18944) and "skinny_mxfp4" in one(256, 1024, 18944)      # 38 us, 33
    assert "wide_kernel<2, 1, 8, true, false, false>" in group(256, (1024, 1024), 8192, 1)          # 21.3 us (rows 20.7: a near tie)
    # the wave tiles of up to 80 rows drift from 18 row blocks on, in more than a round of workgroups and without rectangles
    small = ("<2, 1, 8,", "<3, 2, 4,", "<4, 2, 4,", "<5, 2, 4,")
    assert "<6, 3, 8," in one(1978, 3136, 10240)                                                    # 111 us (80 x 128: 127)
    for plan in (group(2048, (1856,) * 3, 13312, 0), group(2048, (2880,) * 2, 7168, 1),             # 226 us, 131
                 one(1740, 4160, 9216), one(1990, 3136, 12288), one(1850, 2112, 6400)):
        assert not any(t in plan for t in small), plan
    # a short K in more than a round: two workgroups to a CU (286 us on 256 x 256, 246; 92, 75; 111, 99)
    for plan in (group(3309, (31616,) * 2, 512, 1), group(1981, (20544,) * 2, 256, 1), group(6543, (5280,) * 3, 384, 0)):
        assert "big_mxfp4_kernel<8, " in plan and ", 1, 4>" in plan, plan
    for M, N, K in ((300, 4096, 11008), (381, 2112, 4608), (65, 8512, 6400)):  # 44.7 us (in slices 43.7), 16.7 (19.6), 26.8 (28.7)
        assert "wide_sum_kernel" not in one(M, N, K), (M, N, K)
    try:
        monkeypatch.setenv("TPPX_TILED_MIN_M", "0")
        for S, M, N, K in ((2, 65, 160, 1152), (3, 200, 288, 1792), (4, 129, 2080, 2048), (6, 100, 32, 3072), (6, 333, 416, 4224)):
            monkeypatch.setenv("TPPX_TILED_SPLIT", str(S))
            L.tppx_reload_env()
            mt, nt, w = (3, 2, 4) if N * M > 100000 else (2, 1, 8)  # (row tiles and channel tiles of a wave, waves)
            wgs = -(-M // (mt * 16)) * -(-N // (nt * w * 16))
            gemm, add = one(M, N, K).splitlines()
            assert f"wide_kernel<{mt}, {nt}, {w}, false, false, true> grid={wgs}x{S}x1 block={w * 64}" in gemm
            assert f"wide_sum_kernel<{mt}, {nt}, {w}, {S}> grid={wgs * w}x1x1" in add
    finally:
        monkeypatch.undo()
        L.tppx_reload_env()


def test_mxfp4_prompts_of_few_channels_run_a_long_k_in_slices():
    """Fewer than 2048 channels: in slices where the decode kernels end and a few dozen workgroups would walk a long K, whole for
    many row blocks, up to K = 4096 and, on the decode kernels, for few rows."""
    from tpp_pytorch_extension import _lib
    L = _lib.lib()
    buf = ctypes.create_string_buffer(4096)

    def plan(m, n, k):
        _lib.check(L.tppx_plan_linear_mxfp4(m, n, k, 0, 32 << 20, buf, len(buf)))
        return buf.value.decode()

    for shape in ((320, 1024, 18176), (677, 512, 12288), (257, 1920, 8192), (512, 768, 18176), (400, 1344, 12288), (320, 1024, 8192),
                  (3421, 64, 12288)):
        assert "wide_sum_kernel" in plan(*shape), shape  # whole 40.1 us, 24.6, 18.1, 35.0, 24.8, 17.6; in slices 22.5, 17.8, 17.5, 21.9, 22.5, 14.9 (64 x 12288 24.4, 19.3)
    for shape in ((1400, 768, 12288), (1400, 512, 8192), (677, 512, 4096), (1024, 1408, 9216)):
        assert "wide_kernel" in plan(*shape) and "wide_sum_kernel" not in plan(*shape), shape
    assert "skinny_mxfp4" in plan(256, 1024, 18944) and "skinny_mxfp4" in plan(200, 512, 8192)


def test_bf16_prompts_near_the_line_between_the_kernels_run_on_tiles():
    """Launches whose two estimates nearly meet go to the tiles: what decides between two tiles is not weighed against the decode
    kernels."""
    from tpp_pytorch_extension import _lib
    L = _lib.lib()
    for Ns, M, K in (((1120, 1120), 156, 3584), ((192, 192), 541, 2816), ((1184,), 220, 512)):  # 20.3 us (rows 24.0), 14.0 (16.7), 6.1 (7.6)
        assert L.tppx_group_is_one_launch((ctypes.c_int64 * len(Ns))(*Ns), len(Ns), M, K, 2), (Ns, M, K)


def test_environment_switches_are_read_once(monkeypatch):
    """The library keeps a TPPX_* switch after its first read (no getenv per launch, and a captured graph's kernel
    choice cannot drift); tppx_reload_env() makes it read again."""
    import ctypes
    from tpp_pytorch_extension import _lib
    L = _lib.lib()
    buf = ctypes.create_string_buffer(4096)

    def plan():
        _lib.check(L.tppx_plan_linear_qint8(1, 4096, 4096, 256, 1, 0, 0, buf, len(buf)))
        return buf.value.decode()

    L.tppx_reload_env()
    assert "skinny_qint8_fq_kernel" in plan()
    os.environ["TPPX_SKINNY_FUSEDQ"] = "0"
    try:
        assert "skinny_qint8_fq_kernel" in plan(), "the switch was read again without a reload"
        L.tppx_reload_env()
        assert "skinny_qint8_fq_kernel" not in plan() and "quant_act_int8" in plan()
    finally:
        del os.environ["TPPX_SKINNY_FUSEDQ"]
        L.tppx_reload_env()
    assert "skinny_qint8_fq_kernel" in plan()


def test_kernels_of_few_rows_and_uneven_wave_slices():
    """K between 2048 and 4096 whose tiles do not divide by the sixteen waves: the LDS-staged kernel for up to 4 rows, the
    tile-by-tile one for more; single, grouped and as the pair."""
    import ctypes
    from tpp_pytorch_extension import _lib
    L = _lib.lib()
    buf = ctypes.create_string_buffer(4096)
    for M, N, K in ((1, 96, 2176), (4, 4128, 2560), (3, 8224, 3584), (2, 12320, 3968), (4, 32, 3584), (5, 96, 3584), (16, 4128, 2560)):
        name = "skinny_mxfp4_xl_kernel<" if M <= 4 else "skinny_mxfp4_mg_kernel<"
        plans = [(L.tppx_plan_linear_mxfp4, (M, N, K, 0, 1 << 25))]
        for ns, dual in (((N, 32, N), 0), ((N, N), 1)):
            plans.append((L.tppx_plan_multi_linear_mxfp4, ((ctypes.c_int64 * len(ns))(*ns), len(ns), M, K, dual, 0, 1 << 25)))
        for fn, args in plans:
            _lib.check(fn(*args, buf, len(buf)))
            assert name in buf.value.decode(), (M, N, K, buf.value)


def test_forced_prompt_tiles(monkeypatch):
    """TPPX_TILED_BIG_TILE by number, with the workgroups that the tile makes of the launch: 1 .. 4 and, from 7 on, the wave tiles
    of MXFP4 weights, whole and, on the three that have them, with K in slices; what is not built is left to the estimates."""
    import ctypes
    from tpp_pytorch_extension import _lib
    L = _lib.lib()
    buf = ctypes.create_string_buffer(4096)
    M, N, K = 300, 4512, 4096

    def plan(tile, split=0):
        monkeypatch.setenv("TPPX_TILED_MIN_M", "0")
        monkeypatch.setenv("TPPX_TILED_BIG_TILE", str(tile))
        monkeypatch.setenv("TPPX_TILED_SPLIT", str(split))
        L.tppx_reload_env()
        _lib.check(L.tppx_plan_linear_mxfp4(M, N, K, 0, 1 << 25, buf, len(buf)))
        return buf.value.decode()

    def grid(rows, cols, slices=1):
        return f"grid={(M + rows - 1) // rows * ((N + cols - 1) // cols)}x{slices}x1"

    try:
        for tile, name, rows, cols in ((1, "big_mxfp4_kernel<8, false, 2, 4>", 256, 256), (2, "big_mxfp4_kernel<8, false, 1, 4>", 128, 256),
                                       (3, "big_mxfp4_kernel<8, false, 1, 8>", 128, 512), (4, "wide_kernel<4, 2, 4, false, false, false>", 64, 128)):
            assert f"{name} {grid(rows, cols)}" in plan(tile), tile
        forms = ((2, 1, 8), (3, 2, 4), (4, 2, 4), (5, 2, 4), None, (4, 3, 4), (5, 3, 4), (5, 2, 8), (6, 2, 8), (4, 3, 8), (6, 3, 8))
        free = plan(0)
        for tile, form in enumerate(forms, 7):
            if form is None:
                assert plan(tile) == free
                continue
            mt, nt, w = form
            assert f"wide_kernel<{mt}, {nt}, {w}, false, false, false> {grid(mt * 16, nt * w * 16)} block={w * 64}" in plan(tile), tile
        assert plan(5) == free and plan(6) == free and plan(18) == free
        for tile, (mt, nt, w) in ((4, (4, 2, 4)), (7, (2, 1, 8)), (8, (3, 2, 4)), (9, (4, 2, 4))):
            for S in (2, 3, 4, 6):
                lines = plan(tile, S).splitlines()
                rows, cols = mt * 16, nt * w * 16
                fits = (M + rows - 1) // rows * ((N + cols - 1) // cols) * S * rows * cols * 4 <= 1 << 25
                assert f"wide_kernel<{mt}, {nt}, {w}, false, false, {'true' if fits else 'false'}> {grid(rows, cols, S if fits else 1)}" in lines[0]
                assert len(lines) == 1 + fits and (not fits or f"wide_sum_kernel<{mt}, {nt}, {w}, {S}>" in lines[1])
        assert len(plan(10, 4).splitlines()) == 1  # 80 x 128: K whole
    finally:
        monkeypatch.undo()
        L.tppx_reload_env()


def test_cache_lengths_after_graph_replayed_steps():
    """Steps replayed from a graph move the device counter themselves; the host bookkeeping that follows them must
    move every layer's length, so that get_seq_length(layer) and a later update() on any layer see the new keys."""
    from tpp_pytorch_extension.llm.fused_llama_infer import TppCache
    cache = TppCache(64)
    kv = torch.zeros((1, 2, 5, 8), dtype=torch.bfloat16)
    for i in range(3):
        cache.fill_(i, kv, kv)
    cache._advance_host(4)  # what greedy_decode / time_decode_steps do per replay
    assert [cache.get_seq_length(i) for i in range(3)] == [9, 9, 9]
    one = torch.ones((1, 2, 1, 8), dtype=torch.bfloat16)
    k, v = cache.update(one, one, 2)
    assert k.shape[2] == 10 and cache.get_seq_length(2) == 10 and cache.get_seq_length(1) == 9
    assert float(k[0, 0, 9, 0]) == 1.0 and float(k[0, 0, 8, 0]) == 0.0


def test_qwen2_front_end_surface():
    """The Qwen2 front-end mirrors the reference module's names (fused_qwen2_infer.py:45-238) and checks its
    parameter list without touching a GPU."""
    from tpp_pytorch_extension.llm import fused_qwen2_infer as Q
    from tpp_pytorch_extension.llm import fused_llama_infer as F
    from tpp_pytorch_extension._lib import TppxError
    for name in ("Qwen2DecoderLayer", "FixQwen2DecoderLayer", "OptimizeModelForQwen2", "Qwen2Model_forward", "TppCache"):
        assert hasattr(Q, name), name
    assert issubclass(Q.Qwen2DecoderLayer, F.LlamaDecoderLayer)
    with pytest.raises(TppxError):
        Q.Qwen2DecoderLayer([None] * 10, 0, 1e-6, 128, 64, 128)  # the Llama list: three biases short


def test_gptj_and_opt_front_end_surface():
    """The GPT-J and OPT front-ends mirror the reference modules' names (fused_gptj_infer.py:46-193,
    fused_opt_infer.py:45-203) and check their parameter lists without touching a GPU."""
    from tpp_pytorch_extension.llm import fused_gptj_infer as G
    from tpp_pytorch_extension.llm import fused_opt_infer as P
    from tpp_pytorch_extension._lib import TppxError
    for name in ("GPTJBlock", "FixGPTJBlock", "OptimizeModelForGPTJ", "GPTJModel_forward", "create_sinusoidal_positions"):
        assert hasattr(G, name), name
    for name in ("OPTDecoderLayer", "FixOPTDecoderLayer", "OptimizeModelForOPT", "OPTDecoder_forward"):
        assert hasattr(P, name), name
    with pytest.raises(TppxError):
        G.GPTJBlock([None] * 10, 0, 1e-5, 256, 2048, 64)
    with pytest.raises(TppxError):
        P.OPTDecoderLayer([None] * 11, 0, 1e-5, 1e-5, 64, True)
    t = G.create_sinusoidal_positions(8, 4)  # sin | cos of position * 10000^(-2i/dim)
    assert t.shape == (8, 4) and torch.allclose(t[0], torch.tensor([0.0, 0.0, 1.0, 1.0]))
    assert torch.allclose(t[3, :2], torch.sin(torch.tensor([3.0, 0.03]))) and torch.allclose(t[3, 2:], torch.cos(torch.tensor([3.0, 0.03])))


def test_common_module_helpers_one_process():
    """llm_common's process-group helpers in their one-process form, ShardLinear as pure slicing (the shards of all
    ranks tile the weight; a row-parallel split sums back to the whole linear), BlockedLayerNorm on the CPU."""
    import copy
    from tpp_pytorch_extension.llm import llm_common as C
    assert C.get_rank() == 0 and C.get_size() == 1
    C.set_pg()
    t = torch.arange(4.0)
    assert C.all_reduce(t) is t and C.shm_allreduce(t) is t
    torch.manual_seed(3)
    lin = torch.nn.Linear(96, 160)
    x = torch.randn(5, 96)
    full = lin(x)
    def shard(dim, r, size, bs):
        m = copy.deepcopy(lin)
        C.ShardLinear(m, dim, r, size, bs)  # in place, like the reference's
        return m

    cols = [shard(0, r, 3, 32) for r in range(3)]
    assert cols[0].split_sizes == [32, 64, 64] and [c.weight.shape[0] for c in cols] == [32, 64, 64]
    assert torch.equal(torch.cat([c.weight.data for c in cols]), lin.weight.data)
    assert torch.allclose(torch.cat([torch.nn.functional.linear(x, c.weight, c.bias) for c in cols], -1), full, atol=1e-6)
    rows = [shard(1, r, 3, 32) for r in range(3)]
    assert rows[0].split_sizes == [32, 32, 32]
    parts = [torch.nn.functional.linear(x[:, 32 * r:32 * r + 32], m.weight, m.bias) for r, m in enumerate(rows)]
    assert torch.allclose(sum(parts), full, atol=1e-5)  # the bias was divided by the number of ranks
    with pytest.raises(ValueError):
        shard(0, 0, 2, 64)  # 160 is not a multiple of 64
    ln = C.BlockedLayerNorm(64)
    y = ln(torch.randn(3, 64))
    assert torch.allclose(y.mean(-1), torch.zeros(3), atol=1e-5)
    assert C.compare(t, t.clone(), "same") is True and C.compare(t, t + 1, "shifted") is False


def test_cache_allocates_small_layers_together():
    """Layers of a small KV cache share one zeroed allocation (up to eight layers, keys and values), handed out as
    the layers ask for storage; a layer of another shape, or a cache whose layers are large, allocates on its own."""
    import torch
    from tpp_pytorch_extension.llm.fused_llama_infer import TppCache
    c = TppCache(48)
    got = [c._ensure(i, 2, 4, 16, "cpu") for i in range(10)]
    base = got[0][0].untyped_storage().data_ptr()
    assert all(k.untyped_storage().data_ptr() == base and v.untyped_storage().data_ptr() == base for k, v in got[:8])
    assert got[8][0].untyped_storage().data_ptr() != base           # ninth layer: the next group
    ptrs = {t.data_ptr() for kv in got for t in kv}
    assert len(ptrs) == 20                                          # no two layers share memory
    for k, v in got:
        assert k.shape == (2, 4, 48, 16) and k.is_contiguous() and v.is_contiguous()
        assert not k.any() and not v.any()
    assert c._ensure(3, 2, 4, 16, "cpu")[0].data_ptr() == got[3][0].data_ptr()   # a layer keeps its storage
    k, _ = c._ensure(10, 1, 4, 16, "cpu")                            # another shape: not the waiting storage
    assert k.shape == (1, 4, 48, 16) and not k.any()
    big = TppCache(48)
    big.SLAB_BYTES = 4 * 2 * 4 * 48 * 16                            # room for one layer only
    a, b = big._ensure(0, 2, 4, 16, "cpu"), big._ensure(1, 2, 4, 16, "cpu")
    assert a[0].untyped_storage().data_ptr() != b[0].untyped_storage().data_ptr() and not big._spare


def test_w4a8_prompts_take_the_prompt_kernel():
    """W4A8 calls from 64 rows on: row groups stream the 4-bit weights once per 64 rows, so they are for few rows only.
    Long prompts run on the prompt kernel whatever the weight (2048 rows of 28672 x 8192: 1250 us there, 2260 in row
    groups)."""
    from tpp_pytorch_extension import _ops

    shapes = [(28672, 8192), (8192, 28672), (22016, 8192), (8192, 8192), (11008, 4096), (4096, 11008), (4096, 4096), (3584, 18944)]
    for n, k in shapes:
        assert _ops._w4a8_row_groups(64, n, k), (n, k)
        for m in (1024, 1536, 2048, 4096, 16384):
            assert not _ops._w4a8_row_groups(m, n, k), (m, n, k)


def test_w4a8_calls_run_on_the_faster_kernel():
    """Calls where one of the two kernels was measured faster by 10 to 40 % (us in row groups, on the prompt kernel)."""
    from tpp_pytorch_extension import _ops

    for m, n, k in ((1957, 5056, 1280), (1398, 4416, 1024), (1555, 5056, 1280), (964, 8256, 1280), (512, 11008, 1024), (672, 8128, 1024)):
        assert not _ops._w4a8_row_groups(m, n, k), (m, n, k)  # 80 / 60, 42 / 34, 66 / 54, 69 / 57, 39 / 33, 39 / 33
    for m, n, k in ((400, 5120, 5120), (384, 7808, 10752), (323, 7360, 4096), (541, 5184, 9216), (1024, 2560, 10240), (600, 4864, 14336)):
        assert _ops._w4a8_row_groups(m, n, k), (m, n, k)      # 59 / 80, 133 / 186, 56 / 78, 117 / 153, 114 / 149, 180 / 233


def test_mxfp4_prompts_run_k_in_slices_where_that_pays():
    """Launch plans: K in slices where few workgroups have many steps; whole where the launch with whole K was measured
    faster, by 3 to 11 % (most of a round of workgroups, many row blocks) or as fast (4096 x 11008 at 333 rows)."""
    from tpp_pytorch_extension import _lib

    L = _lib.lib()

    def split(n, k, m):
        buf = ctypes.create_string_buffer(4096)
        _lib.check(L.tppx_plan_linear_mxfp4(m, n, k, 0, 32 << 20, buf, len(buf)))
        return "wide_sum_kernel" in buf.value.decode()

    for shape in ((4096, 11008, 100), (4096, 11008, 200), (2560, 10240, 200), (3584, 18944, 333)):
        assert split(*shape), shape
    for shape in ((1408, 9216, 1024), (1408, 11520, 970), (9024, 10496, 183), (4096, 11008, 400), (6400, 9984, 234), (2496, 13056, 725),
                  (1600, 9984, 847), (4096, 11008, 333), (4096, 16384, 420), (3584, 18944, 480)):
        assert not split(*shape), shape
