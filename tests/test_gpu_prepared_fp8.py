"""FP8 operands through arcq_prepare / arcq_linear_prepared / arcq_attention_quant_fp8_fwd (what a block with fp8_operands
runs): the bytes of the stand-alone FP8 kernels, at odd numbers of groups (padding), ragged blocks and the row counts that
choose between the product kernels."""
import ctypes

import pytest
import torch

from arcq_vit_amd import _lib, ops, synth
from test_gpu_prepared import _layer, _stream

pytestmark = pytest.mark.gpu


def _stage1(x, thr, cb, bits, w=None, mult=1.0):
    """arcq_act_quant_fp8_blocked: x8 in the block layout and, with weights, w8 [N, Kp]."""
    m, k = x.shape
    kp = ops.fp8_padded_k(k)
    x8 = torch.empty(m * kp, dtype=torch.uint8, device=x.device)
    n = w[0].shape[0] if w else 0
    w8 = torch.empty(max(n * kp, 1), dtype=torch.uint8, device=x.device)
    code = _lib.ARCQ_F16 if x.dtype == torch.float16 else _lib.ARCQ_F32
    ptrs = [t.data_ptr() for t in w] if w else [None] * 5
    _lib.check(_lib.load().arcq_act_quant_fp8_blocked(x.data_ptr(), code, thr.data_ptr(), cb.data_ptr(), x8.data_ptr(), m, k, bits, 1e-6,
                                                      *ptrs, w8.data_ptr() if w else None, n, mult, _stream()))
    return x8, w8


def _prepare(x, thr, cb, bits, w, mult, row_major):
    n, k = w[0].shape[0], w[2].shape[1] * 64
    kp = ops.fp8_padded_k(k)
    a = _lib.PrepareArgs()
    a.bits, a.fp8 = bits, 1
    a.x_dtype = _lib.ARCQ_F16 if x.dtype == torch.float16 else _lib.ARCQ_F32
    a.rows, a.K = x.shape
    x8 = torch.full((x.shape[0] * kp + 16,), 0x5a, dtype=torch.uint8, device=x.device)
    w8 = torch.full((n * kp + 16,), 0x5a, dtype=torch.uint8, device=x.device)
    a.x, a.thresholds, a.codebook, a.x_hat = x.data_ptr(), thr.data_ptr(), cb.data_ptr(), x8.data_ptr()
    j = a.weights[0]
    j.N, j.K, j.row_major, j.w_mult = n, k, int(row_major), mult
    j.packed, j.codebook, j.center, j.scale, j.code_sum, j.w_hat = [t.data_ptr() for t in w] + [w8.data_ptr()]
    _lib.check(_lib.load().arcq_prepare(ctypes.byref(a), _stream()))
    assert bool((x8[-16:] == 0x5a).all()) and bool((w8[-16:] == 0x5a).all())
    return x8[:-16], w8[:-16]


def _linear(x8, w8, bias, m, n, k, mult, row_major, gelu=False, residual=None, nq=None, bits=4, out=torch.float16):
    a = _lib.LinearPreparedArgs()
    y = torch.empty((m, n), dtype=out, device=x8.device) if nq is None else \
        torch.empty(m * ops.fp8_padded_k(n), dtype=torch.uint8, device=x8.device)
    a.y_dtype = _lib.ARCQ_F32 if out == torch.float32 else _lib.ARCQ_F16
    a.activation, a.w_row_major, a.fp8, a.w_mult = int(gelu), int(row_major), 1, mult
    a.M, a.N, a.K = m, n, k
    a.x_hat, a.w_hat, a.bias, a.y = x8.data_ptr(), w8.data_ptr(), bias.data_ptr(), y.data_ptr()
    if residual is not None:
        a.residual = residual.data_ptr()
    if nq is not None:
        a.next_thresholds, a.next_codebook, a.next_bits = nq[0].data_ptr(), nq[1].data_ptr(), bits
    _lib.check(_lib.load().arcq_linear_prepared(ctypes.byref(a), _stream()))
    return y


@pytest.mark.parametrize("m,k,bits,dtype", [(1, 64, 4, torch.float16), (31, 192, 3, torch.float16), (197, 384, 4, torch.float16),
                                            (591, 1024, 2, torch.float16), (33, 960, 4, torch.float32), (9000, 192, 4, torch.float16)])
def test_prepare_fp8(cuda, oracle, m, k, bits, dtype):
    cb, thr, w, _ = _layer(oracle, cuda, 96, k, bits, 5)
    x = synth.make_activation(m, k, 7).to(cuda, dtype)
    mult = ops.fp8_weight_multiplier(*w[1:])
    want_x, want_w = _stage1(x, thr, cb, bits, w, mult)
    kp = ops.fp8_padded_k(k)
    for row_major in (False, True):
        x8, w8 = _prepare(x, thr, cb, bits, w, mult, row_major)
        assert torch.equal(w8, want_w if row_major else want_w.reshape(3, 32, kp // 16, 16).permute(0, 2, 1, 3).reshape(-1))
        assert torch.equal(x8, want_x)


@pytest.mark.parametrize("m,n,k,bits", [(1, 32, 64, 4), (197, 1152, 384, 3), (100, 3072, 192, 4), (511, 192, 4096, 2), (512, 32, 64, 4),
                                        (591, 1024, 1024, 3), (1001, 2304, 768, 4), (1576, 4096, 1024, 4), (6304, 1184, 448, 2)])
def test_linear_prepared_fp8(cuda, oracle, m, n, k, bits):
    cb, thr, w, bias = _layer(oracle, cuda, n, k, bits, 11)
    x = synth.make_activation(m, k, 13).to(cuda, torch.float16)
    mult = ops.fp8_weight_multiplier(*w[1:])
    res = synth.make_activation(m, n, 17).to(cuda, torch.float16)
    plain = ops.linear_otf_fp8(x, thr, cb, *w, bias, bits, out_dtype=torch.float32)
    for row_major in (False, True):
        x8, w8 = _prepare(x, thr, cb, bits, w, mult, row_major)
        y32 = _linear(x8, w8, bias, m, n, k, mult, row_major, out=torch.float32)
        assert torch.equal(y32, plain)
        y = _linear(x8, w8, bias, m, n, k, mult, row_major)
        assert torch.equal(y, y32.half())
        assert torch.equal(_linear(x8, w8, bias, m, n, k, mult, row_major, gelu=True, residual=res), res + torch.nn.functional.gelu(y))
        if n % 64 == 0:
            for gelu in (False, True):
                want, _ = _stage1(torch.nn.functional.gelu(y) if gelu else y, thr, cb, bits)
                assert torch.equal(_linear(x8, w8, bias, m, n, k, mult, row_major, gelu=gelu, nq=(thr, cb), bits=bits), want), (row_major, gelu)


# (from the fourth: parts of a head with several query tiles, with odd and even numbers of heads; two tiles in a part and all waves
# quantizing from the seventh)
@pytest.mark.parametrize("b,n,h,bits", [(1, 197, 6, 4), (2, 33, 3, 2), (7, 101, 5, 3), (16, 197, 6, 4), (11, 197, 11, 3), (5, 129, 16, 2),
                                        (4, 256, 15, 4), (3, 225, 13, 3), (3, 225, 14, 4)])
def test_attention_quant_fp8(cuda, oracle, b, n, h, bits):
    cb, thr, _, _ = _layer(oracle, cuda, 32, 64, bits, 29)
    qkv = synth.make_activation(b * n, 3 * h * 64, 31).to(cuda, torch.float16).reshape(b, n, 3 * h * 64).contiguous()
    want, _ = _stage1(ops.attention_fwd(qkv, h).reshape(b * n, h * 64), thr, cb, bits)
    got = torch.empty_like(want)
    _lib.check(_lib.load().arcq_attention_quant_fp8_fwd(qkv.data_ptr(), thr.data_ptr(), cb.data_ptr(), bits, got.data_ptr(), b, n, h, 64,
                                                        0.125, _stream()))
    assert torch.equal(got, want)


@pytest.mark.parametrize("fp8", [False, True])
@pytest.mark.parametrize("batch,tokens", [(1, 197), (3, 257), (40, 197)])
def test_block_equals_its_parts(cuda, batch, tokens, fp8):
    """A block from the host extension on prepared operands (FP8, or fp16 without fuse_elementwise) against the same block taken
    apart: LayerNorm, GELU, skips and attention as separate operations around one-layer calls.  The same bits."""
    from arcq_vit_amd.packed_convert import set_fp8_operands
    from arcq_vit_amd.vit import build_packed_vit
    vit = build_packed_vit("deit_tiny", 4, depth=1, own_attention=fp8)
    if fp8:
        set_fp8_operands(vit)
        vit.blocks[0].fuse_elementwise = True
    x = torch.randn(batch, tokens, 192, generator=torch.Generator().manual_seed(3)).half().to(cuda)
    with torch.no_grad():
        got = vit.blocks(x)
        vit.blocks[0].fuse_elementwise = False
        for part in (vit.blocks[0].attn, vit.blocks[0].mlp):      # hooks: the interpreter runs the block part by part
            part.register_forward_hook(lambda *_: None)
        want = vit.blocks(x)
    assert torch.equal(got, want)
