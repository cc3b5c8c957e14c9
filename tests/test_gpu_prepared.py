"""arcq_prepare / arcq_linear_prepared (the layer in two launches on prepared operands): x_hat, w_hat and the outputs have
the bits of the stand-alone kernels, at the edges of the tiles and of the row ranges that choose between the kernels."""
import ctypes

import numpy as np
import pytest
import torch

from arcq_vit_amd import _lib, ops, synth

pytestmark = pytest.mark.gpu


def _layer(oracle, cuda, n, k, bits, seed):
    cb = synth.quantile_codebook(bits)
    thr = synth.midpoint_thresholds(cb)
    codes, center, scale, code_sum = oracle.quantize_weight_torch(synth.make_weight(n, k, seed), thr, cb, 64, 1e-6)
    packed = torch.from_numpy(oracle.pack_codes_np(codes.numpy(), bits))
    w = [t.to(cuda).contiguous() for t in (packed, cb, center, scale, code_sum)]
    return (cb * 1.05).to(cuda), (thr * 1.05).to(cuda), w, synth.make_bias(n, seed).to(cuda)


def _stream():
    return torch.cuda.current_stream().cuda_stream


def _prepare(x, thr, cb, bits, ln=None, weights=(), row_major=False):
    a = _lib.PrepareArgs()
    a.bits = bits
    outs = []
    keep = [x, thr, cb]
    if x is not None:
        a.x_dtype = _lib.ARCQ_F16 if x.dtype == torch.float16 else _lib.ARCQ_F32
        a.rows, a.K = x.shape
        x_hat = torch.empty(x.numel(), dtype=torch.float16, device=x.device)
        a.x, a.thresholds, a.codebook, a.x_hat = x.data_ptr(), thr.data_ptr(), cb.data_ptr(), x_hat.data_ptr()
        if ln is not None:
            a.ln_weight, a.ln_bias, a.ln_eps = ln[0].data_ptr(), ln[1].data_ptr(), ln[2]
        outs.append(x_hat)
    for i, w in enumerate(weights):
        j = a.weights[i]
        j.N, j.K, j.row_major = w[0].shape[0], w[2].shape[1] * 64, int(row_major)
        out = torch.empty(j.N * j.K, dtype=torch.float16, device=w[0].device)
        j.packed, j.codebook, j.center, j.scale, j.code_sum, j.w_hat = [t.data_ptr() for t in w] + [out.data_ptr()]
        outs.append(out)
    _lib.check(_lib.load().arcq_prepare(ctypes.byref(a), _stream()))
    return outs


def _linear(x_hat, w_hat, bias, m, n, k, out_dtype=torch.float16, gelu=False, residual=None, nq=None, bits=4, row_major=False):
    a = _lib.LinearPreparedArgs()
    y = torch.empty((m, n), dtype=out_dtype, device=x_hat.device)
    a.y_dtype = _lib.ARCQ_F16 if out_dtype == torch.float16 else _lib.ARCQ_F32
    a.activation, a.w_row_major = int(gelu), int(row_major)
    a.M, a.N, a.K = m, n, k
    a.x_hat, a.w_hat, a.bias, a.y = x_hat.data_ptr(), w_hat.data_ptr(), bias.data_ptr(), y.data_ptr()
    if residual is not None:
        a.residual = residual.data_ptr()
    if nq is not None:
        a.next_thresholds, a.next_codebook, a.next_bits = nq[0].data_ptr(), nq[1].data_ptr(), bits
    _lib.check(_lib.load().arcq_linear_prepared(ctypes.byref(a), _stream()))
    return y


def _col_blocks(w, n, k):
    return w.reshape(n // 32, 32, k // 8, 8).permute(0, 2, 1, 3).reshape(-1)


@pytest.mark.parametrize("m,k,bits,dtype", [(1, 64, 4, torch.float16), (31, 192, 3, torch.float16), (197, 384, 4, torch.float16),
                                            (591, 1024, 3, torch.float16), (70, 768, 2, torch.float32), (33, 4096, 4, torch.float32),
                                            (1000, 448, 4, torch.float16), (6000, 1536, 4, torch.float16), (40000, 384, 4, torch.float16)])
@pytest.mark.parametrize("ln", [False, True])
def test_prepare_equals_the_stand_alone_kernels(cuda, oracle, m, k, bits, dtype, ln):
    if ln and k > 1024:
        pytest.skip("no stand-alone kernel to compare with")
    cb, thr, w, _ = _layer(oracle, cuda, 96, k, bits, 5)
    _, _, w2, _ = _layer(oracle, cuda, 32, 320, bits, 6)
    x = synth.make_activation(m, k, 7).to(cuda, dtype)
    g = torch.linspace(0.5, 1.5, k, device=cuda)
    b = torch.linspace(-0.2, 0.2, k, device=cuda)
    outs = _prepare(x, thr, cb, bits, (g, b, 1e-6) if ln else None, (w, w2))
    want = (ops.quantize_activation_blocked_ln(x, g, b, 1e-6, thr, cb, bits) if ln
            else ops.quantize_activation_blocked(x, thr, cb, bits)).reshape(-1)
    assert torch.equal(outs[0].view(torch.int16), want.view(torch.int16))
    for got, ww, n, kk in ((outs[1], w, 96, k), (outs[2], w2, 32, 320)):
        dense = ops.unpack_weight_hip(*ww, bits, 64)
        assert torch.equal(got.view(torch.int16), _col_blocks(dense, n, kk).view(torch.int16))
    assert torch.equal(_prepare(None, None, None, bits, None, (w2,))[0], outs[2])          # weights alone
    dense = ops.unpack_weight_hip(*w, bits, 64).reshape(-1)
    assert torch.equal(_prepare(None, None, None, bits, None, (w,), row_major=True)[0], dense)


# below 512 rows: the three tile shapes of the split kernel; from 512 on: the three of the tile kernel; ragged last row
# blocks, column tiles past N, one group and more groups than stages
@pytest.mark.parametrize("m,n,k,bits", [(1, 32, 64, 4), (197, 384, 384, 4), (197, 1152, 384, 3), (100, 3072, 1024, 4), (394, 4096, 1024, 4),
                                        (511, 96, 4096, 2), (512, 32, 64, 4), (591, 1024, 1024, 3), (600, 160, 320, 4), (1001, 2304, 768, 4),
                                        (1576, 4096, 1024, 4), (3152, 768, 3072, 4), (6304, 1184, 448, 2)])
def test_linear_prepared_equals_the_layer_call(cuda, oracle, m, n, k, bits):
    cb, thr, w, bias = _layer(oracle, cuda, n, k, bits, 11)
    x = synth.make_activation(m, k, 13).to(cuda, torch.float16)
    x_hat, w_hat = _prepare(x, thr, cb, bits, None, (w,))
    for out in (torch.float16, torch.float32):
        want = ops.linear_otf(x, thr, cb, *w, bias, bits, 64, out_dtype=out)
        got = _linear(x_hat, w_hat, bias, m, n, k, out)
        assert torch.equal(got, want), (out, (got - want).abs().max().item())
        if m >= 512:
            rows = _prepare(None, None, None, bits, None, (w,), row_major=True)[0]
            assert torch.equal(_linear(x_hat, rows, bias, m, n, k, out, row_major=True), want)
    res = synth.make_activation(m, n, 17).to(cuda, torch.float16)
    want = res + torch.nn.functional.gelu(ops.linear_otf(x, thr, cb, *w, bias, bits, 64))
    assert torch.equal(_linear(x_hat, w_hat, bias, m, n, k, gelu=True, residual=res), want)


@pytest.mark.parametrize("m,n,k,bits", [(1, 64, 64, 4), (197, 1536, 384, 4), (394, 4096, 1024, 3), (197, 4096, 1024, 2), (591, 4096, 1024, 3),
                                        (591, 192, 128, 2), (1576, 3072, 768, 4), (6304, 4096, 1024, 4)])
def test_linear_prepared_quantizes_for_the_next_layer(cuda, oracle, m, n, k, bits):
    cb, thr, w, bias = _layer(oracle, cuda, n, k, bits, 19)
    x = synth.make_activation(m, k, 23).to(cuda, torch.float16)
    x_hat, w_hat = _prepare(x, thr, cb, bits, None, (w,))
    for gelu in (False, True):
        y = _linear(x_hat, w_hat, bias, m, n, k, gelu=gelu)
        got = _linear(x_hat, w_hat, bias, m, n, k, gelu=gelu, nq=(thr, cb), bits=bits).reshape(-1)
        want = ops.quantize_activation_blocked(y, thr, cb, bits).reshape(-1)
        assert torch.equal(got.view(torch.int16), want.view(torch.int16)), gelu


# (from the seventh: parts of a head with several query tiles, whose idle waves leave early, or, at (4, 256, 15) and (3, 225, 13) with
# two tiles in a part, quantize with the others)
@pytest.mark.parametrize("b,n,h,bits", [(1, 197, 6, 4), (3, 197, 12, 3), (2, 33, 3, 2), (5, 1, 1, 4), (7, 101, 2, 4), (2, 256, 16, 3),
                                        (16, 197, 6, 4), (11, 197, 11, 3), (2, 197, 24, 4), (5, 129, 16, 2), (4, 256, 15, 4), (3, 225, 13, 3)])
def test_attention_quantizes_for_the_proj_layer(cuda, oracle, b, n, h, bits):
    cb, thr, _, _ = _layer(oracle, cuda, 32, 64, bits, 29)
    qkv = synth.make_activation(b * n, 3 * h * 64, 31).to(cuda, torch.float16).reshape(b, n, 3 * h * 64).contiguous()
    y = ops.attention_fwd(qkv, h).reshape(b * n, h * 64)
    want = ops.quantize_activation_blocked(y, thr, cb, bits).reshape(-1)
    got = torch.empty(b * n * h * 64, dtype=torch.float16, device=cuda)
    _lib.check(_lib.load().arcq_attention_quant_fwd(qkv.data_ptr(), thr.data_ptr(), cb.data_ptr(), bits, got.data_ptr(), b, n, h, 64,
                                                    0.125, _stream()))
    assert torch.equal(got.view(torch.int16), want.view(torch.int16))


def test_prepared_argument_errors(cuda):
    lib = _lib.load()
    a, b = _lib.PrepareArgs(), _lib.LinearPreparedArgs()
    a.bits = 7
    assert lib.arcq_prepare(ctypes.byref(a), None) == -1
    a.bits, a.rows, a.K = 4, 3, 100
    assert lib.arcq_prepare(ctypes.byref(a), None) == -2
    b.M, b.N, b.K = 4, 33, 64
    assert lib.arcq_linear_prepared(ctypes.byref(b), None) == -4


# one output a thread, and eight behind the tile kernel and the one of large launches; neighbouring columns hold neighbouring values
# (a wave of small values takes a form of its own) or values far apart
@pytest.mark.parametrize("m", [32, 512, 6400])
@pytest.mark.parametrize("apart", [False, True])
def test_gelu_of_every_fp16_value(cuda, m, apart):
    every = torch.arange(65536, dtype=torch.int32).to(torch.int16).view(torch.float16)
    if apart:
        every = every.view(256, 256).t().reshape(-1)
    n, k = 16384, 64
    x_hat = torch.zeros(m * k, dtype=torch.float16, device=cuda)
    w_hat = torch.zeros(n * k, dtype=torch.float16, device=cuda)
    for part in every.to(cuda).split(n):
        y = _linear(x_hat, w_hat, part.float(), m, n, k, gelu=True)               # zero operands: the output is the bias
        want = torch.nn.functional.gelu(part)
        wrong = ~((y == want) | (y.isnan() & want.isnan())).all(0)
        assert not bool(wrong.any()), part[wrong][:8]


# the weight-stationary kernels with a lane per group: every way of dealing the last blocks, ragged rows, a half slab past the last
# column
@pytest.mark.parametrize("m,n,k,bits", [(12608, 1536, 384, 4), (6301, 1600, 320, 3), (9000, 448, 64, 2), (3152, 3072, 768, 4),
                                        (4001, 832, 448, 4), (12577, 3136, 768, 3)])
def test_linear_prepared_quantizes_many_rows(cuda, oracle, m, n, k, bits):
    test_linear_prepared_quantizes_for_the_next_layer(cuda, oracle, m, n, k, bits)
