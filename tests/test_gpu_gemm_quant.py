"""``gemm_quant_kernel`` (products that end with the next layer's stage 1, 64 columns of the weights resident in LDS): the bits of the
weight-stationary kernels, which the row-major weights select."""
import pytest
import torch

import test_gpu_prepared as f16
import test_gpu_prepared_fp8 as f8
from arcq_vit_amd import _lib, ops, synth

pytestmark = pytest.mark.gpu

# One row past a pair of row blocks, past a block, whole pairs; slabs that do not divide the compute units, more slabs than compute
# units; odd numbers of output groups; six units to the eighteen that LDS holds; outputs beyond 200 MB.
SHAPES = [(1153, 4096, 1024, 4, ""), (1249, 4160, 768, 3, ""), (2048, 2304, 1024, 2, ""), (3360, 1536, 384, 4, ""), (513, 17408, 512, 4, ""),
          (1216, 4096, 768, 4, "thresholds"), (1153, 4096, 1024, 3, "large"), (26017, 4160, 512, 4, ""),
          (1601, 3072, 1152, 4, "")]


@pytest.mark.parametrize("m,n,k,bits,case", SHAPES)
def test_fp16(cuda, oracle, m, n, k, bits, case):
    cb, thr, w, bias = f16._layer(oracle, cuda, n, k, bits, 3)
    assert _lib.load().arcq_prepared_quant_row_major(m, n, k, 0) == 0 and _lib.load().arcq_prepared_row_major(m, n, k) == 1
    x = (synth.make_activation(m, k, 5) * (30.0 if case == "large" else 1.0)).to(cuda, torch.float16)
    nthr = thr.clone()
    if case == "thresholds":
        nthr[4] = nthr[5]
    x_hat, cols = f16._prepare(x, thr, cb, bits, None, (w,))
    rows = f16._prepare(None, None, None, bits, None, (w,), row_major=True)[0]
    for gelu in (True, False):
        want = f16._linear(x_hat, rows, bias, m, n, k, gelu=gelu, nq=(nthr, cb), bits=bits, row_major=True)
        got = f16._linear(x_hat, cols, bias, m, n, k, gelu=gelu, nq=(nthr, cb), bits=bits)
        assert torch.equal(got.view(torch.int16), want.view(torch.int16)), gelu


@pytest.mark.parametrize("m,n,k,bits", [(1153, 4096, 1024, 4), (1249, 4160, 768, 3), (2048, 4096, 1536, 2), (513, 17408, 1024, 4), (6304, 3072, 704, 4),
                                        (1601, 3072, 2304, 4)])
def test_fp8(cuda, oracle, m, n, k, bits):
    """Also the padding of a row to 128 values, of the operands (704 values) and of the output (4 160)."""
    cb, thr, w, bias = f16._layer(oracle, cuda, n, k, bits, 3)
    mult = ops.fp8_weight_multiplier(*w[1:5])
    assert _lib.load().arcq_prepared_quant_row_major(m, n, k, 1) == 0
    x = synth.make_activation(m, k, 5).to(cuda, torch.float16)
    x8, cols = f8._prepare(x, thr, cb, bits, w, mult, False)
    _, rows = f8._prepare(x, thr, cb, bits, w, mult, True)
    for gelu in (True, False):
        want = f8._linear(x8, rows, bias, m, n, k, mult, True, gelu=gelu, nq=(thr, cb), bits=bits)
        got = f8._linear(x8, cols, bias, m, n, k, mult, False, gelu=gelu, nq=(thr, cb), bits=bits)
        assert torch.equal(got, want), gelu
