"""Codes and metadata without x_hat (the encoding direction's own kernel) against the kernel that writes everything: one group,
tiles with a remainder, both sides of the line between one tile per wave and walking waves."""
import pytest
import torch

from arcq_vit_amd import _lib, synth

pytestmark = pytest.mark.gpu


def _quantize(x, thr, cb, bits, packed, with_x_hat):
    m, k = x.shape
    code = lambda t: _lib.ARCQ_F16 if t.dtype == torch.float16 else _lib.ARCQ_F32
    out = torch.zeros(m * k * (bits if packed else 8) // 8 + 16, dtype=torch.uint8, device=x.device)
    meta = [torch.zeros(m * k // 64 + 4, device=x.device) for _ in range(3)]
    x_hat = torch.empty_like(x) if with_x_hat else None
    p = out.data_ptr()
    _lib.check(_lib.load().arcq_act_quant(x.data_ptr(), code(x), thr.data_ptr(), cb.data_ptr(), p if packed else None, None if packed else p,
                                          *[t.data_ptr() for t in meta], x_hat.data_ptr() if with_x_hat else None, code(x), m, k, bits, 64,
                                          1e-6, torch.cuda.current_stream().cuda_stream))
    return [out] + meta


@pytest.mark.parametrize("m,k", [(1, 64), (31, 64), (33, 192), (1000, 448), (2048, 2048), (2049, 2048), (12608, 384)])
@pytest.mark.parametrize("bits,packed,dtype", [(4, True, torch.float32), (3, True, torch.float32), (2, True, torch.float16),
                                               (4, False, torch.float16), (3, False, torch.float32)])
def test_codes_kernel(cuda, m, k, bits, packed, dtype):
    cb = synth.quantile_codebook(bits)
    thr = synth.midpoint_thresholds(cb).to(cuda)
    x = synth.make_activation(m, k, 3).to(cuda, dtype)
    if m > 30:
        x[17] = 0.0                      # no deviation: every quotient 0
        x[18] *= 1e-30                   # outside the range of the fast quotient
    for got, want in zip(_quantize(x, thr, cb.to(cuda), bits, packed, False), _quantize(x, thr, cb.to(cuda), bits, packed, True)):
        assert torch.equal(got, want)
