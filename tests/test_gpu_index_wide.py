"""arcq_linear_index (index-space linears with the codebooks at hand): bit-identical to the oracle's serial evaluation, with
the table an outer product of the codebooks (computed entries) and with one that is not (gathered entries)."""
import ctypes

import numpy as np
import pytest
import torch

from arcq_vit_amd import _lib, synth

pytestmark = pytest.mark.gpu


# one row / one output; rows and outputs past the tiles of both launch shapes (one and two rows per lane); one group,
# whole and partial rounds of three and of four waves
@pytest.mark.parametrize("m,n,k", [(1, 1, 64), (3, 65, 128), (70, 300, 192), (197, 768, 192), (257, 2049, 64), (1000, 200, 384), (601, 513, 384), (600, 545, 448)])
@pytest.mark.parametrize("bits", [4, 3, 2])
@pytest.mark.parametrize("outer", [True, False])
def test_linear_index_bitexact(cuda, oracle, m, n, k, bits, outer):
    cb = synth.quantile_codebook(bits)
    thr = synth.midpoint_thresholds(cb)
    a_cb = cb * 1.1
    x = synth.make_activation(m, k, 3)
    xa = oracle.act_quant_c(x.numpy(), thr, a_cb, bits, 64)
    codes, wc, ws, wcs = oracle.quantize_weight_torch(synth.make_weight(n, k, 4), thr, cb, 64, 1e-6)
    packed_w = oracle.pack_codes_np(codes.numpy(), bits)
    table = (a_cb.view(-1, 1) * cb.view(1, -1)).contiguous()
    if not outer:
        table = table + 0.25 * torch.arange(table.numel()).view_as(table) / table.numel()
    bias = synth.make_bias(n, 5)
    d = lambda t: (torch.from_numpy(t) if isinstance(t, np.ndarray) else t).to(cuda).contiguous()
    meta = (xa["center"], xa["scale"], xa["code_sum"]), (wc.numpy(), ws.numpy(), wcs.numpy())
    want = oracle.linear_forward_packed_c(xa["packed"], *meta[0], packed_w, *meta[1], table.numpy(), bias.numpy(), bits, 64, k, n)
    want8 = oracle.linear_forward_u8_c(xa["codes"], *meta[0], codes.numpy().astype(np.uint8), *meta[1], table.numpy(), bias.numpy(), 64)
    for fmt, xq, wq, ref in ((bits, xa["packed"], packed_w, want), (0, xa["codes"], codes.numpy().astype(np.uint8), want8)):
        t = [d(v) for v in (xq, *meta[0], wq, *meta[1], table, a_cb, cb, bias)]
        y = torch.full((m, n), float("nan"), device=cuda)
        a = _lib.LinearIndexArgs(*[v.data_ptr() for v in t], y.data_ptr(), m, n, k, fmt, 64, 1 << bits, 0)
        _lib.check(_lib.load().arcq_linear_index(ctypes.byref(a), torch.cuda.current_stream().cuda_stream))
        assert np.array_equal(y.cpu().numpy(), ref), fmt
