"""Infinities, NaN, overflowing and vanishing values through the kernels of the prepared path: the LayerNorm in front of stage 1
(up to 2 048 inputs), the patch quantizer's fast form, and the products.  What is not finite stays in its group, row or column,
and everything else has the bits it has without it."""
import numpy as np
import pytest
import torch

from arcq_vit_amd import _lib, ops, synth
from test_gpu_patch_conv import _blocked
from test_gpu_prepared import _col_blocks, _layer, _linear, _prepare

pytestmark = pytest.mark.gpu
INF, NAN = float("inf"), float("nan")


def _same(got, want):
    """The same bits, but for the NaN, whose bits are free."""
    nan = np.isnan(want)
    view = np.uint16 if want.dtype == np.float16 else np.uint32
    return np.array_equal(np.isnan(got), nan) and np.array_equal(got.view(view)[~nan], want.view(view)[~nan])


# one and two rows per wave, one to thirty-two groups, four to thirty-two partial sums a row; a ragged last block
@pytest.mark.parametrize("m,k,bits", [(70, 64, 4), (45, 192, 3), (131, 1024, 4), (33, 1088, 4), (64, 1536, 3), (70, 1984, 2), (197, 2048, 4),
                                      (1000, 2048, 3)])
@pytest.mark.parametrize("dtype", [torch.float16, torch.float32])
def test_layernorm_in_front_of_stage_1(cuda, oracle, m, k, bits, dtype):
    cb, thr, _, _ = _layer(oracle, cuda, 32, 64, bits, 5)
    x = (synth.make_activation(m, k, 21) * 1.7 + 0.3).to(dtype)
    x[3, 5], x[4, k - 1], x[5, 0] = NAN, INF, -INF
    x[6], x[7] = 0.0, 3.25                                                # no variance
    x[8] = x[8].clamp(-3, 3) * (2.0e4 if dtype == torch.float16 else 1.0e30)     # large / the sum of squares overflows
    x[9] = x[9] * (1.0e-7 if dtype == torch.float16 else 1.0e-42)         # subnormal
    x[10, ::2], x[10, 1::2] = 6.0e4, -6.0e4
    g = torch.linspace(0.5, 1.5, k)
    b = torch.linspace(-0.2, 0.2, k)
    with np.errstate(all="ignore"):
        ln = oracle.layernorm_rows_np(x.float().numpy(), g.numpy(), b.numpy(), 1e-6, out_f16=dtype == torch.float16)
        want = oracle.act_quant_c(ln, thr.cpu(), cb.cpu(), bits, 64)["x_hat"].astype(np.float16)
    got = _prepare(x.to(cuda), thr, cb, bits, (g.to(cuda), b.to(cuda), 1e-6))[0]
    assert _same(got.cpu().numpy(), _blocked(want))
    others = np.delete(want, [3, 4, 5], 0)
    assert np.isnan(want[3:6]).all() and np.isfinite(others).all()


@pytest.mark.parametrize("dtype", [torch.float16, torch.float32])
@pytest.mark.parametrize("b,h,w,bits", [(1, 16, 16, 4), (2, 64, 48, 3), (3, 224, 224, 2)])
def test_patch_quantizer(cuda, oracle, b, h, w, bits, dtype):
    cb = synth.quantile_codebook(bits)
    thr = synth.midpoint_thresholds(cb)
    img = ((torch.rand(b, 3, h, w, generator=torch.Generator().manual_seed(h)) - 0.45) / 0.23).to(dtype)
    img[0, 0, 0, 0], img[0, 1, 1, 2], img[0, 2, 2, 9], img[0, :, 3, 3] = NAN, INF, -INF, INF
    img[0, 0, 4, :8] = 6.0e4
    if dtype == torch.float32:
        img[0, :, 5, 0] = torch.tensor([1e30, -1e30, 3e38])               # the sum of squares overflows
        img[0, :, 6, 1] = torch.tensor([3e38, 3e38, 3e38])                # the sum does
        img[0, :, 7, 2] = torch.tensor([1e-41, 2e-42, -1e-41])
        bits_of = img.view(torch.int32)
        for i, payload in enumerate((0x7fc00001, 0x7fc01ff8, 0x7fa01008, -0x3ff008, -0x1008)):      # NaN with payloads, both signs
            bits_of[0, i % 3, 8 + i, i] = payload
    else:
        img[0, :, 7, 2] = torch.tensor([6e-8, -6e-8, 1.2e-7])
    pix = img.permute(0, 2, 3, 1).reshape(-1, 3).contiguous()
    with np.errstate(all="ignore"):
        xh = oracle.act_quant_c(pix.float().numpy(), thr, cb, bits, 3)["x_hat"].astype(np.float16)
    rows = xh.reshape(b, h // 16, 16, w // 16, 16, 3).transpose(0, 1, 3, 5, 2, 4).reshape(b * (h // 16) * (w // 16), 768)
    got = ops.quantize_patches(img.to(cuda), thr.to(cuda), cb.to(cuda), bits)
    assert _same(got.cpu().numpy(), rows)
    gotb = ops.quantize_patches(img.to(cuda), thr.to(cuda), cb.to(cuda), bits, blocked=True)
    assert _same(gotb.cpu().numpy(), _blocked(rows))


# the split kernel, the tile kernel and the weight-stationary kernels on row-major weights
@pytest.mark.parametrize("m,n,k", [(37, 96, 192), (197, 384, 1536), (1000, 384, 384), (6304, 1536, 384), (12608, 768, 768)])
@pytest.mark.parametrize("gelu", [False, True])
def test_products(cuda, oracle, m, n, k, gelu):
    bits = 4
    cb, thr, w, bias = _layer(oracle, cuda, n, k, bits, 9)
    row_major = bool(_lib.load().arcq_prepared_row_major(m, n, k))
    dense = ops.unpack_weight_hip(*w, bits, 64)
    residual = synth.make_activation(m, n, 4).half().to(cuda)
    x = ops.dequant_activation_hip(synth.make_activation(m, k, 7).to(cuda), thr, cb, 64).half()
    bad_rows, bad_cols = [0, 5, m - 1], [1, n - 1]
    dirty, dense_dirty = x.clone(), dense.clone()
    dirty[0, 3], dirty[5, k - 1], dirty[m - 1, :] = NAN, INF, -INF
    dense_dirty[1, 7], dense_dirty[n - 1, 0] = NAN, INF

    def run(a, d):
        xb = torch.from_numpy(_blocked(a.cpu().numpy())).to(cuda)
        wd = d.reshape(-1) if row_major else _col_blocks(d, n, k).contiguous()
        return _linear(xb, wd, bias, m, n, k, gelu=gelu, residual=residual, row_major=row_major)

    clean = run(x, dense).cpu()
    ok_rows = [i for i in range(m) if i not in bad_rows]
    ok_cols = [i for i in range(n) if i not in bad_cols]
    assert bool(torch.isfinite(clean).all())
    y = run(dirty, dense).cpu()
    assert torch.equal(y[ok_rows], clean[ok_rows])
    with np.errstate(all="ignore"):
        want = dirty[bad_rows].cpu().double() @ dense.cpu().double().T + bias.cpu().double()
    if gelu:
        want = torch.where(want == -INF, torch.tensor(NAN, dtype=torch.float64), want)       # -inf * 0, as torch's GELU has it
    assert torch.equal(torch.isnan(y[bad_rows]), torch.isnan(want))
    finite = ~torch.isnan(want)
    assert torch.equal(y[bad_rows].double()[finite], want[finite])        # infinities of the right sign
    y = run(x, dense_dirty).cpu()
    assert torch.equal(y[:, ok_cols], clean[:, ok_cols])
    assert bool(torch.isnan(y[:, 1]).all()) and not bool(torch.isfinite(y[:, n - 1]).any())
