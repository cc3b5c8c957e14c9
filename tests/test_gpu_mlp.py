"""GPU tests of the one-launch MLP (``otf_mlp_kernel``): LayerNorm, fc1, GELU, fc2's stage 1, fc2 and the skip connection of 64 rows on
one compute unit, against the two layer calls with the fused options, whose bits it has."""
import ctypes

import pytest
import torch

from arcq_vit_amd import _lib, synth
from arcq_vit_amd.packed_linear import ARCQPackedLinear
from arcq_vit_amd.packed_on_the_fly import ARCQPackedLinearOnTheFly
from arcq_vit_amd.quant_source import QuantLinearPCARCQ

pytestmark = pytest.mark.gpu


def _layer(cuda, n, k, bits, gen, bias=True, thresholds=None):
    src = QuantLinearPCARCQ(k, n, bias, bits, bits, 64)
    with torch.no_grad():
        src.linear.weight.copy_(torch.randn(n, k, generator=gen) * 0.02)
        if bias:
            src.linear.bias.copy_(torch.randn(n, generator=gen) * 0.5)
    cb = synth.quantile_codebook(bits)
    src.act_quant.set_codebook(cb)
    src.weight_quant.set_codebook(cb)
    layer = ARCQPackedLinearOnTheFly.from_packed(ARCQPackedLinear(src, "packed")).to(cuda)
    if thresholds is not None:
        layer.activation_thresholds.copy_(thresholds)
    return layer


def _one_launch(x, norm, fc1, fc2, proj=None, attn=None):
    k, h = x.shape[1], fc1.out_features
    ws = [torch.empty(n * k, dtype=torch.float16, device=x.device) for n in (h, h, k)]
    y = torch.empty_like(x)
    keep = []

    def part(layer, w):
        ts = [layer.activation_thresholds, layer.activation_codebook, layer.packed_weight_codes, layer.weight_codebook,
              layer.weight_center, layer.weight_scale, layer.weight_code_sum]
        keep.extend(ts)
        bias = layer.bias_tensor
        return _lib.MlpLayer(*[t.data_ptr() for t in ts], bias.data_ptr() if bias.numel() else None, w.data_ptr())

    g, b = norm.weight.float().contiguous(), norm.bias.float().contiguous()
    a = _lib.MlpArgs(fc1.bits, 1.0e-6, norm.eps, x.shape[0], k, h, x.data_ptr(), g.data_ptr(), b.data_ptr(), part(fc1, ws[0]),
                     part(fc2, ws[1]), y.data_ptr(), None if attn is None else attn.data_ptr(),
                     part(proj, ws[2]) if proj is not None else _lib.MlpLayer())
    lib = _lib.load()
    rc = lib.arcq_mlp_otf(ctypes.byref(a), torch.cuda.current_stream().cuda_stream)
    assert rc == 0, lib.arcq_last_error()
    torch.cuda.synchronize()
    return y


def _norm(cuda, k, gen):
    norm = torch.nn.LayerNorm(k, eps=1e-6)
    with torch.no_grad():
        norm.weight.copy_(1.0 + 0.2 * torch.randn(k, generator=gen))
        norm.bias.copy_(0.2 * torch.randn(k, generator=gen))
    return norm.half().to(cuda)


@pytest.mark.parametrize("m,k,bits,case", [(512, 192, 4, ""), (577, 192, 2, ""), (1001, 256, 3, ""), (640, 384, 4, ""), (12608, 384, 4, ""),
                                           (703, 384, 3, "no bias"), (513, 768, 4, ""), (12608, 768, 4, ""), (2047, 768, 2, "wide"),
                                           (999, 384, 4, "thresholds"), (530, 768, 3, "zeros"), (530, 192, 4, "inf"),
                                           (700, 768, 4, "no wait"), (1000, 384, 4, "no wait")])
def test_one_launch_mlp_has_the_bits_of_the_two_layers(cuda, monkeypatch, m, k, bits, case):
    """Ragged row counts, every width that it serves, both forms of GELU ("wide": inputs beyond +-2.5), quantizer tables that the
    buckets do not hold, constant groups, infinities, and workgroups that rebuild all weights themselves ("no wait")."""
    gen = torch.Generator().manual_seed(7 * m + k)
    fc1 = _layer(cuda, 4 * k, k, bits, gen, case != "no bias")
    thr = None
    if case == "thresholds":
        thr = synth.midpoint_thresholds(synth.quantile_codebook(bits)).clone()
        thr[3] = thr[4]
    fc2 = _layer(cuda, k, 4 * k, bits, gen, case != "no bias", thr)
    norm = _norm(cuda, k, gen)
    x = torch.randn(m, k, generator=gen) * (1.0 + 3.0 * torch.rand(m, 1, generator=gen))
    if case == "wide":
        with torch.no_grad():
            norm.weight.mul_(6.0)
    if case == "zeros":
        x[5:70] = 0.0
        with torch.no_grad():
            norm.bias.zero_()
    if case == "inf":
        x[3, 7] = float("inf")
    x = x.half().to(cuda)
    assert _lib.load().arcq_mlp_otf_supported(m, k, 4 * k)
    before = _lib.load().arcq_rows_wait_timeouts()
    if case == "no wait":
        monkeypatch.setenv("ARCQ_ROWS_WAIT_TICKS", "0")
    y = _one_launch(x, norm, fc1, fc2)
    assert case != "no wait" or _lib.load().arcq_rows_wait_timeouts() > before
    with torch.no_grad():
        h = fc1(x, layernorm=norm, activation="gelu")
        want = fc2(h, residual=x)
    # (a NaN's payload is nobody's contract)
    same = (y.view(torch.int16) == want.view(torch.int16)) | (torch.isnan(y) & torch.isnan(want))
    assert bool(same.all()), int((~same).sum())
    if case != "inf":
        assert bool(torch.isfinite(y).all())


@pytest.mark.parametrize("m,k,bits,case", [(512, 192, 4, ""), (705, 192, 2, "no wait"), (1001, 256, 3, "no bias"), (12608, 384, 4, ""),
                                           (767, 384, 3, "thresholds"), (1000, 384, 2, "inf"), (513, 768, 4, ""), (12608, 768, 4, ""),
                                           (2047, 768, 3, "zeros"), (700, 768, 2, "no wait")])
def test_one_launch_with_proj_has_the_bits_of_the_three_layers(cuda, monkeypatch, m, k, bits, case):
    """The same with proj and the first skip connection in front: attention's output in, its own quantizer tables, the rows that the
    LayerNorm reads come from the product before it."""
    gen = torch.Generator().manual_seed(11 * m + k)
    thr = None
    if case == "thresholds":
        thr = synth.midpoint_thresholds(synth.quantile_codebook(bits)).clone()
        thr[3] = thr[4]
    proj = _layer(cuda, k, k, bits, gen, case != "no bias", thr)
    fc1, fc2 = _layer(cuda, 4 * k, k, bits, gen), _layer(cuda, k, 4 * k, bits, gen)
    norm = _norm(cuda, k, gen)
    x = torch.randn(m, k, generator=gen) * (1.0 + 3.0 * torch.rand(m, 1, generator=gen))
    attn = torch.randn(m, k, generator=gen)
    if case == "zeros":
        attn[5:70] = 0.0
    if case == "inf":
        attn[3, 7] = float("inf")
        x[65, 2] = float("-inf")
    x, attn = x.half().to(cuda), attn.half().to(cuda)
    before = _lib.load().arcq_rows_wait_timeouts()
    if case == "no wait":
        monkeypatch.setenv("ARCQ_ROWS_WAIT_TICKS", "0")
    y = _one_launch(x, norm, fc1, fc2, proj, attn)
    assert case != "no wait" or _lib.load().arcq_rows_wait_timeouts() > before
    with torch.no_grad():
        x1 = proj(attn, residual=x)
        want = fc2(fc1(x1, layernorm=norm, activation="gelu"), residual=x1)
    same = (y.view(torch.int16) == want.view(torch.int16)) | (torch.isnan(y) & torch.isnan(want))
    assert bool(same.all()), int((~same).sum())
    if case != "inf":
        assert bool(torch.isfinite(y).all())


def test_sizes_that_it_does_not_serve_are_refused_before_a_launch(cuda):
    lib = _lib.load()
    cus = torch.cuda.get_device_properties(cuda).multi_processor_count
    assert lib.arcq_mlp_otf_supported(64 * cus, 384, 1536) == 1
    for m, k, h in ((511, 384, 1536), (64 * cus + 1, 384, 1536), (4096, 512, 2048), (4096, 384, 1152), (4096, 1024, 4096)):
        assert lib.arcq_mlp_otf_supported(m, k, h) == 0
        a = _lib.MlpArgs(4, 1e-6, 1e-6, m, k, h)
        assert lib.arcq_mlp_otf(ctypes.byref(a), None) < 0


@pytest.mark.parametrize("model,k", [("deit_tiny", 192), ("deit_small", 384), ("deit_base", 768)])
def test_blocks_with_lent_buffers_take_it(cuda, model, k):
    """A fused block at a size where it pays: three launches, proj in the last one; the bits of the block that runs proj, fc1 and fc2
    as three, also replayed as a graph."""
    from test_gpu_host_extension import _kernels
    from arcq_vit_amd.vit import build_packed_vit
    net = build_packed_vit(model, 4, device=str(cuda), depth=1, shared_buffers=True, max_rows=64 * 197, fuse_elementwise=True,
                           own_attention=True, own_patch_embed=True)
    block = net.blocks[0]
    x = torch.randn(64, 197, k, generator=torch.Generator().manual_seed(5)).half().to(cuda)
    assert _lib.load().arcq_mlp_otf_pays(64 * 197, k, 4 * k) == 1
    with torch.no_grad():
        block.chain_mlp = False
        want = block(x)
        assert "otf_mlp_kernel" not in _kernels(lambda: block(x))
        block.chain_mlp = True
        assert torch.equal(block(x), want)
        names = _kernels(lambda: block(x))
        assert [names.count(n) for n in ("otf_rows_kernel", "attention_kernel", "otf_mlp_kernel")] == [1, 1, 1], names
        graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(graph):
            y = block(x)
        for i in range(4):
            x.copy_(torch.randn(64, 197, k, generator=torch.Generator().manual_seed(10 + i)).half())
            block.chain_mlp = i % 2 == 0
            eager = block(x)
            torch.cuda.synchronize()
            graph.replay()
            torch.cuda.synchronize()
            assert torch.equal(y, eager), i


@pytest.mark.parametrize("case", ["proj of three bits", "fc2 of three bits"])
def test_blocks_that_it_serves_in_part_or_not(cuda, case):
    """A proj of other code bits is a layer call and the launch starts at the LayerNorm; with other bits in fc2 there is no such launch."""
    from test_gpu_host_extension import _kernels
    from arcq_vit_amd.packed_convert import share_buffers
    from arcq_vit_amd.vit import build_packed_vit
    gen = torch.Generator().manual_seed(9)
    net = build_packed_vit("deit_small", 4, device=str(cuda), depth=1, shared_buffers=True, max_rows=64 * 197, fuse_elementwise=True,
                           own_attention=True, own_patch_embed=True)
    block = net.blocks[0]
    x = torch.randn(64, 197, 384, generator=gen).half().to(cuda)
    if case == "proj of three bits":
        block.attn.proj = _layer(cuda, 384, 384, 3, gen)
    else:
        block.mlp.fc2 = _layer(cuda, 384, 1536, 3, gen)
    share_buffers(net, 64 * 197)
    with torch.no_grad():
        block.chain_mlp = False
        want = block(x)
        block.chain_mlp = True
        assert torch.equal(block(x), want)
        names = _kernels(lambda: block(x))
    assert names.count("otf_mlp_kernel") == (0 if case == "fc2 of three bits" else 1), names
