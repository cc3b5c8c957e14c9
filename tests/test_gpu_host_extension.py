"""What the host extension promises around its hot calls: the plain case only, and the interpreter's results where it takes
over -- types that autocast chooses, flags of any type, copies of modules, grad mode, alignment, memory, threads."""
import collections

import numpy as np
import pytest
import torch
from torch.utils._python_dispatch import TorchDispatchMode

import arcq_vit_amd as A
from arcq_vit_amd import synth
from arcq_vit_amd.vit import build_packed_vit

pytestmark = pytest.mark.gpu


def _packed(k, n, fmt="packed", bits=4, seed=1):
    src = A.QuantLinearPCARCQ(k, n, True, bits, bits, 64)
    cb = synth.quantile_codebook(bits)
    src.act_quant.set_codebook(cb)
    src.weight_quant.set_codebook(cb)
    with torch.no_grad():
        src.linear.weight.copy_(synth.make_weight(n, k, seed))
        src.linear.bias.copy_(synth.make_bias(n, seed))
    return A.ARCQPackedLinear(src.eval(), fmt).cuda()


def _on_the_fly(k, n, bits=4, seed=1):
    return A.ARCQPackedLinearOnTheFly.from_packed(_packed(k, n, bits=bits, seed=seed))


def _vit(**kw):
    return build_packed_vit("deit_tiny", 4, num_classes=10, depth=1, **kw)


def _tokens(*shape, dtype=torch.float16, seed=3):
    rows = int(np.prod(shape[:-1]))
    return synth.make_activation(rows, shape[-1], seed).reshape(shape).cuda().to(dtype)


def _interpreted(block, x):
    """The block as the interpreter runs it, layer by layer: a hook on one of its layers is enough for that."""
    hook = block.attn.qkv.register_forward_hook(lambda *_: None)
    try:
        return block(x)
    finally:
        hook.remove()


class _CountOps(TorchDispatchMode):
    """Counts torch's operations, those of C++ code included (each of them comes back to Python for it)."""

    def __init__(self):
        super().__init__()
        self.seen = collections.Counter()

    def __torch_dispatch__(self, func, types, args=(), kwargs=None):
        self.seen[str(func)] += 1
        return func(*args, **(kwargs or {}))


@pytest.mark.parametrize("fused", [False, True])
@pytest.mark.parametrize("half", [True, False])
@pytest.mark.parametrize("batch,tokens", [(2, 197), (5, 197), (1, 300)])
def test_block_under_bf16_autocast(cuda, batch, tokens, half, fused):
    """torch's attention then hands proj a bf16 tensor, which proj takes rounded to fp16."""
    block = _vit(half_chain=half, fuse_elementwise=fused).blocks[0]
    x = _tokens(batch, tokens, 192, dtype=torch.float16 if half else torch.float32)
    with torch.no_grad(), torch.autocast("cuda", dtype=torch.bfloat16):
        try:
            want = _interpreted(block, x)
        except ValueError:                 # (a skip connection of another type than the layers' outputs does not fuse)
            with pytest.raises(ValueError, match="residual"):
                block(x)
            return
        got = block(x)
        with _CountOps() as ops:
            assert torch.equal(block(x), got)
    assert got.dtype == want.dtype and torch.equal(got, want)
    attentions = sum(n for name, n in ops.seen.items() if "scaled_dot_product" in name)
    assert attentions == 1 and ops.seen["aten.native_layer_norm.default"] == (0 if fused else 2), ops.seen


@pytest.mark.parametrize("yes,no", [(1, 0), (np.bool_(True), np.bool_(False)), ("yes", "")])
def test_flags_of_any_type(cuda, yes, no):
    """Flags decide by their truth, as `if flag:` does, wherever the extension reads them."""
    fc1, fc2 = _on_the_fly(192, 768), _on_the_fly(768, 192)
    x = _tokens(197, 192)
    with torch.no_grad():
        h = fc1(x, activation="gelu", quantize_for=fc2)
        ready = fc2(h, input_is_xhat=True)
        assert torch.equal(fc2(h, input_is_xhat=yes), ready)
        assert not torch.equal(fc2(h, input_is_xhat=no), ready)
        f16 = fc1(x)
        fc1.fp8_operands = True
        f8 = fc1(x)
        fc1.fp8_operands = yes
        assert torch.equal(fc1(x), f8) and not torch.equal(f16, f8)
        fc1.fp8_operands = no
        assert torch.equal(fc1(x), f16)


def test_block_flags_of_any_type(cuda):
    x = _tokens(3, 197, 192)
    results = {}
    for name, yes, no in (("bool", True, False), ("int", 1, 0)):
        block = _vit().blocks[0]
        with torch.no_grad():
            for fuse, own, chain in ((yes, yes, yes), (yes, no, no), (no, yes, yes), (no, no, no)):
                block.fuse_elementwise, block.attn.own_kernel, block.chain_mlp = fuse, own, chain
                results.setdefault((bool(fuse), bool(own), bool(chain)), []).append(block(x))
    assert all(torch.equal(a, b) for a, b in results.values())
    assert not torch.equal(results[True, True, True][0], results[False, False, False][0])


def test_a_flag_that_raises(cuda):
    class Odd:
        def __bool__(self):
            raise KeyError("odd")

    layer = _on_the_fly(192, 768)
    layer.fp8_operands = Odd()
    with pytest.raises(KeyError, match="odd"):
        layer(_tokens(197, 192))


def test_copies_of_a_layer_have_plans_of_their_own(cuda):
    """DataParallel's replicas and shallow copies carry the __dict__ of the layer they were made from."""
    import copy
    layer, x = _on_the_fly(192, 768), _tokens(197, 192)
    with torch.no_grad():
        want = layer(x)
        replica = layer._replicate_for_data_parallel()
        assert replica._host_plan is layer._host_plan                  # handed over by the copy, not to be used by it
        replica._buffers["bias_tensor"] = layer.bias_tensor + 64.0
        shifted = replica(x)
        assert not torch.equal(shifted, want) and replica._host_plan is not layer._host_plan
        plans = layer._host_plan, replica._host_plan
        assert torch.equal(layer(x), want) and torch.equal(replica(x), shifted)
        assert (layer._host_plan, replica._host_plan) == plans         # neither call disturbed the other's
        for other in (copy.copy(layer), copy.deepcopy(layer)):
            assert torch.equal(other(x), want) and other._host_plan is not layer._host_plan


def test_replicas_on_threads_and_streams(cuda):
    """A layer and its replica with other weights, called from two threads on streams of their own while their buffers are
    replaced: with FP8 operands a call then stops to read the metadata back, and the other thread runs meanwhile."""
    import threading
    layer, x = _on_the_fly(192, 768), _tokens(600, 192)
    layer.fp8_operands = True
    replica = layer._replicate_for_data_parallel()
    replica._buffers["weight_scale"] = layer.weight_scale * 64.0
    replica._buffers["weight_center"] = layer.weight_center * 64.0
    with torch.no_grad():
        want = [m(x).clone() for m in (layer, replica)]
    assert not torch.equal(*want)
    torch.cuda.synchronize()
    failures = []

    def work(module, expected):
        with torch.cuda.stream(torch.cuda.Stream()), torch.no_grad():
            for _ in range(20):
                module._buffers["weight_scale"] = module.weight_scale.clone()
                if not torch.equal(module(x), expected):
                    failures.append(module)

    threads = [threading.Thread(target=work, args=a) for a in zip((layer, replica), want)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert not failures


@pytest.mark.parametrize("kind", ["packed", "dequant_gemm", "on_the_fly", "conv"])
def test_a_module_that_moves_away_leaves_no_memory_behind(cuda, kind):
    """Neither the buffers nor the fp32 copies of those that are not fp32 outlive `.cpu()` in the extension's plan."""
    torch.cuda.synchronize()
    before = torch.cuda.memory_allocated()
    if kind == "conv":
        src = A.QuantConv2dPCARCQ(3, 4096, 16, 16, 0, True, 4, 4, 64)
        for q in (src.act_quant, src.weight_quant):
            q.set_codebook(synth.quantile_codebook(4))
        module, x = A.ARCQPackedPatchConv(src).cuda(), synth.make_images(1, 1).cuda()
    else:
        module = _on_the_fly(4096, 4096) if kind == "on_the_fly" else _packed(4096, 4096, kind)
        x = _tokens(600, 4096, dtype=torch.float32)
    module.weight_scale = module.weight_scale.half()                       # needs an fp32 copy
    with torch.no_grad():
        module(x)
    assert module._host_plan is not None
    module.cpu()
    del x
    assert torch.cuda.memory_allocated() - before < 1 << 16


def test_a_replaced_buffer_is_not_kept(cuda):
    layer, x = _packed(4096, 4096, "dequant_gemm"), _tokens(600, 4096, dtype=torch.float32)
    with torch.no_grad():
        want = layer(x)
        before = torch.cuda.memory_allocated()
        layer.weight_dequant = layer.weight_dequant.clone()
        assert torch.cuda.memory_allocated() - before < 1 << 16
        assert torch.equal(layer(x), want)


def test_views_of_a_buffer_are_other_buffers(cuda):
    """The same memory under other sizes or strides: the copies made from it are made again."""
    layer, x = _on_the_fly(192, 192), _tokens(197, 192)
    with torch.no_grad():
        square = torch.rand(192, 192, device=cuda) * 0.02
        layer.weight_scale = square[:, :3]
        a = layer(x)
        layer.weight_scale = square.t()[:, :3]
        b = layer(x)
        layer.weight_scale = square[:, :3].contiguous()
        assert torch.equal(layer(x), a)
        layer.weight_scale = square.t()[:, :3].contiguous()
        assert torch.equal(layer(x), b) and not torch.equal(a, b)


def test_parameters_may_be_swapped(cuda):
    """`torch.__future__.set_swap_module_params_on_conversion` refuses tensors that something else refers to."""
    block, x = _vit(fuse_elementwise=True).blocks[0], _tokens(2, 197, 192)
    with torch.no_grad():
        want = block(x)
    torch.__future__.set_swap_module_params_on_conversion(True)
    try:
        block.cpu().cuda()
    finally:
        torch.__future__.set_swap_module_params_on_conversion(False)
    with torch.no_grad():
        assert torch.equal(block(x), want)


def test_modules_with_a_plan_pickle_without_it(cuda, tmp_path):
    layer, x = _on_the_fly(192, 768), _tokens(197, 192)
    with torch.no_grad():
        want = layer(x)
        torch.save(layer, tmp_path / "layer.pt")
        again = torch.load(tmp_path / "layer.pt", weights_only=False)
        assert again._host_plan is None and torch.equal(again(x), want)


def test_inference_tensors_changed_in_place(cuda):
    """Tensors made under inference_mode carry no version: what a layer derives from its own and from a LayerNorm's (fp32
    copies, the FP8 multiplier) follows a change in place all the same."""
    x, xl = _tokens(197, 192), _tokens(600, 192)
    with torch.inference_mode():
        layer, norm = _on_the_fly(192, 768), torch.nn.LayerNorm(192).cuda().half()
        layer.weight_scale = layer.weight_scale.half()
        assert layer.weight_scale.is_inference() and norm.weight.is_inference()

        def results():
            layer.fp8_operands = True
            f8 = layer(xl)
            layer.fp8_operands = False
            return layer(x), layer(x, layernorm=norm), f8

        before = results()
        layer.weight_scale.mul_(1024)
        layer.weight_center.mul_(1024)
        norm.weight.mul_(2)
        norm.bias.add_(0.5)
        after = results()
        layer, weight, bias = _on_the_fly(192, 768), norm.weight, norm.bias
        layer.weight_scale = layer.weight_scale.half() * 1024
        layer.weight_center = layer.weight_center * 1024
        norm = torch.nn.LayerNorm(192).cuda().half()
        norm.load_state_dict({"weight": weight, "bias": bias})
        assert all(torch.equal(a, b) for a, b in zip(after, results()))
        assert not any(torch.equal(a, b) for a, b in zip(after, before))


def _cut(t):
    return t[:-1].contiguous()


@pytest.mark.parametrize("fmt", ["packed", "u8", "dequant_gemm", "hip_fused", "on_the_fly", "conv"])
def test_buffers_replaced_by_unfit_ones_are_refused(cuda, fmt):
    """The kernels read what the layer's sizes say; a buffer that holds less, or lies in host memory, is refused before anything
    is launched."""
    if fmt == "conv":
        src = A.QuantConv2dPCARCQ(3, 64, 16, 16, 0, True, 4, 4, 64)
        for q in (src.act_quant, src.weight_quant):
            q.set_codebook(synth.quantile_codebook(4))
        layer, inputs = A.ARCQPackedPatchConv(src).cuda(), [synth.make_images(b, 1).cuda() for b in (1, 4)]
    else:
        layer = _on_the_fly(768, 256) if fmt == "on_the_fly" else _packed(768, 256, fmt)
        inputs = [_tokens(m, 768, dtype=torch.float32) for m in (7, 600)]
    index = fmt in ("packed", "u8")
    names = ["packed_weight_codes" if fmt != "u8" else "weight_codes_u8", "weight_center", "weight_scale", "weight_code_sum",
             "activation_codebook", "activation_thresholds", "bias_tensor" if fmt == "on_the_fly" else "bias",
             "product_table" if index else "weight_codebook"] + (["weight_dequant"] if fmt == "dequant_gemm" else [])
    for x in inputs:
        with torch.no_grad():
            want = layer(x)
            for name in names:
                good = layer._buffers[name]
                bad = [_cut(good), good.cpu()] + ([good[:, :-1].contiguous()] if good.dim() == 2 else [])
                for b in bad:
                    layer._buffers[name] = b
                    with pytest.raises(RuntimeError):
                        layer(x)
                layer._buffers[name] = good
                assert torch.equal(layer(x), want)


def _misaligned(t, by=1):
    """The same values, contiguous, `by` elements off a 16-byte boundary."""
    flat = torch.empty(t.numel() + 16, dtype=t.dtype, device=t.device)[by:by + t.numel()]
    return flat.copy_(t.reshape(-1)).view(t.shape)


@pytest.mark.parametrize("m,k,n", [(197, 768, 768), (197, 192, 768), (100, 1536, 384), (511, 1024, 4096)])
def test_layer_on_input_off_the_16_byte_boundary(cuda, m, k, n):
    layer = _on_the_fly(k, n)
    for dtype in (torch.float16, torch.float32):
        x = _tokens(m, k, dtype=dtype)
        with torch.no_grad():
            assert torch.equal(layer(_misaligned(x)), layer(x))


@pytest.mark.parametrize("m", [1, 197, 1000, 5000])
def test_hip_fused_on_input_off_the_16_byte_boundary(cuda, m):
    layer, x = _packed(768, 768, "hip_fused"), _tokens(m, 768, dtype=torch.float32)
    with torch.no_grad():
        assert torch.equal(layer(_misaligned(x)), layer(x))


@pytest.mark.parametrize("batch", [1, 8, 40])
@pytest.mark.parametrize("fp8", [False, True])
def test_block_on_input_off_the_16_byte_boundary(cuda, batch, fp8):
    from arcq_vit_amd.packed_convert import set_fp8_operands
    vit = _vit(fuse_elementwise=fp8, own_attention=fp8)
    if fp8:
        set_fp8_operands(vit)
    x = _misaligned(_tokens(batch, 197, 192))
    with torch.no_grad():
        assert torch.equal(vit.blocks(x), _interpreted(vit.blocks[0], x))


@pytest.mark.parametrize("batch", [8, 40])
def test_block_on_packed_codes_at_a_4_byte_boundary(cuda, batch):
    """The one-launch layer kernels take them (from 512 rows on, with the weight buffer lent); so does the block."""
    vit = _vit(shared_buffers=True, max_rows=batch * 197)
    block, x = vit.blocks[0], _tokens(batch, 197, 192)
    with torch.no_grad():
        for layer in (block.attn.qkv, block.mlp.fc1):
            layer.packed_weight_codes = _misaligned(layer.packed_weight_codes, 4)
        assert torch.equal(block(x), _interpreted(block, x))


def test_weight_buffer_and_layernorm_off_the_16_byte_boundary(cuda):
    layer, x = _on_the_fly(768, 768), _tokens(197, 768)
    norm = torch.nn.LayerNorm(768).cuda()
    with torch.no_grad():
        norm.weight.uniform_(0.5, 1.5)
        want, with_norm = layer(x), layer(x, layernorm=norm)
        layer._weight_buffer = torch.zeros(768 * 768 + 1, dtype=torch.float16, device=cuda)[1:]
        norm.weight = torch.nn.Parameter(_misaligned(norm.weight))
        assert torch.equal(layer(x), want) and torch.equal(layer(x, layernorm=norm), with_norm)


def test_gradients_pass_the_skip_connections(cuda):
    """d block(x) / dx of a default block is the identity (the packed layers pass no gradient), so that what stands in front of
    the blocks is trained; the same for tangents."""
    import torch.autograd.forward_ad as fw
    vit = _vit()
    x = _tokens(2, 197, 192).requires_grad_()
    y = vit.blocks(x)
    weight = torch.rand_like(x)
    (y * weight).sum().backward()
    assert torch.equal(x.grad, weight)
    with torch.no_grad():
        assert torch.equal(vit.blocks(x), y) and not vit.blocks(x).requires_grad
    images = synth.make_images(2, 1).cuda().half()
    vit(images).sum().backward()
    assert all(p.grad is not None for p in (vit.cls_token, vit.pos_embed, vit.patch_embed.proj.weight))
    with torch.no_grad(), fw.dual_level():
        dual = fw.unpack_dual(vit.blocks(fw.make_dual(x.detach(), weight)))
        assert torch.equal(dual.tangent, weight) and torch.equal(dual.primal, y)


@pytest.mark.parametrize("kind", ["on_the_fly", "hip_fused", "packed"])
def test_out_of_memory_keeps_its_type(cuda, kind):
    """A caller that halves its batch on torch.OutOfMemoryError sees that type from the extension's allocations too."""
    layer = _on_the_fly(64, 1 << 14) if kind == "on_the_fly" else _packed(64, 1 << 14, kind)
    x = _tokens(1 << 15, 64, dtype=torch.float32)                         # the output: 1 or 2 GiB
    torch.cuda.synchronize()
    torch.cuda.empty_cache()
    total = torch.cuda.get_device_properties(0).total_memory
    torch.cuda.set_per_process_memory_fraction((torch.cuda.memory_reserved() + (512 << 20)) / total)
    try:
        with torch.no_grad(), pytest.raises(torch.OutOfMemoryError):
            layer(x)
    finally:
        torch.cuda.set_per_process_memory_fraction(1.0)


@pytest.mark.parametrize("kind", ["layer", "block", "packed", "quantize"])
def test_other_threads_run_during_a_call(cuda, kind):
    """A call that has to wait (here for memory: the allocator's cached segments are too small, and giving them back waits for
    the GPU) does not hold the interpreter's lock meanwhile."""
    import threading
    import time
    x = _tokens(1 << 18, 64, dtype=torch.float32)
    if kind == "quantize":
        cb = synth.quantile_codebook(4)
        thr, cb = synth.midpoint_thresholds(cb).cuda(), cb.cuda()
        wide = torch.randn(1 << 18, 1024, device=cuda)
        call = lambda: A.quantize_activation_u8(wide, thr, cb, 4, 64)      # codes of 256 MiB
        small = lambda: A.quantize_activation_u8(wide[:64], thr, cb, 4, 64)
    elif kind == "block":
        block, tokens = _vit().blocks[0], _tokens(1500, 197, 192)          # over 1 GiB of scratch
        call, small = lambda: block(tokens), lambda: block(tokens[:1])
    else:
        layer = _on_the_fly(64, 1024) if kind == "layer" else _packed(64, 1024, kind)
        call, small = lambda: layer(x), lambda: layer(x[:64])              # outputs of 512 MiB / 1 GiB
    total = torch.cuda.get_device_properties(0).total_memory
    longest, stop = [0.0], threading.Event()

    def tick():
        last = time.perf_counter()
        while not stop.is_set():
            time.sleep(0.001)
            now = time.perf_counter()
            longest[0], last = max(longest[0], now - last), now

    with torch.no_grad():
        small()
        torch.cuda.synchronize()
        torch.cuda.empty_cache()
        used = torch.cuda.memory_reserved()
        segments = [torch.empty(100 << 20, dtype=torch.uint8, device=cuda) for _ in range(20)]
        torch.cuda.set_per_process_memory_fraction((used + (2100 << 20)) / total)
        del segments
        ticker = threading.Thread(target=tick)
        ticker.start()
        try:
            torch.cuda._sleep(500_000_000)                                 # GPU busy for some tenths of a second
            start = time.perf_counter()
            call()
            took = time.perf_counter() - start
        finally:
            stop.set()
            ticker.join()
            torch.cuda.synchronize()
            torch.cuda.set_per_process_memory_fraction(1.0)
    if took < 0.05:
        pytest.skip("the call did not have to wait")
    assert longest[0] < took / 2, (took, longest[0])


def test_one_layer_from_several_threads(cuda):
    """Threads on streams of their own call one model; each gets its own input's result."""
    import threading
    vit = _vit(own_attention=True, fuse_elementwise=True)
    inputs = [_tokens(3, 197, 192, seed=s) for s in range(4)]
    with torch.no_grad():
        want = [vit.blocks(x).clone() for x in inputs]
    torch.cuda.synchronize()
    failures = []

    def work(i):
        with torch.cuda.stream(torch.cuda.Stream()), torch.no_grad():
            for _ in range(30):
                if not torch.equal(vit.blocks(inputs[i]), want[i]):
                    failures.append(i)

    threads = [threading.Thread(target=work, args=(i,)) for i in range(len(inputs))]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert not failures


def _without_extension(monkeypatch):
    from arcq_vit_amd import _lib
    monkeypatch.setattr(_lib, "_host", _lib._NoHost)


@pytest.mark.parametrize("m,k,n,bits", [(1, 64, 64, 2), (197, 192, 768, 4), (197, 768, 3072, 3), (394, 1024, 1024, 4), (1000, 384, 1152, 4),
                                        (600, 1536, 200, 3)])
def test_layers_without_the_extension(cuda, monkeypatch, m, k, n, bits):
    """The same kernels through ctypes: the bits of the extension's calls, for every form of a layer's call."""
    layer, norm = _on_the_fly(k, n, bits), torch.nn.LayerNorm(k).cuda().half()
    following = _on_the_fly(n, 64, bits) if n % 64 == 0 else None
    layer._weight_buffer = torch.zeros(n * k, dtype=torch.float16, device=cuda)
    x, skip = _tokens(m, k), _tokens(m, n, seed=4)

    def results():
        out = [layer(x), layer(x.float()), layer(x, activation="gelu"), layer(x, residual=skip), layer(x, layernorm=norm),
               layer(x, layernorm=norm, activation="gelu", residual=skip)]
        if following is not None and layer.can_quantize_for(following, m):
            out.append(following(layer(x, layernorm=norm, activation="gelu", quantize_for=following), input_is_xhat=True))
        layer.fp8_operands = True
        out += [layer(x), layer(x, residual=skip)]
        layer.fp8_operands = False
        return out

    with torch.no_grad():
        want = results()
        _without_extension(monkeypatch)
        got = results()
    assert len(got) == len(want) and all(torch.equal(a, b) for a, b in zip(got, want))


@pytest.mark.parametrize("fused", [False, True])
@pytest.mark.parametrize("batch", [1, 5, 40])
def test_blocks_without_the_extension(cuda, monkeypatch, batch, fused):
    block, x = _vit(fuse_elementwise=fused, own_attention=fused).blocks[0], _tokens(batch, 197, 192)
    with torch.no_grad():
        want = block(x)
        _without_extension(monkeypatch)
        assert torch.equal(block(x), want)


@pytest.mark.parametrize("fmt", ["packed", "u8", "dequant_gemm", "hip_fused"])
def test_formats_without_the_extension(cuda, monkeypatch, fmt):
    layer, xs = _packed(768, 256, fmt), [_tokens(m, 768, dtype=torch.float32) for m in (7, 600)]
    with torch.no_grad():
        want = [layer(x) for x in xs]
        _without_extension(monkeypatch)
        assert all(torch.equal(layer(x), y) for x, y in zip(xs, want))


@pytest.mark.parametrize("fused,fp8", [(False, False), (True, False), (True, True)])
def test_blocks_use_the_lent_buffers(cuda, fused, fp8):
    """With `share_buffers` a forward's peak holds no second copy of what was lent; the results are those without."""
    from arcq_vit_amd.packed_convert import set_fp8_operands, share_buffers
    vit, x = _vit(fuse_elementwise=fused, own_attention=True), _tokens(32, 197, 192)
    if fp8:
        set_fp8_operands(vit)
    rows = 32 * 197

    def peak():
        torch.cuda.synchronize()
        torch.cuda.reset_peak_memory_stats()
        before = torch.cuda.memory_allocated()
        y = vit.blocks(x)
        torch.cuda.synchronize()
        return y, torch.cuda.max_memory_allocated() - before

    with torch.no_grad():
        vit.blocks(x)
        want, alone = peak()
        share_buffers(vit, rows)
        got, lent = peak()
        assert torch.equal(got, want)
        unit = rows * 192 * (1 if fp8 else 2)                             # x_hat of 192 values: one unit, fc2's: four
        assert lent <= alone - 5 * unit + (1 << 20), (alone / unit, lent / unit)
        graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(graph):
            y = vit.blocks(x)
        for _ in range(3):                                                # replays with eager work in the same buffers between
            y.zero_()
            graph.replay()
            assert torch.equal(y, want) and torch.equal(vit.blocks(x), want)
        share_buffers(vit, rows - 1)                                      # too small for fc2's x_hat: allocated again
        assert torch.equal(vit.blocks(x), want)
        for other in (torch.zeros(10, device=cuda), None):                # no fp16 buffer; none
            for layer in (vit.blocks[0].attn.qkv, vit.blocks[0].mlp.fc2):
                layer._x_hat_buffer = other
            assert torch.equal(vit.blocks(x), want)


def _kernels(call):
    from torch.profiler import ProfilerActivity, profile
    torch.cuda.synchronize()
    with profile(activities=[ProfilerActivity.CUDA]) as p:
        call()
        torch.cuda.synchronize()
    return " ".join(e.name for e in p.events())


@pytest.mark.parametrize("batch,buffers,own,layers", [(52, True, False, False), (56, True, False, True), (83, True, False, True),
                                                      (84, True, False, False), (64, False, False, False), (64, True, True, False)])
def test_default_blocks_choose_the_faster_launches(cuda, batch, buffers, own, layers):
    """A default block with lent buffers and torch's attention runs layer by layer where each layer is one launch and that is the
    faster form (10 800 to 16 384 rows), on prepared operands elsewhere; the results are the same."""
    vit = _vit(shared_buffers=buffers, max_rows=batch * 197 if buffers else 0, own_attention=own)
    block, x = vit.blocks[0], _tokens(batch, 197, 192)
    with torch.no_grad():
        one_by_one = "CUDAFunctor_add" in _kernels(lambda: block(x))      # torch's skip connections
        assert one_by_one == layers
        assert torch.equal(block(x), _interpreted(block, x))


def test_copies_made_during_capture_stay_in_the_graph(cuda):
    """A first call under capture records the conversion of its metadata and LayerNorm parameters; an eager call in front of the
    first replay makes its own."""
    x, norm = _tokens(197, 192), torch.nn.LayerNorm(192).cuda().half()
    with torch.no_grad():
        norm.weight.uniform_(0.5, 1.5)
        scale = _on_the_fly(192, 768).weight_scale.half()
        layers = [_on_the_fly(192, 768) for _ in range(2)]
        for layer in layers:
            layer.weight_scale = scale
        want = layers[0](x, layernorm=norm)
        torch.cuda.synchronize()
        graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(graph):
            y = layers[1](x, layernorm=norm)
        assert torch.equal(layers[1](x, layernorm=norm), want)
        for _ in range(3):
            y.zero_()
            graph.replay()
            assert torch.equal(layers[1](x, layernorm=norm), want) and torch.equal(y, want)
        del graph, y
        torch.cuda.empty_cache()
        assert torch.equal(layers[1](x, layernorm=norm), want)


def test_copies_are_ready_for_every_stream(cuda):
    """The stream of the first call makes the fp32 copies; a call on another stream that comes before they are made waits."""
    x = _tokens(197, 192)
    with torch.no_grad():
        norm, scale = torch.nn.LayerNorm(192).cuda().half(), _on_the_fly(192, 768).weight_scale.half()
        norm.weight.uniform_(0.5, 1.5)
        layers = [_on_the_fly(192, 768) for _ in range(2)]
        for layer in layers:
            layer.weight_scale = scale
        want = layers[0](x, layernorm=norm)
        first, second = torch.cuda.Stream(), torch.cuda.Stream()
        torch.cuda.synchronize()
        with torch.cuda.stream(first):
            torch.cuda._sleep(200_000_000)
            a = layers[1](x, layernorm=norm)
        with torch.cuda.stream(second):
            b = layers[1](x, layernorm=norm)
        torch.cuda.synchronize()
        assert torch.equal(a, want) and torch.equal(b, want)
