"""A quantizer's lookup tables as each kernel builds them: thresholds that share a bucket, repeat, lie outside the table or are out of
order (a search over all of them finds the code then: the first threshold that is not below the value), at every bucket width."""
import numpy as np
import pytest
import torch

from arcq_vit_amd import _lib, ops, synth
from test_gpu_patch_conv import _blocked
from test_gpu_prepared import _linear, _prepare, _stream

pytestmark = pytest.mark.gpu
INF = float("inf")


def _tables(bits):
    """name -> thresholds"""
    n = (1 << bits) - 1
    spread = lambda gap: (torch.arange(n) - (n - 1) / 2) * gap
    plain = synth.midpoint_thresholds(synth.quantile_codebook(bits))
    t = {f"gap {g}": spread(g) for g in (0.4, 0.2, 0.1, 0.05, 0.02)}      # 64, 128, 256 and 512 buckets; two in a bucket
    t["at the ends"] = torch.cat([torch.tensor([-8.0]), plain[1:-1], torch.tensor([7.99])]) if n > 1 else plain
    t["repeated"], t["out of order"], t["outside"], t["infinite"] = (plain.clone() for _ in range(4))
    t["repeated"][1] = t["repeated"][0]
    t["out of order"][[0, 2]] = t["out of order"][[2, 0]]
    t["outside"][-1] = 8.0
    t["infinite"][0], t["infinite"][-1] = -INF, INF
    return {k: v.float().contiguous() for k, v in t.items()}


@pytest.mark.parametrize("bits", [2, 3, 4])
def test_tables(cuda, oracle, bits):
    cb = synth.quantile_codebook(bits)
    stage1 = lambda x, thr: oracle.act_quant_c(x.float().numpy(), thr, cb, bits, 64)["x_hat"].astype(np.float16)
    f32 = synth.make_activation(70, 192, 3)
    f16 = {m: synth.make_activation(m, k, 5).half() for m, k in ((197, 384), (20000, 64))}     # a wave that builds; more tiles than that
    bias = synth.make_activation(1, 64, 7).half()
    qkv = synth.make_activation(2 * 33, 3 * 2 * 64, 9).half()
    att = ops.attention_fwd(qkv.to(cuda).view(2, 33, -1), 2).reshape(66, 128).cpu()
    img = synth.make_activation(2 * 3 * 32, 32, 11).view(2, 3, 32, 32)
    pix = img.permute(0, 2, 3, 1).reshape(-1, 3).contiguous()
    zeros = torch.zeros(700 * 64, dtype=torch.float16, device=cuda)
    for name, thr in _tables(bits).items():
        t, c = thr.to(cuda), cb.to(cuda)

        def same(got, want, what):
            assert np.array_equal(got.reshape(-1).cpu().numpy().view(np.uint16), want.reshape(-1).view(np.uint16)), (name, what)

        same(ops.quantize_activation_dequant(f32.to(cuda), t, c, bits, 64).half(), stage1(f32, thr), "row-major")
        for m, x in f16.items():
            same(_prepare(x.to(cuda), t, c, bits)[0], _blocked(stage1(x, thr)), m)
        for m in (33, 700):                                                                  # behind a product: split and tile kernel
            got = _linear(zeros, zeros, bias.to(cuda).float().reshape(-1), m, 64, 64, nq=(t, c), bits=bits)
            same(got, _blocked(stage1(bias.expand(m, 64).contiguous(), thr)), ("product", m))
        got = torch.empty(66 * 128, dtype=torch.float16, device=cuda)
        _lib.check(_lib.load().arcq_attention_quant_fwd(qkv.to(cuda).data_ptr(), t.data_ptr(), c.data_ptr(), bits, got.data_ptr(), 2, 33, 2,
                                                        64, 0.125, _stream()))
        same(got, _blocked(stage1(att, thr)), "attention")
        rows = oracle.act_quant_c(pix.numpy(), thr, cb, bits, 3)["x_hat"].astype(np.float16)
        rows = rows.reshape(2, 2, 16, 2, 16, 3).transpose(0, 1, 3, 5, 2, 4).reshape(8, 768)
        same(ops.quantize_patches(img.to(cuda), t, c, bits), rows, "patches")


# eight, four and two lanes a group: the fewest and the most groups of each, ragged tiles, both sides of two tiles per compute unit
@pytest.mark.parametrize("m,k", [(1, 64), (5, 512), (197, 384), (2049, 192), (2057, 320), (3, 576), (33, 1024), (1700, 640), (5, 1088),
                                 (21, 2048), (16390, 64), (6304, 384)])
@pytest.mark.parametrize("dtype", [torch.float16, torch.float32])
def test_lanes_per_group_behind_a_layernorm(cuda, oracle, m, k, dtype):
    cb = synth.quantile_codebook(4)
    thr = synth.midpoint_thresholds(cb)
    x = (synth.make_activation(m, k, 21) * 1.7 + 0.3).to(dtype)
    g, b = torch.linspace(0.5, 1.5, k), torch.linspace(-0.2, 0.2, k)
    ln = oracle.layernorm_rows_np(x.float().numpy(), g.numpy(), b.numpy(), 1e-6, out_f16=dtype == torch.float16)
    for t in (thr, thr[torch.randperm(15, generator=torch.Generator().manual_seed(m))].contiguous()):      # buckets; a search over the thresholds
        want = oracle.act_quant_c(ln, t, cb, 4, 64)["x_hat"].astype(np.float16)
        got = _prepare(x.to(cuda), t.to(cuda), cb.to(cuda), 4, (g.to(cuda), b.to(cuda), 1e-6))[0]
        assert np.array_equal(got.cpu().numpy().view(np.uint16), _blocked(want).view(np.uint16))


# stage 1 alone: a piece per lane, a tile per wave, walking waves; ragged row tiles, infinities and NaN
@pytest.mark.parametrize("m,k", [(1, 64), (7, 192), (197, 384), (2049, 960), (4097, 512), (6304, 384), (6309, 768), (20011, 384)])
@pytest.mark.parametrize("bits,dtype", [(4, torch.float16), (3, torch.float32), (2, torch.float16)])
def test_stage_1_alone(cuda, oracle, m, k, bits, dtype):
    cb = synth.quantile_codebook(bits)
    thr = synth.midpoint_thresholds(cb)
    x = synth.make_activation(m, k, 23).to(dtype)
    x[m - 1, :4] = torch.tensor([1.0, INF, -INF, float("nan")], dtype=dtype)
    x[m // 2, k - 64:] = 0.25
    x[m // 3] *= 6e-5 if dtype == torch.float16 else 1e-30
    for t in (thr, torch.cat([thr[1:], thr[:1]])):
        with np.errstate(all="ignore"):
            want = _blocked(oracle.act_quant_c(x.float().numpy(), t, cb, bits, 64)["x_hat"].astype(np.float16))
        got = _prepare(x.to(cuda), t.contiguous().to(cuda), cb.to(cuda), bits)[0].cpu().numpy()
        nan = np.isnan(want)
        assert np.array_equal(np.isnan(got), nan) and np.array_equal(got.view(np.uint16)[~nan], want.view(np.uint16)[~nan])


# thresholds in any order with NaN and infinities among them: the search stops at the first one that is not below the value
@pytest.mark.parametrize("bits", [2, 3, 4])
@pytest.mark.parametrize("dtype", [torch.float32, torch.float16])
def test_codes_of_thresholds_in_any_order(cuda, oracle, bits, dtype):
    rng = np.random.default_rng(bits)
    cb = synth.quantile_codebook(bits)
    x = synth.make_activation(301, 192, 41).to(dtype)
    x[7], x[8, :3] = 0.0, torch.tensor([float("nan"), INF, -INF], dtype=dtype)
    for case in range(24):
        thr = np.sort(rng.normal(size=(1 << bits) - 1)).astype(np.float32)
        if case % 3:
            thr = rng.permutation(thr)
        if case % 2:
            thr[rng.integers(thr.size)] = rng.choice(np.float32([np.nan, np.inf, -np.inf, -0.0, 1e-42]))
        thr[rng.integers(thr.size)] = thr[0]
        t = torch.from_numpy(thr)
        with np.errstate(all="ignore"):
            want = oracle.act_quant_c(x.float().numpy(), t, cb, bits, 64)
        packed, _, center, _, total = ops._act_quant(x.to(cuda), t.to(cuda), cb.to(cuda), bits, 64, want_packed=True, want_meta=True, strict_f32=False)
        codes = ops._act_quant(x.to(cuda), t.to(cuda), cb.to(cuda), bits, 64, want_u8=True, strict_f32=False)[1]
        assert np.array_equal(packed.cpu().numpy(), want["packed"]), (case, thr)
        assert np.array_equal(codes.cpu().numpy(), want["codes"]), (case, thr)
        assert np.array_equal(total.cpu().numpy(), want["code_sum"]) and np.array_equal(center.cpu().numpy(), want["center"], equal_nan=True)


# A fitted codebook may repeat a level.  That takes 1.4 times as long as one whose thresholds the buckets hold (every threshold in turn:
# 3 times).
def test_repeated_thresholds_cost_little(cuda):
    cb = synth.quantile_codebook(4)
    thr = synth.midpoint_thresholds(cb)
    x, cb = torch.randn(50432, 1024, device=cuda), cb.to(cuda)

    def microseconds(t):
        best = INF
        for _ in range(8):
            begin, end = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
            begin.record()
            for _ in range(5):
                ops.quantize_activation(x, t, cb, 4, 64)
            end.record()
            torch.cuda.synchronize()
            best = min(best, begin.elapsed_time(end) * 200.0)
        return best

    repeated = thr.clone()
    repeated[1] = repeated[0]
    assert microseconds(repeated.to(cuda)) < 2 * microseconds(thr.to(cuda))
