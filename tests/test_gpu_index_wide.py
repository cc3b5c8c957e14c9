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


# From 512 tiles of 32 x 32 on the packed format runs on the matrix units (sums of the table's entries as integers): ragged rows
# and outputs, one and many groups, and tables that it takes (also with zeros, and all of them zero, and with single-bit entries)
# and leaves to the fp64 loops (entries too far apart, a subnormal, an infinity, a NaN).
@pytest.mark.parametrize("m,n,k", [(545, 1000, 128), (4100, 127, 64), (33, 8225, 320)])
@pytest.mark.parametrize("bits", [4, 3, 2])
@pytest.mark.parametrize("kind", ["outer", "arbitrary", "zeros", "all_zero", "powers", "far_apart", "subnormal", "all_subnormal", "infinity", "nan"])
def test_linear_index_on_the_matrix_units(cuda, oracle, m, n, k, bits, kind):
    levels = 1 << bits
    cb = synth.quantile_codebook(bits)
    table = (1.1 * cb.view(-1, 1) * cb.view(1, -1)).contiguous()
    if kind == "arbitrary":
        table = table + 0.25 * torch.arange(table.numel()).view_as(table) / table.numel()
    elif kind == "zeros":
        table[1] = 0.0
        table[:, 2] = -0.0
    elif kind == "all_zero":
        table = torch.zeros_like(table)
    elif kind == "powers":
        table = torch.sign(table) * 2.0 ** (torch.arange(table.numel()).view_as(table) % 15 - 80)
    elif kind == "all_subnormal":
        table = table * 1.0e-40
    elif kind != "outer":
        table[1, 1] = {"far_apart": 1.0e-6, "subnormal": 1.0e-40, "infinity": float("inf"), "nan": float("nan")}[kind]
    rng = np.random.default_rng(7)
    g = k // 64
    xq = oracle.pack_codes_np(rng.integers(0, levels, (m, k)).astype(np.uint8), bits)
    wq = oracle.pack_codes_np(rng.integers(0, levels, (n, k)).astype(np.uint8), bits)
    meta = [rng.standard_normal((r, g)).astype(np.float32) for r in (m, m, m, n, n, n)]
    bias = synth.make_bias(n, 5)
    want = oracle.linear_forward_packed_c(xq, *meta[:3], wq, *meta[3:], table.numpy(), bias.numpy(), bits, 64, k, n)
    d = lambda t: (torch.from_numpy(t) if isinstance(t, np.ndarray) else t).to(cuda).contiguous()
    t = [d(v) for v in (xq, *meta[:3], wq, *meta[3:], table, cb, cb, bias)]
    y = torch.full((m, n), float("nan"), device=cuda)
    a = _lib.LinearIndexArgs(*[v.data_ptr() for v in t], y.data_ptr(), m, n, k, bits, 64, levels, 0)
    _lib.check(_lib.load().arcq_linear_index(ctypes.byref(a), torch.cuda.current_stream().cuda_stream))
    assert np.array_equal(y.cpu().numpy(), want, equal_nan=True)


# Few rows of very many outputs, on both sides of the rule that leaves tiles which are mostly padding to the wide kernel: waves of the
# matrix-unit launch past the last row leave early.
@pytest.mark.parametrize("m,n,k", [(1, 16416, 64), (16, 16416, 128), (17, 16416, 64), (33, 16390, 128), (64, 8225, 192)])
@pytest.mark.parametrize("bits", [4, 2])
def test_few_rows_of_many_outputs(cuda, m, n, k, bits):
    cb = synth.quantile_codebook(bits)
    a, t = _call(cuda, m, n, k, bits, (cb.view(-1, 1) * cb.view(1, -1)).contiguous(), cb, cb)
    assert torch.equal(*_both_entry_points(cuda, a, t, m, n, k, bits))


# 8 x 768 -> 16416 against its two halves of outputs, which are too small for the matrix units: 28 us against 35 to 40, on the matrix
# units it took 80 to 90.
@pytest.mark.parametrize("bits", [4, 3])
def test_few_rows_of_many_outputs_cost_what_their_halves_do(cuda, bits):
    cb = synth.quantile_codebook(bits)
    table = (cb.view(-1, 1) * cb.view(1, -1)).contiguous()
    stream = torch.cuda.current_stream().cuda_stream
    whole, kept = _call(cuda, 8, 16416, 768, bits, table, cb, cb)
    halves = [_call(cuda, 8, 8208, 768, bits, table, cb, cb) for _ in range(2)]
    assert _microseconds([whole], stream) < 1.5 * _microseconds([h for h, _ in halves], stream)


def _microseconds(calls, stream):
    """The shortest of ten runs of ``calls``, five times over each."""
    best = float("inf")
    for _ in range(10):
        begin, end = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
        begin.record()
        for _ in range(5):
            for a in calls:
                _lib.check(_lib.load().arcq_linear_index(ctypes.byref(a), stream))
        end.record()
        torch.cuda.synchronize()
        best = min(best, begin.elapsed_time(end) * 200.0)
    return best


def _call(cuda, m, n, k, bits, table, a_cb, w_cb):
    g = k // 64
    t = [torch.randint(0, 256, (m, k * bits // 8), dtype=torch.uint8, device=cuda), *(torch.randn(m, g, device=cuda) for _ in range(3)),
         torch.randint(0, 256, (n, k * bits // 8), dtype=torch.uint8, device=cuda), *(torch.randn(n, g, device=cuda) for _ in range(3)),
         table.to(cuda), a_cb.to(cuda), w_cb.to(cuda), torch.randn(n, device=cuda), torch.empty(m, n, device=cuda)]
    return _lib.LinearIndexArgs(*[v.data_ptr() for v in t], m, n, k, bits, 64, 1 << bits, 0), t


def _both_entry_points(cuda, a, t, m, n, k, bits):
    """The outputs with the codebooks at hand, and of the entry point that has only the table."""
    stream = torch.cuda.current_stream().cuda_stream
    y = torch.full_like(t[-1], float("nan"))
    xq, xc, xs, xcs, wq, wc, ws, wcs, table, _, _, bias, _ = (v.data_ptr() for v in t)
    _lib.check(_lib.load().arcq_linear_index(ctypes.byref(a), stream))
    _lib.check(_lib.load().arcq_linear_forward_packed(xq, xc, xs, xcs, wq, wc, ws, wcs, table, bias, y.data_ptr(), m, n, k, bits, 64, 1 << bits, stream))
    return t[-1], y


def _codebook_with_a_level_near_zero(bits):
    cb = synth.quantile_codebook(bits).clone()
    cb[(1 << bits) // 2] = 0.001234567
    return cb, (cb.view(-1, 1) * cb.view(1, -1)).contiguous()


# Such a table runs on the loops, dealt to the workgroups that are resident at once and, of four waves, to those behind them a tile
# each (256 compute units; three and four waves; (5721, 330, 192) has four because of the matrix units): the same bits as the entry
# point without codebooks gives.
@pytest.mark.parametrize("m,n,k", [(1000, 550, 192), (4100, 775, 192), (4100, 2400, 192), (4100, 775, 256), (4100, 2331, 256),
                                   (5721, 330, 192)])
@pytest.mark.parametrize("outer", [True, False])
def test_tables_that_do_not_qualify_in_larger_launches(cuda, m, n, k, outer):
    cb, table = _codebook_with_a_level_near_zero(4)
    if not outer:
        table[1, 1] = 1.0e-6
    a, t = _call(cuda, m, n, k, 4, table, cb, cb)
    assert torch.equal(*_both_entry_points(cuda, a, t, m, n, k, 4))


# 21 groups would be three waves' work in the loops of other tables; on the matrix units three-wave workgroups put more waves on the
# busiest SIMD than four-wave ones here (81 us against 63), and the time is to be 21 / 20 of that of 20 groups.
@pytest.mark.parametrize("bits", [4, 2])
def test_number_of_groups_does_not_unbalance_the_matrix_units(cuda, bits):
    cb = synth.quantile_codebook(bits)
    table = (cb.view(-1, 1) * cb.view(1, -1)).contiguous()
    stream = torch.cuda.current_stream().cuda_stream
    (a, kept), (b, also_kept) = (_call(cuda, 5721, 352, 64 * g, bits, table, cb, cb) for g in (21, 20))
    assert _microseconds([a], stream) < 1.15 * _microseconds([b], stream)


# A fitted codebook with a level near zero (43 bits between the table's entries) is computed with the fp64 loops whatever the size
# of the call: 512 rows cost no more than twice what two calls of 256 rows do, which are too small for the matrix units (29 us,
# 37 both; in the shape of the matrix-unit launch the loops took 100).
@pytest.mark.parametrize("bits", [4, 3, 2])
def test_tables_that_do_not_qualify_fill_the_chip(cuda, bits):
    cb, table = _codebook_with_a_level_near_zero(bits)
    stream = torch.cuda.current_stream().cuda_stream
    whole, kept = _call(cuda, 512, 1024, 384, bits, table, cb, cb)
    halves = [_call(cuda, 256, 1024, 384, bits, table, cb, cb) for _ in range(2)]
    assert _microseconds([whole], stream) < 2 * _microseconds([h for h, _ in halves], stream)
