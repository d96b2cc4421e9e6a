"""MXFP8 GEMMs whose grids run as 128 x 128 quarter tiles only (at most two per
CU), unsplit and split over K through a workspace, at the edges of that range:
one row, one stage pair of K, a K whose pairs do not divide into the splits,
rows that leave dead 32-row groups, one more row than a quarter tile, and the
largest grid (512 quarter tiles on 256 CUs) with its neighbour of one more row
(which runs as 192 x 256 tiles).  And grids of 256 x 256 tiles, at the smallest K
of their ring, with the quarter tiles of their last partial round.
"""
import numpy as np
import pytest
import torch

from oracle import oracle as O
from qwen_image_accel import _native
from qwen_image_accel.kernels import gemm, mxfp8
from tests.helpers import bf16_randn, rel_fro

pytestmark = pytest.mark.gpu


def u8(t):
    return t.view(torch.uint8).cpu().numpy()


@pytest.mark.parametrize("m,n,k", [(1, 128, 128), (33, 384, 2176), (40, 4096, 4096), (129, 1536, 12288),
                                   (2048, 4096, 256), (2049, 4096, 256)])
def test_mxfp8_gemm_quarter_grid(dev, m, n, k):
    """Every epilogue that can split, against the oracle and the unsplit call;
    every operand layout and a strided output, bit for bit."""
    ws = _native.lib().qim_mxfp8_gemm_ws_bytes(m, n, k, _native.EPI_BIAS)
    print("[case] quarter grid", m, n, k, "workspace", ws, flush=True)
    assert (ws > 0) == (1 < m < 2048)
    g = torch.Generator().manual_seed(m + n)
    a, w = bf16_randn(g, (m, k)).to(dev), bf16_randn(g, (n, k), 0.05).to(dev)
    aq, wq = mxfp8.quantize(a), mxfp8.quantize(w)
    at, wt = mxfp8.quantize(a, tiled=True), mxfp8.quantize(w, tiled=True)
    bias = bf16_randn(g, (n,)).to(dev)
    res, gate = bf16_randn(g, (m, n)).to(dev), bf16_randn(g, (2, n)).to(dev)
    seq = (m + 1) // 2
    y32 = gemm.mx_matmul(aq, wq.values, wq.scales, dtype=torch.float32)
    rows = np.unique(np.concatenate([np.arange(min(m, 24)), np.arange(max(0, m - 24), m)]))
    ref = O.mx_gemm(u8(aq.values), u8(aq.scales), u8(wq.values), u8(wq.scales), rows=rows)
    assert rel_fro(y32.cpu().numpy()[rows], ref) < 1e-2
    # The unsplit call: fp32 sums of the same products in another order.
    u32 = torch.empty_like(y32)
    _native.call("qim_mxfp8_gemm_ex", _native.ptr(aq.values), _native.ptr(aq.scales), _native.ptr(wq.values),
                 _native.ptr(wq.scales), m, n, k, _native.EPI_NONE, _native.GEMM_OUT_F32, None, None, None, m,
                 _native.ptr(u32), n, None, _native.stream(dev))
    assert (y32 - u32).abs().max().item() <= 1e-5 * u32.abs().max().item()
    # The epilogues on the call's own fp32 sums, with the reference's rounding points.
    y = gemm.mx_matmul(aq, wq.values, wq.scales)
    assert torch.equal(y, y32.to(torch.bfloat16))
    assert torch.equal(gemm.mx_matmul(aq, wq.values, wq.scales, dtype=torch.float16), y32.to(torch.float16))
    yb = gemm.mx_matmul(aq, wq.values, wq.scales, epilogue="bias", bias=bias)
    assert torch.equal(yb, (y32 + bias.float()).to(torch.bfloat16))
    yg = gemm.mx_matmul(aq, wq.values, wq.scales, epilogue="gated_residual", gate=gate, residual=res, seq=seq)
    assert torch.equal(yg, res + gate.repeat_interleave(seq, 0)[:m] * y)
    # Operand layouts and a strided output.
    wide = torch.zeros(m, n + 8, dtype=torch.bfloat16, device=dev)
    for x, ww, tiled in ((at, wq, False), (aq, wt, True), (at, wt, True)):
        out = gemm.mx_matmul(x, ww.values, ww.scales, epilogue="gated_residual", gate=gate, residual=res, seq=seq,
                             weight_tiled=tiled, out=wide[:, :n])
        assert torch.equal(out, yg) and not wide[:, n:].any()


@pytest.mark.parametrize("m,f,k", [(1, 256, 128), (129, 512, 384), (256, 12288, 256)])
def test_swiglu_quarter_grid(dev, m, f, k):
    """The SwiGLU epilogues of quarter tiles (silu computed, not looked up):
    the unfused GEMM, swiglu and quantizer, byte for byte, gate values outside the
    SiLU estimate's range among them."""
    from qwen_image_accel.kernels.bf16 import swiglu
    print("[case] swiglu quarter grid", m, f, k, flush=True)
    g = torch.Generator().manual_seed(m + f)
    a = bf16_randn(g, (m, k))
    a[0] *= 64
    wg, wu = bf16_randn(g, (f, k), 0.2).to(dev), bf16_randn(g, (f, k), 0.2).to(dev)
    x = mxfp8.quantize(a.to(dev), tiled=True)
    q = mxfp8.quantize(gemm.interleave_swiglu(wg, wu), tiled=True)
    gq, uq = mxfp8.quantize(wg, tiled=True), mxfp8.quantize(wu, tiled=True)
    gate, up = (gemm.mx_matmul(x, w.values, w.scales, weight_tiled=True, dtype=torch.float32).to(torch.bfloat16)
                for w in (gq, uq))
    if _native.lib().qim_mxfp8_gemm_ws_bytes(m, f, k, _native.EPI_NONE):  # the fused form never splits K
        gate, up = torch.empty_like(gate), torch.empty_like(up)
        for w, o in ((gq, gate), (uq, up)):
            _native.call("qim_mxfp8_gemm_ex", _native.ptr(x.values), _native.ptr(x.scales), _native.ptr(w.values),
                         _native.ptr(w.scales), m, f, k, _native.EPI_NONE,
                         _native.GEMM_A_TILED | _native.GEMM_B_TILED, None, None, None, m, _native.ptr(o), f, None,
                         _native.stream(dev))
    want = swiglu(gate, up)
    assert torch.equal(gemm.mx_matmul(x, q.values, q.scales, epilogue="swiglu", weight_tiled=True), want)
    for tiled in (False, True):
        got = gemm.mx_matmul(x, q.values, q.scales, epilogue="swiglu_quant", weight_tiled=True, out_tiled=tiled)
        ref = mxfp8.quantize(want, tiled=tiled)
        assert np.array_equal(u8(got.values), u8(ref.values)) and np.array_equal(u8(got.scales), u8(ref.scales))


# A grid of quarter tiles split over K, and whole tiles whose tail is split (272 tiles).
@pytest.mark.parametrize("m,n,k", [(40, 4096, 4096), (4352, 4096, 1024)])
def test_split_bias_at_any_element(dev, m, n, k):
    """The bias of a split grid may be a slice that starts at any element."""
    assert _native.lib().qim_mxfp8_gemm_ws_bytes(m, n, k, _native.EPI_BIAS) > 0
    print("[case] split, bias at any element", m, n, k, flush=True)
    g = torch.Generator().manual_seed(m + n)
    a, w = bf16_randn(g, (m, k)).to(dev), bf16_randn(g, (n, k), 0.05).to(dev)
    aq, wq = mxfp8.quantize(a), mxfp8.quantize(w)
    buf = bf16_randn(g, (n + 8,)).to(dev)
    y32 = gemm.mx_matmul(aq, wq.values, wq.scales, dtype=torch.float32)
    for at in (0, 1, 2, 5, 7):
        bias = buf[at:at + n]
        y = gemm.mx_matmul(aq, wq.values, wq.scales, epilogue="bias", bias=bias)
        assert torch.equal(y, (y32 + bias.float()).to(torch.bfloat16)), at


@pytest.mark.parametrize("k", [128, 384])
def test_mxfp8_gemm_whole_tile_grid(dev, k):
    """4352 x 4096: 256 whole tiles, then 64 quarter tiles (split over K at K =
    384), at one and three stage pairs, in every output format, against the
    oracle and the same rows as unsplit quarter tiles (bit for bit, but for the
    rows of the split tail)."""
    m, n = 4352, 4096
    ws = _native.lib().qim_mxfp8_gemm_ws_bytes(m, n, k, _native.EPI_NONE)
    print("[case] whole tiles", m, n, k, "workspace", ws, flush=True)
    assert (ws > 0) == (k > 128)
    g = torch.Generator().manual_seed(k)
    a, w, bias = bf16_randn(g, (m, k)).to(dev), bf16_randn(g, (n, k), 0.05).to(dev), bf16_randn(g, (n,)).to(dev)
    aq, wq = mxfp8.quantize(a), mxfp8.quantize(w)
    at, wt = mxfp8.quantize(a, tiled=True), mxfp8.quantize(w, tiled=True)

    def unsplit(x, out, flag):
        _native.call("qim_mxfp8_gemm_ex", _native.ptr(x.values), _native.ptr(x.scales), _native.ptr(wq.values),
                     _native.ptr(wq.scales), x.rows, n, k, _native.EPI_NONE, flag, None, None, None, x.rows,
                     _native.ptr(out), n, None, _native.stream(dev))
        return out
    u32 = unsplit(aq, torch.empty(m, n, device=dev, dtype=torch.float32), _native.GEMM_OUT_F32)
    rows = np.unique(np.concatenate([np.arange(24), np.arange(m - 24, m), np.arange(0, m, 193)]))
    ref = O.mx_gemm(u8(aq.values), u8(aq.scales), u8(wq.values), u8(wq.scales), rows=rows)
    assert rel_fro(u32.cpu().numpy()[rows], ref) < 1e-2
    for r0 in range(0, m, 512):
        x = mxfp8.quantize(a[r0:r0 + 512])
        part = unsplit(x, torch.empty(x.rows, n, device=dev, dtype=torch.float32), _native.GEMM_OUT_F32)
        assert torch.equal(part, u32[r0:r0 + 512]), r0
    assert torch.equal(unsplit(aq, torch.empty(m, n, device=dev, dtype=torch.float16), _native.GEMM_OUT_F16),
                       u32.to(torch.float16))
    assert torch.equal(unsplit(aq, torch.empty(m, n, device=dev, dtype=torch.bfloat16), 0), u32.to(torch.bfloat16))
    # Through the workspace (the tail's rows: fp32 sums of the same products in another order).
    y32 = gemm.mx_matmul(aq, wq.values, wq.scales, dtype=torch.float32)
    assert (y32 - u32).abs().max().item() <= 1e-5 * u32.abs().max().item()
    assert torch.equal(gemm.mx_matmul(aq, wq.values, wq.scales, dtype=torch.float16), y32.to(torch.float16))
    for x, ww, tiled in ((aq, wq, False), (at, wq, False), (aq, wt, True), (at, wt, True)):
        y = gemm.mx_matmul(x, ww.values, ww.scales, epilogue="bias", bias=bias, weight_tiled=tiled)
        assert torch.equal(y, (y32 + bias.float()).to(torch.bfloat16))


def test_swiglu_whole_tile_grid(dev):
    """The SwiGLU epilogues of whole tiles (silu looked up) and of the tail's
    quarter tiles, with gate values outside the table's range and zeros, against
    the unfused GEMM, swiglu and quantizer, byte for byte."""
    from qwen_image_accel.kernels.bf16 import swiglu
    m, f, k = 4352, 2048, 128
    print("[case] swiglu whole tiles", m, f, k, flush=True)
    g = torch.Generator().manual_seed(m)
    a = bf16_randn(g, (m, k))
    a[::7] *= 64
    wg, wu = bf16_randn(g, (f, k), 0.2), bf16_randn(g, (f, k), 0.2).to(dev)
    wg[::5] = 0
    wg = wg.to(dev)
    x = mxfp8.quantize(a.to(dev), tiled=True)
    q = mxfp8.quantize(gemm.interleave_swiglu(wg, wu), tiled=True)
    assert _native.lib().qim_mxfp8_gemm_ws_bytes(m, f, k, _native.EPI_NONE) == 0  # the sums below are unsplit
    gate, up = (gemm.mx_matmul(x, w.values, w.scales, weight_tiled=True)
                for w in (mxfp8.quantize(wg, tiled=True), mxfp8.quantize(wu, tiled=True)))
    assert gate.abs().max() > 100 and (gate[:, ::5] == 0).all() and (up[:, ::5] != 0).any()
    want = swiglu(gate, up)
    assert torch.equal(gemm.mx_matmul(x, q.values, q.scales, epilogue="swiglu", weight_tiled=True), want)
    for tiled in (False, True):
        got = gemm.mx_matmul(x, q.values, q.scales, epilogue="swiglu_quant", weight_tiled=True, out_tiled=tiled)
        ref = mxfp8.quantize(want, tiled=tiled)
        assert np.array_equal(u8(got.values), u8(ref.values)) and np.array_equal(u8(got.scales), u8(ref.scales))
