"""MXFP8 GEMMs that run as 192 x 256 tiles (grids whose 256 x 256 tiles are less
than one round of the CUs and whose 192-row tiles still fit one): the smallest
and the largest grid, one stage pair of K, a last tile with fewer than 64 rows, tiles
that start inside a scale chunk and across the last (128-row) super-block of the
tiled layout, against the oracle and against the same rows computed as quarter
tiles (the same products added in the same order: bit for bit).
"""
import numpy as np
import pytest
import torch

from oracle import oracle as O
from qwen_image_accel import _native
from qwen_image_accel.kernels import attention, gemm, mxfp8
from tests.helpers import bf16_randn, rel_fro

pytestmark = pytest.mark.gpu


def u8(t):
    return t.view(torch.uint8).cpu().numpy()


@pytest.mark.parametrize("m,n,k", [(2049, 4096, 128), (2381, 4096, 384), (3072, 4096, 256), (1280, 7680, 640)])
def test_mxfp8_gemm_192_row_tiles(dev, m, n, k):
    print("[case] 192-row tiles", m, n, k, flush=True)
    g = torch.Generator().manual_seed(m + n)
    a, w = bf16_randn(g, (m, k)).to(dev), bf16_randn(g, (n, k), 0.05).to(dev)
    aq, wq = mxfp8.quantize(a), mxfp8.quantize(w)
    at, wt = mxfp8.quantize(a, tiled=True), mxfp8.quantize(w, tiled=True)
    bias = bf16_randn(g, (n,)).to(dev)
    res, gate = bf16_randn(g, (m, n)).to(dev), bf16_randn(g, (2, n)).to(dev)
    seq = (m + 1) // 2
    y32 = gemm.mx_matmul(aq, wq.values, wq.scales, dtype=torch.float32)
    rows = np.unique(np.concatenate([np.arange(m - 24, m), np.arange(0, m, 97), np.arange(180, 200)]))
    ref = O.mx_gemm(u8(aq.values), u8(aq.scales), u8(wq.values), u8(wq.scales), rows=rows)
    assert rel_fro(y32.cpu().numpy()[rows], ref) < 1e-2
    for r0 in range(0, m, 512):  # a few rows at a time: unsplit quarter tiles
        x = mxfp8.quantize(a[r0:r0 + 512])
        part = torch.empty(x.rows, n, device=dev, dtype=torch.float32)
        _native.call("qim_mxfp8_gemm_ex", _native.ptr(x.values), _native.ptr(x.scales), _native.ptr(wq.values),
                     _native.ptr(wq.scales), x.rows, n, k, _native.EPI_NONE, _native.GEMM_OUT_F32, None, None, None,
                     x.rows, _native.ptr(part), n, None, _native.stream(dev))
        assert torch.equal(part, y32[r0:r0 + 512]), r0
    y = gemm.mx_matmul(aq, wq.values, wq.scales)
    assert torch.equal(y, y32.to(torch.bfloat16))
    assert torch.equal(gemm.mx_matmul(aq, wq.values, wq.scales, dtype=torch.float16), y32.to(torch.float16))
    yb = gemm.mx_matmul(aq, wq.values, wq.scales, epilogue="bias", bias=bias)
    assert torch.equal(yb, (y32 + bias.float()).to(torch.bfloat16))
    yg = gemm.mx_matmul(aq, wq.values, wq.scales, epilogue="gated_residual", gate=gate, residual=res, seq=seq)
    assert torch.equal(yg, res + gate.repeat_interleave(seq, 0)[:m] * y)
    wide = torch.zeros(m, n + 8, dtype=torch.bfloat16, device=dev)
    for x, ww, tiled in ((at, wq, False), (aq, wt, True), (at, wt, True)):
        out = gemm.mx_matmul(x, ww.values, ww.scales, epilogue="gated_residual", gate=gate, residual=res, seq=seq,
                             weight_tiled=tiled, out=wide[:, :n])
        assert torch.equal(out, yg) and not wide[:, n:].any()


# 1280 x 24 heads: 180 whole tiles, 252 of 192 rows; 1408 x 20 heads: two
# batches, the second's first row inside a tile, and a last tile of 64 rows.
@pytest.mark.parametrize("m,heads,k,seq", [(1280, 24, 256, 1280), (1408, 20, 384, 704)])
def test_qkv_gemm_192_row_tiles(dev, m, heads, k, seq):
    """The QK-norm + RoPE epilogue (a head's columns in two waves) against the
    unfused pass on the plain product, and its V^T form against the V columns."""
    print("[case] qkv 192-row tiles", m, heads, k, seq, flush=True)
    g = torch.Generator().manual_seed(m + heads)
    d, b = heads * 128, m // seq
    a, w = bf16_randn(g, (m, k)).to(dev), bf16_randn(g, (3 * d, k), 0.05).to(dev)
    wq, wk = ((torch.rand(128, generator=g) * 0.4 + 0.8).to(torch.bfloat16).to(dev) for _ in range(2))
    ang = torch.rand(seq, 64, generator=g, dtype=torch.float64) * 6.283185307179586
    freqs = torch.polar(torch.ones_like(ang), ang).to(torch.complex64).to(dev)
    x, w8 = mxfp8.quantize(a, tiled=True), mxfp8.quantize(w, tiled=True)
    fused = gemm.mx_matmul_qk_norm_rope(x, w8.values, w8.scales, wq, wk, freqs, heads, seq, weight_tiled=True)
    plain = gemm.mx_matmul(x, w8.values, w8.scales, weight_tiled=True)
    q, kk, v = plain.view(b, seq, 3, heads, 128).unbind(2)
    oq, ok = attention.qk_norm_rope(q, kk, wq, wk, freqs, 1e-6, 1e-6)
    fq, fk, fv = fused.view(b, seq, 3, heads, 128).unbind(2)
    assert torch.equal(fq, oq) and torch.equal(fk, ok) and torch.equal(fv, v)
    ws = attention.workspace(b, seq, seq, heads, dev)
    out = torch.empty_like(fused)
    gemm.mx_matmul_qk_norm_rope(x, w8.values, w8.scales, wq, wk, freqs, heads, seq, weight_tiled=True, out=out,
                                vt=ws)
    assert torch.equal(out[:, :2 * d], fused[:, :2 * d])
    # The tiles: (d, 64 keys) per key block; 16-byte chunk c of row d at chunk c ^ ((d >> 1) & 7), a
    # chunk holding keys 16 (c / 2) + 4 (c % 2) + {0..3, 8..11}.
    nkb = seq // 64
    tiles = ws.view(torch.uint8)[:b * heads * nkb * 16384].view(torch.bfloat16).view(b, heads, nkb, 128, 8, 8)
    c = torch.arange(8, device=dev)
    perm = c[None, :] ^ ((torch.arange(128, device=dev)[:, None] >> 1) & 7)
    chunks = tiles.gather(4, perm.view(1, 1, 1, 128, 8, 1).expand_as(tiles))
    key = (16 * (c // 2) + 4 * (c % 2))[:, None] + torch.tensor([0, 1, 2, 3, 8, 9, 10, 11], device=dev)
    want = fv.reshape(b, nkb, 64, heads, 128).permute(0, 3, 1, 4, 2)[..., key]
    assert torch.equal(chunks, want)
