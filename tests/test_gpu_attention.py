"""The attention core (qim_attention) against softmax(Q K^T * scale) V in
float32 on the CPU, on the same bf16 inputs.

Bar: the kernel rounds P to bf16 for the P V product and writes bf16, so the
output is held to rel-Frobenius <= 1e-2 and a max-abs error of 2 % of the
output's largest magnitude, like the GEMM.  Shapes cover ragged query and key
counts (the last 256-query and 64-key blocks partial), two batches with a
cached prefix (T = P + S), Q/K/V as strided views into one fused QKV output,
and large logits (the running-max subtraction).
"""
import pytest
import torch

from qwen_image_accel.kernels import attention, mxfp8
from tests.helpers import bf16_randn, rel_fro

pytestmark = pytest.mark.gpu


def say(*a):
    print("[case]", *a, flush=True)


def reference(q, k, v, scale):
    """(B, S, H, D) bf16 -> float32 softmax attention, computed on the CPU."""
    qf, kf, vf = (x.float().cpu().permute(0, 2, 1, 3) for x in (q, k, v))  # (B, H, N, D)
    w = torch.softmax(torch.matmul(qf, kf.transpose(-1, -2).contiguous()) * scale, dim=-1)
    return torch.matmul(w, vf).permute(0, 2, 1, 3)


def check(out, ref):
    got = out.float().cpu()
    err = rel_fro(got.numpy(), ref.numpy())
    mx = (got - ref).abs().max().item()
    assert err < 1e-2, err
    assert mx < 0.02 * ref.abs().max().item(), mx


# (1, 64, 1000, 1), (1, 256, 2000, 4) and (2, 520, 1500, 3) run split over key
# ranges (2, 4 and 3 chunks, the last one ragged) and merged.
@pytest.mark.parametrize("b,s,t,h,mag", [(1, 300, 300, 2, 1.0), (2, 256, 333, 3, 1.0), (1, 64, 1000, 1, 1.0),
                                         (1, 520, 520, 2, 8.0), (1, 256, 2000, 4, 1.0), (2, 520, 1500, 3, 4.0)])
def test_attention_packed(dev, b, s, t, h, mag):
    say("attention", b, s, t, h, mag)
    g = torch.Generator().manual_seed(b * 1000 + s + t + h)
    q = (bf16_randn(g, (b, s, h, 128)) * mag).to(torch.bfloat16).to(dev)
    k = bf16_randn(g, (b, t, h, 128)).to(dev)
    v = bf16_randn(g, (b, t, h, 128)).to(dev)
    scale = 128 ** -0.5
    out = attention.attention(q, k, v)
    torch.cuda.synchronize()
    check(out, reference(q, k, v, scale))


@pytest.mark.parametrize("b", [1, 2])
def test_attention_block_shape_with_split_tail(dev, b):
    """The 1024^2 block's shape (S = T = 4352, 24 heads), as views of a fused
    QKV output.  One image: 408 work items on 256 CUs, one whole round and the
    last 152 items split into 3 key chunks; two images: 816 items, three whole
    rounds and the last 48 items split into 5 chunks.  Checked on heads 0, 11
    and 23 (every query of every image)."""
    s, h = 4352, 24
    say("attention block shape", b, s, h)
    g = torch.Generator().manual_seed(4352)
    qkv = bf16_randn(g, (b, s, 3 * h * 128)).to(dev)
    q, k, v = (qkv[:, :, i * h * 128:(i + 1) * h * 128].unflatten(-1, (h, 128)) for i in range(3))
    out = attention.attention(q, k, v)
    torch.cuda.synchronize()
    for hh in (0, 11, 23):
        sl = slice(hh, hh + 1)
        check(out[:, :, sl], reference(q[:, :, sl], k[:, :, sl], v[:, :, sl], 128 ** -0.5))


def test_attention_on_fused_qkv_views(dev):
    """Q, K, V as column blocks of one (B, S, 3HD) projection (token stride 3HD)."""
    b, s, h = 1, 384, 4
    say("attention qkv views", b, s, h)
    g = torch.Generator().manual_seed(5)
    qkv = bf16_randn(g, (b, s, 3 * h * 128)).to(dev)
    q, k, v = (qkv[:, :, i * h * 128:(i + 1) * h * 128].unflatten(-1, (h, 128)) for i in range(3))
    out = attention.attention(q, k, v, scale=0.1)
    torch.cuda.synchronize()
    check(out, reference(q, k, v, 0.1))


# 256 queries read V as rows, 8448 as V^T tiles.
@pytest.mark.parametrize("s", [256, 8448])
@pytest.mark.parametrize("jump", [30.0, 400.0])
def test_attention_score_jump_past_first_block(dev, jump, s):
    """Keys whose scores exceed the scores of the first 32 keys by about
    `jump` (natural-log units).  The kernel's first pass keeps each query's
    reference max from its first key sub-block: a jump of 30 stays within
    its range (P up to ~e^33, l and O finite), one of 400 overflows it, which
    the kernel detects and redoes in the running-max form.  Either way the
    output equals the reference, and the MXFP8 form its quantization."""
    b, t, h = 1, 700, 2
    say("attention score jump", jump, s)
    g = torch.Generator().manual_seed(int(jump))
    # Head 0: every query is q0 plus a little noise; keys 600..609 are q0
    # scaled to a logit of about `jump` against it.
    q0 = bf16_randn(g, (128,)).float()
    q = (q0 + 0.05 * bf16_randn(g, (b, s, h, 128)).float()).to(torch.bfloat16)
    k = bf16_randn(g, (b, t, h, 128))
    v = bf16_randn(g, (b, t, h, 128))
    scale = 128 ** -0.5
    k[0, 600:610, 0] = (q0 * (jump / (scale * q0.square().sum().item()))).to(torch.bfloat16)
    q, k, v = q.to(dev), k.to(dev), v.to(dev)
    out = attention.attention(q, k, v)
    torch.cuda.synchronize()
    ref = reference(q, k, v, scale)
    assert torch.isfinite(out.float()).all()
    check(out, ref)
    got, want = attention.attention_mxfp8(q, k, v, tiled=False), mxfp8.quantize(out.view(s, h * 128))
    assert torch.equal(got.values.view(torch.uint8), want.values.view(torch.uint8))
    assert torch.equal(got.scales.view(torch.uint8), want.scales.view(torch.uint8))
    if s > 256:  # 700 keys are too few to split: the first queries' workgroups, with V as rows
        rows = attention.attention(q[0, :256].unsqueeze(0), k, v)
        assert torch.equal(out[:, :256].contiguous().view(torch.int16), rows.view(torch.int16))


def test_attention_v_tiles_split_ragged(dev):
    """V^T tiles (more than 8192 queries) with the items split over key ranges
    and a last key block of 28 keys."""
    from qwen_image_accel import _native
    b, s, t, h = 1, 8448, 1500, 2
    say("attention v tiles, split, ragged", s, t)
    assert _native.lib().qim_attention_workspace_bytes(b, s, t, h, 128) > b * h * 24 * 16384  # V^T and partials
    g = torch.Generator().manual_seed(t)
    q, k, v = (bf16_randn(g, (b, n, h, 128)).to(dev) for n in (s, t, t))
    out = attention.attention(q, k, v)
    check(out, reference(q, k, v, 128 ** -0.5))
    got, want = attention.attention_mxfp8(q, k, v, tiled=True), mxfp8.quantize(out.view(s, h * 128), tiled=True)
    assert torch.equal(got.values.view(torch.uint8), want.values.view(torch.uint8))
    assert torch.equal(got.scales.view(torch.uint8), want.scales.view(torch.uint8))


# (2, 200, 333, 3): 400 rows, padded to 512, past the last query block's end;
# (1, 256, 2000, 4), (2, 520, 1500, 3) and the 4352 shapes run split and merged.
@pytest.mark.parametrize("b,s,t,h,tiled", [(1, 300, 300, 2, True), (2, 200, 333, 3, False),
                                           (1, 256, 2000, 4, True), (2, 520, 1500, 3, False),
                                           (1, 4352, 4352, 24, True), (2, 4352, 4352, 24, True)])
def test_attention_mxfp8_equals_quantized_output(dev, b, s, t, h, tiled):
    """The fused MXFP8 output is bit-identical to quantizing the bf16 output
    (every code and scale byte, padding rows included: the buffers start
    as 0xff)."""
    say("attention mxfp8", b, s, t, h, tiled)
    g = torch.Generator().manual_seed(7 * b + s + t + h)
    q = bf16_randn(g, (b, s, h, 128)).to(dev)
    kv = bf16_randn(g, (b, t, 2 * h * 128)).to(dev)
    k, v = (kv[:, :, i * h * 128:(i + 1) * h * 128].unflatten(-1, (h, 128)) for i in (0, 1))
    ref = mxfp8.quantize(attention.attention(q, k, v).reshape(b * s, h * 128), tiled=tiled)
    out = mxfp8.empty_quantized(b * s, h * 128, dev, tiled=tiled)
    out.values.view(torch.uint8).fill_(0xff)
    out.scales.view(torch.uint8).fill_(0xff)
    got = attention.attention_mxfp8(q, k, v, tiled=tiled, out=out)
    torch.cuda.synchronize()
    assert torch.equal(got.values.view(torch.uint8), ref.values.view(torch.uint8))
    assert torch.equal(got.scales.view(torch.uint8), ref.scales.view(torch.uint8))


def test_attention_rejects_other_head_dims(dev):
    from qwen_image_accel import _native
    x = torch.zeros(1, 8, 1, 64, dtype=torch.bfloat16, device=dev)
    with pytest.raises(_native.Unsupported):
        attention.attention(x, x, x)


@pytest.mark.parametrize("t", [1, 31, 33, 64, 65, 100, 161, 225, 290, 333, 511])
def test_attention_v_rows_against_v_tiles(dev, t):
    """V read as rows (up to 8192 queries) and as transposed tiles (more): the
    same products in the same order, so the same bits for the same queries, at
    partial sub-blocks and blocks, with an infinity and a NaN in V's last row
    (which the rows past it must not touch), in the plain and the MXFP8 form."""
    say("attention v rows / tiles", t)
    g = torch.Generator().manual_seed(t)
    q, k, v = (bf16_randn(g, (1, n, 2, 128)).to(dev) for n in (8448, t, t))
    v[0, -1, 0, 5], v[0, -1, 1, 7] = float("inf"), float("nan")
    tiles = attention.attention(q, k, v)
    rows = attention.attention(q[0, :1024].unsqueeze(0), k, v)
    assert torch.equal(tiles[:, :1024].contiguous().view(torch.int16), rows.view(torch.int16))
    assert not torch.isfinite(rows[0, :, 0, 5].float()).any() and torch.isnan(rows[0, :, 1, 7].float()).all()
    assert torch.isfinite(rows[0, :, 0, 6:].float()).all() and torch.isfinite(rows[0, :, 1, 8:].float()).all()
    v[0, -1, 0, 5], v[0, -1, 1, 7] = 1.0, -1.0
    tq, rq = attention.attention_mxfp8(q, k, v, tiled=False), attention.attention_mxfp8(q[0, :1024].unsqueeze(0), k, v,
                                                                                      tiled=False)
    assert torch.equal(tq.values[:1024].view(torch.uint8), rq.values.view(torch.uint8))
    ref = mxfp8.quantize(attention.attention(q, k, v).view(8448, 256))
    assert torch.equal(tq.values.view(torch.uint8), ref.values.view(torch.uint8))
    assert torch.equal(tq.scales.view(torch.uint8), ref.scales.view(torch.uint8))


def test_attention_output_stride_of_four(dev):
    """An output whose rows are 8- but not 16-byte aligned, and one that is."""
    say("attention output stride")
    g = torch.Generator().manual_seed(3)
    q, k, v = (bf16_randn(g, (1, n, 3, 128)).to(dev) for n in (300, 200, 200))
    want = attention.attention(q, k, v)
    for pad in (4, 8):
        wide = torch.zeros(1, 300, 384 + pad, device=dev, dtype=torch.bfloat16)
        out = wide[:, :, :384].unflatten(-1, (3, 128))
        attention.attention(q, k, v, out=out)
        assert torch.equal(out, want) and not wide[:, :, 384:].any()


@pytest.mark.parametrize("s", [256, 8448])
@pytest.mark.parametrize("redo", [False, True])
def test_attention_row_sum_rounds_once_per_sub_block(dev, s, redo):
    """The row sum's order: a lane's 16 keys of a sub-block are summed from zero
    and added to its running sum once.  Every lane's sum is 16 after the first 32
    keys (P = 1); each later sub-block brings 16 x 2^-23, one unit in the last
    place of 16, of which any 4 are half lost.  V makes the first keys' mean
    the midpoint 1 + 3 * 2^-8 of two bf16 values, so the 28 units tell on the
    output: 1 + 2^-7, and the tie's 1 + 2^-6 without them.  960 keys (no split
    over key ranges), V as rows and as tiles (more than 8192 queries), in the
    first pass and in the redo (one query of the workgroup overflows it)."""
    say("attention row sum", s, redo)
    t = 960
    q, k, v = (torch.zeros(1, n, 1, 128, dtype=torch.bfloat16) for n in (s, t, t))
    q[..., 0], k[:, 32:, :, 0] = 1.0, -23.0
    if redo:
        q[:, 255, :, 0], q[:, 255, :, 1], k[:, 100, :, 1] = 0.0, 8.0, 64.0
    v[:, 0:16], v[:, 16:32] = 1 + 2.0 ** -7, 1 + 2.0 ** -6
    out = attention.attention(q.to(dev), k.to(dev), v.to(dev), scale=0.6931471805599453)
    rows = [i for i in range(s) if not (redo and i == 255)]
    assert (out.cpu()[:, rows] == 1 + 2.0 ** -7).all()


@pytest.mark.parametrize("t", [520, 1500])
def test_attention_output_over_v(dev, t):
    """The output may lie over V (whole items, and items split over key ranges
    and merged): as bf16 rows, as rows of a fused QKV buffer, and as MXFP8 codes."""
    b, h = 2, 3
    say("attention output over v", t)
    g = torch.Generator().manual_seed(t)
    qkv = bf16_randn(g, (b, t, 3 * h * 128)).to(dev)
    q, k, v = (qkv[:, :, i * h * 128:(i + 1) * h * 128].unflatten(-1, (h, 128)) for i in range(3))
    want = attention.attention(q, k, v).clone()
    ref = mxfp8.quantize(want.view(b * t, h * 128), tiled=True)
    over = v.contiguous()
    assert torch.equal(attention.attention(q, k, over, out=over), want)
    # Codes in V's own memory (a V with rows to spare for the padded code rows).
    buf = torch.empty(ref.values.numel(), device=dev, dtype=torch.bfloat16)
    over = buf[:b * t * h * 128].view(b, t, h, 128)
    over.copy_(v)
    out = ref._replace(values=buf.view(torch.uint8)[:ref.values.numel()].view(ref.values.dtype).view(ref.values.shape),
                       scales=torch.empty_like(ref.scales))
    attention.attention_mxfp8(q, k, over, out=out)
    assert torch.equal(out.values.view(torch.uint8), ref.values.view(torch.uint8))
    assert torch.equal(out.scales.view(torch.uint8), ref.scales.view(torch.uint8))
    # Column blocks of one buffer: beside V, over Q, across two heads of V, over V.
    w = h * 128
    for at in (3 * w, 0, 2 * w + 128, 2 * w):
        wide = torch.zeros(b, t, 4 * w, device=dev, dtype=torch.bfloat16)
        wide[:, :, :3 * w] = qkv
        wq, wk, wv, o = (wide[:, :, c:c + w].unflatten(-1, (h, 128)) for c in (0, w, 2 * w, at))
        attention.attention(wq, wk, wv, out=o)
        assert torch.equal(o, want), at
