"""The fused decoder-layer steps (residual + RMSNorm, head split + rotary,
SwiGLU) against 64-bit forms of the same operations, at the edges of their
vector, register and scalar paths.  Bounds: one rounding to the data type per
rounding the kernel makes (unit roundoff ``u``), plus a few fp32 roundings."""
import pytest
import torch

from hexgen2_amd import ops
from hexgen2_amd.llama import rms_norm

pytestmark = pytest.mark.gpu

DTYPES = [torch.float16, torch.bfloat16, torch.float32]
# half a spacing relative to the value: 2^-p for p significant bits (11, 8, 24)
UNIT = {torch.float16: 2.0 ** -11, torch.bfloat16: 2.0 ** -8, torch.float32: 2.0 ** -24}
FP32 = 2.0 ** -20  # a sum of squares of up to 2^13 terms in pairwise order, rsqrt, a division
TINY = 2.0 ** -24  # spacing of the smallest float16 values


def _within(got, want, bound):
    assert torch.isfinite(got.double()).all()
    assert ((got.double() - want).abs() <= bound).all(), float(((got.double() - want).abs() - bound).max())


@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("hidden", [1, 7, 64, 1024, 2048, 2056, 4096, 4104, 8192, 8200, 8201])
@pytest.mark.parametrize("with_y", [False, True])
def test_add_rms_norm(dtype, hidden, with_y):
    torch.manual_seed(hidden)
    h, y = (torch.randn(2, 3, hidden, device="cuda").to(dtype) for _ in range(2))
    w = torch.randn(hidden, device="cuda").to(dtype)
    want_h = h + y if with_y else h.clone()
    kept = h.clone()
    out = ops.add_rms_norm(kept, y if with_y else None, w, 1e-5)
    assert torch.equal(kept, want_h)
    x = want_h.double()
    want = x * torch.rsqrt(x.square().mean(-1, keepdim=True) + 1e-5) * w.double()
    bound = (2.1 * UNIT[dtype] + FP32) * want.abs() + TINY * (1 + w.double().abs())
    _within(out, want, bound)
    _within(rms_norm(want_h, w, 1e-5), want, bound)
    # the last token of each sequence: rows 3 * hidden apart, h left alone
    last = ops.add_rms_norm(h[:, -1], y[:, -1] if with_y else None, w, 1e-5, keep_sum=False)
    assert torch.equal(last, out[:, -1])


@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("heads,kv_heads,dim", [(4, 4, 16), (32, 4, 64), (8, 1, 128), (32, 32, 128), (3, 1, 6), (5, 5, 20)])
@pytest.mark.parametrize("ragged", [False, True])
def test_rope_split(dtype, heads, kv_heads, dim, ragged):
    torch.manual_seed(dim)
    batch, seqlen, offset = (3, 1, 0) if ragged else (2, 9, 4091)
    qkv = torch.randn(batch, seqlen, (heads + 2 * kv_heads) * dim, device="cuda").to(dtype)
    inv = 1.0 / (10000.0 ** (torch.arange(0, dim, 2, device="cuda", dtype=torch.float32) / dim))
    at = torch.tensor([0, 17, 8191], dtype=torch.int32, device="cuda") if ragged else None
    q, kv = ops.rope_split(qkv, heads, kv_heads, dim, inv, offset, at)
    qk, v = qkv[..., :(heads + kv_heads) * dim], qkv[..., (heads + kv_heads) * dim:]
    pos = at.float()[:, None] if ragged else (offset + torch.arange(seqlen, device="cuda").float())[None].expand(batch, -1)
    angle = (pos[..., None] * inv).double()[:, :, None]  # the fp32 product, as the kernel forms it
    x = qk.double().view(batch, seqlen, heads + kv_heads, dim)
    a, b = x[..., :dim // 2], x[..., dim // 2:]
    want = torch.cat((a * angle.cos() - b * angle.sin(), b * angle.cos() + a * angle.sin()), -1)
    got = torch.cat((q, kv[:, :, 0]), 2)
    size = (a.abs() + b.abs()).repeat(1, 1, 1, 2)
    _within(got, want, UNIT[dtype] * 1.01 * want.abs() + FP32 * size + TINY)
    assert torch.equal(kv[:, :, 1].reshape(v.shape), v)


@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("width", [1, 7, 255, 256, 2048, 2056, 5632])
def test_silu_mul(dtype, width):
    torch.manual_seed(width)
    gate_up = (4 * torch.randn(3, 2, 2 * width, device="cuda")).to(dtype)
    g, u = gate_up.double().chunk(2, -1)
    want = g * torch.sigmoid(g) * u
    _within(ops.silu_mul(gate_up), want, (UNIT[dtype] * 1.01 + FP32) * want.abs() + TINY)


@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("rows", [1, 2])
@pytest.mark.parametrize("hidden,n", [(8, 1), (64, 7), (504, 1023), (512, 2047), (520, 2048), (2048, 2050), (4104, 9),
                                      (5632, 64), (8192, 33)])
def test_norm_linear(dtype, rows, hidden, n):
    """Each lane sums hidden / 64 products in fp32, then six levels of a tree."""
    torch.manual_seed(hidden + n)
    h, y = (torch.randn(rows, 1, hidden, device="cuda").to(dtype) for _ in range(2))
    norm = torch.randn(hidden, device="cuda").to(dtype)
    w = (torch.randn(2 * n, hidden, device="cuda") * hidden ** -0.5).to(dtype)
    total = h.clone()
    x = ops.add_rms_norm(total, y, norm, 1e-5)  # the same roundings
    steps = (hidden + 63) // 64 + 8

    def product(x, w):
        return x.double() @ w.double().T, steps * 2.0 ** -24 * (x.double().abs() @ w.double().abs().T)

    want, err = product(h, w[:n])
    got, same = ops.norm_linear(h, None, None, 0.0, w[:n].contiguous())
    assert same is h
    _within(got, want, 1.01 * UNIT[dtype] * want.abs() + err + TINY)
    # the norm's own sum may round one value of x the other way
    flip = 2 * UNIT[dtype] * (x.double().abs().amax(-1, keepdim=True) * w.double().abs().amax())
    want, err = product(x, w[:n])
    got, kept = ops.norm_linear(h, y, norm, 1e-5, w[:n].contiguous())
    assert torch.equal(kept, total) and not torch.equal(kept, h)
    _within(got, want, 1.01 * UNIT[dtype] * want.abs() + err + 8 * flip + TINY)
    both, err = product(x, w)
    g, u = both[..., :n], both[..., n:]
    silu = g * torch.sigmoid(g)
    eg, eu = (err + 8 * flip)[..., :n], (err + 8 * flip)[..., n:]
    got, kept = ops.norm_linear(h, y, norm, 1e-5, w, glu=True, keep_sum=False)
    assert kept is h
    bound = (1.01 * UNIT[dtype] + FP32) * (silu * u).abs() + 1.1 * u.abs() * eg + silu.abs() * eu + 1.1 * eg * eu
    _within(got, silu * u, bound + TINY)


@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("batch,seqlen,ragged", [(1, 1, False), (1, 2, False), (2, 1, False), (2, 1, True)])
@pytest.mark.parametrize("hidden,heads,kv_heads,dim", [(64, 4, 4, 16), (2048, 32, 4, 64), (520, 8, 1, 128), (16, 3, 1, 6),
                                                       (1024, 48, 8, 64)])
def test_norm_rope_linear(dtype, batch, seqlen, ragged, hidden, heads, kv_heads, dim):
    """Against the product of the same normalised tokens in 64 bits, turned
    by the fp32 angle: the product's error turns with it."""
    torch.manual_seed(hidden + batch)
    offset = 0 if ragged else 4091
    h, y = (torch.randn(batch, seqlen, hidden, device="cuda").to(dtype) for _ in range(2))
    norm = torch.randn(hidden, device="cuda").to(dtype)
    w = (torch.randn((heads + 2 * kv_heads) * dim, hidden, device="cuda") * hidden ** -0.5).to(dtype)
    inv = 1.0 / (10000.0 ** (torch.arange(0, dim, 2, device="cuda", dtype=torch.float32) / dim))
    at = torch.tensor([8191, 17], dtype=torch.int32, device="cuda") if ragged else None
    total = h.clone()
    x = ops.add_rms_norm(total, y, norm, 1e-5)
    q, kv, kept = ops.norm_rope_linear(h, y, norm, 1e-5, w, heads, kv_heads, dim, inv, offset, at)
    assert torch.equal(kept, total)
    full = (x.double() @ w.double().T).view(batch, seqlen, -1, dim)
    flip = 2 * UNIT[dtype] * (x.double().abs().amax() * w.double().abs().amax())
    err = ((hidden + 63) // 64 + 8) * 2.0 ** -24 * (x.double().abs() @ w.double().abs().T).view(full.shape) + 8 * flip
    pos = at.float()[:, None] if ragged else (offset + torch.arange(seqlen, device="cuda").float())[None].expand(batch, -1)
    angle = (pos[..., None] * inv).double()[:, :, None]
    a, b = full[..., :dim // 2], full[..., dim // 2:]
    want = torch.cat((a * angle.cos() - b * angle.sin(), b * angle.cos() + a * angle.sin()), -1)
    want[:, :, heads + kv_heads:] = full[:, :, heads + kv_heads:]
    got = torch.cat((q, kv.flatten(2, 3)), 2)
    size = (a.abs() + b.abs()).repeat(1, 1, 1, 2)
    both = (err[..., :dim // 2] + err[..., dim // 2:]).repeat(1, 1, 1, 2)
    _within(got, want, 1.01 * UNIT[dtype] * want.abs() + both + FP32 * size + TINY)


def test_norm_linear_fits_and_refuses():
    x, w = torch.zeros(2, 1, 64, device="cuda").half(), torch.zeros(16, 64, device="cuda").half()
    assert ops.linear_fits(x, w)
    wide = torch.zeros(1, 1, 32776, device="cuda").half()
    for bad in (torch.zeros(3, 1, 64, device="cuda").half(), wide, x[..., :60], x[:0], x.double()):
        assert not ops.linear_fits(bad, w)
    assert not ops.linear_fits(x, w.T) and not ops.linear_fits(x, w.float())
    with pytest.raises(NotImplementedError):
        ops.norm_linear(wide, None, None, 0.0, torch.zeros(1, 32776, device="cuda").half())
    with pytest.raises(ValueError):
        ops.norm_linear(x, x, None, 0.0, w)
    with pytest.raises(ValueError):
        ops.norm_linear(x, None, None, 0.0, w[:, :32])


def test_layer_steps_refuse_what_they_cannot_address():
    x = torch.zeros(2, 3, 8, device="cuda", dtype=torch.float16)
    w = torch.zeros(8, device="cuda", dtype=torch.float16)
    with pytest.raises(ValueError):
        ops.add_rms_norm(x, None, w[:4], 1e-5)
    with pytest.raises(ValueError):
        ops.add_rms_norm(x.transpose(0, 1), None, w, 1e-5)
    with pytest.raises(ValueError):
        ops.add_rms_norm(x, x.float(), w, 1e-5)
    with pytest.raises(ValueError):
        ops.silu_mul(x[..., :6])
    with pytest.raises(ValueError):
        ops.rope_split(x, 2, 1, 2, torch.zeros(2, device="cuda"))
    assert ops.silu_mul(x[:0]).shape == (0, 3, 4)
