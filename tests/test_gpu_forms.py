"""decode_attention's kept parameter blocks: calls of one geometry on other
tensors, lengths and options give what a first call gives, and a block made
for one geometry is not used for another; and the multi-position cache write
over every batch window and stride it accepts."""
import pytest
import torch

from hexgen2_amd import mha, ops
from hexgen2_amd.generation import InferenceParams

pytestmark = pytest.mark.gpu


def _call(seed, strided=False, out=None, **kw):
    g = torch.Generator(device="cuda").manual_seed(seed)
    q = torch.randn(2, 1, 8, 64, generator=g, device="cuda").half()
    cache = torch.randn(2, 700, 2, 2, 64, generator=g, device="cuda").half()
    if strided:  # the same values behind other strides
        q = torch.stack((q, q), 2)[:, :, 0]
        cache = torch.cat((cache, cache), 1)[:, :700]
    kv = torch.randn(2, 2, 2, 64, generator=g, device="cuda").half()
    lens = torch.tensor([600 - seed, 17 + seed], dtype=torch.int32, device="cuda")
    args = dict(max_seqlen=601, seqlens=lens, kv_new=kv, **kw)
    return ops.decode_attention(q, cache, out=out, **args), cache


@pytest.mark.parametrize("kw", [{}, {"softmax_scale": 0.05}, {"partition": 64}, {"kernel": "valu"}])
def test_kept_blocks_give_the_first_call(device, kw):
    kept = dict(ops._ATTEND_FORMS)
    for seed in (0, 1, 2):
        ops._ATTEND_FORMS.clear()
        want, want_cache = _call(seed, **kw)
        for strided in (False, True, False, True):
            got, cache = _call(seed, strided, out=torch.empty_like(want) if strided else None, **kw)
            assert torch.equal(got, want) and torch.equal(cache, want_cache)
    for seed in (3, 4, 5):  # other tensors on the block seed 2's calls left
        got, cache = _call(seed, **kw)
        ops._ATTEND_FORMS.clear()
        want, want_cache = _call(seed, **kw)
        assert torch.equal(got, want) and torch.equal(cache, want_cache)
    ops._ATTEND_FORMS.update(kept)


def test_kept_blocks_refuse_what_a_first_call_refuses(device):
    _call(0)
    with pytest.raises(ValueError):
        _call(0, kernel="none")
    with pytest.raises(ValueError):
        _call(0, partition=63)
    q, cache = torch.zeros(1, 1, 8, 64, device="cuda").half(), torch.zeros(1, 8, 2, 2, 64, device="cuda").half()
    for _ in range(2):  # refused by the library, with a kept block and without
        with pytest.raises(ValueError):
            ops.decode_attention(q, cache, max_seqlen=9, seqlen_bias=9)
    for i in range(80):  # bounded
        ops.decode_attention(q, cache, max_seqlen=8, seqlen_bias=8, softmax_scale=1.0 + i)
    assert len(ops._ATTEND_FORMS) <= 64


def test_a_growing_view_keeps_one_block(device):
    """A decode loop over cache views one token longer each step keeps a few
    blocks, and a kept block admits no length past the view it is called with."""
    cache = torch.randn(2, 300, 2, 2, 64, device="cuda").half()
    q = torch.randn(2, 1, 8, 64, device="cuda").half()
    ops._ATTEND_FORMS.clear()
    for n in range(200, 300):
        got = ops.decode_attention(q, cache[:, :n], max_seqlen=n, seqlen_bias=n)
    assert len(ops._ATTEND_FORMS) == 1
    assert torch.equal(got, ops.decode_attention(q, cache[:, :299].clone(), max_seqlen=299, seqlen_bias=299))
    with pytest.raises(ValueError):
        ops.decode_attention(q, cache[:, :250], max_seqlen=251, seqlen_bias=251)


@pytest.mark.parametrize("start,batch,offset,length", [(0, 3, 0, 5), (1, 2, 3, 2), (2, 1, 7, 9), (0, 1, 14, 2), (1, 1, 0, 16)])
@pytest.mark.parametrize("pad", [0, 8])
def test_cache_write(device, start, batch, offset, length, pad):
    row = 2 * 2 * 64
    flat = torch.randn(3 * (16 * row + pad), device="cuda").half()
    cache = flat.as_strided((3, 16, 2, 2, 64), (16 * row + pad, row, 128, 64, 1))
    kv = torch.randn(batch, length, 2, 2, 64, device="cuda").half()
    params = InferenceParams(16, 3, offset, start, {0: cache})
    if pad and batch > 1:  # sequences not whole rows apart
        with pytest.raises(ValueError):
            mha._update_kv_cache(kv, params, 0)
        return
    want = cache.clone()
    want[start:start + batch, offset:offset + length] = kv
    view = mha._update_kv_cache(kv, params, 0)
    assert torch.equal(cache, want)
    assert view.data_ptr() == cache[start:].data_ptr() and view.shape == (batch, offset + length, 2, 2, 64)
