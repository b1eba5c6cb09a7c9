"""Attention of several query rows (q_len > 1, 16-bit, head_dim 64 / 128)
against the float64 oracle, at the edges of the query-tile kernel's tiles.  An
explicit partition takes that kernel at any size (4096: keys unsplit); without
one small calls run the per-row kernels.

Tolerances as for decode attention (max-abs, fp16 2e-3, bf16 8e-3): the
output's own rounding plus fp32 sums of hi + lo probabilities (2^-17 relative
for bf16, below the output's 2^-9).
"""
import numpy as np
import pytest
import torch

from hexgen2_amd import ops
from oracle import kv_oracle as oracle

pytestmark = pytest.mark.gpu

TOL = {torch.float16: 2e-3, torch.bfloat16: 8e-3}


def f64(t):
    return t.detach().cpu().double().numpy()


def make(batch, cap, hq, hkv, d, dtype, device, q_len, seed=5):
    g = torch.Generator(device=device).manual_seed(seed)
    q = torch.randn((batch, q_len, hq, d), generator=g, device=device).to(dtype)
    cache = torch.randn((batch, cap, 2, hkv, d), generator=g, device=device).to(dtype)
    return q, cache


def check(out, q, cache, lens, causal):
    err = float(np.abs(f64(out) - oracle.attend(f64(q), f64(cache), lens, causal=causal)).max())
    assert err <= TOL[q.dtype], f"max-abs error {err}"


# (dtype, q heads, KV heads, head_dim): groups 1, 2, 3, 4, 8 and 16
GEOMETRIES = [(torch.float16, 2, 2, 128), (torch.bfloat16, 4, 2, 64), (torch.float16, 6, 2, 64),
              (torch.bfloat16, 8, 2, 128), (torch.float16, 16, 2, 64), (torch.bfloat16, 16, 1, 128)]
# (q_len, keys before the chunk): single rows beyond decode, tile edges
# (32 rows a wave, 128 a workgroup, 32- and 64-key blocks), ragged ones
LENGTHS = [(2, 0), (6, 4090), (31, 0), (32, 1), (33, 31), (64, 0), (65, 63), (127, 129), (128, 0), (129, 500),
           (300, 17)]


@pytest.mark.parametrize("q_len,past", LENGTHS)
@pytest.mark.parametrize("dtype,hq,hkv,d", GEOMETRIES)
@pytest.mark.parametrize("partition", [0, 4096])
def test_tiles_match_the_oracle(device, dtype, hq, hkv, d, q_len, past, partition):
    """With a partition the tile kernel whatever the size, without one the
    kernel that leads."""
    n = past + q_len
    q, cache = make(2, n + 3, hq, hkv, d, dtype, device, q_len)
    out = ops.decode_attention(q, cache, max_seqlen=n, seqlen_bias=n, causal=True, partition=partition)
    check(out, q, cache, [n, n], True)
    if q_len < 130:
        out = ops.decode_attention(q, cache, max_seqlen=n, seqlen_bias=n, partition=partition)
        check(out, q, cache, [n, n], False)


@pytest.mark.parametrize("dtype,hq,hkv,d", GEOMETRIES)
@pytest.mark.parametrize("partition", [0, 64, 192])
def test_ragged_lengths_strides_and_partitions(device, dtype, hq, hkv, d, partition):
    """Per-sequence lengths from the device (one shorter than the chunk: its
    first rows attend nothing and are zero), a strided q and out, a cache
    that is a view into a larger one, every partition count."""
    q_len, cap = 37, 420
    g = torch.Generator(device=device).manual_seed(8)
    wide = torch.randn((3, q_len, hq + 2, d), generator=g, device=device).to(dtype)
    q = wide[:, :, 1:hq + 1]
    cache = torch.randn((5, cap, 2, hkv, d), generator=g, device=device).to(dtype)[1:4]
    out = torch.full((3, q_len, hq + 1, d), 7.0, dtype=dtype, device=device)[:, :, :hq]
    lens = [400, 20, 130]
    seqlens = torch.tensor(lens, dtype=torch.int32, device=device)
    ops.device_status()
    ops.decode_attention(q, cache, max_seqlen=400, seqlens=seqlens, causal=True, out=out, partition=partition)
    for b, n in enumerate(lens):
        first = max(0, q_len - n)  # rows before it attend no key
        assert torch.equal(out[b, :first], torch.zeros_like(out[b, :first]))
        check(out[b:b + 1, first:], q[b:b + 1, first:], cache[b:b + 1], [n], True)
    assert ops.device_status() == 0
    # a bound below the lengths cuts them and says so, as the per-row kernels do
    cut = ops.decode_attention(q, cache, max_seqlen=256, seqlens=seqlens, partition=partition)
    assert ops.device_status() == 2
    check(cut, q, cache, [256, 20, 130], False)


@pytest.mark.parametrize("dtype,hq,hkv,d", [(torch.float16, 4, 2, 64), (torch.bfloat16, 8, 2, 128)])
@pytest.mark.parametrize("partition", [0, 64, 4096])
@pytest.mark.parametrize("where,value", [("v", float("inf")), ("v", float("nan")), ("k", float("nan")),
                                         ("k", float("inf")), ("q", float("nan"))])
def test_non_finite_values_stay_in_their_rows(device, dtype, hq, hkv, d, partition, where, value):
    """An infinity or NaN reaches the rows that attend it, as in the per-row
    kernel, and leaves every other row as it was."""
    q_len, n = 150, 170
    q, cache = make(1, n, hq, hkv, d, dtype, device, q_len, seed=3)
    clean = ops.decode_attention(q, cache, max_seqlen=n, seqlen_bias=n, causal=True, partition=partition)
    at = 95  # first attended by query row 75
    if where == "q":
        q[0, 40, 1, 5] = value
    else:
        cache[0, at, "kv".index(where), 1, 3] = value
    out = ops.decode_attention(q, cache, max_seqlen=n, seqlen_bias=n, causal=True, partition=partition)
    ref = ops.decode_attention(q, cache, max_seqlen=n, seqlen_bias=n, causal=True, partition=partition, kernel="valu")
    assert torch.equal(torch.isfinite(out), torch.isfinite(ref))
    if where == "v" and value == float("inf"):
        # p * inf is inf for every attending row
        assert bool((out[0, 75:, hq // hkv:, 3] == value).all())
    else:
        assert torch.equal(torch.isnan(out), torch.isnan(ref))
    ok = torch.isfinite(ref)
    assert float((out[ok].double() - ref[ok].double()).abs().max()) <= 2 * TOL[dtype]
    if where != "q":
        # rows that do not attend it: recomputed key by key where their tile
        # held it, so two fp32 sums of the same terms, each within TOL
        diff = float((out[0, :75].double() - clean[0, :75].double()).abs().max())
        assert diff <= 2 * TOL[dtype]
        assert torch.equal(out[0, :, :hq // hkv], clean[0, :, :hq // hkv])  # the other KV head


@pytest.mark.parametrize("dtype,hq,hkv,d", [(torch.float16, 4, 2, 64), (torch.bfloat16, 8, 2, 128)])
@pytest.mark.parametrize("partition", [0, 64, 4096])
@pytest.mark.parametrize("value", [float("inf"), float("nan")])
def test_rows_without_keys_are_zero_beside_non_finite_values(device, dtype, hq, hkv, d, partition, value):
    """A row that attends nothing is zero whatever the rows of its tile meet."""
    q_len, n = 37, 20
    q, cache = make(2, 80, hq, hkv, d, dtype, device, q_len)
    cache[:, 0, 1, :, 3] = value
    seqlens = torch.tensor([n, 80], dtype=torch.int32, device=device)
    out = ops.decode_attention(q, cache, max_seqlen=80, seqlens=seqlens, causal=True, partition=partition)
    assert torch.equal(out[0, :q_len - n], torch.zeros_like(out[0, :q_len - n]))
    assert not bool(torch.isfinite(out[0, q_len - n:, :, 3]).any())
    rest = [i for i in range(d) if i != 3]
    assert bool(torch.isfinite(out[..., rest]).all())


@pytest.mark.parametrize("dtype,hq,hkv,d", [(torch.float16, 4, 2, 64), (torch.bfloat16, 8, 2, 128)])
@pytest.mark.parametrize("partition", [0, 64, 4096])
@pytest.mark.parametrize("where,value", [("v", float("inf")), ("v", float("nan")), ("k", float("nan"))])
def test_out_may_be_q(device, dtype, hq, hkv, d, partition, where, value):
    """In place, rows recomputed for a non-finite value read their own query:
    the same results as into another tensor."""
    q_len, n = 150, 170
    q, cache = make(1, n, hq, hkv, d, dtype, device, q_len, seed=3)
    cache[0, 95, "kv".index(where), 1, 3] = value
    args = dict(max_seqlen=n, seqlen_bias=n, causal=True, partition=partition)
    want = ops.decode_attention(q, cache, **args)
    got = ops.decode_attention(q, cache, out=q, **args)
    assert torch.equal(torch.isnan(got), torch.isnan(want))
    assert torch.equal(got.nan_to_num(), want.nan_to_num())


@pytest.mark.parametrize("partition", [0, 4096])
def test_lowest_scores_and_large_scales(device, partition):
    """Scores at the type's lowest and highest values (softmax one-hot)."""
    q, cache = make(1, 90, 2, 1, 64, torch.bfloat16, device, 70)
    q *= 1e4
    cache[:, :, 0] *= 1e4
    out = ops.decode_attention(q, cache, max_seqlen=90, seqlen_bias=90, causal=True, partition=partition)
    check(out, q, cache, [90], True)


def test_sum_keeps_keys_far_below_the_largest(device):
    """A probability of 1 and 2^20 - 1 of 2^-25.2, each below half a spacing of
    the row's running sum: together 2.7% of it.  The call is large enough to
    walk its keys unsplit.  Bound: the output's rounding and 2^-11 (2^20 / 64
    fp32 additions of tile sums, half a spacing each, relative to the sum)."""
    n, q_len, d = 1 << 20, 33024, 64
    cache = torch.zeros(1, n, 2, 1, d, dtype=torch.bfloat16, device=device)
    cache[:, 0, 0, 0, 0] = 17.5
    cache[:, 0, 1] = 1
    q = torch.zeros(1, q_len, 1, d, dtype=torch.bfloat16, device=device)
    q[..., 0] = d ** 0.5  # scores are dimension 0 of the keys
    out = f64(ops.decode_attention(q, cache, max_seqlen=n, seqlen_bias=n)[:, ::997])
    want = 1 / (1 + (n - 1) * np.exp(-17.5))
    assert float(np.abs(out - want).max()) <= (2.0 ** -8 + 2.0 ** -11) * want


@pytest.mark.parametrize("dtype,high", [(torch.float16, 17.46875), (torch.float16, 22.0), (torch.bfloat16, 17.5)])
@pytest.mark.parametrize("first", [True, False])
def test_many_keys_far_below_one(device, dtype, high, first):
    """One score exp(17) above 65535 others, whose values still make up the
    output (the high one's are zero): no probability may be lost.  The call is
    large enough to walk its keys unsplit.  Bound: the output's rounding,
    65536 / 16 fp32 additions (the sum has as many), and for fp16 2^-36 of the
    largest probability per key, times values below 2."""
    n, q_len, heads, d = 65536, 4224, 8, 64
    g = torch.Generator(device=device).manual_seed(1)
    cache = torch.zeros(1, n, 2, heads, d, dtype=dtype, device=device)
    cache[:, :, 1] = (1 + torch.rand(1, n, heads, d, generator=g, device=device)).to(dtype)
    at = 0 if first else n - 1
    cache[:, at, 0, :, 0] = high
    cache[:, at, 1] = 0
    q = torch.zeros(1, q_len, heads, d, dtype=dtype, device=device)
    q[..., 0] = d ** 0.5  # scores are dimension 0 of the keys
    out = f64(ops.decode_attention(q, cache, max_seqlen=n, seqlen_bias=n)[:, ::97])
    want = oracle.attend(f64(q[:, :1]), f64(cache), [n])
    u = {torch.float16: 2.0 ** -11, torch.bfloat16: 2.0 ** -8}[dtype]
    bound = (u + 2 * n / 16 * 2.0 ** -24) * want + 2.0 ** -25 + n * 2.0 ** -36 * 2
    assert (np.abs(out - want) <= bound).all(), float((np.abs(out - want) / bound).max())


@pytest.mark.parametrize("partition", [256, 128])
def test_values_near_the_largest_number(device, partition):
    """Rows whose maximum rises by less than the tile kernel's slack over
    values near bf16's largest: no sum may pass fp32's range, as none does in
    the per-row kernel."""
    q_len, n, d = 40, 200, 64
    cache = torch.zeros(1, n, 2, 1, d, dtype=torch.bfloat16, device=device)
    cache[:, 130, 0, 0, 0] = 5.0  # 2^7.2 times the weight of any other key
    cache[:, 130, 1] = 1e37
    q = torch.zeros(1, q_len, 2, d, dtype=torch.bfloat16, device=device)
    q[..., 0] = d ** 0.5
    out = ops.decode_attention(q, cache, max_seqlen=n, seqlen_bias=n, partition=partition)
    want = oracle.attend(f64(q), f64(cache), [n])
    assert float(np.abs(f64(out) / want - 1).max()) <= 2.0 ** -8 + 2.0 ** -16


@pytest.mark.parametrize("q_len,partition", [(9, 0), (9, 192), (100, 0)])
def test_replay_matches_eager(device, q_len, partition):
    q, cache = make(1, 2100, 8, 1, 128, torch.bfloat16, device, q_len)
    assert ops.attend_kernel(q, cache, partition=partition) == ("mfma" if (q_len, partition) == (9, 0) else "tiles")
    out = torch.empty_like(q)
    ws = torch.zeros(ops.attend_workspace_bytes(q, cache, 2100, partition), dtype=torch.uint8, device=device)
    args = dict(max_seqlen=2100, seqlen_bias=2100, causal=True, workspace=ws, partition=partition)
    want = ops.decode_attention(q, cache, **args)
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        ops.decode_attention(q, cache, out=out, **args)
    for _ in range(3):
        out.fill_(7.0)
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(out, want)
