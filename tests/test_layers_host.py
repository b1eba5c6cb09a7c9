"""Planning of lists that several layers share, on the host: one layer gets
the one-layer rules, several a chunk that every kernel accepts; the checks for
tensors that overlap, of layers and of the steps between products; and the
workspace sizes."""
import ctypes

import pytest
import torch

from hexgen2_amd import _lib


def _params(dtype, batch, hq, hkv, d, longest, kernel=0, xcds=8):
    return _lib.AttendParams(dtype=dtype, batch=batch, q_len=1, q_heads=hq, kv_heads=hkv, head_dim=d, softmax_scale=1.0,
                             capacity=longest + 1, max_seqlen=longest + 1, kv_new=16, kernel=kernel, work_xcds=xcds)


@pytest.mark.parametrize("dtype,hq,hkv,d", [(0, 32, 4, 64), (0, 32, 32, 128), (1, 8, 1, 128), (1, 32, 8, 128), (2, 4, 4, 16)])
@pytest.mark.parametrize("lens", [[0], [1], [5000], [64, 8192, 17], [2048] * 8, [8192] * 64])
@pytest.mark.parametrize("layers", [1, 2, 16, 80])
def test_plan_layers(dtype, hq, hkv, d, lens, layers):
    lib = _lib.load()
    p = _params(dtype, len(lens), hq, hkv, d, max(lens))
    c = (ctypes.c_int32 * len(lens))(*lens)
    kernel, chunk, one_kernel, one_chunk = (ctypes.c_int32() for _ in range(4))
    assert lib.hexkv_attend_plan_layers(p, c, layers, kernel, chunk) == 0
    assert lib.hexkv_attend_plan_kernel(p, c, one_kernel) == 0
    p.kernel = one_kernel.value
    assert lib.hexkv_attend_plan_chunk(p, c, one_chunk) == 0
    if layers == 1 or len(lens) == 64 and hkv >= 8 and d == 128:  # a layer of 512 MB or more runs alone
        assert (kernel.value, chunk.value) == (one_kernel.value, one_chunk.value)
    # the list can be built with it, and its segments merge in the kernel
    p.kernel, p.partition = kernel.value, chunk.value
    n, most = ctypes.c_int32(), ctypes.c_int32()
    assert lib.hexkv_attend_plan(p, c, None, 0, None, 0, n, most) == 0
    assert n.value % 8 == 0 and (layers == 1 or most.value <= 64)


@pytest.mark.parametrize("hq,hkv,rows,kernel", [(8, 8, 1, "valu"), (8, 8, 15, "valu"), (8, 8, 16, "rows"),
                                                (32, 32, 3, "valu"), (32, 32, 4, "rows"), (32, 8, 3, "valu"),
                                                (32, 8, 4, "rows")])
def test_shared_row_blocks_fill_the_xcds(hq, hkv, rows, kernel):
    """A segment's items run on one XCD: row blocks only with two segments for each."""
    lib = _lib.load()
    p = _params(0, rows, hq, hkv, 128, 7570)
    k, chunk = ctypes.c_int32(), ctypes.c_int32()
    assert lib.hexkv_attend_plan_layers(p, (ctypes.c_int32 * rows)(*[7570] * rows), 6, k, chunk) == 0
    assert k.value == _lib.KERNELS[kernel]


def test_plan_layers_keeps_what_the_caller_chose():
    lib = _lib.load()
    p = _params(0, 2, 32, 32, 128, 4000, kernel=1)
    p.partition = 192
    c = (ctypes.c_int32 * 2)(4000, 3000)
    kernel, chunk = ctypes.c_int32(), ctypes.c_int32()
    assert lib.hexkv_attend_plan_layers(p, c, 8, kernel, chunk) == 0
    assert (kernel.value, chunk.value) == (1, 192)
    assert lib.hexkv_attend_plan_layers(p, c, 0, kernel, chunk) == _lib.HEXKV_EINVAL


@pytest.mark.parametrize("change,free", [(None, 1), ("out", 0), ("cache", 0), ("q", 1), ("q_in_out", 0), ("kv_in_cache", 0),
                                         ("touching", 1), ("lengths", 0)])
def test_layers_independent(change, free):
    """Only written bytes shared between layers force an order."""
    lib = _lib.load()
    batch, cap, hkv, hq, d = 2, 64, 2, 4, 64
    p = _params(0, batch, hq, hkv, d, cap - 1)
    p.q_batch_stride = p.out_batch_stride = hq * d
    p.cache_batch_stride, p.cache_pos_stride, p.cache_kv_stride = cap * 2 * hkv * d, 2 * hkv * d, hkv * d
    p.capacity = cap
    cache, row, new = batch * cap * 2 * hkv * d * 2, batch * hq * d * 2, batch * 2 * hkv * d * 2
    base = 1 << 20
    a = _lib.AttendLayer(base, base + (1 << 20), base + (2 << 20), base + (3 << 20))
    b = _lib.AttendLayer(base + (4 << 20), base + (5 << 20), base + (6 << 20), base + (7 << 20))
    if change in ("out", "cache", "q"):
        setattr(b, change, getattr(a, change))
    elif change == "q_in_out":
        b.q = a.out + row - 16
    elif change == "kv_in_cache":
        b.kv_new = a.cache + cache - new
    elif change == "touching":
        b.q, b.kv_new, b.out, b.cache = a.out + row, a.cache + cache, a.out - row, a.cache - cache
    elif change == "lengths":
        p.lengths_out_dev = a.out + 8
    assert lib.hexkv_attend_layers_independent(p, (_lib.AttendLayer * 2)(a, b), 2) == free


@pytest.mark.parametrize("dtype,hq,hkv,d", [(0, 32, 4, 64), (0, 32, 32, 128), (1, 8, 1, 128), (1, 32, 8, 128)])
@pytest.mark.parametrize("batch", [1, 8, 64])
def test_workspace_sizes_follow_the_base_partition(dtype, hq, hkv, d, batch):
    """Decode rows: the size of the call's own partitions of 128, 256 or 512
    positions (not monotone where they double)."""
    lib = _lib.load()
    group = next(g for g in (8, 4, 2, 1) if (hq // hkv) % g == 0)
    for longest in (129, 1024, 1025, 1100, 2048, 4096):
        want = batch * (hq // group) * ((longest + 1) // 2) // 2048
        part = next((p for p in (128, 256) if p >= want), 512)
        parts = (longest + part - 1) // part
        p = _lib.AttendParams(dtype=dtype, batch=batch, q_len=1, q_heads=hq, kv_heads=hkv, head_dim=d, softmax_scale=1.0,
                              capacity=longest, max_seqlen=longest)
        need = _lib.ATTEND_COUNTER_BYTES + batch * hq * parts * (d + 2) * 4 if parts > 1 else 0
        assert lib.hexkv_attend_workspace_bytes(p) == need


@pytest.mark.skipif(torch.cuda.device_count() > 0, reason="calls whose workspace fits would run on made-up addresses")
@pytest.mark.parametrize("dtype,hq,hkv,d", [(0, 32, 4, 64), (0, 32, 32, 128), (1, 8, 1, 128), (1, 32, 8, 128),
                                            (0, 12, 12, 64), (1, 1, 1, 64)])
@pytest.mark.parametrize("batch,q_len", [(1, 2), (1, 8), (3, 8), (1, 40), (2, 128), (1, 700), (16, 5), (1, 8192)])
def test_a_longer_calls_workspace_serves_shorter_chunks(dtype, hq, hkv, d, batch, q_len):
    """Several query rows: the size never falls as the keys grow, and no call
    needs more than it (nor more than the per-row kernels' partitions did)."""
    lib = _lib.load()
    group = next(g for g in (8, 4, 2, 1) if (hq // hkv) % g == 0)
    last = 0
    for n in sorted({*range(q_len, 9000, 61), *(128 * i + j for i in range(1, 70) for j in (0, 1)), 65536}):
        if n < q_len:
            continue
        p = _lib.AttendParams(dtype=dtype, batch=batch, q_len=q_len, q_heads=hq, kv_heads=hkv, head_dim=d, causal=1,
                              softmax_scale=1.0, q=256, cache=256, out=256, capacity=n, max_seqlen=n, seqlen_bias=n,
                              q_batch_stride=q_len * hq * d, q_row_stride=hq * d, out_batch_stride=q_len * hq * d,
                              out_row_stride=hq * d, cache_batch_stride=n * 2 * hkv * d, cache_pos_stride=2 * hkv * d,
                              cache_kv_stride=hkv * d)
        need = lib.hexkv_attend_workspace_bytes(p)
        assert need >= last, n
        last = need
        want = batch * q_len * (hq // group) * ((n + 1) // 2) // 2048
        part = next((s for s in (128, 256) if s >= want), 512)
        per_row = _lib.ATTEND_COUNTER_BYTES + batch * q_len * hq * -(-n // part) * (d + 2) * 4
        for size in (need, per_row):
            # a workspace that is large enough is then refused for its alignment
            rc = lib.hexkv_attend(p, 8, size, None)
            assert rc != _lib.HEXKV_EWORKSPACE and rc != 0, (n, size)


def _linear(lib, h, y, h_out, norm, w, out, rows=2, hidden=64, n=16, glu=0, stride=64):
    return lib.hexkv_norm_linear(h, stride, y, stride, h_out, stride, norm, 1e-5, w, out, rows, hidden, n, glu, 0, None)


def _rope_linear(lib, h, y, h_out, norm, w, q, kv, rows=2):
    return lib.hexkv_norm_rope_linear(h, 64, y, 64, h_out, 64, norm, 1e-5, w, 0x900000, None, 0, q, kv, rows, rows, 64,
                                      4, 2, 16, 0, None)


H, Y, S, N, W, O, K = (0x100000 * i for i in range(1, 8))  # 2 rows of 64 float16 elements: 256 bytes; W 8192 at most


@pytest.mark.skipif(torch.cuda.device_count() > 0, reason="accepted calls would run on made-up addresses")
@pytest.mark.parametrize("clash,call", [
    (False, lambda l: _linear(l, H, Y, S, N, W, O)),
    (True, lambda l: _linear(l, H, Y, H, N, W, O)),           # the sum over h
    (True, lambda l: _linear(l, H, Y, H + 128, N, W, O)),     # over h's second row
    (True, lambda l: _linear(l, H, Y, S, N, W, H)),           # out over h
    (True, lambda l: _linear(l, H, Y, S, N, W, Y, n=64)),     # out over y, as large
    (True, lambda l: _linear(l, H, None, None, N, W, H + 240)),
    (False, lambda l: _linear(l, H, None, None, N, W, H + 256)),
    (False, lambda l: _linear(l, H, None, None, N, W, H + 128, rows=1)),
    (True, lambda l: _linear(l, H, Y, S, N, W, S + 128)),     # out over the sum
    (True, lambda l: _linear(l, H, Y, S, N, W, N)),           # out over the norm's weight
    (True, lambda l: _linear(l, H, Y, S, N, W, W + 16 * 128 - 16)),
    (False, lambda l: _linear(l, H, Y, S, N, W, W + 16 * 128)),
    (True, lambda l: _linear(l, H, Y, S, N, W, W + 16 * 128, glu=1)),
    (False, lambda l: _linear(l, H, H + 128, H + 256, N, W, O, stride=192)),  # rows of one buffer, side by side
    (True, lambda l: _linear(l, H, H + 128, H + 192, N, W, O, stride=192)),
    (False, lambda l: _rope_linear(l, H, Y, S, N, W, O, K)),
    (True, lambda l: _rope_linear(l, H, Y, S, N, W, H, K)),
    (True, lambda l: _rope_linear(l, H, Y, S, N, W, O, Y + 16)),
    (True, lambda l: _rope_linear(l, H, Y, S, N, W, O, O + 128)),
    (True, lambda l: _rope_linear(l, H, Y, S, N, W, W + 8 * 16 * 128 - 16, K)),
    (False, lambda l: l.hexkv_add_rms_norm(H, 64, Y, 64, H, 64, N, Y, 2, 64, 1e-5, 0, None)),   # row for row
    (True, lambda l: l.hexkv_add_rms_norm(H, 64, Y, 64, H + 128, 64, N, O, 2, 64, 1e-5, 0, None)),
    (True, lambda l: l.hexkv_add_rms_norm(H, 128, Y, 64, None, 0, N, H, 2, 64, 1e-5, 0, None)),  # h's rows lie apart
    (False, lambda l: l.hexkv_add_rms_norm(H, 128, Y, 64, None, 0, N, H, 1, 64, 1e-5, 0, None)),
    (True, lambda l: l.hexkv_add_rms_norm(H, 64, Y, 64, None, 0, N, N, 2, 64, 1e-5, 0, None)),
    (True, lambda l: l.hexkv_add_rms_norm(H, 0, Y, 64, H, 0, N, O, 2, 64, 1e-5, 0, None)),      # one row for both
    (False, lambda l: l.hexkv_add_rms_norm(H, 0, Y, 64, None, 0, N, O, 2, 64, 1e-5, 0, None)),
    (False, lambda l: l.hexkv_rope_split(H, 128, 0x900000, None, 0, O, K, 2, 2, 4, 2, 16, 0, None)),
    (True, lambda l: l.hexkv_rope_split(H, 128, 0x900000, None, 0, H, K, 2, 2, 4, 2, 16, 0, None)),
    (False, lambda l: l.hexkv_rope_split(H, 128, 0x900000, None, 0, H, H + 128, 1, 1, 4, 2, 16, 0, None)),
    (True, lambda l: l.hexkv_rope_split(H, 128, 0x900000, None, 0, O, O + 128, 2, 2, 4, 2, 16, 0, None)),
    (False, lambda l: l.hexkv_silu_mul(H, H + 128, 1, 64, 0, None)),
    (True, lambda l: l.hexkv_silu_mul(H, H, 2, 64, 0, None)),
    (True, lambda l: l.hexkv_silu_mul(H, H + 64, 1, 64, 0, None)),
    (False, lambda l: l.hexkv_silu_mul(H, H + 512, 2, 64, 0, None))])
def test_overlapping_outputs_are_refused(clash, call):
    """Workgroups of the layer steps read whole inputs while others store."""
    lib = _lib.load()
    rc = call(lib)
    assert (rc == _lib.HEXKV_EINVAL) == clash, lib.hexkv_last_error()
    assert not clash or b"overlap" in lib.hexkv_last_error()


@pytest.mark.skipif(torch.cuda.device_count() > 0, reason="calls whose workspace fits would run on made-up addresses")
@pytest.mark.parametrize("dtype,d,batch,longest,part", [
    (0, 128, 8, 2048, 192), (1, 64, 16, 1537, 192), (2, 64, 16, 2048, 192),
    (0, 128, 8, 1536, 128),                           # rows too short
    (2, 128, 8, 2048, 128), (1, 256, 8, 2048, 128),   # heads of 512 bytes
    (0, 128, 1, 2048, 128)])                          # too small a call
def test_decode_partition(dtype, d, batch, longest, part):
    """The partition a decode call runs with, by the workspace it accepts (one
    that is large enough is then refused for its alignment)."""
    lib = _lib.load()
    heads = 8
    p = _lib.AttendParams(dtype=dtype, batch=batch, q_len=1, q_heads=heads, kv_heads=heads, head_dim=d, q=256, cache=256,
                          out=256, softmax_scale=1.0, capacity=longest, max_seqlen=longest, seqlen_bias=longest,
                          q_batch_stride=heads * d, out_batch_stride=heads * d,
                          cache_batch_stride=longest * 2 * heads * d, cache_pos_stride=2 * heads * d,
                          cache_kv_stride=heads * d)
    need = _lib.ATTEND_COUNTER_BYTES + batch * heads * -(-longest // part) * (d + 2) * 4
    assert lib.hexkv_attend(p, 8, need - 1, None) == _lib.HEXKV_EWORKSPACE
    assert lib.hexkv_attend(p, 8, need, None) == _lib.HEXKV_EINVAL
