"""hexkv_attend_layers: layers sharing a launch equal one call per layer, bit
for bit, and layers that must not share one (tensors that overlap, counters
or workspace too small) run in order."""
import pytest
import torch

from hexgen2_amd import _lib, ops

pytestmark = pytest.mark.gpu


def _graph(device, layers, lens, hq, hkv, d, dtype, out_layers, partition=0):
    g = torch.Generator(device=device).manual_seed(5)
    cap = max(lens) + 2
    cache = torch.randn((layers, len(lens), cap, 2, hkv, d), generator=g, device=device).to(dtype)
    q = torch.randn((layers, len(lens), 1, hq, d), generator=g, device=device).to(dtype)
    kv = torch.randn((layers, len(lens), 2, hkv, d), generator=g, device=device).to(dtype)
    want_cache, pos = cache.clone(), torch.tensor(lens, dtype=torch.int32, device=device)
    ops.decode_attention(q[0], cache[0].clone(), max_seqlen=max(lens) + 1, seqlens=pos, kv_new=kv[0], lens=lens)
    out = torch.zeros((out_layers, len(lens), 1, hq, d), dtype=dtype, device=device)
    graph = ops.DecodeStepGraph(q, cache, [out[l % out_layers] for l in range(layers)], kv, pos, max(lens) + 1, lens=lens,
                                partition=partition)
    kernel = {v: k for k, v in _lib.KERNELS.items()}[graph.lists.kernels[0]]
    want = [ops.decode_attention(q[l], want_cache[l], max_seqlen=max(lens) + 1, seqlens=pos, kv_new=kv[l], lens=lens,
                                 kernel=kernel, partition=graph.lists.chunks[0]) for l in range(layers)]
    for _ in range(3):  # each replay from the same lengths, with eager work between
        pos.copy_(torch.tensor(lens, dtype=torch.int32, device=device))
        out.zero_()
        graph.restart()
        graph.replay()
        torch.cuda.synchronize()
        assert pos.tolist() == [n + 1 for n in lens]
        assert torch.equal(cache, want_cache)
        for l in range(layers - out_layers, layers):
            assert torch.equal(out[l % out_layers], want[l]), f"layer {l}"
    assert ops.device_status() & _lib.STATUS_ERRORS == 0
    return graph


def _sharing(graph):
    p, table = graph.plan.params, graph.plan.layers[1]
    graph.lists[0].apply(p)
    lib = _lib.load()
    one = int(lib.hexkv_attend_workspace_bytes(p))
    return (int(lib.hexkv_attend_layers_workspace_bytes(p, table, len(table))) - _lib.ATTEND_COUNTER_BYTES) \
        // max(one - _lib.ATTEND_COUNTER_BYTES, 1)


@pytest.mark.parametrize("layers", [1, 2, 7])
@pytest.mark.parametrize("hq,hkv,d,dtype,lens", [
    (8, 1, 128, torch.bfloat16, [600, 1, 4000, 0, 129]),
    (32, 8, 128, torch.bfloat16, [3000, 40, 2500, 4029, 2800, 4000, 12, 3900]),  # the row-block kernel
    (4, 4, 16, torch.float32, [5, 700])])
def test_layers_share_launches(device, layers, hq, hkv, d, dtype, lens):
    graph = _graph(device, layers, lens, hq, hkv, d, dtype, layers)
    assert _sharing(graph) == layers


def test_layers_with_one_output_run_in_order(device):
    assert _sharing(_graph(device, 4, [900, 33], 8, 1, 128, torch.bfloat16, 1)) == 1


def test_layers_beyond_the_counters_or_the_workspace(device):
    # 20 rows x 32 heads: 640 segments (one row of 4 pieces, the others of 1) a layer, 51 layers' worth of counters
    lens = [60] * 19 + [200]
    graph = _graph(device, 55, lens, 32, 32, 16, torch.float32, 55, partition=64)
    assert _sharing(graph) == _lib.ATTEND_COUNTER_WORDS // 640 == 51
    # the least workspace (one layer's) gives the same results, one launch each
    plan, pos = graph.plan, graph.positions
    pos.copy_(torch.tensor(lens, dtype=torch.int32, device=device))
    plan.fix_work_list(graph.lists[0])
    want = [o.clone() for o in graph.out]
    for o in graph.out:
        o.zero_()
    plan.ws_bytes = int(_lib.load().hexkv_attend_workspace_bytes(plan.params))
    plan.call_layers(0, graph.max_seqlen, pos)
    torch.cuda.synchronize()
    assert all(torch.equal(a, b) for a, b in zip(graph.out, want))
