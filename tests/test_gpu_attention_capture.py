"""Paged decode attention in captured graphs.

A graph fixes the grid, the most chunks per segment and the scratch's address;
whether and how a table is cut is decided from its contents in every replay,
in the attention and in the combining kernel apart.  One graph is replayed
while the lengths go from whole segments to split ones, other chunk counts,
empty and short requests and back, its scratch shared by two layers (the
graph's pool hands it to the second after the first), and every replay is
compared with the eager calls, bit for bit, and with the oracle.

A capture that torch did not begin gets no scratch from torch.
"""
import ctypes

import numpy as np
import pytest
import torch

import workloads as W
from oracle import vortex_oracle as O
from vortex_torch import _hip

pytestmark = pytest.mark.gpu


def _bits(t):
    return t.detach().contiguous().cpu().view(torch.int16).numpy().view(np.uint16)


def _step(ic, b, qs, k, v, outs):
    from vortex_torch.decode_attention import dense_decode_attention
    from vortex_torch.indexer.utils_sglang import plan_decode

    plan_decode(b.seq_lens, b.req_to_token, b.req_indices, ic)
    for q, o in zip(qs, outs):
        dense_decode_attention(q, k, v, ic, out=o)


# requests' greatest lengths and the replays' lengths: a few segments, split
# from 520 tokens on average; many, split only where uneven
_FEW = ([6000, 4000, 3000], 2, [[100, 40, 1], [6000, 4000, 3000], [900, 700, 16], [3000, 0, 17], [0, 0, 0],
                                [5999, 3985, 1], [64, 4000, 16], [100, 40, 1]])
_MANY = ([9000] * 18, 8, [[700] * 18, [9000, 8000] + [3000 + 16 * i for i in range(16)], [3500] * 18,
                          [9000] + [0] * 8 + [5000] * 9, [33] * 18, [9000 - 499 * i for i in range(18)]])


@pytest.mark.parametrize("G,D", [(2, 128), (4, 128), (1, 64), (2, 256)])
@pytest.mark.parametrize("requests", ["few", "many"])
def test_replays_follow_the_table(gpu, requests, G, D):
    lens, H, replays = _FEW if requests == "few" else _MANY
    pool = sum((n + 15) // 16 for n in lens) + 3
    batch = W.make_batch(lens, pool_pages=pool, seed=61, num_kv_heads=H, group_size=G, head_dim=D)
    ic, _ = W.make_contexts(batch, gpu)
    b = batch.to(gpu)
    k = W.randn_bf16((pool * H, 16, D), 1, gpu)
    v = W.randn_bf16((pool * H, 16, D), 2, gpu)
    qs = [W.randn_bf16((len(lens) * H, G, D), 3 + i, gpu) for i in range(2)]
    outs, eager = ([torch.zeros_like(q) for q in qs] for _ in range(2))
    side = torch.cuda.Stream(gpu)
    side.wait_stream(torch.cuda.current_stream(gpu))
    with torch.cuda.stream(side):
        _step(ic, b, qs, k, v, outs)
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph, stream=side):
        _step(ic, b, qs, k, v, outs)
    lib = _hip.load_library()
    floats = lib.vtx_paged_decode_attention_workspace_len(len(lens), H, G, D, 16, ic.dense_kv_indices.numel())
    assert floats > 0
    kb, vb = _bits(k), _bits(v)
    for i, now in enumerate(replays):
        b.seq_lens.copy_(torch.tensor(now, dtype=torch.int32))
        for o in outs + eager:
            o.fill_(9.0)
        junk = torch.full((floats,), float("nan"), device=gpu)  # (what eager scratch is made of)
        torch.cuda.synchronize()
        del junk
        graph.replay()
        torch.cuda.synchronize()
        _step(ic, b, qs, k, v, eager)
        for j, (o, e) in enumerate(zip(outs, eager)):
            assert torch.equal(o.view(torch.int16), e.view(torch.int16)), f"replay {i}, layer {j}"
        if requests == "few" or i == 1:
            exp = O.paged_decode_attention(_bits(qs[1]), kb, vb, ic.dense_kv_indptr.cpu().numpy(),
                                           ic.dense_kv_indices.cpu().numpy(), ic.kv_last_page_len.cpu().numpy(),
                                           len(lens), H, 1.0 / np.sqrt(D))
            # the result's bf16 rounding
            np.testing.assert_allclose(O.bf16_to_f32(_bits(outs[1])).reshape(-1, D), O.bf16_to_f32(exp),
                                       rtol=2 ** -7, atol=1e-4)


def _hip_runtime():
    with open("/proc/self/maps") as f:
        path = next(line.split()[-1] for line in f if "libamdhip64" in line)
    return ctypes.CDLL(path)


def test_capture_that_torch_did_not_begin_takes_no_memory(gpu):
    """The call allocates nothing in it, and its replays give what the C entry
    without a workspace gives, bit for bit, whatever torch's free memory was
    handed out for in between."""
    from vortex_torch.decode_attention import paged_decode_attention

    G, D, P, n = 2, 128, 16, 300
    k = W.randn_bf16((2 * n, P, D), 1, gpu)
    v = W.randn_bf16((2 * n, P, D), 2, gpu)
    q = W.randn_bf16((2, G, D), 3, gpu)
    o, whole = torch.zeros_like(q), torch.zeros_like(q)
    ip = torch.tensor([0, n, 2 * n], dtype=torch.int32, device=gpu)
    idx = torch.randperm(2 * n, device=gpu).to(torch.int32)
    last = torch.tensor([P, 3], dtype=torch.int32, device=gpu)
    lib, rt = _hip.load_library(), _hip_runtime()
    assert lib.vtx_paged_decode_attention_workspace_len(2, 1, G, D, P, idx.numel()) > 0
    other = paged_decode_attention(q, k, v, ip, idx, last, 2, 1)  # (a first call outside any capture)
    rc = lib.vtx_paged_decode_attention(q.data_ptr(), whole.data_ptr(), k.data_ptr(), v.data_ptr(), k.shape[0],
                                        ip.data_ptr(), idx.data_ptr(), idx.numel(), last.data_ptr(), 2, 1, G, D, P,
                                        1.0 / np.sqrt(D), torch.cuda.current_stream().cuda_stream)
    assert rc == 0
    side = torch.cuda.Stream(gpu)
    side.wait_stream(torch.cuda.current_stream(gpu))
    torch.cuda.synchronize()
    stream = ctypes.c_void_p(side.cuda_stream)
    graph, run = ctypes.c_void_p(), ctypes.c_void_p()
    with torch.cuda.stream(side):
        before = torch.cuda.memory_stats()["allocation.all.allocated"]
        assert rt.hipStreamBeginCapture(stream, 2) == 0  # relaxed
        try:
            paged_decode_attention(q, k, v, ip, idx, last, 2, 1, out=o)
        finally:
            assert rt.hipStreamEndCapture(stream, ctypes.byref(graph)) == 0
        assert torch.cuda.memory_stats()["allocation.all.allocated"] == before
    assert rt.hipGraphInstantiate(ctypes.byref(run), graph, None, None, ctypes.c_size_t(0)) == 0
    for _ in range(3):
        o.zero_()
        torch.cuda.synchronize()
        assert rt.hipGraphLaunch(run, stream) == 0
        torch.cuda.synchronize()
        assert torch.equal(o, whole)
        del other
        other = torch.full((1 << 20,), 7.0, device=gpu)
    assert rt.hipGraphExecDestroy(run) == 0 and rt.hipGraphDestroy(graph) == 0
