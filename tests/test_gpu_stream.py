"""GPU: the streamed expert tiles (few rows per expert, stream.hip) against the
float64 oracle, at the sizes where their tiling can go wrong: every cut of a
reduction the path takes, rows per expert around its 16- and 32-row tiles,
absent experts, dropped ids, an output that is not 16-byte aligned, and the
block path's fp32 per-slot rows.  The tolerance is tests/util's, which the bf16
rounding of h sets; everything else in the path is fp32.
"""

import ctypes

import numpy as np
import pytest
import torch

from oracle import pmoe_oracle as O
from tests.util import bits_to_bf16_tensor, check_close, fill_slab_gpu, slot_to_expert

pytestmark = pytest.mark.gpu

DEV = "cuda"


def _setup(hidden, inter, bits, experts, seed):
    from pagedmoe_amd._lib import geom
    from pagedmoe_amd.slab import SlabStore
    g = geom(hidden, inter, bits)
    slab = SlabStore(g, experts, DEV)
    fill_slab_gpu(slab, range(experts), seed=seed)
    return g, slab, [slot_to_expert(slab, e) for e in range(experts)]


def _ids(counts, k, rng, n):
    """[n, k] ids (distinct per token, -1 where none is left) with the given
    rows per expert."""
    ids = np.full((n, k), -1, np.int32)
    for e, c in enumerate(counts):
        free = [t for t in range(n) if (ids[t] < 0).any()]
        for t in rng.choice(free, c, replace=False):
            ids[t, np.flatnonzero(ids[t] < 0)[0]] = e
    return ids


def _run(K, g, slab, table, n_experts, xb, ids):
    return K.switch_glu(g, slab.buf, table, n_experts, bits_to_bf16_tensor(xb, DEV),
                        torch.from_numpy(ids).to(DEV))


@pytest.mark.parametrize("hidden,inter,bits", [
    (1024, 512, 4), (1024, 512, 6), (2048, 512, 6), (2048, 1536, 4), (4096, 1536, 4),
    (4096, 1024, 6), (1536, 2048, 6), (7168, 2048, 4),
])
def test_stream_seam_vs_oracle(hidden, inter, bits, monkeypatch):
    """Rows per expert 1, 15, 16, 17, 31, 32, 33, 70 and one absent expert;
    every row against the oracle, dropped and absent ones exact zeros."""
    from pagedmoe_amd import kernels as K
    from pagedmoe_amd._lib import KernelTimer
    monkeypatch.setenv("PMOE_STREAM", "1")
    counts = [1, 15, 16, 17, 31, 32, 33, 70, 20]
    n, k, e = 80, 4, len(counts)
    g, slab, experts = _setup(hidden, inter, bits, e, 80 + bits)
    rng = np.random.default_rng(hidden + inter)
    xb = O.bf16_round(rng.standard_normal((n, hidden), dtype=np.float32))
    ids = _ids(counts, k, rng, n)
    table = torch.arange(e, dtype=torch.int32, device=DEV)
    table[8] = -1
    with KernelTimer() as kt:
        y = _run(K, g, slab, table, e, xb, ids).float().cpu().numpy()
    assert "prefill_gateup" in kt.result and "gateup" not in kt.result, kt.result
    gone = (ids < 0) | (ids == 8)
    assert (y[gone] == 0).all()
    ref = O.switch_glu_f64(xb, np.where(gone, 0, ids), experts)
    check_close(y[~gone], ref[~gone], f"stream {hidden}x{inter} {bits}-bit")
    slab.release()


def test_stream_unaligned_output_matches_aligned(monkeypatch):
    from pagedmoe_amd import kernels as K
    from pagedmoe_amd._lib import check, lib
    monkeypatch.setenv("PMOE_STREAM", "1")
    n, k, e, hidden = 37, 2, 4, 1024
    g, slab, _ = _setup(hidden, 512, 4, e, 90)
    rng = np.random.default_rng(91)
    x = bits_to_bf16_tensor(O.bf16_round(rng.standard_normal((n, hidden), dtype=np.float32)), DEV)
    inds = torch.from_numpy(np.stack([rng.choice(e, k, replace=False) for _ in range(n)])
                            .astype(np.int32)).to(DEV)
    table = torch.arange(e, dtype=torch.int32, device=DEV)
    y = K.switch_glu(g, slab.buf, table, e, x, inds)
    big = torch.full((n * k * hidden + 8,), float("nan"), dtype=torch.bfloat16, device=DEV)
    un = big[1:1 + n * k * hidden]
    ws = K.moe_workspace(g, n, k, 0, e, x.device)
    check(lib().pmoe_switch_glu(ctypes.byref(g), K._ptr(slab.buf), K._table_ptr(table), e,
                                K._ptr(x), K._ptr(inds), n, k, ctypes.c_void_p(un.data_ptr()),
                                K._ptr(ws), ws.numel(), K._stream()), "pmoe_switch_glu")
    torch.cuda.synchronize()
    assert torch.equal(y.reshape(-1).view(torch.int16), un.view(torch.int16))
    assert torch.isnan(big[0]) and torch.isnan(big[-7:]).all()
    slab.release()


@pytest.mark.parametrize("bits", [4, 6])
def test_stream_components_in_arrays_of_their_own(bits, monkeypatch):
    """A slab of one array a component over all experts (components beyond the
    slot's stride) gives what the usual layout gives on the same path."""
    from pagedmoe_amd import kernels as K
    from pagedmoe_amd._lib import geom
    n, k, e, hidden = 37, 2, 4, 1024
    g, slab, _ = _setup(hidden, 512, bits, e, 92)
    src = slab.buf.view(e, g.expert_bytes)
    r, at = geom(hidden, 512, bits), 0
    # every expert's gate weights, then every expert's up weights, ...: the
    # stride of the largest component serves all
    r.expert_bytes = max(g.nbytes)
    dst = torch.empty(9 * e * r.expert_bytes, dtype=torch.uint8, device=DEV)
    for c in range(9):
        r.off[c] = at
        rows = dst[at:at + e * r.expert_bytes].view(e, r.expert_bytes)
        rows[:, :g.nbytes[c]] = src[:, g.off[c]:g.off[c] + g.nbytes[c]]
        at += e * r.expert_bytes
    rng = np.random.default_rng(93)
    x = bits_to_bf16_tensor(O.bf16_round(rng.standard_normal((n, hidden), dtype=np.float32)), DEV)
    inds = torch.from_numpy(np.stack([rng.choice(e, k, replace=False) for _ in range(n)])
                            .astype(np.int32)).to(DEV)
    table = torch.arange(e, dtype=torch.int32, device=DEV)
    monkeypatch.setenv("PMOE_STREAM", "0")
    y = K.switch_glu(g, slab.buf, table, e, x, inds)
    monkeypatch.setenv("PMOE_STREAM", "1")
    yr = K.switch_glu(r, dst, table, e, x, inds)
    assert torch.equal(y.view(torch.int16), yr.view(torch.int16))
    slab.release()


@pytest.mark.parametrize("bits,n", [(4, 2), (4, 12), (4, 13), (4, 17), (6, 50)])
def test_stream_block_vs_oracle(bits, n, monkeypatch):
    """The whole block with a gated shared expert (its rows are every token:
    at 50 tokens two tiles), eager and replayed from a HIP graph."""
    from pagedmoe_amd import kernels as K
    monkeypatch.setenv("PMOE_STREAM", "1")
    spec = O.LayerSpec(1024, 32, 512, 4, bits=bits, shared=1, shared_gate=True)
    g, slab, experts = _setup(1024, 512, bits, 33, 95)
    rng = np.random.default_rng(96 + n)
    gw = O.bf16_round(rng.standard_normal((32, 1024), dtype=np.float32) * np.float32(0.02))
    sg = O.bf16_round(rng.standard_normal((1, 1024), dtype=np.float32) * np.float32(0.02))
    xb = O.bf16_round(rng.standard_normal((n, 1024), dtype=np.float32))
    table = torch.arange(32, dtype=torch.int32, device=DEV)
    rc = K.route_cfg("softmax", 32, spec.top_k)
    args = (g, rc, slab.buf, table, bits_to_bf16_tensor(gw, DEV), bits_to_bf16_tensor(xb, DEV))
    kw = dict(shared_slot=32, shared_gate=bits_to_bf16_tensor(sg, DEV))
    out, gi, gwt = K.moe_block(*args, **kw)
    ref_i, ref_w = O.softmax_topk(O.router_logits(xb, gw), spec.top_k)
    assert np.array_equal(gi.cpu().numpy(), ref_i) and np.array_equal(gwt.cpu().numpy(), ref_w)
    gate = 1.0 / (1.0 + np.exp(-O.router_logits(xb, sg)[:, 0].astype(np.float64)))
    shared = O.expert_ffn_f64(O.bf16_to_f32(xb), experts[32]) * gate[:, None]
    ref = O.combine_f64(O.switch_glu_f64(xb, ref_i, experts), ref_w, shared)
    check_close(out.float().cpu().numpy(), ref, f"stream block n={n} {bits}-bit")
    eager = out.clone()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        gout, _, _ = K.moe_block(*args, **kw)
    for _ in range(3):
        gout.zero_()
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(gout.view(torch.int16), eager.view(torch.int16))
    slab.release()
