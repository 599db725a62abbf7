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


def _streamed(g, n, kk, e, shared=0):
    """The rule that the call itself asks."""
    from pagedmoe_amd._lib import lib
    return lib().pmoe_stream_wanted(ctypes.byref(g), n, kk, e, shared) == 1


def _run(K, g, slab, table, n_experts, xb, ids):
    return K.switch_glu(g, slab.buf, table, n_experts, bits_to_bf16_tensor(xb, DEV),
                        torch.from_numpy(ids).to(DEV))


@pytest.mark.parametrize("hidden,inter,bits", [
    (1024, 512, 4), (1024, 512, 6), (2048, 512, 6), (2048, 1536, 4), (4096, 1536, 4),
    (4096, 1024, 6), (1536, 2048, 6), (7168, 2048, 4),
    # uneven cuts: last slices that overlap the one before, or repeat it whole
    (384, 640, 4), (384, 640, 6), (1408, 896, 4), (1408, 896, 6), (2560, 1152, 4),
    (2560, 1152, 6), (3072, 768, 6), (5120, 768, 4), (5376, 384, 4), (6400, 2304, 4),
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
    assert _streamed(g, n, k, e) and "prefill_gateup" in kt.result, kt.result
    assert "qgemv_gateup" not in kt.result, kt.result
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


@pytest.mark.parametrize("n", [7, 75])
@pytest.mark.parametrize("bits,hidden,inter", [(4, 1024, 512), (6, 1024, 512), (4, 7168, 512)])
def test_stream_huge_activations(bits, hidden, inter, n, monkeypatch):
    """(128 + q) x and 128 s sum(x) of a huge or infinite x leave fp32 where
    (s q + b) x does not.  Finite rows: a 3e38 against weights of ~1e-20 stays
    finite, within tests/util's tolerance.  Infinite ones: NaN and the two
    infinities where float64 has them (weights of one sign: infinities; both
    signs: NaN).  A NaN spoils its own row only, and every other row keeps its
    bits."""
    from pagedmoe_amd import kernels as K
    from pagedmoe_amd._lib import geom
    from pagedmoe_amd.slab import SlabStore
    monkeypatch.setenv("PMOE_STREAM", "1")
    g = geom(hidden, inter, bits)
    table = torch.arange(2, dtype=torch.int32, device=DEV)
    rng = np.random.default_rng(97)
    ids = np.stack([rng.permutation(2) for _ in range(n)]).astype(np.int32)
    for std, positive, values in ((1e-20, False, {1: 3e38, 5: -1e36}),
                                  (0.02, True, {2: np.inf, 6: np.nan}),
                                  (0.02, False, {0: np.inf, 3: np.nan, 4: -np.inf})):
        slab = SlabStore(g, 2, DEV)
        gen = torch.Generator(device=DEV).manual_seed(98)
        for slot in range(2):
            for proj, rows, cols in (("gate_proj", inter, hidden), ("up_proj", inter, hidden),
                                     ("down_proj", hidden, inter)):
                w = torch.randn((rows, cols), generator=gen, device=DEV) * std
                slab.quantize_into(slot, proj, w.abs() if positive else w)
        plain = rng.standard_normal((n, hidden)).astype(np.float32)
        odd = plain.copy()
        for row, v in values.items():
            odd[row, 7 * row + 3] = v
        bits_of = [O.bf16_round(a) for a in (plain, odd)]
        base, y = (_run(K, g, slab, table, 2, xb, ids).float().cpu().numpy() for xb in bits_of)
        rest = [i for i in range(n) if i not in values]
        assert np.array_equal(base[rest].view(np.int32), y[rest].view(np.int32))
        rows = sorted(values)
        with np.errstate(all="ignore"):
            ref = O.switch_glu_f64(bits_of[1][rows], ids[rows], [slot_to_expert(slab, e)
                                                                 for e in range(2)])
        for i, row in enumerate(rows):
            if np.isfinite(values[row]):
                check_close(y[row], ref[i], f"row of {values[row]}")
            else:
                for same in (np.isnan, np.isposinf, np.isneginf):
                    assert np.array_equal(same(y[row]), same(ref[i])), (values[row], same)
        slab.release()


@pytest.mark.parametrize("n", [12, 13])
def test_stream_block_huge_activations(n, monkeypatch):
    """The block path's fp32 rows of a 3e38 against weights of ~1e-20."""
    from pagedmoe_amd import kernels as K
    from pagedmoe_amd._lib import geom
    from pagedmoe_amd.slab import SlabStore
    monkeypatch.setenv("PMOE_STREAM", "1")
    g = geom(1024, 512, 4)
    slab = SlabStore(g, 2, DEV)
    fill_slab_gpu(slab, range(2), seed=103, std=1e-20)
    xb = np.random.default_rng(104).standard_normal((n, 1024)).astype(np.float32)
    xb[4, 100] = 3e38
    xb = O.bf16_round(xb)
    gate = torch.zeros((2, 1024), dtype=torch.bfloat16, device=DEV)
    out, ids, w = K.moe_block(g, K.route_cfg("softmax", 2, 2), slab.buf,
                              torch.arange(2, dtype=torch.int32, device=DEV), gate,
                              bits_to_bf16_tensor(xb, DEV))
    ids, w = ids.cpu().numpy(), w.cpu().numpy()
    assert (w == 0.5).all()
    with np.errstate(over="ignore"):  # exp of a hugely negative gate
        ref = O.combine_f64(O.switch_glu_f64(xb[4:5], ids[4:5], [slot_to_expert(slab, e)
                                                                for e in range(2)]), w[4:5])
    check_close(out[4:5].float().cpu().numpy(), ref, "huge row of a block")
    slab.release()


# the block path's workspace starts with this synchronisation header (pmoe.h)
HEADER = 1_352_960


@pytest.mark.parametrize("n", [2, 12, 13, 28])
@pytest.mark.parametrize("shape", [(1024, 512, 4), (1024, 512, 6), (2048, 768, 4)])
@pytest.mark.parametrize("form", ["softmax", "softmax-shared", "sigmoid", "sigmoid-shared"])
def test_stream_block_forms(form, shape, n, monkeypatch):
    """Routing on both sides of its 12-token line (the router launch's last
    block, a launch of its own), softmax and grouped sigmoid, with an ungated
    shared expert and without one, and the busiest expert absent: its rows are
    written as fp32 zeros, over scratch left full of NaN."""
    from pagedmoe_amd import kernels as K
    monkeypatch.setenv("PMOE_STREAM", "1")
    hidden, inter, bits = shape
    scoring, shared = form.split("-")[0], int(form.endswith("shared"))
    e, k = 32, 6
    sig = dict(scoring="sigmoid", n_group=8, topk_group=4, routed_scale=2.5)
    spec = O.LayerSpec(hidden, e, inter, k, bits=bits, shared=shared,
                       **(sig if scoring == "sigmoid" else {}))
    g, slab, experts = _setup(hidden, inter, bits, e + shared, 101)
    rng = np.random.default_rng(102 + n)
    gw = O.bf16_round(rng.standard_normal((e, hidden), dtype=np.float32) * np.float32(0.02))
    bias = rng.standard_normal(e, dtype=np.float32) * np.float32(0.05)
    xb = O.bf16_round(rng.standard_normal((n, hidden), dtype=np.float32))
    ref_i, ref_w, y, _ = O.moe_layer_f64(spec, xb, gw, experts, bias=bias)
    gone = int(np.bincount(ref_i.reshape(-1)).argmax())
    y[ref_i == gone] = 0.0
    ref = O.combine_f64(y, ref_w,
                        O.expert_ffn_f64(O.bf16_to_f32(xb), experts[e]) if shared else None)
    table = torch.arange(e, dtype=torch.int32, device=DEV)
    table[gone] = -1
    rc = (K.route_cfg("sigmoid", e, k, True, 8, 4, 2.5) if scoring == "sigmoid"
          else K.route_cfg("softmax", e, k))
    x = bits_to_bf16_tensor(xb, DEV)
    assert _streamed(g, n, k + shared, e, shared)
    K.moe_workspace(g, n, k, shared, e, x.device)[HEADER:].fill_(255)
    out, gi, gwt = K.moe_block(g, rc, slab.buf, table, bits_to_bf16_tensor(gw, DEV), x,
                               score_bias=torch.from_numpy(bias).to(DEV)
                               if scoring == "sigmoid" else None,
                               shared_slot=e if shared else -1)
    assert np.array_equal(gi.cpu().numpy(), ref_i) and np.array_equal(gwt.cpu().numpy(), ref_w)
    check_close(out.float().cpu().numpy(), ref, f"{form} n={n}")
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
