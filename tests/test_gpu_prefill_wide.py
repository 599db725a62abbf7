"""GPU: the wide 128-row prefill form (direct loads into LDS, two weight sets a
wave) against the narrow one, bit for bit, and the float64 oracle: rows per
expert around its 32-row blocks and 128-row tiles, reductions of one scale
block (8 groups) and more, absent experts, dropped ids, and an output that is
not 16-byte aligned."""

import ctypes

import numpy as np
import pytest
import torch

from oracle import pmoe_oracle as O
from tests.test_gpu_stream import _ids, _setup
from tests.util import bits_to_bf16_tensor, check_close

pytestmark = pytest.mark.gpu

DEV = "cuda"


def _wide(g, slab, x, n, k, e):
    from pagedmoe_amd._lib import lib
    return lib().pmoe_prefill_wide(ctypes.byref(g), slab.data_ptr, x.data_ptr(), n, k, e)


COUNTS = [300, 129, 128, 127, 97, 96, 1, 31, 32, 33, 64, 65, 90]


@pytest.mark.parametrize("hidden,inter,bits", [(1024, 512, 4), (2048, 1536, 4), (512, 1024, 4),
                                               (4096, 512, 4), (1024, 512, 6), (2048, 1536, 6),
                                               (4096, 1024, 6), (7168, 2048, 4), (1024, 2048, 6)])
def test_wide_matches_narrow_and_oracle(hidden, inter, bits, monkeypatch):
    from pagedmoe_amd import kernels as K
    monkeypatch.setenv("PMOE_STREAM", "0")
    monkeypatch.setenv("PMOE_PREFILL_SMALL", "0")
    n, k, e = 330, 4, len(COUNTS)
    g, slab, experts = _setup(hidden, inter, bits, e, 60)
    rng = np.random.default_rng(hidden + inter)
    xb = O.bf16_round(rng.standard_normal((n, hidden), dtype=np.float32))
    ids = _ids(COUNTS, k, rng, n)
    table = torch.arange(e, dtype=torch.int32, device=DEV)
    table[12] = -1
    x, inds = bits_to_bf16_tensor(xb, DEV), torch.from_numpy(ids).to(DEV)
    got = []
    for pin in ("0", "1"):
        monkeypatch.setenv("PMOE_PREFILL_WIDE", pin)
        assert _wide(g, slab, x, n, k, e) == int(pin)
        got.append(K.switch_glu(g, slab.buf, table, e, x, inds))
    assert torch.equal(got[0].view(torch.int16), got[1].view(torch.int16))
    y = got[1].float().cpu().numpy()
    gone = (ids < 0) | (ids == 12)
    assert (y[gone] == 0).all()
    ref = O.switch_glu_f64(xb, np.where(gone, 0, ids), experts)
    check_close(y[~gone], ref[~gone], f"wide {hidden}x{inter} {bits}-bit")
    # unaligned output rows take the element-wise stores
    big = torch.full((n * k * hidden + 8,), float("nan"), dtype=torch.bfloat16, device=DEV)
    un = big[1:1 + n * k * hidden]
    from pagedmoe_amd._lib import check, lib
    ws = K.moe_workspace(g, n, k, 0, e, x.device)
    check(lib().pmoe_switch_glu(ctypes.byref(g), K._ptr(slab.buf), K._table_ptr(table), e,
                                K._ptr(x), K._ptr(inds), n, k, ctypes.c_void_p(un.data_ptr()),
                                K._ptr(ws), ws.numel(), K._stream()), "pmoe_switch_glu")
    torch.cuda.synchronize()
    assert torch.equal(got[1].reshape(-1).view(torch.int16), un.view(torch.int16))
    assert torch.isnan(big[0]) and torch.isnan(big[-7:]).all()
    slab.release()


@pytest.mark.parametrize("bits", [4, 6])
def test_unaligned_activations(bits, monkeypatch):
    """x at a 2-byte offset (the narrow form) gives the aligned call's bits."""
    from pagedmoe_amd import kernels as K
    monkeypatch.setenv("PMOE_STREAM", "0")
    monkeypatch.setenv("PMOE_PREFILL_SMALL", "0")
    monkeypatch.setenv("PMOE_PREFILL_WIDE", "1")
    n, k, e, hidden = 330, 4, len(COUNTS), 1024
    g, slab, _ = _setup(hidden, 512, bits, e, 63)
    rng = np.random.default_rng(64)
    xb = O.bf16_round(rng.standard_normal((n, hidden), dtype=np.float32))
    inds = torch.from_numpy(_ids(COUNTS, k, rng, n)).to(DEV)
    table = torch.arange(e, dtype=torch.int32, device=DEV)
    x = bits_to_bf16_tensor(xb, DEV)
    un = torch.empty(n * hidden + 8, dtype=torch.bfloat16, device=DEV)[1:1 + n * hidden]
    un = un.view(n, hidden).copy_(x)
    assert x.data_ptr() % 16 == 0 and un.data_ptr() % 16 == 2
    assert _wide(g, slab, x, n, k, e) == 1 and _wide(g, slab, un, n, k, e) == 0
    y, yu = (K.switch_glu(g, slab.buf, table, e, t, inds) for t in (x, un))
    assert torch.equal(y.view(torch.int16), yu.view(torch.int16))
    slab.release()


@pytest.mark.parametrize("bits", [4, 6])
def test_components_in_another_order(bits, monkeypatch):
    """Slots whose components lie in the reverse order (down first, gate last):
    the bits of the usual layout."""
    from pagedmoe_amd import kernels as K
    from pagedmoe_amd._lib import geom
    monkeypatch.setenv("PMOE_STREAM", "0")
    monkeypatch.setenv("PMOE_PREFILL_SMALL", "0")
    monkeypatch.setenv("PMOE_PREFILL_WIDE", "1")
    n, k, e, hidden = 330, 4, len(COUNTS), 1024
    g, slab, _ = _setup(hidden, 512, bits, e, 65)
    r, at = geom(hidden, 512, bits), 0
    for c in reversed(range(9)):
        r.off[c] = at
        at += -(-g.nbytes[c] // 256) * 256
    src = slab.buf.view(e, g.expert_bytes)
    dst = torch.empty_like(src)
    for c in range(9):
        dst[:, r.off[c]:r.off[c] + g.nbytes[c]] = src[:, g.off[c]:g.off[c] + g.nbytes[c]]
    rng = np.random.default_rng(66)
    x = bits_to_bf16_tensor(O.bf16_round(rng.standard_normal((n, hidden), dtype=np.float32)), DEV)
    inds = torch.from_numpy(_ids(COUNTS, k, rng, n)).to(DEV)
    table = torch.arange(e, dtype=torch.int32, device=DEV)
    assert _wide(g, slab, x, n, k, e) == 1 and _wide(r, slab, x, n, k, e) == 0
    y = K.switch_glu(g, slab.buf, table, e, x, inds)
    yr = K.switch_glu(r, dst.view(-1), table, e, x, inds)
    assert torch.equal(y.view(torch.int16), yr.view(torch.int16))
    slab.release()


def test_wide_block_in_a_graph(monkeypatch):
    """The whole block in the wide form, replayed from a HIP graph."""
    from pagedmoe_amd import kernels as K
    monkeypatch.setenv("PMOE_PREFILL_WIDE", "1")
    g, slab, _ = _setup(1024, 512, 4, 8, 61)
    rng = np.random.default_rng(62)
    gw = bits_to_bf16_tensor(O.bf16_round(rng.standard_normal((8, 1024), dtype=np.float32)
                                          * np.float32(0.02)), DEV)
    x = bits_to_bf16_tensor(O.bf16_round(rng.standard_normal((520, 1024), dtype=np.float32)), DEV)
    table = torch.arange(8, dtype=torch.int32, device=DEV)
    rc = K.route_cfg("softmax", 8, 2)
    assert _wide(g, slab, x, 520, 2, 8) == 1
    eager = K.moe_block(g, rc, slab.buf, table, gw, x)[0].clone()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        out, _, _ = K.moe_block(g, rc, slab.buf, table, gw, x)
    for _ in range(3):
        out.zero_()
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(out.view(torch.int16), eager.view(torch.int16))
    slab.release()
