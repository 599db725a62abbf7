"""Where the streamed expert tiles (stream.hip) take over from the decode GEMV
and hand over to the prefill GEMMs: token counts on both sides of each line of
the rule, per shape.  Host code only.
"""

import ctypes

import pytest


@pytest.mark.parametrize("hidden,inter,bits,e,kk,form", [
    (4096, 1536, 4, 128, 8, {11: 0, 12: 1, 255: 1, 512: 1, 513: 0}),
    (2048, 512, 6, 512, 11, {15: 0, 16: 1, 1489: 1, 1490: 0}),
    (7168, 2048, 4, 384, 9, {1: 0, 2: 1, 684: 1, 685: 0}),
    (1024, 512, 4, 32, 4, {37: 0, 38: 1, 255: 1, 256: 0}),
    (1024, 768, 4, 32, 4, {64: 0}),
])
def test_stream_rule(hidden, inter, bits, e, kk, form, monkeypatch):
    for v in ("PMOE_STREAM", "PMOE_PREFILL_SMALL"):
        monkeypatch.delenv(v, raising=False)
    from pagedmoe_amd._lib import geom, lib
    g = geom(hidden, inter, bits)
    shared = 1 if kk in (9, 11) else 0
    for n, want in form.items():
        assert lib().pmoe_stream_wanted(ctypes.byref(g), n, kk, e, shared) == want, n
