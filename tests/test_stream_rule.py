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
    # dims without prefill GEMMs (no multiples of 512) have no upper end
    (2048, 768, 4, 128, 8, {12: 0, 16: 1, 600: 1, 16384: 1}),
    (2304, 1152, 6, 64, 6, {4: 0, 8: 1, 4096: 1}),
    (384, 640, 4, 64, 4, {16: 0, 4096: 1}),
    # 128-row tiles' layers below 1024 rows are the GEMV's otherwise
    (6144, 2560, 4, 16, 2, {4: 0, 8: 1, 511: 1, 512: 0}),
    # the prefill range, by the layer's bytes: 216, 270, 312 and 1224 MiB
    (2048, 512, 4, 128, 8, {255: 1, 257: 0, 512: 0}),
    (2560, 512, 4, 128, 8, {255: 1, 257: 1, 512: 1, 513: 0}),
    (2048, 512, 6, 128, 8, {255: 1, 257: 0}),
    (2048, 512, 6, 512, 10, {820: 1, 1638: 1, 1639: 0}),
    (5120, 1536, 4, 160, 6, {2: 0, 4: 1, 426: 1, 427: 0}),
    # no cut: odd group counts, rows below six groups, 6-bit rows above 4096
    (2880, 2880, 4, 32, 4, {64: 0, 4096: 0}),
    (1024, 704, 4, 32, 4, {64: 0}),
    (1024, 256, 4, 32, 4, {64: 0}),
    (7168, 2048, 6, 64, 8, {64: 0}),
    (8192, 1024, 4, 16, 2, {64: 0}),
])
def test_stream_rule(hidden, inter, bits, e, kk, form, monkeypatch):
    for v in ("PMOE_STREAM", "PMOE_PREFILL_SMALL"):
        monkeypatch.delenv(v, raising=False)
    from pagedmoe_amd._lib import geom, lib
    g = geom(hidden, inter, bits)
    shared = 1 if kk in (9, 11) else 0
    for n, want in form.items():
        assert lib().pmoe_stream_wanted(ctypes.byref(g), n, kk, e, shared) == want, n


@pytest.mark.parametrize("bits", [4, 6])
@pytest.mark.parametrize("pin", [None, "1"])
def test_slots_the_buffer_loads_cannot_address(bits, pin, monkeypatch):
    """A resource spans one slot: components outside the stride (one array a
    component over all experts), strides of 2 GiB and offsets that are not
    whole words stay on the general paths."""
    from pagedmoe_amd._lib import geom, lib
    monkeypatch.delenv("PMOE_STREAM", raising=False)
    if pin:
        monkeypatch.setenv("PMOE_STREAM", pin)

    def wanted(edit):
        g = geom(4096, 1024, bits)
        edit(g)
        return lib().pmoe_stream_wanted(ctypes.byref(g), 64, 8, 128, 0)

    assert wanted(lambda g: None) == 1
    for c in range(9):
        assert wanted(lambda g: g.off.__setitem__(c, g.expert_bytes - g.nbytes[c] + 4)) == 0
        assert wanted(lambda g: g.off.__setitem__(c, -256)) == 0
        assert wanted(lambda g: g.off.__setitem__(c, g.off[c] + 2)) == 0
    assert wanted(lambda g: setattr(g, "expert_bytes", 1 << 31)) == 0
    assert wanted(lambda g: setattr(g, "expert_bytes", (1 << 31) - 256)) == 1
