"""Which prefill calls may take the wide form, and which keep the narrow one:
the wide form loads 16 bytes a lane straight into LDS, so every pointer and
offset it loads from has to lie on 16 bytes.  Host code only."""

import ctypes

import pytest

from pagedmoe_amd._lib import geom, lib

SLAB, X = 1 << 40, 1 << 41  # addresses of the right alignment; never followed


def wide(g, slab=SLAB, x=X, n=4096, kk=8, e=128):
    return lib().pmoe_prefill_wide(ctypes.byref(g), slab, x, n, kk, e)


@pytest.fixture(autouse=True)
def _no_pins(monkeypatch):
    for v in ("PMOE_PREFILL_WIDE", "PMOE_PREFILL_SMALL"):
        monkeypatch.delenv(v, raising=False)


@pytest.mark.parametrize("bits", [4, 6])
@pytest.mark.parametrize("pin", [None, "1"])
def test_unaligned_operands_keep_the_narrow_form(bits, pin, monkeypatch):
    if pin:
        monkeypatch.setenv("PMOE_PREFILL_WIDE", pin)
    g = geom(4096, 1536, bits)
    assert wide(g) == 1
    for shift in (2, 4, 8):
        assert wide(g, x=X + shift) == 0
        assert wide(g, slab=SLAB + shift) == 0
    for c in range(9):
        h = geom(4096, 1536, bits)
        h.off[c] += 8
        assert wide(h) == 0
    h = geom(4096, 1536, bits)
    h.expert_bytes += 8
    assert wide(h) == 0


@pytest.mark.parametrize("bits", [4, 6])
@pytest.mark.parametrize("comp", [0, 1, 2])
def test_up_component_before_its_gate_keeps_the_narrow_form(bits, comp):
    g = geom(4096, 1536, bits)
    g.off[comp], g.off[comp + 3] = g.off[comp + 3], g.off[comp]
    assert wide(g) == 0
    g = geom(4096, 1536, bits)
    g.off[comp + 3] = g.off[comp] + (1 << 31)
    assert wide(g) == 0


def test_pins_and_tile_height(monkeypatch):
    g = geom(4096, 1536, 4)
    assert wide(g, n=512) == 0  # 32-row tiles
    monkeypatch.setenv("PMOE_PREFILL_WIDE", "0")
    assert wide(g) == 0
