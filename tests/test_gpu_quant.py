"""GPU: the format kernels' lane split and reciprocal rounding against the
oracle, bit for bit: group counts that leave a wave or a block part empty,
quotients at and near halves (where the division decides), offsets that push
codes out of range, constant groups, and pointers that are not 16-byte
aligned."""

import numpy as np
import pytest
import torch

from oracle import pmoe_oracle as O
from tests.util import bf16_tensor_bits

pytestmark = pytest.mark.gpu

DEV = "cuda"


def _values(kind, shape, rng):
    x = rng.standard_normal(shape, dtype=np.float32)
    if kind == "normal":
        return x * np.float32(0.02)
    if kind == "halves":  # scale 1 or 0.5: quotients are whole numbers and halves
        return rng.integers(0, 127, shape).astype(np.float32) * np.float32(0.25)
    if kind == "offset":  # the bias' bf16 rounding exceeds the range
        return np.float32(100) + x * np.float32(1e-3)
    if kind == "tiny":  # denormal scales
        return x * np.float32(1e-39)
    return np.full(shape, 0.125, np.float32)


@pytest.mark.parametrize("bits", [4, 6])
@pytest.mark.parametrize("rows,cols", [(1, 64), (3, 448), (11, 192), (33, 1024)])
@pytest.mark.parametrize("kind", ["normal", "halves", "offset", "tiny", "const"])
def test_format_bit_exact(bits, rows, cols, kind):
    from pagedmoe_amd import kernels as K
    w = _values(kind, (rows, cols), np.random.default_rng(rows * cols))
    ref = O.quantize(w, bits)
    for shift in (0, 1):  # 1: a view 4 bytes past an aligned address
        t = torch.zeros(rows * cols + 1, device=DEV)
        v = t[shift:shift + rows * cols].view(rows, cols)
        v.copy_(torch.from_numpy(w))
        assert v.data_ptr() % 16 == 4 * shift
        q, s, b = K.quantize(v, bits)
        assert np.array_equal(q.cpu().numpy().view(np.uint32), ref.weight)
        assert np.array_equal(bf16_tensor_bits(s), ref.scales)
        assert np.array_equal(bf16_tensor_bits(b), ref.biases)
        assert np.array_equal(bf16_tensor_bits(K.dequant(q, s, b, bits)), O.dequant_bf16(ref))


@pytest.mark.parametrize("bits", [4, 6])
def test_dequant_unaligned_output(bits):
    import ctypes
    from pagedmoe_amd import kernels as K
    from pagedmoe_amd._lib import check, lib
    rows, cols = 7, 448
    w = torch.from_numpy(_values("normal", (rows, cols), np.random.default_rng(5))).to(DEV)
    q, s, b = K.quantize(w, bits)
    big = torch.full((rows * cols + 8,), -1, dtype=torch.int16, device=DEV)
    check(lib().pmoe_dequant(K._ptr(q), K._ptr(s), K._ptr(b), rows, cols, bits, 64,
                             ctypes.c_void_p(big.data_ptr() + 2), K._stream()), "pmoe_dequant")
    torch.cuda.synchronize()
    assert torch.equal(big[1:1 + rows * cols],
                       K.dequant(q, s, b, bits).view(torch.int16).reshape(-1))
    assert int(big[0]) == -1 and bool((big[1 + rows * cols:] == -1).all())


def test_more_threads_than_one_launch_holds():
    """2^29 + 40 groups (8 lanes each: over 2^32 threads), 88 GB: the groups
    around each launch's first and last against the same groups alone."""
    from pagedmoe_amd import kernels as K
    cols, rows = 512, (1 << 26) + 5
    if torch.cuda.mem_get_info()[0] < 110e9:
        pytest.skip("needs 88 GB")
    per = cols // 64
    q = torch.empty((rows, cols // 8), dtype=torch.int32, device=DEV)
    s, b = (torch.empty((rows, per), dtype=torch.bfloat16, device=DEV) for _ in range(2))
    w = torch.from_numpy(_values("normal", (16, cols), np.random.default_rng(6))).to(DEV)
    seams = [slice(0, 16), slice((1 << 25) - 8, (1 << 25) + 8), slice((1 << 26) - 11, rows)]
    for at in seams:
        q[at], s[at], b[at] = K.quantize(w, 4)
    out = K.dequant(q, s, b, 4)
    for at in seams:
        assert torch.equal(out[at].view(torch.int16),
                           K.dequant(q[at].clone(), s[at].clone(), b[at].clone(), 4)
                           .view(torch.int16))
    del q, s, b, out
    torch.cuda.empty_cache()
