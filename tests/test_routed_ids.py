"""The routed ids of a paged layer, distinct and ascending, are the same
whether they are made distinct on the host or by torch.unique (the line lies
at HOST_UNIQUE_IDS flat ids); and the library is handed torch's current
stream."""

import pytest
import torch


@pytest.mark.parametrize("shape", [(1, 1), (1, 8), (20, 8), (128, 8), (1025, 1), (700, 3), (0, 8)])
def test_routed_ids_match_unique(shape):
    from pagedmoe_amd import streaming as S
    g = torch.Generator().manual_seed(shape[0])
    ids = torch.randint(-2, 131, shape, dtype=torch.int32, generator=g)  # some out of range
    sw = S.StreamedSwitchGLU.__new__(S.StreamedSwitchGLU)
    torch.nn.Module.__init__(sw)
    sw.n_experts, sw.ring = 128, None
    want = [e for e in torch.unique(ids).tolist() if 0 <= e < 128]
    assert sw.routed_ids(ids) == want


@pytest.mark.gpu
def test_stream_handle_is_torchs_current_stream():
    from pagedmoe_amd import kernels as K
    torch.zeros(1, device="cuda")
    assert (K._stream().value or 0) == torch.cuda.current_stream().cuda_stream
    s = torch.cuda.Stream()
    with torch.cuda.stream(s):
        assert K._stream().value == s.cuda_stream != 0
    assert (K._stream().value or 0) == torch.cuda.current_stream().cuda_stream
