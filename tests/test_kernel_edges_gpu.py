"""Edges of the tiles, splits and dispatch rules of the kernels, against the generic kernels and the oracle."""
import pytest
import torch

from oracle import hash_encoding as O

pytestmark = pytest.mark.gpu
DEV = "cuda"


@pytest.mark.parametrize("N", [2**16 - 1, 2**16, 2**16 + 1, 2**17, 2**17 + 1, 196608, 196609, 2**18 + 1, 304800, 3 * 2**18 + 1, 2**20 - 1, 2**20 + 3])
@pytest.mark.parametrize("dims,dtype", [(3, torch.float16), (2, torch.bfloat16), (3, torch.float32)])
def test_forward_sweep_deals_out_every_point(N, dims, dtype, monkeypatch):
    """The sweep's workgroups take equal shares of one to four points per thread: every output row, also of a ragged last
    wave, has the bits of the per-(point, level) kernel (flag 1)."""
    from triton_helpers_amd.layers.hash_encoding import kernel as hk

    T, L, lo, hi = 2**15, 8, 8, 300
    torch.manual_seed(3)
    x = torch.rand(N, dims, device=DEV)
    table = torch.randn(O.level_row_offsets(L, T, dims, lo, hi)[-1], 2, device=DEV).to(dtype)
    outs = []
    for flags in (0, 1):
        monkeypatch.setattr(hk, "_FLAGS", flags)
        outs.append(hk.hash_encoding(x, table, None, None, T, lo, hi, L))
    assert torch.equal(outs[0], outs[1])
