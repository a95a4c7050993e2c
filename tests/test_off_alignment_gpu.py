"""Tables and weights off their natural alignment, as slices of a flat buffer of parameters are: the same bits, and kernels of about the same speed."""
import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda"


def _off(t, shift):
    """The same values `shift` elements into a buffer of their own."""
    return torch.empty(t.numel() + 8, dtype=t.dtype, device=DEV)[shift : shift + t.numel()].view(t.shape).copy_(t)


def _us(f):
    """Shortest of seven turns of 40 calls, per call."""
    best = float("inf")
    for _ in range(8):
        a, b = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
        a.record()
        for _ in range(40):
            f()
        b.record()
        torch.cuda.synchronize()
        best = min(best, a.elapsed_time(b) * 1e3 / 40)
    return best


@pytest.mark.parametrize("N", [1, 1000, 16383, 16384, 65536, 65537, 131072])
@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("D,T,hi", [(3, 2**19, 4096), (3, 2**14, 512), (2, 2**17, 2048)])
def test_table_a_value_into_its_buffer(N, dtype, D, T, hi):
    from triton_helpers_amd.layers.hash_encoding import hash_encoding
    from triton_helpers_amd.layers.hash_encoding.helpers import total_rows

    torch.manual_seed(N)
    x = torch.rand(N, D, device=DEV)
    table = torch.randn(total_rows(T, 16, D, 16, hi), 2, device=DEV).to(dtype)
    run = lambda t: hash_encoding(x, t, max_entries_per_level=T, min_res=16, max_res=hi, levels=16)  # noqa: E731
    shifted = _off(table, 1)
    assert shifted.data_ptr() % 4 == 2
    assert torch.equal(run(table), run(shifted))
    if N == 1000:  # 4.5 us and as much; through the staged kernel 22 and 51
        assert _us(lambda: run(shifted)) < 2 * _us(lambda: run(table))
