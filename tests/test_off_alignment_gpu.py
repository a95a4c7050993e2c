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


# (offset in values of w_in, w_hid, w_out): one list in 8-byte pieces; the first or last matrix by itself; 16-byte pieces with the first by itself; layer by layer
OFFSETS = [(0, 4, 4), (4, 0, 4), (0, 4, 0), (1, 4, 1), (0, 0, 2), (4, 0, 0), (1, 0, 0), (0, 1, 0)]


@pytest.mark.parametrize("rows", [1, 1000, 40001])
@pytest.mark.parametrize("d_in,hidden,d_out,n_hid,act", [(32, 64, 16, 1, "relu"), (64, 64, 64, 1, "relu"), (35, 64, 3, 1, "relu"), (32, 64, 16, 1, "silu"), (40, 64, 33, 3, "relu"),
                                                         (64, 64, 64, 9, "relu"), (27, 32, 4, 4, "silu"), (8, 16, 20, 2, "relu2")])  # fmt: skip
def test_matrices_of_the_forward(rows, d_in, hidden, d_out, n_hid, act):
    from triton_helpers_amd.layers.fully_fused_mlp import fully_fused_mlp

    torch.manual_seed(rows + d_in)
    u = lambda *s: ((torch.rand(*s, device=DEV) * 2 - 1) / s[-1] ** 0.5).half()  # noqa: E731
    w_in, w_hid, w_out, b_in, b_hid, b_out = u(hidden, d_in), u(n_hid * hidden, hidden), u(d_out, hidden), u(hidden), u(n_hid, hidden), u(d_out)
    x = torch.randn(1, rows, d_in, device=DEV).half()

    def run(a, b, c):
        w = [_off(w_in, a), b_in, _off(w_out, c), b_out, _off(w_hid, b), b_hid]
        return lambda: fully_fused_mlp(x, *w, activation=act)

    with torch.no_grad():
        want = run(0, 0, 0)()
        for offset in OFFSETS:
            assert torch.equal(want, run(*offset)()), offset
        if n_hid == 9 and rows == 1000:  # as a list of 16-byte pieces 8.7 us; layer by layer, two groups of rows to a wave, 17.1
            assert _us(run(0, 4, 4)) < 1.5 * _us(run(0, 0, 0))
