"""The backward kernels stage their weights in both forms from one read of every matrix where those are 16-byte aligned."""
import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda"


@pytest.mark.parametrize("d_in,d_out", [(32, 16), (8, 4), (24, 12), (16, 16), (64, 64), (40, 36), (48, 16), (32, 64)])
@pytest.mark.parametrize("dtype,bias", [(torch.bfloat16, False), (torch.float16, True)])
def test_matrices_off_their_alignment_give_the_same_bits(d_in, d_out, dtype, bias):
    """2^16 + 3 rows of one hidden-to-hidden ReLU layer: the decoder's and the role-split kernel.  Views one element into a buffer are staged form by form."""
    from triton_helpers_amd.layers.fully_fused_mlp import fully_fused_mlp

    torch.manual_seed(d_in + d_out)
    u = lambda *s: ((torch.rand(*s, device=DEV) * 2 - 1) / s[-1] ** 0.5).to(dtype)  # noqa: E731
    w = {"w_in": u(64, d_in), "w_hid": u(64, 64), "w_out": u(d_out, 64)}
    if bias:
        w.update(b_in=u(64), b_hid=u(1, 64), b_out=u(d_out))
    x, dy = torch.randn(1, 2**16 + 3, d_in, device=DEV).to(dtype), torch.randn(1, 2**16 + 3, d_out, device=DEV).to(dtype)

    def grads(shift):
        leaves = {"x": x.clone().requires_grad_()}
        for k, t in w.items():
            flat = torch.empty(t.numel() + 8, dtype=dtype, device=DEV)
            leaves[k] = flat[shift : shift + t.numel()].view(t.shape).copy_(t).detach().requires_grad_()
        y = fully_fused_mlp(activation="relu", **{"b_in": None, "b_out": None, "b_hid": None, **leaves})
        y.backward(dy)
        return [t.grad for t in leaves.values()]

    for a, b in zip(grads(0), grads(1)):
        assert torch.equal(a, b)


@pytest.mark.parametrize("half,blocks,rows", [(64, 1, 33), (64, 3, 64), (64, 5, 4096), (32, 4, 96), (32, 7, 4100), (16, 2, 64)])
@pytest.mark.parametrize("bias", [False, True])
def test_couplings_off_their_alignment_give_the_same_bits(half, blocks, rows, bias):
    """Reversible weights on 16-byte, 8-byte and odd addresses, full and padded widths, a last group and a last pass of fewer couplings."""
    from triton_helpers_amd.layers.reversible_mlp import reversible_mlp

    torch.manual_seed(half + blocks)
    u = lambda *s: ((torch.rand(*s, device=DEV) * 2 - 1) / half**0.5).bfloat16()  # noqa: E731
    w = [u(2 * blocks * half, half), u(2 * blocks, half) if bias else None, u(2 * blocks * half, half), u(2 * blocks, half) if bias else None]
    x, dy = torch.randn(rows, 2 * half, device=DEV).bfloat16(), torch.randn(rows, 2 * half, device=DEV).bfloat16()

    def run(shift):
        leaves = [x.clone().requires_grad_()] + [None if t is None else torch.empty(t.numel() + 8, dtype=t.dtype, device=DEV)[shift : shift + t.numel()].view(t.shape).copy_(t).detach().requires_grad_() for t in w]
        y = reversible_mlp(*leaves, activation="gelu")
        y.backward(dy)
        return [y.detach()] + [t.grad for t in leaves if t is not None]

    want = run(0)
    for shift in (1, 4):
        for a, b in zip(want, run(shift)):
            assert torch.equal(a, b)


@pytest.mark.parametrize("rows", [1, 1000, 40001])
@pytest.mark.parametrize("d_in,hidden,d_out,depth,act", [(32, 64, 16, 2, "relu"), (64, 64, 64, 9, "relu"), (8, 32, 33, 5, "relu"), (24, 16, 3, 1, "silu"), (40, 64, 64, 3, "silu"), (56, 32, 64, 9, "relu2")])
def test_whole_backward_off_its_alignment_gives_the_same_bits(rows, d_in, hidden, d_out, depth, act):
    """The list of 16-byte pieces against the matrices one by one: padded rows and columns of every matrix, the fewest and the most layers."""
    from triton_helpers_amd.layers.fully_fused_mlp import fully_fused_mlp

    torch.manual_seed(rows + d_in)
    u = lambda *s: ((torch.rand(*s, device=DEV) * 2 - 1) / s[-1] ** 0.5).half()  # noqa: E731
    w = {"w_in": u(hidden, d_in), "b_in": u(hidden), "w_out": u(d_out, hidden), "b_out": u(d_out)}
    if depth > 1:
        w.update(w_hid=u((depth - 1) * hidden, hidden), b_hid=u(depth - 1, hidden))
    x, dy = torch.randn(1, rows, d_in, device=DEV).half(), torch.randn(1, rows, d_out, device=DEV).half()

    def grads(shift):
        leaves = {"x": x.clone().requires_grad_()}
        for k, t in w.items():
            leaves[k] = torch.empty(t.numel() + 8, dtype=t.dtype, device=DEV)[shift : shift + t.numel()].view(t.shape).copy_(t).detach().requires_grad_()
        fully_fused_mlp(activation=act, **{"w_hid": None, "b_hid": None, **leaves}).backward(dy)
        return [t.grad for t in leaves.values()]

    for a, b in zip(grads(0), grads(4)):
        assert torch.equal(a, b)
