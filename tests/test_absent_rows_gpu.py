"""Rows that a workgroup rounds its batch up to must not reach a weight gradient.

The networks' biases stand for an input mean (every input is near ``MEAN``, the biases take it out again), so that the activations of every
row of the batch are small, while those of a row of zeros, which the biases alone make, are beyond the type's range: a kernel that lets
such a row into dW = dz^T h adds 0 * inf."""
import pytest
import torch

from oracle import mlp as O
from triton_helpers_amd import _lib

pytestmark = pytest.mark.gpu
NAMES = ("w_in", "b_in", "w_hid", "b_hid", "w_out", "b_out")
# mean of the inputs, and the step between their values: what biases make of zero is beyond the type where the input's deviations are not
MEAN = {torch.float16: (2.0**11, 1.0), torch.float32: (2.0**36, 2.0**22)}


def _network(d_in, H, d_out, depth, act, gen, mean):
    """float32 values that float16 holds (but for float32's bias).  The first layer's pre-activations are exact, and odd multiples of 1/16: none is on a gate's edge."""
    near = lambda *s: (torch.randn(*s, generator=gen) / 12).half().float()  # noqa: E731
    w_in = torch.randint(-2, 2, (H, d_in), generator=gen).float() / 16
    w_in = torch.where(w_in.sum(1, keepdim=True) < 0, w_in, -w_in.abs())
    w_in[:, 0] = -3 / 16
    p = {"w_in": w_in, "b_in": -mean * w_in.sum(1), "w_hid": None, "b_hid": None, "w_out": near(d_out, H), "b_out": near(d_out)}
    if depth > 1:
        p["w_hid"], p["b_hid"] = near((depth - 1) * H, H), near(depth - 1, H)
        if act != "relu2":  # relu2 overflows in the first layer, the others in the second
            p["w_hid"][:H] = 2.0**9 / H
    return p


def _inputs(rows, d_in, d_out, gen, mean, step):
    x = mean + 2.0 * step * torch.randint(-2, 3, (rows, d_in), generator=gen)
    x[:, 0] = mean - step
    return x, torch.randn(rows, d_out, generator=gen).half().float()


def _check(case, entry, dtype=torch.float16):
    rows, d_in, H, d_out, depth, act = case
    gen, mean, half = torch.Generator().manual_seed(rows + depth), MEAN[dtype], torch.float16 if dtype == torch.float16 else None
    p, (x, dy) = _network(d_in, H, d_out, depth, act, gen, mean[0]), _inputs(rows, d_in, d_out, gen, *mean)
    alone = O.mlp_forward(torch.zeros(1, d_in), *(p[k] for k in ("w_in", "b_in", "w_out", "b_out", "w_hid", "b_hid")), act=act, round_to=half)
    assert not torch.isfinite(alone).all(), "the case does not overflow on a row of zeros"
    args = [p[k] for k in ("w_in", "b_in", "w_out", "b_out", "w_hid", "b_hid")]
    want = O.mlp_backward(x, dy, *args, act=act, round_to=half)
    assert all(t is None or torch.isfinite(t).all() for t in want.values())
    dev = {k: None if t is None else t.to(dtype).cuda() for k, t in p.items()}
    dx, got = entry(x.to(dtype).cuda(), dy.to(dtype).cuda(), dev, depth, act)
    # (relu2 doubles a relative error at every layer: at most three of them.)  Each layer's activation, derivative and gradient is rounded to 16 bit (half a unit: 2^-11 of the value), each on its way through at most
    # depth + 1 layers.  As a whole (2-norm) the three add up to less than this.
    # float32: the sums of 64 products (2^-24 of the largest term each) instead, the oracle's in another order.
    eps = 3 * (depth + 1) * (2.0**-11 if half else 64 * 2.0**-24)
    for k, t in {"dx": dx, **{"d" + k: v for k, v in got.items()}}.items():
        if t is None:
            continue
        t, w = t.cpu().double(), want[k].double()
        assert torch.isfinite(t).all(), k
        assert float((t - w).norm()) <= eps * float(w.norm()), k


def _call(function, x, dy, p, depth, act, grads, *tail):
    dx = torch.empty_like(x)
    H, code = p["w_in"].shape[0], _lib.dtype_code(x.dtype)
    rc = function(x.data_ptr(), x.stride(0), dy.data_ptr(), dy.stride(0), dx.data_ptr(), dx.stride(0), *(_lib.ptr(p[k]) for k in NAMES),
                  *(_lib.ptr(grads[k]) for k in NAMES), x.shape[0], x.shape[1], H, dy.shape[1], depth, _lib.NF_ACT[act], code, code, *tail,
                  _lib.current_stream(x.device))
    _lib.check(rc, "backward")
    return dx, grads


def _whole(x, dy, p, depth, act):
    lib = _lib.load()
    n = lib.nf_mlp_bwd_whole_workspace_bytes(x.shape[0], p["w_in"].shape[0], depth, _lib.NF_ACT[act], _lib.NF_F16)
    ws = torch.empty(n, dtype=torch.uint8, device="cuda")
    grads = {k: None if t is None else torch.empty(t.shape, device="cuda") for k, t in p.items()}
    return _call(lib.nf_mlp_bwd_whole, x, dy, p, depth, act, grads, _lib.NF_F32, ws.data_ptr(), n)


@pytest.mark.parametrize("case", [
    # rows, d_in, d_hidden, d_out, depth, act
    (96, 32, 64, 16, 2, "relu2"),   # whole 32-row chunks, half of the second round's 64 rows absent
    (1, 32, 64, 16, 1, "relu2"),
    (97, 48, 64, 33, 2, "relu"),
    (96, 35, 64, 3, 3, "silu"),
    (33, 64, 64, 64, 9, "relu"),
    (96, 32, 64, 16, 5, "gelu"),
    (33, 32, 64, 16, 9, "silu"),
    (96, 32, 32, 16, 2, "relu2"),
    (50, 40, 16, 5, 3, "none"),
    (96, 64, 32, 64, 9, "silu"),
    (16400, 32, 64, 16, 2, "relu2"),  # eight and twelve chain waves
    (16400, 64, 64, 64, 2, "relu"),
    (49200, 32, 32, 16, 3, "relu2"),
], ids=str)
def test_whole_backward(case):
    _check(case, _whole)


def _general(x, dy, p, depth, act):
    lib = _lib.load()
    n = lib.nf_mlp_workspace_bytes(x.shape[0], p["w_in"].shape[0], depth, _lib.NF_ACT[act], 1, _lib.dtype_code(x.dtype))
    ws = torch.empty(max(n, 1), dtype=torch.uint8, device="cuda")
    grads = {k: None if t is None else torch.zeros(t.shape, device="cuda") for k, t in p.items()}
    return _call(lib.nf_mlp_bwd, x, dy, p, depth, act, grads, ws.data_ptr(), n)


@pytest.mark.parametrize("case", [
    # eight waves, role-split (16- and 8-byte rows), four waves (rows off 8-byte boundaries, other activations)
    (33, 32, 64, 16, 2, "relu2"),
    (1, 32, 64, 16, 2, "relu"),
    (4099, 20, 64, 4, 2, "relu"),
    (33, 64, 64, 64, 2, "relu"),
    (8201, 36, 64, 12, 2, "relu"),
    (40003, 16, 64, 64, 2, "relu"),
    (70, 35, 64, 3, 2, "relu"),
    (90, 17, 64, 33, 2, "silu"),
    # two and three hidden-to-hidden layers, and chains of launches
    (49, 32, 64, 16, 3, "relu"),
    (33, 35, 64, 33, 4, "relu"),
    (81, 64, 64, 64, 9, "relu"),
    (50, 32, 64, 16, 5, "silu"),
    # narrow ones
    (33, 32, 32, 16, 2, "relu2"),
    (9, 40, 16, 5, 2, "none"),
    (65, 64, 32, 64, 5, "silu"),
], ids=str)
def test_general_backward(case):
    _check(case, _general)


def _summed(x, dy, p, depth, act):
    lib = _lib.load()
    n = lib.nf_mlp_bwd_rounded_workspace_bytes(x.shape[1], p["w_in"].shape[0], dy.shape[1])
    ws = torch.empty(n, dtype=torch.uint8, device="cuda")
    grads = {k: None if t is None else torch.empty(t.shape, device="cuda") for k, t in p.items()}
    return _call(lib.nf_mlp_bwd_summed, x, dy, p, depth, act, grads, _lib.NF_F32, ws.data_ptr(), n)


@pytest.mark.parametrize("case", [(33, 32, 64, 16, 2, "relu"), (8201, 12, 64, 8, 2, "relu"), (77, 64, 64, 36, 2, "relu"), (40003, 64, 64, 16, 2, "relu")], ids=str)
def test_summed_backward(case):
    _check(case, _summed)


@pytest.mark.parametrize("case", [(33, 32, 64, 16, 2, "relu2"), (17, 64, 32, 64, 2, "relu2"), (4099, 5, 64, 1, 2, "relu2")], ids=str)
def test_float32_backward(case):
    _check(case, _general, torch.float32)
