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
MEAN = 2048.0


def _network(d_in, H, d_out, depth, act, gen):
    """float32 values that float16 holds.  The first layer's pre-activations are exact, and odd multiples of 1/16: none is on a gate's edge."""
    near = lambda *s: (torch.randn(*s, generator=gen) / 12).half().float()  # noqa: E731
    w_in = torch.randint(-2, 2, (H, d_in), generator=gen).float() / 16
    w_in = torch.where(w_in.sum(1, keepdim=True) < 0, w_in, -w_in.abs())
    w_in[:, 0] = -3 / 16
    p = {"w_in": w_in, "b_in": -MEAN * w_in.sum(1), "w_hid": None, "b_hid": None, "w_out": near(d_out, H), "b_out": near(d_out)}
    if depth > 1:
        p["w_hid"], p["b_hid"] = near((depth - 1) * H, H), near(depth - 1, H)
        if act != "relu2":  # relu2 overflows in the first layer, the others in the second
            p["w_hid"][:H] = 2.0**9 / H
    return p


def _inputs(rows, d_in, d_out, gen):
    x = MEAN + 2.0 * torch.randint(-2, 3, (rows, d_in), generator=gen)
    x[:, 0] = MEAN - 1
    return x, torch.randn(rows, d_out, generator=gen).half().float()


def _check(case, entry):
    rows, d_in, H, d_out, depth, act = case
    gen = torch.Generator().manual_seed(rows + depth)
    p, (x, dy) = _network(d_in, H, d_out, depth, act, gen), _inputs(rows, d_in, d_out, gen)
    alone = O.mlp_forward(torch.zeros(1, d_in), *(p[k] for k in ("w_in", "b_in", "w_out", "b_out", "w_hid", "b_hid")), act=act, round_to=torch.float16)
    assert not torch.isfinite(alone).all(), "the case does not overflow on a row of zeros"
    args = [p[k] for k in ("w_in", "b_in", "w_out", "b_out", "w_hid", "b_hid")]
    want = O.mlp_backward(x, dy, *args, act=act, round_to=torch.float16)
    assert all(t is None or torch.isfinite(t).all() for t in want.values())
    dev = {k: None if t is None else t.half().cuda() for k, t in p.items()}
    dx, got = entry(x.half().cuda(), dy.half().cuda(), dev, depth, act)
    # (relu2 doubles a relative error at every layer: at most three of them.)  Each layer's activation, derivative and gradient is rounded to 16 bit (half a unit: 2^-11 of the value), each on its way through at most
    # depth + 1 layers.  As a whole (2-norm) the three add up to less than this.
    eps = 3 * (depth + 1) * 2.0**-11
    for k, t in {"dx": dx, **{"d" + k: v for k, v in got.items()}}.items():
        if t is None:
            continue
        t, w = t.cpu().double(), want[k].double()
        assert torch.isfinite(t).all(), k
        assert float((t - w).norm()) <= eps * float(w.norm()), k


def _call(function, x, dy, p, depth, act, grads, *tail):
    dx = torch.empty_like(x)
    H, code = p["w_in"].shape[0], _lib.NF_F16
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
