"""The whole-network backward (nf_mlp_bwd_whole): against the oracle, and against nf_mlp_bwd, the general path, over the forms both accept."""
import pytest
import torch

from oracle import mlp as O
from triton_helpers_amd import _lib

NAMES = ("w_in", "b_in", "w_hid", "b_hid", "w_out", "b_out")
EPS = {torch.bfloat16: 2.0**-8, torch.float16: 2.0**-11}  # half a unit in the last place, relative


def test_what_it_covers():
    if not _lib.LIB_PATH.exists():
        pytest.skip("libnf_cdna4.so not built")
    lib = _lib.load()
    relu = _lib.NF_ACT["relu"]
    assert lib.nf_mlp_bwd_whole_workspace_bytes(1, 64, 1, relu, _lib.NF_F16) > 0
    assert lib.nf_mlp_bwd_whole_workspace_bytes(1 << 20, 16, 9, relu, _lib.NF_BF16) > 0
    for H, tiles in ((16, 8), (32, 8), (64, 16)):  # one workgroup: a layer's 16 x 16 tiles and its bias sums
        assert lib.nf_mlp_bwd_whole_workspace_bytes(1, H, 9, relu, _lib.NF_F16) == 10 * (tiles + 1) * 256 * 4
    for rows, depth, dtype in ((0, 2, _lib.NF_F16), (100, 10, _lib.NF_F16), (100, 2, _lib.NF_F32)):
        assert lib.nf_mlp_bwd_whole_workspace_bytes(rows, 64, depth, relu, dtype) == 0
        rc = lib.nf_mlp_bwd_whole(1, 32, 1, 16, None, 32, 1, None, 1, None, 1, None, 1, None, 1, None, 1, None,
                                  rows, 32, 64, 16, depth, relu, dtype, dtype, dtype, 16, 1 << 30, None)
        assert rc == _lib.NF_EUNSUPPORTED
    rc = lib.nf_mlp_bwd_whole(1, 32, 1, 16, None, 32, 1, None, 1, None, 1, None, 1, None, 1, None, 1, None,
                              100, 32, 64, 16, 2, relu, _lib.NF_F16, _lib.NF_F16, _lib.NF_F16, None, 0, None)
    assert rc == -1 and b"workspace" in lib.nf_last_error()


def _rows(n, width, pad, shift, dtype, gen):
    """[n, width] with a row stride of width + pad values, `shift` values off an allocation's start."""
    flat = torch.randn(n * (width + pad) + shift + 8, generator=gen, device="cuda").to(dtype)
    return flat[shift:].as_strided((n, width), (width + pad, 1))


CASES = [
    # rows, d_in, d_hidden, d_out, depth, act, bias, dtype, x of the other type, row padding, shift in values
    (1, 32, 64, 16, 1, "relu", True, "f16", False, 0, 0),
    (15, 3, 64, 64, 1, "relu2", True, "bf16", False, 0, 0),
    (16, 64, 64, 1, 2, "silu", False, "f16", False, 0, 0),
    (17, 35, 64, 33, 2, "relu", True, "bf16", False, 1, 1),
    (63, 27, 64, 3, 3, "relu", False, "bf16", False, 0, 0),
    (64, 48, 64, 20, 3, "gelu", True, "f16", False, 4, 4),
    (65, 33, 64, 17, 4, "relu", True, "f16", False, 3, 2),
    (130, 7, 64, 7, 4, "silu", True, "bf16", False, 0, 3),
    (200, 64, 64, 64, 5, "relu", True, "f16", False, 0, 0),
    (513, 32, 64, 16, 6, "silu", True, "bf16", False, 0, 0),
    (300, 9, 64, 8, 8, "relu", True, "bf16", False, 8, 8),
    (1000, 64, 64, 64, 9, "relu", True, "f16", False, 0, 0),
    (1000, 31, 64, 2, 9, "none", False, "bf16", False, 0, 0),
    (40, 64, 32, 64, 1, "relu", True, "bf16", False, 0, 0),
    (70, 33, 32, 33, 2, "relu2", True, "f16", False, 1, 0),
    (129, 32, 16, 16, 2, "relu", True, "bf16", False, 0, 0),
    (127, 5, 16, 3, 3, "silu", True, "f16", False, 0, 1),
    (400, 64, 32, 5, 4, "relu", False, "bf16", False, 2, 0),
    (257, 40, 32, 40, 9, "gelu", True, "f16", False, 0, 0),
    (100, 32, 64, 3, 2, "relu", False, "bf16", True, 0, 0),
    (100, 35, 32, 1, 1, "silu", True, "f16", True, 1, 1),
    # more rows than one round: four or eight (64 wide), twelve chain waves per workgroup
    (16384, 32, 64, 3, 2, "relu", True, "bf16", True, 0, 0),
    (16385, 32, 64, 16, 4, "relu", True, "f16", False, 0, 0),
    (40003, 48, 64, 33, 3, "silu", True, "bf16", False, 0, 0),
    (40003, 64, 64, 64, 9, "relu", False, "bf16", False, 0, 0),
    (40003, 64, 64, 64, 5, "relu", True, "f16", False, 0, 0),
    (80003, 32, 64, 16, 6, "relu", True, "bf16", False, 0, 0),
    (40003, 35, 64, 3, 6, "relu", True, "bf16", False, 1, 1),
    (100003, 33, 32, 16, 4, "relu", True, "f16", False, 0, 0),
    (40003, 32, 16, 33, 6, "relu2", True, "bf16", False, 0, 0),
    # two workgroups per compute unit (narrow deep ReLU) and twelve chain waves of another activation, each in more than one round
    (100003, 32, 32, 16, 6, "relu", True, "bf16", False, 0, 0),
    (100003, 40, 16, 40, 9, "relu", False, "f16", False, 0, 0),
    (100003, 35, 32, 5, 3, "silu", True, "bf16", False, 1, 0),
]


def _params(rows, d_in, H, d_out, depth, bias, dtype, gen):
    def u(shape, fan_in):
        return ((torch.rand(shape, generator=gen, device="cuda") * 2 - 1) * fan_in**-0.5).to(dtype)

    return {"w_in": u((H, d_in), d_in), "w_out": u((d_out, H), H), "w_hid": u(((depth - 1) * H, H), H) if depth > 1 else None,
            "b_in": u((H,), d_in) if bias else None, "b_out": u((d_out,), H) if bias else None,
            "b_hid": u((depth - 1, H), H) if bias and depth > 1 else None}


@pytest.mark.gpu
@pytest.mark.parametrize("case", [c for c in CASES if c[0] <= 1000], ids=lambda c: "-".join(map(str, c)))
def test_whole_backward_is_the_oracles(case):
    rows, d_in, H, d_out, depth, act, bias, dt, other, pad, shift = case
    lib = _lib.load()
    dtype = {"f16": torch.float16, "bf16": torch.bfloat16}[dt]
    xt = dtype if not other else (torch.bfloat16 if dtype == torch.float16 else torch.float16)
    gen = torch.Generator(device="cuda").manual_seed(rows + depth)
    p = _params(rows, d_in, H, d_out, depth, bias, dtype, gen)
    x, dy = _rows(rows, d_in, pad, shift, xt, gen), _rows(rows, d_out, pad, shift, dtype, gen)
    got = {k: None if p[k] is None else torch.empty(p[k].shape, device="cuda") for k in NAMES}
    dx = torch.empty(rows, d_in, dtype=xt, device="cuda")
    code, a = _lib.dtype_code(dtype), _lib.NF_ACT[act]
    n = lib.nf_mlp_bwd_whole_workspace_bytes(rows, H, depth, a, code)
    ws = torch.empty(n, dtype=torch.uint8, device="cuda")
    _lib.check(lib.nf_mlp_bwd_whole(x.data_ptr(), x.stride(0), dy.data_ptr(), dy.stride(0), dx.data_ptr(), d_in, *(_lib.ptr(p[k]) for k in NAMES),
                                    *(_lib.ptr(got[k]) for k in NAMES), rows, d_in, H, d_out, depth, a, code, _lib.dtype_code(xt), _lib.NF_F32,
                                    ws.data_ptr(), n, _lib.current_stream(x.device)), "nf_mlp_bwd_whole")
    cpu = {k: None if t is None else t.cpu() for k, t in p.items()}
    want = O.mlp_backward(x.to(dtype).cpu(), dy.cpu(), *(cpu[k] for k in ("w_in", "b_in", "w_out", "b_out", "w_hid", "b_hid")), act=act, round_to=dtype)
    # As a whole (2-norm): each layer's activation, derivative and gradient is rounded to 16 bit, half a unit each, on its way through at most
    # depth + 1 layers (the oracle rounds the first alone), and dx to x's type.
    eps = 3 * (depth + 1) * EPS[dtype] + EPS[xt]
    for k, t in {"dx": dx, **{"d" + k: v for k, v in got.items()}}.items():
        if t is not None:
            assert float((t.cpu().double() - want[k].double()).norm()) <= eps * float(want[k].double().norm()), k


@pytest.mark.gpu
@pytest.mark.parametrize("case", CASES, ids=lambda c: "-".join(map(str, c)))
def test_whole_backward_is_the_general_one(case):
    rows, d_in, H, d_out, depth, act, bias, dt, other, pad, shift = case
    lib = _lib.load()
    dtype = {"f16": torch.float16, "bf16": torch.bfloat16}[dt]
    xt = dtype if not other else (torch.bfloat16 if dtype == torch.float16 else torch.float16)
    gen = torch.Generator(device="cuda").manual_seed(rows + depth)
    p = _params(rows, d_in, H, d_out, depth, bias, dtype, gen)
    x, dy = _rows(rows, d_in, pad, shift, xt, gen), _rows(rows, d_out, pad, shift, dtype, gen)
    code, a = _lib.dtype_code(dtype), _lib.NF_ACT[act]
    stream = _lib.current_stream(x.device)
    weights = [_lib.ptr(p[k]) for k in NAMES]

    # the general path, on a cast copy where x is stored in the other type
    xc = x.to(dtype).contiguous()
    acc = {k: None if p[k] is None else torch.zeros(p[k].shape, device="cuda") for k in NAMES}
    want_dx = torch.empty_like(xc)
    n = lib.nf_mlp_workspace_bytes(rows, H, depth, a, 1, code)
    ws = torch.empty(max(n, 1), dtype=torch.uint8, device="cuda")
    _lib.check(lib.nf_mlp_bwd(xc.data_ptr(), d_in, dy.data_ptr(), dy.stride(0), want_dx.data_ptr(), d_in, *weights, *(_lib.ptr(acc[k]) for k in NAMES),
                              rows, d_in, H, d_out, depth, a, code, code, ws.data_ptr(), n, stream), "nf_mlp_bwd")

    n = lib.nf_mlp_bwd_whole_workspace_bytes(rows, H, depth, a, code)
    ws = torch.empty(n, dtype=torch.uint8, device="cuda").fill_(0xFF)  # NaN wherever a slot is not written
    runs = []
    for grad_code, grad_dtype in ((_lib.NF_F32, torch.float32), (_lib.NF_F32, torch.float32), (code, dtype)):
        got = {k: None if p[k] is None else torch.full(p[k].shape, float("nan"), dtype=grad_dtype, device="cuda") for k in NAMES}
        room = torch.full((rows * (d_in + pad) + shift + 16,), 7.0, dtype=xt, device="cuda")  # dx between values that must stay
        dx = room[shift:].as_strided((rows, d_in), (d_in + pad, 1))
        _lib.check(lib.nf_mlp_bwd_whole(x.data_ptr(), x.stride(0), dy.data_ptr(), dy.stride(0), dx.data_ptr(), dx.stride(0), *weights,
                                        *(_lib.ptr(got[k]) for k in NAMES), rows, d_in, H, d_out, depth, a, code, _lib.dtype_code(xt), grad_code,
                                        ws.data_ptr(), n, stream), "nf_mlp_bwd_whole")
        runs.append((dx.clone(), got))
        dx.fill_(7.0)
        assert (room == 7.0).all(), "dx was written outside its rows"
    dx, got = runs[0]
    # Layer by layer the two round the same values to 16 bit; sums in another order move one by half a unit in the last place now
    # and then, which every layer in front of it may do again.  The ReLU networks of width 64 sum in the same order.  dx is rounded
    # to the type x is stored in.
    eps = 2 * (depth + 1) * max(EPS[dtype], EPS[xt])
    if act == "relu" and H == 64 and not other:
        assert torch.equal(dx, want_dx)
    else:
        assert float((dx.float() - want_dx.float()).abs().max()) <= eps * float(want_dx.float().abs().max())
    for k in NAMES:
        if p[k] is None:
            continue
        assert torch.isfinite(got[k]).all(), k
        assert float((got[k] - acc[k]).abs().max()) <= eps * float(acc[k].abs().max()) + 1e-30, k
        assert torch.equal(got[k], runs[1][1][k]), f"{k}: two calls differ"
        assert torch.equal(got[k].to(dtype), runs[2][1][k]), f"{k}: rounded"
    assert torch.equal(dx, runs[1][0])
