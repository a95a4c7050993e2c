"""Which kernels the fused MLP's backward runs, on both sides of its rules: the operator's gradients have the bits of the entry point that the rule
names (the chained kernels add weight gradients with atomics: within their order), and agree with the whole-network kernel."""
import pytest
import torch

from triton_helpers_amd import _lib
from triton_helpers_amd.layers.fully_fused_mlp import fully_fused_mlp

pytestmark = pytest.mark.gpu
NAMES = ("w_in", "b_in", "w_hid", "b_hid", "w_out", "b_out")
EPS = {torch.bfloat16: 2.0**-8, torch.float16: 2.0**-11}
CASES = [
    # route, rows, d_in, d_hidden, d_out, depth, act, dtype, row padding, x of the other type
    ("whole", 1 << 16, 32, 64, 16, 2, "relu", "bf16", 0, False),
    ("summed", (1 << 16) + 1, 32, 64, 16, 2, "relu", "bf16", 0, False),
    ("summed", (1 << 16) + 1, 32, 64, 16, 2, "relu", "bf16", 4, True),
    ("summed", (1 << 16) + 1, 64, 64, 64, 2, "relu", "f16", 0, False),
    ("whole", (1 << 16) + 1, 64, 64, 64, 2, "relu", "f16", 0, True),
    ("whole", (1 << 16) + 1, 32, 64, 16, 2, "relu", "bf16", 1, False),
    ("whole", 1 << 19, 32, 64, 16, 1, "relu", "bf16", 0, False),
    ("summed", (1 << 19) + 1, 32, 64, 16, 1, "relu", "bf16", 0, False),
    ("summed", (1 << 19) + 1, 64, 64, 16, 1, "relu", "f16", 0, False),
    ("whole", (1 << 19) + 1, 32, 64, 20, 1, "relu", "bf16", 0, False),
    ("whole", 3 << 18, 32, 64, 16, 2, "silu", "bf16", 0, False),
    ("general", (3 << 18) + 1, 32, 64, 16, 2, "silu", "bf16", 0, False),
    ("general", (3 << 18) + 1, 20, 64, 4, 2, "none", "f16", 4, False),
    ("whole", (3 << 18) + 1, 32, 64, 16, 2, "silu", "bf16", 1, False),
    ("whole", (3 << 18) + 1, 32, 64, 16, 2, "relu", "bf16", 3, False),
    ("whole", (3 << 18) + 1, 32, 64, 16, 2, "silu", "bf16", 0, True),
    ("whole", 3 << 18, 32, 64, 16, 3, "relu", "bf16", 0, False),
    ("general", (3 << 18) + 1, 32, 64, 16, 3, "relu", "f16", 0, False),
    ("whole", (3 << 18) + 1, 64, 64, 16, 3, "relu", "bf16", 0, False),
    ("whole", (7 << 18) + 1, 35, 64, 3, 3, "relu", "bf16", 0, False),
    ("general", (7 << 18) + 1, 64, 64, 16, 3, "relu", "bf16", 0, False),
    ("whole", (5 << 18) + 1, 32, 64, 16, 5, "relu", "bf16", 0, False),
    ("general", (7 << 18) + 1, 32, 64, 16, 5, "relu", "bf16", 0, False),
    ("whole", (7 << 18) + 1, 64, 64, 64, 9, "relu", "f16", 0, False),
    ("general", 1000, 64, 64, 64, 10, "relu", "f16", 0, True),
]


def _rows(n, width, pad, dtype, gen):
    return torch.randn(n, width + pad, generator=gen, device="cuda").to(dtype)[:, :width]


@pytest.mark.parametrize("case", CASES, ids=lambda c: "-".join(map(str, c)))
def test_route(case):
    route, rows, d_in, H, d_out, depth, act, dt, pad, other = case
    lib = _lib.load()
    dtype, xt = (torch.float16, torch.bfloat16) if dt == "f16" else (torch.bfloat16, torch.float16)
    xt = xt if other else dtype
    gen = torch.Generator(device="cuda").manual_seed(depth)

    def u(shape, fan_in):
        return ((torch.rand(shape, generator=gen, device="cuda") * 2 - 1) * fan_in**-0.5).to(dtype).requires_grad_()

    p = {"w_in": u((H, d_in), d_in), "b_in": u((H,), d_in), "w_out": u((d_out, H), H), "b_out": u((d_out,), H),
         "w_hid": u(((depth - 1) * H, H), H) if depth > 1 else None, "b_hid": u((depth - 1, H), H) if depth > 1 else None}
    x, dy = _rows(rows, d_in, pad, xt, gen), _rows(rows, d_out, pad, dtype, gen)
    leaf = x.detach().requires_grad_()
    y = fully_fused_mlp(leaf[None], p["w_in"], p["b_in"], p["w_out"], p["b_out"], p["w_hid"], p["b_hid"], act)
    y.backward(dy[None])
    code, a, st = _lib.dtype_code(dtype), _lib.NF_ACT[act], _lib.current_stream(x.device)
    weights = [_lib.ptr(p[k]) for k in NAMES]

    def entry(which):
        src = x.to(dtype).contiguous() if which == "general" else x
        dx = torch.empty(rows, d_in, dtype=src.dtype, device="cuda")
        grads = {k: None if t is None else torch.zeros(t.shape, dtype=torch.float32 if which == "general" else dtype, device="cuda") for k, t in p.items()}
        head = (src.data_ptr(), src.stride(0), dy.data_ptr(), dy.stride(0), dx.data_ptr(), d_in, *weights, *(_lib.ptr(grads[k]) for k in NAMES), rows, d_in, H,
                d_out, depth, a, code, _lib.dtype_code(src.dtype))
        if which == "whole":
            n = lib.nf_mlp_bwd_whole_workspace_bytes(rows, H, depth, a, code)
        elif which == "summed":
            n = lib.nf_mlp_bwd_rounded_workspace_bytes(d_in, H, d_out)
        else:
            n = lib.nf_mlp_workspace_bytes(rows, H, depth, a, 1, code)
        ws = torch.empty(max(n, 1), dtype=torch.uint8, device="cuda")
        function = {"whole": lib.nf_mlp_bwd_whole, "summed": lib.nf_mlp_bwd_summed, "general": lib.nf_mlp_bwd}[which]
        _lib.check(function(*head, *(() if which == "general" else (code,)), ws.data_ptr(), n, st), which)
        return dx, {k: None if t is None else t.to(dtype) for k, t in grads.items()}

    dx, grads = entry(route)
    assert torch.equal(leaf.grad, dx.to(xt))
    for k, t in p.items():
        if t is None:
            continue
        if route != "general":
            assert torch.equal(t.grad, grads[k]), k
        else:  # float32 sums in another order, rounded: a unit in the last place of the type
            assert float((t.grad.float() - grads[k].float()).abs().max()) <= 2 * EPS[dtype] * float(grads[k].float().abs().max()), k
    if route == "whole" or depth > 9:
        return
    dx, grads = entry("whole")
    # as the kernels round alike, a gradient differs by what sums in another order move at each layer (half a unit of the type, now and then)
    eps = 2 * (depth + 1) * max(EPS[dtype], EPS[xt])
    assert float((leaf.grad.float() - dx.float()).norm()) <= eps * float(dx.float().norm())
    for k, t in p.items():
        if t is not None:
            assert float((t.grad.float() - grads[k].float()).norm()) <= eps * float(grads[k].float().norm()), k
