"""Rows that move in 16-byte pieces (exchanged between lane groups) against the same rows off 16-byte boundaries, which move in
8-byte pieces: the sums are the same, so every output is, bit for bit."""
import pytest
import torch

from triton_helpers_amd import _lib

pytestmark = pytest.mark.gpu
NAMES = ("w_in", "b_in", "w_hid", "b_hid", "w_out", "b_out")


def _rows(t, pad, shift):
    """The same values with a row stride of width + pad, `shift` values off an allocation's start."""
    n, width = t.shape
    out = torch.empty(n * (width + pad) + shift + 8, dtype=t.dtype, device="cuda")[shift:].as_strided((n, width), (width + pad, 1))
    return out.copy_(t)


@pytest.mark.parametrize("rows", [1, 31, 33, 129, 9001])
@pytest.mark.parametrize("d_in,d_out", [(64, 64), (64, 16), (32, 64), (40, 24), (64, 8), (8, 40), (48, 20)])
@pytest.mark.parametrize("dtype,xdtype", [(torch.bfloat16, torch.bfloat16), (torch.float16, torch.bfloat16)])
def test_wide_and_narrow_pieces_agree(rows, d_in, d_out, dtype, xdtype):
    lib = _lib.load()
    H, relu, code, xcode = 64, _lib.NF_ACT["relu"], _lib.dtype_code(dtype), _lib.dtype_code(xdtype)
    gen = torch.Generator(device="cuda").manual_seed(rows)
    u = lambda *s: ((torch.rand(*s, generator=gen, device="cuda") * 2 - 1) / 8).to(dtype)  # noqa: E731
    p = {"w_in": u(H, d_in), "b_in": u(H), "w_hid": u(H, H), "b_hid": u(1, H), "w_out": u(d_out, H), "b_out": u(d_out)}
    x0 = torch.randn(rows, d_in, generator=gen, device="cuda").to(xdtype)
    dy0 = torch.randn(rows, d_out, generator=gen, device="cuda").to(dtype)
    stream = _lib.current_stream(x0.device)
    weights = [_lib.ptr(p[k]) for k in NAMES]
    n = lib.nf_mlp_bwd_rounded_workspace_bytes(d_in, H, d_out)
    ws = torch.empty(n, dtype=torch.uint8, device="cuda")
    results = []
    # x and y on 16-byte boundaries, x alone, neither
    for px, py in ((0, 0), (0, 4), (4, 4)):
        if d_in % 8:
            px = 4
        x, dy, y = _rows(x0, px, px), _rows(dy0, py, py), _rows(torch.zeros_like(dy0), py, py)
        room = torch.full((rows * (d_in + px) + px + 8,), 7.0, dtype=xdtype, device="cuda")
        dx = room[px:].as_strided((rows, d_in), (d_in + px, 1))
        _lib.check(lib.nf_mlp_fwd(x.data_ptr(), x.stride(0), y.data_ptr(), y.stride(0), *weights, rows, d_in, H, d_out, 2, relu, code, xcode, None, 0,
                                  stream), "nf_mlp_fwd")
        out = [y.clone()]
        if xdtype == dtype:
            g = [torch.empty_like(p[k]) for k in NAMES]
            _lib.check(lib.nf_mlp_bwd_rounded(x.data_ptr(), x.stride(0), dy.data_ptr(), dy.stride(0), dx.data_ptr(), dx.stride(0), *weights,
                                              *(_lib.ptr(t) for t in g), rows, d_in, H, d_out, 2, relu, code, xcode, ws.data_ptr(), n, stream),
                       "nf_mlp_bwd_rounded")
            out += [dx.clone(), *g]
            dx.fill_(7.0)
            assert (room == 7.0).all(), "dx was written outside its rows"
        results.append(out)
    for other in results[1:]:
        for a, b in zip(results[0], other):
            assert torch.isfinite(a.float()).all()
            assert torch.equal(a, b)
