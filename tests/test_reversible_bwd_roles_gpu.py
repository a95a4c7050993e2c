"""The reversible backward over its passes (two couplings of 64-wide halves, four of narrower ones), its rounds (16 rows per chain wave) and
both workgroup sizes (eight chain waves from 64 rows per compute unit on), on padded rows: every part of a batch on its own gives the
stream's bits, and the batch's weight gradients are the sum of the parts'."""
import pytest
import torch

from triton_helpers_amd import _lib

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("H,blocks", [(64, 1), (64, 2), (64, 3), (32, 4), (32, 5), (40, 3), (7, 6)])
@pytest.mark.parametrize("act,dtype", [("gelu", torch.bfloat16), ("silu", torch.float16)])
@pytest.mark.parametrize("pad", [0, 8, 3])
@pytest.mark.parametrize("cuts", [(1, 1), (16, 65), (16384, 1), (16385, 30000), (70000, 127)])
def test_a_batch_is_its_parts(cuts, pad, act, dtype, H, blocks):
    lib = _lib.load()
    rows, width = sum(cuts), 2 * H
    gen = torch.Generator(device="cuda").manual_seed(rows + H)
    u = lambda *s: ((torch.rand(*s, generator=gen, device="cuda") * 2 - 1) / H**0.5).to(dtype)  # noqa: E731
    params = [u(blocks * 2 * H, H), u(blocks * 2, H), u(blocks * 2 * H, H), u(blocks * 2, H)]
    room = [torch.full((rows + 1, width + pad), 7.0, dtype=dtype, device="cuda") for _ in range(4)]
    y, dy, dx, x_rec = (t[:, :width] for t in room)
    y[:rows].copy_(torch.randn(rows, width, generator=gen, device="cuda"))
    dy[:rows].copy_(torch.randn(rows, width, generator=gen, device="cuda"))
    stream, code = _lib.current_stream(y.device), _lib.dtype_code(dtype)

    def run(lo, hi):
        g = [torch.full(p.shape, 7.0, device="cuda") for p in params]
        need = lib.nf_revmlp_bwd_workspace_bytes(hi - lo, H, blocks)
        ws = torch.empty(need, dtype=torch.uint8, device="cuda")
        ptrs = [v for t in (y, dy, dx, x_rec) for v in (t[lo:].data_ptr(), t.stride(0))]
        _lib.check(lib.nf_revmlp_bwd_summed(*ptrs, *(_lib.ptr(t) for t in (*params, *g)), hi - lo, H, blocks, _lib.NF_ACT[act], code, _lib.NF_F32,
                                            ws.data_ptr(), need, stream), "nf_revmlp_bwd_summed")
        return g

    whole = run(0, rows)
    kept = dx[:rows].clone(), x_rec[:rows].clone()
    assert all(torch.isfinite(t).all() for t in (*kept, *whole))
    for t in room[2:]:
        assert (t[rows:] == 7.0).all() and (t[:, width:] == 7.0).all(), "written outside the rows"
        t.fill_(7.0)
    parts = [run(0, cuts[0]), run(cuts[0], rows)]
    assert torch.equal(kept[0], dx[:rows]) and torch.equal(kept[1], x_rec[:rows])
    for a, b, c in zip(*([t.cpu() for t in g] for g in (whole, *parts))):
        # both sides add the same products in float32, in another order: at most 2^-24 of a partial sum per matrix instruction (32 rows), which
        # for the 70127 rows here is 2200 * 2^-24 = 1.3e-4 of the largest
        scale = float((b.abs() + c.abs()).max())
        off = (a - b - c).abs()
        i = int(off.argmax())
        assert float(off.max()) <= 1.5e-4 * scale, (tuple(a.shape), i, *(float(t.flatten()[i]) for t in (a, b, c)))
