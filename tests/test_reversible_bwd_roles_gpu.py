"""The reversible backward over its passes (two couplings of 64-wide halves, four of narrower ones), its rounds (16 rows per chain wave) and
both workgroup sizes (eight chain waves from 64 rows per compute unit on), on padded rows: every part of a batch on its own gives the
stream's bits, and the batch's weight gradients are the sum of the parts'."""
import pytest
import torch

from oracle import mlp as O
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


@pytest.mark.parametrize("act", ["gelu", "silu", "relu2"])
@pytest.mark.parametrize("rows,full,H,blocks", [(33, 64, 64, 1), (1, 64, 64, 3), (50, 64, 32, 5), (70, 128, 40, 1), (16400, 16512, 64, 2), (16400, 16512, 32, 1)])
def test_rows_that_are_not_there(rows, full, H, blocks, act):
    """The biases take out a mean of the stream, so every row of the batch stays small, while on a row of zeros they alone drive a
    coupling beyond float16's range.  The kernel rounds a batch up to 16 rows per chain wave: with those rows there (copies of the first with a zero
    gradient, which add nothing) every gradient has the same bits, whatever a kernel makes of rows that are not there."""
    lib = _lib.load()
    gen = torch.Generator().manual_seed(rows + H + blocks)
    mean, step, scale = (2048.0, 1.0, 64.0) if act == "relu2" else (8192.0, 8.0, 4.0)
    w1, w2 = torch.randint(-2, 3, (blocks, 2 * H, H), generator=gen) / 16.0, torch.randint(1, 3, (blocks, 2 * H, H), generator=gen) / scale
    w1[..., 0] = -1.0
    w1 = torch.where(w1.sum(-1, keepdim=True) < 0, w1, -w1)
    k = rows % blocks  # the coupling that overflows; the others change the stream by little
    quiet = torch.arange(blocks) != k
    w1[quiet] /= 64
    w2[quiet] /= 64
    params = [w1.view(-1, H), (-mean * w1.sum(-1)).view(blocks * 2, H), w2.view(-1, H), torch.zeros(blocks * 2, H)]
    t = O.activation(params[1][2 * k + 1].half().float(), act).half().float()  # the hidden layer of a row of zeros
    assert not torch.isfinite((w2[k, H:] @ t).half()).all(), "the case does not overflow on a row of zeros"
    params = [p.half().cuda() for p in params]
    y, dy = mean + step * torch.randint(-2, 3, (full, 2 * H), generator=gen), torch.randn(full, 2 * H, generator=gen)
    y[rows:], dy[rows:] = y[0], 0.0
    y, dy = y.half().cuda(), dy.half().cuda()
    results = []
    for n in (rows, full):
        dx, x_rec = torch.empty_like(y), torch.empty_like(y)
        g = [torch.full(p.shape, 7.0, device="cuda") for p in params]
        need = lib.nf_revmlp_bwd_workspace_bytes(n, H, blocks)
        ws = torch.empty(need, dtype=torch.uint8, device="cuda")
        ptrs = [v for t in (y, dy, dx, x_rec) for v in (t.data_ptr(), t.stride(0))]
        _lib.check(lib.nf_revmlp_bwd_summed(*ptrs, *(_lib.ptr(t) for t in (*params, *g)), n, H, blocks, _lib.NF_ACT[act], _lib.NF_F16, _lib.NF_F32,
                                            ws.data_ptr(), need, _lib.current_stream(y.device)), "nf_revmlp_bwd_summed")
        results.append([dx[:rows], x_rec[:rows], *g])
    for a, b in zip(*results):
        assert torch.isfinite(b).all(), "a row of the batch overflows: the case shows nothing"
        assert torch.equal(a, b)
