"""GPU parity of the reversible MLP against the CPU oracle (through the C ABI).

The reference holds no reversible MLP, so parity with the reference is UNPINNED for this layer; the
oracle is pinned by mathematics (tests/test_oracle_mlp.py).  Tolerance: rtol 2e-2 / atol 1e-2 on y,
dx and (relative to their scale) dw/db, against the oracle on the 16-bit-rounded inputs with the
stream rounded to the storage dtype after every coupling, plus half a storage ulp of the stream's largest
magnitude per coupling (see ``_close``).  ReLU is left out of the gradient check on purpose: the backward rebuilds the
inputs from 16-bit outputs, so pre-activations within rounding of zero switch their gate and move
single gradients by whole weights; the smooth activations (GELU is the BASELINE one) have no such jump.
"""
import pytest
import torch

from oracle import reversible as R

pytestmark = pytest.mark.gpu
DEV = "cuda"
RTOL, ATOL = 2e-2, 1e-2


def _rk():
    from triton_helpers_amd.layers.reversible_mlp import kernel

    return kernel


def _params(blocks, H, bias, dtype, seed=0):
    g = torch.Generator().manual_seed(seed)
    u = lambda *s: ((torch.rand(*s, generator=g) * 2 - 1) / H**0.5).to(dtype)  # noqa: E731
    return u(blocks * 2 * H, H), (u(blocks * 2, H) if bias else None), u(blocks * 2 * H, H), (u(blocks * 2, H) if bias else None)


EPS = {torch.bfloat16: 2.0**-8, torch.float16: 2.0**-11}


def _close(got, want, what, scale_rel=False, blocks=4):
    """rtol 2e-2 / atol 1e-2, plus what the storage format itself costs: the backward hands the stream (x, dx) from
    one coupling to the next in the 16-bit storage dtype, so every element of the stream is rounded once per
    coupling, by at most half an ulp of the stream's magnitude (2^-9 of it in bfloat16, 2^-12 in float16).  An element
    whose terms cancel to ~0 keeps that absolute error, hence the term ``blocks * eps / 2 * max|want|``.  Weight
    gradients (``scale_rel``) are sums over all rows and are compared relative to their largest magnitude."""
    dtype = got.dtype
    got, want = got.detach().cpu().float(), want.float()
    peak = float(want.abs().max())
    atol = ATOL + blocks * 0.5 * EPS.get(dtype, 2.0**-8) * peak
    if scale_rel:
        atol = max(atol, RTOL * peak)
    torch.testing.assert_close(got, want, rtol=RTOL, atol=atol, msg=lambda m: f"{what}: {m}")


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("act", ["gelu", "silu", "none"])
@pytest.mark.parametrize("bias", [False, True])
@pytest.mark.parametrize(
    "rows,H,blocks",
    [(1000, 64, 4), (37, 64, 1), (300, 32, 2), (129, 16, 3), (513, 64, 6), (64, 20, 2),
     # unragged full-width shapes: GELU takes the kernels without per-tile checks and one backward launch for all couplings
     (1024, 64, 4), (96, 64, 1), (640, 64, 6), (512, 32, 3)],
)
def test_forward_backward(rows, H, blocks, bias, act, dtype):
    rk = _rk()
    torch.manual_seed(0)
    w1, b1, w2, b2 = _params(blocks, H, bias, dtype)
    x = torch.randn(rows, 2 * H).to(dtype)
    dy = torch.randn(rows, 2 * H).to(dtype)
    # the forward kernel keeps the stream in float32 for 4 couplings per launch
    want_y = R.rev_forward(x, w1, b1, w2, b2, act, round_to=dtype, stream_round_every=4).to(dtype)
    want = R.rev_backward(x, dy, w1, b1, w2, b2, act, round_to=dtype)
    leaves = [None if t is None else t.to(DEV).requires_grad_(True) for t in (w1, b1, w2, b2)]
    xd = x.to(DEV).requires_grad_(True)
    y = rk.reversible_mlp(xd, *leaves, act)
    assert y.shape == x.shape and y.dtype == dtype
    _close(y, want_y, "y", blocks=(blocks + 3) // 4)  # the forward rounds the stream once per four couplings
    y.backward(dy.to(DEV))
    _close(xd.grad, want["dx"], "dx", blocks=blocks)
    for name, leaf in zip(("dw1", "db1", "dw2", "db2"), leaves):
        if leaf is not None:
            _close(leaf.grad, want[name], name, scale_rel=True, blocks=blocks)


def _misaligned(t):
    """The same values as a view whose rows start 2 bytes off an 8-byte boundary (forces the checked-tile kernels)."""
    buf = torch.zeros(t.shape[0], t.shape[1] + 4, dtype=t.dtype, device=t.device)
    view = buf[:, 1 : 1 + t.shape[1]]
    view.copy_(t)
    assert view.data_ptr() % 8 != 0
    return view


def _offset_8_bytes(t):
    """The same values as a view whose rows start 8 bytes off a 16-byte boundary: fine for the forward's 8-byte tiles, not
    for the backward's 16-byte accesses, so the backward must take its checked kernels."""
    buf = torch.zeros(t.shape[0], t.shape[1] + 8, dtype=t.dtype, device=t.device)
    view = buf[:, 4 : 4 + t.shape[1]]
    view.copy_(t)
    assert view.data_ptr() % 16 == 8 and view.stride(0) % 8 == 0
    return view


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("act", ["gelu", "relu", "silu"])
@pytest.mark.parametrize("rows,H,blocks", [(4096, 64, 4), (1024, 32, 2), (288, 64, 5)])
def test_unchecked_and_checked_kernels_agree(rows, H, blocks, act, dtype):
    """Aligned unragged calls run the kernels without per-tile checks (the backward as one launch over all
    couplings); a misaligned view of the same data runs the checked kernels, one backward launch per coupling.
    Same arithmetic per row: y and dx must agree bit for bit, the weight gradients up to the order of their float32
    atomics.  (This is also what covers ReLU's backward, which the oracle comparison leaves out.)"""
    rk = _rk()
    torch.manual_seed(1)
    w1, b1, w2, b2 = (t.to(DEV) for t in _params(blocks, H, True, dtype))
    x = torch.randn(rows, 2 * H, device=DEV).to(dtype)
    dy = torch.randn(rows, 2 * H, device=DEV).to(dtype)
    results = []
    for variant in (lambda t: t, _misaligned, _offset_8_bytes):
        leaves = [t.clone().requires_grad_(True) for t in (w1, b1, w2, b2)]
        xv = variant(x).detach().requires_grad_(True)
        y = rk.reversible_mlp(xv, *leaves, act)
        y.backward(variant(dy))
        results.append((y.detach(), xv.grad, [t.grad for t in leaves]))
    (y0, dx0, g0) = results[0]
    for y1, dx1, g1 in results[1:]:
        assert torch.equal(y0, y1)
        assert torch.equal(dx0, dx1)
        for a, b in zip(g0, g1):
            scale = float(b.float().abs().max())
            torch.testing.assert_close(a.float(), b.float(), rtol=1e-2, atol=1e-2 * scale)


@pytest.mark.parametrize("act", ["gelu", "relu", "silu"])
@pytest.mark.parametrize("rows,H,blocks", [(4096 + 17, 64, 4), (8192 + 31, 32, 2), (5000, 64, 1)])
def test_large_ragged_batch_runs_as_main_part_plus_tail(rows, H, blocks, act):
    """From 4096 rows a batch whose row count is not a multiple of 32 runs as two calls: the multiple of 32 (the kernels
    without per-tile checks where the rest allows) and the last rows.  Rows are independent, so y and dx equal, bit for
    bit, what the two parts give when the caller splits them, and the weight gradients are the sum of the parts'."""
    rk = _rk()
    dtype = torch.bfloat16
    torch.manual_seed(3)
    w1, b1, w2, b2 = (t.to(DEV) for t in _params(blocks, H, True, dtype))
    x = torch.randn(rows, 2 * H, device=DEV).to(dtype)
    dy = torch.randn(rows, 2 * H, device=DEV).to(dtype)

    def run(xs, dys):
        leaves = [t.clone().requires_grad_(True) for t in (w1, b1, w2, b2)]
        xv = xs.clone().requires_grad_(True)
        y = rk.reversible_mlp(xv, *leaves, act)
        y.backward(dys)
        return y.detach(), xv.grad, [t.grad.float() for t in leaves]

    m = rows - rows % 32
    y, dx, g = run(x, dy)
    y0, dx0, g0 = run(x[:m], dy[:m])
    y1, dx1, g1 = run(x[m:], dy[m:])
    assert torch.equal(y, torch.cat([y0, y1])) and torch.equal(dx, torch.cat([dx0, dx1]))
    for a, b0, b1_ in zip(g, g0, g1):
        want = b0 + b1_
        torch.testing.assert_close(a, want, rtol=2e-2, atol=2e-2 * float(want.abs().max()))


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("rows,H,blocks", [(1000, 64, 4), (1024, 64, 4), (512, 32, 3)])
def test_relu_forward(rows, H, blocks, dtype):
    rk = _rk()
    torch.manual_seed(0)
    w1, b1, w2, b2 = _params(blocks, H, True, dtype)
    x = torch.randn(rows, 2 * H).to(dtype)
    want_y = R.rev_forward(x, w1, b1, w2, b2, "relu", round_to=dtype, stream_round_every=4).to(dtype)
    y = rk.reversible_mlp(x.to(DEV), *(t.to(DEV) for t in (w1, b1, w2, b2)), "relu")
    _close(y, want_y, "y", blocks=(blocks + 3) // 4)  # the forward rounds the stream once per four couplings


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
def test_inverse_round_trip(dtype):
    """inverse(forward(x)) == x up to the 16-bit rounding of the stream (the in-kernel reconstruction)."""
    rk = _rk()
    torch.manual_seed(0)
    w1, b1, w2, b2 = (None if t is None else t.to(DEV) for t in _params(4, 64, True, dtype))
    x = torch.randn(3, 700, 128, device=DEV).to(dtype)
    y = rk.reversible_mlp(x, w1, b1, w2, b2)
    xr = rk.reversible_mlp_inverse(y, w1, b1, w2, b2)
    eps = 2.0**-7 if dtype == torch.bfloat16 else 2.0**-10
    torch.testing.assert_close(xr.float(), x.float(), rtol=8 * eps, atol=8 * eps)


def test_full_size_config3_properties():
    """BASELINE configs[3] at 2^20 rows: round trip, linearity of dx in dy, and a 2048-row sample against the oracle."""
    rk = _rk()
    torch.manual_seed(0)
    w1, b1, w2, b2 = _params(4, 64, False, torch.bfloat16)
    dev = [None if t is None else t.to(DEV) for t in (w1, b1, w2, b2)]
    rows = 2**20
    x = torch.randn(rows, 128, device=DEV).bfloat16()
    y = rk.reversible_mlp(x, *dev)
    idx = torch.randperm(rows)[:2048].to(DEV)
    _close(y[idx], R.rev_forward(x[idx].cpu(), w1, b1, w2, b2), "y sample")
    xr = rk.reversible_mlp_inverse(y, *dev)
    torch.testing.assert_close(xr.float(), x.float(), rtol=2.0**-4, atol=2.0**-4)
    dy = torch.randn(rows, 128, device=DEV).bfloat16()
    xg = x.clone().requires_grad_(True)
    rk.reversible_mlp(xg, *dev).backward(dy)
    xg2 = x.clone().requires_grad_(True)
    rk.reversible_mlp(xg2, *dev).backward(dy * 2)
    torch.testing.assert_close(xg2.grad.float(), xg.grad.float() * 2, rtol=RTOL, atol=ATOL)
    want = R.rev_backward(x[idx].cpu(), dy[idx].cpu(), w1, b1, w2, b2)
    _close(xg.grad[idx], want["dx"], "dx sample")


def test_float32_storage():
    """float32 tensors run with float16 operands and float32 accumulation; everything comes back as float32."""
    rk = _rk()
    torch.manual_seed(0)
    w1, b1, w2, b2 = _params(3, 64, True, torch.float32)
    x = torch.randn(500, 128)
    dy = torch.randn(500, 128)
    want_y = R.rev_forward(x, w1, b1, w2, b2, "gelu")
    want = R.rev_backward(x, dy, w1, b1, w2, b2, "gelu")
    leaves = [t.to(DEV).requires_grad_(True) for t in (w1, b1, w2, b2)]
    xd = x.to(DEV).requires_grad_(True)
    y = rk.reversible_mlp(xd, *leaves, "gelu")
    assert y.dtype == torch.float32
    _close(y, want_y, "y")
    y.backward(dy.to(DEV))
    assert xd.grad.dtype == torch.float32 and all(t.grad.dtype == torch.float32 for t in leaves)
    _close(xd.grad, want["dx"], "dx")
    for name, leaf in zip(("dw1", "db1", "dw2", "db2"), leaves):
        _close(leaf.grad, want[name], name, scale_rel=True)
    xr = rk.reversible_mlp_inverse(y.detach(), *(t.detach() for t in leaves))
    assert xr.dtype == torch.float32
    torch.testing.assert_close(xr.cpu(), x, rtol=2.0**-7, atol=2.0**-7)


def test_module_and_errors():
    from triton_helpers_amd.layers.reversible_mlp import ReversibleMLP

    rk = _rk()
    torch.manual_seed(0)
    layer = ReversibleMLP(128, 4).to(DEV)
    x = torch.randn(2, 50, 128, device=DEV, requires_grad=True)
    with torch.autocast(device_type="cuda", dtype=torch.float16):
        y = layer(x)
    assert y.dtype == torch.float16 and y.shape == x.shape
    y.sum().backward()
    assert layer.w1.grad is not None and layer.b2.grad is not None and x.grad is not None
    assert set(layer.state_dict().keys()) == {"w1", "w2", "b1", "b2"}
    w = torch.zeros(256, 64, device=DEV).half()
    with pytest.raises(AssertionError):
        rk.reversible_mlp(torch.zeros(4, 127, device=DEV).half(), w, None, w, None)
    with pytest.raises(AssertionError):
        rk.reversible_mlp(torch.zeros(4, 128, device=DEV).half(), w[:100], None, w[:100], None)
    with pytest.raises(NotImplementedError):
        rk.reversible_mlp(torch.zeros(4, 128, device=DEV).double(), w.double(), None, w.double(), None)
    # a float32 module without autocast runs too (float16 operands inside) and returns float32
    y32 = layer(x.detach())
    assert y32.dtype == torch.float32
    torch.testing.assert_close(y32, y.detach().float(), rtol=2e-2, atol=1e-2)


@pytest.mark.parametrize(
    "case,rows,H,blocks,act,bias,dtype",
    [
        (22, 1000, 16, 5, "gelu", False, torch.bfloat16),
        (47, 40000, 48, 8, "gelu", False, torch.bfloat16),
        (93, 1024, 64, 4, "none", True, torch.bfloat16),
        (111, 4097, 32, 4, "none", False, torch.bfloat16),
    ],
)
def test_cases_that_once_missed_the_tolerance(case, rows, H, blocks, act, bias, dtype):
    """Four randomly drawn shapes on which a single element of dx came out 10-15 % beyond an absolute tolerance that
    was scaled with the RMS of dx: the element was one whose terms cancel, and its error was the 16-bit rounding of
    the stream at the coupling boundaries, which scales with the stream's magnitude, not with the element's.  They
    are kept as regression cases for the bound stated in ``_close``."""
    rk = _rk()
    torch.manual_seed(case)
    w1, b1, w2, b2 = _params(blocks, H, bias, dtype, seed=case)
    x = torch.randn(rows, 2 * H).to(dtype)
    dy = torch.randn(rows, 2 * H).to(dtype)
    want_y = R.rev_forward(x, w1, b1, w2, b2, act, round_to=dtype, stream_round_every=4).to(dtype)
    want = R.rev_backward(x, dy, w1, b1, w2, b2, act, round_to=dtype)
    leaves = [None if t is None else t.to(DEV).requires_grad_(True) for t in (w1, b1, w2, b2)]
    xd = x.to(DEV).requires_grad_(True)
    y = rk.reversible_mlp(xd, *leaves, act)
    _close(y, want_y, "y", blocks=(blocks + 3) // 4)  # the forward rounds the stream once per four couplings
    y.backward(dy.to(DEV))
    _close(xd.grad, want["dx"], "dx", blocks=blocks)
    for name, leaf in zip(("dw1", "db1", "dw2", "db2"), leaves):
        if leaf is not None:
            _close(leaf.grad, want[name], name, scale_rel=True, blocks=blocks)


@pytest.mark.parametrize("rows,H,blocks,act,bias,dtype", [
    (1, 64, 1, "gelu", True, torch.bfloat16), (96, 64, 4, "gelu", True, torch.bfloat16), (513, 48, 2, "gelu", False, torch.float16),
    (4096 + 17, 64, 2, "silu", True, torch.float16), (8192, 32, 4, "gelu", True, torch.bfloat16), (640, 32, 3, "relu", False, torch.float16),
    (300, 20, 2, "none", True, torch.bfloat16), (256 * 128 * 3, 64, 4, "gelu", True, torch.float16),
])
def test_backward_without_a_workspace(rows, H, blocks, act, bias, dtype):
    """``nf_revmlp_bwd`` adds float32 gradients with atomics and takes no scratch: the stream has the bits of the entry with a workspace,
    and the gradients are its sums of at most 257 float32 parts in another order (257 * 2^-24 of the parts, which cancel a little)."""
    from triton_helpers_amd import _lib as L_

    lib = L_.load()
    g = torch.Generator().manual_seed(rows)
    w1, b1, w2, b2 = (None if t is None else t.to(DEV) for t in _params(blocks, H, bias, dtype, seed=rows))
    y, dy = (torch.randn(rows, 2 * H, generator=g).to(dtype).to(DEV) for _ in range(2))
    dt, code, stream = L_.dtype_code(dtype), L_.NF_ACT[act], L_.current_stream(y.device)
    need = lib.nf_revmlp_bwd_workspace_bytes(rows, H, blocks)
    ws = torch.empty(need, dtype=torch.uint8, device=DEV)
    got = []
    for summed in (False, True):
        dx, x_rec = torch.empty_like(y), torch.empty_like(y)
        grads = [None if t is None else torch.full(t.shape, 0.5, device=DEV) for t in (w1, b1, w2, b2)]
        head = (y.data_ptr(), 2 * H, dy.data_ptr(), 2 * H, dx.data_ptr(), 2 * H, x_rec.data_ptr(), 2 * H, *(L_.ptr(t) for t in (w1, b1, w2, b2, *grads)))
        if summed:
            rc = lib.nf_revmlp_bwd_summed(*head, rows, H, blocks, code, dt, L_.NF_F32, ws.data_ptr(), need, stream)
        else:
            rc = lib.nf_revmlp_bwd(*head, rows, H, blocks, code, dt, stream)
        assert rc == 0, lib.nf_last_error()
        got.append((dx, x_rec, [None if t is None else t - (0.0 if summed else 0.5) for t in grads]))
    assert torch.equal(got[0][0], got[1][0]) and torch.equal(got[0][1], got[1][1])
    for a, b in zip(got[0][2], got[1][2]):
        if b is not None:
            assert float((a - b).norm()) <= 1e-4 * float(b.norm()) + 1e-5 * b.numel() ** 0.5
