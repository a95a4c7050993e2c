"""Edges of the tiles, splits and dispatch rules of the kernels, against the generic kernels and the oracle."""
import pytest
import torch

from oracle import hash_encoding as O

pytestmark = pytest.mark.gpu
DEV = "cuda"


@pytest.mark.parametrize("N", [2**16 - 1, 2**16, 2**16 + 1, 2**17, 2**17 + 1, 196608, 196609, 2**18 + 1, 304800, 3 * 2**18 + 1, 2**20 - 1, 2**20 + 3])
@pytest.mark.parametrize("dims,dtype", [(3, torch.float16), (2, torch.bfloat16), (3, torch.float32)])
def test_forward_sweep_deals_out_every_point(N, dims, dtype, monkeypatch):
    """The sweep's workgroups take equal shares of one to four points per thread: every output row, also of a ragged last
    wave, has the bits of the per-(point, level) kernel (flag 1)."""
    from triton_helpers_amd.layers.hash_encoding import kernel as hk

    T, L, lo, hi = 2**15, 8, 8, 300
    torch.manual_seed(3)
    x = torch.rand(N, dims, device=DEV)
    table = torch.randn(O.level_row_offsets(L, T, dims, lo, hi)[-1], 2, device=DEV).to(dtype)
    outs = []
    for flags in (0, 1):
        monkeypatch.setattr(hk, "_FLAGS", flags)
        outs.append(hk.hash_encoding(x, table, None, None, T, lo, hi, L))
    assert torch.equal(outs[0], outs[1])


@pytest.mark.parametrize("N", [1, 4096, 16384, 16385, 8 * 1024 * 3 + 1, 2**18 - 1, 2**20 + 5])
@pytest.mark.parametrize("dims,F,T,L,dtype", [
    (3, 2, 2**14, 16, torch.float32), (3, 2, 2**14, 4, torch.float16), (3, 2, 2**15, 16, torch.bfloat16), (2, 2, 2**14, 2, torch.float16),
    (3, 4, 2**14, 16, torch.float16), (2, 2, 2**14, 16, torch.float32), (2, 4, 2**13, 2, torch.bfloat16), (3, 2, 2**11, 16, torch.float16),
])
def test_forward_with_levels_in_lds(N, dims, F, T, L, dtype, monkeypatch):
    """Levels of up to 128 KiB are gathered from LDS, one or two to a workgroup: the bits of the per-(point, level) kernel
    (flag 1), on points of the upper edge too, and into rows of a wider output."""
    from triton_helpers_amd.layers.hash_encoding import kernel as hk

    torch.manual_seed(6)
    x = torch.rand(N, dims, device=DEV)
    x[: N // 8, 0] = 1.0
    x[: N // 16] = 1.0
    table = torch.randn(O.level_row_offsets(L, T, dims, 16, 512)[-1], F, device=DEV).to(dtype)
    tail = torch.zeros(N, 4, device=DEV, dtype=dtype)
    outs = []
    for flags in (0, 1):
        monkeypatch.setattr(hk, "_FLAGS", flags)
        outs.append([hk.hash_encoding(x, table, f, None, T, 16, 512, L) for f in (None, tail)])
    assert torch.equal(outs[0][0], outs[1][0]) and torch.equal(outs[0][1], outs[1][1])


@pytest.mark.parametrize("N", [1, 255, 257, 16384, 40960, 40961, 53248, 53249, 65535, 65537])
@pytest.mark.parametrize("dims,F,T,L,dtype", [
    (3, 2, 2**19, 16, torch.float16), (3, 4, 2**19, 16, torch.bfloat16), (3, 4, 2**20, 8, torch.float16), (3, 8, 2**17, 16, torch.float16), (3, 2, 2**18, 4, torch.float32),
    (3, 4, 2**16, 8, torch.float32), (2, 2, 2**16, 2, torch.float32), (2, 4, 2**15, 4, torch.float16), (3, 2, 2**19, 32, torch.float16),
])
def test_forward_per_point_and_level(N, dims, F, T, L, dtype, monkeypatch):
    """Rows of 4, 8 and 16 bytes, units of work dealt out in turn and XCD by XCD: the bits of the generic kernel (flag 1), on the upper edge too,
    and into rows of a wider output, which may not be aligned."""
    from triton_helpers_amd.layers.hash_encoding import kernel as hk

    torch.manual_seed(8)
    x = torch.rand(N, dims, device=DEV)
    x[: N // 8, 0] = 1.0
    x[: N // 16] = 1.0
    table = torch.randn(O.level_row_offsets(L, T, dims, 16, 4000)[-1], F, device=DEV).to(dtype)
    tail = torch.zeros(N, 3, device=DEV, dtype=dtype)
    outs = []
    for flags in (0, 1):
        monkeypatch.setattr(hk, "_FLAGS", flags)
        outs.append([hk.hash_encoding(x, table, f, None, T, 16, 4000, L) for f in (None, tail)])
    assert torch.equal(outs[0][0], outs[1][0]) and torch.equal(outs[0][1], outs[1][1])


def _grads(tensors):
    return [None if t is None else t.grad for t in tensors]


@pytest.mark.parametrize("depth,bias,dtype", [(1, True, torch.bfloat16), (2, False, torch.float16), (2, True, torch.float32), (4, True, torch.float32)])
def test_mlp_node_equals_the_python_function(depth, bias, dtype):
    """The native node and the autograd Function of the same name come to the same launches: the same bits, for the weights' gradients are
    summed in a fixed order (or, four layers deep in float32, are two partial sums)."""
    from triton_helpers_amd.layers.fully_fused_mlp.kernel import _fully_fused_mlp, fully_fused_mlp

    torch.manual_seed(4)
    u = lambda *s: (torch.rand(*s, device=DEV) - 0.5).to(dtype)  # noqa: E731
    H, n = 64, depth - 1
    base = [u(3, 41, 32), u(H, 32), u(H) if bias else None, u(16, H), u(16) if bias else None, u(n * H, H) if n else None, u(n, H) if n and bias else None]
    got = []
    for fn in (fully_fused_mlp, _fully_fused_mlp.apply):
        leaves = [None if t is None else t.clone().requires_grad_() for t in base]
        y = fn(*leaves, "relu")
        y.backward(torch.ones_like(y))
        got.append([y.detach(), *_grads(leaves)])
    for a, b in zip(*got):
        assert (a is None and b is None) or (a.dtype == b.dtype and torch.equal(a, b))


@pytest.mark.parametrize("depth,act", [(2, "relu"), (3, "relu"), (2, "silu")])
def test_mlp_under_autocast(depth, act):
    """float32 parameters under autocast: float16 operands, float32 gradients of the parameters, equal to those of float16
    parameters up to the rounding that those end with."""
    from triton_helpers_amd.layers.fully_fused_mlp import fully_fused_mlp

    torch.manual_seed(5)
    u = lambda *s: torch.rand(*s, device=DEV) - 0.5  # noqa: E731
    H, n = 64, depth - 1
    base = [u(1, 1000, 32), u(H, 32), u(H), u(16, H), u(16), u(n * H, H), u(n, H)]
    got = []
    for cast in (True, False):
        leaves = [(t.clone() if cast else t.half()).requires_grad_() for t in base]
        with torch.autocast("cuda", dtype=torch.float16, enabled=cast):
            y = fully_fused_mlp(*leaves, activation=act)
        assert y.dtype == torch.float16
        y.backward(torch.full_like(y, 0.01))
        got.append([y.detach(), *_grads(leaves)])
    assert torch.equal(got[0][0], got[1][0])
    for a, b in zip(got[0][1:], got[1][1:]):
        assert a.dtype == torch.float32
        torch.testing.assert_close(a, b.float(), rtol=2e-3, atol=2e-3 * float(b.abs().max()))


@pytest.mark.parametrize("case", ["cpu table", "features", "coords grad", "float64", "small table", "strided"])
def test_hash_node_hands_unusual_calls_to_the_python_function(case):
    from triton_helpers_amd.layers.hash_encoding import hash_encoding

    geo = dict(max_entries_per_level=2**10, min_res=4, max_res=32, levels=4)
    E = O.level_row_offsets(4, 2**10, 3, 4, 32)[-1]
    x, table = torch.rand(100, 3, device=DEV), torch.randn(E, 2, device=DEV)
    want = hash_encoding(x, table, **geo)
    if case == "cpu table":
        with pytest.raises(AssertionError):
            hash_encoding(x, table.cpu(), **geo)
    elif case == "features":
        out = hash_encoding(x, table, torch.ones(100, 3, device=DEV), **geo)
        assert torch.equal(out[:, :8], want) and torch.equal(out[:, 8:], torch.ones(100, 3, device=DEV))
    elif case == "coords grad":
        with pytest.raises(AssertionError):
            hash_encoding(x.clone().requires_grad_(), table, **geo)
    elif case == "float64":
        with pytest.raises(TypeError):
            hash_encoding(x.double(), table, **geo)
    elif case == "small table":
        with pytest.raises(AssertionError):
            hash_encoding(x, table[:-1], **geo)
    else:
        wide = torch.zeros(100, 5, device=DEV)
        wide[:, ::2] = x
        assert torch.equal(hash_encoding(wide[:, ::2], table, **geo), want)
        assert torch.equal(hash_encoding(x.view(4, 25, 3), table, **geo).view(100, 8), want)


@pytest.mark.parametrize("N,dims,F,T,L,hi,dtype,layout", [
    (8193, 3, 2, 2**16, 8, 1024, torch.float16, "uniform"),         # one record block and one point
    (16383, 3, 1, 2**15, 8, 512, torch.bfloat16, "uniform"),        # odd feature counts: one feature in the last pass
    (16385, 2, 3, 2**16, 8, 2048, torch.float32, "uniform"),
    (50000, 3, 4, 2**17, 8, 2048, torch.bfloat16, "uniform"),
    (200001, 3, 2, 2**19, 16, 7006, torch.float16, "corner"),       # all points in one corner: bins of many tasks
    (200001, 3, 2, 2**16, 16, 1024, torch.float32, "corner"),
    (2**18 - 1, 3, 2, 2**21, 8, 7006, torch.float16, "uniform"),    # the largest batch of small blocks over a wide level
    (2**18, 3, 2, 2**21, 8, 7006, torch.float16, "uniform"),        # wide blocks, ragged and not
    (2**18 + 2049, 3, 2, 2**21, 8, 7006, torch.float32, "corner"),
    (2**18 + 1, 2, 2, 2**21, 8, 7006, torch.bfloat16, "uniform"),
    (2**18 + 1, 3, 2, 2**21, 16, 7006, torch.float16, "corner"),    # more bins than the table of tasks holds
    (2**18 + 1, 3, 2, 2**21, 16, 7006, torch.float16, "cell"),      # heavy bins behind it, and fewer slots than shares
    (20001, 3, 1, 2**21, 16, 7006, torch.bfloat16, "cell"),
    (2**19, 2, 2, 2**22, 16, 30000, torch.float32, "cell"),
    (150001, 3, 2, 2**23, 8, 4096, torch.float16, "cell"),
])
def test_sorted_backward_writes_the_table(N, dims, F, T, L, hi, dtype, layout, monkeypatch):
    """The backward of the sorted records, added to a float32 table and written in the table's own type: every row against
    float64 sums over the corner rows, rows that no point touches are zeros, and a second run has the same bits."""
    from triton_helpers_amd import _lib
    from triton_helpers_amd.layers.hash_encoding import kernel as hk

    monkeypatch.setattr(hk, "_FLAGS", _lib.NF_HASH_BWD_RECORDS)
    _check_table_gradient(N, dims, F, T, L, hi, dtype, layout, same_bits=True)


@pytest.mark.parametrize("N,dims,F,T,L,hi,dtype,layout", [
    (4096, 3, 2, 2**14, 16, 512, torch.float16, "uniform"),       # two bins a level, one or two slices of the points
    (4097, 3, 2, 2**14, 16, 512, torch.float32, "corner"),
    (2**18 + 77, 3, 2, 2**14, 16, 512, torch.float32, "uniform"),  # a task per unit
    (50001, 2, 4, 2**13, 8, 512, torch.bfloat16, "corner"),       # one bin a level, two feature pairs
    (1024, 3, 1, 2**14, 4, 256, torch.float16, "uniform"),        # odd feature counts, the smallest batch
    (1025, 3, 3, 2**16, 4, 256, torch.float32, "uniform"),
    (5000, 1, 2, 2**12, 4, 9000, torch.bfloat16, "uniform"),
    (6143, 3, 2, 2**16, 16, 1024, torch.float16, "uniform"),      # either side of the smallest batch with bins to choose from
    (6144, 3, 2, 2**16, 16, 1024, torch.float16, "corner"),
    (59000, 3, 2, 2**16, 16, 1024, torch.bfloat16, "corner"),     # slices of bins
    (20000, 3, 4, 2**15 - 3, 8, 512, torch.float16, "uniform"),   # a size that is not a power of two
])
def test_backward_walk_writes_the_table(N, dims, F, T, L, hi, dtype, layout):
    """Small batches and small tables without records: as above."""
    _check_table_gradient(N, dims, F, T, L, hi, dtype, layout, same_bits=N != 6143)


@pytest.mark.parametrize("dims,F,dtype", [(3, 2, torch.float16), (2, 2, torch.bfloat16), (3, 4, torch.float32), (2, 4, torch.float16), (3, 2, torch.float32)])
@pytest.mark.parametrize("N", [1, 17, 1000, 16383])
def test_backward_of_small_batches(N, dims, F, dtype):
    """A lane per (point, level, corner, feature), atomics: every row against float64 sums."""
    _check_table_gradient(N, dims, F, 2**19, 4, 4096, dtype, "uniform", same_bits=False)


def test_backward_atomics_of_a_batch_beyond_one_launch():
    """2^27 + 3 points of four features without a workspace are more threads than a launch has: no point is left out.  Every point's
    weights sum to one, so a gradient of ones sums to the points; 8 * 2^27 / 2^19 = 2048 adds of about 1/8 per row are off by at most
    2048 * 2^-24 of a row's 256."""
    from triton_helpers_amd import _lib as L_
    from triton_helpers_amd.layers.hash_encoding.helpers import level_geometry

    lib, n, T = L_.load(), 2**27 + 3, 2**19
    geom = level_geometry(T, 2, 3, 4, 1000, 2000)
    x = torch.rand(n, 3, device=DEV)
    do = torch.ones(n, 8, device=DEV, dtype=torch.float16)
    do[:, 4:] = 0
    do[-1, :4] = 4096.0
    x[-1] = 0.0  # the last point's weights are all on its first corner
    de = torch.zeros(2 * T, 4, device=DEV)
    pi = torch.tensor(O.PRIMES, dtype=torch.int64, device=DEV)
    rc = lib.nf_hash_encode_bwd(x.data_ptr(), 0, 3, 1, do.data_ptr(), L_.NF_F16, 8, de.data_ptr(), n, geom, pi.data_ptr(), 1.0, None, 0, 0, L_.current_stream(x.device))
    assert rc == 0, lib.nf_last_error()
    total = de[:T].double().sum(0)
    assert not de[T:].any() and float((total - (n - 1 + 4096)).abs().max()) <= 2048 * 2**-24 * n
    assert float(de[0].min()) > 4096.0


def _check_table_gradient(N, dims, F, T, L, hi, dtype, layout, same_bits):
    from triton_helpers_amd.layers.hash_encoding import kernel as hk

    g = torch.Generator(device=DEV).manual_seed(N)
    x = torch.rand(N, dims, generator=g, device=DEV)
    if layout == "corner":
        x[: N // 2] *= 0.05
    if layout == "cell":
        x[: N // 2] = 0.4 + 1e-6 * x[: N // 2]
    *first, E = O.level_row_offsets(L, T, dims, 16, hi)
    first = torch.tensor(first, device=DEV).view(1, L, 1)
    do = torch.randn(N, L * F, generator=g, device=DEV).to(dtype)
    want = torch.zeros(E, F, device=DEV, dtype=torch.float64)
    count = torch.zeros(E, device=DEV)
    for part in range(0, N, 2**16):
        rows, w = hk.hash_encoding_indices(x[part : part + 2**16], None, T, 16, hi, L, return_weights=True)
        rows += first
        d = do[part : part + 2**16].double().view(-1, L, 1, F) * w.double().unsqueeze(-1)
        want.index_add_(0, rows.reshape(-1), d.reshape(-1, F))
        count.index_add_(0, rows.reshape(-1), torch.ones(rows.numel(), device=DEV))
    table = torch.zeros(E, F, device=DEV, dtype=dtype).requires_grad_()
    grads = []
    for _ in range(2):
        table.grad = None
        hk.hash_encoding(x, table, None, None, T, 16, hi, L).backward(do)
        grads.append(table.grad)
    assert grads[0].dtype == dtype and (not same_bits or torch.equal(grads[0], grads[1]))
    added = torch.full((E, F), 0.5, device=DEV)
    hk.hash_encoding_table_grad(x, do, E, F, None, T, 16, hi, L, out=added)
    atol = 1e-4 + 2e-5 * float(want.abs().max())
    torch.testing.assert_close(added.double() - 0.5, want, rtol=1e-3, atol=atol)
    ulp = {torch.float16: 2**-10, torch.bfloat16: 2**-7, torch.float32: 1e-5}[dtype]
    torch.testing.assert_close(grads[0].double(), want, rtol=ulp, atol=atol)
    assert not grads[0][count == 0].any()


@pytest.mark.parametrize("rows,H,blocks,act,dtype", [
    (1, 64, 4, "gelu", torch.bfloat16), (31, 32, 1, "silu", torch.float16), (32, 64, 5, "relu", torch.bfloat16), (128 * 3, 48, 2, "gelu", torch.float16),
    (4096 + 17, 64, 2, "gelu", torch.bfloat16), (256 * 128 + 32, 64, 1, "silu", torch.float16), (3 * 12 * 256 * 32, 32, 4, "gelu", torch.bfloat16),
])
def test_reversible_gradients_of_few_and_many_workgroups(rows, H, blocks, act, dtype):
    """The weights' gradients are summed over one slot per workgroup, the last rows' launch included: against float32 autograd of
    the plain composition, and the same bits in a second run."""
    from triton_helpers_amd.layers.reversible_mlp import reversible_mlp

    g = torch.Generator(device=DEV).manual_seed(rows)
    u = lambda *s: (torch.rand(*s, generator=g, device=DEV) * 2 - 1).mul(H**-0.5).to(dtype)  # noqa: E731
    w = [u(blocks * 2 * H, H), u(blocks * 2, H), u(blocks * 2 * H, H), u(blocks * 2, H)]
    x, dy = torch.randn(rows, 2 * H, generator=g, device=DEV).to(dtype), torch.randn(rows, 2 * H, generator=g, device=DEV).to(dtype)
    got = []
    for _ in range(2):
        leaves = [t.clone().requires_grad_() for t in (x, *w)]
        y = reversible_mlp(*leaves, activation=act)
        y.backward(dy)
        got.append([y.detach(), *_grads(leaves)])
    assert all(torch.equal(a, b) for a, b in zip(*got))
    f = {"gelu": torch.nn.functional.gelu, "silu": torch.nn.functional.silu, "relu": torch.relu}[act]
    leaves = [t.float().requires_grad_() for t in (x, *w)]
    a, b = leaves[0][:, :H], leaves[0][:, H:]
    for k in range(2 * blocks):
        w1, b1, w2, b2 = (t[k * (t.shape[0] // (2 * blocks)) : (k + 1) * (t.shape[0] // (2 * blocks))] for t in leaves[1:])
        s = f((b if k % 2 == 0 else a) @ w1.t() + b1) @ w2.t() + b2
        a, b = (a + s, b) if k % 2 == 0 else (a, b + s)
    ref = torch.cat([a, b], 1)
    ref.backward(dy.float())
    for p, q in zip(got[0], [ref.detach(), *_grads(leaves)]):
        # (a ReLU takes its gates from rebuilt inputs: some open or close)
        assert float((p.float() - q).norm()) <= (6e-2 if act == "relu" else 2e-2) * float(q.norm())


@pytest.mark.parametrize("rows", [1, 16, 17, 2048 * 16 + 5])
@pytest.mark.parametrize("d_in,H,d_out,hidden,act,bias", [
    (3, 64, 1, 0, "relu", True), (32, 64, 16, 1, "silu", True), (33, 64, 16, 1, "relu2", False), (32, 32, 17, 1, "none", True), (64, 64, 64, 1, "relu", True),
    (35, 16, 16, 0, "silu", False), (16, 64, 64, 0, "relu2", True), (64, 32, 33, 0, "relu", True),
])
def test_float32_mlp_gradients(rows, d_in, H, d_out, hidden, act, bias):
    """One and two hidden layers of float32 run backward in one launch: against float64 autograd, with the same bits in a second run."""
    from triton_helpers_amd.layers.fully_fused_mlp import fully_fused_mlp
    from triton_helpers_amd.layers.fully_fused_mlp.kernel import _activate

    g = torch.Generator(device=DEV).manual_seed(rows)
    u = lambda *s: torch.rand(*s, generator=g, device=DEV) * 2 - 1  # noqa: E731
    w = [u(H, d_in), u(H) if bias else None, u(d_out, H), u(d_out) if bias else None, u(H, H) if hidden else None, u(1, H) if hidden and bias else None]
    x, dy = u(1, rows, d_in), u(1, rows, d_out)
    runs = []
    for _ in range(2):
        leaves = [None if t is None else t.clone().requires_grad_() for t in (x, *w)]
        fully_fused_mlp(*leaves, activation=act).backward(dy)
        runs.append(_grads(leaves))
    assert all(a is None or torch.equal(a, b) for a, b in zip(*runs))
    leaves = [None if t is None else t.double().requires_grad_() for t in (x, *w)]
    lin = lambda h, m, b: h @ m.t() + (0 if b is None else b)  # noqa: E731
    h = _activate(lin(leaves[0], leaves[1], leaves[2]), act)
    if hidden:
        h = _activate(lin(h, leaves[5], None if leaves[6] is None else leaves[6][0]), act)
    lin(h, leaves[3], leaves[4]).backward(dy.double())
    for a, b in zip(runs[0], _grads(leaves)):
        if b is not None:
            assert float((a.double() - b).norm()) <= 1e-5 * float(b.norm())


@pytest.mark.parametrize("d_in,H,d_out,depth,act,bias", [(32, 64, 16, 2, "silu", True), (64, 64, 64, 4, "relu2", False), (35, 64, 3, 3, "relu", True), (64, 64, 33, 9, "relu", True),
                                                         (16, 16, 1, 3, "silu", True), (48, 32, 33, 9, "silu", False), (27, 32, 64, 2, "relu", True), (32, 64, 16, 1, "relu", True)])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
def test_mlp_forward_of_every_batch_size(d_in, H, d_out, depth, act, bias, dtype):
    """A wave takes sixteen rows of a small batch at a time and 32 of a large one, and the weights are staged as one list where their matrices are
    16-byte aligned: a row's result has the same bits in every batch, and from matrices that are not."""
    from triton_helpers_amd.layers.fully_fused_mlp import fully_fused_mlp

    torch.manual_seed(depth)
    n = depth - 1
    u = lambda *s: ((torch.rand(*s, device=DEV) * 2 - 1) / s[-1] ** 0.5).to(dtype)  # noqa: E731
    w = {"w_in": u(H, d_in), "w_out": u(d_out, H), "b_in": u(H) if bias else None, "b_out": u(d_out) if bias else None,
         "w_hid": u(n * H, H) if n else None, "b_hid": u(n, H) if n and bias else None}
    x = torch.randn(1, 131_090, d_in, device=DEV).to(dtype)
    want = fully_fused_mlp(x, **w, activation=act)
    for rows in (1, 17, 4097, 32768, 32769, 65536, 65537, 131_072, 131_073):
        assert torch.equal(fully_fused_mlp(x[:, :rows], **w, activation=act), want[:, :rows]), rows
    shifted = {}
    for k, t in w.items():
        if t is not None:
            flat = torch.empty(t.numel() + 1, dtype=dtype, device=DEV)
            flat[1:] = t.flatten()
            t = flat[1:].view(t.shape)
        shifted[k] = t
    assert torch.equal(fully_fused_mlp(x[:, :4097], **shifted, activation=act), want[:, :4097])
