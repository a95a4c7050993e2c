"""The float32 forward's ways to deal rows out: one or two groups of sixteen to a wave, whole pieces or single values."""
import pytest
import torch

pytestmark = pytest.mark.gpu


# single rows, one group of sixteen more or less than the waves or the SIMDs take at once, a share that favours one group, a last round of a few
# chunks, of most and of all, ragged ends
@pytest.mark.parametrize("rows", [1, 17, 4096, 16320, 16384, 16385, 32768, 32769, 40003, 65536, 65537, 88000, 100003, 131089])
@pytest.mark.parametrize("d_in,hidden,d_out,depth,shift", [(32, 64, 16, 2, 0), (64, 64, 64, 8, 0), (36, 32, 4, 7, 0), (35, 64, 3, 2, 0), (32, 64, 16, 1, 1), (64, 16, 64, 9, 0)])
def test_every_share_gives_the_same_rows(rows, d_in, hidden, d_out, depth, shift):
    """A row's result does not depend on its batch.  Against 64 bits: a layer rounds each of its up to 66 additions to 2^-24 of the sum of the
    magnitudes, which the layers behind it (ReLU is 1-Lipschitz) carry on with the magnitudes of their weights."""
    from triton_helpers_amd.layers.fully_fused_mlp import fully_fused_mlp

    g = torch.Generator(device="cuda").manual_seed(rows + depth)
    u = lambda *s: (torch.rand(*s, generator=g, device="cuda") * 2 - 1) * s[-1] ** -0.5  # noqa: E731
    x = torch.empty(rows * d_in + shift, device="cuda")[shift:].view(1, rows, d_in).copy_(torch.randn(1, rows, d_in, generator=g, device="cuda"))
    w = {"w_in": u(hidden, d_in), "b_in": u(hidden), "w_out": u(d_out, hidden), "b_out": u(d_out), "w_hid": None, "b_hid": None}
    if depth > 1:
        w["w_hid"], w["b_hid"] = u((depth - 1) * hidden, hidden), u(depth - 1, hidden)
    with torch.no_grad():
        y = fully_fused_mlp(x, activation="relu", **w)
        pieces = torch.cat([fully_fused_mlp(p, activation="relu", **w) for p in x.split(20000, dim=1)], dim=1)
    assert torch.equal(y, pieces)
    h, a = x.double(), x.double().abs()
    layers = [(w["w_in"], w["b_in"])] + [(w["w_hid"][k * hidden : (k + 1) * hidden], w["b_hid"][k]) for k in range(depth - 1)] + [(w["w_out"], w["b_out"])]
    for k, (m, b) in enumerate(layers):
        h, a = h @ m.double().T + b.double(), a @ m.double().abs().T + b.double().abs()
        if k < depth:
            h = h.relu()
    assert ((y.double() - h).abs() <= a * (66 * (depth + 1) * 2.0**-24)).all()


@pytest.mark.parametrize("rows", [16385, 33000, 70001])
@pytest.mark.parametrize("d_in,hidden,d_out,depth", [(32, 16, 16, 1), (64, 64, 64, 3), (35, 32, 1, 4), (16, 32, 4, 9)])
@pytest.mark.parametrize("act", ["silu", "relu2", "none"])
def test_pairs_of_groups_give_the_rows_of_single_ones(rows, d_in, hidden, d_out, depth, act):
    from triton_helpers_amd.layers.fully_fused_mlp import fully_fused_mlp

    g = torch.Generator(device="cuda").manual_seed(rows + depth)
    u = lambda *s: (torch.rand(*s, generator=g, device="cuda") * 2 - 1) * s[-1] ** -0.5  # noqa: E731
    x, w = torch.randn(1, rows, d_in, generator=g, device="cuda"), [u(hidden, d_in), u(hidden), u(d_out, hidden), u(d_out)]
    w += [u((depth - 1) * hidden, hidden), u(depth - 1, hidden)] if depth > 1 else [None, None]
    with torch.no_grad():
        y = fully_fused_mlp(x, *w, activation=act)
        assert torch.equal(y, torch.cat([fully_fused_mlp(p, *w, activation=act) for p in x.split(4096, dim=1)], dim=1))
    assert y.isfinite().all()


@pytest.mark.parametrize("d_in,hidden,d_out,depth,bias", [(32, 64, 16, 2, True), (64, 64, 64, 2, False), (35, 32, 3, 1, True), (33, 16, 17, 2, True), (16, 64, 64, 1, False)])
@pytest.mark.parametrize("rows", [1, 1000, 4097])
def test_written_gradients_are_the_added_ones(rows, d_in, hidden, d_out, depth, bias):
    """nf_mlp_bwd_f32 over buffers of NaN against nf_mlp_bwd over zeros: the same bits, and nothing beside the gradients is touched."""
    from triton_helpers_amd import _lib

    lib = _lib.load()
    g = torch.Generator(device="cuda").manual_seed(rows + d_in)
    u = lambda *s: (torch.rand(*s, generator=g, device="cuda") * 2 - 1) * s[-1] ** -0.5  # noqa: E731
    x, dy = u(rows, d_in), u(rows, d_out)
    w = [u(hidden, d_in), u(hidden) if bias else None, u(hidden, hidden) if depth == 2 else None, u(1, hidden) if depth == 2 and bias else None,
         u(d_out, hidden), u(d_out) if bias else None]  # fmt: skip
    n = lib.nf_mlp_workspace_bytes(rows, hidden, depth, _lib.NF_ACT["relu"], 1, _lib.NF_F32)
    ws, got = torch.empty(n, dtype=torch.uint8, device="cuda"), []
    for fill in (0.0, float("nan")):
        grads = [None if t is None else torch.full((t.numel() + 64,), fill, device="cuda") for t in w]
        dx = torch.empty_like(x)
        args = [x.data_ptr(), d_in, dy.data_ptr(), d_out, dx.data_ptr(), d_in, *map(_lib.ptr, w), *map(_lib.ptr, grads), rows, d_in, hidden, d_out, depth, _lib.NF_ACT["relu"]]
        types, call = ([_lib.NF_F32, _lib.NF_F32], lib.nf_mlp_bwd) if fill == 0.0 else ([], lib.nf_mlp_bwd_f32)
        _lib.check(call(*args, *types, ws.data_ptr(), n, _lib.current_stream(x.device)), "backward")
        got.append([dx] + [t[:-64] for t in grads if t is not None])
        rest = torch.cat([t[-64:] for t in grads if t is not None])
        assert rest.isnan().all() if fill != fill else (rest == 0).all()
    assert all(torch.equal(a, b) for a, b in zip(*got))


def test_written_gradients_need_rows_and_at_most_two_hidden_layers():
    from triton_helpers_amd import _lib

    lib = _lib.load()
    for rows, depth in ((0, 2), (8, 3)):
        assert lib.nf_mlp_bwd_f32(1, 32, 1, 16, None, 32, 1, None, 1, None, 1, None, 1, None, 1, None, 1, None, rows, 32, 64, 16, depth, 1, None, 0, None) == -2
