"""The float32 forward's ways to deal rows out: one or two groups of sixteen to a wave, whole pieces or single values."""
import pytest
import torch

pytestmark = pytest.mark.gpu


# single rows, one group of sixteen more or less than the waves or the SIMDs take at once, a share that favours one group, ragged ends
@pytest.mark.parametrize("rows", [1, 17, 4096, 16385, 32768, 32769, 40003, 65537, 100003])
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
