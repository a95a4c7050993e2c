"""The operators' native host path beside torch's tracer, forward-mode derivatives, saved-tensor hooks, inference mode and graph capture."""
import pytest
import torch

from oracle import hash_encoding as O

pytestmark = pytest.mark.gpu
DEV = "cuda"
GEO = dict(max_entries_per_level=2**10, min_res=4, max_res=32, levels=4)


def _operator(name, seed=0):
    """(operator, its tensor arguments): the input in front of the parameters."""
    from triton_helpers_amd.layers.fully_fused_mlp import fully_fused_mlp
    from triton_helpers_amd.layers.hash_encoding import hash_encoding
    from triton_helpers_amd.layers.reversible_mlp import reversible_mlp

    g = torch.Generator(device=DEV).manual_seed(seed)
    u = lambda *s: torch.rand(*s, generator=g, device=DEV) - 0.5  # noqa: E731
    if name == "hash":
        rows = O.level_row_offsets(4, 2**10, 3, 4, 32)[-1]
        args = [u(100, 3) + 0.5, u(rows, 2).half()]
        fn = lambda x, table: hash_encoding(x, table, **GEO)  # noqa: E731
        fn(*args)  # the geometry's first call goes through the Python function
        return fn, args
    if name == "mlp":
        return lambda x, w_in, w_hid, w_out: fully_fused_mlp(x, w_in, None, w_out, None, w_hid), [u(*s).half() for s in ((1, 70, 32), (64, 32), (64, 64), (16, 64))]
    return lambda x, w1, w2: reversible_mlp(x, w1, None, w2, None), [u(*s).half() for s in ((70, 64), (64, 32), (64, 32))]


OPERATORS = pytest.mark.parametrize("name", ["hash", "mlp", "reversible"])


@OPERATORS
@pytest.mark.parametrize("train", [False, True])
def test_a_traced_function_runs_the_operator(name, train):
    fn, args = _operator(name)
    _, others = _operator(name, seed=1)
    if train:
        args[1:] = [t.requires_grad_() for t in args[1:]]
    traced = torch.jit.trace(lambda *a: fn(*a) * 2, tuple(args), check_trace=False)
    assert "PythonOp" in str(traced.graph) or "^" in str(traced.graph)
    assert torch.equal(traced(*others), fn(*others) * 2)


@OPERATORS
@pytest.mark.parametrize("which", ["input", "parameter"])
@pytest.mark.parametrize("mode", ["plain", "no_grad", "train"])
def test_forward_mode_derivatives_are_refused(name, which, mode):
    """A tangent that no kernel carries on raises instead of getting lost."""
    import torch.autograd.forward_ad as fw

    fn, args = _operator(name)
    if mode == "train":
        args[-1].requires_grad_()
    with fw.dual_level(), torch.set_grad_enabled(mode != "no_grad"):
        i = 0 if which == "input" else 1
        args[i] = fw.make_dual(args[i], torch.ones_like(args[i]))
        with pytest.raises(NotImplementedError):
            fn(*args)


@OPERATORS
def test_function_transforms_are_refused(name):
    """Inside a transform the autograd Functions refuse, also where the operator's own arguments are plain tensors."""
    fn, args = _operator(name)
    with pytest.raises(RuntimeError):
        torch.func.vmap(lambda s: fn(*args).sum() * s)(torch.ones(3, device=DEV))
    with pytest.raises(RuntimeError):
        torch.func.grad(lambda s: (fn(*args).float() * s).sum())(torch.ones((), device=DEV))
    fn(*args)


@OPERATORS
def test_checkpointed_gradients(name):
    """A saved-tensor hook that recomputes (non-reentrant checkpointing) runs with autograd on inside the operator's backward."""
    from torch.utils.checkpoint import checkpoint

    fn, args = _operator(name)
    scale = torch.full((), 1.5, device=DEV, dtype=torch.float16)

    def step(*a):  # the operator's tensors come out of a differentiable operation inside the checkpointed region
        return fn(a[0], *(t * scale for t in a[1:])) if name == "hash" else fn(*(t * scale for t in a))

    got = []
    for through in (lambda *a: step(*a), lambda *a: checkpoint(step, *a, use_reentrant=False)):
        leaves = [t.clone().requires_grad_(name != "hash" or i > 0) for i, t in enumerate(args)]
        y = through(*leaves)
        y.backward(torch.ones_like(y))
        got.append([y.detach(), *(t.grad for t in leaves if t.requires_grad)])
    assert all(t is not None for t in got[1])
    for a, b in zip(*got):
        torch.testing.assert_close(a, b, rtol=2**-10, atol=2**-10 * float(a.abs().max()))  # (atomics in two of the backwards: a rounding apart)


@OPERATORS
def test_saved_tensors_on_the_host(name):
    fn, args = _operator(name)
    got = []
    for hooks in (False, True):
        leaves = [t.clone().requires_grad_(i > 0) for i, t in enumerate(args)]
        if hooks:
            with torch.autograd.graph.save_on_cpu():
                y = fn(*leaves)
        else:
            y = fn(*leaves)
        y.backward(torch.ones_like(y))
        got.append([t.grad for t in leaves[1:]])
    for a, b in zip(*got):
        torch.testing.assert_close(a, b, rtol=2**-10, atol=2**-10 * float(a.abs().max()))


_PRELUDE = """
import torch
from oracle import hash_encoding as O
from triton_helpers_amd.layers.hash_encoding import hash_encoding
geo = dict(max_entries_per_level=2**10, min_res=4, max_res=32, levels=4)
x = torch.rand(100, 3, device="cuda")
table = torch.rand(O.level_row_offsets(4, 2**10, 3, 4, 32)[-1], 2, device="cuda")
"""
_ORDERS = {
    "ordinary call, inference, training": """
want = hash_encoding(x, table, **geo)
with torch.inference_mode():
    assert torch.equal(hash_encoding(x, table, **geo), want)
hash_encoding(x, table.requires_grad_(), **geo).sum().backward()
assert table.grad.any()
""",
    "inference, training": """
with torch.inference_mode():
    hash_encoding(x, table, **geo)
hash_encoding(x, table.requires_grad_(), **geo).sum().backward()
assert table.grad.any()
""",
    "one call, capture": """
want = hash_encoding(x, table, **geo)
torch.cuda.synchronize()
graph = torch.cuda.CUDAGraph()
with torch.cuda.graph(graph):
    out = hash_encoding(x, table, **geo)
for _ in range(3):
    out.zero_()
    graph.replay()
    torch.cuda.synchronize()
    assert torch.equal(out, want)
""",
}


@pytest.mark.parametrize("order", _ORDERS)
def test_default_primes_whatever_the_first_call_was(order):
    """The primes are made once per process and device, so each order of first calls has a process of its own."""
    import subprocess
    import sys

    done = subprocess.run([sys.executable, "-c", _PRELUDE + _ORDERS[order]], capture_output=True, text=True, timeout=100)
    assert done.returncode == 0, done.stderr


@pytest.mark.parametrize("N,dtype", [(1000, torch.float16), (8192, torch.float32), (20000, torch.float16)])
def test_captured_training_step_of_the_encoder(N, dtype):
    """After one ordinary step, forward and backward replay from a graph: atomics, the walk without records, sorted records."""
    from triton_helpers_amd.layers.hash_encoding import hash_encoding

    geo = dict(max_entries_per_level=2**14 if N == 8192 else 2**18, min_res=16, max_res=512, levels=4)
    E = O.level_row_offsets(4, geo["max_entries_per_level"], 3, 16, 512)[-1]
    x, do = torch.rand(N, 3, device=DEV), torch.randn(N, 8, device=DEV).to(dtype)
    table = torch.randn(E, 2, device=DEV).to(dtype).requires_grad_()

    def step():
        table.grad = None
        y = hash_encoding(x, table, **geo)
        y.backward(do)
        return y.detach(), table.grad

    stream = torch.cuda.Stream()
    stream.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(stream):
        step()
    torch.cuda.current_stream().wait_stream(stream)
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        out = step()
    for _ in range(3):
        x.uniform_()
        do.normal_()
        want = [t.clone() for t in step()]
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(out[0], want[0])
        torch.testing.assert_close(out[1], want[1], rtol=2**-10, atol=2**-10 * float(want[1].abs().max()))
