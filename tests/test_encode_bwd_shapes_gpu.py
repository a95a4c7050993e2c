"""The sorted-record backward at the edges of its work distribution, against the scattered-atomic kernel."""
import ctypes

import pytest
import torch

from oracle import hash_encoding as O

pytestmark = pytest.mark.gpu
DEV = "cuda"


def _grad(x, do, E, F, T, lo, hi, L, flags=0):
    from triton_helpers_amd.layers.hash_encoding import kernel as hk

    before, hk._FLAGS = hk._FLAGS, flags
    try:
        return hk.hash_encoding_table_grad(x, do, E, F, None, T, lo, hi, L)
    finally:
        hk._FLAGS = before


# (points, levels): fill workgroups of 1, 2 and 4 levels, the last group short or of one level, the last block of points ragged
@pytest.mark.parametrize("N,L", [(16384, 16), (16385, 7), (33000, 5), (65537, 17), (70000, 6), (131073, 3), (262144, 9)])
@pytest.mark.parametrize("D,F,T,dtype", [(3, 2, 2**17, torch.float16), (3, 4, 2**15, torch.bfloat16), (2, 3, 2**16, torch.float32), (3, 2, 2**21, torch.float16)])
def test_levels_dealt_to_fill_workgroups(N, L, D, F, T, dtype):
    """A contribution is rounded to 2^-20 of its gradient (a dense cell's to 2^-17) and to 2^-30 of the level's largest, so a row's sum of n of
    them is off by less than 2^-16 of n largest gradients; the atomics' float32 sum by 2^-24 of its n partial sums."""
    torch.manual_seed(N + L)
    lo, hi = 16, 2048
    x = torch.rand(N, D, device=DEV)
    x[0], x[1] = 0.0, 1.0
    E = O.level_row_offsets(L, T, D, lo, hi)[-1]
    do = torch.randn(N, L * F, device=DEV).to(dtype)
    got = _grad(x, do, E, F, T, lo, hi, L, flags=16)
    want = _grad(x, do, E, F, T, lo, hi, L, flags=2)
    torch.testing.assert_close(got, want, rtol=1e-3, atol=1e-3)
    level_sums = lambda t: [t[a:b].double().sum(0) for a, b in zip(O.level_row_offsets(L, T, D, lo, hi)[:-1], O.level_row_offsets(L, T, D, lo, hi)[1:])]  # noqa: E731
    for l, s in enumerate(level_sums(got)):  # the weights of a cell add up to one
        torch.testing.assert_close(s, do[:, l * F : (l + 1) * F].double().sum(0), rtol=0, atol=2**-16 * 5 * 8 * N**0.5)  # independent errors


@pytest.mark.parametrize("N,L,F,dtype", [(470_000, 16, 8, torch.float32), (1_000_001, 15, 4, torch.float32), (1_000_001, 15, 8, torch.float16)])
def test_all_levels_to_a_fill_workgroup(N, L, F, dtype):
    """Gradients of more than 224 MiB.  Bounds as above."""
    assert N * L * F * dtype.itemsize > 224 * 2**20
    torch.manual_seed(N + L)
    T, lo, hi = 2**17, 16, 2048
    x = torch.rand(N, 3, device=DEV)
    E = O.level_row_offsets(L, T, 3, lo, hi)[-1]
    do = torch.randn(N, L * F, device=DEV).to(dtype)
    torch.testing.assert_close(_grad(x, do, E, F, T, lo, hi, L, flags=16), _grad(x, do, E, F, T, lo, hi, L, flags=2), rtol=1e-3, atol=2e-3)


# one block more than a workgroup's threads, a second chunk of blocks, fewer tasks than workgroups
@pytest.mark.parametrize("N", [512 * 1024 + 1, 2**20 + 77])
@pytest.mark.parametrize("cube", [1.0, 0.02])
@pytest.mark.parametrize("F,T,L,dtype", [(2, 2**19, 3, torch.float16), (2, 2**14, 2, torch.bfloat16), (3, 2**17, 2, torch.float32)])
def test_accumulation_in_chunks_of_blocks(N, cube, F, T, L, dtype):
    """Bounds as above; a row of the cube sums up to 2^17 contributions, of which float32 keeps 2^-24 of each partial sum."""
    torch.manual_seed(L)
    lo, hi = 16, 2048
    x = torch.rand(N, 3, device=DEV) * cube
    E = O.level_row_offsets(L, T, 3, lo, hi)[-1]
    do = torch.randn(N, L * F, device=DEV).to(dtype)
    got = _grad(x, do, E, F, T, lo, hi, L, flags=16)
    want = _grad(x, do, E, F, T, lo, hi, L, flags=2)
    torch.testing.assert_close(got, want, rtol=1e-3, atol=2e-3 if cube == 1.0 else 2**-16 * 2**8.5 * 5)
    assert torch.equal(got, _grad(x, do, E, F, T, lo, hi, L, flags=16))


@pytest.mark.parametrize("N", [16384, 40000, 131071, 262143])
@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("F", [2, 3])
def test_shares_of_a_bin_are_rounded_once(N, dtype, F):
    """Points on 64 corners of the cells of two dense levels: a point's weights are one and zeros, and its gradient a multiple of 2^-18 below 2^8, which the
    fixed point keeps whole.  Each of the rows gets hundreds of them, in bins that are cut into many shares: its gradient is their exact
    sum, rounded to float32 once."""
    torch.manual_seed(N)
    T, lo, hi, L = 2**19, 16, 64, 2
    cells = torch.randint(0, 16, (64, 3), device=DEV)[torch.randint(0, 64, (N,), device=DEV)]
    x = cells / 16.0
    offsets = O.level_row_offsets(L, T, 3, lo, hi)
    do = (torch.randint(-127, 128, (N, L * F), device=DEV) * torch.exp2(torch.randint(-18, 2, (N, L * F), device=DEV).float())).to(dtype)
    rows = O.encode_indices(x.cpu(), None, T, L, lo, hi)[:, :, 0].to(DEV)  # of the corner with all the weight
    want = torch.zeros(offsets[-1], F, dtype=torch.float64, device=DEV)
    for l in range(L):
        want.index_add_(0, offsets[l] + rows[:, l], do[:, l * F : (l + 1) * F].double())
    assert torch.equal(_grad(x, do, offsets[-1], F, T, lo, hi, L, flags=16), want.float())


def test_task_of_more_records_than_lds_lists():
    """2^21 points: bins of the first level hold more records than the list of a task names at a time (5760 groups of 16) and fewer than a bin
    that is cut (one and a half shares), in 1024 blocks, which a task takes as one.  Bounds as above."""
    torch.manual_seed(21)
    N, L, T, lo, hi = 2**21, 8, 2**21, 84, 512
    assert max(O.level_row_counts(L, T, 3, lo, hi)) > 128 * 8192  # blocks of 2048 points
    x = torch.rand(N, 3, device=DEV)
    cell = (x * lo).floor().long()
    first = cell[:, 0] + cell[:, 1] * lo + cell[:, 2] * lo * lo
    records = torch.bincount(torch.cat([first + dy * lo + dz * lo * lo for dy in (0, 1) for dz in (0, 1)]) >> 13).max().item()
    assert 5760 * 16 < records < N * L // 192 * 3 // 2
    E = O.level_row_offsets(L, T, 3, lo, hi)[-1]
    do = torch.randn(N, L * 2, device=DEV)
    got = _grad(x, do, E, 2, T, lo, hi, L, flags=16)
    torch.testing.assert_close(got, _grad(x, do, E, 2, T, lo, hi, L, flags=2), rtol=1e-3, atol=2e-3)
    assert torch.equal(got, _grad(x, do, E, 2, T, lo, hi, L, flags=16))


# rows of one piece of 16 bytes, of four, of eight, of numbers between them and of more; blocks of points and chunks that are short, whole and one over
@pytest.mark.parametrize("N", [8192, 8193, 8447, 8449, 9215, 9216, 9999])
@pytest.mark.parametrize("L,F,dtype", [(4, 2, torch.float16), (16, 2, torch.bfloat16), (10, 4, torch.float16), (6, 8, torch.float16), (9, 8, torch.bfloat16),
                                       (2, 2, torch.float32), (16, 2, torch.float32), (7, 4, torch.float32), (13, 4, torch.float32)])  # fmt: skip
def test_gradient_rows_turned_for_the_walk(N, L, F, dtype):
    """Rows that are not 16-byte aligned are read a value at a time and give the same bits (through the library, as the operator packs such rows
    first).  Bounds against the atomics as above."""
    from triton_helpers_amd import _lib
    from triton_helpers_amd.layers.hash_encoding.helpers import level_geometry

    torch.manual_seed(N + L)
    T, lo, hi = 2**14, 8, 512
    x = torch.rand(N, 3, device=DEV)
    E = O.level_row_offsets(L, T, 3, lo, hi)[-1]
    do = torch.randn(N, L * F, device=DEV).to(dtype)
    do[N // 2, -1] = 40.0  # the largest of the last plane
    lib, code, primes = _lib.load(), _lib.dtype_code(dtype), torch.tensor(O.PRIMES, device=DEV)
    geom = ctypes.byref(level_geometry(T, L, 3, F, lo, hi))
    size = lib.nf_hash_encode_bwd_workspace_bytes(N, geom, code, 0)
    ws = torch.empty(size, dtype=torch.uint8, device=DEV)

    def grad(rows):
        out = torch.zeros(E, F, device=DEV)
        _lib.check(lib.nf_hash_encode_bwd(x.data_ptr(), _lib.NF_F32, 3, 1, rows.data_ptr(), code, rows.stride(0), out.data_ptr(), N, geom, primes.data_ptr(), 1.0,
                                          ws.data_ptr(), size, 0, _lib.current_stream(x.device)), "backward")  # fmt: skip
        return out

    got = grad(do)
    off = torch.empty(N * L * F + 2, device=DEV, dtype=dtype)[2:].view(N, L * F).copy_(do)  # 4 or 8 bytes into a buffer
    apart = torch.zeros(N, L * F + 2, device=DEV, dtype=dtype)[:, : L * F].copy_(do)
    assert off.data_ptr() % 16 != 0 and apart.stride(0) * dtype.itemsize % 16 != 0
    assert torch.equal(got, grad(off)) and torch.equal(got, grad(apart))
    assert torch.equal(got, _grad(x, do, E, F, T, lo, hi, L))
    torch.testing.assert_close(got, _grad(x, do, E, F, T, lo, hi, L, flags=2), rtol=1e-3, atol=1e-3)
