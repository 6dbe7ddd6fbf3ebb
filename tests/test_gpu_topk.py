"""GPU parity: the standalone top-k operator (HIP, through the C ABI) against the CPU oracle.

Bar: values and indices bit-exact with the reference's golden, torch.topk(sorted=True)
(framework/tests/st/operation/python/vector_operator_golden.py:2247-2259), under the order its interpreter fixes for
equal values - smaller index first (framework/src/interface/interpreter/calculator/calc_torch.cpp:2481-2494).
"""
import pytest
import torch

from oracle import topk as otopk

pytestmark = pytest.mark.gpu

# the shape / k / largest columns of framework/tests/st/operation/test_case/TopK_st_test_cases.csv (values U[-100, 100])
ST_CASES = [((16, 128), -1, 10, False), ((32, 128), -1, 10, True), ((16, 128), 1, 10, False), ((32, 128), 1, 10, True),
            ((8, 8, 128), -1, 10, False), ((8, 8, 128), -1, 10, True), ((2, 8, 8, 128), -1, 10, False),
            ((2, 8, 8, 128), -1, 10, True), ((209, 40), -1, 40, False), ((739, 4257), -1, 4006, False)]


def check(x, k, dim, largest, dev):
    from pypto_amd.op import topk
    vals, idx = topk(x.to(dev), k, dim, largest)
    torch.cuda.synchronize()
    d = -1 if dim is None else dim
    x2 = x.movedim(d, -1)
    gv, gi = otopk.topk_rows(x2.reshape(-1, x2.shape[-1]), k, largest)
    gv = gv.reshape(*x2.shape[:-1], k).movedim(-1, d)
    gi = gi.reshape(*x2.shape[:-1], k).movedim(-1, d)
    assert vals.dtype == torch.float32 and idx.dtype == torch.int32 and vals.shape == gv.shape
    assert torch.equal(idx.cpu(), gi)
    assert torch.equal(vals.cpu().view(torch.int32), gv.view(torch.int32))  # bit for bit, the sign of zero included


def test_docstring_example(cuda):
    from pypto_amd.op import topk
    x = torch.tensor([[1.0, 2.0, 3.0], [1.0, 2.0, 3.0]])
    vals, idx = topk(x.to(cuda), 2, -1, True)
    assert vals.cpu().tolist() == [[3.0, 2.0], [3.0, 2.0]] and idx.cpu().tolist() == [[2, 1], [2, 1]]


@pytest.mark.parametrize("shape,dim,k,largest", ST_CASES)
def test_st_table_shapes(cuda, shape, dim, k, largest):
    g = torch.Generator().manual_seed(len(shape) * 1000 + k + largest)
    x = torch.rand(shape, generator=g) * 200 - 100
    check(x, k, dim, largest, cuda)


def test_ties_zero_signs_and_whole_rows(cuda):
    g = torch.Generator().manual_seed(5)
    x = torch.randint(-3, 4, (7, 300), generator=g).float()      # many exact ties
    x[0, ::3] = -0.0
    x[0, 1::3] = 0.0
    for largest in (True, False):
        check(x, 50, None, largest, cuda)
        check(x, 300, None, largest, cuda)                        # k = row length: a full stable sort
    check(torch.full((2, 1), 4.0), 1, None, True, cuda)
    check(torch.rand((3, 5, 9), generator=g), 4, 1, True, cuda)    # a middle dimension
    check(torch.rand((6, 17), generator=g), 3, 0, False, cuda)     # the first dimension


def test_row_slices_that_start_off_a_16_byte_boundary(cuda):
    # x[1:] of rows of 3 floats starts 12 bytes into the allocation and is contiguous: a legal operand as it is
    from pypto_amd.op import topk
    g = torch.Generator().manual_seed(9)
    x = torch.rand((5, 3), generator=g)
    xd = x.to(cuda)
    view = xd[1:]
    assert view.is_contiguous() and view.data_ptr() % 16 != 0
    vals, idx = topk(view, 2)
    gv, gi = otopk.topk_rows(x[1:], 2, True)
    assert torch.equal(idx.cpu(), gi) and torch.equal(vals.cpu(), gv)


@pytest.mark.parametrize("n,k", [(300_000, 2048), (1 << 20, 2048), (1 << 20, 64), ((1 << 24) - 3, 2048), (1 << 24, 1)])
def test_rows_up_to_the_longest(cuda, n, k):
    # beyond some 400 K elements the sampled pivot cannot hold 2048 of them and the row is selected by counting passes
    g = torch.Generator().manual_seed(n + k)
    check(torch.randn((1, n), generator=g), k, None, True, cuda)


def test_long_rows_go_through_the_radix_select(cuda):
    g = torch.Generator().manual_seed(6)
    x = torch.randn((3, 131072), generator=g)
    check(x, 2048, None, True, cuda)
    x = torch.randint(-50, 50, (2, 20000), generator=g).float()   # heavy ties across the selection boundary
    check(x, 1000, None, True, cuda)
    check(x, 17, None, False, cuda)


def test_errors(cuda):
    from pypto_amd.error import FeError
    from pypto_amd.op import topk
    x = torch.zeros((2, 10000), device=cuda)
    with pytest.raises(FeError, match="k <= 2048"):
        topk(x, 3000)
    with pytest.raises(FeError, match="1 <= k"):
        topk(x[:, :8].contiguous(), 9)
    with pytest.raises(FeError, match="float32"):
        topk(x.half(), 2)


@pytest.mark.parametrize("n", [128, 129, 1025, 4095, 4096, 4097, 16384, 16385, 32768, 33000, 70001])
def test_row_lengths_at_the_kernels_edges(cuda, n):
    """One element more or less than a lane's, the candidate list's and a request group's capacity; bell-shaped rows (the
    sampled pivot serves), heavy ties, a row in step with the samples (every 16th element of 65536 is large: the pivot
    comes out too high), one far outlier, and infinities."""
    g = torch.Generator().manual_seed(n)
    x = torch.randn((5, n), generator=g)
    x[1] = torch.randint(-2, 3, (n,), generator=g).float()
    x[2, ::max(n // 4096, 2)] += 100.0
    x[3, n // 3] = 1e30
    x[4, n // 2] = float("inf")
    x[4, 0] = float("-inf")
    for k in (1, min(n, 2048)):
        check(x, k, None, True, cuda)
    check(x, min(n, 100), None, False, cuda)


@pytest.mark.parametrize("n,k", [(4097, 2048), (4100, 1), (16383, 2048), (16384, 100), (16385, 2048), (32767, 1000), (32768, 2048),
                                 (32769, 2048), (65537, 5)])
def test_rows_around_the_sample_and_what_registers_hold(cuda, n, k):
    """Rows just within and beyond what a lane's registers hold: the sample comes from them, or from memory.  Scores the sample sees
    as they are (a bell), sorted by position, alternating with the lanes of a wavefront, tied, and with infinities and zeros of both
    signs; selections bit for bit."""
    g = torch.Generator().manual_seed(n)
    bell = torch.randn((1, n), generator=g)
    lanes = bell + 8 * ((torch.arange(n) % 4) == 1).float()        # all the best in one of every four elements
    blocks = bell + 8 * ((torch.arange(n) // 64 % 4) == 2).float()  # all the best in one wavefront of every four
    special = bell.clone()
    special[0, ::7], special[0, 1::7] = 0.0, -0.0
    special[0, 5], special[0, n - 1] = float("inf"), float("-inf")
    tied = torch.randint(-40, 40, (1, n), generator=g).float()
    x = torch.cat([bell, bell.sort(-1).values, lanes, blocks, special, tied])
    for largest in (True, False):
        check(x, k, -1, largest, cuda)
