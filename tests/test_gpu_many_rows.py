"""Matrices of so many rows, panels or clusters that a launch of one wave or work-group for each would
pass 2^32 work-items in one dimension of its grid."""
import pytest

import vcsr_mc_amd as vm
from gpu_util import say

pytestmark = pytest.mark.gpu


def _rows(torch, M, nnz, N, g):
    """CSR of about nnz distinct nonzeros spread over all rows, and the row of each."""
    r = torch.randint(0, M, (nnz,), device="cuda", generator=g)
    c = torch.randint(0, N, (nnz,), device="cuda", generator=g)
    r[0], r[1] = 0, M - 1
    key = torch.unique(r * N + c)
    r = key // N
    rp = torch.zeros(M + 1, dtype=torch.int32, device="cuda")
    rp[1:] = torch.cumsum(torch.bincount(r, minlength=M), 0)
    return rp, (key - r * N).int(), r


@pytest.mark.parametrize("M,nnz", [((1 << 26) + 5, 200000), ((1 << 26) + 5, 1 << 28),
                                   ((1 << 28) + 9, 200000), (1 << 20, 200000),
                                   ((1 << 20) + 1, 1 << 21), ((1 << 20) + 1, (1 << 21) + 6000)])
def test_relabel_rows(M, nnz):
    """Columns relabelled and rows sorted again, each row on its own or all by one sort."""
    import torch
    say("relabel", M, nnz)
    g = torch.Generator(device="cuda")
    g.manual_seed(M % 1000 + 1)
    N = 1000
    rp, col, row = _rows(torch, M, nnz, N, g)
    val = torch.arange(col.numel(), device="cuda", dtype=torch.float32)
    position = torch.randperm(N, device="cuda", generator=g).int()
    new, order = torch.sort(row * N + position[col.long()])
    want_val = val[order]
    vm.apply_column_permutation_device(rp, col, val, M, N, position, None, None, 0)
    torch.cuda.synchronize()
    assert torch.equal(col.long(), new % N)
    assert torch.equal(val, want_val)


@pytest.mark.parametrize("fp32", [True, False])
@pytest.mark.parametrize("M,nnz", [((1 << 28) + 9, 200000), ((1 << 28) + 9, 1 << 28)])
def test_build_many_panels(M, nnz, fp32):
    """2^24 panels and more, few of them or nearly all with nonzeros."""
    import torch
    say("panels", M, nnz, fp32)
    g = torch.Generator(device="cuda")
    g.manual_seed(7)
    N, O = 64, 2
    rp, col, row = _rows(torch, M, nnz, N, g)
    val = torch.randint(1, 5, (col.numel(),), device="cuda", generator=g).float()
    B = torch.randint(-4, 5, (N, O), device="cuda", generator=g).float()  # exact sums
    want = torch.full((M, O), 1.0, device="cuda")
    C = want.clone()
    want.index_add_(0, row, val[:, None] * B[col.long()])
    del row
    with vm.DeviceFormat.from_device_csr(rp, col, val, M, N, fp32, 32) as f:
        f.spmm(B if fp32 else B.half(), C)
        torch.cuda.synchronize()
    # sums of whole numbers; binary16 rounds the scaled values of A
    assert torch.equal(C, want) if fp32 else bool(((C - want).abs() < 0.25).all())


def test_group_many_rows():
    """Row grouping of more than 2^26 clusters: pairs of rows 2^25 apart share their column."""
    import torch
    say("clusters")
    half = (1 << 25) + 64
    M, N, O = 2 * half, half, 1
    rp = torch.arange(M + 1, device="cuda", dtype=torch.int32)
    col = torch.arange(half, device="cuda", dtype=torch.int32).repeat(2)
    val = torch.ones(M, device="cuda")
    B = torch.randint(-4, 5, (N, O), device="cuda").float()
    C = torch.zeros((M, O), device="cuda")
    vm.set_row_grouping(vm.ROW_GROUPING_ALWAYS)
    try:
        with vm.DeviceFormat.from_device_csr(rp, col, val, M, N, True, 32) as f:
            groups = torch.from_numpy(f.row_map().reshape(-1, 16) % half).cuda().sort(1).values
            assert bool((groups[:, ::2] == groups[:, 1::2]).all())  # whole pairs in a panel
            f.spmm(B, C)
            torch.cuda.synchronize()
    finally:
        vm.set_row_grouping(vm.ROW_GROUPING_AUTO)
    assert torch.equal(C, B.repeat(2, 1))
