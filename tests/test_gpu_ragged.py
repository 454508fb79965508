"""Widths and addresses that leave rows of B and C off vector boundaries: the lane that ends at O
takes its columns shifted left, lanes past O repeat the last ones, and C's last piece of a row goes
element by element."""
import numpy as np
import pytest

import vcsr_mc_amd as vm
from conftest import random_csr
from gpu_util import dev, row_l1_parity, say

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("tileK", [16, 64, 128])
@pytest.mark.parametrize("fp32,half_b", [(True, False), (False, True), (False, False)])
@pytest.mark.parametrize("O", [1, 3, 8, 15, 17, 31, 33, 65, 100, 127, 129, 136, 250])
def test_ragged_widths(orc, O, fp32, half_b, tileK):
    """C += A.B and C = A.B with B and C at the first and at an odd element of their buffers, light
    and heavy (shared and split) panels; NaN around B must not reach C, and nothing around C or in
    its untouched rows changes.  Bound per row as in test_gpu_spmm."""
    import torch
    rng = np.random.default_rng(O * 7 + tileK)
    M, N = 330, 2500
    rp, c, v = random_csr(rng, M, N, density=0.01, heavy_rows=2, heavy_nnz=2400, empty_frac=0.1)
    B = rng.uniform(-1, 1, (N, O)).astype(np.float32)
    C0 = rng.uniform(-1, 1, (M, O)).astype(np.float32)
    say("ragged", O, fp32, half_b, tileK)
    tau = 1e-5 if fp32 else 2e-3
    with vm.DeviceFormat.from_device_csr(dev(rp), dev(c), dev(v), M, N, fp32, 32) as f:
        R, L1 = orc.spmm_csr(rp, c, v, M, B, mode=0 if fp32 else 1, scale=f.info()["scale"])
        touched = np.diff(rp) > 0
        for shift, add in ((0, True), (1, True), (1, False)):
            bbuf = torch.full((N * O + 2 * shift + 64,), float("nan"), device="cuda",
                              dtype=torch.float16 if half_b else torch.float32)
            cbuf = torch.full((M * O + 2 * shift + 64,), 7.5, device="cuda")
            bbuf[shift:shift + N * O] = dev(B).reshape(-1)
            cbuf[shift:shift + M * O] = dev(C0).reshape(-1)
            dB = bbuf[shift:shift + N * O].view(N, O)
            dC = cbuf[shift:shift + M * O].view(M, O)
            f.spmm(dB, dC, tileK=tileK, overwrite=not add)
            torch.cuda.synchronize()
            assert bool((cbuf[:shift] == 7.5).all()) and bool((cbuf[shift + M * O:] == 7.5).all())
            C = dC.cpu().numpy()
            want = R + C0 if add else np.where(touched[:, None], R, C0)
            bound = L1 + np.abs(C0).sum(1) * add  # the final sum's rounding counts C0 too
            ok, worst, row = row_l1_parity(C[touched], want[touched], bound[touched], tau)
            assert ok, f"shift {shift} add {add} row {row}: error / bound = {worst:.3g}"
            assert C[~touched].tobytes() == C0[~touched].tobytes()


@pytest.mark.parametrize("fp32,half_b", [(True, False), (False, True)])
@pytest.mark.parametrize("N", [1 << 24, (1 << 24) + 1])
@pytest.mark.parametrize("O", [7, 8])
def test_row_numbers_around_24_bits(O, N, fp32, half_b):
    """B of 2^24 rows, the last that 24-bit row numbers reach, and of one more (64-bit addresses):
    rows that use B's first and last rows, with padding in every tile.  The sums of at most 40
    products are checked against 64 bits: 40 roundings of 2^-24 (FP32) or inputs of 11 bits."""
    import torch
    rng = np.random.default_rng(O + N % 7)
    M = 70
    cols = [np.unique(np.concatenate([rng.integers(0, N, int(rng.integers(0, 38))), [0, N - 1]]))
            for _ in range(M)]
    rp = np.zeros(M + 1, np.int32)
    rp[1:] = np.cumsum([len(x) for x in cols])
    c = np.concatenate(cols).astype(np.int32)
    v = rng.uniform(-1, 1, c.size).astype(np.float32)
    say("24-bit rows", O, N, fp32)
    B = torch.rand((N, O), device="cuda", dtype=torch.float32) - 0.5
    B = B.half() if half_b else B
    row = torch.repeat_interleave(torch.arange(M, device="cuda"), dev(np.diff(rp)).long())
    P = dev(v).double()[:, None] * B[dev(c).long()].double()
    want = torch.zeros((M, O), device="cuda", dtype=torch.float64).index_add_(0, row, P)
    bound = torch.zeros_like(want).index_add_(0, row, P.abs()).sum(1)
    with vm.DeviceFormat.from_device_csr(dev(rp), dev(c), dev(v), M, N, fp32, 32) as f:
        C = torch.zeros((M, O), device="cuda")
        f.spmm(B, C)
        torch.cuda.synchronize()
    err = (C.double() - want).abs().sum(1)
    assert bool((err <= (40 * 2.0 ** -24 if fp32 else 2e-3) * bound + 1e-30).all()), \
        float((err / bound).max())


@pytest.mark.parametrize("more", [0, 1])
@pytest.mark.parametrize("fp32,O", [(True, 256), (True, 65), (False, 128), (False, 137)])
def test_operands_around_the_32_bit_reach(fp32, O, more):
    """The largest B that 32-bit offsets reach (0xff000000 bytes, fewer than 2^24 rows) and one row
    more (64-bit addresses): rows that use its first and last rows and the ones around byte 2^31, an
    Inf in the row after a used one.  Bound as in test_row_numbers_around_24_bits."""
    import torch
    row_bytes = O * (4 if fp32 else 2)
    N = 0xff000000 // row_bytes + more
    if N > 1 << 24:
        N = (1 << 24) + more
    rng = np.random.default_rng(O + more)
    M, half = 70, 2 ** 31 // row_bytes
    edge = [0, half - 1, half, half + 1, N - 1]
    cols = [np.unique(np.concatenate([rng.integers(0, N - 2, int(rng.integers(0, 30))), edge]))
            for _ in range(M)]
    rp = np.zeros(M + 1, np.int32)
    rp[1:] = np.cumsum([len(x) for x in cols])
    c = np.concatenate(cols).astype(np.int32)
    v = rng.uniform(-1, 1, c.size).astype(np.float32)
    say("32-bit reach", fp32, O, N)
    B = torch.empty((N, O), device="cuda", dtype=torch.float32 if fp32 else torch.float16)
    B.uniform_(-0.5, 0.5)
    free = np.setdiff1d(np.array([1, half + 2, N - 2]), c)
    B[torch.from_numpy(free).cuda()] = float("inf")
    row = torch.repeat_interleave(torch.arange(M, device="cuda"), dev(np.diff(rp)).long())
    P = dev(v).double()[:, None] * B[dev(c).long()].double()
    want = torch.zeros((M, O), device="cuda", dtype=torch.float64).index_add_(0, row, P)
    bound = torch.zeros_like(want).index_add_(0, row, P.abs()).sum(1)
    with vm.DeviceFormat.from_device_csr(dev(rp), dev(c), dev(v), M, N, fp32, 32) as f:
        C = torch.zeros((M, O), device="cuda")
        f.spmm(B, C)
        torch.cuda.synchronize()
    err = (C.double() - want).abs().sum(1)
    assert bool((err <= (40 * 2.0 ** -24 if fp32 else 2e-3) * bound + 1e-30).all()), \
        float((err / bound).max())


@pytest.mark.parametrize("add", [True, False])
@pytest.mark.parametrize("empty", [0.0, 0.5])
@pytest.mark.parametrize("fp32,half_b", [(True, False), (False, True), (False, False)])
def test_operand_beyond_the_last_level_cache(fp32, half_b, empty, add):
    """B above 256 MB in tiles of few nonzeros, in natural order and with the empty rows moved last.
    Bound as in test_row_numbers_around_24_bits."""
    import torch
    rng = np.random.default_rng(11)
    M, O = 1500, 128
    N = (270 << 20) // (O * (2 if half_b else 4))
    lens = np.where(rng.random(M) < empty, 0, rng.integers(1, 38, M))
    cols = [np.unique(rng.integers(0, N, k)) for k in lens]
    rp = np.zeros(M + 1, np.int32)
    rp[1:] = np.cumsum([len(x) for x in cols])
    c = np.concatenate(cols).astype(np.int32)
    v = rng.uniform(-1, 1, c.size).astype(np.float32)
    say("far operand", fp32, half_b, empty, add)
    B = torch.empty((N, O), device="cuda", dtype=torch.float16 if half_b else torch.float32)
    B.uniform_(-0.5, 0.5)
    C0 = torch.rand((M, O), device="cuda")
    row = torch.repeat_interleave(torch.arange(M, device="cuda"), dev(np.diff(rp)).long())
    P = dev(v).double()[:, None] * B[dev(c).long()].double()
    sums = torch.zeros((M, O), device="cuda", dtype=torch.float64).index_add_(0, row, P)
    used = dev(np.diff(rp) > 0)[:, None]
    want = C0.double() + sums if add else torch.where(used, sums, C0.double())
    bound = torch.zeros_like(want).index_add_(0, row, P.abs()).sum(1) + C0.double().sum(1) * add
    with vm.DeviceFormat.from_device_csr(dev(rp), dev(c), dev(v), M, N, fp32, 32) as f:
        assert (f.row_map() is not None) == (empty > 0) and c.size < 48 * f.info()["num_chunks"]
        C = C0.clone()
        f.spmm(B, C, overwrite=not add)
        torch.cuda.synchronize()
    err = (C.double() - want).abs().sum(1)
    assert bool((err <= (40 * 2.0 ** -24 if fp32 else 2e-3) * bound + 1e-30).all()), \
        float((err / bound).max())
