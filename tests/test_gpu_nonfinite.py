"""An Inf or NaN of B stays in its own output column: the padding slots of a tile, and of a row-step
batch, multiply zeros, whatever the B row they are loaded from holds."""
import numpy as np
import pytest

import vcsr_mc_amd as vm
from conftest import random_csr
from gpu_util import dev, say

pytestmark = pytest.mark.gpu

# (FP32 format, FP32 row steps, binary16 B)
KINDS = [(False, False, True), (False, False, False), (True, False, False), (True, True, False)]
BAD = [np.inf, np.nan]


def _format(rp, c, v, M, N, fp32, steps):
    vm.set_fp32_row_steps(vm.FP32_ROW_STEPS_ALWAYS if steps else vm.FP32_ROW_STEPS_OFF)
    try:
        f = vm.DeviceFormat.from_device_csr(dev(rp), dev(c), dev(v), M, N, fp32, 32)
    finally:
        vm.set_fp32_row_steps(vm.FP32_ROW_STEPS_AUTO)
    assert (f.info()["num_row_step_batches"] > 0) == steps
    return f


def _product(f, B, b16, M, tileK, add):
    import torch
    C = torch.zeros((M, B.shape[1]), dtype=torch.float32, device="cuda")
    f.spmm(dev(B).half() if b16 else dev(B), C, tileK=tileK, overwrite=not add)
    torch.cuda.synchronize()
    return C.cpu().numpy()


@pytest.mark.parametrize("bad", BAD)
@pytest.mark.parametrize("per_row", [1, 5, 31, 32, 33, 37])
@pytest.mark.parametrize("fp32,steps,b16", KINDS)
def test_every_row_holds_the_column(fp32, steps, b16, per_row, bad):
    """Rows that all hold the same columns, the last of them `bad` in one element B[last, k]: every
    row's output is `bad` there, every other element what it is without it."""
    M, N = 37, 64
    cols = np.arange(1, 1 + per_row)
    rp = (np.arange(M + 1) * per_row).astype(np.int32)
    c = np.tile(cols, M).astype(np.int32)
    v = np.full(c.size, 0.5, np.float32)
    say("holder", fp32, steps, b16, per_row, bad)
    with _format(rp, c, v, M, N, fp32, steps) as f:
        for tileK, O in ((16, 16), (32, 64), (64, 40), (128, 128), (128, 100), (32, 7)):
            for k in sorted({0, 1, O // 2, O - 1}):
                B = np.ones((N, O), np.float32)
                B[cols[-1], k] = bad
                want = np.full((M, O), 0.5 * per_row, np.float32)
                want[:, k] = bad
                for add in (True, False):
                    C = _product(f, B, b16, M, tileK, add)
                    assert np.array_equal(C, want, equal_nan=True), (tileK, O, k, add)


@pytest.mark.parametrize("bad", BAD)
@pytest.mark.parametrize("fp32,steps,b16", KINDS)
def test_other_columns_unchanged(fp32, steps, b16, bad):
    """A whole column of B bad, for a matrix with tiles and batches of every fill (light, heavy and
    split panels): the other output columns are, bit for bit, those of a clean B (split panels, whose
    parts meet in any order: finite)."""
    rng = np.random.default_rng(5)
    M, N = 700, 1500
    rp, c, v = random_csr(rng, M, N, density=0.01, heavy_rows=3, heavy_nnz=1400, empty_frac=0.2)
    say("columns", fp32, steps, b16, bad)
    with _format(rp, c, v, M, N, fp32, steps) as f:
        split = f.info()["num_split_panels"] > 0
        for tileK, O in ((16, 16), (32, 96), (64, 64), (128, 128), (128, 99)):
            B = rng.uniform(-1, 1, (N, O)).astype(np.float32)
            clean = _product(f, B, b16, M, tileK, True)
            for k in sorted({0, 3, O // 2, O - 1}):
                P = B.copy()
                P[:, k] = bad
                C = _product(f, P, b16, M, tileK, True)
                others = np.arange(O) != k
                assert np.isfinite(C[:, others]).all(), (tileK, O, k)
                if not split:
                    assert np.array_equal(C[:, others], clean[:, others]), (tileK, O, k)
                used = np.diff(rp) > 0
                assert not np.isfinite(C[used, k]).any()
                assert not C[~used].any()


@pytest.mark.parametrize("bad", BAD + [1e6])
@pytest.mark.parametrize("tileK", [32, 128])
def test_converted_b(tileK, bad):
    """FP16 formats that convert an FP32 B first, row-major and O-tile-major (1e6 overflows
    binary16): the bad column alone changes."""
    rng = np.random.default_rng(6)
    M, O, k = 30000, 128, 64
    key = np.unique(rng.integers(0, M, (M, 16)) + M * np.arange(M)[:, None])
    rp = np.searchsorted(key, M * np.arange(M + 1)).astype(np.int32)
    c, v = (key % M).astype(np.int32), rng.uniform(-1, 1, key.size).astype(np.float32)
    B = rng.uniform(-1, 1, (M, O)).astype(np.float32)
    say("converted", tileK, bad)
    with _format(rp, c, v, M, M, False, False) as f:
        info = f.info()
        assert c.size >= 12 * M and c.size < 48 * info["num_chunks"] and info["num_split_panels"] == 0
        clean = _product(f, B, False, M, tileK, True)
        B[:, k] = bad
        C = _product(f, B, False, M, tileK, True)
        others = np.arange(O) != k
        assert np.array_equal(C[:, others], clean[:, others])
        assert not np.isfinite(C[np.diff(rp) > 0, k]).any()
