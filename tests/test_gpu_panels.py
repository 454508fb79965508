"""Panels around the sizes where the layout's sort changes: one work-group in LDS up to 1024 and up
to 8192 nonzeros, through memory above, with empty rows and panels between them."""
import numpy as np
import pytest

import vcsr_mc_amd as vm
from gpu_util import dev, row_l1_parity, say

pytestmark = pytest.mark.gpu


def _csr(rng, panels, N):
    """Rows of 16-row panels with the given nonzero counts, dealt unevenly to the panel's rows."""
    lens = []
    for n in panels:
        k = np.zeros(16, np.int64)
        if n:
            w = rng.random(16) * (rng.random(16) < 0.7)
            w[rng.integers(16)] += 1.0
            k = np.minimum((n * w / w.sum()).astype(np.int64), N)
            while k.sum() < n:  # the remainder, to rows with room
                r = int(rng.integers(16))
                k[r] += min(n - int(k.sum()), N - int(k[r]))
        lens.extend(k)
    cols = [np.sort(rng.choice(N, size=int(k), replace=False)) for k in lens]
    rp = np.zeros(len(lens) + 1, np.int32)
    rp[1:] = np.cumsum(lens)
    col = np.concatenate(cols).astype(np.int32)
    return rp, col, rng.uniform(-1, 1, col.size).astype(np.float32)


@pytest.mark.parametrize("upload", [False, True])
@pytest.mark.parametrize("grouping", [0, 1, 2])
@pytest.mark.parametrize("fp32", [True, False])
def test_panel_sizes(orc, fp32, grouping, upload):
    import torch
    rng = np.random.default_rng(31)
    N, O = 9000, 40
    panels = [1, 0, 1024, 1025, 8192, 0, 8193, 3, 0, 0, 40000, 0, 144000, 700, 9001]
    rp, c, v = _csr(rng, panels, N)
    M = rp.size - 1 - 5  # the last panel is not whole
    rp = rp[:M + 1].copy()
    c, v = c[:rp[-1]], v[:rp[-1]]
    assert [int(rp[min(M, 16 * (j + 1))] - rp[16 * j]) for j in range(len(panels) - 1)] == \
        panels[:-1]
    B = rng.uniform(-1, 1, (N, O)).astype(np.float32)
    C0 = rng.uniform(-1, 1, (M, O)).astype(np.float32)
    say("panel sizes", fp32, grouping, upload)
    try:
        vm.set_row_grouping(grouping)
        f = vm.DeviceFormat.from_device_csr(dev(rp), dev(c), dev(v), M, N, fp32, 32)
        if upload:
            V = f.download()
            f.close()
            f = vm.DeviceFormat.from_host_format(V)
    finally:
        vm.set_row_grouping(1)
    with f:
        info = f.info()
        C = dev(C0)
        f.spmm(dev(B), C, tileK=64)
        torch.cuda.synchronize()
        C = C.cpu().numpy()
    if grouping == 0:
        assert info["num_panels"] == sum(n > 0 for n in panels[:-1]) + (rp[M] > rp[M // 16 * 16])
    R, L1 = orc.spmm_csr(rp, c, v, M, B, mode=0 if fp32 else 1, scale=info["scale"])
    ok, worst, row = row_l1_parity(C, R + C0, L1 + np.abs(C0).sum(1), 1e-5 if fp32 else 2e-3)
    assert ok, f"row {row}: error / bound = {worst:.3g}"
    empty = np.diff(rp) == 0
    assert C[empty].tobytes() == C0[empty].tobytes()
