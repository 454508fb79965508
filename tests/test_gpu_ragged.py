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
