"""Handles on several host threads at once.  A handle holds all of its format's state; what the
library shares between handles is read-only or synchronised (the row-grouping mode and the RCM
limits are atomics, the per-device scratch lookup takes a mutex).  So four threads that each
build their own format and multiply on their own stream, at the same time, must produce bit for
bit what the same calls produce one after another on one thread.  The matrices have no split
panels, so every product is deterministic (no atomics)."""
import threading

import numpy as np
import pytest

import vcsr_mc_amd as vm
from conftest import random_csr
from gpu_util import row_l1_parity, say

pytestmark = pytest.mark.gpu

TAU = {True: 1e-5, False: 2e-3}


def _cases():
    out = []
    for i in range(4):
        rng = np.random.default_rng(4100 + i)
        M, N = 2500 + 700 * i, 2000 + 300 * i
        rp, c, v = random_csr(rng, M, N, nnz_per_row=5 + 2 * i, empty_frac=0.1 * i)
        fp32 = bool(i % 2)
        O = 40 + 32 * i
        B = rng.uniform(-1, 1, (N, O)).astype(np.float32)
        if not fp32:
            B = B.astype(np.float16).astype(np.float32)
        C0 = rng.uniform(-1, 1, (M, O)).astype(np.float32)
        out.append(dict(rp=rp, c=c, v=v, M=M, N=N, fp32=fp32, B=B, C0=C0))
    return out


def _run(case, stream):
    """Build, then C += A.B and C = A.B twice each on `stream`; returns the four results."""
    import torch
    with torch.cuda.stream(stream):
        d = {k: torch.from_numpy(case[k]).to("cuda", non_blocking=False)
             for k in ("rp", "c", "v", "B", "C0")}
        outs = []
        with vm.DeviceFormat.from_device_csr(d["rp"], d["c"], d["v"], case["M"], case["N"],
                                             case["fp32"], 32, stream=stream) as f:
            info = f.info()
            for overwrite in (False, False, True, True):
                C = d["C0"].clone()
                f.spmm(d["B"], C, tileK=128, overwrite=overwrite, stream=stream)
                outs.append(C)
        stream.synchronize()
        return info, [C.cpu().numpy() for C in outs]


def test_handles_on_threads(orc):
    import torch
    cases = _cases()
    say("threads: serial")
    serial = [_run(case, torch.cuda.Stream()) for case in cases]
    for (info, outs), case in zip(serial, cases):
        assert info["num_split_panels"] == 0, info
        R, L1 = orc.spmm_csr(case["rp"], case["c"], case["v"], case["M"], case["B"],
                             mode=0 if case["fp32"] else 1, scale=info["scale"])
        touched = np.diff(case["rp"]) > 0
        for k, got in enumerate(outs):
            base = case["C0"].astype(np.float64).copy()
            if k >= 2:
                base[touched] = 0.0
            ok, worst, row = row_l1_parity(got, R + base, L1 + np.abs(base).sum(axis=1),
                                           TAU[case["fp32"]])
            assert ok, f"serial call {k}: row {row}: error / bound = {worst:.3g}"
    for rep in range(3):
        say("threads: concurrent", rep)
        results = [None] * len(cases)
        errors = []
        start = threading.Barrier(len(cases))

        def worker(i):
            try:
                stream = torch.cuda.Stream()
                start.wait(timeout=60)
                results[i] = _run(cases[i], stream)
            except BaseException as e:  # reported on the main thread
                errors.append((i, repr(e)))

        threads = [threading.Thread(target=worker, args=(i,)) for i in range(len(cases))]
        for t in threads:
            t.start()
        for t in threads:
            t.join(timeout=120)
        assert not any(t.is_alive() for t in threads), "a worker did not finish"
        assert not errors, errors
        for i, ((info_s, outs_s), (info_c, outs_c)) in enumerate(zip(serial, results)):
            assert info_s == info_c, i
            for k, (a, b) in enumerate(zip(outs_s, outs_c)):
                assert np.array_equal(a, b), (rep, i, k)


def test_scratch_kept_between_calls_is_bounded():
    """Scratch blocks of finished builds serve later ones: builds of growing sizes, with a refused
    one between them, multiply as the first did, and leave at most 2 GiB (and the runtime's own
    granules) held once the formats are closed."""
    import torch
    say("kept scratch")
    rng = np.random.default_rng(77)
    rp, c, v = random_csr(rng, 3000, 2500, nnz_per_row=9)
    B = rng.uniform(-1, 1, (2500, 48)).astype(np.float32)
    d = lambda a: torch.from_numpy(a).cuda()
    dB, first = d(B), None
    torch.cuda.synchronize()
    free0 = torch.cuda.mem_get_info()[0]
    for k in range(6):
        n = 200000 << k  # rows of one nonzero each, in a column of its own
        ones = torch.ones(n, device="cuda")
        seq = torch.arange(n + 1, device="cuda", dtype=torch.int32)
        with vm.DeviceFormat.from_device_csr(seq, seq[:n], ones, n, n, True, 32) as big:
            assert big.info()["nnz"] == n
        with pytest.raises(vm.VCSRMCError):
            vm.DeviceFormat.from_device_csr(seq, torch.zeros_like(seq[:n]) - 1, ones, n, n, True, 32)
        del ones, seq
        with vm.DeviceFormat.from_device_csr(d(rp), d(c), d(v), 3000, 2500, True, 32) as f:
            C = torch.zeros((3000, 48), device="cuda")
            f.spmm(dB, C)
            torch.cuda.synchronize()
        first = C if first is None else first
        assert torch.equal(C, first)
    del C, first
    torch.cuda.synchronize()
    torch.cuda.empty_cache()
    assert free0 - torch.cuda.mem_get_info()[0] <= (2 << 30) + (256 << 20)
