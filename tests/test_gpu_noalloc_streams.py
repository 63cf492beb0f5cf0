"""The allocation-free batched network solve on streams that have not run it:
it takes no device memory, nor does the runtime on its behalf (a kernel that
needs scratch memory has it allocated when a queue first runs one: 64 bytes per
lane are some 30 MB).  Systems of every row count per lane, FP64 and FP32; the
results are those of the allocating call, bit for bit."""
import ctypes as C

import numpy as np
import pytest

import cfdrs_amd as ca
from cfdrs_amd import _native as N
from cfdrs_amd import network as NW
from cfdrs_amd.sparse import bind_torch_stream

pytestmark = pytest.mark.gpu


def solve(fn, batch, cfg, x):
    reps = (N.Report * batch.n_sys)()
    x.zero_()
    bind_torch_stream()
    N.call(fn, batch.handle, C.byref(cfg), None, x.data_ptr(), reps)
    return [(r.iterations, r.final_residual_norm, r.termination) for r in reps]


def test_no_memory_is_taken_on_a_new_stream():
    import torch

    nets = NW.synth_networks(count=96, seed_base=4600, nmin=50, nmax=2000)
    batch = NW.channel_batch(nets)
    rows = np.diff(nets.node_offset)
    assert {-(-int(r) // 256) for r in rows} == set(range(1, 9))  # 1 to 8 rows per lane
    x = torch.zeros(batch.n_rows, dtype=torch.float64, device="cuda")
    cfgs = [ca.IterativeSolverConfig.new(1e-10).with_max_iterations(20000).with_precision(p).native(N.KIND_CG)
            for p in (ca.Precision.FP64, ca.Precision.FP32_REFINED)]
    want = []
    for cfg in cfgs:
        reps = solve("cfdla_batch_solve_device", batch, cfg, x)
        assert all(r[2] == N.TERM_CONVERGED for r in reps)
        want.append((reps, x.clone()))
    got = torch.empty_like(x)
    for _ in range(5):
        stream = torch.cuda.Stream()
        with torch.cuda.stream(stream):
            for _ in range(3):
                x.zero_()  # the stream's queue is there
            torch.cuda.synchronize()
            for cfg, (reps, y) in zip(cfgs, want):
                before = torch.cuda.mem_get_info()[0]
                assert solve("cfdla_batch_solve_device_noalloc", batch, cfg, x) == reps
                torch.cuda.synchronize()
                assert before - torch.cuda.mem_get_info()[0] < 1 << 20
                got.copy_(x)
                assert torch.equal(got, y)
    bind_torch_stream()
