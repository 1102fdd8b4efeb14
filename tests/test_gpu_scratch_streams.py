"""Calls that take scratch memory from the library's list, on several streams and threads
at once: forward projections through the padded copy, re-pitched 16-bit views and paired
RTK views.  The blocks pass from stream to stream; every result equals the same call made
alone."""
import threading

import numpy as np
import pytest

import fdk_amd as F
from test_gpu_fp_runs import takes_the_copy

pytestmark = pytest.mark.gpu


class Work:
    """One of the three kinds of calls, of a size that depends on `seed`."""

    def __init__(self, torch, kind, seed):
        g = torch.Generator(device="cuda")
        g.manual_seed(seed)
        n = 60 + 8 * seed
        self.kind, self.n = kind, n
        if kind == "fp":
            self.p = F.Parameter(nx=n, ny=n, nz=n, nu=n + 9, nv=n + 5, du=2.0, dv=2.0, nproj=24)
            assert takes_the_copy(self.p, 0, 24, 0.25)
            self.src = torch.rand((n, n, n), device="cuda", generator=g)
            self.shape = (24, n + 5, n + 9)
        elif kind == "rtk":
            n = self.n = n + 100
            self.p = F.Parameter(nx=n, ny=n, nz=n, nu=n, nv=n, du=1.6, dv=1.6, nproj=32)
            self.src = torch.rand((32, n, n), device="cuda", generator=g)
            self.vin = torch.rand((n, n, n), device="cuda", generator=g)
            self.shape = (n, n, n)
        else:
            self.p = F.Parameter(nx=n, ny=n, nz=n, nu=n + 4, nv=n + 3 - n % 2, du=2.0, dv=2.0, nproj=32)
            self.src = torch.rand((32, self.p.nu, self.p.nv), device="cuda", generator=g).half()
            self.shape = (n, n, n)
        self.m = self.p.proj_matrices().astype(np.float32)

    def run(self, torch, out):
        p, n = self.p, self.n
        if self.kind == "fp":
            F.forward_project(p, self.src, 0, 24, out, 0.25)
        elif self.kind == "rtk":
            F.reconstruct_conebeam((n, n, 32), (n, n, n), self.m, self.vin, out, self.src)
        else:
            h = F.BackProjectionFDK(p.nv, p.nu, 32, n, n, n, (0, 0, 0, n, n, n), (0, 0, 0, 0, 0, 0))
            h.set_stream(torch.cuda.current_stream().cuda_stream)
            for _ in range(3):
                h.bp_device(self.src, p.nv, p.nu, self.m, 32, dtype=F.FDK_F16,
                            scale_offset=np.tile(np.float32([1, 0]), (32, 1)))
            h.get_volume_device(out)
            h.close()


@pytest.mark.parametrize("threads", [False, True])
def test_results_are_those_of_calls_made_alone(torch_cuda, threads):
    torch = torch_cuda
    jobs = [Work(torch, kind, seed) for seed in range(4) for kind in ("fp", "pitched", "rtk")]
    ref = [torch.empty(j.shape, device="cuda") for j in jobs]
    for j, r in zip(jobs, ref):
        j.run(torch, r)
        torch.cuda.synchronize()
    lanes = 3
    streams = [torch.cuda.Stream() for _ in range(lanes)]
    out = [torch.full_like(r, 7.0) for r in ref for _ in range(2)]
    torch.cuda.synchronize()
    failed = []

    def lane(k, only=None):
        try:
            with torch.cuda.stream(streams[k]):
                for i in range(k, 2 * len(jobs), lanes) if only is None else [only]:
                    jobs[i // 2].run(torch, out[i])
        except Exception as e:  # the threads' errors fail the test
            failed.append(e)

    if threads:
        t = [threading.Thread(target=lane, args=(k,)) for k in range(lanes)]
        [q.start() for q in t]
        [q.join() for q in t]
    else:
        for i in range(2 * len(jobs)):
            lane(i % lanes, i)
    torch.cuda.synchronize()
    assert not failed, failed
    for i, o in enumerate(out):
        assert torch.equal(o, ref[i // 2]), jobs[i // 2].kind


def test_release_gives_the_memory_back(torch_cuda):
    """A projection's copy stays with the library until it is released."""
    torch = torch_cuda
    n = 200
    p = F.Parameter(nx=n, ny=n, nz=n, nu=n, nv=n, du=2.0, dv=2.0, nproj=24)
    assert takes_the_copy(p, 0, 24, 0.5)
    vol, out = torch.rand((n, n, n), device="cuda"), torch.empty((24, n, n), device="cuda")
    F.release_scratch()
    before = torch.cuda.mem_get_info()[0]
    F.forward_project(p, vol, 0, 24, out, 0.5)
    torch.cuda.synchronize()
    kept = before - torch.cuda.mem_get_info()[0]
    assert 8 * n ** 3 <= kept <= 1 << 29
    F.release_scratch()
    assert torch.cuda.mem_get_info()[0] >= before
    again = torch.empty_like(out)
    F.forward_project(p, vol, 0, 24, again, 0.5)
    torch.cuda.synchronize()
    assert torch.equal(out, again)
