"""Calls of one geometry with many different pose counts.

The tile kernels' work depends on the pose count, their lists must not: after a first pass over a few
counts, calls with other counts only enqueue.  A sleeping kernel is put on the stream first, and every
call must return while it still sleeps (making a list or growing the workspace waits for the stream).
The results are those of the same calls on another stream.
"""
import pytest
import torch

from torch_projectors import capi

pytestmark = pytest.mark.gpu

T = torch.ops.torch_projectors


def _rel(a, b):
    return ((a - b).norm() / b.norm()).item()


@pytest.fixture(scope="module")
def stream(gpu):
    return torch.cuda.Stream()


@pytest.mark.parametrize("interp,os_", [("linear", 2.0), ("cubic", 1.0)])
def test_other_pose_counts_only_enqueue(gpu, stream, interp, os_):
    n, B, most = 48, 2, 640
    N = capi.rec_boxsize(n, os_)
    g = torch.Generator().manual_seed(515)
    vol = torch.randn(B, N, N, N // 2 + 1, generator=g, dtype=torch.complex64).to(gpu)
    rot = torch.linalg.qr(torch.randn(1, most, 3, 3, generator=g, dtype=torch.float64))[0].float()
    rot[:, 3::7] *= 1.1
    rot = rot.to(gpu)
    sh = (torch.rand(1, most, 2, generator=g) * 4 - 2).to(gpu)
    w = torch.rand(B, most, n, n // 2 + 1, generator=g).to(gpu)

    def step(P):
        r, s = rot[:, :P].contiguous(), sh[:, :P].contiguous()
        proj = T.project_3d_to_2d_forw(vol, r, s, [n, n], interp, os_, None)
        data, wrec = T.backproject_2d_to_3d_forw(proj, w[:, :P].contiguous(), r, s, interp, os_, None)
        gradients = T.project_3d_to_2d_back(proj, vol, r.requires_grad_(True), s.requires_grad_(True), interp, os_, None)
        return proj, data, wrec, *gradients

    was = capi.lib().tp_set_gather_route(capi.ROUTE_TILES)
    try:
        stream.wait_stream(torch.cuda.current_stream())
        with torch.cuda.stream(stream):
            for P in (most, 320, 160, 80, 40, 20, 10):
                step(P)
        torch.cuda.synchronize()
        for P in (611, 570, 530, 487, 451, 402, 377, 341, 303, 266, 231, 199, 173, 151, 127, 103, 91, 77, 61, 47, 33, 21):
            print(f"[pose counts] {interp} P={P}", flush=True)
            expected = step(P)
            torch.cuda.synchronize()
            with torch.cuda.stream(stream):
                torch.cuda._sleep(100_000_000)  # tens of milliseconds
                slept = torch.cuda.Event()
                slept.record()
                got = step(P)
                waited = slept.query()
            torch.cuda.synchronize()
            assert not waited, f"P={P}: a call waited for the stream"
            assert torch.equal(got[0], expected[0])
            for a, b in zip(got[1:], expected[1:]):
                assert _rel(a, b) <= 1e-5
    finally:
        capi.lib().tp_set_gather_route(was)
