"""The fp32 scatters and gathers at pose counts around the edges of their pose ranges.

Small calls split a tile's poses into short ranges to fill the GPU; these cases put the pose count
just below, at and above the lengths where the split changes (one range, a last range of one pose,
ranges of unequal length), with scaled poses among the rotations, against the oracle with the bars
of tests/parity.py.
"""
import pytest

from tests.golden.cases import _case, make_inputs
from tests.parity import check_outputs, scatter_cells
from torch_projectors import capi

pytestmark = pytest.mark.gpu


def _cases():
    out, seed = [], 771000
    # 3D: tiles in one, two and three levels of pieces (few and many poses for the box), one-pose pieces
    for op in ("project_3d_to_2d_forw", "project_3d_to_2d_back", "backproject_2d_to_3d_forw",
               "backproject_2d_to_3d_back"):
        for interp, os_ in (("linear", 2.0), ("cubic", 1.0), ("linear", 1.5)):
            for n, P in ((16, 47), (16, 49), (32, 130), (48, 260)):
                seed += 1
                out.append(_case(f"{op}_{interp}_n{n}_os{os_:g}_P{P}", op, interp=interp, os=os_,
                                 cutoff=11.0 if n == 32 else None, B=2, P=P, n=n, B_rot=2, seed=seed,
                                 weights=(seed % 2 == 0)))
    for op in ("backproject_2d_forw", "project_2d_back"):
        for interp, os_ in (("linear", 1.0), ("cubic", 1.0), ("cubic", 2.0)):
            for n, P in ((32, 1), (32, 15), (30, 31), (48, 33), (40, 65)):
                seed += 1
                out.append(_case(f"{op}_{interp}_n{n}_os{os_:g}_P{P}", op, interp=interp, os=os_, cutoff=None, B=2, P=P,
                                 n=n, B_rot=2, seed=seed, weights=(seed % 2 == 0)))
    # 3D batches whose work balances without levels: one level of two pieces, and the levels just below
    for op, interp, B in (("project_3d_to_2d_forw", "cubic", 80), ("project_3d_to_2d_back", "cubic", 120),
                          ("project_3d_to_2d_back", "cubic", 40), ("backproject_2d_to_3d_forw", "linear", 90),
                          ("backproject_2d_to_3d_forw", "linear", 60), ("backproject_2d_to_3d_back", "cubic", 80)):
        seed += 1
        out.append(_case(f"{op}_{interp}_n16_B{B}_P520", op, interp=interp, os=2.0, cutoff=None, B=B, P=520, n=16, B_rot=B,
                         seed=seed, weights=True))
    return out


CASES = _cases()


def _rotations_at(args):
    return next(i for i, a in enumerate(args) if hasattr(a, "shape") and a.dim() == 4 and a.shape[-2:] in ((2, 2), (3, 3)))


@pytest.mark.parametrize("case", CASES, ids=[c["name"] for c in CASES])
def test_pose_ranges_match_oracle(case, hip, oracle):
    args, tensors = make_inputs(case)
    at = _rotations_at(args)
    rot = args[at].detach().clone()
    rot[:, 2::5] *= 1.1
    args[at] = rot.requires_grad_(args[at].requires_grad)
    print(f"[pose ranges] {case['name']}", flush=True)
    got = getattr(hip, case["op"])(*args)
    exp = getattr(oracle, case["op"])(*args)
    check_outputs(case["op"], got, exp, has_shifts=tensors.get("shifts") is not None, label=case["name"],
                  cells=scatter_cells(case["op"], args, oracle))


@pytest.mark.parametrize("op,n,os_,P,cut", [
    ("project_3d_to_2d_forw", 64, 2.0, 40, None), ("project_2d_forw", 1024, 2.0, 2, None),
    ("project_3d_to_2d_back", 48, 1.0, 60, None), ("backproject_2d_to_3d_back", 48, 2.0, 60, 9.0),
    ("project_2d_back", 64, 0.5, 40, None), ("backproject_2d_back", 100, 3.0, 40, 30.0)])
def test_small_calls_run_per_pixel(op, n, os_, P, cut, hip, oracle):
    case = _case("small", op, interp="linear", os=os_, cutoff=cut, B=1, P=P, n=n, seed=775000 + n)
    args, tensors = make_inputs(case)
    got = getattr(hip, op)(*args)
    assert capi.lib().tp_last_gather_route() == capi.ROUTE_PER_PIXEL
    exp = getattr(oracle, op)(*args)
    check_outputs(op, got, exp, has_shifts=tensors.get("shifts") is not None, label=op,
                  cells=scatter_cells(op, args, oracle))


# Calls just past the size where the tile-owner gathers take over from the per-pixel ones (the other tests'
# small calls run per pixel): volumes small and large for the caches, every oversampling range, cutoffs,
# 2D images beyond an XCD's L2 and poses of many blocks.
def _large_cases():
    out, seed = [], 772000
    for op, interp, n, os_, P, B, cut in (
            ("project_3d_to_2d_forw", "linear", 66, 2.0, 1400, 1, None), ("project_3d_to_2d_forw", "linear", 63, 3.0, 1000, 1, None),
            ("project_3d_to_2d_forw", "linear", 128, 1.3, 500, 1, 60.0),
            ("project_3d_to_2d_forw", "cubic", 50, 2.0, 400, 1, None), ("project_3d_to_2d_forw", "cubic", 62, 1.3, 600, 2, 25.0),
            ("project_3d_to_2d_back", "linear", 70, 2.0, 2100, 1, None), ("project_3d_to_2d_back", "cubic", 80, 1.5, 400, 1, None),
            ("backproject_2d_to_3d_back", "linear", 70, 2.0, 2100, 1, None), ("backproject_2d_to_3d_back", "cubic", 90, 1.0, 500, 2, 40.0),
            ("project_2d_forw", "cubic", 48, 3.0, 6000, 1, None), ("project_2d_forw", "linear", 513, 2.0, 65, 1, None),
            ("project_2d_forw", "cubic", 514, 2.0, 10, 2, None),
            ("project_2d_back", "linear", 150, 1.5, 21, 2, None), ("project_2d_back", "cubic", 200, 2.0, 18, 1, 90.0),
            ("backproject_2d_back", "linear", 150, 0.75, 500, 2, 50.0), ("backproject_2d_back", "cubic", 146, 2.0, 18, 1, None)):
        seed += 1
        out.append(_case(f"large_{op}_{interp}_n{n}_os{os_:g}_P{P}", op, interp=interp, os=os_, cutoff=cut, B=B, P=P, n=n,
                         B_rot=B, seed=seed, weights=(seed % 2 == 0)))
    return out


LARGE = _large_cases()


@pytest.mark.parametrize("case", LARGE, ids=[c["name"] for c in LARGE])
def test_tiled_gathers_past_the_per_pixel_sizes(case, hip, oracle):
    args, tensors = make_inputs(case)
    at = _rotations_at(args)
    rot = args[at].detach().clone()
    rot[:, 1::3] *= 1.1
    rot[:, 2::7] *= 2.5  # beyond the tiled range
    args[at] = rot.requires_grad_(args[at].requires_grad)
    print(f"[large] {case['name']}", flush=True)
    got = getattr(hip, case["op"])(*args)
    assert capi.lib().tp_last_gather_route() == capi.ROUTE_TILES
    exp = getattr(oracle, case["op"])(*args)
    check_outputs(case["op"], got, exp, has_shifts=tensors.get("shifts") is not None, label=case["name"],
                  cells=scatter_cells(case["op"], args, oracle))


# 2D scatters of many short pose ranges on small images: rotations alone, with scaled poses among them
# (their kernel adds onto the rotations' tiles), and scaled poses alone; tiles beyond the cutoff's reach.
MANY = [(op, interp, n, os_, P, B, cut, scale)
        for op in ("backproject_2d_forw", "project_2d_back")
        for interp, n, os_, P, B, cut, scale in (
            ("linear", 32, 1.0, 4099, 1, None, None), ("linear", 40, 1.0, 517, 3, 9.0, "some"),
            ("cubic", 24, 1.0, 1031, 2, None, "all"), ("cubic", 36, 2.0, 700, 1, 7.5, "some"),
            ("linear", 48, 1.75, 333, 2, None, "some"), ("linear", 33, 2.0, 97, 1, None, "all"))]


@pytest.mark.parametrize("op,interp,n,os_,P,B,cut,scale", MANY)
def test_many_ranges_match_oracle(op, interp, n, os_, P, B, cut, scale, hip, oracle):
    case = _case("many", op, interp=interp, os=os_, cutoff=cut, B=B, P=P, n=n, B_rot=B, seed=773000 + P + n,
                 weights=True)
    args, tensors = make_inputs(case)
    at = _rotations_at(args)
    rot = args[at].detach().clone()
    if scale:
        rot[:, ::(3 if scale == "some" else 1)] *= 1.3
    args[at] = rot.requires_grad_(args[at].requires_grad)
    print(f"[many ranges] {op} {interp} n={n} os={os_} P={P} {scale}", flush=True)
    got = getattr(hip, op)(*args)
    exp = getattr(oracle, op)(*args)
    check_outputs(op, got, exp, has_shifts=tensors.get("shifts") is not None, label=f"{op} {P}",
                  cells=scatter_cells(op, args, oracle))


@pytest.mark.parametrize("scale", [1.0, 1.1])
def test_precision_does_not_fall_with_the_pose_count(gpu, scale):
    """The weight image of 4096 poses of a small image, against the complex128 path: a range's sum rounds
    to fp32 once and the ranges' sum once (2^-24 each, relative), the taps' weight products round
    independently over the poses: together below 2^-23.  (256 ranges added in fp32 gave 2.1e-7.)"""
    import torch
    n, P = 64, 4096
    g = torch.Generator(device="cuda").manual_seed(774000)
    pr = torch.randn(1, P, n, n // 2 + 1, generator=g, device="cuda", dtype=torch.complex64)
    w = torch.rand(1, P, n, n // 2 + 1, generator=g, device="cuda")
    a = torch.rand(P, generator=g, device="cuda", dtype=torch.float64) * 6.283
    rot = (scale * torch.stack([a.cos(), -a.sin(), a.sin(), a.cos()], 1)).reshape(1, P, 2, 2).float()
    f = torch.ops.torch_projectors.backproject_2d_forw
    data, wrec = f(pr, w, rot, None, "linear", 1.0, None)
    data64, wrec64 = f(pr.to(torch.complex128), w.double(), rot.double(), None, "linear", 1.0, None)
    print(f"[precision] scale {scale}", flush=True)
    assert ((wrec.double() - wrec64).norm() / wrec64.norm()).item() < 2.0 ** -23
    assert ((data.to(torch.complex128) - data64).norm() / data64.norm()).item() < 2e-6
