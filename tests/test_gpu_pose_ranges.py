"""The fp32 scatters and gathers at pose counts around the edges of their pose ranges.

Small calls split a tile's poses into short ranges to fill the GPU; these cases put the pose count
just below, at and above the lengths where the split changes (one range, a last range of one pose,
ranges of unequal length), with scaled poses among the rotations, against the oracle with the bars
of tests/parity.py.
"""
import pytest

from tests.golden.cases import _case, make_inputs
from tests.parity import check_outputs, scatter_cells

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


# Calls just past the size where the tile-owner gathers take over from the per-pixel ones: small boxes
# with many poses (the other tests' small calls run per pixel).
def _large_cases():
    out, seed = [], 772000
    for op, interp, n, os_, P, B, cut in (
            ("project_3d_to_2d_forw", "linear", 30, 2.0, 3001, 1, None), ("project_3d_to_2d_forw", "linear", 32, 3.0, 700, 2, 9.5),
            ("project_3d_to_2d_forw", "cubic", 24, 2.0, 1100, 1, None), ("project_3d_to_2d_forw", "cubic", 34, 1.3, 1500, 1, 15.0),
            ("project_3d_to_2d_back", "linear", 30, 2.0, 3300, 1, None), ("project_3d_to_2d_back", "cubic", 26, 1.5, 1200, 1, None),
            ("backproject_2d_to_3d_back", "linear", 30, 2.0, 3300, 1, None), ("backproject_2d_to_3d_back", "cubic", 28, 1.0, 500, 2, 12.0),
            ("project_2d_forw", "cubic", 48, 3.0, 4000, 1, None), ("project_2d_forw", "linear", 256, 1.0, 1900, 1, None),
            ("project_2d_back", "linear", 150, 1.5, 21, 2, None), ("project_2d_back", "cubic", 146, 2.0, 18, 1, 60.0),
            ("backproject_2d_back", "linear", 150, 0.75, 21, 2, 50.0), ("backproject_2d_back", "cubic", 146, 2.0, 18, 1, None)):
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
