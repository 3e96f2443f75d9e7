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


@pytest.mark.parametrize("case", CASES, ids=[c["name"] for c in CASES])
def test_pose_ranges_match_oracle(case, hip, oracle):
    args, tensors = make_inputs(case)
    rot = args[2].detach().clone()
    rot[:, 2::5] *= 1.1
    args[2] = rot.requires_grad_(args[2].requires_grad)
    print(f"[pose ranges] {case['name']}", flush=True)
    got = getattr(hip, case["op"])(*args)
    exp = getattr(oracle, case["op"])(*args)
    check_outputs(case["op"], got, exp, has_shifts=tensors.get("shifts") is not None, label=case["name"],
                  cells=scatter_cells(case["op"], args, oracle))
