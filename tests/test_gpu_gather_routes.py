"""The tile-owner gathers on calls that are small enough to run per pixel by themselves.

The calls of most GPU tests are small, so their forward projections and pose gradients take the
per-pixel kernels.  Here the same tests (their functions, cases, references and bars) run once more
with tp_set_gather_route(TP_ROUTE_TILES): pose classes, carried windows, complex-half volumes, sizes,
oversamplings, layouts, streams, host threads, captured graphs and the entry point without
allocations.  Cases without a choice of gathers (TP_F64, backprojections) are left out, and every test
checks that the last call of each of its threads did not run per pixel.
"""
import threading
import types

import pytest

from tests import (test_gpu_carried_windows, test_gpu_golden, test_gpu_graph, test_gpu_half_storage, test_gpu_layouts,
                   test_gpu_oversampling, test_gpu_parity, test_gpu_pose_classes, test_gpu_pose_ranges,
                   test_gpu_random, test_gpu_streams, test_gpu_tiled2d, test_zz_no_alloc)
from torch_projectors import capi

pytestmark = [pytest.mark.gpu, pytest.mark.filterwarnings("ignore:ComplexHalf support is experimental")]

MODULES = (test_gpu_carried_windows, test_gpu_golden, test_gpu_graph, test_gpu_half_storage, test_gpu_layouts,
           test_gpu_oversampling, test_gpu_parity, test_gpu_pose_classes, test_gpu_pose_ranges, test_gpu_random,
           test_gpu_streams, test_gpu_tiled2d, test_zz_no_alloc)
# no gathers, or no small calls
LEFT_OUT = ("test_pose_class_predicate_bounds", "test_fourier_transforms_replayed_after_plan_eviction",
            "test_2d_backprojection_replayed", "test_3d_scatters_replayed_without_a_workspace",
            "test_many_ranges_match_oracle", "test_precision_does_not_fall_with_the_pose_count",
            "test_strided_inputs_backprojection", "test_half_volume_through_autograd",
            "test_tiled_gathers_past_the_per_pixel_sizes", "test_small_calls_run_per_pixel")


def _has_gathers(param):
    case = test_gpu_golden.load_fixture(param)[0] if isinstance(param, str) else param
    return case["dtype"] == "f32" and case["op"] not in ("backproject_2d_forw", "backproject_2d_to_3d_forw")


def _filtered(fn):
    """A copy of a test function whose cases (or golden paths) are those with a choice of gathers."""
    out = types.FunctionType(fn.__code__, fn.__globals__, fn.__name__, fn.__defaults__, fn.__closure__)
    out.pytestmark = []
    for m in getattr(fn, "pytestmark", []):
        if m.name == "parametrize" and m.args[0] in ("case", "path"):
            keep = [i for i, p in enumerate(m.args[1]) if _has_gathers(p)]
            m = pytest.mark.parametrize(m.args[0], [m.args[1][i] for i in keep],
                                        ids=[m.kwargs["ids"][i] for i in keep]).mark
        out.pytestmark.append(m)
    return out


for _m in MODULES:
    for _name, _fn in list(vars(_m).items()):
        if _name.startswith("test_") and isinstance(_fn, types.FunctionType) and _name not in LEFT_OUT:
            globals()[f"test_tiles_{_m.__name__.split('test_')[-1]}_{_name[5:]}"] = _filtered(_fn)


@pytest.fixture(autouse=True)
def tiles(gpu, monkeypatch):
    lib, run, took = capi.lib(), threading.Thread.run, []

    def routed(self):  # (the setting is each thread's own)
        lib.tp_set_gather_route(capi.ROUTE_TILES)
        run(self)
        took.append(lib.tp_last_gather_route())

    monkeypatch.setattr(threading.Thread, "run", routed)
    was = lib.tp_set_gather_route(capi.ROUTE_TILES)
    yield
    lib.tp_set_gather_route(was)
    assert capi.ROUTE_PER_PIXEL not in took + [lib.tp_last_gather_route()]


@pytest.mark.parametrize("route", [capi.ROUTE_BY_SIZE, capi.ROUTE_TILES, capi.ROUTE_PER_PIXEL])
def test_setting_of_the_calling_thread(route):
    lib = capi.lib()
    assert lib.tp_set_gather_route(route) == capi.ROUTE_TILES
    assert lib.tp_set_gather_route(7) == route and lib.tp_set_gather_route(-1) == route  # unknown: unchanged
    seen = []
    t = threading.Thread(target=lambda: seen.append(lib.tp_set_gather_route(capi.ROUTE_PER_PIXEL)))
    t.start()
    t.join()
    assert seen == [capi.ROUTE_TILES]  # (as the fixture starts its threads, not as this one is set)
    assert lib.tp_set_gather_route(capi.ROUTE_TILES) == route
