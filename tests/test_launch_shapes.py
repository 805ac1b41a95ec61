"""CPU checks of the launch shapes that a plan's host code works out: the
routes of its levels and the room for the block sums of their launches."""
import itertools
import os
import subprocess
import sys

import numpy as np
import pytest


def _shape(n, bc=(1, 1, 1, 1, 2, 2), level=0, **policy):
    import hundun_flow as H
    faces = [np.linspace(0.0, 1.0, v + 1) for v in n]
    pol = H.default_policy(anisotropy_threshold=1e9, **policy)
    return H.launch_shape(n, faces, bc, pol, level)


@pytest.mark.parametrize("n,policy,blocks", [
    # no leg: six colour passes and the defect before a restriction
    ((58, 9, 50), dict(pre_sweeps=3), 2 * 2 * 50),
    ((58, 17, 42), dict(pre_sweeps=3), 2 * 3 * 42),
    # an F-cycle whose second level takes more boxes than a leg may have
    ((64, 12, 52), dict(f_cycle=1), 2 * 2 * 52),
    ((64, 12, 64), dict(f_cycle=1), 2 * 2 * 64),
])
def test_slim_march_sums_fit(n, policy, blocks):
    """The march that ends a cycle of a closed domain sums a mean in each of
    its blocks: tiles of 56x8 columns (FP64), a plane each on a slim grid,
    are more than the 64x4 tiles of the plane kernels."""
    s = _shape(n, **policy)
    assert s["route"] == "march"
    assert s["sum_blocks"] == blocks
    assert s["sum_blocks"] <= s["sum_capacity"]


@pytest.mark.parametrize("env", [{}, {"HF_LEG_CELLS": "0"},
                                 {"HF_LEG_CELLS": "0", "HF_TAIL_CELLS": "0",
                                  "HF_SWEEP_MIN_CELLS": "0",
                                  "HF_SWEEP_ZC": "1"}])
@pytest.mark.parametrize("precision", ["fp64", "fp32", "bf16"])
def test_block_sums_fit_everywhere(monkeypatch, precision, env):
    """No launch on any level makes more block sums than the plan holds, over
    slim and odd grids, sweep counts and coarsest extents."""
    for k, v in env.items():
        monkeypatch.setenv(k, v)
    grids = list(itertools.product((32, 58, 64, 114), (8, 9, 12, 17),
                                   (8, 9, 50, 200)))
    grids += [(1, 40, 33), (3, 5, 700), (2, 2, 4000), (4096, 2, 2),
              (97, 13, 9), (130, 41, 21), (512, 8, 8), (32, 8, 2000)]
    policies = [dict(), dict(pre_sweeps=1, post_sweeps=1),
                dict(pre_sweeps=3), dict(pre_sweeps=4, post_sweeps=2),
                dict(f_cycle=1), dict(minimum_coarse_extent=8),
                dict(minimum_coarse_extent=16, f_cycle=1),
                dict(minimum_coarse_extent=2, pre_sweeps=3, post_sweeps=4),
                dict(point_smoother=1, f_cycle=1, pre_sweeps=1)]
    routes = set()
    for n, policy in itertools.product(grids, policies):
        level, levels = 0, 1
        while level < levels:
            try:
                s = _shape(n, level=level, precision=precision, **policy)
            except RuntimeError:  # refused: no coarse level, or too large one
                break
            assert s["sum_blocks"] <= s["sum_capacity"], (n, policy, level, s)
            routes.add(s["route"])
            levels = s["levels"]
            level += 1
    assert {"march", "tail"} <= routes


@pytest.mark.parametrize("n", [(1, 1, 9_000_000), (1, 2, 8_388_609),
                               (512, 512, 512)])
def test_folded_sums_fit(n):
    """The first fold's spans grow where spans of the usual length would be
    more than its buffer holds: a plane of few cells takes a block each."""
    s = _shape(n)
    assert 0 < s["fold_blocks"] <= s["fold_capacity"]


@pytest.mark.parametrize("n", [(0, 4, 4), (2147483647, 1, 1)])
def test_shape_of_a_refused_grid(n):
    """A grid that no plan takes has no shape either."""
    import hundun_flow as H
    faces = [np.linspace(0.0, 1.0, 5)] * 3
    with pytest.raises(H.HundunFlowError) as err:
        H.launch_shape(n, faces, (1,) * 6, H.default_policy())
    assert err.value.code == 2


_STARVED = """
import ctypes, resource, sys
import numpy as np
sys.path.insert(0, sys.argv[1])
import hundun_flow as H
lib = H.load_library()
n = (1, 1, 500_000_000)
faces = [np.linspace(0.0, 1.0, 2)] * 2 + [np.zeros(n[2] + 1)]
grid = H._grid_desc(n, faces, (1,) * 6)
policy = H.default_policy()
size = int(open("/proc/self/statm").read().split()[0]) * 4096
resource.setrlimit(resource.RLIMIT_AS, (size + (1 << 30),) * 2)
shape, plan = H.hf_launch_shape(), ctypes.c_void_p()
for st in (lib.hf_launch_shape_of(ctypes.byref(grid), ctypes.byref(policy), 0,
                                  ctypes.byref(shape)),
           lib.hf_plan_create(ctypes.byref(grid), ctypes.byref(policy), None,
                              ctypes.byref(plan))):
    assert (st.code, st.detail) == (3, 9102), (st.code, st.detail)
"""


def test_out_of_host_memory_is_a_status():
    """A grid whose face coordinates no longer fit into host memory is an
    allocation failure, not an exception through the C interface."""
    import hundun_flow as H
    run = subprocess.run([sys.executable, "-c", _STARVED,
                          os.path.dirname(H.__file__)], timeout=120,
                         capture_output=True, text=True)
    assert run.returncode == 0, run.stderr[-2000:]
