"""GPU parity of the multigrid kernels route by route: every case asks the
library which kernels its levels take and holds the cycle to the CPU oracle or
to another route (bit for bit, or to 1e-12 where a mean is summed in another
order)."""
import sys

import numpy as np
import pytest

import hf_cases
import hf_oracle as O

pytestmark = pytest.mark.gpu


def _say(msg):
    print(msg, flush=True)
    sys.stdout.flush()


def _case(n, bc, seed, radius=0.2):
    """A sphere case on an n grid with six boundary kinds."""
    case = hf_cases.lognormal_sphere(n=n, seed=seed, radius=radius)
    act = case["cell_active"].reshape(n[2], n[1], n[0])
    fx, fy, fz = hf_cases.face_activity(act, bc)
    case.update(bc=list(bc), x_active=fx, y_active=fy, z_active=fz)
    return case


def _plan(case, **policy):
    import hundun_flow as H
    return H.plan_from_case(case, H.default_policy(**policy))


def _route(case, level=0, **policy):
    import hundun_flow as H
    return H.launch_shape(case["n"], case["faces"], case["bc"],
                          H.default_policy(**policy), level)["route"]


def _t(torch, a):
    return torch.from_numpy(np.ascontiguousarray(a)).cuda()


@pytest.mark.parametrize("n,policy", [
    ((58, 9, 50), dict(pre_sweeps=3)),
    ((58, 17, 42), dict(pre_sweeps=3)),
    ((64, 12, 52), dict(f_cycle=1)),
    ((64, 12, 64), dict(f_cycle=1)),
])
def test_slim_march_means(torch_cuda, n, policy):
    """Closed domains on slim grids, whose last march sums a mean in more
    blocks than the grid has plane tiles: the projected cycle equals the
    oracle's to rounding, and the solve on the static scratch, which packs
    the block sums, the plain one's bit for bit."""
    torch = torch_cuda
    _say(f"[slim march] n={n} policy={policy}")
    case = _case(n, (1, 1, 1, 1, 2, 2), seed=61)
    pol = dict(policy, anisotropy_threshold=1e9)
    assert _route(case, **pol) == "march"
    plan = _plan(case, **pol)
    _, mg = O.from_case(case, O.policy(**pol))
    b = _t(torch, case["rhs"])
    z, zo = plan.mg_apply(b).cpu().numpy(), mg.apply(case["rhs"])
    assert np.linalg.norm(z - zo) <= 1e-12 * np.linalg.norm(zo)
    x, res = plan.solve_pcg(b, rtol=1e-9)
    y, static = plan.solve_pcg(b, rtol=1e-9, static=True)
    assert res.final_true_residual <= 1e-9 * res.rhs_norm
    assert torch.equal(x, y)
    assert static.iterations == res.iterations
    plan.close()


def test_sums_of_single_cell_planes(torch_cuda):
    """A grid of nine million planes of one cell: the norms of the right-hand
    side and the residual, folded with the entry's mean (to 1e-12 of
    torch's)."""
    import hundun_flow as H
    torch = torch_cuda
    n = (1, 1, 9_000_000)
    _say(f"[single-cell planes] n={n}")
    faces = [np.linspace(0.0, 1.0, v + 1) for v in n[:2]]
    faces.append(np.linspace(0.0, float(n[2]), n[2] + 1))
    plan = H.Plan(n, faces, (1,) * 6, H.default_policy(
        anisotropy_threshold=1e9))
    plan.set_coefficients(*plan.assemble(
        torch.ones(n[2], dtype=torch.float64, device="cuda")))
    gen = torch.Generator(device="cuda").manual_seed(3)
    b = torch.randn(n[2], dtype=torch.float64, device="cuda", generator=gen)
    b -= b.mean()
    _, res = plan.solve_pcg(b, rtol=1e-10, maximum_iterations=1, check=False)
    norm = torch.linalg.vector_norm(b).item()
    assert abs(res.rhs_norm - norm) <= 1e-12 * norm
    assert abs(res.initial_true_residual - norm) <= 1e-12 * norm
    plan.close()


@pytest.mark.parametrize("n", [(3, 4, 600_001),   # two planes to a lane
                               (1, 7, 100_003),   # rows of one cell
                               (16, 15, 501),     # two planes to a block
                               (16, 17, 500)])    # one, half a block
def test_operator_on_planes_of_few_cells(torch_cuda, n):
    """A x where a block holds several planes: bit for bit the same sums of
    products by torch, whose elementwise operations round one by one."""
    import hundun_flow as H
    torch = torch_cuda
    _say(f"[planes of few cells] n={n}")
    nx, ny, nz = n
    faces = [np.linspace(0.0, v / 8.0, v + 1) for v in n]
    plan = H.Plan(n, faces, (1,) * 6, H.default_policy(
        anisotropy_threshold=1e9))
    gen = torch.Generator(device="cuda").manual_seed(7)

    def normal():
        return torch.randn(nx * ny * nz, dtype=torch.float64, device="cuda",
                           generator=gen)
    d, bx, by, bz = plan.assemble(normal().exp())
    plan.set_coefficients(d, bx, by, bz)
    x = normal()
    y = plan.operator_apply(x)
    v = x.view(nz, ny, nx)
    ref = d.view(nz, ny, nx) * v
    for dim, f in ((2, bx.view(nz, ny, nx + 1)), (1, by.view(nz, ny + 1, nx)),
                   (0, bz.view(nz + 1, ny, nx))):
        m = v.shape[dim]  # a wall's neighbour is the cell itself
        first, last = v.narrow(dim, 0, 1), v.narrow(dim, m - 1, 1)
        low = torch.cat([first, v.narrow(dim, 0, m - 1)], dim)
        high = torch.cat([v.narrow(dim, 1, m - 1), last], dim)
        ref = ref - f.narrow(dim, 0, m) * low
        ref = ref - f.narrow(dim, 1, m) * high
    assert torch.equal(y.view(nz, ny, nx), ref)
    b = x - x.mean()
    _, res = plan.solve_pcg(b, maximum_iterations=1, check=False)
    norm = torch.linalg.vector_norm(b).item()
    assert abs(res.initial_true_residual - norm) <= 1e-12 * norm
    plan.close()


def test_operator_on_unaligned_arrays(torch_cuda):
    """A x of the smallest grid whose operator runs over aligned pairs in
    tiles, on arrays that begin in the middle of a pair: bit for bit that of
    aligned ones."""
    import hundun_flow as H
    torch = torch_cuda
    n = (256, 256, 192)
    _say(f"[unaligned operator] n={n}")
    cells = n[0] * n[1] * n[2]
    faces = [np.linspace(0.0, 1.0, v + 1) for v in n]
    plan = H.Plan(n, faces, (1, 1, 0, 1, 2, 2))
    gen = torch.Generator(device="cuda").manual_seed(5)

    def normal(count):
        return torch.randn(count, dtype=torch.float64, device="cuda",
                           generator=gen)
    plan.set_coefficients(*plan.assemble(normal(cells).exp()))
    x = normal(cells + 1)[1:]
    y = torch.empty(cells + 1, dtype=torch.float64, device="cuda")[1:]
    assert x.data_ptr() % 16 == 8 and y.data_ptr() % 16 == 8
    aligned = plan.operator_apply(x.clone())
    plan.operator_apply(x, out=y)
    assert torch.equal(y, aligned)
    assert torch.equal(plan.operator_apply(x), aligned)
    plan.close()


_GRID_LEVELS = {"HF_TAIL_CELLS": "0", "HF_LEG_CELLS": "0",
                "HF_SWEEP_MIN_CELLS": "0"}
# smoothing of the finest level by two sweeps, by one and by one colour a
# launch
_RED_BLACK = {"march": {},
              "sweep": {"HF_SWEEP_MARCH": "0"},
              "colours": {"HF_SWEEP_MARCH": "0", "HF_FUSED_SWEEP": "0"}}


def _cycle_on(torch, monkeypatch, env, case, r, **policy):
    """The cycle of a plan made under `env`, and the finest level's route."""
    with monkeypatch.context() as m:
        for k, v in {**_GRID_LEVELS, **env}.items():
            m.setenv(k, v)
        route = _route(case, **policy)
        plan = _plan(case, **policy)
        z = plan.mg_apply(_t(torch, r)).cpu().numpy()
        plan.close()
    return z, route


MARCH_GRIDS = [
    ((32, 8, 8), (0, 0, 1, 1, 2, 2)),      # the smallest grid it takes
    ((56, 24, 9), (1, 1, 0, 1, 1, 0)),     # one FP32 tile, three FP64 ones
    ((58, 25, 10), (2, 2, 1, 0, 2, 2)),    # a partial tile of two columns
    ((114, 18, 12), (0, 1, 2, 2, 1, 1)),   # wrapped rows, walls in z
    ((64, 40, 36), (1, 1, 1, 1, 1, 1)),    # a coarse level that marches too
]


@pytest.mark.parametrize("zc", ["", "1", "5"])
@pytest.mark.parametrize("n,bc", MARCH_GRIDS)
def test_red_black_routes(torch_cuda, monkeypatch, n, bc, zc):
    """V(2,2) cycles by marches, sweeps and colours, with the tail and the
    legs out of the way, on tile and chunk edges and every boundary kind: one
    result in every storage type, in FP64 the oracle's."""
    torch = torch_cuda
    _say(f"[red-black] n={n} bc={bc} zc={zc or 'planned'}")
    case = _case(n, bc, seed=23)
    pol = dict(null_space_constant=0, anisotropy_threshold=64.0)
    _, mg = O.from_case(case, O.policy(**pol))
    r = np.random.default_rng(17).standard_normal(n[0] * n[1] * n[2])
    zo = mg.apply(r)
    for precision in ("fp64", "fp32", "bf16"):
        first = None
        for name, env in _RED_BLACK.items():
            z, route = _cycle_on(torch, monkeypatch, {
                **env, **({"HF_SWEEP_ZC": zc} if zc else {})}, case, r,
                precision=precision, **pol)
            assert route == name
            first = z if first is None else first
            assert np.array_equal(z, first), (precision, name)
        if precision == "fp64":
            assert np.array_equal(first, zo)


@pytest.mark.parametrize("unit_linear", [1, 0])
@pytest.mark.parametrize("f_cycle", [0, 1])
@pytest.mark.parametrize("n,bc", MARCH_GRIDS)
def test_red_black_routes_projected(torch_cuda, monkeypatch, n, bc, f_cycle,
                                    unit_linear):
    """The same cycles with the constant null space, whose means the marches
    and sweeps take from and leave to other launches: 1e-12 of the oracle."""
    torch = torch_cuda
    _say(f"[red-black means] n={n} bc={bc} f={f_cycle} unit={unit_linear}")
    case = _case(n, bc, seed=23)
    pol = dict(anisotropy_threshold=64.0, f_cycle=f_cycle,
               unit_linear=unit_linear)
    _, mg = O.from_case(case, O.policy(**pol))
    zo = mg.apply(case["rhs"])
    for name, env in _RED_BLACK.items():
        z, route = _cycle_on(torch, monkeypatch, env, case, case["rhs"], **pol)
        assert route == name
        assert np.linalg.norm(z - zo) <= 1e-12 * np.linalg.norm(zo), name


@pytest.mark.parametrize("sweeps", [(1, 1), (1, 2), (2, 1), (3, 2), (2, 3),
                                    (4, 4)])
@pytest.mark.parametrize("n,route", [((66, 20, 10), "march"),
                                     ((66, 20, 6), "sweep")])
def test_sweep_counts(torch_cuda, monkeypatch, n, route, sweeps):
    """Smoothings that march and smoothings that cannot (other counts than
    two, too few planes) in one cycle: bit for bit the colour passes and, in
    FP64, the oracle; projected to 1e-12 of it."""
    torch = torch_cuda
    _say(f"[sweep counts] n={n} sweeps={sweeps}")
    case = _case(n, (1, 1, 1, 1, 2, 2), seed=29)
    pol = dict(null_space_constant=0, anisotropy_threshold=64.0,
               pre_sweeps=sweeps[0], post_sweeps=sweeps[1])
    _, mg = O.from_case(case, O.policy(**pol))
    r = np.random.default_rng(31).standard_normal(n[0] * n[1] * n[2])
    zo = mg.apply(r)
    for precision in ("fp64", "fp32", "bf16"):
        z, got = _cycle_on(torch, monkeypatch, {}, case, r,
                           precision=precision, **pol)
        assert got == route
        c, got = _cycle_on(torch, monkeypatch, _RED_BLACK["colours"], case, r,
                           precision=precision, **pol)
        assert got == "colours"
        assert np.array_equal(z, c), precision
        if precision == "fp64":
            assert np.array_equal(z, zo)
    pol["null_space_constant"] = 1
    _, mg = O.from_case(case, O.policy(**pol))
    zo = mg.apply(case["rhs"])
    z, _ = _cycle_on(torch, monkeypatch, {}, case, case["rhs"], **pol)
    assert np.linalg.norm(z - zo) <= 1e-12 * np.linalg.norm(zo)


@pytest.mark.parametrize("precision", ["fp64", "fp32", "bf16"])
@pytest.mark.parametrize("smoother", ["red_black", "chebyshev"])
@pytest.mark.parametrize("n,bc", [
    ((32, 32, 32), (1, 1, 1, 1, 2, 2)),
    ((128, 16, 8), (1, 1, 0, 1, 2, 2)),
    ((34, 10, 14), (2, 2, 2, 2, 0, 1)),    # a wavefront's rows partly full
])
def test_defect_restriction_routes(torch_cuda, monkeypatch, n, bc, smoother,
                                   precision):
    """The retained defect and its restriction in one launch and in two, on
    levels that neither the tail nor a leg takes: one result, and the single
    launch seen to be taken."""
    torch = torch_cuda
    _say(f"[defect, restriction] n={n} {smoother} {precision}")
    case = _case(n, bc, seed=37)
    pol = dict(null_space_constant=0, anisotropy_threshold=64.0,
               precision=precision)
    if smoother == "chebyshev":
        pol.update(point_smoother=1, f_cycle=1, pre_sweeps=1, post_sweeps=2)
    z, launches = {}, {}
    for fused in ("1", "0"):
        with monkeypatch.context() as m:
            for k, v in {**_GRID_LEVELS, "HF_DEFECT_RESTRICT": fused}.items():
                m.setenv(k, v)
            plan = _plan(case, **pol)
        r = _t(torch, case["rhs"])
        z[fused] = plan.mg_apply(r).cpu().numpy()
        plan.set_profiling(True)
        plan.solve_pcg(r, maximum_iterations=1, check=False)
        launches[fused] = plan.profile()["restrict"][1]
        plan.close()
    assert launches["1"] < launches["0"]
    assert np.array_equal(z["1"], z["0"])
