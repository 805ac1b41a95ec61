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
    """A grid of nine million planes of one cell: the residual's norm and the
    entry's mean, two accumulators of a block sum per plane, are folded apart
    (the norm to 1e-12 of torch's)."""
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
