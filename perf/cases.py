"""The pressure-solve work that a low-Mach step gives this library.

Every case goes through the Python binding (`hundun_flow.Plan`), on inputs
made on the GPU from a seed: a flame-sheet density with log-normal noise on a
Cartesian grid, an immersed solid, Neumann walls with a periodic span (or a
closed box, or an outlet), and cubic cells whose y spacing may be stretched.

kind      one pass
operator  y = A x, the level-0 operator a Krylov method of the user's own calls
cycle     z = M r, one V(2,2) multigrid cycle as such a method's preconditioner
solve     PCG from zero to a relative residual of 1e-10, then the gauge (zero
          fluid mean): the projection step of an incompressible flow
step      a compressible time step's pressure work: face coefficients, the
          pressure-correction system, the refresh of the hierarchy and FGMRES
          with the Chebyshev F-cycle
adjoint   the gradients with respect to the right-hand side and log(rho)

exact() is the same mathematics in plain float64 torch: the linear systems by
Jacobi-preconditioned CG run to rounding, the cycle level by level.
"""
import math
import os
import sys

import numpy as np
import torch

sys.path.insert(0, os.path.join(os.path.dirname(os.path.dirname(
    os.path.abspath(__file__))), "hundun-flow_amd"))
import hundun_flow as H  # noqa: E402

DIRICHLET, NEUMANN, PERIODIC = 0, 1, 2
BOUNDARIES = {
    "span": (NEUMANN,) * 4 + (PERIODIC,) * 2,    # walls, periodic in z
    "box": (NEUMANN,) * 6,                       # closed box
    "outlet": (NEUMANN, DIRICHLET, NEUMANN, NEUMANN, PERIODIC, PERIODIC),
}
DENSITY_RATIO = 7.0
GAMMA = 1.4
ACOUSTIC_CFL = 4.0
RTOL = 1e-10
OMEGA = 0.72  # the smoother's relaxation factor


def _case(name, kind, nx, ny, nz, precision="fp64", solid="sphere",
          bc="span", stretch=1.0):
    return {"name": name, "kind": kind, "nx": nx, "ny": ny, "nz": nz,
            "precision": precision, "solid": solid, "bc": bc,
            "stretch": stretch}


def listed():
    return [
        # a user's own Krylov loop on a grid cut to its geometry
        _case("operator_ragged", "operator", 201, 149, 97, bc="box"),
        # the preconditioner alone, for the same loop
        _case("cycle_fp64_256", "cycle", 256, 256, 128, solid="cylinder"),
        # the smallest solve: every launch and every wait counts
        _case("solve_fp64_32", "solve", 32, 32, 32),
        # the log-normal sphere in a unit cube
        _case("solve_fp64_64", "solve", 64, 64, 64),
        # odd extents in every direction, an outlet, a stretched y
        _case("solve_fp32_odd", "solve", 143, 101, 75, "fp32", "cylinder",
              "outlet", 2.5),
        # even extents that no tile divides
        _case("solve_fp32_ragged", "solve", 300, 180, 140, "fp32", "sphere",
              "box"),
        # BF16 storage of the cycle
        _case("solve_bf16_192", "solve", 192, 192, 128, "bf16", "cylinder"),
        # the flame sheet with a cylinder, all in FP64
        _case("solve_fp64_256", "solve", 256, 256, 256, solid="cylinder"),
        # the flame sheet behind a step: the benchmark's grid
        _case("solve_fp32_512", "solve", 512, 256, 256, "fp32", "step"),
        # a compressible time step, small in FP64 and production-sized in FP32
        _case("step_fp64_64", "step", 64, 64, 64, solid="cylinder"),
        _case("step_fp32_256", "step", 256, 256, 256, "fp32", "cylinder"),
        # the backward pass of a loss on the pressure
        _case("adjoint_fp64_128", "adjoint", 128, 128, 128, solid="cylinder"),
    ]


def draw(rng):
    kind = rng.choice(["operator", "cycle", "solve", "solve", "solve",
                       "step", "step", "adjoint"])
    cells = 2.0 ** rng.uniform(13.0, 23.5)
    # aspect ratios up to about four between the axes
    ax, ay, az = (2.0 ** rng.uniform(-1.0, 1.0) for _ in range(3))
    unit = (cells / (ax * ay * az)) ** (1.0 / 3.0)
    n = [max(12, int(round(unit * a))) for a in (ax, ay, az)]
    layout = rng.choice(["any", "even", "sixteen"])
    if layout == "even":
        n = [v + (v & 1) for v in n]
    elif layout == "sixteen":
        n = [max(16, 16 * int(round(v / 16.0))) for v in n]
    precision = "fp64"
    if kind in ("solve", "step"):
        precision = rng.choice(["fp64", "fp32", "fp32", "bf16"]
                               if kind == "solve" else ["fp64", "fp32"])
    case = _case("", kind, n[0], n[1], n[2], precision,
                 rng.choice(["sphere", "cylinder", "step", "none"]),
                 # (the adjoint projects dL/dp: for closed domains only)
                 rng.choice(["span", "span", "box", "box" if kind == "adjoint"
                             else "outlet"]),
                 rng.choice([1.0, 1.0, 2.5]))
    del case["name"]
    return case


def work(case):
    """Every input read once and every output written once."""
    nx, ny, nz = case["nx"], case["ny"], case["nz"]
    cells = nx * ny * nz
    faces = (nx + 1) * ny * nz + nx * (ny + 1) * nz + nx * ny * (nz + 1)
    stencil = 8 * (cells + faces)  # D and the face coefficients
    if case["kind"] == "step":
        # mobility, three face fluxes, rho three times, drho/dp and a source
        # in; D, b and the pressure out
        return {"bytes": 8 * (6 * cells + faces + 3 * cells),
                "flops": 60 * cells}
    if case["kind"] == "adjoint":
        # mobility, pressure and dL/dp in, two gradients out
        return {"bytes": stencil + 5 * 8 * cells, "flops": 60 * cells}
    # one vector in, one out
    return {"bytes": stencil + 2 * 8 * cells, "flops": 13 * cells}


# -- inputs -----------------------------------------------------------------
def _grid(case):
    """Face coordinates per axis (x, y, z) and the boundary kinds."""
    n = (case["nx"], case["ny"], case["nz"])
    h = 1.0 / case["ny"]
    faces = [np.arange(v + 1, dtype=np.float64) * h for v in n]
    if case["stretch"] > 1.0:
        s = math.acosh(math.sqrt(case["stretch"]))
        eta = np.arange(n[1] + 1, dtype=np.float64) / n[1]
        faces[1] = 0.5 + 0.5 * np.tanh(s * (2.0 * eta - 1.0)) / math.tanh(s)
        faces[1][0], faces[1][-1] = 0.0, 1.0
    return n, faces, BOUNDARIES[case["bc"]]


def _along(values, axis, device):
    """A 1-D array as a (z, y, x) tensor along `axis` (0: x)."""
    shape = [1, 1, 1]
    shape[2 - axis] = -1
    return torch.as_tensor(values, dtype=torch.float64,
                           device=device).reshape(shape)


def _face_mask(fluid, axis, bc):
    """Faces between two fluid cells; a physical boundary face follows its
    inside cell, a periodic one its two wrapped cells."""
    dim = 2 - axis
    n = fluid.shape[dim]
    first, last = fluid.narrow(dim, 0, 1), fluid.narrow(dim, n - 1, 1)
    periodic = bc[2 * axis] == PERIODIC
    low = torch.cat([last if periodic else first, fluid], dim)
    high = torch.cat([fluid, first if periodic else last], dim)
    return low & high


def _inputs(case, seed):
    """Density, activity masks, and what the case's kind takes beside them."""
    dev = torch.device("cuda")
    gen = torch.Generator(device=dev).manual_seed(seed)
    n, faces, bc = _grid(case)
    shape = (n[2], n[1], n[0])

    def normal(shape=shape):
        return torch.randn(shape, dtype=torch.float64, device=dev,
                           generator=gen)

    width = [np.diff(f) for f in faces]
    x, y, z = (_along(f[:-1] + 0.5 * w, a, dev)
               for a, (f, w) in enumerate(zip(faces, width)))
    rho = 1.0 + (DENSITY_RATIO - 1.0) * 0.5 * (1.0 + torch.tanh(
        (y - 0.5) / 0.02))
    rho = rho * torch.exp(0.05 * normal())
    # the solid sits where the seed puts it, away from the walls
    place = torch.rand(4, dtype=torch.float64, generator=torch.Generator(
        ).manual_seed(seed)).tolist()
    mx, mz = 0.5 * faces[0][-1], 0.5 * faces[2][-1]
    size = min(1.0, faces[0][-1], faces[2][-1])
    cx, cy = mx + 0.1 * size * (place[0] - 0.5), 0.45 + 0.1 * place[1]
    radius = (0.12 + 0.08 * place[2]) * size
    solid = torch.zeros(shape, dtype=torch.bool, device=dev)
    if case["solid"] == "sphere":
        solid |= (x - cx) ** 2 + (y - cy) ** 2 + (z - mz) ** 2 < radius ** 2
    elif case["solid"] == "cylinder":
        solid |= (x - cx) ** 2 + (y - cy) ** 2 < radius ** 2
    elif case["solid"] == "step":
        solid |= (x < 0.125 * faces[0][-1]) & (y < 0.2 + 0.1 * place[3])
    fluid = ~solid
    inputs = {"n": n, "faces": faces, "bc": bc, "fluid": fluid, "rho": rho,
              "face_fluid": [_face_mask(fluid, a, bc) for a in range(3)]}
    singular = case["bc"] != "outlet"

    def right_hand_side():
        b = torch.where(fluid, normal(), 0.0)
        return torch.where(fluid, b - b.sum() / fluid.sum(), 0.0) \
            if singular else b

    if case["kind"] == "step":
        widths = [_along(w, a, dev) for a, w in enumerate(width)]
        spacing = min(float(w.min()) for w in width)
        dt = ACOUSTIC_CFL * spacing * math.sqrt(float(rho.min()) / GAMMA)
        inputs["dt"] = dt
        inputs["bdf"] = (1.5 / dt, -2.0 / dt, 0.5 / dt)
        inputs["rho_n"] = rho * (1.0 + 0.01 * normal())
        inputs["rho_nm1"] = rho * (1.0 + 0.01 * normal())
        inputs["drho_dp"] = rho / GAMMA
        inputs["source"] = 0.01 * normal()
        inputs["phi"] = []
        for a in range(3):
            extent = list(shape)
            extent[2 - a] += 1
            u = normal(extent)
            if bc[2 * a] == PERIODIC:
                u.narrow(2 - a, n[a], 1).copy_(u.narrow(2 - a, 0, 1))
            else:
                u.narrow(2 - a, 0, 1).zero_()
                u.narrow(2 - a, n[a], 1).zero_()
            area = widths[(a + 1) % 3] * widths[(a + 2) % 3]
            inputs["phi"].append(u * area)
    elif case["kind"] == "adjoint":
        wave = torch.cos(math.pi * x / faces[0][-1]) * torch.cos(math.pi * y)
        inputs["pressure"] = torch.where(
            fluid, wave + torch.sin(2.0 * math.pi * z / faces[2][-1]), 0.0)
        # dL/dp of L = the sum of p over a box of the domain
        probe = ((x - 1.5 * mx).abs() < 0.25 * mx) & ((y - 0.5).abs() < 0.125)
        inputs["grad_p"] = (probe & fluid).to(torch.float64) * (1.0 + 0.1 *
                                                                normal())
    elif case["kind"] == "operator":
        inputs["x"] = normal()
    else:
        inputs["rhs"] = right_hand_side()
    return inputs


def _policy(case):
    if case["kind"] == "step":
        return H.default_policy(
            pre_sweeps=1, post_sweeps=2, point_smoother=1, f_cycle=1,
            chebyshev_lower_fraction=0.3, diagonal_shortcut_ratio=0.1,
            null_space_constant=0, precision=case["precision"])
    return H.default_policy(precision=case["precision"],
                            coarse_face_scaling=1,
                            null_space_constant=int(case["bc"] != "outlet"))


def prepare(case, seed):
    inputs = _inputs(case, seed)
    flat = {k: v.reshape(-1) for k, v in inputs.items()
            if isinstance(v, torch.Tensor) and k not in ("fluid", "rho")}
    scale = inputs["dt"] if case["kind"] == "step" else 1.0
    state = {"case": case, **flat, "rho": inputs["rho"].reshape(-1),
             "mobility": (scale / inputs["rho"]).reshape(-1),
             "masks": [m.to(torch.uint8).reshape(-1) for m in
                       [inputs["fluid"]] + inputs["face_fluid"]]}
    state["plan"] = H.Plan(inputs["n"], inputs["faces"], inputs["bc"],
                           _policy(case))
    if case["kind"] == "step":
        state["phi"] = [p.reshape(-1) for p in inputs["phi"]]
        state["bdf"] = inputs["bdf"]
        state["fluid"] = state["masks"][0].to(torch.float64)
    else:
        # the coefficients that stand while the user's program solves
        state["plan"].set_coefficients(
            *state["plan"].assemble(state["mobility"]), *state["masks"])
    return state


def run(state):
    case, plan = state["case"], state["plan"]
    kind = case["kind"]
    if kind == "operator":
        return plan.operator_apply(state["x"])
    if kind == "cycle":
        return plan.mg_apply(state["rhs"])
    if kind == "solve":
        x, _ = plan.solve_pcg(state["rhs"], rtol=RTOL,
                              flexible=case["precision"] != "fp64")
        return plan.project_mean(x) if case["bc"] != "outlet" else x
    if kind == "adjoint":
        grad_b, grad_logrho, _ = plan.adjoint(
            state["mobility"], state["pressure"], state["grad_p"], rtol=RTOL)
        return grad_b, grad_logrho
    _, bx, by, bz = plan.assemble(state["mobility"])
    diag, rhs = plan.assemble_pressure_system(
        bx, by, bz, state["phi"], state["rho"], state["rho_n"],
        state["drho_dp"], state["bdf"], rho_nm1=state["rho_nm1"],
        source=state["source"])
    rhs = rhs * state["fluid"]
    plan.set_coefficients(diag, bx, by, bz, *state["masks"])
    pressure, _ = plan.solve_fgmres(rhs, rtol=RTOL)
    return diag, rhs, pressure


# -- the same in plain float64 torch ----------------------------------------
def _face_coefficients(mobility, faces, bc):
    """beta = A / (d_L / m_L + d_R / m_R) per axis; 0 on a Neumann face, the
    half cell alone on a Dirichlet face."""
    dev = mobility.device
    out = []
    for a in range(3):
        dim = 2 - a
        n = mobility.shape[dim]
        half = _along(0.5 * np.diff(faces[a]), a, dev)
        d_over_m = half / mobility
        first, last = d_over_m.narrow(dim, 0, 1), d_over_m.narrow(dim, n - 1,
                                                                  1)
        inner = d_over_m.narrow(dim, 0, n - 1) + d_over_m.narrow(dim, 1,
                                                                 n - 1)
        if bc[2 * a] == PERIODIC:
            sums = [last + first, inner, last + first]
        else:
            ends = [e if bc[2 * a + s] == DIRICHLET
                    else torch.full_like(e, math.inf)
                    for s, e in enumerate((first, last))]
            sums = [ends[0], inner, ends[1]]
        area = 1.0
        for t in range(3):
            if t != a:
                area = area * _along(np.diff(faces[t]), t, dev)
        out.append(area / torch.cat(sums, dim))
    return out


def _face_sum(beta):
    total = 0.0
    for a, b in enumerate(beta):
        dim = 2 - a
        n = b.shape[dim] - 1
        total = total + b.narrow(dim, 0, n) + b.narrow(dim, 1, n)
    return total


def _masked(diag, beta, fluid, face_fluid):
    """The operator with its solid rows the identity and no face across the
    solid's surface."""
    masked = [b * m for b, m in zip(beta, face_fluid)]
    diag = torch.where(fluid, diag - _face_sum(beta) + _face_sum(masked), 1.0)
    return diag, masked


def _neighbours(x, axis, bc):
    """The low and high neighbours' values of every cell along `axis`."""
    dim = 2 - axis
    n = x.shape[dim]
    first, last = x.narrow(dim, 0, 1), x.narrow(dim, n - 1, 1)

    def edge(kind, own, wrapped):
        if kind == PERIODIC:
            return wrapped
        return own if kind == NEUMANN else torch.zeros_like(own)

    low = torch.cat([edge(bc[2 * axis], first, last),
                     x.narrow(dim, 0, n - 1)], dim)
    high = torch.cat([x.narrow(dim, 1, n - 1),
                      edge(bc[2 * axis + 1], last, first)], dim)
    return low, high


def _apply(diag, beta, bc, x):
    y = diag * x
    for a, b in enumerate(beta):
        dim = 2 - a
        n = x.shape[dim]
        low, high = _neighbours(x, a, bc)
        y -= b.narrow(dim, 0, n) * low
        y -= b.narrow(dim, 1, n) * high
    return y


def _solve(diag, beta, bc, b, weight=None):
    """Jacobi-preconditioned CG, corrected on the true residual while that
    falls.  weight: the fluid cells of a singular system, whose residual is
    held in the range of the operator."""
    x, best = torch.zeros_like(b), math.inf
    correction = torch.zeros_like(b)
    for _ in range(4):
        r = b - _apply(diag, beta, bc, x + correction)
        if weight is not None:
            r = _zero_mean(r, weight)
        norm = float(torch.linalg.vector_norm(r))
        if not norm < best:
            break
        x, best = x + correction, norm
        if norm == 0.0:
            break
        correction = torch.zeros_like(b)
        z = r / diag
        p, rho = z.clone(), (r * z).sum()
        for it in range(1, 6001):
            q = _apply(diag, beta, bc, p)
            alpha = rho / (p * q).sum()
            correction += alpha * p
            r -= alpha * q
            z = r / diag
            rho, old = (r * z).sum(), rho
            p = z + (rho / old) * p
            if it % 50 == 0 and not float(torch.linalg.vector_norm(r)) > \
                    1e-8 * norm:
                break
    return x


def _zero_mean(x, weight):
    return torch.where(weight > 0.0, x - (x * weight).sum() / weight.sum(),
                       0.0)


def _pairs(v, axis):
    """Sums of neighbouring pairs along `axis`, an odd last entry alone."""
    dim = 2 - axis
    if v.shape[dim] % 2:
        v = torch.cat([v, torch.zeros_like(v.narrow(dim, 0, 1))], dim)
    return v.unflatten(dim, (-1, 2)).sum(dim + 1)


def _hierarchy(diag, beta, volume):
    """Aggregation of two cells per axis while it has more than three, the
    faces whose normal axis was coarsened halved; (D, faces, volume, axes
    coarsened) per level."""
    levels = []
    while True:
        axes = [a for a in range(3) if diag.shape[2 - a] > 3]
        levels.append((diag, beta, volume, axes))
        if not axes:
            return levels
        reaction = torch.where(volume > 0.0, diag - _face_sum(beta),
                               0.0).clamp(min=0.0)
        coarse = []
        for a, b in enumerate(beta):
            dim = 2 - a
            for t in axes:
                if t != a:
                    b = _pairs(b, t)
            if a in axes:
                last = b.shape[dim] - 1
                at = torch.arange(0, last + 2, 2, device=b.device).clamp(
                    max=last).unique()
                b = 0.5 * b.index_select(dim, at)
            coarse.append(b)
        for t in axes:
            reaction, volume = _pairs(reaction, t), _pairs(volume, t)
        beta = coarse
        diag = torch.where(volume > 0.0, reaction + _face_sum(beta), 1.0)


def _interpolate(x, axis, fine, periodic):
    """Linear interpolation (3/4, 1/4) from coarse to `fine` cells."""
    dim = 2 - axis
    n = x.shape[dim]
    i = torch.arange(fine, device=x.device)
    near = i // 2
    far = near + torch.where(i % 2 == 0, -1, 1)
    far = far % n if periodic else torch.where((far < 0) | (far >= n), near,
                                               far)
    return 0.75 * x.index_select(dim, near) + 0.25 * x.index_select(dim, far)


def _smooth(level, bc, x, b, sweeps, reverse):
    diag, beta = level[:2]
    nz, ny, nx = x.shape
    k, j, i = (torch.arange(v, device=x.device) for v in (nz, ny, nx))
    colour = (k[:, None, None] + j[None, :, None] + i[None, None, :]) % 2
    for _ in range(sweeps):
        for c in ((1, 0) if reverse else (0, 1)):
            defect = b - _apply(diag, beta, bc, x)
            x = torch.where(colour == c, x + OMEGA * defect / diag, x)
    return x


def _cycle(levels, at, bc, b, singular):
    """V(2,2) from zero, 24 sweeps on the coarsest level."""
    level = levels[at]
    diag, beta, volume, axes = level
    if singular:
        b = _zero_mean(b, volume)
    x = torch.zeros_like(b)
    if not axes:
        return _smooth(level, bc, x, b, 24, False)
    x = _smooth(level, bc, x, b, 2, False)
    coarse = b - _apply(diag, beta, bc, x)
    for a in axes:
        coarse = _pairs(coarse, a)
    e = _cycle(levels, at + 1, bc, coarse, singular)
    for a in axes:
        e = _interpolate(e, a, x.shape[2 - a], bc[2 * a] == PERIODIC)
    x = torch.where(volume > 0.0, x + e, 0.0)
    return _smooth(level, bc, x, b, 2, True)


def exact(case, seed):
    inputs = _inputs(case, seed)
    faces, bc, fluid = inputs["faces"], inputs["bc"], inputs["fluid"]
    face_fluid = inputs["face_fluid"]
    kind, singular = case["kind"], case["bc"] != "outlet"
    dev = fluid.device
    volume = 1.0
    for a in range(3):
        volume = volume * _along(np.diff(faces[a]), a, dev)
    weight = fluid.to(torch.float64)
    mobility = (inputs["dt"] if kind == "step" else 1.0) / inputs["rho"]
    beta = _face_coefficients(mobility, faces, bc)
    diag = _face_sum(beta)
    if kind == "step":
        a0, a1, a2 = inputs["bdf"]
        diag = a0 * volume * inputs["drho_dp"] + diag
        flux = 0.0
        for a, phi in enumerate(inputs["phi"]):
            flux = flux + phi.diff(dim=2 - a)
        rhs = -(volume * (a0 * inputs["rho"] + a1 * inputs["rho_n"] +
                          a2 * inputs["rho_nm1"] - inputs["source"]) + flux)
        rhs = rhs * weight
        pressure = _solve(*_masked(diag, beta, fluid, face_fluid), bc, rhs)
        return diag.reshape(-1), rhs.reshape(-1), pressure.reshape(-1)
    diag, beta = _masked(diag, beta, fluid, face_fluid)
    if kind == "operator":
        return _apply(diag, beta, bc, inputs["x"]).reshape(-1)
    if kind == "cycle":
        volume = volume * weight
        z = _cycle(_hierarchy(diag, beta, volume), 0, bc, inputs["rhs"],
                   singular)
        z = _zero_mean(z, volume) if singular else z * weight
        return z.reshape(-1)
    if kind == "solve":
        x = _solve(diag, beta, bc, inputs["rhs"],
                   weight if singular else None)
        return (_zero_mean(x, weight) if singular else x).reshape(-1)
    # adjoint: A lambda = P dL/dp, then -d/dlog(rho) of lambda . A(rho) p
    adjoint = _zero_mean(_solve(
        diag, beta, bc, _zero_mean(inputs["grad_p"], weight),
        weight), weight)
    log_rho = torch.log(inputs["rho"]).requires_grad_()
    beta = _face_coefficients(torch.exp(-log_rho), faces, bc)
    action = 0.0
    for a, b in enumerate(beta):
        dim = 2 - a

        # the two ends of a periodic axis are one face
        count = b.shape[dim] - (bc[2 * a] == PERIODIC)

        def jump(v):
            low, high = _neighbours(v, a, bc)
            return torch.cat([v.narrow(dim, 0, 1) - low.narrow(dim, 0, 1),
                              high - v], dim)

        terms = (b * face_fluid[a] * jump(adjoint) *
                 jump(inputs["pressure"]))
        action = action + terms.narrow(dim, 0, count).sum()
    gradient, = torch.autograd.grad(-action, log_rho)
    return adjoint.reshape(-1), gradient.reshape(-1)
