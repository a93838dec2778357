"""The work that programs built on easyfsi_amd have it do, as measurable cases.

A time step of such a program is: advect and diffuse the velocity (``predict``), project it
(``project``: multigrid-preconditioned CG), step the solid (``NeoHookeanMpmState.step``), classify
the grid nodes around the marker surface (``HibmMpmIbNodeSearch``) and hand the marker forces to the
solid's particles.  Beside it stand the learned initial guess's network (inference before a solve)
and its training.  Each family has a case at the sizes its users run; ``draw`` gives others of the
same ranges: small grids where launches and latency count, ordinary ones, odd and ragged extents.

Every case is a dict of plain values; ``family`` names the path, the other keys its sizes and options.
"""

import ctypes
import math

import numpy as np
import torch

RHO, MU, DT = 1000.0, 1.0e-3, 1.0e-3  # water-like fluid and a 1 ms step, as the package's own solvers use


# ---------------------------------------------------------------------------------------------
# The cases
# ---------------------------------------------------------------------------------------------

def listed():
    return [
        # A small closed box at the default precision, the report read: the tightest tolerance, and so few
        # cells that launches and host reads set the time.
        {"name": "project_64_default", "family": "project", "nx": 64, "ny": 64, "nz": 64, "growth": 1.0,
         "precision": "ref64", "tolerance": 1e-10, "outlet": False, "report": True, "radius": 0.0},
        # An ordinary graded grid around an obstacle at the default precision.
        {"name": "project_128_default", "family": "project", "nx": 128, "ny": 128, "nz": 128, "growth": 1.04,
         "precision": "ref64", "tolerance": 1e-8, "outlet": False, "report": True, "radius": 0.1},
        # Odd extents, three different ones, with the pressure outlet: the mixed solver.
        {"name": "project_ragged_mixed", "family": "project", "nx": 150, "ny": 97, "nz": 118, "growth": 1.03,
         "precision": "mixed", "tolerance": 1e-8, "outlet": True, "report": False, "radius": 0.12},
        # The large graded grid of the benchmark, mixed precision, no report.
        {"name": "project_256_mixed", "family": "project", "nx": 256, "ny": 256, "nz": 256, "growth": 1.04,
         "precision": "mixed", "tolerance": 1e-8, "outlet": False, "report": False, "radius": 0.06},
        # The predictor at its default scheme on the large grid.
        {"name": "predict_256_euler", "family": "predict", "nx": 256, "ny": 256, "nz": 256, "growth": 1.04,
         "scheme": "euler", "cfl": 1.0, "radius": 0.06},
        # The second-order back-trace on odd extents, with steps of two cells.
        {"name": "predict_ragged_rk2", "family": "predict", "nx": 141, "ny": 96, "nz": 203, "growth": 1.02,
         "scheme": "rk2", "cfl": 2.0, "radius": 0.1},
        # A small solid, loaded on its surface, whose report is read at every step: the smallest call.
        {"name": "mpm_32k", "family": "mpm", "px": 32, "py": 32, "pz": 32, "nodes": 64, "loaded": True, "report": True},
        # A large solid on a large grid, stepped without reading the report.
        {"name": "mpm_1m", "family": "mpm", "px": 100, "py": 100, "pz": 100, "nodes": 256, "loaded": False,
         "report": False},
        # The guess network as the 256^3 solve uses it (the 2:1-coarsened grid).
        {"name": "unet_infer_128", "family": "unet_infer", "nx": 128, "ny": 128, "nz": 128},
        # Training on the 2:1-coarsened grid of 128^3 projections: four Adam steps, then the weights are read.
        {"name": "unet_train_64", "family": "unet_train", "nx": 64, "ny": 64, "nz": 64, "steps": 4},
        # Marker forces handed to the particles of a large solid.
        {"name": "scatter_1m", "family": "scatter", "lattice": 100, "per_face": 64},
        # Node classification around a closed surface, far nodes included.
        {"name": "ib_search_128", "family": "ib_search", "nx": 128, "ny": 128, "nz": 128, "rings": 48, "segments": 64,
         "far": True},
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    family = rng.choice(["project", "project", "predict", "mpm", "mpm", "unet_infer", "unet_train", "scatter",
                         "ib_search"])
    if family == "project":
        precision = rng.choice(["ref64", "ref64", "fp32", "mixed", "mixed"])
        top = 220 if precision == "mixed" else 120
        n = [_log_int(rng, 40, top) for _ in range(3)]
        return {"family": family, "nx": n[0], "ny": n[1], "nz": n[2], "growth": rng.choice([1.0, 1.02, 1.04]),
                "precision": precision, "tolerance": rng.choice([1e-7, 1e-8]), "outlet": rng.random() < 0.4,
                "report": rng.random() < 0.5, "radius": rng.choice([0.0, round(rng.uniform(0.06, 0.2), 3)])}
    if family == "predict":
        n = [_log_int(rng, 32, 256) for _ in range(3)]
        return {"family": family, "nx": n[0], "ny": n[1], "nz": n[2], "growth": rng.choice([1.0, 1.02, 1.04]),
                "scheme": rng.choice(["euler", "rk2"]), "cfl": round(rng.uniform(0.5, 3.0), 2),
                "radius": rng.choice([0.0, round(rng.uniform(0.06, 0.2), 3)])}
    if family == "mpm":
        n = [_log_int(rng, 12, 100) for _ in range(3)]
        return {"family": family, "px": n[0], "py": n[1], "pz": n[2], "nodes": _log_int(rng, 48, 256),
                "loaded": rng.random() < 0.5, "report": rng.random() < 0.5}
    if family == "unet_infer":
        n = [4 * _log_int(rng, 6, 32) for _ in range(3)]
        return {"family": family, "nx": n[0], "ny": n[1], "nz": n[2]}
    if family == "unet_train":
        n = [4 * _log_int(rng, 6, 22) for _ in range(3)]
        return {"family": family, "nx": n[0], "ny": n[1], "nz": n[2], "steps": rng.choice([2, 4])}
    if family == "scatter":
        return {"family": family, "lattice": _log_int(rng, 20, 100), "per_face": _log_int(rng, 12, 64)}
    n = [_log_int(rng, 40, 128) for _ in range(3)]
    return {"family": family, "nx": n[0], "ny": n[1], "nz": n[2], "rings": _log_int(rng, 12, 48),
            "segments": _log_int(rng, 16, 64), "far": rng.random() < 0.7}


def _cells(c):
    return c["nx"] * c["ny"] * c["nz"]


# (cin, cout, level) of the network's 3x3x3 convolutions
_UNET = [(16, 16, 1), (16, 16, 1), (16, 32, 2), (32, 32, 2), (32, 64, 3), (64, 64, 3), (96, 32, 2), (32, 32, 2),
         (48, 16, 1), (16, 16, 1)]


def work(case):
    f = case["family"]
    if f == "project":  # velocity read and written, obstacle read, pressure written
        return {"bytes": 36.0 * _cells(case), "flops": 0.0}
    if f == "predict":  # velocity read and written, obstacle read
        return {"bytes": 28.0 * _cells(case), "flops": 0.0}
    if f == "mpm":
        # a particle: x, v, C, F read and written, mass, volume, external force, fixed, region, rest position read
        p = case["px"] * case["py"] * case["pz"]
        return {"bytes": (2 * 96.0 + 40.0) * p, "flops": 0.0}
    if f in ("unet_infer", "unet_train"):
        n = _cells(case)
        flops = sum(2.0 * 27 * a * b * n / 8 ** (lvl - 1) for a, b, lvl in _UNET) + 32.0 * n
        if f == "unet_infer":
            return {"bytes": 24.0 * n, "flops": flops}
        return {"bytes": 25.0 * n * case["steps"], "flops": 3.0 * flops * case["steps"]}
    if f == "scatter":
        p, m = case["lattice"] ** 3, 6 * case["per_face"] ** 2
        return {"bytes": 36.0 * p + 36.0 * m, "flops": 0.0}
    return {"bytes": 56.0 * _cells(case) + 36.0 * case["rings"] * case["segments"], "flops": 0.0}


def tolerance(case):
    f = case["family"]
    if f == "project":
        # two solves that stop at the same residual differ by the error that residual leaves in the pressure
        # (measured against 64 bits: up to 1e-7 at 1e-8) and by float32 rounding of the velocity (4e-8)
        return {"rel": 1e-5, "max": 1e-3} if case["tolerance"] > 3e-8 else {"rel": 1e-6, "max": 1e-4}
    if f == "predict":
        return "exact"  # every operation is the correctly rounded one of a fixed expression
    if f == "mpm":
        return {"rel": 2e-5, "max": 2e-3}  # float32 sums over particles and nodes, in another order
    if f == "unet_infer":
        return {"rel": 1e-2, "max": 1e-1}  # bf16 activations
    if f == "unet_train":
        return {"rel": 2e-2, "max": 0.8}  # bf16 activations and gradients, through Adam's normalised steps
    if f == "scatter":
        return {"rel": 1e-6, "max": 1e-4}  # float32 weight sums and atomics
    return "exact"  # choices between candidates by strict comparison in index order


# ---------------------------------------------------------------------------------------------
# Inputs
# ---------------------------------------------------------------------------------------------

def _gen(seed):
    g = torch.Generator(device="cuda")
    g.manual_seed(int(seed) + 1)
    return g


def _axis(n, growth):
    """Unit-length widths: half the cells equal in the middle, the rest growing towards both walls."""
    if growth == 1.0:
        return np.full(n, 1.0 / n)
    core = n - 2 * (n // 4)
    side = growth ** np.arange(1, n // 4 + 1)
    w = np.concatenate([side[::-1], np.ones(core), side])
    return w / w.sum()


def _smooth_velocity(shape, seed, kmax):
    """Random Fourier modes up to kmax per component, unit RMS, float32 [nx, ny, nz, 3]."""
    nx, ny, nz = shape
    k = [torch.fft.fftfreq(nx, 1.0 / nx, device="cuda"), torch.fft.fftfreq(ny, 1.0 / ny, device="cuda"),
         torch.fft.rfftfreq(nz, 1.0 / nz, device="cuda")]
    k2 = k[0][:, None, None] ** 2 + k[1][None, :, None] ** 2 + k[2][None, None, :] ** 2
    m = ((k2 > 0) & (k2 <= kmax * kmax)).to(torch.float32)
    g = _gen(seed)
    out = torch.empty(shape + (3,), dtype=torch.float32, device="cuda")
    for d in range(3):
        re, im = (torch.randn(m.shape, generator=g, device="cuda") for _ in range(2))
        f = torch.fft.irfftn(torch.complex(re * m, im * m), s=shape)
        out[..., d] = f / f.square().mean().sqrt()
    return out


def _fluid_inputs(case, seed):
    shape = (case["nx"], case["ny"], case["nz"])
    widths = [_axis(n, case["growth"]) for n in shape]
    rs = np.random.RandomState(seed % (2 ** 31))
    centre = 0.5 + rs.uniform(-0.05, 0.05, 3)
    if case["radius"] > 0:
        c = [torch.as_tensor(np.cumsum(w) - 0.5 * w, device="cuda") for w in widths]
        r2 = ((c[0][:, None, None] - centre[0]) ** 2 + (c[1][None, :, None] - centre[1]) ** 2
              + (c[2][None, None, :] - centre[2]) ** 2)
        obstacle = (r2 <= case["radius"] ** 2).to(torch.int32)
    else:
        obstacle = torch.zeros(shape, dtype=torch.int32, device="cuda")
    velocity = _smooth_velocity(shape, seed, 16 if min(shape) >= 64 else 8)
    return widths, obstacle, velocity


def _solver(widths, precision):
    from easyfsi_amd.simulation_core.fluid import CartesianFluidSolver
    from easyfsi_amd.simulation_core.grid import CartesianGrid, FluidDomainSpec

    g = CartesianGrid(bounds_min_m=(0.0, 0.0, 0.0), cell_widths_x_m=tuple(float(v) for v in widths[0]),
                      cell_widths_y_m=tuple(float(v) for v in widths[1]),
                      cell_widths_z_m=tuple(float(v) for v in widths[2]))
    spec = FluidDomainSpec(bounds_min_m=g.bounds_min_m, bounds_max_m=g.bounds_max_m, grid_nodes=None,
                           density_kgm3=RHO, viscosity_pa_s=MU, dt_s=DT, cartesian_grid=g)
    return CartesianFluidSolver(spec, solver_precision=precision)


def _solid_inputs(case, seed):
    """A block deformed by a smooth displacement, moving as a rotating body with a wave on it."""
    rs = np.random.RandomState(seed % (2 ** 31))
    counts = (case["px"], case["py"], case["pz"])
    longest = max(counts)
    half = [0.15 * c / longest for c in counts]
    lo, hi = [0.5 - h for h in half], [0.5 + h for h in half]
    amp, phase = 2e-3 * rs.uniform(0.5, 1.0, (3, 3)), rs.uniform(0, 2 * math.pi, (3, 3))
    return {"counts": counts, "lo": lo, "hi": hi, "amp": amp, "phase": phase, "omega": rs.uniform(-3, 3, 3),
            "drift": rs.uniform(-0.1, 0.1, 3)}


def _solid_fields(rest, s):
    """(x, v, C, F, force) of the rest positions [P, 3], float32."""
    X = rest.double()
    k = 2 * math.pi / 0.3
    amp = torch.as_tensor(s["amp"], device="cuda")
    ph = torch.as_tensor(s["phase"], device="cuda")
    arg = k * X[:, None, :] + ph[None]  # component, axis
    u = (amp * torch.sin(arg)).sum(2)
    G = amp * k * torch.cos(arg)  # du_i / dX_j
    x = X + u
    F = torch.eye(3, dtype=torch.float64, device="cuda") + G
    w = torch.as_tensor(s["omega"], device="cuda")
    v = torch.linalg.cross(w.expand_as(x), x - 0.5) + torch.as_tensor(s["drift"], device="cuda") + 10.0 * u
    W = torch.tensor([[0, -w[2], w[1]], [w[2], 0, -w[0]], [-w[1], w[0], 0]], dtype=torch.float64, device="cuda")
    C = W + 10.0 * G
    edge = ((X - 0.5).abs() / torch.as_tensor(s["hi"], device="cuda").sub(0.5)).amax(1) > 0.97
    force = torch.where(edge[:, None], 1e-3 * torch.sin(arg[:, :, 0]), torch.zeros_like(u))
    return x.float(), v.float(), C.float(), F.float(), force.float()


_SOLID = {"mu": 1.0e5 / (2 * 1.4), "lam": 1.0e5 * 0.4 / (1.4 * 0.2), "dt": 5.0e-5, "rho": 1000.0}


def _surface(case, seed):
    """A closed latitude-longitude sphere: positions, outward normals, triangles (float32, int32, on the GPU)."""
    rs = np.random.RandomState(seed % (2 ** 31))
    centre = 0.5 + rs.uniform(-0.03, 0.03, 3)
    rings, segs, radius = case["rings"], case["segments"], 0.3
    pts, idx = [(0.0, 0.0, 1.0)], []
    for r in range(1, rings):
        th = math.pi * r / rings
        for q in range(segs):
            ph = 2 * math.pi * q / segs
            pts.append((math.sin(th) * math.cos(ph), math.sin(th) * math.sin(ph), math.cos(th)))
    pts.append((0.0, 0.0, -1.0))
    at = lambda r, q: 1 + (r - 1) * segs + q % segs  # noqa: E731
    for q in range(segs):
        idx.append((0, at(1, q), at(1, q + 1)))
        for r in range(1, rings - 1):
            idx.append((at(r, q), at(r + 1, q), at(r + 1, q + 1)))
            idx.append((at(r, q), at(r + 1, q + 1), at(r, q + 1)))
        idx.append((len(pts) - 1, at(rings - 1, q + 1), at(rings - 1, q)))
    n = np.asarray(pts)
    return ((centre + radius * n).astype(np.float32), n.astype(np.float32), np.asarray(idx, np.int32))


def _marker_block(case, seed):
    n, m, g = case["lattice"], case["per_face"], _gen(seed)
    rs = np.random.RandomState(seed % (2 ** 31))
    shift = rs.uniform(-0.02, 0.02, 3)
    a = 0.35 + (torch.arange(n, device="cuda", dtype=torch.float64) + 0.5) * (0.3 / n)
    xp = torch.stack(torch.meshgrid(a, a, a, indexing="ij"), -1).reshape(-1, 3)
    xp = xp + (torch.rand(xp.shape, generator=g, device="cuda", dtype=torch.float64) - 0.5) * (0.2 * 0.3 / n)
    u = 0.35 + (torch.arange(m, device="cuda", dtype=torch.float64) + 0.5) * (0.3 / m)
    uu, vv = torch.meshgrid(u, u, indexing="ij")
    faces = []
    for axis in range(3):
        for side in (0.35, 0.65):
            f = torch.zeros((m * m, 3), dtype=torch.float64, device="cuda")
            f[:, axis] = side
            f[:, (axis + 1) % 3], f[:, (axis + 2) % 3] = uu.reshape(-1), vv.reshape(-1)
            faces.append(f)
    t = torch.as_tensor(shift, device="cuda")
    xm = (torch.cat(faces) + t).float()
    fm = torch.randn(xm.shape, generator=g, device="cuda", dtype=torch.float64)
    return (xp + t).float(), xm, fm, 2.0 * 0.3 / n


def _network_inputs(case, seed, count):
    """Features (normalised divergence, solid fraction, log2 widths), pressure-like targets and masks."""
    shape = (case["nx"], case["ny"], case["nz"])
    out = []
    for s in range(count):
        q = _smooth_velocity(shape, seed * 31 + s, 8)
        f = torch.empty(shape + (5,), dtype=torch.float32, device="cuda")
        f[..., 0] = q[..., 0]
        grid = [torch.linspace(-0.5, 0.5, n, device="cuda") for n in shape]
        r2 = grid[0][:, None, None] ** 2 + grid[1][None, :, None] ** 2 + grid[2][None, None, :] ** 2
        solid = (r2 < 0.15 ** 2)
        f[..., 1] = solid.float()
        for a in range(3):
            sh = [1, 1, 1]
            sh[a] = shape[a]
            f[..., 2 + a] = (6.0 * (grid[a].abs() - 0.25).clamp_min(0.0)).reshape(sh)
        out.append((f.reshape(-1, 5).contiguous(), (3.0 * q[..., 1] + q[..., 0]).contiguous(),
                    (~solid).reshape(-1).to(torch.uint8).contiguous()))
    return out


_WEIGHT_SEED = 7


def prepare(case, seed):
    f = case["family"]
    if f in ("project", "predict"):
        widths, obstacle, velocity = _fluid_inputs(case, seed)
        s = _solver(widths, case.get("precision", "ref64"))
        s.obstacle.tensor.copy_(obstacle)
        s.velocity.tensor.copy_(velocity)
        dt = case.get("cfl", 1.0) * min(float(w.min()) for w in widths) / float(velocity.abs().max())
        return {"case": case, "solver": s, "velocity": velocity, "dt": dt}
    if f == "mpm":
        from easyfsi_amd.simulation_core.neo_hookean_mpm import NeoHookeanMpmState

        i = _solid_inputs(case, seed)
        p = int(np.prod(i["counts"]))
        s = NeoHookeanMpmState(p, (0.0, 0.0, 0.0), (1.0, 1.0, 1.0), (case["nodes"],) * 3)
        s.initialize_box(particle_counts=i["counts"], box_min_m=i["lo"], box_max_m=i["hi"],
                         density_kgm3=_SOLID["rho"])
        x, v, C, F, force = _solid_fields(s.rest_x.tensor, i)
        for field, value in ((s.x, x), (s.v, v), (s.C, C), (s.F, F)):
            field.tensor.copy_(value)
        if case["loaded"]:
            s.external_force_n.tensor.copy_(force)
        s.region_id.tensor.fill_(1)
        return {"case": case, "solid": s}
    if f in ("unet_infer", "unet_train"):
        from easyfsi_amd.learned import GuessNetwork

        net = GuessNetwork((case["nx"], case["ny"], case["nz"]), train=f == "unet_train", seed=_WEIGHT_SEED)
        return {"case": case, "net": net, "data": _network_inputs(case, seed, case.get("steps", 1))}
    if f == "scatter":
        xp, xm, fm, h = _marker_block(case, seed)
        return {"case": case, "xp": xp, "xm": xm, "fm": fm, "h": h, "ext": torch.zeros_like(xp)}
    from easyfsi_amd import hibm

    x, n, tris = _surface(case, seed)
    markers = hibm.HibmMpmSurfaceMarkers(marker_capacity=len(x), projection_triangle_capacity=len(tris))
    markers.x_gamma_m.tensor.copy_(torch.from_numpy(x))
    markers.n_gamma.tensor.copy_(torch.from_numpy(n))
    markers.projection_triangle_indices.tensor.copy_(torch.from_numpy(tris))
    markers.marker_count, markers.projection_triangle_count = len(x), len(tris)
    search = hibm.HibmMpmIbNodeSearch(grid_nodes=(case["nx"], case["ny"], case["nz"]), bounds_min_m=(0.0, 0.0, 0.0),
                                      bounds_max_m=(1.0, 1.0, 1.0), marker_capacity=len(x))
    return {"case": case, "markers": markers, "search": search}


# ---------------------------------------------------------------------------------------------
# One pass
# ---------------------------------------------------------------------------------------------

def run(state):
    case = state["case"]
    f = case["family"]
    if f == "project":
        s = state["solver"]
        s.velocity.tensor.copy_(state["velocity"])
        s.project(iterations=500, pressure_outlet_zmin=case["outlet"], pressure_solver="fv_cg",
                  cg_preconditioner="fv_multigrid", cg_tolerance=case["tolerance"], reset_pressure=True,
                  read_report=case["report"])
        return {"velocity": s.velocity.tensor, "pressure": s.pressure.tensor}
    if f == "predict":
        s = state["solver"]
        s.predict(state["dt"], advection_scheme=case["scheme"])
        return s.velocity.tensor
    if f == "mpm":
        s = state["solid"]
        s.step(dt_s=_SOLID["dt"], mu_pa=_SOLID["mu"], lambda_pa=_SOLID["lam"], primary_region_id=1,
               secondary_region_id=2, read_report=case["report"])
        return {"x": s.x.tensor, "v": s.v.tensor, "C": s.C.tensor, "F": s.F.tensor}
    if f == "unet_infer":
        return state["net"].forward(state["data"][0][0])
    if f == "unet_train":
        from easyfsi_amd import _lib

        net = state["net"]
        for features, target, mask in state["data"]:
            net.train_step(features, target, mask, lr=1e-4)
        grads = np.empty(net.num_params, np.float32)
        _lib.check(_lib.lib().hfsi_unet_get_grads(net._h, grads.ctypes.data_as(ctypes.c_void_p), _lib.stream_handle()),
                   "hfsi_unet_get_grads")
        return {"params": net.get_params(), "grads": grads}
    if f == "scatter":
        from easyfsi_amd import hibm

        state["ext"].zero_()
        rep = hibm.scatter_marker_forces_to_mpm_particles(
            state["xm"], state["fm"], state["ext"], state["xp"], particle_count=state["xp"].shape[0],
            support_radius_m=state["h"])
        return {"force": state["ext"], "pairs": rep.active_particle_count, "markers": rep.active_marker_count}
    s = state["search"]
    h = max(s.spacing_m)
    rep = s.search_and_classify(state["markers"], search_radius_m=2 * h, interior_probe_distance_m=h,
                                classify_far_internal_nodes=case["far"])
    return {"kind": s.node_kind_code.tensor, "marker": s.nearest_marker.tensor,
            "signed_distance": s.node_signed_distance_m.tensor, "point": s.node_boundary_point_m.tensor,
            "interior": s.node_interior_fluid_point_m.tensor, "indices": s.node_projection_marker_indices.tensor,
            "weights": s.node_projection_marker_weights.tensor, "near": rep.near_boundary_node_count,
            "internal": rep.internal_node_count}


# ---------------------------------------------------------------------------------------------
# The same results in 64 bits
# ---------------------------------------------------------------------------------------------

def exact(case, seed):
    f = case["family"]
    with torch.no_grad():
        if f == "project":
            return _exact_project(case, seed)
        if f == "predict":
            return _exact_predict(case, seed)
        if f == "mpm":
            return _exact_mpm(case, seed)
        if f in ("unet_infer", "unet_train"):
            return _exact_network(case, seed)
        if f == "scatter":
            return _exact_scatter(case, seed)
        return _exact_ib(case, seed)


def _metrics(widths):
    """Widths and distances of neighbouring centres, rounded as the solver stores them, in 64 bits."""
    w, d = [], []
    for a in widths:
        edges = np.concatenate([[0.0], np.cumsum(a)])
        c = 0.5 * (edges[1:] + edges[:-1])
        w.append(torch.as_tensor(a.astype(np.float32).astype(np.float64), device="cuda"))
        d.append(torch.as_tensor(np.diff(c).astype(np.float32).astype(np.float64), device="cuda"))
    return w, d


def _on(axis, v):
    sh = [1, 1, 1]
    sh[axis] = -1
    return v.reshape(sh)


def _exact_project(case, seed):
    widths, obstacle, velocity = _fluid_inputs(case, seed)
    w, d = _metrics(widths)
    outlet, free = case["outlet"], obstacle == 0
    u = velocity.double()
    shape = obstacle.shape

    def boundary(u):
        if outlet:
            z = u[:, :, 0, 2]
            u[:, :, 0, 2] = torch.where(free[:, :, 0] & (z > 0), torch.zeros_like(z), z)
            u[0, :, :, 0] = 0.0
            u[:, 0, :, 1] = 0.0

    boundary(u)
    V = _on(0, w[0]) * _on(1, w[1]) * _on(2, w[2]) * free
    T, open_ = [], []
    for a in range(3):
        lo, hi = free.narrow(a, 0, shape[a] - 1), free.narrow(a, 1, shape[a] - 1)
        open_.append(lo & hi)
        area = _on((a + 1) % 3, w[(a + 1) % 3]) * _on((a + 2) % 3, w[(a + 2) % 3])
        T.append(torch.where(open_[a], area / _on(a, d[a]), torch.zeros((), dtype=torch.float64, device="cuda")))
    t_out = 2.0 / w[2][0] ** 2 * V[:, :, 0] if outlet else None

    def divergence(u):
        out = torch.zeros(shape, dtype=torch.float64, device="cuda")
        for a in range(3):
            face = torch.where(open_[a], u[..., a].narrow(a, 1, shape[a] - 1), torch.zeros((), dtype=torch.float64,
                                                                                        device="cuda"))
            out.narrow(a, 0, shape[a] - 1).add_(face / _on(a, w[a][:-1]))
            out.narrow(a, 1, shape[a] - 1).sub_(face / _on(a, w[a][1:]))
        if outlet:
            out[:, :, 0] -= u[:, :, 0, 2] / w[2][0]
        return out * free

    def apply(p):  # V times the operator
        q = torch.zeros_like(p)
        for a in range(3):
            flux = T[a] * (p.narrow(a, 1, shape[a] - 1) - p.narrow(a, 0, shape[a] - 1))
            q.narrow(a, 1, shape[a] - 1).add_(flux)
            q.narrow(a, 0, shape[a] - 1).sub_(flux)
        if outlet:
            q[:, :, 0] += t_out * p[:, :, 0]
        return q

    diag = torch.zeros(shape, dtype=torch.float64, device="cuda")
    for a in range(3):
        diag.narrow(a, 0, shape[a] - 1).add_(T[a])
        diag.narrow(a, 1, shape[a] - 1).add_(T[a])
    if outlet:
        diag[:, :, 0] += t_out
    inv = torch.where(diag > 0, 1.0 / diag, torch.zeros_like(diag))
    b = -(RHO / DT) * divergence(u) * V
    if not outlet:
        b = b - V * (b.sum() / V.sum())
    x, r = torch.zeros_like(b), b.clone()
    z = inv * r
    p, rz, stop = z.clone(), float((r * z).sum()), 1e-11 * float((b * inv * b).sum()) ** 0.5
    for _ in range(6000):
        q = apply(p)
        alpha = rz / float((p * q).sum())
        x.add_(p, alpha=alpha)
        r.sub_(q, alpha=alpha)
        z = inv * r
        new = float((r * z).sum())
        if new ** 0.5 <= stop:
            break
        p.mul_(new / rz).add_(z)
        rz = new
    if not outlet:
        x = (x - (V * x).sum() / V.sum()) * free
    for a in range(3):
        g = torch.where(open_[a], (x.narrow(a, 1, shape[a] - 1) - x.narrow(a, 0, shape[a] - 1)) / _on(a, d[a]),
                        torch.zeros((), dtype=torch.float64, device="cuda"))
        u[..., a].narrow(a, 1, shape[a] - 1).sub_(DT / RHO * g)
    if outlet:
        u[:, :, 0, 2] -= DT / RHO * 2.0 * x[:, :, 0] / w[2][0]
    u = u * free[..., None]
    boundary(u)
    u[0, :, :, 0] = 0.0
    u[:, 0, :, 1] = 0.0
    if not outlet:
        u[:, :, 0, 2] = 0.0
    return {"velocity": u, "pressure": x}


def _exact_predict(case, seed):
    widths, obstacle, velocity = _fluid_inputs(case, seed)
    dt = case["cfl"] * min(float(v.min()) for v in widths) / float(velocity.abs().max())
    w, d = _metrics(widths)
    shape = obstacle.shape
    u, free = velocity.double(), obstacle == 0
    edges = [torch.as_tensor(np.concatenate([[0.0], np.cumsum(a)]), device="cuda") for a in widths]
    c = [0.5 * (e[1:] + e[:-1]) for e in edges]
    flat_u, flat_free = u.reshape(-1, 3), free.reshape(-1)

    def coordinate(pos, a):
        ca, n = c[a], shape[a]
        lo = (torch.searchsorted(ca, pos, right=True) - 1).clamp(0, n - 2)
        g = lo.double() + (pos - ca[lo]) / (ca[lo + 1] - ca[lo])
        g = torch.where(pos <= ca[0], -0.5 * (ca[0] - pos) / (ca[0] - edges[a][0]), g)
        return torch.where(pos >= ca[-1], n - 1 + 0.5 * (pos - ca[-1]) / (edges[a][-1] - ca[-1]), g)

    def sample(trace, step):
        i0, t = [], []
        for a in range(3):
            g = coordinate(_on(a, c[a]).expand(shape).contiguous() - step * trace[..., a], a)
            k = g.floor().clamp(0, shape[a] - 2)
            i0.append(k.long())
            t.append((g - k).clamp(0, 1))
        value, weight = torch.zeros_like(u), torch.zeros(shape, dtype=torch.float64, device="cuda")
        for o in range(8):
            off = (o >> 2 & 1, o >> 1 & 1, o & 1)
            q = t[0] * 0 + 1
            for a in range(3):
                q = q * (t[a] if off[a] else 1 - t[a])
            at = ((i0[0] + off[0]) * shape[1] + i0[1] + off[1]) * shape[2] + i0[2] + off[2]
            q = q * flat_free[at]
            value += q[..., None] * flat_u[at]
            weight += q
        some = weight > 1e-12
        return torch.where(some[..., None], value / torch.where(some, weight, 1.0)[..., None], u)

    trace = sample(u, 0.5 * dt) if case["scheme"] == "rk2" else u
    out = sample(trace, dt)
    for a in range(3):
        n = shape[a] - 1
        both = free.narrow(a, 1, n), free.narrow(a, 0, n)
        diff = (u.narrow(a, 1, n) - u.narrow(a, 0, n)) / _on(a, d[a])[..., None]
        lap = torch.zeros_like(u)
        lap.narrow(a, 0, n).add_(diff * both[0][..., None])
        lap.narrow(a, 1, n).sub_(diff * both[1][..., None])
        out += (dt * MU / RHO) * lap / _on(a, w[a])[..., None]
    return out * free[..., None]


def _exact_mpm(case, seed):
    i = _solid_inputs(case, seed)
    n, p = case["nodes"], int(np.prod(i["counts"]))
    axes, lo, hi = [], np.float32(i["lo"]), np.float32(i["hi"])
    for a, m in enumerate(i["counts"]):
        axes.append((lo[a] + (np.arange(m, dtype=np.float32) + np.float32(0.5)) * (hi[a] - lo[a]) / np.float32(m)))
    z, y, x0 = (torch.as_tensor(v.astype(np.float32), device="cuda") for v in axes[::-1])
    grid = torch.meshgrid(z, y, x0, indexing="ij")  # x fastest
    rest = torch.stack([grid[2].reshape(-1), grid[1].reshape(-1), grid[0].reshape(-1)], 1)
    x, v, C, F, force = (t.double() for t in _solid_fields(rest, i))
    vol = float(np.float32(np.prod((hi - lo).astype(np.float32)) / np.float32(p)))
    mass, dx, dt = float(np.float32(np.float32(_SOLID["rho"]) * np.float32(vol))), 1.0 / n, _SOLID["dt"]
    force = force if case["loaded"] else torch.zeros_like(force)
    J = torch.linalg.det(F)
    Fit = torch.linalg.inv(F).transpose(1, 2)
    P = _SOLID["mu"] * (F - Fit) + _SOLID["lam"] * J.log()[:, None, None] * Fit
    A = -dt * vol * (4 / dx ** 2) * torch.matmul(P, F.transpose(1, 2).contiguous()) + mass * C
    X = x / dx
    base = (X - 0.5).floor()
    fx = X - base
    w = [0.5 * (1.5 - fx) ** 2, 0.75 - (fx - 1) ** 2, 0.5 * (fx - 0.5) ** 2]
    gm = torch.zeros(n ** 3, dtype=torch.float64, device="cuda")
    gp = torch.zeros((n ** 3, 3), dtype=torch.float64, device="cuda")
    nodes = []
    for o in range(27):
        off = torch.tensor([o // 9, o // 3 % 3, o % 3], dtype=torch.float64, device="cuda")
        k = (o // 9, o // 3 % 3, o % 3)
        wt = w[k[0]][:, 0] * w[k[1]][:, 1] * w[k[2]][:, 2]
        b = (base + off).long()
        at = (b[:, 0] * n + b[:, 1]) * n + b[:, 2]
        r = (off - fx) * dx
        gm.index_add_(0, at, wt * mass)
        gp.index_add_(0, at, wt[:, None] * (mass * v + (A * r[:, None, :]).sum(2) + dt * force))
        nodes.append((wt, at, r))
    gv = gp / torch.where(gm > 1e-20, gm, 1.0)[:, None] * (gm > 1e-20)[:, None]
    nv, nC = torch.zeros_like(v), torch.zeros_like(C)
    for wt, at, r in nodes:
        q = wt[:, None] * gv[at]
        nv += q
        nC += q[:, :, None] * (4.0 / dx ** 2 * r)[:, None, :]
    nF = F + dt * torch.matmul(nC, F)
    return {"x": x + dt * nv, "v": nv, "C": nC, "F": nF}


class _Conv3(torch.autograd.Function):
    """3x3x3 convolution, zero padding, as 27 matrix products: x [D, H, W, cin], w [cout, 27, cin]."""

    @staticmethod
    def taps(x):
        D, H, W, _ = x.shape
        p = torch.nn.functional.pad(x, (0, 0, 1, 1, 1, 1, 1, 1))
        for t in range(27):
            a, b, c = t // 9, t // 3 % 3, t % 3
            yield t, p[a:a + D, b:b + H, c:c + W].reshape(-1, x.shape[3])

    @staticmethod
    def forward(ctx, x, w):
        ctx.save_for_backward(x, w)
        out = 0
        for t, s in _Conv3.taps(x):
            out = out + s @ w[:, t].T.contiguous()
        return out.reshape(x.shape[:3] + (w.shape[0],))

    @staticmethod
    def backward(ctx, g):
        x, w = ctx.saved_tensors
        flat = g.reshape(-1, w.shape[0])
        dw = torch.stack([flat.T @ s for _, s in _Conv3.taps(x)], 1)
        dx = 0
        for t, s in _Conv3.taps(g.contiguous()):
            dx = dx + s @ w[:, 26 - t].contiguous()
        return dx.reshape(x.shape), dw


def _exact_network(case, seed):
    from easyfsi_amd.learned import GuessNetwork

    shape = (case["nx"], case["ny"], case["nz"])
    start = GuessNetwork((8, 8, 8), seed=_WEIGHT_SEED).get_params()  # the initial weights are the handle's
    theta = torch.as_tensor(start, dtype=torch.float64, device="cuda")

    def forward(theta, features):
        at = 0
        wb = []
        for ci, co, _ in _UNET:
            wb.append((theta[at:at + co * 27 * ci].reshape(co, 27, ci), theta[at + co * 27 * ci:at + co * 27 * ci + co]))
            at += co * 27 * ci + co
        x = torch.zeros(shape + (16,), dtype=torch.float64, device="cuda")
        x[..., :5] = features.double().reshape(shape + (5,))
        conv = lambda x, k: torch.relu(_Conv3.apply(x, wb[k][0]) + wb[k][1])  # noqa: E731

        def pool(x):
            D, H, W, c = x.shape
            return x.reshape(D // 2, 2, H // 2, 2, W // 2, 2, c).mean((1, 3, 5))

        def up(x):
            return x.repeat_interleave(2, 0).repeat_interleave(2, 1).repeat_interleave(2, 2)

        s1 = conv(conv(x, 0), 1)
        s2 = conv(conv(pool(s1), 2), 3)
        b3 = conv(conv(pool(s2), 4), 5)
        d2 = conv(conv(torch.cat([up(b3), s2], 3), 6), 7)
        d1 = conv(conv(torch.cat([up(d2), s1], 3), 8), 9)
        return (d1 * theta[at:at + 16]).sum(3) + theta[at + 16]

    data = _network_inputs(case, seed, case.get("steps", 1))
    if case["family"] == "unet_infer":
        return forward(theta, data[0][0])
    m, v, g = torch.zeros_like(theta), torch.zeros_like(theta), None
    for k, (features, target, mask) in enumerate(data, 1):
        with torch.enable_grad():
            th = theta.clone().requires_grad_(True)
            on = mask.reshape(shape).bool()
            t = target.double()
            loss = (forward(th, features) - t)[on].square().sum() / t[on].square().sum()
            g, = torch.autograd.grad(loss, th)
        m, v = 0.9 * m + 0.1 * g, 0.999 * v + 0.001 * g * g
        theta = theta - 1e-4 * (m / (1 - 0.9 ** k)) / ((v / (1 - 0.999 ** k)).sqrt() + 1e-8)
    return {"params": theta, "grads": g}


def _exact_scatter(case, seed):
    xp, xm, fm, h = _marker_block(case, seed)
    h = float(np.float32(h))
    p, out = xp.double(), torch.zeros(xp.shape, dtype=torch.float64, device="cuda")
    order = torch.argsort(p[:, 0])
    first = p[order, 0].contiguous()
    # the markers by x, in groups whose particles are a slab of the sorted ones
    by_x = torch.argsort(xm[:, 0])
    for part in by_x.split(512):
        y = xm[part].double()
        a = int(torch.searchsorted(first, (y[:, 0].min() - h).reshape(1)))
        b = int(torch.searchsorted(first, (y[:, 0].max() + h).reshape(1), right=True))
        idx = order[a:b]
        w_sum = torch.zeros(len(part), dtype=torch.float64, device="cuda")
        kept = []
        for at in idx.split(1 << 16):
            w = torch.ones((len(part), len(at)), dtype=torch.float64, device="cuda")
            for axis in range(3):
                w *= (1 - (p[at, axis][None] - y[:, axis][:, None]).abs() / h).clamp_min(0)
            w_sum += w.sum(1)
            mk, pk = w.nonzero(as_tuple=True)
            kept.append((mk, at[pk], w[mk, pk]))
        for mk, pk, w in kept:
            out.index_add_(0, pk, (w / w_sum[mk])[:, None] * fm[part][mk])
    return {"force": out, "pairs": None, "markers": None}


def _exact_ib(case, seed):
    x, _, tris = _surface(case, seed)
    shape = (case["nx"], case["ny"], case["nz"])
    v = torch.as_tensor(x, device="cuda").double()
    t = torch.as_tensor(tris.astype(np.int64), device="cuda")
    a, b, c = v[t[:, 0]], v[t[:, 1]], v[t[:, 2]]
    axes = [(torch.arange(n, device="cuda", dtype=torch.float64) + 0.5) / n for n in shape]
    nodes = torch.stack(torch.meshgrid(*axes, indexing="ij"), -1).reshape(-1, 3)
    radius = 2.0 / min(shape)
    centre = v.mean(0)
    r = (nodes - centre).norm(dim=1)
    inside_only = float((v - centre).norm(dim=1).max())
    pick = (r < inside_only + radius) if case["far"] else ((r - 0.3).abs() < radius + 0.03)
    pick = pick.nonzero().reshape(-1)
    ab, ac, bc = b - a, c - a, c - b
    normal = torch.linalg.cross(ab, ac)
    normal = normal / normal.norm(dim=1, keepdim=True)
    point = torch.zeros_like(nodes)
    for at in pick.split(max(1, (1 << 23) // len(t))):
        p = nodes[at][:, None, :]
        best_d = torch.full((len(at), len(t)), 1e30, dtype=torch.float64, device="cuda")
        best = torch.zeros((len(at), len(t), 3), dtype=torch.float64, device="cuda")
        for o, e in ((a, ab), (a, ac), (b, bc)):  # the edges
            s = (((p - o) * e).sum(2) / (e * e).sum(1)).clamp(0, 1)
            q = o + s[..., None] * e
            dist = (p - q).square().sum(2)
            near = dist < best_d
            best_d, best = torch.where(near, dist, best_d), torch.where(near[..., None], q, best)
        height = ((p - a) * normal).sum(2)
        q = p - height[..., None] * normal  # the plane, where its foot is inside the triangle
        foot = ((torch.linalg.cross(ab.expand_as(q), q - a) * normal).sum(2) >= 0) \
            & ((torch.linalg.cross(bc.expand_as(q), q - b) * normal).sum(2) >= 0) \
            & ((torch.linalg.cross(-ac.expand_as(q), q - c) * normal).sum(2) >= 0) & (height.square() < best_d)
        best_d, best = torch.where(foot, height.square(), best_d), torch.where(foot[..., None], q, best)
        d, k = best_d.min(1)
        row = torch.arange(len(at), device="cuda")
        found = d.sqrt() < radius
        if case["far"]:  # deep nodes: behind every face of the closed surface
            found |= r[at] < 0.3 - radius
        point[at] = best[row, k] * found[:, None]
    out = {k: None for k in ("kind", "marker", "signed_distance", "interior", "indices", "weights", "near", "internal")}
    out["point"] = point.reshape(shape + (3,))
    return out
