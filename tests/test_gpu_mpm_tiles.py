"""The tile path of the binned MPM step: per-cell P2G scatter, force pass, stale-block clearing, binned G2P.

  - A block of particles moving one grid cell per step crosses 8^3-node block boundaries for 12 steps:
    every step's grid (mass, momentum/velocity, force) and particle state equal those of the atomic
    scatter, which clears the whole grid every step, from the same particle state, to float32 summation
    order (grid mass and force 1e-5, grid momentum m v and particle v 1e-4 of their maxima, C 1e-5 of its
    natural scale 4 max|v| / dx), and every
    node the atomic path leaves at zero is exactly zero (the blocks the previous step wrote are cleared).
  - Dense cells: 40 particles stacked in each of a few cells (ranks up to 39, past the 32 layers) and
    1500 particles in one 8^3 block (more than one 1024-particle pass), against the float64 oracle
    (same tolerances as the other MPM parity tests).
  - External forces on a subset of the particles reach the grid force through the force pass only in
    the blocks that hold them (against the atomic path).
  - Arrays written between steps are cleared by the next step after invalidate_grid.
"""

import numpy as np
import pytest
import torch

from easyfsi_amd.simulation_core.hyperelastic import ecoflex_0010_material
from oracle import mpm as M

pytestmark = pytest.mark.gpu

MAT = ecoflex_0010_material()
MU, LAM = MAT.shear_modulus_pa, MAT.lame_lambda_pa


def _say(msg):
    print(msg, flush=True)


def _state(nodes, counts, box_lo, box_hi, p2g, capacity=None):
    from easyfsi_amd.simulation_core.neo_hookean_mpm import NeoHookeanMpmState

    P = int(np.prod(counts))
    s = NeoHookeanMpmState(capacity or P, (0.0, 0.0, 0.0), (1.0, 1.0, 1.0), nodes)
    s.set_p2g_mode(p2g)
    s.initialize_box(particle_counts=counts, box_min_m=box_lo, box_max_m=box_hi, density_kgm3=MAT.density_kgm3)
    return s


def _max_rel(a, b):
    a, b = np.asarray(a, np.float64), np.asarray(b, np.float64)
    return float(np.abs(a - b).max()) / max(float(np.abs(b).max()), 1e-30)


def _grid(s):
    return s.grid_mass_kg.to_numpy(), s.grid_velocity_mps.to_numpy(), s.grid_force_n.to_numpy()


def test_moving_block_matches_atomic_scatter_and_clears_left_blocks():
    _say("moving 20^3-particle block on a 64^3 grid, 12 steps of one cell, binned tiles vs atomic scatter")
    states = {m: _state((64, 64, 64), (20, 20, 20), (0.2, 0.25, 0.3), (0.3, 0.35, 0.4), m) for m in ("binned", "atomic")}
    for s in states.values():
        n = s.particle_count
        x = s.x.tensor[:n]
        v = torch.zeros_like(x)
        # one cell per step along x at dt = 2e-4 (the material's wave speed, 39 m/s, crosses half a cell)
        v[:, 0], v[:, 1], v[:, 2] = 80.0, -30.0, 42.5
        v[:, 0] += -25.0 * (x[:, 1] - 0.3)
        v[:, 1] += 25.0 * (x[:, 0] - 0.25)
        s.v.tensor[:n] = v
        s.external_force_n.tensor[: n // 3] = torch.tensor([0.0, 0.0, -2e-5], device="cuda")
    sb, sa = states["binned"], states["atomic"]
    for step in range(12):
        # both steps start from the binned run's particle state, so they differ by summation order only
        n = sb.particle_count
        for f in ("x", "v", "C", "F", "external_force_n"):
            getattr(sa, f).tensor[:n] = getattr(sb, f).tensor[:n]
        reps = {m: s.step(dt_s=2e-4, mu_pa=MU, lambda_pa=LAM, primary_region_id=1, secondary_region_id=2)
                for m, s in states.items()}
        gb, ga = _grid(sb), _grid(sa)
        # grid velocity as momentum m v: p / m at nodes of tiny mass amplifies the float32 rounding of both
        e_m, e_v, e_f = (_max_rel(gb[0], ga[0]), _max_rel(gb[0][..., None] * gb[1], ga[0][..., None] * ga[1]),
                         _max_rel(gb[2], ga[2]))
        zero = ga[0] == 0.0
        stray = int(np.count_nonzero(gb[0][zero])) + int(np.count_nonzero(gb[1][zero])) + \
            int(np.count_nonzero(gb[2][zero]))
        n = states["binned"].particle_count
        e_pv = _max_rel(states["binned"].v.to_numpy()[:n], states["atomic"].v.to_numpy()[:n])
        # C sums node velocities times 4 dpos / dx^2 (terms of size 4 |v| / dx that cancel down to |C|): its
        # float32 summation-order floor is relative to that natural scale
        va = states["atomic"].v.to_numpy()[:n]
        c_nat = 4.0 * float(np.abs(va).max()) * 64.0
        e_pc = float(np.abs(states["binned"].C.to_numpy()[:n].astype(np.float64)
                            - states["atomic"].C.to_numpy()[:n]).max()) / c_nat
        if step in (0, 5, 11):
            _say(f"  step {step}: grid mass {e_m:.1e}, momentum {e_v:.1e}, force {e_f:.1e}, particle v {e_pv:.1e}, "
                 f"C {e_pc:.1e} of 4 max|v|/dx; nonzero nodes where the atomic grid is zero: {stray}; active "
                 f"{reps['binned'].active_grid_nodes}")
        assert reps["binned"].active_grid_nodes == reps["atomic"].active_grid_nodes, step
        assert stray == 0, step
        assert e_m <= 1e-5 and e_v <= 1e-4 and e_f <= 1e-5, (step, e_m, e_v, e_f)
        assert e_pv <= 1e-4 and e_pc <= 1e-5, (step, e_pv, e_pc)
    xb = states["binned"].x.to_numpy()[:n]
    assert reps["binned"].grid_out_of_bounds_particle_count == 0
    assert float(xb[:, 0].min()) > 0.2 + 10.0 / 64  # the block has moved by more than one 8-node block


def _compare_oracle(s, o, rep, ref):
    n = s.particle_count
    assert rep.active_grid_nodes == ref.values["active_grid_nodes"]
    errs = {"x": float(np.abs(s.x.to_numpy()[:n] - o.x).max()),
            "v": _max_rel(s.v.to_numpy()[:n], o.v), "F": float(np.abs(s.F.to_numpy()[:n] - o.F).max()),
            "grid mass": _max_rel(s.grid_mass_kg.to_numpy(), ref.grid_mass)}
    _say("  errors vs oracle: " + ", ".join(f"{k} {v:.2e}" for k, v in errs.items()))
    assert errs["x"] <= 1e-6 and errs["v"] <= 2e-4 and errs["F"] <= 1e-5 and errs["grid mass"] <= 1e-5


def test_dense_cells_and_a_crowded_block_match_oracle():
    _say("dense cells (40 per cell) and a 1500-particle block on a 32^3 grid vs the oracle")
    rng = np.random.default_rng(5)
    dx = 1.0 / 32
    # 12 cells with 40 particles each sharing one stencil-base node (X - 0.5 inside [c, c + 1)), plus 1500
    # particles whose base nodes all lie in the 8^3-node block 1..1..1 (X - 0.5 inside [8, 16))
    cells = rng.integers(4, 27, size=(12, 3))
    stacked = (cells[:, None, :] + 0.5 + rng.uniform(0.02, 0.98, size=(12, 40, 3))) * dx
    crowd = (8.5 + rng.uniform(0.01, 7.99, size=(1500, 3))) * dx
    pts = np.concatenate([stacked.reshape(-1, 3), crowd]).astype(np.float32)
    n = len(pts)
    s = _state((32, 32, 32), (1, 1, n), (0.4,) * 3, (0.6,) * 3, "binned", capacity=n)
    s.x.tensor[:n] = torch.from_numpy(pts).cuda()
    s.rest_x.tensor[:n] = s.x.tensor[:n]
    s.v.tensor[:n] = torch.from_numpy(rng.normal(0.0, 0.05, size=(n, 3)).astype(np.float32)).cuda()
    Fd = np.eye(3) + rng.normal(0.0, 0.02, size=(n, 3, 3))
    s.F.tensor[:n] = torch.from_numpy(Fd.astype(np.float32)).cuda()
    s.external_force_n.tensor[:200] = torch.from_numpy(rng.normal(0, 1e-4, size=(200, 3)).astype(np.float32)).cuda()
    s.invalidate_grid()
    for step in range(3):
        o = M.MpmState(x=s.x.to_numpy()[:n].astype(np.float64), v=s.v.to_numpy()[:n].astype(np.float64),
                       C=s.C.to_numpy()[:n].astype(np.float64), F=s.F.to_numpy()[:n].astype(np.float64),
                       mass=s.mass_kg.to_numpy()[:n].astype(np.float64),
                       volume=s.volume_m3.to_numpy()[:n].astype(np.float64),
                       rest_x=s.rest_x.to_numpy()[:n].astype(np.float64), fixed=np.zeros(n, np.int32),
                       region=np.zeros(n, np.int32), f_ext=s.external_force_n.to_numpy()[:n].astype(np.float64),
                       normal=np.zeros((n, 3)), rest_normal=np.zeros((n, 3)), area=np.zeros(n), rest_area=np.zeros(n))
        ref = M.step(o, bounds_min=(0.0, 0.0, 0.0), bounds_max=(1.0, 1.0, 1.0), grid_nodes=(32, 32, 32), dt=1e-4,
                     mu=MU, lam=LAM)
        rep = s.step(dt_s=1e-4, mu_pa=MU, lambda_pa=LAM, primary_region_id=1, secondary_region_id=2)
        _compare_oracle(s, o, rep, ref)
        gf = s.grid_force_n.to_numpy()
        assert _max_rel(gf, ref.grid_force) <= 1e-5


def test_invalidate_grid_clears_arrays_written_between_steps():
    s = _state((48, 48, 48), (10, 10, 10), (0.3,) * 3, (0.5,) * 3, "binned")
    a = _state((48, 48, 48), (10, 10, 10), (0.3,) * 3, (0.5,) * 3, "atomic")
    for st in (s, a):
        st.set_uniform_velocity((0.5, 0.0, 0.0))
        st.step(dt_s=1e-4, mu_pa=MU, lambda_pa=LAM, primary_region_id=1, secondary_region_id=2)
    s.grid_mass_kg.tensor.fill_(3.0)
    s.grid_velocity_mps.tensor.fill_(-1.0)
    s.invalidate_grid()
    for st in (s, a):
        st.step(dt_s=1e-4, mu_pa=MU, lambda_pa=LAM, primary_region_id=1, secondary_region_id=2)
    gb, ga = _grid(s), _grid(a)
    assert int(np.count_nonzero(gb[0][ga[0] == 0.0])) == 0
    assert _max_rel(gb[0], ga[0]) <= 1e-5 and _max_rel(gb[1], ga[1]) <= 1e-4


@pytest.mark.parametrize("capacity", [None, (1 << 19) + 1])  # blocks of 4^3 nodes, of 8^3 nodes
@pytest.mark.parametrize("nodes", [(33, 30, 21), (8, 7, 6)])
def test_both_block_edges_match_oracle(nodes, capacity):
    """1100 particles in one cell (more than either kernel orders at once), particles in every other part of a
    grid that neither block edge divides, fixed and out-of-bounds ones among them.  The tolerances are
    _compare_oracle's, but the mass is a float32 sum of 1100 terms at one node: its error is up to
    1100 * 2^-24 = 6.6e-5 of the largest node's mass, and a velocity p / m takes both sums' errors."""
    rng = np.random.default_rng(11)
    dx = 1.0 / np.asarray(nodes)
    pile = (np.asarray(nodes) // 2 + 0.5 + rng.uniform(0.02, 0.98, size=(1100, 3))) * dx
    spread = (0.6 + rng.uniform(0.0, 1.0, size=(700, 3)) * (np.asarray(nodes) - 2.2)) * dx
    outside = rng.uniform(1.1, 1.3, size=(70, 3))
    pts = np.concatenate([spread, outside, pile]).astype(np.float32)
    n = len(pts)
    s = _state(nodes, (1, 1, n), (0.4,) * 3, (0.6,) * 3, "binned", capacity=capacity)
    s.x.tensor[:n] = torch.from_numpy(pts).cuda()
    s.rest_x.tensor[:n] = s.x.tensor[:n]
    s.v.tensor[:n] = torch.from_numpy(rng.normal(0.0, 0.05, size=(n, 3)).astype(np.float32)).cuda()
    s.F.tensor[:n] = torch.from_numpy((np.eye(3) + rng.normal(0.0, 0.02, size=(n, 3, 3))).astype(np.float32)).cuda()
    s.external_force_n.tensor[:900] = torch.from_numpy(rng.normal(0, 1e-4, size=(900, 3)).astype(np.float32)).cuda()
    s.fixed_particle.tensor[5:n:9] = 1
    s.invalidate_grid()
    for _ in range(2):
        g = lambda f: f.to_numpy()[:n].astype(np.float64)  # noqa: E731
        o = M.MpmState(x=g(s.x), v=g(s.v), C=g(s.C), F=g(s.F), mass=g(s.mass_kg), volume=g(s.volume_m3),
                       rest_x=g(s.rest_x), fixed=s.fixed_particle.to_numpy()[:n].copy(), region=np.zeros(n, np.int32),
                       f_ext=g(s.external_force_n), normal=np.zeros((n, 3)), rest_normal=np.zeros((n, 3)),
                       area=np.zeros(n), rest_area=np.zeros(n))
        ref = M.step(o, bounds_min=(0.0,) * 3, bounds_max=(1.0,) * 3, grid_nodes=nodes, dt=2e-5, mu=MU, lam=LAM)
        rep = s.step(dt_s=2e-5, mu_pa=MU, lambda_pa=LAM, primary_region_id=1, secondary_region_id=2)
        assert rep.active_grid_nodes == ref.values["active_grid_nodes"]
        assert rep.grid_out_of_bounds_particle_count == ref.values["oob_count"] == 70
        e = {"x": float(np.abs(s.x.to_numpy()[:n] - o.x).max()), "v": _max_rel(s.v.to_numpy()[:n], o.v),
             "F": float(np.abs(s.F.to_numpy()[:n] - o.F).max()),
             "mass": _max_rel(s.grid_mass_kg.to_numpy(), ref.grid_mass),
             "force": _max_rel(s.grid_force_n.to_numpy(), ref.grid_force)}
        _say(f"  {nodes}, capacity {capacity}: " + ", ".join(f"{k} {v:.2e}" for k, v in e.items()))
        assert e["x"] <= 1e-6 and e["v"] <= 2e-4 and e["F"] <= 1e-5 and e["mass"] <= 7e-5 and e["force"] <= 7e-5
        assert int(np.count_nonzero(s.grid_mass_kg.to_numpy()[ref.grid_mass == 0.0])) == 0
