"""GPU parity of hfsi_ib_node_search (HIBM immersed-boundary node search) against
oracle/ib_search.py, and the reference's node-search tests (tests/test_hibm.py:903-1318)
through easyfsi_amd.hibm.HibmMpmIbNodeSearch.

Tolerance: bit for bit (np.array_equal on every node field, equal report counts): the kernel
and the oracle run the same float32 operations in the same order, and the tile culling keeps
every triangle within the search radius of a node.
"""

import sys

import numpy as np
import pytest
import torch

from oracle import ib_search as S
from tests.test_oracle_ib_search import SIX, SIX_N, icosphere

pytestmark = pytest.mark.gpu

FIELDS = (("kind", "node_kind_code"), ("nearest_marker", "nearest_marker"),
          ("signed_distance", "node_signed_distance_m"), ("boundary_point", "node_boundary_point_m"),
          ("interior_point", "node_interior_fluid_point_m"), ("projection_indices", "node_projection_marker_indices"),
          ("projection_weights", "node_projection_marker_weights"))


def _say(msg):
    print(msg, flush=True)
    sys.stdout.flush()


def _markers(xm, nm, tris=None):
    from easyfsi_amd.hibm import HibmMpmSurfaceMarkers

    m = HibmMpmSurfaceMarkers(marker_capacity=len(xm), projection_triangle_capacity=max(1, len(tris or ())))
    m.load_markers(positions_m=[tuple(map(float, p)) for p in xm], velocities_mps=[(0.0, 0.0, 0.0)] * len(xm),
                   normals=[tuple(map(float, n)) for n in nm], areas_m2=[1.0] * len(xm), region_ids=[7] * len(xm))
    if tris:
        m.set_projection_triangles(tris)
    return m


def _search(shape, bmin=(0.0, 0.0, 0.0), bmax=(1.0, 1.0, 1.0), capacity=1):
    from easyfsi_amd.hibm import HibmMpmIbNodeSearch

    return HibmMpmIbNodeSearch(grid_nodes=shape, bounds_min_m=bmin, bounds_max_m=bmax, marker_capacity=capacity)


def _compare(search, want, rep_want, rep):
    n = int(np.prod(search.grid_nodes))
    for key, attr in FIELDS:
        got = getattr(search, attr).to_numpy().reshape(n, -1).squeeze()
        exp = want[key].reshape(n, -1).squeeze()
        assert np.array_equal(got, exp), f"{key}: {np.count_nonzero(got != exp)} differing entries"
    assert rep.__dict__ == rep_want


def _positions(search):
    return S.node_positions(search.grid_nodes, bounds_min=search.bounds_min_m, spacing=search.spacing_m)


@pytest.mark.parametrize("far", [False, True])
@pytest.mark.parametrize("use_triangles", [False, True])
def test_sphere_surface_matches_oracle_bit_for_bit(far, use_triangles):
    _say(f"ib search: icosphere level 2 on 20x22x24, triangles={use_triangles} far={far}")
    xm, nm, tris = icosphere(2, (0.47, 0.52, 0.5), 0.27)
    shape = (20, 22, 24)
    search = _search(shape, bmin=(-0.05, 0.0, 0.02), bmax=(1.05, 1.0, 0.98), capacity=len(xm))
    tri_list = [tuple(int(v) for v in t) for t in tris] if use_triangles else None
    markers = _markers(xm, nm, tri_list)
    x32 = markers.x_gamma_m.to_numpy()[: len(xm)]
    n32 = markers.n_gamma.to_numpy()[: len(xm)]
    rep = search.search_and_classify(markers, search_radius_m=0.09, interior_probe_distance_m=0.04,
                                     classify_far_internal_nodes=far)
    want, rep_want = S.search_and_classify(_positions(search), x32, n32, tris if use_triangles else None,
                                           search_radius=0.09, interior_probe_distance=0.04,
                                           sign_tolerance=search._default_sign_tolerance_m(),
                                           classify_far_internal_nodes=far)
    _compare(search, want, rep_want, rep)
    near_internal = rep.near_boundary_node_count - rep.external_ib_node_count
    assert rep.near_boundary_node_count > 100 and (rep.internal_node_count > near_internal if far
                                                   else rep.internal_node_count == near_internal)


def test_graded_cell_centres_and_duplicate_triangles_match_oracle():
    """Cell-centre nodes of a graded grid; a duplicated triangle (equal distances, the first index
    must win) and a degenerate one (skipped)."""
    from easyfsi_amd.simulation_core.grid import CartesianGrid, FluidDomainSpec
    from easyfsi_amd.simulation_core.fluid import CartesianFluidSolver

    rng = np.random.default_rng(4)
    shape = (18, 16, 20)
    widths = [rng.uniform(0.6, 1.4, size=n) / n for n in shape]
    g = CartesianGrid(bounds_min_m=(0.0, 0.0, 0.0), cell_widths_x_m=tuple(widths[0]),
                      cell_widths_y_m=tuple(widths[1]), cell_widths_z_m=tuple(widths[2]))
    fluid = CartesianFluidSolver(FluidDomainSpec(bounds_min_m=g.bounds_min_m, bounds_max_m=g.bounds_max_m,
                                                 grid_nodes=None, density_kgm3=1000.0, viscosity_pa_s=1e-3,
                                                 dt_s=1e-3, cartesian_grid=g))
    _say("ib search: graded cell centres 18x16x20, duplicated + degenerate triangles, far classification")
    xm, nm, tris = icosphere(1, (0.5, 0.45, 0.55), 0.3)
    tris = [tuple(int(v) for v in t) for t in tris]
    tris = tris[:7] + [tris[3]] + [(0, 0, 1)] + tris[7:]
    search = _search(fluid.grid.grid_nodes, fluid.grid.bounds_min_m, fluid.grid.bounds_max_m, capacity=len(xm))
    markers = _markers(xm, nm, tris)
    rep = search.search_and_classify_grid_fields(markers, cell_center_x_m=fluid.cell_center_x_m,
                                                 cell_center_y_m=fluid.cell_center_y_m,
                                                 cell_center_z_m=fluid.cell_center_z_m, search_radius_m=0.1,
                                                 interior_probe_distance_m=0.05, classify_far_internal_nodes=True)
    centres = [fluid.cell_center_x_m.to_numpy(), fluid.cell_center_y_m.to_numpy(), fluid.cell_center_z_m.to_numpy()]
    want, rep_want = S.search_and_classify(S.node_positions(shape, centers=centres),
                                           markers.x_gamma_m.to_numpy(), markers.n_gamma.to_numpy(), tris,
                                           search_radius=0.1, interior_probe_distance=0.05,
                                           sign_tolerance=search._default_sign_tolerance_m(),
                                           classify_far_internal_nodes=True)
    _compare(search, want, rep_want, rep)


def test_sampled_nodes_of_a_fine_surface_at_128():
    """128^3 nodes against a 5120-triangle sphere with far classification; 20 000 sampled nodes
    checked against the oracle, all counts against the analytic sphere."""
    _say("ib search: 128^3 nodes, icosphere level 4 (5120 triangles), far classification")
    xm, nm, tris = icosphere(4, (0.5, 0.5, 0.5), 0.3)
    shape = (128, 128, 128)
    search = _search(shape, capacity=len(xm))
    tri_list = [tuple(int(v) for v in t) for t in tris]
    markers = _markers(xm, nm, tri_list)
    torch.cuda.synchronize()
    start, end = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
    rep = search.search_and_classify(markers, search_radius_m=2.0 / 128, interior_probe_distance_m=1.0 / 128,
                                     classify_far_internal_nodes=True)
    start.record()
    rep = search.search_and_classify(markers, search_radius_m=2.0 / 128, interior_probe_distance_m=1.0 / 128,
                                     classify_far_internal_nodes=True)
    end.record()
    torch.cuda.synchronize()
    _say(f"  {rep}, {start.elapsed_time(end):.3f} ms (the full loop would be {128 ** 3 * 5120:.3g} node-triangle tests)")
    pos = _positions(search)
    rng = np.random.default_rng(0)
    pick = rng.choice(pos.shape[0], size=20000, replace=False)
    want, _ = S.search_and_classify(pos[pick], markers.x_gamma_m.to_numpy(), markers.n_gamma.to_numpy(), tris,
                                    search_radius=2.0 / 128, interior_probe_distance=1.0 / 128,
                                    sign_tolerance=search._default_sign_tolerance_m(),
                                    classify_far_internal_nodes=True)
    n = pos.shape[0]
    for key, attr in FIELDS:
        got = getattr(search, attr).to_numpy().reshape(n, -1)[pick].squeeze()
        assert np.array_equal(got, want[key].reshape(len(pick), -1).squeeze()), key
    r = np.linalg.norm(pos.astype(np.float64) - 0.5, axis=1)
    kind = search.node_kind_code.to_numpy().ravel()
    assert np.all(kind[r < 0.3 * 0.995 - 2.0 / 128] == 2)
    assert np.all(kind[r > 0.3 + 2.0 / 128] == 0)


# ---- the reference's tests (tests/test_hibm.py) ----------------------------------------------

def test_plane_search_classifies_external_and_internal_nodes():  # test_hibm.py:903-941
    markers = _markers([(0.5, 0.5, 0.5)], [(0.0, 0.0, 1.0)])
    search = _search((1, 1, 4))
    report = search.search_and_classify(markers, search_radius_m=0.26, interior_probe_distance_m=0.125)
    assert (report.near_boundary_node_count, report.external_ib_node_count, report.internal_node_count,
            report.invalid_projection_count) == (2, 1, 1, 0)
    assert search.node_kind((0, 0, 2)) == "external_ib" and search.node_kind((0, 0, 1)) == "internal"
    assert search.nearest_marker_index((0, 0, 2)) == 0 and search.nearest_marker_index((0, 0, 1)) == 0
    assert search.boundary_point_m((0, 0, 2)) == (0.5, 0.5, 0.5)
    assert search.interior_fluid_point_m((0, 0, 2)) == (0.5, 0.5, 0.75)
    assert search.signed_distance_m((0, 0, 2)) > 0.0 > search.signed_distance_m((0, 0, 1))


def test_triangle_projection_finds_closest_surface_point_between_markers():  # :943-988
    markers = _markers([(0.25, 0.25, 0.5), (0.75, 0.25, 0.5), (0.25, 0.75, 0.5)], [(0.0, 0.0, 1.0)] * 3, [(0, 1, 2)])
    search = _search((8, 8, 8), capacity=3)
    report = search.search_and_classify(markers, search_radius_m=0.08, interior_probe_distance_m=0.05)
    assert report.near_boundary_node_count >= 1 and report.external_ib_node_count >= 1
    assert search.node_kind((2, 2, 4)) == "external_ib"
    np.testing.assert_allclose(search.boundary_point_m((2, 2, 4)), (0.3125, 0.3125, 0.5), atol=1.0e-6)
    assert search.signed_distance_m((2, 2, 4)) == pytest.approx(0.0625)
    np.testing.assert_allclose(search.interior_fluid_point_m((2, 2, 4)), (0.3125, 0.3125, 0.6125), atol=1.0e-6)


def test_closed_surface_search_classifies_deep_internal_nodes():  # :990-1031
    markers = _markers(SIX, SIX_N)
    search = _search((1, 1, 1), capacity=6)
    report = search.search_and_classify(markers, search_radius_m=0.1, interior_probe_distance_m=0.125,
                                        classify_far_internal_nodes=True)
    assert (report.near_boundary_node_count, report.external_ib_node_count, report.internal_node_count) == (0, 0, 1)
    assert search.node_kind((0, 0, 0)) == "internal" and search.nearest_marker_index((0, 0, 0)) >= 0


def test_closed_surface_grid_field_search_classifies_deep_internal_nodes():  # :1033-1091 (search part)
    from easyfsi_amd.simulation_core.fluid import CartesianFluidSolver
    from easyfsi_amd.simulation_core.grid import FluidDomainSpec

    markers = _markers(SIX, SIX_N)
    fluid = CartesianFluidSolver(FluidDomainSpec.unit_box(grid_nodes=(4, 4, 4), dt_s=1.0e-3))
    search = _search(fluid.grid.grid_nodes, fluid.grid.bounds_min_m, fluid.grid.bounds_max_m, capacity=6)
    report = search.search_and_classify_grid_fields(
        markers, cell_center_x_m=fluid.cell_center_x_m, cell_center_y_m=fluid.cell_center_y_m,
        cell_center_z_m=fluid.cell_center_z_m, search_radius_m=0.08, interior_probe_distance_m=0.125,
        classify_far_internal_nodes=True)
    assert report.near_boundary_node_count == 0 and report.internal_node_count == 8
    assert search.node_kind((1, 1, 1)) == "internal" and search.node_kind((2, 2, 2)) == "internal"
    assert search.node_kind((0, 0, 0)) == "none"


def test_default_sign_tolerance_flags_f32_scale_ambiguous_nodes():  # :1093-1116
    markers = _markers([(0.5, 0.5, 0.5 - 5.0e-8)], [(0.0, 0.0, 1.0)])
    search = _search((1, 1, 1))
    report = search.search_and_classify(markers, search_radius_m=0.01, interior_probe_distance_m=0.125)
    assert report.near_boundary_node_count == 1 and report.invalid_projection_count == 1
    assert search.node_kind((0, 0, 0)) == "internal" and search.signed_distance_m((0, 0, 0)) > 0.0


def test_search_uses_nonuniform_fluid_cell_center_fields():  # :1118-1175
    from easyfsi_amd.simulation_core.fluid import CartesianFluidSolver
    from easyfsi_amd.simulation_core.grid import CartesianGrid, FluidDomainSpec

    grid = CartesianGrid(bounds_min_m=(0.0, 0.0, 0.0), cell_widths_x_m=(0.25,) * 4, cell_widths_y_m=(0.25,) * 4,
                         cell_widths_z_m=(0.1, 0.1, 0.2, 0.6))
    fluid = CartesianFluidSolver(FluidDomainSpec(bounds_min_m=(0.0, 0.0, 0.0), bounds_max_m=(1.0, 1.0, 1.0),
                                                 grid_nodes=(4, 4, 4), density_kgm3=1000.0, viscosity_pa_s=1.0e-3,
                                                 dt_s=1.0e-3, cartesian_grid=grid))
    markers = _markers([(0.625, 0.625, 0.28)], [(0.0, 0.0, 1.0)])
    search = _search(fluid.grid.grid_nodes, fluid.grid.bounds_min_m, fluid.grid.bounds_max_m)
    report = search.search_and_classify_grid_fields(
        markers, cell_center_x_m=fluid.cell_center_x_m, cell_center_y_m=fluid.cell_center_y_m,
        cell_center_z_m=fluid.cell_center_z_m, search_radius_m=0.04, interior_probe_distance_m=0.05)
    assert (report.near_boundary_node_count, report.external_ib_node_count, report.internal_node_count) == (1, 1, 0)
    assert search.node_kind((2, 2, 2)) == "external_ib" and search.node_kind((2, 2, 1)) == "none"
    assert search.signed_distance_m((2, 2, 2)) == pytest.approx(0.02, abs=1.0e-6)
    bp = search.boundary_point_m((2, 2, 2))
    assert bp[0] == pytest.approx(0.625, abs=1e-6) and bp[1] == pytest.approx(0.625, abs=1e-6)
    assert bp[2] == pytest.approx(0.28, abs=1e-6)
    assert search.interior_fluid_point_m((2, 2, 2))[2] == pytest.approx(0.35, abs=1.0e-6)


def test_search_treats_node_as_external_if_any_local_normal_is_positive():  # :1177-1203
    markers = _markers([(0.5, 0.5, 0.55), (0.5, 0.5, 0.45)], [(0.0, 0.0, -1.0), (0.0, 0.0, 1.0)])
    search = _search((1, 1, 1), capacity=2)
    report = search.search_and_classify(markers, search_radius_m=0.08, interior_probe_distance_m=0.05)
    assert (report.near_boundary_node_count, report.external_ib_node_count, report.internal_node_count) == (1, 1, 0)
    assert search.node_kind((0, 0, 0)) == "external_ib"


def test_external_search_stores_external_projection_candidate():  # :1205-1240
    markers = _markers([(0.5, 0.5, 0.49), (0.5, 0.5, 0.46)], [(0.0, 0.0, -1.0), (0.0, 0.0, 1.0)])
    search = _search((1, 1, 1), capacity=2)
    report = search.search_and_classify(markers, search_radius_m=0.05, interior_probe_distance_m=0.05,
                                        sign_tolerance_m=1.0e-8)
    assert (report.near_boundary_node_count, report.external_ib_node_count, report.internal_node_count) == (1, 1, 0)
    assert search.node_kind((0, 0, 0)) == "external_ib" and search.nearest_marker_index((0, 0, 0)) == 1
    assert search.signed_distance_m((0, 0, 0)) > 0.0
    assert search.boundary_point_m((0, 0, 0))[2] == pytest.approx(0.46, abs=1.0e-6)
    assert search.interior_fluid_point_m((0, 0, 0))[2] > 0.5


def test_sphere_local_radial_marker_classifies_inside_and_outside_nodes():  # :1242-1270
    markers = _markers([(0.75, 0.5, 0.5)], [(1.0, 0.0, 0.0)])
    search = _search((4, 1, 1))
    report = search.search_and_classify(markers, search_radius_m=0.14, interior_probe_distance_m=0.125)
    assert (report.near_boundary_node_count, report.external_ib_node_count, report.internal_node_count) == (2, 1, 1)
    assert search.node_kind((3, 0, 0)) == "external_ib" and search.node_kind((2, 0, 0)) == "internal"
    assert search.signed_distance_m((3, 0, 0)) > 0.0 > search.signed_distance_m((2, 0, 0))


def test_tangent_projection_fallback_records_invalid_count():  # :1272-1300
    markers = _markers([(0.5, 0.5, 0.5)], [(0.0, 0.0, 1.0)])
    search = _search((1, 1, 1))
    report = search.search_and_classify(markers, search_radius_m=0.1, interior_probe_distance_m=0.125,
                                        sign_tolerance_m=1.0e-9)
    assert report.near_boundary_node_count == 1 and report.invalid_projection_count == 1
    assert search.nearest_marker_index((0, 0, 0)) == 0
    assert search.boundary_point_m((0, 0, 0)) == (0.5, 0.5, 0.5)
    assert search.interior_fluid_point_m((0, 0, 0)) == (0.5, 0.5, 0.625)


@pytest.mark.parametrize("sizes", [(0.6,), (0.05,), (0.3, 0.1), (0.001,)])
@pytest.mark.parametrize("sliver", [1.0, 40.0])
def test_far_bounds_skip_nothing_that_counts(sizes, sliver):
    """Far classification below open patches that face up, so that most nodes under them are internal and
    take the nearest of all triangles: large, small and tiny patches far from most nodes (where the
    closest-point formula loses digits and nothing may be skipped), two at different heights, slivers
    (one axis squeezed), every fifth triangle twice (equal distances: the lower index)."""
    rng = np.random.default_rng(int(1000 * sizes[0]) + int(sliver))
    xm, nm, tris = [], [], []
    m = 9
    for q, size in enumerate(sizes):
        u, v = np.meshgrid(np.linspace(-0.5, 0.5, m), np.linspace(-0.5, 0.5, m), indexing="ij")
        h = 0.05 * (u * u + v * v) + 0.002 * rng.normal(size=u.shape)
        x = np.stack([u.ravel() * size / sliver, v.ravel() * size, h.ravel() * size], -1)
        at = len(xm) * m * m
        xm.append((x + (0.3 + 0.3 * q, 0.47, 0.62 + 0.1 * q)).astype(np.float32))
        nm.append(np.tile(np.array([0, 0, 1], np.float32), (m * m, 1)))
        for i in range(m - 1):
            for j in range(m - 1):
                c = at + i * m + j
                tris += [(c, c + m, c + m + 1), (c, c + m + 1, c + 1)]
    xm, nm = np.concatenate(xm), np.concatenate(nm)
    tris = [t for k, t in enumerate(tris) for _ in range(2 if k % 5 == 0 else 1)]
    shape = (21, 18, 23)
    _say(f"ib search: open patches {sizes}, sliver {sliver}, {len(tris)} triangles")
    search = _search(shape, capacity=len(xm))
    markers = _markers(xm, nm, tris)
    rep = search.search_and_classify(markers, search_radius_m=0.03, interior_probe_distance_m=0.02,
                                     classify_far_internal_nodes=True)
    want, rep_want = S.search_and_classify(_positions(search), markers.x_gamma_m.to_numpy(),
                                           markers.n_gamma.to_numpy(), tris, search_radius=0.03,
                                           interior_probe_distance=0.02,
                                           sign_tolerance=search._default_sign_tolerance_m(),
                                           classify_far_internal_nodes=True)
    _compare(search, want, rep_want, rep)
    assert rep.internal_node_count > 50
