"""Both forms of the column walk (GPU), equal to the oracle.

Few columns take the quad walk by themselves, and every small case here has few:
the tests of the other files that reach the column rows (boundary rows, nudging,
discharges, small depths, vertical schemes, implicit restarts, launch shapes) run
again with the lane walk set on every handle.  Batched runs of several steps
over ragged floors compare every cell of Size, the inert rows below the floor
included, in both forms and orders.
"""
import itertools

import numpy as np
import pytest

from mohid_amd import _lib as L
from mohid_amd import advection_diffusion as AD
from mohid_amd import fixtures as fx
from oracle import oracle as ora

from . import (test_gpu_boundaries, test_gpu_fluxes, test_gpu_implicit, test_gpu_nudging,
               test_gpu_options, test_gpu_parity, test_gpu_state, test_gpu_tiles)
from .cases import GRID

pytestmark = pytest.mark.gpu

TESTS = [
    test_gpu_boundaries.test_open_boundary_drop_in, test_gpu_boundaries.test_orlanski_drop_in,
    test_gpu_boundaries.test_null_gradient_without_open_boundary,
    test_gpu_fluxes.test_cell_fluxes_drop_in,
    test_gpu_implicit.test_implicit_drop_in_matches_oracle,
    test_gpu_implicit.test_implicit_mixed_directions_within_a_step,
    test_gpu_implicit.test_implicit_one_layer,
    test_gpu_implicit.test_implicit_batched_matches_oracle,
    test_gpu_implicit.test_implicit_batched_launch_shapes,
    test_gpu_implicit.test_implicit_fast_mode,
    test_gpu_implicit.test_batched_masks_change_between_steps,
    test_gpu_nudging.test_nudging_drop_in, test_gpu_nudging.test_nudging_with_open_boundary,
    test_gpu_nudging.test_nudging_one_layer,
    test_gpu_options.test_nodifflux_drop_in, test_gpu_options.test_small_depths_drop_in,
    test_gpu_options.test_options_batched, test_gpu_options.test_noadvflux_drop_in,
    test_gpu_options.test_discharges_drop_in,
    test_gpu_options.test_discharges_with_open_boundary_and_fluxes,
    test_gpu_parity.test_advection_diffusion_matches_oracle,
    test_gpu_parity.test_advection_diffusion_options,
    test_gpu_parity.test_batched_transport_chunks_match_oracle,
    test_gpu_parity.test_batched_transport_matches_oracle,
    test_gpu_parity.test_fast_transport_matches_oracle,
    test_gpu_parity.test_batched_graph_replays_agree,
    test_gpu_parity.test_every_launch_shape_gives_identical_results,
    test_gpu_parity.test_edge_shapes_match_oracle,
    test_gpu_parity.test_moving_surface_matches_oracle,
    test_gpu_state.test_tracers_set_between_runs,
    test_gpu_tiles.test_columns, test_gpu_tiles.test_columns_vertical_schemes,
    test_gpu_tiles.test_batched_columns,
]


def _runs():
    """Every test of TESTS with each of its own parameters."""
    for fn in TESTS:
        sets = [[dict()]]
        for m in getattr(fn, "pytestmark", ()):
            if m.name != "parametrize":
                continue
            names = [n.strip() for n in m.args[0].split(",")]
            sets.append([dict(zip(names, v if len(names) > 1 else (v,))) for v in m.args[1]])
        for n, combo in enumerate(itertools.product(*sets)):
            kw = {k: v for d in combo for k, v in d.items()}
            yield pytest.param(fn, kw, id=f"{fn.__name__}-{n}")


@pytest.mark.parametrize("fn,kw", _runs())
def test_lane_walk(fn, kw, monkeypatch):
    for cls in (AD.AdvectionDiffusion, AD.Transport):
        def init(self, *a, _of=cls.__init__, **k):
            _of(self, *a, **k)
            self.set_column_walk(L.MGPU_WALK_LANES)
        monkeypatch.setattr(cls, "__init__", init)
    fn(**kw)


@pytest.mark.parametrize("walk", (L.MGPU_WALK_LANES, L.MGPU_WALK_QUADS))
@pytest.mark.parametrize("order", (L.MGPU_COLUMNS_MEMORY, L.MGPU_COLUMNS_BY_DEPTH))
@pytest.mark.parametrize("tracers,optimize", [(1, True), (2, False), (3, True), (8, True)])
def test_inert_rows_over_several_steps(tracers, optimize, order, walk):
    """The inert rows' null_real is stored in a run's first two steps only: runs
    of one to five steps, captured and not, after tracers that had other values
    there, in each of them."""
    names = ("temperature", "salinity") + ("lognormal",) * 6
    case = fx.make_case(fx.config("c3", ni=37, nj=23, nk=21, kfloor=(1, 21), land_frac=0.3,
                                  tracers=names[:tracers], **GRID))
    case.params["Optimize"] = optimize
    tr = AD.Transport(case.size, case.worksize, case.geom, tracers)
    tr.set_column_order(order)
    tr.set_column_walk(walk)
    tr.set_hydro(case.hydro, case.params)
    rng = np.random.default_rng(7)
    props = [np.asfortranarray(p + rng.uniform(0, 1, p.shape)) for p in case.tracers]
    refs = {n: ora.run_case(case, n, nthreads=1, tracers=props) for n in (1, 2, 3, 5)}
    for steps, graph, lanes in ((3, False, 0), (5, True, 1), (1, False, 2), (2, True, 0),
                                (5, False, 4), (3, True, 8)):
        tr.set_lanes(0, 0, lanes)
        for t, p in enumerate(props):
            tr.set_tracer(t, p)
        tr.run(steps, use_graph=graph)
        for t in range(tracers):
            assert np.array_equal(tr.get_tracer(t), refs[steps][t]), (steps, graph, lanes, t)
    tr.close()


def test_walk_is_checked():
    case = fx.make_case(fx.config("c1", ni=4, nj=3, nk=2))
    for h in (AD.AdvectionDiffusion(case.size, case.worksize, case.geom),
              AD.Transport(case.size, case.worksize, case.geom, 1)):
        for bad in (-1, 3):
            with pytest.raises(L.MgpuError) as e:
                h.set_column_walk(bad)
            assert e.value.code == L.MGPU_ERR_BADARG
        h.set_column_walk(L.MGPU_WALK_QUADS)
        h.set_column_walk(L.MGPU_WALK_AUTO)
