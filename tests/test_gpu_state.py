"""Tracers and fields into and out of a batched handle (GPU): tracers set again
between runs reach both state buffers, no step runs after refused masks, and
device arrays at any 8-byte (fields) or 4-byte (masks) alignment give the same
step, equal to the oracle."""
import numpy as np
import pytest

from mohid_amd import fixtures as fx
from oracle import oracle as ora

from .cases import GRID

pytestmark = pytest.mark.gpu


def _case(names):
    return fx.make_case(fx.config("c3", ni=45, nj=21, nk=7, kfloor=(2, 7), land_frac=0.4,
                                  tracers=names, **GRID))


@pytest.mark.parametrize("steps", (1, 2))
def test_tracers_set_between_runs(steps):
    """Every cell of Size, solved or not, after the tracers are set to other
    values (on land too) under the same hydrodynamics."""
    from mohid_amd.advection_diffusion import Transport
    names = ("temperature", "salinity", "lognormal")
    case = _case(names)
    tr = Transport(case.size, case.worksize, case.geom, len(names))
    tr.set_hydro(case.hydro, case.params)
    for t, p in enumerate(case.tracers):
        tr.set_tracer(t, p)
    tr.run(1)
    rng = np.random.default_rng(3)
    props = [np.asfortranarray(p + rng.uniform(0, 1, p.shape)) for p in case.tracers]
    for t, p in enumerate(props):
        tr.set_tracer(t, p)
    tr.run(steps)
    ref = ora.run_case(case, steps, nthreads=1, tracers=props)
    for t in range(len(names)):
        assert np.array_equal(tr.get_tracer(t), ref[t]), t
    tr.close()


@pytest.mark.parametrize("use_graph", (False, True))
def test_masks_refused_between_runs(use_graph):
    """No step runs after a hydrodynamic state whose masks were refused, not even
    one captured before it; the tracers set meanwhile are whole once the next
    state is accepted."""
    from mohid_amd import _lib as L
    from mohid_amd.advection_diffusion import Transport
    names = ("temperature", "salinity", "lognormal")
    case = _case(names)
    tr = Transport(case.size, case.worksize, case.geom, len(names))
    tr.set_hydro(case.hydro, case.params)
    for t, p in enumerate(case.tracers):
        tr.set_tracer(t, p)
    tr.run(1, use_graph=use_graph)
    rng = np.random.default_rng(5)
    props = [np.asfortranarray(p + rng.uniform(0, 1, p.shape)) for p in case.tracers]
    for t, p in enumerate(props):
        tr.set_tracer(t, p)
    # a W face missing above the floor of a column: not what KFloor says
    cfw = np.array(case.hydro["ComputeFacesW3D"], order="F", copy=True)
    i, j, k = np.argwhere(cfw[:, :, :case.worksize[5]] == 1)[0]   # below the surface one
    cfw[i, j, k] = 0
    with pytest.raises(L.MgpuError) as e:
        tr.set_hydro(dict(case.hydro, ComputeFacesW3D=cfw), case.params)
    assert e.value.code == L.MGPU_ERR_MASKS
    with pytest.raises(L.MgpuError) as e:
        tr.run(1, use_graph=use_graph)
    assert e.value.code == L.MGPU_ERR_STATE
    for t, p in enumerate(props):
        assert np.array_equal(tr.get_tracer(t), p), t
    tr.set_hydro(case.hydro, case.params)
    tr.run(2, use_graph=use_graph)
    ref = ora.run_case(case, 2, nthreads=1, tracers=props)
    for t in range(len(names)):
        assert np.array_equal(tr.get_tracer(t), ref[t]), t
    tr.close()


@pytest.mark.parametrize("shift", (0, 1))
def test_device_arrays_at_any_alignment(shift):
    import torch
    from mohid_amd.advection_diffusion import Transport
    names = ("temperature", "salinity")
    case = _case(names)

    def dev(a):
        a = np.asarray(a)
        flat = torch.from_numpy(np.ascontiguousarray(a.T).reshape(-1).copy())
        room = torch.zeros(flat.numel() + 1, dtype=flat.dtype, device="cuda")
        view = room[shift:shift + flat.numel()]
        view.copy_(flat)
        return view.view(a.T.shape)

    geom = {n: dev(v) for n, v in case.geom.items()}
    hydro = {n: dev(v) for n, v in case.hydro.items()}
    props = [dev(p) for p in case.tracers]
    tr = Transport(case.size, case.worksize, geom, len(names))
    tr.set_hydro(hydro, case.params)
    for t, p in enumerate(props):
        tr.set_tracer(t, p)
    tr.set_geometry(geom)
    tr.run(3)
    for t, p in enumerate(props):
        tr.get_tracer(t, out=p)
    torch.cuda.synchronize()
    ref = ora.run_case(case, 3, nthreads=1)
    for t in range(len(names)):
        assert np.array_equal(props[t].cpu().numpy().T, ref[t]), t
    tr.close()
