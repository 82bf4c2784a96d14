"""The one-tracer explicit kernel at the edges of its 64 x 8 tiles and the
column walk's two forms (GPU), equal to the oracle on every cell: extents
around a tile, one level, every branch of the face, fields with exact zeros
and with values far below 1; few columns (four lanes each) and many, of depths
around a group of four levels."""
import numpy as np
import pytest

from mohid_amd import constants as C
from mohid_amd import fixtures as fx
from oracle import oracle as ora

from .cases import GRID

pytestmark = pytest.mark.gpu


def _check(case, props, optimize):
    from mohid_amd.advection_diffusion import AdvectionDiffusion
    case.params["Optimize"] = optimize
    inst = ora.Instance(case, nthreads=1)
    gpu = AdvectionDiffusion(case.size, case.worksize, case.geom)
    got = [np.array(p, order="F", copy=True) for p in props]
    ref = [np.array(p, order="F", copy=True) for p in props]
    for s in range(2):
        for t in range(len(props)):
            assert inst.step(ref[t], first_property=t == 0,
                             now=(s + 1) * case.params["DTProp"]) == 0
            gpu(got[t], case.hydro, case.params, first_property=t == 0)
            assert np.array_equal(got[t], ref[t]), (s, t)
    gpu.kill()
    inst.close()


@pytest.mark.parametrize("optimize", (False, True))
@pytest.mark.parametrize("ni,nj,nk,kfloor,land", [
    (3, 3, 1, (1, 1), 0.0), (63, 7, 3, (1, 3), 0.2), (64, 8, 2, (1, 1), 0.0),
    (65, 9, 4, (2, 4), 0.4), (129, 17, 5, (1, 5), 0.3), (2, 40, 6, (1, 6), 0.1),
    (2, 70000, 2, (1, 2), 0.0), (70000, 2, 2, (1, 2), 0.0)])
def test_extents(ni, nj, nk, kfloor, land, optimize):
    case = fx.make_case(fx.config("c3", ni=ni, nj=nj, nk=nk, kfloor=kfloor, land_frac=land,
                                  tracers=("temperature", "lognormal"), **GRID))
    _check(case, case.tracers, optimize)


@pytest.mark.parametrize("method,limiter,up2", [
    (C.UPWIND_ORDER1, C.SUPERBEE, False), (C.P2_TVD, C.MINMOD, True),
    (C.P2_TVD, C.VANLEER, True), (C.P2_TVD, C.MUSCL, True), (C.P2_TVD, C.SUPERBEE, True),
    (C.P2_TVD, C.PDM, True), (C.CENTRAL_DIF, C.SUPERBEE, False)])
def test_faces(method, limiter, up2):
    case = fx.make_case(fx.config("c3", ni=70, nj=19, nk=5, kfloor=(1, 5), land_frac=0.3,
                                  tracers=("lognormal",), **GRID))
    case.params.update(AdvMethodH=method, TVDLimitationH=limiter, Upwind2H=up2)
    _check(case, case.tracers, False)


@pytest.mark.parametrize("ni,closed", [(2, ()), (3, (3,))])
def test_limiter_that_no_face_uses(ni, closed):
    """A limiter id that does not exist matters only where a face takes its value:
    not beside a closed cell with Upwind2H, nor at a face with a closed cell."""
    from mohid_amd import _lib as L
    from mohid_amd.advection_diffusion import AdvectionDiffusion
    case = fx.make_case(fx.config("c2", ni=ni, nj=2, nk=4, depth=(8.0, 20.0), **GRID))
    for i in closed:
        case.hydro["OpenPoints3D"][i] = 0
    case.params.update(TVDLimitationH=99, Upwind2H=True)
    _check(case, case.tracers, False)
    # where one does, the call says so
    case.params["Upwind2H"] = False
    gpu = AdvectionDiffusion(case.size, case.worksize, case.geom)
    with pytest.raises(L.MgpuError) as e:
        gpu(np.array(case.tracers[0], order="F", copy=True), case.hydro, case.params)
    assert e.value.code == L.MGPU_ERR_OPTION
    gpu.kill()


@pytest.mark.parametrize("optimize", (False, True))
def test_zero_and_small_values(optimize):
    """Exact zeros beside a patch, and the patch at 1e-200: every quotient is
    zero, or too small for the shared-reciprocal form."""
    case = fx.make_case(fx.config("c3", ni=70, nj=19, nk=5, kfloor=(1, 5), land_frac=0.3,
                                  tracers=("lognormal", "lognormal"), **GRID))
    wet = case.hydro["WaterPoints3D"] == 1
    props = []
    for scale in (1.0, 1e-200):
        p = np.array(case.tracers[0], order="F", copy=True)
        far = np.zeros_like(wet)
        far[30:] = True
        p[wet & far] = 0.0
        p[wet & ~far] *= scale
        props.append(p)
    _check(case, props, optimize)


@pytest.mark.parametrize("optimize", (False, True))
@pytest.mark.parametrize("ni,nj,nk,kfloor", [
    (5, 3, 2, (1, 2)), (9, 7, 3, (3, 3)), (17, 5, 4, (1, 4)), (16, 4, 5, (1, 5)),
    (11, 6, 37, (1, 37)), (4, 4, 259, (1, 259)), (230, 230, 4, (1, 4)),
    (330, 310, 3, (1, 3))])
def test_columns(ni, nj, nk, kfloor, optimize):
    """Depths around groups of four levels and past what LDS holds (259), and
    column counts either side of the change of walk."""
    case = fx.make_case(fx.config("c3", ni=ni, nj=nj, nk=nk, kfloor=kfloor, land_frac=0.0,
                                  tracers=("temperature", "lognormal"), **GRID))
    _check(case, case.tracers, optimize)


@pytest.mark.parametrize("impV,difV", [(C.EXPLICIT_SCHEME, 1.0), (C.EXPLICIT_SCHEME, 0.5),
                                       (C.IMPLICIT_SCHEME, C.EXPLICIT_SCHEME)])
@pytest.mark.parametrize("optimize", (False, True))
def test_columns_vertical_schemes(impV, difV, optimize):
    case = fx.make_case(fx.config("c3", ni=21, nj=13, nk=11, kfloor=(1, 11), land_frac=0.2,
                                  tracers=("temperature", "lognormal"), **GRID))
    case.params.update(ImpExp_AdvV=impV, ImpExp_DifV=difV)
    _check(case, case.tracers, optimize)


@pytest.mark.parametrize("tracers", (2, 4, 8))
def test_batched_zero_and_small_values(tracers):
    """Launches of several tracers: a patch in exact zeros, at 1 and at 1e-200,
    and the values beside it, in one launch."""
    from mohid_amd.advection_diffusion import Transport
    case = fx.make_case(fx.config("c3", ni=70, nj=19, nk=5, kfloor=(1, 5), land_frac=0.3,
                                  tracers=("lognormal",) * tracers, **GRID))
    wet = case.hydro["WaterPoints3D"] == 1
    props = []
    for t in range(tracers):
        p = np.array(case.tracers[t], order="F", copy=True)
        far = np.zeros_like(wet)
        far[30:] = True
        if t % 2 == 0:
            p[wet & far] = 0.0
        if t % 4 == 0:
            p[wet & ~far] *= 1e-200
        props.append(p)
    tr = Transport(case.size, case.worksize, case.geom, tracers)
    tr.set_hydro(case.hydro, case.params)
    for t, p in enumerate(props):
        tr.set_tracer(t, p)
    tr.run(3)
    ref = ora.run_case(case, 3, nthreads=1, tracers=props)
    solved = np.zeros(props[0].shape, dtype=bool)
    solved[:, :, 1:] = (case.hydro["WaterPoints3D"][:, :, case.worksize[5]] == 1)[:, :, None]
    for t in range(tracers):
        assert np.array_equal(tr.get_tracer(t)[solved], ref[t][solved]), t
    tr.close()


@pytest.mark.parametrize("tracers,order", [(3, 0), (3, 1), (5, 0), (5, 1)])
def test_batched_columns(tracers, order):
    """Interleaved tracers, columns in memory order and by first row."""
    from mohid_amd.advection_diffusion import Transport
    names = ("temperature", "salinity", "lognormal", "lognormal", "lognormal")[:tracers]
    case = fx.make_case(fx.config("c3", ni=37, nj=23, nk=13, kfloor=(2, 13), land_frac=0.3,
                                  tracers=names, **GRID))
    tr = Transport(case.size, case.worksize, case.geom, tracers)
    tr.set_column_order(order)
    tr.set_hydro(case.hydro, case.params)
    for t, p in enumerate(case.tracers):
        tr.set_tracer(t, p)
    tr.run(2)
    ref = ora.run_case(case, 2, nthreads=1)
    solved = np.zeros(case.tracers[0].shape, dtype=bool)
    solved[:, :, 1:] = (case.hydro["WaterPoints3D"][:, :, case.worksize[5]] == 1)[:, :, None]
    for t in range(tracers):
        assert np.array_equal(tr.get_tracer(t)[solved], ref[t][solved]), t
    tr.close()
