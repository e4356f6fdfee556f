"""GPU parity of the Joseph projector pair against the ref-compat oracle
(bar: <= 1e-5 relative L2 in FP32, projector-parallel-joseph.cl semantics)."""
import numpy as np
import pytest

import oracle as O
import uir
from phantoms import ellipse_phantom, shepp_logan

pytestmark = pytest.mark.gpu

TOL = 1e-5

SHAPES = [  # (image edge, detectors, angles, step)
    (367, 367, 180, np.float32(np.pi / 180)),     # config-1 shape on the reference D x D grid
    (256, 367, 180, np.float32(np.pi / 180)),     # config-1 native grid
    (1024, 1448, 720, np.float32(np.pi / 720)),   # config-2 / metric shape, native grid
    (1448, 1448, 720, np.float32(np.pi / 720)),   # config-2 reference grid
    (96, 96, 90, np.float32(0.034906585)),        # json-sample step (2 degrees)
    (64, 64, 120, np.float32(2 * np.pi / 120)),   # full circle: five direction runs
]


def _projector(n, d, a, step, forward, **extra):
    p = uir.Task("parallel-projector", step=float(step), is_forward=forward, angles_num=a,
                 image_size=n, detectors_num=d, **extra)
    return p


@pytest.mark.parametrize("n,d,a,step", SHAPES)
def test_fp_matches_oracle(res, n, d, a, step):
    print("case fp", n, d, a, flush=True)
    g = O.Geometry(n, d, a, step)
    x = ellipse_phantom(n, seed=n + a)
    ref = O.fp(g, x)
    p = _projector(n, d, a, step, True).setup(res)
    dx = uir.DeviceArray.from_numpy(x)
    assert p.requisition(dx) == (a, d)
    out = uir.DeviceArray((a, d))
    p.process(dx, out)
    got = out.numpy()
    err = O.rel_l2(got, ref)
    assert err <= TOL, (err, np.abs(got - ref).max())


@pytest.mark.parametrize("n,d,a,step", SHAPES)
def test_bp_matches_oracle(res, n, d, a, step):
    print("case bp", n, d, a, flush=True)
    g = O.Geometry(n, d, a, step)
    sino = O.fp(g, ellipse_phantom(n, seed=3 * n))
    ref = O.bp(g, sino)
    p = _projector(n, d, a, step, False).setup(res)
    ds = uir.DeviceArray.from_numpy(sino)
    assert p.requisition(ds) == (n, n)
    out = uir.DeviceArray((n, n))
    p.process(ds, out)
    got = out.numpy()
    err = O.rel_l2(got, ref)
    assert err <= TOL, (err, np.abs(got - ref).max())


@pytest.mark.parametrize("n,d,a,axis", [
    (1, 1, 1, -1.0), (3, 5, 2, -1.0), (64, 64, 9, -1.0),
    (71, 101, 12, -1.0), (130, 184, 10, 85.25),   # a last block of 7 and of 2 lines; inactive detectors
    (640, 906, 6, -1.0), (641, 907, 6, -1.0), (200, 283, 40, 260.5),
    (1024, 1449, 5, -1.0), (1025, 1450, 5, -1.0),  # both sides of the work table's line in the edge
    (9, 17, 5294, -1.0), (9, 17, 5295, -1.0),      # and in the rays: 89998 and 90015
    (71, 101, 900, 30.25), (63, 200, 460, -1.0),   # last chunks of 7 and 31 lines; inactive detectors
    (33, 91, 13000, -1.0),                         # items of 8 angles
])
def test_fp_bit_exact(res, n, d, a, axis):
    """The FP runs the reference's operations in its order
    (projector-parallel-joseph.cl:51-94): equal to the oracle bit for bit,
    adding to what the sinogram holds."""
    print("case fp bit-exact", n, d, a, axis, flush=True)
    step = np.float32(np.pi / a)
    g = O.Geometry(n, d, a, step, axis=axis)
    rng = np.random.default_rng(n + a)
    x = rng.standard_normal((n, n)).astype(np.float32)
    base = rng.standard_normal((a, d)).astype(np.float32)
    p = _projector(n, d, a, step, True, axis_position=axis).setup(res)
    dx, ds = uir.DeviceArray.from_numpy(x), uir.DeviceArray.from_numpy(base)
    assert p.requisition(dx) == (a, d)
    p["correction_scale"] = 0.75
    p.forward(dx, ds)
    assert np.array_equal(ds.numpy(), O.fp(g, x, sino=base, corr=0.75))


@pytest.mark.parametrize("n,d,a,axis", [
    (1, 1, 1, -1.0), (3, 5, 2, -1.0),
    (63, 90, 7, -1.0), (65, 65, 9, -1.0),       # no clamp; detector as wide as the image: clamped corners
    (511, 723, 17, -1.0), (513, 726, 15, -1.0),  # one and two pixels a thread, odd last rows, angles not in eights
    (512, 725, 8, 355.25),                       # off-centre axis: the clamp window shrinks
    (64, 91, 24, 0.2), (64, 91, 24, 95.0),       # no active detector: the clamp's two edges cross
])
def test_bp_bit_exact(res, n, d, a, axis):
    """The BP runs the reference's operations in its order
    (projector-parallel-joseph.cl:196-216): equal to the oracle bit for bit."""
    print("case bp bit-exact", n, d, a, axis, flush=True)
    step = np.float32(np.pi / a)
    g = O.Geometry(n, d, a, step, axis=axis)
    sino = np.random.default_rng(n + a).standard_normal((a, d)).astype(np.float32)
    p = _projector(n, d, a, step, False, axis_position=axis).setup(res)
    ds, out = uir.DeviceArray.from_numpy(sino), uir.DeviceArray((n, n))
    assert p.requisition(ds) == (n, n)
    p.process(ds, out)
    assert np.array_equal(out.numpy(), O.bp(g, sino))


@pytest.mark.parametrize("n,a", [(96, 20), (700, 20), (300, 301)])
def test_forward_again_and_with_another_step(res, n, a):
    """A forward projector keeps its tables between calls and takes a changed
    step property at the next one, on both sides of the work table's line
    (90000 rays)."""
    print("case forward, changed step", n, a, flush=True)
    d = n
    x = ellipse_phantom(n, seed=n)
    steps = [np.float32(np.pi / a), np.float32(np.pi / a), np.float32(0.1)]
    p = _projector(n, d, a, steps[0], True).setup(res)
    dx, ds = uir.DeviceArray.from_numpy(x), uir.DeviceArray((a, d))
    for step in steps:
        p["step"] = float(step)
        p.process(dx, ds)
        assert np.array_equal(ds.numpy(), O.fp(O.Geometry(n, d, a, step), x))


@pytest.mark.parametrize("forward", [True, False])
def test_lut_of_an_input_as_high_as_the_angle_count_stays(res, forward):
    """The LUT is rebuilt when the angle count differs from the input's height
    (ufo-ir-parallel-projector-task.c:305-347): a projector whose input is as
    high as its angle count keeps the angles of its first call."""
    n, a = 96, 96
    print("case kept LUT", forward, flush=True)
    first, later = np.float32(np.pi / a), np.float32(0.1)
    g = O.Geometry(n, n, a, first)
    x = np.random.default_rng(8).random((n, n)).astype(np.float32)
    p = _projector(n, n, a, first, forward).setup(res)
    dx, out = uir.DeviceArray.from_numpy(x), uir.DeviceArray((n, n))
    for step in (first, later):
        p["step"] = float(step)
        assert p.requisition(dx) == (n, n)
        p.process(dx, out)
        assert np.array_equal(out.numpy(), O.fp(g, x) if forward else O.bp(g, x))


def test_luts_and_runs_match_oracle(res):
    a, step = 720, np.float32(np.pi / 720)
    g = O.Geometry(1448, 1448, a, step)
    p = _projector(1448, 1448, a, step, False).setup(res)
    p.requisition(uir.DeviceArray((a, 1448)))
    s, c = p.luts()
    assert np.array_equal(s, g.sin) and np.array_equal(c, g.cos)
    assert p.subsets() == g.runs == [(0, 181, 1), (181, 359, 0), (540, 180, 1)]


@pytest.mark.parametrize("axis", [180.0, 190.25])
def test_off_centre_axis(res, axis):
    """axis_position != n_dets / 2 switches detectors off in FP and shrinks the
    BP clamp window (projector-parallel-joseph.cl:62-66,180-182)."""
    n = d = 367
    a, step = 180, np.float32(np.pi / 180)
    g = O.Geometry(n, d, a, step, axis=axis)
    x = shepp_logan(n, extent=256)
    p = _projector(n, d, a, step, True, axis_position=axis).setup(res)
    out = uir.DeviceArray((a, d))
    p.process(uir.DeviceArray.from_numpy(x), out)
    ref = O.fp(g, x)
    assert O.rel_l2(out.numpy(), ref) <= TOL
    q = _projector(n, d, a, step, False, axis_position=axis).setup(res)
    vol = uir.DeviceArray((n, n))
    q.process(uir.DeviceArray.from_numpy(ref), vol)
    assert O.rel_l2(vol.numpy(), O.bp(g, ref)) <= TOL


def test_subset_fp_bp_accumulate(res):
    """subset_fp / subset_bp accumulate with correction_scale / relaxation
    (ufo-ir-parallel-projector-task.c:167-195)."""
    n = d = 128
    a, step = 60, np.float32(np.pi / 60)
    g = O.Geometry(n, d, a, step)
    x = ellipse_phantom(n, seed=11)
    base = np.random.default_rng(1).random((a, d)).astype(np.float32)
    p = _projector(n, d, a, step, False).setup(res)
    p.requisition(uir.DeviceArray((a, d)))
    p["correction_scale"] = 2.5
    p["relaxation"] = 0.75
    dx = uir.DeviceArray.from_numpy(x)
    ds = uir.DeviceArray.from_numpy(base)
    for sub in g.angle_subsets[::7]:
        p.subset_fp(dx, ds, sub)
    ref = base.copy()
    for sub in g.angle_subsets[::7]:
        ref = O.fp(g, x, sino=ref, corr=2.5, subsets=[sub])
    assert O.rel_l2(ds.numpy(), ref) <= TOL
    vol = uir.DeviceArray.from_numpy(x)
    for sub in g.runs:
        p.subset_bp(vol, ds, sub)
    vref = O.bp(g, ref, vol=x, relax=0.75)
    assert O.rel_l2(vol.numpy(), vref) <= TOL
