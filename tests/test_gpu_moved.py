"""The updated-geometry step without element frames, at every lane width and row mapping: it follows
the kernel of the divided element frames, and a system without fan entries takes the frames.  Six
steps of some 250 roundings of 1.1e-16 each are 1.7e-13 of the largest displacement: 1e-12."""
import numpy as np
import pytest

from tests.test_gpu_tiles import wall

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("kind,S,interval,beta,damp", [
    ("tube", 1, 1, 0.0, 0.0), ("grid", 2, 1, 1e-7, 5.0), ("isolated", 33, 3, 1e-7, 0.0), ("grid", 64, 1, 0.0, 5.0),
    ("tube", 97, 3, 0.0, 5.0), ("isolated", 100, 1, 1e-7, 5.0), ("fan9", 128, 3, 1e-7, 5.0), ("fan40", 6, 1, 0.0, 0.0),
    ("grid", 130, 1, 0.0, 0.0)])
@pytest.mark.parametrize("form", ["auto", "rowload1"])
def test_moved_equals_frames(require_gpu, kind, S, interval, beta, damp, form):
    from cvfes_amd.system import MembraneSystem
    nodes, el, bdy = wall(kind)
    rng = np.random.default_rng(S)
    E = 7e6 * np.exp(0.1 * rng.standard_normal((el.shape[0], S)))
    u0 = 1e-3 * rng.standard_normal(3 * nodes.shape[0])
    ga, q = rng.standard_normal(3 * nodes.shape[0]), np.linspace(1.0, 2.0, 6)
    dt, p = 1e-6, 1.33e4 * (1.0 + 0.1 * np.sin(np.arange(6)))
    got = []
    for variant, fan in (("generic", True), (form, True), (form, False)):
        s = MembraneSystem(nodes, el, bdy, S, vthickness=np.full(nodes.shape[0], 0.07), elmE=E, density=1.0,
                           nu=0.45, store_values=False)
        s.set_variant(variant)
        if not fan:
            s.fan = None
            s._sys = s._make_struct()
        ls = s.loads(p, ga=ga, qa=q)
        s.initial_state(u0, 0.0 * u0, ls, dt, beta=beta, damp=damp, method="matfree")
        s.step_updated(ls, dt, interval, beta=beta, damp=damp)
        got.append(s.u.cpu().numpy())
    top = np.max(np.abs(got[0]))
    assert top > 0 and all(np.all(np.isfinite(g)) for g in got)
    assert np.max(np.abs(got[1] - got[0])) < 1e-12 * top
    assert np.max(np.abs(got[1] - got[2])) < 1e-12 * top


@pytest.mark.parametrize("S,interval,beta", [(200, 1, 1e-7), (255, 3, 0.0)])
def test_rows_by_tiles_equal_natural_order(require_gpu, S, interval, beta):
    """Systems large enough for the tiles' row order give the bits of the natural order."""
    from cvfes_amd.mesh import tube_geometry
    from cvfes_amd.system import MembraneSystem
    nodes, el, bdy = tube_geometry(96, 97, 0.3, 2.0)
    assert 24 * nodes.shape[0] * S > 32 << 20
    E = 7e6 * np.exp(0.1 * np.random.default_rng(S).standard_normal((el.shape[0], S)))
    u0 = 1e-3 * np.random.default_rng(1).standard_normal(3 * nodes.shape[0])
    s = MembraneSystem(nodes, el, bdy, S, vthickness=np.full(nodes.shape[0], 0.07), elmE=E, density=1.0, nu=0.45,
                       store_values=False)
    got, tiles = [], s.n_tiles
    assert tiles > 0
    for n in (tiles, 0):
        s.n_tiles = n
        s._sys = s._make_struct()
        ls = s.loads(np.full(5, 1.33e4))
        s.initial_state(u0, 0.0 * u0, ls, 1e-6, beta=beta, damp=5.0, method="matfree")
        s.step_updated(ls, 1e-6, interval, beta=beta, damp=5.0)
        got.append(s.u.cpu().numpy())
    # the initial product runs by rows either way
    assert np.max(np.abs(got[0])) > 0 and np.array_equal(got[0], got[1])


@pytest.mark.parametrize("S,interval,beta", [(128, 3, 1e-7), (192, 3, 0.0), (256, 1, 1e-7)])
def test_row_order_rule_keeps_the_bits(require_gpu, S, interval, beta):
    """The shortest rows that take the tiles' order with a damped state and a saved geometry, and with
    one of them."""
    from cvfes_amd.mesh import tube_geometry
    from cvfes_amd.system import MembraneSystem
    nodes, el, bdy = tube_geometry(128, 97, 0.3, 2.0)
    assert 24 * nodes.shape[0] * S > 32 << 20
    E = 7e6 * np.exp(0.1 * np.random.default_rng(S).standard_normal((el.shape[0], S)))
    u0 = 1e-3 * np.random.default_rng(1).standard_normal(3 * nodes.shape[0])
    s = MembraneSystem(nodes, el, bdy, S, vthickness=np.full(nodes.shape[0], 0.07), elmE=E, density=1.0, nu=0.45,
                       store_values=False)
    got = []
    for n in (s.n_tiles, 0):
        s.n_tiles = n
        s._sys = s._make_struct()
        ls = s.loads(np.full(5, 1.33e4))
        s.initial_state(u0, 0.0 * u0, ls, 1e-6, beta=beta, damp=5.0, method="matfree")
        s.step_updated(ls, 1e-6, interval, beta=beta, damp=5.0)
        got.append(s.u.cpu().numpy())
    assert np.max(np.abs(got[0])) > 0 and np.array_equal(got[0], got[1])
