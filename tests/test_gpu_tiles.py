"""Matrix-free kernels by node tiles (GPU) and the tiles themselves (CPU).

* every node sits in exactly one tile and a tile's columns fit its slots, for tubes, an irregular
  wall, isolated nodes and coordinates that are not numbers (CPU);
* the tile kernels (step, adjoint step) give the bits of the row kernels at sample counts around
  the lane and chunk edges, per-node and per-sample masses, with and without damping, on meshes
  with 6 and with 8 elements around a node, boundary fans and an isolated node; the row kernels
  they are compared with follow the oracle (1e-10 relative max-norm, the bar of every step);
* meshes with more elements around a node than a tile or a fan takes run the row kernels, within
  the same bar, and walking block by block without fan entries agrees with the fans to rounding.
"""
import ctypes

import numpy as np
import pytest

from cvfes_amd import _lib
from cvfes_amd.mesh import tube_geometry
from cvfes_amd.sparse import block_structure
from oracle import solid_oracle as so


def wall(kind, seed=0):
    """Nodes, triangles and fixed nodes of a test wall."""
    rng = np.random.default_rng(seed)
    if kind == "tube":
        return tube_geometry(20, 9, 0.3, 2.0)
    if kind == "isolated":                       # and a node in no element
        nodes, el, bdy = tube_geometry(20, 9, 0.3, 2.0)
        return np.vstack([nodes, [[4.0, 4.0, 4.0]]]), el, bdy
    if kind.startswith("fan"):                   # a flat fan of n triangles about node 0, a grid beside it
        n = int(kind[3:])
        t = 2.0 * np.pi * np.arange(n) / n
        nodes = np.vstack([[[0.0, 0.0, 0.1]], np.stack([np.cos(t), np.sin(t), 0.0 * t], 1)])
        el = np.array([[0, 1 + i, 1 + (i + 1) % n] for i in range(n)])
        el = el[rng.permutation(n)]
        el = np.array([np.roll(e, rng.integers(3)) for e in el])
        bdy = np.array([1])
    else:                                        # "grid": a bumpy rectangle, diagonals at random
        n = 13
        x, y = np.meshgrid(np.arange(n), np.arange(n), indexing="ij")
        nodes = np.stack([x, y, 0.3 * np.sin(x) * np.cos(0.7 * y)], -1).reshape(-1, 3) * 0.05
        el = []
        for i in range(n - 1):
            for j in range(n - 1):
                a, b, c, d = i * n + j, (i + 1) * n + j, (i + 1) * n + j + 1, i * n + j + 1
                el += [[a, b, c], [a, c, d]] if (i + j) % 2 else [[a, b, d], [b, c, d]]
        el = np.array(el)[rng.permutation(len(el))]
        bdy = np.arange(n)
    return nodes, el.astype(np.int64), bdy.astype(np.int64)


def tile_rows(nodes, el):
    ip, ix = block_structure(el, nodes.shape[0])
    ip, ix = ip.astype(np.int32), ix.astype(np.int32)
    xyz = np.ascontiguousarray(nodes, np.float64)
    rows = np.full((nodes.shape[0], _lib.TILE_ROWS), -7, np.int32)
    n = _lib.lib().cvfes_tile_rows(nodes.shape[0], xyz.ctypes.data, ip.ctypes.data, ix.ctypes.data,
                                   rows.ctypes.data, nodes.shape[0])
    assert n > 0
    return rows[:n], ip, ix


@pytest.mark.parametrize("kind", ["tube", "isolated", "grid", "fan8", "nan", "point"])
def test_tiles_hold_every_node_once(kind):
    if not _lib.LIB_PATH.exists():
        pytest.skip("libcvfes_mi355x.so not built")
    nodes, el, _ = wall("tube" if kind in ("nan", "point") else kind)
    if kind == "nan":
        nodes = nodes.copy()
        nodes[::3] = np.nan
    if kind == "point":
        nodes = np.zeros_like(nodes)
    rows, ip, ix = tile_rows(nodes, el)
    assert np.array_equal(np.sort(rows[rows >= 0]), np.arange(nodes.shape[0]))
    for r in rows:
        own = r[r >= 0]
        assert np.all(r[len(own):] == -1)
        cols = np.unique(np.concatenate([ix[ip[a]:ip[a + 1]] for a in own] + [own]))
        assert len(cols) - len(own) <= _lib.TILE_COLS - _lib.TILE_ROWS


def build(kind, S, seed=0, thick_samples=False):
    from cvfes_amd.system import MembraneSystem
    nodes, el, bdy = wall(kind, seed)
    rng = np.random.default_rng(seed)
    E = 7e6 * np.exp(0.1 * rng.standard_normal((el.shape[0], S)))
    n = nodes.shape[0]
    h = 0.07 * rng.uniform(0.9, 1.1, (n, S)) if thick_samples else np.full(n, 0.07)
    s = MembraneSystem(nodes, el, bdy, S, vthickness=h, elmE=E, density=1.0, nu=0.45, store_values=False)
    return nodes, el, bdy, s


def run(s, u0, dt, beta, damp, nsteps=6):
    """Steps, then one adjoint step from the states, by the system's current matrix-free path."""
    import torch
    p = 1.33e4 * (1.0 + 0.1 * np.sin(np.arange(nsteps)))
    s._sys = s._make_struct()
    s.initial_state(u0, 0.0 * u0, s.loads(p), dt, beta=beta, damp=damp, method="matfree")
    s.step(p, dt, beta=beta, damp=damp, method="matfree")
    mu = torch.empty_like(s.u)
    w = torch.linspace(0.5, 1.5, s.n_smp, dtype=torch.float64, device=s.device)
    _lib.check(s.lib.cvfes_adjoint_step(s.stream, ctypes.byref(s._sys), _lib.METHOD_MATFREE, s.u.data_ptr(),
                                        s.up.data_ptr(), mu.data_ptr(), s.state[2].data_ptr(), None,
                                        w.data_ptr(), dt, beta, damp, 1))
    return s.u.cpu().numpy(), mu.cpu().numpy(), p


@pytest.mark.gpu
@pytest.mark.parametrize("kind,S,beta,damp,thick", [
    ("tube", 1, 1e-7, 0.0, False), ("isolated", 2, 0.0, 5.0, True), ("tube", 3, 1e-7, 5.0, False),
    ("grid", 5, 0.0, 0.0, False), ("fan8", 7, 1e-7, 5.0, True), ("tube", 8, 0.0, 0.0, False), ("tube", 9, 1e-7, 0.0, False), ("tube", 31, 0.0, 5.0, True),
    ("tube", 33, 1e-7, 5.0, False), ("tube", 64, 1e-7, 0.0, False), ("tube", 66, 0.0, 0.0, False),
    ("isolated", 128, 1e-7, 5.0, False), ("isolated", 130, 0.0, 0.0, True), ("tube", 200, 1e-7, 5.0, True),
    ("grid", 16, 1e-7, 5.0, True), ("grid", 97, 0.0, 0.0, False), ("fan7", 24, 1e-7, 5.0, False),
    ("fan8", 34, 0.0, 5.0, True)])
def test_tile_kernels_equal_row_kernels(require_gpu, kind, S, beta, damp, thick):
    nodes, el, bdy, s = build(kind, S, seed=S, thick_samples=thick)
    assert s.n_tiles > 0
    dt = 1e-6
    u0 = 1e-4 * np.random.default_rng(S).standard_normal(3 * nodes.shape[0])
    u, mu, p = run(s, u0, dt, beta, damp)
    tiles, s.n_tiles = s.n_tiles, 0
    ur, mur, _ = run(s, u0, dt, beta, damp)
    s.n_tiles = tiles
    assert np.all(np.isfinite(u)) and np.max(np.abs(mu)) > 0
    assert np.array_equal(u, ur) and np.array_equal(mu, mur)
    ref = oracle_run(nodes, el, bdy, s, u0, p, dt, beta, damp)
    assert np.max(np.abs(u.reshape(-1, S) - ref)) < 1e-10 * np.max(np.abs(ref))


def oracle_run(nodes, el, bdy, s, u0, p, dt, beta, damp):
    ip, ix = so.sparse_info_loops(el, nodes.shape[0])
    h = np.broadcast_to(s.vthick.cpu().numpy().reshape(nodes.shape[0], -1), (nodes.shape[0], s.n_smp))
    gth = so.gauss_properties(np.ones_like(h), h, el)[1]
    _, K, f1, LM = so.assemble_reference(nodes, el, 1.0, so.d_matrix(0.45), s.coef.cpu().numpy(), gth, 1.0, ip, ix)
    bd = (3 * bdy[:, None] + np.arange(3)).ravel()
    return so.run(ip, ix, K, LM, f1, p, u0, 0.0 * u0, dt, beta=beta, damp=damp, bdy_dofs=bd)[0]


@pytest.mark.gpu
@pytest.mark.parametrize("kind,S", [("fan9", 16), ("fan40", 5), ("fan9", 3)])
def test_untiled_meshes_and_block_walk(require_gpu, kind, S):
    """More elements around a node than a tile takes (9, and 40: beyond the sorted fans)."""
    nodes, el, bdy, s = build(kind, S, seed=3)
    dt, beta, damp = 1e-6, 1e-7, 5.0
    assert s.fan is not None and s.n_tiles == 0
    u0 = 1e-4 * np.random.default_rng(1).standard_normal(3 * nodes.shape[0])
    u, mu, p = run(s, u0, dt, beta, damp)
    ref = oracle_run(nodes, el, bdy, s, u0, p, dt, beta, damp)
    assert np.max(np.abs(u.reshape(-1, S) - ref)) < 1e-10 * np.max(np.abs(ref))
    fan, s.fan = s.fan, None
    ub, mub, _ = run(s, u0, dt, beta, damp)
    s.fan = fan
    # the two walks sum the same products in another order: a few ulp per step of the largest value
    assert np.max(np.abs(u - ub)) < 1e-13 * np.max(np.abs(ub))
    assert np.max(np.abs(mu - mub)) < 1e-12 * np.max(np.abs(mub))


@pytest.mark.gpu
def test_batched_tiles_and_rows_in_one_ensemble(require_gpu):
    """Tiled meshes of three shapes beside meshes with wave tasks: eager and replayed steps give the
    single-mesh bits."""
    from cvfes_amd.batch import BatchedEnsemble
    n = 24
    specs = [("tube", 64, 1e-7, 5.0), ("tube", 5, 0.0, 0.0), ("fan8", 33, 0.0, 5.0), ("grid", 12, 0.0, 0.0),
             ("fan9", 16, 1e-7, 0.0)]
    systems = [build(k, S, seed=S)[3] for k, S, _, _ in specs]
    loads = [s.loads(np.full(n, 1.33e4)) for s in systems]
    u0s = [1e-4 * np.random.default_rng(i).standard_normal(3 * s.n_nodes) for i, s in enumerate(systems)]
    outs = []
    for mode in ("single", "eager", "graph"):
        ens = BatchedEnsemble(systems, loads, dts=1e-6, methods="matfree", betas=[c[2] for c in specs],
                              damps=[c[3] for c in specs])
        ens.initial_state(u0s=u0s)
        assert [int(m.tiled) for m in ens.host_meshes] == [1, 0, 1, 1, 0]
        if mode == "single":
            ens.run_per_mesh(n)
        else:
            ens.run(n, graph=mode == "graph", block=6)
        outs.append([s.u.cpu().numpy() for s in systems])
    for o in outs[1:]:
        for a, b in zip(outs[0], o):
            assert np.all(np.isfinite(a)) and np.array_equal(a, b)


def free_nodes(nodes, el, bdy, share, seed=0):
    """The wall with `share` of its node count in nodes of no element, scattered among its own."""
    rng = np.random.default_rng(seed)
    n = int(round(share * nodes.shape[0]))
    lo, hi = nodes.min(0), nodes.max(0)
    near = nodes[rng.integers(nodes.shape[0], size=n)] + 0.02 * (hi - lo) * rng.standard_normal((n, 3))
    every = np.vstack([nodes, near])
    place = rng.permutation(every.shape[0])            # node i of the wall becomes place[i]
    out = np.empty_like(every)
    out[place] = every
    return out, place[el], place[bdy]


def walls_with_free_nodes(kind, share):
    if kind == "large":
        return free_nodes(*tube_geometry(64, 32, 0.3, 2.0), share)
    if kind == "two":                                  # one wall inside the other, a spacing apart
        a, ea, ba = tube_geometry(40, 24, 0.30, 2.0)
        b, eb, bb = tube_geometry(40, 24, 0.33, 2.0)
        return free_nodes(np.vstack([a, b]), np.vstack([ea, eb + a.shape[0]]), np.concatenate([ba, bb + a.shape[0]]), share)
    return free_nodes(*wall(kind), share)


@pytest.mark.parametrize("kind", ["tube", "grid", "large", "two"])
@pytest.mark.parametrize("share", [0.05, 0.2, 0.5, 1.0])
def test_tiles_hold_their_halo_among_free_nodes(kind, share):
    """Nodes of no element have empty block rows: they take a row slot of a tile and no column."""
    if not _lib.LIB_PATH.exists():
        pytest.skip("libcvfes_mi355x.so not built")
    nodes, el, _ = walls_with_free_nodes(kind, share)
    rows, ip, ix = tile_rows(nodes, el)
    assert np.array_equal(np.sort(rows[rows >= 0]), np.arange(nodes.shape[0]))
    for r in rows:
        own = r[r >= 0]
        cols = np.unique(np.concatenate([ix[ip[a]:ip[a + 1]] for a in own] + [own]))
        assert len(cols) - len(own) <= _lib.TILE_COLS - _lib.TILE_ROWS


@pytest.mark.gpu
@pytest.mark.parametrize("kind,share,S", [("two", 0.2, 33), ("large", 0.05, 16), ("two", 1.0, 5)])
def test_tile_kernels_among_free_nodes(require_gpu, kind, share, S):
    from cvfes_amd.system import MembraneSystem
    nodes, el, bdy = walls_with_free_nodes(kind, share)
    n, dt, beta, damp = nodes.shape[0], 1e-6, 1e-7, 5.0
    E = 7e6 * np.exp(0.1 * np.random.default_rng(S).standard_normal((el.shape[0], S)))
    s = MembraneSystem(nodes, el, bdy, S, vthickness=np.full(n, 0.07), elmE=E, density=1.0, nu=0.45, store_values=False)
    assert s.n_tiles > 0
    u0 = 1e-4 * np.random.default_rng(S).standard_normal(3 * n)
    u, mu, p = run(s, u0, dt, beta, damp)
    tiles, s.n_tiles = s.n_tiles, 0
    ur, mur, _ = run(s, u0, dt, beta, damp)
    s.n_tiles = tiles
    assert np.array_equal(u, ur) and np.array_equal(mu, mur)
    ref = oracle_run(nodes, el, bdy, s, u0, p, dt, beta, damp)
    used = np.repeat(np.isin(np.arange(n), el), 3)     # a node of no element has no mass: 0 / 0 in the oracle
    assert np.max(np.abs(u.reshape(-1, S) - ref)[used]) < 1e-10 * np.max(np.abs(ref[used]))


@pytest.mark.gpu
def test_lists_refuse_a_tile_that_does_not_fit(require_gpu):
    import torch
    nodes, el, bdy, s = build("tube", 2)
    far = np.full((1, _lib.TILE_ROWS), -1, np.int32)
    far[0, :4] = [40, 65, 90, 115]                     # four rows of six neighbours each, none in common
    out = [torch.empty(k, dtype=torch.int32, device="cuda")
           for k in (4 * _lib.TILE_ROWS, _lib.TILE_COLS - _lib.TILE_ROWS, 2 * _lib.TILE_ROWS * _lib.TILE_ELEMS)]
    for take, good in ((3, True), (4, False)):
        rows = torch.as_tensor(np.where(np.arange(_lib.TILE_ROWS) < take, far, -1).astype(np.int32)).cuda()
        rc = s.lib.cvfes_tile_lists(s.stream, 1, rows.data_ptr(), s.nptr.data_ptr(), s.fan.data_ptr(),
                                    s.max_node_elems, *[t.data_ptr() for t in out])
        assert (rc == 0) == good


@pytest.mark.gpu
@pytest.mark.parametrize("nz,S,beta,damp,tiled", [
    (42, 128, 1e-7, 5.0, True), (42, 100, 0.0, 0.0, True), (42, 128, 1e-7, 0.0, False), (9, 128, 0.0, 5.0, True),
    (42, 96, 0.0, 5.0, False), (42, 66, 1e-7, 0.0, True)])
def test_fused_step_is_its_two_steps(require_gpu, nz, S, beta, damp, tiled):
    """Two samples per lane of wave-uniform rows, large and small (two launches and one), with tiles and
    by rows; 66 samples: packed rows."""
    import torch
    from cvfes_amd.system import MembraneSystem
    nodes, el, bdy = tube_geometry(64, nz, 0.3, 2.0)
    E = 7e6 * np.exp(0.1 * np.random.default_rng(S).standard_normal((el.shape[0], S)))
    s = MembraneSystem(nodes, el, bdy, S, vthickness=np.full(nodes.shape[0], 0.07), elmE=E, density=1.0, nu=0.45,
                       store_values=False)
    if not tiled:
        s.n_tiles = 0
        s._sys = s._make_struct()
    load, dt = s.loads(np.full(3, 1.33e4)), 1e-6
    u0 = 1e-4 * np.random.default_rng(1).standard_normal(3 * nodes.shape[0])
    s.initial_state(u0, 0.0 * u0, load, dt, beta=beta, damp=damp, method="matfree")
    gen = torch.Generator(device="cuda").manual_seed(S)
    m1, m2 = (torch.randn(s.state_shape(), generator=gen, dtype=torch.float64, device="cuda") for _ in range(2))
    w = torch.linspace(0.5, 1.5, S, dtype=torch.float64, device="cuda")
    p, got = _lib.ptr, []
    for fused in (True, False):
        out, mu = torch.full_like(s.u, np.nan), torch.full_like(s.u, np.nan)
        arr = (ctypes.c_void_p * 3)(p(s.u), p(s.up), p(out))
        ls, sys = ctypes.byref(load.struct(1)), ctypes.byref(s._sys)
        if fused:
            _lib.check(s.lib.cvfes_adjoint_fused_step(s.stream, sys, 1, arr, ls, p(m1), p(m2), p(mu), p(s.up), None, p(w),
                                                      dt, beta, damp))
        else:
            _lib.check(s.lib.cvfes_step(s.stream, sys, 1, arr, ls, 1, dt, beta, damp))
            _lib.check(s.lib.cvfes_adjoint_step(s.stream, sys, 1, p(m1), p(m2), p(mu), p(s.up), None, p(w), dt, beta,
                                                damp, 1))
        got.append((out.cpu().numpy(), mu.cpu().numpy()))
    for a, b in zip(*got):
        assert np.all(np.isfinite(a)) and np.max(np.abs(a)) > 0 and np.array_equal(a, b)
