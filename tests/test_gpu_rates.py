"""Calls that a rule of a dispatch once sent to the slower of two kernels, timed against what they can
be held to on the same card and in the same minute: a device copy of the bytes the call has to move,
or the other kernel.  Best of several interleaved rounds, and limits that leave a wide margin to what
was measured on either side."""
import ctypes

import numpy as np
import pytest
import torch

from cvfes_amd import _lib
from cvfes_amd.mesh import tube_geometry

pytestmark = pytest.mark.gpu


def microseconds(calls, rounds=9, n=20):
    """Best time of each call over interleaved rounds of n."""
    best = [np.inf] * len(calls)
    for c in calls:
        c()
    for _ in range(rounds):
        for i, c in enumerate(calls):
            e0, e1 = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
            e0.record()
            for _ in range(n):
                c()
            e1.record()
            e1.synchronize()
            best[i] = min(best[i], 1e3 * e0.elapsed_time(e1) / n)
    return best


def system(nt, nz, S, **kw):
    from cvfes_amd.system import MembraneSystem
    nodes, el, bdy = tube_geometry(nt, nz, 0.5, 6.0)
    E = 7e6 * np.exp(0.1 * np.random.default_rng(S).standard_normal((el.shape[0], S)))
    return MembraneSystem(nodes, el, bdy, S, vthickness=np.full(nodes.shape[0], 0.07), elmE=E, density=1.0, nu=0.45, **kw)


def copy_of(n_bytes):
    """A device copy that reads and writes n_bytes together."""
    a = torch.zeros(int(n_bytes) // 16, dtype=torch.float64, device="cuda")
    b = torch.empty_like(a)
    return lambda: b.copy_(a)


# Stores past L2 of rows of a few samples took 5.4 (blocks) and 2.3 times as long as stores through it.
@pytest.mark.parametrize("S", [1, 2, 4])
def test_assembly_of_few_samples(require_gpu, S):
    s = system(256, 400, S)
    moved = 72 * s.nnzu * S + 8 * s.coef.numel() + 8 * s.khat.numel()
    t, copy = microseconds([s.assemble_upper, copy_of(moved)])
    print(f"{S} samples: {t:.1f} us, copy {copy:.1f}")
    assert t <= 2.5 * copy + 5.0


@pytest.mark.parametrize("S", [2, 6])
def test_stress_of_few_samples(require_gpu, S):
    s = system(256, 400, S, store_values=False)
    u = torch.zeros(s.state_shape(), dtype=torch.float64, device="cuda")
    moved = 8 * (6 * s.n_elms * S + u.numel()) + 12 * s.n_elms
    t, copy = microseconds([lambda: s.element_stress(u=u), copy_of(moved)])
    print(f"{S} samples: {t:.1f} us, copy {copy:.1f}")
    assert t <= 2.5 * copy + 5.0


def irregular(nt, nz, seed=0):
    """A tube with every quad's diagonal at random: 4 to 8 elements around a node, 5 to 9 blocks a row."""
    t, z = np.meshgrid(2.0 * np.pi * np.arange(nt) / nt, 6.0 * np.arange(nz) / (nz - 1))
    nodes = np.stack([0.5 * np.cos(t), 0.5 * np.sin(t), z], -1).reshape(-1, 3)
    i, j = np.meshgrid(np.arange(nz - 1), np.arange(nt), indexing="ij")
    a, b = (i * nt + j).ravel(), (i * nt + (j + 1) % nt).ravel()
    c, d = b + nt, a + nt
    side = np.random.default_rng(seed).random(a.size) < 0.5
    el = np.concatenate([np.where(side[:, None], np.stack([a, b, c], 1), np.stack([a, b, d], 1)),
                         np.where(side[:, None], np.stack([a, c, d], 1), np.stack([b, c, d], 1))])
    return nodes, el, np.concatenate([np.arange(nt), nt * (nz - 1) + np.arange(nt)])


def irregular_system(nt, nz, S, **kw):
    from cvfes_amd.system import MembraneSystem
    nodes, el, bdy = irregular(nt, nz)
    E = 7e6 * np.exp(0.1 * np.random.default_rng(S).standard_normal((el.shape[0], S)))
    return MembraneSystem(nodes, el, bdy, S, vthickness=np.full(nodes.shape[0], 0.07), elmE=E, density=1.0, nu=0.45, **kw)


# Walking the symmetric storage, a step of 8 samples took 1.6 times its product (16 -> 23 us at 16,384
# nodes): the compiler waited for each block's entries a few at a time.  It reads two states and the
# masses besides, and measures 1.1 to 1.2 times the product.
def test_walked_step_keeps_to_its_product(require_gpu):
    s = irregular_system(128, 128, 8)
    s.row_records, s.record_width = None, 0
    s._sys = s._make_struct()
    load, z = s.loads(np.zeros(20)), np.zeros(3 * s.n_nodes)
    s.initial_state(z, z, load, 1e-7, damp=1.0)
    x, y = torch.zeros_like(s.u), torch.empty_like(s.u)
    step, product = microseconds([lambda: s.step(load, 1e-7, damp=1.0, nsteps=20), lambda: s.spmv(x, out=y)], n=5)
    print(f"step {step / 20:.1f} us, product {product:.1f}")
    assert step / 20 <= 1.35 * product


# Row records against the walk over indptr, indices and vblk, where records once took 1.1 to 1.2 times as
# long.  The kernel that the rule takes has to be the faster one, within the noise.
@pytest.mark.parametrize("kind,call", [("irregular", "product"), ("irregular", "adjoint"), ("tube", "adjoint")])
def test_records_only_where_they_pay(require_gpu, kind, call):
    S = 48
    s = irregular_system(128, 128, S) if kind == "irregular" else system(128, 128, S)
    x, y, z = (torch.zeros(s.state_shape(), dtype=torch.float64, device="cuda") for _ in range(3))
    structs = [s._make_struct()]
    assert structs[0].row_records
    s.row_records, s.record_width, kept = None, 0, s.row_records
    structs.append(s._make_struct())
    p = _lib.ptr

    def run(sys):
        if call == "product":
            return lambda: _lib.check(s.lib.cvfes_bcsr_spmv(s.stream, ctypes.byref(sys), 0, p(x), p(y)))
        return lambda: _lib.check(s.lib.cvfes_adjoint_step(s.stream, ctypes.byref(sys), 0, p(x), p(z), p(y), None, None,
                                                           None, 1e-7, 0.0, 1.0, 1))
    ruled, walked = microseconds([run(sys) for sys in structs])
    print(f"by the rule {ruled:.1f} us, walked {walked:.1f}")
    assert ruled <= 1.08 * walked
    del kept


# The fused forward + adjoint step exists to be faster than its two launches; matrix-free, with two
# samples per lane of wave-uniform rows, it once took 1.2 to 1.5 times as long.
@pytest.mark.parametrize("S", [128, 256])
def test_fused_step_keeps_to_its_two_launches(require_gpu, S):
    s = system(128, 128, S, store_values=False)
    load, z = s.loads(np.zeros(4)), np.zeros(3 * s.n_nodes)
    s.initial_state(z, z, load, 1e-7, damp=1.0, method="matfree")
    a, b, c = (torch.zeros_like(s.u) for _ in range(3))
    p, sys, ls = _lib.ptr, ctypes.byref(s._sys), load.struct(0)
    state = (ctypes.c_void_p * 3)(*[t.data_ptr() for t in s.state])

    def fused():
        _lib.check(s.lib.cvfes_adjoint_fused_step(s.stream, sys, 1, state, ctypes.byref(ls), p(a), p(b), p(c), None, None,
                                                  None, 1e-7, 0.0, 1.0))

    def separate():
        _lib.check(s.lib.cvfes_step(s.stream, sys, 1, state, ctypes.byref(ls), 1, 1e-7, 0.0, 1.0))
        _lib.check(s.lib.cvfes_adjoint_step(s.stream, sys, 1, p(a), p(b), p(c), None, None, None, 1e-7, 0.0, 1.0, 1))

    one, two = microseconds([fused, separate])
    print(f"fused {one:.1f} us, two launches {two:.1f}")
    assert one <= 1.1 * two


# The updated-geometry step in the rows' natural order against the order of the node tiles, in which
# rows of 64 samples once took 1.1 to 1.3 times as long.
def test_updated_step_takes_the_faster_row_order(require_gpu):
    s = system(206, 320, 64, store_values=False)
    load, u0 = s.loads(np.zeros(5)), 1e-4 * np.random.default_rng(0).standard_normal(3 * s.n_nodes)
    s.initial_state(u0, 0.0 * u0, load, 1e-7, beta=1e-7, damp=1e-3, method="matfree")
    tiles = s.n_tiles
    assert tiles > 0

    def steps(n_tiles):
        def call():
            s.n_tiles = n_tiles
            s._sys = s._make_struct()
            s.step_updated(load, 1e-7, 5, beta=1e-7, damp=1e-3)
        return call
    ruled, natural = microseconds([steps(tiles), steps(0)], n=5)
    print(f"by the rule {ruled:.1f} us, natural {natural:.1f}")
    assert ruled <= 1.06 * natural
