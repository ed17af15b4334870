"""The symmetric-storage kernels that read a row's structure from its record, at every lane width and
row mapping: the step, the adjoint step and the fused step give the bits of the kernels that walk
indptr, indices and vblk, and the step follows the oracle (1e-10 relative max-norm)."""
import ctypes

import numpy as np
import pytest

from cvfes_amd import _lib
from tests.test_gpu_tiles import oracle_run, wall

pytestmark = pytest.mark.gpu


def run(s, u0, p, dt, beta, damp):
    import torch
    s._sys = s._make_struct()
    ls = s.loads(p)
    s.initial_state(u0, 0.0 * u0, ls, dt, beta=beta, damp=damp)
    s.step(ls, dt, beta=beta, damp=damp)
    u, up, w = s.u, s.up, torch.linspace(0.5, 1.5, s.n_smp, dtype=torch.float64, device=s.device)
    mu, out, mu_f = (torch.empty_like(u) for _ in range(3))
    _lib.check(s.lib.cvfes_adjoint_step(s.stream, ctypes.byref(s._sys), 0, u.data_ptr(), up.data_ptr(),
                                        mu.data_ptr(), up.data_ptr(), None, w.data_ptr(), dt, beta, damp, 1))
    arr = (ctypes.c_void_p * 3)(u.data_ptr(), up.data_ptr(), out.data_ptr())
    m1, m2 = u.clone(), up.clone()
    _lib.check(s.lib.cvfes_adjoint_fused_step(s.stream, ctypes.byref(s._sys), 0, arr, ctypes.byref(ls.struct(0)),
                                              m1.data_ptr(), m2.data_ptr(), mu_f.data_ptr(), up.data_ptr(), None,
                                              w.data_ptr(), dt, beta, damp))
    return [t.cpu().numpy() for t in (u, mu, out, mu_f)]


@pytest.mark.parametrize("kind,S,beta,damp,order", [
    ("tube", 1, 1e-7, 0.0, "natural"), ("tube", 2, 0.0, 5.0, "natural"), ("tube", 5, 1e-7, 5.0, "strips"),
    ("isolated", 16, 0.0, 0.0, "natural"), ("tube", 33, 1e-7, 5.0, "natural"), ("isolated", 64, 1e-7, 0.0, "strips"),
    ("tube", 97, 0.0, 5.0, "natural"), ("tube", 100, 1e-7, 5.0, "natural"), ("grid", 34, 1e-7, 5.0, "natural"),
    ("grid", 130, 0.0, 0.0, "natural")])
def test_records_equal_walk(require_gpu, kind, S, beta, damp, order):
    from cvfes_amd.system import MembraneSystem
    nodes, el, bdy = wall(kind)
    E = 7e6 * np.exp(0.1 * np.random.default_rng(S).standard_normal((el.shape[0], S)))
    s = MembraneSystem(nodes, el, bdy, S, vthickness=np.full(nodes.shape[0], 0.07), elmE=E, density=1.0, nu=0.45)
    s.set_variant("generic")
    s.set_row_order(order, width=8)
    assert s.record_width == (24 - 2 if kind == "grid" else 16)     # 10 or 7 block slots
    dt, p = 1e-6, 1.33e4 * (1.0 + 0.1 * np.sin(np.arange(5)))
    u0 = 1e-4 * np.random.default_rng(S + 1).standard_normal(3 * nodes.shape[0])
    a = run(s, u0, p, dt, beta, damp)
    s.row_records, s.record_width = None, 0
    b = run(s, u0, p, dt, beta, damp)
    for x, y in zip(a, b):
        assert np.all(np.isfinite(x)) and np.max(np.abs(x)) > 0 and np.array_equal(x, y)
    ref = oracle_run(nodes, el, bdy, s, u0, p, dt, beta, damp)
    assert np.max(np.abs(a[0].reshape(-1, S) - ref)) < 1e-10 * np.max(np.abs(ref))
