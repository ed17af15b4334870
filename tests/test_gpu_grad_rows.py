"""The gradient accumulation at every lane width, row mapping and alignment against the element form
in 64 bits over all nine unit blocks: 81 products and sums of 1.1e-16 on either side, the vectors
relative to a node at most twice the nodes' own, so 1e-13 of the sum of magnitudes."""
import ctypes

import numpy as np
import pytest
import torch

from tests.test_gpu_element_rows import shifted, system

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("kind,S", [("tube", 1), ("grid", 7), ("tube", 8), ("isolated", 15), ("grid", 16), ("tube", 31),
                                    ("grid", 32), ("isolated", 63), ("tube", 64), ("grid", 100), ("tube", 128),
                                    ("isolated", 192), ("fan40", 256), ("grid", 257)])
@pytest.mark.parametrize("beta,strided,inverse,by", [(0.0, False, True, 0), (1e-7, True, True, 0),
                                                     (0.0, True, False, 1), (1e-7, False, False, 0)])
def test_gradient_rows(require_gpu, kind, S, beta, strided, inverse, by):
    from cvfes_amd import _lib
    nodes, el, E, s = system(kind, S, store_values=False)
    n, rng, dt = nodes.shape[0], np.random.default_rng(S), 1e-6
    mu, xc, xp = rng.standard_normal((3, n, 3, S))
    m = np.exp(0.1 * rng.standard_normal((n, S) if strided else (n, 1)))
    m[n // 2] = 0.0
    g0 = rng.standard_normal((el.shape[0], S))
    coef = s.coef.cpu().numpy()
    minv = np.divide(1.0, m, out=np.zeros_like(m), where=m != 0.0)
    d = [shifted(x, by) for x in (mu, xc, xp, m, minv, g0)]
    sys = s._make_struct()
    sys.lm, sys.lm_sstride, sys.minv = _lib.ptr(d[3]), int(strided), _lib.ptr(d[4]) if inverse else None
    cpos = s.cpos if getattr(s, "cpos", None) is not None else torch.as_tensor(s.maps.cpos).to("cuda", torch.int32)
    p = _lib.ptr
    _lib.check(s.lib.cvfes_grad_accum(s.stream, ctypes.byref(sys), p(s.elems), p(cpos), p(d[0]), p(d[1]),
                                      p(d[2]) if beta else None, dt, beta, 2.5, p(d[5])))
    kh = s.khat.cpu().numpy().reshape(-1, 9)[np.asarray(s.maps.cpos).reshape(-1)].reshape(-1, 3, 3, 3, 3)
    nu = (2.5 * minv[:, None] * mu)[el]
    x = (xc + beta / dt * (xc - xp))[el] if beta else xc[el]
    form = np.einsum("eais,eabij,ebjs->es", nu, kh, x)
    size = np.einsum("eais,eabij,ebjs->es", np.abs(nu), np.abs(kh), np.abs(x))
    ref = g0 - coef * form
    got = d[5].cpu().numpy()
    assert np.all(np.abs(got - ref) <= 1e-13 * (np.abs(g0) + coef * size))


@pytest.mark.parametrize("kind,S", [("tube", 1), ("grid", 7), ("tube", 8), ("isolated", 15), ("grid", 16), ("fan40", 33),
                                    ("tube", 64), ("grid", 100), ("isolated", 128), ("grid", 257)])
@pytest.mark.parametrize("beta,strided,by", [(0.0, False, 0), (1e-7, True, 0), (1e-7, False, 1)])
def test_gradient_rows_of_any_blocks(require_gpu, kind, S, beta, strided, by):
    """A system without fan entries makes no claim on its unit blocks: blocks that are neither symmetric
    nor sum to zero (an elastic bedding, say), all nine of them, to the same bound."""
    from cvfes_amd import _lib
    nodes, el, E, s = system(kind, S, store_values=False)
    n, rng, dt = nodes.shape[0], np.random.default_rng(S), 1e-6
    mu, xc, xp = rng.standard_normal((3, n, 3, S))
    m = np.exp(0.1 * rng.standard_normal((n, S) if strided else (n, 1)))
    m[n // 2] = 0.0
    g0 = rng.standard_normal((el.shape[0], S))
    coef = s.coef.cpu().numpy()
    kh_all = rng.standard_normal((9 * el.shape[0], 9))
    d = [shifted(x, by) for x in (mu, xc, xp, m, g0, kh_all)]
    sys = s._make_struct()
    sys.lm, sys.lm_sstride, sys.minv = _lib.ptr(d[3]), int(strided), None
    sys.fan, sys.n_tiles, sys.khat = None, 0, _lib.ptr(d[5])
    cpos = s.cpos if getattr(s, "cpos", None) is not None else torch.as_tensor(s.maps.cpos).to("cuda", torch.int32)
    p = _lib.ptr
    _lib.check(s.lib.cvfes_grad_accum(s.stream, ctypes.byref(sys), p(s.elems), p(cpos), p(d[0]), p(d[1]),
                                      p(d[2]) if beta else None, dt, beta, 2.5, p(d[4])))
    kh = kh_all[np.asarray(s.maps.cpos).reshape(-1)].reshape(-1, 3, 3, 3, 3)
    minv = np.divide(1.0, m, out=np.zeros_like(m), where=m != 0.0)
    nu = (2.5 * minv[:, None] * mu)[el]
    x = (xc + beta / dt * (xc - xp))[el] if beta else xc[el]
    ref = g0 - coef * np.einsum("eais,eabij,ebjs->es", nu, kh, x)
    size = np.einsum("eais,eabij,ebjs->es", np.abs(nu), np.abs(kh), np.abs(x))
    assert np.all(np.abs(d[4].cpu().numpy() - ref) <= 1e-13 * (np.abs(g0) + coef * size))
