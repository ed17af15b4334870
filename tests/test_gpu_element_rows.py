"""The kernels with a row per element or block at every lane width, row mapping and alignment: the
stresses against the oracle (some 100 roundings of 1.1e-16 and gradients no worse conditioned than
10: 1e-12 of the largest), the assembled blocks against the contributions summed in 64 bits (at most
40 products and sums: 1e-14 of the sum of magnitudes), the coefficients against NumPy."""
import numpy as np
import pytest
import torch

from oracle import solid_oracle as so
from tests.test_gpu_tiles import wall

pytestmark = pytest.mark.gpu


def system(kind, S, **kw):
    from cvfes_amd.system import MembraneSystem
    nodes, el, bdy = wall(kind)
    E = 7e6 * np.exp(0.1 * np.random.default_rng(S).standard_normal((el.shape[0], S)))
    return nodes, el, E, MembraneSystem(nodes, el, bdy, S, vthickness=np.full(nodes.shape[0], 0.07), elmE=E,
                                        density=1.0, nu=0.45, **kw)


def shifted(x, by):
    """`x` on the device, its first element `by` doubles behind an allocation's start."""
    buf = torch.empty(x.size + by, dtype=torch.float64, device="cuda")
    out = buf[by:].view(x.shape)
    out.copy_(torch.as_tensor(x))
    return out


@pytest.mark.parametrize("S", [1, 2, 33, 50, 63, 64, 97, 100, 128, 130])
@pytest.mark.parametrize("geom,by", [("reference", 0), ("moved", 0), ("same", 0), ("moved", 1), ("reference", 1)])
def test_stress_rows(require_gpu, S, geom, by):
    nodes, el, E, s = system("grid" if S % 2 else "isolated", S, store_values=False)
    rng = np.random.default_rng(S)
    u = 2e-3 * rng.standard_normal((nodes.shape[0], 3, S))
    ug = {"reference": 0.0 * u, "moved": 2e-3 * rng.standard_normal(u.shape), "same": u}[geom]
    ud = shifted(u, by)
    st = s.element_stress(u=ud, ug={"reference": None, "moved": shifted(ug, by), "same": ud}[geom],
                          ave_E=shifted(E, by)).cpu().numpy()
    ref = so.calculate_stress(nodes[None] + np.moveaxis(ug, 2, 0), el, so.d_matrix(0.45), E, u.reshape(-1, S))
    assert np.max(np.abs(np.moveaxis(st, 1, 2) - ref)) < 1e-12 * np.max(np.abs(ref))


@pytest.mark.parametrize("kind,S", [("tube", 1), ("grid", 2), ("isolated", 33), ("grid", 50), ("fan40", 64),
                                    ("tube", 97), ("fan9", 100), ("grid", 128), ("isolated", 130)])
@pytest.mark.parametrize("symmetric", [False, True])
@pytest.mark.parametrize("by", [0, 1])
def test_assembled_rows(require_gpu, kind, S, symmetric, by):
    from cvfes_amd import _lib
    nodes, el, E, s = system(kind, S)
    coef = shifted(s.coef.cpu().numpy(), by)
    n = s.nnzu if symmetric else s.nnzb
    out = shifted(np.full((n, 9, S), np.nan), by)
    p = _lib.ptr
    if symmetric:
        _lib.check(s.lib.cvfes_assemble_upper(s.stream, n, S, p(s.ublk), p(s.cptr), p(s.celem), p(s.khat), p(coef),
                                              p(out)))
    else:
        _lib.check(s.lib.cvfes_assemble_bcsr(s.stream, n, S, p(s.cptr), p(s.celem), p(s.khat), p(coef), p(out)))
    cp, ce = s.cptr.cpu().numpy(), s.celem.cpu().numpy()
    kh, cf = s.khat.cpu().numpy().reshape(-1, 9), s.coef.cpu().numpy()
    blocks = s.ublk.cpu().numpy() if symmetric else np.arange(n)
    got = out.cpu().numpy()
    for i, b in enumerate(blocks):
        terms = kh[cp[b]:cp[b + 1], :, None] * cf[ce[cp[b]:cp[b + 1]], None, :]
        assert np.all(np.abs(got[i] - terms.sum(0)) <= 1e-14 * np.abs(terms).sum(0))


@pytest.mark.parametrize("S", [1, 2, 33, 64, 97, 100, 130])
@pytest.mark.parametrize("thick_samples,node_field,log,by", [
    (False, False, False, 0), (True, False, True, 0), (True, True, False, 1), (False, True, False, 0)])
def test_coefficient_rows(require_gpu, S, thick_samples, node_field, log, by):
    from cvfes_amd import _lib
    nodes, el, E, s = system("grid", 2)
    n, rng, p = nodes.shape[0], np.random.default_rng(S), _lib.ptr
    h = 0.07 * rng.uniform(0.5, 1.5, (n, S) if thick_samples else (n, 1))
    E = np.exp(rng.standard_normal((n if node_field else el.shape[0], S)))
    out = shifted(np.full((el.shape[0], S), np.nan), by)
    hd, Ed = shifted(h, by), shifted(np.log(E) if log else E, by)
    _lib.check(s.lib.cvfes_element_coef(s.stream, el.shape[0], S, p(s.elems), p(hd), int(thick_samples),
                                        p(Ed) if node_field else None, None if node_field else p(Ed), int(log), p(out)))
    i, j = el[:, [0, 0, 1]], el[:, [1, 2, 2]]
    Eq = 0.5 * (E[i] + E[j]) if node_field else E[:, None]
    ref = (0.5 * (h[i] + h[j]) * Eq).sum(1) / 3.0
    # a dozen roundings, and with the logarithm an argument off by an ulp and exp's own
    assert np.all(np.abs(out.cpu().numpy() - ref) <= 1e-14 * ref)
