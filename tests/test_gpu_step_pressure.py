"""A pressure that travels with the launch (LoadTables.set_pressure) gives the bits of the same
pressure in a table, in every kernel form of the step, and the table holds it when it is read."""
import numpy as np
import pytest
import torch

from tests.test_gpu_element_rows import system

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("S,method,variant,storage", [
    (1, "stored", "auto", "full"), (16, "stored", "auto", "sym"), (33, "stored", "generic", "full"),
    (128, "stored", "auto", "sym"), (128, "stored", "rowload", "full"), (128, "stored", "lds", "full"),
    (4, "matfree", "auto", "full"), (64, "matfree", "auto", "full"), (128, "matfree", "generic", "full"),
    (128, "matfree", "lds", "full"), (128, "matfree", "cached", "full"), (6, "matfree", "ebe", "full")])
def test_pressure_with_the_launch(require_gpu, S, method, variant, storage):
    nodes, el, E, s = system("tube", S)
    s.set_storage(storage)
    s.set_variant(variant)
    u0, dt, got = 1e-4 * np.random.default_rng(S).standard_normal(3 * nodes.shape[0]), 1e-6, []
    pressures = [1.2e4, 0.0, -3.5e3]
    for deferred in (False, True):
        load = s.loads(np.zeros(1))
        s.initial_state(u0, 0.0 * u0, load, dt, beta=1e-7, damp=5.0, method=method)
        for p in pressures:
            if deferred:
                load.set_pressure(p)
            else:
                load.p.fill_(p)
            s.step(load, dt, beta=1e-7, damp=5.0, method=method)
        got.append([t.cpu() for t in s.state[:2]])
        assert float(load.p[0]) == pressures[-1]
        load.p = torch.full_like(load.p, 7.0)
        assert load.value is None and load.struct(0).p == load.p.data_ptr()
    assert all(torch.equal(a, b) and bool(a.abs().max() > 0) for a, b in zip(*got))


def test_set_pressure_is_for_one_entry(require_gpu):
    nodes, el, E, s = system("tube", 2)
    with pytest.raises(ValueError):
        s.loads(np.zeros(2)).set_pressure(1.0)
    with pytest.raises(ValueError):
        s.loads(np.zeros(1), ga=np.zeros(3 * nodes.shape[0]), qa=np.zeros(1)).set_pressure(1.0)
