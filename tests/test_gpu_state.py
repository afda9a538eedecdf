"""A call's result depends on its arguments and the context's settings, not on the calls before it."""
import numpy as np
import pytest

from oracle import equiprop_oracle as eo
from tests.helpers import gue

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("prec, x, m", [("fp64", 0.03, 7), ("fp64", 0.3, 11), ("fp32", 0.4, 7)])
@pytest.mark.parametrize("d", [5, 32])
@pytest.mark.parametrize("manual_first", [False, True])
def test_gradient_manual_and_automatic_order(prec, x, m, d, manual_first):
    """The table's order and the same order set by hand take different polynomials: after repeated
    gradients with one of them (replayed as a graph), the other gives a fresh context's bits.  Controls
    of modulus 3 put the two polynomials further apart than rounding."""
    import parament_amd as parament
    from parament_amd.workloads import haar_unitary
    rng = np.random.default_rng(40 + d)
    hs = [gue(rng, d) for _ in range(3)]
    c = rng.uniform(2, 3, (2, 40)) * rng.choice([-1, 1], (2, 40))
    dt, target = x / eo.hamiltonian_norm(hs[0], hs[1:]), haar_unitary(rng, d)

    def gradients(manual, p):
        p.set_iteration_cycles(m) if manual else p.automatic_iteration_cycles()
        for _ in range(4):
            f, g = p.gate_fidelity_gradient(dt, *c, target=target)
            assert p.iteration_cycles == m
        return f, g

    fresh = []
    for manual in (manual_first, not manual_first):
        with parament.Parament(prec) as p:
            p.set_hamiltonian(hs[0], *hs[1:])
            fresh.append(gradients(manual, p))
    with parament.Parament(prec) as p:
        p.set_hamiltonian(hs[0], *hs[1:])
        for manual, (f, g) in zip((manual_first, not manual_first, manual_first), (*fresh, fresh[0])):
            fp, gp = gradients(manual, p)
            assert fp == f and np.array_equal(gp, g)
