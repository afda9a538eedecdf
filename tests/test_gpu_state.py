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


@pytest.mark.parametrize("prec, d", [("fp32", 16), ("fp32", 33), ("fp64", 9), ("fp64", 64)])
def test_precision_mode_before_and_after_the_hamiltonian(prec, d):
    """The mixed mode gives the same bits whether it is chosen before the Hamiltonian is set, after, or again after
    calls in the other mode; a new Hamiltonian is not computed with the former one's operators."""
    import parament_amd as parament
    rng = np.random.default_rng(d)
    sets = [[gue(rng, d) for _ in range(3)] for _ in range(2)]
    c = rng.uniform(-1, 1, (2, 300))
    dt = 0.4 / eo.hamiltonian_norm(sets[0][0], sets[0][1:])
    ref = {}
    for k, hs in enumerate(sets):
        for mode in ("native", "mixed"):
            with parament.Parament(prec) as p:
                p.set_precision_mode(mode)
                p.set_hamiltonian(hs[0], *hs[1:])
                ref[k, mode] = p.equiprop(dt, *c)
    with parament.Parament(prec) as p:
        for k in (0, 1, 0):
            p.set_precision_mode("native")
            p.set_hamiltonian(sets[k][0], *sets[k][1:])
            for mode in ("mixed", "native", "mixed"):
                p.set_precision_mode(mode)
                for _ in range(3):
                    assert np.array_equal(p.equiprop(dt, *c), ref[k, mode])


def test_operators_are_padded_only_where_the_mode_reads_them():
    """120 operators of dim 64: the padded FP64 copy (7.9 MB) belongs to the mixed mode alone."""
    import torch
    import parament_amd as parament
    rng = np.random.default_rng(3)
    hs = [np.diag(rng.uniform(-1, 1, 64)) + 0j for _ in range(120)]
    used = {}
    for mode in ("mixed", "native"):
        with parament.Parament("fp64") as p:
            p.set_precision_mode(mode)
            p.set_hamiltonian(hs[0], hs[1])   # the context's first allocations
            torch.cuda.synchronize()
            free = torch.cuda.mem_get_info()[0]
            p.set_hamiltonian(hs[0], *hs[1:])
            torch.cuda.synchronize()
            used[mode] = free - torch.cuda.mem_get_info()[0]
    assert used["mixed"] - used["native"] > 5e6, used
