"""The product-saving slice schemes (degree 8 on three products for the orders M = 5 and 7, degree 12 on
four for M = 9 and 11) against the oracle's recurrence at order M, at the edges of the dimension
classes.  Tolerance: the complex128 bar of 1e-12; the truncation differs by at most the table's own
tail (0.05 eps per slice) and the coefficients are formed from the same Bessel values."""
import numpy as np
import pytest

from oracle import equiprop_oracle as eo
from tests.helpers import gue, rel_err

pytestmark = pytest.mark.gpu

STEPS = {5: 0.004, 7: 0.03, 9: 0.1, 11: 0.3}   # tau Hnorm that the complex128 table maps to M


def problem(d, amps, pts, x, doubled):
    rng = np.random.default_rng(7000 + d)
    h = [gue(rng, d) for _ in range(amps + 1)]
    dt = x / eo.hamiltonian_norm(h[0], h[1:]) / (2 if doubled else 1)
    return h[0], h[1:], rng.uniform(-1, 1, (amps, pts)), dt


@pytest.mark.parametrize("m", sorted(STEPS))
@pytest.mark.parametrize("d, pts", [(17, 9), (32, 1030), (33, 6), (48, 65), (49, 2), (64, 1), (64, 1031)])
def test_complex128_schemes(m, d, pts):
    import parament_amd as parament
    mode = "none" if pts < 9 else "simpson" if pts < 1000 else "midpoint"
    h0, hks, c, dt = problem(d, 2, pts, STEPS[m], mode == "simpson")
    with parament.Parament("fp64") as p:
        p.set_hamiltonian(h0, *hks, quadrature_mode=mode)
        u = p.equiprop(dt, *c)
        assert p.iteration_cycles == m
    assert rel_err(u, eo.equiprop(h0, hks, c, dt, mode=mode, cycles=m)) < 1e-12


@pytest.mark.parametrize("m", sorted(STEPS))
@pytest.mark.parametrize("d, pts", [(5, 9), (65, 2), (96, 33), (100, 1), (128, 5), (129, 34)])
def test_complex128_stepwise_schemes(m, d, pts):
    """The schemes on the batched GEMMs (32- and 64-wide tiles, with and without edges)."""
    import parament_amd as parament
    mode = "simpson" if pts == 33 else "none"
    h0, hks, c, dt = problem(d, 2, pts, STEPS[m], mode == "simpson")
    with parament.Parament("fp64") as p:
        p.set_kernel_path("stepwise")
        p.set_hamiltonian(h0, *hks, quadrature_mode=mode)
        u = p.equiprop(dt, *c)
        assert p.iteration_cycles == m
    assert rel_err(u, eo.equiprop(h0, hks, c, dt, mode=mode, cycles=m)) < 1e-12


@pytest.mark.parametrize("x, m", [(0.1, 5), (0.4, 7), (0.9, 9)])
@pytest.mark.parametrize("mode", ["native", "mixed"])
@pytest.mark.parametrize("d", [40, 65, 100, 128])
def test_complex64_stepwise_schemes(x, m, mode, d):
    """The same for complex64 contexts, within the complex64 bar of 1e-5 of FP64 on the rounded inputs."""
    import parament_amd as parament
    from tests.helpers import as_c64_inputs
    h0, hks, c, dt = problem(d, 2, 33, x, False)
    with parament.Parament("fp32") as p:
        p.set_kernel_path("stepwise")
        p.set_precision_mode(mode)
        p.set_hamiltonian(h0, *hks)
        u = p.equiprop(dt, *c)
        assert p.iteration_cycles == m
    h0, hks, c = as_c64_inputs(h0, hks, c)
    assert rel_err(u, eo.equiprop(h0, hks, c, dt, cycles=m)) < 1e-5


def test_workspace_without_room_for_the_scheme():
    """The allocation-free entry point where the recurrence's three buffers fit its 256 MiB and the scheme's
    four do not: still accepted, with the same result to the complex128 bar."""
    import torch
    import parament_amd as parament
    d, pts = 128, 300   # 3 x 78.6 MB fit, 4 do not
    h0, hks, c, dt = problem(d, 1, pts, STEPS[7], False)
    carr = torch.tensor(c, dtype=torch.complex128, device="cuda")
    out = torch.empty((d, d), dtype=torch.complex128, device="cuda")
    torch.cuda.synchronize()
    with parament.Parament("fp64") as p:
        p.set_hamiltonian(h0, *hks)
        lib, args = p._lib, (dt, pts, 1)
        import ctypes
        code = lib.Parament_equipropDeviceNoAlloc_fp64(p._handle, ctypes.c_void_p(carr.data_ptr()), *args,
                                                       ctypes.c_void_p(out.data_ptr()))
        assert code == 0
        p.synchronize()
        u = out.cpu().numpy()
        assert rel_err(p.equiprop(dt, *c), u) < 1e-12


@pytest.mark.parametrize("x, m", [(0.02, 3), (0.1, 5), (0.4, 7), (0.9, 9)])
@pytest.mark.parametrize("d, n, amps", [(17, 1, 1), (31, 257, 2), (32, 1031, 3), (33, 2, 4), (63, 258, 3), (64, 4099, 2)])
def test_mixed_slice_kernel(x, m, d, n, amps):
    """The fp16 split kernel's schemes (degree 8 at M = 7, Horner's rule otherwise) at both padded sizes, with
    up to three operators loaded at once and more in a loop, every fold depth and ragged blocks;
    1e-5 of FP64 on the complex64 inputs."""
    import parament_amd as parament
    from tests.helpers import as_c64_inputs
    h0, hks, c, dt = problem(d, amps, n, x, False)
    with parament.Parament("fp32") as p:
        p.set_hamiltonian(h0, *hks)
        u = p.equiprop(dt, *c)
        assert p.iteration_cycles == m
    h0, hks, c = as_c64_inputs(h0, hks, c)
    assert rel_err(u, eo.equiprop(h0, hks, c, dt, cycles=m)) < 1e-5


SMALL = [("fp32", 1, 1, 5), ("fp32", 4, 1, 256), ("fp32", 4, 2, 257), ("fp32", 3, 3, 16385), ("fp32", 8, 4, 64),
         ("fp32", 8, 1, 65), ("fp32", 5, 5, 4097), ("fp32", 8, 2, 40000), ("fp64", 2, 1, 1), ("fp64", 4, 2, 65),
         ("fp64", 8, 1, 16), ("fp64", 8, 2, 17), ("fp64", 7, 3, 1025), ("fp64", 8, 4, 4096), ("fp64", 5, 1, 4097),
         ("fp64", 8, 1, 8200), ("fp64", 9, 2, 33), ("fp64", 16, 2, 4100)]


@pytest.mark.parametrize("prec, d, amps, n", SMALL)
@pytest.mark.parametrize("x, mode", [(0.004, "none"), (0.03, "midpoint"), (0.1, "simpson"), (0.3, "magnus"), (0.9, "none"),
                                     (1.4, "none")])
def test_small_dims(prec, d, amps, n, x, mode):
    """Dims up to 8: slices and tree in one launch, at the edges of a wave's slices, of a work-group and
    of each fold depth, with up to three operators in registers and more in LDS; dims 9 and 16 the
    padded kernel.  complex128: its bar.  complex64: the recurrence in FP32 throughout rounds its constant
    coefficients by up to 2^-23 of E = O(x) in every slice alike, which adds up linearly: 1e-5 + 2^-23 n x."""
    import parament_amd as parament
    from tests.helpers import as_c64_inputs
    doubled = mode in ("simpson", "magnus")
    pts = 2 * n + 1 if doubled else n + (mode == "midpoint")
    h0, hks, c, dt = problem(d, amps, pts, x, doubled)
    quad = "simpson" if doubled else mode
    with parament.Parament(prec) as p:
        p.set_hamiltonian(h0, *hks, quadrature_mode=quad, use_magnus=mode == "magnus")
        u = p.equiprop(dt, *c)
        m = p.iteration_cycles
    if prec == "fp32":
        h0, hks, c = as_c64_inputs(h0, hks, c)
    ref = eo.equiprop(h0, hks, c, dt, mode=quad, use_magnus=mode == "magnus", cycles=m)
    assert rel_err(u, ref) < (1e-12 if prec == "fp64" else 1e-5 + 2.0 ** -23 * n * x)


@pytest.mark.parametrize("prec, x, m", [("fp64", 0.004, 5), ("fp64", 0.03, 7), ("fp64", 0.1, 9), ("fp64", 0.3, 11),
                                        ("fp32", 0.1, 5), ("fp32", 0.4, 7), ("fp32", 0.9, 9)])
@pytest.mark.parametrize("d, n, mode", [(3, 1, "none"), (16, 34, "simpson"), (17, 2, "midpoint"), (32, 19, "none")])
def test_fused_gradient_schemes(prec, x, m, d, n, mode):
    """The derivative of the schemes in the fused gradient kernel against the block-exponential oracle: 1e-10
    of the largest entry in complex128 (the truncation is below the table's 0.05 eps per slice), 1e-4 in complex64."""
    import parament_amd as parament
    from oracle.grape_oracle import fidelity_gradient
    from parament_amd.workloads import haar_unitary
    from tests.helpers import as_c64_inputs
    pts = 2 * n + 1 if mode == "simpson" else n + (mode == "midpoint")
    h0, hks, c, dt = problem(d, 2, pts, x, mode == "simpson")
    t = haar_unitary(np.random.default_rng(d), d)
    with parament.Parament(prec) as p:
        p.set_hamiltonian(h0, *hks, quadrature_mode=mode)
        f, g = p.gate_fidelity_gradient(dt, *c, target=t)
        assert p.iteration_cycles == m
    if prec == "fp32":
        h0, hks, c = as_c64_inputs(h0, hks, c)
        c, t = c.real, t.astype(np.complex64).astype(complex)
    fr, gr = fidelity_gradient(h0, hks, c, dt, mode, t)
    tol = 1e-10 if prec == "fp64" else 1e-4
    assert abs(f - fr) < tol * max(fr, 1e-2)
    assert np.abs(g - gr).max() < tol * max(np.abs(gr).max(), 1e-3)


@pytest.mark.parametrize("prec, d, amps, n", [("fp32", 2, 1, 100), ("fp32", 4, 2, 256), ("fp32", 4, 2, 257), ("fp64", 8, 1, 256),
                                              ("fp64", 8, 1, 257), ("fp64", 64, 4, 8192), ("fp64", 64, 1, 32769),
                                              ("fp64", 65, 2, 33), ("fp32", 90, 1, 9), ("fp32", 91, 1, 9)])
def test_host_arrays(prec, d, amps, n):
    """Host-array calls at the edges of their staging (controls read in place, staged or copied, results
    written in place or copied) give the device-array call's result bit for bit, and a second call with
    other controls its own."""
    import torch
    import parament_amd as parament
    ct, rt = (torch.complex64, np.complex64) if prec == "fp32" else (torch.complex128, np.complex128)
    h0, hks, c, dt = problem(d, amps, n, 0.02, False)
    with parament.Parament(prec) as p:
        p.set_hamiltonian(h0, *hks)
        for k in (1.0, -0.5):
            block = (k * c).astype(rt)
            u = p.equiprop(dt, *block)
            carr = torch.tensor(block, dtype=ct, device="cuda")
            out = torch.empty((d, d), dtype=ct, device="cuda")
            torch.cuda.synchronize()
            p.equiprop_device(dt, carr.data_ptr(), n, amps, out.data_ptr())
            p.synchronize()
            assert np.array_equal(u, out.cpu().numpy())


@pytest.mark.parametrize("d, n", [(192, 130), (193, 70), (256, 67), (256, 63), (100, 300)])
def test_complex128_tiles(d, n):
    """The batched FP64 products on 64-wide tiles (full launches at dims from 192) and on 32-wide ones
    (narrow tree levels, smaller dims), propagator against the oracle and the gradient's two-product launches
    on full launches against chunks of eight slices: the complex128 bar."""
    import parament_amd as parament
    h0, hks, c, dt = problem(d, 2, n, 0.1, False)
    target = np.linalg.qr(gue(np.random.default_rng(d), d))[0]
    with parament.Parament("fp64") as p:
        p.set_hamiltonian(h0, *hks)
        assert rel_err(p.equiprop(dt, *c), eo.equiprop(h0, hks, c, dt, cycles=p.iteration_cycles)) < 1e-12
        f, g = p.gate_fidelity_gradient(dt, *c, target=target)
        p.set_gradient_checkpointing(0, 8)
        f8, g8 = p.gate_fidelity_gradient(dt, *c, target=target)
    assert abs(f - f8) < 1e-12 and rel_err(g, g8) < 1e-12


@pytest.mark.parametrize("x, m", [(0.4, 7), (0.9, 9)])
@pytest.mark.parametrize("d, n", [(2, 300), (40, 33), (65, 2), (100, 33)])
def test_complex64_stepwise_is_the_power_form(x, m, d, n):
    """The FP32 step-wise path evaluates the degree-M polynomial in powers of tau X whether M is the table's
    choice or set by hand, bit for bit (the product-saving schemes are less accurate in FP32)."""
    import parament_amd as parament
    h0, hks, c, dt = problem(d, 2, n, x, False)
    us = []
    for manual in (False, True):
        with parament.Parament("fp32") as p:
            p.set_kernel_path("stepwise")
            p.set_precision_mode("native")
            if manual:
                p.set_iteration_cycles(m)
            p.set_hamiltonian(h0, *hks)
            us.append(p.equiprop(dt, *c))
            assert p.iteration_cycles == m
    assert np.array_equal(*us)


@pytest.mark.parametrize("d, n", [(5, 40), (16, 1), (32, 9)])
def test_complex64_gradient_keeps_the_power_form(d, n):
    """At M = 9 the complex64 gradient evaluates the degree-9 polynomial in powers of tau X whether M is the
    table's choice or set by hand, bit for bit."""
    import parament_amd as parament
    from parament_amd.workloads import haar_unitary
    h0, hks, c, dt = problem(d, 2, n, 0.9, False)
    t = haar_unitary(np.random.default_rng(d), d)
    res = []
    for manual in (False, True):
        with parament.Parament("fp32") as p:
            if manual:
                p.set_iteration_cycles(9)
            p.set_hamiltonian(h0, *hks)
            res.append(p.gate_fidelity_gradient(dt, *c, target=t))
            assert p.iteration_cycles == 9
    assert res[0][0] == res[1][0] and np.array_equal(res[0][1], res[1][1])


@pytest.mark.parametrize("prec, d, amps, n", [("fp32", 3, 4, 50), ("fp32", 4, 7, 4097), ("fp32", 8, 16, 65), ("fp32", 8, 64, 20000),
                                              ("fp32", 5, 17, 1), ("fp64", 4, 16, 129), ("fp64", 2, 33, 300), ("fp64", 8, 64, 1030),
                                              ("fp64", 7, 20, 17)])
@pytest.mark.parametrize("mode", ["none", "midpoint", "magnus"])
def test_small_dims_many_operators(prec, d, amps, n, mode):
    """Dims up to 8 with more operators than registers hold: coefficients dealt to the lanes in full and
    partial rounds, at up to 64 of them (Magnus: as many controls as stay within 64 terms)."""
    import parament_amd as parament
    from tests.helpers import as_c64_inputs
    if mode == "magnus":
        amps = min(amps, 9)   # 9 + 9 + 36 terms
    pts = 2 * n + 1 if mode == "magnus" else n + (mode == "midpoint")
    h0, hks, c, dt = problem(d, amps, pts, 0.1, mode == "magnus")
    quad = "simpson" if mode == "magnus" else mode
    with parament.Parament(prec) as p:
        p.set_hamiltonian(h0, *hks, quadrature_mode=quad, use_magnus=mode == "magnus")
        u = p.equiprop(dt, *c)
        m = p.iteration_cycles
    if prec == "fp32":
        h0, hks, c = as_c64_inputs(h0, hks, c)
    ref = eo.equiprop(h0, hks, c, dt, mode=quad, use_magnus=mode == "magnus", cycles=m)
    assert rel_err(u, ref) < (1e-12 if prec == "fp64" else 1e-5 + 2.0 ** -23 * n * 0.1)


@pytest.mark.parametrize("prec, d", [("fp32", 2), ("fp64", 8), ("fp64", 40)])
def test_host_arrays_of_changing_length(prec, d):
    """One context over host arrays that grow and shrink, within the pinned memory's sizes, past their
    doublings and beyond them: each call the device-array call's bits."""
    import torch
    import parament_amd as parament
    ct, rt = (torch.complex64, np.complex64) if prec == "fp32" else (torch.complex128, np.complex128)
    h0, hks, c, dt = problem(d, 2, 40000, 0.02, False)
    c = c.astype(rt)
    with parament.Parament(prec) as p:
        p.set_hamiltonian(h0, *hks)
        for n in (5, 64, 65, 3, 1000, 1000, 1000, 20000, 7, 40000, 300):
            block = np.ascontiguousarray(c[:, n // 3:n // 3 + n] if n < 20000 else c[:, :n])
            u = p.equiprop(dt, *block)
            carr = torch.tensor(block, dtype=ct, device="cuda")
            out = torch.empty((d, d), dtype=ct, device="cuda")
            torch.cuda.synchronize()
            p.equiprop_device(dt, carr.data_ptr(), n, 2, out.data_ptr())
            p.synchronize()
            assert np.array_equal(u, out.cpu().numpy()), n


@pytest.mark.parametrize("d, amps, n", [(2, 1, 1), (4, 2, 257), (3, 3, 16385), (8, 2, 40000), (5, 5, 4097), (8, 4, 64)])
@pytest.mark.parametrize("x", [0.1, 0.3, 0.9, 1.4])
def test_small_dims_rounding_complex64(d, amps, n, x):
    """complex64 at dims up to 8 against the recurrence with the kernel's own FP32 constants, evaluated in 64 bits:
    what is left are the roundings of single operations, M + 2 of them a slice at 2^-24 of E = O(x), which
    differ from slice to slice (random controls) and add up as sqrt(n), twice that allowed; and the tree's, below
    2^-20 in all."""
    import parament_amd as parament
    from tests.helpers import as_c64_inputs
    h0, hks, c, dt = problem(d, amps, n, x, False)
    with parament.Parament("fp32") as p:
        p.set_hamiltonian(h0, *hks)
        u = p.equiprop(dt, *c)
        m = p.iteration_cycles
    h0, hks, c = as_c64_inputs(h0, hks, c)
    hnorm = eo.hamiltonian_norm(h0, hks)
    a = eo.bessel_coefficients(m, dt * hnorm)
    a0 = complex(np.complex64(a[0] - 1)) + 1
    a = np.concatenate([[a0], a[1:].astype(np.complex64).astype(complex)])
    s = float(np.float32(2 / hnorm))
    r = eo.clenshaw(eo.assemble(h0, hks, c), a, 2 / s)
    ref = eo.pairwise_tree(r)
    assert rel_err(u, ref) < 2 * (m + 2) * 2.0 ** -24 * x * n ** 0.5 + 2.0 ** -20


@pytest.mark.parametrize("d, n", [(192, 116), (256, 66)])
def test_complex128_tiles_gradient(d, n):
    """The gradient's two-product launches on 64-wide FP64 tiles against fourth-order differences of the oracle's
    fidelity along a random direction (truncation below 1e-12, 1e-14 / h = 1e-10 of rounding): 1e-8."""
    import parament_amd as parament
    h0, hks, c, dt = problem(d, 2, n, 0.1, False)
    rng = np.random.default_rng(d)
    with parament.Parament("fp64") as p:
        p.set_hamiltonian(h0, *hks)
        target = p.equiprop(dt, *(c + 0.5))
        f, g = p.gate_fidelity_gradient(dt, *c, target=target)
        m = p.iteration_cycles
    v, h = rng.uniform(-1, 1, c.shape), 1e-4
    fid = lambda x: abs(np.sum(target.conj() * eo.equiprop(h0, hks, x, dt, cycles=m))) ** 2 / d ** 2
    assert abs(f - fid(c)) < 1e-12
    ref = (8 * (fid(c + h * v) - fid(c - h * v)) - (fid(c + 2 * h * v) - fid(c - 2 * h * v))) / (12 * h)
    assert abs(ref) > 1e-4   # a direction in which F changes
    assert abs(np.sum(g * v) - ref) < 1e-8
