"""Circuits on resident states, through the C ABI, against the oracle.

Both executors (one launch per gate, and fused tiles of up to 13 qubits in
LDS) must equal the oracle's gate-by-gate application bit for bit: every op
does the reference's arithmetic (sum over inputs in row-major order from
zero, products without FMA) on the same values in the same order.
<Z_q> is checked against numpy brute force; large states through norm
preservation and fused == per-gate.
"""
import numpy as np
import pytest
import torch

import oracle
from qtnh_amd import _lib, ops

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module", autouse=True)
def _gpu():
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    yield
    ops.tune_circuit(12)


def dev(a):
    return torch.from_numpy(np.ascontiguousarray(a, dtype=np.complex128)).cuda()


def host(t):
    torch.cuda.synchronize()
    return t.cpu().numpy()


def same_bits(a, b):
    return np.array_equal(np.asarray(a).view(np.uint64), np.asarray(b).view(np.uint64))


def rnd_state(n, seed):
    rng = np.random.default_rng(seed)
    x = rng.standard_normal(1 << n) + 1j * rng.standard_normal(1 << n)
    return x / np.linalg.norm(x)


def oracle_run(circuit, x):
    x = np.array(x, dtype=np.complex128, copy=True)
    dims = [2] * circuit.n
    for kind, q, co in circuit.ops():
        if kind == 0:
            oracle.gate_apply(x, dims, q, co, inplace=True)
        else:
            oracle.diag_apply(x, dims, q, co, inplace=True)
    return x


@pytest.mark.parametrize("n", [1, 3, 8, 12, 14, 16])
@pytest.mark.parametrize("mode", [_lib.RUN_FUSED, _lib.RUN_PER_GATE])
def test_qft_bitexact(n, mode):
    phases = np.exp(1j * np.pi / 2.0 ** np.arange(n + 1))
    x = rnd_state(n, n)
    ref = oracle.qft(x, n, phases)
    c = ops.Circuit(n).qft(phases)
    s = dev(x)
    c.run(s, mode)
    assert same_bits(host(s), ref)


def test_qft_plus_state_known_answer():
    # QFT of |+>^n is |0...0> (reference tests/gen/qft.hpp, c2-network.cpp:155-198)
    n = 12
    s = dev(np.full(1 << n, 2.0 ** (-n / 2), dtype=np.complex128))
    ops.Circuit(n).qft().run(s)
    out = host(s)
    assert abs(out[0] - 1) < 1e-12
    assert np.abs(out[1:]).max() < 1e-12


@pytest.mark.parametrize("n,depth", [(5, 6), (13, 3), (17, 2), (20, 2)])
def test_random_circuit_bitexact_both_modes(n, depth):
    c = ops.Circuit(n).random(depth, 100 + n)
    x = rnd_state(n, 7)
    ref = oracle_run(c, x)
    for mode in (_lib.RUN_FUSED, _lib.RUN_PER_GATE):
        s = dev(x)
        c.run(s, mode)
        assert same_bits(host(s), ref), mode


@pytest.mark.parametrize("tb", [3, 5, 8, 10, 11, 12, 13])
def test_every_tile_size_bitexact(tb):
    n = 15
    c = ops.Circuit(n).random(2, 5)
    # also 3-qubit dense gates and 3-qubit diagonals
    rng = np.random.default_rng(tb)
    g3 = rng.standard_normal(64) + 1j * rng.standard_normal(64)
    c.gate([14, 0, 7], g3).diag([3, 12, 1], np.exp(1j * rng.standard_normal(8))).gate([2, 9], rng.standard_normal(16))
    x = rnd_state(n, 9)
    ref = oracle_run(c, x)
    ops.tune_circuit(tb)
    try:
        s = dev(x)
        c.run(s)
        assert same_bits(host(s), ref)
    finally:
        ops.tune_circuit(12)


@pytest.mark.parametrize("mode", [3, 2, 1, 0])
def test_large_state_kernels_bitexact(mode):
    """22 qubits: 1024 tiles of 12 bits.  Register-blocked with the next tile
    in flight (3), register-blocked (2), pipelined (1) and plain (0) fused
    kernels all equal the oracle; the circuit mixes 1-, 2- and 3-qubit gates
    and diagonals on low and high qubits."""
    n = 22
    c = ops.Circuit(n).random(2, 2222)
    rng = np.random.default_rng(mode)
    g3 = rng.standard_normal(64) + 1j * rng.standard_normal(64)
    c.gate([21, 20, 19], g3).diag([0, 21, 10], np.exp(1j * rng.standard_normal(8))).gate([20, 3], rng.standard_normal(16))
    c.gate([21], [0, 1, 1, 0]).diag([18, 21], [1, 1j, -1, -1j])
    x = rnd_state(n, 22)
    ref = oracle_run(c, x)
    ops.tune_circuit_pipeline(mode)
    try:
        s = dev(x)
        c.run(s)
        assert same_bits(host(s), ref), mode
    finally:
        ops.tune_circuit_pipeline(2)


@pytest.mark.parametrize("mode,tb", [(3, 12), (2, 12), (1, 12), (0, 12), (0, 6)])
def test_diagonals_outside_the_tile_bitexact(mode, tb):
    """Diagonals on qubits outside a run's tile take the coefficient block
    those qubits select per tile.  Random unequal coefficients (so a wrong
    index order or outer bit shows) on 1-3 qubits mixing tile and outer ones,
    between layers of dense gates; every large-state kernel and a 6-bit tile."""
    n = 22
    rng = np.random.default_rng(10 * mode + tb)
    c = ops.Circuit(n)
    for layer in range(2):
        for q in range(n):
            c.gate([q], rng.standard_normal(4) + 1j * rng.standard_normal(4))
        for _ in range(10):
            k = int(rng.integers(1, 4))
            qs = [int(v) for v in rng.choice(n, k, replace=False)]
            c.diag(qs, np.exp(1j * rng.standard_normal(1 << k)) * (1 + 0.25 * rng.standard_normal(1 << k)))
    x = rnd_state(n, 23)
    ref = oracle_run(c, x)
    ops.tune_circuit(tb)
    ops.tune_circuit_pipeline(mode)
    try:
        s_ = dev(x)
        c.run(s_)
        assert same_bits(host(s_), ref), (mode, tb)
    finally:
        ops.tune_circuit(12)
        ops.tune_circuit_pipeline(2)


def test_batch_equals_individual_runs():
    sizes = [3, 9, 12, 13, 14, 16, 12, 5]
    circuits = [ops.Circuit(n).random(3, 40 + i) for i, n in enumerate(sizes)]
    xs = [rnd_state(n, 60 + i) for i, n in enumerate(sizes)]
    states = [dev(x) for x in xs]
    ops.run_batch(circuits, states)
    for c, x, s in zip(circuits, xs, states):
        assert same_bits(host(s), oracle_run(c, x))


def test_batch_rejects_aliased_states():
    c = ops.Circuit(4).random(1, 1)
    s = dev(rnd_state(4, 1))
    with pytest.raises(_lib.QtnhError):
        ops.run_batch([c, c], [s, s])


@pytest.mark.parametrize("n", [1, 4, 11, 12, 13, 18])
def test_expect_z_matches_brute_force(n):
    x = rnd_state(n, 3 * n)
    qs = list(range(n))
    got = ops.expect_z(dev(x), n, qs)
    p = np.abs(x) ** 2
    idx = np.arange(1 << n)
    for q, v in zip(qs, got):
        bit = (idx >> (n - 1 - q)) & 1
        assert abs(v - np.sum(p * (1 - 2 * bit))) < 1e-12


def test_expect_z_basis_states_exact():
    n = 14
    for x0 in (0, 1, 5000, (1 << n) - 1):
        e = np.zeros(1 << n, dtype=np.complex128)
        e[x0] = 1
        got = ops.expect_z(dev(e), n, list(range(n)))
        want = [1.0 - 2.0 * ((x0 >> (n - 1 - q)) & 1) for q in range(n)]
        assert got == want


def test_large_random_circuit_keeps_norm_and_modes_agree():
    n = 24
    c = ops.Circuit(n).random(2, 77)
    a = ops.fill_(ops.empty(1 << n), 5)
    ops.scale_(a, 1 / np.sqrt(ops.norm2(a)))
    b = a.clone()
    c.run(a, _lib.RUN_FUSED)
    c.run(b, _lib.RUN_PER_GATE)
    torch.cuda.synchronize()
    assert torch.equal(a.view(torch.float64), b.view(torch.float64))
    assert abs(ops.norm2(a) - 1) < 1e-12
    z = ops.expect_z(a, n, [0, n // 2, n - 1])
    assert all(abs(v) <= 1 for v in z)


@pytest.mark.parametrize("kind,n", [("qft", 12), ("random", 12), ("random", 16)])
def test_circuit_tune_keeps_results(kind, n):
    """A circuit tuned to its own fastest tile gives the per-gate executor's bits."""
    c = ops.Circuit(n).qft() if kind == "qft" else ops.Circuit(n).random(6, 3)
    x = rnd_state(n, 40 + n)
    want = dev(x)
    c.run(want, _lib.RUN_PER_GATE)
    tb, lb, us = c.tune()
    assert 7 <= tb <= 12 and lb in (2, 4) and us > 0
    got = dev(x)
    c.run(got, _lib.RUN_FUSED)
    assert same_bits(host(got), host(want))


def _mixed_circuit(n, n_ops, dense3, seed):
    """Random ops of every form: dense gates of 1, 2 (both qubit orders) and
    optionally 3 qubits, diagonals of 1-3, all with unequal coefficients."""
    rng = np.random.default_rng(seed)
    c = ops.Circuit(n)
    for _ in range(n_ops):
        k = int(rng.integers(1, min(n, 3) + 1))
        q = [int(v) for v in rng.choice(n, k, replace=False)]
        if rng.random() < 0.5 and (k < 3 or dense3):
            c.gate(q, (rng.standard_normal(1 << 2 * k) + 1j * rng.standard_normal(1 << 2 * k)) / (1 << k))
        else:
            c.diag(q, np.exp(1j * rng.standard_normal(1 << k)))
    return c


@pytest.mark.parametrize("dense3", [False, True])
@pytest.mark.parametrize("n,tb,low", [(4, 4, 4), (5, 12, 4), (8, 6, 2), (9, 9, 3), (11, 10, 3), (13, 11, 3),
                                      (12, 12, 4), (14, 12, 0), (15, 7, 4)])
def test_register_runs_bitexact(n, tb, low, dense3):
    """Every width of the register form (2 to 4 register bits; the smallest and
    largest tiles; tiles of less than a wave), with more ops than one staged
    chunk holds and gates on the lowest bits, where the state cannot be read
    under the first gates' register bits."""
    c = _mixed_circuit(n, 130, dense3, 100 * n + tb)
    x = rnd_state(n, n)
    ref = oracle_run(c, x)
    ops.tune_circuit(tb, low)
    try:
        s = dev(x)
        c.run(s)
        assert same_bits(host(s), ref), (n, tb, low, dense3)
    finally:
        ops.tune_circuit(12)


@pytest.mark.parametrize("dense3", [False, True])
def test_register_runs_of_several_widths_in_one_launch(dense3):
    """A batch whose circuits want different register bits and tile sizes."""
    sizes = [4, 7, 10, 11, 13, 16]
    cs = [_mixed_circuit(n, 60, dense3 and n == 11, n) for n in sizes]
    xs = [rnd_state(n, 50 + n) for n in sizes]
    refs = [oracle_run(c, x) for c, x in zip(cs, xs)]
    states = [dev(x) for x in xs]
    ops.run_batch(cs, states)
    for n, s, ref in zip(sizes, states, refs):
        assert same_bits(host(s), ref), n


@pytest.mark.parametrize("dense3", [False, True])
@pytest.mark.parametrize("sizes", [[28], [27, 26, 20]])
def test_register_runs_walk_several_tiles(sizes, dense3):
    """4-bit tiles of large states: more tiles than a launch has workgroups, so
    a workgroup takes several, of one run and of several in turn, with more ops
    than one staged chunk holds."""
    ops.tune_circuit(4, 1)
    try:
        cs = []
        for n in sizes:
            c = _mixed_circuit(n, 20, dense3, n)
            for i in range(60):  # one run, two chunks of ops
                c.diag([i % n, (i + 5) % n], np.exp(1j * np.arange(4)))
            cs.append(c)
        got = [ops.fill_(ops.empty(1 << n), n) for n in sizes]
        want = [ops.fill_(ops.empty(1 << n), n) for n in sizes]
        ops.run_batch(cs, got)
        for c, w in zip(cs, want):
            c.run(w, _lib.RUN_PER_GATE)
        for g, w in zip(got, want):
            assert torch.equal(torch.view_as_real(g).view(torch.int64), torch.view_as_real(w).view(torch.int64))
    finally:
        ops.tune_circuit(12)


def _underflowing(rng, size):
    """Nine in ten magnitudes near 1e-170, whose products underflow to zeros of
    either sign; the others ordinary."""
    x = (1e-170 * (1 + rng.random(size))) * rng.choice([-1.0, 1.0], size)
    return np.where(rng.random(size) < 0.9, x, rng.standard_normal(size))


@pytest.mark.parametrize("k", [1, 2, 3])
@pytest.mark.parametrize("tb", [4, 9, 10, 11, 12])
def test_signs_of_underflowing_products_bitexact(tb, k):
    """A gate's sums start from +0, so none is -0 whatever its products underflow
    to; diagonals after the gate and the stored state show the sign."""
    n = 13
    ops.tune_circuit(tb)
    try:
        for seed in range(4):
            rng = np.random.default_rng(seed)
            c = ops.Circuit(n)
            for _ in range(seed + 1):
                for _ in range(2):
                    c.gate([int(v) for v in rng.choice(n, k, replace=False)],
                           _underflowing(rng, 1 << 2 * k) + 1j * _underflowing(rng, 1 << 2 * k))
                c.diag([int(v) for v in rng.choice(n, 2, replace=False)], rng.choice([1, -1, 1j, -1j], 4))
            if seed == 3:
                c.gate([0], [1, 0, 0, 1])
            x = _underflowing(rng, 1 << n) + 1j * _underflowing(rng, 1 << n)
            ref = oracle_run(c, x)
            assert np.isfinite(ref.view(np.float64)).all() and (ref == 0).any()
            s = dev(x)
            c.run(s)
            assert same_bits(host(s), ref), seed
    finally:
        ops.tune_circuit(12)


@pytest.mark.parametrize("n", [9, 10, 11, 17, 18, 19, 20, 21])
def test_default_tiles_bitexact(n):
    """The tiles that the state's size picks, around the sizes where they change."""
    c = _mixed_circuit(n, 60, False, n)
    x = rnd_state(n, n)
    ref = oracle_run(c, x)
    s = dev(x)
    c.run(s)
    assert same_bits(host(s), ref)


@pytest.mark.parametrize("tb", [0, 9, 11, 12])
def test_batches_of_several_widths_bitexact(tb):
    """Circuits of several widths in one launch, under the default and set tiles."""
    sizes = [3, 4, 7, 10, 11, 13, 16]
    cs = [_mixed_circuit(n, 60, n == 13, n) for n in sizes]
    xs = [rnd_state(n, 50 + n) for n in sizes]
    refs = [oracle_run(c, x) for c, x in zip(cs, xs)]
    ops.tune_circuit(tb)
    for first in (0, 1):  # with and without a width that has no register form
        states = [dev(x) for x in xs[first:]]
        ops.run_batch(cs[first:], states)
        for n, s, ref in zip(sizes[first:], states, refs[first:]):
            assert same_bits(host(s), ref), n


def test_tuning_tries_the_untuned_tile():
    """240 gates on 12 qubits above the lowest 4: 12-bit tiles that keep no low
    bits take one run, the tuner's own shapes 30 or more."""
    n = 20
    c = ops.Circuit(n)
    for i in range(240):
        c.gate([n - 5 - i % 12], [0.6, 0.8, 0.8, -0.6])
    ops.tune_circuit(12, 0)
    assert c.info()[2] == 1
    tb, low, us = c.tune()
    assert (tb, low) == (12, 0) and us > 0
    ops.tune_circuit()
    assert c.info()[2] == 1  # the circuit keeps it


def test_ops_appended_after_runs_under_several_tiles():
    """A circuit keeps what it compiled for each tile shape; appended ops reach
    every shape, on states seen before and new ones."""
    n = 13
    c = _mixed_circuit(n, 30, True, 1)
    x = rnd_state(n, 3)
    s = dev(x)
    for more in range(3):
        for tb in (12, 8, 0, 12):
            ops.tune_circuit(tb)
            for t in (s, dev(x)):
                x0 = host(t)
                c.run(t)
                assert same_bits(host(t), oracle_run(c, x0)), (more, tb)
        c.gate([more], [0.6, 0.8, 0.8, -0.6]).diag([12, more], [1, 1j, -1, -1j])


@pytest.mark.parametrize("n,count", [(11, 8), (12, 7), (12, 8), (15, 16), (16, 16), (18, 2), (18, 4), (19, 2), (19, 4)])
def test_batch_tiles_by_all_states_bitexact(n, count):
    """The tile of a batch goes by the amplitudes of all its states; circuits that
    run alone before and after keep their own."""
    cs = [_mixed_circuit(n, 40, i == 1, i) for i in range(count)]
    want = [ops.fill_(ops.empty(1 << n), i) for i in range(count)]
    got = [w.clone() for w in want]
    for c, g, w in zip(cs, got, want):
        for _ in range(4):
            c.run(w, _lib.RUN_PER_GATE)
    cs[0].run(got[0])
    ops.run_batch(cs[1:], got[1:])
    ops.run_batch(cs, got)
    for c, g in zip(cs[1:], got[1:]):
        c.run(g)
    ops.run_batch(cs[:1], got[:1])
    ops.run_batch(cs, got)
    for g, w in zip(got, want):
        assert torch.equal(torch.view_as_real(g).view(torch.int64), torch.view_as_real(w).view(torch.int64))


@pytest.mark.parametrize("dense3", [False, True])
@pytest.mark.parametrize("n", [20, 21, 22, 23])
def test_few_and_many_tiles_bitexact(n, dense3):
    """One and two tiles for a compute unit, and more (other registers and LDS):
    every form of op, against one launch per gate."""
    c = _mixed_circuit(n, 150, dense3, n)
    got = ops.fill_(ops.empty(1 << n), n)
    want = got.clone()
    c.run(got)
    c.run(want, _lib.RUN_PER_GATE)
    assert torch.equal(torch.view_as_real(got).view(torch.int64), torch.view_as_real(want).view(torch.int64))
