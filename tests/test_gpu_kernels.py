"""Parity of the gfx950 kernels with the oracle, through the C ABI.

Bit-exact for data movement (permute, swap), seeded fill, gates and diagonal
gates (the kernels keep the reference's summation order and separate
rounding), and for small contractions (direct route).  The GEMM route is
checked at relative error <= 1e-12 (the FP64 target).
"""
import ctypes
import math
import random

import numpy as np
import pytest
import torch

import oracle
from _fixtures import contraction_cases, iden_tensor, swap_tensor
from qtnh_amd import _lib, ops

pytestmark = pytest.mark.gpu

X = _lib.X


@pytest.fixture(scope="module", autouse=True)
def _gpu():
    if not torch.cuda.is_available():
        pytest.skip("no GPU")


def dev(a):
    return torch.from_numpy(np.ascontiguousarray(a, dtype=np.complex128)).cuda()


def host(t):
    torch.cuda.synchronize()
    return t.cpu().numpy()


def rnd(n, seed):
    rng = np.random.default_rng(seed)
    return rng.standard_normal(n) + 1j * rng.standard_normal(n)


def same_bits(a, b):
    return np.array_equal(np.asarray(a).view(np.uint64), np.asarray(b).view(np.uint64))


# ------------------------------------------------------------------ fill
@pytest.mark.parametrize("dist", [0, 1])
def test_fill_matches_oracle_bitwise(dist):
    n = 100003
    for seed in (0, 1, 2 ** 63 + 5):
        x = ops.fill_(ops.empty(n), seed, dist)
        assert same_bits(host(x), oracle.fill(n, seed, dist)), (seed, dist)


# ------------------------------------------------------------------ permute
def _perm_cases():
    pyr = random.Random(5)
    cases = []
    for rank in list(range(1, 21)) + [20, 21]:
        dims = [2] * rank
        p = list(range(rank))
        pyr.shuffle(p)
        cases.append((dims, p))
    for _ in range(12):  # power-of-two dims of several widths
        rank = pyr.randint(2, 8)
        dims = [pyr.choice([1, 2, 4, 8, 16]) for _ in range(rank)]
        p = list(range(rank))
        pyr.shuffle(p)
        cases.append((dims, p))
    for _ in range(12):  # general dims
        rank = pyr.randint(1, 7)
        dims = [pyr.choice([1, 2, 3, 5, 6]) for _ in range(rank)]
        p = list(range(rank))
        pyr.shuffle(p)
        cases.append((dims, p))
    # fixed structures: reversal, rotation, identity, swap of the two lowest / highest
    for rank in (12, 18):
        cases.append(([2] * rank, list(range(rank))[::-1]))
        cases.append(([2] * rank, [(i + 1) % rank for i in range(rank)]))
        cases.append(([2] * rank, list(range(rank))))
        cases.append(([2] * rank, list(range(rank - 2)) + [rank - 1, rank - 2]))
        cases.append(([2] * rank, [1, 0] + list(range(2, rank))))
        # low source bits kept in place (the tile grows past the kept bits)
        hi = list(range(rank - 8))
        pyr.shuffle(hi)
        cases.append(([2] * rank, hi + list(range(rank - 8, rank))))
        # lowest bit exchanged with the highest
        sw = list(range(rank))
        sw[0], sw[rank - 1] = rank - 1, 0
        cases.append(([2] * rank, sw))
    return cases


def test_permute_every_tile_shape():
    """Results do not depend on the tile parameters: a random permutation, and
    ones whose natural tile is small (a rotation, the low 8 axes kept), where
    the tile grows or is filled with outer bits."""
    dims = [2] * 16
    rng = random.Random(16)
    p = list(range(16))
    rng.shuffle(p)
    hi = list(range(8))
    rng.shuffle(hi)
    x = rnd(1 << 16, 16)
    perms = [p, [(i + 1) % 16 for i in range(16)], hi + list(range(8, 16))]
    # order + 2: the tile is filled with outer bits instead of longer runs;
    # order + 4: tiles are walked by the outer bits' distance from bit 10
    shapes = [(6, 6, 12, 0, 0, 16), (4, 4, 8, 1, 1, 2), (6, 3, 9, 1, 0, 4), (3, 6, 12, 0, 1, 8), (2, 2, 4, 0, 0, 1),
              (8, 8, 12, 1, 1, 16), (6, 6, 12, 3, 1, 2), (5, 6, 11, 2, 0, 8), (4, 6, 12, 3, 1, 4), (6, 6, 10, 3, 1, 16),
              (6, 6, 12, 4, 1, 2), (5, 5, 11, 6, 1, 8)]
    try:
        for p in perms:
            ref = oracle.permute(x, dims, p)
            for a, b, u, order, nt, bpc in shapes:
                ops.tune_permute(a, b, u, order, nt, bpc)
                assert same_bits(host(ops.permute(dev(x), dims, p)), ref), (p, a, b, u, order, nt, bpc)
    finally:
        ops.tune_permute_auto(True)


def test_permute_tuning_keeps_bits():
    """Per-permutation tuning gives the default tile's bits: on the tuning call
    (candidate shapes timed into dst), on the cached call after it, and in a
    graph captured before the signature was tuned (tuning skipped), replayed
    with eager work and synchronisation between replays."""
    r = 24
    dims = [2] * r
    rng = random.Random(2400)
    rand = list(range(r))
    rng.shuffle(rand)
    low = list(range(r - 8))
    rng.shuffle(low)
    swap = list(range(r))
    swap[0], swap[r - 1] = r - 1, 0
    perms = [rand, list(range(r))[::-1], low + list(range(r - 8, r)), swap]
    x = ops.fill_(ops.empty(1 << r), 31)
    try:
        ops.tune_permute_auto(False)
        refs = [ops.permute(x, dims, p) for p in perms]
        ops.tune_permute_auto(True)
        for p, ref in zip(perms, refs):
            for rep in range(2):
                y = ops.permute(x, dims, p)
                torch.cuda.synchronize()
                assert torch.equal(torch.view_as_real(y), torch.view_as_real(ref)), (p, rep)
        ops.tune_permute_auto(True)  # forget the tuned shapes
        y = ops.empty(1 << r)
        s = torch.cuda.Stream()
        ops.context(stream=s)
        g = torch.cuda.CUDAGraph()
        with torch.cuda.graph(g, stream=s):
            ops.permute(x, dims, perms[0], out=y)
        for rep in range(3):
            ops.fill_(y, 5)
            g.replay()
            torch.cuda.synchronize()
            assert torch.equal(torch.view_as_real(y), torch.view_as_real(refs[0])), rep
    finally:
        ops.tune_permute_auto(True)


@pytest.mark.parametrize("case", _perm_cases(), ids=lambda c: "%s-%s" % (c[0][:3], c[1][:3]))
def test_permute_bitexact(case):
    dims, p = case
    n = int(np.prod(dims))
    x = rnd(n, n + len(dims))
    y = ops.permute(dev(x), dims, p)
    assert same_bits(host(y), oracle.permute(x, dims, p))


def _ragged_cases():
    rng = np.random.default_rng(15)
    cases = [([63, 65], [1, 0]), ([64, 129], [1, 0]), ([127, 3, 62], [2, 1, 0]), ([5000, 3], [1, 0]),
             ([3, 4097], [1, 0]), ([2, 3, 2, 5, 2, 7, 2, 3], [7, 5, 3, 1, 6, 4, 2, 0]), ([3] * 11, None),
             ([17, 1, 16, 9, 1], [3, 4, 0, 2, 1]), ([40, 30, 16], [1, 0, 2]), ([40, 30, 15], [1, 0, 2]),
             ([7, 11, 13, 2], [2, 0, 1, 3]), ([1, 6, 1], [2, 1, 0]), ([48, 35, 21, 22, 18], [4, 1, 3, 0, 2]),
             ([200, 300, 11], [2, 1, 0]), ([6, 0, 5], [2, 0, 1])]
    for i in range(24):
        r = int(rng.integers(2, 8))
        d = [int(v) for v in rng.integers(1, [3, 12, 40][i % 3], r)]
        while np.prod(d) > 2000000:
            d[int(np.argmax(d))] //= 2
        cases.append((d, [int(v) for v in rng.permutation(r)]))
    return [(d, p if p else [int(v) for v in rng.permutation(len(d))]) for d, p in cases]


@pytest.mark.parametrize("case", _ragged_cases(), ids=lambda c: "x".join(map(str, c[0])))
def test_permute_ragged_bitexact(case):
    """Dims that are no powers of two: cut axes with and without remainders,
    tiles from one element run to the largest, dims of 1 and 0, merged axes,
    inner axes kept (above and below the gather's line) and moved."""
    dims, ptup = case
    x = rnd(int(np.prod(dims)), len(dims))
    got = host(ops.permute(dev(x), dims, ptup))
    assert same_bits(got, oracle.permute(x, dims, ptup))


def test_permute_roundtrip_rank24():
    dims = [2] * 24
    p = list(range(24))
    random.Random(24).shuffle(p)
    inv = list(np.argsort(p))
    x = ops.fill_(ops.empty(1 << 24), 77)
    y = ops.permute(x, dims, p)
    z = ops.permute(y, ops.permuted_dims(dims, p), inv)
    torch.cuda.synchronize()
    assert torch.equal(torch.view_as_real(x), torch.view_as_real(z))


def test_permute_rejects_bad_tuple():
    """Refused by the Python front end, and by the C ABI itself."""
    x = ops.empty(8)
    y = ops.empty(8)
    with pytest.raises(ValueError):
        ops.permute(x, [2, 2, 2], [0, 1, 1])
    d, dp = ops._u64([2, 2, 2])
    p, pp = ops._u16([0, 1, 1])
    ctx = ops.context()
    st = _lib.lib().qtnh_permute_c128(ctx, ops._ptr(x), ops._ptr(y), 3, dp, pp)
    assert st == 1, st
    assert b"permutation" in _lib.lib().qtnh_ctx_last_error(ctx)


# ------------------------------------------------------------------ swap
@pytest.mark.parametrize("dims,i,j", [([2] * 10, 0, 9), ([2] * 10, 3, 4), ([2] * 12, 11, 0), ([2] * 3, 1, 2),
                                      ([4, 2, 4, 2], 0, 2), ([3, 2, 3], 0, 2), ([2, 5, 5, 2], 1, 2),
                                      ([2, 2], 1, 1)])
def test_swap_bitexact(dims, i, j):
    n = int(np.prod(dims))
    x = rnd(n, 3)
    y = ops.swap_(dev(x), dims, i, j)
    assert same_bits(host(y), oracle.swap(x, dims, i, j))


def test_swap_rejects_unequal_dims():
    with pytest.raises(_lib.QtnhError):
        ops.swap_(ops.empty(6), [2, 3], 0, 1)


# ------------------------------------------------------------------ gates
# Placements that reach every gate kernel shape: all gate bits among the lowest
# 6 (lane exchange, registers; 3-qubit: LDS-staged tiles, in any bit order),
# some low and some high (lane exchange, LDS coefficients, one or two high
# bits), all high (one thread per group).
_GATE_PLACEMENTS = {1: [[13], [0]], 2: [[13, 12], [13, 0], [0, 13], [1, 2]],
                    3: [[13, 12, 11], [13, 12, 0], [13, 0, 5], [0, 13, 11], [0, 1, 2], [7, 13, 3],
                        [13, 9, 11], [12, 13, 8]]}


@pytest.mark.parametrize("k", [1, 2, 3])
def test_gate_bitexact_binary(k):
    pyr = random.Random(k)
    rank = 14
    dims = [2] * rank
    fixed = _GATE_PLACEMENTS[k]
    for trial in range(6 + len(fixed)):
        axes = pyr.sample(range(rank), k)
        if trial == 0:
            axes = list(range(rank - k, rank))  # lowest bits
        if trial == 1:
            axes = list(range(k))               # highest bits
        if trial >= 6:
            axes = fixed[trial - 6]
        x = rnd(1 << rank, trial)
        g = rnd(4 ** k, 100 + trial)
        y = ops.gate_apply_(dev(x), dims, axes, g)
        assert same_bits(host(y), oracle.gate_apply(x, dims, axes, g)), (k, axes)


@pytest.mark.parametrize("dims,axes", [([4, 2, 4], [2, 0]), ([2, 3, 3], [1, 2]), ([3, 3, 3, 2], [0]),
                                       ([2] * 10, [1, 5, 7, 8]), ([2] * 8, [0, 2, 4, 6, 7])])
def test_gate_bitexact_general(dims, axes):
    n = int(np.prod(dims))
    K = int(np.prod([dims[a] for a in axes]))
    x = rnd(n, 9)
    g = rnd(K * K, 10)
    y = ops.gate_apply_(dev(x), dims, axes, g)
    assert same_bits(host(y), oracle.gate_apply(x, dims, axes, g))


@pytest.mark.parametrize("dims,axes", [([2] * 12, [3]), ([2] * 12, [11, 0]), ([2] * 12, [5, 6, 1]),
                                       ([2] * 12, [0, 1, 2, 3, 4, 5]), ([3, 2, 3], [0, 2]), ([4, 2, 2], [0, 2])])
def test_diag_bitexact(dims, axes):
    n = int(np.prod(dims))
    K = int(np.prod([dims[a] for a in axes]))
    x = rnd(n, 4)
    d = np.exp(1j * np.random.default_rng(1).uniform(0, 2 * np.pi, K))
    y = ops.diag_apply_(dev(x), dims, axes, d)
    assert same_bits(host(y), oracle.diag_apply(x, dims, axes, d))


def test_gate_unitary_roundtrip_rank22():
    dims = [2] * 22
    x = ops.fill_(ops.empty(1 << 22), 5)
    x0 = x.clone()
    q, _ = np.linalg.qr(rnd(16, 8).reshape(4, 4))
    g = q.T.reshape(-1)                   # [in, out] = q^T: applies q
    ops.gate_apply_(x, dims, [3, 17], g)
    ops.gate_apply_(x, dims, [3, 17], q.conj().reshape(-1))  # applies q^dagger
    torch.cuda.synchronize()
    err = (x - x0).norm().item() / x0.norm().item()
    assert err < 1e-14


# ------------------------------------------------------------------ contraction: golden vectors
def _check_case(t1, d1, t2, d2, t3, d3, wires, repls=None):
    out, dc, _ = ops.contract(dev(t1), d1, dev(t2), d2, wires, *(repls or (None, None)))
    got = host(out)
    assert dc == d3
    if repls is None:
        repls = oracle.default_repls(len(d1), 0, len(d2), 0, wires)
    ref, _ = oracle.contract(t1, d1, t2, d2, wires, *repls)
    assert same_bits(got, ref)
    np.testing.assert_allclose(got, t3, rtol=0, atol=1e-12)


@pytest.mark.parametrize("case", list(contraction_cases("dense_vals")), ids=lambda c: c[0])
def test_contract_dense_vals(case):
    name, t1, d1, t2, d2, t3, d3, wires = case
    _check_case(t1, d1, t2, d2, t3, d3, wires)


@pytest.mark.parametrize("case", list(contraction_cases("swap_vals")), ids=lambda c: c[0])
def test_contract_swap_vals(case):
    name, t1, d1, _, d2, t3, d3, wires = case
    n = d2[0]
    _check_case(t1, d1, swap_tensor(n), [n] * 4, t3, d3, wires, ops.symm_repls(len(d1), 0, 4, 0, wires))


@pytest.mark.parametrize("case", list(contraction_cases("id_vals")), ids=lambda c: c[0])
def test_contract_id_vals(case):
    name, t1, d1, _, d2, t3, d3, wires = case
    k = len(d2) // 2
    _check_case(t1, d1, iden_tensor(d2[:k]), d2, t3, d3, wires, ops.symm_repls(len(d1), 0, len(d2), 0, wires))


@pytest.mark.parametrize("group,nd1,nd2", [("mpi2r_vals", 1, 0), ("mpi3r_vals", 1, 0), ("mpi4r_vals", 1, 1),
                                           ("mpi6r_vals", 1, 1), ("mpi8r_vals", 2, 1)])
def test_contract_distributed_goldens(group, nd1, nd2):
    for name, t1, d1, t2, d2, t3, d3, wires in contraction_cases(group):
        r = ops.default_repls(len(d1), nd1, len(d2), nd2, wires)
        _check_case(t1, d1, t2, d2, t3, d3, wires, r)


# ------------------------------------------------------------------ contraction: small dense gate, outputs last
@pytest.mark.parametrize("da,db,wires", [
    ([2] * 16, [2, 2, 2, 2], [(15, 0), (3, 1)]),             # 2-qubit gate: 4 terms, 4 results per row
    ([2] * 15, [2, 2], [(0, 0)]),                             # 1-qubit gate on the top axis
    ([2] * 16, [2] * 5, [(2, 0), (9, 1), (11, 2), (4, 3)]),   # 16 terms, 2 results per row
    ([2] * 16, [2] * 5, [(14, 0)]),                           # 2 terms, 16 results per row
    ([2] * 16, [2] * 5, [(1, 0), (12, 1), (6, 2)]),           # 8 terms, 4 results per row
    ([4] * 8, [4, 4], [(5, 0)]),                              # dim-4 axes: 4 terms, 4 results
    ([4] * 7 + [2], [2, 4, 2, 2], [(7, 0), (2, 1)]),           # mixed widths: 8 terms, 4 results
])
def test_contract_small_gate_outputs_last_bitexact(da, db, wires):
    """Default placement puts the gate's open axes last: the row kernel (one
    thread per row of gate results) must equal the oracle bit for bit."""
    a = rnd(int(np.prod(da)), 11)
    b = rnd(int(np.prod(db)), 12)
    out, dc, _ = ops.contract(dev(a), da, dev(b), db, wires)
    ref, rdc = oracle.contract(a, da, b, db, wires)
    assert dc == rdc
    assert same_bits(host(out), ref)


_ROW_SHAPES = [(nb, kb) for nb in range(1, 5) for kb in range(1, 6 - nb)]


@pytest.mark.parametrize("nb,kb", _ROW_SHAPES)
def test_contract_row_kernel_every_shape_bitexact(nb, kb):
    """Every (result bits, term bits) shape of the row kernel: staged reads
    (up to 8 terms) or direct ones (16), one or two rows per thread, one or two
    result passes; contracted axes scattered over a rank-16 state (>= 12 row bits)."""
    rng = np.random.default_rng(100 * nb + kb)
    da = [2] * 16
    db = [2] * (kb + nb)
    axes = rng.choice(16, size=kb, replace=False)
    wires = [(int(a), i) for i, a in enumerate(axes)]
    a = rnd(1 << 16, 31 + nb)
    b = rnd(1 << (kb + nb), 41 + kb)
    out, dc, _ = ops.contract(dev(a), da, dev(b), db, wires)
    ref, rdc = oracle.contract(a, da, b, db, wires)
    assert dc == rdc
    assert same_bits(host(out), ref)


@pytest.mark.parametrize("rank,axes,flip", [
    (16, [15, 14], False),  # the state's two lowest bits
    (17, [0, 1], False),    # its two highest
    (18, [3, 12], True),    # mixed, the wires given in the other order (other term order)
    (20, [19, 0], True),    # lowest and highest
    (19, [6, 7], False),
    (16, [7], False),       # 1-qubit gates
    (19, [18], False),
    (19, [0], False),
    (16, [15, 14, 13], False),  # 3-qubit gates
    (18, [0, 9, 17], True),
    (17, [2, 11, 5], False),
])
def test_contract_dense_gate_fused_permute_bitexact(rank, axes, flip):
    """A square dense gate (1 to 3 term bits) contracted into a state of at
    least 2^16 elements with the default placement runs as the bit permutation
    that moves the gate's axes last, each row of results formed in the
    permute's tiles: equal to the oracle bit for bit."""
    k = len(axes)
    da, db = [2] * rank, [2] * (2 * k)
    wires = [(a, i) for i, a in enumerate(axes)]
    if flip:
        wires = wires[::-1]
    a = rnd(1 << rank, 60 + rank)
    b = rnd(1 << (2 * k), 70 + k)
    out, dc, _ = ops.contract(dev(a), da, dev(b), db, wires)
    ref, rdc = oracle.contract(a, da, b, db, wires)
    assert dc == rdc
    assert same_bits(host(out), ref)


def test_contract_small_gate_custom_placement_bitexact():
    """Gate outputs placed below the state's open axes too (not only last)."""
    da, db = [2] * 15, [2, 2, 2, 2]
    wires = [(4, 0), (10, 1)]
    # state open axes keep their order at 0..12; gate outputs go to 14 and 13 (swapped)
    open1 = [i for i in range(15) if i not in (4, 10)]
    r1 = [X] * 15
    for k, i in enumerate(open1):
        r1[i] = k
    r2 = [X, X, 14, 13]
    a = rnd(1 << 15, 21)
    b = rnd(16, 22)
    out, dc, _ = ops.contract(dev(a), da, dev(b), db, wires, r1, r2)
    ref, _ = oracle.contract(a, da, b, db, wires, r1, r2)
    assert same_bits(host(out), ref)


# ------------------------------------------------------------------ contraction: GEMM route
@pytest.mark.parametrize("da,db,wires", [
    ([2] * 16, [2] * 16, [(i + 8, i) for i in range(8)]),                          # 256x256x256, no permutes
    ([2] * 16, [2] * 16, [(0, 15), (3, 2), (9, 7), (12, 0), (5, 9), (14, 11), (7, 4), (1, 13)]),
    ([3, 5, 7, 4, 9], [4, 9, 6, 11], [(3, 0), (4, 1)]),                             # odd sizes, tile edges
    ([8, 16, 32], [32, 16, 40], [(2, 0), (1, 1)]),
    ([2] * 20, [2] * 21, [(7 + i, i) for i in range(13)]),                        # 128x256x8192: 16 depth chunks
    ([2] * 20, [2] * 20, [(8 + i, 11 - i) for i in range(12)]),                   # 256x256x4096: 8 chunks, permuted B
])
def test_contract_gemm_route(da, db, wires):
    a = rnd(int(np.prod(da)), 1)
    b = rnd(int(np.prod(db)), 2)
    out, dc, _ = ops.contract(dev(a), da, dev(b), db, wires)
    ref, rdc = oracle.contract(a, da, b, db, wires)
    got = host(out)
    assert dc == rdc
    err = np.linalg.norm(got - ref) / np.linalg.norm(ref)
    assert err < 1e-12, err


def test_contract_gemm_route_placement():
    """GEMM route with a non-natural placement: the output permute follows repl1/repl2."""
    da, db = [2] * 14, [2] * 14
    wires = [(i, 13 - i) for i in range(7)]
    rng = random.Random(3)
    perm = list(range(14))
    rng.shuffle(perm)
    # wires use t1 axes 0..6 and t2 axes 13..7; open t1 axes 7..13, open t2 axes 0..6
    r1 = [X] * 7 + perm[:7]
    r2 = perm[7:] + [X] * 7
    a = rnd(1 << 14, 5)
    b = rnd(1 << 14, 6)
    out, dc, _ = ops.contract(dev(a), da, dev(b), db, wires, r1, r2)
    ref, _ = oracle.contract(a, da, b, db, wires, r1, r2)
    err = np.linalg.norm(host(out) - ref) / np.linalg.norm(ref)
    assert err < 1e-12, err


@pytest.mark.parametrize("da,db,wires", [
    ([2] * 16, [2] * 16, [(i, i) for i in range(16)]),                   # inner product to a scalar, K = 65536
    ([2] * 15, [2] * 15, [(i, 14 - i) for i in range(15)]),              # reversed wires: permutes before the sums
    ([4, 2] + [2] * 12, [2] * 12 + [3, 2], [(2 + i, i) for i in range(12)]),  # 8 x 6 outputs, K = 4096
    ([5, 7, 9, 11, 13], [9, 13, 11, 2], [(2, 0), (3, 2), (4, 1)]),        # ragged dims, K = 1287
])
def test_contract_few_outputs_long_sums(da, db, wires):
    """Few outputs over long sums (split into ordered chunks): within 1e-12 of the oracle."""
    a = rnd(int(np.prod(da)), 11)
    b = rnd(int(np.prod(db)), 12)
    out, dc, _ = ops.contract(dev(a), da, dev(b), db, wires)
    ref, rdc = oracle.contract(a, da, b, db, wires)
    assert dc == rdc
    got = host(out)
    err = np.linalg.norm(got - ref) / np.linalg.norm(ref)
    assert err < 1e-12, err
    # deterministic: the same call gives the same bits
    out2, _, _ = ops.contract(dev(a), da, dev(b), db, wires)
    assert same_bits(host(out2), got)


def test_kernels_are_ordered_on_the_torch_stream():
    """Results are visible to torch work queued after them on the same stream,
    with no explicit synchronisation (the context runs on torch's stream)."""
    dims = [2] * 20
    p = list(range(20))[::-1]
    for _ in range(3):
        x = ops.fill_(ops.empty(1 << 20), 9)
        y = ops.permute(x, dims, p)
        z = ops.permute(y, dims, p)
        assert torch.equal(torch.view_as_real(z), torch.view_as_real(x))  # no synchronize() before this
        ops.gate_apply_(x, dims, [19], [0, 1, 1, 0])  # X gate on the last axis
        w = x.view(-1, 2).flip(1).reshape(-1)
        assert torch.equal(torch.view_as_real(w), torch.view_as_real(z))


def test_norm2_and_scale():
    x = rnd(12345, 3)
    t = dev(x)
    assert abs(ops.norm2(t) - np.vdot(x, x).real) < 1e-9
    ops.scale_(t, 0.5 - 2j)
    y = host(t)
    exp = (x.real * 0.5 - x.imag * -2.0) + 1j * (x.real * -2.0 + x.imag * 0.5)
    assert same_bits(y, exp)


@pytest.mark.parametrize("m,n,k", [(33, 1025, 33), (64, 1024, 17), (31, 65, 1040), (65, 2049, 32), (100, 700, 31),
                                   (257, 129, 47), (63, 64, 1025), (200, 300, 257), (129, 1000, 512), (96, 96, 2049),
                                   (1, 5000, 300), (5000, 2, 300), (513, 511, 49), (1500, 1400, 48)])
def test_contract_gemm_every_tile_and_depth(m, n, k):
    """Tiles of 64 x 64, 32 x 64 and 32 x 32, with and without depth chunks;
    results one below and above tile edges; depths of whole stages and of one
    term more or less.  A NaN in the last row of A and an infinity in the last
    column of B reach only that row and column (rows, columns and terms past
    the operands' ends are read again or zeroed, never mixed in)."""
    rng = np.random.default_rng(m + n + k)
    a = rng.standard_normal((m, k)) + 1j * rng.standard_normal((m, k))
    b = rng.standard_normal((k, n)) + 1j * rng.standard_normal((k, n))
    ref = a @ b
    got, _, _ = ops.contract(dev(a), [m, k], dev(b), [k, n], [(1, 0)])
    got = host(got).reshape(m, n)
    assert np.linalg.norm(got - ref) <= 1e-12 * np.linalg.norm(ref)
    a[-1, k // 2] = np.nan
    b[k - 1, -1] = np.inf
    got, _, _ = ops.contract(dev(a), [m, k], dev(b), [k, n], [(1, 0)])
    got = host(got).reshape(m, n)
    assert np.isnan(got[-1]).all() and not np.isfinite(got[:, -1]).any()
    inner = np.linalg.norm(got[:-1, :-1] - ref[:-1, :-1])
    assert inner <= 1e-12 * max(np.linalg.norm(ref[:-1, :-1]), 1e-300)


@pytest.mark.parametrize("m,n,k", [(2, 14, 5), (12, 2, 8), (9, 10, 6), (8, 8, 9), (3, 17, 5), (3, 18, 5)])
@pytest.mark.parametrize("form", ["bits", "wider"])
def test_contract_permutes_both_operands_bitwise(m, n, k, form):
    """A contraction whose operands both have to be permuted (operands below a
    tile, at and above the size that goes in one launch, axes of one and more
    bits) equals the one whose operands lie in order, bit for bit."""
    rng = np.random.default_rng(m + 100 * n)
    def split(bits):
        dims = []
        while bits:
            b = 1 if form == "bits" else min(bits, int(rng.integers(1, 4)))
            dims.append(1 << b)
            bits -= b
        return dims
    dm, dn, dk = split(m), split(n), split(k)
    A = rng.standard_normal(dm + dk) + 1j * rng.standard_normal(dm + dk)
    B = rng.standard_normal(dk + dn) + 1j * rng.standard_normal(dk + dn)
    a, b, c = len(dm), len(dn), len(dk)
    want = host(ops.contract(dev(A.reshape(-1)), dm + dk, dev(B.reshape(-1)), dk + dn, [(a + i, i) for i in range(c)])[0])
    # Open axes keep their order among themselves; the wired ones go anywhere, and
    # the wires are taken in the order of B's.
    def shuffled(no, wired):
        labels = ["o%d" % i for i in range(no)] + wired
        places = sorted(rng.choice(no + c, no, replace=False))
        out, o, w = [], iter(labels[:no]), iter(wired)
        for i in range(no + c):
            out.append(next(o) if i in places else next(w))
        return out
    wired = ["k%d" % i for i in range(c)]
    la, lb = shuffled(a, list(rng.permutation(wired))), shuffled(b, wired)
    pa = [["o%d" % i for i in range(a)].index(v) if v[0] == "o" else a + int(v[1:]) for v in la]
    pb = [c + int(v[1:]) if v[0] == "o" else int(v[1:]) for v in lb]
    At, Bt = np.ascontiguousarray(A.transpose(pa)), np.ascontiguousarray(B.transpose(pb))
    wires = [(la.index(w), lb.index(w)) for w in wired]
    got = host(ops.contract(dev(At.reshape(-1)), At.shape, dev(Bt.reshape(-1)), Bt.shape, wires)[0])
    assert np.array_equal(got.view(np.uint64), want.view(np.uint64))


@pytest.mark.parametrize("m,n,k", [
    (0, 15, 3), (16, 0, 4), (14, 1, 2), (1, 13, 4), (9, 9, 4), (10, 9, 1), (2, 17, 0),  # register tiles
    (5, 8, 3), (2, 10, 4), (12, 1, 1), (0, 0, 0), (1, 0, 3),                             # one result a thread
    (3, 3, 10), (4, 4, 9), (0, 0, 10), (1, 7, 6), (5, 5, 8), (5, 6, 9), (6, 6, 5),        # long sums
])
@pytest.mark.parametrize("widest", [1, 3])
def test_contract_direct_matches_oracle_bitwise(m, n, k, widest):
    """Direct contractions over power-of-two dims, with shuffled axes, wires and
    result placement, at the edges of the kernel's forms."""
    rng = np.random.default_rng(1000 * m + 100 * n + k)
    def split(bits):
        dims = []
        while bits:
            b = min(bits, int(rng.integers(1, widest + 1)))
            dims.append(1 << b)
            bits -= b
        return dims
    dm, dn, dk = split(m), split(n), split(k)
    a = [("m", i) for i in range(len(dm))] + [("k", i) for i in range(len(dk))]
    b = [("n", i) for i in range(len(dn))] + [("k", i) for i in range(len(dk))]
    rng.shuffle(a), rng.shuffle(b)
    a, b = [(x, int(i)) for x, i in a], [(x, int(i)) for x, i in b]
    size = {"m": dm, "n": dn, "k": dk}
    da, db = [size[x][i] for x, i in a], [size[x][i] for x, i in b]
    wires = [(a.index(("k", i)), b.index(("k", i))) for i in rng.permutation(len(dk))]
    place = iter(int(v) for v in rng.permutation(len(dm) + len(dn)))
    r1 = [X if x == "k" else next(place) for x, _ in a]
    r2 = [X if x == "k" else next(place) for x, _ in b]
    A, B = rnd(1 << (m + k), 1), rnd(1 << (n + k), 2)
    want, _ = oracle.contract(A, da, B, db, wires, r1, r2)
    got, _, _ = ops.contract(dev(A), da, dev(B), db, wires, r1, r2)
    assert same_bits(host(got), want)


@pytest.mark.parametrize("dm,dn,dk", [
    ([3], [5], [3]), ([7, 3], [2, 2], [4]), ([5], [1], [5, 3]), ([], [], [7]),
    ([3], [3], [9, 7]), ([3, 2], [3], [64]), ([1], [3, 1], [5, 13]), ([3], [1], [10, 10]),  # 63, 64, 65, 100 terms
    ([31], [33], [2, 32, 3]), ([5, 5], [41], [3, 43]), ([3], [21], [8, 125]),                # to and past 2^10 results
    ([], [3], [1023]), ([3], [], [2, 512]), ([50, 20], [61], [3, 5]), ([600], [700], [3]),
])
def test_contract_direct_ragged_matches_oracle_bitwise(dm, dn, dk):
    """Direct contractions over any dims, with shuffled axes, wires and result
    placement: remainders of four and of 64 terms, the lines between the forms."""
    rng = np.random.default_rng(len(dm) + 10 * len(dn) + 100 * sum(dk))
    a = [("m", i) for i in range(len(dm))] + [("k", i) for i in range(len(dk))]
    b = [("n", i) for i in range(len(dn))] + [("k", i) for i in range(len(dk))]
    a, b = [a[i] for i in rng.permutation(len(a))], [b[i] for i in rng.permutation(len(b))]
    size = {"m": dm, "n": dn, "k": dk}
    da, db = [size[x][i] for x, i in a], [size[x][i] for x, i in b]
    wires = [(a.index(("k", i)), b.index(("k", i))) for i in rng.permutation(len(dk))]
    place = iter(int(v) for v in rng.permutation(len(dm) + len(dn)))
    r1 = [X if x == "k" else next(place) for x, _ in a]
    r2 = [X if x == "k" else next(place) for x, _ in b]
    A, B = rnd(int(np.prod(da)), 1), rnd(int(np.prod(db)), 2)
    want, _ = oracle.contract(A, da, B, db, wires, r1, r2)
    got, _, _ = ops.contract(dev(A), da, dev(B), db, wires, r1, r2)
    assert same_bits(host(got), want)


@pytest.mark.parametrize("dims", [[2] * 3, [2] * 9, [2] * 10, [2] * 11, [4, 2, 8, 2, 4], [1, 16, 1, 64, 2], [2] * 16,
                                  [2] * 23, [2] * 24, [8, 4, 16, 2, 2, 32, 64, 8]])
def test_permute_tiles_bitwise(dims):
    """Power-of-two dims below, at and above a tile and on both sides of the
    largest tensor that is moved a tile per block."""
    x = ops.fill_(ops.empty(int(np.prod(dims))), 3)
    rng = np.random.default_rng(len(dims))
    n = len(dims)
    for p in (rng.permutation(n), rng.permutation(n), np.arange(n)[::-1], np.roll(np.arange(n), 1)):
        p = [int(v) for v in p]
        # Source index of every result element, axis by axis from the last of the result.
        left, source = torch.arange(x.numel(), device="cuda"), torch.zeros(x.numel(), dtype=torch.int64, device="cuda")
        for i in reversed([p.index(k) for k in range(n)]):
            source += left % dims[i] * int(np.prod(dims[i + 1:]))
            left = left // dims[i]
        got = ops.permute(x, dims, p)
        assert torch.equal(torch.view_as_real(got).view(torch.int64),
                           torch.view_as_real(x[source]).view(torch.int64)), p


@pytest.mark.parametrize("precision", [_lib.PREC_FP64, _lib.PREC_SPLIT])
@pytest.mark.parametrize("opened,closed", [
    ([9], [0]), ([2] * 3, [0, 3]),                   # few axes
    ([9], [1] * 30 + [0]), ([2] * 4, [0] + [2] * 25),  # more wires than the direct kernels take
    ([3] * 2 + [1] * 26, [5, 0]),                    # more result axes than they take
])
def test_contract_empty_sums(opened, closed, precision):
    """A closed dim of 0: every result is zero, whatever the axes."""
    da, db = opened + closed, closed + opened
    wires = [(len(opened) + i, i) for i in range(len(closed))]
    empty = torch.empty(0, dtype=torch.complex128, device="cuda")
    n = int(np.prod(opened)) ** 2
    out = torch.full((n,), float("nan"), dtype=torch.complex128, device="cuda")
    got, dc, err = ops.contract(empty, da, empty, db, wires, precision=precision, out=out)
    assert dc == opened + opened and err == 0.0
    assert np.array_equal(host(got).view(np.uint64), np.zeros(2 * n, dtype=np.uint64))
    out.fill_(float("nan"))
    u64, u16 = ops._u64, ops._u16
    r1, r2 = ops.default_repls(len(da), 0, len(db), 0, wires)
    args = [u64(da), u64(db), u16([v for w in wires for v in w]), u16(r1), u16(r2)]
    eta = ctypes.c_double(-1.0)
    _lib.check(_lib.lib().qtnh_contract_c128_noalloc(
        ops.context(), None, len(da), args[0][1], None, len(db), args[1][1], len(wires), args[2][1], args[3][1],
        args[4][1], ctypes.c_void_p(out.data_ptr()), precision, ctypes.byref(eta)), ops.context())
    assert eta.value == 0.0
    assert np.array_equal(host(out).view(np.uint64), np.zeros(2 * n, dtype=np.uint64))


def test_gates_beyond_one_launch_of_threads():
    """32 qubits (64 GiB), an element or a row for each of 2^32 threads: a gate
    on the lowest bit and a diagonal, on stretches over the whole state."""
    n = 32
    x = ops.fill_(ops.empty(1 << n), 5)
    at = [0, (1 << 31) - (1 << 12), 1 << 31, 3 << 30, (1 << n) - (1 << 12)]
    before = [host(x[i:i + (1 << 12)]) for i in at]
    g = rnd(4, 1)
    d = rnd(2, 2)
    ops.gate_apply_(x, [2] * n, [n - 1], g)
    ops.diag_apply_(x, [2] * n, [0], d)
    for i, b in zip(at, before):
        want = oracle.gate_apply(b, [2] * 12, [11], g)
        want = oracle.diag_apply(want, [2] * 12, [0], [d[i >> 31]] * 2)
        assert same_bits(host(x[i:i + (1 << 12)]), want), i


@pytest.mark.parametrize("short_first", [False, True])
def test_permute_axis_beyond_32_bits(short_first):
    """An axis of more than 2^32 elements beside one of 2 (128 GiB a side)."""
    d = (1 << 32) + 7
    torch.cuda.empty_cache()
    if torch.cuda.mem_get_info()[0] < 260 << 30:
        pytest.skip("needs 256 GiB of free device memory")
    dims = [2, d] if short_first else [d, 2]
    x = ops.fill_(ops.empty(2 * d), 3)
    y = ops.permute(x, dims, [1, 0])
    a, b = x.view(dims), y.view(dims[::-1])
    for i in (0, (1 << 31) - 512, (1 << 32) - 512, d - 1024):
        for j in range(2):
            s, t = (a[j, i:i + 1024], b[i:i + 1024, j]) if short_first else (a[i:i + 1024, j], b[j, i:i + 1024])
            assert torch.equal(s, t), (i, j)
    del x, y, a, b, s, t
    torch.cuda.empty_cache()


def test_contract_gemm_more_small_tiles_than_a_launch_takes():
    """2^29 rows and few columns: 32 x 32 tiles would be 2^24 workgroups of 256
    threads (a 136 GiB operand, the shortest depth of this route)."""
    m, n, k = (1 << 29) + 3, 2, 17
    torch.cuda.empty_cache()
    if torch.cuda.mem_get_info()[0] < 170 << 30:
        pytest.skip("needs 160 GiB of free device memory")
    a = ops.fill_(ops.empty(m * k), 7)
    b = rnd(k * n, 8)
    got, _, _ = ops.contract(a, [m, k], dev(b), [k, n], [(1, 0)])
    rows = a.view(m, k)
    for i in (0, (1 << 28) - 32, m // 2, m - 64):
        want = host(rows[i:i + 64]) @ b.reshape(k, n)
        assert np.linalg.norm(host(got.view(m, n)[i:i + 64]) - want) <= 1e-12 * np.linalg.norm(want), i
    del a, got, rows
    torch.cuda.empty_cache()


@pytest.mark.parametrize("da,db,wires,repl1,repl2", [
    # 2^33 elements of dims 2; the open axis of B first in the result
    ([2] * 33, [2, 2, 2, 2, 2], [(0, 0), (1, 1), (2, 3), (3, 4)], [X] * 4 + list(range(1, 30)), [X, X, 0, X, X]),
    # 3 x 2^31 elements; the open axis of B last
    ([16, 3, 1 << 27], [2, 16], [(0, 1)], [X, 0, 1], [2, X]),
    # the largest that the kernels with 32-bit offsets take
    ([2] * 32, [2, 2, 2, 2, 2], [(0, 0), (1, 1), (2, 3), (3, 4)], [X] * 4 + list(range(1, 29)), [X, X, 0, X, X]),
    ([16, 3, 89478485], [2, 16], [(0, 1)], [X, 0, 1], [2, X]),
])
def test_contract_direct_around_32_bits_bitexact(da, db, wires, repl1, repl2):
    """The direct kernels of tensors of 2^32 elements and more, against the
    oracle on stretches of the result (16 terms each, from all over A)."""
    torch.cuda.empty_cache()
    n = math.prod(da)
    if torch.cuda.mem_get_info()[0] < 160 << 30:
        pytest.skip("needs 150 GiB of free device memory")
    a = ops.fill_(ops.empty(n), 11)
    b = rnd(math.prod(db), 12)
    got, dc, _ = ops.contract(a, da, dev(b), db, wires, repl1, repl2)
    inner = n // 16  # results of each B output, consecutive elements of A for each term
    A = a.view(16, inner)
    C = got.view(2, inner) if repl2[0] == X else got.view(inner, 2)
    for i in (0, inner // 3, inner - 1024):
        piece = host(A[:, i:i + 1024].contiguous()).reshape(-1)
        if repl2[0] == X:
            ref, _ = oracle.contract(piece, [2] * 4 + [1024], b, db, wires, [X] * 4 + [1], [X, X, 0, X, X])
            part = host(C[:, i:i + 1024].contiguous()).reshape(-1)
        else:
            ref, _ = oracle.contract(piece, [16, 1024], b, db, wires, [X, 0], [1, X])
            part = host(C[i:i + 1024].contiguous()).reshape(-1)
        assert same_bits(part, np.asarray(ref).reshape(-1)), i
    del a, got, A, C
    torch.cuda.empty_cache()


@pytest.mark.parametrize("dims,ptup", [([65537, 65537], [1, 0]), ([48, 35, 81, 22, 1500], [4, 1, 3, 0, 2])])
def test_permute_ragged_beyond_32_bits(dims, ptup):
    """Boxes with 64-bit offsets (64 GiB a side), on slices of the first, the
    middle and the last index of every axis."""
    torch.cuda.empty_cache()
    if torch.cuda.mem_get_info()[0] < 150 << 30:
        pytest.skip("needs 140 GiB of free device memory")
    x = ops.fill_(ops.empty(math.prod(dims)), 4)
    y = ops.permute(x, dims, ptup)
    inv = [ptup.index(i) for i in range(len(ptup))]
    want, got = x.view(dims).permute(inv), y.view([dims[i] for i in inv])
    for axis, d in enumerate(got.shape):
        for i in (0, d // 2, d - 1):
            assert torch.equal(want.select(axis, i), got.select(axis, i)), (axis, i)
    del x, y, want, got
    torch.cuda.empty_cache()


@pytest.mark.parametrize("axes", [[3], [20], [2, 12], [5, 1], [4, 12, 19]])
def test_gate_grids_bitwise(axes):
    """A thread per group and grids that walk the state give the same bits."""
    n = 22
    g = rnd(1 << 2 * len(axes), 3)
    outs = []
    try:
        for blocks in (0, 256, 1000, 1 << 20):
            ops.tune_stream(blocks)
            x = ops.fill_(ops.empty(1 << n), 6)
            outs.append(host(ops.gate_apply_(x, [2] * n, axes, g)))
    finally:
        ops.tune_stream()
    for o in outs[1:]:
        assert same_bits(o, outs[0])
