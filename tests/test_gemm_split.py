"""fp32 products on the bf16 matrix cores (three bf16 values per fp32 one):
tile edges, partial steps of K, operand layouts, both tile sizes, split K,
and the values that the split cannot hold (recomputed with fp32 MFMAs)."""

import numpy as np
import pytest

import porch_amd as porch
from oracle import host
from tests.helpers import placeholder
from tests.kernel_emu import emulate as emu

T = porch.transpose


def ints(shape, rng):
    return rng.integers(-8, 9, size=shape).astype(np.float32)


def strided(x, rows, cols):
    # every second row and column of a larger matrix: contiguous along neither
    return x[porch.slice(0, 2 * rows, 2), porch.slice(1, 2 * cols + 1, 2)]


# name: (shapes of A, B; graph).  K = 65 .. 130 covers partial steps of 1 to
# 31 values (steps of 32) and none; extents around the 128-row tile, odd ones
# for the two-row loads along the rows.
SMALL = {
    "one row past a tile": ([129, 66], [66, 130], lambda a, b: porch.matmul(a, b)),
    "odd columns, epilogue": ([127, 97], [97, 129], lambda a, b: porch.relu(porch.matmul(a, b) - 3.0) * 0.5),
    "both transposed, odd": ([65, 131], [67, 65], lambda a, b: porch.matmul(T(a), T(b))),
    "transposed A, whole steps": ([96, 130], [96, 34], lambda a, b: porch.matmul(T(a), b)),
    "strided operands": ([140, 141], [142, 261], lambda a, b: porch.matmul(strided(a, 70, 70), strided(b, 70, 130))),
    "one column": ([2050, 130], [130, 1], lambda a, b: porch.batched_matmul(
        porch.reshape(a, [1, 2050, 130]), porch.reshape(b, [1, 130, 1]))),
    "batched, shared right side": ([3, 70, 100], [100, 35], lambda a, b: porch.batched_matmul(
        a, porch.broadcast_to(b, [3, 100, 35]))),
    "split K, partial step": ([40, 1030], [1030, 37], lambda a, b: porch.matmul(a, b) + 1.0),
}

# chunks of K with uneven numbers of steps: 17 whole ones (the fewest that are split), 16 and a partial one
UNEVEN = {"whole steps": (70, 544, 131), "partial step": (129, 515, 40), "odd K, odd columns": (33, 1001, 257)}


def build(name, make):
    sa, sb, f = SMALL[name]
    return f(make(sa), make(sb))


def filled(shape, values):
    t = placeholder(shape)
    t._state.storage = porch._Storage(None, np.ascontiguousarray(values, np.float32).reshape(-1))
    return t


@pytest.mark.skipif(not emu.available(), reason="no clang for the emulation")
@pytest.mark.parametrize("name", ["both transposed, odd", "strided operands"])
def test_emulated_products_bit_exact(name):
    rng = np.random.default_rng(1)
    sa, sb, f = SMALL[name]
    a, b = ints(sa, rng), ints(sb, rng)
    expr = f(filled(sa, a), filled(sb, b))
    assert [k["kind"] for k in porch.plan(expr)["kernels"]] == ["gemm.mfma"]
    assert all(r["ok"] for r in emu.emulate(expr, timeout=300))
    got = emu.evaluate(expr, [a, b], timeout=300)
    assert np.array_equal(got, host.evaluate(expr).reshape(got.shape))


def uneven(name, make, rng):
    m, k, n = UNEVEN[name]
    a, b, c = ints((m, k), rng), ints((k, n), rng), ints((1, n), rng)
    expr = porch.relu(porch.matmul(make(a), make(b)) + porch.broadcast_to(make(c), [m, n])) - 0.5
    assert [x["kind"] for x in porch.plan(expr)["kernels"]] == ["gemm.mfma", "gemm.combine"]
    return [a, b, c], expr


@pytest.mark.skipif(not emu.available(), reason="no clang for the emulation")
@pytest.mark.parametrize("name", sorted(UNEVEN))
def test_emulated_uneven_chunks(name):
    values, expr = uneven(name, lambda x: filled(list(x.shape), x), np.random.default_rng(7))
    assert all(r["ok"] for r in emu.emulate(expr, timeout=300))
    got = emu.evaluate(expr, values, timeout=300)
    assert np.array_equal(got, host.evaluate(expr).reshape(got.shape))


@pytest.mark.gpu
@pytest.mark.parametrize("name", sorted(UNEVEN))
def test_uneven_chunks(gpu, name):
    _, expr = uneven(name, lambda x: gpu.tensor(list(x.shape), x.reshape(-1)), np.random.default_rng(8))
    out = gpu.materialize(expr).cpu().reshape(expr.shape())
    assert np.array_equal(out, host.evaluate(expr).reshape(out.shape))


@pytest.mark.skipif(not emu.available(), reason="no clang for the emulation")
def test_emulated_large_tiles_at_the_edges():
    # 256 x 256 tiles (16 x 16 of them), a partial step of 3, ragged edges
    rng = np.random.default_rng(2)
    m, k, n = 3901, 67, 3999
    a, b = ints((m, k), rng), ints((k, n), rng)
    expr = porch.matmul(filled([m, k], a), filled([k, n], b))
    (kernel,) = porch.plan(expr)["kernels"]
    assert kernel["grid"][0] == 256
    assert emu.check_edges(expr, [a, b], host.evaluate(expr).reshape(m, n)) > 4 * 150 * 150


# Operand values past what three bf16 values hold, planted into A: the
# results are the fp32 MFMA's, in the oracle's (sequential) order here.
SPECIAL = {
    "infinity": [np.inf], "both infinities": [np.inf, -np.inf], "nan": [np.nan],
    "largest": [3.4028235e38], "rounds up to an infinite bf16": [-3.4e38],
    "denormal": [1e-40], "least denormal": [1.4e-45], "below 2^-109": [1.5e-33 * 0.9],
}


def special_inputs(name, m, k, n):
    rng = np.random.default_rng(3)
    a = rng.uniform(0.5, 2.0, size=(m, k)).astype(np.float32)
    b = rng.uniform(0.5, 2.0, size=(k, n)).astype(np.float32)
    a[1] = 0.0  # a row of its own: nothing hides the value
    for i, x in enumerate(SPECIAL[name]):
        a[1, 3 + i] = np.float32(x)
        a[2, 5 + i] = np.float32(x)
        if abs(x) > 1e30:
            b[3 + i] = 2.0 ** -20
        elif abs(x) < 1e-30:
            b[3 + i] = 2.0 ** 100
            b[3 + i, : n // 2] = 3.0
    return a, b


def check_special(got, a, b, want):
    assert np.array_equal(np.isnan(got), np.isnan(want))
    fin = np.isfinite(want)
    assert np.array_equal(got[~fin & ~np.isnan(want)], want[~fin & ~np.isnan(want)])
    a64, b64 = a.astype(np.float64), b.astype(np.float64)
    with np.errstate(invalid="ignore", over="ignore"):
        exact, scale = a64 @ b64, np.abs(a64) @ np.abs(b64)
    # K roundings of fp32, or half the least denormal where that is more
    assert np.all(np.abs(got[fin] - exact[fin]) <= (a.shape[1] * 2.0 ** -24 * scale)[fin] + 2.0 ** -150)


@pytest.mark.skipif(not emu.available(), reason="no clang for the emulation")
@pytest.mark.parametrize("name", ["both infinities", "least denormal"])
def test_emulated_special_values(name):
    m, k, n = 40, 96, 72
    a, b = special_inputs(name, m, k, n)
    expr = porch.matmul(filled([m, k], a), filled([k, n], b))
    got = emu.evaluate(expr, [a, b], timeout=300)
    check_special(got.reshape(m, n), a, b, host.evaluate(expr).reshape(m, n))


@pytest.mark.gpu
@pytest.mark.parametrize("name", sorted(SMALL))
def test_products_bit_exact_on_integers(gpu, name):
    rng = np.random.default_rng(4)
    expr = build(name, lambda s: gpu.tensor(s, ints(s, rng).reshape(-1)))
    out = gpu.materialize(expr).cpu().reshape(expr.shape())
    assert np.array_equal(out, host.evaluate(expr).reshape(out.shape))


@pytest.mark.gpu
@pytest.mark.parametrize("m, k, n, ta, tb", [(3901, 67, 3999, False, False), (3901, 80, 3999, True, True)])
def test_large_tiles_bit_exact_on_integers(gpu, m, k, n, ta, tb):
    rng = np.random.default_rng(5)
    a, b = ints((k, m) if ta else (m, k), rng), ints((n, k) if tb else (k, n), rng)
    x, y = gpu.tensor(list(a.shape), a.reshape(-1)), gpu.tensor(list(b.shape), b.reshape(-1))
    expr = porch.matmul(T(x) if ta else x, T(y) if tb else y)
    assert gpu.plan(expr)["kernels"][0]["grid"][0] == 256
    out = gpu.materialize(expr).cpu().reshape(m, n)
    want = (a.T if ta else a).astype(np.float64) @ (b.T if tb else b).astype(np.float64)
    assert np.array_equal(out, want.astype(np.float32))


@pytest.mark.gpu
@pytest.mark.parametrize("name", sorted(SPECIAL))
def test_special_values(gpu, name):
    for m, k, n in [(200, 96, 300), (130, 1100, 150)]:
        a, b = special_inputs(name, m, k, n)
        expr = porch.matmul(gpu.tensor([m, k], a.reshape(-1)), gpu.tensor([k, n], b.reshape(-1)))
        out = gpu.materialize(expr).cpu().reshape(m, n)
        check_special(out, a, b, host.evaluate(expr).reshape(m, n))


@pytest.mark.gpu
def test_tiny_values_beside_ordinary_results(gpu):
    # values below 2^-109 in a product whose results are all 2^-56 and more:
    # the split's own results, within K roundings of fp32
    rng = np.random.default_rng(6)
    m, k, n = 300, 200, 260
    a = rng.uniform(0.5, 1.0, size=(m, k)).astype(np.float32)
    a[:, 7] = 1e-38
    b = rng.uniform(0.5, 1.0, size=(k, n)).astype(np.float32)
    out = gpu.materialize(porch.matmul(gpu.tensor([m, k], a.reshape(-1)), gpu.tensor([k, n], b.reshape(-1))))
    exact = a.astype(np.float64) @ b.astype(np.float64)
    assert np.all(np.abs(out.cpu().reshape(m, n) - exact) <= k * 2.0 ** -24 * exact)


# Below 16 values of K the fp32 MFMAs: no more than K roundings.  Aligned and
# not, one tile a workgroup and persistent, 128- and 256-row tiles.
SHORT = [(1, 700, 701, False), (2, 400, 390, True), (3, 300, 512, False), (4, 256, 300, False), (7, 200, 333, True),
         (12, 180, 260, False), (15, 130, 141, True), (1, 4100, 4101, False), (4, 3900, 4000, False)]


def short_k(make, k, m, n, transposed, rng):
    a = rng.standard_normal((m, k)).astype(np.float32)
    b = rng.standard_normal((k, n)).astype(np.float32)
    y = T(make(np.ascontiguousarray(b.T))) if transposed else make(b)
    expr = porch.matmul(make(a), y)
    (kernel,) = porch.plan(expr)["kernels"]
    assert (kernel["kind"], kernel["block"]) == ("gemm.mfma", 256)
    return a, b, expr


def check_short(got, a, b):
    exact = a.astype(np.float64) @ b.astype(np.float64)
    scale = np.abs(a).astype(np.float64) @ np.abs(b).astype(np.float64)
    assert np.all(np.abs(got - exact) <= a.shape[1] * 2.0 ** -24 * scale)
    if a.shape[1] == 1:
        assert np.array_equal(got, a * b)


@pytest.mark.skipif(not emu.available(), reason="no clang for the emulation")
@pytest.mark.parametrize("case", [s for s in SHORT if s[0] in (1, 3, 15) and s[1] < 1000])
def test_emulated_short_k(case):
    a, b, expr = short_k(lambda x: filled(list(x.shape), x), *case, np.random.default_rng(9))
    assert all(r["ok"] for r in emu.emulate(expr, timeout=300))
    values = [a, np.ascontiguousarray(b.T) if case[3] else b]
    check_short(emu.evaluate(expr, values, timeout=300).reshape(case[1], case[2]), a, b)


@pytest.mark.gpu
@pytest.mark.parametrize("case", SHORT)
def test_short_k(gpu, case):
    a, b, expr = short_k(lambda x: gpu.tensor(list(x.shape), x.reshape(-1)), *case, np.random.default_rng(10))
    check_short(gpu.materialize(expr).cpu().reshape(case[1], case[2]), a, b)


def test_plans_stay_within_a_launch():
    # a launch holds fewer than 2^32 threads
    for a, b in (([1 << 23, 17, 17], [1 << 23, 17, 17]), ([(1 << 23) + 5, 33, 49], [(1 << 23) + 5, 49, 33]),
                 ([1 << 23, 9, 9], [1 << 23, 9, 9]), ([1 << 23, 10, 3], [1 << 23, 3, 10])):
        expr = porch.batched_matmul(placeholder(a), placeholder(b))
        (kernel,) = porch.plan(expr)["kernels"]
        assert kernel["kind"] == "gemm.mfma" and kernel["grid"][0] * kernel["block"] < 1 << 32


@pytest.mark.gpu
def test_more_tiles_than_512_threads_each_can_be_launched_for(gpu):
    # the same two 17 x 17 matrices for every entry, each product times a
    # value of its own
    rng = np.random.default_rng(14)
    batch = (1 << 23) + 5
    a, b = ints((1, 17, 17), rng), ints((1, 17, 17), rng)
    x = rng.integers(1, 8, size=(batch, 1, 1)).astype(np.float32)
    t = lambda v: gpu.tensor(list(v.shape), v.reshape(-1))
    product = porch.batched_matmul(porch.broadcast_to(t(a), [batch, 17, 17]), porch.broadcast_to(t(b), [batch, 17, 17]))
    expr = porch.sum(porch.sum(product * porch.broadcast_to(t(x), [batch, 17, 17]), 2), 1)
    assert any(k["kind"] == "gemm.mfma" and k["grid"][0] == batch for k in gpu.plan(expr)["kernels"])
    out = gpu.materialize(expr).cpu().reshape(batch)
    assert np.array_equal(out, x.reshape(-1) * (a[0] @ b[0]).sum())


# (batch, m, k, n, transposed B) on either side of the rule for many tiles: 256 tiles,
# K of 48, small matrices of a side of 32 and K of 256; True: fp32 MFMAs
MANY = [((256, 33, 48, 65, False), True), ((255, 33, 48, 65, False), False), ((256, 33, 49, 65, True), False),
        ((256, 32, 80, 41, False), True), ((256, 33, 80, 41, False), False), ((256, 17, 255, 43, True), True),
        ((256, 17, 257, 43, False), False), ((512, 9, 65, 201, False), True), ((1, 4097, 17, 4099, False), True),
        ((16, 31, 389, 32, True), True), ((16, 33, 389, 32, True), False)]


def many(make, size, rng):
    batch, m, k, n, transposed = size
    a, b = ints((batch, m, k), rng), ints((batch, n, k) if transposed else (batch, k, n), rng)
    y = porch.permute(make(b), [0, 2, 1]) if transposed else make(b)
    return [a, b], porch.relu(porch.batched_matmul(make(a), y) - 3.0)


@pytest.mark.parametrize("size, fp32", MANY)
def test_many_tiles_plans(size, fp32):
    _, expr = many(lambda x: placeholder(list(x.shape)), size, np.random.default_rng(11))
    (kernel,) = porch.plan(expr)["kernels"]
    assert (kernel["kind"], kernel["block"]) == ("gemm.mfma", 256 if fp32 else 512)


@pytest.mark.skipif(not emu.available(), reason="no clang for the emulation")
@pytest.mark.parametrize("size", [(256, 33, 48, 65, False), (256, 17, 255, 43, True)])
def test_emulated_many_tiles(size):
    values, expr = many(lambda x: filled(list(x.shape), x), size, np.random.default_rng(12))
    want = host.evaluate(expr).reshape(size[0], size[1], size[3])
    assert emu.check_edges(expr, values, want) == 4 * size[1] * size[3]


@pytest.mark.gpu
@pytest.mark.parametrize("size", [s for s, _ in MANY])
def test_many_tiles(gpu, size):
    _, expr = many(lambda x: gpu.tensor(list(x.shape), x.reshape(-1)), size, np.random.default_rng(13))
    out = gpu.materialize(expr).cpu().reshape(expr.shape())
    assert np.array_equal(out, host.evaluate(expr).reshape(out.shape))


# What each of the six products of parts adds, exactly: integers whose bits
# reach into the second and third bf16 value of one side, or the second of
# both, with sums below 2^24.  (name: bits of A, of B, nonzeros a column of B)
PARTS = {"three values of A": (20, 1, 7), "three values of B": (1, 20, 7), "two values of either": (11, 11, 3)}


def part_inputs(name, m, k, n, rng):
    bits_a, bits_b, nonzeros = PARTS[name]
    draw = lambda shape, bits: (rng.integers(1 << (bits - 1), 1 << bits, size=shape) * rng.choice([-1, 1], size=shape))
    a = draw((m, k), bits_a).astype(np.float32)
    b = np.zeros((k, n), np.float32)
    for j in range(n):
        b[rng.choice(k, nonzeros, replace=False), j] = draw(nonzeros, bits_b)
    return a, b


@pytest.mark.skipif(not emu.available(), reason="no clang for the emulation")
@pytest.mark.parametrize("name", sorted(PARTS))
def test_emulated_parts(name):
    a, b = part_inputs(name, 100, 70, 90, np.random.default_rng(15))
    expr = porch.matmul(filled([100, 70], a), filled([70, 90], b))
    assert porch.plan(expr)["kernels"][0]["block"] == 512
    got = emu.evaluate(expr, [a, b], timeout=300).reshape(100, 90)
    assert np.array_equal(got, (a.astype(np.float64) @ b.astype(np.float64)).astype(np.float32))


# one tile of 128 x 128, a K of one step and of 16, split K, 256 x 256 tiles
@pytest.mark.gpu
@pytest.mark.parametrize("name", sorted(PARTS))
def test_parts(gpu, name):
    for m, k, n in [(100, 70, 90), (128, 16, 130), (500, 33, 200), (40, 1030, 37), (3901, 67, 3999)]:
        a, b = part_inputs(name, m, k, n, np.random.default_rng(16))
        expr = porch.matmul(gpu.tensor([m, k], a.reshape(-1)), gpu.tensor([k, n], b.reshape(-1)))
        assert gpu.plan(expr)["kernels"][0]["block"] == 512
        got = gpu.materialize(expr).cpu().reshape(m, n)
        assert np.array_equal(got, (a.astype(np.float64) @ b.astype(np.float64)).astype(np.float32))
