"""softmax(f(q k^T)) v in one kernel: tile remainders, operand layouts,
masks, head dimensions, the plans that take it and those that don't, and the
values its bf16 split cannot hold."""

import numpy as np
import pytest

import porch_amd as porch
from oracle import host
from tests.helpers import placeholder
from tests.kernel_emu import emulate as emu


def attention(q, k, v, scale, mask=None):
    """q [b, sq, d], k [b, sk, d], v [b, sk, d]."""
    scores = porch.batched_matmul(q, porch.permute(k, [0, 2, 1])) * scale
    if mask is not None:
        scores = scores + porch.broadcast_to(mask, scores.shape())
    return porch.batched_matmul(porch.softmax(scores, 2), v)


def reference(q, k, v, scale, mask=None):
    s = np.matmul(q.astype(np.float64), k.astype(np.float64).transpose(0, 2, 1)) * np.float64(np.float32(scale))
    if mask is not None:
        s = s + mask
    with np.errstate(invalid="ignore", over="ignore"):
        top = np.maximum(np.max(np.where(np.isnan(s), -np.inf, s), -1, keepdims=True), -np.finfo(np.float32).max)
        p = np.exp(s - top)
        p = p / p.sum(-1, keepdims=True)
        return np.matmul(p, v.astype(np.float64)), np.matmul(p, np.abs(v.astype(np.float64)))


def close(got, want, scale):
    """Sums of `dim` products inside exp, then of weights: each rounding of a
    score moves its weight by as much, relatively; 64 covers dim and the
    scores' size here (|s| up to about 8)."""
    with np.errstate(over="ignore"):
        want32 = want.astype(np.float32)
    assert np.array_equal(np.isnan(got), np.isnan(want32))
    assert np.array_equal(got[np.isinf(want32)], want32[np.isinf(want32)])
    ok = np.isfinite(want32)
    assert np.all(np.abs(got[ok] - want[ok]) <= 64 * 2.0 ** -23 * scale[ok] + 1e-37)


# (batch, queries, keys, dim, masked): around the tiles of 32 queries, of
# 128 / 64 / 32 keys (dim 32 / 64 / 128), keys of one partial tile alone,
# none, and one past; 40 entries take workgroups of eight waves
SIZES = [(1, 32, 32, 64, False), (2, 33, 64, 64, True), (1, 127, 65, 64, False), (3, 129, 200, 64, True),
         (1, 40, 130, 32, True), (2, 100, 128, 32, False), (1, 64, 33, 128, True), (2, 70, 96, 128, False),
         (40, 1000, 321, 64, False), (40, 900, 100, 128, True), (40, 900, 300, 32, False)]


def inputs(size, rng):
    b, sq, sk, d, masked = size
    q, k, v = (rng.standard_normal((b, n, d)).astype(np.float32) for n in (sq, sk, sk))
    mask = np.where(rng.random((1, sq, sk)) < 0.3, np.float32(-1e9), np.float32(0)) if masked else None
    return q, k, v, mask


def graph(make, q, k, v, mask):
    return attention(make(q), make(k), make(v), q.shape[2] ** -0.5, None if mask is None else make(mask))


def host_only(x):
    return placeholder(list(x.shape), np.ascontiguousarray(x, np.float32).reshape(-1))


def emulated(q, k, v, mask):
    expr = graph(host_only, q, k, v, mask)
    assert [x["kind"] for x in porch.plan(expr)["kernels"]] == ["attention"]
    assert all(r["ok"] for r in emu.emulate(expr, timeout=300))
    values = [q, k] + ([] if mask is None else [mask]) + [v]
    return emu.evaluate(expr, values, timeout=300)


@pytest.mark.skipif(not emu.available(), reason="no clang for the emulation")
@pytest.mark.parametrize("size", [(1, 33, 70, 64, True), (1, 32, 33, 128, False)])
def test_emulated(size):
    q, k, v, mask = inputs(size, np.random.default_rng(1))
    want, scale = reference(q, k, v, size[3] ** -0.5, mask)
    close(emulated(q, k, v, mask), want, scale)


def special(name, q, k, v, mask):
    if name == "infinite value":
        v[0, 5, 3] = np.inf
    elif name == "nan key":
        k[0, 7, 1] = np.nan
    elif name == "large values":
        v *= np.float32(1e38)
    elif name == "tiny queries and keys":
        q *= np.float32(1e-36)
        k[:] = np.where(np.abs(k) < 1.5, np.float32(0.0), k) * np.float32(1e36)
    elif name == "tiny values":
        v *= np.float32(1e-37)
    elif name == "masked rows":
        mask[0, :3] = -np.inf
    elif name == "masked to the lowest value":
        mask[0, 1] = -np.finfo(np.float32).max
        mask[0, 2, 4:] = -np.inf


SPECIAL = ["infinite value", "nan key", "large values", "tiny queries and keys", "tiny values", "masked rows",
           "masked to the lowest value"]


@pytest.mark.skipif(not emu.available(), reason="no clang for the emulation")
@pytest.mark.parametrize("name", ["infinite value", "masked rows", "tiny values"])
def test_emulated_special_values(name):
    size = (1, 34, 70, 64, True)
    q, k, v, mask = inputs(size, np.random.default_rng(2))
    special(name, q, k, v, mask)
    with np.errstate(invalid="ignore"):
        want, scale = reference(q, k, v, 0.125, mask)
    close(emulated(q, k, v, mask), want, scale)


def kinds(expr):
    return [x["kind"] for x in porch.plan(expr)["kernels"]]


def test_plans():
    P = placeholder
    d = 64
    q, k, v = P([4, 128, d]), P([4, 256, d]), P([4, 256, d])
    assert kinds(attention(q, k, v, 0.125)) == ["attention"]
    assert kinds(porch.relu(attention(q, k, v, 0.125)) + 1.0) == ["attention"]
    # rank 2, k stored transposed
    s = porch.matmul(P([64, 32]), P([32, 96])) * 0.5
    assert kinds(porch.matmul(porch.softmax(s, 1), P([96, 32]))) == ["attention"]
    # other head dimensions, fewer than 32 rows, another axis
    for shape in ([4, 128, 48], [4, 128, 256], [4, 20, 64]):
        assert "attention" not in kinds(attention(P(shape), P(shape), P(shape), 0.125))
    # as many threads as a launch holds, and more
    for batch, fused in (((1 << 23) - 1, True), (1 << 23, False)):
        shape = [batch, 32, 32]
        assert ("attention" in kinds(attention(P(shape), P(shape), P(shape), 0.125))) == fused
    s = porch.batched_matmul(q, porch.permute(k, [0, 2, 1]))
    assert "attention" not in kinds(porch.batched_matmul(porch.softmax(s, 1), v))
    # the weights or the scores are read elsewhere too
    p = porch.softmax(s, 2)
    both = porch.batched_matmul(p, v) + porch.broadcast_to(porch.sum(p, 2, True), [4, 128, d])
    assert "attention" not in kinds(both)
    both = porch.batched_matmul(p, v) + porch.broadcast_to(porch.max(s * 2.0, 2, True), [4, 128, d])
    assert "attention" not in kinds(both)
    # the weights times themselves: they are made all the same, once
    p = porch.softmax(porch.batched_matmul(P([4, 64, 64]), P([4, 64, 64])), 2)
    assert "attention" not in kinds(porch.batched_matmul(p, p))
    p = porch.softmax(porch.matmul(P([128, 128]), P([128, 128])), 1)
    assert "attention" not in kinds(porch.matmul(p, p))
    # a softmax in all but its last step
    e = porch.exp(s - porch.broadcast_to(porch.max(s, 2, True), s.shape()))
    assert "attention" not in kinds(porch.batched_matmul(e, v))


@pytest.mark.gpu
@pytest.mark.parametrize("size", SIZES)
def test_sizes(gpu, size):
    q, k, v, mask = inputs(size, np.random.default_rng(3))
    expr = graph(lambda x: gpu.tensor(list(x.shape), x.reshape(-1)), q, k, v, mask)
    assert kinds(expr) == ["attention"]
    want, scale = reference(q, k, v, size[3] ** -0.5, mask)
    close(gpu.materialize(expr).cpu().reshape(want.shape), want, scale)


@pytest.mark.gpu
@pytest.mark.parametrize("name", SPECIAL)
def test_special_values(gpu, name):
    for size in [(1, 34, 70, 64, True), (2, 200, 130, 32, True)]:
        q, k, v, mask = inputs(size, np.random.default_rng(4))
        special(name, q, k, v, mask)
        with np.errstate(invalid="ignore"):
            want, scale = reference(q, k, v, size[3] ** -0.5, mask)
        expr = graph(lambda x: gpu.tensor(list(x.shape), x.reshape(-1)), q, k, v, mask)
        assert kinds(expr) == ["attention"]
        got = gpu.materialize(expr).cpu().reshape(want.shape)
        close(got, want, scale)


def layouts(make, rng):
    """Every way a tile is read: q, k, v interleaved by heads (one read in
    place), k^T and v^T stored, and strided along both."""
    b, s, d = 2, 75, 64
    x = [rng.standard_normal((b, s, d)).astype(np.float32) for _ in range(3)]
    heads = [np.ascontiguousarray(a.transpose(1, 0, 2)) for a in x]
    yield x, [porch.permute(make(a), [1, 0, 2]) for a in heads]
    turned = [np.ascontiguousarray(a.transpose(0, 2, 1)) for a in x]
    yield x, [porch.permute(make(a), [0, 2, 1]) for a in turned]
    # two entries of three heads each, in [batch, seq, heads, dim]
    six = [rng.standard_normal((6, s, d)).astype(np.float32) for _ in range(3)]
    apart = [np.ascontiguousarray(a.reshape(2, 3, s, d).transpose(0, 2, 1, 3)) for a in six]
    yield six, [porch.reshape(porch.permute(make(a), [0, 2, 1, 3]), [6, s, d]) for a in apart]
    wide = []
    for a in x:
        w = np.zeros((b, 2 * s, 2 * d), np.float32)
        w[:, 1::2, ::2] = a
        wide.append(w)
    yield x, [make(w)[porch.all, porch.slice(1, 2 * s, 2), porch.slice(0, 2 * d, 2)] for w in wide]


def test_layouts_are_read_in_place():
    for _, views in layouts(host_only, np.random.default_rng(5)):
        assert kinds(attention(*views, 0.125)) == ["attention"]


@pytest.mark.gpu
def test_layouts(gpu):
    for x, views in layouts(lambda a: gpu.tensor(list(a.shape), a.reshape(-1)), np.random.default_rng(5)):
        want, scale = reference(*x, 0.125)
        close(gpu.materialize(attention(*views, 0.125)).cpu().reshape(want.shape), want, scale)


# (batch, queries, keys, dim, masked): past the blocks of 32 queries whose
# keys are split over waves (512 of them, 256 at dim 128): the shared tiles
SHARED = [(19, 865, 130, 64, True), (19, 865, 64, 32, False), (19, 865, 200, 32, True), (10, 831, 65, 128, False)]


@pytest.mark.gpu
@pytest.mark.parametrize("size", SHARED + [(16, 1024, 40, 64, True), (8, 1024, 100, 128, True), (1, 32, 1000, 64, True)])
def test_either_side_of_the_key_split(gpu, size):
    q, k, v, mask = inputs(size, np.random.default_rng(6))
    expr = graph(lambda x: gpu.tensor(list(x.shape), x.reshape(-1)), q, k, v, mask)
    (kernel,) = gpu.plan(expr)["kernels"]
    blocks = size[0] * -(-size[1] // 32)
    assert (kernel["grid"][0] == blocks) == (size not in SHARED)
    want, scale = reference(q, k, v, size[3] ** -0.5, mask)
    close(gpu.materialize(expr).cpu().reshape(want.shape), want, scale)


@pytest.mark.gpu
@pytest.mark.parametrize("name", SPECIAL)
def test_special_values_in_shared_tiles(gpu, name):
    size = (19, 865, 70, 64, True)
    q, k, v, mask = inputs(size, np.random.default_rng(7))
    special(name, q, k, v, mask)
    with np.errstate(invalid="ignore"):
        want, scale = reference(q, k, v, 0.125, mask)
    expr = graph(lambda x: gpu.tensor(list(x.shape), x.reshape(-1)), q, k, v, mask)
    close(gpu.materialize(expr).cpu().reshape(want.shape), want, scale)


@pytest.mark.gpu
def test_keys_masked_to_minus_infinity_for_whole_waves(gpu):
    # causal: most waves' keys weigh nothing for the first queries
    size = (2, 256, 256, 64, True)
    q, k, v, mask = inputs(size, np.random.default_rng(8))
    mask[:] = np.where(np.tri(256, dtype=bool), np.float32(0), np.float32(-np.inf))
    want, scale = reference(q, k, v, 0.125, mask)
    expr = graph(lambda x: gpu.tensor(list(x.shape), x.reshape(-1)), q, k, v, mask)
    close(gpu.materialize(expr).cpu().reshape(want.shape), want, scale)


# Products that the split cannot form, under a score function that gives a
# number for NaN (a > b ? a : b): the score is f of the fp32 product.
FUNCTIONS = {"relu": porch.relu, "at most 4": lambda s: porch.minimum(s, 4.0), "at least -4": lambda s: porch.maximum(s, -4.0)}
PRODUCTS = ["key past bf16", "query past bf16", "infinite key", "infinite query", "nan key", "products past fp32"]


def product_inputs(name, size, rng):
    q, k, v, _ = inputs((*size, False), rng)
    tiny = lambda n: (rng.uniform(0.5, 1.0, n) * rng.choice([-1.0, 1.0], n)).astype(np.float32) * np.float32(1e-31)
    if name == "key past bf16":
        q[0, :, 3] = tiny(size[1])
        k[0, 5, 3] = np.float32(3.4e38)
    elif name == "query past bf16":
        q[0, 2, 3] = np.float32(3.4e38)
        k[0, :, 3] = tiny(size[2])
    elif name == "infinite key":
        k[0, 5, 3] = -np.inf
    elif name == "infinite query":
        q[0, 2, 3] = np.inf
    elif name == "nan key":
        k[0, 5, 3] = np.nan
    else:
        q[0, 2, 3:5] = np.float32(1e30)
        k[0, 5, 3] = np.float32(1e30)
        k[0, 6, 3] = np.float32(-1e30)
        k[0, 7, 3:5] = np.float32([1e30, -1e30])
    return q, k, v


def product_graph(make, q, k, v, f):
    scores = FUNCTIONS[f](porch.batched_matmul(make(q), porch.permute(make(k), [0, 2, 1])) * 0.125)
    return porch.batched_matmul(porch.softmax(scores, 2), make(v))


def check_products(got, expr, v):
    want = host.evaluate(expr).reshape(got.shape)
    assert np.array_equal(np.isnan(got), np.isnan(want))
    ok = ~np.isnan(want)
    # as in close(), with the weights' sum of 1 bounding the scale
    assert np.all(np.abs(got[ok].astype(np.float64) - want[ok]) <= 64 * 2.0 ** -23 * np.abs(v).max())


@pytest.mark.skipif(not emu.available(), reason="no clang for the emulation")
@pytest.mark.parametrize("name", PRODUCTS)
def test_emulated_products_hidden_by_the_scores(name):
    for f in ("relu", "at most 4"):
        q, k, v = product_inputs(name, (1, 33, 40, 64), np.random.default_rng(11))
        expr = product_graph(host_only, q, k, v, f)
        assert kinds(expr) == ["attention"]
        got = emu.evaluate(expr, [q, k, v], timeout=300)
        check_products(got.reshape(v.shape[0], -1, v.shape[2]), expr, v)


@pytest.mark.skipif(not emu.available(), reason="no clang for the emulation")
def test_emulated_products_hidden_by_the_scores_in_shared_tiles():
    for name in ("key past bf16", "products past fp32"):
        q, k, v = product_inputs(name, (19, 865, 70, 64), np.random.default_rng(12))
        expr = product_graph(host_only, q, k, v, "relu")
        (kernel,) = porch.plan(expr)["kernels"]
        assert kernel["kind"] == "attention" and kernel["grid"][0] < 19 * 28
        got = emu.evaluate(expr, [q, k, v], timeout=300, only=[0])
        rows = kernel["block"] // 2  # 32 queries a wave
        got = got.reshape(v.shape[0], -1, v.shape[2])[:1, :rows]
        check_products(got, product_graph(host_only, q[:1, :rows], k[:1], v[:1], "relu"), v)


@pytest.mark.gpu
@pytest.mark.parametrize("f", sorted(FUNCTIONS))
@pytest.mark.parametrize("name", PRODUCTS)
def test_products_hidden_by_the_scores(gpu, name, f):
    for size in [(1, 33, 40, 64), (19, 865, 70, 64), (19, 865, 70, 32)]:
        q, k, v = product_inputs(name, size, np.random.default_rng(13))
        expr = product_graph(lambda x: gpu.tensor(list(x.shape), x.reshape(-1)), q, k, v, f)
        assert kinds(expr) == ["attention"]
        check_products(gpu.materialize(expr).cpu().reshape(v.shape[0], size[1], size[3]), expr, v)


# Whole rows masked with a finite value: their scores are that value (it
# absorbs them), their weights equal.  fp32 values of 2^31 and more lie 256
# and more apart, 2^369 in weights.  One value per entry: nothing else sends
# its workgroups to the fp32 MFMAs.
MASKS = [-1e9, -4.1e9, -1.26e10, -2.21e10, 4.1e9, -6e9, -3.4028235e38]


def masked_rows_graph(make, size, seed):
    q, k, v, _ = inputs((*size, False), np.random.default_rng(seed))
    mask = np.zeros((size[0], size[1], size[2]), np.float32)
    for i, x in enumerate(MASKS):
        mask[i, 0] = x          # the row
        mask[i, 1, 1::2] = x    # half of its keys
        mask[i, 2, 33:] = x     # the keys behind the first tile
        mask[i, 3, :33] = x     # and those of the first
    return (q, k, mask, v), graph(make, q, k, v, mask)


@pytest.mark.skipif(not emu.available(), reason="no clang for the emulation")
def test_emulated_rows_masked_with_finite_values():
    values, expr = masked_rows_graph(host_only, (len(MASKS), 32, 50, 64), 14)
    assert kinds(expr) == ["attention"]
    check_products(emu.evaluate(expr, values, timeout=300), expr, values[3])


@pytest.mark.gpu
def test_rows_masked_with_finite_values(gpu):
    for size in [(7, 32, 50, 64), (7, 100, 300, 64), (19, 865, 70, 64), (19, 865, 130, 32), (10, 831, 65, 128)]:
        values, expr = masked_rows_graph(lambda x: gpu.tensor(list(x.shape), x.reshape(-1)), size, 15)
        assert kinds(expr) == ["attention"]
        got = gpu.materialize(expr).cpu().reshape(size[0], size[1], size[3])
        check_products(got, expr, values[3])


def faint_inputs(size, value, seed):
    """The first key has the largest score of every query, 88 to 94 above the
    others': V is zero there, and `value` at two keys of weights around 2^-130."""
    rng = np.random.default_rng(seed)
    q, k, v, _ = inputs((*size, False), rng)
    q[:], k[:], v[:] = 0, 0, 0
    q[:, :, 0] = rng.uniform(28.0, 30.0, q.shape[:2])
    k[:, 0, 0] = 3.125 * size[3] ** 0.5
    v[:, 3, 5] = value
    v[:, size[2] - 2, 7] = -value
    return q, k, v


def check_faint(got, q, k, v):
    want, scale = reference(q, k, v, q.shape[2] ** -0.5)
    # a denormal weight's last bit, 2^-149, on top of close()'s
    assert np.all(np.abs(got - want) <= 64 * 2.0 ** -23 * scale + 2.0 ** -148 * np.abs(v).max())
    assert np.all(got[:, :, 5] != 0) and np.all(got[:, :, 7] != 0)


@pytest.mark.skipif(not emu.available(), reason="no clang for the emulation")
def test_emulated_faint_weights_of_large_values():
    for value in (2.0 ** 31, 2.0 ** 100):
        q, k, v = faint_inputs((1, 32, 70, 64), np.float32(value), 16)
        check_faint(emulated(q, k, v, None), q, k, v)


@pytest.mark.gpu
def test_faint_weights_of_large_values(gpu):
    for value in (2.0 ** 31, 2.0 ** 100):
        for size in [(1, 32, 70, 64), (19, 865, 70, 64), (19, 865, 130, 32)]:
            q, k, v = faint_inputs(size, np.float32(value), 17)
            expr = graph(lambda x: gpu.tensor(list(x.shape), x.reshape(-1)), q, k, v, None)
            check_faint(gpu.materialize(expr).cpu().reshape(q.shape), q, k, v)


# (batch, queries, keys, dim): few queries over many keys are left to the
# products and the softmax, which use every compute unit
@pytest.mark.parametrize("size, fused", [
    ((1, 32, 262144, 64), False), ((8, 32, 32768, 64), False), ((8, 256, 16384, 64), False), ((4, 1000, 40000, 128), False),
    ((1, 100, 4096, 32), False), ((64, 32, 4096, 64), True), ((16, 2048, 16384, 64), True), ((8, 256, 512, 64), True),
    ((4096, 32, 4096, 32), True), ((1, 65536, 65536, 64), True), ((8, 32, 1000, 128), False), ((8, 32, 512, 128), True),
    ((4, 1024, 1024, 128), True), ((4, 2048, 2048, 64), True), ((16, 520, 520, 32), True)])
def test_plans_of_few_queries(size, fused):
    b, sq, sk, d = size
    q, kv = placeholder([b, sq, d]), placeholder([b, sk, d])
    assert (kinds(attention(q, kv, kv, 0.125)) == ["attention"]) == fused


@pytest.mark.parametrize("size", [(1 << 22, 64, 129, 32), (1 << 23, 64, 100, 64), ((1 << 23) - 1, 33, 32, 32)])
def test_plans_of_many_queries_stay_within_a_launch(size):
    b, sq, sk, d = size
    q, kv = placeholder([b, sq, d]), placeholder([b, sk, d])
    for kernel in porch.plan(attention(q, kv, kv, 0.125))["kernels"]:
        assert kernel["grid"][0] * kernel["block"] < 1 << 32


@pytest.mark.gpu
@pytest.mark.parametrize("size, fused", [((2, 33, 6000, 64, True), False), ((1, 100, 5001, 128, False), False),
                                         ((3, 64, 4100, 32, True), False), ((1024, 32, 100, 64, False), True),
                                         ((260, 64, 300, 128, True), True), ((520, 40, 70, 128, True), False)])
def test_few_queries(gpu, size, fused):
    q, k, v, mask = inputs(size, np.random.default_rng(18))
    expr = graph(lambda x: gpu.tensor(list(x.shape), x.reshape(-1)), q, k, v, mask)
    assert (kinds(expr) == ["attention"]) == fused
    want, scale = reference(q, k, v, size[3] ** -0.5, mask)
    close(gpu.materialize(expr).cpu().reshape(want.shape), want, scale)


def part_inputs(batch, sq, dim, rng):
    """One nonzero a query and a diagonal V over `dim` keys: a score is one
    product, an output one weight times one value, all of 24 bits."""
    value = lambda *shape: (rng.uniform(0.5, 1.0, shape) * rng.choice([-1.0, 1.0], shape)).astype(np.float32)
    q = np.zeros((batch, sq, dim), np.float32)
    q[:, np.arange(sq), np.arange(sq) % dim] = value(batch, sq)
    k = value(batch, dim, dim)
    v = np.zeros((batch, dim, dim), np.float32)
    v[:, np.arange(dim), np.arange(dim)] = value(batch, dim)
    return q, k, v


def check_parts(got, q, k, v):
    # Scores of at most 1, rounded once (2^-25); a weight's exponent (up to
    # 2.9) rounded twice, exp2 within an ulp, a product and a quotient and the
    # sum of up to 128 weights of one sign: below 16 roundings.  Without
    # one of the six products of parts: 2^-18 or more.
    want, _ = reference(q, k, v, 1.0)
    nonzero = want != 0
    assert np.all(got[~nonzero] == 0)
    assert np.all(np.abs(got[nonzero] / want[nonzero] - 1) <= 16 * 2.0 ** -24)


@pytest.mark.skipif(not emu.available(), reason="no clang for the emulation")
@pytest.mark.parametrize("dim", [32, 64])
def test_emulated_parts(dim):
    q, k, v = part_inputs(1, 40, dim, np.random.default_rng(19))
    expr = attention(host_only(q), host_only(k), host_only(v), 1.0)
    assert kinds(expr) == ["attention"]
    check_parts(emu.evaluate(expr, [q, k, v], timeout=300), q, k, v)


@pytest.mark.gpu
@pytest.mark.parametrize("batch, sq, dim", [(1, 40, 32), (1, 40, 64), (1, 40, 128), (19, 865, 32), (19, 865, 64),
                                            (10, 831, 128), (40, 1000, 64)])
def test_parts(gpu, batch, sq, dim):
    q, k, v = part_inputs(batch, sq, dim, np.random.default_rng(20))
    expr = attention(*(gpu.tensor(list(x.shape), x.reshape(-1)) for x in (q, k, v)), 1.0)
    assert kinds(expr) == ["attention"]
    check_parts(gpu.materialize(expr).cpu().reshape(q.shape), q, k, v)


@pytest.mark.gpu
def test_wide_indices(gpu):
    # 2^30 scores: 64-bit indices, in shared tiles; the first, a middle and the
    # last entry
    size = (4, 16384, 16384, 32, False)
    q, k, v, _ = inputs(size, np.random.default_rng(21))
    expr = graph(lambda x: gpu.tensor(list(x.shape), x.reshape(-1)), q, k, v, None)
    assert kinds(expr) == ["attention"] and "typedef long long idx_t" in gpu.kernel_source(expr, 0)
    got = gpu.materialize(expr).cpu().reshape(q.shape)
    for b, rows in ((0, slice(0, 200)), (2, slice(8000, 8200)), (3, slice(16184, 16384))):
        want, scale = reference(q[b:b + 1, rows], k[b:b + 1], v[b:b + 1], size[3] ** -0.5)
        close(got[b:b + 1, rows], want, scale)
