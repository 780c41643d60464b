"""Parity of the matrix product (forward and both gradients) with the NumPy restatement of the
reference, through the C ABI and through ``Tensor.backward()``.

Bar: the convolution's -- maximum absolute error relative to the largest magnitude of the
expected array <= 1e-10 in float64, <= 2e-4 in float32 (the product runs on the convolution's
MFMA kernels; against a float64 evaluation for float32 inputs)."""

import numpy as np
import pytest

from oracle import np_oracle as ora

pytestmark = pytest.mark.gpu

TOL = {np.dtype(np.float32): 2e-4, np.dtype(np.float64): 1e-10}


@pytest.fixture(scope="module")
def abi():
    import mygrad_amd

    if not mygrad_amd.is_available():
        pytest.fail("libmygrad_hip.so / gfx950 device not available: the GPU tests need both")
    from tests import abi as module

    return module


def err(got, want):
    want = np.asarray(want, dtype=np.float64)
    scale = float(np.max(np.abs(want))) or 1.0
    return float(np.max(np.abs(np.asarray(got, dtype=np.float64) - want))) / scale


# (batch, M, K, N): vectors, ragged sizes that are no multiple of any tile, one long reduction,
# tall / wide / batched operands
SIZES = [
    (1, 1, 1, 1),
    (1, 2, 2, 2),
    (1, 1, 7, 1),
    (1, 5, 3, 1),
    (1, 1, 3, 9),
    (1, 17, 33, 65),
    (3, 17, 33, 65),
    (1, 128, 128, 128),
    (1, 200, 1000, 72),
    (1, 64, 4099, 48),
    (2, 256, 96, 300),
    (1, 1024, 64, 16),
    (5, 16, 64, 1024),
    (1, 513, 257, 255),
    # large enough, with a reduction or a row count that is no multiple of 16: zero-padded operands
    (1, 520, 1000, 700),
    (2, 300, 330, 1100),
    (1, 512, 1000, 512),
    (1, 1001, 512, 512),
]


@pytest.mark.parametrize("dtype", [np.float32, np.float64])
@pytest.mark.parametrize("batch, M, K, N", SIZES)
def test_product_and_gradients_match_the_oracle(abi, batch, M, K, N, dtype):
    dtype = np.dtype(dtype)
    rng = np.random.default_rng([batch, M, K, N])
    a = rng.standard_normal((M, K)).astype(dtype)
    x = rng.standard_normal((batch, K, N)).astype(dtype)
    g = rng.standard_normal((batch, M, N)).astype(dtype)
    wide = [v.astype(np.float64) for v in (a, x, g)]
    assert err(abi.matmul(a, x), ora.matmul_forward(wide[0], wide[1])) <= TOL[dtype]
    assert err(abi.matmul_da(g, x, M), ora.matmul_backward(wide[2], wide[0], wide[1], 0)) <= TOL[dtype]
    assert err(abi.matmul_dx(g, a), ora.matmul_backward(wide[2], wide[0], wide[1], 1)) <= TOL[dtype]


def test_results_repeat_exactly(abi):
    rng = np.random.default_rng(3)
    a = rng.standard_normal((96, 500)).astype(np.float32)
    x = rng.standard_normal((4, 500, 130)).astype(np.float32)
    g = rng.standard_normal((4, 96, 130)).astype(np.float32)
    for fn, args in ((abi.matmul, (a, x)), (abi.matmul_da, (g, x, 96)), (abi.matmul_dx, (g, a))):
        assert np.array_equal(fn(*args), fn(*args))


# (batch, M, K, N) of products on three bf16 parts: one value; one past, and short of, a panel of 128, a tile of 256 and a K step of 32, with
# octets that end early; whole rounds of tiles and a rest that blocks share; batches along the columns and along the terms
PARTS = [(1, 1, 1, 1), (1, 129, 31, 257), (1, 255, 33, 127), (2, 100, 65, 515), (3, 300, 129, 77), (1, 384, 1000, 640), (1, 4200, 40, 4100), (1, 96, 5000, 70)]


@pytest.mark.parametrize("batch, M, K, N", PARTS)
def test_large_products_on_three_bf16_parts(abi, monkeypatch, batch, M, K, N):
    from mygrad_amd import _hip

    rng = np.random.default_rng([7, batch, M, K, N])

    def run(a, x, g, parts=True):
        monkeypatch.setenv("MYGRAD_HIP_SPLIT", "1" if parts else "0")
        monkeypatch.setenv("MYGRAD_HIP_SPLIT_MIN", "0")
        results = []
        for fn, args in ((abi.matmul, (a, x)), (abi.matmul_da, (g, x, M)), (abi.matmul_dx, (g, a))):
            results.append(fn(*args))
            assert ("three bf16 parts" in _hip.last_plan()) == parts
        return results

    def exact(a, x, g):
        a, x, g = (v.astype(np.float64) for v in (a, x, g))
        return a @ x, sum(g[b] @ x[b].T for b in range(batch)), a.T @ g

    normal = lambda *shape: rng.standard_normal(shape).astype(np.float32)
    a, x, g = normal(M, K), normal(batch, K, N), normal(batch, M, N)
    # small integers: every sum is exact, and no value of a neighbour is in it
    ints = [rng.integers(-2, 3, v.shape).astype(np.float32) for v in (a, x, g)]
    whole = run(*ints)
    for got, ref in zip(whole, exact(*ints)):
        assert np.array_equal(got, ref)
    # a sum of large products rounds off once in 32 terms, 5.06e-8 of itself as it stands then (cut off towards zero: 2^-23 * E[m^-2]^1/2 /
    # 3^1/2, significands m spread evenly in their logarithm), what is left out of it and the last roundings 3.5e-8
    plain, refs, terms = run(a, x, g, parts=False), exact(a, x, g), (K, batch * N, M)
    for got, single, ref, count in zip(run(a, x, g), plain, refs, terms):
        off = np.linalg.norm(got - ref)
        assert off <= (1.25 * 5.06e-8 * np.sqrt(-(-count // 32) / 2) + 3.5e-8) * np.linalg.norm(ref)
        # no further off than the single-precision instruction, which rounds once in a term
        assert count < 30 or off <= np.linalg.norm(single - ref)
    # one product a sum, the low bits of an operand below the smallest number of bf16 or not: what the six products leave out is 2^-24 of
    # it, the five small ones round off 2^-29 each and the last sum 2^-24
    few = np.zeros_like(a)
    few[np.arange(min(M, K)), np.arange(min(M, K))] = rng.uniform(1, 2, min(M, K))
    for tiny, other in ((1.0, 1.0), (1e-41, 3e4), (1e-38, 3e4), (1e-35, 3e36)):
        for left, right in ((tiny, other), (other, tiny)):
            args = few * np.float32(left), x * np.float32(right), g * np.float32(right)
            for i in (0, 2):
                got, ref = run(*args)[i], exact(*args)[i]
                assert np.all(np.abs(got - ref) <= (2 + 5 / 32) * 2.0**-24 * np.abs(ref) + 2.0**-149)
    # one value of low bits that parts lose, in the last row and column: no sum can tell, and all stay on the parts
    for which in range(3):
        args = [v.copy() for v in (a, x, g)]
        where = tuple(n - 1 for n in args[which].shape)
        args[which][where] = 0
        without = run(*args)
        args[which][where] = 1e-36
        for got, was, count in zip(run(*args), without, terms):
            assert count < 100 or np.array_equal(got.view(np.uint32), was.view(np.uint32))
    # infinities, NaN and sums that overflow are those of single precision
    for value in (np.inf, np.nan, 3e38):
        odd = [v.copy() for v in (a * np.float32(4), x, g)]
        for v in odd[1:]:
            v[0, 0, 0] = value
        odd[0][-1, -1] = value
        with np.errstate(all="ignore"):
            for got, single in zip(run(*odd), run(*odd, parts=False)):
                finite = np.isfinite(single)
                assert not finite.all() and np.array_equal(got[~finite], single[~finite], equal_nan=True)
                assert np.all(np.isfinite(got[finite]))
    for got, was in zip(run(*ints), whole):
        assert np.array_equal(got, was)


@pytest.mark.parametrize("sizes, parts", [((4096, 4096, 1024), (True, True, True)), ((1411, 3000, 3000), (True, True, True)),
                                          ((72, 8611, 3924), (False, False, False)), ((1024, 1024, 1024), (False, False, False)),
                                          ((4096, 24, 8192), (False, False, False)),
                                          # stacks: a run of `a`'s gradient has no more terms than a matrix has columns, and is padded to eight on parts
                                          ((1024, 1024, 1, 8192), (True, False, True)), ((4096, 4096, 1, 64), (False, False, False)),
                                          ((1024, 1024, 2, 4096), (True, False, True)), ((1024, 1024, 9, 2048), (True, False, True)),
                                          ((2000, 2000, 33, 64), (True, True, True))])
def test_which_products_run_on_three_bf16_parts(abi, sizes, parts):
    from mygrad_amd import _hip

    M, K, N, batch = (*sizes, 1)[:4]
    a, x, g = (np.ones(shape, np.float32) for shape in ((M, K), (batch, K, N), (batch, M, N)))
    for fn, args, terms, expected in zip((abi.matmul, abi.matmul_da, abi.matmul_dx), ((a, x), (g, x, M), (g, a)), (K, batch * N, M), parts):
        assert np.all(fn(*args) == terms)
        assert ("three bf16 parts" in _hip.last_plan()) == expected


def test_benchmark_prices_products_on_parts_against_their_own_peak():
    import bench

    kernels = bench.run_gpu("mm4k", 2, 1, prewarm=0.0)["kernels"]
    assert all(0 < kernels[key]["frac"] < 1 for key in ("conv_fwd", "conv_dgrad", "conv_wgrad")), kernels


BATCHED = [(1, 1, 1, 1), (3, 16, 16, 16), (5, 17, 3, 33), (2, 1, 70, 1), (300, 8, 8, 8), (7, 64, 40, 48), (4, 33, 6, 2), (2, 5, 0, 4),
           (3, 100, 129, 50),
           # 32 x 32 results or more per pair: 64 x 64 tiles staged in LDS -- whole tiles, ragged edges in M, N
           # and K, several K chunks, row lengths that are and are not whole 16-byte pieces
           (9, 64, 64, 64), (3, 130, 70, 96), (2, 32, 200, 32), (5, 47, 33, 61), (2, 128, 64, 192),
           # tiles of 128 x 32 and 32 x 128, one past a wavefront's part, a K of one and of one past a chunk, nine blocks
           (2, 127, 33, 32), (3, 31, 65, 129), (1, 33, 1, 33), (2, 17, 17, 97), (9, 65, 32, 33)]


@pytest.mark.parametrize("dtype", [np.float32, np.float64])
@pytest.mark.parametrize("batch, M, K, N", BATCHED)
def test_batched_product_with_and_without_transposed_operands(abi, batch, M, K, N, dtype):
    """mg_matmul_batched against float64 products of the same values, to the bar of the other
    matrix products (max abs error over the largest |entry|: 2e-4 float32, 1e-10 float64)."""
    dtype = np.dtype(dtype)
    rng = np.random.default_rng([batch, M, K, N])
    a, b = rng.standard_normal((batch, M, K)).astype(dtype), rng.standard_normal((batch, K, N)).astype(dtype)
    want = np.matmul(a.astype(np.float64), b.astype(np.float64))
    at, bt = np.ascontiguousarray(a.transpose(0, 2, 1)), np.ascontiguousarray(b.transpose(0, 2, 1))
    for ta, tb in ((False, False), (True, False), (False, True), (True, True)):
        got = abi.matmul_batched(at if ta else a, bt if tb else b, ta, tb)
        assert got.shape == want.shape and got.dtype == dtype
        assert err(got, want) <= TOL[dtype], (ta, tb)
    if K:  # a column and a row of the result must not see their neighbours: exact small integers
        ai, bi = np.round(a * 2), np.round(b * 2)
        assert np.array_equal(abi.matmul_batched(ai, bi), np.matmul(ai, bi))


@pytest.mark.parametrize("dtype", [np.float32, np.float64])
@pytest.mark.parametrize("tile", ["32,0", "64,0", "128,0", "32,1", "64,1", "128,1"])
def test_every_staged_tile_of_a_batched_product(abi, monkeypatch, tile, dtype):
    """Edges of the tiles and of the chunks (16, 32 or 64 values of k), rows shorter than a 16-byte piece and of every
    remainder; what lies beside a pair in its stack stays out of its product, NaN and all."""
    from mygrad_amd import _hip

    monkeypatch.setenv("MYGRAD_HIP_BMM_TILE", tile)
    for batch, M, K, N in ((3, 17, 1, 18), (2, 33, 3, 31), (2, 65, 2, 129), (3, 129, 17, 66), (2, 64, 64, 64), (2, 63, 65, 33), (9, 35, 130, 37), (64, 40, 19, 21)):
        rng = np.random.default_rng([batch, M, K, N])
        a, b = rng.integers(-4, 5, (batch, M, K)).astype(dtype), rng.integers(-4, 5, (batch, K, N)).astype(dtype)
        want = np.matmul(a, b)
        a[1::2], b[1::2] = np.nan, np.inf
        at, bt = np.ascontiguousarray(a.transpose(0, 2, 1)), np.ascontiguousarray(b.transpose(0, 2, 1))
        print("tile", tile, np.dtype(dtype).name, batch, M, K, N, flush=True)
        for ta, tb in ((False, False), (True, False), (False, True), (True, True)):
            got = abi.matmul_batched(at if ta else a, bt if tb else b, ta, tb)
            assert f"{tile.split(',')[0]} x" in _hip.last_plan()
            assert np.array_equal(got[::2], want[::2]), (M, K, N, ta, tb)


@pytest.mark.parametrize("dtype,batch,M,K,N,short", [
    (np.float64, 24, 64, 64, 64, False), (np.float32, 4, 200, 100, 60, False), (np.float32, 9, 300, 500, 40, False), (np.float64, 16, 64, 197, 197, False),
    (np.float32, 500, 86, 117, 322, True), (np.float32, 300, 20, 100, 20, False),
])
def test_small_stacks_take_few_trips(abi, dtype, batch, M, K, N, short):
    """A stack of few blocks is bound by the trips of one block's chain, a large one by the work of a unit."""
    from mygrad_amd import _hip

    a, b = np.ones((batch, M, K), dtype=dtype), np.ones((batch, K, N), dtype=dtype)
    assert np.array_equal(abi.matmul_batched(a, b), np.full((batch, M, N), K, dtype=dtype))
    assert _hip.last_plan().startswith("batched") and ("short" in _hip.last_plan()) == short, _hip.last_plan()


def test_batched_product_of_more_blocks_than_a_launch_has(abi):
    """2^26 + 5 products of one element are 2^24 + 2 blocks of four; a launch is limited to fewer than 2^32 threads."""
    batch = 2**26 + 5
    a = (np.arange(batch) % 251).astype(np.float32).reshape(batch, 1, 1)
    b = (np.arange(batch) % 127).astype(np.float32).reshape(batch, 1, 1)
    assert np.array_equal(abi.matmul_batched(a, b), a * b)


def test_batched_product_bad_arguments(abi):
    from mygrad_amd import _device, _hip

    buf, lib = _device.DeviceBuffer(4096), _hip.lib()
    assert lib.mg_matmul_batched(0, 2, 4, 4, 4, 0, 0, buf.ptr, buf.ptr, buf.ptr) == _hip.MG_OK
    assert lib.mg_matmul_batched(2, 2, 4, 4, 4, 0, 0, buf.ptr, buf.ptr, buf.ptr) == _hip.MG_ERR_UNSUPPORTED
    assert lib.mg_matmul_batched(0, 2, -1, 4, 4, 0, 0, buf.ptr, buf.ptr, buf.ptr) == _hip.MG_ERR_BAD_ARG
    assert lib.mg_matmul_batched(0, 2, 4, 4, 4, 0, 0, None, buf.ptr, buf.ptr) == _hip.MG_ERR_BAD_ARG
    assert lib.mg_matmul_batched(0, 2, 4, 4, 4, 0, 0, buf.ptr, buf.ptr, None) == _hip.MG_ERR_BAD_ARG
    assert lib.mg_matmul_batched(0, 2, 1 << 24, 4, 4, 0, 0, buf.ptr, buf.ptr, buf.ptr) == _hip.MG_ERR_UNSUPPORTED
    assert lib.mg_matmul_batched(0, 0, 4, 4, 4, 0, 0, None, None, None) == _hip.MG_OK  # nothing to do


SHAPES = [
    ((3, 4), (4, 5)),
    ((4,), (4, 5)),
    ((3, 4), (4,)),
    ((4,), (4,)),
    ((2, 3, 4), (4, 5)),
    ((3, 4), (2, 4, 5)),
    ((2, 3, 4), (2, 4, 5)),
    ((4,), (2, 3, 4, 5)),
    ((2, 3, 4), (4,)),
    ((2, 2, 30, 40), (2, 2, 40, 50)),
    ((2, 800, 810), (2, 810, 790)),  # pairs large enough for a launch of the tiled kernels each
    ((60, 70), (70, 80)),
    # stacks that broadcast against each other
    ((2, 1, 3, 4), (2, 4, 5)),
    ((1, 3, 4), (2, 4, 5)),
    ((3, 1, 2, 6, 4), (2, 1, 4, 5)),
    ((2, 3, 4), (5, 1, 4, 3)),
]


@pytest.mark.parametrize("dtype", [np.float32, np.float64])
@pytest.mark.parametrize("sa, sb", SHAPES)
def test_matmul_through_the_tensor_api(sa, sb, dtype):
    import mygrad_amd as mg

    dtype = np.dtype(dtype)
    rng = np.random.default_rng([len(sa), len(sb), int(np.prod(sa)), int(np.prod(sb))])
    a, b = mg.Tensor(rng.standard_normal(sa).astype(dtype)), mg.Tensor(rng.standard_normal(sb).astype(dtype))
    out = mg.matmul(a, b)
    wa, wb = a.data.astype(np.float64), b.data.astype(np.float64)
    want = ora.matmul_forward(wa, wb)
    assert out.shape == want.shape and out.dtype == dtype and err(out.data, want) <= TOL[dtype]
    g = rng.standard_normal(out.shape).astype(dtype)
    out.backward(g)
    assert a.grad.shape == sa and b.grad.shape == sb and a.grad.dtype == b.grad.dtype == dtype
    assert err(a.grad, ora.matmul_backward(g.astype(np.float64), wa, wb, 0)) <= TOL[dtype]
    assert err(b.grad, ora.matmul_backward(g.astype(np.float64), wa, wb, 1)) <= TOL[dtype]


def test_reference_vectors_operator_and_errors(kats):
    import mygrad_amd as mg
    for case in kats["matmul"]:
        if "a" not in case:
            out = mg.matmul(np.zeros(case["a_shape"]), np.zeros(case["b_shape"]))
            assert list(out.shape) == case["out_shape"]
            continue
        a, b = mg.Tensor(np.array(case["a"], dtype=float)), mg.Tensor(np.array(case["b"], dtype=float))
        out = a @ b
        assert np.array_equal(out.data, np.array(case["out"], dtype=float)), case["source"]
        out.backward()
        if "da" in case:
            assert np.array_equal(a.grad, case["da"]) and np.array_equal(b.grad, case["db"])
    x = mg.Tensor(np.eye(3))
    assert np.array_equal((np.arange(9.0).reshape(3, 3) @ x).data, np.arange(9.0).reshape(3, 3))  # __rmatmul__

    with pytest.raises(ValueError):
        mg.matmul(mg.Tensor(np.ones((2, 3))), 3.0)  # scalars are not allowed
    with pytest.raises(ValueError):
        mg.matmul(mg.Tensor(np.ones((2, 3))), np.ones((4, 2)))  # core dimensions differ
    with pytest.raises(ValueError):
        mg.matmul(mg.Tensor(np.ones((2, 1, 3, 4))), np.ones((3, 2, 4, 5)))  # stacks that do not broadcast
    with pytest.raises(TypeError):
        mg.matmul(mg.Tensor(np.ones((2, 3), dtype=np.int64)), np.ones((3, 2), dtype=np.int64))
    assert mg.matmul(np.ones((0, 3)), np.ones((3, 2))).shape == (0, 2)
    assert np.array_equal(mg.matmul(np.ones((2, 0)), np.ones((0, 3))).data, np.zeros((2, 3)))


def test_dense_layer_chain_stays_on_the_device():
    """relu(x @ w1) @ w2 summed against g: the hidden activations never leave the device."""
    import mygrad_amd as mg
    from mygrad_amd import _device
    from mygrad_amd.nnet import relu

    rng = np.random.default_rng(21)
    x = mg.Tensor(rng.standard_normal((64, 100)))
    w1, w2 = mg.Tensor(rng.standard_normal((100, 80)) * 0.1), mg.Tensor(rng.standard_normal((80, 10)) * 0.1)
    g = rng.standard_normal((64, 10))
    before = dict(_device.stats)
    h = relu(x @ w1)
    out = h @ w2
    h_data = h.data
    out.backward(g)
    assert _device.stats["uploads"] - before["uploads"] == 4  # x, w1, w2 and the seed gradient
    want_h = ora.relu_forward(ora.matmul_forward(x.data, w1.data))
    assert err(h_data, want_h) <= 1e-10
    dh = ora.relu_backward(x.data @ w1.data, ora.matmul_backward(g, want_h, w2.data, 0))
    assert err(w2.grad, ora.matmul_backward(g, want_h, w2.data, 1)) <= 1e-10
    assert err(w1.grad, ora.matmul_backward(dh, x.data, w1.data, 1)) <= 1e-10
    assert err(x.grad, ora.matmul_backward(dh, x.data, w1.data, 0)) <= 1e-10


@pytest.mark.parametrize("dtype", [np.float32, np.float64])
@pytest.mark.parametrize("shapes", [
    [(10, 100), (100, 5), (5, 50)], [(3, 4), (4, 5), (5, 6), (6, 2)], [(4,), (4, 5), (5, 3)], [(3, 4), (4, 5), (5,)],
    [(4,), (4, 6), (6, 5), (5,)], [(7, 2), (2, 9), (9, 1), (1, 8), (8, 3)], [(3, 4), (4, 5)],
])
def test_multi_matmul_and_its_gradients(shapes, dtype):
    """Same bar as the single product; the expected values are NumPy's chained product and the
    chain rule through the restated matmul gradients, in float64."""
    import mygrad_amd as mg

    dtype = np.dtype(dtype)
    rng = np.random.default_rng([len(shapes), sum(int(np.prod(s)) for s in shapes)])
    arrays = [rng.standard_normal(s).astype(dtype) for s in shapes]
    tensors = [mg.Tensor(a) for a in arrays]
    out = mg.multi_matmul(tensors)
    wide = [a.astype(np.float64) for a in arrays]
    want = wide[0]
    for w in wide[1:]:
        want = ora.matmul_forward(want, w)
    assert out.shape == want.shape and out.dtype == dtype and err(out.data, want) <= TOL[dtype]
    g = rng.standard_normal(want.shape).astype(dtype)
    out.backward(g)
    # d out / d A_i = (A_0 ... A_{i-1})^T g (A_{i+1} ... A_n)^T, by the chain rule from the left
    for i, t in enumerate(tensors):
        left = None
        for w in wide[:i]:
            left = w if left is None else ora.matmul_forward(left, w)
        right = None
        for w in wide[i + 1:]:
            right = w if right is None else ora.matmul_forward(right, w)
        grad = g.astype(np.float64)
        chain = wide[i] if right is None else ora.matmul_forward(wide[i], right)
        if left is not None:
            grad = ora.matmul_backward(grad, left, chain, 1)  # through left @ (A_i right)
        if right is not None:
            grad = ora.matmul_backward(grad, wide[i], right, 0)  # through A_i @ right
        assert t.grad.shape == t.shape and err(t.grad, grad) <= TOL[dtype]
