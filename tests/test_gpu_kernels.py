"""Parity of the HIP kernels (called through the C ABI) against the CPU oracle.

Bars: pooling bit-exact (raw bit patterns); convolution
max|gpu - ref| / max|ref| <= 1e-10 in float64 and <= 2e-4 in float32.
"""

import os

import numpy as np
import pytest

from oracle import direct
from oracle import np_oracle as ora

pytestmark = pytest.mark.gpu

TOL = {np.dtype(np.float64): 1e-10, np.dtype(np.float32): 2e-4}


@pytest.fixture(scope="module")
def abi():
    import mygrad_amd

    if not mygrad_amd.is_available():
        pytest.fail("libmygrad_hip.so / gfx950 device not available: the GPU tests need both")
    from tests import abi as module

    return module


def rel_err(got, want):
    scale = float(np.max(np.abs(want))) or 1.0
    return float(np.max(np.abs(got.astype(np.float64) - want.astype(np.float64)))) / scale


def bits(a):
    return a.view(np.uint32 if a.dtype == np.float32 else np.uint64)


# ----------------------------------------------------------------------------- pooling
class _Remembered:
    """The pair of entry points that keeps each window's argmax from the forward pass,
    behind the calling convention of the pair that recomputes it from x."""

    def __init__(self, abi):
        self.abi = abi

    def pool_fwd(self, x, pool, stride):
        out, argmax = self.abi.pool_fwd_argmax(x, pool, stride)
        # what was recorded is np.argmax over each flattened window (pooling.py:109-111)
        if x.size <= 1 << 22:
            assert argmax.dtype == np.uint8 and np.array_equal(argmax, ora.pool_argmax(x, pool, stride))
        return out

    def pool_bwd(self, x, grad, pool, stride, dx_dtype=None):
        _, argmax = self.abi.pool_fwd_argmax(x, pool, stride)
        return self.abi.pool_bwd_argmax(argmax, x.shape, x.dtype, grad, pool, stride, dx_dtype=dx_dtype)


@pytest.fixture(params=["recompute", "remember"])
def pools(request, abi):
    return abi if request.param == "recompute" else _Remembered(abi)


def test_pool_reference_known_answers(pools, kats):
    for case in kats["pool"]:
        x = np.array(case["x"], dtype=case["dtype"])
        pool, stride = tuple(case["pool"]), tuple(case["stride"])
        out = pools.pool_fwd(x, pool, stride)
        assert np.array_equal(out, np.array(case["out"], dtype=x.dtype)), case["source"]
        if case["grad"] is None:
            continue
        g = np.ones(out.shape) if case["grad"] == "ones" else np.arange(out.size).reshape(out.shape)
        for dx_dtype in (x.dtype, np.float64):
            dx = pools.pool_bwd(x, g, pool, stride, dx_dtype=dx_dtype)
            assert dx.dtype == dx_dtype
            assert np.array_equal(dx, np.array(case["dx"], dtype=float)), case["source"]


@pytest.mark.parametrize("m,lead", [(1, (3,)), (1, (2, 5)), (2, (2, 3)), (3, (2,)), (2, ()), (3, (1, 2))])
@pytest.mark.parametrize("dtype", [np.float32, np.float64])
def test_pool_ties_and_overlap_bit_exact(pools, m, lead, dtype):
    rng = np.random.default_rng(300 + 10 * m + len(lead))
    for trial in range(12):
        pool = tuple(int(v) for v in rng.integers(1, 5, m))
        stride = tuple(int(v) for v in rng.integers(1, 5, m))
        grid = tuple(int(v) for v in rng.integers(1, 9, m))
        slack = tuple(int(v) for v in rng.integers(0, 2, m))
        X = tuple((g - 1) * s + p + (e if e < s else 0) for g, s, p, e in zip(grid, stride, pool, slack))
        print("pool case", m, lead, dtype.__name__, pool, stride, X, flush=True)
        if trial % 3 == 0:
            x = rng.standard_normal((*lead, *X)).astype(dtype)
        else:
            x = rng.integers(0, 4, (*lead, *X)).astype(dtype)  # few distinct values: ties everywhere
        out_shape = (*lead, *(((xk - pk) // sk + 1) for xk, pk, sk in zip(X, pool, stride)))
        g = (rng.standard_normal(out_shape) * 10.0 ** rng.integers(-6, 6, out_shape)).astype(dtype)
        want_out = ora.pool_forward(x, pool, stride, validate=False)
        want_dx = ora.pool_backward(x, g, pool, stride)  # float64
        out = pools.pool_fwd(x, pool, stride)
        assert np.array_equal(bits(out), bits(want_out))
        dx64 = pools.pool_bwd(x, g, pool, stride, dx_dtype=np.float64)
        assert np.array_equal(bits(dx64), bits(want_dx))
        dx = pools.pool_bwd(x, g, pool, stride)
        assert np.array_equal(bits(dx), bits(want_dx.astype(dtype)))
        hits = pools.pool_bwd(x, np.ones(out_shape, dtype), pool, stride)
        assert np.array_equal(hits, ora.pool_backward(x, np.ones(out_shape), pool, stride))


@pytest.mark.parametrize("dtype", [np.float32, np.float64])
@pytest.mark.parametrize("lead,X,pool,stride", [
    ((3, 2), (11, 16), (3, 3), (2, 2)),   # an odd number of rows: the last row group is half empty
    ((5,), (56, 56), (3, 3), (2, 2)),     # the benchmark's plane (rows 55 and columns 55 are never covered)
    ((2,), (9, 12), (3, 3), (1, 1)),      # every element under up to nine windows
    ((4,), (7, 8), (2, 2), (1, 1)),
    ((2,), (3, 6, 8), (1, 3, 3), (1, 2, 2)),  # a leading pooled axis of extent one folds into the planes
    ((1,), (3, 4), (3, 3), (2, 2)),       # a single window per plane
    # exact window grids over an odd last extent (what the reference's validator admits for 3 x 3 windows
    # placed every other column): rows start on no 16-byte boundary and end in a short piece
    ((3, 2), (11, 15), (3, 3), (2, 2)),
    ((5,), (55, 55), (3, 3), (2, 2)),     # the valid neighbour of the benchmark's plane
    ((2,), (5, 7), (3, 3), (2, 2)),       # short pieces of three (float32) and one (float64) columns
    ((2,), (5, 5), (3, 3), (2, 2)),       # of one column in either precision
    ((3,), (9, 13), (3, 3), (1, 1)),
    ((3,), (7, 9), (2, 2), (1, 1)),
    ((2,), (5, 6), (3, 3), (1, 1)),       # a short piece of two float32 columns
    ((2,), (3, 3), (3, 3), (2, 2)),       # a float32 row shorter than one piece
    # 3 x 3 x 3 windows at every other position: the same kernels with a pooled leading axis
    ((2, 2), (7, 9, 13), (3, 3, 3), (2, 2, 2)),
    ((3,), (5, 7, 8), (3, 3, 3), (2, 2, 2)),     # flooring placement along the last axis
    ((2,), (8, 10, 12), (3, 3, 3), (2, 2, 2)),   # the last plane, row and column are never covered
    ((1,), (9, 65, 65), (3, 3, 3), (2, 2, 2)),   # planes too large for a band in LDS
    ((2,), (3, 5, 9), (3, 3, 3), (2, 2, 2)),     # a single window plane
])
def test_pool_backward_gather_for_windows_known_at_compile_time(pools, dtype, lead, X, pool, stride):
    """2-D windows of 3x3 / stride 2, 3x3 / stride 1 and 2x2 / stride 1 over rows of whole 16-byte
    pieces: the backward pass from the recorded argmax gathers per element in registers.  Ties,
    NaNs, gradients of -0.0 and huge / tiny magnitudes (the order of the additions shows), the
    float64 dx of a float32 input."""
    rng = np.random.default_rng(370 + X[-1] + X[-2])
    for trial in range(5):
        if trial == 0:
            x = rng.standard_normal((*lead, *X)).astype(dtype)
        else:
            x = rng.integers(0, 3, (*lead, *X)).astype(dtype)
        if trial == 2:
            x[rng.random(x.shape) < 0.1] = np.nan
        out_shape = (*lead, *(((xk - pk) // sk + 1) for xk, pk, sk in zip(X, pool, stride)))
        g = (rng.standard_normal(out_shape) * 10.0 ** rng.integers(-6, 6, out_shape)).astype(dtype)
        if trial == 3:
            g = rng.choice(np.array([1e16, 1.0, -1e16], dtype=dtype), out_shape)  # sums that depend on their order
        g[rng.random(out_shape) < 0.2] = -0.0
        want_dx = ora.pool_backward(x, g, pool, stride)  # float64
        assert np.array_equal(bits(pools.pool_fwd(x, pool, stride)), bits(ora.pool_forward(x, pool, stride, validate=False)))
        assert np.array_equal(bits(pools.pool_bwd(x, g, pool, stride, dx_dtype=np.float64)), bits(want_dx))
        assert np.array_equal(bits(pools.pool_bwd(x, g, pool, stride)), bits(want_dx.astype(dtype)))


@pytest.mark.parametrize("dtype", [np.float32, np.float64])
@pytest.mark.parametrize("lead,X,pool", [
    ((3, 5), (8, 12), (2, 2)),        # 2-D, rows of whole 16-byte pieces: the exact-tiling kernel
    ((2,), (6, 4, 8), (2, 2, 2)),     # 3-D
    ((7,), (2, 2, 4), (2, 2, 2)),     # a single window slab per volume
    ((4,), (10, 6), (2, 2)),          # float32 rows of 4k + 2 columns: pieces of 8 bytes
    ((3, 2), (14, 14), (2, 2)),
    ((2,), (4, 6, 10), (2, 2, 2)),
    ((1,), (2, 2), (2, 2)),           # one window in all
])
def test_pool_windows_that_tile_the_input_exactly(pools, dtype, lead, X, pool):
    """Stride == pool extent and X == G * P: the kernels that work straight from global
    memory.  Ties, NaNs, -0.0 gradients and the float64 dx of a float32 input included."""
    rng = np.random.default_rng(350 + len(X) + X[-1])
    for trial in range(4):
        if trial == 0:
            x = rng.standard_normal((*lead, *X)).astype(dtype)
        else:
            x = rng.integers(0, 3, (*lead, *X)).astype(dtype)  # ties in almost every window
        if trial == 2:
            x[rng.random(x.shape) < 0.1] = np.nan
        out_shape = (*lead, *(xk // pk for xk, pk in zip(X, pool)))
        g = (rng.standard_normal(out_shape) * 10.0 ** rng.integers(-6, 6, out_shape)).astype(dtype)
        g[rng.random(out_shape) < 0.2] = -0.0
        want_out = ora.pool_forward(x, pool, pool, validate=False)
        want_dx = ora.pool_backward(x, g, pool, pool)  # float64
        assert np.array_equal(bits(pools.pool_fwd(x, pool, pool)), bits(want_out))
        assert np.array_equal(bits(pools.pool_bwd(x, g, pool, pool, dx_dtype=np.float64)), bits(want_dx))
        assert np.array_equal(bits(pools.pool_bwd(x, g, pool, pool)), bits(want_dx.astype(dtype)))


@pytest.mark.parametrize("dtype", [np.float32, np.float64])
@pytest.mark.parametrize("X,pool,stride", [((7, 9001), (3, 3), (2, 2)), ((2, 5, 7000), (2, 3, 2), (1, 2, 3)),
                                           ((7, 70, 70), (2, 3, 3), (1, 2, 2)), ((5, 9000), (4, 2), (1, 1))])
def test_pool_rows_too_long_for_the_staged_kernels(pools, dtype, X, pool, stride):
    """One row of windows with its halo exceeds the LDS budget: the kernels that work
    element by element from global memory take over."""
    rng = np.random.default_rng(360 + len(X))
    x = rng.integers(0, 5, (3, *X)).astype(dtype)
    out_shape = (3, *(((xk - pk) // sk + 1) for xk, pk, sk in zip(X, pool, stride)))
    g = (rng.standard_normal(out_shape) * 10.0 ** rng.integers(-6, 6, out_shape)).astype(dtype)
    want_dx = ora.pool_backward(x, g, pool, stride)
    assert np.array_equal(bits(pools.pool_fwd(x, pool, stride)), bits(ora.pool_forward(x, pool, stride, validate=False)))
    assert np.array_equal(bits(pools.pool_bwd(x, g, pool, stride, dx_dtype=np.float64)), bits(want_dx))
    assert np.array_equal(bits(pools.pool_bwd(x, g, pool, stride)), bits(want_dx.astype(dtype)))


def test_pool_window_of_256_positions_fills_the_argmax_byte(pools):
    rng = np.random.default_rng(361)
    x = rng.integers(0, 50, (2, 20, 19)).astype(np.float64)
    g = rng.standard_normal((2, 5, 4))
    assert np.array_equal(pools.pool_fwd(x, (16, 16), 1), ora.pool_forward(x, (16, 16), 1))
    assert np.array_equal(bits(pools.pool_bwd(x, g, (16, 16), 1)), bits(ora.pool_backward(x, g, (16, 16), 1)))


def test_pool_order_of_summation_and_signed_zero(pools):
    x = np.array([[0.0, 0.0, 9.0, 0.0, 0.0]])
    for g in ([1e16, 1.0, -1e16], [1e16, -1e16, 1.0], [-0.0, -0.0, -0.0]):
        g = np.array([g])
        dx = pools.pool_bwd(x, g, (3,), (1,))
        assert np.array_equal(bits(dx), bits(ora.pool_backward(x, g, (3,), (1,))))
    dx = pools.pool_bwd(np.array([[1.0, 0.0]]), np.array([[-0.0]]), (2,), (2,))
    assert not np.signbit(dx).any()


def test_pool_nan_first_nan_wins(pools):
    x = np.array([[1.0, np.nan, 5.0, np.nan, 2.0, 3.0]])
    out = pools.pool_fwd(x, (4,), (1,))
    want = ora.pool_forward(x, (4,), (1,))
    assert np.array_equal(np.isnan(out), np.isnan(want)) and np.isnan(out).all()
    g = np.array([[2.0, 3.0, 5.0]])
    assert np.array_equal(pools.pool_bwd(x, g, (4,), (1,)), ora.pool_backward(x, g, (4,), (1,)))


@pytest.mark.parametrize("ties", [False, True])
def test_pool_config2_literal_full_size(pools, ties):
    # x (64,64,56,56) f64, pool 3x3 stride 2, floor placement -> (64,64,27,27);
    # the reference's validator rejects it ((56-3)/2+1 = 27.5), its window helper floors
    rng = np.random.default_rng(1002)
    shape = (64, 64, 56, 56)
    x = rng.integers(0, 8, shape).astype(np.float64) if ties else rng.standard_normal(shape)
    g = rng.standard_normal((64, 64, 27, 27))
    out = pools.pool_fwd(x, (3, 3), 2)
    dx = pools.pool_bwd(x, g, (3, 3), 2)
    want_out, want_dx = direct.pool(x, g, (3, 3), (2, 2))
    assert np.array_equal(bits(out), bits(want_out))
    assert np.array_equal(bits(dx), bits(want_dx))
    assert not dx[..., 55, :].any() and not dx[..., :, 55].any()  # never covered by a window
    # the NumPy restatement of the reference agrees on a slice it finishes quickly
    sl = slice(0, 4)
    assert np.array_equal(bits(out[sl]), bits(ora.pool_forward(x[sl], (3, 3), 2, validate=False)))
    assert np.array_equal(bits(dx[sl]), bits(ora.pool_backward(x[sl], g[sl], (3, 3), 2)))


@pytest.mark.parametrize("ties", [False, True])
@pytest.mark.parametrize("dtype", [np.float64, np.float32])
def test_pool_config2_valid_full_size(pools, ties, dtype):
    # the neighbour of config 2 that the reference accepts: x (64,64,55,55), pool 3x3 stride 2 ->
    # (64,64,27,27) exactly; rows of 55 elements start on no 16-byte boundary
    rng = np.random.default_rng(1002)
    shape = (64, 64, 55, 55)
    x = (rng.integers(0, 8, shape) if ties else rng.standard_normal(shape)).astype(dtype)
    g = rng.standard_normal((64, 64, 27, 27)).astype(dtype)
    out = pools.pool_fwd(x, (3, 3), 2)
    dx = pools.pool_bwd(x, g, (3, 3), 2)
    dx64 = pools.pool_bwd(x, g, (3, 3), 2, dx_dtype=np.float64)
    want_out, want_dx = direct.pool(x, g, (3, 3), (2, 2))
    assert np.array_equal(bits(out), bits(want_out))
    assert np.array_equal(bits(dx64), bits(want_dx))
    assert np.array_equal(bits(dx), bits(want_dx.astype(dtype)))
    sl = slice(0, 4)
    assert np.array_equal(bits(out[sl]), bits(ora.pool_forward(x[sl], (3, 3), 2)))
    assert np.array_equal(bits(dx64[sl]), bits(ora.pool_backward(x[sl], g[sl], (3, 3), 2)))


def test_pool_config5_shape_full_size(pools):
    rng = np.random.default_rng(1006)
    x = rng.standard_normal((8, 32, 32, 64, 64)).astype(np.float32)
    g = rng.standard_normal((8, 32, 16, 32, 32)).astype(np.float32)
    out = pools.pool_fwd(x, (2, 2, 2), 2)
    dx = pools.pool_bwd(x, g, (2, 2, 2), 2)
    want_out, want_dx = direct.pool(x, g, (2, 2, 2), (2, 2, 2))
    assert np.array_equal(bits(out), bits(want_out))
    assert np.array_equal(bits(dx), bits(want_dx.astype(np.float32)))


# ----------------------------------------------------------------------------- convolution
def test_conv_reference_known_answers(abi, kats):
    for dtype in (np.float64, np.float32):
        for case in kats["conv"]:
            x, w = np.array(case["x"], dtype=dtype), np.array(case["w"], dtype=dtype)
            conf = (tuple(case["stride"]), tuple(case["padding"]), tuple(case["dilation"]))
            out = abi.conv_fwd(x, w, *conf)
            assert np.array_equal(out, np.array(case["out"], dtype=dtype)), case["source"]
            if "dx_of_ones" in case:
                g = np.ones_like(out)
                assert np.array_equal(abi.conv_dgrad(g, x.shape, w, *conf), np.array(case["dx_of_ones"], dtype=dtype))
                assert np.array_equal(abi.conv_wgrad(g, x, w.shape, *conf), np.array(case["dw_of_ones"], dtype=dtype))


def _random_case(rng, m, big):
    hi = 40 if big else 6
    N = int(rng.integers(1, 4))
    C = int(rng.integers(1, hi))
    F = int(rng.integers(1, hi))
    taps = tuple(int(v) for v in rng.integers(1, 4, m))
    dil = tuple(int(v) for v in rng.integers(1, 3, m))
    stride = tuple(int(v) for v in rng.integers(1, 4, m))
    pad = tuple(int(v) for v in rng.integers(0, 3, m))
    grid = tuple(int(v) for v in rng.integers(1, 12 if m < 3 else 6, m))
    extra = tuple(int(v) for v in rng.integers(0, 2, m))  # rows the floor rule never uses
    X = tuple(
        (g - 1) * s + (t - 1) * d + 1 - 2 * p + (e if e < s else 0)
        for g, s, t, d, p, e in zip(grid, stride, taps, dil, pad, extra)
    )
    if any(v < 1 for v in X):
        return None
    return (N, C, *X), (F, C, *taps), stride, pad, dil


@pytest.fixture(params=["small problems planned as such", "planned like large ones"])
def plan_mode(request, monkeypatch):
    """A convolution of a few microseconds is planned for few launches (table-driven kernels
    that read the filter bank in place); MYGRAD_HIP_TINY=0 plans it like a large one, which
    is how shapes this small reach the tap-major kernels' edge cases."""
    if request.param == "planned like large ones":
        monkeypatch.setenv("MYGRAD_HIP_TINY", "0")
    return request.param


@pytest.mark.parametrize("dtype", [np.float64, np.float32])
@pytest.mark.parametrize("m", [1, 2, 3])
@pytest.mark.parametrize("big", [False, True])
def test_conv_random_cases_vs_oracle(abi, dtype, m, big, plan_mode):
    rng = np.random.default_rng(400 + 10 * m + big)
    tol = TOL[np.dtype(dtype)]
    done = 0
    while done < 10:
        case = _random_case(rng, m, big)
        if case is None:
            continue
        x_shape, w_shape, s, p, d = case
        print("conv case", np.dtype(dtype).name, x_shape, w_shape, s, p, d, flush=True)
        x = rng.standard_normal(x_shape).astype(dtype)
        w = rng.standard_normal(w_shape).astype(dtype)
        want_out = direct.conv_forward(x, w, s, p, d)
        g = rng.standard_normal(want_out.shape).astype(dtype)
        out = abi.conv_fwd(x, w, s, p, d)
        assert out.shape == want_out.shape and out.dtype == dtype
        assert rel_err(out, want_out) <= tol
        assert rel_err(abi.conv_dgrad(g, x_shape, w, s, p, d), direct.conv_backward_x(g, x_shape, w, s, p, d)) <= tol
        assert rel_err(abi.conv_wgrad(g, x, w_shape, s, p, d), direct.conv_backward_w(g, x, w_shape, s, p, d)) <= tol
        done += 1


@pytest.mark.parametrize("dtype", [np.float64, np.float32])
@pytest.mark.parametrize("m", [1, 2, 3])
def test_conv_channel_counts_that_take_the_tap_major_kernels(abi, dtype, m, plan_mode):
    # channel / filter counts that are multiples of the K tile (8 or 16) select the
    # tap-major kernels; mix them with counts that do not, strides, dilation, padding
    rng = np.random.default_rng(500 + m)
    tol = TOL[np.dtype(dtype)]
    done = 0
    while done < 14:
        C = int(rng.choice([8, 16, 32, 48, 64]))
        F = int(rng.choice([8, 16, 24, 32, 64, 80, 128, 144]))
        N = int(rng.integers(1, 4))
        taps = tuple(int(v) for v in rng.integers(1, 4, m))
        dil = tuple(int(v) for v in rng.integers(1, 3, m))
        stride = tuple(int(v) for v in rng.integers(1, 4, m))
        pad = tuple(int(v) for v in rng.integers(0, 3, m))
        grid = tuple(int(v) for v in rng.integers(1, [40, 14, 7][m - 1], m))
        extra = tuple(int(v) for v in rng.integers(0, 2, m))
        X = tuple(
            (g - 1) * s + (t - 1) * d + 1 - 2 * p + (e if e < s else 0)
            for g, s, t, d, p, e in zip(grid, stride, taps, dil, pad, extra)
        )
        if any(v < 1 for v in X):
            continue
        x_shape, w_shape = (N, C, *X), (F, C, *taps)
        print("tap-major case", np.dtype(dtype).name, x_shape, w_shape, stride, pad, dil, flush=True)
        x = rng.standard_normal(x_shape).astype(dtype)
        w = rng.standard_normal(w_shape).astype(dtype)
        want_out = direct.conv_forward(x, w, stride, pad, dil)
        g = rng.standard_normal(want_out.shape).astype(dtype)
        assert rel_err(abi.conv_fwd(x, w, stride, pad, dil), want_out) <= tol
        assert rel_err(abi.conv_dgrad(g, x_shape, w, stride, pad, dil),
                       direct.conv_backward_x(g, x_shape, w, stride, pad, dil)) <= tol
        assert rel_err(abi.conv_wgrad(g, x, w_shape, stride, pad, dil),
                       direct.conv_backward_w(g, x, w_shape, stride, pad, dil)) <= tol
        done += 1


# Stride 2 along the last axis (float32, filter count a multiple of 16): every tile of the data
# gradient computes all 2 / 4 stride phases of its patch and writes them interleaved.  Even and
# odd extents (vector and element-wise stores, phases with fewer positions than the coarse grid),
# 1, 2 and 3 convolved axes, channel counts for every fused tile shape (16 .. 128 rows), filters
# with taps that some phases never see (1x1: three of four phases are all zero), dilation, and
# enough positions for persistent blocks, tail tiles and K slices.
FUSED_PHASE_CASES = [
    ((4, 64, 28, 28), (32, 64, 3, 3), (2, 2), (1, 1), (1, 1)),
    ((3, 128, 27, 27), (48, 128, 3, 3), (2, 2), (1, 1), (1, 1)),
    ((2, 32, 30, 36), (16, 32, 1, 1), (2, 2), (0, 0), (1, 1)),
    ((5, 16, 19, 24), (64, 16, 5, 3), (2, 2), (2, 1), (1, 2)),
    ((2, 48, 40, 44), (32, 48, 2, 2), (1, 2), (0, 1), (1, 1)),
    ((3, 64, 130), (16, 64, 7), (2,), (3,), (1,)),
    ((2, 24, 9, 16, 20), (32, 24, 3, 3, 3), (1, 2, 2), (1, 1, 1), (1, 1, 1)),
    ((40, 128, 28, 28), (256, 128, 3, 3), (2, 2), (1, 1), (1, 1)),
    ((2, 8, 12, 10), (16, 8, 3, 3), (2, 2), (0, 0), (1, 1)),
    # exact window grids under stride 2 (odd extents): rows of dx start on no 16-byte boundary; an even
    # and an odd number of coarse positions per row (pairs of positions / single positions per store)
    ((3, 64, 13, 13), (32, 64, 3, 3), (2, 2), (1, 1), (1, 1)),
    ((2, 32, 55, 55), (64, 32, 3, 3), (2, 2), (1, 1), (1, 1)),
    ((2, 128, 9, 27), (16, 128, 3, 3), (1, 2), (1, 1), (1, 1)),
    ((2, 16, 5, 7, 11), (32, 16, 3, 3, 3), (1, 2, 2), (1, 1, 1), (1, 1, 1)),
    ((2, 64, 15, 15), (32, 64, 1, 1), (2, 2), (0, 0), (1, 1)),
]


@pytest.mark.parametrize("rows", ["short rows fused too", "short rows phase by phase"])
@pytest.mark.parametrize("case", range(len(FUSED_PHASE_CASES)))
def test_conv_dgrad_with_fused_stride_phases(abi, case, plan_mode, rows, monkeypatch):
    # four phases of rows shorter than 20 elements are planned phase by phase unless told otherwise
    if rows == "short rows fused too":
        monkeypatch.setenv("MYGRAD_HIP_FUSE_MIN_ROW", "0")
    x_shape, w_shape, s, p, d = FUSED_PHASE_CASES[case]
    rng = np.random.default_rng(900 + case)
    w = (rng.standard_normal(w_shape) / np.sqrt(np.prod(w_shape[1:]))).astype(np.float32)
    grid = tuple((x + 2 * pp - ((t - 1) * dd + 1)) // ss + 1 for x, t, ss, pp, dd in zip(x_shape[2:], w_shape[2:], s, p, d))
    g = rng.standard_normal((x_shape[0], w_shape[0], *grid)).astype(np.float32)
    dx = abi.conv_dgrad(g, x_shape, w, s, p, d)
    assert rel_err(dx, direct.conv_backward_x(g, x_shape, w, s, p, d)) <= 2e-4
    assert np.array_equal(dx, abi.conv_dgrad(g, x_shape, w, s, p, d))  # no atomics: run-to-run identical
    # dx of an all-ones gradient counts, per input element, the windows that reach it: exact
    # in float32 with a filter of ones, which isolates the routing from the rounding
    ones_w = np.ones(w_shape, dtype=np.float32)
    ones_g = np.ones_like(g)
    assert np.array_equal(abi.conv_dgrad(ones_g, x_shape, ones_w, s, p, d),
                          direct.conv_backward_x(ones_g, x_shape, ones_w, s, p, d).astype(np.float32))


@pytest.mark.parametrize("dtype", [np.float32, np.float64])
@pytest.mark.parametrize("x_shape,w_shape,s,p,d", [
    ((5, 64, 7, 7), (64, 64, 3, 3), (1, 1), (1, 1), (1, 1)),       # 49 positions per sample
    ((3, 64, 27, 27), (128, 64, 3, 3), (1, 1), (1, 1), (1, 1)),    # 729
    ((2, 48, 5, 9, 3), (64, 48, 3, 3, 1), (1, 1, 1), (1, 1, 0), (1, 1, 1)),
    ((7, 128, 13), (64, 128, 5), (1,), (2,), (1,)),
    ((4, 64, 30, 31), (64, 64, 3, 3), (2, 2), (1, 1), (1, 1)),     # forward only: a 15 x 15 grid
])
def test_conv_samples_that_are_no_whole_16_byte_pieces(abi, dtype, x_shape, w_shape, s, p, d, monkeypatch):
    """An odd number of positions per sample: a lane's positions are adjacent in the result but
    not 16-byte aligned, and the last lane of a sample holds positions of two samples."""
    monkeypatch.setenv("MYGRAD_HIP_TINY", "0")
    rng = np.random.default_rng(1450 + x_shape[-1])
    tol = TOL[np.dtype(dtype)]
    x = rng.standard_normal(x_shape).astype(dtype)
    w = (rng.standard_normal(w_shape) / np.sqrt(np.prod(w_shape[1:]))).astype(dtype)
    want = direct.conv_forward(x, w, s, p, d)
    g = rng.standard_normal(want.shape).astype(dtype)
    assert rel_err(abi.conv_fwd(x, w, s, p, d), want) <= tol
    assert rel_err(abi.conv_dgrad(g, x_shape, w, s, p, d), direct.conv_backward_x(g, x_shape, w, s, p, d)) <= tol
    assert rel_err(abi.conv_wgrad(g, x, w_shape, s, p, d), direct.conv_backward_w(g, x, w_shape, s, p, d)) <= tol
    # exact with ones: an element stored to the wrong place changes a count
    ones_x, ones_w = np.ones(x_shape, dtype), np.ones(w_shape, dtype)
    assert np.array_equal(abi.conv_fwd(ones_x, ones_w, s, p, d), direct.conv_forward(ones_x, ones_w, s, p, d).astype(dtype))
    ones_g = np.ones_like(g)
    assert np.array_equal(abi.conv_dgrad(ones_g, x_shape, ones_w, s, p, d),
                          direct.conv_backward_x(ones_g, x_shape, ones_w, s, p, d).astype(dtype))


# Few channels (filters, in the forward pass), a 3-tap "same" last axis whose rows are a power of
# two up to 64 long (float32, the other count a multiple of 16): the data gradient and the forward
# pass compute the three taps of the last axis as separate rows and add them, shifted, in the epilogue.  1, 2 and 3 convolved axes,
# row lengths 4 .. 64, channel counts that do and do not fill the tile, other axes with padding,
# dilation and even tap counts, position counts that are no multiple of the tile.
FOLDED_TAP_CASES = [
    ((2, 16, 8, 64, 64), (32, 16, 3, 3, 3), (1, 1, 1), (1, 1, 1), (1, 1, 1)),
    ((3, 16, 40, 32), (16, 16, 3, 3), (1, 1), (1, 1), (1, 1)),
    ((5, 8, 21, 16), (48, 8, 2, 3), (1, 1), (0, 1), (1, 1)),
    ((7, 5, 9, 8), (16, 5, 5, 3), (1, 1), (4, 1), (2, 1)),
    ((9, 12, 64), (32, 12, 3), (1,), (1,), (1,)),
    ((2, 3, 6, 10, 4), (16, 3, 1, 3, 3), (1, 1, 1), (0, 0, 1), (1, 1, 1)),
    ((1, 16, 33, 64), (64, 16, 1, 3), (1, 1), (0, 1), (1, 1)),
    ((2, 32, 16, 32), (16, 32, 3, 3), (1, 1), (1, 1), (1, 1)),       # 32 channels: 96-row tiles
    ((3, 24, 10, 16), (32, 24, 3, 3), (1, 1), (1, 1), (1, 1)),       # 24 channels in a 96-row tile
    ((2, 48, 12, 9, 32), (24, 48, 2, 3, 3), (2, 1, 1), (0, 2, 1), (1, 2, 1)),  # forward only folds (24 filters; stride on axis 0)
    # rows that are no power of two: padded to one (at most an eighth of padding), the padding never stored
    ((3, 16, 28, 28), (16, 16, 3, 3), (1, 1), (1, 1), (1, 1)),
    ((2, 8, 5, 14, 14), (32, 8, 3, 3, 3), (1, 1, 1), (1, 1, 1), (1, 1, 1)),
    ((5, 16, 9, 7), (16, 16, 3, 3), (1, 1), (1, 1), (1, 1)),
    ((2, 16, 20, 56), (32, 16, 3, 3), (1, 1), (1, 1), (1, 1)),
    ((3, 10, 11, 30), (16, 10, 2, 3), (1, 1), (1, 1), (1, 1)),       # rows of 30: no whole 16-byte pieces, element-wise stores
    ((4, 16, 6, 15), (16, 16, 3, 3), (1, 1), (1, 1), (1, 1)),
    ((7, 32, 61), (32, 32, 3), (1,), (1,), (1,)),
]


@pytest.mark.parametrize("dtype", [np.float32, np.float64])
@pytest.mark.parametrize("case", range(len(FOLDED_TAP_CASES)))
def test_conv_with_the_last_axis_taps_folded_into_rows(abi, case, dtype, monkeypatch):
    monkeypatch.setenv("MYGRAD_HIP_TINY", "0")  # small shapes: planned like large ones, or they take the table-driven kernel
    x_shape, w_shape, s, p, d = FOLDED_TAP_CASES[case]
    rng = np.random.default_rng(1300 + case)
    tol = TOL[np.dtype(dtype)]
    w = (rng.standard_normal(w_shape) / np.sqrt(np.prod(w_shape[1:]))).astype(dtype)
    grid = tuple((x + 2 * pp - ((t - 1) * dd + 1)) // ss + 1 for x, t, ss, pp, dd in zip(x_shape[2:], w_shape[2:], s, p, d))
    g = rng.standard_normal((x_shape[0], w_shape[0], *grid)).astype(dtype)
    dx = abi.conv_dgrad(g, x_shape, w, s, p, d)
    assert rel_err(dx, direct.conv_backward_x(g, x_shape, w, s, p, d)) <= tol
    assert np.array_equal(dx, abi.conv_dgrad(g, x_shape, w, s, p, d))
    # exact with ones: per input element, the number of (filter, tap) pairs that reach it -- a
    # shift in the wrong direction or a neighbour taken across a row end changes the counts
    ones_w = np.ones(w_shape, dtype=dtype)
    ones_g = np.ones_like(g)
    assert np.array_equal(abi.conv_dgrad(ones_g, x_shape, ones_w, s, p, d),
                          direct.conv_backward_x(ones_g, x_shape, ones_w, s, p, d).astype(dtype))
    # and with a filter that is not symmetric along the last axis (tap t2 weighs t2 + 1), so that
    # tap 0 and tap 2 cannot be swapped unnoticed
    ramp_w = np.ones(w_shape, dtype=dtype) * np.arange(1, w_shape[-1] + 1, dtype=dtype)
    assert np.array_equal(abi.conv_dgrad(ones_g, x_shape, ramp_w, s, p, d),
                          direct.conv_backward_x(ones_g, x_shape, ramp_w, s, p, d).astype(dtype))
    # the forward pass folds the same way when there are few filters (and channels in whole K tiles)
    x = rng.standard_normal(x_shape).astype(dtype)
    out = abi.conv_fwd(x, w, s, p, d)
    assert rel_err(out, direct.conv_forward(x, w, s, p, d)) <= tol
    assert np.array_equal(out, abi.conv_fwd(x, w, s, p, d))
    # exact: x counts along the last axis (small integers), ramp filter
    steps = np.broadcast_to(np.arange(x_shape[-1], dtype=dtype) % 5, x_shape).copy()
    assert np.array_equal(abi.conv_fwd(steps, ramp_w, s, p, d), direct.conv_forward(steps, ramp_w, s, p, d).astype(dtype))


# Channel counts that fill no K tile (the one or three channels of a first layer), on problems
# large enough not to be planned as tiny: the forward pass runs the tap-major kernel with K tiles
# made of rows of the gather table (the last tile padded with rows that lie outside every input).
FIRST_LAYER_CASES = [
    ((16, 3, 64, 64), (32, 3, 5, 5), (1, 1), (2, 2), (1, 1)),
    ((8, 3, 115, 115), (64, 3, 7, 7), (2, 2), (3, 3), (1, 1)),      # the stem's geometry, flooring placement
    ((32, 1, 28, 28), (20, 1, 5, 5), (1, 1), (0, 0), (1, 1)),       # one channel, 20 filters (padded packed rows)
    ((4, 5, 20, 24, 24), (16, 5, 3, 3, 3), (1, 2, 1), (1, 0, 1), (1, 1, 2)),
    ((64, 7, 500), (48, 7, 9), (3,), (4,), (2,)),
    ((64, 1, 28, 28), (64, 1, 5, 5), (1, 1), (0, 0), (1, 1)),       # 25 columns of dw: one 32-column tile
    ((16, 3, 48, 48), (128, 3, 7, 7), (1, 1), (3, 3), (1, 1)),      # 147 columns: two 80-column tiles, two row tiles
    # filter counts that fill no K tile either: the data gradient on table rows, the filter gradient
    # with a short last row tile
    ((256, 1, 28, 28), (20, 1, 5, 5), (1, 1), (0, 0), (1, 1)),
    ((256, 20, 12, 12), (10, 20, 5, 5), (1, 1), (0, 0), (1, 1)),
    ((32, 24, 41, 40), (20, 24, 3, 4), (2, 2), (1, 1), (1, 1)),     # four stride phases with different tap counts
    ((6, 16, 10, 18, 18), (35, 16, 3, 3, 3), (1, 1, 1), (1, 1, 1), (1, 1, 1)),
    ((64, 40, 301), (19, 40, 7), (2,), (3,), (3,)),
]


@pytest.mark.parametrize("dtype", [np.float32, np.float64])
@pytest.mark.parametrize("case", range(len(FIRST_LAYER_CASES)))
def test_conv_with_channel_or_filter_counts_that_fill_no_k_tile(abi, dtype, case):
    x_shape, w_shape, s, p, d = FIRST_LAYER_CASES[case]
    rng = np.random.default_rng(1500 + case)
    tol = TOL[np.dtype(dtype)]
    x = rng.standard_normal(x_shape).astype(dtype)
    w = (rng.standard_normal(w_shape) / np.sqrt(np.prod(w_shape[1:]))).astype(dtype)
    want = direct.conv_forward(x, w, s, p, d)
    out = abi.conv_fwd(x, w, s, p, d)
    assert rel_err(out, want) <= tol
    assert np.array_equal(out, abi.conv_fwd(x, w, s, p, d))
    # exact: small integers, every (channel, tap) weighted differently
    xi = rng.integers(-2, 3, x_shape).astype(dtype)
    wi = (np.arange(np.prod(w_shape[1:])).reshape(w_shape[1:]) % 7 - 3).astype(dtype) * np.ones(w_shape, dtype=dtype)
    assert np.array_equal(abi.conv_fwd(xi, wi, s, p, d), direct.conv_forward(xi, wi, s, p, d).astype(dtype))
    g = rng.standard_normal(want.shape).astype(dtype)
    assert rel_err(abi.conv_dgrad(g, x_shape, w, s, p, d), direct.conv_backward_x(g, x_shape, w, s, p, d)) <= tol
    assert rel_err(abi.conv_wgrad(g, x, w_shape, s, p, d), direct.conv_backward_w(g, x, w_shape, s, p, d)) <= tol
    # exact: gradients of small integers
    gi = rng.integers(-2, 3, want.shape).astype(dtype)
    assert np.array_equal(abi.conv_dgrad(gi, x_shape, wi, s, p, d), direct.conv_backward_x(gi, x_shape, wi, s, p, d).astype(dtype))
    assert np.array_equal(abi.conv_wgrad(gi, xi, w_shape, s, p, d), direct.conv_backward_w(gi, xi, w_shape, s, p, d).astype(dtype))


# Up to four channels in single precision, on enough positions to fill the device: the data
# gradient runs one position of the coarse grid ceil(X / stride) per lane on the 4x4x1 MFMA, all
# stride phases of the position at once (1, 2 or 4 of them).  Between them the cases cover every
# phase count, entries that fill their chunks of 16 / phases and ones that need padding or
# several channels per chunk, odd extents (phases with different numbers of positions, no paired
# stores), dilation, and one to three convolved axes.  float64 runs the other kernels.
THIN_ROW_CASES = [
    ((16, 3, 130, 130), (16, 3, 7, 7), (2, 2), (3, 3), (1, 1)),     # the stem's geometry (even extent, flooring placement): 4 phases, 16 entries
    ((16, 3, 131, 131), (8, 3, 7, 7), (2, 2), (3, 3), (1, 1)),      # odd extents: the phases differ in size
    ((64, 3, 64, 64), (32, 3, 5, 5), (1, 1), (2, 2), (1, 1)),       # one phase, 25 entries, two filters per chunk step
    ((64, 1, 128, 128), (10, 1, 3, 3), (1, 1), (1, 1), (1, 1)),     # one channel; 9 entries x 2 filters, padded
    ((16, 4, 96, 97), (16, 4, 3, 4), (1, 2), (1, 1), (1, 1)),       # two phases along the last axis
    ((16, 2, 140, 70), (24, 2, 5, 3), (2, 1), (2, 1), (1, 1)),      # two phases along the first axis: no paired stores
    ((64, 3, 64, 64), (32, 3, 3, 3), (1, 1), (2, 2), (2, 2)),       # dilation 2; 9 entries x 16 filters fill their chunks
    ((4, 3, 18, 64, 64), (12, 3, 3, 3, 3), (1, 2, 2), (1, 1, 1), (1, 1, 1)),  # three axes, four phases
    ((64, 2, 2100), (48, 2, 9), (2,), (4,), (1,)),                  # one axis, two phases
    ((64, 3, 128, 128), (16, 3, 2, 2), (2, 2), (0, 0), (1, 1)),     # window = stride: every phase has one tap
]


@pytest.mark.parametrize("dtype", [np.float32, np.float64])
@pytest.mark.parametrize("case", range(len(THIN_ROW_CASES)))
def test_data_gradient_with_up_to_four_channels(abi, dtype, case):
    x_shape, w_shape, s, p, d = THIN_ROW_CASES[case]
    rng = np.random.default_rng(2300 + case)
    tol = TOL[np.dtype(dtype)]
    w = (rng.standard_normal(w_shape) / np.sqrt(np.prod(w_shape[1:]))).astype(dtype)
    grid = direct.conv_forward(np.zeros(x_shape, dtype=dtype), w, s, p, d).shape
    g = rng.standard_normal(grid).astype(dtype)
    got = abi.conv_dgrad(g, x_shape, w, s, p, d)
    assert rel_err(got, direct.conv_backward_x(g, x_shape, w, s, p, d)) <= tol
    assert np.array_equal(got, abi.conv_dgrad(g, x_shape, w, s, p, d))
    # exact: small integers, every (filter, channel, tap) weighted differently
    gi = rng.integers(-2, 3, grid).astype(dtype)
    wi = (np.arange(np.prod(w_shape)).reshape(w_shape) % 11 - 5).astype(dtype)
    assert np.array_equal(abi.conv_dgrad(gi, x_shape, wi, s, p, d), direct.conv_backward_x(gi, x_shape, wi, s, p, d).astype(dtype))
    if dtype == np.float32:
        # MYGRAD_HIP_THIN=0 plans the same problem on the 16-row tiles: same bar
        os.environ["MYGRAD_HIP_THIN"] = "0"
        try:
            other = abi.conv_dgrad(g, x_shape, w, s, p, d)
        finally:
            del os.environ["MYGRAD_HIP_THIN"]
        assert rel_err(other, direct.conv_backward_x(g, x_shape, w, s, p, d)) <= tol


@pytest.mark.parametrize("dtype", [np.float32, np.float64])
@pytest.mark.parametrize("x_shape,w_shape,s,p,d", [
    ((8, 3, 101, 100), (64, 3, 7, 7), (2, 2), (3, 3), (1, 1)),     # too few positions for the kernel above in float32
    ((6, 4, 75, 81), (32, 4, 5, 5), (2, 2), (2, 2), (1, 1)),       # sixteen rows: four channels x four phases, odd extents
    ((4, 8, 90, 64), (48, 8, 3, 4), (2, 1), (1, 2), (1, 1)),       # two phases along the first axis only: no paired stores
    ((3, 2, 30, 41, 44), (16, 2, 3, 3, 3), (1, 2, 2), (1, 1, 1), (1, 1, 1)),
    ((16, 5, 4000), (32, 5, 9), (2,), (4,), (2,)),                 # dilation 2 under stride 2: one phase has no tap at all
])
def test_data_gradient_with_the_stride_phases_as_rows(abi, dtype, x_shape, w_shape, s, p, d):
    """A few channels under a stride where the one-position-per-lane kernel does not apply (double
    precision, or too few positions): the rows of the GEMM are (channel, stride phase) over the
    coarse grid.  MYGRAD_HIP_PHASE_ROWS=0 plans the same problem phase by phase: same bar."""
    rng = np.random.default_rng(2500 + x_shape[-1])
    tol = TOL[np.dtype(dtype)]
    w = (rng.standard_normal(w_shape) / np.sqrt(np.prod(w_shape[1:]))).astype(dtype)
    grid = direct.conv_forward(np.zeros(x_shape, dtype=dtype), w, s, p, d).shape
    g = rng.standard_normal(grid).astype(dtype)
    want = direct.conv_backward_x(g, x_shape, w, s, p, d)
    got = abi.conv_dgrad(g, x_shape, w, s, p, d)
    assert rel_err(got, want) <= tol
    assert np.array_equal(got, abi.conv_dgrad(g, x_shape, w, s, p, d))
    gi = rng.integers(-2, 3, grid).astype(dtype)
    wi = (np.arange(np.prod(w_shape)).reshape(w_shape) % 11 - 5).astype(dtype)
    assert np.array_equal(abi.conv_dgrad(gi, x_shape, wi, s, p, d), direct.conv_backward_x(gi, x_shape, wi, s, p, d).astype(dtype))
    os.environ["MYGRAD_HIP_PHASE_ROWS"] = "0"
    try:
        other = abi.conv_dgrad(g, x_shape, w, s, p, d)
    finally:
        del os.environ["MYGRAD_HIP_PHASE_ROWS"]
    assert rel_err(other, want) <= tol


# Every tile shape of the forward / data-gradient kernels, forced in turn (the planner would take
# one or two of them for any given problem): rows x positions, and for the data gradient under a
# stride the shapes of its fused stride phases.
ALL_TILES = ["128,128", "128,64", "64,256", "64,128", "32,256", "32,128", "16,256", "64,64", "96,128", "48,256"]
TILE_PROBLEMS = [
    # (x, w, stride, padding, dilation): odd extents, so that row ends and sample ends fall inside tiles
    ((3, 32, 29, 27), (160, 32, 3, 3), (1, 1), (1, 1), (1, 1)),       # 160 rows: one and a quarter tiles of 128
    ((2, 48, 31, 33), (48, 48, 3, 3), (2, 2), (1, 1), (1, 1)),        # stride 2 both ways: four fused phases
    ((2, 32, 20, 45), (64, 32, 3, 5), (1, 2), (1, 2), (1, 1)),        # stride 2 along the last axis only: two fused phases
    ((2, 16, 9, 17, 19), (32, 16, 3, 3, 3), (1, 1, 1), (1, 1, 1), (1, 1, 1)),  # three axes; folded taps where the tile allows
]


@pytest.mark.parametrize("dtype", [np.float32, np.float64])
@pytest.mark.parametrize("tile", ALL_TILES)
@pytest.mark.parametrize("problem", range(len(TILE_PROBLEMS)))
def test_every_tile_shape_of_the_gather_gemm(abi, monkeypatch, problem, tile, dtype):
    from mygrad_amd import _hip

    monkeypatch.setenv("MYGRAD_HIP_TINY", "0")
    monkeypatch.setenv("MYGRAD_HIP_TILE", tile)
    monkeypatch.setenv("MYGRAD_HIP_FUSE_MIN_ROW", "0")
    x_shape, w_shape, s, p, d = TILE_PROBLEMS[problem]
    rng = np.random.default_rng(2700 + problem)
    tol = TOL[np.dtype(dtype)]
    x = rng.standard_normal(x_shape).astype(dtype)
    w = (rng.standard_normal(w_shape) / np.sqrt(np.prod(w_shape[1:]))).astype(dtype)
    want = direct.conv_forward(x, w, s, p, d)
    got = abi.conv_fwd(x, w, s, p, d)
    print("forward:", _hip.last_plan(), flush=True)
    assert rel_err(got, want) <= tol
    g = rng.standard_normal(want.shape).astype(dtype)
    dx = abi.conv_dgrad(g, x_shape, w, s, p, d)
    print("data gradient:", _hip.last_plan(), flush=True)
    assert rel_err(dx, direct.conv_backward_x(g, x_shape, w, s, p, d)) <= tol
    # small integers: every sum is exact whatever the tile and however its K tiles are shared out
    xi = rng.integers(-3, 4, x_shape).astype(dtype)
    wi = rng.integers(-2, 3, w_shape).astype(dtype)
    gi = rng.integers(-2, 3, want.shape).astype(dtype)
    assert np.array_equal(abi.conv_fwd(xi, wi, s, p, d), direct.conv_forward(xi, wi, s, p, d).astype(dtype))
    assert np.array_equal(abi.conv_dgrad(gi, x_shape, wi, s, p, d), direct.conv_backward_x(gi, x_shape, wi, s, p, d).astype(dtype))


@pytest.mark.parametrize("x_shape,w_shape,row_tiles", [
    ((16, 32, 32, 32), (512, 32, 3, 3), 4),
    ((8, 16, 32, 32), (1024, 16, 3, 3), 8),
])
def test_row_tiles_of_a_position_block_on_one_xcd(abi, monkeypatch, x_shape, w_shape, row_tiles):
    """As many tiles as the device has block slots, 4 or 8 row tiles per position block: the blocks
    start on the tiles in chunks per XCD (every tile must still be computed exactly once), and with
    MYGRAD_HIP_XCD_CHUNK=0 on the tile of their own number; same results bit for bit."""
    from mygrad_amd import _hip

    monkeypatch.setenv("MYGRAD_HIP_TILE", "128,128,2")
    rng = np.random.default_rng(2900 + row_tiles)
    x = rng.standard_normal(x_shape).astype(np.float32)
    w = (rng.standard_normal(w_shape) / np.sqrt(np.prod(w_shape[1:]))).astype(np.float32)
    got = abi.conv_fwd(x, w, 1, 1, 1)
    assert f"x {row_tiles} row tiles" in _hip.last_plan() and "tile 128x128" in _hip.last_plan()
    assert rel_err(got, direct.conv_forward(x, w, (1, 1), (1, 1), (1, 1))) <= 2e-4
    monkeypatch.setenv("MYGRAD_HIP_XCD_CHUNK", "0")  # read at every launch
    assert np.array_equal(bits(got), bits(abi.conv_fwd(x, w, 1, 1, 1)))


WGRAD_TILES = ["48,64", "128,128", "64,64", "32,128", "32,64", "16,64"]


@pytest.mark.parametrize("dtype", [np.float32, np.float64])
@pytest.mark.parametrize("tile", WGRAD_TILES)
@pytest.mark.parametrize("x_shape,w_shape,s,p,d", [
    ((3, 32, 29, 27), (128, 32, 3, 3), (1, 1), (1, 1), (1, 1)),   # 288 columns: tiles of 128 overhang
    ((2, 48, 31, 33), (64, 48, 3, 3), (2, 2), (1, 1), (1, 1)),    # rows of grad that are no whole 16-byte pieces
])
def test_every_tile_shape_of_the_filter_gradient(abi, monkeypatch, x_shape, w_shape, s, p, d, tile, dtype):
    from mygrad_amd import _hip

    monkeypatch.setenv("MYGRAD_HIP_TINY", "0")
    monkeypatch.setenv("MYGRAD_HIP_WGRAD_TILE", tile)
    rng = np.random.default_rng(2800 + x_shape[-1])
    x = rng.standard_normal(x_shape).astype(dtype)
    grid = direct.conv_forward(x, np.zeros(w_shape, dtype=dtype), s, p, d).shape
    g = rng.standard_normal(grid).astype(dtype)
    got = abi.conv_wgrad(g, x, w_shape, s, p, d)
    print("filter gradient:", _hip.last_plan(), flush=True)
    assert rel_err(got, direct.conv_backward_w(g, x, w_shape, s, p, d)) <= TOL[np.dtype(dtype)]
    xi = rng.integers(-3, 4, x_shape).astype(dtype)
    gi = rng.integers(-2, 3, grid).astype(dtype)
    assert np.array_equal(abi.conv_wgrad(gi, xi, w_shape, s, p, d), direct.conv_backward_w(gi, xi, w_shape, s, p, d).astype(dtype))


# The filter gradient's K index is the position: the single-precision tap-major kernel reads, per
# position, a row of a table (window origin in x, which taps exist, what the sample adds to the
# offset into grad) instead of dividing the position into coordinates for every K tile.
POS_TABLE_CASES = [
    ((6, 16, 23, 23), (32, 16, 3, 3), (1, 1), (1, 1), (1, 1)),         # rows of grad that are no whole 16-byte pieces
    ((4, 32, 20, 24), (16, 32, 3, 3), (2, 2), (1, 1), (1, 1)),         # stride: taps missing on one side only
    ((3, 16, 31, 36), (64, 16, 7, 7), (2, 1), (3, 3), (1, 1)),         # 49 taps: both words of the tap mask
    ((2, 16, 9, 20, 20), (32, 16, 3, 3, 3), (1, 1, 1), (1, 1, 1), (1, 1, 1)),  # 27 taps, padding on three axes
    ((5, 48, 40, 40), (128, 48, 5, 5), (1, 1), (4, 4), (2, 2)),        # dilation; wide tiles, several column groups per thread
    ((2, 16, 12, 12), (16, 16, 3, 3), (1, 1), (2, 2), (1, 1)),         # padding wider than a tap step; one short K tile per split
    # channels that fill no group of 16 columns: one table row per column, its tap looked up in the position's mask
    ((8, 3, 45, 45), (64, 3, 7, 7), (2, 2), (3, 3), (1, 1)),           # 147 columns in two tiles of 80
    ((6, 5, 22, 26), (24, 5, 3, 3), (1, 1), (1, 1), (1, 1)),           # a short last row tile; rows of grad that are no whole pieces
    ((4, 20, 15, 15), (10, 20, 5, 5), (1, 1), (0, 0), (1, 1)),         # no padding: every tap exists everywhere
]


@pytest.mark.parametrize("x_shape,w_shape,s,p,d", POS_TABLE_CASES)
def test_filter_gradient_with_and_without_the_position_table(abi, monkeypatch, x_shape, w_shape, s, p, d):
    monkeypatch.setenv("MYGRAD_HIP_TINY", "0")  # small shapes: planned like large ones, or they take the table-driven kernel
    rng = np.random.default_rng(2600 + x_shape[-1])
    x = rng.standard_normal(x_shape).astype(np.float32)
    grid = direct.conv_forward(x, np.zeros(w_shape, dtype=np.float32), s, p, d).shape
    g = rng.standard_normal(grid).astype(np.float32)
    want = direct.conv_backward_w(g, x, w_shape, s, p, d)
    got = abi.conv_wgrad(g, x, w_shape, s, p, d)
    from mygrad_amd import _hip

    assert "tap-major" in _hip.last_plan()
    assert rel_err(got, want) <= TOL[np.dtype(np.float32)]
    # small integers: every sum is exact, so the result is the definition's bit for bit
    xi = rng.integers(-3, 4, x_shape).astype(np.float32)
    gi = rng.integers(-2, 3, grid).astype(np.float32)
    assert np.array_equal(abi.conv_wgrad(gi, xi, w_shape, s, p, d), direct.conv_backward_w(gi, xi, w_shape, s, p, d).astype(np.float32))
    # the same kernel on its own position arithmetic adds the same terms in the same order
    monkeypatch.setenv("MYGRAD_HIP_POS_TABLE", "0")
    assert np.array_equal(bits(got), bits(abi.conv_wgrad(g, x, w_shape, s, p, d)))


# Up to four filters in single precision (a layer that ends in one map or in the three colours
# of an image), or a first layer (channels that fill no K tile): the forward pass on the same
# kernel, one output position per lane.
THIN_FILTER_CASES = [
    ((64, 16, 64, 64), (3, 16, 3, 3), (1, 1), (1, 1), (1, 1)),
    ((256, 64, 64, 64), (1, 64, 1, 1), (1, 1), (0, 0), (1, 1)),     # one tap: sixteen channels per chunk
    ((112, 8, 97, 97), (4, 8, 7, 7), (2, 2), (3, 3), (1, 1)),       # strided reads
    ((4, 6, 20, 64, 64), (2, 6, 3, 3, 3), (1, 1, 1), (1, 1, 1), (1, 1, 1)),
    ((128, 48, 2048), (3, 48, 5), (1,), (4,), (2,)),
    ((64, 9, 64, 64), (4, 9, 5, 5), (1, 1), (2, 2), (1, 1)),        # 25 taps, 9 channels: one channel per group, chunks padded
    # a first layer with more than 64 filters: passes of 64 rows over the same positions
    ((128, 3, 64, 64), (96, 3, 4, 4), (2, 2), (1, 1), (1, 1)),      # a pass of 64 and one of 32
    ((64, 1, 64, 64), (130, 1, 3, 3), (1, 1), (1, 1), (1, 1)),      # three passes, two rows in the last
    # a first layer of 8, 16 and 32 filters: two, four and eight groups of four rows
    ((64, 3, 64, 64), (8, 3, 3, 3), (1, 1), (1, 1), (1, 1)),
    ((32, 3, 96, 96), (16, 3, 5, 5), (2, 2), (2, 2), (1, 1)),
    ((64, 2, 64, 64), (32, 2, 3, 3), (1, 1), (1, 1), (1, 1)),
]


@pytest.mark.parametrize("dtype", [np.float32, np.float64])
@pytest.mark.parametrize("case", range(len(THIN_FILTER_CASES)))
def test_forward_pass_with_up_to_four_filters(abi, dtype, case):
    x_shape, w_shape, s, p, d = THIN_FILTER_CASES[case]
    rng = np.random.default_rng(2400 + case)
    tol = TOL[np.dtype(dtype)]
    x = rng.standard_normal(x_shape).astype(dtype)
    w = (rng.standard_normal(w_shape) / np.sqrt(np.prod(w_shape[1:]))).astype(dtype)
    got = abi.conv_fwd(x, w, s, p, d)
    assert rel_err(got, direct.conv_forward(x, w, s, p, d)) <= tol
    assert np.array_equal(got, abi.conv_fwd(x, w, s, p, d))
    xi = rng.integers(-2, 3, x_shape).astype(dtype)
    wi = (np.arange(np.prod(w_shape)).reshape(w_shape) % 11 - 5).astype(dtype)
    assert np.array_equal(abi.conv_fwd(xi, wi, s, p, d), direct.conv_forward(xi, wi, s, p, d).astype(dtype))
    if dtype == np.float32:
        os.environ["MYGRAD_HIP_THIN"] = "0"  # the same problem on the 16-row tiles: same bar
        try:
            other = abi.conv_fwd(x, w, s, p, d)
        finally:
            del os.environ["MYGRAD_HIP_THIN"]
        assert rel_err(other, direct.conv_forward(x, w, s, p, d)) <= tol


def _random_medium_case(rng, m):
    """A random problem of 0.12 - 3 GFLOP: large enough to be planned like the benchmark's
    layers (whichever family its channel and filter counts select), small enough for the oracle."""
    C = int(rng.choice([1, 3, 8, 16, 20, 32, 48, 64]))
    F = int(rng.choice([2, 4, 10, 16, 24, 32, 64, 96]))
    taps = tuple(int(v) for v in rng.integers(1, 6 if m < 3 else 4, m))
    dil = tuple(int(v) for v in rng.integers(1, 3, m))
    stride = tuple(int(v) for v in rng.integers(1, 4, m))
    pad = tuple(int(v) for v in rng.integers(0, 3, m))
    grid = tuple(int(v) for v in rng.integers(6, {1: 900, 2: 60, 3: 20}[m], m))
    X = tuple((g - 1) * s + (t - 1) * d + 1 - 2 * p + int(rng.integers(0, s)) for g, s, t, d, p in zip(grid, stride, taps, dil, pad))
    if any(v < 1 for v in X):
        return None
    per_sample = 2 * int(np.prod(grid)) * C * F * int(np.prod(taps))
    N = max(1, -(-150_000_000 // per_sample))
    if N > 512 or N * per_sample > 3_000_000_000 or N * max(C * int(np.prod(X)), F * int(np.prod(grid))) > 50_000_000:
        return None
    return (N, C, *X), (F, C, *taps), stride, pad, dil


@pytest.mark.parametrize("dtype", [np.float32, np.float64])
@pytest.mark.parametrize("m", [1, 2, 3])
def test_conv_random_problems_of_benchmark_size(abi, dtype, m):
    rng = np.random.default_rng(2700 + m)
    tol = TOL[np.dtype(dtype)]
    done = 0
    while done < 10:
        case = _random_medium_case(rng, m)
        if case is None:
            continue
        x_shape, w_shape, s, p, d = case
        print("medium case", np.dtype(dtype).name, x_shape, w_shape, s, p, d, flush=True)
        x = rng.standard_normal(x_shape).astype(dtype)
        w = (rng.standard_normal(w_shape) / np.sqrt(np.prod(w_shape[1:]))).astype(dtype)
        want = direct.conv_forward(x, w, s, p, d)
        g = rng.standard_normal(want.shape).astype(dtype)
        assert rel_err(abi.conv_fwd(x, w, s, p, d), want) <= tol
        assert rel_err(abi.conv_dgrad(g, x_shape, w, s, p, d), direct.conv_backward_x(g, x_shape, w, s, p, d)) <= tol
        assert rel_err(abi.conv_wgrad(g, x, w_shape, s, p, d), direct.conv_backward_w(g, x, w_shape, s, p, d)) <= tol
        done += 1


@pytest.mark.parametrize("dtype", [np.float32, np.float64])
@pytest.mark.parametrize("filters", [10, 16])
def test_conv_whose_windows_step_over_the_only_row(abi, dtype, filters):
    """An axis of one element, padded by one, under a one-element window with stride 2: the
    windows sit on the two padding rows and never on x.  The output is zero, dw is zero, and dx
    is zero because no stride phase has a tap (the data gradient's tables are empty) -- on a
    problem large enough to be planned like any other."""
    x_shape, w_shape, s, p, d = (64, 20, 1, 2048), (filters, 20, 1, 3), (2, 1), (1, 1), (1, 1)
    rng = np.random.default_rng(2600 + filters)
    x = rng.standard_normal(x_shape).astype(dtype)
    w = rng.standard_normal(w_shape).astype(dtype)
    out = abi.conv_fwd(x, w, s, p, d)
    assert out.shape == (64, filters, 2, 2048) and not out.any()
    g = rng.standard_normal(out.shape).astype(dtype)
    dx = abi.conv_dgrad(g, x_shape, w, s, p, d)
    assert dx.shape == x_shape and not dx.any()
    assert not direct.conv_backward_x(g, x_shape, w, s, p, d).any()
    dw = abi.conv_wgrad(g, x, w_shape, s, p, d)
    assert dw.shape == w_shape and not dw.any()


def _random_thin_case(rng, m, rows_are_channels):
    """A random problem with few rows (channels for the data gradient, filters for the forward
    pass) and enough positions for the one-position-per-lane kernel: strides of 1 or 2 (1, 2 or 4
    stride phases, or more: then the other kernels run), windows of 1 to 5, dilation, padding."""
    few = int(rng.integers(1, 5))
    many = int(rng.choice([8, 16, 20, 33]))
    C, F = (few, many) if rows_are_channels else (many, few)
    taps = tuple(int(v) for v in rng.integers(1, 6 if m < 3 else 4, m))
    dil = tuple(int(v) for v in rng.integers(1, 3, m))
    stride = tuple(int(v) for v in rng.integers(1, 3, m))
    pad = tuple(int(v) for v in rng.integers(0, 3, m))
    grid = tuple(int(v) for v in rng.integers(20, {1: 600, 2: 70, 3: 24}[m], m))
    X = tuple((g - 1) * s + (t - 1) * d + 1 - 2 * p + int(rng.integers(0, s)) for g, s, t, d, p in zip(grid, stride, taps, dil, pad))
    if any(v < 1 for v in X):
        return None
    coarse = int(np.prod([-(-v // s) for v, s in zip(X, stride)])) if rows_are_channels else int(np.prod(grid))
    # enough positions, and enough work not to be planned as a problem of a few microseconds
    N = max(-(-300000 // coarse), -(-120_000_000 // (2 * coarse * C * F * int(np.prod(taps)))))
    if N * max(C, F) * int(np.prod(X)) > 60_000_000:
        return None
    return (N, C, *X), (F, C, *taps), stride, pad, dil


@pytest.mark.parametrize("m", [1, 2, 3])
@pytest.mark.parametrize("which", ["data gradient, few channels", "forward, few filters"])
def test_random_problems_with_few_rows(abi, m, which):
    rows_are_channels = which.startswith("data")
    rng = np.random.default_rng(2500 + 10 * m + rows_are_channels)
    done = 0
    while done < 8:
        case = _random_thin_case(rng, m, rows_are_channels)
        if case is None:
            continue
        x_shape, w_shape, s, p, d = case
        print("thin case", which, x_shape, w_shape, s, p, d, flush=True)
        w = (rng.standard_normal(w_shape) / np.sqrt(np.prod(w_shape[1:]))).astype(np.float32)
        wi = (np.arange(np.prod(w_shape)).reshape(w_shape) % 11 - 5).astype(np.float32)
        if rows_are_channels:
            grid = direct.conv_forward(np.zeros(x_shape, dtype=np.float32), w, s, p, d).shape
            g = rng.standard_normal(grid).astype(np.float32)
            assert rel_err(abi.conv_dgrad(g, x_shape, w, s, p, d), direct.conv_backward_x(g, x_shape, w, s, p, d)) <= 2e-4
            gi = rng.integers(-2, 3, grid).astype(np.float32)
            assert np.array_equal(abi.conv_dgrad(gi, x_shape, wi, s, p, d), direct.conv_backward_x(gi, x_shape, wi, s, p, d).astype(np.float32))
        else:
            x = rng.standard_normal(x_shape).astype(np.float32)
            assert rel_err(abi.conv_fwd(x, w, s, p, d), direct.conv_forward(x, w, s, p, d)) <= 2e-4
            xi = rng.integers(-2, 3, x_shape).astype(np.float32)
            assert np.array_equal(abi.conv_fwd(xi, wi, s, p, d), direct.conv_forward(xi, wi, s, p, d).astype(np.float32))
        done += 1


AWKWARD_CHANNEL_CASES = [
    # (x shape, w shape, stride, pad, dilation): channel / filter counts that are no multiple of 16
    ((8, 24, 48, 48), (40, 24, 3, 3), (1, 1), (1, 1), (1, 1)),
    ((6, 40, 40, 40), (32, 40, 3, 3), (2, 2), (1, 1), (1, 1)),
    ((4, 32, 64, 64), (56, 32, 3, 3), (1, 1), (0, 0), (2, 2)),
    ((16, 100, 400), (72, 100, 5), (1,), (2,), (1,)),
    ((2, 24, 12, 20, 20), (24, 24, 3, 3, 3), (1, 1, 1), (1, 1, 1), (1, 1, 1)),
]


@pytest.mark.parametrize("dtype", [np.float64, np.float32])
@pytest.mark.parametrize("case", range(len(AWKWARD_CHANNEL_CASES)))
def test_conv_awkward_channel_counts(abi, dtype, case):
    x_shape, w_shape, s, p, d = AWKWARD_CHANNEL_CASES[case]
    rng = np.random.default_rng(700 + case)
    tol = TOL[np.dtype(dtype)]
    x = rng.standard_normal(x_shape).astype(dtype)
    w = (rng.standard_normal(w_shape) / np.sqrt(np.prod(w_shape[1:]))).astype(dtype)
    want_out = direct.conv_forward(x, w, s, p, d)
    g = rng.standard_normal(want_out.shape).astype(dtype)
    assert rel_err(abi.conv_fwd(x, w, s, p, d), want_out) <= tol
    assert rel_err(abi.conv_dgrad(g, x_shape, w, s, p, d), direct.conv_backward_x(g, x_shape, w, s, p, d)) <= tol
    assert rel_err(abi.conv_wgrad(g, x, w_shape, s, p, d), direct.conv_backward_w(g, x, w_shape, s, p, d)) <= tol


# Counts that fill no K tile (channels forward, filters in the data gradient) or no row tile, read where they lie:
# one row short of and one beyond a K tile, of each row tile and of a group of 16 columns; an odd number of
# positions.  From 2e8 flops on such counts are contracted in K tiles with dead rows; which kernel a pass
# takes is part of the case: (x, w, stride, padding, dilation, forward, data gradient in float32, in float64).
RAGGED_CASES = [
    ((2, 47, 41, 37), (83, 47, 3, 3), (1, 1), (1, 1), (1, 1), "tap-major tile", "tap-major tile", "tap-major tile"),
    # four fused stride phases, K tiles 16 and 32 deep; two
    ((12, 45, 47, 43), (65, 45, 3, 3), (2, 2), (1, 1), (1, 1), "tap-major tile", "x16, 1 phase(s) (4 fused", "4 phase(s) (1 fused"),
    ((12, 31, 47, 43), (93, 31, 3, 3), (2, 2), (1, 1), (1, 1), "tap-major tile", "x32, 1 phase(s) (4 fused", "4 phase(s) (1 fused"),
    ((6, 45, 33, 41), (61, 45, 3, 3), (1, 2), (1, 1), (1, 1), "tap-major tile", "(2 fused", "2 phase(s) (1 fused"),
    # the taps of the last axis folded into the rows: forward (96 x 128), data gradient (48 x 256)
    ((6, 45, 30, 64), (31, 45, 3, 3), (1, 1), (1, 1), (1, 1), "folded taps tile 96x128", "tap-major tile", "tap-major tile"),
    ((12, 13, 30, 64), (45, 13, 3, 3), (1, 1), (1, 1), (1, 1), "tap-major tile", "folded taps tile 48x256", "folded taps tile 48x256"),
    # the stride phases of a few channels as rows
    ((4, 4, 113, 113), (95, 4, 5, 5), (2, 2), (2, 2), (1, 1), "fwd", "stride phases as rows", "stride phases as rows"),
    ((2, 49, 1501), (129, 49, 9), (1,), (4,), (1,), "tap-major tile", "tap-major tile", "tap-major tile"),
    # one tap: the filter gradient written without a pass over partial sums
    ((1, 81, 9001), (161, 81, 1), (1,), (0,), (1,), "tap-major tile", "tap-major tile", "tap-major tile"),
    ((10, 29, 6, 25, 25), (47, 29, 3, 3, 1), (1, 2, 2), (1, 0, 0), (1, 1, 1), "tap-major tile", "(4 fused", "4 phase(s) (1 fused"),
]


@pytest.mark.parametrize("dtype", [np.float64, np.float32])
@pytest.mark.parametrize("case", range(len(RAGGED_CASES)))
def test_conv_counts_that_fill_no_tile_in_place(abi, dtype, case):
    from mygrad_amd import _hip

    x_shape, w_shape, s, p, d, fwd, dx32, dx64 = RAGGED_CASES[case]
    rng = np.random.default_rng(1700 + case)
    print("ragged", np.dtype(dtype).name, x_shape, w_shape, s, p, d, flush=True)
    # small integers: every sum is exact in both precisions, so the results are compared as they are
    x = rng.integers(-3, 4, x_shape).astype(dtype)
    w = rng.integers(-2, 3, w_shape).astype(dtype)
    want = direct.conv_forward(x, w, s, p, d).astype(dtype)
    assert 2.0 * want.size * w[0].size >= 2e8
    g = rng.integers(-2, 3, want.shape).astype(dtype)
    assert np.array_equal(abi.conv_fwd(x, w, s, p, d), want)
    assert fwd in _hip.last_plan(), _hip.last_plan()
    assert np.array_equal(abi.conv_dgrad(g, x_shape, w, s, p, d), direct.conv_backward_x(g, x_shape, w, s, p, d).astype(dtype))
    assert (dx32 if dtype == np.float32 else dx64) in _hip.last_plan(), _hip.last_plan()
    assert np.array_equal(abi.conv_wgrad(g, x, w_shape, s, p, d), direct.conv_backward_w(g, x, w_shape, s, p, d).astype(dtype))
    # what lies behind a sample's channels (the next sample's first ones) stays out of its sums, NaN and all
    if x_shape[0] > 1:
        xn, gn = x.copy(), g.copy()
        xn[1:], gn[1:] = np.nan, np.nan
        assert np.array_equal(abi.conv_fwd(xn, w, s, p, d)[0], want[0])
        dx = direct.conv_backward_x(g[:1], (1, *x_shape[1:]), w, s, p, d).astype(dtype)
        assert np.array_equal(abi.conv_dgrad(gn, x_shape, w, s, p, d)[0], dx[0])


@pytest.mark.parametrize("tile", ["128,128", "128,64", "96,128", "64,256", "64,128", "48,256", "32,256", "32,128", "16,256"])
def test_dead_rows_in_every_tile(abi, monkeypatch, tile):
    """float32, one K tile of dead rows per tap, in every tile shape of the forward and data-gradient kernels (some
    have an instance of their own for it)."""
    from mygrad_amd import _hip

    monkeypatch.setenv("MYGRAD_HIP_TILE", tile)
    rng = np.random.default_rng(45)
    x_shape, w_shape, conf = (3, 45, 41, 37), (61, 45, 3, 3), ((1, 1), (1, 1), (1, 1))
    x, w = rng.integers(-3, 4, x_shape).astype(np.float32), rng.integers(-2, 3, w_shape).astype(np.float32)
    want = direct.conv_forward(x, w, *conf).astype(np.float32)
    g = rng.integers(-2, 3, want.shape).astype(np.float32)
    print("dead rows", tile, flush=True)
    for got, ref in ((abi.conv_fwd(x, w, *conf), want), (abi.conv_dgrad(g, x_shape, w, *conf), direct.conv_backward_x(g, x_shape, w, *conf).astype(np.float32))):
        assert f"tap-major tile {tile.replace(',', 'x')}x" in _hip.last_plan(), _hip.last_plan()
        assert np.array_equal(got, ref)


@pytest.mark.parametrize("dtype", [np.float64, np.float32])
@pytest.mark.parametrize("x_shape,w_shape,s", [
    ((2, 45, 41, 37), (128, 45, 3, 3), 1),   # ragged channels, forward on 128-row tiles
    ((2, 128, 41, 37), (45, 128, 3, 3), 1),  # ragged filters, data gradient on 128-row tiles
    ((5, 128, 41, 37), (45, 128, 3, 3), 2),
    ((3, 1001, 400), (512, 1001, 1), 1),     # a matrix product
])
def test_ragged_counts_in_tensors_too_large_for_buffer_loads(abi, monkeypatch, dtype, x_shape, w_shape, s):
    """What tensors of 2 GiB and more run on, reached with small ones: every pass launches a kernel and
    writes its result."""
    from mygrad_amd import _hip

    monkeypatch.setenv("MYGRAD_HIP_BUFFER_LIMIT", "4096")
    rng = np.random.default_rng(list(x_shape))
    nd = len(w_shape) - 2
    conf = (s,) * nd, (w_shape[2] // 2,) * nd, (1,) * nd
    print("large", np.dtype(dtype).name, x_shape, w_shape, s, flush=True)
    x, w = rng.integers(-3, 4, x_shape).astype(dtype), rng.integers(-2, 3, w_shape).astype(dtype)
    want = direct.conv_forward(x, w, *conf).astype(dtype)
    g = rng.integers(-2, 3, want.shape).astype(dtype)
    assert np.array_equal(abi.conv_fwd(x, w, *conf), want)
    assert "table-driven" in _hip.last_plan()
    assert np.array_equal(abi.conv_dgrad(g, x_shape, w, *conf), direct.conv_backward_x(g, x_shape, w, *conf).astype(dtype))
    assert "table-driven" in _hip.last_plan()
    assert np.array_equal(abi.conv_wgrad(g, x, w_shape, *conf), direct.conv_backward_w(g, x, w_shape, *conf).astype(dtype))
    assert "table-driven" in _hip.last_plan()


# A pass that does not fill the device is shared out by how many blocks its tiles make, not only by their
# padding: (dtype, x, w, stride, padding, pass, what the plan must say, what it must not)
SMALL_PASSES = [
    (np.float32, (1, 7, 17, 28), (37, 7, 3, 3), 1, 0, "fwd", "tile 16x64x", None),      # 24 blocks, 2 on 64 rows
    (np.float32, (4, 4, 14, 69), (84, 4, 5, 3), (1, 2), (0, 1), "fwd", "tile 16x64x", None),
    (np.float32, (64, 8, 56, 56), (24, 8, 1, 1), 1, 0, "fwd", "table-driven", "tile 16x64x"),  # thousands of blocks either way
    (np.float64, (25, 7, 19, 29), (102, 7, 1, 3), 2, 0, "fwd", "tile 16x64x", None),
    (np.float64, (8, 259, 26, 31), (27, 259, 3, 3), (1, 2), (0, 2), "dx", "tap-major", "tile 96x128x"),
    (np.float64, (1, 808, 3317), (93, 808, 1), 1, 0, "dx", "tap-major", "tile 96x128x"),
    (np.float64, (1, 184, 375), (41, 184, 1), 1, 0, "fwd", "tap-major", "tile 48x256x"),
    (np.float32, (1, 72, 23, 42), (55, 72, 3, 1), 1, (1, 0), "fwd", "tap-major", "tile 64x256x"),
    (np.float32, (1, 216, 171), (96, 216, 1), 1, 0, "fwd", "tap-major", "tile 96x128x"),
]


@pytest.mark.parametrize("case", range(len(SMALL_PASSES)))
def test_small_passes_are_spread_over_the_device(abi, case):
    from mygrad_amd import _hip

    dtype, x_shape, w_shape, s, p, which, has, has_not = SMALL_PASSES[case]
    nd = len(x_shape) - 2
    s, p = ((v,) * nd if isinstance(v, int) else v for v in (s, p))
    rng = np.random.default_rng(case)
    x, w = rng.integers(-3, 4, x_shape).astype(dtype), rng.integers(-2, 3, w_shape).astype(dtype)
    want = direct.conv_forward(x, w, s, p, (1,) * nd).astype(dtype)
    if which == "fwd":
        got = abi.conv_fwd(x, w, s, p, 1)
    else:
        g = rng.integers(-2, 3, want.shape).astype(dtype)
        want = direct.conv_backward_x(g, x_shape, w, s, p, (1,) * nd).astype(dtype)
        got = abi.conv_dgrad(g, x_shape, w, s, p, 1)
    plan = _hip.last_plan()
    assert np.array_equal(got, want)
    assert has in plan and (has_not is None or has_not not in plan), plan


@pytest.mark.parametrize("m,k,n", [(353, 777, 2631), (622, 1357, 491), (463, 102, 2473)])
def test_small_products_add_up_no_longer_chains(abi, m, k, n):
    """Spreading K over blocks also shortens the sum that one accumulator takes: the bound is what these products
    showed where their K was cut (2.4e-7, 2.2e-7, 1.6e-7), a third above it; uncut they show up to 5.0e-7."""
    rng = np.random.default_rng(m)
    a, b = rng.standard_normal((m, k)).astype(np.float32), rng.standard_normal((k, n)).astype(np.float32)
    want = a.astype(np.float64) @ b
    got = abi.conv_fwd(b[None], a[:, :, None], 1, 0, 1)[0]
    assert np.linalg.norm(got - want) <= 3.3e-7 * np.linalg.norm(want)


@pytest.mark.parametrize("x_shape,w_shape,bound", [
    ((1, 2639, 1862), (329, 2639, 1), 3.5e-7),   # what these showed against 64 bits with their K cut into 8, 7, 5
    ((1, 2294, 1235), (473, 2294, 1), 3.1e-7),   # splits (2.9e-7, 2.5e-7, 2.5e-7, ...), a fifth above it; in one run
    ((1, 747, 877), (1947, 747, 1), 3.1e-7),     # 7.7e-7, 6.3e-7, 5.3e-7
    ((1, 693, 664), (2112, 693, 1), 2.8e-7),
    ((15, 51, 12603), (24, 51, 5), 7.8e-7),      # 6.5e-7; 8.9e-7 with half as many splits
    ((32, 24, 56, 56), (24, 24, 3, 3), 5.7e-7),  # 4.7e-7; 6.3e-7
])
def test_filter_gradient_adds_up_runs_of_a_bounded_length(abi, x_shape, w_shape, bound):
    rng = np.random.default_rng(w_shape[0])
    pad = (w_shape[2] // 2 if len(x_shape) == 4 else 0,) * (len(x_shape) - 2)
    ones = (1,) * len(pad)
    grid = tuple(a + 2 * q - t + 1 for a, q, t in zip(x_shape[2:], pad, w_shape[2:]))
    x = rng.standard_normal(x_shape).astype(np.float32)
    g = rng.standard_normal((x_shape[0], w_shape[0], *grid)).astype(np.float32)
    got = abi.conv_wgrad(g, x, w_shape, 1, pad, 1)
    g64, x64 = g.astype(np.float64), np.pad(x.astype(np.float64), [(0, 0), (0, 0)] + [(q, q) for q in pad])
    want = np.empty(w_shape)
    for tap in np.ndindex(*w_shape[2:]):
        part = x64[(slice(None), slice(None), *(slice(t, t + n) for t, n in zip(tap, grid)))]
        want[(slice(None), slice(None), *tap)] = sum(a.reshape(a.shape[0], -1) @ b.reshape(b.shape[0], -1).T for a, b in zip(g64, part))
    assert np.linalg.norm(got - want) <= bound * np.linalg.norm(want)


@pytest.mark.parametrize("dtype", [np.float64, np.float32])
@pytest.mark.parametrize("filters", [1, 5, 12, 15, 17, 33, 60])
def test_filter_gradient_of_filters_that_fill_no_row_tile(abi, dtype, filters):
    """The rows beyond the last filter are computed from whatever follows in grad, or zeros, and not stored."""
    from mygrad_amd import _hip

    for x_shape, w_shape in (((7, 32, 23, 21), (filters, 32, 3, 3)), ((1, 16, 999), (filters, 16, 1)), ((1, 48, 40, 41), (filters, 48, 1, 3))):
        nd = len(x_shape) - 2
        rng = np.random.default_rng(filters)
        x = rng.integers(-3, 4, x_shape).astype(dtype)
        grid = tuple(a - t + 1 for a, t in zip(x_shape[2:], w_shape[2:]))
        g = rng.integers(-2, 3, (x_shape[0], filters, *grid)).astype(dtype)
        conf = (1,) * nd, (0,) * nd, (1,) * nd
        print("few filters", np.dtype(dtype).name, x_shape, w_shape, flush=True)
        assert np.array_equal(abi.conv_wgrad(g, x, w_shape, *conf), direct.conv_backward_w(g, x, w_shape, *conf).astype(dtype))
        assert "tap-major tile" in _hip.last_plan()


@pytest.mark.parametrize("dtype,channels,has", [(np.float32, 5, "one position per lane"), (np.float32, 11, "one position per lane"),
                                                (np.float32, 13, "tap-major tile"), (np.float64, 8, "x8, 1 phase")])
def test_single_taps_of_few_channels(abi, dtype, channels, has):
    """1x1 convolutions whose channels fill no K tile of 16 mostly: no dead rows where a kernel without them is faster."""
    from mygrad_amd import _hip

    rng = np.random.default_rng(channels)
    x_shape, w_shape = (24, channels, 56, 56), (1600 // channels, channels, 1, 1)
    x, w = rng.integers(-3, 4, x_shape).astype(dtype), rng.integers(-2, 3, w_shape).astype(dtype)
    want = direct.conv_forward(x, w, (1, 1), (0, 0), (1, 1)).astype(dtype)
    got = abi.conv_fwd(x, w, 1, 0, 1)
    assert np.array_equal(got, want)
    assert 2 * want.size * channels >= 2e8 and has in _hip.last_plan(), _hip.last_plan()


@pytest.mark.parametrize("dtype", [np.float64, np.float32])
def test_filter_gradient_of_a_tap_with_one_channel_beyond_a_group(abi, dtype):
    """17 channels are 32 columns of two groups, fifteen of them computed twice: on table rows they are 17 of 32."""
    from mygrad_amd import _hip

    rng = np.random.default_rng(17)
    x, g = rng.integers(-3, 4, (2, 17, 61, 63)).astype(dtype), rng.integers(-2, 3, (2, 800, 61, 63)).astype(dtype)
    conf = (1, 1), (0, 0), (1, 1)
    assert np.array_equal(abi.conv_wgrad(g, x, (800, 17, 1, 1), *conf), direct.conv_backward_w(g, x, (800, 17, 1, 1), *conf).astype(dtype))
    assert "table rows tile 64x32" in _hip.last_plan(), _hip.last_plan()


# Shapes picked so that, between them, the code paths of the tap-major kernels run: persistent blocks that
# stream through several tiles and K slices, strided dgrad phases, filter counts that are not a multiple of
# four (padded packed rows), wide and square filter-gradient tiles, and an odd number of positions per
# sample (grad tile loaded element by element instead of 16 bytes per lane).  (Every tile shape is
# forced in tests of its own, above.)
KERNEL_VARIANT_CASES = [
    # x shape, w shape, stride, padding, dilation
    ((8, 128, 28, 28), (128, 128, 3, 3), (1, 1), (1, 1), (1, 1)),   # wgrad 128x128
    ((32, 64, 28, 28), (64, 64, 3, 3), (1, 1), (1, 1), (1, 1)),     # wgrad 64x64
    ((64, 64, 28, 28), (64, 64, 2, 2), (1, 1), (0, 0), (1, 1)),
    ((16, 128, 29, 29), (256, 128, 3, 3), (2, 2), (1, 1), (1, 1)),  # four dgrad phases
    ((4, 16, 15, 15), (32, 16, 3, 3), (1, 1), (1, 1), (1, 1)),      # 225 positions per sample (odd)
    ((6, 16, 20, 20), (10, 16, 3, 3), (1, 1), (1, 1), (1, 1)),      # F = 10: packed rows padded to 12
    ((5, 48, 9, 33), (16, 48, 3, 5), (1, 2), (1, 0), (1, 2)),       # 16-row tiles, dilation, mixed strides
    ((3, 32, 12, 12, 12), (32, 32, 3, 3, 3), (1, 1, 1), (1, 1, 1), (1, 1, 1)),  # 3-D, 32-row tiles
]


@pytest.mark.parametrize("dtype", [np.float32, np.float64])
@pytest.mark.parametrize("case", range(len(KERNEL_VARIANT_CASES)))
def test_conv_shapes_that_reach_every_kernel_variant(abi, dtype, case):
    x_shape, w_shape, s, p, d = KERNEL_VARIANT_CASES[case]
    rng = np.random.default_rng(700 + case)
    tol = TOL[np.dtype(dtype)]
    print("variant case", np.dtype(dtype).name, x_shape, w_shape, s, p, d, flush=True)
    x = rng.standard_normal(x_shape).astype(dtype)
    w = (rng.standard_normal(w_shape) * (2.0 / np.prod(w_shape[1:])) ** 0.5).astype(dtype)
    want_out = direct.conv_forward(x, w, s, p, d)
    g = rng.standard_normal(want_out.shape).astype(dtype)
    assert rel_err(abi.conv_fwd(x, w, s, p, d), want_out) <= tol
    assert rel_err(abi.conv_dgrad(g, x_shape, w, s, p, d), direct.conv_backward_x(g, x_shape, w, s, p, d)) <= tol
    dw = abi.conv_wgrad(g, x, w_shape, s, p, d)
    assert rel_err(dw, direct.conv_backward_w(g, x, w_shape, s, p, d)) <= tol
    assert np.array_equal(bits(dw), bits(abi.conv_wgrad(g, x, w_shape, s, p, d)))  # fixed summation order


def _check_conv_config(abi, seed, dtype, x_shape, w_shape, w_scale, s, p, d, np_oracle_batch):
    """Full-size check: against the definition-level C reference everywhere, and
    against the NumPy restatement of the reference on the leading batch items."""
    rng = np.random.default_rng(seed)
    tol = TOL[np.dtype(dtype)]
    x = rng.standard_normal(x_shape).astype(dtype)
    w = (rng.standard_normal(w_shape) * w_scale).astype(dtype)
    out = abi.conv_fwd(x, w, s, p, d)
    g = rng.standard_normal(out.shape).astype(dtype)
    dx = abi.conv_dgrad(g, x_shape, w, s, p, d)
    dw = abi.conv_wgrad(g, x, w_shape, s, p, d)

    assert rel_err(out, direct.conv_forward(x, w, s, p, d)) <= tol
    assert rel_err(dx, direct.conv_backward_x(g, x_shape, w, s, p, d)) <= tol
    assert rel_err(dw, direct.conv_backward_w(g, x, w_shape, s, p, d)) <= tol

    # adjoint identity <conv(x,w), g> = <x, dx> = <w, dw>, in float64
    lhs = np.vdot(out.astype(np.float64), g.astype(np.float64))
    eps = 1e-9 if dtype == np.float64 else 1e-3
    scale = np.linalg.norm(out.astype(np.float64)) * np.linalg.norm(g.astype(np.float64))
    assert abs(lhs - np.vdot(x.astype(np.float64), dx.astype(np.float64))) <= eps * scale
    assert abs(lhs - np.vdot(w.astype(np.float64), dw.astype(np.float64))) <= eps * scale

    nb = np_oracle_batch
    conf = dict(stride=s, padding=p, dilation=d)
    ref_out = ora.conv_forward(x[:nb], w, validate=False, **conf)
    assert rel_err(out[:nb], ref_out) <= tol
    ref_dx = ora.conv_backward_x(g[:nb], x[:nb].shape, x.dtype, w, **conf)
    assert rel_err(dx[:nb], ref_dx) <= tol
    if nb == x_shape[0]:
        assert rel_err(dw, ora.conv_backward_w(g, x, w_shape, **conf)) <= tol


def test_conv_config1(abi):
    _check_conv_config(abi, 1001, np.float64, (32, 3, 32, 32), (16, 3, 3, 3), 1 / np.sqrt(27), (1, 1), (1, 1), (1, 1), 32)


def test_conv_config3a(abi):
    _check_conv_config(abi, 1003, np.float32, (128, 64, 56, 56), (64, 64, 3, 3), np.sqrt(2 / 576), (1, 1), (1, 1), (1, 1), 2)


def test_conv_config3b_literal(abi):
    _check_conv_config(abi, 1004, np.float32, (128, 128, 28, 28), (256, 128, 3, 3), np.sqrt(2 / 1152), (2, 2), (1, 1), (1, 1), 4)


def test_conv_config4_shape(abi):
    _check_conv_config(abi, 1005, np.float64, (16, 32, 128, 128), (32, 32, 5, 5), 1 / np.sqrt(800), (2, 1), (4, 4), (2, 2), 1)


def test_conv_config4_literal(abi):
    _check_conv_config(abi, 1005, np.float64, (16, 32, 128, 128), (32, 32, 5, 5), 1 / np.sqrt(800), (2, 1), (4, 2), (2, 2), 1)


def test_conv_config5(abi):
    _check_conv_config(abi, 1006, np.float32, (8, 16, 32, 64, 64), (32, 16, 3, 3, 3), np.sqrt(2 / 432), (1, 1, 1), (1, 1, 1), (1, 1, 1), 1)


def test_conv_stem_three_channels_seven_by_seven_stride_two(abi):
    # a quarter of the batch of bench.py's `stem` workload, its literal (flooring) shape
    _check_conv_config(abi, 1017, np.float32, (32, 3, 224, 224), (64, 3, 7, 7), np.sqrt(2 / 147), (2, 2), (3, 3), (1, 1), 1)


def test_conv_wgrad_is_run_to_run_identical(abi):
    rng = np.random.default_rng(5)
    x = rng.standard_normal((16, 24, 30, 30)).astype(np.float32)
    g = rng.standard_normal((16, 40, 28, 28)).astype(np.float32)
    first = abi.conv_wgrad(g, x, (40, 24, 3, 3), 1, 0, 1)
    for _ in range(3):
        assert np.array_equal(bits(first), bits(abi.conv_wgrad(g, x, (40, 24, 3, 3), 1, 0, 1)))


def test_abi_rejects_bad_arguments(abi):
    import ctypes

    from mygrad_amd import _hip

    lib = _hip.lib()
    desc, _ = abi.conv_desc((1, 1, 4, 4), (1, 1, 3, 3), np.float32, 1, 0, 1)
    assert lib.mg_conv_fwd(desc, None, None, None) == _hip.MG_ERR_BAD_ARG
    assert "null" in _hip.last_error()
    desc.dtype = 7
    assert lib.mg_conv_fwd(desc, 1, 1, 1) == _hip.MG_ERR_UNSUPPORTED
    desc.dtype = 0
    desc.G[2] = 99
    assert lib.mg_conv_fwd(desc, 1, 1, 1) == _hip.MG_ERR_BAD_ARG
    pdesc, _ = abi.pool_desc((2, 4, 4), np.float32, (2, 2), 2)
    pdesc.nd = 5
    assert lib.mg_maxpool_fwd(pdesc, 1, 1) == _hip.MG_ERR_UNSUPPORTED
    pdesc, _ = abi.pool_desc((2, 4, 4), np.float32, (2, 2), 2)
    assert lib.mg_maxpool_fwd_argmax(pdesc, 1, 1, None) == _hip.MG_ERR_BAD_ARG
    assert lib.mg_maxpool_bwd_argmax(pdesc, None, 1, 1) == _hip.MG_ERR_BAD_ARG
    wide, _ = abi.pool_desc((2, 20, 20), np.float32, (17, 16), 1)  # 272 positions: more than a byte tells apart
    assert lib.mg_maxpool_fwd_argmax(wide, 1, 1, 1) == _hip.MG_ERR_UNSUPPORTED
    assert lib.mg_maxpool_bwd_argmax(wide, 1, 1, 1) == _hip.MG_ERR_UNSUPPORTED
    assert "256" in _hip.last_error()
    huge = ctypes.c_void_p()
    assert lib.mg_malloc(ctypes.byref(huge), 1 << 60) == _hip.MG_ERR_OOM


def test_blocks_given_back_are_handed_out_again_in_stream_order(abi):
    """mg_free keeps the block, mg_malloc of a like size returns it without touching the
    driver; work enqueued on the block before it was given back runs before its next use."""
    import os

    from mygrad_amd import _device, _hip

    if os.environ.get("MYGRAD_HIP_POOL", "")[:1] == "0":
        pytest.skip("block reuse is switched off (MYGRAD_HIP_POOL=0)")
    size = 3 << 20
    first = _device.DeviceBuffer(size)
    ptr = first.ptr
    first.free()
    again = _device.DeviceBuffer(size - 4096)  # rounds to the same block size
    assert again.ptr == ptr
    # a kernel still writing the block when it is given back: the next owner's upload lands after it
    x = np.arange(size // 8, dtype=np.float64)
    src = _device.DeviceBuffer(size)
    src.upload(x)
    _hip.check(_hip.lib().mg_memcpy_d2d(again.ptr, src.ptr, size))  # enqueued, not waited for
    again.free()
    reused = _device.DeviceBuffer(size)
    assert reused.ptr == ptr
    reused.upload(-x)
    got = np.empty_like(x)
    reused.download_into(got)
    assert np.array_equal(got, -x)
    # a block of another size class does not take this one
    small = _device.DeviceBuffer(1024)
    assert small.ptr != ptr


@pytest.mark.gpu
def test_mfma_probe_reports_plausible_rates():
    """The diagnostic entry point runs and its figures are ordered the way the fp64
    kernels rely on: the four-block 4x4x4 MFMA outruns the 16x16x4 one."""
    from mygrad_amd import _hip

    f32 = _hip.probe_mfma("f32_16x16x4", 2)
    wide = _hip.probe_mfma("f64_16x16x4", 2)
    quad = _hip.probe_mfma("f64_4x4x4_4b", 2)
    assert 20.0 < f32 < 200.0 and 5.0 < wide < 100.0 and 5.0 < quad < 100.0
    assert quad > wide
    with pytest.raises(_hip.HipError):
        _hip.probe_mfma("f32_16x16x4", 9)


@pytest.mark.gpu
def test_stream_probe_moves_what_it_says():
    """The memory diagnostic stores every 16-byte piece of the large buffer from piece
    i / share of the small one (first value plus one), or loads the large buffer and stores
    every share-th piece to the small one; sizes and alignment are checked."""
    from mygrad_amd import _device, _hip

    pieces = 1000
    small_host = np.arange(4 * pieces, dtype=np.float32).reshape(pieces, 4)
    big, small = _device.DeviceBuffer(16 * pieces), _device.DeviceBuffer(16 * pieces)
    small.upload(small_host)
    got = np.empty((pieces, 4), dtype=np.float32)
    for share in (1, 2, 8):
        assert _hip.probe_stream(big.ptr, small.ptr, 16 * pieces, share, True) > 0.0
        big.download_into(got)
        want = small_host[np.arange(pieces) // share].copy()
        want[:, 0] += 1.0
        assert np.array_equal(got, want)
    _hip.probe_stream(big.ptr, small.ptr, 16 * pieces, 0, True)
    big.download_into(got)
    assert np.array_equal(got, np.tile(np.array([2.0, 2.0, 3.0, 4.0], dtype=np.float32), (pieces, 1)))
    big.upload(small_host)
    _hip.check(_hip.lib().mg_memset_zero(small.ptr, 16 * pieces))
    _hip.probe_stream(big.ptr, small.ptr, 16 * pieces, 4, False)
    small.download_into(got)
    assert np.array_equal(got[: pieces // 4], small_host[::4]) and not got[pieces // 4:].any()
    _hip.probe_stream(big.ptr, small.ptr, 16 * pieces, 0, False)  # loads only
    small.download_into(got)
    assert np.array_equal(got[: pieces // 4], small_host[::4])
    with pytest.raises(_hip.HipError):
        _hip.probe_stream(big.ptr, small.ptr, 24, 1, True)
    with pytest.raises(_hip.HipError):
        _hip.probe_stream(big.ptr + 4, small.ptr, 16, 1, True)


def test_per_launch_timing_records_chains_and_pauses():
    """``mg_timing_enable`` / ``mg_timing_read`` give one (kernel, milliseconds) record per timed
    launch, in order; ``mg_timing_pause`` suspends the recording without dropping what was
    recorded (what bench.py uses to time a sample of its steps)."""
    import mygrad_amd as mg
    from mygrad_amd import _hip

    a = mg.device_tensor(np.ones((256, 1024), dtype=np.float32))
    b = mg.device_tensor(np.full((256, 1024), 2.0, dtype=np.float32))
    with mg.no_autodiff:
        _hip.timing_enable(True)
        try:
            mg.multiply(a, b)
            _hip.timing_pause(True)
            for _ in range(3):
                mg.multiply(a, b)
            _hip.timing_pause(False)
            mg.multiply(a, b)
            mg.multiply(a, b)
            records = _hip.timing_read()
        finally:
            _hip.timing_enable(False)
    assert [k for k, _ in records] == ["elementwise"] * 3
    assert all(0.0 < ms < 5.0 for _, ms in records)
    with mg.no_autodiff:
        mg.multiply(a, b)  # timing off: nothing is recorded, nothing is left over
    _hip.timing_enable(True)
    try:
        assert _hip.timing_read() == []
    finally:
        _hip.timing_enable(False)


# float32 on operands split into three bf16 parts: (x, w, padding, dilation, tile; "" leaves the tile to the plan).  Odd
# extents, so that row ends and sample ends fall inside tiles; channels and filters that fill no 16.
SPLIT_PROBLEMS = [
    ((3, 32, 29, 27), (160, 32, 3, 3), (1, 1), (1, 1), "128,128"),           # odd window; a quarter row tile
    ((9, 45, 31, 33), (101, 45, 2, 3), (1, 2), (1, 1), "64,192"),            # even window, ragged counts
    ((2, 16, 23, 300), (64, 16, 3, 3), (1, 1), (1, 1), "48,256"),            # rows longer than a tile: stages of one row of taps
    ((17, 61, 13, 13), (64, 61, 5, 5), (2, 2), (1, 2), "64,128"),             # the tiles of several samples; dilation
    ((2, 48, 5000), (48, 48, 8), (3,), (2,), "48,256"),                      # one axis, even window
    ((310, 24, 7, 7), (32, 24, 3, 3), (2, 2), (2, 2), "32,256"),              # planes of 49: samples rounded up to whole loads
    ((1, 16, 4099), (16, 16, 31), (15,), (1,), "16,256"),                    # as many taps as a position's bits
    ((4, 45, 9, 11, 13), (76, 45, 2, 3, 3), (1, 0, 1), (1, 2, 1), ""),       # three axes
    ((11, 32, 19, 21), (48, 32, 5, 3), (0, 0), (1, 1), ""),                  # no padding: the data gradient's positions outnumber
    ((37, 32, 61), (80, 32, 9), (0,), (2,), ""),                             # its rows along every axis, and samples overlap in them
    ((3, 32, 9, 11, 12), (48, 32, 3, 3, 3), (1, 0, 0), (1, 1, 2), ""),
    ((2, 512, 6, 5), (512, 512, 3, 3), (1, 1), (1, 1), ""),                  # every tile shared out
    ((7, 45, 27, 31), (70, 45, 3, 3), (1, 1), (1, 1), "64,192"),             # odd window
    ((2, 32, 70, 75), (64, 32, 3, 3), (1, 1), (1, 1), "64,128"),             # patches of more rows than threads
    ((9, 16, 4099), (64, 16, 3), (1,), (1,), "64,192"),                      # enough tiles for a pass over marked ones to go by waves
    ((17, 16, 4099), (48, 16, 4), (2,), (1,), "48,256"),
    ((17, 16, 4099), (32, 16, 4), (2,), (1,), "32,256"),
    ((17, 16, 4099), (16, 16, 3), (1,), (1,), "16,256"),
]


def _split_passes(abi, monkeypatch, problem):
    """passes(x, w, g, split=True): forward pass and data gradient of a problem, on split operands or without."""
    from mygrad_amd import _hip

    x_shape, _, p, d, tile = SPLIT_PROBLEMS[problem]
    s = (1,) * len(p)

    def passes(x, w, g, split=True):
        with monkeypatch.context() as m:
            m.setenv("MYGRAD_HIP_TINY", "0")
            m.setenv("MYGRAD_HIP_SPLIT_MIN", "0")
            m.setenv("MYGRAD_HIP_SPLIT", "1" if split else "0")
            if tile:
                m.setenv("MYGRAD_HIP_TILE", tile)
            out = abi.conv_fwd(x, w, s, p, d)
            plans = [_hip.last_plan()]
            dx = abi.conv_dgrad(g, x_shape, w, s, p, d)
            plans.append(_hip.last_plan())
        print(*plans, sep="\n", flush=True)
        for plan in plans:
            assert plan.endswith("three bf16 parts") == split
            assert not split or tile.replace(",", "x") in plan
        return out, dx

    return passes


@pytest.mark.parametrize("problem", range(len(SPLIT_PROBLEMS)))
def test_products_of_three_bf16_parts(abi, monkeypatch, problem):
    x_shape, w_shape, p, d, _ = SPLIT_PROBLEMS[problem]
    s = (1,) * len(p)
    rng = np.random.default_rng(3100 + problem)
    passes = _split_passes(abi, monkeypatch, problem)

    # small integers: every sum is exact
    xi, wi = rng.integers(-3, 4, x_shape).astype(np.float32), rng.integers(-2, 3, w_shape).astype(np.float32)
    want = direct.conv_forward(xi, wi, s, p, d).astype(np.float32)
    gi = rng.integers(-2, 3, want.shape).astype(np.float32)
    out, dx = passes(xi, wi, gi)
    assert np.array_equal(out, want)
    assert np.array_equal(dx, direct.conv_backward_x(gi, x_shape, wi, s, p, d).astype(np.float32))
    # against 64 bits: a sum of K terms takes six roundings into its accumulator for every 32 of them (three for 16).  Rounded off towards
    # zero, a number is off by 2^-23 * E[m^-2]^1/2 / 3^1/2 = 5.06e-8 of itself on average (significands m of 1 to 2, evenly in
    # their logarithm), and after a share of its roundings a sum of normal terms has that share of its variance: together 5.06e-8 *
    # (6 K / 32 / 2)^1/2 of the result; a quarter for the spread of a sample, K in whole blocks of 16 channels
    x, w, g = (rng.standard_normal(shape).astype(np.float32) for shape in (x_shape, w_shape, want.shape))
    x64, w64, g64 = (a.astype(np.float64) for a in (x, w, g))
    exact = direct.conv_forward(x64, w64, s, p, d), direct.conv_backward_x(g64, x_shape, w64, s, p, d)
    for got, plain, ref, count in zip(passes(x, w, g), passes(x, w, g, split=False), exact, (w_shape[1], w_shape[0])):
        assert not np.array_equal(got, plain)  # (nothing was left to the single-precision kernels)
        terms = -(-count // 16) * 16 * np.prod(w_shape[2:])
        assert np.linalg.norm(got - ref) <= 1.25 * 5.06e-8 * np.sqrt(6 * terms / 64) * np.linalg.norm(ref)
    # what the parts cannot hold: infinite and NaN operands, sums that overflow, and near the smallest numbers; and the pass after it
    at = tuple(n // 2 for n in x_shape)
    for value in (np.inf, np.nan, 3e38):
        xs, gs = x.copy(), g.copy()
        xs[at] = value
        gs[tuple(n // 2 for n in g.shape)] = value
        with np.errstate(all="ignore"):
            ws = w * np.float32(4)
        for got, plain in zip(passes(xs, ws, gs), passes(xs, ws, gs, split=False)):
            finite = np.isfinite(plain)
            assert not finite.all() and np.array_equal(got[~finite], plain[~finite], equal_nan=True)
            # (two sums in single precision: each off by the bound above, with an accumulator that rounds a third more often)
            terms = max(w_shape[:2]) * np.prod(w_shape[2:])
            off = np.linalg.norm((got[finite] - plain[finite]).astype(np.float64)) / np.linalg.norm(plain[finite].astype(np.float64))
            assert off <= 2 * 1.25 * 5.06e-8 * np.sqrt(8 * terms / 64)
    scales = (1e-30, 1.0, 1e-30), (1e-36, 1e9, 1e-36), (1e9, 1e-36, 1e9), (1e-20, 1e-20, 1e-20)
    for scale in scales:
        xs, ws, gs = (v * np.float32(c) for v, c in zip((x, w, g), scale))
        x64, w64, g64 = (a.astype(np.float64) for a in (xs, ws, gs))
        exact = direct.conv_forward(x64, w64, s, p, d), direct.conv_backward_x(g64, x_shape, w64, s, p, d)
        for got, ref, count in zip(passes(xs, ws, gs), exact, (w_shape[1], w_shape[0])):
            terms = -(-count // 16) * 16 * np.prod(w_shape[2:])
            # (subnormal sums round to multiples of 2^-149)
            grain = 2.0**-149 * np.sqrt(8 * terms / 32 * ref.size) if max(np.abs(ref).max(), 1e-30) == 1e-30 else 0.0
            assert np.linalg.norm(got - ref) <= 1.25 * 5.06e-8 * np.sqrt(8 * terms / 64) * np.linalg.norm(ref) + grain
    again = passes(xi, wi, gi)
    assert np.array_equal(bits(again[0]), bits(out)) and np.array_equal(bits(again[1]), bits(dx))


@pytest.mark.parametrize("problem", [0, 1, 3, 5, 8, 11, 12])
def test_products_of_three_bf16_parts_keep_single_precision(abi, monkeypatch, problem):
    """Sums of few terms, where an error that long dense sums hide would show."""
    x_shape, w_shape, p, d, _ = SPLIT_PROBLEMS[problem]
    s = (1,) * len(p)
    rng = np.random.default_rng(3200 + problem)
    passes = _split_passes(abi, monkeypatch, problem)
    normal = lambda shape: rng.standard_normal(shape).astype(np.float32)
    x, w = normal(x_shape), normal(w_shape)
    g = normal(direct.conv_forward(x, w, s, p, d).shape)

    def exact(x, w, g):
        x, w, g = (a.astype(np.float64) for a in (x, w, g))
        return direct.conv_forward(x, w, s, p, d), direct.conv_backward_x(g, x_shape, w, s, p, d)

    # one tap of one channel per filter, and no channel twice: every sum is one product.  What the six products leave out is at
    # most 2^-24 of it (second parts of at most 2^-8 and third ones of 2^-17 of their values), x0 w0 is exact, the five small products
    # round off 2^-29 each and their sum with x0 w0 2^-24
    few = np.zeros_like(w)
    for f in range(min(w_shape[:2])):
        at = np.unravel_index(f * 7 % np.prod(w_shape[2:]), w_shape[2:])
        few[(f, f, *at)] = w[(f, f, *at)]
    for got, ref in zip(passes(x, few, g), exact(x, few, g)):
        assert np.all(np.abs(got - ref) <= (2 + 5 / 32) * 2.0**-24 * np.abs(ref))
    # dense, behind a relu, and few values not zero: a sum of large products rounds off once in a step, of 32 terms or of 16 under an odd
    # tap, 5.06e-8 of itself each time (see above), the rest 3.5e-8.  (All six products in one sum: twice as much.)
    for share in (1.0, 0.5, 0.02):
        xs, gs = (np.where(rng.random(a.shape) < share, a if share == 1.0 else np.abs(a), np.float32(0)) for a in (x, g))
        for got, ref, count in zip(passes(xs, w, gs), exact(xs, w, gs), (w_shape[1], w_shape[0])):
            steps = -(-count // 16) * (np.prod(w_shape[2:]) + 1) / 2
            assert np.linalg.norm(got - ref) <= (1.25 * 5.06e-8 * np.sqrt(steps / 2) + 3.5e-8) * np.linalg.norm(ref)


@pytest.mark.parametrize("problem", [0, 1, 3, 5, 8, 12, 14, 15, 16, 17])
def test_products_of_three_bf16_parts_lose_no_operand(abi, monkeypatch, problem):
    """Operands whose low bits, or all of them, are below the smallest number of bf16: the products are normal numbers all the same."""
    x_shape, w_shape, p, d, _ = SPLIT_PROBLEMS[problem]
    s = (1,) * len(p)
    rng = np.random.default_rng(3300 + problem)
    passes = _split_passes(abi, monkeypatch, problem)
    few = np.zeros(w_shape, np.float32)  # one product a sum, as above
    for f in range(min(w_shape[:2])):
        few[(f, f, *np.unravel_index(f * 7 % np.prod(w_shape[2:]), w_shape[2:]))] = rng.uniform(1, 2)
    x = rng.uniform(1, 2, x_shape).astype(np.float32)
    g = rng.uniform(1, 2, direct.conv_forward(x, few, s, p, d).shape).astype(np.float32)
    for tiny, other in ((1e-41, 3e4), (1e-38, 3e4), (1e-43, 1e7), (1e-35, 3e36)):
        for a, b, some in ((tiny, other, 1), (other, tiny, 1), (tiny, other, 9), (1.0, tiny, 1)):
            # one element in nine is tiny, the others are as they are: the pass has sums of either kind
            where = np.arange(x.size).reshape(x.shape) % some == 0, np.arange(g.size).reshape(g.shape) % some == 0
            xs, gs = (np.where(i, v * np.float32(a), v).astype(np.float32) for i, v in zip(where, (x, g)))
            ws = few * np.float32(b)
            x64, w64, g64 = (v.astype(np.float64) for v in (xs, ws, gs))
            exact = direct.conv_forward(x64, w64, s, p, d), direct.conv_backward_x(g64, x_shape, w64, s, p, d)
            for got, ref in zip(passes(xs, ws, gs), exact):
                assert np.all(np.abs(got - ref) <= (2 + 5 / 32) * 2.0**-24 * np.abs(ref) + 2.0**-149)


@pytest.mark.parametrize("problem", [0, 1, 5, 7, 10, 12])
def test_products_of_three_bf16_parts_keep_odd_values_apart(abi, monkeypatch, problem):
    """What the parts cannot hold in one sample leaves every bit of another one alone."""
    x_shape, w_shape, p, d, _ = SPLIT_PROBLEMS[problem]
    rng = np.random.default_rng(3400 + problem)
    passes = _split_passes(abi, monkeypatch, problem)
    x, w = (rng.standard_normal(shape).astype(np.float32) for shape in (x_shape, w_shape))
    g = rng.standard_normal(direct.conv_forward(x, w, (1,) * len(p), p, d).shape).astype(np.float32)
    plain = passes(x, w, g)
    # samples that no tile of 256 positions shares with the first one
    apart = [1 + -(-256 // np.prod(out.shape[2:])) for out in plain]
    for value in (np.inf, np.nan, 1e-40):
        xs, gs = x.copy(), g.copy()
        for v in (xs, gs):
            if value == 1e-40:
                v[0] *= np.float32(1e-40)
            else:
                v[(0, *(n // 2 for n in v.shape[1:]))] = value
        for got, was, first in zip(passes(xs, w, gs), plain, apart):
            assert first < len(was)
            assert np.array_equal(bits(got[first:]), bits(was[first:])) and not np.array_equal(got[0], was[0])


# (x, w, padding, whether the forward pass runs on split operands, and why not)
SPLIT_RULES = [
    ((128, 64, 56, 56), (64, 64, 3, 3), (1, 1), True),
    ((16, 45, 16001), (83, 45, 9), (4,), True),
    ((28, 64, 56, 56), (64, 64, 3, 3), (1, 1), False),        # 6.5 GFLOP
    ((2, 57, 16936), (125, 57, 15), (0,), False),             # K in fewer slices
    ((70, 113, 38, 78), (17, 113, 3, 5), (0, 0), False),      # patches that only fit tiles of twice the rows
    ((40, 285, 34, 55), (36, 285, 5, 1), (2, 0), False),      # large patches for their products
    ((59, 56, 930), (443, 56, 3), (1,), False),               # three taps
]


@pytest.mark.parametrize("rule", range(len(SPLIT_RULES)))
def test_which_passes_run_on_three_bf16_parts(abi, monkeypatch, rule):
    from mygrad_amd import _hip

    x_shape, w_shape, p, split = SPLIT_RULES[rule]
    rng = np.random.default_rng(3500 + rule)
    x, w = (rng.standard_normal(shape, dtype=np.float32) for shape in (x_shape, w_shape))
    out = abi.conv_fwd(x, w, (1,) * len(p), p, (1,) * len(p))
    plan = _hip.last_plan()
    print(plan, flush=True)
    assert plan.endswith("three bf16 parts") == split
    single = None
    if split:
        monkeypatch.setenv("MYGRAD_HIP_SPLIT", "0")
        single = abi.conv_fwd(x, w, (1,) * len(p), p, (1,) * len(p))
        assert not _hip.last_plan().endswith("three bf16 parts")
    # 200 of the results, each from its window; single precision rounds once a term, 2.5e-8 of the sum as it stands on average
    padded = np.pad(x, ((0, 0), (0, 0), *((q, q) for q in p)))
    flat = w.reshape(w_shape[0], -1).astype(np.float64)
    terms = flat.shape[1]
    off = norm = off_single = 0.0
    for _ in range(200):
        n, *at = (rng.integers(size) for size in (x_shape[0], *out.shape[2:]))
        window = padded[(n, slice(None), *(slice(i, i + k) for i, k in zip(at, w_shape[2:])))]
        ref = flat @ window.reshape(-1).astype(np.float64)
        off, norm = off + np.sum((out[(n, slice(None), *at)] - ref) ** 2), norm + np.sum(ref**2)
        if split:
            off_single += np.sum((single[(n, slice(None), *at)] - ref) ** 2)
    assert np.sqrt(off / norm) <= 1.25 * 2.5e-8 * np.sqrt(terms / 2)
    # no further off than the single-precision instruction, which rounds eight times as often
    assert not split or off <= off_single


def lost_bits_of_operands(gradient, g, x, distinct=True):
    """Values below 2**-109 have bits that three bf16 parts lose.  One among others (and a filter or channel that is zero throughout): no sum can
    tell, and the gradient stays on the parts.  A filter's or a channel's worth of them: the single-precision gradient, bit for bit."""
    for odd in range(2):
        operands = [g.copy(), x.copy()]
        middle = tuple(n // 2 for n in operands[odd].shape)
        if middle[1] + 1 < operands[odd].shape[1]:
            operands[odd][:, -1] = 0
        operands[odd][middle] = 0
        without = gradient(*operands)
        assert not distinct or not np.array_equal(without, gradient(*operands, False))
        for value in (1e-36, 1e-40):
            operands[odd][middle] = value
            assert np.array_equal(bits(gradient(*operands)), bits(without))
        operands[odd][:, 0] *= np.float32(1e-41)
        operands[1 - odd] *= np.float32(2.0**40)
        assert np.array_equal(bits(gradient(*operands)), bits(gradient(*operands, False)))


# (x, w, stride, padding, dilation, tile): filter gradients on three bf16 parts, a kernel each (waves along filters, column tiles, quads of a row)
SPLIT_GRADIENTS = [
    ((8, 64, 9, 17), (64, 64, 3, 3), (1, 1), (1, 1), (1, 1), "2,2,2"),        # whole tiles; rows that end among four columns
    ((5, 17, 13, 30), (70, 17, 2, 7), (1, 1), (0, 3), (1, 1), "2,2,2"),       # 14 taps: two chunks; runs of columns; one channel past a group
    ((16, 33, 14, 13), (65, 33, 3, 3), (1, 2), (1, 1), (1, 1), "2,2,2"),      # strided: two tasks a wave; three column tiles
    ((9, 16, 5, 7, 12), (33, 16, 3, 3, 3), (2, 1, 1), (1, 1, 0), (1, 1, 2), "1,2,4"),  # planes of a volume that are outside
    ((8, 32, 11, 20), (31, 32, 2, 3), (1, 1), (1, 1), (1, 1), "1,2,2"),       # two rows a stage
    ((8, 16, 27, 27), (130, 16, 3, 3), (2, 2), (1, 1), (1, 1), "4,2,1"),      # every other row and column; one column tile for two
    ((3, 48, 12, 67), (40, 48, 3, 3), (1, 1), (1, 1), (1, 1), "1,1,8"),
    ((1, 40, 6, 45), (32, 40, 1, 3), (1, 1), (0, 1), (1, 1), "1,1,4"),        # one sample: eight runs of columns
    ((8, 45, 501), (83, 45, 9), (1,), (4,), (1,), "1,1,8"),                   # along the only axis
    ((3, 16, 1003), (64, 16, 4), (1,), (2,), (2,), "2,2,2"),
    ((2, 30, 301), (20, 30, 5), (2,), (0,), (2,), "1,2,4"),
    ((64, 16, 1, 5), (16, 16, 1, 3), (1, 1), (0, 1), (1, 1), "1,1,8"),        # fewer columns than a stage has
    # single-precision kernels behind them whose splits are added in sixteen and in four runs
    ((8, 16, 4001), (16, 16, 9), (1,), (4,), (1,), "1,1,8"),
    ((8, 32, 4001), (64, 32, 9), (1,), (4,), (1,), "2,2,2"),
    # Along the only axis, padded by more than a stage's columns: the second stage of a walk, or a later one, begins one to three columns
    # ahead of its rows too.  (Filters enough that a block has several stages of a walk.)
    *(((8, 32, 701), (300, 32, 9), (1,), (p,), (1,), "2,2,2") for p in (9, 10, 11)),
    *(((8, 16, 1501), (256, 16, t), (1,), (p,), (1,), "1,2,4") for p, t in ((17, 18), (18, 18), (19, 20), (26, 27))),
    *(((8, 16, 2001), (300, 16, 5), (1,), (p,), (1,), "1,1,8") for p in (33, 34, 35)),
    *(((8, 32, 1401), (300, 32, 2), (2,), (p,), (1,), "2,2,2") for p in (17, 18, 19)),
    ((8, 16, 1501), (256, 16, 9), (2,), (35,), (1,), "1,2,4"),
    ((8, 16, 1501), (256, 16, 8), (1,), (21,), (3,), "1,2,4"),
    ((8, 16, 3, 901), (250, 16, 3, 9), (1, 1), (0, 18), (1, 1), "1,2,4"),     # three rows to the only row of results
]


@pytest.mark.parametrize("problem", range(len(SPLIT_GRADIENTS)))
def test_filter_gradients_on_three_bf16_parts(abi, monkeypatch, problem):
    from mygrad_amd import _hip

    x_shape, w_shape, s, p, d, tile = SPLIT_GRADIENTS[problem]
    rng = np.random.default_rng(3600 + problem)

    def gradient(g, x, split=True):
        with monkeypatch.context() as m:
            m.setenv("MYGRAD_HIP_SPLIT_MIN", "0")
            m.setenv("MYGRAD_HIP_SPLIT", "1" if split else "0")
            m.setenv("MYGRAD_HIP_SPLIT_TILE", tile)
            dw = abi.conv_wgrad(g, x, w_shape, s, p, d)
            plan = _hip.last_plan()
            print(plan, flush=True)
            assert plan.endswith("three bf16 parts") == split
        return dw

    xi = rng.integers(-3, 4, x_shape).astype(np.float32)
    grid = direct.conv_forward(xi, np.zeros(w_shape, np.float32), s, p, d).shape
    gi = rng.integers(-2, 3, grid).astype(np.float32)
    # small integers: every sum is exact
    want = direct.conv_backward_w(gi, xi, w_shape, s, p, d).astype(np.float32)
    whole = gradient(gi, xi)
    assert np.array_equal(whole, want)
    # against 64 bits: a sum takes two roundings for every 32 terms (its large products, and the small ones), each 5.06e-8 of it as it stands
    # then (see test_products_of_three_bf16_parts), the rest 3.5e-8; 32 terms are four positions of eight segments, of which some are dead
    x, g = rng.standard_normal(x_shape).astype(np.float32), rng.standard_normal(grid).astype(np.float32)
    exact = direct.conv_backward_w(g.astype(np.float64), x.astype(np.float64), w_shape, s, p, d)
    got, single = gradient(g, x), gradient(g, x, split=False)
    assert not np.array_equal(got, single)
    off, norm = np.linalg.norm(got - exact), np.linalg.norm(exact)
    terms = grid[0] * np.prod(grid[2:])
    assert off <= (1.25 * 5.06e-8 * np.sqrt(2 * 2 * terms / 64) + 3.5e-8) * norm
    assert off <= np.linalg.norm(single - exact)
    # what the parts cannot hold: the single-precision kernel's gradient, bit for bit, and the one after it on the parts again
    for value in (np.inf, np.nan):
        for odd in range(2):
            operands = [g.copy(), x.copy()]
            operands[odd][tuple(n // 2 for n in operands[odd].shape)] = value
            assert np.array_equal(bits(gradient(*operands)), bits(gradient(*operands, split=False)))
    lost_bits_of_operands(gradient, g, x)
    assert np.array_equal(bits(gradient(gi, xi)), bits(whole))
    assert np.array_equal(bits(gradient(g, x)), bits(got))


# (x, w, stride, padding, whether the filter gradient runs on parts)
SPLIT_GRADIENT_RULES = [
    ((128, 64, 56, 56), (64, 64, 3, 3), (1, 1), (1, 1), True),
    ((16, 45, 16001), (83, 45, 9), (1,), (4,), True),
    ((8, 16, 32, 64, 64), (32, 16, 3, 3, 3), (1, 1, 1), (1, 1, 1), True),
    ((16, 64, 28, 28), (64, 64, 3, 3), (1, 1), (1, 1), False),         # 0.9 GFLOP
    ((69, 205, 38, 11), (481, 205, 3, 1), (1, 1), (1, 0), False),      # three taps of a tile's nine
    ((128, 64, 55, 55), (128, 64, 3, 3), (2, 2), (1, 1), False),       # stages of one quad, seven of which share a row's lines of memory
]


@pytest.mark.parametrize("rule", range(len(SPLIT_GRADIENT_RULES)))
def test_which_filter_gradients_run_on_three_bf16_parts(abi, rule):
    from mygrad_amd import _hip

    x_shape, w_shape, s, p, split = SPLIT_GRADIENT_RULES[rule]
    grid = tuple((n + 2 * q - t) // v + 1 for n, q, t, v in zip(x_shape[2:], p, w_shape[2:], s))
    x, g = np.ones(x_shape, np.float32), np.ones((x_shape[0], w_shape[0], *grid), np.float32)
    dw = abi.conv_wgrad(g, x, w_shape, s, p, (1,) * len(p))
    print(_hip.last_plan(), flush=True)
    assert _hip.last_plan().endswith("three bf16 parts") == split
    centre = tuple(t // 2 for t in w_shape[2:])  # of the window: without padding there
    assert np.all(dw[(slice(None), slice(None), *centre)] == x_shape[0] * np.prod(grid))


def test_launches_behind_filter_gradients_on_parts_are_timed_apart(abi):
    from mygrad_amd import _hip

    x, g = np.ones((64, 64, 56, 56), np.float32), np.ones((64, 64, 56, 56), np.float32)
    _hip.timing_enable(True)
    try:
        abi.conv_wgrad(g, x, (64, 64, 3, 3), (1, 1), (1, 1), (1, 1))
        assert _hip.last_plan().endswith("three bf16 parts")
        kernels = [kernel for kernel, _ in _hip.timing_read() if kernel != "copy"]
    finally:
        _hip.timing_enable(False)
    assert kernels == ["conv_wgrad", "gated", "wgrad_reduce"]


# (x, w, stride, padding, dilation, shape): forward passes with few terms on three bf16 parts (10 * (16 filters) + 16 positions of a wave)
FEW_TERMS = [
    ((3, 3, 33, 45), (64, 3, 7, 7), (2, 2), (3, 3), (1, 1), 43),    # a first layer; the last tile of a plane is short
    ((2, 3, 40, 67), (70, 3, 3, 3), (1, 1), (1, 1), (1, 1), 42),    # two tiles of filters, most of the second one's beyond the last
    ((5, 1, 9, 9), (8, 1, 5, 5), (1, 1), (0, 0), (1, 1), 22),       # fewer positions than a wave has
    ((2, 5, 30, 21), (33, 5, 3, 4), (3, 1), (2, 0), (2, 3), 24),    # unequal axes
    ((3, 21, 1501), (17, 21, 9), (1,), (4,), (1,), 24),             # 189 terms; runs of a row
    ((2, 2, 4000), (40, 2, 15), (2,), (0,), (2,), 43),
    ((1, 24, 6, 700), (48, 24, 1, 3), (1, 1), (0, 1), (1, 1), 42),  # rows longer than a tile: along them
    ((4, 7, 5, 600), (65, 7, 2, 2), (1, 1), (0, 0), (1, 1), 43),
    ((1, 1, 3), (1, 1, 1), (1,), (0,), (1,), 22),                   # one term
    ((8, 3, 64, 64), (16, 3, 3, 3), (1, 1), (1, 1), (1, 1), 22),    # a single-precision filter gradient whose splits are added in sixteen runs
]


@pytest.mark.parametrize("problem", range(len(FEW_TERMS)))
def test_forward_of_few_terms_on_three_bf16_parts(abi, monkeypatch, problem):
    from mygrad_amd import _hip

    x_shape, w_shape, s, p, d, shape = FEW_TERMS[problem]
    rng = np.random.default_rng(3700 + problem)

    def forward(x, w, few=True):
        with monkeypatch.context() as m:
            m.setenv("MYGRAD_HIP_FEW", str(shape if few else 0))
            m.setenv("MYGRAD_HIP_SPLIT", "1" if few else "0")
            out = abi.conv_fwd(x, w, s, p, d)
            assert ("few terms" in _hip.last_plan()) == few
        return out

    xi, wi = rng.integers(-3, 4, x_shape).astype(np.float32), rng.integers(-2, 3, w_shape).astype(np.float32)
    # small integers: every sum is exact
    whole = forward(xi, wi)
    assert np.array_equal(whole, direct.conv_forward(xi, wi, s, p, d))
    # against 64 bits: as in test_filter_gradients_on_three_bf16_parts, a rounding for every 32 terms
    x, w = rng.standard_normal(x_shape).astype(np.float32), rng.standard_normal(w_shape).astype(np.float32)
    exact = direct.conv_forward(x.astype(np.float64), w.astype(np.float64), s, p, d)
    got, single = forward(x, w), forward(x, w, few=False)
    off, norm, terms = np.linalg.norm(got - exact), np.linalg.norm(exact), int(np.prod(w_shape[1:]))
    assert off <= (1.25 * 5.06e-8 * np.sqrt(-(-terms // 32) / 2) + 3.5e-8) * norm
    assert terms < 6 or off <= np.linalg.norm(single - exact)
    # what the parts cannot hold: single precision's values, and the bits of far results as they were
    for value in (np.inf, np.nan, 3e38, 1e-40):
        for odd in range(2):
            operands = [x * np.float32(4), w * np.float32(4)]
            operands[odd][tuple(n // 2 for n in operands[odd].shape)] = value
            with np.errstate(all="ignore"):
                some, plain, far = forward(*operands), forward(*operands, few=False), forward(x * np.float32(4), w * np.float32(4))
            finite = np.isfinite(plain)
            assert np.array_equal(some[~finite], plain[~finite], equal_nan=True) and np.all(np.isfinite(some[finite]))
            if odd == 0 and x_shape[0] > 1:
                assert np.array_equal(bits(some[0]), bits(far[0]))
    # one value of low bits that parts lose, beside a filter and a sample of zeros: no sum can tell, and all stay on the parts
    for odd in range(2):
        operands = [x.copy(), w.copy()]
        for v in operands:
            v[len(v) // 2 + 1 :][:1] = 0
        middle = tuple(n // 2 for n in operands[odd].shape)
        operands[odd][middle] = 0
        without = forward(*operands)
        operands[odd][middle] = 1e-36
        assert terms < 6 or np.array_equal(bits(forward(*operands)), bits(without))
    # one term a sum, of values below the smallest number of bf16: the single-precision instruction's results, to its rounding
    tiny = np.zeros_like(w)
    tiny.reshape(w_shape[0], -1)[:, 0] = 1e-41
    assert np.array_equal(forward(x * np.float32(2.0**40), tiny), forward(x * np.float32(2.0**40), tiny, few=False))
    assert np.array_equal(bits(forward(xi, wi)), bits(whole))


@pytest.mark.parametrize("x_shape, w_shape, s, p, few", [((64, 3, 225, 225), (64, 3, 7, 7), 2, 3, True), ((25, 24, 6716), (178, 24, 5), 1, 2, True),
                                                         ((111, 1, 211, 211), (11, 1, 3, 3), 2, 2, False), ((100, 16, 16, 16), (32, 16, 3, 3), 1, 1, False),
                                                         ((4, 3, 16, 64, 64), (32, 3, 3, 3, 3), 1, 1, False), ((128, 64, 56, 56), (64, 64, 3, 3), 1, 1, False)])
def test_which_forward_passes_run_as_few_terms(abi, x_shape, w_shape, s, p, few):
    from mygrad_amd import _hip

    out = abi.conv_fwd(np.ones(x_shape, np.float32), np.ones(w_shape, np.float32), s, p)
    assert ("few terms" in _hip.last_plan()) == few
    middle = tuple(n // 2 for n in out.shape[2:])
    assert np.all(out[(slice(None), slice(None), *middle)] == np.prod(w_shape[1:]))


@pytest.mark.parametrize("problem", [n for n, case in enumerate(FEW_TERMS) if np.prod(case[1][1:]) <= 160])
def test_filter_gradients_of_few_terms_on_three_bf16_parts(abi, monkeypatch, problem):
    from mygrad_amd import _hip

    x_shape, w_shape, s, p, d, _ = FEW_TERMS[problem]
    rng = np.random.default_rng(3800 + problem)

    def gradient(g, x, few=True):
        with monkeypatch.context() as m:
            m.setenv("MYGRAD_HIP_FEW", "1" if few else "0")
            m.setenv("MYGRAD_HIP_SPLIT", "1" if few else "0")
            dw = abi.conv_wgrad(g, x, w_shape, s, p, d)
            assert ("few terms" in _hip.last_plan()) == few
        return dw

    xi = rng.integers(-3, 4, x_shape).astype(np.float32)
    grid = direct.conv_forward(xi, np.zeros(w_shape, np.float32), s, p, d).shape
    gi = rng.integers(-2, 3, grid).astype(np.float32)
    # small integers: every sum is exact
    whole = gradient(gi, xi)
    assert np.array_equal(whole, direct.conv_backward_w(gi, xi, w_shape, s, p, d))
    # against 64 bits: two roundings for every 32 terms, as in test_filter_gradients_on_three_bf16_parts
    x, g = rng.standard_normal(x_shape).astype(np.float32), rng.standard_normal(grid).astype(np.float32)
    exact = direct.conv_backward_w(g.astype(np.float64), x.astype(np.float64), w_shape, s, p, d)
    got, single = gradient(g, x), gradient(g, x, few=False)
    off, terms = np.linalg.norm(got - exact), grid[0] * np.prod(grid[2:])
    assert off <= (1.25 * 5.06e-8 * np.sqrt(2 * 2 * terms / 64) + 3.5e-8) * np.linalg.norm(exact)
    assert terms < 30 or off <= np.linalg.norm(single - exact)
    # what the parts cannot hold: the single-precision kernel's gradient, bit for bit, and the one after it on the parts again
    for value in (np.inf, np.nan):
        for odd in range(2):
            operands = [g.copy(), x.copy()]
            operands[odd][tuple(n // 2 for n in operands[odd].shape)] = value
            assert np.array_equal(bits(gradient(*operands)), bits(gradient(*operands, few=False)))
    lost_bits_of_operands(gradient, g, x, terms >= 30)
    assert np.array_equal(bits(gradient(gi, xi)), bits(whole))


@pytest.mark.parametrize("x_shape, w_shape, s, p, few", [((64, 3, 225, 225), (64, 3, 7, 7), 2, 3, True), ((91, 8, 14715), (26, 8, 15), 1, 7, False),
                                                         ((32, 3, 224, 224), (64, 3, 3, 3), 1, 1, False), ((128, 64, 56, 56), (64, 64, 3, 3), 1, 1, False)])
def test_which_filter_gradients_run_as_few_terms(abi, x_shape, w_shape, s, p, few):
    from mygrad_amd import _hip

    x = np.ones(x_shape, np.float32)
    grid = tuple((n + 2 * p - t) // s + 1 for n, t in zip(x_shape[2:], w_shape[2:]))
    dw = abi.conv_wgrad(np.ones((x_shape[0], w_shape[0], *grid), np.float32), x, w_shape, s, p)
    assert ("few terms" in _hip.last_plan()) == few
    assert np.all(dw[(slice(None), slice(None), *(t // 2 for t in w_shape[2:]))] == x_shape[0] * np.prod(grid))
