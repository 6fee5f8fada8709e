"""The FP32 GEMM on the bf16 matrix cores (three exact bf16 terms per value):
every tile shape and operand form at ragged sizes, exact products where the
three terms must hold them, and the values the terms do not hold (infinities,
NaN, tiny and largest values), which the kernel recomputes on the FP32
instruction.
"""

from __future__ import annotations

import ctypes
import threading

import numpy as np
import pytest

import helpers

pytestmark = pytest.mark.gpu
U = helpers.U32


@pytest.fixture(scope="module")
def gpu():
    helpers.ensure_built()
    return helpers.load_package().Engine()


def gemm(gpu, A, B):
    dA, dB = gpu.upload(A), gpu.upload(B)
    dC = gpu.empty((A.shape[0], B.shape[1]), np.float32)
    dC.fill_bytes(0xFF)
    gpu.call("eng_matmul_f32", dA.ptr, dB.ptr, dC.ptr, A.shape[0], B.shape[1], A.shape[1], None)
    gpu.sync()
    return dC.download()


# (M, N, K): the tile, operand form and split that a card of 256 CUs gives eng_matmul_f32
# there (test_gemm_choice.py holds them to the launcher's rules)
FLOAT64 = {
    (1536, 4096, 512): "256x128 ALIGNED",
    (1531, 4093, 515): "256x128 SHIFT",       # every edge ragged, a partial K tile
    (2041, 2056, 530): "256x128 ANY",
    (500, 4096, 4096): "256x128 ALIGNED split",  # (records and the fix-up pass)
    (509, 4090, 4090): "256x128 SHIFT split",
    (2048, 2048, 512): "128x128 ALIGNED",
    (2030, 2040, 300): "128x128 ANY",
    (1000, 4090, 1030): "128x128 SHIFT",
    (640, 1024, 4096): "128x128 ALIGNED split",
    (640, 2000, 2050): "128x128 ANY split",
    (1000, 2050, 1030): "128x128 SHIFT split",
    (1531, 1024, 1024): "128x64 ALIGNED",     # (two K groups, as in all smaller tiles)
    (512, 4096, 1000): "128x64 ANY",
    (509, 2051, 1023): "128x64 SHIFT",
    (128, 768, 4096): "128x64 ALIGNED split",
    (128, 1024, 4096): "64x64 ALIGNED split",
    (65, 8, 1001): "64x64 ANY split",
    (130, 250, 1000): "64x64 SHIFT split",
    (129, 257, 993): "64x64 SHIFT split",     # one column past a tile, 31 whole K tiles and one value
    (300, 999, 4000): "64x64 SHIFT split",
    (70, 56, 8190): "64x64 ANY split",        # 32 records to a tile
    (70, 57, 4100): "64x64 SHIFT split",      # 16
    (4096, 5, 300): "64x64 SHIFT",            # N below one column chunk
    (100, 3, 700): "64x64 SHIFT",
    (1000, 3000, 200): "fp32 staged",         # 16-byte loads of both operands,
    (438, 521, 132): "fp32 staged",           # of A,
    (300, 336, 85): "fp32 staged",            # of B,
    (200, 3001, 63): "fp32 staged",           # of neither
}
SPECIAL = {
    (300, 1024, 704): "fp32 direct",
    (300, 999, 701): "64x64 SHIFT",
    (300, 512, 4096): "64x64 ALIGNED split",
    (1531, 1024, 1024): "128x64 ALIGNED",
    (640, 2000, 2050): "128x128 ANY split",
    (1536, 4096, 512): "256x128 ALIGNED",
}
# M, N, K, weight type, layout of eng_rmsnorm_linear_*
FORMS = {
    (1531, 4093, 515, "f32", "nk"): "256x128 ANY",
    (1531, 4093, 515, "f16", "nk"): "256x128 ANY",
    (1531, 4093, 515, "f16", "kn"): "256x128 SHIFT",
    (2030, 2040, 300, "f16", "kn"): "128x128 ANY",
    (2030, 2041, 300, "f16", "kn"): "128x128 SHIFT",
    (640, 2000, 2050, "f32", "nk"): "128x128 ANY split",
    (640, 2000, 2050, "f16", "nk"): "128x128 ANY split",
    (640, 2000, 2050, "f16", "kn"): "128x128 ANY split",
    (509, 2051, 1023, "f32", "nk"): "128x64 ANY",
    (509, 2051, 1023, "f16", "nk"): "128x64 ANY",
    (509, 2051, 1023, "f16", "kn"): "128x64 SHIFT",
    (129, 257, 993, "f32", "nk"): "64x64 ANY split",
    (129, 257, 993, "f16", "nk"): "64x64 ANY split",
    (129, 257, 993, "f16", "kn"): "64x64 SHIFT split",
}


@pytest.mark.parametrize("M,N,K", FLOAT64)
def test_split_gemm_against_float64(gpu, M, N, K):
    rng = np.random.default_rng(M + 3 * N + 7 * K)
    A = rng.uniform(-1, 1, (M, K)).astype(np.float32)
    B = rng.uniform(-1, 1, (K, N)).astype(np.float32)
    got = gemm(gpu, A, B)
    y64 = helpers.as_f64(A) @ helpers.as_f64(B)
    derived, stat = helpers.dot_bounds(helpers.absdot(A, B), y64, K)
    helpers.assert_within(got, y64, np.minimum(derived, stat), f"{M}x{N}x{K}")


@pytest.mark.parametrize("M,N,K", [
    (1536, 4096, 1024),   # 256 x 128 tiles
    (2048, 2048, 512),    # 128 x 128
    (509, 2051, 1023),    # 128 x 64 in two K groups
    (130, 250, 1000),     # 64 x 64 in two K groups
])
@pytest.mark.parametrize("kind", ["mixed", "same sign", "half zero", "one product"])
def test_split_gemm_error_is_that_of_one_rounding_per_slice(gpu, M, N, K, kind):
    """The leading products' sum is rounded once per 16 k. Independent roundings of
    a sum that grows to y (in the mean half its square) to 2^-24 of it at most add
    up to 2^-24 sqrt(K / 32) |y|; all six products on one sum exceed this, as does
    the FP32 instruction with its eight roundings. A sum of one product is rounded
    once, 0.42 x 2^-24 in the root mean square, without a bias; the products left
    out add at most 2 x 2^-24."""
    rng = np.random.default_rng(M + N + K)
    A = rng.uniform(-1, 1, (M, K)).astype(np.float32)
    B = rng.uniform(-1, 1, (K, N)).astype(np.float32)
    if kind == "same sign":
        A, B = np.abs(A), np.abs(B)
    elif kind == "half zero":
        A = np.maximum(A, 0)
    elif kind == "one product":
        n = min(K, N)
        B = np.zeros((K, N), np.float32)
        B[np.arange(n), np.arange(n)] = rng.uniform(1, 2, n).astype(np.float32)
    y64 = helpers.as_f64(A) @ helpers.as_f64(B)
    err = gemm(gpu, A, B) - y64
    if kind == "one product":
        rel = err[:, :n] / np.abs(y64[:, :n]) / U
        assert np.abs(rel).max() <= 3.1
        assert np.sqrt((rel * rel).mean()) <= 0.5
        assert abs(rel.mean()) <= 0.05
    else:
        assert np.linalg.norm(err) / np.linalg.norm(y64) <= U * np.sqrt(K / 32)


@pytest.mark.parametrize("M,N,K", [(1531, 1024, 1024), (300, 999, 999)])
def test_split_gemm_times_identity_is_exact(gpu, M, N, K):
    """A . I = A bit for bit: the three terms of a value add up to it, over 200
    binary orders of magnitude."""
    rng = np.random.default_rng(3)
    A = (rng.uniform(1, 2, (M, K)) * 2.0 ** rng.integers(-100, 100, (M, K))).astype(np.float32)
    A *= rng.choice(np.float32([-1, 1]), A.shape)
    B = np.zeros((K, N), np.float32)
    B[np.arange(min(K, N)), np.arange(min(K, N))] = 1.0
    got = gemm(gpu, A, B)
    assert np.array_equal(got[:, :min(K, N)], A[:, :min(K, N)])


@pytest.mark.parametrize("M,N,K", [(1531, 1024, 1024), (300, 999, 999)])
def test_split_gemm_subnormal_third_terms_are_exact(gpu, M, N, K):
    """The smallest values that three terms hold, with third terms (and for the
    smallest first ones) below bf16's and fp32's normal range: A . I = A bit for bit
    without a recompute, which the matrix instruction has to keep subnormals for."""
    rng = np.random.default_rng(7)
    A = (rng.uniform(1, 2, (M, K)) * 2.0 ** rng.integers(-110, -101, (M, K))).astype(np.float32)
    A[::2] = (rng.integers(1, 2**16, A[::2].shape) * 2.0**-133).astype(np.float32)
    A *= rng.choice(np.float32([-1, 1]), A.shape)
    n = min(K, N)
    B = np.zeros((K, N), np.float32)
    B[np.arange(n), np.arange(n)] = 1.0
    assert np.array_equal(gemm(gpu, A, B)[:, :n], A[:, :n])


@pytest.mark.parametrize("M,N,K,w,layout", FORMS)
def test_split_gemm_weight_types_and_layouts(gpu, M, N, K, w, layout):
    """fp16 and output-major B at every tile (the normalised rows are the A operand)."""
    rng = np.random.default_rng(M + N + K)
    x = rng.standard_normal((M, K), dtype=np.float32)
    W = (0.02 * rng.standard_normal((K, N))).astype(np.float32)
    if w == "f16":
        W = W.astype(np.float16).view(np.uint16)
    dx, dW = gpu.upload(x), gpu.upload(np.ascontiguousarray(W.T) if layout == "nk" else W)
    dy = gpu.empty((M, N), np.float32)
    dy.fill_bytes(0xFF)
    gpu.call(f"eng_rmsnorm_linear_{w}{'w' if w == 'f16' else ''}{'_nk' if layout == 'nk' else ''}",
             dx.ptr, None, dW.ptr, dy.ptr, M, N, K, 1e-5, None)
    gpu.sync()
    x64 = helpers.as_f64(x)
    y64 = x64 / np.sqrt((x64 * x64).mean(1, keepdims=True) + 1e-5) @ helpers.as_f64(W)
    got = dy.download()
    derived, stat = helpers.rmsnorm_linear_bounds(x, None, W, y64, K)
    helpers.assert_within(got, y64, np.minimum(derived, stat), f"{w} {layout} {M}x{N}x{K}")
    # one rounding per 16 k, and a few of the row scale
    assert np.linalg.norm(got - y64) / np.linalg.norm(y64) <= U * (np.sqrt(K / 32) + 8)


@pytest.mark.parametrize("M,N,K", SPECIAL)
def test_split_gemm_infinities_nan_and_extreme_values(gpu, M, N, K):
    rng = np.random.default_rng(11)
    A = rng.uniform(-1, 1, (M, K)).astype(np.float32)
    B = rng.uniform(-1, 1, (K, N)).astype(np.float32)
    A[3, 5] = np.inf
    A[7, 6] = -np.inf
    A[7, 9] = np.inf        # meets both signs: NaN where the products disagree
    A[11, K - 1] = np.nan
    A[130] *= np.float32(1e-37)             # down to fp32 subnormals
    A[131, ::2] *= np.float32(1e-42)
    A[140] *= np.float32(1e36)
    A[141, 17] = np.finfo(np.float32).max   # rounds past bf16's range
    B[17] *= np.float32(1e-30)
    B[20, 200] = np.inf
    B[21, 201] = np.nan
    B[:, 202] = 0.0
    got = gemm(gpu, A, B)
    with np.errstate(invalid="ignore"):
        y64 = helpers.as_f64(A) @ helpers.as_f64(B)
    fin = np.isfinite(y64)
    assert np.array_equal(np.isnan(got), np.isnan(y64))
    assert np.array_equal(got[~fin & ~np.isnan(y64)], y64[~fin & ~np.isnan(y64)].astype(np.float32))
    with np.errstate(invalid="ignore"):
        a = helpers.absdot(A, B)
    # each of the K products and sums also rounds to at most half of the
    # smallest subnormal, 2^-150
    bound = K * U * np.where(fin, a, 0) + U * np.abs(np.where(fin, y64, 0)) + 2 * K * 2.0**-150
    err = np.abs(np.where(fin, got, 0).astype(np.float64) - np.where(fin, y64, 0))
    assert (err <= bound).all(), float((err / bound).max())


@pytest.mark.parametrize("M,N,K", SPECIAL)
def test_split_gemm_tiny_values_beside_ordinary_ones(gpu, M, N, K):
    """Probabilities down to e^-87 (values the three terms do not hold, in every
    tile) times ordinary values, and rows of nothing but tiny ones."""
    rng = np.random.default_rng(5)
    A = np.exp(-rng.uniform(0, 87, (M, K))).astype(np.float32)
    A[256:290] = A[256:290] * np.float32(1e-36)
    B = rng.uniform(-1, 1, (K, N)).astype(np.float32)
    got = gemm(gpu, A, B)
    y64 = helpers.as_f64(A) @ helpers.as_f64(B)
    bound = K * U * helpers.absdot(A, B) + U * np.abs(y64) + 2 * K * 2.0**-150
    err = np.abs(got - y64)
    assert (err <= bound).all(), float((err / bound).max())


@pytest.mark.parametrize("M,N,K", [(1536, 4096, 512), (509, 2051, 1023), (300, 999, 4000)])
def test_split_gemm_recomputes_no_more_than_it_must(gpu, M, N, K):
    """Infinities and NaN change the elements they reach and no others, bit for bit;
    neither do exact zeros beside values the three terms do not hold."""
    rng = np.random.default_rng(23)
    A = np.exp(-rng.uniform(0, 87, (M, K))).astype(np.float32)
    A[:, : K // 2] = rng.uniform(-1, 1, (M, K // 2)).astype(np.float32)
    B = rng.uniform(-1, 1, (K, N)).astype(np.float32)
    want = gemm(gpu, A, B)
    A2, B2 = A.copy(), B.copy()
    rows, cols = [5, 131, M - 1], [7, 130, N - 1]
    A2[rows[0], 3], A2[rows[1], K - 1], A2[rows[2], 9] = np.nan, np.inf, -np.inf
    B2[:, cols] = 0.0
    zero_rows = [6, 200]
    A2[zero_rows] = 0.0
    got = gemm(gpu, A2, B2)
    keep = np.ones((M, N), bool)
    keep[rows + zero_rows] = False
    keep[:, cols] = False
    assert np.array_equal(got[keep], want[keep])
    assert (got[zero_rows] == 0).all()
    ordinary = np.setdiff1d(np.arange(M), rows)
    assert (got[np.ix_(ordinary, cols)] == 0).all()
    other = np.setdiff1d(np.arange(N), cols)
    assert np.isnan(got[rows[0]]).all() and np.isnan(got[np.ix_(rows, cols)]).all()
    assert np.array_equal(got[rows[1], other], np.sign(B2[K - 1, other]) * np.inf)
    assert np.array_equal(got[rows[2], other], -np.sign(B2[9, other]) * np.inf)


@pytest.mark.parametrize("M,N,K", [(640, 1024, 4096), (1280, 4096, 2048)])
def test_split_gemm_captured_with_no_eager_call_before(gpu, M, N, K):
    """Sizes whose K is split over workgroups, captured on a stream with no
    scratch yet: the call runs on a cut that needs none, as it does for another
    stream's eager call that cannot disturb the capture."""
    rng = np.random.default_rng(M + N + K)
    A = rng.uniform(-1, 1, (M, K)).astype(np.float32)
    B = rng.uniform(-1, 1, (K, N)).astype(np.float32)
    y64 = helpers.as_f64(A) @ helpers.as_f64(B)
    derived, stat = helpers.dot_bounds(helpers.absdot(A, B), y64, K)
    bound = np.minimum(derived, stat)
    dA, dB, dC, dE = gpu.upload(A), gpu.upload(B), gpu.empty((M, N), np.float32), gpu.empty((M, N), np.float32)
    s, other, graph = gpu.stream(), gpu.stream(), None
    try:
        graph = gpu.graph(s)
        with graph:
            gpu.call("eng_matmul_f32", dA.ptr, dB.ptr, dC.ptr, M, N, K, s.handle)
            gpu.call("eng_matmul_f32", dA.ptr, dB.ptr, dE.ptr, M, N, K, other.handle)
        other.sync()
        eager = dE.download().copy()
        helpers.assert_within(eager, y64, bound, f"eager {M}x{N}x{K}")
        for _ in range(3):
            dC.fill_bytes(0xFF)
            gpu.sync()
            graph.launch()
            s.sync()
            helpers.assert_within(dC.download(), y64, bound, f"captured {M}x{N}x{K}")
    finally:
        if graph is not None:
            graph.destroy()
        s.destroy()
        other.destroy()


class NativeGraph:
    """A capture of `stream` begun and ended with HIP's own calls."""

    def __init__(self, stream):
        self.hip = ctypes.CDLL("libamdhip64.so")
        self.stream = ctypes.c_void_p(stream)
        self.graph, self.exec = ctypes.c_void_p(0), ctypes.c_void_p(0)

    def ok(self, status):
        assert status == 0, f"HIP status {status}"

    def __enter__(self):
        self.ok(self.hip.hipStreamBeginCapture(self.stream, 1))  # thread-local mode
        return self

    def __exit__(self, *exc):
        self.ok(self.hip.hipStreamEndCapture(self.stream, ctypes.byref(self.graph)))
        self.ok(self.hip.hipGraphInstantiate(ctypes.byref(self.exec), self.graph, None, None,
                                             ctypes.c_size_t(0)))

    def nodes(self):
        n = ctypes.c_size_t(0)
        self.ok(self.hip.hipGraphGetNodes(self.graph, None, ctypes.byref(n)))
        return n.value

    def launch(self, stream):
        self.ok(self.hip.hipGraphLaunch(self.exec, ctypes.c_void_p(stream)))

    def destroy(self):
        self.ok(self.hip.hipGraphExecDestroy(self.exec))
        self.ok(self.hip.hipGraphDestroy(self.graph))


def test_split_gemm_in_a_capture_of_the_program_and_on_the_per_thread_stream(gpu):
    """Sizes whose K is split over workgroups, where no records of their own can be
    had: in a capture begun with HIP itself, on a stream that has an arena, and on
    hipStreamPerThread, one handle for every thread's stream. Both run as one
    launch without records; a capture begun here still has them."""
    M, N, K = 512, 4096, 4096
    per_thread = 2  # hipStreamPerThread
    rng = np.random.default_rng(17)
    A = [rng.uniform(-1, 1, (M, K)).astype(np.float32) for _ in range(2)]
    B = rng.uniform(-1, 1, (K, N)).astype(np.float32)
    dA, dB = [gpu.upload(a) for a in A], gpu.upload(B)
    dC = [gpu.empty((M, N), np.float32) for _ in range(2)]

    def call(i, stream):
        gpu.call("eng_matmul_f32", dA[i].ptr, dB.ptr, dC[i].ptr, M, N, K, stream)

    s, other = gpu.stream(), gpu.stream()
    native, own = NativeGraph(s.handle), gpu.graph(s)
    try:
        call(0, s.handle)
        s.sync()
        eager = dC[0].download().copy()
        y64 = helpers.as_f64(A[0]) @ helpers.as_f64(B)
        derived, stat = helpers.dot_bounds(helpers.absdot(A[0], B), y64, K)
        with own:
            call(0, s.handle)
        with native:
            call(0, s.handle)
        assert native.nodes() == 1
        for _ in range(3):
            dC[0].fill_bytes(0xFF)
            gpu.sync()
            native.launch(other.handle)
            call(1, s.handle)  # the stream's eager calls go on meanwhile
            gpu.sync()
            one = dC[0].download().copy()
            helpers.assert_within(one, y64, np.minimum(derived, stat), "replay")
        own.launch(s)
        s.sync()
        assert np.array_equal(dC[0].download(), eager)
        assert not np.array_equal(eager, one)  # (the split's sums are in another order)

        want = []
        for i in range(2):
            with NativeGraph(s.handle) as g:
                call(i, s.handle)
            g.launch(s.handle)
            s.sync()
            g.destroy()
            want.append(dC[i].download().copy())
            dC[i].fill_bytes(0xFF)
        gpu.sync()
        done = []

        def work(i):
            for _ in range(20):
                call(i, per_thread)
            gpu.call("eng_stream_sync", per_thread)
            done.append(i)

        threads = [threading.Thread(target=work, args=(i,)) for i in range(2)]
        for t in threads:
            t.start()
        for t in threads:
            t.join()
        assert sorted(done) == [0, 1]
        for i in range(2):
            assert np.array_equal(dC[i].download(), want[i])
    finally:
        native.destroy()
        own.destroy()
        s.destroy()
        other.destroy()
