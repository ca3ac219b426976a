"""GPU parity of the matmuls that the reference runs token by token (matmul, fastgguf.c:3004-3017):
every type below 8 tokens, and the types without a prompt GEMM at every batch. Each token's
outputs equal the reference's row kernel bit for bit (the oracle's matvec of that token)."""
import numpy as np
import pytest
from conftest import bits_equal, bits_equal_or_nan

from fastgguf_amd import synth as S
from fastgguf_amd.backend import MATMUL_DECODE, MATMUL_TOKENS, ORDER_AUTO, ORDER_ROW, Backend, matmul_path

pytestmark = pytest.mark.gpu


def check(backend, oracle, type_, rows, cols, T, order=ORDER_AUTO, n_mats=1, w=None, X=None, seed=0, path=MATMUL_TOKENS):
    assert matmul_path(type_, oracle_order(type_, rows, n_mats, order), cols, rows, T, n_mats) == path
    if w is None:
        w = S.weights(type_, rows * n_mats, cols, 900 + seed)
    if X is None:
        X = S.activations(cols, 910 + seed, rows=T)
    t = backend.upload(type_, cols, w, rows=rows, n_mats=n_mats, order=order)
    got = backend.matmul(t, X)
    t.free()
    for k in range(T):
        want = oracle.matvec(type_, w, cols, X[k], oracle_order(type_, rows, n_mats, order))
        assert bits_equal(got[k], want), f"{S.TYPE_NAME[type_]} {rows}x{cols} x{n_mats}, token {k} of {T}"


def oracle_order(type_, rows, n_mats, order):
    from oracle import ORDER_REPACKED, ORDER_ROW as ROW
    if order == ORDER_AUTO and n_mats == 1 and rows % 8 == 0 and type_ in (S.T_Q4_K, S.T_Q4_0):
        return ORDER_REPACKED
    return ROW


@pytest.mark.parametrize("rows,cols,order,n_mats,T,path", [
    (72, 1792, ORDER_AUTO, 1, 7, MATMUL_DECODE), (16390, 2048, ORDER_AUTO, 1, 5, MATMUL_DECODE),
    (14344, 1024, ORDER_AUTO, 1, 7, MATMUL_TOKENS), (8208, 3328, ORDER_AUTO, 1, 7, MATMUL_TOKENS),
    (16360, 1792, ORDER_AUTO, 1, 7, MATMUL_TOKENS), (16376, 2048, ORDER_AUTO, 1, 6, MATMUL_TOKENS),
    (16376, 2816, ORDER_AUTO, 1, 6, MATMUL_TOKENS), (17608, 1536, ORDER_AUTO, 1, 7, MATMUL_TOKENS),
    (10256, 1792, ORDER_ROW, 1, 7, MATMUL_TOKENS), (16380, 2048, ORDER_AUTO, 1, 7, MATMUL_TOKENS),
    (32776, 768, ORDER_ROW, 1, 7, MATMUL_TOKENS), (15990, 2304, ORDER_AUTO, 1, 7, MATMUL_TOKENS),
    (5400, 1280, ORDER_AUTO, 3, 6, MATMUL_TOKENS), (5456, 1536, ORDER_AUTO, 3, 7, MATMUL_TOKENS)])
def test_q4_k_few_tokens(backend, oracle, rows, cols, order, n_mats, T, path):
    """Both fp32 orders (rows that are no multiple of 8 and 3 matrices: the row order) on either side of
    the rule that picks the kernel: block counts that end anywhere in a ring round (rings of 6 and 4),
    below and above one wavefront per SIMD, a last tile and a last workgroup that are not full."""
    check(backend, oracle, S.T_Q4_K, rows, cols, T, order, n_mats, seed=cols, path=path)


@pytest.mark.parametrize("rows,cols,n_mats,T,path", [
    (50, 256, 1, 17, MATMUL_DECODE), (1020, 4096, 1, 64, MATMUL_DECODE), (4090, 2048, 1, 16, MATMUL_DECODE),
    (700, 1280, 3, 33, MATMUL_DECODE), (2050, 2304, 1, 17, MATMUL_DECODE),
    (14330, 768, 1, 7, MATMUL_TOKENS), (16370, 768, 1, 16, MATMUL_TOKENS), (16380, 256, 1, 16, MATMUL_TOKENS),
    (16380, 512, 1, 13, MATMUL_TOKENS), (5400, 1280, 3, 9, MATMUL_TOKENS),
    (4090, 2048, 1, 24, MATMUL_TOKENS), (1340, 1280, 3, 33, MATMUL_TOKENS), (700, 1280, 3, 64, MATMUL_TOKENS),
    (4090, 1792, 1, 48, MATMUL_TOKENS),
    (6160, 768, 1, 50, MATMUL_TOKENS), (14330, 768, 1, 17, MATMUL_TOKENS), (13000, 1536, 1, 33, MATMUL_TOKENS)])
def test_q5_k_tokens(backend, oracle, rows, cols, n_mats, T, path):
    """One group of 16 tokens, several apart, and two per wavefront (the last three; the last group not
    full), block counts below and beyond a ring round."""
    check(backend, oracle, S.T_Q5_K, rows, cols, T, n_mats=n_mats, seed=cols + T, path=path)


@pytest.mark.parametrize("type_", [S.T_Q4_K, S.T_Q5_K], ids=["Q4_K", "Q5_K"])
def test_extreme_blocks(backend, oracle, type_):
    """Every quant, scale and min at its largest against activations at +-127: the largest integers the
    f16 products and sums meet (row order: 8 * 4 * 31 * 63 * 127), and a token of zeros, through the
    shared kernels of both orders."""
    cols, T = 1024, 7
    w = S.weights(type_, 16400, cols, 3)
    blk = w.reshape(-1, S.BLOCK[type_][1])
    blk[:, 4:] = 0xFF
    X = np.ones((T, cols), np.float32)
    X[1] = -1.0
    X[2, ::2] = -1.0
    X[3] = 0.0
    X[4:] *= np.repeat(np.float32(2.0) ** np.arange(cols // 256), 256)
    for rows in (16376, 16400):
        for order in (ORDER_AUTO, ORDER_ROW):
            check(backend, oracle, type_, rows, cols, T, order, w=w[:rows], X=X)


@pytest.mark.parametrize("type_,rows,cols,n_mats,T", [
    (S.T_F32, 6200, 520, 1, 5), (S.T_F32, 3001, 1003, 1, 17), (S.T_F32, 1500, 77, 2, 64), (S.T_F32, 6200, 136, 1, 61),
    (S.T_F16, 2000, 1003, 1, 64), (S.T_F16, 12400, 136, 1, 61), (S.T_F16, 6200, 520, 2, 17), (S.T_F16, 6600, 776, 1, 29),
    (S.T_BF16, 8000, 325, 1, 64), (S.T_BF16, 5000, 1003, 2, 17), (S.T_BF16, 9001, 256, 1, 33), (S.T_BF16, 40, 77, 1, 9)])
def test_float_tokens(backend, oracle, type_, rows, cols, n_mats, T):
    """Whole and partial steps and stages, the scalar tail (cols % 8), row tiles and matrices that are not
    full, 1, 2 and 4 groups of 16 tokens per wavefront (F16 6600, 12400 rows)."""
    check(backend, oracle, type_, rows, cols, T, n_mats=n_mats, seed=cols + T, path=MATMUL_DECODE if rows == 40 else MATMUL_TOKENS)


@pytest.mark.parametrize("type_", [S.T_F32, S.T_F16, S.T_BF16], ids=["F32", "F16", "BF16"])
def test_float_bit_patterns(backend, oracle, type_):
    """Random finite bit patterns, subnormals and zeros among them, at every token kernel."""
    for rows, T in ((66, 3), (8000, 20), (14000, 20), (8000, 64)):
        w = S.random_float_bits(type_, rows, 325, 40 + T)
        decode = rows == 66 or (type_ == S.T_BF16 and (rows, T) == (8000, 20))
        check(backend, oracle, type_, rows, 325, T, w=w, seed=T, path=MATMUL_DECODE if decode else MATMUL_TOKENS)


def float_specials(type_, rows, cols, seed):
    """Weights of every kind: infinities and NaN (a few rows), subnormals, zeros of both signs, normals."""
    rng = np.random.default_rng(seed)
    w = rng.standard_normal((rows, cols)).astype(np.float32)
    sub = np.float32({S.T_F32: 1e-41, S.T_F16: 3e-7, S.T_BF16: 1e-39}[type_])
    w[rng.random((rows, cols)) < 0.1] = sub
    w[rng.random((rows, cols)) < 0.1] = -0.0
    for r, v in ((1, np.inf), (2, -np.inf), (5, np.nan), (rows - 1, np.inf)):
        w[r, rng.integers(0, cols)] = v
    w[7, :2] = np.inf, -np.inf
    if type_ == S.T_F16:
        return w.astype(np.float16).view(np.uint8).reshape(rows, -1)
    if type_ == S.T_BF16:
        return (w.view(np.uint32) >> 16).astype(np.uint16).view(np.uint8).reshape(rows, -1)
    return w.view(np.uint8).reshape(rows, -1)


@pytest.mark.parametrize("type_,rows,T", [(S.T_F32, 8000, 20), (S.T_F16, 8000, 20), (S.T_F16, 8000, 64), (S.T_BF16, 14000, 20)],
                         ids=["F32", "F16", "F16_64", "BF16"])
def test_float_specials(backend, oracle, type_, rows, T):
    """The fp32 MFMAs add each product as one fmaf also for infinities, NaN, subnormals and signed zeros,
    in weights and in activations: outputs equal bit for bit, any NaN as any NaN."""
    cols = 325
    w = float_specials(type_, rows, cols, 3)
    X = S.activations(cols, 4, rows=T)
    X[1] *= np.float32(1e-38)  # subnormal products and sums
    X[2, ::3] = 0.0
    X[2, 1::3] = -0.0
    X[3, 17] = np.inf
    X[4, 18] = np.nan
    X[5] = np.float32(1e-42)
    assert matmul_path(type_, 0, cols, rows, T) == MATMUL_TOKENS
    t = backend.upload(type_, cols, w, rows=rows)
    got = backend.matmul(t, X)
    t.free()
    for k in range(T):
        want = oracle.matvec(type_, w, cols, X[k], oracle_order(type_, rows, 1, ORDER_AUTO))
        assert bits_equal_or_nan(got[k], want), f"{S.TYPE_NAME[type_]}, token {k}"


@pytest.mark.parametrize("type_,rows,cols,T", [(S.T_Q4_K, 16376, 1024, 7), (S.T_Q5_K, 16376, 1024, 9), (S.T_F16, 8000, 325, 20)],
                         ids=["Q4_K", "Q5_K", "F16"])
def test_graph_replays(type_, rows, cols, T):
    """A matmul of several tokens captured on a fresh context, first without its scratch (Q4_K, Q5_K: the
    decode launches take the call; the float kernels need none), then after an eager call (the shared
    kernels): every replay, with new tokens and eager work in between, equals the eager result."""
    assert matmul_path(type_, oracle_order(type_, rows, 1, ORDER_AUTO), cols, rows, T) == MATMUL_TOKENS
    Xs = [S.activations(cols, 60 + i, rows=T) for i in range(3)]
    with Backend(0) as be:
        t = be.upload(type_, cols, S.weights(type_, rows, cols, 5))
        xd, yd, ye = be.dev_alloc(Xs[0].nbytes), be.dev_alloc(4 * T * rows), be.dev_alloc(4 * T * rows)
        graphs = []
        for _ in range(2):
            be.graph_begin()
            be.matmul_dev(t, xd, yd, T)
            graphs.append(be.graph_end())
            for X in Xs:
                be.h2d(xd, X)
                for g in graphs:
                    be.h2d(yd, np.full(T * rows, np.nan, np.float32))
                    be.graph_launch(g)
                    be.sync()
                    be.matmul_dev(t, xd, ye, T)  # eager: also grows the scratch
                    be.sync()
                    got, want = np.empty(T * rows, np.float32), np.empty(T * rows, np.float32)
                    be.d2h(got, yd)
                    be.d2h(want, ye)
                    assert not np.isnan(want).any() and bits_equal(got, want)
        for g in graphs:
            be.graph_destroy(g)
        for p in (xd, yd, ye):
            be.dev_free(p)
        t.free()
