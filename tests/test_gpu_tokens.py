"""GPU parity of the matmuls that the reference runs token by token (matmul, fastgguf.c:3004-3017):
every type below 8 tokens, and the types without a prompt GEMM at every batch. Each token's
outputs equal the reference's row kernel bit for bit (the oracle's matvec of that token)."""
import numpy as np
import pytest
from conftest import bits_equal

from fastgguf_amd import synth as S
from fastgguf_amd.backend import ORDER_AUTO, ORDER_ROW

pytestmark = pytest.mark.gpu


def check(backend, oracle, type_, rows, cols, T, order=ORDER_AUTO, n_mats=1, w=None, X=None, seed=0):
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


@pytest.mark.parametrize("rows,cols,order,n_mats,T", [(72, 1792, ORDER_AUTO, 1, 7), (14344, 1024, ORDER_AUTO, 1, 7), (16390, 2048, ORDER_AUTO, 1, 5),
                                                      (10256, 1792, ORDER_ROW, 1, 7), (5400, 1280, ORDER_AUTO, 3, 6), (8208, 3328, ORDER_AUTO, 1, 7)])
def test_q4_k_few_tokens(backend, oracle, rows, cols, order, n_mats, T):
    """Both fp32 orders (16390 rows and 3 matrices: the row order) on either side of the rule that
    picks the kernel, block counts that end inside a ring round, a last tile and a last workgroup
    that are not full."""
    check(backend, oracle, S.T_Q4_K, rows, cols, T, order, n_mats, seed=cols)


@pytest.mark.parametrize("rows,cols,n_mats,T", [(50, 256, 1, 17), (14330, 768, 1, 7), (4090, 2048, 1, 16), (6160, 768, 1, 50), (1020, 4096, 1, 64),
                                                (700, 1280, 3, 33), (2050, 2304, 1, 17)])
def test_q5_k_tokens(backend, oracle, rows, cols, n_mats, T):
    """One group of 16 tokens, several apart, and two per wavefront (6160 rows; the last group not full)."""
    check(backend, oracle, S.T_Q5_K, rows, cols, T, n_mats=n_mats, seed=cols + T)


@pytest.mark.parametrize("type_", [S.T_Q4_K, S.T_Q5_K], ids=["Q4_K", "Q5_K"])
def test_extreme_blocks(backend, oracle, type_):
    """Every quant, scale and min at its largest against activations at +-127: the largest integers the
    f16 products and sums meet (row order: 8 * 4 * 31 * 63 * 127), and a token of zeros."""
    rows, cols, T = 16400, 1024, 7
    w = S.weights(type_, rows, cols, 3)
    blk = w.reshape(-1, S.BLOCK[type_][1])
    blk[:, 4:] = 0xFF
    X = np.ones((T, cols), np.float32)
    X[1] = -1.0
    X[2, ::2] = -1.0
    X[3] = 0.0
    X[4:] *= np.repeat(np.float32(2.0) ** np.arange(cols // 256), 256)
    for order in (ORDER_AUTO, ORDER_ROW):
        check(backend, oracle, type_, rows, cols, T, order, w=w, X=X)


@pytest.mark.parametrize("type_,rows,cols,n_mats,T", [
    (S.T_F32, 6200, 520, 1, 5), (S.T_F32, 3001, 1003, 1, 17), (S.T_F32, 1500, 77, 2, 64), (S.T_F32, 6200, 136, 1, 61),
    (S.T_F16, 2000, 1003, 1, 64), (S.T_F16, 12400, 136, 1, 61), (S.T_F16, 6200, 520, 2, 17), (S.T_F16, 6600, 776, 1, 29),
    (S.T_BF16, 8000, 325, 1, 64), (S.T_BF16, 5000, 1003, 2, 17), (S.T_BF16, 9001, 256, 1, 33), (S.T_BF16, 40, 77, 1, 9)])
def test_float_tokens(backend, oracle, type_, rows, cols, n_mats, T):
    """Whole and partial steps and stages, the scalar tail (cols % 8), row tiles and matrices that are not
    full, 1, 2 and 4 groups of 16 tokens per wavefront (F16 6600, 12400 rows)."""
    check(backend, oracle, type_, rows, cols, T, n_mats=n_mats, seed=cols + T)


@pytest.mark.parametrize("type_", [S.T_F32, S.T_F16, S.T_BF16], ids=["F32", "F16", "BF16"])
def test_float_bit_patterns(backend, oracle, type_):
    """Random finite bit patterns, subnormals and zeros among them, at every token kernel."""
    for rows, T in ((66, 3), (8000, 20), (8000, 64)):
        w = S.random_float_bits(type_, rows, 325, 40 + T)
        check(backend, oracle, type_, rows, 325, T, w=w, seed=T)
