"""Which kernels a matmul of several tokens runs (fgh_matmul_path; host code, no device): the kernels
that share a matrix's weights between tokens only where they were measured to be the faster side, and
never for types without them."""
import pytest

from fastgguf_amd import synth as S
from fastgguf_amd.backend import MATMUL_DECODE, MATMUL_GEMM, MATMUL_TOKENS, BackendError, matmul_path

ROW, REPACKED = 0, 1
# (type, order, rows, cols, tokens, us of the decode launches, us of the shared kernels), measured on MI355X
MEASURED = [
    (S.T_Q4_K, REPACKED, 14336, 4096, 2, 11.8, 16.6), (S.T_Q4_K, REPACKED, 14336, 4096, 5, 20.0, 16.4),
    (S.T_Q4_K, REPACKED, 14336, 4096, 7, 25.5, 16.2), (S.T_Q4_K, REPACKED, 8192, 8192, 6, 20.7, 24.1),
    (S.T_Q4_K, REPACKED, 4096, 14336, 7, 25.5, 36.9), (S.T_Q4_K, REPACKED, 32000, 4096, 5, 50.2, 23.8),
    (S.T_Q4_K, REPACKED, 512, 2048, 7, 4.4, 10.6), (S.T_Q4_K, REPACKED, 16376, 1024, 7, 10.4, 9.0),
    (S.T_Q4_K, ROW, 14336, 4096, 3, 15.2, 19.5), (S.T_Q4_K, ROW, 14336, 4096, 6, 24.2, 19.1),
    (S.T_Q4_K, ROW, 32000, 4096, 4, 42.6, 26.5), (S.T_Q4_K, ROW, 5120, 13824, 6, 31.7, 45.4),
    (S.T_Q5_K, ROW, 14336, 4096, 4, 20.8, 23.6), (S.T_Q5_K, ROW, 14336, 4096, 7, 31.4, 23.1),
    (S.T_Q5_K, ROW, 14336, 4096, 64, 263.2, 36.3), (S.T_Q5_K, ROW, 4096, 4096, 16, 20.1, 22.8),
    (S.T_Q5_K, ROW, 4096, 4096, 24, 26.9, 21.9), (S.T_Q5_K, ROW, 4096, 14336, 12, 46.9, 62.1),
    (S.T_Q5_K, ROW, 4096, 14336, 32, 118.4, 60.2), (S.T_Q5_K, ROW, 8192, 8192, 6, 29.2, 38.4),
    (S.T_Q5_K, ROW, 8192, 2048, 8, 11.6, 14.9), (S.T_Q5_K, ROW, 1024, 4096, 64, 18.9, 22.0),
    (S.T_Q5_K, ROW, 4096, 1536, 16, 10.2, 12.7), (S.T_Q5_K, ROW, 2048, 2048, 64, 19.4, 14.3),
    (S.T_Q5_K, ROW, 16376, 1024, 5, 9.4, 10.7), (S.T_Q5_K, ROW, 16376, 1024, 16, 22.2, 10.8),
    (S.T_Q5_K, ROW, 12464, 5888, 3, 28.1, 30.2), (S.T_Q5_K, ROW, 12464, 5888, 5, 41.2, 29.9),
    (S.T_F32, ROW, 640, 2048, 40, 15.6, 20.0), (S.T_F32, ROW, 512, 4096, 64, 29.7, 34.6),
    (S.T_F32, ROW, 896, 4864, 28, 35.0, 41.4), (S.T_F32, ROW, 1024, 1024, 20, 9.1, 12.4),
    (S.T_F32, ROW, 4096, 4096, 4, 33.0, 35.9), (S.T_F32, ROW, 4096, 4096, 8, 65.2, 36.0),
    (S.T_F32, ROW, 14336, 2048, 64, 991.1, 69.9), (S.T_F32, ROW, 1003, 1003, 64, 35.5, 14.2),
    (S.T_F16, ROW, 3072, 3072, 14, 18.2, 22.9), (S.T_F16, ROW, 3072, 3072, 32, 30.6, 23.0),
    (S.T_F16, ROW, 1024, 4096, 64, 25.5, 28.9), (S.T_F16, ROW, 1536, 8960, 24, 47.7, 57.1),
    (S.T_F16, ROW, 14336, 2048, 64, 379.4, 50.2), (S.T_F16, ROW, 2048, 512, 64, 20.9, 8.2),
    (S.T_F16, ROW, 3120, 4192, 16, 55.8, 29.7), (S.T_F16, ROW, 4096, 4096, 12, 29.8, 28.9),
    (S.T_BF16, ROW, 4096, 4096, 48, 100.2, 107.1), (S.T_BF16, ROW, 4096, 4096, 64, 139.2, 107.4),
    (S.T_BF16, ROW, 14336, 2048, 8, 39.3, 56.9), (S.T_BF16, ROW, 14336, 2048, 64, 291.8, 56.8),
]


@pytest.mark.parametrize("case", MEASURED, ids=lambda c: f"{S.TYPE_NAME[c[0]]}_o{c[1]}_{c[2]}x{c[3]}_T{c[4]}")
def test_the_faster_side(case):
    type_, order, rows, cols, tokens, decode, shared = case
    assert matmul_path(type_, order, cols, rows, tokens) == (MATMUL_TOKENS if shared < decode else MATMUL_DECODE)


def test_other_paths():
    assert matmul_path(S.T_Q4_K, REPACKED, 4096, 14336, 1) == MATMUL_DECODE
    for t in (S.T_Q4_K, S.T_Q6_K, S.T_Q8_0, S.T_Q4_0):
        assert matmul_path(t, ROW, 4096, 14336, 8) == MATMUL_GEMM
    for t in (S.T_Q6_K, S.T_Q8_0, S.T_Q3_K, S.T_IQ4_XS):
        assert matmul_path(t, ROW, 4096, 14336, 7) == MATMUL_DECODE
    assert matmul_path(S.T_IQ4_XS, ROW, 4096, 14336, 64) == MATMUL_DECODE


@pytest.mark.parametrize("args", [(S.T_Q4_K, ROW, 4095, 16, 2), (S.T_Q4_K, ROW, 4096, 0, 2), (S.T_Q4_K, ROW, 4096, 16, 65), (99, ROW, 4096, 16, 2)])
def test_refusals(args):
    with pytest.raises(BackendError):
        matmul_path(*args)
