"""GPU parity of attention over the KV ring cache (attn_rows, fastgguf.c:3273-3326) through the C ABI.

Every output is compared bit for bit: against the compiled reference's golden outputs and against
the oracle's restatement (pinned to those outputs) on decode and prompt-batch ranges, GQA head
groups, ring wrap, head sizes 32 .. 256, every range length mod 8 (the softmax tail), and scores
spread past exp_neg_ps's -87 cut-off. Head sizes that are not multiples of 32 (the reference's
per-row path, dot_f32v's score order) run with 16-value chunks only, an extra group of 8, a
scalar tail, and odd sizes whose rows are not 16-byte aligned.
"""
import numpy as np
import pytest
from conftest import bits_equal, bits_equal_or_nan

from fastgguf_amd.backend import BackendError

pytestmark = pytest.mark.gpu


def oracle_attention(oracle, q, ck, cv, st, en, n_head_kv, scale):
    n_tok, n_head, hd = q.shape
    g = n_head // n_head_kv
    rows_st = np.repeat(np.asarray(st, np.int32), n_head)
    rows_en = np.repeat(np.asarray(en, np.int32), n_head)
    kvo = np.tile(np.arange(n_head) // g * hd, n_tok).astype(np.int32)
    return oracle.attn_rows(q.reshape(-1, hd), rows_st, rows_en, ck, cv, kvo, hd, scale).reshape(q.shape)


def test_attention_matches_golden(backend):
    """The golden calls (up to 4 rows sharing a head offset) as one head of kv_dim / hd heads."""
    from test_oracle import attn_golden
    rng = np.random.default_rng(3)
    for c in attn_golden():
        hd, kvo = c["hd"], c["kvo"]
        n_head = c["ck"].shape[1] // hd
        q = rng.standard_normal((len(c["st"]), n_head, hd)).astype(np.float32)
        q[:, kvo // hd] = c["q"]
        o = backend.attention(q, c["ck"], c["cv"], c["st"], c["en"], n_head, c["scale"])
        assert bits_equal_or_nan(o[:, kvo // hd], c["o"]), (hd, kvo, c["st"], c["en"])


CASES = [  # (n_tok, n_head, n_head_kv, hd, cap, first position, magnitude)
    (1, 4, 4, 32, 64, 0, 1.0),        # one position
    (1, 8, 2, 64, 100, 90, 1.0),      # decode over a wrapped ring
    (9, 8, 2, 128, 200, 180, 1.0),    # causal prompt batch over a wrapped ring, every length mod 8
    (5, 6, 3, 96, 40, 33, 1.0),       # hd 96, ring shorter than the range start
    (3, 4, 1, 256, 70, 60, 1.0),      # hd 256, multi-query
    (4, 2, 2, 32, 50, 10, 30.0),      # scores past the -87 cut-off
    (1, 32, 32, 80, 300, 250, 1.0),   # per-row path: hd 80 decode (five 16-value chunks)
    (9, 8, 2, 112, 60, 50, 1.0),      # hd 112: chunks and one group of 8, prompt batch, GQA
    (5, 6, 3, 100, 40, 33, 1.0),      # hd 100: a scalar tail of 4
    (70, 4, 2, 72, 100, 20, 1.0),     # hd 72, 70 tokens x 2 heads per K head: the 16-row value kernel
    (3, 5, 5, 13, 30, 25, 2.0),       # odd hd: unaligned rows, values read one by one
    (66, 2, 1, 6, 80, 0, 1.0),        # tiny hd: the tail only; 66 rows per K head
]


@pytest.mark.parametrize("case", CASES, ids=lambda c: f"t{c[0]}h{c[1]}kv{c[2]}d{c[3]}cap{c[4]}")
def test_attention_matches_oracle(backend, oracle, case):
    n_tok, n_head, n_kv, hd, cap, p0, mag = case
    rng = np.random.default_rng(hd + cap)
    kv_dim = n_kv * hd
    ck = rng.standard_normal((cap, kv_dim)).astype(np.float32)
    cv = rng.standard_normal((cap, kv_dim)).astype(np.float32)
    q = (rng.standard_normal((n_tok, n_head, hd)) * mag).astype(np.float32)
    en = p0 + np.arange(n_tok, dtype=np.int32) + min(cap - n_tok, 30)
    st = np.maximum(en - (cap - 1), p0).astype(np.int32)  # as long as the cache allows
    if n_tok > 1:
        st[:] = p0  # causal: token t sees p0 .. p0 + (offset) + t
    scale = float(np.float32(1 / np.sqrt(hd)))
    o = backend.attention(q, ck, cv, st, en, n_kv, scale)
    assert bits_equal(o, oracle_attention(oracle, q, ck, cv, st, en, n_kv, scale))


@pytest.mark.parametrize("case", [(70, 4, 2, 72, 100, 20), (66, 2, 1, 6, 80, 0), (3, 5, 5, 13, 30, 25)],
                         ids=["d72_16row", "d6_16row_unaligned", "d13_4row_unaligned"])
def test_attention_per_row_path_nonfinite_v(backend, oracle, case):
    """The per-row path (hd % 32 != 0) walks each row's own positions only (fastgguf.c:3318-3323):
    inf and NaN in V at the last position of a causal batch, which only the last token attends,
    leave every other token's outputs finite, in the value kernel's 16-row and 4-row groups alike.
    (The vector path walks its call's whole span, with NaN where fma(0, inf) falls: the golden
    case with hd 64 covers that.)"""
    n_tok, n_head, n_kv, hd, cap, p0 = case
    rng = np.random.default_rng(hd + 7)
    kv_dim = n_kv * hd
    ck = rng.standard_normal((cap, kv_dim)).astype(np.float32)
    cv = rng.standard_normal((cap, kv_dim)).astype(np.float32)
    q = rng.standard_normal((n_tok, n_head, hd)).astype(np.float32)
    en = (p0 + 5 + np.arange(n_tok)).astype(np.int32)
    st = np.full(n_tok, p0, np.int32)
    last = int(en[-1]) % cap
    cv[last, 0] = np.inf
    cv[last, kv_dim - 1] = np.nan
    scale = float(np.float32(1 / np.sqrt(hd)))
    o = backend.attention(q, ck, cv, st, en, n_kv, scale)
    want = oracle_attention(oracle, q, ck, cv, st, en, n_kv, scale)
    assert np.isfinite(want[:-1]).all() and not np.isfinite(want[-1]).all()
    assert bits_equal_or_nan(o, want)


def test_attention_long_decode(backend, oracle):
    """A Llama-3-8B-shaped decode step (32 heads over 8 KV heads, hd 128) at 4096 positions of a
    wrapped 4096-slot ring, and a 64-token prompt batch at the end of the same cache."""
    rng = np.random.default_rng(11)
    cap, hd, n_head, n_kv = 4096, 128, 32, 8
    ck = rng.standard_normal((cap, n_kv * hd)).astype(np.float32)
    cv = rng.standard_normal((cap, n_kv * hd)).astype(np.float32)
    scale = float(np.float32(1 / np.sqrt(hd)))
    q = rng.standard_normal((1, n_head, hd)).astype(np.float32)
    st, en = np.array([5000], np.int32), np.array([5000 + cap - 1], np.int32)
    o = backend.attention(q, ck, cv, st, en, n_kv, scale)
    assert bits_equal(o, oracle_attention(oracle, q, ck, cv, st, en, n_kv, scale))
    q = rng.standard_normal((64, n_head, hd)).astype(np.float32)
    en = (2000 + np.arange(64)).astype(np.int32)
    st = np.zeros(64, np.int32)
    o = backend.attention(q, ck, cv, st, en, n_kv, scale)
    assert bits_equal(o, oracle_attention(oracle, q, ck, cv, st, en, n_kv, scale))


def test_attention_dev_bad_rows_are_nan(backend, oracle):
    """On device pointers the ranges are not checked on the host: a token whose range is empty or
    longer than max_len gets NaN outputs and the other tokens are unaffected."""
    rng = np.random.default_rng(12)
    cap, hd, n_head, n_kv = 64, 64, 4, 2
    ck = rng.standard_normal((cap, n_kv * hd)).astype(np.float32)
    cv = rng.standard_normal((cap, n_kv * hd)).astype(np.float32)
    q = rng.standard_normal((4, n_head, hd)).astype(np.float32)
    st = np.array([0, 10, 20, 5], np.int32)
    en = np.array([9, 9, 60, 30], np.int32)  # token 1 empty, token 2 longer than max_len 32
    scale = 0.125
    bufs = [backend.dev_alloc(a.nbytes) for a in (q, q, ck, cv, st, en)]
    try:
        for b, a in zip(bufs, (q, q, ck, cv, st, en)):
            backend.h2d(b, a)
        backend.attention_dev(4, n_head, n_kv, hd, bufs[0], bufs[1], bufs[2], bufs[3], n_kv * hd, cap, bufs[4],
                              bufs[5], 32, scale)
        o = np.empty_like(q)
        backend.d2h(o, bufs[1])
    finally:
        for b in bufs:
            backend.dev_free(b)
    assert np.all(np.isnan(o[1])) and np.all(np.isnan(o[2]))
    for t in (0, 3):
        want = oracle_attention(oracle, q[t:t + 1], ck, cv, st[t:t + 1], en[t:t + 1], n_kv, scale)
        assert bits_equal(o[t:t + 1], want)


def test_attention_refusals(backend):
    rng = np.random.default_rng(13)
    ck = rng.standard_normal((16, 96)).astype(np.float32)
    q = rng.standard_normal((1, 1, 288)).astype(np.float32)
    with pytest.raises(BackendError):  # hd above 256
        backend.attention(q, np.zeros((16, 288), np.float32), np.zeros((16, 288), np.float32), [0], [3], 1, 0.1)
    q = rng.standard_normal((1, 3, 32)).astype(np.float32)
    with pytest.raises(BackendError):  # 3 heads over 2 KV heads
        backend.attention(q, ck, ck, [0], [3], 2, 0.1)
    q = rng.standard_normal((1, 2, 32)).astype(np.float32)
    with pytest.raises(BackendError):  # range longer than the cache
        backend.attention(q, ck, ck, [0], [16], 2, 0.1)
    with pytest.raises(BackendError):  # empty range
        backend.attention(q, ck, ck, [5], [4], 2, 0.1)


@pytest.mark.parametrize("n_tok,n_head,n_kv,hd", [(1, 4, 1, 64), (3, 2, 2, 72), (17, 4, 1, 32), (70, 3, 3, 36), (33, 8, 2, 96)],
                         ids=["4row", "4row_per_row_path", "16row", "16row_per_row_path", "16row_hd96"])
@pytest.mark.parametrize("length", [1, 15, 33, 127, 128, 129, 256, 257, 385, 512, 600])
def test_attention_value_tile_edges(backend, oracle, n_tok, n_head, n_kv, hd, length):
    """The value kernels' tiles of 128 (64 rows and more per K head) and 256 positions: ranges that
    end around whole tiles, start anywhere in the ring and wrap inside a tile, groups with rows of
    other ranges and a last group that is not full. Each sum is the reference's chain of fmas, so
    every output is equal bit for bit."""
    rng = np.random.default_rng(length * 7 + hd)
    cap = length + n_tok + 5
    ck = rng.standard_normal((cap, n_kv * hd)).astype(np.float32)
    cv = rng.standard_normal((cap, n_kv * hd)).astype(np.float32)
    q = rng.standard_normal((n_tok, n_head, hd)).astype(np.float32)
    st = np.full(n_tok, cap // 2 + 3, np.int32)
    en = (st + length - 1 + np.arange(n_tok)).astype(np.int32)
    st[n_tok // 2:] += 2 if length > 2 else 0  # rows of one group that start apart
    scale = float(np.float32(1 / np.sqrt(hd)))
    o = backend.attention(q, ck, cv, st, en, n_kv, scale)
    assert bits_equal(o, oracle_attention(oracle, q, ck, cv, st, en, n_kv, scale))


# rows per K head (token x query heads of the K head): the 4-row score kernel up to 15, the 16-row one with 1, 2
# and 4 wavefronts from 16, 17 and 33; the 16-row value kernel from 64
@pytest.mark.parametrize("n_tok,g", [(1, 1), (5, 3), (4, 4), (17, 1), (8, 4), (11, 3), (16, 4), (13, 5)], ids=lambda v: str(v))
@pytest.mark.parametrize("hd", [32, 64, 96, 128, 160, 192, 224, 256])
def test_attention_score_kernel_forms(backend, oracle, hd, n_tok, g):
    """Every head size of the vector path in every score kernel form, ranges that end around its 64-key
    tiles (63, 64, 65 and 130 keys for the first token) over a ring that wraps inside one, two K heads."""
    rng = np.random.default_rng(hd + 7 * n_tok + g)
    n_kv = 2
    scale = float(np.float32(1 / np.sqrt(hd)))
    for length in (63, 64, 65, 130):
        cap = length + n_tok + 2
        ck = rng.standard_normal((cap, n_kv * hd)).astype(np.float32)
        cv = rng.standard_normal((cap, n_kv * hd)).astype(np.float32)
        q = rng.standard_normal((n_tok, g * n_kv, hd)).astype(np.float32)
        st = np.full(n_tok, cap - 20, np.int32)
        en = (st + length - 1 + np.arange(n_tok)).astype(np.int32)
        o = backend.attention(q, ck, cv, st, en, n_kv, scale)
        assert bits_equal(o, oracle_attention(oracle, q, ck, cv, st, en, n_kv, scale)), length


@pytest.mark.parametrize("n_tok,n_head", [(1, 2), (65, 4)], ids=["1024_threads", "256_threads"])
@pytest.mark.parametrize("length", [12288, 12289, 12300, 2 * 12288 + 5])
def test_attention_rows_beyond_lds(backend, oracle, n_tok, n_head, length):
    """Rows around and past the softmax's 12,288 resident positions (longer ones go through LDS in
    chunks that carry the ordered lane sums), in both of its workgroup sizes."""
    rng = np.random.default_rng(length + n_tok)
    hd, cap = 32, length + n_tok
    ck = rng.standard_normal((cap, hd)).astype(np.float32)
    cv = rng.standard_normal((cap, hd)).astype(np.float32)
    q = (rng.standard_normal((n_tok, n_head, hd)) * 2).astype(np.float32)
    st = np.full(n_tok, 77, np.int32)
    en = (st + length - 1).astype(np.int32)
    en[-1] += n_tok > 1
    scale = float(np.float32(1 / np.sqrt(hd)))
    o = backend.attention(q, ck, cv, st, en, 1, scale)
    assert bits_equal(o, oracle_attention(oracle, q, ck, cv, st, en, 1, scale))


@pytest.mark.parametrize("n_tok,g", [(2, 2), (4, 4), (16, 2), (20, 4)], ids=["scores4_values4", "scores16_1", "scores16_2", "scores16_4_values16"])
@pytest.mark.parametrize("hd", [64, 128])
def test_attention_mfma_specials(backend, oracle, hd, n_tok, g):
    """The fp32 MFMAs add each product as one fmaf: scores of subnormal products (scaled back up), -inf
    scores from an infinity in K, and value sums over subnormals, infinities and NaN in V. All rows
    attend the same positions; outputs equal bit for bit, any NaN as any NaN."""
    rng = np.random.default_rng(hd + n_tok)
    n = 150
    q = rng.standard_normal((n_tok, g, hd)).astype(np.float32)
    q[..., 5] = np.abs(q[..., 5])
    ck = rng.standard_normal((n, hd)).astype(np.float32)
    cv = rng.standard_normal((n, hd)).astype(np.float32)
    ck[7, 5] = ck[90, 5] = -np.inf
    cv[:, 1] *= np.float32(1e-39)
    cv[:, 2] = np.float32(1e-44)
    cv[:, 3] = -0.0
    cv[100, 8], cv[101, 9] = np.inf, -np.inf
    cv[3, 10], cv[140, 10] = np.inf, -np.inf
    cv[77, 11] = np.nan
    st, en = np.zeros(n_tok, np.int32), np.full(n_tok, n - 1, np.int32)
    for qs, ks, scale in ((1.0, 1.0, float(np.float32(1 / np.sqrt(hd)))), (1e-20, 1e-20, 3e38)):
        qq, kk = (q * np.float32(qs)).astype(np.float32), (ck * np.float32(ks)).astype(np.float32)
        o = backend.attention(qq, kk, cv, st, en, 1, scale)
        want = oracle_attention(oracle, qq, kk, cv, st, en, 1, scale)
        assert np.isnan(want[..., 10:12]).all() and np.isinf(want[..., 8:10]).all()
        assert np.isfinite(want[..., 12:]).all() and np.abs(want[..., 1]).max() < 1.2e-38
        assert bits_equal_or_nan(o, want)
