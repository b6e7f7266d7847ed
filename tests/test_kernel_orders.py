"""Kernels of csrc/indexer.hip run on the host, in orders of their waves and
lanes that a GPU takes rarely: the results must not depend on them."""
import ctypes

import numpy as np
import pytest

import host_kernels

I64, P = ctypes.c_int64, ctypes.c_void_p
ORDERS = [(0, 0), (0, 1), (1, 0), (1, 1)]   # waves, lanes: ascending or descending


@pytest.fixture(scope="module")
def lib(tmp_path_factory):
    return host_kernels.build("indexer.hip", tmp_path_factory.mktemp("indexer"))


def topk(lib, x, lens, k, max_len):
    ws = lib.glm53_indexer_topk_workspace_bytes
    ws.restype, ws.argtypes = I64, [I64, I64, I64]
    run = lib.glm53_indexer_topk
    run.argtypes = [P, I64, P, I64, I64, I64, P, I64, P, I64, P]
    rows = x.shape[0]
    out = np.full((rows, k + 2 * max_len), -7, np.int32)     # room past each row: a stray rank shows
    need = ws(rows, max_len, k)
    scratch = np.zeros(need + 64, np.uint8)
    at = (scratch.ctypes.data + 63) // 64 * 64
    assert run(x.ctypes.data, x.shape[1], lens.ctypes.data, rows, max_len, k, at, need, out.ctypes.data,
               out.shape[1], None) == 0
    assert (out[:, k:] == -7).all()
    return out[:, :k]


def rows_of(n, k):
    """Rows that take every way through the selection: values that differ, a
    tie that holds most of a row with fewer than k keys above it (zeros, -inf
    or NaN), with more above it, few values, one value."""
    rng = np.random.default_rng(n + k)
    x = rng.standard_normal((8, n)).astype(np.float32)
    few = np.zeros(n, bool)
    few[::max(53, 2 * n // k)] = True
    x[1] = np.where(few, np.abs(x[1]), 0)
    x[2] = np.where(few, x[2], -np.inf)
    x[3] = np.where(few, x[3], np.nan)
    x[4] = np.where(rng.random(n) < 0.5, x[4], 0)
    x[5] = rng.integers(0, 3, n)
    x[6] = -1.5
    x[7] = np.arange(n)
    return x


# the one-workgroup selection (4097..131072 columns, k <= 1024) at 1024 threads, its row as one list, its edges
@pytest.mark.parametrize("n,k", [(4097, 512), (5001, 1024), (12001, 40), (16384, 512), (4000, 700)])
@pytest.mark.parametrize("order", ORDERS)
def test_topk_any_order(lib, oracle, n, k, order):
    lib.host_hip_order(*order)
    x = rows_of(n, k)
    lens = np.array([n, n, n - 1, n, n - 3, n, n, k], np.int32)
    assert np.array_equal(topk(lib, x, lens, k, n), oracle.indexer_topk(x, lens, k))


@pytest.mark.parametrize("order", ORDERS)
def test_topk_any_order_other_plans(lib, oracle, order):
    """512-thread workgroups (256 rows), the two stages (few rows of 20000
    columns) and the sweeps (more candidates than the final stage takes)."""
    lib.host_hip_order(*order)
    x = np.zeros((256, 5001), np.float32)
    x[:8] = rows_of(5001, 512)
    lens = np.zeros(256, np.int32)
    lens[:8] = 5001
    assert np.array_equal(topk(lib, x, lens, 512, 5001), oracle.indexer_topk(x, lens, 512))
    for n, k in ((20000, 512), (34000, 20000)):
        x = rows_of(n, k)[1:4]
        lens = np.array([n, n - 5, n], np.int32)
        assert np.array_equal(topk(lib, x, lens, k, n), oracle.indexer_topk(x, lens, k)), (n, k)


def sampled(n):
    """The 4096 positions of a row of n columns that the one-workgroup
    selection ranks for its bound (either workgroup size takes the same)."""
    part = np.arange(1024)
    at = (part * n // 1024 + ((part * 159 & 255) * (n // 1024 - 3) >> 8)) & ~3
    return (at[:, None] + np.arange(4)).reshape(-1)


# columns, k and rows of the call: 1024 threads, 512 threads, and few long rows
@pytest.mark.parametrize("n,k,rows", [(16384, 512, 6), (9001, 1024, 256), (40000, 1024, 24)])
def test_topk_misleading_sample(lib, oracle, n, k, rows):
    """Rows whose sample says the wrong thing: the sampled keys below all
    others (the list overflows) or above them (too few listed), one sampled
    value whose copies complete the list, too few copies of it, NaN all over
    the sample, and a row that repeats with the parts' length."""
    lib.host_hip_order(0, 0)
    rng = np.random.default_rng(n)
    x = np.zeros((rows, n), np.float32)
    x[:6] = rng.standard_normal((6, n))
    s = sampled(n)
    assert len(np.unique(s)) == 4096 and s.max() < n
    x[0, s] -= 20
    x[1, s] += np.where(np.arange(4096) < k // 2, 20, 0)
    x[2, s] = 5
    x[3, s[::8][:k - 300]] = 5
    x[4, s] = np.nan
    x[5, np.arange(n) % (n // 1024) < 4] -= 6
    lens = np.zeros(rows, np.int32)
    lens[:6] = n
    got = topk(lib, x, lens, k, n)
    assert np.array_equal(got[:6], oracle.indexer_topk(x[:6], lens[:6], k))


@pytest.mark.parametrize("order", ORDERS)
@pytest.mark.parametrize("heads,tokens,keys,clean", [(16, 17, 130, 1), (32, 16, 200, 0)])
def test_logits_rows_any_order(lib, heads, tokens, keys, clean, order):
    """The logits of rows that share one block table (keys staged in LDS,
    results handed between lanes for the stores) against the same rows with a
    table each: bit-identical, whichever lane of a wave runs first."""
    fn = lib.glm53_fp8_paged_mqa_logits
    fn.argtypes = [P, I64, I64, P, I64, I64, I64, P, I64, P, P, I64, I64, I64, I64, I64, I64, ctypes.c_int, P, I64, P]
    lib.host_hip_order(*order)
    rng = np.random.default_rng(heads + keys)
    block, pages = 16, (keys + 15) // 16
    q = rng.integers(0, 120, tokens * heads * 128 + 16, dtype=np.uint8)     # E4M3 of either sign, no NaN
    q ^= (rng.random(q.shape) < 0.5).astype(np.uint8) << 7
    kv = rng.integers(0, 120, pages * block * 132 + 16, dtype=np.uint8)
    qa, kva = (a.ctypes.data + 15 & ~15 for a in (q, kv))
    page = kv[kva - kv.ctypes.data:][:pages * block * 132].reshape(pages, block * 132)
    page[:, block * 128:] = (rng.random((pages, block), dtype=np.float32) - 0.2).view(np.uint8)
    w = rng.standard_normal((tokens, heads)).astype(np.float32)
    lens = rng.integers(0, keys + 1, tokens).astype(np.int32)
    lens[0] = keys
    table = rng.permutation(pages).astype(np.int32)
    out = []
    for bt, stride in ((table, 0), (np.tile(table, (tokens, 1)), pages)):
        o = np.full((tokens, keys), 7, np.float32)
        assert fn(qa, heads * 128, 128, kva, block * 132, block, pages, w.ctypes.data, heads, lens.ctypes.data,
                  bt.ctypes.data, stride, pages, tokens, heads, 128, keys, clean, o.ctypes.data, keys, None) == 0
        out.append(o)
    assert np.array_equal(out[0], out[1])
