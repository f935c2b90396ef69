"""GPU parity tests of the Flat paths (through the C ABI) against the CPU oracle.

int8: exact int32 distances and ids, bit for bit.  fp32: the final candidates are re-evaluated in
the canonical scalar arithmetic, so distances and ids equal the oracle's bit for bit as well.
"""
import ctypes
import os

import numpy as np
import pytest
import torch

from indexsdk_amd import _capi

pytestmark = pytest.mark.gpu
GOLDEN = os.path.join(os.path.dirname(os.path.abspath(__file__)), "golden", "ivfpq_small.npz")


@pytest.fixture(scope="module")
def ix():
    import indexsdk_amd
    return indexsdk_amd


@pytest.mark.parametrize("d,n,nq,k", [(64, 5000, 33, 10), (512, 20000, 130, 100), (96, 3000, 7, 128), (40, 1000, 5, 3),
                                      # query rows in every 128-row block of several 256-row tiles, with and
                                      # without the staged epilogue operands (nq % 4)
                                      (128, 9000, 516, 20), (256, 6000, 301, 7)])
def test_flat_i8_exact(ix, oracle, d, n, nq, k):
    rng = np.random.default_rng(d + n)
    base = rng.integers(-127, 128, size=(n, d), dtype=np.int8)
    base[17] = base[5]                 # exact duplicates: ties resolve to the vector added first
    q = rng.integers(-127, 128, size=(nq, d), dtype=np.int8)
    q[0] = base[5]
    ids = (np.arange(n, dtype=np.int64) * 7 + 3)
    # a small scratch forces several base chunks, exercising the streaming top-k
    index = ix.AscendIndexInt8Flat(d, ix.METRIC_L2, scratch_bytes=4 << 20)
    index.add_with_ids(base[: n // 2], ids[: n // 2])
    index.add_with_ids(base[n // 2:], ids[n // 2:])
    assert index.ntotal == n
    assert np.array_equal(index.getBase(3, 10), base[3:13])
    D, I = index.search_int32(q, k)
    Dr, Ir = oracle.flat_i8(base, q, k, ids=ids)
    assert np.array_equal(D, Dr)
    assert np.array_equal(I, Ir)
    assert D[0, 0] == 0 and I[0, 0] == ids[5] and I[0, 1] == ids[17]
    Df, If = index.search(q, k)
    assert np.array_equal(If, Ir) and np.array_equal(Df, Dr.astype(np.float32))


def test_flat_i8_extremes_and_padding(ix, oracle):
    base = np.full((3, 512), -127, dtype=np.int8)
    base[1] = 127
    q = np.full((2, 512), 127, dtype=np.int8)
    index = ix.AscendIndexInt8Flat(512)
    index.add(base)
    D, I = index.search_int32(q, 5)
    Dr, Ir = oracle.flat_i8(base, q, 5)
    assert np.array_equal(D, Dr) and np.array_equal(I, Ir)
    assert D[0].tolist() == [0, 512 * 254 * 254, 512 * 254 * 254, 2**31 - 1, 2**31 - 1]
    assert I[0].tolist() == [1, 0, 2, -1, -1]
    index.reset()
    assert index.ntotal == 0
    D, I = index.search_int32(q, 2)
    assert np.all(I == -1)


def test_flat_i8_golden(ix):
    g = np.load(GOLDEN, allow_pickle=False)
    index = ix.AscendIndexInt8Flat(64)
    index.add(g["flat_i8_base"])
    D, I = index.search_int32(g["flat_i8_queries"], 12)
    assert np.array_equal(D, g["flat_i8_D"]) and np.array_equal(I, g["flat_i8_I"])


@pytest.mark.parametrize("d", [64, 128, 256, 384, 512, 768, 1024])
def test_flat_i8_every_dimension_of_the_resident_kernel(ix, oracle, d):
    """The dimensions of the reference's Int8Flat (AscendIndexInt8FlatImpl.cpp:55), each a kernel instance of its own:
    a base long enough for the seeded stretch (stored scores) and several bound-filtered launches, queries in more
    than one query tile with a ragged last block, a base that ends inside a tile of 256 and inside a block of 32."""
    n, nq, k = 41000 + 77, 300, 20
    rng = np.random.default_rng(d)
    base = rng.integers(-127, 128, size=(n, d), dtype=np.int8)
    q = rng.integers(-127, 128, size=(nq, d), dtype=np.int8)
    q[:5] = base[[0, 255, 256, n - 1, 31999]]          # tile edges come back at distance 0
    base[n - 3] = base[100]                             # a tie across launches: the vector added first wins
    index = ix.AscendIndexInt8Flat(d, ix.METRIC_L2, scratch_bytes=4 << 20)
    index.add(base[:1000])
    index.add(base[1000:1037])                          # adds that start and end inside blocks of 32
    index.add(base[1037:])
    D, I = index.search_int32(q, k)
    Dr, Ir = oracle.flat_i8(base, q, k)
    assert np.array_equal(D, Dr) and np.array_equal(I, Ir)
    assert index.last_search_stats()["score_launches"] >= 3
    assert D[:5, 0].tolist() == [0] * 5 and I[:5, 0].tolist() == [0, 255, 256, n - 1, 31999]


def test_flat_i8_storage_in_matrix_core_order_round_trips(ix, oracle):
    """What goes into the tiled base comes back row-major, across blocks of 32 and tiles of 256, for a dimension
    that is padded (100 -> 128 bytes per row) and one that is not; removal moves vectors inside that layout."""
    rng = np.random.default_rng(3)
    for d in (100, 64):
        n = 3000 + 19
        base = rng.integers(-127, 128, size=(n, d), dtype=np.int8)
        index = ix.AscendIndexInt8Flat(d)
        for s, e in ((0, 1), (1, 33), (33, 300), (300, n)):
            index.add(base[s:e])
        assert np.array_equal(index.getBase(0, n), base)
        assert np.array_equal(index.getBase(31, 2), base[31:33])
        assert np.array_equal(index.getBase(250, 600), base[250:850])
        gone = np.array([0, 31, 32, 255, 256, 1000, n - 1, n - 40], dtype=np.int64)
        assert index.remove_ids(gone) == len(gone)
        order = oracle.flat_remove_order(n, np.sort(gone))
        assert np.array_equal(index.getBase(0, n - len(gone)), base[order])
        q = rng.integers(-127, 128, size=(9, d), dtype=np.int8)
        D, I = index.search_int32(q, 7)
        Dr, Ir = oracle.flat_i8(base[order], q, 7, ids=order.astype(np.int64))
        assert np.array_equal(D, Dr) and np.array_equal(I, Ir)


@pytest.mark.parametrize("metric_name", ["L2", "IP"])
@pytest.mark.parametrize("d,n,nq,k", [(128, 20000, 100, 10), (96, 7000, 40, 100), (30, 900, 9, 5), (64, 9000, 300, 10)])
def test_flat_f32_bit_exact(ix, oracle, metric_name, d, n, nq, k):
    metric = ix.METRIC_L2 if metric_name == "L2" else ix.METRIC_INNER_PRODUCT
    rng = np.random.default_rng(n + d)
    centres = rng.standard_normal((20, d)).astype(np.float32)
    base = (centres[rng.integers(0, 20, n)] + 0.3 * rng.standard_normal((n, d))).astype(np.float32)
    q = (centres[rng.integers(0, 20, nq)] + 0.3 * rng.standard_normal((nq, d))).astype(np.float32)
    index = ix.AscendIndexFlat(d, metric, scratch_bytes=2 << 20)
    index.add(base[: n // 3])
    index.add(base[n // 3:])
    D, I = index.search(q, k)
    Dr, Ir = oracle.flat_f32(base, q, k, metric)
    assert np.array_equal(I, Ir)
    assert np.array_equal(D.view(np.uint32), Dr.view(np.uint32))
    assert np.array_equal(index.getBase(10, 5), base[10:15])


def test_flat_f32_padding_and_golden(ix, oracle):
    g = np.load(GOLDEN, allow_pickle=False)
    x, q = g["base"].astype(np.float32), g["queries"].astype(np.float32)
    index = ix.AscendIndexFlatL2(32)
    index.add(x[:400])
    D, I = index.search(q[:6], 12)
    assert np.array_equal(D.view(np.uint32), g["flat_f32_D"].view(np.uint32)) and np.array_equal(I, g["flat_f32_I"])
    small = ix.AscendIndexFlatL2(32)
    small.add(x[:5])
    D, I = small.search(q[:3], 9)
    Dr, Ir = oracle.flat_f32(x[:5], q[:3], 9)
    assert np.array_equal(I, Ir) and np.array_equal(D, Dr)
    assert np.all(I[:, 5:] == -1) and np.all(D[:, 5:] == np.finfo(np.float32).max)


def test_flat_i8_many_fused_chunks_and_overflow_fallback(ix, oracle):
    # 150k rows: one seeded stretch through the score scratch, then several filtered chunks
    rng = np.random.default_rng(77)
    d, n, nq, k = 64, 150_000, 70, 50
    base = rng.integers(-127, 128, size=(n, d), dtype=np.int8)
    q = rng.integers(-127, 128, size=(nq, d), dtype=np.int8)
    index = ix.AscendIndexInt8Flat(d, ix.METRIC_L2, scratch_bytes=8 << 20)
    index.add(base)
    D, I = index.search_int32(q, k)
    Dr, Ir = oracle.flat_i8(base, q, k)
    assert np.array_equal(D, Dr) and np.array_equal(I, Ir)
    # adversarial order: every later row is closer to the query than all earlier ones, so the
    # filtered chunks admit everything and overflow their candidate buffers -> exact fallback path
    n2 = 60_000
    ramp = np.zeros((n2, d), dtype=np.int8)
    steps = np.linspace(127, 0, n2).astype(np.int64)
    ramp[:, 0] = steps.astype(np.int8)
    ramp[:, 1] = (np.arange(n2) % 100).astype(np.int8)      # breaks ties between equal first coordinates
    q2 = np.zeros((3, d), dtype=np.int8)
    index2 = ix.AscendIndexInt8Flat(d, ix.METRIC_L2)
    index2.add(ramp)
    D, I = index2.search_int32(q2, 20)
    Dr, Ir = oracle.flat_i8(ramp, q2, 20)
    assert np.array_equal(D, Dr) and np.array_equal(I, Ir)


def test_flat_f32_many_fused_chunks(ix, oracle):
    rng = np.random.default_rng(78)
    d, n, nq, k = 32, 120_000, 40, 20
    base = rng.standard_normal((n, d)).astype(np.float32)
    q = rng.standard_normal((nq, d)).astype(np.float32)
    for metric in (ix.METRIC_L2, ix.METRIC_INNER_PRODUCT):
        index = ix.AscendIndexFlat(d, metric, scratch_bytes=8 << 20)
        index.add(base)
        D, I = index.search(q, k)
        Dr, Ir = oracle.flat_f32(base, q, k, metric)
        assert np.array_equal(I, Ir) and np.array_equal(D.view(np.uint32), Dr.view(np.uint32))


@pytest.mark.parametrize("metric_name", ["L2", "IP"])
def test_flat_f32_near_duplicates_are_redone_exactly(ix, oracle, metric_name):
    """3000 base vectors within 1e-6 of each other: for queries near them the matrix-core scores can
    neither rank them nor prove a candidate list complete; those queries are redone from canonical
    scores of the whole base and every result still equals the oracle's bit for bit."""
    metric = ix.METRIC_L2 if metric_name == "L2" else ix.METRIC_INNER_PRODUCT
    rng = np.random.default_rng(71)
    d, n, nq, k = 64, 12000, 60, 20
    base = rng.standard_normal((n, d)).astype(np.float32)
    base[:3000] = base[0] + (1e-6 * rng.standard_normal((3000, d))).astype(np.float32)
    q = rng.standard_normal((nq, d)).astype(np.float32)
    q[:10] = base[0] + (0.05 * rng.standard_normal((10, d))).astype(np.float32)
    if metric == ix.METRIC_INNER_PRODUCT:
        q[:10] = 3.0 * base[0] + (0.05 * rng.standard_normal((10, d))).astype(np.float32)
    index = ix.AscendIndexFlat(d, metric)
    index.add(base)
    D, I = index.search(q, k)
    reruns = index.last_search_stats()["exact_reruns"]
    assert 10 <= reruns < nq, reruns
    Dr, Ir = oracle.flat_f32(base, q, k, metric)
    assert np.array_equal(I, Ir)
    assert np.array_equal(D.view(np.uint32), Dr.view(np.uint32))


# Score rows of 4096 .. 98304 columns with k <= 384 are selected from registers (bound from group
# minima); the cases below hold a ragged last segment, every group count, running keys from an
# earlier chunk, and rows of many equal scores, which overflow the candidate list and are redone by
# the streaming selection.
@pytest.mark.parametrize("n,k,scratch", [(20003, 100, 0), (20003, 300, 0), (33000, 150, 0), (40000, 60, 6 << 20)])
def test_flat_f32_rows_selected_from_registers(ix, oracle, n, k, scratch):
    d, nq = 64, 50
    rng = np.random.default_rng(n + k)
    centres = rng.standard_normal((30, d)).astype(np.float32)
    base = (centres[rng.integers(0, 30, n)] + 0.3 * rng.standard_normal((n, d))).astype(np.float32)
    q = (centres[rng.integers(0, 30, nq)] + 0.3 * rng.standard_normal((nq, d))).astype(np.float32)
    index = ix.AscendIndexFlat(d, ix.METRIC_L2, scratch_bytes=scratch)
    index.add(base)
    D, I = index.search(q, k)
    Dr, Ir = oracle.flat_f32(base, q, k, ix.METRIC_L2)
    assert np.array_equal(I, Ir)
    assert np.array_equal(D.view(np.uint32), Dr.view(np.uint32))


def test_flat_rows_of_equal_scores_overflow_the_register_selection(ix, oracle):
    d, n, nq, k = 64, 24000, 20, 100
    rng = np.random.default_rng(5)
    protos = rng.standard_normal((5, d)).astype(np.float32)
    base = protos[rng.integers(0, 5, n)]
    q = (protos[rng.integers(0, 5, nq)] + 0.05 * rng.standard_normal((nq, d))).astype(np.float32)
    index = ix.AscendIndexFlat(d, ix.METRIC_L2)
    index.add(base)
    D, I = index.search(q, k)
    Dr, Ir = oracle.flat_f32(base, q, k, ix.METRIC_L2)
    assert np.array_equal(I, Ir) and np.array_equal(D.view(np.uint32), Dr.view(np.uint32))
    b8 = rng.integers(-127, 128, size=(4, d), dtype=np.int8)[rng.integers(0, 4, n)]
    q8 = rng.integers(-127, 128, size=(nq, d), dtype=np.int8)
    i8 = ix.AscendIndexInt8Flat(d)
    i8.add(b8)
    D, I = i8.search_int32(q8, k)
    Dr, Ir = oracle.flat_i8(b8, q8, k)
    assert np.array_equal(I, Ir) and np.array_equal(D, Dr)


def test_flat_i8_rows_selected_from_registers(ix, oracle):
    d, n, nq, k = 64, 30001, 40, 200
    rng = np.random.default_rng(6)
    base = rng.integers(-127, 128, size=(n, d), dtype=np.int8)
    q = rng.integers(-127, 128, size=(nq, d), dtype=np.int8)
    index = ix.AscendIndexInt8Flat(d)
    index.add(base)
    D, I = index.search_int32(q, k)
    Dr, Ir = oracle.flat_i8(base, q, k)
    assert np.array_equal(I, Ir) and np.array_equal(D, Dr)


@pytest.mark.parametrize("n,nq,scratch", [(9000, 37, 0), (2049, 129, 1 << 20), (50000, 5, 4 << 20), (1500, 3, 0)])
def test_flat_largest_k(ix, oracle, n, nq, scratch):
    """k = 2048, the API's maximum, on all three Flat variants: the streaming selection then runs on two
    scanning wavefronts (four pools of 4096 keys do not fit LDS), over one block of the base or several,
    and with fewer rows than k the tail is padding."""
    d, k = 64, 2048
    rng = np.random.default_rng(n + nq)
    bi = rng.integers(-127, 128, size=(n, d), dtype=np.int8)
    qi = rng.integers(-127, 128, size=(nq, d), dtype=np.int8)
    bi[n // 3] = bi[1]
    index = ix.AscendIndexInt8Flat(d, ix.METRIC_L2, scratch_bytes=scratch)
    index.add(bi)
    D, I = index.search_int32(qi, k)
    Dr, Ir = oracle.flat_i8(bi, qi, k)
    assert np.array_equal(I, Ir) and np.array_equal(D, Dr)
    centres = rng.standard_normal((16, d)).astype(np.float32)
    base = (centres[rng.integers(0, 16, n)] + 0.3 * rng.standard_normal((n, d))).astype(np.float32)
    q = (centres[rng.integers(0, 16, nq)] + 0.3 * rng.standard_normal((nq, d))).astype(np.float32)
    base[n // 3] = base[1]
    for metric in (ix.METRIC_L2, ix.METRIC_INNER_PRODUCT):
        flat = ix.AscendIndexFlat(d, metric, scratch_bytes=scratch)
        flat.add(base)
        D, I = flat.search(q, k)
        Dr, Ir = oracle.flat_f32(base, q, k, metric)
        assert np.array_equal(I, Ir)
        assert np.array_equal(D.view(np.uint32), Dr.view(np.uint32))


@pytest.mark.parametrize("kind", ["fp32_L2", "fp32_IP", "int8"])
def test_flat_remove_ids_follows_the_reference_order(ix, oracle, kind):
    """remove_ids with a batch of ids (some absent, some repeated, some held by two vectors) and with an id
    range: the count, the storage order afterwards (getIdxMap / getBase: every hole, highest first, is
    refilled with the vector that is last at that moment; Index.cpp:86-113) and the searches on what is left
    equal the oracle's, and vectors added afterwards land behind the survivors."""
    rng = np.random.default_rng(31)
    d, n = 48, 30000
    if kind == "int8":
        index = ix.AscendIndexInt8Flat(d, ix.METRIC_L2, scratch_bytes=4 << 20)
        base = rng.integers(-127, 128, size=(n, d), dtype=np.int8)
        q = rng.integers(-127, 128, size=(40, d), dtype=np.int8)
    else:
        metric = ix.METRIC_L2 if kind == "fp32_L2" else ix.METRIC_INNER_PRODUCT
        index = ix.AscendIndexFlat(d, metric, scratch_bytes=4 << 20)
        base = rng.standard_normal((n, d)).astype(np.float32)
        q = rng.standard_normal((40, d)).astype(np.float32)
    ids = rng.permutation(10 * n)[:n].astype(np.int64)
    ids[100] = ids[7]                                   # one id held by two vectors: both leave
    index.add_with_ids(base[:20000], ids[:20000])
    index.add_with_ids(base[20000:], ids[20000:])

    def check(base, ids, k=12):
        assert index.ntotal == len(ids)
        assert np.array_equal(index.getIdxMap(), ids)
        assert np.array_equal(index.getBase(), base)
        if kind == "int8":
            D, I = index.search_int32(q, k)
            Dr, Ir = oracle.flat_i8(base, q, k, ids=ids)
            assert np.array_equal(D, Dr) and np.array_equal(I, Ir)
        else:
            D, I = index.search(q, k)
            Dr, Ir = oracle.flat_f32(base, q, k, index.metric_type, ids=ids)
            assert np.array_equal(I, Ir) and np.array_equal(D.view(np.uint32), Dr.view(np.uint32))

    check(base, ids)
    victims = np.concatenate([rng.choice(ids, 2500, replace=False), ids[-3:], [ids[7]], [-5, 10 * n + 1], ids[:4], ids[:4]])
    gone = np.nonzero(np.isin(ids, victims))[0]
    assert index.remove_ids(victims) == len(gone)
    order = oracle.flat_remove_order(n, gone)
    base, ids = base[order], ids[order]
    check(base, ids)
    assert index.remove_ids(np.array([-5], dtype=np.int64)) == 0 and index.remove_ids(np.empty(0, dtype=np.int64)) == 0
    lo, hi = 1000, 40000
    gone = np.nonzero((ids >= lo) & (ids < hi))[0]
    assert len(gone) > 1000 and index.remove_range(lo, hi) == len(gone)
    order = oracle.flat_remove_order(len(ids), gone)
    base, ids = base[order], ids[order]
    check(base, ids)
    assert index.remove_range(hi, lo) == 0
    extra = base[:50][::-1].copy()
    extra_ids = np.arange(50, dtype=np.int64) + 20 * n
    index.add_with_ids(extra, extra_ids)
    base, ids = np.concatenate([base, extra]), np.concatenate([ids, extra_ids])
    check(base, ids)
    assert index.remove_range(-1, 30 * n) == len(ids) and index.ntotal == 0      # everything leaves
    if kind == "int8":
        D, I = index.search_int32(q[:2], 3)
    else:
        D, I = index.search(q[:2], 3)
    assert (I == -1).all()


@pytest.mark.parametrize("kind", ["fp32_L2", "fp32_IP", "int8"])
def test_flat_search_with_masks(ix, oracle, kind):
    """search_with_masks: every query has its own bit mask over the storage positions (bit p % 8 of byte p / 8;
    FR/test/DTascendhost/TestAscendIndexInt8Flat.cpp:230-240 reads it that way); the answer is the oracle's
    brute force over the vectors that take part, bit for bit, with sentinels when fewer than k do.  A full
    mask gives the plain search; the base has a length that is no multiple of eight and spans several
    stretches of the score scratch."""
    rng = np.random.default_rng(61)
    d, n, nq, k = 40, 20003, 24, 30
    if kind == "int8":
        index = ix.AscendIndexInt8Flat(d, ix.METRIC_L2, scratch_bytes=1 << 20)
        base = rng.integers(-127, 128, size=(n, d), dtype=np.int8)
        q = rng.integers(-127, 128, size=(nq, d), dtype=np.int8)
        base[101] = base[7]                              # a tie across the mask
    else:
        metric = ix.METRIC_L2 if kind == "fp32_L2" else ix.METRIC_INNER_PRODUCT
        index = ix.AscendIndexFlat(d, metric, scratch_bytes=1 << 20)
        base = rng.standard_normal((n, d)).astype(np.float32)
        q = rng.standard_normal((nq, d)).astype(np.float32)
    ids = rng.permutation(5 * n)[:n].astype(np.int64)
    index.add_with_ids(base, ids)
    stride = (n + 7) // 8
    allowed = rng.random((nq, n)) < 0.5
    allowed[0] = True                                    # everything takes part
    allowed[1] = False                                   # nothing does
    allowed[2] = False
    allowed[2, rng.choice(n, 11, replace=False)] = True  # fewer than k
    allowed[3] = False
    allowed[3, -1] = True                                # only the last vector (a bit of the last, partial byte)
    allowed[4, 7] = False                                # of two equal vectors only the later one
    allowed[4, 101] = True
    mask = np.packbits(allowed, axis=1, bitorder="little")
    assert mask.shape == (nq, stride)
    if kind == "int8":
        q[4] = base[7]
        search = lambda qq, m: index.search_with_masks_int32(qq, k, m)
        plain = index.search_int32(q, k)
        brute = lambda sel, qq: oracle.flat_i8(base[sel], qq, k, ids=ids[sel])
    else:
        search = lambda qq, m: index.search_with_masks(qq, k, m)
        plain = index.search(q, k)
        brute = lambda sel, qq: oracle.flat_f32(base[sel], qq, k, index.metric_type, ids=ids[sel])
    D, I = search(q, mask)
    assert np.array_equal(I[0], plain[1][0]) and np.array_equal(D[0], plain[0][0])
    for i in range(nq):
        sel = np.nonzero(allowed[i])[0]
        if len(sel) == 0:
            assert (I[i] == -1).all()
            continue
        Dr, Ir = brute(sel, q[i:i + 1])
        assert np.array_equal(I[i], Ir[0]), i
        assert np.array_equal(D[i].view(np.uint32), Dr[0].view(np.uint32)), i
    assert (I[2, 11:] == -1).all() and (I[2, :11] >= 0).all()
    assert I[3, 0] == ids[-1] and (I[3, 1:] == -1).all()
    if kind == "int8":
        assert I[4, 0] == ids[101] and D[4, 0] == 0
    # the index answers plain searches as before
    again = index.search_int32(q, k) if kind == "int8" else index.search(q, k)
    assert np.array_equal(again[1], plain[1]) and np.array_equal(again[0], plain[0])


def test_flat_int8_mask_precision_recipe(ix, oracle):
    """The reference's own mask test (testMaskPrecision, FR/test/DTascendhost/TestAscendIndexInt8Flat.cpp:287-325):
    300000 vectors of 384 int8 (more than one 262144-row block of the reference), top 100, every second mask
    byte 255 and the others 0, for 1, 32 and 128 queries taken from the base.  Its check -- every label of the
    plain search that passes the mask is among the masked results with the same distance -- and the stricter
    one here: the masked results are the brute-force answer over the vectors that pass, bit for bit."""
    rng = np.random.default_rng(2024)
    n, d, k = 300_000, 384, 100
    base = rng.integers(-127, 128, size=(n, d), dtype=np.int8)
    index = ix.AscendIndexInt8Flat(d, ix.METRIC_L2)
    index.add(base)
    stride = (n + 7) // 8
    row = np.zeros(stride, dtype=np.uint8)
    row[1::2] = 255
    passes = np.unpackbits(row, bitorder="little")[:n].astype(bool)
    sel = np.nonzero(passes)[0]
    for nq in (1, 32, 128):
        q = base[:nq]
        mask = np.ascontiguousarray(np.broadcast_to(row, (nq, stride)))
        D, I = index.search_int32(q, k)
        Dm, Im = index.search_with_masks_int32(q, k, mask)
        for i in range(nq):
            keep = passes[I[i]]
            found = {int(l): int(v) for l, v in zip(Im[i], Dm[i])}
            assert all(found.get(int(l)) == int(v) for l, v in zip(I[i][keep], D[i][keep])), i
        Dr, Ir = oracle.flat_i8(base[sel], q, k, ids=sel.astype(np.int64))
        assert np.array_equal(Im, Ir) and np.array_equal(Dm, Dr)
        assert passes[Im].all()


# Batches of more than 256 queries (1024 where rows are short) over bases of 32768 rows and more form their candidate scores from
# bf16 x 3 splits; the results are canonical scores all the same, so they equal the fp32 plan's bit for bit.
@pytest.mark.parametrize("metric_name", ["L2", "IP"])
@pytest.mark.parametrize("d,n,nq,k,scratch", [(64, 32768, 1027, 1, 0), (100, 34817, 259, 100, 0), (33, 70001, 1027, 20, 32 << 20),
                                              (200, 50001, 259, 300, 64 << 20)])
def test_flat_f32_large_batches_equal_small_ones(ix, oracle, metric_name, d, n, nq, k, scratch):
    metric = ix.METRIC_L2 if metric_name == "L2" else ix.METRIC_INNER_PRODUCT
    rng = np.random.default_rng(n + d)
    centres = rng.standard_normal((200, d)).astype(np.float32)
    base = (centres[rng.integers(0, 200, n)] + 0.4 * rng.standard_normal((n, d))).astype(np.float32)
    base[n - 3] = base[100]
    base[5] *= 50.0
    q = (centres[rng.integers(0, 200, nq)] + 0.4 * rng.standard_normal((nq, d))).astype(np.float32)
    q[0] = base[100]
    q[3] *= 1e-3
    q[7, 1] = np.nan
    q[8, 2] = np.inf
    q[9, 0] = -np.inf
    index = ix.AscendIndexFlat(d, metric, scratch_bytes=scratch)
    index.add(base)
    D, I = index.search(q, k)
    for s in range(0, nq, 130):
        Ds, Is = index.search(q[s:s + 130], k)
        assert np.array_equal(I[s:s + 130], Is)
        assert np.array_equal(D[s:s + 130].view(np.uint32), Ds.view(np.uint32))
    Dr, Ir = oracle.flat_f32(base, q[10:40], k, metric)
    assert np.array_equal(I[10:40], Ir) and np.array_equal(D[10:40].view(np.uint32), Dr.view(np.uint32))


def test_flat_f32_base_with_values_out_of_range_keeps_the_fp32_plan(ix):
    rng = np.random.default_rng(5)
    d, n, k = 32, 40000, 10
    base = rng.standard_normal((n, d)).astype(np.float32)
    base[17, 3] = np.inf
    base[18, 3] = np.nan
    q = rng.standard_normal((1100, d)).astype(np.float32)
    for metric in (ix.METRIC_L2, ix.METRIC_INNER_PRODUCT):
        index = ix.AscendIndexFlat(d, metric)
        index.add(base)
        D, I = index.search(q, k)
        Ds, Is = index.search(q[:100], k)
        assert np.array_equal(I[:100], Is) and np.array_equal(D[:100].view(np.uint32), Ds.view(np.uint32))


# The kernel that keeps a tile of 256, 128, 64 or 32 queries in LDS and splits fp32 base rows in registers (dimensions that are a
# multiple of 4): remainders of the dimension, of the 256-row tile, of a wavefront's 32 rows and of four rows, tiles that the batch
# does not fill, scores stored and bound-filtered (scratch of 8 MB).  Canonical results: the oracle's, bit for bit.
@pytest.mark.parametrize("metric_name", ["L2", "IP"])
@pytest.mark.parametrize("d,n,nq,k,scratch", [(36, 2048, 1, 1, 0), (64, 2049, 257, 10, 0), (100, 2303, 33, 300, 0),
                                              (128, 4095, 129, 100, 0), (132, 3001, 300, 20, 0), (256, 2050, 65, 5, 0),
                                              (388, 2305, 64, 100, 0), (512, 2559, 31, 10, 0), (768, 2561, 40, 384, 0),
                                              (1024, 2100, 3, 7, 0), (44, 65537, 300, 10, 8 << 20), (96, 65794, 385, 100, 8 << 20),
                                              (200, 70001, 259, 3, 8 << 20), (384, 65567, 70, 60, 2 << 20)])
def test_flat_f32_split_in_the_score_kernel(ix, oracle, metric_name, d, n, nq, k, scratch):
    metric = ix.METRIC_L2 if metric_name == "L2" else ix.METRIC_INNER_PRODUCT
    rng = np.random.default_rng(d + n)
    centres = rng.standard_normal((50, d)).astype(np.float32)
    base = (centres[rng.integers(0, 50, n)] + 0.5 * rng.standard_normal((n, d))).astype(np.float32)
    base[n - 1] = base[0]
    q = (centres[rng.integers(0, 50, nq)] + 0.5 * rng.standard_normal((nq, d))).astype(np.float32)
    q[nq - 1] = base[0]
    index = ix.AscendIndexFlat(d, metric, scratch_bytes=scratch)
    index.add(base)
    some = np.unique(np.concatenate([np.arange(min(nq, 3)), [nq - 1], np.arange(31, nq, 32), np.arange(32, nq, 32)]))
    Dr, Ir = oracle.flat_f32(base, q[some], k, metric)
    D, I = index.search(q, k)
    assert np.array_equal(I[some], Ir) and np.array_equal(D[some].view(np.uint32), Dr.view(np.uint32))
    # queries in device memory that are not 16-byte aligned keep the fp32 kernels
    room = torch.zeros(nq * d + 1, device="cuda")
    room[1:] = torch.from_numpy(q).reshape(-1)
    Dd, Id = torch.empty(nq, k, device="cuda"), torch.empty(nq, k, device="cuda", dtype=torch.int64)
    torch.cuda.synchronize()
    _capi.check(_capi.load().flat_search_device(index._h, nq, ctypes.c_void_p(room.data_ptr() + 4), k,
                                                ctypes.c_void_p(Dd.data_ptr()), ctypes.c_void_p(Id.data_ptr())))
    assert np.array_equal(Id.cpu().numpy(), I) and np.array_equal(Dd.cpu().numpy().view(np.uint32), D.view(np.uint32))


# Up to 64 queries over 32768 rows and more: every row of scores is selected by several workgroups, whose keys one more orders.
@pytest.mark.parametrize("nq,k,scratch", [(1, 1, 0), (8, 128, 0), (64, 300, 0), (65, 128, 0), (3, 384, 20 << 20), (3, 385, 0)])
def test_flat_few_queries_over_a_long_base(ix, oracle, nq, k, scratch):
    rng = np.random.default_rng(nq + k)
    n, d = 100_003, 64
    base = rng.integers(-20, 21, size=(n, d), dtype=np.int8)
    base[50_000:50_400] = base[7]          # equal scores on both sides of a stretch's end
    q = rng.integers(-20, 21, size=(nq, d), dtype=np.int8)
    q[0] = base[7]
    index = ix.AscendIndexInt8Flat(d, ix.METRIC_L2, scratch_bytes=scratch) if scratch else ix.AscendIndexInt8Flat(d, ix.METRIC_L2)
    index.add(base)
    D, I = index.search_int32(q, k)
    Dr, Ir = oracle.flat_i8(base, q, k)
    assert np.array_equal(D, Dr) and np.array_equal(I, Ir)
    x, y = base.astype(np.float32), q.astype(np.float32)
    index = ix.AscendIndexFlat(d, ix.METRIC_L2, scratch_bytes=scratch)
    index.add(x)
    D, I = index.search(y, k)
    Dr, Ir = oracle.flat_f32(x, y, k, ix.METRIC_L2)
    assert np.array_equal(D, Dr) and np.array_equal(I, Ir)


# Vectors so short that fp32 sums of their squares lose everything (components below 1e-19): the length that the completeness
# proof multiplies its error bound with is 0, so the proof may not be believed.  1100 queries take the bf16 x 3 plan, 100 the fp32
# one; the base lies so close around one point that its inner products differ by less than either plan's scores err.
@pytest.mark.parametrize("metric_name", ["L2", "IP"])
@pytest.mark.parametrize("qscale,bscale", [(1e-24, 1.0), (1e-30, 1.0), (1e-36, 1.0), (1.0, 1e-24), (1e-19, 1e-17)])
def test_flat_f32_queries_and_bases_of_vanishing_norm(ix, oracle, metric_name, qscale, bscale):
    metric = ix.METRIC_L2 if metric_name == "L2" else ix.METRIC_INNER_PRODUCT
    rng = np.random.default_rng(24)
    d, n, k = 64, 40000, 10
    point = rng.standard_normal(d)
    for spread in (1e-5, 1e-6):
        base = (bscale * (point + spread * rng.standard_normal((n, d)))).astype(np.float32)
        q = (qscale * rng.standard_normal((1100, d))).astype(np.float32)
        index = ix.AscendIndexFlat(d, metric)
        index.add(base)
        Dr, Ir = oracle.flat_f32(base, q[:40], k, metric)
        for nq in (1100, 100):
            D, I = index.search(q[:nq], k)
            assert np.array_equal(I[:40], Ir) and np.array_equal(D[:40].view(np.uint32), Dr.view(np.uint32)), (nq, spread)


def test_flat_f32_a_batch_that_splits_do_not_pay_for(ix):
    """Splitting the base costs the same for every batch: 256 queries over 65536 rows bring too few products for it and keep
    the plan of 255 queries (371 us; with splits 455)."""
    rng = np.random.default_rng(1)
    d, n, k = 768, 65536, 100
    base = rng.standard_normal((n, d)).astype(np.float32)
    q = rng.standard_normal((256, d)).astype(np.float32)
    index = ix.AscendIndexFlat(d, ix.METRIC_L2)
    index.add(base)

    def milliseconds(nq):
        best = 1e9
        for _ in range(30):
            index.search(q[:nq], k)
            best = min(best, index.last_search_stats()["ms_total"])
        return best

    assert milliseconds(256) < 1.1 * milliseconds(255)


@pytest.mark.parametrize("offset", [10.0, 14.0, 20.0, 28.0, 60.0])
def test_flat_f32_queries_that_splits_leave_unproven(ix, offset):
    """Vectors with a common offset: inner products grow against the gaps between distances, until first the splits' error bound
    and then that of fp32 scores exceeds the gap behind the k-th.  Whatever the plan of the batch, a query is redone from
    canonical scores only where fp32 scores do not prove it either, and the answers are those of small batches."""
    rng = np.random.default_rng(3)
    d, n, nq, k = 128, 60000, 510, 10
    centres = rng.standard_normal((256, d))
    base = (centres[rng.integers(0, 256, n)] + 0.5 * rng.standard_normal((n, d)) + offset).astype(np.float32)
    q = (centres[rng.integers(0, 256, nq)] + 0.5 * rng.standard_normal((nq, d)) + offset).astype(np.float32)
    index = ix.AscendIndexFlat(d, ix.METRIC_L2)
    index.add(base)
    parts, redone = [], 0
    for s in range(0, nq, 255):
        parts.append(index.search(q[s:s + 255], k))
        redone += index.last_search_stats()["exact_reruns"]
    for _ in range(20):   # also where batches of this base have stopped taking splits, and when one tries again
        D, I = index.search(q, k)
        assert index.last_search_stats()["exact_reruns"] <= redone   # (a few less: the splits' list has more spare candidates)
        assert np.array_equal(I, np.concatenate([p[1] for p in parts]))
        assert np.array_equal(D.view(np.uint32), np.concatenate([p[0] for p in parts]).view(np.uint32))


@pytest.mark.parametrize("metric_name", ["L2", "IP"])
def test_flat_f32_an_undefined_vector_does_not_hide_the_longest(ix, oracle, metric_name):
    """The margin of the completeness proof grows with the longest vector of the base, also when a vector with an undefined
    norm was added along with it: a base so close around one point that fp32 scores cannot order it is redone exactly."""
    metric = ix.METRIC_L2 if metric_name == "L2" else ix.METRIC_INNER_PRODUCT
    rng = np.random.default_rng(8)
    d, n, k = 64, 40000, 10
    short = (1e-3 * rng.standard_normal((100, d))).astype(np.float32)
    base = (8.0 * rng.standard_normal(d) + 2e-5 * rng.standard_normal((n, d))).astype(np.float32)
    undefined = np.full((1, d), np.nan, dtype=np.float32)
    q = (8.0 * rng.standard_normal((40, d))).astype(np.float32)
    index = ix.AscendIndexFlat(d, metric)
    index.add(short)
    index.add(np.concatenate([base, undefined]))
    D, I = index.search(q, k)
    Dr, Ir = oracle.flat_f32(np.concatenate([short, base]), q, k, metric)
    assert np.array_equal(I, Ir) and np.array_equal(D.view(np.uint32), Dr.view(np.uint32))


@pytest.mark.parametrize("way", ["reset", "remove_ids", "remove_range", "remove all"])
def test_flat_f32_forgets_a_vector_without_a_finite_norm(ix, way):
    """An index that has lost an infinite and an undefined vector plans its searches like one that never had them: the same
    launches, nothing redone exactly (with an infinite margin every query is)."""
    rng = np.random.default_rng(6)
    d, n, nq, k = 128, 60000, 512, 10
    base = rng.standard_normal((n, d)).astype(np.float32)
    q = rng.standard_normal((nq, d)).astype(np.float32)
    odd = np.ones((2, d), dtype=np.float32)
    odd[0, 3], odd[1, 4] = np.inf, np.nan
    fresh = ix.AscendIndexFlat(d, ix.METRIC_L2, scratch_bytes=48 << 20)
    fresh.add(base)
    D, I = fresh.search(q, k)
    index = ix.AscendIndexFlat(d, ix.METRIC_L2, scratch_bytes=48 << 20)
    if way in ("reset", "remove all"):
        index.add(np.concatenate([base[:100], odd]))
        if way == "reset":
            index.reset()
        else:
            assert index.remove_range(0, 102) == 102
        index.add(base)
    else:
        index.add(np.concatenate([base, odd]))
        assert (index.remove_ids(np.array([n, n + 1])) if way == "remove_ids" else index.remove_range(n, n + 2)) == 2
    Dn, In = index.search(q, k)
    got, want = index.last_search_stats(), fresh.last_search_stats()
    assert got["exact_reruns"] == want["exact_reruns"] == 0
    assert got["score_launches"] == want["score_launches"]
    assert np.array_equal(In % n, I) and np.array_equal(Dn.view(np.uint32), D.view(np.uint32))


def test_flat_f32_split_queries_stay_within_the_scratch(ix, oracle):
    """Queries are split a page at a time: a larger batch costs its own inputs, results and candidate lists in memory (here 12
    bytes for each of 17 candidates), not 6 bytes per component for every query; the pages' results stand where the batch's do."""
    import ctypes
    rt = ctypes.CDLL("libamdhip64.so")

    def free_bytes():
        free, total = ctypes.c_size_t(), ctypes.c_size_t()
        assert rt.hipDeviceSynchronize() == 0 and rt.hipMemGetInfo(ctypes.byref(free), ctypes.byref(total)) == 0
        return free.value

    rng = np.random.default_rng(12)
    d, n, nq, k = 256, 33000, 70000, 1
    base = rng.standard_normal((n, d)).astype(np.float32)
    q = base[rng.integers(0, n, nq)] + np.float32(0.5) * rng.standard_normal((nq, d)).astype(np.float32)
    q[16383, 0], q[16384, 0], q[nq - 1, 0] = np.nan, np.inf, np.nan     # redone: on both sides of a page's end
    index = ix.AscendIndexFlat(d, ix.METRIC_L2)
    index.add(base)
    D, I = index.search(q[:16384], k)
    before = free_bytes()
    D, I = index.search(q, k)
    assert before - free_bytes() < (nq - 16384) * (4 * d + 17 * 12 + 64) + (32 << 20)
    for s in (0, 16300, 32700, 65500, nq - 200):
        Ds, Is = index.search(q[s:s + 200], k)
        assert np.array_equal(I[s:s + 200], Is) and np.array_equal(D[s:s + 200].view(np.uint32), Ds.view(np.uint32))
    Dr, Ir = oracle.flat_f32(base, q[16385:16405], k, ix.METRIC_L2)
    assert np.array_equal(I[16385:16405], Ir) and np.array_equal(D[16385:16405].view(np.uint32), Dr.view(np.uint32))


# Masked searches write every chunk of the score matrix: with 20 MB of scratch chunks of 40960, 40960 and 18083 columns.  The second is
# cut into stretches whose keys are ordered together with those the first has left.
@pytest.mark.parametrize("kind", ["int8", "float"])
@pytest.mark.parametrize("nq,k", [(1, 1), (5, 300), (64, 100)])
def test_flat_masked_few_queries_over_several_long_chunks(ix, kind, nq, k):
    rng = np.random.default_rng(nq)
    n, d = 100_003, 64
    base = rng.integers(-20, 21, size=(n, d), dtype=np.int8)
    base[40_700:41_300] = base[7]                                       # equal scores on both sides of a chunk's end
    q = rng.integers(-20, 21, size=(nq, d), dtype=np.int8)
    q[0] = base[7]
    passes = rng.random((nq, n)) < 0.5
    if nq > 2:
        passes[1] = False
        passes[1, [3, 40_959, 40_960, 50_000, n - 1]] = True            # fewer vectors take part than are asked for
        passes[2, :81_920] = False                                      # none of the first two chunks
    mask = np.packbits(passes, axis=1, bitorder="little")
    if kind == "int8":
        index = ix.AscendIndexInt8Flat(d, ix.METRIC_L2, scratch_bytes=20 << 20)
        index.add(base)
        D, I = index.search_with_masks_int32(q, k, mask)
    else:
        index = ix.AscendIndexFlat(d, ix.METRIC_L2, scratch_bytes=20 << 20)
        index.add(base.astype(np.float32))
        D, I = index.search_with_masks(q.astype(np.float32), k, mask)
    b = base.astype(np.float32)   # (sums of products up to 64 * 400: exact)
    dist = (b * b).sum(1) - 2 * (q.astype(np.float32) @ b.T) + (q.astype(np.float32) ** 2).sum(1, keepdims=True)
    dist[~passes] = np.inf
    want = np.argsort(dist, axis=1, kind="stable")[:, :k]
    best = np.take_along_axis(dist, want, 1)
    assert np.array_equal(I, np.where(np.isinf(best), -1, want))
    assert np.array_equal(D[np.isfinite(best)].astype(np.float32), best[np.isfinite(best)])


def _flat_on_device(ix, base, k):
    """An index over rows in device memory, and the seconds of one search of it."""
    import time

    index = ix.AscendIndexFlat(base.shape[1], ix.METRIC_L2)
    torch.cuda.synchronize()
    _capi.check(_capi.load().flat_add_with_ids_device(index._h, len(base), ctypes.c_void_p(base.data_ptr()), None))

    def search(q):
        D, I = torch.empty(len(q), k, device="cuda"), torch.empty(len(q), k, device="cuda", dtype=torch.int64)
        torch.cuda.synchronize()
        t = time.perf_counter()
        _capi.check(_capi.load().flat_search_device(index._h, len(q), ctypes.c_void_p(q.data_ptr()), k, ctypes.c_void_p(D.data_ptr()),
                                                    ctypes.c_void_p(I.data_ptr())))
        return time.perf_counter() - t
    search.index = index   # (lives as long as the function)
    return search


def test_flat_queries_without_proof_do_not_change_the_plan_of_the_next_batch(ix):
    """An undefined query, or one amid more near ties than its candidate list has room for, is served by other plans; the next
    batches keep the fast one (sixteen of them took up to three times as long when one such query was enough)."""
    gen = torch.Generator(device="cuda").manual_seed(3)
    base = torch.randn(500000, 128, generator=gen, device="cuda")
    base[:2000] = base[0] + 1e-5 * torch.randn(2000, 128, generator=gen, device="cuda")
    search = _flat_on_device(ix, base, 10)
    for nq in (1, 10, 300):
        q = torch.randn(nq, 128, generator=gen, device="cuda")
        undefined, tied = q.clone(), q.clone()
        undefined[0, 5] = float("nan")
        tied[0] = base[0]
        best = min(search(q) for _ in range(10))
        for odd in (undefined, tied):
            search(odd)
            assert min(search(q) for _ in range(10)) < 1.6 * best, nq


def test_flat_batches_with_some_unproven_queries_keep_the_faster_plan(ix):
    """An offset of 2 leaves a few of 300 queries unproven by splits: their second plan is cheaper than the older plan for all of them
    (2.4 times as long when any such batch sent the next sixteen there)."""
    gen = torch.Generator(device="cuda").manual_seed(4)
    centres = torch.randn(1024, 128, generator=gen, device="cuda")

    def rows(n):
        which = torch.randint(0, 1024, (n,), generator=gen, device="cuda")
        return centres[which] + 0.25 * torch.randn(n, 128, generator=gen, device="cuda")

    base, batches, mean = rows(500000), [rows(300) for _ in range(24)], []
    for offset in (0, 2):
        search = _flat_on_device(ix, base + offset, 100)
        times = [search(q + offset) for q in batches]
        mean.append(sum(times[4:]) / len(times[4:]))
    assert mean[1] < 1.8 * mean[0], mean
