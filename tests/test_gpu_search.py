"""GPU brute-force search (k_search.hip, sg_search.cpp) against the CPU
oracle's restatement of search/brute: every score bit-exact, the top-k
identical (ids and distances, ties included), the storage format byte-exact.
"""
import struct
import sys

import numpy as np
import pytest

import oracle as o

pytestmark = pytest.mark.gpu

MODES = [0, 1, 2]  # float32, int8, int16 (brute.QuantizationMode)
MODE_NAMES = {0: "f32", 1: "i8", 2: "i16"}


def say(*a):
    print(*a, flush=True)
    sys.stdout.flush()


def _build(ctx, ids, vecs, mode):
    from semantica_gpu import search
    b = search.Builder(ctx, dimension=vecs.shape[1], quantization=mode)
    b.add_vectors(ids, vecs)
    return b.build()


def _oracle(vecs, ids, mode, queries, k, normalized):
    data = o.bf_quantize(o.bf_normalize(vecs), mode)
    out = []
    for q in queries:
        out.append(o.bf_search(data, mode, ids, q if normalized else o.bf_normalize(q), k))
    return data, out


def _check(idx, vecs, ids, mode, queries, k, normalized, tag):
    gi, gd, gn = idx.search_batch(queries, k, normalized=normalized)
    _, want = _oracle(vecs, ids, mode, queries, k, normalized)
    for q, (wi, wd) in enumerate(want):
        assert gn[q] == len(wi), (tag, q)
        assert np.array_equal(gi[q, :gn[q]], wi), (tag, q)
        assert np.array_equal(gd[q, :gn[q]].view(np.uint32), wd.view(np.uint32)), (tag, q)


@pytest.mark.parametrize("mode", MODES)
@pytest.mark.parametrize("dim", [1, 3, 4, 5, 7, 8, 9, 12, 64, 127, 768])
def test_every_score_bit_exact(gpu_ctx, mode, dim):
    """top_k = count returns every score, in the reference's order: all of
    them must equal the oracle's bit for bit (the 8-lane part, its reduction
    and the scalar tail for every dim % 8)."""
    rng = np.random.default_rng(dim * 3 + mode)
    n, nq = 700, 9  # 9 queries: one block of 8 and one of 1
    vecs = (rng.standard_normal((n, dim)) * rng.uniform(0.1, 10, (n, 1))).astype(np.float32)
    ids = rng.permutation(10 * n)[:n].astype(np.int32) - 3 * n
    queries = rng.standard_normal((nq, dim)).astype(np.float32)
    say(f"scores mode={MODE_NAMES[mode]} dim={dim}")
    idx = _build(gpu_ctx, ids, vecs, mode)
    try:
        _check(idx, vecs, ids, mode, queries, n, False, "all")
    finally:
        idx.close()


@pytest.mark.parametrize("mode", MODES)
def test_top_k_matches_oracle(gpu_ctx, mode):
    rng = np.random.default_rng(40 + mode)
    n, dim = 20000, 256
    vecs = rng.standard_normal((n, dim)).astype(np.float32)
    ids = np.arange(n, dtype=np.int32) * 7 + 1
    queries = rng.standard_normal((21, dim)).astype(np.float32)
    idx = _build(gpu_ctx, ids, vecs, mode)
    try:
        for k in (1, 10, 100, 1000):
            for normalized in (False, True):
                say(f"top-k mode={MODE_NAMES[mode]} k={k} normalized={normalized}")
                q = o.bf_normalize(queries) if normalized else queries
                _check(idx, vecs, ids, mode, q, k, normalized, f"k={k}")
    finally:
        idx.close()


@pytest.mark.parametrize("mode", MODES)
def test_ties_straddling_the_kth_place(gpu_ctx, mode):
    """Every vector stored three times under different ids (shuffled): equal
    scores straddle the k-th place for most k, which the reference resolves
    by its slot order (index.go:84-131).  The GPU must keep the same ids."""
    rng = np.random.default_rng(90 + mode)
    base = rng.standard_normal((500, 48)).astype(np.float32)
    rep = np.repeat(base, 3, axis=0)
    perm = rng.permutation(rep.shape[0])
    vecs = rep[perm]
    ids = (np.arange(vecs.shape[0], dtype=np.int32) * 13) % 100003
    queries = rng.standard_normal((16, 48)).astype(np.float32)
    idx = _build(gpu_ctx, ids, vecs, mode)
    try:
        for k in (1, 2, 3, 4, 5, 10, 31, 64, 65, 100, 1499, 1500):
            say(f"ties mode={MODE_NAMES[mode]} k={k}")
            _check(idx, vecs, ids, mode, queries, k, False, f"k={k}")
    finally:
        idx.close()


def test_zero_scores_of_both_signs_tie(gpu_ctx):
    """Vectors orthogonal to the query score +0 or -0 (a product with a
    negative code is -0); the reference compares them as equal.  k lands
    inside that run of zeros."""
    rng = np.random.default_rng(5)
    dim = 16
    pos = np.abs(rng.standard_normal((40, dim))).astype(np.float32)
    zero = rng.standard_normal((200, dim)).astype(np.float32)
    zero[:, 0] = 0.0
    vecs = np.concatenate([pos, zero])[rng.permutation(240)]
    ids = np.arange(240, dtype=np.int32)[::-1].copy()
    q = np.zeros((2, dim), np.float32)
    q[:, 0] = 1.0
    q[1, 0] = -1.0
    for mode in MODES:
        idx = _build(gpu_ctx, ids, vecs, mode)
        try:
            for k in (39, 40, 41, 60, 239, 240):
                _check(idx, vecs, ids, mode, q, k, False, f"{MODE_NAMES[mode]} k={k}")
        finally:
            idx.close()


def test_reference_known_answer_and_round_trip(gpu_ctx):
    """TestBuilderSearchAndRoundTrip (search/brute/index_test.go:10-36)."""
    from semantica_gpu import search
    b = search.Builder(gpu_ctx, dimension=3, quantization=search.QUANTIZE_INT8)
    for i, v in {10: [1, 0, 0], 11: [0, 1, 0], 12: [0, 0, 1]}.items():
        b.add_vector(i, v)
    idx = b.build()
    res = idx.search_vector([1, 0, 0], 2)
    assert res[0].id == 10 and len(res) == 2
    data = search.Serializer().serialize(idx)
    loaded = search.Serializer().deserialize(gpu_ctx, data)
    assert loaded.dimension() == idx.dimension() == 3
    assert loaded.count() == 3
    for i in (10, 11, 12):
        vec, ok = loaded.vector(i)
        assert ok and len(vec) == 3
    assert loaded.vector(99) == (None, False)
    idx.close()
    loaded.close()


@pytest.mark.parametrize("mode", MODES)
@pytest.mark.parametrize("dim", [5, 8, 13, 768])
def test_storage_format_byte_exact(gpu_ctx, mode, dim):
    """storage.go:47-91: "BRUT", version 1 (u16), dim (u16), count (u32),
    mode (u8), 7 zero bytes, ids (i32), row-major data -- little-endian.
    Serialize must produce exactly that; Deserialize of it must search like
    the built index; Vector must dequantize as quant.go:43-55 does."""
    from semantica_gpu import search
    rng = np.random.default_rng(dim + 10 * mode)
    n = 300
    vecs = rng.standard_normal((n, dim)).astype(np.float32)
    ids = rng.permutation(5000)[:n].astype(np.int32)
    idx = _build(gpu_ctx, ids, vecs, mode)
    data = o.bf_quantize(o.bf_normalize(vecs), mode)
    want = b"BRUT" + struct.pack("<HHIB7x", 1, dim, n, mode) + ids.tobytes() + data.tobytes()
    got = search.Serializer().serialize(idx)
    assert got == want
    loaded = search.Serializer().deserialize(gpu_ctx, want)
    q = rng.standard_normal((3, dim)).astype(np.float32)
    a, b = idx.search_batch(q, 17), loaded.search_batch(q, 17)
    assert all(np.array_equal(x, y) for x, y in zip(a, b))
    scale = {0: None, 1: np.float32(1 / 127), 2: np.float32(1 / 32767)}[mode]
    for j in (0, n // 2, n - 1):
        vec, ok = loaded.vector(int(ids[j]))
        expect = data[j].astype(np.float32) * scale if scale is not None else data[j]
        assert ok and np.array_equal(vec, expect)
    seen = []
    loaded.for_each(lambda i, v: seen.append((i, v)))
    assert [i for i, _ in seen] == ids.tolist()
    idx.close()
    loaded.close()


def test_deserialize_errors(gpu_ctx):
    """readIndex (storage.go:94-153) error cases and an empty index."""
    from semantica_gpu import SemanticaError, search
    ser = search.Serializer()
    good = b"BRUT" + struct.pack("<HHIB7x", 1, 4, 2, 1) + np.array([1, 2], np.int32).tobytes() + bytes(8)

    def err(data):
        with pytest.raises(SemanticaError) as e:
            ser.deserialize(gpu_ctx, data)
        return str(e.value)

    assert "EOF" in err(b"") and "unexpected" not in err(b"")
    assert "unexpected EOF" in err(good[:10])
    assert 'brute: invalid magic: "BRUX"' in err(b"BRUX" + good[4:])
    assert 'invalid magic: "\\x00AB\\n"' in err(b"\x00AB\n" + good[4:])
    assert "brute: unsupported version 2" in err(good[:4] + struct.pack("<H", 2) + good[6:])
    assert "EOF" in err(good[:20]) and "unexpected" not in err(good[:20])
    assert "unexpected EOF" in err(good[:22])
    assert "unexpected EOF" in err(good[:-1])
    assert "brute: unsupported quantization 3" in err(good[:12] + bytes([3]) + good[13:])
    empty = ser.deserialize(gpu_ctx, b"BRUT" + struct.pack("<HHIB7x", 1, 4, 0, 1))
    assert empty.count() == 0 and empty.search_vector([1, 0, 0, 0], 5) == []
    empty.close()
    idx = ser.deserialize(gpu_ctx, good)
    assert idx.count() == 2 and len(idx.search_vector([1, 0, 0, 0], 5)) == 2
    idx.close()


def test_builder_and_search_errors(gpu_ctx):
    """builder.go:52-80 and index.go:27-51 error cases."""
    from semantica_gpu import SemanticaError, search
    b = search.Builder(gpu_ctx, quantization=search.QUANTIZE_INT16)
    with pytest.raises(SemanticaError, match="brute: no vectors added"):
        b.build()
    b.add_vector(1, [1, 2, 3])
    with pytest.raises(SemanticaError, match="brute: duplicate id 1"):
        b.add_vector(1, [1, 2, 3])
    with pytest.raises(SemanticaError, match="brute: vector dimension mismatch: got 2 want 3"):
        b.add_vector(2, [1, 2])
    idx = b.build()
    with pytest.raises(SemanticaError, match="brute: builder already built"):
        b.build()
    with pytest.raises(SemanticaError, match="brute: topK must be positive"):
        idx.search_vector([1, 0, 0], 0)
    with pytest.raises(SemanticaError, match="brute: query dimension mismatch: got 2 want 3"):
        idx.search_vector([1, 0], 3)
    bad = search.Builder(gpu_ctx, quantization=7)
    bad.add_vector(1, [1, 0])
    with pytest.raises(SemanticaError, match="brute: unsupported quantization 7"):
        bad.build()
    idx.close()


def test_device_build_matches_host_build(gpu_ctx):
    """Index.from_device (vectors already in HBM) stores the same bytes as the
    Builder path."""
    import torch
    from semantica_gpu import search
    rng = np.random.default_rng(77)
    n, dim = 5000, 768
    vecs = rng.standard_normal((n, dim)).astype(np.float32)
    ids = np.arange(n, dtype=np.int32)
    for mode in MODES:
        host = _build(gpu_ctx, ids, vecs, mode)
        padded = torch.zeros((n, dim + 3), dtype=torch.float32, device="cuda")
        padded[:, :dim] = torch.from_numpy(vecs).cuda()
        torch.cuda.synchronize()
        devi = search.Index.from_device(gpu_ctx, ids, padded.data_ptr(), dim, n, mode, ld=dim + 3)
        ser = search.Serializer()
        assert ser.serialize(host) == ser.serialize(devi), mode
        host.close()
        devi.close()


def test_large_index(gpu_ctx):
    """300k x 768 int8 vectors (the embedding width), 40 queries in one call
    (query blocks of 8), top 10: three queries against the oracle in full, and
    every returned distance equal to the oracle's score of the returned id."""
    rng = np.random.default_rng(11)
    n, dim = 300_000, 768
    vecs = rng.standard_normal((n, dim), dtype=np.float32)
    ids = rng.permutation(n).astype(np.int32)
    queries = rng.standard_normal((40, dim), dtype=np.float32)
    say("large index build")
    idx = _build(gpu_ctx, ids, vecs, 1)
    try:
        gi, gd, gn = idx.search_batch(queries, 10)
        assert np.all(gn == 10)
        data = o.bf_quantize(o.bf_normalize(vecs), 1)
        pos = np.empty(n, np.int64)
        pos[ids] = np.arange(n)
        for q in range(40):
            qn = o.bf_normalize(queries[q])
            for j in range(10):
                s = np.float32(o.load().sgo_bf_dot(o._p(data), 1, int(pos[gi[q, j]]), o._p(qn), dim))
                assert s.view(np.uint32) == gd[q, j].view(np.uint32)
            assert np.all(np.diff(gd[q]) <= 0)
        for q in (0, 17, 39):
            say(f"large index oracle query {q}")
            wi, wd = o.bf_search(data, 1, ids, o.bf_normalize(queries[q]), 10)
            assert np.array_equal(gi[q], wi) and np.array_equal(gd[q].view(np.uint32), wd.view(np.uint32))
    finally:
        idx.close()


@pytest.mark.parametrize("mode", MODES)
@pytest.mark.parametrize("dim,n,nq,k", [
    (16, 20011, 1, 10),     # one k-step; one query
    (23, 20011, 33, 1),     # odd group count (2) and a 7-element tail; two column tiles
    (136, 17664, 40, 20),   # odd group count (17), whole blocks only
    (257, 13312, 65, 10),   # a 1-element tail; the smallest index taken at k = 10; two passes
    (768, 26001, 64, 37),
    (1300, 9000, 34, 1),    # fragments of 32 queries fill the LDS: two passes of one column tile
])
def test_prefiltered_search_matches_oracle(gpu_ctx, mode, dim, n, nq, k):
    """Indexes large enough for the matrix-core prefilter (at least twice the
    listed-block capacity): ids and distances identical to the oracle's, over
    clustered vectors (many scores close to the k-th), with queries that are
    stored vectors, and with ones the prefilter hands back: zero, not finite
    in its fp16 scaling (1e-35, 1e35), a tie straddling the k-th place (a
    vector stored twice and searched for with k = 1)."""
    rng = np.random.default_rng(dim * 7 + mode)
    topics = rng.standard_normal((12, dim)).astype(np.float32)
    vecs = (0.3 * rng.standard_normal((n, dim)) + topics[rng.integers(0, 12, n)]).astype(np.float32)
    vecs[n - 1] = vecs[5]
    ids = rng.permutation(3 * n)[:n].astype(np.int32)
    idx = _build(gpu_ctx, ids, vecs, mode)
    q = (topics[rng.integers(0, 12, nq)] + 0.4 * rng.standard_normal((nq, dim))).astype(np.float32)
    q[0] = vecs[5]
    if nq > 8:
        q[3] = 0.0
        q[5] = vecs[n // 2]
        q[6] = -vecs[7]
    say(f"prefilter mode={MODE_NAMES[mode]} dim={dim} n={n} q={nq} k={k}")
    _check(idx, vecs, ids, mode, q, k, False, "normalized by the search")
    q[nq - 1] *= np.float32(1e-35) if mode else np.float32(1e35)
    _check(idx, vecs, ids, mode, q, k, True, "as given")


@pytest.mark.parametrize("mode", MODES)
def test_prefilter_hands_back_crowded_queries(gpu_ctx, mode):
    """Vectors so alike that every block can hold one of the k best: more
    blocks than the list takes, so the queries run through the full scoring."""
    rng = np.random.default_rng(91 + mode)
    n, dim, k = 20000, 64, 10
    base = rng.standard_normal(dim)
    vecs = (base + 1e-5 * rng.standard_normal((n, dim))).astype(np.float32)
    ids = np.arange(n, dtype=np.int32)
    q = np.stack([base, base + 0.1 * rng.standard_normal(dim), rng.standard_normal(dim)]).astype(np.float32)
    say(f"crowded mode={MODE_NAMES[mode]}")
    _check(_build(gpu_ctx, ids, vecs, mode), vecs, ids, mode, q, k, False, "crowded")


@pytest.mark.parametrize("crowd", [12, 900, 1030, 3000])
@pytest.mark.parametrize("mode", MODES)
def test_prefilter_ranks_or_selects(gpu_ctx, mode, crowd):
    """Candidates that reach the cut: fewer than the 1024 that are ranked
    against each other, and more (radix selection), near the query and side by
    side; once with a tie inside the k best and once with one that straddles
    the k-th place."""
    rng = np.random.default_rng(crowd + mode)
    n, dim, k = 30000, 40, 10
    base = rng.standard_normal(dim)
    vecs = rng.standard_normal((n, dim)).astype(np.float32)
    vecs[640:640 + crowd] = base + 0.2 * rng.standard_normal((crowd, dim))
    vecs[7] = vecs[8] = base  # a tie for the first place
    vecs[9], vecs[20000] = base + 1e-3, base + 1e-3
    ids = rng.permutation(n).astype(np.int32)
    idx = _build(gpu_ctx, ids, vecs, mode)
    q = np.stack([base, base + 0.1 * rng.standard_normal(dim)]).astype(np.float32)
    say(f"crowd={crowd} mode={MODE_NAMES[mode]}")
    _check(idx, vecs, ids, mode, q, k, False, "ties inside")
    _check(idx, vecs, ids, mode, q, 1, False, "tie at the first place")
    _check(idx, vecs, ids, mode, q, 3, False, "tie at the third place")


@pytest.mark.parametrize("n", [1, 1023, 1025, 4096, 4097, 16384, 16385, 32768, 32769])
def test_selection_sizes_match_oracle(gpu_ctx, n):
    """The one-launch selection at the edges of its sizes and the general one
    past them (9 dimensions: never prefiltered), with the k-th place tied and
    not, k = 1 and k = all included."""
    rng = np.random.default_rng(n)
    vecs = rng.standard_normal((n, 9)).astype(np.float32)
    if n > 8:
        vecs[n // 2] = vecs[n - 1] = vecs[3]
    ids = rng.permutation(2 * n)[:n].astype(np.int32)
    idx = _build(gpu_ctx, ids, vecs, MODES[0])
    q = np.stack([vecs[min(3, n - 1)], rng.standard_normal(9)]).astype(np.float32)
    for k in sorted({1, 2, 3, 100, n} if n <= 1025 else {1, 2, 3, 100}):
        say(f"selection n={n} k={k}")
        _check(idx, vecs, ids, MODES[0], q, k, False, f"k={k}")


@pytest.mark.parametrize("dim,n", [(1, 3), (7, 64), (64, 65), (71, 200), (200, 129)])
@pytest.mark.parametrize("mode", MODES)
def test_build_tiles_match_oracle(gpu_ctx, mode, dim, n):
    """The tiled index build at the edges of its 64 x 64 tiles: stored codes
    byte-exact (serialized), a zero vector and one with an element past 1e19
    (its float32 square overflows) among them."""
    from semantica_gpu import search
    rng = np.random.default_rng(dim + n + mode)
    vecs = rng.standard_normal((n, dim)).astype(np.float32)
    vecs[1] = 0.0
    vecs[2, 0] = 1e20
    ids = rng.permutation(5 * n)[:n].astype(np.int32)
    raw = search.Serializer().serialize(_build(gpu_ctx, ids, vecs, mode))
    want = o.bf_quantize(o.bf_normalize(vecs), mode)
    assert raw[20 + 4 * n:] == np.ascontiguousarray(want).tobytes()


def _image(ids, data, mode):
    """A serialized index (storage.go:14-92) of rows as given: codes and norms
    that Build never stores, which a file may hold."""
    n, dim = data.shape
    head = struct.pack("<4sHHIB7x", b"BRUT", 1, dim, n, mode)
    return head + np.ascontiguousarray(ids, np.int32).tobytes() + np.ascontiguousarray(data).tobytes()


def _check_image(ctx, data, mode, queries, k, tag):
    from semantica_gpu import search
    ids = np.random.default_rng(k).permutation(2 * len(data))[:len(data)].astype(np.int32)
    idx = search.Serializer().deserialize(ctx, _image(ids, data, mode))
    try:
        for normalized in (True, False):
            gi, gd, gn = idx.search_batch(queries, k, normalized=normalized)
            for q, x in enumerate(queries):
                wi, wd = o.bf_search(data, mode, ids, x if normalized else o.bf_normalize(x), k)
                assert gn[q] == len(wi), (tag, normalized, q)
                assert np.array_equal(gi[q], wi), (tag, normalized, q)
                assert np.array_equal(gd[q].view(np.uint32), wd.view(np.uint32)), (tag, normalized, q)
    finally:
        idx.close()


@pytest.mark.parametrize("mode", MODES[1:])
@pytest.mark.parametrize("dim,n,k", [(23, 9000, 1), (20, 9800, 3), (23, 13400, 10), (257, 9000, 1), (24, 9000, 1)])
def test_prefilter_most_negative_codes(gpu_ctx, mode, dim, n, k):
    """Deserialized indexes with the most negative code, which the tail clamps
    to -127 / -32767 and the whole groups do not (quant.go:57-77,
    dot_amd64.s).  k vectors whose tails are all most negative score below one
    whose clamped tail and first element beat them, but above it by the codes
    as they are."""
    rng = np.random.default_rng(dim + k + mode)
    dt, lo, unit = ((np.int8, -128, 1), (np.int16, -32768, 256))[mode - 1]
    R = dim % 8
    data = (rng.integers(-3, 4, (n, dim)) * unit).astype(dt)
    data[rng.integers(0, n, n // 100), rng.integers(1, dim - R, n // 100)] = lo
    at = 64 * 8 * (1 + np.arange(k)) + 5  # one per block, the blocks eight apart
    best = 64 * 8 * (k + 2) + 9
    data[at, dim - R:] = lo
    data[at, 0] = -np.arange(k) * unit
    data[best, dim - R:] = lo + 1
    data[best, 0] = unit
    q = (1e-3 * rng.standard_normal((3, dim))).astype(np.float32)
    q[0, 0] = 0.5
    q[0, dim - R:] = -1.0
    q[1, dim - R:] = 1.0
    say(f"most negative codes mode={MODE_NAMES[mode]} dim={dim} k={k}")
    _check_image(gpu_ctx, data, mode, q, k, "most negative codes")


@pytest.mark.parametrize("norm,query", [(1e10, 1e30), (1e18, 1e22), (1e7, 2e29), (1e-20, 1e-25), (1e-14, 1e-30),
                                        (1e-16, 3e-26), (1e-20, 1e-20), (1e-10, 1e-10), (1e8, 1e8)])
@pytest.mark.parametrize("dim", [16, 257])
def test_prefilter_scores_outside_float32(gpu_ctx, norm, query, dim):
    """Deserialized float32 indexes searched as given, where products leave
    float32's range: scores that differ become +inf, or fall on a few steps
    of the subnormal grid or on zero, and the reference resolves these ties
    by stored order.  k strong vectors, weaker ones that tie with them, and
    the rest negative."""
    rng = np.random.default_rng(dim)
    n, k = 14000, 10
    data = np.zeros((n, dim), np.float32)
    data[:, 0] = -norm * rng.uniform(0.5, 1.0, n)
    data[:, dim - 1] = 1e-3 * norm
    data[64 * (2 * np.arange(100) + 1) + 7, 0] = norm * rng.uniform(0.8, 0.97, 100)  # other blocks than the strong ones
    data[64 * 4 * (3 + 2 * np.arange(k)) + 11, 0] = norm * rng.uniform(0.98, 1.0, k)
    q = np.zeros((3, dim), np.float32)
    q[0, 0] = query
    q[1, 0] = query * 2.2
    q[2, dim - 1] = query
    say(f"score range dim={dim} norm={norm:g} query={query:g}")
    _check_image(gpu_ctx, data, o.BF_F32, q, k, "score range")


def test_prefilter_norms_below_float32_squares(gpu_ctx):
    """Deserialized float32 vectors whose squares underflow: their norms
    (3e-22, over 1024 dimensions) are ten times that of the one vector whose
    single element's square does not.  The best vector rounds down to fp16 in
    every element, the second best up, by nearly half a unit each."""
    n, dim, k = 9000, 1024, 1
    rng = np.random.default_rng(3)
    data = (2e-25 * rng.standard_normal((n, dim))).astype(np.float32)
    unit, h, t = 2.0 ** -77, 2.0 ** -11, 2.0 ** -20  # 6.6e-24
    data[1000] = unit * (1 + h + t)
    data[5000, :512] = unit * (1 + 3 * h - t)
    data[5000, 512:] = unit * (1 + h - t)
    data[7000] = 0.0
    data[7000, 3] = 4e-23
    q = np.stack([np.full(dim, 2.0 ** 66), rng.standard_normal(dim)]).astype(np.float32)
    say("norms below float32 squares")
    _check_image(gpu_ctx, data, o.BF_F32, q, k, "tiny norms")


def test_prefilter_backs_off_from_crowded_collections(gpu_ctx):
    """Searches of one index in a row, of queries that the prefilter leaves open
    (near-duplicates) and ones that it decides, alone and in batches of several
    passes, so that searches with it and without it follow on each other."""
    rng = np.random.default_rng(17)
    n, dim, k = 20000, 64, 10
    base = rng.standard_normal(dim)
    vecs = rng.standard_normal((n, dim)).astype(np.float32)
    vecs[:15000] = base + 1e-5 * rng.standard_normal((15000, dim))
    ids = rng.permutation(n).astype(np.int32)
    idx = _build(gpu_ctx, ids, vecs, MODES[0])
    near = (base + 0.05 * rng.standard_normal((70, dim))).astype(np.float32)
    far = (-base + 0.5 * rng.standard_normal((70, dim))).astype(np.float32)
    say("back-off: crowded and clear queries in turn")
    for i, q in enumerate([near[:1], near[1:2], near[2:3], far[:1], far[1:2], near, far, np.zeros((1, dim), np.float32),
                           near[:5], far[:5], far, np.concatenate([near[:6], far[:2]]), far[2:4]]):
        _check(idx, vecs, ids, MODES[0], q, k, False, i)


@pytest.mark.parametrize("mode", MODES)
def test_prefilter_large_k(gpu_ctx, mode):
    """k at the edge of what few queries are prefiltered for, and past it with
    few and with many: selections of more candidates than are ranked against
    each other."""
    rng = np.random.default_rng(23 + mode)
    n, dim = 320000, 17
    vecs = rng.standard_normal((n, dim)).astype(np.float32)
    ids = rng.permutation(n).astype(np.int32)
    idx = _build(gpu_ctx, ids, vecs, mode)
    q = rng.standard_normal((16, dim)).astype(np.float32)
    for nq, k in ((1, 512), (3, 512), (1, 513), (16, 600)):
        say(f"large k mode={MODE_NAMES[mode]} q={nq} k={k}")
        _check(idx, vecs, ids, mode, q[:nq], k, False, (nq, k))
