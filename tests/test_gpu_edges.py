"""GPU: kernels at the sizes where their tiles end, against the CPU oracle
(integers and topics bit for bit)."""
import numpy as np
import pytest

from conftest import make_corpus
from lda_sc20_amd import ezlda
from oracle import binding as ob

pytestmark = pytest.mark.gpu

BETA = 0.01


def _pair(off, words, V, K, seed=21, z0=None, **kw):
    ctx = ezlda.Context(K=K, alpha=50.0 / K, beta=BETA, seed=seed, **kw)
    ctx.load(ezlda.Corpus(V, off, words), z0=z0)
    return ctx, ob.Oracle(K, float(np.float32(50.0 / K)), BETA, seed, V, off, words, z0=z0)


# groups of 4 values, workgroups of 64 topics, a bitmap word of 32 topics
@pytest.mark.parametrize("K", [1, 2, 3, 4, 5, 31, 32, 33, 63, 64, 65, 127, 129, 255, 257, 1023, 1025, 4099, 16383])
def test_top3_of_sparse_words(K):
    off, words = make_corpus(K, 60, 90, 50, zipf=1.2)
    for z0 in (None, np.zeros(len(words), np.uint16), (np.arange(len(words)) % min(K, 3)).astype(np.uint16)):
        # many topics without a token: equal values, ordered by topic
        ctx, orc = _pair(off, words, 90, K, z0=z0, dense_words=5)
        for x in (ctx, orc):
            x.build_wt()
            x.topk()
        assert np.array_equal(ctx.get_inv().view(np.uint32), orc.get_inv().view(np.uint32))
        assert np.array_equal(ctx.get_top(), orc.get_top())
        ctx.close()


# readback pieces: below, at and past a piece (2^19 topics) and a lane's eight
@pytest.mark.parametrize("n", [1, 7, 8, 9, 2047, 2049, (1 << 19) - 1, (1 << 19), (1 << 19) + 1, (1 << 20) + 11])
def test_topics_are_read_back_in_the_corpus_order(n):
    rng = np.random.default_rng(n)
    cuts = np.sort(rng.choice(np.arange(1, n), min(n - 1, max(1, n // 60)), replace=False)) if n > 1 else []
    off = np.concatenate([[0], cuts, [n]]).astype(np.int64)
    words = rng.integers(0, 300, n).astype(np.int32)
    z = rng.integers(0, 9, n).astype(np.uint16)
    ctx = ezlda.Context(K=9, alpha=0.5, beta=BETA, seed=1)
    ctx.load(ezlda.Corpus(300, off, words), z0=z)
    assert np.array_equal(ctx.get_topics(), z)
    ctx.close()


# where the topics stop coming through the host's loop, and a lane's eight behind it
@pytest.mark.parametrize("n", [65535, 65536, 65537, 65543, 65544, 65545])
@pytest.mark.parametrize("chunks", [1, 3])
def test_topics_of_corpora_around_the_host_readback(n, chunks):
    rng = np.random.default_rng(n)
    off = np.append(np.arange(0, n, 61, dtype=np.int64), n)
    words = rng.integers(0, 300, n).astype(np.int32)
    z = rng.integers(0, 9, n).astype(np.uint16)
    ctx = ezlda.Context(K=9, alpha=0.5, beta=BETA, seed=1, num_chunks=chunks)
    ctx.load(ezlda.Corpus(300, off, words), z0=z)
    assert np.array_equal(ctx.get_topics(), z)
    ctx.set_topics(z[::-1].copy())
    assert np.array_equal(ctx.get_topics(), z[::-1])
    ctx.close()


# items cut by cost: documents of up to 5,000 tokens holding a word hundreds of
# times, rows of more than a block per checkpoint (16- and 32-bit), and
# corpora of fewer items than workgroups; the run cap does not change a draw
@pytest.mark.parametrize("K,D,lens,kw", [
    (700, 24, (4000, 5000), {}),
    (1500, 24, (4000, 5000), {"run_cap": 7}),
    (2048, 40, (300, 5000), {"run_cap": 3, "grid_dim": 24}),
    (4096, 30, (1500, 5000), {"dense_words": 4, "grid_dim": 16}),
    (9000, 24, (2000, 5000), {"grid_dim": 16}),
    (20, 300, (1, 90), {}),
])
def test_sweeps_of_long_documents(K, D, lens, kw):
    rng = np.random.default_rng(K)
    n = rng.integers(lens[0], lens[1], D)
    off = np.concatenate([[0], np.cumsum(n)]).astype(np.int64)
    words = np.minimum(rng.geometric(0.02, int(off[-1])) - 1, 399).astype(np.int32)
    ctx, orc = _pair(off, words, 400, K, **kw)
    for s in range(2):
        ctx.sweep(1)
        orc.sweep(1)
        assert np.array_equal(ctx.get_topics(), orc.get_topics()), s
    assert abs(ctx.loglik() - orc.loglik()) <= 1e-9 * abs(orc.loglik())
    ctx.close()


# fold-in: tokens a wavefront draws (1, 2, 4 by length), pieces of 256 row
# entries, more than 64 slabs (K > 4096), empty documents
@pytest.mark.parametrize("K", [7, 64, 300, 1024, 4096, 5000, 16383])
def test_fold_in_at_the_edges_of_its_tiles(K):
    lens = [0, 1, 3, 4, 5, 63, 255, 256, 257, 512, 513, 1023, 1024, 1025, 2048, 2049, 4500]
    off, words = make_corpus(4, 200, 300, 60, zipf=1.2)
    ctx, orc = _pair(off, words, 300, K)
    ctx.sweep(2)
    orc.sweep(2)
    rng = np.random.default_rng(K)
    doff = np.concatenate([[0], np.cumsum(lens)]).astype(np.int64)
    dw = ((rng.zipf(1.2, int(doff[-1])) - 1) % 300).astype(np.int32)
    rids = np.arange(50, 50 + len(lens), dtype=np.uint32)
    zo, co = orc.foldin(doff, dw, rids, 3, 77)
    srv = ezlda.Server(ctx, max_slots=len(lens), sweeps=3, hbm_budget_bytes=1 << 22, seed=77)
    srv.submit_many(rids, doff, dw)
    for r, rid in enumerate(rids.tolist()):
        z, c, _ = srv.wait(rid, timeout_ms=60000)
        assert np.array_equal(z, zo[doff[r]: doff[r + 1]]) and np.array_equal(c, co[r]), lens[r]
        z, c = srv.plain(rid, dw[doff[r]: doff[r + 1]])
        assert np.array_equal(z, zo[doff[r]: doff[r + 1]]) and np.array_equal(c, co[r]), lens[r]
    srv.close()


# steps of more and of fewer tokens than are drawn without buckets by word
@pytest.mark.parametrize("K,D", [(128, 900), (1024, 700)])
def test_fold_in_of_a_full_house(K, D):
    off, words = make_corpus(4, 200, 300, 60, zipf=1.2)
    ctx, orc = _pair(off, words, 300, K)
    rng = np.random.default_rng(K)
    lens = rng.integers(200, 600, D)
    doff = np.concatenate([[0], np.cumsum(lens)]).astype(np.int64)
    dw = ((rng.zipf(1.2, int(doff[-1])) - 1) % 300).astype(np.int32)
    rids = np.arange(D, dtype=np.uint32)
    ctx.build_wt()
    orc.build_wt()
    orc.topk()
    zo, co = orc.foldin(doff, dw, rids, 2, 5)
    srv = ezlda.Server(ctx, max_slots=D, sweeps=2, hbm_budget_bytes=1 << 24, seed=5)
    srv.submit_many(rids, doff, dw)
    for r in rids.tolist():
        z, c, _ = srv.wait(r, timeout_ms=60000)
        assert np.array_equal(z, zo[doff[r]: doff[r + 1]]) and np.array_equal(c, co[r]), r
    assert srv.stats().max_active * 400 > 196608
    srv.close()


def _fold_in_case(K, lens, sweeps, V=300):
    """A frozen model and documents of these lengths, with the oracle's topics and counts."""
    off, words = make_corpus(4, 200, V, 60, zipf=1.2)
    ctx, orc = _pair(off, words, V, K)
    rng = np.random.default_rng(K + len(lens))
    doff = np.concatenate([[0], np.cumsum(lens)]).astype(np.int64)
    dw = ((rng.zipf(1.2, int(doff[-1])) - 1) % V).astype(np.int32)
    rids = np.arange(len(lens), dtype=np.uint32)
    ctx.build_wt()
    orc.build_wt()
    orc.topk()
    return ctx, doff, dw, rids, orc.foldin(doff, dw, rids, sweeps, 5)


def _serve(ctx, doff, dw, rids, want, sweeps, slots):
    srv = ezlda.Server(ctx, max_slots=slots, sweeps=sweeps, hbm_budget_bytes=1 << 24, seed=5)
    srv.submit_many(rids, doff, dw)
    for r in rids.tolist():
        z, c, _ = srv.wait(r, timeout_ms=60000)
        assert np.array_equal(z, want[0][doff[r]: doff[r + 1]]) and np.array_equal(c, want[1][r]), r
    st = srv.stats()
    srv.close()
    return st


# a step's tokens decide how many a wavefront draws (1, 2, 4: lines at 4,096 and 8,192)
@pytest.mark.parametrize("total", [4096, 4097, 6000, 8192, 8193])
@pytest.mark.parametrize("K", [64, 1024])
def test_fold_in_steps_by_their_tokens(K, total):
    lens = [300] * (total // 300) + [total % 300]
    ctx, doff, dw, rids, want = _fold_in_case(K, lens, 2)
    st = _serve(ctx, doff, dw, rids, want, 2, len(lens))
    assert st.max_active == len(lens)  # all in one step


# documents in flight while the steps go from unbucketed to bucketed and back: half of them are admitted at a time
@pytest.mark.parametrize("K", [128, 1024])
def test_fold_in_steps_change_their_path(K):
    lens = np.random.default_rng(K).integers(120, 360, 840)
    ctx, doff, dw, rids, want = _fold_in_case(K, lens, 4)
    st = _serve(ctx, doff, dw, rids, want, 4, len(lens))
    assert st.max_active == len(lens) and int(doff[-1]) > 196608 > int(doff[430])


# a long row among short documents: a launch of its own (16,383 topics, more workgroups than the CUs hold), and
# steps of few workgroups or of rows that leave room, in one
@pytest.mark.parametrize("K,short,long", [(16383, 60, 20000), (16383, 5, 20000), (16383, 60, 4097), (9000, 130, 16500)])
def test_fold_in_of_a_long_row_among_short_ones(K, short, long):
    lens = np.random.default_rng(K).integers(200, 400, short)
    lens = np.concatenate([lens[: short // 2], [long], lens[short // 2:], [0]])
    ctx, doff, dw, rids, want = _fold_in_case(K, lens, 2)
    _serve(ctx, doff, dw, rids, want, 2, len(lens))


# words of few tokens drawn by groups (K <= 512): slabs and topics that fill no
# whole load, groups of dense words, of sparse words and at the border of the
# two, unused words, long words between; stages in any order
@pytest.mark.parametrize("K", [1, 2, 5, 20, 63, 64, 65, 127, 130, 256, 300, 512, 513])
@pytest.mark.parametrize("kw", [{"dense_words": 0}, {"dense_words": 37, "run_cap": 2}, {"dense_words": 10**6},
                                {"grid_dim": 24, "shortcut": 0}])
def test_groups_of_small_words(K, kw):
    rng = np.random.default_rng(K)
    n = rng.integers(1, 120, 90)
    off = np.concatenate([[0], np.cumsum(n)]).astype(np.int64)
    words = np.where(rng.random(int(off[-1])) < 0.3, rng.integers(0, 3, int(off[-1])),
                     rng.integers(0, 1500, int(off[-1]))).astype(np.int32)
    ctx, orc = _pair(off, words, 1600, K, **kw)
    for s in range(2):
        ctx.sweep(1)
        orc.sweep(1)
        assert np.array_equal(ctx.get_topics(), orc.get_topics()), s
        assert abs(ctx.loglik() - orc.loglik()) <= 1e-9 * abs(orc.loglik())
    for stages in (("sample_tail", "shortcut", "sample_head"), ("shortcut", "sample_head", "sample_tail")):
        ctx.build_wt()
        ctx.topk()
        ctx.build_dt()
        for name in stages:
            getattr(ctx, name)()
        ctx.commit_head()
        orc.sweep(1)
        assert np.array_equal(ctx.get_topics(), orc.get_topics()), stages
    ctx.set_layout(block_dim=128)  # no groups there
    ctx.sweep(1)
    orc.sweep(1)
    assert np.array_equal(ctx.get_topics(), orc.get_topics())
    ctx.close()


@pytest.mark.parametrize("D,V,mean,chunks,run_cap", [(3, 2, 300, 3, 32),      # runs of every length, chunks of one document
                                                     (700, 1, 3, 2, 4),       # one word: items of many runs, empty documents
                                                     (129, 4000, 40, 2, 1),   # runs of one token
                                                     (2500, 30, 25, 2, 5)])   # items above and below 64 runs
def test_chunk_layouts_made_on_the_device(D, V, mean, chunks, run_cap):
    """A chunk's runs, ordered and numbered on the device from their slots and
    lengths: topics, model and draw counts equal to the resident layout's and
    the oracle's (exact)."""
    rng = np.random.default_rng(D)
    lens = rng.integers(0, 2 * mean + 1, D)
    lens[0] = mean
    off = np.concatenate([[0], np.cumsum(lens)]).astype(np.int64)
    words = np.minimum(rng.integers(0, V, off[-1]), rng.integers(0, V, off[-1])).astype(np.int32)
    K = 48
    res = ezlda.Context(K=K, alpha=50.0 / K, beta=0.01, seed=9, run_cap=run_cap)
    chk = ezlda.Context(K=K, alpha=50.0 / K, beta=0.01, seed=9, run_cap=run_cap, num_chunks=chunks)
    orc = ob.Oracle(K, float(np.float32(50.0 / K)), 0.01, 9, V, off, words)
    for c in (res, chk):
        c.load(ezlda.Corpus(V, off, words))
        c.sweep(3)
    orc.sweep(3)
    assert np.array_equal(chk.get_topics(), orc.get_topics())
    assert np.array_equal(res.get_topics(), orc.get_topics())
    assert abs(chk.loglik() - res.loglik()) <= 1e-9 * abs(res.loglik())
    chk.set_topics(orc.get_topics())
    chk.sweep(1)
    orc.sweep(1)
    assert np.array_equal(chk.get_topics(), orc.get_topics())
    assert chk.info().num_chunks == min(chunks, D)


# half wavefronts of words of up to 128 tokens beside workgroups of larger
# ones (32-bit rows): 31 to 33 and 127 to 129 tokens, an odd and an even number
# of words, words cut by block_dim, rows past the checkpoints
@pytest.mark.parametrize("K,kw", [(8192, {}), (8193, {}), (8256, {"shortcut": 0}), (10000, {"grid_dim": 0}),
                                  (16383, {}), (16383, {"block_dim": 64, "run_cap": 1})])
@pytest.mark.parametrize("odd", [0, 1])
def test_words_of_few_tokens_at_large_k(K, kw, odd):
    rng = np.random.default_rng(K + odd)
    counts = np.array([700, 300, 257, 256, 130, 129, 128, 128, 127, 65, 64, 63, 33, 32, 31] + [5] * 20 + [1] * (30 + odd))
    bag = np.repeat(rng.permutation(len(counts)), counts)  # the words' order of frequency is not that of their numbers
    rng.shuffle(bag)
    lens = np.concatenate([[len(bag) // 2], rng.multinomial(len(bag) - len(bag) // 2, np.ones(90) / 90)])
    off = np.concatenate([[0], np.cumsum(lens)]).astype(np.int64)
    for z0 in (None, (np.arange(len(bag)) % 7).astype(np.uint16)):
        ctx, orc = _pair(off, bag.astype(np.int32), len(counts), K, z0=z0, dense_words=2, **kw)
        for n in (1, 2):
            ctx.sweep(n)
            orc.sweep(n)
            assert np.array_equal(ctx.get_topics(), orc.get_topics()), n
        ctx.sweep_graph(2)
        orc.sweep(2)
        assert np.array_equal(ctx.get_topics(), orc.get_topics())


# enough of them for the launch of half wavefronts (32, 14 or 10 a CU of 256, as
# four, three or two of the sampler's tables fit a CU), and one less
@pytest.mark.parametrize("K,n", [(8200, 8191), (8200, 8192), (10000, 3583), (10000, 3584), (16383, 2559), (16383, 2560)])
def test_many_words_of_few_tokens_at_large_k(K, n):
    rng = np.random.default_rng(K + n)
    counts = np.concatenate([[900, 400, 200, 129], np.full(9, 128), rng.integers(1, 7, n - 9)])
    bag = rng.permutation(np.repeat(rng.permutation(len(counts)), counts)).astype(np.int32)
    off = np.linspace(0, len(bag), 301).astype(np.int64)
    ctx, orc = _pair(off, bag, len(counts), K, dense_words=2)
    for n in (1, 2):
        ctx.sweep(n)
        orc.sweep(n)
        assert np.array_equal(ctx.get_topics(), orc.get_topics()), n
    ctx.close()


# dense rows of one segment (32,768 tokens) are written whole, of several added
# up; words without a token; K with and without 16-byte rows
@pytest.mark.parametrize("K", [64, 65, 1026, 2600])
def test_dense_rows_with_and_without_tokens(K):
    rng = np.random.default_rng(K)
    counts = [65537, 32769, 32768, 700, 3, 1, 1]
    bag = rng.permutation(np.repeat(rng.permutation(len(counts)), counts)).astype(np.int32)
    off = np.linspace(0, len(bag), 41).astype(np.int64)
    V = len(counts) + 5  # five words of the vocabulary do not occur
    for dense in (V, 4):
        ctx, orc = _pair(off, bag, V, K, dense_words=dense)
        for _ in range(2):
            for c in (ctx, orc):
                c.sweep(1)
                c.build_wt()
                c.topk()
            assert np.array_equal(ctx.get_topics(), orc.get_topics())
            assert np.array_equal(ctx.get_wt_dense(), orc.get_wt_dense())
            assert np.array_equal(ctx.get_nk(), orc.get_nk()) and np.array_equal(ctx.get_top(), orc.get_top())


# where rows are sorted instead of counted (K > 4819): tail words and documents
# of 0, 1 and 64, 128, 256, 512 topics and one more or less, equal and distinct
@pytest.mark.parametrize("K", [4800, 4900, 8193, 16383])
def test_rows_of_sorted_topics(K):
    sizes = [1, 2, 63, 64, 65, 127, 128, 129, 255, 256, 257, 511, 512, 513, 600]
    rng = np.random.default_rng(K)
    words = rng.permutation(np.repeat(np.arange(len(sizes)), sizes)).astype(np.int32)
    rest = len(words) - sum(sizes[:-2])
    off = np.concatenate([[0, 0], np.cumsum(sizes[:-2] + [rest // 2, rest - rest // 2])]).astype(np.int64)
    for z0 in (None, np.full(len(words), K - 1, np.uint16), (np.arange(len(words)) % 5).astype(np.uint16)):
        ctx, orc = _pair(off, words, len(sizes) + 1, K, z0=z0, dense_words=0)
        for c in (ctx, orc):
            c.build_wt()
            c.topk()
        assert np.array_equal(ctx.get_wt_dense(), orc.get_wt_dense())
        assert np.array_equal(ctx.get_top(), orc.get_top())
        for n in (1, 2):
            ctx.sweep(n)
            orc.sweep(n)
            assert np.array_equal(ctx.get_topics(), orc.get_topics())
        assert abs(ctx.loglik() - orc.loglik()) <= 1e-9 * abs(orc.loglik())


# tail words none of which is longer than those sorted; and beside longer words as
# many short ones as are counted with them (2^31 / K^2 a CU of 256), and one more
@pytest.mark.parametrize("K,longer,short", [(4900, 0, 0), (16383, 0, 0), (8000, 2, 8589), (8000, 2, 8590), (16383, 2, 2048), (16383, 2, 2049)])
def test_rows_sorted_beside_rows_counted(K, longer, short):
    sizes = [1, 2, 63, 64, 65, 127, 128, 129, 255, 256, 257, 511, 512]
    counts = [700, 513][:longer] + sizes + [1] * (short - len(sizes))
    rng = np.random.default_rng(K + short)
    words = rng.permutation(np.repeat(rng.permutation(len(counts)), counts)).astype(np.int32)
    off = np.linspace(0, len(words), 101).astype(np.int64)
    ctx, orc = _pair(off, words, len(counts) + 1 if short == 0 else len(counts), K, dense_words=0)
    for n in (1, 2):
        for c in (ctx, orc):
            c.sweep(n)
            c.build_wt()
            c.topk()
        assert np.array_equal(ctx.get_topics(), orc.get_topics())
        assert np.array_equal(ctx.get_top(), orc.get_top())
    assert abs(ctx.loglik() - orc.loglik()) <= 1e-9 * abs(orc.loglik())
    ctx.close()


# DT rows compacted 128 topics a step (K <= 1024), from a bitmap above it;
# counts below, at and above one entry's 63 (K <= 1024), 31 and 15
@pytest.mark.parametrize("K", [1, 2, 3, 64, 127, 128, 129, 255, 257, 1023, 1024, 1025, 2049])
def test_rows_of_many_counts(K):
    n = np.array([0, 1, 63, 64, 65, 126, 127, 300, 513, 700])
    off = np.concatenate([[0], np.cumsum(n)]).astype(np.int64)
    words = (np.arange(off[-1]) * 7 % 50).astype(np.int32)
    last = np.full(off[-1], K - 1, np.uint16)
    pair = (np.arange(off[-1]) % 130 < 65) * (K - 1)  # two topics, next to each other's counts in turn
    spread = np.arange(off[-1]) * 5 % K
    for z0 in (last, pair.astype(np.uint16), spread.astype(np.uint16)):
        ctx, orc = _pair(off, words, 50, K, z0=z0)
        for c in (1, 2):
            ctx.sweep(c)
            orc.sweep(c)
            assert np.array_equal(ctx.get_topics(), orc.get_topics()), c
        for c in (ctx, orc):
            c.build_wt()
            c.topk()
            c.build_dt()
        (ge, gn), (oe, on) = ctx.get_dt_raw(), orc.get_dt_raw()
        assert np.array_equal(gn, on)
        for d, b in enumerate(ezlda.dt_offsets(off, K)[: len(gn)]):
            assert np.array_equal(ge[b: b + gn[d]], oe[b: b + gn[d]]), d
        assert np.array_equal(ctx.get_aux(), orc.get_aux())
