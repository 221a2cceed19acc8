"""The scan and its launches on the GPU against the oracle, at the sizes where a rule changes over:
slice and window ends, kinds of pair mixed in a batch, the shares a strand's lags are split into
(to 32, 128 and 768 strands), a workgroup per channel (to 128 strands), the record counts' scan
(1024 at a time), run ordering and probabilities around their tiles.
Bar: coordinates, lengths, strands, identities bit-exact; prob within 1e-11 relative (the device's
erf/exp; keep decisions near min_prob are made on the host)."""
import numpy as np
import pytest

import oracle
from conftest import dense_run_pair
from scan_cases import GATES, LENGTHS, LETTERS, composed, related, short_runs

pytestmark = pytest.mark.gpu

EXACT = ["query_id", "target_id", "query_size", "qstart", "tstart", "len", "reverse", "ident"]


@pytest.fixture(scope="module")
def ctx():
    from satsuma2_amd.api import Context

    c = Context(0)
    yield c
    c.close()


def chunk_pairs(shapes):
    from satsuma2_amd.api import ChunkPair

    out = []
    for k, (lt, lq, letters) in enumerate(shapes):
        t, q = related(lt, lq, letters, 17 * k + 1, reverse=k % 3 == 0)
        out.append(ChunkPair(t, q, t_record=k, q_record=k, q_record_len=len(q), fast=int(k % 5 == 4)))
    return out


def check(ctx, pairs, t_chunk, target_total=1e6, resident=True):
    from satsuma2_amd.api import HomologyByXCorr, ResidentBatch, SlaveParams

    prm = SlaveParams(t_chunk=t_chunk, q_chunk=t_chunk, target_total=target_total)
    ref = oracle.align_batch([dict(tseq=p.tseq, qseq=p.qseq, t_record=p.t_record, q_record=p.q_record,
                                   q_record_len=p.q_record_len, fast=p.fast) for p in pairs],
                             oracle.make_params(N=2 * t_chunk, q_chunk=t_chunk, target_total=target_total), threads=16,
                             cap_per_pair=2048)
    ref = np.concatenate(ref)
    results = [HomologyByXCorr(ctx, prm).align_batch(pairs)]
    if resident:
        b = ResidentBatch(ctx, pairs, prm)
        b.run()
        results.append(b.results())
        b.close()
    for got in results:
        assert len(got) == len(ref)
        for f in EXACT:
            assert np.array_equal(got[f], ref[f]), f
        assert np.all(np.abs(got["prob"] - ref["prob"]) <= 1e-11 * np.abs(ref["prob"]))
    return ref


@pytest.mark.parametrize("letters", LETTERS)
@pytest.mark.parametrize("t_chunk", [1024, 2048, 4096])
def test_lengths(ctx, letters, t_chunk):
    """Diagonals around the ends of windows, words and slices (t_chunk 4096: up to 5 slices)."""
    ends = [n for n in LENGTHS] + [n + 928 * k for n in (960, 961, 962) for k in (1, 2, 3) if n + 928 * k <= t_chunk]
    shapes = [(n, (n, t_chunk, t_chunk - 31)[k % 3], letters) for k, n in enumerate(ends) if n <= t_chunk]
    assert len(check(ctx, chunk_pairs(shapes), t_chunk)) > 0


@pytest.mark.parametrize("n", [1, 16, 17, 64, 65, 128, 384, 385, 512, 513, 1025])
def test_batch_sizes(ctx, n):
    """Launch rules by the number of pairs, kinds mixed; two strands each."""
    kinds = ["acgt", "acgt", "n_gap", "few", "acgt", "dense", "words", "zero"]
    shapes = [(256 - k % 7, 256 - k % 11, kinds[k % len(kinds)]) for k in range(n)]
    check(ctx, chunk_pairs(shapes), 256)


@pytest.mark.parametrize("t_chunk", [256, 512, 1024, 2048, 4096, 8192, 16384])
@pytest.mark.parametrize("letters", ["acgt", "few"])
def test_few_pairs_of_every_length(ctx, t_chunk, letters):
    """A workgroup per channel and 16 shares per strand, odd chunk lengths, every N."""
    shapes = [(t_chunk, t_chunk, letters), (t_chunk - 1, t_chunk // 2 + 3, letters), (t_chunk // 3, t_chunk, letters)]
    assert len(check(ctx, chunk_pairs(shapes), t_chunk)) > 0


@pytest.mark.parametrize("target_total", [1.0, 30.0, 1e3])
def test_small_targets(ctx, target_total):
    """Every gate: kept runs of less than 8, 4 and 2 positions above the threshold."""
    shapes = [(700, 1000, k) for k in ("acgt", "few", "n_gap", "dense")]
    assert len(check(ctx, chunk_pairs(shapes), 1024, target_total)) > 0


@pytest.mark.parametrize("letter", [b"", b"N", b"R"])
def test_run_counts(ctx, letter):
    """A resident batch's count of runs, and more blocks than the queue holds."""
    from satsuma2_amd.api import ChunkPair, ResidentBatch, SlaveParams

    t = dense_run_pair()
    t = t[:700] + letter + t[700 + len(letter):]
    b = ResidentBatch(ctx, [ChunkPair(t, t, q_record_len=len(t))], SlaveParams(target_total=100.0))
    b.run()
    lags, runs = b.stats()
    b.close()
    want = [0, 0]
    for qs in (t, oracle.reverse_complement(t)):
        xc = oracle.xcorr(oracle.encode(t, 8192), oracle.encode(qs, 8192))
        want[0] += len(oracle.findtop(xc, 1.8))
        want[1] += len(oracle.matchup(qs, t, xc, 1.8))
    assert [lags, runs] == want


@pytest.mark.parametrize("letters", ["acgt", "n_gap", "few"])
def test_matchup_runs_and_probabilities(ctx, letters):
    """MatchUp's runs in order (tiles of 256), their probabilities (64 at a time, 16 bases each step)."""
    for n in (80, 1023, 4096):
        t, q = related(n, n, letters, n)
        xc = oracle.xcorr(oracle.encode(t, 2 * 4096), oracle.encode(q, 2 * 4096))
        ref = oracle.matchup(q, t, xc, 1.8)
        got = ctx.matchup(q, t, xc, 1.8)
        got = np.stack([got[f] for f in got.dtype.names], 1) if got.dtype.names else got
        assert np.array_equal(got, ref)
    rng = np.random.default_rng(5)
    for k in (1, 63, 64, 65, 1025):
        length = rng.choice([1, 15, 16, 17, 46, 300], k)
        runs = np.stack([rng.integers(0, len(t) - 300, k), rng.integers(0, len(q) - 300, k), length], 1).astype(np.int32)
        prob, ident = ctx.match_probability(t, q, runs, 1e6)
        for (st, sq, n), p, i in zip(runs, prob, ident):
            want = oracle.match_probability(t, q, int(st), int(sq), int(n), 1e6)
            assert p == want or abs(p - want) <= 1e-11 * abs(want) or (np.isnan(p) and np.isnan(want))
            assert i == oracle.print_match_ident(q, t, int(st), int(sq), int(n))


@pytest.mark.parametrize("odd", [b"N", b"R", b""])
def test_one_pair_of_a_rare_kind_in_a_large_batch(ctx, odd):
    """More than 2^19 pairs, one of another kind: that pair's strands are shared between 16
    workgroups each, and 2^20 strands times 16 workgroups of 256 threads are more than a launch takes.
    (odd empty: one pure pair, all others with an N.)"""
    from satsuma2_amd.api import ChunkPair, HomologyByXCorr, SlaveParams

    n, at = (1 << 19) + 9, 77777
    t, q = related(256, 256, "acgt", 3)
    other = t[:100] + (odd or b"N") + t[101:]
    seqs = {False: t if odd else other, True: other if odd else t}
    prm = SlaveParams(t_chunk=256, q_chunk=256, target_total=1e6)
    want = {}
    for rare, s in seqs.items():
        want[rare] = np.concatenate(oracle.align_batch([dict(tseq=s, qseq=q, q_record_len=256)],
                                                       oracle.make_params(N=512, q_chunk=256, target_total=1e6)))
        assert len(want[rare]) > 0
    pairs = [ChunkPair(seqs[k == at], q, q_record=k) for k in range(n)]
    print(f"[rare kind] {n} pairs, one with {odd or b'A/C/G/T only'}", flush=True)
    got = HomologyByXCorr(ctx, prm).align_batch(pairs)
    m, r = len(want[False]), len(want[True])
    assert len(got) == m * (n - 1) + r
    parts = np.concatenate([got[:m * at], got[m * at + r:]]).reshape(n - 1, m)
    ids = np.array([k for k in range(n) if k != at], np.uint64)
    for f in EXACT:
        ref = want[False][f][None, :] if f != "query_id" else ids[:, None]
        assert np.all(parts[f] == ref), f
        assert np.array_equal(got[m * at:m * at + r][f], want[True][f] if f != "query_id" else np.full(r, at, np.uint64)), f


def test_server_launches_of_mixed_kinds(ctx):
    """A serving launch holds its pairs and, behind them, their list by kind: requests with every kind
    of pair, one kind alone, full launches and a last one of a single pair."""
    from satsuma2_amd.api import Chunk, Server, SlaveParams
    from test_gpu_server import assert_records

    kinds = ["acgt", "n_gap", "few", "acgt", "dense", "words"]
    T, Q = [], []
    for k in range(24):
        t, q = related(1024 - k % 5, 1024, kinds[k % 6], 40 + k, reverse=k % 3 == 0)
        T.append((t, 700 * k, 0, 20000))
        Q.append((q[:500] + b"N" * 9 + q[509:] if k % 8 == 3 else q, 900 * k, k % 2, 30000))
    prm = SlaveParams(t_chunk=1024, q_chunk=1024, target_total=20000.0)
    srv = Server(ctx, prm, [Chunk(*c) for c in T], [Chunk(*c) for c in Q], max_pairs_per_launch=96, max_slots=2)

    def want(blocks):
        pairs = [dict(tseq=T[ti][0], qseq=Q[qi][0], t_chunk_start=T[ti][1], q_chunk_start=Q[qi][1], t_record=0,
                      q_record=Q[qi][2], q_record_len=30000, fast=f)
                 for tf, tt, qf, qt, f in blocks for qi in range(qf, qt + 1) for ti in range(tf, tt + 1)]
        return np.concatenate(oracle.align_batch(pairs, oracle.make_params(N=2048, q_chunk=1024, target_total=20000.0),
                                                 threads=16))

    requests = [[(k, k, k, k, 0)] for k in range(6)] + [[(0, 23, 0, 3, 0)], [(0, 23, 4, 8, 1), (5, 5, 5, 5, 0)], [(0, 0, 0, 2, 0)]]
    tickets = [srv.submit(r) for r in requests]
    refs = [want(r) for r in requests]
    assert sum(map(len, refs)) > 24
    for r, ticket, ref in zip(requests, tickets, refs):
        assert_records(srv.results(ticket), ref, r)
    srv.close()


@pytest.mark.parametrize("letters", ["n_gap", "few", "dense"])
@pytest.mark.parametrize("t_chunk,n", [(2048, 320), (2048, 321), (4096, 128), (4096, 171), (4096, 256), (8192, 64), (8192, 86),
                                       (8192, 128), (16384, 16), (16384, 32), (16384, 64), (16384, 86), (16384, 129)])
def test_shares_of_resident_workgroups(ctx, t_chunk, n, letters):
    """Numbers of strands around those where as many shares as before no longer fit the device at once."""
    shapes = [(t_chunk - k % 3, (t_chunk, t_chunk // 3)[k % 2], letters) for k in range(4)]
    four = chunk_pairs(shapes)
    ref = oracle.align_batch([dict(tseq=p.tseq, qseq=p.qseq, q_record_len=len(p.qseq)) for p in four],
                             oracle.make_params(N=2 * t_chunk, q_chunk=t_chunk, target_total=1e6), threads=4,
                             cap_per_pair=2048)
    from satsuma2_amd.api import ChunkPair, HomologyByXCorr, SlaveParams

    pairs = [ChunkPair(four[k % 4].tseq, four[k % 4].qseq, q_record=k) for k in range(n)]
    got = HomologyByXCorr(ctx, SlaveParams(t_chunk=t_chunk, q_chunk=t_chunk, target_total=1e6)).align_batch(pairs)
    assert np.array_equal(got["query_id"], np.repeat(np.arange(n), [len(ref[k % 4]) for k in range(n)]))
    want = np.concatenate([ref[k % 4] for k in range(n)])
    assert len(want) > 0
    for f in EXACT[1:]:
        assert np.array_equal(got[f], want[f]), f
    assert np.all(np.abs(got["prob"] - want["prob"]) <= 1e-11 * np.abs(want["prob"]))


@pytest.mark.parametrize("letters", ["acgt", "few", "words", "n_gap"])
@pytest.mark.parametrize("target_total", [g[0] for g in GATES])
def test_every_gate(ctx, target_total, letters):
    """Target sizes whose shortest kept run asks for each gate (tests/test_scan_slices.py says which)."""
    from satsuma2_amd.api import ChunkPair

    pairs = [ChunkPair(*(short_runs(500, letters, k) if k < 64 else related(900, 1000, letters, k, reverse=k % 2 == 1)),
                       t_record=k, q_record=k, q_record_len=500) for k in range(68)]
    assert len(check(ctx, pairs, 1024, target_total)) >= (3 if target_total > 1e8 else 40)


@pytest.mark.parametrize("strands", [1, 2])
@pytest.mark.parametrize("t_chunk", [0, 512])
def test_mixed_kinds_by_strands_and_lengths(ctx, strands, t_chunk):
    """The list of a mixed batch's strands, forward only too, and one list per length class (t_chunk 0)."""
    from satsuma2_amd.api import ChunkPair, HomologyByXCorr, ResidentBatch, SlaveParams

    kinds, pairs = ["acgt", "few", "n_gap", "dense", "acgt"], []
    for k in range(90):
        n = (500, 300, 900)[k % 3] if t_chunk == 0 else 512 - k % 9
        t, q = related(n, n - k % 4, kinds[(k * k) % 5], 300 + k, reverse=k % 4 == 1)
        pairs.append(ChunkPair(t, q, t_record=k, q_record=k, q_record_len=len(q)))
    want = []
    for p in pairs:
        N = 2 * t_chunk or max(512, 1 << (len(p.tseq) + len(p.qseq) - 1).bit_length())
        want += oracle.align_batch([dict(tseq=p.tseq, qseq=p.qseq, t_record=p.t_record, q_record=p.q_record,
                                         q_record_len=p.q_record_len)],
                                   oracle.make_params(N=N, strands=strands, q_chunk=512, target_total=1e6))
    want = np.concatenate(want)
    assert len(want) > 20
    prm = SlaveParams(t_chunk=t_chunk, q_chunk=512, strands=strands, target_total=1e6)
    b = ResidentBatch(ctx, pairs, prm)
    got = [HomologyByXCorr(ctx, prm).align_batch(pairs)]
    for _ in range(3):  # eager, captured, replayed
        b.run()
        got.append(b.results())
    b.close()
    for g in got:
        assert len(g) == len(want)
        for f in EXACT:
            assert np.array_equal(g[f], want[f]), f


@pytest.mark.parametrize("target_total", [1e3, 1e6, 1e9])
@pytest.mark.parametrize("t_chunk,n", [(256, 3), (256, 600), (1024, 3), (1024, 60), (2048, 30), (4096, 3), (4096, 40), (16384, 3)])
def test_slices_or_segments(ctx, t_chunk, n, target_total):
    """General pairs on both sides of slices_pay's limits, in launches of few shares and many."""
    from satsuma2_amd.api import ChunkPair

    pairs = []
    for k in range(n):
        gc, other = ((0.15, 0.0), (0.41, 0.0), (0.41, 0.004), (0.3, 0.002), (0.5, 0.02))[k % 5]
        t, q = composed(t_chunk - k % 4, t_chunk - k % 6, gc, other, 700 + k)
        pairs.append(ChunkPair(t, q, t_record=k, q_record=k, q_record_len=len(q)))
    assert len(check(ctx, pairs, t_chunk, target_total)) > 0
